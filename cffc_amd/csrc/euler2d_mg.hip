// euler2d_mg.hip -- the level-transfer kernels of the FAS multigrid solver
// (FASMultigrid2D/FASMultigrid2D.h), gfx950.
//
// Each multigrid level is its own context (padded SoA layout, BlockMeta per
// block); level l+1 halves level l block by block, so coarse cell (ic, jc)
// of block b (padded indices, 2 ghost layers) covers the fine cells
// (2*(ic-2)+2 + {0,1}, 2*(jc-2)+2 + {0,1}) of block b.  One thread per coarse
// interior cell (grid: x over the block's coarse cells, y over blocks), FP64,
// built with -ffp-contract=off in the reference's operation order.  These are
// memory-bound elementwise passes over a level (tens of bytes per cell) next
// to the stage kernels' hundreds of flops per cell.
#include <hip/hip_runtime.h>

#include "euler2d_device.hpp"
#include "euler2d_kernels.hpp"
#include "euler2d_state.hpp"

namespace cffc {

namespace {

__device__ __forceinline__ int64_t cell(const BlockMeta &m, int i, int j) { return m.coff + (int64_t)j * m.pitch + i; }

__device__ __forceinline__ CS<double> ldU(const double *U, int64_t ncp, int64_t c) {
    CS<double> u = {U[c], U[ncp + c], U[2 * ncp + c], U[3 * ncp + c]};
    return u;
}
__device__ __forceinline__ void stU(double *U, int64_t ncp, int64_t c, const CS<double> &u) {
    U[c] = u.d; U[ncp + c] = u.mx; U[2 * ncp + c] = u.my; U[3 * ncp + c] = u.E;
}

// Restrict_Solution_Blocks :996-1037 (U -> Uc, with Update_Primitive_Variables
// :2423-2445 into Wc) and, where R is given, Restrict_Residuals :1053-1095
// (R -> P): the area-weighted average of the four fine cells, SW, SE, NW, NE
// in that order.  One pass: both averages share the areas and their quotients
// the coarse area's reciprocal.
__global__ void mg_restrict_kernel(const BlockMeta *mf, const BlockMeta *mc, const double *U, const double *R,
                                   const double *Af, int64_t ncpf, double *Uc, double *Wc, double *P, const double *Ac,
                                   int64_t ncpc) {
    const BlockMeta f = mf[blockIdx.y], c = mc[blockIdx.y];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= c.ni * c.nj || c.skip) return;
    const int ic = q % c.ni + 2, jc = q / c.ni + 2;
    const int i0 = 2 * (ic - 2) + 2, j0 = 2 * (jc - 2) + 2;
    const int64_t q0 = cell(f, i0, j0), q1 = q0 + 1, q2 = q0 + f.pitch, q3 = q2 + 1;
    const double A0 = Af[q0], A1 = Af[q1], A2 = Af[q2], A3 = Af[q3];
    const int64_t cc = cell(c, ic, jc);
    const Recip<double> rA = recip(Ac[cc]);
    auto average = [&](const double *src, int v) {
        const double *s = src + v * ncpf;
        return rdiv(s[q0] * A0 + s[q1] * A1 + s[q2] * A2 + s[q3] * A3, rA);
    };
    const CS<double> u = {average(U, 0), average(U, 1), average(U, 2), average(U, 3)};
    stU(Uc, ncpc, cc, u);
    const PS<double> w = W_of_U(u);
    Wc[cc] = w.d; Wc[ncpc + cc] = w.vx; Wc[2 * ncpc + cc] = w.vy; Wc[3 * ncpc + cc] = w.p;
    if (R) {
#pragma unroll
        for (int v = 0; v < 4; ++v) P[v * ncpc + cc] = average(R, v);
    }
}

// Evaluate_Solution_Changes :2454-2478 over every cell of each block,
// ghosts included (U -= uo); a converged case of a batch is skipped
__global__ void mg_changes_kernel(const BlockMeta *meta, double *U, const double *uo, int64_t ncp) {
    const BlockMeta m = meta[blockIdx.y];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m.nci * m.ncj || m.skip) return;
    const int64_t c = cell(m, q % m.nci, q / m.nci);
#pragma unroll
    for (int v = 0; v < 4; ++v) U[v * ncp + c] -= uo[v * ncp + c];
}

// uo = U over every cell of each block, ghosts included
// (Store_Current_Solution_in_uo_MG); a kernel rather than a copy node, so
// that a captured cycle holds kernels only
__global__ void mg_copy_kernel(const BlockMeta *meta, double *dst, const double *src, int64_t ncp) {
    const BlockMeta m = meta[blockIdx.y];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m.nci * m.ncj || m.skip) return;
    const int64_t c = cell(m, q % m.nci, q / m.nci);
#pragma unroll
    for (int v = 0; v < 4; ++v) dst[v * ncp + c] = src[v * ncp + c];
}

// Bilinear_Interpolation, CFD.h:1367-1416 (Zingg and Yarrow)
__device__ bool bilinear(const CS<double> &U1, double x1, double y1, const CS<double> &U2, double x2, double y2,
                         const CS<double> &U3, double x3, double y3, const CS<double> &U4, double x4, double y4,
                         double x0, double y0, CS<double> &U0) {
    const double TOL = 0.0000001;
    const double a0 = x1, a1 = x4 - x1, a2 = x2 - x1, a3 = x1 + x3 - x2 - x4;
    const double b0 = y1, b1 = y4 - y1, b2 = y2 - y1, b3 = y1 + y3 - y2 - y4;
    const double a = a1 * b3 - a3 * b1;
    const double b = a0 * b3 - b3 * x0 + a1 * b2 - a2 * b1 + a3 * y0 - a3 * b0;
    const double c = a0 * b2 - b2 * x0 + a2 * y0 - a2 * b0;
    double zeta0;
    if (a > TOL || a < -TOL) {
        if (b * b - 4.0 * a * c < 0.0) return false;
        zeta0 = (-b + sqrt(b * b - 4.0 * a * c)) / (2.0 * a);
        if (zeta0 < 0.0 || zeta0 > 1.0) {
            zeta0 = (-b - sqrt(b * b - 4.0 * a * c)) / (2.0 * a);
            if (zeta0 < 0.0 || zeta0 > 1.0) return false;
        }
    } else if (b > TOL || b < -TOL) {
        zeta0 = -c / b;
        if (zeta0 < 0.0 || zeta0 > 1.0) return false;
    } else {
        return false;
    }
    if (b2 + b3 * zeta0 < TOL && b2 + b3 * zeta0 > -TOL) return false;
    const double eta0 = (y0 - b0 - b1 * zeta0) / (b2 + b3 * zeta0);
    U0.d = U1.d + (U4.d - U1.d) * zeta0 + (U2.d - U1.d) * eta0 + (U1.d + U3.d - U2.d - U4.d) * zeta0 * eta0;
    U0.mx = U1.mx + (U4.mx - U1.mx) * zeta0 + (U2.mx - U1.mx) * eta0 + (U1.mx + U3.mx - U2.mx - U4.mx) * zeta0 * eta0;
    U0.my = U1.my + (U4.my - U1.my) * zeta0 + (U2.my - U1.my) * eta0 + (U1.my + U3.my - U2.my - U4.my) * zeta0 * eta0;
    U0.E = U1.E + (U4.E - U1.E) * zeta0 + (U2.E - U1.E) * eta0 + (U1.E + U3.E - U2.E - U4.E) * zeta0 * eta0;
    return true;
}

__device__ __forceinline__ bool unphysical(const CS<double> &U) { return U.d <= 0.0 || U.E <= 0.0 || U_e(U) <= 0.0; }

// interpolation quadrilaterals per fine cell (SW, SE, NE, NW), by the offset
// of the quadrilateral's SW coarse cell (:1718-2211)
__constant__ int8_t kQuad[4][4][2] = {
    {{-1, -1}, {-1, 0}, {0, -1}, {0, 0}},
    {{0, -1}, {0, 0}, {-1, -1}, {-1, 0}},
    {{0, 0}, {0, -1}, {-1, 0}, {-1, -1}},
    {{-1, 0}, {0, 0}, {-1, -1}, {0, -1}},
};

// Prolong_and_Update_Solution_Blocks :1627-2213.  Uc: the coarse solution
// change (ghosts included).  A coarse cell next to a fixed boundary injects
// into its four fine cells; otherwise each fine cell interpolates from the
// first quadrilateral that contains it, and a cell none contains restarts
// the coarse cell with injection from the SW fine cell (cells already
// updated are updated again, as in the reference).  Updates that leave the
// state unphysical are halved up to max_red times, then dropped.  Wf (if not
// null) takes the fine cells' W(U) (Update_Primitive_Variables).
//
// neumann: a ghost cell of the interior span next to a constant-extrapolation
// boundary takes the adjacent interior change (:1640-1669).
//
// assign (Prolong_Solution_Blocks :1200-1625, full multigrid): Uc is the
// coarse solution; the fine cells take it (same quadrilateral order and
// injection fall-back), with neither Dirichlet injection nor reduction.
__global__ void mg_prolong_kernel(const BlockMeta *mc, const BlockMeta *mf, const int32_t *bc, const double *Uc,
                                  const double *gc, int64_t ncpc, double *Uf, double *Wf, const double *gf,
                                  int64_t ncpf, int neumann, int inj_dirichlet, int inj_always, int stability,
                                  int max_red, int assign) {
    const BlockMeta c = mc[blockIdx.y], f = mf[blockIdx.y];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= c.ni * c.nj || c.skip) return;
    const int ic = q % c.ni + 2, jc = q / c.ni + 2;
    const int i0 = 2 * (ic - 2) + 2, j0 = 2 * (jc - 2) + 2;
    const int32_t *bW = bc + c.bcoff, *bE = bW + c.ncj, *bS = bE + c.ncj, *bN = bS + c.nci;
    const CS<double> Ucc = ldU(Uc, ncpc, cell(c, ic, jc));
    // the coarse change at (a, e)
    auto change = [&](int a, int e) {
        if (neumann) {
            if (e >= 2 && e <= c.nj + 1) {
                if (a == c.ni + 2 && bE[e] == 4001) a = c.ni + 1;
                else if (a == 1 && bW[e] == 4001) a = 2;
            } else if (a >= 2 && a <= c.ni + 1) {
                if (e == 1 && bS[a] == 4001) e = 2;
                else if (e == c.nj + 2 && bN[a] == 4001) e = c.nj + 1;
            }
        }
        return ldU(Uc, ncpc, cell(c, a, e));
    };
    auto primitive = [&](int64_t fc, const CS<double> &u) {
        if (!Wf) return;
        const PS<double> w = W_of_U(u);
        Wf[fc] = w.d; Wf[ncpf + fc] = w.vx; Wf[2 * ncpf + fc] = w.vy; Wf[3 * ncpf + fc] = w.p;
    };
    const int fdi[4] = {0, 1, 1, 0}, fdj[4] = {0, 0, 1, 1};
    const bool dirichlet = (ic == 2 && bW[jc] == 11000) || (ic == c.ni + 1 && bE[jc] == 11000) ||
                           (jc == 2 && bS[ic] == 11000) || (jc == c.nj + 1 && bN[ic] == 11000);
    if (!assign && inj_dirichlet && dirichlet) {
        for (int k = 0; k < 4; ++k) {
            const int64_t fc = cell(f, i0 + fdi[k], j0 + fdj[k]);
            CS<double> u = ldU(Uf, ncpf, fc);
            u.d += Ucc.d; u.mx += Ucc.mx; u.my += Ucc.my; u.E += Ucc.E;
            stU(Uf, ncpf, fc, u);
            primitive(fc, u);
        }
        return;
    }
    const double *xc = gc + GEO_XC * ncpc, *yc = gc + GEO_YC * ncpc;
    bool inject = inj_always != 0;
    for (int k = 0; k < 4; ++k) {
        const int64_t fc = cell(f, i0 + fdi[k], j0 + fdj[k]);
        CS<double> dU;
        if (!inject) {
            bool ok = false;
            for (int t = 0; t < 4 && !ok; ++t) {
                const int a = ic + kQuad[k][t][0], e = jc + kQuad[k][t][1];
                const int64_t p1 = cell(c, a, e), p2 = p1 + c.pitch, p3 = p2 + 1, p4 = p1 + 1;
                ok = bilinear(change(a, e), xc[p1], yc[p1], change(a, e + 1), xc[p2], yc[p2], change(a + 1, e + 1),
                              xc[p3], yc[p3], change(a + 1, e), xc[p4], yc[p4], gf[GEO_XC * ncpf + fc],
                              gf[GEO_YC * ncpf + fc], dU);
            }
            if (!ok) {
                inject = true;
                k = -1;   // restart the coarse cell with injection
                continue;
            }
        } else {
            dU = Ucc;
        }
        if (assign) {
            stU(Uf, ncpf, fc, dU);
            continue;
        }
        CS<double> u = ldU(Uf, ncpf, fc);
        if (stability) {
            CS<double> un = {u.d + dU.d, u.mx + dU.mx, u.my + dU.my, u.E + dU.E};
            if (unphysical(un)) {
                int n = 1;
                while (n <= max_red) {
                    dU.d *= 0.5; dU.mx *= 0.5; dU.my *= 0.5; dU.E *= 0.5;
                    CS<double> um = {u.d + dU.d, u.mx + dU.mx, u.my + dU.my, u.E + dU.E};
                    if (!unphysical(um)) break;
                    n++;
                }
                if (n > max_red) { dU.d = 0.0; dU.mx = 0.0; dU.my = 0.0; dU.E = 0.0; }
            }
        }
        u.d += dU.d; u.mx += dU.mx; u.my += dU.my; u.E += dU.E;
        stU(Uf, ncpf, fc, u);
        primitive(fc, u);   // a restarted cell's last write is its final state
    }
}

// ---------------------------------------------------------------------------
// Smoothing of a first-order level (HLLE, zero limiter, so a face takes the
// states of its two cells): a cell needs its four neighbours and nothing else,
// which the host lists per cell across blocks.  No window, no LDS, no ghost cells,
// two dependent loads to the states; the price is that both cells of a face
// evaluate its flux.  The launches of the coarse levels are bound by that load
// chain (a 12,288-cell case: 9.6 us a stage with windows, whatever the level).
struct FirstCell {
    PS<double> W;
    double A, lW, lE, lS, lN, nWx, nWy, nEx, nEy, nSx, nSy, nNx, nNy;
};
__device__ __forceinline__ void load_geometry(const FirstArgs &a, const MgCell &k, FirstCell &f) {
    const double *G = a.geom;
    const int64_t n = a.ncp, c = k.c, w = k.c - 1, s = k.south;
    f.A = G[GEO_A * n + c];
    f.lW = G[GEO_LE * n + w]; f.lE = G[GEO_LE * n + c]; f.lS = G[GEO_LN * n + s]; f.lN = G[GEO_LN * n + c];
    f.nWx = G[GEO_NEX * n + w]; f.nWy = G[GEO_NEY * n + w]; f.nEx = G[GEO_NEX * n + c]; f.nEy = G[GEO_NEY * n + c];
    f.nSx = G[GEO_NNX * n + s]; f.nSy = G[GEO_NNY * n + s]; f.nNx = G[GEO_NNX * n + c]; f.nNy = G[GEO_NNY * n + c];
}
// flux through the face to neighbour state Wn, or to the boundary entry -(nb + 1)
// of the bc / wo arrays; (nx, ny): the face's normal (E or N of its low cell), low:
// this cell is on the high side
__device__ __forceinline__ CS<double> first_flux(const FirstArgs &a, const PS<double> &Wc, PS<double> Wn, int nb, bool low,
                                                 double nx, double ny) {
    if (nb < 0) {
        const int e = -(nb + 1), t = a.bc[e];
        const PS<double> wo = {a.wo[4 * (int64_t)e], a.wo[4 * (int64_t)e + 1], a.wo[4 * (int64_t)e + 2],
                               a.wo[4 * (int64_t)e + 3]};
        const double sg = low ? -1.0 : 1.0;   // outward
        if (t == 7001) Wn = reflect(Wc, sg * nx, sg * ny);
        else if (t == 8001) Wn = bc_characteristic_pressure(Wc, wo, sg * nx, sg * ny);
        else if (t == 11000) Wn = wo;
        else Wn = Wc;
    }
    return low ? flux_hlle_n(Wn, Wc, nx, ny) : flux_hlle_n(Wc, Wn, nx, ny);
}
// (CFL dt)(+W -E +S -N)/A + (CFL dt) P, in the stage kernel's order
template <typename State>
__device__ __forceinline__ void first_residual(const FirstArgs &a, const FirstCell &f, const int (&nb)[4], double cdt,
                                               const double (&P)[4], State state, double (&dU)[4]) {
    const Recip<double> rA = recip(f.A);
    CS<double> F = first_flux(a, f.W, state(0), nb[0], true, f.nWx, f.nWy);
    dU[0] = 0.0 + rdivf(cdt * F.d * f.lW, rA); dU[1] = 0.0 + rdivf(cdt * F.mx * f.lW, rA);
    dU[2] = 0.0 + rdivf(cdt * F.my * f.lW, rA); dU[3] = 0.0 + rdivf(cdt * F.E * f.lW, rA);
    F = first_flux(a, f.W, state(1), nb[1], false, f.nEx, f.nEy);
    dU[0] -= rdivf(cdt * F.d * f.lE, rA); dU[1] -= rdivf(cdt * F.mx * f.lE, rA);
    dU[2] -= rdivf(cdt * F.my * f.lE, rA); dU[3] -= rdivf(cdt * F.E * f.lE, rA);
    F = first_flux(a, f.W, state(2), nb[2], true, f.nSx, f.nSy);
    dU[0] += rdivf(cdt * F.d * f.lS, rA); dU[1] += rdivf(cdt * F.mx * f.lS, rA);
    dU[2] += rdivf(cdt * F.my * f.lS, rA); dU[3] += rdivf(cdt * F.E * f.lS, rA);
    F = first_flux(a, f.W, state(3), nb[3], false, f.nNx, f.nNy);
    dU[0] -= rdivf(cdt * F.d * f.lN, rA); dU[1] -= rdivf(cdt * F.mx * f.lN, rA);
    dU[2] -= rdivf(cdt * F.my * f.lN, rA); dU[3] -= rdivf(cdt * F.E * f.lN, rA);
    if (a.P) {
#pragma unroll
        for (int v = 0; v < 4; ++v) dU[v] += cdt * P[v];
    }
}
// update_kernel's rule; returns W^(s+1), Wc where the state stays unphysical
__device__ __forceinline__ PS<double> first_update(const FirstArgs &a, const MgCell &k, const CS<double> &U0, double om,
                                                   const PS<double> &Wc, double &dtl, double (&dU)[4], CS<double> &Un) {
    Un = {U0.d + om * dU[0], U0.mx + om * dU[1], U0.my + om * dU[2], U0.E + om * dU[3]};
    bool bad = unphysical(Un);
    if (bad && a.halve) {
        double f = 1.0;
        for (int n = 1; n <= 10; ++n) {
            f = 0.5 * f;
            dtl = f * dtl;
#pragma unroll
            for (int v = 0; v < 4; ++v) dU[v] = f * dU[v];
            Un = {U0.d + om * dU[0], U0.mx + om * dU[1], U0.my + om * dU[2], U0.E + om * dU[3]};
            if (!unphysical(Un)) break;
        }
        bad = unphysical(Un);
    }
    if (bad) atomicMin(a.err, ((unsigned long long)(unsigned)k.blk << 32) | (unsigned long long)(unsigned)k.ji);
    return bad ? Wc : W_of_U(Un);
}
__device__ __forceinline__ PS<double> ldW4(const double *W, int64_t ncp, int64_t c) {
    return {W[c], W[ncp + c], W[2 * ncp + c], W[3 * ncp + c]};
}

// one smoothing stage of a level, one thread per cell, from Win to Wout
__global__ __launch_bounds__(256) void mg_first_step_kernel(FirstArgs a, double om, int first_stage) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= a.n) return;
    const MgCell k = a.cells[q];
    if (a.meta[k.blk].skip) return;
    const int4 n4 = a.nb[q];
    const int nb[4] = {n4.x, n4.y, n4.z, n4.w};
    const int64_t ncp = a.ncp, c = k.c;
    FirstCell f;
    f.W = ldW4(a.Win, ncp, c);
    PS<double> Wn[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) Wn[s] = ldW4(a.Win, ncp, nb[s] >= 0 ? nb[s] : k.c);
    load_geometry(a, k, f);
    const CS<double> U0 = ldU(first_stage ? a.U : a.Uo, ncp, c);
    double P[4] = {0.0, 0.0, 0.0, 0.0}, dtl = a.dt[c], dU[4];
    if (a.P) {
#pragma unroll
        for (int v = 0; v < 4; ++v) P[v] = a.P[v * ncp + c];
    }
    const double dt0 = dtl;
    first_residual(a, f, nb, a.cfl * dtl, P, [&](int s) { return Wn[s]; }, dU);
    CS<double> Un;
    const PS<double> w = first_update(a, k, U0, om, f.W, dtl, dU, Un);
    if (dtl != dt0) a.dt[c] = dtl;
    stU(a.U, ncp, c, Un);
    if (first_stage) stU(a.Uo, ncp, c, U0);
    a.Wout[c] = w.d; a.Wout[ncp + c] = w.vx; a.Wout[2 * ncp + c] = w.vy; a.Wout[3 * ncp + c] = w.p;
}

// All smoothings of a level whose connected groups of blocks have at most 1,024
// cells, in one launch: a workgroup per group, a thread per cell, W in LDS,
// everything else of the cell in registers.  nsm smoothings of a.nstage stages;
// each starts with the cell's CFL time step and the finer level's rule
// (cfl_kernel).  18 launches of the coarsest level of a V cycle (3 smoothings)
// become one.
__global__ __launch_bounds__(1024) void mg_first_smooth_kernel(FirstArgs a, const int32_t *group0, const int4 *local,
                                                               int nsm, FineLevel fl) {
    __shared__ double sW[4][1024];
    const int g0 = group0[blockIdx.x], n = group0[blockIdx.x + 1] - g0, t = threadIdx.x;
    const bool on = t < n;
    const int q = g0 + (on ? t : 0);
    const MgCell k = a.cells[q];
    if (a.meta[k.blk].skip) return;   // a group lies in one case: uniform
    const int4 n4 = a.nb[q], l4 = local[q];
    const int nb[4] = {n4.x, n4.y, n4.z, n4.w}, lo[4] = {l4.x, l4.y, l4.z, l4.w};
    const int64_t ncp = a.ncp, c = k.c;
    FirstCell f;
    f.W = ldW4(a.Win, ncp, c);
    load_geometry(a, k, f);
    CS<double> U = ldU(a.U, ncp, c), U0 = U;
    double P[4] = {0.0, 0.0, 0.0, 0.0};
    if (a.P) {
#pragma unroll
        for (int v = 0; v < 4; ++v) P[v] = a.P[v * ncp + c];
    }
    // the finer level's part of the time step (CFL_Multigrid)
    double dtf = MILLION;
    const bool fine = fl.meta != nullptr;
    if (fine) {
        const BlockMeta m = fl.meta[k.blk];
        const int i = k.ji & 0xFFFF, j = k.ji >> 16;
        const int64_t sw = cell(m, 2 * (i - 2) + 2, 2 * (j - 2) + 2), se = sw + 1, nw = sw + m.pitch, ne = nw + 1;
        const double dt_NE = qsqrt(qdiv(f.A, fl.A[ne])) * fl.dt[ne], dt_SE = qsqrt(qdiv(f.A, fl.A[se])) * fl.dt[se];
        const double dt_NW = qsqrt(qdiv(f.A, fl.A[nw])) * fl.dt[nw], dt_SW = qsqrt(qdiv(f.A, fl.A[sw])) * fl.dt[sw];
        dtf = dmin(dt_NE, dmin(dt_SE, dmin(dt_NW, dt_SW)));
    }
    double dtl = 0.0;
    for (int nu = 0; nu < nsm; ++nu) {
        {
            const double d_i = 2.0 * qdiv(f.A, f.lE + f.lW), d_j = 2.0 * qdiv(f.A, f.lN + f.lS);
            const double v_i = 0.5 * (f.W.vx * (f.nEx - -f.nWx) + f.W.vy * (f.nEy - -f.nWy));
            const double v_j = 0.5 * (f.W.vx * (f.nNx - -f.nSx) + f.W.vy * (f.nNy - -f.nSy));
            const double so = W_a(f.W);
            dtl = dmin(qdiv(d_i, so + fabs(v_i)), qdiv(d_j, so + fabs(v_j)));
            if (fine) dtl = dmin(dtl, dtf);
        }
        U0 = U;
        for (int st = 0; st < a.nstage; ++st) {
            if (on) { sW[0][t] = f.W.d; sW[1][t] = f.W.vx; sW[2][t] = f.W.vy; sW[3][t] = f.W.p; }
            __syncthreads();
            if (on) {
                double dU[4];
                first_residual(a, f, nb, a.cfl * dtl, P, [&](int s) -> PS<double> {
                    const int q = lo[s] >= 0 ? lo[s] : t;   // at a boundary: not used
                    return {sW[0][q], sW[1][q], sW[2][q], sW[3][q]};
                }, dU);
                f.W = first_update(a, k, U0, a.omega[st], f.W, dtl, dU, U);
            }
            __syncthreads();
        }
    }
    if (!on) return;
    stU(a.U, ncp, c, U);
    stU(a.Uo, ncp, c, U0);
    a.dt[c] = dtl;
    a.Wout[c] = f.W.d; a.Wout[ncp + c] = f.W.vx; a.Wout[2 * ncp + c] = f.W.vy; a.Wout[3 * ncp + c] = f.W.p;
}

}  // namespace
}  // namespace cffc

using namespace cffc;

extern "C" hipError_t cffc_launch_mg_restrict(const BlockMeta *mf, const BlockMeta *mc, int nblk, int max_int_c,
                                   const double *U, const double *R, const double *Af, int64_t ncpf, double *Uc,
                                   double *Wc, double *P, const double *Ac, int64_t ncpc, hipStream_t st) {
    dim3 grid((max_int_c + 255) / 256, nblk);
    hipLaunchKernelGGL(mg_restrict_kernel, grid, dim3(max_int_c <= 64 ? 64 : 256), 0, st, mf, mc, U, R, Af, ncpf, Uc,
                       Wc, P, Ac, ncpc);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_changes(const BlockMeta *meta, int nblk, int max_cells, double *U,
                                             const double *uo, int64_t ncp, hipStream_t st) {
    hipLaunchKernelGGL(mg_changes_kernel, dim3((max_cells + 255) / 256, nblk), dim3(256), 0, st, meta, U, uo, ncp);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_copy(const BlockMeta *meta, int nblk, int max_cells, double *dst,
                                          const double *src, int64_t ncp, hipStream_t st) {
    hipLaunchKernelGGL(mg_copy_kernel, dim3((max_cells + 255) / 256, nblk), dim3(256), 0, st, meta, dst, src, ncp);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_prolong(const BlockMeta *mc, const BlockMeta *mf, int nblk, int max_int_c,
                                  const int32_t *bc, const double *Uc, const double *gc, int64_t ncpc, double *Uf,
                                  double *Wf, const double *gf, int64_t ncpf, int neumann, int inj_dirichlet,
                                  int inj_always, int stability, int max_red, int assign, hipStream_t st) {
    // one thread per coarse cell, in the smallest workgroup that holds a block's
    const int nt = max_int_c <= 64 ? 64 : max_int_c <= 128 ? 128 : 256;
    hipLaunchKernelGGL(mg_prolong_kernel, dim3((max_int_c + nt - 1) / nt, nblk), dim3(nt), 0, st, mc, mf, bc, Uc, gc,
                       ncpc, Uf, Wf, gf, ncpf, neumann, inj_dirichlet, inj_always, stability, max_red, assign);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_first_step(const FirstArgs *a, double omega, int first_stage, hipStream_t st) {
    hipLaunchKernelGGL(mg_first_step_kernel, dim3((a->n + 255) / 256), dim3(256), 0, st, *a, omega, first_stage);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_first_smooth(const FirstArgs *a, int ngroup, int max_group, const int32_t *group0,
                                       const int4 *local, int nsm, const FineLevel *fl, hipStream_t st) {
    hipLaunchKernelGGL(mg_first_smooth_kernel, dim3(ngroup), dim3((max_group + 63) / 64 * 64), 0, st, *a, group0, local,
                       nsm, *fl);
    return hipGetLastError();
}
