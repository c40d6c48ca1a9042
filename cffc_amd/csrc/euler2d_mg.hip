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

// Restrict_Boundary_Ref_States :1112-1186: the reference state of a coarse
// boundary face is the area-weighted mean of its two fine ones.  The states stay
// on the device: through the host this was four copies a level, one of them every
// cell's area.
__global__ __launch_bounds__(64) void mg_restrict_wo_kernel(const BlockMeta *mf, const BlockMeta *mc, const double *Af,
                                                            const double *wf, double *wc) {
    const BlockMeta F = mf[blockIdx.x], C = mc[blockIdx.x];
    const int n = 2 * (C.ni + C.nj);
    for (int q = blockIdx.y * 64 + threadIdx.x; q < n; q += gridDim.y * 64) {
        // sides W, E (nj entries each), S, N (ni each)
        const int side = q < C.nj ? 0 : q < 2 * C.nj ? 1 : q < 2 * C.nj + C.ni ? 2 : 3;
        const int k = q - (side == 0 ? 0 : side == 1 ? C.nj : side == 2 ? 2 * C.nj : 2 * C.nj + C.ni);
        const int k0 = 2 * k + 2;
        const int64_t c0 = side == 0 ? cell(F, 2, k0) : side == 1 ? cell(F, F.ni + 1, k0)
                                     : side == 2 ? cell(F, k0, 2) : cell(F, k0, F.nj + 1);
        const int64_t c1 = c0 + (side < 2 ? F.pitch : 1);
        const int fb = side == 0 ? 0 : side == 1 ? F.ncj : side == 2 ? 2 * F.ncj : 2 * F.ncj + F.nci;
        const int cb = side == 0 ? 0 : side == 1 ? C.ncj : side == 2 ? 2 * C.ncj : 2 * C.ncj + C.nci;
        const double A0 = Af[c0], A1 = Af[c1];
        const double *w0 = wf + 4 * (int64_t)(F.bcoff + fb + k0), *w1 = w0 + 4;
        double *o = wc + 4 * (int64_t)(C.bcoff + cb + k + 2);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = (w0[v] * A0 + w1[v] * A1) / (A0 + A1);
    }
}

// ---------------------------------------------------------------------------
// Smoothing of a first-order level (HLLE, zero limiter, so a face takes the
// states of its two cells): a cell needs its four neighbours and nothing else,
// which the host lists per cell across blocks.  No window, no LDS, no ghost cells,
// two dependent loads to the states; the price is that both cells of a face
// evaluate its flux.  The launches of the coarse levels are bound by that load
// chain (a 12,288-cell case: 9.6 us a stage with windows, whatever the level, 6.7 us
// so).  Without the gradient that the limiter would multiply by zero (0 * NaN is
// NaN) a state that is no longer finite spreads through faces alone, a cell a
// stage, not through the stencils of both cells of a face.
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
// state beyond a boundary face of cell Wc; (nx, ny): the face's normal (E or N of
// its low cell), low: the cell is on the high side, the boundary on the low one
__device__ __forceinline__ PS<double> first_ghost(int t, const PS<double> &wo, const PS<double> &Wc, bool low, double nx,
                                                  double ny) {
    const double sg = low ? -1.0 : 1.0;   // outward
    if (t == 7001) return reflect(Wc, sg * nx, sg * ny);
    if (t == 8001) return bc_characteristic_pressure(Wc, wo, sg * nx, sg * ny);
    return t == 11000 ? wo : Wc;
}
// (CFL dt)(+W -E +S -N)/A in the stage kernel's order
__device__ __forceinline__ void first_sum(const CS<double> &W, const CS<double> &E, const CS<double> &S, const CS<double> &N,
                                          double lW, double lE, double lS, double lN, const Recip<double> &rA, double cdt,
                                          double (&dU)[4]) {
    dU[0] = 0.0 + rdivf(cdt * W.d * lW, rA); dU[1] = 0.0 + rdivf(cdt * W.mx * lW, rA);
    dU[2] = 0.0 + rdivf(cdt * W.my * lW, rA); dU[3] = 0.0 + rdivf(cdt * W.E * lW, rA);
    dU[0] -= rdivf(cdt * E.d * lE, rA); dU[1] -= rdivf(cdt * E.mx * lE, rA);
    dU[2] -= rdivf(cdt * E.my * lE, rA); dU[3] -= rdivf(cdt * E.E * lE, rA);
    dU[0] += rdivf(cdt * S.d * lS, rA); dU[1] += rdivf(cdt * S.mx * lS, rA);
    dU[2] += rdivf(cdt * S.my * lS, rA); dU[3] += rdivf(cdt * S.E * lS, rA);
    dU[0] -= rdivf(cdt * N.d * lN, rA); dU[1] -= rdivf(cdt * N.mx * lN, rA);
    dU[2] -= rdivf(cdt * N.my * lN, rA); dU[3] -= rdivf(cdt * N.E * lN, rA);
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

// CFL_Multigrid: the finer level's bound on a cell's time step
__device__ __forceinline__ double first_dt_fine(const FineLevel &fl, const MgCell &k, double A) {
    const BlockMeta m = fl.meta[k.blk];
    const int i = k.ji & 0xFFFF, j = k.ji >> 16;
    const int64_t sw = cell(m, 2 * (i - 2) + 2, 2 * (j - 2) + 2), se = sw + 1, nw = sw + m.pitch, ne = nw + 1;
    const double dt_NE = qsqrt(qdiv(A, fl.A[ne])) * fl.dt[ne], dt_SE = qsqrt(qdiv(A, fl.A[se])) * fl.dt[se];
    const double dt_NW = qsqrt(qdiv(A, fl.A[nw])) * fl.dt[nw], dt_SW = qsqrt(qdiv(A, fl.A[sw])) * fl.dt[sw];
    return dmin(dt_NE, dmin(dt_SE, dmin(dt_NW, dt_SW)));
}
// cfl_kernel's time step; s?i, s?j: sums of the opposite faces' normals
__device__ __forceinline__ double first_dt(const PS<double> &W, double A, double lW, double lE, double lS, double lN,
                                           double sxi, double syi, double sxj, double syj) {
    const double d_i = 2.0 * qdiv(A, lE + lW), d_j = 2.0 * qdiv(A, lN + lS);
    const double v_i = 0.5 * (W.vx * sxi + W.vy * syi), v_j = 0.5 * (W.vx * sxj + W.vy * syj);
    const double so = W_a(W);
    return dmin(qdiv(d_i, so + fabs(v_i)), qdiv(d_j, so + fabs(v_j)));
}

// One smoothing stage of a level, one thread per cell, from Win to Wout.  The first
// one of a smoothing forms the time step from the geometry it has loaded anyway; as
// a launch of its own that took 4 us (one case) to 18 us (64 cases).
__global__ __launch_bounds__(256) void mg_first_step_kernel(FirstArgs a, double om, int first_stage, FineLevel fl) {
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
    double P[4] = {0.0, 0.0, 0.0, 0.0}, dtl, dU[4];
    if (first_stage) {
        dtl = first_dt(f.W, f.A, f.lW, f.lE, f.lS, f.lN, f.nEx - -f.nWx, f.nEy - -f.nWy, f.nNx - -f.nSx, f.nNy - -f.nSy);
        if (fl.meta) dtl = dmin(dtl, first_dt_fine(fl, k, f.A));
    } else {
        dtl = a.dt[c];
    }
    if (a.P) {
#pragma unroll
        for (int v = 0; v < 4; ++v) P[v] = a.P[v * ncp + c];
    }
    const double dt0 = dtl;
    auto flux = [&](int h, bool low, double nx, double ny) -> CS<double> {
        if (nb[h] < 0) {
            const int e = -(nb[h] + 1);
            const double *w = a.wo + 4 * (int64_t)e;
            Wn[h] = first_ghost(a.bc[e], PS<double>{w[0], w[1], w[2], w[3]}, f.W, low, nx, ny);
        }
        return low ? flux_hlle_n(Wn[h], f.W, nx, ny) : flux_hlle_n(f.W, Wn[h], nx, ny);
    };
    const double cdt = a.cfl * dtl;
    first_sum(flux(0, true, f.nWx, f.nWy), flux(1, false, f.nEx, f.nEy), flux(2, true, f.nSx, f.nSy),
              flux(3, false, f.nNx, f.nNy), f.lW, f.lE, f.lS, f.lN, recip(f.A), cdt, dU);
    if (a.P) {
#pragma unroll
        for (int v = 0; v < 4; ++v) dU[v] += cdt * P[v];
    }
    CS<double> Un;
    const PS<double> w = first_update(a, k, U0, om, f.W, dtl, dU, Un);
    if (first_stage || dtl != dt0) a.dt[c] = dtl;
    stU(a.U, ncp, c, Un);
    if (first_stage) stU(a.Uo, ncp, c, U0);
    a.Wout[c] = w.d; a.Wout[ncp + c] = w.vx; a.Wout[2 * ncp + c] = w.vy; a.Wout[3 * ncp + c] = w.p;
}

// All smoothings of a level whose connected groups of blocks are small (at most
// MG_GROUP_CELLS cells, MG_GROUP_FACES faces, MG_GROUP_EDGES of them on boundaries),
// in one launch: a workgroup per group.  nsm smoothings of a.nstage stages; each
// starts with the cell's CFL time step and the finer level's rule (cfl_kernel).
// In a stage a thread first evaluates one to three faces of the group's list into
// LDS, then updates its cell from its four faces; W, the fluxes, the faces' normals
// and the boundaries' states live in LDS (102 of 160 KB), the cells' geometry and U
// in registers.  A wave alone on its SIMD is bound by the flux's own dependent
// instructions, so faces, not cells, are spread over the threads.  15 stages of 192
// cells take 52 us, 3.4 us each, against 6.7 us for a launch per stage; of 768 cells
// (16 waves at 128 registers, some spilled) 10 us each, no less than by launches:
// hence the limit of 512 cells and threads (40 cycles of one case 16.4 -> 15.3 ms; 64
// cases of up to 768 cells on that level 28.0 and 28.3 ms, runs differing by 0.5%).
__global__ __launch_bounds__(512) void mg_first_smooth_kernel(FirstArgs a, GroupArgs ga, int nsm, FineLevel fl) {
    __shared__ double sW[4][MG_GROUP_CELLS], sF[4][MG_GROUP_FACES], sn[2][MG_GROUP_FACES];
    __shared__ double swo[4][MG_GROUP_EDGES];
    __shared__ int16_t sLR[2][MG_GROUP_FACES];   // negative: the boundary's kind, -1 ... -4
    const int32_t *gr = ga.groups + 3 * blockIdx.x;
    const int g0 = gr[0], n = gr[3] - g0, f0 = gr[1], nf = gr[4] - f0, inner = gr[2] - f0;
    const int t = threadIdx.x, nt = blockDim.x;
    const bool on = t < n;
    const int q = g0 + (on ? t : 0);
    const MgCell k = a.cells[q];
    if (a.meta[k.blk].skip) return;   // a group lies in one case: uniform
    const double *G = a.geom;
    const int64_t ncp = a.ncp, c = k.c;
    for (int f = t; f < nf; f += nt) {
        const MgFace k = ga.faces[f0 + f];
        int l = k.l, r = k.r;
        if (k.e >= 0) {
            const int bc = a.bc[k.e], kind = bc == 7001 ? -2 : bc == 8001 ? -3 : bc == 11000 ? -4 : -1;
            if (l < 0) l = kind;
            else r = kind;
            const double *w = a.wo + 4 * (int64_t)k.e;
#pragma unroll
            for (int v = 0; v < 4; ++v) swo[v][f - inner] = w[v];
        }
        sLR[0][f] = (int16_t)l;
        sLR[1][f] = (int16_t)r;
        sn[0][f] = G[(k.north ? GEO_NNX : GEO_NEX) * ncp + k.g];
        sn[1][f] = G[(k.north ? GEO_NNY : GEO_NEY) * ncp + k.g];
    }
    // the thread's cell
    const int4 cf = ga.cell_faces[q];
    const int fW = cf.x, fE = cf.y, fS = cf.z, fN = cf.w;
    PS<double> W = ldW4(a.Win, ncp, c);
    CS<double> U = ldU(a.U, ncp, c), U0 = U;
    double P[4] = {0.0, 0.0, 0.0, 0.0};
    if (a.P) {
#pragma unroll
        for (int v = 0; v < 4; ++v) P[v] = a.P[v * ncp + c];
    }
    const int64_t wc = c - 1, sc = k.south;
    const double lW = G[GEO_LE * ncp + wc], lE = G[GEO_LE * ncp + c], lS = G[GEO_LN * ncp + sc], lN = G[GEO_LN * ncp + c];
    const double A = G[GEO_A * ncp + c];
    const Recip<double> rA = recip(A);
    const bool fine = fl.meta != nullptr;
    const double dtf = fine ? first_dt_fine(fl, k, A) : MILLION;
    double dtl = 0.0;
    if (on) { sW[0][t] = W.d; sW[1][t] = W.vx; sW[2][t] = W.vy; sW[3][t] = W.p; }
    for (int nu = 0; nu < nsm; ++nu) {
        // the normals are read again rather than held in registers
        dtl = first_dt(W, A, lW, lE, lS, lN, G[GEO_NEX * ncp + c] - -G[GEO_NEX * ncp + wc],
                       G[GEO_NEY * ncp + c] - -G[GEO_NEY * ncp + wc], G[GEO_NNX * ncp + c] - -G[GEO_NNX * ncp + sc],
                       G[GEO_NNY * ncp + c] - -G[GEO_NNY * ncp + sc]);
        if (fine) dtl = dmin(dtl, dtf);
        U0 = U;
        for (int st = 0; st < a.nstage; ++st) {
            __syncthreads();
#pragma unroll 1
            for (int f = t; f < nf; f += nt) {
                const int l = sLR[0][f], r = sLR[1][f], il = l >= 0 ? l : r, ir = r >= 0 ? r : l;
                PS<double> Wl = {sW[0][il], sW[1][il], sW[2][il], sW[3][il]};
                PS<double> Wr = {sW[0][ir], sW[1][ir], sW[2][ir], sW[3][ir]};
                const double nx = sn[0][f], ny = sn[1][f];
                if ((l | r) < 0) {
                    const int q = f - inner, kind = l < 0 ? l : r;
                    const PS<double> wo = {swo[0][q], swo[1][q], swo[2][q], swo[3][q]};
                    const PS<double> g = first_ghost(kind == -2 ? 7001 : kind == -3 ? 8001 : kind == -4 ? 11000 : 0, wo, Wl,
                                                     l < 0, nx, ny);
                    if (l < 0) Wl = g;
                    else Wr = g;
                }
                const CS<double> F = flux_hlle_n(Wl, Wr, nx, ny);
                sF[0][f] = F.d; sF[1][f] = F.mx; sF[2][f] = F.my; sF[3][f] = F.E;
            }
            __syncthreads();
            if (on) {
                auto F = [&](int x) -> CS<double> { return {sF[0][x], sF[1][x], sF[2][x], sF[3][x]}; };
                const double cdt = a.cfl * dtl;
                double dU[4];
                first_sum(F(fW), F(fE), F(fS), F(fN), lW, lE, lS, lN, rA, cdt, dU);
                if (a.P) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) dU[v] += cdt * P[v];
                }
                W = first_update(a, k, U0, a.omega[st], W, dtl, dU, U);
                sW[0][t] = W.d; sW[1][t] = W.vx; sW[2][t] = W.vy; sW[3][t] = W.p;
            }
        }
    }
    if (!on) return;
    stU(a.U, ncp, c, U);
    stU(a.Uo, ncp, c, U0);
    a.dt[c] = dtl;
    a.Wout[c] = W.d; a.Wout[ncp + c] = W.vx; a.Wout[2 * ncp + c] = W.vy; a.Wout[3 * ncp + c] = W.p;
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
extern "C" hipError_t cffc_launch_mg_restrict_wo(const BlockMeta *mf, const BlockMeta *mc, int nblk, int max_faces,
                                       const double *Af, const double *wf, double *wc, hipStream_t st) {
    hipLaunchKernelGGL(mg_restrict_wo_kernel, dim3(nblk, (max_faces + 63) / 64), dim3(64), 0, st, mf, mc, Af, wf, wc);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_first_step(const FirstArgs *a, double omega, int first_stage, const FineLevel *fl,
                                       hipStream_t st) {
    hipLaunchKernelGGL(mg_first_step_kernel, dim3((a->n + 255) / 256), dim3(256), 0, st, *a, omega, first_stage, *fl);
    return hipGetLastError();
}
extern "C" hipError_t cffc_launch_mg_first_smooth(const FirstArgs *a, const GroupArgs *ga, int ngroup, int nt, int nsm,
                                       const FineLevel *fl, hipStream_t st) {
    hipLaunchKernelGGL(mg_first_smooth_kernel, dim3(ngroup), dim3(nt), 0, st, *a, *ga, nsm, *fl);
    return hipGetLastError();
}
