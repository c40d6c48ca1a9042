// unet_kernels.hip -- BF16 MFMA kernels of the warm-start U-Net (gfx950).
//
// The network has no counterpart in the reference: it predicts an initial
// state for the steady bump solves.  Activations are NHWC.  BF16: the operands
// of every product, that is weights, activations and the masked gradients of
// convolution outputs.  FP32: accumulation, weight and bias gradients, the
// gradient that a skip connection brings, master weights and moments.
//
// 3x3 "same" convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16:
//   forward      Y[p,co]  = act( sum_k X[p+off(k), ci(k)] * Wt[co][k] + b[co] )
//                M = Cout, N = pixels, K = 9*Cin (k = tap*Cin + ci)
//   backward-in  dX[p,ci] = sum_k' G[p-off(k'), co(k')] * Wd[ci][k']
//                M = Cin,  N = pixels, K = 9*Cout (k' = tap*Cout + co)
//   backward-w   dW[co][k] = sum_p G[p,co] * X[p+off(k), ci(k)]
//                M = co, N = ci of one tap, K = pixels
// with G = BF16(dY * relu'(Y)): every product of the backward pass takes the
// gradient rounded to BF16 after the mask, so the kernel that forms dY in FP32
// rounds it once and sums the bias gradient from the FP32 values.  The first
// two are one kernel (conv_tile_kernel): a 16-pixel-wide input tile with its
// halo is staged in LDS once and serves all nine taps; weights are kept in
// the order in which a wavefront reads them.  The pooling after and the
// upsampling before a convolution, and their backward passes, are done in its
// epilogue and staging.  Operand layout of the 16x16x32 MFMA (wave64): lane l
// holds A[l%16][8*(l/16)+0..7], B[8*(l/16)+0..7][l%16] and
// D[4*(l/16)+0..3][l%16]; mfma_layout_kernel checks it on the device
// against a host product.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "unet_kernels.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace unetk {

__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7F800000u) == 0x7F800000u) return (bf16_t)(u >> 16);  // inf/nan
    u += 0x7FFFu + ((u >> 16) & 1u);                                  // round to nearest even
    return (bf16_t)(u >> 16);
}

union Frag {
    bf16x8 v;
    uint4 u;
    bf16_t h[8];
};

__device__ __forceinline__ Frag zero_frag() {
    Frag f;
    f.u = make_uint4(0, 0, 0, 0);
    return f;
}

// ---------------------------------------------------------------------------
// layout self-test: D = A(16x32) * B(32x16) with A[m][k] = m + k/64,
// B[k][n] = (k == n) + (k == n + 16); each lane writes its 4 D values.
__global__ void mfma_layout_kernel(float *out) {
    const int l = threadIdx.x;
    Frag a, b;
    for (int i = 0; i < 8; ++i) {
        const int m = l % 16, k = 8 * (l / 16) + i;
        a.h[i] = f2bf((float)m + (float)k / 64.0f);
        const int kb = 8 * (l / 16) + i, n = l % 16;
        b.h[i] = f2bf((kb == n || kb == n + 16) ? 1.0f : 0.0f);
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
    for (int i = 0; i < 4; ++i) out[l * 4 + i] = acc[i];
}

// ---------------------------------------------------------------------------
// Packed weights: row n (an output channel of the product) of chunk c (32 of
// the K values) sits where lane n%16 + 16*(k%32/8) of the wavefront that
// multiplies it reads 16 bytes, so a chunk of 16 rows is 1 KiB in order.
__device__ __forceinline__ int64_t packed_index(int n, int k, int nchunk) {
    return (((int64_t)(n >> 4) * nchunk + (k >> 5)) * 64 + (n & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

// ---------------------------------------------------------------------------
// One tile of a 3x3 convolution: 4 waves x MB rows of 16 pixels, NB x 16
// output channels (blockIdx.y picks them).  CIN: channels of the staged input
// (two tensors in the forward pass of a decoder's first convolution).
//
// Bound by staging and launch: 0.2 to 1.3 GFLOP and 6 to 38 MB a layer of a
// 16-image batch.  A tile's halo is read once from HBM or L2 (the nine taps
// come from LDS), the pixels of a wave share each weight fragment, and the
// output channels lie along a lane's accumulators, so that it stores 8 bytes of
// a pixel at once.  The sums run over k in chunks of 32 from k = 0 up whatever
// the tile.
struct ConvArgs {
    const bf16_t *xA, *xB;   // staged input: CA channels of xA, the rest of xB
    int CA, upA;             // upA: xA has half the resolution (nearest upsampling)
    int B, H, W;
    const bf16_t *w;         // packed weights
    int Cout;                // output channels (a multiple of 16)
    // forward
    const float *bias;
    int relu;
    bf16_t *y;               // [P][Cout]
    float *y4;               // first 4 channels in FP32 [P][4], or null
    bf16_t *pool;            // 2x2 average of y at half the resolution, or null
    // backward-in: channels below CT go to the target tensor, the rest to gB
    int CT, kind;            // BwdKind of the target
    const bf16_t *act;       // target's activation (its relu mask)
    bf16_t *G;               // target's masked gradient, BF16
    float *dbp;              // [tile][CT] bias partials of the target's convolution
    float *gB;               // FP32 gradient [P][Cout - CT] (skip connection), or null
    const float *gskip;      // BWD_POOL: FP32 gradient of the target through its skip connection
};
__device__ __forceinline__ bool relu_on(bf16_t y) { return y != 0 && !(y & 0x8000u); }   // Y > 0

union Half4 {
    uint2 u;
    bf16_t h[4];
};

// masked gradient of four channels at element q of the target: stored in BF16,
// added to the bias sums in FP32
__device__ __forceinline__ void put_gradient(const ConvArgs &a, int64_t q, const float (&g)[4], float (&db)[4]) {
    Half4 y, o;
    y.u = *(const uint2 *)(a.act + q);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = relu_on(y.h[i]) ? g[i] : 0.f;
        db[i] += v;
        o.h[i] = f2bf(v);
    }
    *(uint2 *)(a.G + q) = o.u;
}

template <int CIN, int MB, int NB, bool BWD>
__global__ __launch_bounds__(256) void conv_tile_kernel(ConvArgs a) {
    constexpr int TH = 4 * MB, TW = 16, HW = TW + 2, C8 = CIN / 8;
    // row stride of a pixel in LDS: 16 bytes past a multiple of 128 for wide
    // inputs, so that a wave's 16 pixels fall on different banks
    constexpr int CS = CIN + (CIN >= 64 ? 8 : 0);
    constexpr int NCH = (9 * CIN + 31) / 32;
    __shared__ __align__(16) bf16_t sx[(TH + 2) * HW * CS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ntx = (a.W + TW - 1) / TW, nty = (a.H + TH - 1) / TH;
    const int tx = blockIdx.x % ntx, ty = (blockIdx.x / ntx) % nty, b = blockIdx.x / (ntx * nty);
    const int x0 = tx * TW, y0 = ty * TH;
    // six 16-byte loads in flight per thread before their LDS stores: one after
    // the other, the 17 of a 192-channel tile are 17 memory latencies
    constexpr int NU = (TH + 2) * HW * C8, NIT = (NU + 255) / 256, UB = NIT < 6 ? NIT : 6;
    for (int k0 = 0; k0 < NIT; k0 += UB) {
        uint4 v[UB];
#pragma unroll
        for (int k = 0; k < UB; ++k) {
            const int u = tid + (k0 + k) * 256;
            const int pix = u / C8, c = (u - pix * C8) * 8;
            const int row = pix / HW, yy = y0 + row - 1, xx = x0 + (pix - row * HW) - 1;
            v[k] = make_uint4(0, 0, 0, 0);
            if (u < NU && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W) {
                if (c < a.CA) {
                    const int64_t q = a.upA ? ((int64_t)b * (a.H >> 1) + (yy >> 1)) * (a.W >> 1) + (xx >> 1)
                                            : ((int64_t)b * a.H + yy) * a.W + xx;
                    v[k] = *(const uint4 *)(a.xA + q * a.CA + c);
                } else {
                    const int64_t q = ((int64_t)b * a.H + yy) * a.W + xx;
                    v[k] = *(const uint4 *)(a.xB + q * (CIN - a.CA) + (c - a.CA));
                }
            }
        }
#pragma unroll
        for (int k = 0; k < UB; ++k) {
            const int u = tid + (k0 + k) * 256;
            const int pix = u / C8, c = (u - pix * C8) * 8;
            if (u < NU) *(uint4 *)(sx + pix * CS + c) = v[k];
        }
    }
    __syncthreads();
    const int px = lane & 15, kg = lane >> 4;
    f32x4 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const bf16_t *sp = sx + ((wave * MB) * HW + px) * CS;
    const int nb0 = blockIdx.y * NB;
    const bf16_t *wp = a.w + (int64_t)nb0 * NCH * 512 + lane * 8;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        // this lane's eight k of the chunk: one tap, eight channels
        const int k = 32 * c + 8 * kg;
        int tap, ci;
        if constexpr (CIN % 32 == 0) { tap = 32 * c / CIN; ci = 32 * c % CIN + 8 * kg; }
        else { tap = k / CIN; ci = k - tap * CIN; }
        const bool in = CIN % 32 == 0 || tap < 9;   // past K: the weights are zero, and so is the input
        if (CIN % 32 != 0 && !in) { tap = 8; ci = 0; }
        // forward reads X at p + off(tap), backward G at p - off(tap)
        const int t = BWD ? 8 - tap : tap;
        const int off = ((t / 3) * HW + t % 3) * CS + ci;
        Frag w[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) w[n].u = *(const uint4 *)(wp + ((int64_t)n * NCH + c) * 512);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            Frag x;
            x.u = *(const uint4 *)(sp + m * HW * CS + off);
            if (!in) x.u = make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int n = 0; n < NB; ++n)
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[n].v, x.v, acc[m][n], 0, 0, 0);
        }
    }
    // D: lane holds channels n0 + 4*kg + 0..3 of pixel (row, px)
    const int xx = x0 + px;
    if constexpr (!BWD) {
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int co = (nb0 + n) * 16 + 4 * kg;
            const float4 bv = *(const float4 *)(a.bias + co);
            float pa[4];
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const int yy = y0 + wave * MB + m;
                const bool ok = yy < a.H && xx < a.W;
                const int64_t q = ((int64_t)b * a.H + yy) * a.W + xx;
                float v[4] = {acc[m][n][0] + bv.x, acc[m][n][1] + bv.y, acc[m][n][2] + bv.z, acc[m][n][3] + bv.w};
                Half4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (a.relu) v[i] = v[i] > 0.f ? v[i] : 0.f;
                    o.h[i] = f2bf(v[i]);
                }
                if (ok) {
                    *(uint2 *)(a.y + q * a.Cout + co) = o.u;
                    if (a.y4 && co == 0) *(float4 *)(a.y4 + 4 * q) = make_float4(v[0], v[1], v[2], v[3]);
                }
                if (a.pool) {
                    // (x0,y0) + (x0+1,y0) + (x0,y0+1) + (x0+1,y0+1) of the stored values, times 1/4
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float e = bf2f(o.h[i]), f = __shfl_xor(e, 1);
                        if ((m & 1) == 0) pa[i] = e + f;
                        else pa[i] = (pa[i] + e) + f;
                    }
                    if ((m & 1) && ok && !(px & 1)) {
                        Half4 po;
#pragma unroll
                        for (int i = 0; i < 4; ++i) po.h[i] = f2bf(0.25f * pa[i]);
                        const int64_t r = ((int64_t)b * (a.H >> 1) + (yy >> 1)) * (a.W >> 1) + (xx >> 1);
                        *(uint2 *)(a.pool + r * a.Cout + co) = po.u;
                    }
                }
            }
        }
    } else {
        __shared__ float sdb[4][NB * 16];
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int n0 = (nb0 + n) * 16, ch = n0 + 4 * kg;
            float db[4] = {0.f, 0.f, 0.f, 0.f};
            float pa[4];
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const int yy = y0 + wave * MB + m;
                const bool ok = yy < a.H && xx < a.W;
                const int64_t q = ((int64_t)b * a.H + yy) * a.W + xx;
                const float g[4] = {acc[m][n][0], acc[m][n][1], acc[m][n][2], acc[m][n][3]};
                if (n0 >= a.CT) {
                    if (ok) *(float4 *)(a.gB + q * (a.Cout - a.CT) + (ch - a.CT)) = make_float4(g[0], g[1], g[2], g[3]);
                } else if (a.kind == BWD_SAME) {
                    if (ok) put_gradient(a, q * a.CT + ch, g, db);
                } else if (a.kind == BWD_UP) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float f = __shfl_xor(g[i], 1);
                        if ((m & 1) == 0) pa[i] = g[i] + f;
                        else pa[i] = (pa[i] + g[i]) + f;
                    }
                    if ((m & 1) && ok && !(px & 1)) {
                        const int64_t r = ((int64_t)b * (a.H >> 1) + (yy >> 1)) * (a.W >> 1) + (xx >> 1);
                        put_gradient(a, r * a.CT + ch, pa, db);
                    }
                } else if (ok) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int64_t r = ((int64_t)b * (2 * a.H) + 2 * yy + (k >> 1)) * (2 * a.W) + 2 * xx + (k & 1);
                        const float4 s = *(const float4 *)(a.gskip + r * a.CT + ch);
                        const float t[4] = {s.x + 0.25f * g[0], s.y + 0.25f * g[1], s.z + 0.25f * g[2],
                                            s.w + 0.25f * g[3]};
                        put_gradient(a, r * a.CT + ch, t, db);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                for (int o = 1; o < 16; o <<= 1) db[i] += __shfl_xor(db[i], o);
                if (px == 0) sdb[wave][n * 16 + 4 * kg + i] = db[i];
            }
        }
        __syncthreads();
        if (tid < NB * 16) {
            const int ch = nb0 * 16 + tid;
            if (ch < a.CT)
                a.dbp[(int64_t)blockIdx.x * a.CT + ch] = (sdb[0][tid] + sdb[1][tid]) + (sdb[2][tid] + sdb[3][tid]);
        }
    }
}

// ---------------------------------------------------------------------------
// backward wrt the weights.  A workgroup keeps dW of 16 input channels (all nine
// taps) by COB x 16 output channels in its accumulators while it walks tiles of 8 x
// 16 pixels (blockIdx.x, += gridDim.x) and writes one partial at the end
// (grad_reduce_kernel sums them; no atomics, so the sums are the same every
// time).  Pixels are the contracted index, channels the contiguous one in
// memory: the operands come out of LDS with the transposing 64-bit read
// (ds_read_b64_tr_b16: four pixels by 16 channels per 16 lanes), each tap a
// shifted address in the same tile.  COB < 4: the four waves also split a tile's
// pixels and add up at the end.  C8: an 8-channel input, two taps per 16 columns.
// Per layer of a 16-image batch of 64 x 192: 8 to 11 us; with per-tap gathers,
// transposing stores and atomics it was 86 us.
struct WgradArgs {
    const bf16_t *G;
    int Cout;
    const bf16_t *xA, *xB;
    int CA, CB, upA;
    int B, H, W, ntiles;
    float *part;   // [gridDim.x][Cout][9*Cin]
};
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ s16x4 lds_read_tr(const bf16_t *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
}
union FragT {
    bf16x8 v;
    s16x4 q[2];
};

template <int COB, bool C8>
__global__ __launch_bounds__(256) void conv_wgrad_kernel(WgradArgs a) {
    constexpr int TH = 8, TW = 16, HW = TW + 2, PS = 4 / COB;
    constexpr int NX = C8 ? 8 : 16, NBK = C8 ? 5 : 9;
    constexpr int GS = COB * 16 + (COB == 4 ? 8 : 0);
    constexpr int NG = TH * TW * GS, NXE = (TH + 2) * HW * NX;
    constexpr int RED = PS > 1 ? PS * COB * NBK * 256 * 2 : 0;   // floats as bf16 units
    __shared__ __align__(16) bf16_t sm[NG + NXE > RED ? NG + NXE : RED];
    bf16_t *sG = sm, *sX = sm + NG;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cob = wave % COB, slice = wave / COB;
    const int ci0 = blockIdx.y * NX, co0 = blockIdx.z * COB * 16;
    const int ntx = (a.W + TW - 1) / TW, nty = (a.H + TH - 1) / TH;
    const bool fromA = ci0 < a.CA;
    const bf16_t *x = fromA ? a.xA : a.xB;
    const int xc = fromA ? a.CA : a.CB, xc0 = fromA ? ci0 : ci0 - a.CA;
    const bool up = fromA && a.upA;
    const int g = lane >> 4, li = lane & 15;
    f32x4 acc[NBK];
#pragma unroll
    for (int n = 0; n < NBK; ++n) acc[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // the next tile's operands are loaded into registers while this one's are
    // multiplied
    constexpr int NUG = TH * TW * COB * 2 / 256, NUX = ((TH + 2) * HW * (NX / 8) + 255) / 256;
    uint4 vg[NUG], vx[NUX];
    auto load_tile = [&](int t) {
        const int x0 = (t % ntx) * TW, y0 = ((t / ntx) % nty) * TH, b = t / (ntx * nty);
#pragma unroll
        for (int k = 0; k < NUG; ++k) {
            const int u = tid + k * 256;
            const int pix = u / (COB * 2), c = (u - pix * (COB * 2)) * 8;
            const int yy = y0 + (pix >> 4), xx = x0 + (pix & 15);
            vg[k] = make_uint4(0, 0, 0, 0);
            if (yy < a.H && xx < a.W)
                vg[k] = *(const uint4 *)(a.G + (((int64_t)b * a.H + yy) * a.W + xx) * a.Cout + co0 + c);
        }
#pragma unroll
        for (int k = 0; k < NUX; ++k) {
            const int u = tid + k * 256;
            const int pix = u / (NX / 8), c = (u - pix * (NX / 8)) * 8;
            const int row = pix / HW, yy = y0 + row - 1, xx = x0 + (pix - row * HW) - 1;
            vx[k] = make_uint4(0, 0, 0, 0);
            if (row < TH + 2 && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W) {
                const int64_t q = up ? ((int64_t)b * (a.H >> 1) + (yy >> 1)) * (a.W >> 1) + (xx >> 1)
                                     : ((int64_t)b * a.H + yy) * a.W + xx;
                vx[k] = *(const uint4 *)(x + q * xc + xc0 + c);
            }
        }
    };
    if ((int)blockIdx.x < a.ntiles) load_tile(blockIdx.x);
    for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
#pragma unroll
        for (int k = 0; k < NUG; ++k) {
            const int u = tid + k * 256;
            const int pix = u / (COB * 2), c = (u - pix * (COB * 2)) * 8;
            *(uint4 *)(sG + pix * GS + c) = vg[k];
        }
#pragma unroll
        for (int k = 0; k < NUX; ++k) {
            const int u = tid + k * 256;
            if (u < (TH + 2) * HW * (NX / 8)) *(uint4 *)(sX + u * 8) = vx[k];   // rows of NX, no padding
        }
        __syncthreads();
        if (t + (int)gridDim.x < a.ntiles) load_tile(t + gridDim.x);
        // 32 pixels a step: two rows of 16; lane group g takes pixels 8g..8g+7,
        // four of them (row, 8*(g&1) + 4h + ...) with each of two reads
#pragma unroll
        for (int s = 0; s < 4; s += PS) {
            const int row = 2 * (s + slice) + (g >> 1), col = 8 * (g & 1) + (li >> 2);
            FragT ga;
            const bf16_t *pg = sG + (row * TW + col) * GS + cob * 16 + 4 * (li & 3);
            ga.q[0] = lds_read_tr(pg);
            ga.q[1] = lds_read_tr(pg + 4 * GS);
#pragma unroll
            for (int n = 0; n < NBK; ++n) {
                int tap, c;
                if constexpr (C8) {
                    tap = 2 * n + ((li & 3) >> 1);
                    c = 4 * (li & 1);
                    if (tap > 8) tap = 8;   // columns past K: never stored
                } else {
                    tap = n;
                    c = 4 * (li & 3);
                }
                const bf16_t *pb = sX + ((row + tap / 3) * HW + col + tap % 3) * NX + c;
                FragT xb;
                xb.q[0] = lds_read_tr(pb);
                xb.q[1] = lds_read_tr(pb + 4 * NX);
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga.v, xb.v, acc[n], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    const int K = 9 * (a.CA + a.CB);
    float *out = a.part + (int64_t)blockIdx.x * a.Cout * K;
    if constexpr (PS > 1) {
        float *r = (float *)sm;
#pragma unroll
        for (int n = 0; n < NBK; ++n) *(f32x4 *)(r + ((wave * NBK + n) * 64 + lane) * 4) = acc[n];
        __syncthreads();
        if (slice > 0) return;
        for (int s = 1; s < PS; ++s)
#pragma unroll
            for (int n = 0; n < NBK; ++n) acc[n] += *(const f32x4 *)(r + (((s * COB + cob) * NBK + n) * 64 + lane) * 4);
    }
#pragma unroll
    for (int n = 0; n < NBK; ++n) {
        const int k = C8 ? 16 * n + li : n * (a.CA + a.CB) + ci0 + li;
        if (k >= K) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) out[(int64_t)(co0 + cob * 16 + 4 * g + i) * K + k] = acc[n][i];
    }
}

// Sums of partials, every layer's weight and bias gradients and the loss in one
// launch: out[e] = sum over c of part[c*n + e].  A workgroup takes 32
// elements, 8 threads per element over the partials, added in a fixed order.
__global__ __launch_bounds__(256) void grad_reduce_kernel(SumList L) {
    __shared__ float sm[8][32];
    int d = 0;
    while ((int)blockIdx.x >= L.first[d + 1]) ++d;
    const int e = ((int)blockIdx.x - L.first[d]) * 32 + (threadIdx.x & 31), s = threadIdx.x >> 5;
    const int n = L.n[d];
    float v = 0.f;
    if (e < n) {
        const float *p = L.part[d] + e;
#pragma unroll 4
        for (int c = s; c < L.chunks[d]; c += 8) v += p[(int64_t)c * n];
    }
    sm[s][threadIdx.x & 31] = v;
    __syncthreads();
    if (s == 0 && e < n) {
        for (int k = 1; k < 8; ++k) v += sm[k][threadIdx.x & 31];
        L.out[d][e] = v;
    }
}

// FP32 -> BF16, eight values a thread (n a multiple of 8)
__global__ void to_bf16_kernel(const float4 *src, uint4 *dst, int64_t n8) {
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= n8) return;
    const float4 a = src[2 * q], b = src[2 * q + 1];
    Frag f;
    f.h[0] = f2bf(a.x); f.h[1] = f2bf(a.y); f.h[2] = f2bf(a.z); f.h[3] = f2bf(a.w);
    f.h[4] = f2bf(b.x); f.h[5] = f2bf(b.y); f.h[6] = f2bf(b.z); f.h[7] = f2bf(b.w);
    dst[q] = f.u;
}

// MSE of the first 4 of 16 output channels (y4 [P][4]); dy = 2*(y-t)/N, stored
// in BF16 over all 16 (zero past the fourth) with its FP32 sums per channel and
// workgroup in dbp [gridDim.x][16]; each workgroup's share of the loss in
// lossp.  One thread per pixel.
__global__ __launch_bounds__(256) void mse_kernel(const float *y4, const float *t, int64_t P, bf16_t *G, float *dbp,
                                                  float *lossp) {
    __shared__ float sm[4][5];
    const float inv = 1.0f / (float)(P * 4);
    float s = 0.f, db[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < P; p += (int64_t)gridDim.x * blockDim.x) {
        const float4 y = *(const float4 *)(y4 + 4 * p), r = *(const float4 *)(t + 4 * p);
        const float d[4] = {y.x - r.x, y.y - r.y, y.z - r.z, y.w - r.w};
        Frag o = zero_frag();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            s += d[c] * d[c];
            const float gv = 2.f * d[c] * inv;
            db[c] += gv;
            o.h[c] = f2bf(gv);
        }
        *(uint4 *)(G + 16 * p) = o.u;
        *(uint4 *)(G + 16 * p + 8) = make_uint4(0, 0, 0, 0);
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o);
#pragma unroll
        for (int c = 0; c < 4; ++c) db[c] += __shfl_xor(db[c], o);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sm[w][4] = s;
        for (int c = 0; c < 4; ++c) sm[w][c] = db[c];
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        const int c = threadIdx.x;
        dbp[blockIdx.x * 16 + c] = c < 4 ? (sm[0][c] + sm[1][c]) + (sm[2][c] + sm[3][c]) : 0.f;
        if (c == 4) lossp[blockIdx.x] = ((sm[0][4] + sm[1][4]) + (sm[2][4] + sm[3][4])) * inv;
    }
}

// Adam on FP32 master weights [Cout][K] and biases of every layer in one
// launch; refreshes the packed BF16 copies of the forward product (rows Cout, k
// = tap*Cin + ci) and of the backward-input product (rows Cin, k' = tap*Cout +
// co).  update 0: only the copies.
__device__ __forceinline__ float adam_step(float w, float g, float &m, float &v, float lr, float b1, float b2,
                                           float eps, float c1, float c2) {
    m = b1 * m + (1.f - b1) * g;
    v = b2 * v + (1.f - b2) * g * g;
    return w - lr * (m / c1) / (sqrtf(v / c2) + eps);
}
__global__ __launch_bounds__(256) void adam_kernel(AdamList A, float lr, float b1, float b2, float eps, float c1,
                                                   float c2, int update) {
    int d = 0;
    while (d + 1 < A.count && (int)blockIdx.x >= A.l[d + 1].first) ++d;
    const AdamLayer L = A.l[d];
    const int K = 9 * L.Cin, nw = L.Cout * K;
    int q = ((int)blockIdx.x - L.first) * 256 + threadIdx.x;
    if (q < nw) {
        float wv = L.w[q];
        if (update) {
            float mv = L.m[q], vv = L.v[q];
            wv = adam_step(wv, L.g[q], mv, vv, lr, b1, b2, eps, c1, c2);
            L.m[q] = mv;
            L.v[q] = vv;
            L.w[q] = wv;
        }
        const int co = q / K, k = q - co * K;
        const int tap = k / L.Cin, ci = k - tap * L.Cin;
        const bf16_t hb = f2bf(wv);
        L.wt[packed_index(co, k, (K + 31) / 32)] = hb;
        L.wd[packed_index(ci, tap * L.Cout + co, (9 * L.Cout + 31) / 32)] = hb;
    } else if (update && (q -= nw) < L.Cout) {
        float mv = L.mb[q], vv = L.vb[q];
        L.b[q] = adam_step(L.b[q], L.gb[q], mv, vv, lr, b1, b2, eps, c1, c2);
        L.mb[q] = mv;
        L.vb[q] = vv;
    }
}

// gather a batch of samples: dst[r] = src[idx[r]] (rows of n16 16-byte units, blockIdx.y = r)
__global__ void gather_rows_kernel(const uint4 *src, const int32_t *idx, int64_t n16, uint4 *dst) {
    const int r = blockIdx.y;
    const uint4 *s = src + (int64_t)idx[r] * n16;
    uint4 *d = dst + (int64_t)r * n16;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n16; q += (int64_t)gridDim.x * blockDim.x)
        d[q] = s[q];
}

}  // namespace unetk

using namespace unetk;

// ---------------------------------------------------------------------------
// Shape of a convolution's launch.  MB rows per wave: 4 (tiles of 16 x 16
// pixels) while that gives every compute unit a workgroup, else 2; NB: 32
// output channels a workgroup while that does, else 16.
struct ConvShape {
    int mb, nb, tiles, groups;
};
static ConvShape conv_shape(int B, int H, int W, int Cout) {
    ConvShape s;
    auto tiles = [&](int mb) { return B * ((W + 15) / 16) * ((H + 4 * mb - 1) / (4 * mb)); };
    s.mb = Cout <= 48 && tiles(4) >= 256 ? 4 : 2;
    s.tiles = tiles(s.mb);
    s.nb = Cout % 32 == 0 && (int64_t)s.tiles * (Cout / 32) >= 256 ? 2 : 1;
    s.groups = Cout / (16 * s.nb);
    return s;
}

template <int CIN, bool BWD> static hipError_t launch_conv(const ConvArgs &a, hipStream_t st) {
    const ConvShape s = conv_shape(a.B, a.H, a.W, a.Cout);
    dim3 grid(s.tiles, s.groups);
    if constexpr (CIN <= 96) {   // mb 4 comes with at most 48 output channels, so with at most 96 input channels
        if (s.mb == 4) {
            if (s.nb == 2) hipLaunchKernelGGL((conv_tile_kernel<CIN, 4, 2, BWD>), grid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((conv_tile_kernel<CIN, 4, 1, BWD>), grid, dim3(256), 0, st, a);
            return hipGetLastError();
        }
    } else if (s.mb == 4) {
        return hipErrorInvalidValue;
    }
    if (s.nb == 2) hipLaunchKernelGGL((conv_tile_kernel<CIN, 2, 2, BWD>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((conv_tile_kernel<CIN, 2, 1, BWD>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

// pixel chunks (partials) of a weight gradient: about 256 workgroups over the
// channel blocks (a training pass of 16 images: 430 us; with 128 workgroups
// 481 us, with 512, whose partials take longer to add, 451 us)
static int wgrad_chunks(int B, int H, int W, int Cin, int Cout) {
    const int tiles = B * ((W + 15) / 16) * ((H + 7) / 8);
    const int blocks = ((Cin + 15) / 16) * (Cout >= 64 ? Cout / 64 : 1);
    return std::max(1, std::min(tiles, 256 / blocks));
}

extern "C" {

hipError_t cffc_unet_launch_mfma_layout(float *out, hipStream_t st) {
    hipLaunchKernelGGL(mfma_layout_kernel, dim3(1), dim3(64), 0, st, out);
    return hipGetLastError();
}

int cffc_unet_conv_tiles(int B, int H, int W, int Cout) { return conv_shape(B, H, W, Cout).tiles; }
int cffc_unet_wgrad_chunks(int B, int H, int W, int Cin, int Cout) { return wgrad_chunks(B, H, W, Cin, Cout); }

hipError_t cffc_unet_launch_conv_fwd(const bf16_t *xA, int CA, int upA, const bf16_t *xB, int CB, int B, int H, int W,
                                     const bf16_t *wt, const float *bias, int Cout, int relu, bf16_t *y, float *y4,
                                     bf16_t *pool, hipStream_t st) {
    ConvArgs a = {};
    a.xA = xA; a.xB = xB; a.CA = CA; a.upA = upA;
    a.B = B; a.H = H; a.W = W;
    a.w = wt; a.Cout = Cout; a.bias = bias; a.relu = relu;
    a.y = y; a.y4 = y4; a.pool = pool;
    if (Cout % 16) return hipErrorInvalidValue;
    switch (CA + CB) {
    case 8: return launch_conv<8, false>(a, st);
    case 16: return launch_conv<16, false>(a, st);
    case 32: return launch_conv<32, false>(a, st);
    case 48: return launch_conv<48, false>(a, st);
    case 64: return launch_conv<64, false>(a, st);
    case 96: return launch_conv<96, false>(a, st);
    case 128: return launch_conv<128, false>(a, st);
    case 192: return launch_conv<192, false>(a, st);
    default: return hipErrorInvalidValue;
    }
}

// gradient of a convolution's input from its masked output gradient G (C
// channels): Cout = the input's channels, of which CT go to the target tensor
hipError_t cffc_unet_launch_conv_bwd_data(const bf16_t *G, int C, int B, int H, int W, const bf16_t *wd, int Cout,
                                          int CT, int kind, const bf16_t *act, bf16_t *Gt, float *dbp, float *gB,
                                          const float *gskip, hipStream_t st) {
    ConvArgs a = {};
    a.xA = G; a.CA = C;
    a.B = B; a.H = H; a.W = W;
    a.w = wd; a.Cout = Cout; a.CT = CT; a.kind = kind;
    a.act = act; a.G = Gt; a.dbp = dbp; a.gB = gB; a.gskip = gskip;
    if (Cout % 16 || CT % 16) return hipErrorInvalidValue;
    switch (C) {
    case 16: return launch_conv<16, true>(a, st);
    case 32: return launch_conv<32, true>(a, st);
    case 64: return launch_conv<64, true>(a, st);
    case 128: return launch_conv<128, true>(a, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t cffc_unet_launch_conv_bwd_weight(const bf16_t *G, int Cout, const bf16_t *xA, int CA, int upA,
                                            const bf16_t *xB, int CB, int B, int H, int W, float *part,
                                            hipStream_t st) {
    WgradArgs a;
    a.G = G; a.Cout = Cout; a.xA = xA; a.xB = xB; a.CA = CA; a.CB = CB; a.upA = upA;
    a.B = B; a.H = H; a.W = W;
    a.ntiles = B * ((W + 15) / 16) * ((H + 7) / 8);
    a.part = part;
    const int Cin = CA + CB, chunks = wgrad_chunks(B, H, W, Cin, Cout);
    if (Cin == 8) {
        if (Cout != 16) return hipErrorInvalidValue;
        hipLaunchKernelGGL((conv_wgrad_kernel<1, true>), dim3(chunks), dim3(256), 0, st, a);
        return hipGetLastError();
    }
    if (Cin % 16 || CA % 16) return hipErrorInvalidValue;
    if (Cout == 16) hipLaunchKernelGGL((conv_wgrad_kernel<1, false>), dim3(chunks, Cin / 16), dim3(256), 0, st, a);
    else if (Cout == 32) hipLaunchKernelGGL((conv_wgrad_kernel<2, false>), dim3(chunks, Cin / 16), dim3(256), 0, st, a);
    else if (Cout % 64 == 0)
        hipLaunchKernelGGL((conv_wgrad_kernel<4, false>), dim3(chunks, Cin / 16, Cout / 64), dim3(256), 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t cffc_unet_launch_reduce(const SumList *L, hipStream_t st) {
    hipLaunchKernelGGL(grad_reduce_kernel, dim3(L->first[L->count]), dim3(256), 0, st, *L);
    return hipGetLastError();
}
hipError_t cffc_unet_launch_mse(const float *y4, const float *t, int64_t P, int nwg, bf16_t *G, float *dbp,
                                float *lossp, hipStream_t st) {
    hipLaunchKernelGGL(mse_kernel, dim3(nwg), dim3(256), 0, st, y4, t, P, G, dbp, lossp);
    return hipGetLastError();
}
hipError_t cffc_unet_launch_adam(const AdamList *A, int nwg, float lr, float b1, float b2, float eps, float c1,
                                 float c2, int update, hipStream_t st) {
    hipLaunchKernelGGL(adam_kernel, dim3(nwg), dim3(256), 0, st, *A, lr, b1, b2, eps, c1, c2, update);
    return hipGetLastError();
}
// rows of a multiple of 16 bytes
hipError_t cffc_unet_launch_gather(const void *src, const int32_t *idx, int nrows, int64_t row_bytes, void *dst,
                                   hipStream_t st) {
    const int64_t n16 = row_bytes / 16;
    dim3 grid((unsigned)std::min<int64_t>((n16 + 255) / 256, 1024), nrows);
    hipLaunchKernelGGL(gather_rows_kernel, grid, dim3(256), 0, st, (const uint4 *)src, idx, n16, (uint4 *)dst);
    return hipGetLastError();
}
hipError_t cffc_unet_launch_to_bf16(const float *src, bf16_t *dst, int64_t n, hipStream_t st) {
    hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, st, (const float4 *)src,
                       (uint4 *)dst, n / 8);
    return hipGetLastError();
}

}  // extern "C"
