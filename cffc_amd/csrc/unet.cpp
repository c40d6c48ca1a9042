// unet.cpp -- host runtime of the warm-start U-Net (include/cffc_unet.h).
//
// Four resolution levels (H x W down to H/8 x W/8), channels 16-32-64-128,
// two 3x3 conv + ReLU per level, 2x2 average pooling down, nearest 2x
// upsampling up, skip connections by channel concatenation (a conv reads its
// input from two NHWC tensors, so no copy is made), and a final 3x3 conv to
// 16 channels of which the first CFFC_UNET_OUT are the prediction.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <thread>
#include <vector>

#include "../../include/cffc_euler2d.h"
#include "../../include/cffc_unet.h"

#include "unet_kernels.hpp"

using namespace unetk;

static thread_local std::string u_err;
static int ufail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    u_err = buf;
    fprintf(stderr, "cffc_unet: %s\n", buf);
    return code;
}
#define UCHK(x)                                                                                   \
    do {                                                                                          \
        hipError_t e_ = (x);                                                                      \
        if (e_ != hipSuccess) return ufail(CFFC_E_HIP, "%s: %s", #x, hipGetErrorString(e_));      \
    } while (0)

// Activations, and the masked BF16 gradient of a convolution's output; gskip:
// the FP32 gradient a skip connection brings to it.
struct Tensor {
    int C, level;
    int producer = -1;   // conv that writes it
    bf16_t *act = nullptr, *G = nullptr;
    float *gskip = nullptr;
};

struct Conv {
    int inA, inB, out;   // tensor ids (inB = -1: none); inA is read through the upsampling if upA
    int upA;
    int pool = -1;       // pooled copy of the output, or -1
    int CA, CB, Cout, level, relu;
    int kind = -1, target = -1;   // where the input's gradient goes (BwdKind, tensor); -1: not needed
    int K, Kpad, Kpad2;
    float *w = nullptr, *b = nullptr, *m = nullptr, *v = nullptr, *mb = nullptr, *vb = nullptr;
    float *gw = nullptr, *gb = nullptr;
    bf16_t *wt = nullptr, *wd = nullptr;
    float *part = nullptr, *dbp = nullptr;   // weight-gradient and bias-gradient partials
};

constexpr int MSE_WG = 256;   // workgroups of the loss kernel

struct cffc_unet {
    int H = 0, W = 0, maxB = 0;
    hipStream_t stream = nullptr;
    // the weight gradients run beside the chain of input gradients, a few
    // layers at a time: they wait for their outputs' gradients (ready), the sums
    // wait for them (joined)
    hipStream_t side = nullptr;
    hipEvent_t ready[4] = {nullptr, nullptr, nullptr, nullptr}, joined = nullptr;
    std::vector<Tensor> t;
    std::vector<Conv> L;
    int x0 = -1, yout = -1;
    float *y4 = nullptr, *target = nullptr, *loss = nullptr, *lossp = nullptr, *x32 = nullptr;
    // predictions of several batches: the second of each buffer, the streams of the
    // copies, a batch computed
    float *x32b = nullptr, *y4b = nullptr;
    hipStream_t up = nullptr, down = nullptr;
    hipEvent_t computed[2] = {nullptr, nullptr};
    int32_t *idx = nullptr;
    bf16_t *ds_in = nullptr;
    float *ds_tg = nullptr;
    int ds_n = 0;
    int step = 0;
    std::vector<void *> allocs;
};

// hipMemset of device memory only enqueues on the null stream, which the network's
// streams (hipStreamNonBlocking) do not wait for: wait_cleared comes between the
// allocations and their first use there, or a clear could run after it (a wait
// in every allocation: a network created in 24 ms instead of 21).
static int ualloc(cffc_unet *n, void **p, size_t bytes) {
    if (hipMalloc(p, bytes) != hipSuccess) return ufail(CFFC_E_NOMEM, "hipMalloc(%zu) failed", bytes);
    n->allocs.push_back(*p);
    if (hipMemset(*p, 0, bytes) != hipSuccess) return ufail(CFFC_E_HIP, "hipMemset failed");
    return 0;
}
static int wait_cleared() {
    UCHK(hipStreamSynchronize(nullptr));
    return 0;
}

static int npix(const cffc_unet *n, int level, int B) { return B * (n->H >> level) * (n->W >> level); }

static int add_tensor(cffc_unet *n, int C, int level) {
    Tensor x;
    x.C = C;
    x.level = level;
    n->t.push_back(x);
    return (int)n->t.size() - 1;
}

static int add_conv(cffc_unet *n, int inA, int upA, int inB, int Cout, int relu) {
    Conv c;
    c.inA = inA;
    c.upA = upA;
    c.inB = inB;
    c.CA = n->t[inA].C;
    c.CB = inB >= 0 ? n->t[inB].C : 0;
    c.Cout = Cout;
    c.level = n->t[inA].level - upA;
    c.relu = relu;
    c.out = add_tensor(n, Cout, c.level);
    n->t[c.out].producer = (int)n->L.size();
    c.K = 9 * (c.CA + c.CB);
    c.Kpad = (c.K + 31) / 32 * 32;
    c.Kpad2 = (9 * Cout + 31) / 32 * 32;
    if (inA != n->x0) {
        // the input's gradient: to the tensor, to the low-resolution tensor, or
        // (a pooled input, which has no producer) to the tensor it was pooled from
        c.kind = upA ? BWD_UP : BWD_SAME;
        c.target = inA;
        if (n->t[inA].producer < 0) {
            c.kind = BWD_POOL;
            for (const Conv &q : n->L)
                if (q.pool == inA) c.target = q.out;
        }
    }
    n->L.push_back(c);
    return c.out;
}

static int add_pool(cffc_unet *n, int src) {
    const int dst = add_tensor(n, n->t[src].C, n->t[src].level + 1);
    n->L[n->t[src].producer].pool = dst;
    return dst;
}

static void build_graph(cffc_unet *n) {
    const int ch[4] = {16, 32, 64, 128};
    n->x0 = add_tensor(n, CFFC_UNET_IN, 0);
    int cur = n->x0;
    int skip[3];
    for (int l = 0; l < 4; ++l) {
        cur = add_conv(n, cur, 0, -1, ch[l], 1);
        cur = add_conv(n, cur, 0, -1, ch[l], 1);
        if (l < 3) {
            skip[l] = cur;
            cur = add_pool(n, cur);
        }
    }
    for (int l = 2; l >= 0; --l) {
        cur = add_conv(n, cur, 1, skip[l], ch[l], 1);
        cur = add_conv(n, cur, 0, -1, ch[l], 1);
    }
    n->yout = add_conv(n, cur, 0, -1, 16, 0);
}

// Adam on every layer, or (update 0) only the packed BF16 copies of layer
// first .. last
static int run_adam(cffc_unet *n, int first, int last, int update, float lr, float b1, float b2, float eps, float c1,
                    float c2) {
    AdamList A = {};
    int wg = 0;
    for (int l = first; l <= last; ++l) {
        const Conv &c = n->L[l];
        AdamLayer &a = A.l[A.count++];
        a = {c.w, c.gw, c.m, c.v, c.b, c.gb, c.mb, c.vb, c.wt, c.wd, c.Cout, c.CA + c.CB, wg};
        wg += (c.Cout * c.K + c.Cout + 255) / 256;
    }
    UCHK(cffc_unet_launch_adam(&A, wg, lr, b1, b2, eps, c1, c2, update, n->stream));
    return 0;
}

extern "C" void cffc_unet_destroy(cffc_unet *n) {
    if (!n) return;
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    if (n->side) (void)hipStreamSynchronize(n->side);
    for (void *p : n->allocs) (void)hipFree(p);
    for (hipEvent_t e : n->ready)
        if (e) (void)hipEventDestroy(e);
    if (n->joined) (void)hipEventDestroy(n->joined);
    if (n->side) (void)hipStreamDestroy(n->side);
    for (hipStream_t q : {n->up, n->down})
        if (q) (void)hipStreamDestroy(q);
    for (hipEvent_t q : n->computed)
        if (q) (void)hipEventDestroy(q);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

extern "C" int cffc_unet_create(int H, int W, int max_batch, uint64_t seed, cffc_unet **out) {
    if (!out || H <= 0 || W <= 0 || H % 8 || W % 8 || max_batch <= 0) return ufail(CFFC_E_ARG, "bad network shape");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return ufail(CFFC_E_NODEVICE, "no HIP device");
    cffc_unet *n = new cffc_unet();
    n->H = H;
    n->W = W;
    n->maxB = max_batch;
    if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) {
        delete n;
        return ufail(CFFC_E_HIP, "stream creation failed");
    }
    build_graph(n);
    bool ok = hipStreamCreateWithFlags(&n->side, hipStreamNonBlocking) == hipSuccess &&
              hipEventCreateWithFlags(&n->joined, hipEventDisableTiming) == hipSuccess;
    for (hipEvent_t &ev : n->ready) ok = ok && hipEventCreateWithFlags(&ev, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        cffc_unet_destroy(n);
        return ufail(CFFC_E_HIP, "stream or event creation failed");
    }
    int e = 0;
    for (auto &x : n->t) {
        const size_t np = (size_t)npix(n, x.level, max_batch) * x.C;
        if ((e = ualloc(n, (void **)&x.act, np * sizeof(bf16_t))) ||
            (x.producer >= 0 && (e = ualloc(n, (void **)&x.G, np * sizeof(bf16_t))))) {
            cffc_unet_destroy(n);
            return e;
        }
    }
    for (auto &c : n->L) {
        if (c.inB < 0) continue;
        Tensor &x = n->t[c.inB];
        if ((e = ualloc(n, (void **)&x.gskip, (size_t)npix(n, x.level, max_batch) * x.C * sizeof(float)))) {
            cffc_unet_destroy(n);
            return e;
        }
    }
    // rows of the bias-gradient partials of every convolution, written by the
    // kernel that forms its output's gradient, for the largest batch and any
    // smaller one (a smaller batch may take smaller tiles)
    std::vector<size_t> dbrows(n->L.size(), MSE_WG), parts(n->L.size(), 0);
    for (const Conv &c : n->L)
        for (int B = 1; B <= max_batch; ++B) {
            const int ch = H >> c.level, cw = W >> c.level, Cin = c.CA + c.CB;
            size_t &p = parts[&c - n->L.data()];
            p = std::max(p, (size_t)cffc_unet_wgrad_chunks(B, ch, cw, Cin, c.Cout));
            if (c.target < 0) continue;
            size_t &r = dbrows[n->t[c.target].producer];
            r = std::max(r, (size_t)cffc_unet_conv_tiles(B, ch, cw, Cin));
        }
    std::mt19937_64 rng(seed);
    for (size_t li = 0; li < n->L.size(); ++li) {
        Conv &c = n->L[li];
        const size_t nw = (size_t)c.Cout * c.K;
        const int Cin = c.CA + c.CB;
        if ((e = ualloc(n, (void **)&c.w, nw * 4)) || (e = ualloc(n, (void **)&c.m, nw * 4)) ||
            (e = ualloc(n, (void **)&c.v, nw * 4)) || (e = ualloc(n, (void **)&c.gw, nw * 4)) ||
            (e = ualloc(n, (void **)&c.b, c.Cout * 4)) || (e = ualloc(n, (void **)&c.mb, c.Cout * 4)) ||
            (e = ualloc(n, (void **)&c.vb, c.Cout * 4)) || (e = ualloc(n, (void **)&c.gb, c.Cout * 4)) ||
            (e = ualloc(n, (void **)&c.wt, (size_t)c.Cout * c.Kpad * 2)) ||
            (e = ualloc(n, (void **)&c.wd, (size_t)((Cin + 15) / 16 * 16) * c.Kpad2 * 2)) ||
            (e = ualloc(n, (void **)&c.part, parts[li] * nw * 4)) ||
            (e = ualloc(n, (void **)&c.dbp, dbrows[li] * c.Cout * 4))) {
            cffc_unet_destroy(n);
            return e;
        }
        // He-normal initialisation; the output layer starts near zero so
        // the untrained prediction is the freestream
        std::vector<float> hw(nw);
        const double sd = std::sqrt(2.0 / (9.0 * Cin)) * (li + 1 == n->L.size() ? 0.05 : 1.0);
        std::normal_distribution<double> nd(0.0, sd);
        for (auto &x : hw) x = (float)nd(rng);
        UCHK(hipMemcpy(c.w, hw.data(), nw * 4, hipMemcpyHostToDevice));
    }
    const size_t np0 = (size_t)npix(n, 0, max_batch);
    if ((e = ualloc(n, (void **)&n->y4, np0 * CFFC_UNET_OUT * 4)) ||
        (e = ualloc(n, (void **)&n->target, np0 * CFFC_UNET_OUT * 4)) ||
        (e = ualloc(n, (void **)&n->x32, np0 * CFFC_UNET_IN * 4)) || (e = ualloc(n, (void **)&n->loss, 4)) ||
        (e = ualloc(n, (void **)&n->lossp, MSE_WG * 4)) || (e = ualloc(n, (void **)&n->idx, max_batch * 4)) ||
        (e = wait_cleared()) || (e = run_adam(n, 0, (int)n->L.size() - 1, 0, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f))) {
        cffc_unet_destroy(n);
        return e;
    }
    UCHK(hipStreamSynchronize(n->stream));
    *out = n;
    return 0;
}

extern "C" int cffc_unet_num_layers(const cffc_unet *n) { return n ? (int)n->L.size() : 0; }
extern "C" int cffc_unet_layer_shape(const cffc_unet *n, int l, int shape[4]) {
    if (!n || l < 0 || l >= (int)n->L.size()) return ufail(CFFC_E_ARG, "bad layer");
    shape[0] = n->L[l].CA;
    shape[1] = n->L[l].CB;
    shape[2] = n->L[l].Cout;
    shape[3] = n->L[l].level;
    return 0;
}
extern "C" int cffc_unet_get_weights(cffc_unet *n, int l, float *w, float *b) {
    if (!n || l < 0 || l >= (int)n->L.size()) return ufail(CFFC_E_ARG, "bad layer");
    Conv &c = n->L[l];
    UCHK(hipStreamSynchronize(n->stream));
    if (w) UCHK(hipMemcpy(w, c.w, (size_t)c.Cout * c.K * 4, hipMemcpyDeviceToHost));
    if (b) UCHK(hipMemcpy(b, c.b, (size_t)c.Cout * 4, hipMemcpyDeviceToHost));
    return 0;
}
extern "C" int cffc_unet_set_weights(cffc_unet *n, int l, const float *w, const float *b) {
    if (!n || l < 0 || l >= (int)n->L.size()) return ufail(CFFC_E_ARG, "bad layer");
    Conv &c = n->L[l];
    if (w) UCHK(hipMemcpy(c.w, w, (size_t)c.Cout * c.K * 4, hipMemcpyHostToDevice));
    if (b) UCHK(hipMemcpy(c.b, b, (size_t)c.Cout * 4, hipMemcpyHostToDevice));
    if (int e = run_adam(n, l, l, 0, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f)) return e;
    UCHK(hipStreamSynchronize(n->stream));
    return 0;
}

extern "C" int cffc_unet_set_dataset(cffc_unet *n, int ns, const float *inputs, const float *targets) {
    if (!n || ns <= 0 || !inputs || !targets) return ufail(CFFC_E_ARG, "bad dataset");
    const size_t per_in = (size_t)n->H * n->W * CFFC_UNET_IN, per_tg = (size_t)n->H * n->W * CFFC_UNET_OUT;
    // a call that fails from here on leaves the network without a dataset
    n->ds_n = 0;
    for (void *q : {(void *)n->ds_in, (void *)n->ds_tg}) {
        if (!q) continue;
        (void)hipFree(q);
        n->allocs.erase(std::remove(n->allocs.begin(), n->allocs.end(), q), n->allocs.end());
    }
    n->ds_in = nullptr;
    n->ds_tg = nullptr;
    int e;
    if ((e = ualloc(n, (void **)&n->ds_in, per_in * ns * 2)) ||
        (e = ualloc(n, (void **)&n->ds_tg, per_tg * ns * 4)) || (e = wait_cleared()))
        return e;
    // rounded to BF16 on the device, max_batch samples at a time
    for (int s = 0; s < ns; s += n->maxB) {
        const size_t k = per_in * std::min(n->maxB, ns - s);
        UCHK(hipMemcpyAsync(n->x32, inputs + per_in * s, k * 4, hipMemcpyHostToDevice, n->stream));
        UCHK(cffc_unet_launch_to_bf16(n->x32, n->ds_in + per_in * s, (int64_t)k, n->stream));
    }
    UCHK(hipMemcpyAsync(n->ds_tg, targets, per_tg * ns * 4, hipMemcpyHostToDevice, n->stream));
    UCHK(hipStreamSynchronize(n->stream));
    n->ds_n = ns;
    return 0;
}

static int forward(cffc_unet *n, int B, float *y4 = nullptr) {
    for (const Conv &c : n->L) {
        const int H = n->H >> c.level, W = n->W >> c.level;
        UCHK(cffc_unet_launch_conv_fwd(n->t[c.inA].act, c.CA, c.upA, c.inB >= 0 ? n->t[c.inB].act : nullptr, c.CB, B, H,
                                       W, c.wt, c.b, c.Cout, c.relu, n->t[c.out].act,
                                       c.out == n->yout ? (y4 ? y4 : n->y4) : nullptr,
                                       c.pool >= 0 ? n->t[c.pool].act : nullptr, n->stream));
    }
    return 0;
}

// Weight and input gradients from the last convolution to the first, then the
// sums of all partials.  A skip tensor's gradient comes first through its
// decoder (gskip), then through the pooling, where the two are added.
static int backward(cffc_unet *n, int B) {
    SumList S = {};
    auto sum = [&](const float *part, float *out, int len, int chunks) {
        S.part[S.count] = part;
        S.out[S.count] = out;
        S.n[S.count] = len;
        S.chunks[S.count] = chunks;
        S.first[S.count + 1] = S.first[S.count] + (len + 31) / 32;
        S.count++;
    };
    sum(n->lossp, n->loss, 1, MSE_WG);
    sum(n->L.back().dbp, n->L.back().gb, n->L.back().Cout, MSE_WG);
    const int nl = (int)n->L.size();
    int pending = nl - 1, group = 0;   // weight gradients not launched yet: layers q..pending
    for (int q = nl - 1; q >= 0; --q) {
        const Conv &c = n->L[q];
        if (q == 0 || (q & 3) == 3) {
            // every gradient down to layer q's output is in the stream
            UCHK(hipEventRecord(n->ready[group], n->stream));
            UCHK(hipStreamWaitEvent(n->side, n->ready[group], 0));
            group++;
            for (; pending >= q; --pending) {
                const Conv &w = n->L[pending];
                const int H = n->H >> w.level, W = n->W >> w.level;
                UCHK(cffc_unet_launch_conv_bwd_weight(n->t[w.out].G, w.Cout, n->t[w.inA].act, w.CA, w.upA,
                                                      w.inB >= 0 ? n->t[w.inB].act : nullptr, w.CB, B, H, W, w.part,
                                                      n->side));
                sum(w.part, w.gw, w.Cout * w.K, cffc_unet_wgrad_chunks(B, H, W, w.CA + w.CB, w.Cout));
            }
        }
        if (c.target < 0) continue;
        const int H = n->H >> c.level, W = n->W >> c.level, Cin = c.CA + c.CB;
        const Tensor &t = n->t[c.target];
        const Conv &pr = n->L[t.producer];
        UCHK(cffc_unet_launch_conv_bwd_data(n->t[c.out].G, c.Cout, B, H, W, c.wd, Cin, c.CA, c.kind, t.act, t.G, pr.dbp,
                                            c.inB >= 0 ? n->t[c.inB].gskip : nullptr, t.gskip, n->stream));
        sum(pr.dbp, pr.gb, pr.Cout, cffc_unet_conv_tiles(B, H, W, Cin));
    }
    UCHK(hipEventRecord(n->joined, n->side));
    UCHK(hipStreamWaitEvent(n->stream, n->joined, 0));
    UCHK(cffc_unet_launch_reduce(&S, n->stream));
    return 0;
}

static int load_batch(cffc_unet *n, const int32_t *idx, int B) {
    if (!n->ds_n) return ufail(CFFC_E_ARG, "no dataset");
    for (int i = 0; i < B; ++i)
        if (idx[i] < 0 || idx[i] >= n->ds_n) return ufail(CFFC_E_ARG, "sample index out of range");
    UCHK(hipMemcpyAsync(n->idx, idx, B * 4, hipMemcpyHostToDevice, n->stream));
    const int64_t px = (int64_t)n->H * n->W;
    UCHK(cffc_unet_launch_gather(n->ds_in, n->idx, B, px * CFFC_UNET_IN * 2, n->t[n->x0].act, n->stream));
    UCHK(cffc_unet_launch_gather(n->ds_tg, n->idx, B, px * CFFC_UNET_OUT * 4, n->target, n->stream));
    return 0;
}

static int loss_and_grad(cffc_unet *n, int B, float *loss) {
    UCHK(cffc_unet_launch_mse(n->y4, n->target, (int64_t)npix(n, 0, B), MSE_WG, n->t[n->yout].G, n->L.back().dbp,
                              n->lossp, n->stream));
    if (int e = backward(n, B)) return e;
    if (loss) {
        UCHK(hipMemcpyAsync(loss, n->loss, 4, hipMemcpyDeviceToHost, n->stream));
    }
    return 0;
}

extern "C" int cffc_unet_train_step(cffc_unet *n, const int32_t *idx, int B, float lr, float *loss) {
    if (!n || B <= 0 || B > n->maxB) return ufail(CFFC_E_ARG, "bad batch");
    if (int e = load_batch(n, idx, B)) return e;
    if (int e = forward(n, B)) return e;
    float l = 0.f;
    if (int e = loss_and_grad(n, B, &l)) return e;
    n->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)n->step), c2 = 1.f - std::pow(b2, (float)n->step);
    if (int e = run_adam(n, 0, (int)n->L.size() - 1, 1, lr, b1, b2, 1e-8f, c1, c2)) return e;
    UCHK(hipStreamSynchronize(n->stream));
    if (loss) *loss = l;
    return 0;
}

extern "C" int cffc_unet_loss_grad(cffc_unet *n, const int32_t *idx, int B, float *loss, int l, float *gw, float *gb) {
    if (!n || B <= 0 || B > n->maxB) return ufail(CFFC_E_ARG, "bad batch");
    if (int e = load_batch(n, idx, B)) return e;
    if (int e = forward(n, B)) return e;
    float lv = 0.f;
    if (int e = loss_and_grad(n, B, &lv)) return e;
    UCHK(hipStreamSynchronize(n->stream));
    if (loss) *loss = lv;
    if (l >= 0 && l < (int)n->L.size()) {
        Conv &c = n->L[l];
        if (gw) UCHK(hipMemcpy(gw, c.gw, (size_t)c.Cout * c.K * 4, hipMemcpyDeviceToHost));
        if (gb) UCHK(hipMemcpy(gb, c.gb, (size_t)c.Cout * 4, hipMemcpyDeviceToHost));
    }
    return 0;
}

extern "C" int cffc_unet_predict(cffc_unet *n, const float *inputs, int B, float *outputs) {
    if (!n || B <= 0 || B > n->maxB || !inputs || !outputs) return ufail(CFFC_E_ARG, "bad batch");
    const size_t px = (size_t)n->H * n->W;
    // rounded to BF16 on the device; the four FP32 output channels come back as
    // the last convolution stores them
    UCHK(hipMemcpyAsync(n->x32, inputs, px * CFFC_UNET_IN * B * 4, hipMemcpyHostToDevice, n->stream));
    UCHK(cffc_unet_launch_to_bf16(n->x32, n->t[n->x0].act, (int64_t)px * CFFC_UNET_IN * B, n->stream));
    if (int e = forward(n, B)) return e;
    UCHK(hipMemcpyAsync(outputs, n->y4, px * CFFC_UNET_OUT * B * 4, hipMemcpyDeviceToHost, n->stream));
    UCHK(hipStreamSynchronize(n->stream));
    return 0;
}

static int ensure_pipeline(cffc_unet *n) {
    if (n->computed[1]) return 0;
    const size_t px = (size_t)n->H * n->W * n->maxB;
    int e;
    if (!n->x32b && (e = ualloc(n, (void **)&n->x32b, px * CFFC_UNET_IN * 4))) return e;
    if (!n->y4b && (e = ualloc(n, (void **)&n->y4b, px * CFFC_UNET_OUT * 4))) return e;
    for (hipStream_t *q : {&n->up, &n->down})
        if (!*q) UCHK(hipStreamCreateWithFlags(q, hipStreamNonBlocking));
    if ((e = wait_cleared())) return e;
    for (hipEvent_t &q : n->computed)
        if (!q) UCHK(hipEventCreateWithFlags(&q, hipEventDisableTiming));
    return 0;
}

// Batches of maxB samples through two buffers of each kind: this thread sends the
// inputs of a batch while the one before it is computed and a second thread
// fetches the outputs of the one before that.  64 samples of 64 x 192, of which the
// kernels take 0.5 ms: 2.1 ms one after the other, 1.57 ms this way.
extern "C" int cffc_unet_predict_all(cffc_unet *n, const float *inputs, int count, float *outputs) {
    if (!n || count <= 0 || !inputs || !outputs) return ufail(CFFC_E_ARG, "bad batch");
    if (count <= n->maxB) return cffc_unet_predict(n, inputs, count, outputs);
    if (int e = ensure_pipeline(n)) return e;
    const size_t px = (size_t)n->H * n->W, per_in = px * CFFC_UNET_IN, per_out = px * CFFC_UNET_OUT;
    const int nb = (count + n->maxB - 1) / n->maxB;
    float *x[2] = {n->x32, n->x32b}, *y[2] = {n->y4, n->y4b};
    int device = 0;
    UCHK(hipGetDevice(&device));
    std::mutex mu;
    std::condition_variable cv;
    int launched = 0, fetched = 0;   // batches
    bool stop = false;
    hipError_t down_err = hipSuccess;
    auto size = [&](int i) { return std::min(n->maxB, count - i * n->maxB); };
    auto fetch = [&](int i) -> hipError_t {
        hipError_t e = hipEventSynchronize(n->computed[i & 1]);
        if (e == hipSuccess)
            e = hipMemcpyAsync(outputs + per_out * n->maxB * i, y[i & 1], per_out * size(i) * 4, hipMemcpyDeviceToHost,
                               n->down);
        return e == hipSuccess ? hipStreamSynchronize(n->down) : e;
    };
    auto fetch_all = [&]() {
        hipError_t e = hipSetDevice(device);
        for (int i = 0; i < nb && e == hipSuccess; ++i) {
            {
                std::unique_lock<std::mutex> l(mu);
                cv.wait(l, [&] { return launched > i || stop; });
                if (launched <= i) return;
            }
            e = fetch(i);
            std::lock_guard<std::mutex> l(mu);
            if (e == hipSuccess) fetched = i + 1;
            cv.notify_all();
        }
        std::lock_guard<std::mutex> l(mu);
        down_err = e;
        if (e != hipSuccess) stop = true;
        cv.notify_all();
    };
    std::thread second;
    try {
        second = std::thread(fetch_all);
    } catch (...) {
        // no second thread: one batch after the other
        for (int i = 0; i < nb; ++i)
            if (int e = cffc_unet_predict(n, inputs + per_in * n->maxB * i, size(i), outputs + per_out * n->maxB * i))
                return e;
        return 0;
    }
    auto send = [&](int i) -> int {
        {
            // batch i - 2 has left both of its buffers
            std::unique_lock<std::mutex> l(mu);
            cv.wait(l, [&] { return fetched >= i - 1 || stop; });
            if (stop) return 0;   // reported below
        }
        const int B = size(i);
        UCHK(hipMemcpyAsync(x[i & 1], inputs + per_in * n->maxB * i, per_in * B * 4, hipMemcpyHostToDevice, n->up));
        UCHK(hipStreamSynchronize(n->up));
        UCHK(cffc_unet_launch_to_bf16(x[i & 1], n->t[n->x0].act, (int64_t)per_in * B, n->stream));
        if (int e = forward(n, B, y[i & 1])) return e;
        UCHK(hipEventRecord(n->computed[i & 1], n->stream));
        std::lock_guard<std::mutex> l(mu);
        launched = i + 1;
        cv.notify_all();
        return 0;
    };
    int rc = 0;
    for (int i = 0; i < nb && !rc; ++i) rc = send(i);
    if (rc) {
        std::lock_guard<std::mutex> l(mu);
        stop = true;
        cv.notify_all();
    }
    second.join();
    (void)hipStreamSynchronize(n->stream);
    if (rc) return rc;
    UCHK(down_err);
    return 0;
}

extern "C" int cffc_unet_mfma_layout_probe(float out[256]) {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return ufail(CFFC_E_NODEVICE, "no HIP device");
    float *d = nullptr;
    UCHK(hipMalloc((void **)&d, 256 * 4));
    hipError_t e = cffc_unet_launch_mfma_layout(d, nullptr);
    if (e == hipSuccess) e = hipMemcpy(out, d, 256 * 4, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) return ufail(CFFC_E_HIP, "probe: %s", hipGetErrorString(e));
    return 0;
}

extern "C" void *cffc_unet_stream(cffc_unet *n) { return n ? (void *)n->stream : nullptr; }
