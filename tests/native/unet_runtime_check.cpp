// The U-Net's host runtime (unet.cpp) on a stand-in for the HIP runtime: device
// memory is host memory, work on the null stream runs as late as that stream
// allows (when something waits for it), work on the network's own streams, which
// do not order with the null stream, as early as it can.  Both are orders that a
// device may take.
#include "../../cffc_amd/csrc/unet.cpp"

#include <functional>
#include <map>

static std::map<char *, size_t> live;                 // device allocations
static std::vector<std::function<void()>> null_work;  // not run yet
static int mallocs_left = -1;                         // allocations that succeed; -1: all

static void drain() {
    for (auto &w : null_work) w();
    null_work.clear();
}
static void must_be_live(const void *p, size_t n, const char *what) {
    auto it = live.upper_bound((char *)p);
    if (it != live.begin() && (--it, (char *)p + n <= it->first + it->second)) return;
    fprintf(stderr, "FAIL: %s touches memory that is not allocated\n", what);
    _Exit(1);
}

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMalloc(void **p, size_t n) {
    if (mallocs_left == 0) return hipErrorOutOfMemory;
    if (mallocs_left > 0) --mallocs_left;
    *p = malloc(n);
    memset(*p, 0xA5, n);
    live[(char *)*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    drain();
    if (!live.erase((char *)p)) {
        fprintf(stderr, "FAIL: freed twice\n");
        _Exit(1);
    }
    free(p);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
    null_work.push_back([=] { memset(p, v, n); });
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t st) {
    if (!st) return hipMemset(p, v, n);
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    drain();
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    if (!st) return hipMemcpy(d, s, n, k);
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { drain(); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) {
    if (!st) drain();
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

// the kernels: those that move data do so, the others only succeed
hipError_t cffc_unet_launch_to_bf16(const float *src, bf16_t *dst, int64_t n, hipStream_t) {
    for (int64_t i = 0; i < n; ++i) {
        uint32_t u;
        memcpy(&u, src + i, 4);
        dst[i] = (bf16_t)(u >> 16);   // values of few bits
    }
    return hipSuccess;
}
hipError_t cffc_unet_launch_gather(const void *src, const int32_t *idx, int nrows, int64_t row_bytes, void *dst,
                                   hipStream_t) {
    for (int r = 0; r < nrows; ++r) {
        must_be_live((const char *)src + idx[r] * row_bytes, row_bytes, "gather");
        memcpy((char *)dst + r * row_bytes, (const char *)src + idx[r] * row_bytes, row_bytes);
    }
    return hipSuccess;
}
int cffc_unet_conv_tiles(int, int, int, int) { return 1; }
int cffc_unet_wgrad_chunks(int, int, int, int, int) { return 1; }
hipError_t cffc_unet_launch_mfma_layout(float *, hipStream_t) { return hipSuccess; }
hipError_t cffc_unet_launch_conv_fwd(const bf16_t *, int, int, const bf16_t *, int, int, int, int, const bf16_t *,
                                     const float *, int, int, bf16_t *, float *, bf16_t *, hipStream_t) {
    return hipSuccess;
}
hipError_t cffc_unet_launch_conv_bwd_data(const bf16_t *, int, int, int, int, const bf16_t *, int, int, int,
                                          const bf16_t *, bf16_t *, float *, float *, const float *, hipStream_t) {
    return hipSuccess;
}
hipError_t cffc_unet_launch_conv_bwd_weight(const bf16_t *, int, const bf16_t *, int, int, const bf16_t *, int, int,
                                            int, int, float *, hipStream_t) {
    return hipSuccess;
}
hipError_t cffc_unet_launch_reduce(const SumList *, hipStream_t) { return hipSuccess; }
hipError_t cffc_unet_launch_mse(const float *, const float *, int64_t, int, bf16_t *, float *, float *, hipStream_t) {
    return hipSuccess;
}
hipError_t cffc_unet_launch_adam(const AdamList *, int, float, float, float, float, float, float, int, hipStream_t) {
    return hipSuccess;
}
}

#define CHECK(c)                                                  \
    do {                                                          \
        if (!(c)) {                                               \
            fprintf(stderr, "FAIL line %d: %s\n", __LINE__, #c); \
            return 1;                                             \
        }                                                         \
    } while (0)

enum { H = 8, W = 16, PX = H * W, NS = 5 };

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    cffc_unet *n = nullptr;
    CHECK(cffc_unet_create(H, W, 2, 1, &n) == 0);
    std::vector<float> x(NS * PX * CFFC_UNET_IN), y(NS * PX * CFFC_UNET_OUT);
    for (size_t i = 0; i < x.size(); ++i) x[i] = (float)(1 + i % 100);
    for (size_t i = 0; i < y.size(); ++i) y[i] = (float)(1 + i % 77);
    if (what == "create") {
        CHECK(null_work.empty());   // nothing that clears a buffer is still to come
    } else if (what == "order") {
        CHECK(cffc_unet_set_dataset(n, NS, x.data(), y.data()) == 0);
        drain();
        for (size_t i = 0; i < x.size(); ++i) {
            uint32_t u;
            memcpy(&u, &x[i], 4);
            CHECK(n->ds_in[i] == (bf16_t)(u >> 16));
        }
        CHECK(memcmp(n->ds_tg, y.data(), y.size() * 4) == 0);
    } else if (what == "dataset") {
        const int32_t idx[2] = {0, NS - 1};
        float loss;
        for (int ok : {0, 1}) {   // neither buffer of the new dataset can be allocated, or only the first
            CHECK(cffc_unet_set_dataset(n, NS, x.data(), y.data()) == 0);
            CHECK(cffc_unet_train_step(n, idx, 2, 1e-3f, &loss) == 0);
            mallocs_left = ok;
            CHECK(cffc_unet_set_dataset(n, NS, x.data(), y.data()) == CFFC_E_NOMEM);
            mallocs_left = -1;
            CHECK(cffc_unet_train_step(n, idx, 2, 1e-3f, &loss) == CFFC_E_ARG);   // no dataset
        }
        CHECK(cffc_unet_set_dataset(n, NS, x.data(), y.data()) == 0);
        CHECK(cffc_unet_train_step(n, idx, 2, 1e-3f, &loss) == 0);
    } else {
        return 2;
    }
    cffc_unet_destroy(n);
    CHECK(live.empty());
    printf("ok\n");
    return 0;
}
