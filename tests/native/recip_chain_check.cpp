// The FP64 division and square root of the kernels (euler2d_state.hpp, its device
// side) on the host: v_rcp_f64 and v_rsq_f64 are stood in for by the correctly
// rounded value moved by up to 2^29 units of the last place, the accuracy their
// documentation states, at random and at its ends.  Every result has to equal the
// host's IEEE operation, from whatever value the hardware starts.  For recip one kind of
// quotient depends on that value and is left to a test on the device: a power of two
// over a divisor whose mantissa is all ones lies 2^-107 above the middle of two
// doubles.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

static std::mt19937_64 rng(7);
static double perturbed(double v) {
    if (!(v > 0x1p-1000 && v < 0x1p1000) && !(v < -0x1p-1000 && v > -0x1p1000)) return v;
    const int64_t lim = (int64_t)1 << 29;
    const uint64_t r = rng();
    const int64_t off = (r & 7) == 0 ? lim : (r & 7) == 1 ? -lim : (int64_t)(r >> 8) % (2 * lim + 1) - lim;
    int64_t b;
    memcpy(&b, &v, 8);
    b += off;
    memcpy(&v, &b, 8);
    return v;
}
static double hw_rcp(double b) { return perturbed(1.0 / b); }
static double hw_rsq(double b) { return perturbed(1.0 / std::sqrt(b)); }
static double fixup(double q, double b, double a) {
    if (a == 0 || b == 0 || std::isinf(a) || std::isinf(b) || a != a || b != b) return a / b;
    return std::copysign(q, std::signbit(a) != std::signbit(b) ? -1.0 : 1.0);
}
#define __HIP_DEVICE_COMPILE__ 1
#define __builtin_amdgcn_rcp hw_rcp
#define __builtin_amdgcn_rsq hw_rsq
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_div_fixup fixup
#define __builtin_amdgcn_ballot_w64(x) ((x) ? 1 : 0)
static int __double2loint(double x) {
    uint64_t u;
    memcpy(&u, &x, 8);
    return (int)(uint32_t)u;
}
static int __double2hiint(double x) {
    uint64_t u;
    memcpy(&u, &x, 8);
    return (int)(uint32_t)(u >> 32);
}
static double __hiloint2double(int hi, int lo) {
    const uint64_t u = ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
    double x;
    memcpy(&x, &u, 8);
    return x;
}
#define __builtin_amdgcn_class(x, m) ((x) == 0 || ((x) > 0 && std::isinf(x)))
#include "../../cffc_amd/csrc/euler2d_state.hpp"
using namespace cffc;

// random, or near the ends where quotients lie next to the middle of two doubles, or
// with a low word of ones
static double mantissa() {
    const uint64_t r = rng(), k = (r >> 8) % 64;
    uint64_t f = r >> 12;
    switch (r & 15) {
    case 0: f = 0; break;
    case 1: f = ~(uint64_t)0 >> 12; break;
    case 2: f = k; break;
    case 3: f = (~(uint64_t)0 >> 12) - k; break;
    case 4: f |= 0xFFFFFFFFu; break;
    }
    return 1.0 + (double)f * 0x1p-52;
}
static double value(int e) { return std::ldexp(mantissa(), (int)(rng() % (2 * e + 1)) - e); }

static long bad = 0;
static void same(const char *what, double got, double want, double a, double b) {
    if (memcmp(&got, &want, 8) == 0) return;
    if (bad++ < 20) printf("%s: %a, not %a, for %a and %a\n", what, got, want, a, b);
}
static uint64_t fraction(double x) {
    uint64_t u;
    memcpy(&u, &x, 8);
    return u & (((uint64_t)1 << 52) - 1);
}
static bool from_estimate(double a, double b) { return fraction(a) == 0 && fraction(b) == ((uint64_t)1 << 52) - 1; }
static void quotient(const char *what, double got, double a, double b) { same(what, got, a / b, a, b); }

int main(int argc, char **argv) {
    const long n = argc > 1 ? atol(argv[1]) : 1000000;
    const double g1i = 1.0 / (1.40 - 1.0);
    for (long k = 0; k < n; ++k) {
        const double s = rng() & 1 ? -1.0 : 1.0;
        {   // any pair
            const double a = s * value(300), b = value(300) * (rng() & 1 ? -1.0 : 1.0);
            if (!from_estimate(a, b)) {
                quotient("rdivf(a, recip(b))", rdivf(a, recip(b)), a, b);
                quotient("rdiv(a, recip(b))", rdiv(a, recip(b)), a, b);
                quotient("qdivf(a, b)", qdivf(a, b), a, b);
            }
        }
        {   // gamma p / ((gamma - 1) d) from 1/d
            const double d = value(60), x = value(60), b = gm1<double>() * d;
            quotient("recip_near(gm1 d)", rdivf(x, recip_near(b, recip(d).r * g1i)), x, b);
            const Recip<double> rgam = {gam<double>(), 1.0 / 1.40};
            quotient("division by gamma", rdivf(x, rgam), x, 1.40);
        }
        {   // any divisor from a value a few units to 2^-41 away
            const double b = s * value(60), x = value(60), d = std::ldexp(1.0, -41 - (int)(rng() % 14));
            quotient("recip_near(b)", rdivf(x, recip_near(b, 1.0 / b * (1.0 + (rng() & 1 ? d : -d)))), x, b);
        }
        {   // a2 -> c, and 1/c, 1/c^2, 1/a2 one from the other
            const double a2 = value(60), x = s * value(60);
            double h;
            const double c = qsqrt_h(a2, h);
            same("qsqrt_h", c, std::sqrt(a2), a2, 0.0);
            same("qsqrt", qsqrt(a2), std::sqrt(a2), a2, 0.0);
            const Recip<double> rc = recip_near(c, 2.0 * h), rc2 = recip_near(c * c, rc.r * rc.r);
            quotient("recip_near(c)", rdivf(x, rc), x, c);
            quotient("recip_near(c^2)", rdivf(0.5, rc2), 0.5, c * c);
            quotient("recip_near(a2)", rdivf(-1.0, recip_near(a2, rc2.r)), -1.0, a2);
        }
    }
    printf("%ld of %ld\n", bad, n);
    return bad != 0;
}
