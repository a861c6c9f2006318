// pp_noise.h -- the reference's Gaussian white noise on the device.
//
// fill_noise_threefry! / _threefry_gaussian (src/InitialConditions/
// RandomField.jl:46-81): cell idx (1-based, x fastest) of an N^3 grid takes
// the first normal of counter pair (idx-1) >> 1 when idx-1 is even, the
// second otherwise; each pair is Threefry-2x64-20 of counter (pair, 0) under
// key (seed, 0) (Salmon et al. 2011), two 53-bit uniforms in (0, 1] and
// Box-Muller in Float64.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pp {

// 64-bit rotation by 0 < r < 64 on the two halves (a 64-bit shift costs four
// times a 32-bit operation)
__device__ __forceinline__ uint64_t rotl64(uint64_t x, int r)
{
    uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    if (r >= 32) {
        const uint32_t t = lo;
        lo = hi;
        hi = t;
    }
    if (r & 31) {
        const uint32_t h = __builtin_amdgcn_alignbit(hi, lo, 32 - (r & 31));
        lo = __builtin_amdgcn_alignbit(lo, hi, 32 - (r & 31));
        hi = h;
    }
    return (uint64_t)hi << 32 | lo;
}

// -2 ln(x / 2^53) for a whole x in [1, 2^53].  x = 2^e m with m in
// [sqrt(1/2), sqrt 2): a fraction 1.f from sqrt 2 on (by its leading 20 bits) is
// halved.  ln m = 2 atanh(s), s = (m - 1) / (m + 1): the series in s^2 as its
// polynomial through seven Chebyshev nodes on [0, (3 - 2 sqrt 2)^2] (5e-18 of
// the whole); the quotient by the hardware's reciprocal, one Newton step and
// the remainder.
__device__ __forceinline__ double noise_neg2log(double x)
{
    constexpr double A[7] = {0.33333333333333348,  0.19999999999949722,  0.14285714313001635, 0.11111105565129939,
                             0.090914447278374735, 0.076658553091053863, 0.073082927124443114};
    const uint64_t bits = (uint64_t)__double_as_longlong(x);
    const uint32_t hi = (uint32_t)(bits >> 32), frac = hi & 0xfffffu;
    const uint32_t over = frac >= 434334u ? 1u : 0u;  // (sqrt 2 - 1) 2^20 = 434334.4
    const int n = 53 + 1023 - (int)(hi >> 20) - (int)over;
    const double m = __longlong_as_double((long long)((uint64_t)(frac + ((1023u - over) << 20)) << 32 | (uint32_t)bits));
    const double f = m - 1.0, d = m + 1.0;
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    double s = f * r;
    s = fma(fma(-d, s, f), r, s);
    const double z = s * s;
    double p = A[6];
#pragma unroll
    for (int q = 5; q >= 0; q--) p = fma(p, z, A[q]);
    const double s4 = 4.0 * s;
    return fma((double)n, 1.3862943611198906, -fma(s4, z * p, s4));
}

// sqrt(v) for v in [0, 2^7]: the hardware's reciprocal root, one coupled
// (Goldschmidt) step and the remainder; 0 gives 1e-100
__device__ __forceinline__ double noise_sqrt(double v)
{
    const double a = fmax(v, 1e-200);
    const double y = __builtin_amdgcn_rsq(a);
    double g = a * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    return fma(fma(-g, g, a), h, g);
}

// cos and sin of 2 pi x / 2^53 for a whole x in [0, 2^53]: 4 x / 2^53 less its
// nearest whole number is exact; over that quarter turn the two series as
// polynomials through seven Chebyshev nodes (5e-18)
__device__ __forceinline__ void noise_sincos(double x, double &c, double &s)
{
    constexpr double S[7] = {1.5707963267948966,     -0.64596409750624428,    0.079692626246043008, -0.0046817541323409756,
                             0.00016044115074219091, -3.5986433529823099e-06, 5.6339337815378543e-08};
    constexpr double C[7] = {1.2337005501361697,     -0.25366950790104781,    0.020863480763340773, -0.00091926027454684465,
                             2.5202039028029178e-05, -4.7106784055052271e-07, 6.3293963449674238e-09};
    double t = x * 4.4408920985006262e-16;  // 2^-51
    const double q = rint(t);
    t -= q;
    const uint32_t k = (uint32_t)(int)q;
    const double w = t * t;
    double ps = S[6], pc = C[6];
#pragma unroll
    for (int a = 5; a >= 0; a--) {
        ps = fma(ps, w, S[a]);
        pc = fma(pc, w, C[a]);
    }
    ps *= t;
    pc = fma(-pc, w, 1.0);
    const uint64_t bc = (uint64_t)__double_as_longlong(k & 1 ? ps : pc), bs = (uint64_t)__double_as_longlong(k & 1 ? pc : ps);
    c = __longlong_as_double((long long)(bc ^ (uint64_t)((k + 1) & 2) << 62));
    s = __longlong_as_double((long long)(bs ^ (uint64_t)(k & 2) << 62));
}

// the two Float64 normals of counter pair `pair`
//
// Every kernel that draws them is bound by the issue of these instructions,
// 229 of them (505 with the general log, cos and sin, whose ranges, signs and
// special values a uniform of 53 bits does not need).  Against 113 bits over
// 10^7 pairs the normals are right to 3.6e-16 of their radius (1.2e-16 rms),
// where the angle 2 pi u, rounded before its cosine is taken, left 7.3e-16
// (3.0e-16 rms).
__device__ __forceinline__ void threefry_normals(uint64_t pair, uint64_t seed, double &g1, double &g2)
{
    constexpr int ROT[8] = {16, 42, 12, 31, 16, 32, 24, 21};
    const uint64_t ks[3] = {seed, 0ull, 0x1BD11BDAA9FC1A22ull ^ seed};
    uint64_t x0 = pair + ks[0], x1 = ks[1];
#pragma unroll
    for (int blk = 0; blk < 5; blk++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            x0 += x1;
            x1 = rotl64(x1, ROT[(4 * blk + r) & 7]);
            x1 ^= x0;
        }
        const int inj = blk + 1;
        x0 += ks[inj % 3];
        x1 += ks[(inj + 1) % 3] + (uint64_t)inj;
    }
    const double r = noise_sqrt(noise_neg2log((double)(x0 >> 11) + 1.0));
    double c, s;
    noise_sincos((double)(x1 >> 11) + 1.0, c, s);
    g1 = r * c;
    g2 = r * s;
}

}  // namespace pp
