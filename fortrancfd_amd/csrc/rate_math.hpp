// rate_math.hpp -- the exponentials and logarithms of the rate code, with the bits of fcfd_math.h's, for the
// kernels that run them most (chem_coop.hip, chem_lane.hip).
#pragma once

#include "chem_device.hpp"
#include "fluid_coop.hpp"

namespace fcfd {

// The constants of the exponential and logarithm series, read through the constant address space: as
// scalar loads they are an operand of the multiply-add they belong to, where a 64-bit literal takes two
// moves first.  Users hold an opaque pointer (a compiler that sees the table turns it into literals).
struct Series {
    double exp[13];          // 1/14! .. 1/2! (fm_exp_series)
    double log[12];          // 2/25, 2/23 .. 2/3 (fm_log_dd)
    double inv_ln2, shift, ln2_hi, ln2_lo, limit;
    double inv_ln10_hi, inv_ln10_lo, ln10_hi, ln10_lo;
};
static __constant__ Series series = {
    {0x1.93974a8c07c9dp-37, 0x1.6124613a86d09p-33, 0x1.1eed8eff8d898p-29, 0x1.ae64567f544e4p-26, 0x1.27e4fb7789f5cp-22,
     0x1.71de3a556c734p-19, 0x1.a01a01a01a01ap-16, 0x1.a01a01a01a01ap-13, 0x1.6c16c16c16c17p-10, 0x1.1111111111111p-7,
     0x1.5555555555555p-5, 0x1.5555555555555p-3, 0.5},
    {2.0 / 25.0, 2.0 / 23.0, 2.0 / 21.0, 2.0 / 19.0, 2.0 / 17.0, 2.0 / 15.0, 2.0 / 13.0, 2.0 / 11.0, 2.0 / 9.0, 2.0 / 7.0,
     2.0 / 5.0, 2.0 / 3.0},
    FM_INV_LN2, FM_SHIFT, FM_LN2_HI, FM_LN2_LO, 1000.0, FM_INV_LN10_HI, FM_INV_LN10_LO, FM_LN10_HI, FM_LN10_LO};
using CSeries = const __attribute__((address_space(4))) Series;
__device__ __forceinline__ CSeries *get_series() {
    CSeries *k = (CSeries *)&series;
    asm volatile("" : "+s"(k));
    return k;
}

// a b + k with k a scalar operand (left to itself the compiler moves k into the destination first)
__device__ __forceinline__ double fma_k(double a, double b, double k) {
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(k));
    return r;
}

// exp of the two-term value x + xl with fm_exp's bits (arguments beyond +-1000 give infinity or 0)
__device__ __forceinline__ double exp2term(CSeries *k, double x, double xl) {
    const double xc = __builtin_fmin(__builtin_fmax(x, -k->limit), k->limit);
    const double kd = (xc * k->inv_ln2 + k->shift) - k->shift;
    const double r0 = __builtin_fma(-kd, k->ln2_hi, xc);
    const double r1 = xl - kd * k->ln2_lo;
    const double rh = r0 + r1;
    const double rl = r1 - (rh - r0);
    double p = k->exp[0];
#pragma unroll
    for (int i = 1; i < 13; ++i) p = fma_k(p, rh, k->exp[i]);
    const double q = (rh * rh) * p;
    const double s = 1.0 + rh;
    const double e = rh - (s - 1.0);
    return __builtin_amdgcn_ldexp(s + (e + (rl + (rh * rl + q))), int(kd));
}
// fm_exp for |x| < 2^128, NaN included: no clamp, one term.  (Far from 0 the reduction leaves more than ln2 / 2, but
// the power of two decides: 0 or infinity.  Beyond 2^128 the series overflows.)
__device__ __forceinline__ double exp_near(CSeries *k, double x) {
    const double kd = (x * k->inv_ln2 + k->shift) - k->shift;
    const double r0 = __builtin_fma(-kd, k->ln2_hi, x);
    const double r1 = -kd * k->ln2_lo;
    const double rh = r0 + r1;
    const double rl = r1 - (rh - r0);
    double p = k->exp[0];
#pragma unroll
    for (int i = 1; i < 13; ++i) p = fma_k(p, rh, k->exp[i]);
    const double q = (rh * rh) * p;
    const double s = 1.0 + rh;
    const double e = rh - (s - 1.0);
    return __builtin_amdgcn_ldexp(s + (e + (rl + (rh * rl + q))), int(kd));
}
// fm_exp, NaN included
__device__ __forceinline__ double exp_rate(CSeries *k, double x) {
    const double r = exp2term(k, x, 0.0);
    return x == x ? r : x;
}

// fm_log's two-term value for x > 0 in the normal range, its two quotients by one reciprocal
__device__ __forceinline__ double log_dd_rate(CSeries *k, double x, double &lo) {
    uint64_t b = fm_to_bits(x);
    int e = int(b >> 52) - 1023;
    b = (b & 0x000fffffffffffffULL) | 0x3ff0000000000000ULL;
    const bool half = b > 0x3ff6a09e667f3bcdULL;
    b -= half ? 0x0010000000000000ULL : 0ULL;
    e += half ? 1 : 0;
    const double f = fm_from_bits(b) - 1.0;
    const double u = 2.0 + f;
    const double ul = f - (u - 2.0);
    const double ru = recip(u);
    const double sh = quot(f, u, ru);
    const double sl = quot(__builtin_fma(-sh, u, f) - sh * ul, u, ru);
    const double z = sh * sh;
    double p = k->log[0];
#pragma unroll
    for (int i = 1; i < 12; ++i) p = fma_k(p, z, k->log[i]);
    const double small = 2.0 * sl + ((sh * z) * p + 2.0 * z * sl);
    const double ed = double(e);
    const double ph = ed * k->ln2_hi;
    const double pl = __builtin_fma(ed, k->ln2_hi, -ph);
    const double b2 = 2.0 * sh;
    const double t = ph + b2;
    const double bv = t - ph;
    const double err = (ph - (t - bv)) + (b2 - bv);
    const double tl = err + (pl + (ed * k->ln2_lo + small));
    const double hi = t + tl;
    lo = tl - (hi - t);
    return hi;
}

// fm_log10 for x > 0 in the normal range or +infinity
__device__ __forceinline__ double log10_rate(CSeries *k, double x) {
    double lo;
    const double hi = log_dd_rate(k, x, lo);
    const double qh = hi * k->inv_ln10_hi;
    const double ql = __builtin_fma(hi, k->inv_ln10_hi, -qh) + (hi * k->inv_ln10_lo + lo * k->inv_ln10_hi);
    return x == __builtin_inf() ? x : qh + ql;
}

// fm_exp10 (its argument carried as a two-term value)
__device__ __forceinline__ double exp10_rate(CSeries *k, double y) {
    const double xh = y * k->ln10_hi;
    const double xl = __builtin_fma(y, k->ln10_hi, -xh) + y * k->ln10_lo;
    const double r = exp2term(k, xh, xl);
    return y == y ? r : y;
}

// The temperature of an evaluation, the same in all lanes: T and what the rates take from it.  Outside
// den_ok's range (an iteration that has come apart) log T is NaN, and with it every rate.
struct Temp {
    double T, rT, logT;
    bool usual;
};

__device__ __forceinline__ Temp temperature(CSeries *k, double T) {
    Temp t;
    t.T = T;
    t.rT = recip(T);
    t.usual = den_ok(T);
    double lo;
    const double lg = log_dd_rate(k, T, lo);
    t.logT = t.usual ? lg : __builtin_nan("");
    return t;
}

// a / T for a table constant (DevKin::usual: zero or well inside the normal range)
__device__ __forceinline__ double over(double a, const Temp &t) { return quot(a, t.T, t.rT); }

// x ** m, 0 <= m <= 3 (ipow3 without branches)
__device__ __forceinline__ double pow3(double x, int m) {
    const double x2 = x * x, x3 = x * x2;
    double r = m == 1 ? x : 1.0;
    r = m == 2 ? x2 : r;
    return m == 3 ? x3 : r;
}

}  // namespace fcfd
