// fluid_coop.hpp -- the fluid kernels' workgroup functions: the species of a column (or of one side
// of an interface) split over the four waves of a workgroup, and quotients by a shared divisor.
//
// A lane of each of the four waves holds the same column; wave w owns the species block w*M ..
// w*M + M - 1.  A wave's species index is uniform, so coefficients are scalar operands; its species
// values stay in registers, M = 14 of 53 instead of all of them, which leaves room for several
// waves per SIMD and divides the length of the dependent chain of one column by four.  The
// reference adds its mixture sums in species order; chain_sum keeps that order exactly: wave 0 adds
// its block, hands the partial sum to wave 1 through LDS, and so on.
#pragma once

#include "columns.hpp"
#include "fcfd_device.hpp"

namespace fcfd {

constexpr int GW = SPECIES_BLOCKS;                               // waves per workgroup
template <int NSP> constexpr int group_m() { return (NSP + GW - 1) / GW; }   // species per wave

// The value of lane 0: of indices that grow with the lane, a workgroup's smallest (column_bytes).
__device__ __forceinline__ unsigned lane0(unsigned v) { return unsigned(__builtin_amdgcn_readfirstlane(int(v))); }

// The thermo tables through the constant address space: reads at a wave-uniform index are scalar
// loads wherever they stand (behind a store or a barrier the compiler would otherwise take them for
// possibly changed memory and read them through the vector caches).
using CThermo = const __attribute__((address_space(4))) DevThermo;
using CCoef = const __attribute__((address_space(4))) double;
__device__ __forceinline__ CThermo *constant(const DevThermo *m) { return (CThermo *)m; }

struct CoopShared {
    double c[2][4][64];      // partial sums in transit, two sets used in turn
};

// ---------------------------------------------------------------------------------------------
// Correctly rounded quotients by a divisor that serves many numerators.  recip() is 1 / d to half
// an ulp (hardware estimate, one cubic and one linear correction, all fused); quot() is the
// closing step of the division sequence itself: q = n r, one exact remainder, one fused correction
// (Markstein).  3 instructions a quotient instead of the 12 of n / d.  Both need d, n and n / d
// well inside the normal range; callers test that (in_range) and divide otherwise.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double recip(double d) {
    const double r0 = __builtin_amdgcn_rcp(d);
    const double e0 = __builtin_fma(-d, r0, 1.0);
    const double r1 = __builtin_fma(r0, __builtin_fma(e0, e0, e0), r0);     // error e0^3
    return __builtin_fma(r1, __builtin_fma(-d, r1, 1.0), r1);
}

__device__ __forceinline__ double quot(double n, double d, double r) {
    const double q = n * r;
    return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// r refined to 1 / d from an estimate at most 2^-51 off (relative).  Its error, half an ulp and 2^-102, leaves every
// quotient right but for divisors whose mantissa is within 2^-49 of 2: with the mantissas of d and of a
// quotient's middle as whole numbers the quotient is at least 1 / (2 d) ulps from the middle, and the closing step
// moves it by half of r's relative error, at most d 2^-107 + 2^-103.
__device__ __forceinline__ double refine(double d, double r) {
    return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}

// sqrt for x in the normal range: Goldschmidt's iteration on g -> sqrt(x), h -> 1 / (2 sqrt(x)) from the hardware's
// estimate of 1 / sqrt(x), closed by two residual corrections (x - g g exact under the fused multiply-add).
__device__ __forceinline__ double sqrt_core(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// numerators: 0 or 2^-700 <= |v| <= 2^60; divisors: 2^-60 <= d <= 2^60.  With these every quotient,
// remainder and reciprocal of the fluid kernels stays normal.  NaN is out of range.
__device__ __forceinline__ bool num_ok(double v) {
    const double a = fabs(v);
    return a <= 0x1p60 && (a >= 0x1p-700 || v == 0.0);
}
__device__ __forceinline__ bool den_ok(double d) { return d >= 0x1p-60 && d <= 0x1p60; }

// Sums of NC terms over all species, in species order from 0.0, the same in the four waves; term(c, j)
// is term c of the wave's species j (0 past the last species).  Every wave of the workgroup calls it
// (GW barriers).  buf alternates between consecutive calls: a wave may read the last call's totals
// while wave 0 already writes the next one's.
template <int NC, int M, class Term>
__device__ __forceinline__ void chain_sum(double (&buf)[4][64], int w, int lane, Term term, double (&out)[NC]) {
#pragma unroll 1
    for (int p = 0; p < GW; ++p) {
        if (w == p) {
            double s[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) s[c] = p == 0 ? 0.0 : buf[c][lane];
#pragma unroll
            for (int j = 0; j < M; ++j)
#pragma unroll
                for (int c = 0; c < NC; ++c) s[c] = s[c] + term(c, j);
#pragma unroll
            for (int c = 0; c < NC; ++c) buf[c][lane] = s[c];
        }
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) out[c] = buf[c][lane];
}

// ---------------------------------------------------------------------------------------------
// WENO5 on one side of an interface, side = lane half (0 left, 1 right), without the divisions' range
// handling: the weights' reciprocals take recip().  A multiplication by a power of two is exact, so
// it is fused with the addition it feeds; every other operation rounds as in reconstruct_side.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double at_byte(const double *__restrict__ row, unsigned off) {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(row) + off);
}

// The five stencil values of WENO5.
__device__ __forceinline__ void load5(const double *__restrict__ row, const unsigned (&o)[5], double (&u)[5]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) u[i] = at_byte(row, o[i]);
}

// The reconstruction from them; big collects whether a smoothness indicator is too large for recip()
// (or NaN), in which case the value is not to be used.
template <int RK>
__device__ __forceinline__ double weno5_lane(const double (&u)[5], int side, bool &big) {
    const double u0 = u[0], u1 = u[1], u2 = u[2], u3 = u[3], u4 = u[4];
    const double c13 = 13.0 / 12.0, eps = 1.0e-6;
    const double m3 = 3.0 * u2, m7 = 7.0 * u1, m11 = 11.0 * u2;
    double b3 = __builtin_fma(0.25, sq(__builtin_fma(-4.0, u1, u0) + m3), c13 * sq(__builtin_fma(-2.0, u1, u0) + u2));
    double b2 = __builtin_fma(0.25, sq(u1 - u3), c13 * sq(__builtin_fma(-2.0, u2, u1) + u3));
    double b1 = __builtin_fma(0.25, sq(__builtin_fma(-4.0, u3, m3) + u4), c13 * sq(__builtin_fma(-2.0, u3, u2) + u4));
    big = big || !(b3 + b2 + b1 < 0x1p200);
    if (RK == R_WENO5JS) {
        b3 = recip(sq(eps + b3));
        b2 = recip(sq(eps + b2));
        b1 = recip(sq(eps + b1));
    } else {
        const double tau = fabs(b3 - b1);
        const double d3 = eps + b3, d2 = eps + b2, d1 = eps + b1;
        b3 = 1.0 + sq(quot(tau, d3, recip(d3)));
        b2 = 1.0 + sq(quot(tau, d2, recip(d2)));
        b1 = 1.0 + sq(quot(tau, d1, recip(d1)));
    }
    const double a2 = 6.0 * b2, a1 = 3.0 * b1;
    const double ai = recip(b3 + a2 + a1);
    const double x2 = 2.0 * u0;
    const double t3 = ((side ? m11 : x2) - m7) + (side ? x2 : m11);
    const double t2 = __builtin_fma(2.0, u3, 5.0 * u2 - u1);
    const double t1 = __builtin_fma(2.0, u2, 5.0 * u3) - u4;
    return (1.0 / 6.0) * ai * (b3 * t3 + a2 * t2 + a1 * t1);
}

// tpow (fcfd_device.hpp) without its divisions: T in the range of den_ok
__device__ __forceinline__ TPow tpow_fast(double T, double ru) {
    TPow p;
    const double t2 = T * T, t3 = T * t2, t4 = t2 * t2;
    p.T = T;
    p.rut = T * ru;
    p.tnh1 = T / 2.0; p.tnh2 = quot(t2, 3.0, 1.0 / 3.0); p.tnh3 = t3 / 4.0; p.tnh4 = quot(t4, 5.0, 1.0 / 5.0);
    p.rtn0 = ru * 1.0; p.rtn1 = ru * T; p.rtn2 = ru * t2; p.rtn3 = ru * t3; p.rtn4 = ru * t4;
    return p;
}

// h_mol with T's reciprocal
__device__ __forceinline__ double h_mol_r(const Nasa &a, const TPow &p, double rT) {
    double s = a.a0;
    s = s + p.tnh1 * a.a1;
    s = s + p.tnh2 * a.a2;
    s = s + p.tnh3 * a.a3;
    s = s + p.tnh4 * a.a4;
    return p.rut * (s + quot(a.a5, p.T, rT));
}

// Molar u (with H: h; erg/mol) and cp (erg/(mol K)) of the wave's species at the lanes' temperatures T (fast:
// every T of the wave in den_ok's range).  One pass per temperature class among the lanes, nearly
// always one, two or three where a flame front crosses the wave: the class's coefficients are
// scalar operands.  Selected per lane they cost 24 moves and 12 selects a species, more than the
// polynomials.
template <int NSP, bool U, bool CP, bool H = false>
__device__ __forceinline__ void species_thermo(CThermo *m, int w, double T, bool fast,
                                               double (&u)[group_m<NSP>()], double (&c)[group_m<NSP>()]) {
    constexpr int M = group_m<NSP>();
    if (fast && m->nclass[w] > 0) {
        int cls = 0;
        for (int i = 0; i + 1 < m->nclass[w]; ++i) cls += T > m->cut[w][i] ? 1 : 0;
        const TPow p = tpow_fast(T, m->ru);
        const double rT = recip(T);
        auto one = [&](CCoef *b, double &uj, double &cj) {
            const Nasa a{b[0], b[1], b[2], b[3], b[4], b[5], 0.0};
            if (U) uj = H ? h_mol_r(a, p, rT) : h_mol_r(a, p, rT) - p.rut;
            if (CP) cj = cp_mol(a, p);
        };
        // (rows past the last species: unused rows of the table)
        const int c0 = __builtin_amdgcn_readfirstlane(cls);
        if (__all(cls == c0)) {
            CCoef *tab = &m->coef[w][c0][0][0];
#pragma unroll
            for (int j = 0; j < M; ++j) one(tab + 6 * j, u[j], c[j]);
        } else {
            unsigned long long todo = ~0ull;
#pragma unroll
            for (int j = 0; j < M; ++j) u[j] = c[j] = 0.0;
#pragma unroll 1
            while (todo) {
                const int c1 = __builtin_amdgcn_readlane(cls, __ffsll((long long)todo) - 1);
                const bool mine = cls == c1;
                CCoef *tab = &m->coef[w][c1][0][0];
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    double uj = 0.0, cj = 0.0;
                    one(tab + 6 * j, uj, cj);
                    if (U) u[j] = mine ? uj : u[j];
                    if (CP) c[j] = mine ? cj : c[j];
                }
                todo &= ~__ballot(mine);
            }
        }
    } else {
        const TPow p = tpow(T, m->ru);
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int k = min(w * M + j, NSP - 1);
            CCoef *lo = m->alo[k], *hi = m->ahi[k];
            const bool up = T > m->tmid[k];
            const Nasa a{up ? hi[0] : lo[0], up ? hi[1] : lo[1], up ? hi[2] : lo[2], up ? hi[3] : lo[3],
                         up ? hi[4] : lo[4], up ? hi[5] : lo[5], 0.0};
            if (U) u[j] = H ? h_mol(a, p) : h_mol(a, p) - p.rut;
            if (CP) c[j] = cp_mol(a, p);
            __builtin_amdgcn_sched_barrier(0);     // a rare path: no registers for overlap
        }
    }
}

// CKYTX of the wave's species: x = y / (sum_k y_k / wt_k * wt), not clipped.  fast: the y in num_ok's
// range.  Returns false (per wave) where the quotients left the fast range.
template <int NSP>
__device__ __forceinline__ void ytx_coop(CThermo *m, int w, bool fast, double sw,
                                         const double (&y)[group_m<NSP>()], double (&x)[group_m<NSP>()]) {
    constexpr int M = group_m<NSP>();
    if (fast && __all(den_ok(sw))) {
        const double rs = recip(sw);
        unsigned most = 0;        // the divisors' lower halves: refine() does not serve mantissas next to 2
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int k = min(w * M + j, NSP - 1);
            const double d = sw * m->wt[k];
            most = max(most, unsigned(__double2loint(d)));
            x[j] = quot(y[j], d, refine(d, rs * m->rwt[k]));
        }
        if (__any(most >= 0xfffffff0u)) {
#pragma unroll
            for (int j = 0; j < M; ++j) {
                const double d = sw * m->wt[min(w * M + j, NSP - 1)];
                x[j] = quot(y[j], d, recip(d));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            x[j] = y[j] / (sw * m->wt[min(w * M + j, NSP - 1)]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// v / s for the wave's species
template <int M>
__device__ __forceinline__ void scale_coop(bool fast, double s, double (&v)[M]) {
    if (fast && __all(den_ok(s))) {
        const double r = recip(s);
#pragma unroll
        for (int j = 0; j < M; ++j) v[j] = quot(v[j], s, r);
    } else {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            v[j] = v[j] / s;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// y / wt for the wave's species
template <int NSP>
__device__ __forceinline__ void over_wt_coop(CThermo *m, int w, bool fast,
                                             const double (&y)[group_m<NSP>()], double (&t)[group_m<NSP>()]) {
    constexpr int M = group_m<NSP>();
    if (fast) {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int k = min(w * M + j, NSP - 1);
            t[j] = quot(y[j], m->wt[k], m->rwt[k]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            t[j] = y[j] / m->wt[min(w * M + j, NSP - 1)];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// temperature_con (SRC/thermo.f90:211-257) from the wave's mole fractions x, with wtm = sum x wt.  The four
// waves iterate on the same values, so they take the same decisions and meet at the same barriers.
// Its sums use sh.c[1], then sh.c[0] and sh.c[1] in turn: the caller's last sum went through sh.c[0].
template <int NSP>
__device__ __forceinline__ double temperature_coop(CThermo *m, CoopShared &sh, int w, int lane, double e,
                                                   const double (&x)[group_m<NSP>()], double &wtm) {
    constexpr int M = group_m<NSP>();
    double s1[1];
    chain_sum<1, M>(sh.c[1], w, lane, [&](int, int j) { return x[j] * m->wt[min(w * M + j, NSP - 1)]; }, s1);
    wtm = s1[0];
    const double spe = e * 1.e4 * wtm;
    double T = 1000.0, f = 1.e30, dT = 1.e30;
    const double ru_gas = m->ru;
    for (int it = 0; it < 10; ++it) {
        const bool go = fabs(f) >= fabs(spe) * 1.e-9 && fabs(dT) >= T * 1.e-6;
        if (!__any(go)) break;
        double tu[M], tc[M], s[2];
        species_thermo<NSP, true, true>(m, w, T, true, tu, tc);       // 20 <= T <= 6000
#pragma unroll
        for (int j = 0; j < M; ++j) {
            tu[j] = x[j] * tu[j];
            tc[j] = x[j] * (tc[j] - ru_gas);
        }
        chain_sum<2, M>(sh.c[it & 1], w, lane, [&](int c, int j) { return c == 0 ? tu[j] : tc[j]; }, s);
        if (go) {
            f = s[0] - spe;
            dT = -f / s[1];
            T = T + dT;
            T = fmax(20.0, fmin(6000.0, T));
        }
    }
    return T;
}

// QcToqf (SRC/eos.f90:49-83) of one column per lane by the workgroup's four waves: rho, rho u and
// rho E in every wave, q the wave's rho Y (0 past the last species).  Gives u, T and the wave's
// renormalised mass fractions (store_y(j, y), before the temperature iteration, so that they need no
// registers during it).  The operations and their order are those of qc_to_qf_store.
template <int NSP, class StoreY>
__device__ __forceinline__ void qc_to_qf_coop(CThermo *m, CoopShared &sh, int w, int lane,
                                              double rho, double ru, double rE, const double (&q)[group_m<NSP>()],
                                              double &u, double &T, StoreY store_y) {
    constexpr int M = group_m<NSP>();
    double y[M];
    bool ok = den_ok(rho);
#pragma unroll
    for (int j = 0; j < M; ++j) ok = ok && num_ok(q[j]);
    const bool fast = __all(ok);
    u = ru / rho;
    const double e = rE / rho - 0.5 * (u * u);
    double s1[1];
#pragma unroll
    for (int j = 0; j < M; ++j) y[j] = q[j];
    scale_coop<M>(fast, rho, y);
#pragma unroll
    for (int j = 0; j < M; ++j) y[j] = fmax(y[j], 0.0);
    chain_sum<1, M>(sh.c[0], w, lane, [&](int, int j) { return y[j]; }, s1);      // adjust_sum
    scale_coop<M>(fast, s1[0], y);
#pragma unroll
    for (int j = 0; j < M; ++j) store_y(j, y[j]);
    double x[M];
    over_wt_coop<NSP>(m, w, fast, y, x);
    chain_sum<1, M>(sh.c[1], w, lane, [&](int, int j) { return x[j]; }, s1);      // CKYTX
    ytx_coop<NSP>(m, w, fast, s1[0], y, x);
#pragma unroll
    for (int j = 0; j < M; ++j) x[j] = fmax(x[j], 0.0);
    chain_sum<1, M>(sh.c[0], w, lane, [&](int, int j) { return x[j]; }, s1);      // adjust_sum
    scale_coop<M>(fast, s1[0], x);
    T = temperature_coop<NSP>(m, sh, w, lane, e, x, s1[0]);
}

}  // namespace fcfd
