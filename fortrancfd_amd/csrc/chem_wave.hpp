// chem_wave.hpp -- what the two integrator kernels (chem.hip, chem_coop.hip) share: the method's
// constants, wave reductions, the pivot search and the per-cell sums.
#pragma once

#include "chem.hpp"
#include "chem_device.hpp"
#include "fcfd_device.hpp"

namespace fcfd {

constexpr double CH_G = 0.435866521508459;
constexpr double CH_A21 = 0.2820667392457705;
constexpr double CH_B1 = 1.20849664917601;
constexpr double CH_B2 = -0.6443631706844692;
constexpr double CH_E1 = 0.43586652150845895;
constexpr double CH_E2 = -0.8717330430169181;
constexpr double CH_E3 = 0.435866521508459;
constexpr double CH_KAPPA = 0.03;
constexpr int CH_MAXIT = 7;
constexpr int CH_MAXSTEPS = 5000;

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// Largest value over the wave: row_shr 1/2/4/8 within each row of 16 lanes, then row_bcast 15 / 31
// across rows; lane 63 ends with the maximum.  fmax returns one of its operands, so the result is
// bitwise one of the inputs (NaN inputs are passed over).
__device__ __forceinline__ double wave_max(double v) {
    v = fmax(v, dpp_f64<0x111>(v));
    v = fmax(v, dpp_f64<0x112>(v));
    v = fmax(v, dpp_f64<0x114>(v));
    v = fmax(v, dpp_f64<0x118>(v));
    v = fmax(v, dpp_f64<0x142, 0xA>(v));
    v = fmax(v, dpp_f64<0x143, 0xC>(v));
    return bcast(v, 63);
}

// Largest value over the wave of an unsigned key, the same scheme as wave_max with one DPP max per
// stage (lanes without a source and rows outside the mask contribute 0, the identity).  Every lane
// of the wave must be active.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, true));
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, true));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// The pivot of an elimination step: the open row with the largest |entry| rk in the pivot column, the
// lowest such row on ties (NaN entries are passed over).  For |x| >= 0 the upper 32 bits of the
// double order like the value, so one 32-bit wave max finds the candidates; only when several rows
// share those bits are their full values compared.  If the column of every open row is NaN, the
// lowest open row, and ok = false.  Called by every lane of the wave (wave-wide reductions).
__device__ __forceinline__ int pivot_row(double rk, bool open, bool &ok) {
    const double av = fabs(rk);
    const bool num = open && av == av;
    const unsigned key = num ? (unsigned)__double2hiint(av) : 0u;
    const unsigned kmax = wave_max_u32(key);
    const bool top = num && key == kmax;
    unsigned long long hit = __ballot(top);
    if (__popcll(hit) > 1) {
        const double v = top ? av : -1.0;
        const double vmax = wave_max(v);
        hit = __ballot(top && v == vmax);
    }
    if (hit == 0ull) {
        hit = __ballot(open);
        ok = false;
    }
    return __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
}

__device__ __forceinline__ double wnorm(double v, double w, int n) {
    const double t = v * w;
    return sqrt(wsum(t * t) / n);
}

// Mixture e = sum Y u / W and cv = sum Y cv / W at T (wave sums); y_l this lane's Y.
template <int NSP>
__device__ __forceinline__ void energy(const DevThermo *__restrict__ th, double y_l, double T, double &e, double &cv) {
    const int lane = lane_id();
    double eu = 0.0, ec = 0.0;
    if (lane < NSP) {
        const Nasa a = nasa(th, lane, T);
        const TPow p = tpow(T, th->ru);
        eu = y_l * (h_mol(a, p) - p.rut) / th->wt[lane];
        ec = y_l * (cp_mol(a, p) - th->ru) / th->wt[lane];
    }
    e = wsum(eu);
    cv = wsum(ec);
}

__device__ __forceinline__ double adjusted(double y_l, int lane, int nsp) {
    const double v = lane < nsp ? fmax(y_l, 0.0) : 0.0;
    return v / wsum(v);
}

}  // namespace fcfd
