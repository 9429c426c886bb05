// tran.hip -- calc_flux_tran (SRC/flux.f90:18-127) with the TRANLIB mixture rules it calls.
//
// Three kernels per flux evaluation:
//   k_tran_state: 64 cells per workgroup of four waves, the species split over the waves
//     (fluid_coop.hpp), for the cells on both sides of every interface (interior cells plus one
//     ghost layer per block end): T from the conserved state (temperature_con on the unnormalised Y,
//     SRC/flux.f90:33-55), p and log T.
//   k_tran_pairs: ONE WAVE PER CELL OR TWO CELLS (lanes over species): the Wilke mixture viscosity
//     (MCAVIS, tranlib.f:734-762), the mixture conductivity (MCACON, tranlib.f:876-891) and the
//     mixture-averaged diffusion coefficients (MCADIF -> MCEDIF, tranlib.f:1022-1024, 1095-1148),
//     then dif_k = (1 - X_k) / (1 - Y_k) D_km (SRC/flux.f90:62-72).
//   k_flux_tran: 64 interfaces per workgroup of four waves: central differences of u, T and Y
//     between the two cells and arithmetic means of the coefficients (SRC/flux.f90:74-123);
//     F = 0 + transport flux, and the advection kernel then adds its flux on top, as Fplus
//     accumulates in the reference (SRC/timeintegration.f90:138-146).
//
// SRC/flux.f90:56-57 takes mu from viscosity_ea -> MCAVIS_EA, a routine the reference does not
// ship; the Wilke mixture rule of MCAVIS (the routine SRC/trans.f90:46-59 wraps) stands in for it.
#include <algorithm>
#include <cmath>

#include "fluid_coop.hpp"
#include "tran.hpp"

namespace fcfd {

namespace {

// MCEVAL (tranlib.f:1335) of a fit of at most four coefficients, absent ones 0
__device__ __forceinline__ double mceval(const double *c, double x) {
    return ((c[3] * x + c[2]) * x + c[1]) * x + c[0];
}

template <int NSP>
__global__ void __launch_bounds__(64 * GW, 3) k_tran_state(TranArgs a) {
    constexpr int M = group_m<NSP>();
    __shared__ CoopShared sh;
    CThermo *m = constant(a.thermo);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned nc = unsigned(a.ncell) + 2u, n = unsigned(a.nblk) * nc;
    const unsigned t0 = xcd_block() * 64u + unsigned(lane);
    const bool live = t0 < n;
    const unsigned t = live ? t0 : n - 1u;
    const unsigned b = t / nc;
    const unsigned c = b * unsigned(a.S) + unsigned(a.lv) - 1u + (t - b * nc);
    const unsigned cb = column_bytes(c, lane0(c));
    const double *Qc = a.Qc + lane0(c);
    double *props = a.props + lane0(t);
    double y[M], x[M], s1[1];
#pragma unroll
    for (int j = 0; j < M; ++j) y[j] = at_byte(Qc + long(3 + min(w * M + j, NSP - 1)) * a.P, cb);
    const double rho = at_byte(Qc, cb);
    const double u = at_byte(Qc + a.P, cb) / rho;
    const double et = at_byte(Qc + 2 * a.P, cb) / rho;
    bool ok = den_ok(rho);
#pragma unroll
    for (int j = 0; j < M; ++j) {
        y[j] = w * M + j < NSP ? y[j] : 0.0;
        ok = ok && num_ok(y[j]);
    }
    const bool fast = __all(ok);
    scale_coop<M>(fast, rho, y);
    // Yi2Xi (CKYTX), no adjust_sum
    over_wt_coop<NSP>(m, w, fast, y, x);
    chain_sum<1, M>(sh.c[0], w, lane, [&](int, int j) { return x[j]; }, s1);
    ytx_coop<NSP>(m, w, fast, s1[0], y, x);
    const unsigned pb = column_bytes(t, lane0(t));
    auto put = [pb, live](double *row, double v) {
        if (live) *reinterpret_cast<double *>(reinterpret_cast<char *>(row) + pb) = v;
    };
#pragma unroll
    for (int j = 0; j < M; ++j) {
        if (w * M + j >= NSP) break;
        put(props + long(5 + w * M + j) * a.PP, y[j]);
        put(props + long(5 + NSP + w * M + j) * a.PP, x[j]);
    }
    double wtm;
    const double ek = 0.5 * (u * u);
    const double T = temperature_coop<NSP>(m, sh, w, lane, et - ek, x, wtm);
    if (w == 0) {
        put(props, rho);
        put(props + a.PP, u);
        put(props + 2 * a.PP, T);
        put(props + 3 * a.PP, (rho * 1.e-3) * m->ru * T / wtm * 0.1);     // pressure (CKPX, SI)
        put(props + 4 * a.PP, fm_log(T));
    }
}

// Lane k < NSP is species k; it walks its row j = 0 .. NSP - 1 of the Wilke and binary-diffusion sums in
// TRANLIB's order.  A row's table entries are read by neighbouring lanes and serve CPW cells; the
// quotients and the square root go through reciprocals where a cell's values allow it (FAST), with
// the same bits.  Bound: FP64 issue, two thirds of it the exponential of D_jk.  Before, every lane of a
// cell's wave repeated the temperature iteration and gathered its D fit per lane, with two square
// roots and three divisions per pair: 786 us for 16,384 cells, 90 us for 510 (now k_tran_state and
// this kernel, 195 and 47 us).  Forming D_jk once for
// both rows and rotating it between the lanes, the sums in offset order, is 1.5 times faster again, but
// those sums round differently, and a flame's heat release feels it.  (Kept in LDS, D_jk could be summed in
// TRANLIB's order: not tried.)
template <int NSP, int CPW>
struct PairLds {
    double2 xv[4 * CPW][64];                            // X_j, 1 / vis_j
    double v[4 * CPW][64];                              // vis_j
    double xw[4 * CPW][64];                             // max(X_j, 1e-50) w_j
    double y[4 * CPW][64];                              // Y_j, then dif_j
    double t[4 * CPW][4][64];                           // terms of the sums over all species
};

template <int NSP, int CPW, bool FAST>
__device__ __forceinline__ void pair_rows(const DevTran *__restrict__ tr, const PairLds<NSP, CPW> &sh, int q0, int lane,
                                          const double (&lt)[CPW], const double (&vis)[CPW], double (&si)[CPW],
                                          double (&sxod)[CPW], double (&sw)[CPW]) {
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        si[c] = 0.0;
        sxod[c] = 0.0;
        sw[c] = -sh.xw[q0 + c][lane];
    }
    for (int j = 0; j < NSP; ++j) {
        const double d0 = tr->pair_d[j][0][lane], d1 = tr->pair_d[j][1][lane], d2 = tr->pair_d[j][2][lane],
                     d3 = tr->pair_d[j][3][lane];
        const double sq_w = tr->pair_w[j][0][lane], cw = tr->pair_w[j][1][lane], rc = tr->pair_w[j][2][lane];
#pragma unroll
        for (int c = 0; c < CPW; ++c) {
            const double2 xv = sh.xv[q0 + c][j];
            const double vj = sh.v[q0 + c][j];
            // MCAVIS (tranlib.f:752-758)
            const double ratio = FAST ? quot(vis[c], vj, xv.y) : vis[c] / vj;
            const double arg = ratio * sq_w;
            const double aa = 1.0 + (FAST ? sqrt_core(arg) : sqrt(arg));
            const double num = xv.x * (aa * aa);
            si[c] = si[c] + (FAST ? quot(num, cw, rc) : num / cw);
            // MCEDIF (tranlib.f:1130-1146): D_jk; the term of j = k is zero in sxod, and sw runs from
            // -x_k w_k over all j
            const double D = exp_core(((d3 * lt[c] + d2) * lt[c] + d1) * lt[c] + d0);
            sw[c] = sw[c] + sh.xw[q0 + c][j];
            sxod[c] = sxod[c] + fmax(xv.x, 1.0e-50) * (j == lane ? 0.0 : D);
        }
    }
}

template <int NSP, int CPW>
__global__ void __launch_bounds__(256) k_tran_pairs(TranArgs a) {
    constexpr int NCW = 4 * CPW;
    __shared__ PairLds<NSP, CPW> sh;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, q0 = w * CPW;
    const unsigned n = unsigned(a.nblk) * (unsigned(a.ncell) + 2u);
    const unsigned c0 = blockIdx.x * unsigned(NCW);
    const DevTran *__restrict__ tr = a.tran;
    const long PP = a.PP;
    for (int i = threadIdx.x; i < NCW * 64; i += 256) {
        const int c = i % NCW, k = i / NCW;
        const unsigned pc = min(c0 + unsigned(c), n - 1u);
        sh.xv[c][k].x = k < NSP ? a.props[long(5 + NSP + k) * PP + pc] : 0.0;
        sh.y[c][k] = k < NSP ? a.props[long(5 + k) * PP + pc] : 0.0;
    }
    __syncthreads();
    const double wk = lane < NSP ? tr->twt[lane] : 0.0;
    double x[CPW], lt[CPW], vis[CPW], si[CPW], sxod[CPW], sw[CPW], p[CPW];
    bool ok = true;
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        const unsigned pc = min(c0 + unsigned(q0 + c), n - 1u);
        p[c] = a.props[3 * PP + pc];
        lt[c] = a.props[4 * PP + pc];
        x[c] = sh.xv[q0 + c][lane].x;
        vis[c] = exp_core(mceval(tr->cofeta[lane], lt[c]));
        const double lam = exp_core(mceval(tr->coflam[lane], lt[c]));
        sh.xv[q0 + c][lane].y = 1.0 / vis[c];
        sh.v[q0 + c][lane] = vis[c];
        sh.xw[q0 + c][lane] = fmax(x[c], 1.0e-50) * wk;
        sh.t[q0 + c][1][lane] = x[c] * lam;
        sh.t[q0 + c][2][lane] = x[c] / lam;
        sh.t[q0 + c][3][lane] = wk * x[c];
        ok = ok && num_ok(x[c]) && den_ok(vis[c]);
    }
    __syncthreads();
    if (__all(ok)) pair_rows<NSP, CPW, true>(tr, sh, q0, lane, lt, vis, si, sxod, sw);
    else pair_rows<NSP, CPW, false>(tr, sh, q0, lane, lt, vis, si, sxod, sw);
#pragma unroll
    for (int c = 0; c < CPW; ++c) sh.t[q0 + c][0][lane] = x[c] * vis[c] / si[c];
    __syncthreads();
    // the sums over all species in species order, one per lane: lane 4 c + s takes sum s of cell c
    double sum = 0.0;
    {
        const double *t = sh.t[q0 + min(lane >> 2, CPW - 1)][lane & 3];
        for (int k = 0; k < NSP; ++k) sum = sum + t[k];
    }
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        const int q = q0 + c;
        const double so = bcast(sum, 4 * c), sl = bcast(sum, 4 * c + 1), slr = bcast(sum, 4 * c + 2),
                     wtm = bcast(sum, 4 * c + 3);
        // MCADIF: D_km = sxw / (wtm sxod) * patmos / p (p in dyn/cm^2), cm^2/s -> m^2/s
        double D = sw[c] / (wtm * sxod[c]);
        D = D * tr->patmos / (p[c] * 10.0);
        D = D * 1.e-4;
        const double y = sh.y[q][lane];
        const double dif = (1.0 - x[c]) / (1.0 - y) * D;
        sh.y[q][lane] = y == 1.0 ? 0.0 : dif;
        const unsigned pc = c0 + unsigned(q);
        if (lane == 0 && pc < n) {
            a.props[3 * PP + pc] = so * sqrt(8.0) * 0.1;                     // SRC/trans.f90:57-59 (cgs -> SI)
            a.props[4 * PP + pc] = 0.5 * (sl + 1.0 / slr) * 1.e-5;           // SRC/trans.f90:74-76
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NCW * NSP; i += 256) {
        const int c = i % NCW, k = i / NCW;
        if (c0 + unsigned(c) < n) a.props[long(5 + NSP + k) * PP + c0 + c] = sh.y[c][k];
    }
}

template <int NSP>
__global__ void __launch_bounds__(64 * GW, 3) k_flux_tran(TranArgs a) {
    constexpr int M = group_m<NSP>();
    __shared__ CoopShared sh;
    CThermo *m = constant(a.thermo);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned n1 = unsigned(a.ncell) + 1u, n = unsigned(a.nblk) * n1;
    const unsigned t0 = xcd_block() * 64u + unsigned(lane);
    const bool live = t0 < n;
    const unsigned t = live ? t0 : n - 1u;
    const unsigned b = t / n1, j = t - b * n1;
    const unsigned c = b * (n1 + 1u) + j;              // cell ista-1+j; ista+j follows
    const unsigned pb = column_bytes(c, lane0(c));
    const double *props = a.props + lane0(c);
    const long PP = a.PP;
    auto pair = [&](int row, double &v0, double &v1) {
        const double *q = props + long(row) * PP;
        v0 = at_byte(q, pb);
        v1 = at_byte(q + 1, pb);
    };
    double dy[M], da[M], rho0, rho1, u0, u1, T0, T1, mu0, mu1, ka0, ka1;
    pair(0, rho0, rho1); pair(1, u0, u1); pair(2, T0, T1); pair(3, mu0, mu1); pair(4, ka0, ka1);
    const double dx = a.dxb ? a.dxb[b] : a.dx;                // b_obj(ib)%smr_dx
    bool ok = true;
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const int k = min(w * M + i, NSP - 1);
        double y0, y1, d0, d1;
        pair(5 + k, y0, y1);
        pair(5 + NSP + k, d0, d1);
        da[i] = 0.5 * (d0 + d1);
        dy[i] = y1 - y0;
        ok = ok && num_ok(dy[i]);
    }
    scale_coop<M>(__all(ok), dx, dy);
    const double rho_a = 0.5 * (rho0 + rho1), u_a = 0.5 * (u0 + u1);
    const double T_a = 0.5 * (T0 + T1), mu_a = 0.5 * (mu0 + mu1);
    const double kap_a = 0.5 * (ka0 + ka1);
    const double tau = -(2.0 / 3.0 * mu_a * (2.0 * ((u1 - u0) / dx)));
    double h[M], hw[M], unused[M], hs[1];
    species_thermo<NSP, true, false, true>(m, w, T_a, __all(den_ok(T_a)), h, unused);
    ok = true;
#pragma unroll
    for (int i = 0; i < M; ++i) ok = ok && num_ok(h[i]);
    over_wt_coop<NSP>(m, w, __all(ok), h, hw);
    char *F = reinterpret_cast<char *>(a.F) + t * 8ul;
    const long PF8 = a.PF * 8;
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const int k = min(w * M + i, NSP - 1);
        const double f = rho_a * da[i] * dy[i];
        if (live && w * M + i < NSP) *reinterpret_cast<double *>(F + (3 + k) * PF8) = 0.0 - f;
        h[i] = w * M + i < NSP ? -(hw[i] * 1.e-4 * da[i] * dy[i]) : 0.0;     // CKHMS, SI
    }
    chain_sum<1, M>(sh.c[0], w, lane, [&](int, int i) { return h[i]; }, hs);
    if (w == 0 && live) {
        *reinterpret_cast<double *>(F) = 0.0 + 0.0;
        *reinterpret_cast<double *>(F + PF8) = 0.0 + tau;
        *reinterpret_cast<double *>(F + 2 * PF8) = 0.0 + (tau * u_a + rho_a * hs[0] - kap_a * ((T1 - T0) / dx));
    }
}

// Cells from which a wave takes two of them (the pair tables, 190 kB, are read once for two cells)
// instead of one.  The whole flux at 16,384 / 65,536 cells takes 262 / 792 us with one cell per wave,
// 219 / 638 with two, 223 / 643 with three, 226 / 634 with four; at 2,048 cells 85, 86, 82, 90 us.
constexpr unsigned TRAN_WIDE = 4096;

}  // namespace

hipError_t launch_flux_tran(const TranArgs &a, int nsp, hipStream_t st) {
    const unsigned ncells = unsigned(a.nblk * (a.ncell + 2));
    const unsigned nif = unsigned(a.nblk * (a.ncell + 1));
#define FCFD_CASE(N)                                                                               \
    if (nsp == N) {                                                                                \
        hipLaunchKernelGGL((k_tran_state<N>), dim3((ncells + 63) / 64), dim3(64 * GW), 0, st, a); \
        hipError_t e = hipGetLastError();                                                          \
        if (e != hipSuccess) return e;                                                             \
        if (ncells >= TRAN_WIDE) hipLaunchKernelGGL((k_tran_pairs<N, 2>), dim3((ncells + 7) / 8), dim3(256), 0, st, a); \
        else hipLaunchKernelGGL((k_tran_pairs<N, 1>), dim3((ncells + 3) / 4), dim3(256), 0, st, a); \
        if ((e = hipGetLastError()) != hipSuccess) return e;                                       \
        hipLaunchKernelGGL((k_flux_tran<N>), dim3((nif + 63) / 64), dim3(64 * GW), 0, st, a);     \
        return hipGetLastError();                                                                  \
    }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

void build_dev_tran(const Mech &m, DevTran &t) {
    t.no = m.no;
    t.patmos = m.patmos;
    for (int k = 0; k < m.kk; ++k) {
        t.twt[k] = m.twt[k];
        for (int i = 0; i < m.no && i < 4; ++i) {
            t.cofeta[k][i] = m.cofeta[size_t(k) * m.no + i];
            t.coflam[k][i] = m.coflam[size_t(k) * m.no + i];
        }
        for (int j = 0; j < m.kk; ++j) {
            const int hi = std::max(j, k), lo = std::min(j, k);       // the link file's triangle
            for (int i = 0; i < m.no && i < 4 && j != k; ++i)
                t.pair_d[j][i][k] = -m.cofd[(size_t(hi) * m.kk + lo) * m.no + i];
            t.pair_w[j][0][k] = std::sqrt(m.twt[j] / m.twt[k]);
            t.pair_w[j][1][k] = std::sqrt(1.0 + m.twt[k] / m.twt[j]);
            t.pair_w[j][2][k] = 1.0 / t.pair_w[j][1][k];
        }
    }
}

}  // namespace fcfd
