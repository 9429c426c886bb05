// chem_lane.hip -- explicit screen of the chemistry source: ONE CELL PER LANE.
//
// Every cell first tries the integrator's explicit pre-step (Heun over the whole dt with the
// embedded Euler error estimate, accepted when the weighted RMS error is <= 1, then the
// energy-consistent temperature).  Quiescent cells -- the cold bulk of a reacting domain -- end
// here; the others are appended to a work list for the wave-per-cell SDIRK kernel (chem.hip),
// which then starts from the unchanged state.  The arithmetic is the pre-step of that kernel; only
// the order of the species sums differs.  k_chem_retry runs the integrator's next explicit attempt
// (two half steps) the same way over a long work list, before the SDIRK kernel sees it.
//
// Mapping: a workgroup of RW = 16 waves owns NC = 64 cells (lane l of every wave is cell l; with
// NC < 64, lanes NC..63 would repeat cell NC - 1 and store nothing).  Concentrations and S/R - H/RT of
// the cells live in LDS as species-major [k][NC] blocks.  The reactions are taken in chunks of
// CH = 112 rows: the waves draw rows from a counter, evaluate each for all cells and put its rates of
// progress in LDS; after a barrier every wave adds the chunk's contributions to the species it was given
// (LaneSeg: by their number of terms), in row order, into one shared production-rate block.  Each
// species' production rate is therefore one sequential sum over the rows, independent of which wave does
// what.  Species-wise work (thermo, state update, norms) is split over the first NW = 8 waves by k mod
// NW; cell-wise scalars (T, sums) are combined through LDS in wave order, by every wave.
//
// Bound: the issue of one SIMD's four waves.  A plain row takes some 110 vector operations (two
// exponentials, a division), a fall-off row 500.  LDS (144 KB) holds one workgroup per compute unit; 128
// registers a lane allow its 16 waves.  65,536 cells (four rounds of 256 workgroups): 574 us a launch, 510
// cells: 155 us.  (682 and 181 while the series' constants went through vector registers and empty slots
// were selected away.)  Eight waves with 32-row chunks, one fixed row in
// eight each, and table reads that went through the vector cache at each branch took 1,098 and 334 us.
#include <algorithm>

#include "chem.hpp"
#include "chem_device.hpp"
#include "fcfd_device.hpp"
#include "rate_math.hpp"

namespace fcfd {

namespace {

constexpr int NW = LANE_NW;    // waves that own species
constexpr int RW = LANE_RW;    // waves per workgroup, each with rows of a chunk
constexpr int NC = LANE_NC;    // cells per workgroup
constexpr int CH = LANE_CHUNK; // reaction rows per chunk

template <int NSP>
struct LaneShared {
    double C[(NSP + 1) * NC];  // concentrations, mol/cm^3; the last row, for empty slots, is 1
    double G[(NSP + 1) * NC];  // S/R - H/RT; the last row is 0
    double W[NSP * NC];        // production rates
    double Q[CH * NC];         // rates of progress (forward minus reverse) of the current chunk; outside
                               // the reaction loop, the per-wave values of cross-wave sums
    int next[2];               // rows of a chunk handed out, by the chunk's parity
    double PF[7 * NC];         // pfac**m for m = -3 .. 3 (row m + 3), the equilibrium constants' factor
};

// The tables through the constant address space: reads at a wave-uniform index are scalar loads wherever
// they stand (behind a barrier or an LDS store they would otherwise go through the vector caches, one
// after the other as a row's branches ask for them).
using CKin = const __attribute__((address_space(4))) DevKin;
using CLanePlain = const __attribute__((address_space(4))) LanePlain;

// Both coefficient sets as scalars, the range selected per lane.  (Opaque: a compiler that sees the loads
// selects their address instead, which makes each a memory access per lane.)
__device__ __forceinline__ Nasa nasa(CThermo *m, int k, double T) {
    const bool up = T > m->tmid[k];
    auto pick = [&](int n) {
        double lo = m->alo[k][n], hi = m->ahi[k][n];
        asm("" : "+s"(lo));
        asm("" : "+s"(hi));
        return up ? hi : lo;
    };
    return Nasa{pick(0), pick(1), pick(2), pick(3), pick(4), pick(5), pick(6)};
}

// a / T for a table constant
__device__ __forceinline__ double over(double a, const Temp &t, bool usual) {
    double q = over(a, t);
    if (__builtin_expect(!usual, 0)) q = a / t.T;       // (the same in all lanes)
    return q;
}

// reaction() (chem_device.hpp) for a row the whole wave evaluates, as forward minus reverse rate of
// progress: the same operations, with the exponentials and logarithms of rate_math.hpp and T's
// reciprocal.
__device__ __forceinline__ double lane_row_q(CKin *K, CSeries *ks, int i, const Temp &tp, bool usual,
                                             double pfac, double ctot, const double *__restrict__ c,
                                             const double *__restrict__ smh) {
    auto nu = &K->nu[i][0], nk = &K->nk[i][0];
    if (nu[0] == 0) return 0.0;
    double kf = K->A[i];
    if (!K->arr0[i]) kf = kf * exp_rate(ks, K->B[i] * tp.logT - over(K->E[i], tp, usual));
    double kr = 0.0;
    if (K->rev[i]) {
        double s = 0.0;
        for (int n = 0; n < 6; ++n) {
            const int k = nk[n];
            if (k >= 0) s = s + (double)nu[n] * smh[k * NC];
        }
        double eqk = s != 0.0 ? exp_rate(ks, fmin(s, K->exparg)) : 1.0;
        eqk = eqk * ipow(pfac, K->nus[i]);
        kr = kf / fmax(eqk, K->small);
    }
    double ctb = 1.0;
    const int t = K->tb[i];
    if (t >= 0) {
        ctb = ctot;
        const int nl = K->ntbs[t];
        for (int l = 0; l < nl; ++l) {
            const int tk = K->tbk[t][l];
            ctb = ctb + (K->tba[t][l] - 1.0) * c[(tk >= 0 ? tk : 0) * NC];
        }
    }
    const int f = K->fo[i];
    if (f >= 0) {
        auto fp = &K->fpar[f][0];
        const double rklow = fp[0] * exp_rate(ks, fp[1] * tp.logT - over(fp[2], tp, usual));
        double pr;
        if (K->kfal[f] < 0) { pr = rklow * ctb / kf; ctb = 1.0; }
        else pr = rklow * c[K->kfal[f] * NC] / kf;
        double pcor = pr / (1.0 + pr);
        if (K->ifop[f] > 1) {
            const double prlog = log10_rate(ks, fmax(pr, K->small));
            double fc;
            if (K->ifop[f] == 2) {
                const double xp = 1.0 / (1.0 + prlog * prlog);
                fc = fm_pow(fp[3] * fm_exp(-fp[4] / tp.T) + fm_exp(-tp.T / fp[5]), xp) * fp[6] * fm_pow(tp.T, fp[7]);
            } else {
                double fcent = (1.0 - fp[3]) * exp_rate(ks, -tp.T / fp[4]) + fp[3] * exp_rate(ks, -tp.T / fp[5]);
                if (K->ifop[f] == 4) fcent = fcent + exp_rate(ks, -over(fp[6], tp, usual));
                const double fclog = log10_rate(ks, fmax(fcent, K->small));
                // single-precision literals of cklib.f:6915-6917
                const double xn = 0.75 - (double)1.27f * fclog;
                const double cprlog = prlog - ((double)0.4f + (double)0.67f * fclog);
                const double q = cprlog / (xn - (double)0.14f * cprlog);
                fc = exp10_rate(ks, fclog / (1.0 + q * q));
            }
            pcor = fc * pcor;
        }
        kf = kf * pcor;
        kr = kr * pcor;
    }
    kf = kf * ctb * 1.0;
    kr = kr * ctb * 1.0;
    double qf = kf * ipow(c[nk[0] * NC], abs(nu[0]));
    double qr = kr * ipow(c[nk[3] * NC], nu[3]);
    if (nk[1] >= 0) {
        qf = qf * ipow(c[nk[1] * NC], abs(nu[1]));
        if (nk[2] >= 0) qf = qf * ipow(c[nk[2] * NC], abs(nu[2]));
    }
    if (nk[4] >= 0) {
        qr = qr * ipow(c[nk[4] * NC], nu[4]);
        if (nk[5] >= 0) qr = qr * ipow(c[nk[5] * NC], nu[5]);
    }
    return qf - qr;
}

// reaction_plain (chem_device.hpp) for a row the whole wave evaluates, as forward minus reverse rate of
// progress: the same operations, with the powers and flags
// of K->lane_plain taken as scalar branches instead of selects, the species rows read at byte offsets
// from this lane's column of the C and G blocks, and pfac**nus from the lane's PF column.
__device__ __forceinline__ double ipow_u(double x, int m) {      // ipow3 for a wave-uniform m; 0 only for x = 1
    if (m <= 1) return x;
    const double x2 = x * x;
    return m == 2 ? x2 : x * x2;
}

__device__ __forceinline__ double lane_plain_q(CLanePlain *L, CSeries *ks, const Temp &tp, bool usual,
                                               double small, double exparg, const char *Cb, int dG,
                                               const double *Pf) {
    // the whole record at once: one wait instead of one at each branch
    const int bits = L->bits;
    const double A = L->A, B = L->B, E = L->E;
    const double nud[6] = {L->nud[0], L->nud[1], L->nud[2], L->nud[3], L->nud[4], L->nud[5]};
    const int off[6] = {L->off[0], L->off[1], L->off[2], L->off[3], L->off[4], L->off[5]};
    if (bits & LP_DEAD) return 0.0;
    // concentrations and S/R - H/RT of the slots (G follows C at a constant distance); an empty slot reads the
    // row that changes nothing: coefficient 0, concentration 1
    double c[6], g[6];
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const char *at = Cb + off[n];
        c[n] = *reinterpret_cast<const double *>(at);
        g[n] = *reinterpret_cast<const double *>(at + dG);
    }
    double kf = A;
    if (!(bits & LP_ARR0)) kf = kf * exp_near(ks, B * tp.logT - over(E, tp, usual));
    double kr = 0.0;
    if (bits & LP_REV) {
        // reaction_plain starts from 0.0 + t0; the two differ at most in the sign of a zero sum,
        // which the test s != 0 and exp(+-0) = 1 do not see
        double s = nud[0] * g[0];
#pragma unroll
        for (int n = 1; n < 6; ++n) s = s + nud[n] * g[n];
        double eqk = exp_near(ks, fmin(s, exparg));      // (1 for s = 0)
        eqk = eqk * Pf[((bits >> LP_NUS) & 7) * NC];
        kr = kf / fmax(eqk, small);
    }
    if (bits & LP_POW) {
        const int pw = bits >> LP_PW;
#pragma unroll
        for (int n = 0; n < 6; ++n) c[n] = ipow_u(c[n], (pw >> (2 * n)) & 3);
    }
    const double qf = kf * c[0] * c[1] * c[2], qr = kr * c[3] * c[4] * c[5];
    return qf - qr;
}

// Species slots of wave w < NW: k = w + NW * j; the other waves have none (species_base: past the last).
__device__ __forceinline__ int species_base(int w) { return w < NW ? w : 1 << 20; }
template <int NSP>
constexpr int slots() { return (NSP + NW - 1) / NW; }

// Sum over the NW waves of one value per cell, in wave order, through a block of NW * NC doubles
// (the start of the rate block Q, free outside the reaction loop).
__device__ __forceinline__ double sum_waves(double *slot, int w, int cl, double v) {
    if (w < NW) slot[w * NC + cl] = v;
    __syncthreads();
    double s = slot[cl];
#pragma unroll
    for (int u = 1; u < NW; ++u) s = s + slot[u * NC + cl];
    __syncthreads();
    return s;
}

// The same for two values at once through a block of 2 * NW * NC doubles (the rate block Q, free
// outside the reaction loop): one pair of barriers instead of two.
__device__ __forceinline__ void sum_waves2(double *pair, int w, int cl, double va, double vb, double &ra, double &rb) {
    if (w < NW) {
        pair[w * NC + cl] = va;
        pair[(NW + w) * NC + cl] = vb;
    }
    __syncthreads();
    const double *q = pair + NW * NC;
    ra = pair[cl];
    rb = q[cl];
#pragma unroll
    for (int u = 1; u < NW; ++u) {
        ra = ra + pair[u * NC + cl];
        rb = rb + q[u * NC + cl];
    }
    __syncthreads();
}

// f = dy/dt at (y + s d, T) for this wave's species slots (f[j] of species w + NW*j) and fT for
// all waves (SHIFT = false: at y).  rho in g/cm^3.  cl: this lane's LDS column.
template <int NSP, bool SHIFT>
__device__ __forceinline__ void rhs_lane(CThermo *th, CKin *K, LaneShared<NSP> &sh,
                         int w, int cl, double rho, const double (&y)[slots<NSP>()],
                         const double (&d)[slots<NSP>()], double s, double T, double (&f)[slots<NSP>()],
                         double &fT) {
    constexpr int NS = slots<NSP>();
    const TPow p = tpow(T, th->ru);
    double uk[NS];
    double ctot_w = 0.0, cvm_w = 0.0;
    CSeries *ks = get_series();
    Temp tp = temperature(ks, T);
    // beyond any temperature of a state that can be accepted: NaN rates, the cell goes on to the integrator.
    // (Arguments of exp_near stay below 2^128 for activation temperatures below 2^121 K.)
    tp.logT = T >= 0x1p-7 && T <= 0x1p27 ? tp.logT : __builtin_nan("");
    const double lnT = tp.logT;
    const bool usual = K->usual != 0;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int k = species_base(w) + NW * j;
        uk[j] = 0.0;
        if (k < NSP) {
            const double yj = SHIFT ? y[j] + s * d[j] : y[j];
            const double ck = rho * yj / th->wt[k];
            sh.C[k * NC + cl] = ck;
            sh.W[k * NC + cl] = 0.0;
            ctot_w = ctot_w + ck;
            const Nasa a = nasa(th, k, T);
            uk[j] = h_mol(a, p) - p.rut;
            cvm_w = cvm_w + yj * (cp_mol(a, p) - th->ru) / th->wt[k];
            const double t2 = T * T, t3 = T * t2, t4 = t2 * t2;     // CKSMH, as smh_species
            double s = (lnT - 1.0) * a.a0;
            s = s + T / 2.0 * a.a1;
            s = s + t2 / 6.0 * a.a2;
            s = s + t3 / 12.0 * a.a3;
            s = s + t4 / 20.0 * a.a4;
            sh.G[k * NC + cl] = s + a.a6 - a.a5 / T;
        }
    }
    const double pfac = th->pa / (th->ru * T);
    {
        // pfac**m as reaction_plain forms it (x**3 = x * (x * x), x**-m = 1 / x**m); row m + 3 of PF,
        // row r written by wave r mod NW
        const double p2 = pfac * pfac, p3 = pfac * p2;
        const double pm[7] = {1.0 / p3, 1.0 / p2, 1.0 / pfac, 1.0, pfac, p2, p3};
#pragma unroll
        for (int r = 0; r < 7; ++r)
            if (r % NW == w) sh.PF[r * NC + cl] = pm[r];
    }
    static_assert(CH >= 2 * NW, "the rate block holds a pair of cross-wave sums");
    double ctot, cvm;
    sum_waves2(sh.Q, w, cl, ctot_w, cvm_w, ctot, cvm);     // its barrier also publishes C, G and PF
    const double *Cp = sh.C + cl, *Gp = sh.G + cl;
    const char *Cb = reinterpret_cast<const char *>(Cp);
    const int dG = int(reinterpret_cast<const char *>(sh.G) - reinterpret_cast<const char *>(sh.C));
    const double *Pf = sh.PF + cl;
    double *Wp = sh.W + cl;
    char *Wb = reinterpret_cast<char *>(Wp);
    const double *Qp = sh.Q + cl;
    const char *Qb = reinterpret_cast<const char *>(Qp);
    const int ii = K->ii, np0 = K->nplain0;
    const double small = K->small, exparg = K->exparg;
    for (int c0 = 0, chunk = 0; c0 < ii; c0 += CH, ++chunk) {
        // the chunk's rows, handed out one by one: the waves of a SIMD do not run at the same speed (the
        // oldest goes first), and the fall-off rows, the first ones, take five times as long
        const int n = min(CH, ii - c0);
        for (;;) {
            int r = 0;
            if ((threadIdx.x & 63) == 0) r = atomicAdd(&sh.next[chunk & 1], 1);
            r = __builtin_amdgcn_readfirstlane(r);
            if (r >= n) break;
            const int i = c0 + r;
            const double q = i >= np0 ? lane_plain_q(&K->lane_plain[i], ks, tp, usual, small, exparg, Cb, dG, Pf)
                                      : lane_row_q(K, ks, i, tp, usual, pfac, ctot, Cp, Gp);
            sh.Q[r * NC + cl] = q;
        }
        __syncthreads();
        if (threadIdx.x == 0) sh.next[chunk & 1] = 0;       // (used again two chunks on)
        // the chunk's contributions, species by species
        const int s1 = K->lane_seg0[chunk * RW + w + 1];
        for (int sg = K->lane_seg0[chunk * RW + w]; sg < s1; ++sg) {
            const int goff = K->lane_seg[sg].off, e0 = K->lane_seg[sg].e0, n = K->lane_seg[sg].n;
            double *wk = reinterpret_cast<double *>(Wb + goff);
            double s = *wk;
#pragma unroll 4
            for (int e = e0; e < e0 + n; ++e)
                s = s + *reinterpret_cast<const double *>(Qb + K->lane_ent[e].off) * K->lane_ent[e].nu;
            *wk = s;
        }
        __syncthreads();                   // Q is rewritten by the next chunk
    }
    double su_w = 0.0;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int k = species_base(w) + NW * j;
        f[j] = 0.0;
        if (k < NSP) {
            const double wd = Wp[k * NC];
            f[j] = wd * th->wt[k] / rho;
            su_w = su_w + uk[j] * wd;
        }
    }
    const double su = sum_waves(sh.Q, w, cl, su_w);     // after the last chunk's closing barrier
    fT = -su / (rho * cvm);
}

// Mixture e = sum Y u / W and cv (erg/g) over all species at T for this cell.
template <int NSP>
__device__ __forceinline__ void energy_lane(CThermo *th, double *pair, int w, int lane,
                            const double (&y)[slots<NSP>()], double T, double &e, double &cv) {
    constexpr int NS = slots<NSP>();
    const TPow p = tpow(T, th->ru);
    double eu = 0.0, ec = 0.0;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int k = species_base(w) + NW * j;
        if (k < NSP) {
            const Nasa a = nasa(th, k, T);
            eu = eu + y[j] * (h_mol(a, p) - p.rut) / th->wt[k];
            ec = ec + y[j] * (cp_mol(a, p) - th->ru) / th->wt[k];
        }
    }
    sum_waves2(pair, w, lane, eu, ec, e, cv);
}

// adjust_sum (SRC/thermo.f90:136-149) of this wave's slots: clip at 0, divide by the cell's sum.
template <int NSP>
__device__ __forceinline__ void adjust_lane(double *slot, int w, int lane, double (&y)[slots<NSP>()]) {
    constexpr int NS = slots<NSP>();
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        y[j] = (species_base(w) + NW * j < NSP) ? fmax(y[j], 0.0) : 0.0;
        s = s + y[j];
    }
    const double tot = sum_waves(slot, w, lane, s);
#pragma unroll
    for (int j = 0; j < NS; ++j) y[j] = y[j] / tot;
}

template <int NSP>
__global__ void __launch_bounds__(64 * RW) k_chem_screen(ChemArgs a) {
    constexpr int NS = slots<NSP>();
    __shared__ LaneShared<NSP> sh;
    // the wave index is uniform across the wave; saying so turns every table read indexed by it
    // (reactions i = w + NW n, species k = w + NW j) into a scalar load and every branch on the
    // reaction kind into a scalar branch
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = min(int(threadIdx.x & 63), NC - 1);   // the LDS column (lanes >= NC repeat NC - 1)
    CThermo *th = constant(a.thermo);
    CKin *K = (CKin *)a.kin;
    const int cell0 = int(xcd_block()) * NC;   // neighbouring cell ranges share their XCD's L2
    const int cell = cell0 + lane;
    // every lane of a column takes the column's decisions (lanes >= NC share column NC - 1 and must
    // write the same LDS values as its owner); only the owner lane stores to global memory
    const bool live = cell < a.ncells;
    const bool owner = live && int(threadIdx.x & 63) < NC;
    const int c = live ? cell : cell0;          // columns past the end shadow a live cell
    double *slot = sh.Q;
    // (barriers follow before the first rows)
    if (threadIdx.x < 2) sh.next[threadIdx.x] = 0;
    if (w == 0) {
        sh.C[NSP * NC + lane] = 1.0;
        sh.G[NSP * NC + lane] = 0.0;
    }

    long col = 0;
    double rho_si, dt, T0;
    double y[NS];
    if (a.layout == 0) {
        const int b = c / a.ncell, i = c % a.ncell;
        col = long(b) * a.S + a.lv + i;
        rho_si = a.qf[col];
        T0 = a.qf[2 * a.P + col];
        dt = a.dt_dev ? *a.dt_dev : a.dt;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            y[j] = k < NSP ? a.qf[(3 + k) * a.P + col] : 0.0;
        }
        adjust_lane<NSP>(slot, w, lane, y);
    } else {
        rho_si = a.b_rho[c];
        dt = a.b_dt[c];
        T0 = a.b_T[c];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            y[j] = k < NSP ? a.b_y[long(k) * a.ncells + c] : 0.0;
        }
    }
    const double rho = rho_si * 1.e-3;
    double e0, cv0;
    {
        double ya[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) ya[j] = y[j];
        adjust_lane<NSP>(slot, w, lane, ya);
        energy_lane<NSP>(th, sh.Q, w, lane, ya, T0, e0, cv0);
    }

    // ---- Heun over dt with the embedded Euler error estimate ----
    double f0[NS], f0T;
    rhs_lane<NSP, false>(th, K, sh, w, lane, rho, y, y, 0.0, T0, f0, f0T);
    const double T1 = T0 + dt * f0T;
    double f1[NS], f1T;
    rhs_lane<NSP, true>(th, K, sh, w, lane, rho, y, f0, dt, T1, f1, f1T);   // at y + dt f0
    double err_w = 0.0;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        if (species_base(w) + NW * j < NSP) {
            const double wt = 1.0 / (a.atol + a.rtol * fabs(y[j]));
            const double t = ((dt * 0.5) * (f1[j] - f0[j])) * wt;
            err_w = err_w + t * t;
        }
    }
    if (w == 0) {
        const double t = ((dt * 0.5) * (f1T - f0T)) * (1.0 / (a.rtol * fabs(T0)));
        err_w = err_w + t * t;
    }
    const double err = sqrt(sum_waves(slot, w, lane, err_w) / double(NSP + 1));
    const bool ok = live && err <= 1.0;

    if (!ok && owner && a.f0) {   // f at the start state, for the retry of a long list
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            if (k < NSP) a.f0[long(k) * a.ncells + cell] = f0[j];
        }
        if (w == 0) a.f0[long(NSP) * a.ncells + cell] = f0T;
    }
    if (!ok) {
        if (owner && w == 0) {
            const unsigned long long bal = __ballot(1);
            const int leader = __ffsll((long long)bal) - 1;
            const int rank = __popcll(bal & ((1ull << lane) - 1ull));
            unsigned base = 0;
            if (lane == leader) base = atomicAdd(a.stiff_n, unsigned(__popcll(bal)));
            base = __shfl(base, leader, 64);
            a.stiff[base + rank] = cell;
            if (a.route) a.route[cell] = 0;
        }
    }
    // ---- accepted cells: state update and energy-consistent temperature ----
#pragma unroll
    for (int j = 0; j < NS; ++j) y[j] = y[j] + (dt * 0.5) * (f0[j] + f1[j]);
    double T = T0 + (dt * 0.5) * (f0T + f1T);
    adjust_lane<NSP>(slot, w, lane, y);
    bool done = !ok;
    for (int it = 0; it < 20; ++it) {
        if (!__syncthreads_or(done ? 0 : 1)) break;
        double ek, cvk;
        energy_lane<NSP>(th, sh.Q, w, lane, y, T, ek, cvk);
        if (!done) {
            const double d = (e0 - ek) / cvk;
            T = T + d;
            if (fabs(d) <= 1.0e-12 * T) done = true;
        }
    }
    double hrr_s = 0.0, hrr_d = 0.0;
    if (a.hrr) {
        // heat_release_rate (SRC/thermo.f90:98-101) and heat_release_rate_omegadot
        // (SRC/thermo.f90:128-132): the creation minus destruction rates of CKCDYR are the net
        // production rates, evaluated at the new state.
        double fn[NS], fnT;
        rhs_lane<NSP, false>(th, K, sh, w, lane, rho, y, y, 0.0, T, fn, fnT);
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            if (k < NSP) {
                const double y_in = a.layout == 0 ? a.qf[(3 + k) * a.P + col] : a.b_y[long(k) * a.ncells + c];
                s1 = s1 + rho * th->h298[k] * (y[j] - y_in) / dt;
                s2 = s2 + th->h298[k] * fn[j] * rho;     // W_k h_k wdot_k = h_k (W_k wdot_k / rho) rho
            }
        }
        sum_waves2(sh.Q, w, lane, s1, s2, hrr_s, hrr_d);
    }
    if (!ok || !owner) return;
    if (a.layout == 0) {
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            if (k < NSP) a.qf[(3 + k) * a.P + col] = y[j];
        }
        if (w == 0) {
            a.qf[2 * a.P + col] = T;
            if (a.hrr) {
                a.hrr[cell] = -hrr_s * 1.e-1;
                a.hrr_dot[cell] = -hrr_d * 1.e-1;
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            if (k < NSP) a.b_y[long(k) * a.ncells + cell] = y[j];
        }
        if (w == 0) a.b_T[cell] = T;
    }
    if (w == 0) {
        if (a.stats) a.stats[cell] = ChemCellStats{1, 0, 0, 0};
        if (a.route) a.route[cell] = 2;
        if (a.hmem) a.hmem[cell] = 0.0;
    }
}

// Explicit retry of a LONG stiff list, ONE CELL PER LANE like k_chem_screen: two Heun steps of dt/2,
// each accepted by its own embedded Euler estimate with weights at its start -- the retry k_chem
// makes before its implicit steps, with the same formulas.  In: cells a.list[0 .. *a.list_n), and
// (when a.f0 is given) f at their start states, which the screen computed at the same states.
// Accepted cells are final (state, heat release, stats {2, 0, 0, 0}, step-size memory 0); the
// others go to a.stiff (*a.stiff_n zero before the launch) for the implicit integrator, which
// *a.retry_done = 1 tells to skip its own retry.  A list of at most a.coop_max cells is copied to
// a.stiff unchanged with *a.retry_done = 0: the integrator then runs it several waves per cell and
// retries each cell itself.  Domain layout only.
template <int NSP>
__global__ void __launch_bounds__(64 * RW) k_chem_retry(ChemArgs a) {
    constexpr int NS = slots<NSP>();
    __shared__ LaneShared<NSP> sh;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = min(int(threadIdx.x & 63), NC - 1);   // the LDS column (lanes >= NC repeat NC - 1)
    CThermo *th = constant(a.thermo);
    CKin *K = (CKin *)a.kin;
    const int n = int(*a.list_n);
    if (coop_list(a, n)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *a.retry_done = 0;
            *a.stiff_n = unsigned(n);
        }
        for (int i = int(blockIdx.x) * (64 * RW) + int(threadIdx.x); i < n; i += int(gridDim.x) * (64 * RW)) a.stiff[i] = a.list[i];
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.retry_done = 1;
    const int item0 = int(blockIdx.x) * NC;
    if (item0 >= n) return;                     // the whole workgroup: no barrier is skipped
    const int item = item0 + lane;
    // every lane of a column takes the column's decisions (lanes >= NC share column NC - 1); only the
    // owner lane stores to global memory
    const bool live = item < n;
    const bool owner = live && int(threadIdx.x & 63) < NC;
    const int cell = a.list[live ? item : item0];   // columns past the end shadow a live cell
    double *slot = sh.Q;
    // (barriers follow before the first rows)
    if (threadIdx.x < 2) sh.next[threadIdx.x] = 0;
    if (w == 0) {
        sh.C[NSP * NC + lane] = 1.0;
        sh.G[NSP * NC + lane] = 0.0;
    }

    const int b = cell / a.ncell, i = cell % a.ncell;
    const long col = long(b) * a.S + a.lv + i;
    const double rho_si = a.qf[col];
    const double T0 = a.qf[2 * a.P + col];
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    double y[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int k = species_base(w) + NW * j;
        y[j] = k < NSP ? a.qf[(3 + k) * a.P + col] : 0.0;
    }
    adjust_lane<NSP>(slot, w, lane, y);
    const double rho = rho_si * 1.e-3;
    double e0, cv0;
    {
        double ya[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) ya[j] = y[j];
        adjust_lane<NSP>(slot, w, lane, ya);
        energy_lane<NSP>(th, sh.Q, w, lane, ya, T0, e0, cv0);
    }

    // ---- two Heun steps of dt/2; a lane keeps going only while its half steps are accepted ----
    const double hs = dt * 0.5;
    double Th = T0;
    bool ok = live;
    for (int sub = 0; sub < 2; ++sub) {
        double fa[NS], faT, fb[NS], fbT;
        if (sub == 0 && a.f0) {   // f at the start state, stored by the screen
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                const int k = species_base(w) + NW * j;
                fa[j] = k < NSP ? a.f0[long(k) * a.ncells + cell] : 0.0;
            }
            faT = a.f0[long(NSP) * a.ncells + cell];
        } else {
            rhs_lane<NSP, false>(th, K, sh, w, lane, rho, y, y, 0.0, Th, fa, faT);
        }
        rhs_lane<NSP, true>(th, K, sh, w, lane, rho, y, fa, hs, Th + hs * faT, fb, fbT);   // at y + hs fa
        double err_w = 0.0;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            if (species_base(w) + NW * j < NSP) {
                const double wt = 1.0 / (a.atol + a.rtol * fabs(y[j]));
                const double t = ((hs * 0.5) * (fb[j] - fa[j])) * wt;
                err_w = err_w + t * t;
            }
        }
        if (w == 0) {
            const double t = ((hs * 0.5) * (fbT - faT)) * (1.0 / (a.rtol * fabs(Th)));
            err_w = err_w + t * t;
        }
        const double err = sqrt(sum_waves(slot, w, lane, err_w) / double(NSP + 1));
        ok = ok && err <= 1.0;
        if (ok) {
#pragma unroll
            for (int j = 0; j < NS; ++j) y[j] = y[j] + (hs * 0.5) * (fa[j] + fb[j]);
            Th = Th + (hs * 0.5) * (faT + fbT);
        }
        // no lane of the workgroup passed the first half step: the second would be wasted work.
        // ok is the same in all waves of a lane (err comes from sum_waves), and every wave reaches
        // this barrier, so the exit is uniform
        if (sub == 0 && !__syncthreads_or(ok ? 1 : 0)) break;
    }
    if (!ok) {
        if (owner && w == 0) {
            const unsigned long long bal = __ballot(1);
            const int leader = __ffsll((long long)bal) - 1;
            const int rank = __popcll(bal & ((1ull << lane) - 1ull));
            unsigned base = 0;
            if (lane == leader) base = atomicAdd(a.stiff_n, unsigned(__popcll(bal)));
            base = __shfl(base, leader, 64);
            a.stiff[base + rank] = cell;
        }
    }
    // ---- accepted cells: energy-consistent temperature ----
    adjust_lane<NSP>(slot, w, lane, y);
    double T = Th;
    bool done = !ok;
    for (int it = 0; it < 20; ++it) {
        if (!__syncthreads_or(done ? 0 : 1)) break;
        double ek, cvk;
        energy_lane<NSP>(th, sh.Q, w, lane, y, T, ek, cvk);
        if (!done) {
            const double d = (e0 - ek) / cvk;
            T = T + d;
            if (fabs(d) <= 1.0e-12 * T) done = true;
        }
    }
    double hrr_s = 0.0, hrr_d = 0.0;
    if (a.hrr) {
        // heat_release_rate and heat_release_rate_omegadot (SRC/thermo.f90:98-101, 128-132), as
        // in k_chem_screen
        double fn[NS], fnT;
        rhs_lane<NSP, false>(th, K, sh, w, lane, rho, y, y, 0.0, T, fn, fnT);
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const int k = species_base(w) + NW * j;
            if (k < NSP) {
                const double y_in = a.qf[(3 + k) * a.P + col];
                s1 = s1 + rho * th->h298[k] * (y[j] - y_in) / dt;
                s2 = s2 + th->h298[k] * fn[j] * rho;
            }
        }
        sum_waves2(sh.Q, w, lane, s1, s2, hrr_s, hrr_d);
    }
    if (!ok || !owner) return;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int k = species_base(w) + NW * j;
        if (k < NSP) a.qf[(3 + k) * a.P + col] = y[j];
    }
    if (w == 0) {
        a.qf[2 * a.P + col] = T;
        if (a.hrr) {
            a.hrr[cell] = -hrr_s * 1.e-1;
            a.hrr_dot[cell] = -hrr_d * 1.e-1;
        }
        if (a.stats) a.stats[cell] = ChemCellStats{2, 0, 0, 0};
        if (a.route) a.route[cell] = 3;
        if (a.hmem) a.hmem[cell] = 0.0;
    }
}

}  // namespace

hipError_t launch_chem_retry(const ChemArgs &a, int nsp, hipStream_t st) {
    const unsigned nb = unsigned((a.ncells + NC - 1) / NC);
    if (nb == 0) return hipSuccess;
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_chem_retry<N>), dim3(nb), dim3(64 * RW), 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_chem_screen(const ChemArgs &a, int nsp, hipStream_t st) {
    const unsigned nb = unsigned((a.ncells + NC - 1) / NC);
    if (nb == 0) return hipSuccess;
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_chem_screen<N>), dim3(nb), dim3(64 * RW), 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

}  // namespace fcfd
