// chem_coop.hip -- the stiff integrator for short work lists: ONE CELL PER EIGHT-WAVE WORKGROUP.
//
// The method is the one-wave kernel's (chem.hip).  A launch over a short list lasts as long as its
// slowest cells' chain of steps, so here a cell's work is split by kind over the waves, and only what
// the method makes sequential stays sequential:
//   wave 0      runs the integrator (stages, Newton, norms, triangular solves, step control) and the
//               species part of a rate evaluation; it posts commands to the other waves through LDS;
//   waves 1..6  evaluate 64 reaction rows each, one row per lane (one row's chain of an exponential, a
//               logarithm and divisions is what an evaluation cannot be shorter than);
//   wave 7      evaluates the fall-off rows' terms that depend on temperature alone.
// A rate evaluation has three barriers: concentrations and temperature terms | rates of progress |
// sums per species.  The sums (production rates, Jacobian entries) gather the rates of progress from
// LDS by precomputed lists instead of scattering them with LDS atomics, whose conflicts serialised.
// The lists hold each sum's terms in the order in which a four-wave scatter added them (four
// partial sums: rows 0..63, then every third block of 64 rows; within a block by slot, then by row), so
// every sum is the same bits as there.  The Newton matrix is factored in registers, seven columns a
// wave, a panel at a time.  80 kB of LDS and 128 registers: two workgroups per CU.
//
// What bounds it: the latency of one cell's chain.  Cycles of the slowest part per event, GRI-3.0 (53
// species, 325 rows): rate evaluation 13.6k (temperature terms 2.3k, fall-off rows 4.3k, sums 3.6k,
// species 1k), substitutions of a Newton iteration 4.2k, Jacobian with its temperature column 33k, LU
// about 38k; some seven Newton iterations an attempt.  Four waves that each evaluated blocks of rows,
// scattered into their own partial sums and Jacobian (155 kB of LDS, one workgroup per CU) and ran the
// integrator redundantly took 18.8k, 6.3k, 67k and 58k.  256 cells of the chemistry batch: 111 -> 62
// ms; 3,000 cells, which two workgroups per CU serve: 375 -> 137 ms; 200 H2/O2 cells: 24.5 -> 12.4 ms.  (That
// kernel, k_chem<NSP, 4>, still takes the mechanisms that the tables here do not hold.)
#include <algorithm>

#include "chem_wave.hpp"
#include "rate_math.hpp"

namespace fcfd {

namespace {

constexpr int CW = COOP_WAVES;

constexpr int FR = COOP_AT(3) + COOP_Q;      // split: the reverse rates behind the forward ones

enum { CMD_RHS, CMD_SPLIT, CMD_JAC, CMD_LU, CMD_EXIT };

template <int NSP>
struct Cell {
    static constexpr int N = NSP + 1;
    static constexpr int NCW = (N + CW - 1) / CW;                 // matrix columns per wave
    static constexpr int NP = NCW * CW;                           // matrix order, padded by the identity
    static constexpr int LDF = NP | 1;                            // odd: rows of one column in different banks
    static constexpr int max3(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }
    static constexpr int FW = max3((NP + 1) * LDF, 6 * COOP_MAXR + 1, 2 * COOP_AT(3) + 2 * COOP_Q);
    double F[FW];               // LU factors; while rates are evaluated the rates of progress' derivatives
                                // [slot][COOP_MAXR], or the forward and reverse rates (each as in q)
    double J[NSP * NSP];        // concentration Jacobian d(wdot_r) / d(c_k), unscaled
    double trow[64], tcol[64];  // temperature row and column of df/dy
    double tsum[64];            // sum_j u_j J_jk
    double S[8][64];            // partial sums per species (split: creation, then destruction)
    double c[64], smh[64], u[64];
    double q[max3(2 * NCW * 64 + COOP_Q, COOP_AT(3) + COOP_Q, 0)];      // rates: the net rates of progress
                                // (COOP_AT) with the fall-off terms [2][COOP_FAL] after the first COOP_Q;
                                // LU: there the multipliers of the last two panels
    double z[64];               // state of a rate evaluation: Y, T
    double lo[7][64], hi[7][64], wt[64], rwt[64], tmid[64];   // thermo tables, species per lane
    unsigned long long list[COOP_LIST / 4];                   // DevKin::coop_sum
    double rho, ctot, hg;
    int perm[64];
    int cmd, lu_ok;
};

#define FCFD_LDS __attribute__((address_space(3)))
#define FCFD_GLB __attribute__((address_space(1)))

// The SRI fall-off factor
__device__ __forceinline__ double sri_factor(double a, double b, double c, double d, double e, double prlog,
                                                       double T) {
    const double xp = 1.0 / (1.0 + prlog * prlog);
    return fm_pow(a * fm_exp(-b / T) + fm_exp(-T / c), xp) * d * fm_pow(T, e);
}

// Table values that stay in registers while the kernel runs.
struct Consts {
    int ii, nfal;
    double small, exparg, pa, ru;
};
// A lane's own: in waves 1 .. 6 its reaction row (DevKin::coop_row; A, B, E), in wave 7 its fall-off row's
// form and parameters; in waves 1 .. 4 its species' list of the sums (entries in fours; mx: the longest of
// the wave).
struct Own {
    unsigned w[4];
    double v[5];
    int off, len, mx;
};

// The block of 64 rows of waves 1 .. 6.  Waves w and w + 4 share a SIMD: block 0, which holds the fall-off
// rows, goes to wave 3, whose partner has no rows.
__device__ __forceinline__ int row_block(int w) { return w == 3 ? 0 : (w < 3 ? w : w - 1); }

__device__ __forceinline__ Own load_own(const DevKin *__restrict__ K, const Consts &cs, int w) {
    const int lane = lane_id();
    Own o{};
    if (w < 7) {
        const int i = min(row_block(w) * 64 + lane, cs.ii - 1);
#pragma unroll
        for (int n = 0; n < 4; ++n) o.w[n] = K->coop_row[n][i];
        o.v[0] = K->A[i];
        o.v[1] = K->B[i];
        o.v[2] = K->E[i];
    } else if (cs.nfal > 0) {
        const int f = min(lane & 31, cs.nfal - 1);
        const double *fp = K->fpar[f];
        o.w[0] = unsigned(K->ifop[f]);
        o.v[0] = fp[1];
        o.v[1] = fp[2];
        o.v[2] = fp[3];
        o.v[3] = fp[lane < 32 ? 4 : 5];
        o.v[4] = fp[6];
    }
    if (w <= 4) {
        o.off = K->sum_off[w - 1][lane] / 4;
        o.len = K->sum_len[w - 1][lane] / 4;
        o.mx = int(wave_max_u32(unsigned(o.len)));
    }
    return o;
}

// What a row has before the concentrations are known: the Arrhenius factor, (pa / RT) ** (coefficient
// sum), the entries of the third-body and fall-off tables.
struct Row {
    double kf, pn;
    unsigned tk[COOP_TB / 4];
    double ta[COOP_TB];
    double f0;
    int ifop, kfal;
};

__device__ __forceinline__ Row row_begin(const DevKin *__restrict__ K, const Consts &cs, const Own &own, CSeries *k, int i, const Temp &tp) {
    Row o;
    if (__any(own.w[3] != 0)) {
        const int f = int(own.w[3] >> 16), ff = f > 0 ? f - 1 : 0;
#pragma unroll
        for (int u = 0; u < COOP_TB / 4; ++u) o.tk[u] = K->coop_tbk[u][i];
#pragma unroll
        for (int u = 0; u < COOP_TB; ++u) o.ta[u] = K->coop_tba[u][i];
        o.f0 = K->fpar[ff][0];
        o.ifop = K->ifop[ff];
        o.kfal = K->kfal[ff];
    }
    const double ek = exp_rate(k, own.v[1] * tp.logT - over(own.v[2], tp));
    o.kf = (own.w[2] & CR_ARR0) ? own.v[0] : own.v[0] * ek;
    const int ns = int((own.w[2] >> CR_NUS) & 7u) - 3;
    const double pp = pow3(cs.pa / (cs.ru * tp.T), ns < 0 ? -ns : ns);
    o.pn = ns < 0 ? 1.0 / pp : pp;
    return o;
}

// Rates of progress of row i (CKRATT + CKRATX, as reaction()), into sh.q; CMD_JAC: their derivatives by
// the slots' concentrations into sh.F; CMD_SPLIT: the forward and reverse rates into sh.F.  An empty slot's
// concentration is 1 and its coefficient 0, so its factors and terms change no bit.
template <int NSP>
__device__ __forceinline__ void row_end(const DevKin *__restrict__ K, Cell<NSP> &sh, const Consts &cs, const Own &own,
                                        CSeries *k, const Row &r, int i, double T, int cmd) {
    const bool any_tb = __any(own.w[3] != 0), any_pow = __any((own.w[2] & CR_POW) != 0);
    double x[6], h[6], an[6];
    int m[6];
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const int sp = int((own.w[n / 4] >> (8 * (n % 4))) & 255u);
        h[n] = sh.smh[sp];
        x[n] = sh.c[sp];
    }
    double tc[COOP_TB], low = 0.0, fcl = 0.0, cm = 0.0, ctot = 0.0;
    const int f = int(own.w[3] >> 16) - 1;
    if (any_tb) {
        ctot = sh.ctot;
#pragma unroll
        for (int u = 0; u < COOP_TB; ++u) tc[u] = sh.c[(r.tk[u / 4] >> (8 * (u % 4))) & 255u];
        low = sh.q[COOP_Q + max(f, 0)];
        fcl = sh.q[COOP_Q + COOP_FAL + max(f, 0)];
        cm = sh.c[max(r.kfal, 0)];
    }
    __builtin_amdgcn_sched_barrier(0);          // (all LDS reads are on their way)
    double s = 0.0;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const int nu = int(own.w[2] << (20 - 4 * n)) >> 28;
        s = s + double(nu) * h[n];
        m[n] = n < 3 ? -nu : nu;
        an[n] = double(m[n] < 0 ? -m[n] : m[n]);
    }
    double kf = r.kf;
    double eqk = exp_rate(k, fmin(s, cs.exparg));
    eqk = (s != 0.0 ? eqk : 1.0) * r.pn;
    double kr = (own.w[2] & CR_REV) ? kf / fmax(eqk, cs.small) : 0.0;
    if (any_tb) {
        double ctb = ctot;
#pragma unroll
        for (int u = 0; u < COOP_TB; ++u) ctb = ctb + r.ta[u] * tc[u];
        ctb = (own.w[3] & 0xffffu) ? ctb : 1.0;
        if (f >= 0) {
            double pr;
            const double cb = r.kfal < 0 ? ctb : cm;
            pr = r.f0 * low * cb / kf;
            ctb = r.kfal < 0 ? 1.0 : ctb;
            double pcor = pr / (1.0 + pr);
            if (r.ifop > 1) {
                const double prlog = log10_rate(k, fmax(pr, cs.small));
                double fc;
                if (__builtin_expect(r.ifop == 2, 0)) {
                    const double *fp = K->fpar[f];
                    fc = sri_factor(fp[3], fp[4], fp[5], fp[6], fp[7], prlog, T);
                } else {
                    // single-precision literals of cklib.f:6915-6917
                    const double xn = 0.75 - (double)1.27f * fcl;
                    const double cprlog = prlog - ((double)0.4f + (double)0.67f * fcl);
                    const double q = cprlog / (xn - (double)0.14f * cprlog);
                    fc = exp10_rate(k, fcl / (1.0 + q * q));
                }
                pcor = fc * pcor;
            }
            kf = kf * pcor;
            kr = kr * pcor;
        }
        kf = kf * ctb * 1.0;
        kr = kr * ctb * 1.0;
    }
    double pw[6];
#pragma unroll
    for (int n = 0; n < 6; ++n) pw[n] = x[n];
    if (any_pow)
#pragma unroll
        for (int n = 0; n < 6; ++n) pw[n] = pow3(x[n], m[n] < 0 ? -m[n] : m[n]);
    const bool live = m[0] != 0;
    double qf = kf * pw[0] * pw[1] * pw[2];
    double qr = kr * pw[3] * pw[4] * pw[5];
    qf = live ? qf : 0.0;
    qr = live ? qr : 0.0;
    if (i >= cs.ii) return;
    auto store = [&](double *at, double v) {
        at[i] = v;
        if (any_pow) {
            at[COOP_AT(2) + i] = 2.0 * v;
            at[COOP_AT(3) + i] = 3.0 * v;
        }
    };
    store(sh.q, qf - qr);
    if (cmd == CMD_SPLIT) {
        store(sh.F, qf);
        store(sh.F + FR, qr);
    }
    if (cmd != CMD_JAC) return;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const int lo = n < 3 ? 0 : 3;
        double d = an[n];
        if (any_pow) d = an[n] * pow3(x[n], (m[n] < 0 ? -m[n] : m[n]) - 1);
#pragma unroll
        for (int o = lo; o < lo + 3; ++o)
            if (o != n) d = d * pw[o];
        sh.F[n * COOP_MAXR + i] = n < 3 ? kf * d : -(kr * d);
    }
}

// The fall-off terms that depend on temperature alone, into sh.q (wave 7): two lanes a row, which share
// its four exponentials.
template <int NSP>
__device__ __forceinline__ void falloff_terms(Cell<NSP> &sh, const Consts &cs, const Own &own, CSeries *k, int lane, const Temp &tp) {
    const bool half = lane >= 32;
    const double ea = exp_rate(k, -tp.T / own.v[3]);
    const double eb = exp_rate(k, half ? -over(own.v[4], tp) : own.v[0] * tp.logT - over(own.v[1], tp));
    const double e5 = __shfl_xor(ea, 32, 64), e6 = __shfl_xor(eb, 32, 64);
    double fcent = (1.0 - own.v[2]) * ea + own.v[2] * e5;
    fcent = own.w[0] == 4 ? fcent + e6 : fcent;
    const double lf = log10_rate(k, fmax(fcent, cs.small));
    if (lane < cs.nfal) {               // (at most COOP_FAL)
        sh.q[COOP_Q + lane] = eb;
        sh.q[COOP_Q + COOP_FAL + lane] = lf;
    }
}

// A sum over a list of terms (DevKin::coop_sum; SPLIT: coop_split, product slots' rates in base1).  len: this
// lane's entries in fours; mx: the wave's largest.  Eight terms at a time, the next eight's entries and
// rates on their way meanwhile.
template <bool SPLIT, class List>
__device__ __forceinline__ double list_sum(List *e, int len, int mx, const double *base0, const double *base1) {
    constexpr unsigned long long pad = (unsigned long long)(COOP_MAXR << 3) * 0x0001000100010001ULL;
    auto rate = [&](unsigned long long v, int u) {
        const unsigned x = unsigned(v >> (32 * (u / 2))) >> (16 * (u % 2));
        const char *b = reinterpret_cast<const char *>(SPLIT && (x & 0x8000u) ? base1 : base0);
        return *reinterpret_cast<const double *>(b + (x & 0x7ff8u));
    };
    auto term = [](double q, unsigned long long v, int u) {
        if (SPLIT) return q;
        const unsigned x = unsigned(v >> (32 * (u / 2))) << (u % 2 ? 0 : 16);
        return __hiloint2double(__double2hiint(q) ^ int(x & 0x80000000u), __double2loint(q));
    };
    auto entry = [&](int l) { return l < len ? e[l] : pad; };
    unsigned long long a0 = entry(0), a1 = entry(1), b0 = entry(2), b1 = entry(3);
    double q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) q[u] = rate(u < 4 ? a0 : a1, u % 4);
    double s = 0.0;
    for (int l = 0; l < mx; l += 2) {
        double n[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) n[u] = rate(u < 4 ? b0 : b1, u % 4);
        const unsigned long long c0 = entry(l + 4), c1 = entry(l + 5);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u) s = s + term(q[u], u < 4 ? a0 : a1, u % 4);
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = n[u];
        a0 = b0;
        a1 = b1;
        b0 = c0;
        b1 = c1;
    }
    return s;
}

using Uint4 = unsigned __attribute__((ext_vector_type(4)));

// This wave's share of the Jacobian entries (DevKin::coop_jac).
template <int NSP>
__device__ __forceinline__ void jac_gather(const DevKin *__restrict__ K, Cell<NSP> &sh, int lane, int w) {
    const int steps = __builtin_amdgcn_readfirstlane(K->jac_steps[w]);
    // (a pointer read from memory: said to be global, else the loads are flat and wait for LDS as well)
    auto *e = (FCFD_GLB const Uint4 *)(K->coop_jac + K->jac_off[w]) + 2 * lane;
    const unsigned char *end = K->jac_end[w];
    const char *base = reinterpret_cast<const char *>(sh.F);
    // the steps' words come two iterations ahead
    auto load = [&](int l, Uint4 &a, Uint4 &b, unsigned &m) {
        const int lc = min(l, steps - 8);
        a = e[lc * 16];
        b = e[lc * 16 + 1];
        m = end[lc / 8];
    };
    Uint4 a0, b0, a1, b1;
    unsigned m0, m1;
    load(0, a0, b0, m0);
    load(8, a1, b1, m1);
    double s = 0.0;
    for (int l = 0; l < steps; l += 8) {
        Uint4 a2, b2;
        unsigned m2;
        load(l + 16, a2, b2, m2);
        const unsigned v[8] = {a0.x, a0.y, a0.z, a0.w, b0.x, b0.y, b0.z, b0.w};
        double d[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) d[u] = *reinterpret_cast<const double *>(base + (v[u] & 0x7ff8u));
        __builtin_amdgcn_sched_barrier(0);
        const unsigned bits = __builtin_amdgcn_readfirstlane(m0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (bits >> u & 1u) {
                const double tot = s + dpp_f64<0x55>(s) + dpp_f64<0xAA>(s) + dpp_f64<0xFF>(s);
                if ((lane & 3) == 0 && v[u] != JE_NONE) sh.J[v[u]] = tot;
                s = 0.0;
            } else {
                s = s + __hiloint2double(int(v[u] & 0xffff0000u), 0) * d[u];
            }
        }
        a0 = a1;
        b0 = b1;
        m0 = m1;
        a1 = a2;
        b1 = b2;
        m1 = m2;
    }
}

struct Rates {
    double f;         // this lane's component of dy/dt
    double cvm, cvk;  // mixture cv (erg/(g K)), this lane's species cv (erg/(mol K))
    double cd, dd;    // split: this lane's creation / destruction rate
};

// f = dy/dt at the state sh.z (Y, T) and density sh.rho: wave 0's part, three barriers.
template <int NSP>
__device__ __attribute__((noinline)) Rates rates(FCFD_GLB const DevThermo *th1, FCFD_GLB const DevKin *K1,
                                                 FCFD_LDS Cell<NSP> *shl, int cmd1) {
    const int cmd = __builtin_amdgcn_readfirstlane(cmd1);
    const DevThermo *__restrict__ th = (const DevThermo *)th1;
    const DevKin *__restrict__ K = (const DevKin *)K1;
    Cell<NSP> &sh = *(Cell<NSP> *)shl;
    const int lane = lane_id();
    const double rho = sh.rho, T = sh.z[NSP];
    Rates o{0.0, 0.0, 0.0, 0.0, 0.0};
    const bool up = T > sh.tmid[lane];
    const double wt = sh.wt[lane], rw = sh.rwt[lane];
    const double y = lane < NSP ? sh.z[lane] : 0.0;
    Nasa a;
    a.a0 = up ? sh.hi[0][lane] : sh.lo[0][lane];
    a.a1 = up ? sh.hi[1][lane] : sh.lo[1][lane];
    a.a2 = up ? sh.hi[2][lane] : sh.lo[2][lane];
    a.a3 = up ? sh.hi[3][lane] : sh.lo[3][lane];
    a.a4 = up ? sh.hi[4][lane] : sh.lo[4][lane];
    a.a5 = up ? sh.hi[5][lane] : sh.lo[5][lane];
    a.a6 = up ? sh.hi[6][lane] : sh.lo[6][lane];
    const Temp tp = temperature(get_series(), T);
    const double ry = rho * y;
    // every divisor's reciprocal, where all numerators allow it
    const bool fast = __builtin_amdgcn_ballot_w64(tp.usual && num_ok(ry) && num_ok(a.a5)) == ~0ull;
    const double t2 = T * T, t3 = T * t2, t4 = t2 * t2;
    double ck, smh;
    if (__builtin_expect(fast, 1)) {
        ck = quot(ry, wt, rw);
        smh = (tp.logT - 1.0) * a.a0;
        smh = smh + T * 0.5 * a.a1;
        smh = smh + quot(t2, 6.0, 1.0 / 6.0) * a.a2;
        smh = smh + quot(t3, 12.0, 1.0 / 12.0) * a.a3;
        smh = smh + quot(t4, 20.0, 1.0 / 20.0) * a.a4;
        smh = smh + a.a6 - quot(a.a5, T, tp.rT);
    } else {
        ck = ry / wt;
        smh = smh_species(a, T);
    }
    if (lane < NSP) {
        sh.c[lane] = ck;
        sh.smh[lane] = smh;
    }
    const double ct = wsum(ck);
    if (lane == 0) sh.ctot = ct;
    __syncthreads();
    const double ru = th->ru;
    double uk;
    {
        const TPow p = tpow(T, ru);
        uk = h_mol(a, p) - p.rut;
        o.cvk = cp_mol(a, p) - ru;
    }
    sh.u[lane] = uk;
    o.cvm = wsum(lane < NSP ? y * o.cvk / wt : 0.0);
    __syncthreads();
    if (cmd == CMD_JAC) jac_gather(K, sh, lane, 0);
    __syncthreads();
    double wdot = 0.0;
    if (cmd == CMD_SPLIT) {
        o.cd = sh.S[0][lane];
        o.dd = sh.S[4][lane];
#pragma unroll
        for (int g = 1; g < 4; ++g) {
            o.cd = o.cd + sh.S[g][lane];
            o.dd = o.dd + sh.S[4 + g][lane];
        }
    } else {
        wdot = sh.S[0][lane];
#pragma unroll
        for (int g = 1; g < 4; ++g) wdot = wdot + sh.S[g][lane];
    }
    const double su = wsum(lane < NSP ? uk * wdot : 0.0);
    o.f = lane < NSP ? wdot * wt / rho : (lane == NSP ? -su / (rho * o.cvm) : 0.0);
    return o;
}

// LU with partial pivoting of M = I - hg*J in the waves' registers: wave w holds columns w*NCW ..
// w*NCW + NCW - 1 of every row (lane r: row r).  Panel w: wave w factors its own columns without a
// barrier -- pivot (the open row with the largest entry, the lower row on ties), multipliers l = rk /
// piv, fma(-l, u_j, m_j) on its columns to the right -- and publishes multipliers and pivot rows; after
// one barrier the waves right of it apply its steps to their columns in order.  Every entry sees the
// operations of an elimination step by step, so the factors do not depend on the split.  They go to
// sh.F (rows unswapped, sh.perm[k] the pivot row of step k).  The multipliers alternate between two
// buffers: wave w + 2 overwrites panel w's after the barrier of panel w + 1, which every wave passes
// after applying panel w.
template <int NSP>
__device__ __forceinline__ void factor(Cell<NSP> &sh, int lane, int w) {
    constexpr int N = Cell<NSP>::N, NCW = Cell<NSP>::NCW, NP = Cell<NSP>::NP, LDF = Cell<NSP>::LDF;
    static_assert(NP <= 64, "one row per lane");
    const double hg = sh.hg;
    const int j0 = w * NCW;
    double col[NCW];
    {
        const double wr = lane < NSP ? sh.wt[lane] : 1.0;
        const int rl = min(lane, NSP - 1);
        double v[NCW];
        bool in = true;
#pragma unroll
        for (int jj = 0; jj < NCW; ++jj) {
            v[jj] = sh.J[rl * NSP + min(j0 + jj, NSP - 1)] * wr;
            const unsigned hi = (unsigned)__double2hiint(v[jj]) & 0x7fffffffu;
            in = in & ((hi - 0x14000000u < 0x3f000000u) | (v[jj] == 0.0));      // 2^-703 .. 2^305
        }
        in = __all(in);
        if (in) {
#pragma unroll
            for (int jj = 0; jj < NCW; ++jj) {
                const int jc = min(j0 + jj, NSP - 1);
                v[jj] = quot(v[jj], sh.wt[jc], sh.rwt[jc]);
            }
        } else {
#pragma unroll 1
            for (int jj = 0; jj < NCW; ++jj) {
                const int jc = min(j0 + jj, NSP - 1);
                v[0] = v[0] / sh.wt[jc];
#pragma unroll
                for (int n = 0; n < NCW; ++n) {      // (rotates: each column once through the one division)
                    const double t = v[n];
                    v[n] = n + 1 < NCW ? v[n + 1] : v[n];
                    if (n == 0) col[0] = t;
                }
                v[NCW - 1] = col[0];
            }
        }
        const double tc = sh.tcol[lane];
#pragma unroll
        for (int jj = 0; jj < NCW; ++jj) {
            const int j = j0 + jj;
            const double tr = sh.trow[min(j, NSP - 1)];
            double u = lane == NSP ? tr : v[jj];
            u = j == NSP ? tc : u;
            double m = -hg * u;
            const double m1 = m + 1.0;
            m = j == lane ? m1 : m;
            col[jj] = ((lane < N) & (j < N)) ? m : (lane == j ? 1.0 : 0.0);
        }
    }
    bool open = lane < NP;              // this lane's row has not been a pivot row
    if ((w == 0) & (lane == 0)) sh.lu_ok = 1;
    __syncthreads();                    // every matrix entry is read: sh.q and sh.F may be written
    for (int blk = 0; blk < (N + NCW - 1) / NCW; ++blk) {
        double *lb = sh.q + COOP_Q + (blk & 1) * NCW * 64;
        if (w == blk) {
            // Steps without a branch for the usual columns: the upper 32 bits of the open rows' |entries|
            // (which order like the values) have one largest, and its quotients stay in the normal range by
            // the pivot's reciprocal (|entry| <= |pivot|).  The whole panel is taken again by the full
            // pivot search and plain division if a column was not like that.
            double *out = sh.F + min(lane, NP) * LDF + j0;      // (lanes past the matrix: a row of their own)
            double c[NCW];
            bool op = open;
            unsigned long long ties = 0;
            unsigned kmin = ~0u, kmost = 0, lmin = ~0u;
#pragma unroll
            for (int jn = 0; jn < NCW; ++jn) c[jn] = col[jn];
#pragma unroll
            for (int jj = 0; jj < NCW; ++jj) {
                const double rk = c[jj];
                const unsigned key = op ? (unsigned)__double2hiint(rk) & 0x7fffffffu : 0u;
                const unsigned kmax = wave_max_u32(key);
                const unsigned long long hit = __builtin_amdgcn_ballot_w64(key == kmax);
                const int p = __builtin_ctzll(hit);
                const double piv = bcast(rk, p);
                double u[NCW];
#pragma unroll
                for (int jn = jj + 1; jn < NCW; ++jn) u[jn] = bcast(c[jn], p);
                const double lq = quot(rk, piv, recip(piv));
                op = op & (lane != p);
                const double l = op ? lq : 0.0;
#pragma unroll
                for (int jn = jj + 1; jn < NCW; ++jn) c[jn] = fma(-l, u[jn], c[jn]);
                ties |= hit & (hit - 1);
                kmin = min(kmin, kmax);
                kmost = max(kmost, kmax);
                lmin = min(lmin, ((unsigned)__double2hiint(l) & 0x7fffffffu) - 1u);     // (0: none)
                sh.perm[j0 + jj] = p;
                out[jj] = op ? lq : rk;
                lb[jj * 64 + lane] = l;
                __builtin_amdgcn_sched_barrier(0);
            }
            // pivots in 2^-100 .. 2^102, multipliers from 2^-790 on (below 2^-1042 they are denormal and
            // change nothing)
            const bool odd = ties != 0 || kmin < 0x39b00000u || kmost >= 0x46500000u || __any(lmin < 0x0e900000u);
            if (__builtin_expect(odd, 0)) {
                bool good = true;
#pragma unroll 1
                for (int jj = 0; jj < NCW; ++jj) {
                    const double rk = col[0];
                    bool ok = true;
                    const int p = pivot_row(rk, open, ok);
                    const double piv = bcast(rk, p);
                    good = good & ok & (piv != 0.0);
                    sh.perm[j0 + jj] = p;
                    open = open & (lane != p);
                    const double l = open ? rk / piv : 0.0;
                    out[jj] = open ? l : rk;
                    lb[jj * 64 + lane] = l;
#pragma unroll
                    for (int jn = 1; jn < NCW; ++jn) col[jn - 1] = fma(-l, bcast(col[jn], p), col[jn]);
                }
                if (!good && lane == 0) sh.lu_ok = 0;
            }
        }
        __syncthreads();
        if (w > blk) {
            double l[NCW];
            int pv[NCW];
#pragma unroll
            for (int jj = 0; jj < NCW; ++jj) {
                l[jj] = lb[jj * 64 + lane];
                pv[jj] = sh.perm[blk * NCW + jj];
            }
#pragma unroll
            for (int jj = 0; jj < NCW; ++jj) {
                const int p = __builtin_amdgcn_readfirstlane(pv[jj]);
                double u[NCW];
#pragma unroll
                for (int jn = 0; jn < NCW; ++jn) u[jn] = bcast(col[jn], p);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int jn = 0; jn < NCW; ++jn) col[jn] = fma(-l[jj], u[jn], col[jn]);
                open = open & (lane != p);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    __syncthreads();
}

// A rate evaluation, the part of waves 1 .. 7.
template <int NSP>
__device__ __forceinline__ void serve_rates(const DevKin *__restrict__ K, Cell<NSP> &sh, const Consts &cs, const Own &own,
                                            int lane, int w, int cmd) {
    CSeries *k = get_series();
    const Temp tp = temperature(k, sh.z[NSP]);
    if (w < 7 && row_block(w) * 64 < cs.ii) {
        const int i = row_block(w) * 64 + lane;
        const Row row = row_begin(K, cs, own, k, min(i, cs.ii - 1), tp);
        __syncthreads();
        row_end(K, sh, cs, own, k, row, i, tp.T, cmd);
    } else {
        if (w == 7) falloff_terms(sh, cs, own, k, lane, tp);
        __syncthreads();
        if (w == 7 && lane == 0) {
            if (cmd == CMD_JAC) sh.F[6 * COOP_MAXR] = 0.0;
            if (cmd == CMD_SPLIT) sh.F[COOP_MAXR] = sh.F[FR + COOP_MAXR] = 0.0;
        }
    }
    __syncthreads();
    if (w <= 4) {
        const int g = w - 1;
        if (cmd == CMD_SPLIT) {
            const unsigned long long *e = reinterpret_cast<const unsigned long long *>(K->coop_split) + own.off;
            sh.S[g][lane] = list_sum<true>(e, own.len, own.mx, sh.F + FR, sh.F);        // reactant slots, product slots
            sh.S[4 + g][lane] = list_sum<true>(e, own.len, own.mx, sh.F, sh.F + FR);
        } else {
            sh.S[g][lane] = list_sum<false>(sh.list + own.off, own.len, own.mx, sh.q, sh.q);
        }
    }
    if (cmd == CMD_JAC) jac_gather(K, sh, lane, w);
    __syncthreads();
    if (cmd == CMD_JAC && w == 7) {
        // sum_j u_j J_jk for the temperature row, while wave 0 goes on
        double s = 0.0;
        const int l = min(lane, NSP - 1);
#pragma unroll 8
        for (int j = 0; j < NSP; ++j) s = s + sh.u[j] * sh.J[j * NSP + l];
        sh.tsum[lane] = s;
    }
}

// The compiler's own lane write (clang has no builtin for it): a vector instruction may read a scalar register
// that another vector instruction wrote only two wait states later, and the compiler provides them for
// instructions that it knows, not inside inline assembly.
extern "C" __device__ int fcfd_writelane(int v, int k, int old) __asm("llvm.amdgcn.writelane.i32");

// v, the same in all lanes, into lane k of x
__device__ __forceinline__ double put_lane(double x, double v, const int k) {
    const int lo = fcfd_writelane(__double2loint(v), k, __double2loint(x));
    const int hi = fcfd_writelane(__double2hiint(v), k, __double2hiint(x));
    return __hiloint2double(hi, lo);
}

// Solves M x = b with the factors in sh.F; b and x one component per lane of wave 0.  Lane r carries the
// right-hand side of the row pivoted at step r (pr), dg its reciprocal pivot.  A step of either
// substitution broadcasts its unknown and takes it from the right-hand sides by one fused multiply-add
// (the back substitution multiplies by the reciprocal pivot first).  The steps do not mask lanes: an
// unknown is put aside as it is broadcast, what later steps do to its lane is not read.
template <int NSP>
__device__ __attribute__((noinline)) double solve(FCFD_LDS const Cell<NSP> *shl, double b, int pr, double dg) {
    constexpr int N = Cell<NSP>::N;
    const Cell<NSP> &sh = *(const Cell<NSP> *)shl;
    const double *row = sh.F + pr * Cell<NSP>::LDF;
    double rv[8], nv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) rv[u] = row[u];
    double bq = __shfl(b, pr, 64), x = 0.0;
#pragma unroll
    for (int k0 = 0; k0 < N - 1; k0 += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) nv[u] = row[k0 + 8 < N - 1 ? k0 + 8 + u : N - 1 - u >= 0 ? N - 1 - u : 0];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k0 + u < N - 1) {
                const double v = bcast(bq, k0 + u);
                bq = fma(-rv[u], v, bq);
                x = put_lane(x, v, k0 + u);
            }
#pragma unroll
        for (int u = 0; u < 8; ++u) rv[u] = nv[u];
    }
    bq = put_lane(x, bcast(bq, N - 1), N - 1);
#pragma unroll
    for (int k1 = N - 1; k1 > 0; k1 -= 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) nv[u] = row[k1 - 8 - u >= 0 ? k1 - 8 - u : 0];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k1 - u > 0) {
                const double v = bcast(bq * dg, k1 - u);
                bq = fma(-rv[u], v, bq);
                x = put_lane(x, v, k1 - u);
            }
#pragma unroll
        for (int u = 0; u < 8; ++u) rv[u] = nv[u];
    }
    x = put_lane(x, bcast(bq * dg, 0), 0);
    return lane_id() < N ? x : 0.0;
}

template <int NSP>
__global__ void __launch_bounds__(64 * CW, 4) k_chem_coop(ChemArgs a) {
    __shared__ Cell<NSP> sh;
    constexpr int N = Cell<NSP>::N;
    const int lane = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    FCFD_GLB const DevThermo *thg = (FCFD_GLB const DevThermo *)a.thermo;
    FCFD_GLB const DevKin *Kg = (FCFD_GLB const DevKin *)a.kin;
    FCFD_LDS Cell<NSP> *shl = (FCFD_LDS Cell<NSP> *)&sh;
    const DevThermo *__restrict__ th = a.thermo;
    const DevKin *__restrict__ K = a.kin;
    const int nitems = a.list_n ? int(*a.list_n) : a.ncells;
    if (!coop_list(a, nitems) || int(blockIdx.x) >= nitems) return;       // (no more workgroups than cells)
    // entries that no reaction reaches are never written again
    for (int e = threadIdx.x; e < NSP * NSP; e += 64 * CW) sh.J[e] = 0.0;
    for (int e = threadIdx.x; e < COOP_LIST / 4; e += 64 * CW)
        sh.list[e] = reinterpret_cast<const unsigned long long *>(K->coop_sum)[e];
    if (w == 0) {
        const int k = min(lane, NSP - 1);
#pragma unroll
        for (int n = 0; n < 7; ++n) {
            sh.lo[n][lane] = th->alo[k][n];
            sh.hi[n][lane] = th->ahi[k][n];
        }
        sh.wt[lane] = th->wt[k];
        sh.rwt[lane] = th->rwt[k];
        sh.tmid[lane] = th->tmid[k];
        sh.c[lane] = 1.0;               // COOP_EMPTY
        sh.smh[lane] = 0.0;
        if (lane == 0) sh.q[COOP_MAXR] = 0.0;
    }
    __syncthreads();
    if (w != 0) {
        const Consts cs{K->ii, K->nfal, K->small, K->exparg, th->pa, th->ru};
        const Own own = load_own(K, cs, w);
        for (;;) {
            // opaque copies: what depends on them alone is computed where it is used, not kept in registers
            // across the loop (there are too few)
            int l = lane, wl = w;
            FCFD_GLB const DevKin *Kl = Kg;
            Own o = own;
            asm volatile("" : "+v"(l), "+s"(wl), "+s"(Kl), "+v"(o.w[0]), "+v"(o.w[1]), "+v"(o.w[2]), "+v"(o.w[3]),
                              "+v"(o.off), "+v"(o.len));
            __syncthreads();                               // wave 0 has posted a command
            const int cmd = __builtin_amdgcn_readfirstlane(sh.cmd);
            if (cmd == CMD_EXIT) return;
            if (cmd == CMD_LU) factor<NSP>(sh, l, wl);
            else serve_rates<NSP>((const DevKin *)Kl, sh, cs, o, l, wl, cmd);
        }
    }
    auto post = [&](int cmd) {
        if (lane == 0) sh.cmd = cmd;
        __syncthreads();
    };
    // f at the state z (lane NSP: T)
    auto rhs = [&](double z) {
        sh.z[lane] = z;
        post(CMD_RHS);
        return rates<NSP>(thg, Kg, shl, CMD_RHS).f;
    };
    for (;;) {
        int item = 0;
        if (lane == 0) item = int(atomicAdd(a.counter, 1u));
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= nitems) break;
        const int cell = a.list ? a.list[item] : item;

        // ---- load (reaction_macks, SRC/source.f90:44-56) ----
        long col = 0;
        double rho_si, dt, T0, y_raw = 0.0;
        if (a.layout == 0) {
            const int b = cell / a.ncell, i = cell % a.ncell;
            col = long(b) * a.S + a.lv + i;
            rho_si = a.qf[col];
            T0 = a.qf[2 * a.P + col];
            dt = a.dt_dev ? *a.dt_dev : a.dt;
            if (lane < NSP) y_raw = a.qf[(3 + lane) * a.P + col];
        } else {
            rho_si = a.b_rho[cell];
            dt = a.b_dt[cell];
            T0 = a.b_T[cell];
            if (lane < NSP) y_raw = a.b_y[long(lane) * a.ncells + cell];
        }
        const double rho = rho_si * 1.e-3;
        if (lane == 0) sh.rho = rho;
        double y = a.layout == 0 ? adjusted(y_raw, lane, NSP) : y_raw;   // adjust_sum(y_sp)
        double e0, cv0;
        energy<NSP>(th, adjusted(y, lane, NSP), T0, e0, cv0);
        if (lane == NSP) y = T0;

        double t = 0.0, h = dt;
        if (a.hmem) {   // the last call's proposal for this cell, if smaller than dt
            const double hp = a.hmem[cell];
            if (hp > 0.0 && hp < dt) h = hp;
        }
        bool expl = false;
        int steps = 0, rejects = 0, newton = 0;
        // ---- explicit retry: two Heun steps of dt/2, each accepted by its own embedded Euler
        //      estimate (weights at the step's start).  Trace radicals at the atol level in a cold
        //      mixture relax so fast that one explicit step of dt overshoots (dt times their
        //      consumption rate near 2) while a half step does not; such cells need no Jacobian.  (The
        //      step over dt itself has already failed for every listed cell.) ----
        if (t < dt && !(a.retry_done && *a.retry_done)) {
            const double hs = dt * 0.5;
            double yh = y;
            bool ok = true;
            for (int sub = 0; sub < 2 && ok; ++sub) {
                const double wt = lane < NSP ? 1.0 / (a.atol + a.rtol * fabs(yh))
                                             : (lane == NSP ? 1.0 / (a.rtol * fabs(yh)) : 0.0);
                const double fa = rhs(yh);
                const double fb = rhs(lane < N ? yh + hs * fa : 0.0);
                const double err = wnorm(lane < N ? (hs * 0.5) * (fb - fa) : 0.0, wt, N);
                if (err <= 1.0) {
                    if (lane < N) yh = yh + (hs * 0.5) * (fa + fb);
                } else {
                    ok = false;
                }
            }
            if (ok) {
                y = yh;
                t = dt;
                steps = 2;
                expl = true;
            }
        }
        // ---- SDIRK3 over [0, dt] ----
        while (t < dt && steps + rejects < CH_MAXSTEPS) {
            if (h > dt - t) h = dt - t;
            const double Tn = bcast(y, NSP);
            const double wt = lane < NSP ? 1.0 / (a.atol + a.rtol * fabs(y))
                                         : (lane == NSP ? 1.0 / (a.rtol * fabs(y)) : 0.0);
            // J at (y, Tn) and f there, the first Newton evaluation of stage 0; a rejected attempt (same
            // y) finds J unchanged
            sh.z[lane] = lane < N ? y : 0.0;
            post(CMD_JAC);
            const Rates fy = rates<NSP>(thg, Kg, shl, CMD_JAC);
            {
                // temperature column by a forward difference, temperature row from the concentration
                // Jacobian
                const double dT = Tn * 1.0e-6;
                const double f1 = rhs(lane == NSP ? Tn + dT : (lane < N ? y : 0.0));
                if (lane < N) sh.tcol[lane] = (f1 - fy.f) / dT;
                const double fT = bcast(fy.f, NSP);
                if (lane < NSP) {
                    const double s = sh.tsum[lane] * rho / th->wt[lane];
                    sh.trow[lane] = -s / (rho * fy.cvm) - fT * (fy.cvk / th->wt[lane]) / fy.cvm;
                }
            }
            for (;;) {
                const double hg = h * CH_G;
                if (lane == 0) sh.hg = hg;
                post(CMD_LU);
                factor<NSP>(sh, lane, 0);
                bool ok = sh.lu_ok != 0;
                const int pr = lane < N ? sh.perm[lane] : 0;
                const double dg = lane < N ? 1.0 / sh.F[pr * Cell<NSP>::LDF + lane] : 0.0;
                double k0 = 0.0, k1 = 0.0, k2 = 0.0, z = 0.0;
                for (int st = 0; st < 3 && ok; ++st) {
                    double base = y;
                    if (st == 1) base = base + h * CH_A21 * k0;
                    if (st == 2) base = base + h * CH_B1 * k0 + h * CH_B2 * k1;
                    z = st == 0 ? base : base + hg * (st == 1 ? k0 : k1);
                    double prev = 0.0;
                    bool conv = false;
                    for (int it = 0; it < CH_MAXIT; ++it) {
                        const double f = st == 0 && it == 0 ? fy.f : rhs(z);      // z = y there
                        double r = lane < N ? -(z - base - hg * f) : 0.0;
                        r = solve<NSP>(shl, r, pr, dg);
                        if (lane < N) z = z + r;
                        ++newton;
                        const double nrm = wnorm(lane < N ? r : 0.0, wt, N);
                        if (!(nrm == nrm) || (it > 0 && nrm > 0.9 * prev)) break;
                        if (nrm <= CH_KAPPA) { conv = true; break; }
                        prev = nrm;
                    }
                    if (!conv) { ok = false; break; }
                    const double kv = (z - base) / hg;
                    if (st == 0) k0 = kv; else if (st == 1) k1 = kv; else k2 = kv;
                }
                if (!ok) {
                    ++rejects;
                    h = h * 0.25;
                    if (steps + rejects >= CH_MAXSTEPS) break;
                    continue;
                }
                double ev = lane < N ? h * (CH_E1 * k0 + CH_E2 * k1 + CH_E3 * k2) : 0.0;
                ev = solve<NSP>(shl, ev, pr, dg);
                const double err = wnorm(lane < N ? ev : 0.0, wt, N);
                const double fac = 0.9 * fm_pow(fmax(err, 1.0e-10), -1.0 / 3.0);
                if (err <= 1.0) {
                    if (lane < N) y = z;
                    t = t + h;
                    ++steps;
                    h = h * fmin(4.0, fmax(0.2, fac));
                    break;
                }
                ++rejects;
                h = h * fmax(0.2, fac);
                if (steps + rejects >= CH_MAXSTEPS) break;
            }
        }
        const int failed = t < dt ? 1 : 0;

        // ---- energy-consistent temperature ----
        const double ya = adjusted(lane < NSP ? y : 0.0, lane, NSP);
        double T = bcast(y, NSP);
        for (int it = 0; it < 20; ++it) {
            double ek, cvk;
            energy<NSP>(th, ya, T, ek, cvk);
            const double d = (e0 - ek) / cvk;
            T = T + d;
            if (fabs(d) <= 1.0e-12 * T) break;
        }

        // ---- store (SRC/source.f90:60-73) ----
        if (a.layout == 0) {
            if (lane < NSP) a.qf[(3 + lane) * a.P + col] = ya;
            if (lane == 0) a.qf[2 * a.P + col] = T;
            if (a.hrr) {
                // heat_release_rate (SRC/thermo.f90:98-101)
                const double term = lane < NSP ? rho * th->h298[lane] * (ya - y_raw) / dt : 0.0;
                const double s1 = wsum(term);
                // heat_release_rate_omegadot via CKCDYR at the new state (SRC/thermo.f90:128-132)
                sh.z[lane] = lane == NSP ? T : ya;
                post(CMD_SPLIT);
                const Rates fc = rates<NSP>(thg, Kg, shl, CMD_SPLIT);
                const double s2 = wsum(lane < NSP ? th->wt[lane] * th->h298[lane] * (fc.cd - fc.dd) : 0.0);
                if (lane == 0) {
                    a.hrr[cell] = -s1 * 1.e-1;
                    a.hrr_dot[cell] = -s2 * 1.e-1;
                }
            }
        } else {
            if (lane < NSP) a.b_y[long(lane) * a.ncells + cell] = y;
            if (lane == 0) a.b_T[cell] = T;
        }
        if (a.stats && lane == 0) a.stats[cell] = ChemCellStats{steps, rejects, newton, failed};
        // route of a cell the explicit attempts finished: 3 the two half steps
        if (a.route && expl && lane == 0) a.route[cell] = 3;
        if (a.hmem && lane == 0) a.hmem[cell] = expl ? 0.0 : h;
    }
    post(CMD_EXIT);
}

}  // namespace

hipError_t launch_chem_coop(const ChemArgs &a, int nsp, int nwg, hipStream_t st) {
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_chem_coop<N>), dim3(unsigned(nwg)), dim3(64 * CW), 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

}  // namespace fcfd
