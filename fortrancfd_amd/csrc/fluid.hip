// fluid.hip -- kernels of the hydrodynamic part of one time step.
//
// Device layout ("SoA, ghost-padded"): variable v of padded column c lives at q[v*P + c].  Block b
// owns columns [b*S, (b+1)*S), S = ncell + 2*lv; its interior cell i (0-based) is column
// b*S + lv + i, exactly the reference's b_obj(ib)%qf(:, ista-lv : iend+lv) column range.
// Interface j (0..ncell) of block b -- the reference's Fplus(:, ista-1+j) -- is F[v*PF + b*(ncell+1)+j].
#include <algorithm>

#include "fluid_coop.hpp"
#include "fluid.hpp"

namespace fcfd {

// ---------------------------------------------------------------------------------------------
// Per-side interface state: what qfToQc + pressure + sonic_speed give for one reconstructed
// primitive vector (SRC/flux.f90:247-268, SRC/eos.f90:11-46).
// ---------------------------------------------------------------------------------------------
struct Side {
    double rho, u, p, a, E;
};

__device__ __forceinline__ double pair_other(double v) { return __shfl_xor(v, 32, 64); }

__device__ __forceinline__ Side pair_other(const Side &me) {
    Side o;
    o.rho = pair_other(me.rho); o.u = pair_other(me.u);
    o.p = pair_other(me.p); o.a = pair_other(me.a); o.E = pair_other(me.E);
    return o;
}

// ---------------------------------------------------------------------------------------------
// calc_flux_advection: 32 interfaces per workgroup of four waves.  Lanes 0..31 of every wave build
// the left states of the workgroup's interfaces, lanes 32..63 the right states (the right-state
// formulas are the left-state ones on the mirrored stencil); wave w reconstructs the species
// w*M .. w*M + M - 1 and one of rho, u, T, and keeps its species in registers.  The mixture sums
// run over the waves in species order (chain_sum); wave 0 completes the two side records, exchanges
// them between the lane halves, evaluates the Riemann branch and the first three components, and
// publishes what the species components need; with HLLC only the upwind side's lanes write those.
// Every output is the same expression of the same operands as in a one-lane evaluation.
//
// Bound: FP64 issue (WENO weights, NASA-7 sums).  A whole side per lane, with its 53 mass fractions in
// 27 KB of LDS per wave, left one wave per SIMD, full divisions and per-lane coefficient selects: 54 us
// for 400 cells, 144 us for 65,536, 560 us for 262,144 (GRI-3.0, WENO5-JS + HLLC).  Split over four
// waves (142 registers, three waves per SIMD), with scalar coefficients and quotients by shared
// reciprocals: 16, 55 and 195 us.  The mass fractions wait in LDS while the sums run: kept in
// registers they cost the third wave (236 us).
// ---------------------------------------------------------------------------------------------
template <int NSP, int RK, bool SPH, int RS, int WPE = 3>
__global__ void __launch_bounds__(64 * GW, WPE) k_flux(FluxArgs a) {
    constexpr int M = group_m<NSP>();
    __shared__ CoopShared sh;
    __shared__ double prim[3][64];                        // rho, u, T of this lane's side
    __shared__ double pub[3][64];                         // the Riemann solution, for the species components
    __shared__ double park[M][64 * GW];                   // each lane's mass fractions while the sums run
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int s = lane >> 5;                              // 0: left state, 1: right state
    const unsigned nif = unsigned(a.ncell) + 1u, total = unsigned(a.nblk) * nif;
    const unsigned g0 = xcd_block() * 32u + unsigned(lane & 31);
    const bool live = g0 < total;
    const unsigned g = live ? g0 : total - 1u;            // lanes past the end shadow the last interface
    const unsigned bl = g / nif, j0 = g - bl * nif;
    const unsigned c0 = bl * unsigned(a.S) + unsigned(a.lv) + j0 - 1u;   // the interface's left cell
    CThermo *m = constant(a.thermo);
    const double *__restrict__ q = a.qf;

    double y[M];
    if constexpr (RK == R_WENO5JS || RK == R_WENO5Z) {
        // byte offsets of the side's stencil: left q[c0 - 2 .. c0 + 2], right q[c0 + 3 .. c0 - 1]
        unsigned o[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) o[i] = (c0 + unsigned(s ? 3 - i : i - 2)) * 8u;
        bool big = false;
        // two variables' stencils in flight ahead of the one being reconstructed (more would spill)
        auto row = [&](int j) { return q + long(j < 0 ? min(w, 2) : 3 + min(w * M + j, NSP - 1)) * a.P; };
        double v[2][5];
        load5(row(-1), o, v[0]);
        load5(row(0), o, v[1]);
#pragma unroll
        for (int j = -1; j < M; ++j) {
            double r = weno5_lane<RK>(v[(j + 1) & 1], s, big);
            asm volatile("" : "+v"(r));                   // finished here, not behind the test of big
            if (j < 0) { if (w < 3) prim[w][lane] = r; }
            else y[j] = r;
            if (j + 2 < M) load5(row(j + 2), o, v[(j + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (__any(big)) {                                 // far out of any gas: with plain divisions
            if (w < 3) prim[w][lane] = reconstruct_side<RK>(q + long(w) * a.P, c0, a.muscl, s);
#pragma unroll
            for (int j = 0; j < M; ++j) {
                y[j] = reconstruct_side<RK>(q + long(3 + min(w * M + j, NSP - 1)) * a.P, c0, a.muscl, s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else {
        if (w < 3) prim[w][lane] = reconstruct_side<RK>(q + long(w) * a.P, c0, a.muscl, s);
#pragma unroll
        for (int j = 0; j < M; ++j) y[j] = reconstruct_side<RK>(q + long(3 + min(w * M + j, NSP - 1)) * a.P, c0, a.muscl, s);
    }
    bool ok = true;
#pragma unroll
    for (int j = 0; j < M; ++j) {
        y[j] = w * M + j < NSP ? y[j] : 0.0;
        ok = ok && num_ok(y[j]);
    }
    const bool fast = __all(ok);
    double sy, syw;
    {
        double yw[M], r[2];
        over_wt_coop<NSP>(m, w, fast, y, yw);             // CKYTX on the raw reconstructed Y
        // (its barriers also publish prim)
        chain_sum<2, M>(sh.c[0], w, lane, [&](int c, int j) { return c == 0 ? fmax(y[j], 0.0) : yw[j]; }, r);
        sy = r[0];                                        // adjust_sum(Y) denominator
        syw = r[1];
    }
    const double rho = prim[0][lane], u = prim[1][lane], T = prim[2][lane];
    double mix[4];                                        // mean molar mass, u, cp, cv (molar)
    {
        // mole fractions, clipped and renormalised (SRC/flux.f90:250-253)
        double x[M], r[1];
        ytx_coop<NSP>(m, w, fast, syw, y, x);
#pragma unroll
        for (int j = 0; j < M; ++j) park[j][threadIdx.x] = y[j];
#pragma unroll
        for (int j = 0; j < M; ++j) x[j] = fmax(x[j], 0.0);
        chain_sum<1, M>(sh.c[1], w, lane, [&](int, int j) { return x[j]; }, r);
        scale_coop<M>(fast, r[0], x);
        double hu[M], cp[M];
        species_thermo<NSP, true, true>(m, w, T, __all(den_ok(T)), hu, cp);
        const double ru = m->ru;
        // the products are formed as they are added: the terms of four sums would not fit beside y
        chain_sum<4, M>(sh.c[0], w, lane, [&](int c, int j) {
            return x[j] * (c == 0 ? m->wt[min(w * M + j, NSP - 1)] : c == 1 ? hu[j] : c == 2 ? cp[j] : cp[j] - ru);
        }, mix);
    }

    double *__restrict__ F = a.F;
    const long PF = a.PF;
    // Fplus accumulates (SRC/flux.f90:358): on top of the transport flux when there is one
    const bool acc = a.accumulate != 0;
    auto put = [acc](double *row, unsigned at, double val) {
        double *d = reinterpret_cast<double *>(reinterpret_cast<char *>(row) + at);
        *d = acc ? *d + val : val;
    };
    const unsigned gb = g * 8u;
    if (w == 0) {
        Side me;
        me.rho = rho; me.u = u;
        const double wtm = mix[0];
        me.p = (rho * 1.e-3) * m->ru * T / wtm * 0.1;                // pressure(), CKPX
        const double e = mix[1] * 1.e-4 / wtm;                       // specific_energy()
        me.E = rho * (e + 0.5 * (u * u));
        const double cp = mix[2] * 1.e-4 / wtm, cv = mix[3] * 1.e-4 / wtm;
        me.a = sqrt(cp / cv * me.p / rho);                           // sonic_speed()
        const Side ot = pair_other(me);
        const Side L = s ? ot : me;
        const Side R = s ? me : ot;
        // physical fluxes of mass, momentum, energy (SRC/flux.f90:270-280)
        const double fl0 = L.rho * L.u, fr0 = R.rho * R.u;
        // spherical: no pressure in the momentum flux; the update adds its gradient (SRC/flux.f90:272-278)
        const double fl1 = SPH ? L.rho * L.u * L.u : L.rho * L.u * L.u + L.p;
        const double fr1 = SPH ? R.rho * R.u * R.u : R.rho * R.u * R.u + R.p;
        const double fl2 = (L.E + L.p) * L.u, fr2 = (R.E + R.p) * R.u;
        double f0, f1, f2;
        if (RS == 0) {                                                // LxF (SRC/flux.f90:291-294)
            const double lL = fmax(fmax(fabs(L.u - L.a), fabs(L.u)), fabs(L.u + L.a));
            const double lR = fmax(fmax(fabs(R.u - R.a), fabs(R.u)), fabs(R.u + R.a));
            const double al = fmax(lL, lR);
            f0 = 0.5 * (fl0 + fr0 - al * (R.rho - L.rho));
            f1 = 0.5 * (fl1 + fr1 - al * (R.rho * R.u - L.rho * L.u));
            f2 = 0.5 * (fl2 + fr2 - al * (R.E - L.E));
            pub[0][lane] = al;
        } else {
            const double rt = sqrt(R.rho / L.rho);
            const double uro = (L.u + rt * R.u) / (1.0 + rt);
            const double aro = (L.a + rt * R.a) / (1.0 + rt);
            const double sL = fmin(L.u - L.a, uro - aro), sR = fmax(R.u + R.a, uro + aro);
            if (RS == 1) {                                            // HLL (SRC/flux.f90:300-315)
                const int br = (0.0 <= sL) ? 0 : ((sL <= 0.0 && 0.0 <= sR) ? 1 : 2);
                auto hll = [&](double fL, double fR, double QL, double QR) {
                    return br == 0 ? fL : (br == 1 ? (sR * fL - sL * fR + sL * sR * (QR - QL)) / (sR - sL) : fR);
                };
                f0 = hll(fl0, fr0, L.rho, R.rho);
                f1 = hll(fl1, fr1, L.rho * L.u, R.rho * R.u);
                f2 = hll(fl2, fr2, L.E, R.E);
                pub[0][lane] = sL;
                pub[1][lane] = sR;
                pub[2][lane] = double(br);
            } else {                                                  // HLLC (SRC/flux.f90:321-354)
                const double sM = (L.p - R.p + R.rho * R.u * (sR - R.u) - L.rho * L.u * (sL - L.u)) /
                                  (R.rho * (sR - R.u) - L.rho * (sL - L.u));
                // branch chain of SRC/flux.f90:332-354
                const int br = (0.0 <= sL) ? 0 : ((sL <= 0.0 && 0.0 <= sM) ? 1 : ((sM <= 0.0 && 0.0 <= sR) ? 2 : 3));
                const bool left = br <= 1;
                const Side S = left ? L : R;
                f0 = left ? fl0 : fr0;
                f1 = left ? fl1 : fr1;
                f2 = left ? fl2 : fr2;
                // 0: this lane's side is not the upwind one; 1: supersonic, upwind flux; 2: star state
                double mode = left == (s == 0) ? 1.0 : 0.0;
                if (!(br == 0 || br == 3)) {                          // star state of the upwind side
                    const double sK = left ? sL : sR;
                    const double c = S.rho * (sK - S.u) / (sK - sM);
                    const double v2 = S.E / S.rho + (sM - S.u) * (sM + S.p / (S.rho * (sK - S.u)));
                    f0 = f0 + sK * (c * 1.0 - S.rho);
                    f1 = f1 + sK * (c * sM - S.rho * S.u);
                    f2 = f2 + sK * (c * v2 - S.E);
                    mode = 2.0 * mode;
                    pub[1][lane] = sK;
                    pub[2][lane] = c;
                }
                pub[0][lane] = live ? mode : 0.0;
            }
        }
        if (live) {
            if (s == 0) {
                put(F, gb, f0);
                put(F + 2 * PF, gb, f2);
            } else {
                put(F + PF, gb, f1);
            }
            if (a.godunov && s == 0) {                                // SRC/flux.f90:360-367
                const double rt = sqrt(R.rho / L.rho);
                double *G = a.godunov + g;
                G[0] = sqrt(R.rho * L.rho);
                G[PF] = (L.u + rt * R.u) / (1.0 + rt);
                G[2 * PF] = (L.p + rt * R.p) / (1.0 + rt);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < M; ++j) y[j] = park[j][threadIdx.x];
    // adjust_sum(Y) where QcL/R needs it: Q_k = rho (max(Y_k, 0) / sy)
    const bool fd = fast && __all(den_ok(sy) && den_ok(rho));
    const double rsy = recip(sy), rrho = recip(rho);
    if (RS == 2) {
        const double mode = pub[0][lane], sK = pub[1][lane], c = pub[2][lane];
        // star state: F + s_K (c Q_k / rho - Q_k); supersonic: the upwind flux
        double f[M];
        if (__any(mode == 2.0)) {
            if (fd) {
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    const double Qk = rho * quot(fmax(y[j], 0.0), sy, rsy);
                    f[j] = rho * y[j] * u + sK * (c * quot(Qk, rho, rrho) - Qk);
                }
            } else {
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    const double Qk = rho * (fmax(y[j], 0.0) / sy);
                    f[j] = rho * y[j] * u + sK * (c * (Qk / rho) - Qk);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if (__any(mode == 1.0)) {
#pragma unroll
            for (int j = 0; j < M; ++j) f[j] = mode == 1.0 ? rho * y[j] * u : f[j];
        }
        if (mode != 0.0) {
            if (acc) {
#pragma unroll
                for (int j = 0; j < M; ++j)
                    if (w * M + j < NSP) f[j] = at_byte(F + long(3 + w * M + j) * PF, gb) + f[j];
            }
#pragma unroll
            for (int j = 0; j < M; ++j)
                if (w * M + j < NSP) *reinterpret_cast<double *>(reinterpret_cast<char *>(F + long(3 + w * M + j) * PF) + gb) = f[j];
        }
    } else {
        // both sides enter: this lane's Q_k and physical flux go to the interface's other lane, and
        // the two lanes write alternate species
        const double w0 = pub[0][lane], w1 = pub[1][lane], w2 = pub[2][lane];
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int k = w * M + j;
            if (k >= NSP) break;
            const double yc = fmax(y[j], 0.0);
            const double Qm = rho * (fd ? quot(yc, sy, rsy) : yc / sy), fm = rho * y[j] * u;
            const double Qo = pair_other(Qm), fo = pair_other(fm);
            const double QL = s ? Qo : Qm, QR = s ? Qm : Qo, fL = s ? fo : fm, fR = s ? fm : fo;
            if ((k & 1) != s || !live) continue;
            double v;
            if (RS == 0) {
                v = 0.5 * (fL + fR - w0 * (QR - QL));
            } else {
                v = w2 == 0.0 ? fL : (w2 == 1.0 ? (w1 * fL - w0 * fR + w0 * w1 * (QR - QL)) / (w1 - w0) : fR);
            }
            put(F + (3 + k) * PF, gb, v);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// QcToqf on one column, writing qf (SRC/eos.f90:49-83).
// ---------------------------------------------------------------------------------------------
template <int NSP>
__device__ __forceinline__ void qc_to_qf_store(const DevThermo *__restrict__ m, const double (&Qv)[NSP + 3],
                                               double *__restrict__ qf, long P, long c) {
    const double rho = Qv[0];
    const double u = Qv[1] / rho;
    double y[NSP];
#pragma unroll
    for (int k = 0; k < NSP; ++k) y[k] = Qv[3 + k] / rho;
    adjust_sum<NSP>(y);
#pragma unroll
    for (int k = 0; k < NSP; ++k) qf[(3 + k) * P + c] = y[k];
    ytx<NSP>(m, y);
    adjust_sum<NSP>(y);
    const double e = Qv[2] / rho - 0.5 * (u * u);
    qf[c] = rho;
    qf[P + c] = u;
    qf[2 * P + c] = temperature_con<NSP>(m, e, y);
}

// Stage end: RK combine of the source cell, ghost fill, primitive recovery -- the interior update
// of SRC/timeintegration.f90:150-175 (or :48-56 for Euler), then update_boundary /
// interpolation_block / QcToqf on every column (:201-215).  mode 0: Q = Qin - dt/dx*dF;
// mode 1: Q = h1*Q0 + h2*(Qin - dt/dx*dF); mode 2: no update (ghost fill + QcToqf only).
// 64 columns per workgroup of four waves, wave w with the species w*M .. w*M + M - 1.  Bound: the FP64
// issue of the temperature Newton iteration and its chain from one iteration to the next.  One
// lane per column (56 values in registers, the coefficients selected per lane) took 75 us however
// few columns there were, 111 us for 65,536 and 382 us for 262,144; split over four waves (three per
// SIMD) 29, 50 and 160 us.
template <int NSP, int MODE, bool SPH, int WPE = 3>
__global__ void __launch_bounds__(64 * GW, WPE) k_stage_end(StageArgs a) {
    constexpr int M = group_m<NSP>();
    __shared__ CoopShared sh;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned cend = a.col0 + a.ncol;
    const unsigned cq = a.col0 + xcd_block() * 64u + unsigned(lane);
    const unsigned c = min(cq, cend - 1u);                // lanes past the end shadow the last column
    const int b = int(c / unsigned(a.S)), i = int(c - unsigned(b) * unsigned(a.S)) - a.lv;
    const bool ghost = (i < 0 || i >= a.ncell);
    const bool live = cq < cend && (ghost || !a.ghosts_only);
    if (!__any(live)) return;                             // the same in the four waves
    int sb, si;
    double sgn;
    ghost_source(a.left, a.right, a.ncell, b, i, sb, si, sgn);
    const unsigned sc = (unsigned(sb) * unsigned(a.S) + unsigned(a.lv + si)) * 8u;      // byte offsets
    const unsigned fj = (unsigned(sb) * unsigned(a.ncell + 1) + unsigned(si)) * 8u;
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const double dx = a.dxb ? a.dxb[sb] : a.dx;         // the source cell's block spacing
    const double dtdx = dt / dx;
    // spherical (SRC/timeintegration.f90:58-72, 177-196): face areas (r -+ dx/2)^2 and volume
    // r^2 dx at the source cell's centre
    constexpr bool sph = SPH && MODE != 2;
    double Al = 0.0, Ar = 0.0, dtdV = 0.0;
    if (sph) {
        const double rm = a.xm[long(sb) * a.ncell + si];
        const double tl = rm - (dx / 2.0), tr = rm + (dx / 2.0);
        Al = tl * tl;
        Ar = tr * tr;
        dtdV = dt / (rm * rm * dx);
    }
    auto value = [&](int v) {
        const double qi = at_byte(a.Qin + long(v) * a.P, sc);
        double Q = qi;
        if (MODE != 2) {
            const double *f = a.F + long(v) * a.PF;
            const double fr = at_byte(f + 1, fj), fl = at_byte(f, fj);
            const double base = sph ? qi - dtdV * (Ar * fr - Al * fl) : qi - dtdx * (fr - fl);
            if (MODE == 0) Q = base;
            else Q = a.h1 * at_byte(a.Q0 + long(v) * a.P, sc) + a.h2 * base;
        }
        return Q;
    };
    const double rho = value(0), rE = value(2);
    double ru = value(1);
    if (sph) ru = ru - dtdx * (at_byte(a.god + 2 * a.PF + 1, fj) - at_byte(a.god + 2 * a.PF, fj));
    ru = sgn < 0.0 ? -ru : ru;
    double q[M], u, T;
    // (species past the last one: the last one's column, then 0, so that no load waits on a branch)
#pragma unroll
    for (int j = 0; j < M; ++j) q[j] = value(3 + min(w * M + j, NSP - 1));
#pragma unroll
    for (int j = 0; j < M; ++j) q[j] = w * M + j < NSP ? q[j] : 0.0;
    const unsigned cb = c * 8u;
    auto put = [cb, live](double *row, double v) {
        if (live) *reinterpret_cast<double *>(reinterpret_cast<char *>(row) + cb) = v;
    };
    // a refresh runs in place (Qout = Qin): ghost columns read interior columns, whose owners write
    // back the value they read
    if (w == 0) {
        put(a.Qout, rho);
        put(a.Qout + a.P, ru);
        put(a.Qout + 2 * a.P, rE);
    }
#pragma unroll
    for (int j = 0; j < M; ++j)
        if (w * M + j < NSP) put(a.Qout + long(3 + w * M + j) * a.P, q[j]);
    qc_to_qf_coop<NSP>(constant(a.thermo), sh, w, lane, rho, ru, rE, q, u, T, [&](int j, double y) {
        if (w * M + j < NSP) put(a.qf + long(3 + w * M + j) * a.P, y);
    });
    if (w == 0) {
        put(a.qf, rho);
        put(a.qf + a.P, u);
        put(a.qf + 2 * a.P, T);
    }
}

// RK4 stage (SRC/timeintegration.f90:222-356) with the reference's semantics: within the step the
// advection fluxes keep reading the primitives of the step start (only the left wall ghosts' are
// refreshed, by update_boundary), interior cells move by a quarter, a quarter and a full dt/dx
// flux difference in stages 1-3, k_s = -dt/dx dF_s accumulate as k1 + 2 k2 + 2 k3 (+ k4 at the end),
// the walls are mirrored after every stage and the block-interface ghosts are not refreshed; the
// last stage sets Q = Q0 + (1/6)(k1 + 2 k2 + 2 k3 + k4) and recovers the primitives everywhere.
template <int NSP>
__global__ void __launch_bounds__(64) k_rk4_stage(StageArgs a) {
    const long c = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= long(a.nblk) * a.S) return;
    const int b = int(c / a.S), i = int(c % a.S) - a.lv;
    const int st = a.mode;
    const bool interior = i >= 0 && i < a.ncell;
    const bool lwall = b == 0 && i < 0, rwall = b == a.nblk - 1 && i >= a.ncell;
    double Qv[NSP + 3];
    if (!interior && !lwall && !rwall) {                  // block-interface ghost: unchanged
#pragma unroll
        for (int v = 0; v < NSP + 3; ++v) {
            Qv[v] = a.Qin[v * a.P + c];
            a.Qout[v * a.P + c] = Qv[v];
        }
        if (st == 3) qc_to_qf_store<NSP>(a.thermo, Qv, a.qf, a.P, c);
        return;
    }
    int sb, si;
    double sgn;
    ghost_source(0, a.nblk - 1, a.ncell, b, i, sb, si, sgn);
    const long sc = long(sb) * a.S + a.lv + si;
    const long fj = long(sb) * (a.ncell + 1) + si;
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const double dx = a.dxb ? a.dxb[sb] : a.dx;
#pragma unroll
    for (int v = 0; v < NSP + 3; ++v) {
        const double d = a.F[v * a.PF + fj + 1] - a.F[v * a.PF + fj];
        const double k = -(dt / dx) * d;
        const double qi = a.Qin[v * a.P + sc];
        double Q;
        if (st < 2) Q = qi - 0.5 * (0.5 * dt / dx) * d;
        else if (st == 2) Q = qi - (dt / dx) * d;
        else Q = a.Q0[v * a.P + sc] + (1.0 / 6.0) * (a.acc[v * a.P + sc] + k);
        if (interior && st < 3) {
            const double prev = st == 0 ? 0.0 : a.acc[v * a.P + c];
            a.acc[v * a.P + c] = st == 0 ? k : prev + 2.0 * k;
        }
        if (v == 1) Q = sgn < 0.0 ? -Q : Q;
        Qv[v] = Q;
        a.Qout[v * a.P + c] = Q;
    }
    if (st == 3 || lwall) qc_to_qf_store<NSP>(a.thermo, Qv, a.qf, a.P, c);
}

// ---------------------------------------------------------------------------------------------
// Halo between blocks of unequal cell size (interpolation_block, SRC/block.f90:499-563), after the
// kernel that filled every halo as a plain copy.  k_smr_fill: one thread per (block pair,
// variable): the coarse block's lv ghosts average pairs of fine cells, then the fine block's lv
// ghosts take the coarse cell they lie in, -+ a quarter of its minmod slope (the slope stencil
// reaches the coarse ghost just written).  k_smr_qf: QcToqf on those ghost columns.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double smr_slope(double m, double p) {
    return 0.5 * (copysign(1.0, m) + copysign(1.0, p)) * fmin(fabs(m), fabs(p));
}

__global__ void __launch_bounds__(64) k_smr_fill(SmrArgs a) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nif * a.nequ) return;
    const int ib = a.ifb[t / a.nequ], v = t % a.nequ;
    const long L = long(ib) * a.S + a.lv, R = long(ib + 1) * a.S + a.lv;   // interior cell 0 of each
    const int nc = a.ncell, lv = a.lv;
    double *__restrict__ Q = a.Q + long(v) * a.P;
    if (a.dxb[ib] > a.dxb[ib + 1]) {                   // coarse | fine
        for (int g = 1; g <= lv; ++g)
            Q[L + nc - 1 + g] = (Q[R + 2 * (g - 1)] + Q[R + 2 * (g - 1) + 1]) / 2.0;
        for (int g = 1; g <= lv; ++g) {
            const long c = L + nc - 1 - (g - 1) / 2;
            const double s = smr_slope(Q[c] - Q[c - 1], Q[c + 1] - Q[c]);
            Q[R - g] = (g % 2 == 1) ? Q[c] + 0.25 * s : Q[c] - 0.25 * s;
        }
    } else {                                            // fine | coarse
        for (int g = 1; g <= lv; ++g)
            Q[R - g] = (Q[L + nc - 1 - 2 * (g - 1)] + Q[L + nc - 1 - (2 * (g - 1) + 1)]) / 2.0;
        for (int g = 1; g <= lv; ++g) {
            const long c = R + (g - 1) / 2;
            const double s = smr_slope(Q[c] - Q[c - 1], Q[c + 1] - Q[c]);
            Q[L + nc - 1 + g] = (g % 2 == 1) ? Q[c] - 0.25 * s : Q[c] + 0.25 * s;
        }
    }
}

template <int NSP>
__global__ void __launch_bounds__(64) k_smr_qf(SmrArgs a) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nif * 2 * a.lv) return;
    const int ib = a.ifb[t / (2 * a.lv)], g = t % (2 * a.lv);
    // the left block's right ghosts, then the right block's left ghosts
    const long c = g < a.lv ? long(ib) * a.S + a.lv + a.ncell + g : long(ib + 1) * a.S + (g - a.lv);
    double Qv[NSP + 3];
#pragma unroll
    for (int v = 0; v < NSP + 3; ++v) Qv[v] = a.Q[v * a.P + c];
    qc_to_qf_store<NSP>(a.thermo, Qv, a.qf, a.P, c);
}

// ---------------------------------------------------------------------------------------------
// calc_dt (SRC/update.f90:13-59): max wave speed over interior cells -> dt on the device.  64 cells
// per workgroup of four waves, the species split over the waves as in k_stage_end; at most
// 2048 workgroups, which stride over the cells; the last one to finish writes dt.  13 / 18 / 48 us for
// 400 / 65,536 / 262,144 cells; one lane per cell and a launch of its own for dt took 18 / 25 / 53 us.
// ---------------------------------------------------------------------------------------------
template <int NSP>
__global__ void __launch_bounds__(64 * GW, 4) k_wave_speed(DtArgs a) {
    constexpr int M = group_m<NSP>();
    __shared__ CoopShared sh;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned n = unsigned(a.nblk) * unsigned(a.ncell);
    CThermo *m = constant(a.thermo);
    double most = 0.0;
    for (unsigned t0 = blockIdx.x * 64u; t0 < n; t0 += gridDim.x * 64u) {
        const unsigned t = min(t0 + unsigned(lane), n - 1u);      // a repeated cell changes no maximum
        const unsigned b = t / unsigned(a.ncell), i = t - b * unsigned(a.ncell);
        const unsigned c = b * unsigned(a.S) + unsigned(a.lv) + i;
        const unsigned cb = column_bytes(c, lane0(c));
        const double *qf = a.qf + lane0(c);
        double y[M], x[M], s1[1];
        bool ok = true;
#pragma unroll
        for (int j = 0; j < M; ++j) {
            y[j] = at_byte(qf + long(3 + min(w * M + j, NSP - 1)) * a.P, cb);
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
            y[j] = w * M + j < NSP ? y[j] : 0.0;
            ok = ok && num_ok(y[j]);
        }
        const double rho = at_byte(qf, cb), u = at_byte(qf + a.P, cb), T = at_byte(qf + 2 * a.P, cb);
        const bool fast = __all(ok);
        over_wt_coop<NSP>(m, w, fast, y, x);
        chain_sum<1, M>(sh.c[0], w, lane, [&](int, int j) { return x[j]; }, s1);
        ytx_coop<NSP>(m, w, fast, s1[0], y, x);                   // no adjust_sum here (update.f90:396)
        double cp_k[M], unused[M], mix[3];
        species_thermo<NSP, false, true>(m, w, T, __all(den_ok(T)), unused, cp_k);
        const double ru = m->ru;
        chain_sum<3, M>(sh.c[1], w, lane, [&](int c, int j) {
            return x[j] * (c == 0 ? m->wt[min(w * M + j, NSP - 1)] : c == 1 ? cp_k[j] : cp_k[j] - ru);
        }, mix);
        if (w == 0) {
            const double wtm = mix[0];
            const double p = (rho * 1.e-3) * m->ru * T / wtm * 0.1;
            const double cp = mix[1] * 1.e-4 / wtm, cv = mix[2] * 1.e-4 / wtm;
            const double as = sqrt(cp / cv * p / rho);
            most = fmax(most, fmax(fmax(fabs(u - as), fabs(u)), fabs(u + as)));
        }
    }
    if (w == 0) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) most = fmax(most, __shfl_xor(most, off, 64));
        // One address for every workgroup's maximum and arrival serialises them (1024 workgroups: 10 us);
        // they meet at DT_SLOTS slots a cache line apart, and the last arrivals of the slots at one more.
        // Non-negative doubles order like their bit patterns.  Everything passes through atomics, so
        // no fence is needed (an agent-scope fence writes the L2 back, more than the whole kernel):
        // each arrival only has to follow the atomic before it, whose returned value it takes in.
        unsigned long long *slots = a.slots;
        const unsigned g = blockIdx.x % DT_SLOTS, in_slot = (gridDim.x - g + DT_SLOTS - 1) / DT_SLOTS;
        const unsigned nslots = min(gridDim.x, unsigned(DT_SLOTS));
        int last = 0;
        if (lane == 0) {
            // (the sign bit of a maximum is 0)
            const unsigned long long m0 = atomicMax(slots + g * 8, (unsigned long long)__double_as_longlong(most));
            const unsigned long long n0 = atomicAdd(slots + g * 8 + 1, 1ull + (m0 >> 63));
            if (n0 == in_slot - 1) last = atomicAdd(slots + DT_SLOTS * 8, 1ull) == nslots - 1;
        }
        if (__builtin_amdgcn_readfirstlane(last)) {
            // the last workgroup of all: the maximum of the slots gives dt; every word is zero again
            // for the next call
            double cvel = 0.0;
            if (unsigned(lane) < nslots) {
                cvel = __longlong_as_double((long long)atomicExch(slots + lane * 8, 0ull));
                atomicExch(slots + lane * 8 + 1, 0ull);
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) cvel = fmax(cvel, __shfl_xor(cvel, off, 64));
            if (lane == 0) {
                atomicExch(slots + DT_SLOTS * 8, 0ull);
                const double dt = (a.cfl * a.dx) / cvel;
                *a.dt_out = dt;
                if (a.time) *a.time = *a.time + dt;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Initial state (SRC/params.f90:305-580 + SRC/block.f90:413-429): interior columns.
// ---------------------------------------------------------------------------------------------
template <int NSP>
__global__ void __launch_bounds__(64) k_init_cells(InitArgs a) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= long(a.nblk) * a.ncell) return;
    const int b = int(t / a.ncell), i = int(t % a.ncell);
    const long c = long(b) * a.S + a.lv + i;
    const DevThermo *__restrict__ m = a.thermo;
    const double *cell = a.cells + t * (3 + NSP);
    const double T = cell[0], p = cell[1], u = cell[2];
    double x[NSP];
#pragma unroll
    for (int k = 0; k < NSP; ++k) x[k] = cell[3 + k];
    adjust_sum<NSP>(x);
    const double wx = mix_w<NSP>(m, x);
    const double rho = wx * (p * 10.0) / (m->ru * T) * 1.e3;      // density(): CKRHOX
    const MixSums ms = mix_sums<NSP>(m, x, T, true, false, false);
    const double e = ms.ubml * 1.e-4 / wx;                        // specific_energy()
    a.qf[c] = rho; a.qf[a.P + c] = u; a.qf[2 * a.P + c] = T;
    a.Qc[c] = rho; a.Qc[a.P + c] = rho * u; a.Qc[2 * a.P + c] = rho * (e + 0.5 * (u * u));
#pragma unroll
    for (int k = 0; k < NSP; ++k) {
        const double y = x[k] * m->wt[k] / wx;                    // CKXTY
        a.qf[(3 + k) * a.P + c] = y;
        a.Qc[(3 + k) * a.P + c] = rho * y;
    }
}

// ---------------------------------------------------------------------------------------------
// Conversions and reconstruction on host-array batches (stateless entry points).
// ---------------------------------------------------------------------------------------------
template <int NSP>
__global__ void k_qf_to_qc(const DevThermo *__restrict__ m, int n, const double *__restrict__ qf,
                           double *__restrict__ Qc, long P) {
    const long c = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= n) return;
    double y[NSP];
    const double rho = qf[c], u = qf[P + c], T = qf[2 * P + c];
#pragma unroll
    for (int k = 0; k < NSP; ++k) y[k] = qf[(3 + k) * P + c];
    double ya[NSP];
#pragma unroll
    for (int k = 0; k < NSP; ++k) ya[k] = y[k];
    adjust_sum<NSP>(ya);
#pragma unroll
    for (int k = 0; k < NSP; ++k) Qc[(3 + k) * P + c] = rho * ya[k];
    ytx<NSP>(m, y);
    adjust_sum<NSP>(y);
    const double wtm = mix_w<NSP>(m, y);
    const MixSums ms = mix_sums<NSP>(m, y, T, true, false, false);
    const double e = ms.ubml * 1.e-4 / wtm;
    Qc[c] = rho;
    Qc[P + c] = rho * u;
    Qc[2 * P + c] = rho * (e + 0.5 * (u * u));
}

template <int NSP>
__global__ void k_qc_to_qf(const DevThermo *__restrict__ m, int n, const double *__restrict__ Qc,
                           double *__restrict__ qf, long P) {
    const long c = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= n) return;
    double Qv[NSP + 3];
#pragma unroll
    for (int v = 0; v < NSP + 3; ++v) Qv[v] = Qc[v * P + c];
    qc_to_qf_store<NSP>(m, Qv, qf, P, c);
}

// qfToQc on the interior columns of a padded domain (reaction_macks' final loop,
// SRC/source.f90:78-82): 64 cells per workgroup of four waves, the species split as in k_stage_end
// (18 us for 65,536 cells; 33 us with one lane per cell).
template <int NSP>
__global__ void __launch_bounds__(64 * GW, 4) k_qf_to_qc_interior(const DevThermo *thermo, int nblk, int ncell, int lv,
                                                                  int S, const double *qf, double *Qc, long P) {
    constexpr int M = group_m<NSP>();
    __shared__ CoopShared sh;
    CThermo *m = constant(thermo);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const unsigned n = unsigned(nblk) * unsigned(ncell);
    const unsigned t0 = xcd_block() * 64u + unsigned(lane);
    const bool live = t0 < n;
    const unsigned t = live ? t0 : n - 1u;
    const unsigned b = t / unsigned(ncell);
    const unsigned c = b * unsigned(S) + unsigned(lv) + (t - b * unsigned(ncell));
    const unsigned cb = column_bytes(c, lane0(c));
    qf += lane0(c);
    Qc += lane0(c);
    auto put = [cb, live](double *row, double v) {
        if (live) *reinterpret_cast<double *>(reinterpret_cast<char *>(row) + cb) = v;
    };
    double y[M], x[M], s1[1];
#pragma unroll
    for (int j = 0; j < M; ++j) y[j] = at_byte(qf + long(3 + min(w * M + j, NSP - 1)) * P, cb);
    const double rho = at_byte(qf, cb), u = at_byte(qf + P, cb), T = at_byte(qf + 2 * P, cb);
    bool ok = true;
#pragma unroll
    for (int j = 0; j < M; ++j) {
        y[j] = w * M + j < NSP ? y[j] : 0.0;
        ok = ok && num_ok(y[j]);
    }
    const bool fast = __all(ok);
    // rho Y from adjust_sum(Y), X = adjust_sum(CKYTX(Y)) from the raw Y
    double s2[2];
    over_wt_coop<NSP>(m, w, fast, y, x);
    chain_sum<2, M>(sh.c[0], w, lane, [&](int c, int j) { return c == 0 ? fmax(y[j], 0.0) : x[j]; }, s2);
    ytx_coop<NSP>(m, w, fast, s2[1], y, x);
#pragma unroll
    for (int j = 0; j < M; ++j) {
        y[j] = fmax(y[j], 0.0);
        x[j] = fmax(x[j], 0.0);
    }
    scale_coop<M>(fast, s2[0], y);
#pragma unroll
    for (int j = 0; j < M; ++j)
        if (w * M + j < NSP) put(Qc + long(3 + w * M + j) * P, rho * y[j]);
    chain_sum<1, M>(sh.c[1], w, lane, [&](int, int j) { return x[j]; }, s1);
    scale_coop<M>(fast, s1[0], x);
    double hu[M], unused[M];
    species_thermo<NSP, true, false>(m, w, T, __all(den_ok(T)), hu, unused);
    chain_sum<2, M>(sh.c[0], w, lane, [&](int c, int j) {
        return x[j] * (c == 0 ? m->wt[min(w * M + j, NSP - 1)] : hu[j]);
    }, s2);
    if (w == 0) {
        const double e = s2[1] * 1.e-4 / s2[0];
        put(Qc, rho);
        put(Qc + P, rho * u);
        put(Qc + 2 * P, rho * (e + 0.5 * (u * u)));
    }
}

__global__ void k_recon(int n, const double *__restrict__ s, double *__restrict__ out) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    double st[8];
    for (int j = 0; j < 8; ++j) st[j] = s[r * 8 + j];
    double *o = out + r * 18;
    weno3z(st, o[0], o[1]);
    weno5<2>(st, o[2], o[3]);
    weno5<3>(st, o[4], o[5]);
    weno7z(st, o[6], o[7]);
    for (int f = 1; f <= 4; ++f) muscl3(st, o[6 + 2 * f], o[7 + 2 * f], f);
    o[16] = 0.0;
    o[17] = 0.0;
}

// ---------------------------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------------------------
static int recon_kind(int flag_acu, int flag_weno) {
    if (flag_acu == 0) return R_FIRST;
    if (flag_acu == 1) return R_MUSCL;
    switch (flag_weno) {
        case 1: return R_WENO3Z;
        case 2: return R_WENO5JS;
        case 3: return R_WENO5Z;
        case 4: return R_WENO7Z;
        default: return -1;
    }
}

template <int NSP, bool SPH, int RK>
static hipError_t launch_flux_slice(const FluxArgs &a, hipStream_t st) {
    const long n = long(a.nblk) * (a.ncell + 1);
    const dim3 grid(unsigned((n + 31) / 32)), blk(64 * GW);     // 32 interfaces, both sides, per workgroup
    switch (a.riemann) {
        case 0: hipLaunchKernelGGL((k_flux<NSP, RK, SPH, 0>), grid, blk, 0, st, a); break;
        case 1: hipLaunchKernelGGL((k_flux<NSP, RK, SPH, 1>), grid, blk, 0, st, a); break;
        default:
            if constexpr (RK == R_WENO5JS || RK == R_WENO5Z)
                if (a.variant == 1) { hipLaunchKernelGGL((k_flux<NSP, RK, SPH, 2, 4>), grid, blk, 0, st, a); break; }
            hipLaunchKernelGGL((k_flux<NSP, RK, SPH, 2>), grid, blk, 0, st, a);
            break;
    }
    return hipGetLastError();
}

// Launches of the blocks b0 .. b0 + nblk - 1 (the coarse blocks of a refined mesh reconstruct at first order in
// launches of their own, SRC/flux.f90:240) over slices of them, and of a block alone where it is longer than a slice: the cells between its interfaces j and
// j + n are a block of their own to the kernel.
template <int NSP, bool SPH, int RK>
static hipError_t launch_flux_rk(const FluxArgs &whole, hipStream_t st) {
    return for_slices(whole.nblk, whole.S, SLICE, [&](int b, int n) {
        FluxArgs a = whole;
        const long blk = a.b0 + b;
        a.qf += blk * a.S;
        a.F += blk * (a.ncell + 1);
        if (a.godunov) a.godunov += blk * (a.ncell + 1);
        a.nblk = n;
        if (a.S <= SLICE) return launch_flux_slice<NSP, SPH, RK>(a, st);
        return for_slices(whole.ncell + 1, 1, SLICE, [&](int j, int m) {
            FluxArgs p = a;
            p.qf += j;
            p.F += j;
            if (p.godunov) p.godunov += j;
            p.ncell = m - 1;
            return launch_flux_slice<NSP, SPH, RK>(p, st);
        });
    });
}

template <int NSP, bool SPH>
static hipError_t launch_flux_nsp(const FluxArgs &a, int rk, hipStream_t st) {
    switch (rk) {
        case R_FIRST: return launch_flux_rk<NSP, SPH, R_FIRST>(a, st);
        case R_MUSCL: return launch_flux_rk<NSP, SPH, R_MUSCL>(a, st);
        case R_WENO3Z: return launch_flux_rk<NSP, SPH, R_WENO3Z>(a, st);
        case R_WENO5JS: return launch_flux_rk<NSP, SPH, R_WENO5JS>(a, st);
        case R_WENO5Z: return launch_flux_rk<NSP, SPH, R_WENO5Z>(a, st);
        case R_WENO7Z: return launch_flux_rk<NSP, SPH, R_WENO7Z>(a, st);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_smr_halo(const SmrArgs &a, int nsp, hipStream_t st) {
    if (a.nif == 0) return hipSuccess;
    hipLaunchKernelGGL(k_smr_fill, dim3(unsigned((a.nif * a.nequ + 63) / 64)), dim3(64), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid(unsigned((a.nif * 2 * a.lv + 63) / 64)), blk(64);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_smr_qf<N>), grid, blk, 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_flux(const FluxArgs &a, int nsp, int flag_acu, int flag_weno, hipStream_t st) {
    const int rk = recon_kind(flag_acu, flag_weno);
    if (rk < 0) return hipErrorInvalidValue;
#define FCFD_CASE(N) if (nsp == N) return a.spherical ? launch_flux_nsp<N, true>(a, rk, st) : launch_flux_nsp<N, false>(a, rk, st);
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

template <int NSP, int MODE, bool SPH>
static hipError_t launch_stage_end_mode(const StageArgs &whole, hipStream_t st) {
    return for_slices(whole.nblk, whole.S, SLICE, [&](int b, int n) {
        const StageSlice s = stage_slice(whole.nblk, whole.S, b, n);
        StageArgs a = whole;
        const long c = long(s.first) * a.S, f = long(s.first) * (a.ncell + 1);
        if (a.Q0) a.Q0 += c;
        a.Qin += c; a.Qout += c; a.qf += c; a.F += f;
        if (a.god) a.god += f;
        if (a.xm) a.xm += long(s.first) * a.ncell;
        if (a.dxb) a.dxb += s.first;
        a.col0 = s.col0; a.ncol = s.ncol; a.left = s.left; a.right = s.right;
        const dim3 grid((s.ncol + 63u) / 64u), blk(64 * GW);    // 64 columns per workgroup
        if (a.variant == 1) hipLaunchKernelGGL((k_stage_end<NSP, MODE, SPH, 4>), grid, blk, 0, st, a);
        else hipLaunchKernelGGL((k_stage_end<NSP, MODE, SPH>), grid, blk, 0, st, a);
        return hipGetLastError();
    });
}

template <int NSP>
static hipError_t launch_stage_end_nsp(const StageArgs &a, hipStream_t st) {
    if (a.mode == 2) return launch_stage_end_mode<NSP, 2, false>(a, st);
    if (a.spherical) return a.mode == 0 ? launch_stage_end_mode<NSP, 0, true>(a, st) : launch_stage_end_mode<NSP, 1, true>(a, st);
    return a.mode == 0 ? launch_stage_end_mode<NSP, 0, false>(a, st) : launch_stage_end_mode<NSP, 1, false>(a, st);
}

hipError_t launch_stage_end(const StageArgs &a, int nsp, hipStream_t st) {
#define FCFD_CASE(N) if (nsp == N) return launch_stage_end_nsp<N>(a, st);
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_rk4_stage(const StageArgs &a, int nsp, hipStream_t st) {
    const long n = long(a.nblk) * a.S;
    const dim3 grid(unsigned((n + 63) / 64)), blk(64);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_rk4_stage<N>), grid, blk, 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_dt(const DtArgs &a, int nsp, hipStream_t st) {
    const long n = long(a.nblk) * a.ncell;
    const dim3 grid(unsigned(std::min<long>((n + 63) / 64, 2048))), blk(64 * GW);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_wave_speed<N>), grid, blk, 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_init(const InitArgs &a, int nsp, hipStream_t st) {
    const long n = long(a.nblk) * a.ncell;
    const dim3 grid(unsigned((n + 63) / 64)), blk(64);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_init_cells<N>), grid, blk, 0, st, a); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_qf_to_qc(const DevThermo *m, int nsp, int n, const double *qf, double *Qc, long P, hipStream_t st) {
    const dim3 grid(unsigned((n + 63) / 64)), blk(64);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_qf_to_qc<N>), grid, blk, 0, st, m, n, qf, Qc, P); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_qc_to_qf(const DevThermo *m, int nsp, int n, const double *Qc, double *qf, long P, hipStream_t st) {
    const dim3 grid(unsigned((n + 63) / 64)), blk(64);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_qc_to_qf<N>), grid, blk, 0, st, m, n, Qc, qf, P); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_qf_to_qc_interior(const DevThermo *m, int nsp, int nblk, int ncell, int lv, int S,
                                    const double *qf, double *Qc, long P, hipStream_t st) {
    const long n = long(nblk) * ncell;
    const dim3 grid(unsigned((n + 63) / 64)), blk(64 * GW);
#define FCFD_CASE(N) if (nsp == N) { hipLaunchKernelGGL((k_qf_to_qc_interior<N>), grid, blk, 0, st, m, nblk, ncell, lv, S, qf, Qc, P); return hipGetLastError(); }
    FCFD_FOR_EACH_NSP(FCFD_CASE)
#undef FCFD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_recon(int n, const double *s, double *out, hipStream_t st) {
    hipLaunchKernelGGL(k_recon, dim3(unsigned((n + 63) / 64)), dim3(64), 0, st, n, s, out);
    return hipGetLastError();
}

}  // namespace fcfd
