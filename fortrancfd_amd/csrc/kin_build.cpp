// kin_build.cpp -- device kinetics tables from the CHEMKIN-II link-file data (host side).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstdint>
#include <cstring>
#include <vector>

#include "chem.hpp"

namespace fcfd {

// Device rows are the mechanism's reactions re-ordered by kind -- fall-off first, then plain
// third-body, then the remaining reactions whose coefficients exceed 3 in magnitude (or whose
// product coefficients are negative), then the rest, by falling count of exponentials -- so a wave,
// which evaluates 64 consecutive rows at once, runs the fall-off and third-body code paths in as
// few row chunks as possible, and the last group (from row nplain0) can take the branch-free
// evaluation.  Every per-reaction result
// is independent of the row order; only the order of the species-sum additions changes.
void build_dev_kin(const Mech &m, DevKin &k) {
    std::memset(&k, 0, sizeof(DevKin));
    k.ii = m.ii;
    k.kk = m.kk;
    k.nthb = int(m.itb.size());
    k.nfal = int(m.ifl.size());
    k.small = std::pow(10.0, -300);        // CKINIT SMALL / EXPARG (cklib.f:4054-4057)
    k.exparg = std::log(std::pow(10.0, 300));
    std::vector<int> tb_of(m.ii, -1), fo_of(m.ii, -1), order;
    for (int t = 0; t < k.nthb; ++t) tb_of[m.itb[t] - 1] = t;
    for (int f = 0; f < k.nfal; ++f) fo_of[m.ifl[f] - 1] = f;
    // the branch-free rows also store their reactants in slots 0 .. nr-1 and products in 3 .. 3+np-1
    auto small = [&](int i) {
        int sum = 0;
        for (int n = 0; n < 6; ++n) {
            const int v = m.nu[size_t(i) * 6 + n];
            if (v > 3 || v < -3 || (n >= 3 && v < 0)) return false;
            sum += v;
        }
        for (int h = 0; h < 2; ++h)
            for (int n = 1; n < 3; ++n)
                if (m.nk[size_t(i) * 6 + 3 * h + n] > 0 && m.nk[size_t(i) * 6 + 3 * h + n - 1] <= 0) return false;
        return sum >= -3 && sum <= 3 && m.nk[size_t(i) * 6] > 0;
    };
    // exponentials a branch-free row evaluates: the Arrhenius factor unless B = E = 0, the
    // equilibrium constant if reversible
    const int np1 = m.npar + 1;
    auto n_exp = [&](int i) {
        const bool arr0 = m.par[size_t(i) * np1 + 1] == 0.0 && m.par[size_t(i) * np1 + 2] == 0.0;
        return (arr0 ? 0 : 1) + (m.ns[i] > 0 ? 1 : 0);
    };
    for (int pass = 0; pass < 6; ++pass) {
        if (pass == 3) k.nplain0 = int(order.size());
        for (int i = 0; i < m.ii; ++i) {
            const int kind = fo_of[i] >= 0 ? 0 : (tb_of[i] >= 0 ? 1 : (small(i) ? 3 : 2));
            // the branch-free rows by falling cost, so that the waves that share a chunk of rows
            // (and its barriers) get rows of equal cost
            if (kind == 3 ? pass == 5 - n_exp(i) : kind == pass) order.push_back(i);
        }
    }
    for (int r = 0; r < m.ii; ++r) {
        const int i = order[r];
        k.orig[r] = i;
        k.A[r] = m.par[size_t(i) * np1 + 0];
        k.B[r] = m.par[size_t(i) * np1 + 1];
        k.E[r] = m.par[size_t(i) * np1 + 2];
        k.rev[r] = m.ns[i] > 0 ? 1 : 0;
        k.arr0[r] = (k.B[r] == 0.0 && k.E[r] == 0.0) ? 1 : 0;
        int s = 0;
        for (int n = 0; n < 6; ++n) {
            k.nu[r][n] = m.nu[size_t(i) * 6 + n];
            k.nk[r][n] = m.nk[size_t(i) * 6 + n] - 1;
            s += k.nu[r][n];
        }
        k.nus[r] = s;
        k.tb[r] = tb_of[i];
        k.fo[r] = fo_of[i];
    }
    // lists of the lane-per-cell kernels, over the device rows
    int ne = 0, ns = 0;
    const int nchunk = (m.ii + LANE_CHUNK - 1) / LANE_CHUNK;
    for (int c = 0; c < nchunk; ++c) {
        std::vector<std::vector<LaneEnt>> of(size_t(m.kk));
        for (int r = 0; r < LANE_CHUNK && c * LANE_CHUNK + r < m.ii; ++r)
            for (int n = 0; n < 6; ++n) {
                const int row = c * LANE_CHUNK + r, sp = k.nk[row][n];
                if (sp >= 0) of[size_t(sp)].push_back(LaneEnt{double(k.nu[row][n]), r * LANE_NC * 8, 0});
            }
        std::vector<int> order;
        for (int sp = 0; sp < m.kk; ++sp)
            if (!of[size_t(sp)].empty()) order.push_back(sp);
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return of[size_t(x)].size() > of[size_t(y)].size(); });
        std::vector<int> mine[LANE_RW];
        size_t load[LANE_RW] = {};
        for (int sp : order) {
            const int w = int(std::min_element(load, load + LANE_RW) - load);
            mine[w].push_back(sp);
            load[w] += of[size_t(sp)].size() + 2;
        }
        for (int w = 0; w < LANE_RW; ++w) {
            k.lane_seg0[c * LANE_RW + w] = ns;
            for (int sp : mine[w]) {
                k.lane_seg[ns++] = LaneSeg{sp * LANE_NC * 8, ne, int(of[size_t(sp)].size())};
                for (const LaneEnt &e : of[size_t(sp)]) k.lane_ent[ne++] = e;
            }
        }
    }
    k.lane_seg0[nchunk * LANE_RW] = ns;
    for (int r = k.nplain0; r < m.ii; ++r) {
        LanePlain &p = k.lane_plain[r];
        p.A = k.A[r];
        p.B = k.B[r];
        p.E = k.E[r];
        int pw = 0, big = 0;
        for (int n = 0; n < 6; ++n) {
            const int sp = k.nk[r][n];
            p.nud[n] = sp >= 0 ? double(k.nu[r][n]) : 0.0;
            p.off[n] = (sp >= 0 ? sp : m.kk) * LANE_NC * 8;
            const int a = k.nu[r][n] < 0 ? -k.nu[r][n] : k.nu[r][n];
            pw |= (sp >= 0 ? a : 0) << (2 * n);
            if (sp >= 0 && a > 1) big = 1;
        }
        p.bits = (k.rev[r] ? LP_REV : 0) | (k.arr0[r] ? LP_ARR0 : 0) |
                 ((k.nus[r] + 3) << LP_NUS) | (big ? LP_POW : 0) | (pw << LP_PW) | (k.nu[r][0] == 0 ? LP_DEAD : 0);
    }
    for (int t = 0; t < k.nthb; ++t) {
        k.ntbs[t] = m.ntbs[t];
        for (int l = 0; l < m.mxtb && l < MAXTB; ++l) {
            k.tbk[t][l] = m.nktb[size_t(t) * m.mxtb + l] - 1;
            k.tba[t][l] = m.aik[size_t(t) * m.mxtb + l];
        }
    }
    for (int f = 0; f < k.nfal; ++f) {
        k.ifop[f] = m.ifo[f];
        k.kfal[f] = m.kfl[f] - 1;
        for (int c = 0; c < 8 && c < m.nfar; ++c) k.fpar[f][c] = m.fpar[size_t(f) * m.nfar + c];
    }
}

void build_coop_lists(DevKin &k, std::vector<unsigned> &jac) {
    const int ii = k.ii, nb = (ii + 63) / 64;
    bool fits = ii <= COOP_MAXR && k.kk < COOP_EMPTY && k.nfal <= COOP_FAL;
    auto usual = [](double v) { return v == 0.0 || (std::fabs(v) >= 0x1p-700 && std::fabs(v) <= 0x1p60); };
    k.usual = 1;
    for (int f = 0; f < k.nfal; ++f)
        if (!usual(k.fpar[f][2]) || !usual(k.fpar[f][6])) k.usual = 0;
    for (int r = 0; r < ii; ++r)
        if (!usual(k.E[r]) || !(std::fabs(k.E[r]) <= 0x1p22 && std::fabs(k.B[r]) <= 0x1p20)) k.usual = 0;
    fits = fits && k.usual;
    for (int r = 0; r < ii; ++r) {
        const int *nu = k.nu[r], *nk = k.nk[r];
        fits = fits && std::abs(k.nus[r]) <= 3 && nk[0] >= 0 && nk[3] >= 0 && (nk[1] >= 0 || nk[2] < 0) &&
               (nk[4] >= 0 || nk[5] < 0) && (k.tb[r] < 0 || k.ntbs[k.tb[r]] <= COOP_TB);
        bool pow = false;
        unsigned w[4] = {0, 0, 0, 0};
        for (int n = 0; n < 6; ++n) {
            fits = fits && std::abs(nu[n]) <= 3 && (n < 3 || nu[n] >= 0) && (nk[n] >= 0 || nu[n] == 0);
            pow = pow || std::abs(nu[n]) > 1;
            w[n / 4] |= unsigned(nk[n] >= 0 ? nk[n] : COOP_EMPTY) << (8 * (n % 4));
            w[2] |= (unsigned(nu[n]) & 15u) << (8 + 4 * n);
        }
        w[2] |= (k.rev[r] ? CR_REV : 0u) | (k.arr0[r] ? CR_ARR0 : 0u) | (pow ? CR_POW : 0u) |
                (unsigned(k.nus[r] + 3) & 7u) << CR_NUS;
        w[3] = unsigned(k.tb[r] + 1) | unsigned(k.fo[r] + 1) << 16;
        for (int n = 0; n < 4; ++n) k.coop_row[n][r] = w[n];
        const int t = k.tb[r];
        for (int l = 0; l < COOP_TB; ++l) {
            const bool on = t >= 0 && l < k.ntbs[t];
            if (l % 4 == 0) k.coop_tbk[l / 4][r] = 0;
            k.coop_tbk[l / 4][r] |= unsigned(on ? std::max(k.tbk[t][l], 0) : COOP_EMPTY) << (8 * (l % 4));
            k.coop_tba[l][r] = on ? k.tba[t][l] - 1.0 : 0.0;
        }
    }
    k.coop = fits ? 1 : 0;
    if (!fits) return;
    auto group = [](int b) { return b == 0 ? 0 : 1 + (b - 1) % 3; };
    // production rates, and the creation / destruction split
    auto place = [](int r, int nu) {
        const int m = std::abs(nu);
        return (unsigned short)((m == 0 ? COOP_MAXR : COOP_AT(m) + r) << 3);
    };
    const unsigned short pad = place(0, 0);
    int at = 0;
    for (int g = 0; g < 4; ++g) {
        std::vector<std::vector<unsigned short>> sum(64), split(64);
        for (int b = 0; b < nb; ++b) {
            if (group(b) != g) continue;
            const int r0 = b * 64, r1 = std::min(ii, r0 + 64);
            for (int n = 0; n < 6; ++n)
                for (int r = r0; r < r1; ++r)
                    if (k.nk[r][n] >= 0) sum[k.nk[r][n]].push_back((unsigned short)(place(r, k.nu[r][n]) | (k.nu[r][n] < 0 ? 0x8000 : 0)));
            for (int n = 0; n < 3; ++n)
                for (int half = 0; half < 2; ++half)
                    for (int r = r0; r < r1; ++r) {
                        const int s = n + 3 * half;
                        if (k.nk[r][s] >= 0)
                            split[k.nk[r][s]].push_back((unsigned short)(place(r, k.nu[r][s]) | half << 15));
                    }
        }
        for (int s = 0; s < 64; ++s) {
            while (sum[s].size() % 4) {
                sum[s].push_back(pad);
                split[s].push_back(pad);
            }
            k.sum_off[g][s] = (unsigned short)at;
            k.sum_len[g][s] = (unsigned short)sum[s].size();
            for (size_t e = 0; e < sum[s].size(); ++e, ++at) {
                k.coop_sum[at] = sum[s][e];
                k.coop_split[at] = split[s][e];
            }
        }
    }
    // Jacobian entries d(wdot_r) / d(c_c) = sum nu[t] dq[s] over slots t holding r and s holding c
    auto upper16 = [](int v) {
        const double d = v;
        uint64_t b;
        std::memcpy(&b, &d, sizeof b);
        return unsigned(b >> 32) & 0xffff0000u;      // (small whole numbers: all other bits are 0)
    };
    struct Entry { unsigned dst; std::vector<unsigned> e[4]; size_t steps; };
    std::vector<Entry> all(size_t(k.kk) * k.kk);
    for (int b = 0; b < nb; ++b)
        for (int s = 0; s < 6; ++s)
            for (int t = 0; t < 6; ++t)
                for (int r = b * 64; r < std::min(ii, b * 64 + 64); ++r) {
                    if (k.nu[r][0] == 0 || k.nk[r][s] < 0 || k.nk[r][t] < 0) continue;
                    all[size_t(k.nk[r][t]) * k.kk + k.nk[r][s]].e[group(b)].push_back(
                        unsigned(s * COOP_MAXR + r) << 3 | upper16(k.nu[r][t]));
                }
    std::vector<Entry> entries;
    for (size_t i = 0; i < all.size(); ++i) {
        all[i].dst = unsigned(i);
        all[i].steps = 0;
        for (auto &g : all[i].e) all[i].steps = std::max(all[i].steps, g.size());
        if (all[i].steps) entries.push_back(all[i]);
    }
    std::stable_sort(entries.begin(), entries.end(), [](const Entry &a, const Entry &b) { return a.steps > b.steps; });
    // Rounds of sixteen entries, longest first, each to the wave with the fewest steps so far.  Waves 1 ..
    // 4 also add up the production rates before: they start with those steps' share.
    constexpr unsigned none = unsigned(6 * COOP_MAXR) << 3;
    std::vector<std::vector<unsigned>> lane(COOP_WAVES * 64);
    size_t load[COOP_WAVES];
    for (int w = 0; w < COOP_WAVES; ++w) {
        load[w] = 0;
        if (w >= 1 && w <= 4)
            for (int s = 0; s < 64; ++s) load[w] = std::max(load[w], size_t(k.sum_len[w - 1][s]));
    }
    std::vector<size_t> ends[COOP_WAVES];
    for (size_t e0 = 0; e0 < entries.size(); e0 += 16) {
        const int w = int(std::min_element(load, load + COOP_WAVES) - load);
        const size_t steps = entries[e0].steps;
        load[w] += steps + 2;
        for (int i = 0; i < 16; ++i) {
            const Entry *en = e0 + i < entries.size() ? &entries[e0 + i] : nullptr;
            for (int g = 0; g < 4; ++g) {
                std::vector<unsigned> &l = lane[w * 64 + i * 4 + g];
                for (size_t e = 0; e < steps; ++e) l.push_back(en && e < en->e[g].size() ? en->e[g][e] : none);
                l.push_back(en ? en->dst : JE_NONE);
            }
        }
        ends[w].push_back(lane[w * 64].size() - 1);
    }
    for (int w = 0; w < COOP_WAVES; ++w) {
        const size_t mx = std::max<size_t>((lane[w * 64].size() + 7) / 8 * 8, 8);      // the kernel loads eight steps at a time
        k.coop = k.coop && mx <= COOP_JAC ? 1 : 0;
        if (!k.coop) return;
        k.jac_steps[w] = int(mx);
        k.jac_off[w] = int(jac.size());
        std::memset(k.jac_end[w], 0, sizeof k.jac_end[w]);
        for (size_t e : ends[w]) k.jac_end[w][e / 8] |= (unsigned char)(1u << (e % 8));
        jac.resize(jac.size() + mx * 64, none);
        for (int i = 0; i < 64; ++i)
            for (size_t e = 0; e < lane[w * 64 + i].size(); ++e) jac[k.jac_off[w] + e / 8 * 512 + i * 8 + e % 8] = lane[w * 64 + i][e];
    }
}

// Values that follow from the tables: CKHMS(298.15) (cklib.f:3598-3618), the formation enthalpies of
// the heat-release diagnostics; 1 / wt; the coefficient sets by temperature class.
void thermo_derived(DevThermo &t) {
    for (int k = 0; k < t.kk; ++k) t.rwt[k] = 1.0 / t.wt[k];
    const int M = (t.kk + SPECIES_BLOCKS - 1) / SPECIES_BLOCKS;
    for (int w = 0; w < SPECIES_BLOCKS; ++w) {
        const int k0 = std::min(w * M, t.kk), k1 = std::min(k0 + M, t.kk);
        std::vector<double> cut(t.tmid + k0, t.tmid + k1);
        std::sort(cut.begin(), cut.end());
        cut.erase(std::unique(cut.begin(), cut.end()), cut.end());
        t.nclass[w] = int(cut.size()) < MAXCLS ? int(cut.size()) + 1 : 0;
        for (int c = 0; c < t.nclass[w]; ++c) {
            if (c > 0) t.cut[w][c - 1] = cut[c - 1];
            for (int k = k0; k < k1; ++k) {
                const bool up = c > 0 && cut[c - 1] >= t.tmid[k];      // T > cut[c - 1] >= tmid
                for (int i = 0; i < 6; ++i) t.coef[w][c][k - k0][i] = up ? t.ahi[k][i] : t.alo[k][i];
            }
        }
    }
    const double T = 298.15, rut = T * t.ru;
    const double t2 = T * T, t3 = T * t2, t4 = t2 * t2;
    const double tn1 = T / 2.0, tn2 = t2 / 3.0, tn3 = t3 / 4.0, tn4 = t4 / 5.0;
    for (int k = 0; k < t.kk; ++k) {
        const double *a = T > t.tmid[k] ? t.ahi[k] : t.alo[k];
        double s = a[0];
        s = s + tn1 * a[1];
        s = s + tn2 * a[2];
        s = s + tn3 * a[3];
        s = s + tn4 * a[4];
        t.h298[k] = rut * (s + a[5] / T) / t.wt[k];
    }
}

}  // namespace fcfd
