// chem.hpp -- kinetics tables and launchers of the chemistry source kernels (chem.hip).
#pragma once

#include "fcfd_common.hpp"

namespace fcfd {

constexpr int LANE_NW = 8;       // waves of a lane-per-cell workgroup that share the species
constexpr int LANE_RW = 16;      // waves of it that share the reactions
constexpr int LANE_CHUNK = 7 * LANE_RW;   // reaction rows between two barriers (seven per wave)
constexpr int LANE_NC = 64;      // cells per workgroup of the lane-per-cell kernels

// A row of the branch-free range (nplain0 .. ii-1) as the lane-per-cell kernels read it, with one
// row index for the whole wave: coefficients as doubles, and the species of each slot as the byte
// offset k * LANE_NC * 8 of its row in a species-major [k][LANE_NC] LDS block (an empty slot: coefficient 0,
// the row after the last species).
struct LanePlain {
    double A, B, E;
    double nud[6];
    int off[6];
    int bits;                    // LP_* fields
};
// LanePlain::bits
constexpr int LP_REV = 1 << 4;   // reverse rate from the equilibrium constant
constexpr int LP_ARR0 = 1 << 5;  // B = E = 0
constexpr int LP_NUS = 6;        // bits 6-8: coefficient sum + 3
constexpr int LP_POW = 1 << 9;   // some slot has |coefficient| > 1
constexpr int LP_PW = 10;        // bits 10-21: |coefficient| of slot n in bits 10 + 2n .. 11 + 2n
constexpr int LP_DEAD = 1 << 22; // coefficient of slot 0 is 0: no rate
// The lane-per-cell kernels' sums: a segment is one species' terms of a chunk, n entries from e0 on, added to
// the production rate at byte offset off; an entry is a rate's byte offset in the chunk's block and the
// coefficient.
struct LaneSeg {
    int off, e0, n;
};
struct LaneEnt {
    double nu;
    int off, pad;
};

// ---- tables of the integrator that gives a cell eight waves (chem_coop.hip) ----
constexpr int COOP_WAVES = 8;        // waves per cell
constexpr int COOP_MAXR = 384;       // reactions: six waves of one row per lane
constexpr int COOP_LIST = COOP_MAXR * 6 + 4 * 64 * 3;      // list entries, padding included
constexpr int COOP_TB = 8;           // enhanced third bodies of a row
constexpr int COOP_FAL = 32;         // fall-off rows: two lanes of a wave each
constexpr int COOP_EMPTY = 63;       // species index of an empty slot (concentration 1, coefficient 0)
constexpr unsigned CR_REV = 1, CR_ARR0 = 2;   // DevKin::coop_row[2]: reversible; B = E = 0
constexpr unsigned CR_POW = 4;       // some |coefficient| is 2 or 3
constexpr int CR_NUS = 4;            // bits 4-6: coefficient sum + 3
constexpr unsigned JE_NONE = 0xffff;
constexpr int COOP_JAC = 1024;       // steps of a wave
// Doubles per rate array: a place for each row and one that stays 0.  The arrays of 1, 2 and 3 times the
// rates start at COOP_AT(1), (2), (3) of one LDS array, which holds the fall-off terms in between.
constexpr int COOP_Q = COOP_MAXR + 1;
constexpr int COOP_AT(int m) { return m == 1 ? 0 : (m - 1) * COOP_Q + 2 * COOP_FAL; }

// Reaction data in the form CKRATT / CKRATX / CKWYR consume it (cklib.f:6630-6993, 9107-9204),
// re-indexed 0-based with one row per reaction.
struct DevKin {
    int ii, kk, nthb, nfal;
    int nplain0;                        // rows nplain0 .. ii-1 suit reaction_plain (chem_device.hpp)
    double small, exparg;
    double A[MAXR], B[MAXR], E[MAXR];   // PAR(1..3): A, temperature exponent, E/R
    int rev[MAXR];                      // NSPEC > 0: reverse rate from equilibrium
    int arr0[MAXR];                     // B = E = 0: the rate constant is A (exp(0) = 1)
    int nus[MAXR];                      // sum of the six stoichiometric coefficients
    int nu[MAXR][6], nk[MAXR][6];       // coefficients and 0-based species (-1: empty slot)
    int tb[MAXR], fo[MAXR];             // third-body / fall-off table row, -1 if none
    int ntbs[MAXR], tbk[MAXR][MAXTB];   // enhanced third bodies (species, 0-based)
    double tba[MAXR][MAXTB];            // their efficiencies
    int ifop[MAXR], kfal[MAXR];         // fall-off form (1 Lindemann, 2 SRI, 3/4 Troe), [M] species
    double fpar[MAXR][8];
    int orig[MAXR];                     // the mechanism's (0-based) index of each device row
    // lists of the lane-per-cell kernels (chem_lane.hip): rows are taken in chunks of LANE_CHUNK; after
    // chunk c, wave w sums the segments lane_seg[lane_seg0[c * LANE_RW + w] .. lane_seg0[c * LANE_RW + w +
    // 1]), each in row then slot order.  The species of a chunk go to the waves by their entries, most
    // first.
    int lane_seg0[(MAXR + LANE_CHUNK - 1) / LANE_CHUNK * LANE_RW + 1];
    LaneSeg lane_seg[(MAXR + LANE_CHUNK - 1) / LANE_CHUNK * 64];
    LaneEnt lane_ent[MAXR * 6];
    int usual;                          // 1: the constants that are divided by T are 0 or in 2^-700 .. 2^60
    LanePlain lane_plain[MAXR];         // rows nplain0 .. ii-1 (other entries unused)
    // Packed rows of the eight-wave integrator: [0] species of slots 0-3, a byte each (COOP_EMPTY: none);
    // [1] those of slots 4 and 5; [2] CR_* and the coefficients as four-bit two's complement in bits
    // 8 + 4 slot; [3] third-body row + 1, fall-off row + 1 in the upper half.
    unsigned coop_row[4][MAXR];
    // Third bodies of a row: species, a byte each (COOP_EMPTY: none), and efficiency - 1 (0)
    unsigned coop_tbk[COOP_TB / 4][MAXR];
    double coop_tba[COOP_TB][MAXR];
    // 1: the mechanism suits that integrator (else its short lists take k_chem's four-wave mode): at most COOP_MAXR rows, |coefficients| and their sums at
    // most 3, no negative product coefficient, no gap before a filled slot, at most COOP_TB third bodies
    // and COOP_FAL fall-off rows, constants that over() may divide by T's reciprocal.
    int coop;
    // Its sums as lists of terms.  Row blocks of 64 form four groups (block 0; every third block from
    // 1, 2, 3), each with a partial sum; within one the terms stand in the order block, slot, row.
    //   coop_sum (production rates): group g's terms of species k are sum_len[g][k] entries from
    //   sum_off[g][k] on, both multiples of four (padded by terms of rate 0).  A row's rate times 1, 2
    //   and 3 stands in LDS; an entry is the place in bits 3-14 and the coefficient's sign in bit 15
    //   coop_split (creation, destruction): place and, in bit 15, product slot (magnitude as above)
    alignas(8) unsigned short coop_sum[COOP_LIST];
    alignas(8) unsigned short coop_split[COOP_LIST];
    unsigned short sum_off[4][64], sum_len[4][64];          // of either list
    //   coop_jac (Jacobian entries): wave w takes jac_steps[w] steps (a multiple of eight), step l of its
    //   lane at [jac_off[w] + 512 (l / 8) + 8 lane + l mod 8].  Four neighbouring lanes work on one entry, lane mod 4 on its
    //   group's partial sum; the sixteen entries of a wave end at the same step.  A step: slot *
    //   COOP_MAXR + row of the derivative in bits 3-14 (6 * COOP_MAXR: none), the upper half of the
    //   coefficient as a double in bits 16-31; or, where jac_end[w] has its bit set, the place r * kk + c
    //   of the finished entry (JE_NONE: none).  A device buffer of the mechanism.
    const unsigned *coop_jac;
    int jac_steps[COOP_WAVES], jac_off[COOP_WAVES];
    unsigned char jac_end[COOP_WAVES][COOP_JAC / 8];        // bit u of byte b: step 8 b + u
};

// Fills the eight-wave integrator's tables of k; jac receives coop_jac's contents.
void build_coop_lists(DevKin &k, std::vector<unsigned> &jac);
void build_dev_kin(const Mech &m, DevKin &k);

// Per-cell integrator counters (optional output).
struct ChemCellStats {
    int steps, rejects, newton, failed;
};

struct ChemArgs {
    const DevThermo *thermo;
    const DevKin *kin;
    unsigned int *counter;       // work-queue head, zeroed before launch
    int ncells;
    double rtol, atol;
    // layout A (solve_source): primitive state of a padded SoA domain, updated in place
    double *qf;
    long P;
    int ncell, lv, S;
    double dt;
    const double *dt_dev;        // device dt (overrides dt when non-null)
    double *hrr, *hrr_dot;       // per interior cell (may be null)
    // layout B (batched cells): arrays of length ncells; y is [KK][ncells]
    const double *b_rho, *b_dt;
    double *b_T, *b_y;
    ChemCellStats *stats;        // may be null
    // optional work list: cells list[0 .. *list_n) instead of 0 .. ncells (both device memory)
    const int *list;
    const unsigned *list_n;
    int skip_explicit;           // 1: the explicit pre-step already failed for every listed cell
    // explicit screen output: cells that need the implicit integrator (list + length)
    int *stiff;
    unsigned *stiff_n;
    int *route;                  // optional per-cell route: 2 explicit step over dt, 3 two explicit half
                                 // steps, 1 surrogate, 0 implicit (SDIRK) integrator
    int layout;                  // 0: domain, 1: batch
    int coop;                    // 1: the mechanism suits the eight-wave integrator (fcfd_mech::coop)
    int coop_max;                // set by launch_chem: lists up to this length run several waves per cell
    // optional (domain layout with stats): buffer of the list's capacity that receives the list
    // reordered with the cells whose previous integration took the most attempts first
    int *order;
    // optional (domain layout): per interior cell, the integrator's last step-size proposal, carried
    // from one call to the next (0: none; the screen and the surrogate reset it for cells they finish)
    double *hmem;
    // optional (domain layout): set by k_chem_retry to 1 when every listed cell has already failed
    // the explicit half-step retry (k_chem then goes straight to its implicit steps), else 0
    int *retry_done;
    // optional (domain layout): f at the start state of each cell the explicit screen rejects,
    // [NSP + 1][ncells] (species, then T); k_chem_retry starts from it instead of evaluating it again
    double *f0;
};

// SDIRK integrator over all cells or over a work list (persistent grid): one cell per wave for long
// lists, one cell per workgroup for short ones: eight waves (launch_chem_coop), or four for a mechanism
// beyond that kernel's tables.
hipError_t launch_chem_coop(const ChemArgs &a, int nsp, int nwg, hipStream_t st);
hipError_t launch_chem(const ChemArgs &a, int nsp, int n_workgroups, hipStream_t st);
// Lane-per-cell explicit screen over cells 0 .. ncells: accepted cells are final, the others are
// appended to a.stiff (a.stiff_n must be zero before the launch).
hipError_t launch_chem_screen(const ChemArgs &a, int nsp, hipStream_t st);
// Lane-per-cell explicit half-step retry of the list a.list[0 .. *a.list_n) when it is longer than
// a.coop_max: accepted cells are final, the others go to a.stiff (a.stiff_n must be zero before
// the launch) and *a.retry_done = 1; a shorter list is copied to a.stiff unchanged, *a.retry_done = 0.
hipError_t launch_chem_retry(const ChemArgs &a, int nsp, hipStream_t st);
// Longest list that gets eight waves per cell: the tuned factor (default 8) times the workgroup count
// (api.hip).
int chem_coop_max(int n_workgroups, int nsp);
// The same for these cells: a sixth of it, 1,706 cells by default, where a cell gets four waves.  Batches of GRI-3.0 with
// ten third bodies, four waves and one: 1,536 cells 203 and 232 ms, 1,792: 231 and 235, 2,048: 272 and 240; 8,192:
// 869 and 499.  (Eight waves are the faster at every length: 8,192 cells 292 ms and 499, 65,536: 2.08 s and 2.89.)
inline int coop_limit(const ChemArgs &a, int n_workgroups, int nsp) {
    return chem_coop_max(n_workgroups, nsp) / (a.coop ? 1 : 6);
}
hipError_t launch_zero_u32(unsigned *p, hipStream_t st, unsigned *q = nullptr);      // *p = 0, *q = 0
// *out = f * *in on the device (one thread), e.g. the half step of Strang splitting.
hipError_t launch_scale_scalar(const double *in, double *out, double f, hipStream_t st);
// CKWYR / CKCDYR (cklib.f:9107-9204, 1422-1541) on n states with the one-wave integrator's rate code:
// rho [g/cm^3], T [K], Y [n][KK] in; wdot, cdot, ddot [n][KK] (mol/(cm^3 s)) and the rates of
// progress qf, qr [n][II] (mechanism order) out.  One state per wave.
hipError_t launch_rates(const DevThermo *th, const DevKin *K, int nsp, int n, const double *rho, const double *T,
                        const double *Y, double *wdot, double *cdot, double *ddot, double *qf, double *qr,
                        hipStream_t st);
// FP64 verification of surrogate answers for the cells cand_list[0 .. *ncand): accepted when the
// trapezoidal-rule residual Y1 - Y0 - dt/2 (f(Y0) + f(Y1)) of the candidate (Y1, T1) = cand[i],
// weighted by the integrator's tolerances, has an RMS <= tol (1: the integrator's own bar); accepted
// answers are written to the state, the others appended to the fallback list.  One candidate per
// wave (chem.hip).
hipError_t launch_chem_verify(const ChemArgs &a, int nsp, const int *cand_list, const unsigned *ncand,
                              const double *cand, int rows_max, int *fallback, unsigned *nfallback, double tol,
                              hipStream_t st);
// Screen, then SDIRK on the cells the screen rejected; list / list_n are scratch for ncells cells.
hipError_t launch_chem_full(ChemArgs a, int nsp, int n_workgroups, int *list, unsigned *list_n,
                            hipStream_t st);

}  // namespace fcfd
