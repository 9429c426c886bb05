// surrogate.hip -- host side of the chemistry surrogate: parameter and workspace management,
// the forward / backward / update sequence of one training step, batched inference with FP64
// fallback, and the surrogate branch of solve_source.  All work is stream-ordered and
// allocation-free once the workspace is sized, so a solve_source with the surrogate can be
// captured in a HIP graph.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/fcfd.h"
#include "chem.hpp"
#include "fcfd_common.hpp"
#include "surrogate_impl.hpp"

namespace fcfd {

void set_error(const std::string &msg);

namespace {

constexpr float ADAM_B1 = 0.9f, ADAM_B2 = 0.999f, ADAM_EPS = 1.0e-8f;

long wsize(int l) { return long(MLP_K[l]) * MLP_N[l]; }

// Split-K factor for a weight-gradient GEMM with `tiles` output tiles and K = rows: about 256
// workgroups, each K slice a multiple of 16 rows.
int choose_split(int rows, int tiles) {
    int s = std::max(1, 256 / tiles);
    while (s > 1 && rows % (s * 16) != 0) --s;
    return s;
}

template <class T>
hipError_t grow(T *&p, size_t &cap, size_t n) {
    if (n <= cap) return hipSuccess;
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    hipError_t e = hipMalloc(&p, n * sizeof(T));
    if (e == hipSuccess) cap = n;
    return e;
}

}  // namespace

hipError_t Surrogate::reserve(int rows, bool training) {
    hipError_t e;
    const size_t r = size_t(rows);
    if ((e = grow(X, capX, r * MLP_INP)) != hipSuccess) return e;
    if ((e = grow(Yh, capYh, r * MLP_OUTP)) != hipSuccess) return e;
    if ((e = grow(in_range, capIR, r)) != hipSuccess) return e;
    if ((e = grow(fb_list, capFB, r)) != hipSuccess) return e;
    if ((e = grow(stiff, capST, r)) != hipSuccess) return e;
    if ((e = grow(cand_list, capCL, r)) != hipSuccess) return e;
    if ((e = grow(cand, capCD, r * size_t(mech->host.kk + 1))) != hipSuccess) return e;
    if (!training) return hipSuccess;
    for (int l = 0; l < 4; ++l) {
        if ((e = grow(H[l], capHl[l], r * MLP_HID)) != hipSuccess) return e;
        if ((e = grow(Pre[l], capPre[l], r * MLP_HID)) != hipSuccess) return e;
    }
    if ((e = grow(Yt, capYt, r * MLP_OUTP)) != hipSuccess) return e;
    if ((e = grow(dY, capdY, r * MLP_OUTP)) != hipSuccess) return e;
    for (int i = 0; i < 4; ++i)
        if ((e = grow(dZ[i], capdZ[i], r * MLP_HID)) != hipSuccess) return e;
    if ((e = grow(cs_part, capCS, ((r + 63) / 64) * (4 * MLP_HID + MLP_OUTP))) != hipSuccess) return e;
    if ((e = grow(loss_part, capLP, (r * MLP_OUTP + 255) / 256 + 1)) != hipSuccess) return e;
    return hipSuccess;
}

NetParams Surrogate::params() const {
    NetParams p{};
    int f = 0, r = 0;
    for (int l = 0; l < MLP_LAYERS; ++l) {
        p.K[l] = MLP_K[l]; p.N[l] = MLP_N[l];
        p.W[l] = W32[l]; p.b[l] = b32[l]; p.gW[l] = gW[l]; p.gb[l] = gb[l];
        p.mW[l] = mW[l]; p.vW[l] = vW[l]; p.mb[l] = mb[l]; p.vb[l] = vb[l];
        p.fwd0[l] = f;
        f += int(wsize(l));
    }
    for (int l = MLP_LAYERS - 1; l > 0; --l) {
        p.bwd0[l] = r;
        r += int(wsize(l));
    }
    p.fwd = Wfwd; p.bwd = Wbwd;
    return p;
}

// Forward of `rows` rows of x (rows multiple of 64).  Training keeps every layer's activations and
// pre-activations.
hipError_t Surrogate::forward(const uint16_t *x, int rows, float *out, bool training, hipStream_t st,
                              const unsigned *m_dev, const int *row_live) {
    NetArgs a{};
    a.x = x; a.w = Wfwd; a.rows = rows; a.out = out;
    a.wide = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
    a.m_dev = m_dev; a.row_live = row_live;
    for (int l = 0; l < MLP_LAYERS; ++l) a.bias[l] = b32[l];
    if (training)
        for (int l = 0; l < 4; ++l) { a.H[l] = H[l]; a.P[l] = Pre[l]; }
    return net_forward(a, training, st);
}

hipError_t Surrogate::train(int rows, float lr, hipStream_t st) {
    hipError_t e;
    if ((e = forward(X, rows, Yh, true, st)) != hipSuccess) return e;
    if ((e = mlp_mse(Yh, Yt, dY, rows, loss_part, d_loss, st)) != hipSuccess) return e;
    NetArgs a{};
    a.x = dY; a.w = Wbwd; a.rows = rows; a.wide = 1;
    for (int i = 0; i < 4; ++i) { a.H[i] = dZ[3 - i]; a.P[i] = Pre[3 - i]; }     // from the last hidden layer down
    if ((e = net_backward(a, st)) != hipSuccess) return e;
    NetGrad g{};
    g.rows = rows; g.part = gpart; g.csum = cs_part;
    long p0 = 0, c0 = 0;
    for (int l = 0; l < MLP_LAYERS; ++l) {
        const int tiles = (MLP_K[l] / 64) * (MLP_N[l] / 64);
        g.K[l] = MLP_K[l]; g.N[l] = MLP_N[l];
        g.in[l] = l == 0 ? X : H[l - 1];
        g.z[l] = l == MLP_LAYERS - 1 ? dY : dZ[l];
        g.split[l] = choose_split(rows, tiles);
        g.chunk[l] = rows / g.split[l];
        g.wg[l] = tiles * g.split[l];
        g.part0[l] = p0; g.csum0[l] = c0;
        p0 += long(g.split[l]) * wsize(l);
        c0 += long(rows / 64) * MLP_N[l];
    }
    if ((e = net_gradients(g, st)) != hipSuccess) return e;
    NetParams p = params();
    if (lr > 0.0f) {
        ++step;
        p.lr = lr; p.b1 = ADAM_B1; p.b2 = ADAM_B2; p.eps = ADAM_EPS;
        p.c1 = 1.0f - std::pow(ADAM_B1, float(step));
        p.c2 = 1.0f - std::pow(ADAM_B2, float(step));
    }
    return net_update(p, g, st);
}

hipError_t Surrogate::network(FeatArgs fa, const int *list, const unsigned *list_n, int rows_max, hipStream_t st) {
    fa.norm = d_norm;
    fa.thermo = mech->d_thermo;
    fa.kk = mech->host.kk;
    fa.list = list;
    fa.list_n = list_n;
    fa.X = X;
    fa.in_range = in_range;
    const int rows = int((long(rows_max) + 63) / 64 * 64);
    hipError_t e = mlp_features(fa, rows, st);
    if (e != hipSuccess) return e;
    // rows outside the training range go to the FP64 integrator whatever the network says: tiles of
    // 64 such rows are not evaluated
    return forward(X, rows, Yh, false, st, list_n, in_range);
}

hipError_t Surrogate::accept(ApplyArgs ap, const ChemArgs &ca, const int *list, const unsigned *list_n, int rows_max,
                             hipStream_t st) {
    ap.thermo = mech->d_thermo;
    ap.norm = d_norm;
    ap.ncf = d_ncf;
    ap.mm = mech->host.mm;
    ap.list = list;
    ap.list_n = list_n;
    ap.Yh = Yh;
    ap.in_range = in_range;
    ap.nfallback = d_nfb;
    ap.fallback = fb_list;
    ap.resid_tol = resid_tol;
    ap.t_tol = t_tol;
    ap.n = rows_max;
    ap.ncand = d_ncand;
    ap.cand_list = cand_list;
    ap.cand = cand;
    hipError_t e = launch_zero_u32(d_nfb, st);
    if (e != hipSuccess) return e;
    if ((e = launch_zero_u32(d_ncand, st)) != hipSuccess) return e;
    if ((e = mlp_apply(ap, mech->host.kk, st)) != hipSuccess) return e;
    return launch_chem_verify(ca, mech->host.kk, cand_list, d_ncand, cand, rows_max, fb_list, d_nfb, verify_tol, st);
}

hipError_t Surrogate::fallback(ChemArgs ca, int chem_wg, hipStream_t st) {
    ca.list = fb_list;
    ca.list_n = d_nfb;
    ca.skip_explicit = 1;
    return launch_chem(ca, mech->host.kk, chem_wg, st);
}

Surrogate::~Surrogate() {
    auto f = [](void *p) { if (p) (void)hipFree(p); };
    f(flat);
    for (int l = 0; l < 4; ++l) { f(H[l]); f(Pre[l]); }
    for (int i = 0; i < 4; ++i) f(dZ[i]);
    f(Wfwd); f(Wbwd);
    f(X); f(Yh); f(Yt); f(dY); f(gpart); f(cs_part); f(loss_part); f(d_loss); f(in_range); f(fb_list);
    f(stiff); f(d_stiff_n); f(d_nfb); f(d_norm); f(d_ncf); f(cand_list); f(cand); f(d_ncand);
    if (stream) (void)hipStreamDestroy(stream);
}

}  // namespace fcfd

using namespace fcfd;

#define HIP_TRY(expr)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) {                                                                \
            set_error(std::string(#expr) + ": " + hipGetErrorString(e_));                      \
            return FCFD_E_HIP;                                                                 \
        }                                                                                      \
    } while (0)

extern "C" {

int fcfd_sur_create(const fcfd_mech *m, fcfd_surrogate **out) {
    if (!m || !out) { set_error("fcfd_sur_create: invalid argument"); return FCFD_E_ARG; }
    *out = nullptr;
    if (m->host.kk + 3 != MLP_IN || m->host.kk + 1 != MLP_OUT) {
        set_error("the surrogate network is sized for 53 species");
        return FCFD_E_UNSUPPORTED;
    }
    if (m->host.mm > 8) { set_error("at most 8 elements"); return FCFD_E_UNSUPPORTED; }
    if (int rc = ensure_dev_tables(m)) return rc;
    auto s = std::make_unique<fcfd_surrogate>();
    s->mech = m;
    HIP_TRY(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
    // parameters, gradients and moments: each one array in the order of fcfd_sur_set_params
    const size_t np = size_t(fcfd_sur_nparams());
    HIP_TRY(hipMalloc(&s->flat, 4 * np * 4));
    HIP_TRY(hipMemset(s->flat, 0, 4 * np * 4));
    float *at = s->flat;
    for (int l = 0; l < MLP_LAYERS; ++l) {
        s->W32[l] = at; s->gW[l] = at + np; s->mW[l] = at + 2 * np; s->vW[l] = at + 3 * np;
        at += wsize(l);
        s->b32[l] = at; s->gb[l] = at + np; s->mb[l] = at + 2 * np; s->vb[l] = at + 3 * np;
        at += MLP_N[l];
    }
    size_t gp = 0, nw = 0;               // largest split-K partial sets (see choose_split), weights
    for (int l = 0; l < MLP_LAYERS; ++l) {
        const int tiles = (MLP_K[l] / 64) * (MLP_N[l] / 64);
        gp += size_t(std::max(1, 256 / tiles)) * size_t(wsize(l));
        nw += size_t(wsize(l));
    }
    HIP_TRY(hipMalloc(&s->Wfwd, nw * 2)); HIP_TRY(hipMalloc(&s->Wbwd, nw * 2));
    HIP_TRY(hipMemset(s->Wfwd, 0, nw * 2)); HIP_TRY(hipMemset(s->Wbwd, 0, nw * 2));
    HIP_TRY(hipMalloc(&s->gpart, gp * 4));
    HIP_TRY(hipMalloc(&s->d_loss, 4));
    HIP_TRY(hipMalloc(&s->d_nfb, sizeof(unsigned)));
    HIP_TRY(hipMalloc(&s->d_stiff_n, sizeof(unsigned)));
    HIP_TRY(hipMalloc(&s->d_ncand, sizeof(unsigned)));
    HIP_TRY(hipMalloc(&s->d_norm, sizeof(SurrogateNorm)));
    SurrogateNorm nm{};
    for (int c = 0; c < MLP_INP; ++c) { nm.in_std[c] = 1.0; nm.lo[c] = -1e300; nm.hi[c] = 1e300; }
    for (int c = 0; c < MLP_OUTP; ++c) nm.out_std[c] = 1.0;
    s->h_norm = nm;
    HIP_TRY(hipMemcpy(s->d_norm, &nm, sizeof nm, hipMemcpyHostToDevice));
    const int kk = m->host.kk, mm = m->host.mm;
    std::vector<double> ncf(size_t(kk) * mm);
    for (size_t i = 0; i < ncf.size(); ++i) ncf[i] = double(m->host.ncf[i]);
    HIP_TRY(hipMalloc(&s->d_ncf, ncf.size() * sizeof(double)));
    HIP_TRY(hipMemcpy(s->d_ncf, ncf.data(), ncf.size() * sizeof(double), hipMemcpyHostToDevice));
    *out = s.release();
    return FCFD_OK;
}

void fcfd_sur_free(fcfd_surrogate *s) { delete s; }

int fcfd_sur_nparams(void) {
    int n = 0;
    for (int l = 0; l < MLP_LAYERS; ++l) n += int(wsize(l)) + MLP_N[l];
    return n;
}

int fcfd_sur_set_params(fcfd_surrogate *s, const float *params) {
    if (!s || !params) { set_error("fcfd_sur_set_params: invalid argument"); return FCFD_E_ARG; }
    const size_t np = size_t(fcfd_sur_nparams());
    HIP_TRY(hipMemcpyAsync(s->flat, params, np * 4, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemsetAsync(s->flat + 2 * np, 0, 2 * np * 4, s->stream));
    HIP_TRY(net_pack(s->params(), s->stream));
    s->step = 0;
    HIP_TRY(hipStreamSynchronize(s->stream));
    return FCFD_OK;
}

int fcfd_sur_get_params(fcfd_surrogate *s, float *params) {
    if (!s || !params) { set_error("fcfd_sur_get_params: invalid argument"); return FCFD_E_ARG; }
    HIP_TRY(hipMemcpyAsync(params, s->flat, size_t(fcfd_sur_nparams()) * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return FCFD_OK;
}

int fcfd_sur_get_grads(fcfd_surrogate *s, float *grads) {
    if (!s || !grads) { set_error("fcfd_sur_get_grads: invalid argument"); return FCFD_E_ARG; }
    const size_t np = size_t(fcfd_sur_nparams());
    HIP_TRY(hipMemcpyAsync(grads, s->flat + np, np * 4, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return FCFD_OK;
}

int fcfd_sur_set_norm(fcfd_surrogate *s, const double *norm) {
    if (!s || !norm) { set_error("fcfd_sur_set_norm: invalid argument"); return FCFD_E_ARG; }
    SurrogateNorm nm{};
    std::memcpy(&nm, norm, sizeof nm);
    for (int c = 0; c < MLP_INP; ++c)
        if (!(nm.in_std[c] > 0.0)) { set_error("fcfd_sur_set_norm: input scales must be positive"); return FCFD_E_ARG; }
    for (int c = 0; c < MLP_OUTP; ++c)
        if (!(nm.out_std[c] > 0.0)) { set_error("fcfd_sur_set_norm: output scales must be positive"); return FCFD_E_ARG; }
    s->h_norm = nm;
    HIP_TRY(hipMemcpy(s->d_norm, &nm, sizeof nm, hipMemcpyHostToDevice));
    return FCFD_OK;
}

int fcfd_sur_set_thresholds(fcfd_surrogate *s, double resid_tol, double t_tol, double verify_tol) {
    if (!s || !(resid_tol > 0.0) || !(t_tol > 0.0) || !(verify_tol > 0.0)) { set_error("fcfd_sur_set_thresholds: invalid argument"); return FCFD_E_ARG; }
    s->resid_tol = resid_tol;
    s->t_tol = t_tol;
    s->verify_tol = verify_tol;
    return FCFD_OK;
}

int fcfd_sur_features(fcfd_surrogate *s, int n, const double *rho, const double *dt, const double *T,
                      const double *Y, void *X, int *in_range, void *stream) {
    if (!s || n < 1 || !rho || !dt || !T || !Y || !X) { set_error("fcfd_sur_features: invalid argument"); return FCFD_E_ARG; }
    hipStream_t st = static_cast<hipStream_t>(stream);
    FeatArgs f{};
    f.norm = s->d_norm; f.thermo = s->mech->d_thermo; f.kk = s->mech->host.kk; f.layout = 1;
    f.n = n; f.npad = int((long(n) + 63) / 64 * 64);
    f.rho = rho; f.dtv = dt; f.T = T; f.Y = Y;
    f.X = static_cast<uint16_t *>(X); f.in_range = in_range;
    HIP_TRY(mlp_features(f, f.npad, st));
    HIP_TRY(hipStreamSynchronize(st));
    return FCFD_OK;
}

int fcfd_sur_targets(fcfd_surrogate *s, int n, const double *T0, const double *Y0, const double *T1,
                     const double *Y1, float *Tg, void *stream) {
    if (!s || n < 1 || !T0 || !Y0 || !T1 || !Y1 || !Tg) { set_error("fcfd_sur_targets: invalid argument"); return FCFD_E_ARG; }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int npad = int((long(n) + 63) / 64 * 64);
    HIP_TRY(mlp_targets(s->d_norm, s->mech->host.kk, n, npad, T0, Y0, T1, Y1, Tg, st));
    HIP_TRY(hipStreamSynchronize(st));
    return FCFD_OK;
}

int fcfd_sur_forward(fcfd_surrogate *s, int rows, const void *X, float *Yh, void *stream) {
    if (!s || rows < 64 || rows % 64 || !X || !Yh) { set_error("fcfd_sur_forward: rows must be a positive multiple of 64"); return FCFD_E_ARG; }
    hipStream_t st = static_cast<hipStream_t>(stream);
    HIP_TRY(s->forward(static_cast<const uint16_t *>(X), rows, Yh, false, st));
    HIP_TRY(hipStreamSynchronize(st));
    return FCFD_OK;
}

int fcfd_sur_train_step(fcfd_surrogate *s, const void *X_all, const float *Tg_all, const int *idx, int batch,
                        float lr, float *loss, void *stream) {
    if (!s || !X_all || !Tg_all || !idx || batch < 64 || batch % 64 || !(lr >= 0.0f)) {
        set_error("fcfd_sur_train_step: invalid argument (batch must be a positive multiple of 64)");
        return FCFD_E_ARG;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    HIP_TRY(s->reserve(batch, true));
    HIP_TRY(mlp_gather_bf16(static_cast<const uint16_t *>(X_all), s->X, idx, batch, MLP_INP, st));
    HIP_TRY(mlp_gather_f32(Tg_all, s->Yt, idx, batch, MLP_OUTP, st));
    HIP_TRY(s->train(batch, lr, st));
    if (loss) {
        HIP_TRY(hipMemcpyAsync(loss, s->d_loss, 4, hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        *loss /= float(batch) * float(MLP_OUT);
    }
    return FCFD_OK;
}

int fcfd_sur_infer_batch(fcfd_surrogate *s, const fcfd_opts *o, int n, const double *rho, const double *dt,
                         double *T, double *Y, int *accepted, int *n_fallback, int *stats, void *stream) {
    if (!s || !o || n < 1 || !rho || !dt || !T || !Y) { set_error("fcfd_sur_infer_batch: invalid argument"); return FCFD_E_ARG; }
    if (!(o->rtol > 0.0 && o->atol > 0.0)) { set_error("fcfd_sur_infer_batch: atol and rtol must be positive"); return FCFD_E_ARG; }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int npad = int((long(n) + 63) / 64 * 64);
    HIP_TRY(s->reserve(npad, false));
    ChemArgs ca{};
    ca.thermo = s->mech->d_thermo; ca.kin = static_cast<const DevKin *>(s->mech->d_kin); ca.counter = s->mech->d_counter;
    ca.coop = s->mech->coop;
    ca.ncells = n; ca.rtol = o->rtol; ca.atol = o->atol;
    ca.b_rho = rho; ca.b_dt = dt; ca.b_T = T; ca.b_y = Y;
    ca.stats = reinterpret_cast<ChemCellStats *>(stats);
    ca.layout = 1;
    ca.route = accepted;
    HIP_TRY(launch_zero_u32(s->d_stiff_n, st));
    ca.stiff = s->stiff; ca.stiff_n = s->d_stiff_n;
    HIP_TRY(launch_chem_screen(ca, s->mech->host.kk, st));
    FeatArgs fa{};
    fa.layout = 1; fa.n = n; fa.rho = rho; fa.dtv = dt; fa.T = T; fa.Y = Y;
    HIP_TRY(s->network(fa, s->stiff, s->d_stiff_n, n, st));
    ApplyArgs ap{};
    ap.layout = 1; ap.rho = rho; ap.T = T; ap.Y = Y; ap.route = accepted;
    HIP_TRY(s->accept(ap, ca, s->stiff, s->d_stiff_n, n, st));
    HIP_TRY(s->fallback(ca, chem_workgroups(s->mech), st));
    if (n_fallback) {
        unsigned nf = 0;
        HIP_TRY(hipMemcpyAsync(&nf, s->d_nfb, sizeof nf, hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        *n_fallback = int(nf);
    }
    HIP_TRY(hipStreamSynchronize(st));
    return FCFD_OK;
}

int fcfd_bf16_gemm(int M, int N, int K, const void *A, long sam, long sak, const void *B, long sbk, long sbn,
                   float *C, long ldc, int ksplit, void *stream) {
    if (!A || !B || !C || M < 64 || N < 64 || K < 16 || ksplit < 1) { set_error("fcfd_bf16_gemm: invalid argument"); return FCFD_E_ARG; }
    GemmArgs g{};
    g.A = static_cast<const uint16_t *>(A); g.B = static_cast<const uint16_t *>(B);
    g.sam = sam; g.sak = sak; g.sbk = sbk; g.sbn = sbn; g.M = M; g.N = N; g.K = K; g.ksplit = ksplit;
    g.C32 = C; g.ldc = ldc;
    hipError_t e = launch_gemm(g, static_cast<hipStream_t>(stream));
    if (e == hipErrorInvalidValue) { set_error("fcfd_bf16_gemm: M, N must be multiples of 64 and K / ksplit a multiple of 16"); return FCFD_E_ARG; }
    HIP_TRY(e);
    HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    return FCFD_OK;
}

}  // extern "C"
