// surrogate.hpp -- device-side records of the chemistry surrogate and the launchers of mlp.hip.
#pragma once

#include <cstdint>

#include "fcfd_common.hpp"
#include "mlp.hpp"

namespace fcfd {

// Feature / target scaling and the training range (raw feature units), columns as the network's.
struct SurrogateNorm {
    double in_mean[MLP_INP], in_std[MLP_INP];
    double lo[MLP_INP], hi[MLP_INP];
    double out_mean[MLP_OUTP], out_std[MLP_OUTP];
};

// Feature rows (k_features).
struct FeatArgs {
    const SurrogateNorm *norm;
    const DevThermo *thermo;
    int kk, layout;
    int n, npad;                 // cells; rows written when list is null
    const int *list;             // optional: row r <- cell list[r], r < *list_n
    const unsigned *list_n;
    const double *qf;            // layout 0
    long P;
    int ncell, lv, S;
    const double *dt_dev;
    double dt;
    const double *rho, *dtv, *T, *Y;   // layout 1 (Y [KK][n])
    uint16_t *X;
    int *in_range;
};

// Inference epilogue (k_apply): network output -> accepted state or a fallback-list entry.
struct ApplyArgs {
    const DevThermo *thermo;
    const SurrogateNorm *norm;
    const double *ncf;          // [KK][MM] element counts
    int mm, n, layout;          // layout 0: padded SoA domain (qf), 1: batch arrays
    double *qf;
    long P;
    int ncell, lv, S;
    const double *rho;          // layout 1
    double *T, *Y;              // layout 1: T[n], Y[KK][n]
    const int *list;            // optional: row r is cell list[r], r < *list_n (else row = cell < n)
    const unsigned *list_n;
    const float *Yh;            // [rows][MLP_OUTP] normalised network output
    const int *in_range;        // [rows]
    int *route;                 // [n] or null: 1 surrogate accepted, 0 sent to the FP64 integrator
    unsigned *nfallback;        // fallback-list length (zeroed before the launch)
    int *fallback;              // fallback list (cell indices)
    unsigned *ncand;            // candidate-list length (zeroed before the launch)
    int *cand_list;             // candidate cells
    double *cand;               // [candidate][KK + 1]: Y1, T1
    double resid_tol, t_tol;
};

// A pass through the network (mlp_net.hip); rows a multiple of 64.
struct NetArgs {
    const uint16_t *x;           // [rows][64]: features (forward) or the output's gradient (backward)
    const uint16_t *w;           // packed weights (NetParams::fwd or bwd)
    const float *bias[MLP_LAYERS];
    int rows;
    int wide;                    // 1: x and out are aligned to 16 bytes
    float *out;                  // forward: [rows][64]
    // hidden layers, in the order the pass meets them: training's forward writes pre-activations P and
    // activations H, backward reads P and writes the gradients of the pre-activations to H
    uint16_t *H[4];
    float *P[4];
    // inference, optional: device count of live rows and, with it, per-row flags; 64-row tiles past the
    // count or without a flag set are not evaluated, their output rows left as they were
    const unsigned *m_dev;
    const int *row_live;
};
hipError_t net_forward(const NetArgs &a, bool training, hipStream_t st);
hipError_t net_backward(const NetArgs &a, hipStream_t st);

// Weight and bias gradients: inputs and output gradients of every layer, the split of the rows and the
// partial sums' places.
struct NetGrad {
    int rows;
    int K[MLP_LAYERS], N[MLP_LAYERS];
    const uint16_t *in[MLP_LAYERS], *z[MLP_LAYERS];
    int split[MLP_LAYERS], chunk[MLP_LAYERS], wg[MLP_LAYERS];      // slices, rows each, workgroups
    float *part, *csum;
    long part0[MLP_LAYERS], csum0[MLP_LAYERS];
};
hipError_t net_gradients(const NetGrad &g, hipStream_t st);

struct NetParams {
    int K[MLP_LAYERS], N[MLP_LAYERS];
    float *W[MLP_LAYERS], *b[MLP_LAYERS], *gW[MLP_LAYERS], *gb[MLP_LAYERS];
    float *mW[MLP_LAYERS], *vW[MLP_LAYERS], *mb[MLP_LAYERS], *vb[MLP_LAYERS];
    uint16_t *fwd, *bwd;         // packed BF16 weights
    int fwd0[MLP_LAYERS], bwd0[MLP_LAYERS];
    float lr, b1, b2, eps, c1, c2;
};
hipError_t net_pack(const NetParams &p, hipStream_t st);
hipError_t net_update(const NetParams &p, const NetGrad &g, hipStream_t st);

hipError_t mlp_features(const FeatArgs &f, int rows, hipStream_t st);
hipError_t mlp_targets(const SurrogateNorm *nm, int kk, int n, int npad, const double *T0, const double *Y0,
                       const double *T1, const double *Y1, float *Tg, hipStream_t st);
hipError_t mlp_gather_bf16(const uint16_t *src, uint16_t *dst, const int *idx, int rows, int w, hipStream_t st);
hipError_t mlp_gather_f32(const float *src, float *dst, const int *idx, int rows, int w, hipStream_t st);
hipError_t mlp_mse(const float *Yh, const float *Yt, uint16_t *dY, int rows, float *partial, float *loss,
                   hipStream_t st);
hipError_t mlp_zero_u32(unsigned *p, hipStream_t st);
hipError_t mlp_apply(const ApplyArgs &a, int nsp, hipStream_t st);

}  // namespace fcfd
