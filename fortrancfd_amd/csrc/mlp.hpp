// mlp.hpp -- the chemistry surrogate: a 56 -> 4x256 GELU -> 54 multilayer perceptron with BF16
// weights and activations and FP32 accumulation on MFMA (mlp.hip).
#pragma once

#include <cstdint>

#include "fcfd_common.hpp"

namespace fcfd {

constexpr int MLP_IN = 56;       // Box-Cox Y (53), T, log p, log dt
constexpr int MLP_OUT = 54;      // dY (53), dT
constexpr int MLP_HID = 256;
constexpr int MLP_LAYERS = 5;
constexpr int MLP_INP = 64;      // padded widths (multiples of the 16-wide MFMA tiles)
constexpr int MLP_OUTP = 64;

// Layer l maps K[l] -> N[l] columns.
constexpr int MLP_K[MLP_LAYERS] = {MLP_INP, MLP_HID, MLP_HID, MLP_HID, MLP_HID};
constexpr int MLP_N[MLP_LAYERS] = {MLP_HID, MLP_HID, MLP_HID, MLP_HID, MLP_OUTP};

struct GemmArgs {
    const uint16_t *A;   // bf16, element (m, k) at A[m*sam + k*sak]
    const uint16_t *B;   // bf16, element (k, n) at B[k*sbk + n*sbn]
    long sam, sak, sbk, sbn;
    int M, N, K;         // M, N multiples of 64; K multiple of 16
    int ksplit;          // split-K factor: partial s goes to C32 + s*M*ldc
    float *C32;
    long ldc;
};

hipError_t launch_gemm(const GemmArgs &a, hipStream_t st);

}  // namespace fcfd
