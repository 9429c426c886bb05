// mlp_net.hip -- the surrogate network as whole passes: forward (inference or training), backward through
// the layers, weight and bias gradients, and Adam.
//
// Forward and backward keep a row's activations in the registers of one wave from layer to layer.  The
// product is formed transposed, (features x rows) = W^T (features x inputs) * X^T (inputs x rows): in
// v_mfma_f32_16x16x16bf16_1k the result lane (quad h, column c) holds features 4h .. 4h+3 of row c, which
// is the operand fragment the next layer takes for those four inputs.  So activations pass neither
// through LDS nor through memory; what streams is the weights, 16 KB stages in fragment order (packed
// when they change), double-buffered in LDS for the four waves of a workgroup.  Every product sums its
// inputs 16 at a time in ascending order in one accumulator, as a GEMM of 16-deep steps does.
#include "mlp_device.hpp"
#include "surrogate.hpp"

namespace fcfd {

namespace {

constexpr int STAGE = 8192;                    // BF16 values of a stage: two 16 x 256 (or eight 16 x 64) blocks
constexpr int HID = MLP_HID, FB = HID / 16;    // feature blocks of a hidden layer
static_assert(MLP_INP == 64 && MLP_OUTP == 64 && MLP_HID == 256, "stages per layer");

enum { INFER, TRAIN, BACK };

__device__ __forceinline__ v4s frag(uint32_t lo, uint32_t hi) {
    const uint2 v{lo, hi};
    v4s r;
    __builtin_memcpy(&r, &v, sizeof r);
    return r;
}

// The weight stream: 64 bytes a thread and stage, fetched DEPTH stages ahead of their use.
template <int DEPTH>
struct Stream {
    const uint4 *src;
    uint4 (*lds)[STAGE / 8];
    uint4 r[DEPTH][4];
    int left;                                  // stages not fetched yet
    __device__ __forceinline__ void fetch(int slot) {
        if (left <= 0) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[slot][i] = src[i * 256 + threadIdx.x];
        src += STAGE / 8;
        --left;
    }
    __device__ __forceinline__ void store(int slot, int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) lds[buf][i * 256 + threadIdx.x] = r[slot][i];
    }
};

// acc = W^T act over KB input blocks and this wave's part of the NB feature blocks; the stages alternate
// between the buffers from 0 on (every layer has an even number of them).
template <int RT, int FS, int KB, int NB, int D>
__device__ __forceinline__ void layer(Stream<D> &s, const v4s (&act)[FB][RT], v4f (&acc)[FB / FS][RT], int lane, int part,
                                      bool live) {
    constexpr int PER = STAGE / 256 / NB;      // input blocks of a stage
    constexpr int NW = NB / FS;
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[n][t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < KB / PER; ++st) {
        s.fetch(st % D);                       // stage st + D, into the slot of stage st
        if (live) {
            const v4s *w = reinterpret_cast<const v4s *>(s.lds[st & 1]) + part * NW * 64;
#pragma unroll
            for (int kk = 0; kk < PER; ++kk)
#pragma unroll
                for (int n = 0; n < NW; ++n) {
                    const v4s a = w[(kk * NB + n) * 64 + lane];
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        acc[n][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, act[st * PER + kk][t], acc[n][t], 0, 0, 0);
                }
        }
        s.store((st + 1) % D, (st + 1) & 1);
        __syncthreads();
    }
}

}  // namespace

// A workgroup of four waves: 16 RT rows a wave (RT = 1: 64 rows, 2: 128), or 16 rows for FS waves that share
// the features of each layer and pass their activations to each other through LDS (FS = 2: 32 rows, 4: 16).
// Bound: the activation function -- erff takes some 45 vector operations, 1,024 of them a row -- and the
// half-rate MFMA of this depth, which keeps the sums' order: for 65,536 rows about 65 and 29 us.  With 128 rows
// the accumulators and activations do not all fit 256 registers: inference, training's forward and backward keep
// 132, 172 and 156 bytes a lane in scratch, traffic that those figures leave out.  (64 rows and fewer: 136 to
// 186 registers, no scratch.)  65,536 rows: 110 us a pass; five GEMMs of 64 x 64 tiles, loading two bytes a lane and passing every layer through
// memory, took 5 x 72 us.
template <int MODE, int RT, int FS>
__global__ void __launch_bounds__(256, 2) k_mlp(NetArgs a) {
    static_assert(RT == 1 || FS == 1, "rows or features are split");
    constexpr int ROWS = 64 * RT / FS, NT = RT > 1 ? RT : 1, NF = FB / FS;
    __shared__ uint4 stage[2][STAGE / 8];
    __shared__ v4s pass[FS > 1 ? 4 / FS : 1][FS > 1 ? FB * 64 : 1];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, h = lane >> 4, part = wave % FS, group = wave / FS;
    const int wg0 = blockIdx.x * ROWS;
    // tiles of 64 rows: past the rows, past the live row count, or without a live row: left as they are
    bool on[NT], any = false;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int r0 = (wg0 & ~63) + 64 * i;
        on[i] = r0 < a.rows;
        if (MODE == INFER && a.m_dev && on[i]) {
            const int m = int(*a.m_dev);
            on[i] = r0 < m;
            if (on[i] && a.row_live) on[i] = __any(r0 + lane < m && a.row_live[r0 + lane] != 0);
        }
        any = any || on[i];
    }
    if (!any) return;                          // the same in the four waves: before any barrier
    const int row0 = wg0 + 16 * RT * group;    // this wave's rows lie in one tile
    bool live = on[0];
#pragma unroll
    for (int i = 1; i < NT; ++i)
        if (row0 >= wg0 + 64 * i) live = on[i];
    live = __builtin_amdgcn_readfirstlane(live);
    // (two stages ahead where a stage is short: 8 or 16 MFMA blocks, less than the loads take)
    constexpr int D = RT == 1 ? 2 : 1;
    Stream<D> s{reinterpret_cast<const uint4 *>(a.w), stage, {}, MODE == BACK ? 26 : 28};
#pragma unroll
    for (int d = 0; d < D; ++d) s.fetch(d);
    v4s act[FB][RT];
    v4f acc[NF][RT];
    if (live) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const uint16_t *x = a.x + long(row0 + 16 * t + c) * 64 + 4 * h;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (a.wide) {
                    const uint2 v = *reinterpret_cast<const uint2 *>(x + 16 * k);
                    act[k][t] = frag(v.x, v.y);
                } else {
                    act[k][t] = v4s{short(x[16 * k]), short(x[16 * k + 1]), short(x[16 * k + 2]), short(x[16 * k + 3])};
                }
            }
        }
    }
    s.store(0, 0);
    __syncthreads();
#pragma unroll 1
    for (int l = 0; l < 4; ++l) {
        if (l == 0) layer<RT, FS, 4, FB>(s, act, acc, lane, part, live);
        else layer<RT, FS, FB, FB>(s, act, acc, lane, part, live);
        if (!live) continue;                   // (with FS > 1 every wave of the workgroup is live)
#pragma unroll
        for (int n = 0; n < NF; ++n) {
            const int f = 16 * (part * NF + n) + 4 * h;      // features f .. f + 3
            v4f b{};
            if (MODE != BACK) b = *reinterpret_cast<const v4f *>(a.bias[l] + f);
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const long at = long(row0 + 16 * t + c) * HID + f;
                v4f v = acc[n][t];
                float g[4];
                if (MODE == BACK) {
                    const v4f p = *reinterpret_cast<const v4f *>(a.P[l] + at);
#pragma unroll
                    for (int q = 0; q < 4; ++q) g[q] = v[q] * gelu_d(p[q]);
                } else {
                    v = v + b;
                    if (MODE == TRAIN) *reinterpret_cast<v4f *>(a.P[l] + at) = v;
#pragma unroll
                    for (int q = 0; q < 4; ++q) g[q] = gelu(v[q]);
                }
                const uint2 o{f2bf2(g[0], g[1]), f2bf2(g[2], g[3])};
                if (FS == 1) act[n][t] = frag(o.x, o.y);
                else pass[group][(part * NF + n) * 64 + lane] = frag(o.x, o.y);
                if (MODE != INFER) *reinterpret_cast<uint2 *>(a.H[l] + at) = o;
            }
        }
        if (FS > 1) {
            __syncthreads();                   // (the next layer's stages keep writers behind these reads)
#pragma unroll
            for (int n = 0; n < FB; ++n) act[n][0] = pass[group][n * 64 + lane];
        }
    }
    if (MODE == BACK) return;
    layer<RT, FS, FB, 4>(s, act, acc, lane, part, live);
    if (!live) return;
#pragma unroll
    for (int n = 0; n < 4 / FS; ++n) {
        const int f = 16 * (part * (4 / FS) + n) + 4 * h;
        const v4f b = *reinterpret_cast<const v4f *>(a.bias[4] + f);
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            float *o = a.out + long(row0 + 16 * t + c) * MLP_OUTP + f;
            const v4f v = acc[n][t] + b;
            if (a.wide) *reinterpret_cast<v4f *>(o) = v;
            else
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = v[q];
        }
    }
}

// As many rows a workgroup as still give each of 256 CUs one: 16 or 32 (features split), 64, else 128, which
// stream the weights least often.  Both sides, by calls: 8,192 rows, training's forward: 64 rows a workgroup 61 us,
// 32 rows 41; 65,536 rows, inference: 64 rows 128 us, 128 rows 125.  The line between 64 and 128 serves large
// inference only: just above it two rounds of 64 rows are the faster (32,768 rows, inference: 73 us, 128 rows
// 103), and training's passes, which spill more, are so throughout (four steps of 32,768 rows 1.37 ms, 128 rows
// 1.91; of 65,536: 2.46 and 2.95).
template <int MODE>
static hipError_t launch_net(const NetArgs &a, hipStream_t st) {
    if (a.rows <= 0 || a.rows % 64) return hipErrorInvalidValue;
    const int n = a.rows / 64;
    if (n <= 64) hipLaunchKernelGGL((k_mlp<MODE, 1, 4>), dim3(unsigned(4 * n)), dim3(256), 0, st, a);
    else if (n <= 128) hipLaunchKernelGGL((k_mlp<MODE, 1, 2>), dim3(unsigned(2 * n)), dim3(256), 0, st, a);
    else if (n <= 256) hipLaunchKernelGGL((k_mlp<MODE, 1, 1>), dim3(unsigned(n)), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_mlp<MODE, 2, 1>), dim3(unsigned((n + 1) / 2)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t net_forward(const NetArgs &a, bool training, hipStream_t st) {
    return training ? launch_net<TRAIN>(a, st) : launch_net<INFER>(a, st);
}
hipError_t net_backward(const NetArgs &a, hipStream_t st) { return launch_net<BACK>(a, st); }

// ---------------------------------------------------------------------------------------------
// Weight gradients of all layers, H^T dZ with the rows split over NetGrad::split workgroups: 64 x 64 tiles
// of four waves (32 x 32 each), 32 rows a step.  A thread reads the same four columns of four rows and
// writes them as four columns' fragments of four rows, so LDS is read and written eight bytes at a time.
// Partial sums go to g.part, split by split.  Bound: the latency of a workgroup's few steps (16 of 32 rows at
// 8,192 rows and 16 slices) and the partial sums' 21 MB.  8,192 rows, all layers in one launch: 21 us; a launch
// a layer of the two-byte GEMM took 5 x 36 us.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_wgrad(NetGrad g) {
    __shared__ uint16_t As[2][64][36], Bs[2][64][36];
    int l = 0, blk = int(blockIdx.x);
    for (; blk >= g.wg[l]; ++l) blk -= g.wg[l];
    const int K = g.K[l], N = g.N[l], tn = N / 64, tiles = (K / 64) * tn;
    const int tile = blk % tiles, split = blk / tiles;
    const int m0 = tile / tn * 64, n0 = tile % tn * 64;
    const int kbeg = split * g.chunk[l], kend = kbeg + g.chunk[l];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    // loads: threads 0 .. 127 the A tile, the others the B tile; four columns mq of the four rows 4 kq ..
    const bool isb = tid >= 128;
    const int id = tid & 127, kq = id >> 4, mq = id & 15;
    const uint16_t *src = isb ? g.z[l] + n0 : g.in[l] + m0;
    const long ld = isb ? N : K;
    uint2 r[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = min(k0 + 4 * kq + i, kend - 1);          // (rows past the chunk: not used below)
            r[i] = *reinterpret_cast<const uint2 *>(src + k * ld + 4 * mq);
        }
    };
    auto store = [&](int buf) {
        uint16_t (*d)[36] = isb ? Bs[buf] : As[buf];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const unsigned sel = j & 1 ? 0x07060302u : 0x05040100u;      // upper or lower halves
            const uint2 o{__builtin_amdgcn_perm(j < 2 ? r[1].x : r[1].y, j < 2 ? r[0].x : r[0].y, sel),
                          __builtin_amdgcn_perm(j < 2 ? r[3].x : r[3].y, j < 2 ? r[2].x : r[2].y, sel)};
            *reinterpret_cast<uint2 *>(&d[4 * mq + j][4 * kq]) = o;
        }
    };
    v4f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    fetch(kbeg);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = kbeg; k0 < kend; k0 += 32, buf ^= 1) {
        const bool more = k0 + 32 < kend;
        if (more) fetch(k0 + 32);
        const int rr = lane & 15, kf = (lane >> 4) * 4;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            if (kk == 1 && k0 + 16 >= kend) break;                 // a last step of 16 rows
            v4s av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                av[i] = *reinterpret_cast<const v4s *>(&As[buf][wm + i * 16 + rr][16 * kk + kf]);
                bv[i] = *reinterpret_cast<const v4s *>(&Bs[buf][wn + i * 16 + rr][16 * kk + kf]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if (more) store(buf ^ 1);
        __syncthreads();
    }
    float *out = g.part + g.part0[l] + long(split) * K * N;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                out[long(m0 + wm + i * 16 + (lane >> 4) * 4 + q) * N + n0 + wn + j * 16 + (lane & 15)] = acc[i][j][q];
}

// Column sums of dZ (bias gradients) over 64-row chunks, all layers: block (64 columns, chunk).
__global__ void __launch_bounds__(64) k_colsum(NetGrad g) {
    int l = 0, b = int(blockIdx.x);
    for (; b >= g.N[l] / 64; ++l) b -= g.N[l] / 64;
    const int j = b * 64 + threadIdx.x, chunk = blockIdx.y, N = g.N[l];
    const uint16_t *d = g.z[l] + long(chunk) * 64 * N + j;
    float s = 0.f;
#pragma unroll 16
    for (int r = 0; r < 64; ++r) s += bf2f(d[long(r) * N]);
    g.csum[g.csum0[l] + long(chunk) * N + j] = s;
}

hipError_t net_gradients(const NetGrad &g, hipStream_t st) {
    unsigned nb = 0, nc = 0;
    for (int l = 0; l < MLP_LAYERS; ++l) {
        if (g.chunk[l] % 16) return hipErrorInvalidValue;
        nb += unsigned(g.wg[l]);
        nc += unsigned(g.N[l] / 64);
    }
    hipLaunchKernelGGL(k_wgrad, dim3(nb), dim3(256), 0, st, g);
    hipLaunchKernelGGL(k_colsum, dim3(nc, unsigned(g.rows / 64)), dim3(64), 0, st, g);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Parameters.  Element i of the parameters: weights layer by layer, then biases.  Weight (k, n) of a layer
// goes to two packed BF16 streams: forward, blocks of 16 inputs by 16 features as the feature-row fragment
// reads them, layers 0 .. 4; backward the transpose, layers 4 .. 1.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void pack(const NetParams &p, int l, int k, int n, float w) {
    const int K = p.K[l], N = p.N[l];
    const uint16_t v = f2bf(w);
    p.fwd[p.fwd0[l] + ((k >> 4) * (N >> 4) + (n >> 4)) * 256 + (((k >> 2) & 3) * 16 + (n & 15)) * 4 + (k & 3)] = v;
    if (l > 0)
        p.bwd[p.bwd0[l] + ((n >> 4) * (K >> 4) + (k >> 4)) * 256 + (((n >> 2) & 3) * 16 + (k & 15)) * 4 + (n & 3)] = v;
}

__global__ void __launch_bounds__(256) k_pack(NetParams p) {
    int l = 0, i = int(blockIdx.x) * 256 + int(threadIdx.x);
    for (; l < MLP_LAYERS && i >= p.K[l] * p.N[l]; ++l) i -= p.K[l] * p.N[l];
    if (l < MLP_LAYERS) pack(p, l, i / p.N[l], i % p.N[l], p.W[l][i]);
}

// Gradients from the partial sums (in split order), and, with p.lr > 0, Adam on the FP32 parameters and
// their packed copies.  One launch, sixteen partial sums in flight a thread: 9.5 us at 8,192 rows, bound by
// reading them; ten reductions that loaded one at a time (20 us each) and ten Adam launches (4.6) before.
__global__ void __launch_bounds__(256) k_update(NetParams p, NetGrad g) {
    int l = 0, i = int(blockIdx.x) * 256 + int(threadIdx.x);
    for (; l < MLP_LAYERS && i >= p.K[l] * p.N[l]; ++l) i -= p.K[l] * p.N[l];
    const bool bias = l == MLP_LAYERS;
    if (bias) {
        l = 0;
        for (; l < MLP_LAYERS && i >= p.N[l]; ++l) i -= p.N[l];
        if (l == MLP_LAYERS) return;
    }
    const long len = bias ? p.N[l] : long(p.K[l]) * p.N[l];
    const float *part = bias ? g.csum + g.csum0[l] + i : g.part + g.part0[l] + i;
    const int n = bias ? g.rows / 64 : g.split[l];
    float gi = 0.f;
    int q = 0;
    for (; q + 16 <= n; q += 16) {
        float t[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = part[(q + u) * len];
#pragma unroll
        for (int u = 0; u < 16; ++u) gi += t[u];
    }
    for (; q < n; ++q) gi += part[q * len];
    (bias ? p.gb[l] : p.gW[l])[i] = gi;
    if (!(p.lr > 0.f)) return;
    float *w = bias ? p.b[l] : p.W[l], *m = bias ? p.mb[l] : p.mW[l], *v = bias ? p.vb[l] : p.vW[l];
    const float mi = p.b1 * m[i] + (1.f - p.b1) * gi;
    const float vi = p.b2 * v[i] + (1.f - p.b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - p.lr * (mi / p.c1) / (sqrtf(vi / p.c2) + p.eps);
    w[i] = wi;
    if (!bias) pack(p, l, i / p.N[l], i % p.N[l], wi);
}

static unsigned param_blocks(const NetParams &p, bool with_bias) {
    long n = 0;
    for (int l = 0; l < MLP_LAYERS; ++l) n += long(p.K[l]) * p.N[l] + (with_bias ? p.N[l] : 0);
    return unsigned((n + 255) / 256);
}

hipError_t net_pack(const NetParams &p, hipStream_t st) {
    hipLaunchKernelGGL(k_pack, dim3(param_blocks(p, false)), dim3(256), 0, st, p);
    return hipGetLastError();
}

hipError_t net_update(const NetParams &p, const NetGrad &g, hipStream_t st) {
    hipLaunchKernelGGL(k_update, dim3(param_blocks(p, true)), dim3(256), 0, st, p, g);
    return hipGetLastError();
}

}  // namespace fcfd
