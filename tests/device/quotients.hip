// quotients.hip -- the shared-divisor quotients and the square root of fluid_coop.hpp on arrays of operands, for
// tests/test_gpu_quotients.py.
#include "fluid_coop.hpp"

namespace {

enum { RECIP, QUOT, ROOT };

__global__ void __launch_bounds__(256) k_eval(int op, int n, const double *a, const double *b, double *out) {
    const int i = int(blockIdx.x) * 256 + int(threadIdx.x);
    if (i >= n) return;
    const double x = a[i], d = b[i];
    double r = 0.0;
    if (op == RECIP) r = fcfd::recip(d);
    if (op == QUOT) r = fcfd::quot(x, d, fcfd::recip(d));
    if (op == ROOT) r = fcfd::sqrt_core(d);
    out[i] = r;
}

// Mole fractions of three species a lane: y_k / (sw wt_k)
constexpr int NS = 11, M = fcfd::group_m<NS>();
__global__ void __launch_bounds__(64) k_mole(const fcfd::DevThermo *m, int n, const double *sw, const double *y, double *out) {
    const int i = min(int(blockIdx.x) * 64 + int(threadIdx.x), n - 1);
    double yj[M], x[M];
    for (int j = 0; j < M; ++j) yj[j] = y[j * n + i];
    fcfd::ytx_coop<NS>(fcfd::constant(m), 0, true, sw[i], yj, x);
    for (int j = 0; j < M; ++j) out[j * n + i] = x[j];
}

struct Buf {
    double *p = nullptr;
    ~Buf() { (void)hipFree(p); }
    bool get(size_t n) { return hipMalloc(&p, n * sizeof(double)) == hipSuccess; }
    bool put(const double *h, size_t n) { return get(n) && hipMemcpy(p, h, n * sizeof(double), hipMemcpyHostToDevice) == hipSuccess; }
    bool read(double *h, size_t n) { return hipMemcpy(h, p, n * sizeof(double), hipMemcpyDeviceToHost) == hipSuccess; }
};

}  // namespace

// out = 1 / b, a / b, sqrt(b); host arrays of n.  0: done.
extern "C" int quotients_eval(int op, int n, const double *a, const double *b, double *out) {
    if (n < 1 || op < RECIP || op > ROOT) return -1;
    Buf da, db, dout;
    if (!da.put(a, size_t(n)) || !db.put(b, size_t(n)) || !dout.get(size_t(n))) return 1;
    hipLaunchKernelGGL(k_eval, dim3(unsigned((n + 255) / 256)), dim3(256), 0, nullptr, op, n, da.p, db.p, dout.p);
    return hipGetLastError() == hipSuccess && dout.read(out, size_t(n)) ? 0 : 2;
}

// x[3][n] = y[3][n] / (sw[n] wt[3]) as CKYTX forms it.  0: done.
extern "C" int quotients_mole(int n, const double *wt, const double *sw, const double *y, double *x) {
    if (n < 1) return -1;
    static fcfd::DevThermo th;
    for (int j = 0; j < M; ++j) {
        th.wt[j] = wt[j];
        th.rwt[j] = 1.0 / wt[j];
    }
    Buf dt, ds, dy, dx;
    const size_t N = size_t(n);
    if (!dt.put(reinterpret_cast<const double *>(&th), (sizeof th + 7) / 8) || !ds.put(sw, N) || !dy.put(y, M * N) || !dx.get(M * N)) return 1;
    hipLaunchKernelGGL(k_mole, dim3(unsigned((n + 63) / 64)), dim3(64), 0, nullptr,
                       reinterpret_cast<const fcfd::DevThermo *>(dt.p), n, ds.p, dy.p, dx.p);
    return hipGetLastError() == hipSuccess && dx.read(x, M * N) ? 0 : 2;
}
