// The library's device functions one at a time, for tests (test_gpu_functions.py):
// built by the package's Makefile into lib/libnmlmc_probe.so, not a part of the library.
#include "../nested-risk-mlmc_amd/csrc/model_batched.hip"
#include "../nested-risk-mlmc_amd/csrc/portfolio_dev.hpp"

using namespace nmlmc;

namespace {

enum { LOG, SQRT, SINCOS, EXP, PAIR_F64, PAIR_F64_LIB, PAIR_F32 };

__device__ double as_double(uint64_t u) { return __longlong_as_double((long long)u); }

// out[i], out[n + i]: the results for the words a[i], b[i] (or a[i] as a double).
__global__ void k_functions(int which, uint64_t n, const uint64_t* a, const uint64_t* b, double* out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double x = 0., y = 0.;
    if (which == LOG) x = log_unit(as_double(a[i]));
    if (which == SQRT) x = sqrt_pos(as_double(a[i]));
    if (which == SINCOS) sincos_small(as_double(a[i]), x, y);
    if (which == EXP) x = exp_d(as_double(a[i]));
    if (which == PAIR_F64) boxmuller_f64(a[i], b[i], x, y);
    if (which == PAIR_F64_LIB) boxmuller_f64_lib(a[i], b[i], x, y);
    if (which == PAIR_F32) {
        float s, c, r, r2;
        bm_polar_f32(a[i], b[i], s, c, r, r2);
        x = (double)s * (double)r;
        y = (double)c * (double)r;
    }
    out[i] = x;
    out[n + i] = y;
}

// Exact option i (columns of p: S0, sigma, strike, maturity, weight over probability; type[i]) and a
// draw (words a, b; level R over S0): the mixed form's term and error scale, and the FP64 term.
__global__ void k_exact(uint64_t n, double r, double tau, int anti, int cv, const double* p, const uint64_t* words,
                        double* out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double S0 = p[i], sigma = p[n + i], K = p[2 * n + i], T = p[3 * n + i], wp = p[4 * n + i], R = p[5 * n + i];
    const int type = (int)p[6 * n + i];
    const double Tt = T - tau, dcoef = r - 0.5 * sigma * sigma, discp = wp * exp(-r * T), log2e = 0x1.71547652b82fep+0;
    const uint32_t stype = (uint32_t)(type + 2);
    const MixRec q{(float)(K / S0), (float)sqrt(Tt), (float)(is_digital(type) ? 0.5 * discp : 0.5 * discp * S0), stype};
    const MixStock ms{(float)(sigma * log2e), (float)(dcoef * log2e), (float)(sigma * sqrt(tau) * log2e), (float)exp(dcoef * tau)};
    const ExactRec e{K, Tt, sqrt(Tt), discp, stype, 0};
    const ExactStock es{sigma, dcoef, dcoef * tau, sqrt(tau), S0, 1. / S0};
    float x, y, mag;
    double X, Y;
    boxmuller_f32(words[i], words[n + i], x, y);
    boxmuller_f64(words[i], words[n + i], X, Y);
    out[i] = (double)inner_exact_mix(q, ms, anti, cv, (float)R, x, y, mag);
    out[n + i] = (double)mag;
    out[2 * n + i] = inner_exact_d(e, es, anti, cv, R * S0, X, Y);
}

// A lane sums the units [u[i], u[n + i]) of outer sample i's first final group of `count` inner samples:
// s1, s2, sab, smm.
template <int VAR, bool F32>
__global__ void k_units(typename ModelPolicy<VAR>::Args A, uint64_t n, uint64_t count, const double* Y, const uint64_t* m,
                        const uint64_t* u, double* out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    ItemState it{};
    it.Y = Y[i];
    SegAcc s;
    ModelPolicy<VAR>::template units<F32, true>(A, (uint32_t)m[i], it, TAG_FINAL, u[i], u[n + i], 0, count, s);
    out[i] = s.s1;
    out[n + i] = s.s2;
    out[2 * n + i] = s.sab;
    out[3 * n + i] = s.smm;
}

struct Buffers {
    void* p[4] = {};
    int used = 0;
    ~Buffers() {
        for (int i = 0; i < used; i++) (void)hipFree(p[i]);
    }
    void* take(const void* from, size_t bytes) {
        void* d = nullptr;
        if (hipMalloc(&d, bytes) != hipSuccess) return nullptr;
        p[used++] = d;
        if (from && hipMemcpy(d, from, bytes, hipMemcpyHostToDevice) != hipSuccess) return nullptr;
        return d;
    }
};

template <int VAR, bool F32>
hipError_t run_units(double tau, uint64_t seed, uint64_t n, uint64_t count, const double* Y, const uint64_t* m,
                     const uint64_t* u, double* out) {
    typename ModelPolicy<VAR>::Args A{};
    A.c.seed = seed;
    A.mp.stau = sqrt(tau);
    A.mp.s1tau = sqrt(1. - tau);
    hipLaunchKernelGGL((k_units<VAR, F32>), dim3((uint32_t)((n + 63) / 64)), dim3(64), 0, 0, A, n, count, Y, m, u, out);
    return hipGetLastError();
}

}  // namespace

extern "C" {

int probe_functions(int which, uint64_t n, const uint64_t* a, const uint64_t* b, double* out) {
    Buffers bufs;
    uint64_t* da = (uint64_t*)bufs.take(a, 8 * n);
    uint64_t* db = (uint64_t*)bufs.take(b, 8 * n);
    double* dout = (double*)bufs.take(nullptr, 16 * n);
    if (!da || !db || !dout) return 1;
    hipLaunchKernelGGL(k_functions, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, 0, which, n, da, db, dout);
    if (hipGetLastError() != hipSuccess) return 2;
    return hipMemcpy(out, dout, 16 * n, hipMemcpyDeviceToHost) == hipSuccess ? 0 : 3;
}

int probe_exact(uint64_t n, double r, double tau, int anti, int cv, const double* p, const uint64_t* words, double* out) {
    Buffers bufs;
    const double* dp = (const double*)bufs.take(p, 56 * n);
    const uint64_t* dw = (const uint64_t*)bufs.take(words, 16 * n);
    double* dout = (double*)bufs.take(nullptr, 24 * n);
    if (!dp || !dw || !dout) return 1;
    hipLaunchKernelGGL(k_exact, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, 0, n, r, tau, anti, cv, dp, dw, dout);
    if (hipGetLastError() != hipSuccess) return 2;
    return hipMemcpy(out, dout, 24 * n, hipMemcpyDeviceToHost) == hipSuccess ? 0 : 3;
}

int probe_units(int variant, int f32, double tau, uint64_t seed, uint64_t n, uint64_t count, const double* Y,
                const uint64_t* m, const uint64_t* u, double* out) {
    Buffers bufs;
    const double* dY = (const double*)bufs.take(Y, 8 * n);
    const uint64_t* dm = (const uint64_t*)bufs.take(m, 8 * n);
    const uint64_t* du = (const uint64_t*)bufs.take(u, 16 * n);
    double* dout = (double*)bufs.take(nullptr, 32 * n);
    if (!dY || !dm || !du || !dout) return 1;
    const hipError_t e =
        variant == MODEL_REF ? (f32 ? run_units<MODEL_REF, true>(tau, seed, n, count, dY, dm, du, dout)
                                    : run_units<MODEL_REF, false>(tau, seed, n, count, dY, dm, du, dout))
                             : (f32 ? run_units<MODEL_SHIFT, true>(tau, seed, n, count, dY, dm, du, dout)
                                    : run_units<MODEL_SHIFT, false>(tau, seed, n, count, dY, dm, du, dout));
    if (e != hipSuccess) return 2;
    return hipMemcpy(out, dout, 32 * n, hipMemcpyDeviceToHost) == hipSuccess ? 0 : 3;
}

}  // extern "C"
