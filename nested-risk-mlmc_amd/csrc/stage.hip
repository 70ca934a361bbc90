// Device side of portfolio staging: the option-search guides and the Exact
// records, built from the uploaded options and CDFs.
#include "portfolio.hpp"
#include "portfolio_dev.hpp"

namespace nmlmc {

// The smallest x whose product with scale (one IEEE multiply, as in pick_cdf)
// reaches b: bucket b of the guide starts there.
__device__ __forceinline__ double guide_edge(uint64_t b, double scale) {
    if (b == 0) return 0.;
    const double want = (double)b;
    auto step = [](double x, int64_t by) { return __longlong_as_double(__double_as_longlong(x) + by); };
    double x = want / scale;
    while (x > 0. && step(x, -1) * scale >= want) x = step(x, -1);
    while (x * scale < want) x = step(x, 1);
    return x;
}

// Blocks [blk[k], blk[k + 1]) take part k: the guides of methods 0, 1, 2 (one
// thread a bucket), the Exact options' records, the stocks' constants.
//
// Bound by the latency of the binary search (log2 n dependent loads from L2).
// The host built these tables in one thread, 30 ns a bucket of the guide (a
// division and neighbouring doubles) and an exponential a record, and uploaded each by
// itself: 0.6 ms a book of 9000 options, now 0.1 ms.  Staging and sweep of 16 such
// books 20.4 -> 13.1 ms, of 8 with Asians 16.2 -> 13.7 ms.
__global__ __launch_bounds__(256) void k_stage(StageArgs A) {
    uint32_t k = 0;
    while (k < 4 && blockIdx.x >= A.blk[k + 1]) k++;
    const uint64_t t = (uint64_t)(blockIdx.x - A.blk[k]) * 256 + threadIdx.x;
    if (k < 3) {
        // guide[b]: the answer max{i : cdf[i] <= u} at the bucket's lower edge,
        // marked when the next edge's differs; the last bucket is open above.
        __shared__ uint32_t at[257];
        const uint32_t n = A.n[k];
        const uint64_t nb = 4 * (uint64_t)n;
        const double* __restrict__ cdf = A.cdf[k];
        auto answer = [&](uint64_t b) -> uint32_t {
            if (b >= nb) return n - 1;
            const double x = guide_edge(b, A.scale[k]);
            uint32_t lo = 0, hi = n;
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (cdf[mid] <= x) lo = mid;
                else hi = mid;
            }
            return lo;
        };
        at[threadIdx.x] = answer(t);
        if (threadIdx.x == 255) at[256] = answer(t + 1);
        __syncthreads();
        if (t < nb) A.guide[k][t] = at[threadIdx.x] | (at[threadIdx.x + 1] != at[threadIdx.x] ? kGuideMulti : 0u);
        else if (t == nb) A.guide[k][t] = n - 1;
    } else if (k == 3) {
        if (t >= A.n[1]) return;
        const OptionRec o = A.opt1[t];
        const double w = o.w * exp_d(-A.r * o.maturity);
        const double Tt = o.maturity - A.tau, sTt = sqrt(Tt);
        const uint32_t stype = (o.stock_ind << 8) | (uint32_t)(o.type + 2);
        const double S0 = A.stocks[o.stock_ind].S0, h = 0.5 * w * A.prob_norm / o.prob;
        A.mix[t] = MixRec{(float)(o.strike / S0), (float)sTt, (float)(is_digital(o.type) ? h : h * S0), stype};
        const double discp = A.subsample == 1    ? w / (o.prob / A.prob_norm)
                             : A.subsample == -1 ? w * A.options_count
                                                 : w;
        A.ext[t] = ExactRec{o.strike, Tt, sTt, discp, stype, 0};
    } else {
        if (t >= A.d) return;
        const StockRec st = A.stocks[t];
        const double dcoef = A.r - 0.5 * st.sigma * st.sigma;
        const double log2e = 0x1.71547652b82fep+0;
        A.ms[t] = MixStock{(float)(st.sigma * log2e), (float)(dcoef * log2e), (float)(st.sigma * A.stau * log2e),
                           (float)exp_d(dcoef * A.tau)};
        A.es[t] = ExactStock{st.sigma, dcoef, dcoef * A.tau, A.stau, st.S0, 1. / st.S0};
    }
}

hipError_t launch_stage(StageArgs A, hipStream_t s) {
    uint64_t b = 0;
    for (int k = 0; k < 5; k++) {
        A.blk[k] = (uint32_t)b;
        const uint64_t items = k < 3 ? (A.n[k] ? 4 * (uint64_t)A.n[k] + 1 : 0) : k == 3 ? A.n[1] : A.d;
        b += (items + 255) / 256;
    }
    A.blk[5] = (uint32_t)b;
    hipLaunchKernelGGL(k_stage, dim3((uint32_t)b), dim3(256), 0, s, A);
    return hipGetLastError();
}

}  // namespace nmlmc
