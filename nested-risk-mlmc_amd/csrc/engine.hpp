// Shared definitions of the nested-sampler engine (host and device).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rng.hpp"

namespace nmlmc {

constexpr int kMaxPhi = 4;
constexpr int kMaxMoments = 4;
constexpr int kStats = 6;       // inner_stats reported through the ABI
constexpr int kStatsExt = 9;    // + mixed-form diagnostics: FP64 re-evaluations, flips, rechecked decisions

// One record of per-group partial results, reduced in a fixed order by
// k_reduce_partials: the per-level block of the reference (nested_sampler.hpp:587).
struct Partial {
    double f[kMaxPhi * kMaxMoments];
    double d[kMaxPhi * kMaxMoments];
    double work;
    uint64_t stats[kStatsExt];
};
constexpr int kPartialFields = 2 * kMaxPhi * kMaxMoments + 1 + kStatsExt;
// The reduced record of a level call is followed by this many staging records
// of the two-pass reduction (launch_reduce_partials).
constexpr uint32_t kReduceBlocks = 256;

// get_samples_count's constructor state (nested_sampler.hpp:225-239), computed on
// the host with the host libm so that tmp matches the reference bit for bit.
struct LevelCounts {
    uint64_t base;
    uint64_t max;
    double tmp;
    int adaptive;
    int rule;
};

struct EngineParams {
    uint32_t N0, beta;
    int antithetic;
    uint32_t fine_moments, diff_moments;
    double adaptive_r;
    uint32_t adapt_rule, cap_log2;
};

enum { PHI_INDICATOR = 0, PHI_MAX = 1, PHI_MOMENTS = 2, PHI_FMOMENTS = 3 };

// One step of a butterfly over aligned groups of lanes: v plus the value O lanes
// across (lane ^ O), by register moves (DPP, gfx950's row swaps) instead of the
// LDS permute that a shuffle is: a wave's FP64 sum in a fraction of the latency.
// DPP has no lane ^ 4 and, upward, no lane ^ 8: a mirror of 8 or 16 lanes where the
// steps go up (the smaller groups' lanes are equal already), a rotation by 4
// where they go down (lanes 8 apart are).
template <int O, bool UP>
__device__ __forceinline__ uint32_t lane_across(uint32_t v) {
    static_assert(O == 1 || O == 2 || O == 4 || O == 8, "within a row of 16 lanes");
    constexpr int quad = O == 1 ? 0xB1 : 0x4E, mirror = O == 4 ? 0x141 : 0x140, rotate = O == 4 ? 0x124 : 0x128;
    constexpr int ctrl = O <= 2 ? quad : UP ? mirror : rotate;
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, 0xf, 0xf, false);
}
template <int O, bool UP = true, class T>
__device__ __forceinline__ T add_across(T v) {
    static_assert(sizeof(T) == 8, "64-bit sums");
    uint32_t w[2], a[2], b[2];
    __builtin_memcpy(w, &v, 8);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        if constexpr (O < 16) {
            a[i] = w[i];
            b[i] = lane_across<O, UP>(w[i]);
        } else if constexpr (O == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(w[i], w[i], false, false);
            a[i] = r[0];
            b[i] = r[1];
        } else {
            const auto r = __builtin_amdgcn_permlane32_swap(w[i], w[i], false, false);
            a[i] = r[0];
            b[i] = r[1];
        }
    }
    T x, y;
    __builtin_memcpy(&x, a, 8);
    __builtin_memcpy(&y, b, 8);
    return x + y;
}

// Sum over the G lanes of an aligned lane group: every lane of the group ends
// with the same, bit-identical, total.
template <int G, class T>
__device__ __forceinline__ T group_total(T v) {
    if constexpr (G > 1) v = add_across<1>(v);
    if constexpr (G > 2) v = add_across<2>(v);
    if constexpr (G > 4) v = add_across<4>(v);
    if constexpr (G > 8) v = add_across<8>(v);
    if constexpr (G > 16) v = add_across<16>(v);
    if constexpr (G > 32) v = add_across<32>(v);
    return v;
}
template <int G>
__device__ __forceinline__ double group_sum(double v) {
    return group_total<G>(v);
}

// Sums over the 64 lanes of a wave, halves first.
template <class T>
__device__ __forceinline__ T wave_total(T v) {
    v = add_across<32, false>(v);
    v = add_across<16, false>(v);
    v = add_across<8, false>(v);
    v = add_across<4, false>(v);
    v = add_across<2, false>(v);
    return add_across<1, false>(v);
}
__device__ __forceinline__ double wave_sum(double v) { return wave_total(v); }
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) { return wave_total(v); }

// Lane `lane`'s value for every lane (lane the same in all lanes; it need not
// be active for the read, but its value is only meaningful when it is).
__device__ __forceinline__ uint32_t bcast_u32(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
__device__ __forceinline__ uint64_t bcast_u64(uint64_t v, uint32_t lane) {
    const uint32_t lo = bcast_u32((uint32_t)v, lane), hi = bcast_u32((uint32_t)(v >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ double bcast_f64(double v, uint32_t lane) {
    return __longlong_as_double((long long)bcast_u64((uint64_t)__double_as_longlong(v), lane));
}

// add_moments (nested_sampler.hpp:87-100): out[i*m + j] += phi_i^(j+1).
__device__ __forceinline__ void add_moments(const double* phi, uint32_t phi_size, double* out,
                                            uint32_t moments) {
    for (uint32_t i = 0; i < phi_size; i++) {
        double p = 1.;
        for (uint32_t j = 0; j < moments; j++) {
            p *= phi[i];
            out[i * moments + j] += p;
        }
    }
}

// Single-component add_phi of the model sampler (model_sampler.cpp:81-91) and of
// the portfolio sampler's Indicator / Max cases (portfolio_sampler.cpp:261-291).
__device__ __forceinline__ double phi_scalar(int phi_type, double u, double coeff, double phi) {
    if (phi_type == PHI_MAX) return phi + coeff * (u > 0 ? u : 0.);
    return phi + coeff * (double)(u >= 0.);
}

}  // namespace nmlmc
