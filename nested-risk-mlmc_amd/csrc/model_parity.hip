// Plain FP64 form of the model problem with the reference's keying.
//
// Restates kernel_sample<false, model::sampler> (nested_sampler.hpp:369-485) for
// the OpenMP build's semantics: T virtual threads, thread t owning two streams
// keyed {seed, t} whose positions persist across calls, thread t taking the
// libgomp static-schedule block of [0, M) and walking its outer samples in
// order.  On the GPU a virtual thread is an aligned group of G lanes (G | 64),
// or a whole block of G = 256 lanes (four waves) when few virtual threads hold
// outer samples and their inner loops are long: the group walks the outer
// samples in order while its lanes split every inner loop, each lane computing
// the draws at the stream positions it owns.  Every decision (adaptive counts,
// phi, moments) is group-uniform, so the draws and the per-sample results
// equal those of the sequential reference.
#include "engine.hpp"
#include "model.hpp"
#include "plain_help.hpp"

namespace nmlmc {

struct ModelParityArgs {
    ModelParams mp;
    EngineParams ep;
    LevelCounts cf, cc;      // fine (ell) and coarse (ell - 1) sample counts
    uint64_t seed;
    uint64_t M;
    uint32_t T;
    uint32_t ell;
    PlainHelp* help;         // G = 256 only
    uint32_t help_base;
    StreamState* states;     // [2 T]: sync, inner
    Partial* partials;       // [T]
    double* tr_phi_f;
    double* tr_phi_c;
    uint64_t* tr_nf;
    uint64_t* tr_nc;
};

// Sums of a and b over the G lanes of a virtual thread.  G = 256 is the whole
// block (one virtual thread per block, so every thread reaches the barriers): wave
// sums, then the waves' added in wave order.  Two buffers by turns need one
// barrier a sum.
template <int G>
__device__ __forceinline__ void vt_sum(double& a, double& b, uint32_t& turn) {
    if constexpr (G <= 64) {
        a = group_sum<G>(a);
        b = group_sum<G>(b);
    } else {
        constexpr int W = G / 64;
        __shared__ double red[2][2][W];
        a = wave_sum(a);
        b = wave_sum(b);
        const uint32_t wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) {
            red[turn][0][wave] = a;
            red[turn][1][wave] = b;
        }
        __syncthreads();
        a = red[turn][0][0];
        b = red[turn][1][0];
#pragma unroll
        for (int w = 1; w < W; w++) {
            a += red[turn][0][w];
            b += red[turn][1][w];
        }
        turn ^= 1;
    }
}

// One lane's share of the Box-Muller pairs [lo, hi) of a draw group of `count`
// inner samples whose pair p is block blk0 + p of the stream (k0, k1): sums of the
// losses and of their squares.  Two pairs an iteration: the last outer samples
// of a level run one wave a SIMD, where a lone pair's chain of dependent FP64
// operations leaves half the issue slots empty.
template <int VAR, int G>
__device__ __forceinline__ void pair_sums(const ModelParams& mp, uint64_t k0, uint64_t k1, double Y, uint64_t blk0,
                                          uint64_t count, uint64_t lo, uint64_t hi, uint32_t gl, double& s1, double& s2) {
    auto add = [&](double d) {
        s1 += d;
        s2 += d * d;
    };
    auto pair = [&](uint64_t b, double x, double y) {
        if (VAR == MODEL_REF) {
            add(model_ref_inner(mp, Y, x, y));
        } else {
            add(Y + x);
            if (2 * b + 1 < count) add(Y + y);
        }
    };
    // All lanes while a pair is left for the second half of them: with each lane for
    // itself, groups that end between G and 2 G pairs ran the loop for some lanes and
    // then the last pair for the others (80 pairs on 64 lanes: 592 us a call, 510 so).
    uint64_t b = lo + gl;
    for (uint64_t first = lo; first + G < hi; first += 2 * G, b += 2 * G) {
        const u64x2 w = threefry2x64_20(blk0 + b, 0, k0, k1), v = threefry2x64_20(blk0 + b + G, 0, k0, k1);
        double x, y, z, t;
        boxmuller_f64(w.a, w.b, x, y);
        boxmuller_f64(v.a, v.b, z, t);
        pair(b, x, y);
        if (b + G < hi) pair(b + G, z, t);
    }
    if (b < hi) {
        const u64x2 w = threefry2x64_20(blk0 + b, 0, k0, k1);
        double x, y;
        boxmuller_f64(w.a, w.b, x, y);
        pair(b, x, y);
    }
}

// Words that blocks on other XCDs read or write during the kernel.
template <class T>
__device__ __forceinline__ T shared_load(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void shared_store(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A segment of block `slot`'s posting, or -1.  Segments are numbered from above, so
// that one counter holds them; a claim that succeeds holds the posting open, and its
// words are read after it.
__device__ __forceinline__ int claim_segment(PlainHelp* h, uint32_t slot) {
    int32_t* avail = &h->job[slot].avail;
    if (shared_load(avail) <= 0) return -1;
    return __hip_atomic_fetch_add(avail, -1, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) - 1;
}

// Runs segment seg of the posting with the whole block.
template <int VAR>
__device__ __forceinline__ void run_segment(const ModelParams& mp, PlainHelp* h, uint32_t slot, int seg, uint64_t k0,
                                            uint32_t& turn) {
    PlainJob* j = &h->job[slot];
    const uint64_t size = shared_load(&j->segment), pairs = shared_load(&j->pairs);
    const uint64_t lo = seg * size, hi = lo + size < pairs ? lo + size : pairs;
    double s1 = 0., s2 = 0.;
    pair_sums<VAR, 256>(mp, k0, slot, shared_load(&j->Y), shared_load(&j->blk0), shared_load(&j->count), lo, hi,
                        threadIdx.x, s1, s2);
    vt_sum<256>(s1, s2, turn);
    if (threadIdx.x == 0) {
        shared_store(&h->sums[slot][seg][0], s1);
        shared_store(&h->sums[slot][seg][1], s2);
        __hip_atomic_fetch_add(&j->finished, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The draw group of this block's virtual thread through a posting.
template <int VAR>
__device__ __forceinline__ void posted_sums(const ModelParams& mp, PlainHelp* h, uint64_t k0, double Y, uint64_t blk0,
                                            uint64_t count, uint64_t pairs, uint32_t& turn, double& s1, double& s2) {
    __shared__ int taken;
    const uint32_t slot = blockIdx.x;
    PlainJob* j = &h->job[slot];
    uint64_t size = (pairs + kMaxSegments - 1) / kMaxSegments;
    size = size < kMinSegment ? kMinSegment : (size + 511) & ~(uint64_t)511;
    const uint32_t segments = (uint32_t)((pairs + size - 1) / size);
    if (threadIdx.x == 0) {
        shared_store(&j->finished, 0u);
        shared_store(&j->segment, (uint32_t)size);
        shared_store(&j->blk0, blk0);
        shared_store(&j->pairs, pairs);
        shared_store(&j->count, count);
        shared_store(&j->Y, Y);
        __hip_atomic_store(&j->avail, (int32_t)segments, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_or(&h->open[slot / 64], 1ull << (slot & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    while (true) {
        if (threadIdx.x == 0) taken = claim_segment(h, slot);
        __syncthreads();
        const int seg = taken;
        __syncthreads();
        if (seg < 0) break;
        run_segment<VAR>(mp, h, slot, seg, k0, turn);
    }
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_and(&h->open[slot / 64], ~(1ull << (slot & 63)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while (__hip_atomic_load(&j->finished, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < segments)
            __builtin_amdgcn_s_sleep(4);
    }
    __syncthreads();
    s1 = threadIdx.x < segments ? shared_load(&h->sums[slot][threadIdx.x][0]) : 0.;
    s2 = threadIdx.x < segments ? shared_load(&h->sums[slot][threadIdx.x][1]) : 0.;
    vt_sum<256>(s1, s2, turn);
}

// A block whose virtual thread has ended: segments of others' postings until
// every block has ended, or at once if some have not even started (they need the room).
template <int VAR>
__device__ __forceinline__ void help_others(const ModelParams& mp, PlainHelp* h, uint32_t base, uint64_t k0,
                                            uint32_t& turn) {
    __shared__ int job[2];  // slot (-1: none, -2: leave) and segment
    const uint32_t words = (gridDim.x + 63) / 64, lane = threadIdx.x;
    if (lane == 0) __hip_atomic_fetch_add(&h->ended, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t turnstile = blockIdx.x;
    while (true) {
        if (lane < 64) {
            // The lanes look at the words of postings from a place of this block's
            // own onward, so that helpers spread over the postings.
            const uint32_t w = words ? (lane + turnstile) % 64 : 0;
            const uint64_t open = w < words ? shared_load(&h->open[w]) : 0;
            const uint64_t some = __ballot(open != 0);
            int slot = -1, seg = -1;
            if (some) {
                const int at = __builtin_ctzll(some);
                if ((int)lane == at) {
                    const uint32_t r = (turnstile >> 3) & 63;
                    const uint64_t turned = (open >> r) | (r ? open << (64 - r) : 0);
                    slot = (int)(w * 64 + ((__builtin_ctzll(turned) + r) & 63));
                    seg = claim_segment(h, (uint32_t)slot);
                }
                slot = __shfl(slot, at);
                seg = __shfl(seg, at);
                if (seg < 0) slot = -1;
            }
            if (lane == 0) {
                if (slot < 0 && helper_leaves(shared_load(&h->started), shared_load(&h->ended), base, gridDim.x))
                    slot = -2;
                job[0] = slot;
                job[1] = seg;
            }
        }
        __syncthreads();
        const int slot = job[0], seg = job[1];
        __syncthreads();
        if (slot == -2) return;
        if (slot >= 0) run_segment<VAR>(mp, h, (uint32_t)slot, seg, k0, turn);
        else __builtin_amdgcn_s_sleep(16);
        turnstile += 9;
    }
}

// Inner loop over `count` model samples from stream state st (the group's
// inner stream), lanes of the group splitting the Box-Muller pairs
// (inner_sampler::sample_inner, nested_sampler.hpp:131-161).
template <int VAR, int G>
__device__ __forceinline__ void parity_inner(const ModelParams& mp, PlainHelp* help, uint64_t k0, uint64_t k1,
                                             StreamState& st, double Y, uint64_t count, uint32_t gl, uint32_t& turn,
                                             double& s1_out, double& s2_out) {
    constexpr int nps = (VAR == MODEL_REF) ? 2 : 1;
    const uint64_t K = count * nps;
    double s1 = 0., s2 = 0.;
    if (!st.is_saved && (st.P & 1) == 0) {
        const uint64_t pairs = (K + 1) >> 1;
        const uint64_t blk0 = st.P >> 1;
        if (G == 256 && help && pairs >= kPostPairs) {
            posted_sums<VAR>(mp, help, k0, Y, blk0, count, pairs, turn, s1_out, s2_out);
            st = advance_normals_f64(k0, k1, st, K);
            return;
        }
        pair_sums<VAR, G>(mp, k0, k1, Y, blk0, count, 0, pairs, gl, s1, s2);
    } else {
        for (uint64_t i = gl; i < count; i += G) {
            double d;
            if (VAR == MODEL_REF) {
                d = model_ref_inner(mp, Y, normal_at_f64(k0, k1, st, 2 * i), normal_at_f64(k0, k1, st, 2 * i + 1));
            } else {
                d = Y + normal_at_f64(k0, k1, st, i);
            }
            s1 += d;
            s2 += d * d;
        }
    }
    vt_sum<G>(s1, s2, turn);
    s1_out = s1;
    s2_out = s2;
    st = advance_normals_f64(k0, k1, st, K);
}

// Waves per SIMD the kernels are compiled for: at 2 they take 225 to 235 VGPRs, at 4
// they spill 250 to 510 B a lane, at 3 the reference model's sweep (levels 0 to 8 from
// 2 10^6 outer samples) is as fast within 2%.  The sweep is bound by FP64 issue: 18.9 ms
// with one call of the inner loop, two pairs an iteration and register-move sums
// (22.3 ms before), 9.4 ms with the lane rule of the level call and the blocks'
// helping: there level 8's 488 outer samples waited 5.5 ms for the few that
// draw 2^21 inner samples a round on one CU each (6.2 ms, now 0.62; level 7 1.8, now 0.74).
#ifndef NMLMC_PLAIN_MODEL_WAVES
#define NMLMC_PLAIN_MODEL_WAVES 2
#endif

template <int VAR, int G>
__global__ __launch_bounds__(256, NMLMC_PLAIN_MODEL_WAVES) void k_model_parity(ModelParityArgs A) {
    const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t t = gtid / G;
    const uint32_t gl = gtid % G;
    const bool active = t < A.T;  // whole groups share this flag (G divides the block)
    constexpr int nps = (VAR == MODEL_REF) ? 2 : 1;
    const ModelParams& mp = A.mp;
    const EngineParams& ep = A.ep;
    const uint64_t k0 = A.seed, k1 = t;

    // libgomp static schedule of [0, M) over T threads.
    uint64_t q = A.M / A.T, rr = A.M % A.T;
    if (t < rr) {
        q++;
        rr = 0;
    }
    const uint64_t s0 = active ? q * t + rr : 0, e0 = active ? s0 + q : 0;

    if (G == 256 && A.help && threadIdx.x == 0)
        __hip_atomic_fetch_add(&A.help->started, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    StreamState ss{}, si{};
    if (active) {
        ss = A.states[2 * t];
        si = A.states[2 * t + 1];
    }
    double f_sums[kMaxMoments] = {0, 0, 0, 0}, d_sums[kMaxMoments] = {0, 0, 0, 0};
    // stats[0 .. 3] of inner_stats; the model draws no uniforms.
    uint64_t inner = 0, outers = 0, at_max = 0, at_base = 0, randn_count = 0;
    uint32_t turn = 0;
    const bool fine_only = (A.ell == 0);
    const double start = -mp.max_loss;

    for (uint64_t m = s0; m < e0; m++) {
        // model::sampler::sample_outer (model_sampler.cpp:57-59).
        const double Y = st_randn_f64(k0, k1, ss);
        randn_count++;
        // The outer sample's draw groups one after another, from one call of the
        // inner loop: the test rounds (get_samples_count::operator(),
        // nested_sampler.hpp:240-273, with sample_inner_delta2, 120-129) of the fine
        // count (phase 0) and of the coarse one (1), then the finals (2):
        // sample_phi / sample_phi_antithetic (164-216).
        uint64_t nf = 0, nc = 0, cur = A.cf.base;
        uint64_t group = 0, groups = 1, small = 0, big = 0;
        bool f_big = true;
        double f_phi = 0., c_phi = 0., phi_small = 0., s1_big = 0.;
        int phase = 0;
        while (true) {
            bool decided = false;
            uint64_t n;
            if (phase < 2) {
                const uint64_t lmax = phase == 0 ? A.cf.max : A.cc.max;
                n = cur;
                if (lmax <= 2 * cur) {
                    cur = lmax;
                    decided = true;
                } else {
                    inner += cur;
                }
            } else {
                n = (fine_only || ep.antithetic) ? small : group == 0 ? nf : nc;
            }
            if (!decided) {
                double s1, s2;
                parity_inner<VAR, G>(mp, A.help, k0, k1, si, Y, n, gl, turn, s1, s2);
                randn_count += n * nps;
                const double mean = start + s1 / (double)n;
                if (phase < 2) {
                    const double tmp = phase == 0 ? A.cf.tmp : A.cc.tmp;
                    const double out_var = s2 / (double)(n - 1) - (s1 * s1) / (double)(n * (n - 1));
                    const double delta2 = mean * mean / out_var;
                    const double want = A.cf.rule == 1 ? tmp / delta2 : pow(delta2, -ep.adaptive_r / 2) * tmp;
                    if (want <= (double)n) decided = true;
                    else cur *= 2;
                } else if (fine_only) {
                    f_phi = phi_scalar(mp.phi_type, mean, 1., 0.);
                } else if (ep.antithetic) {
                    phi_small = phi_scalar(mp.phi_type, mean, (double)(1.f / (float)groups), phi_small);
                    s1_big += s1;
                } else {
                    (group == 0 ? f_phi : c_phi) = phi_scalar(mp.phi_type, mean, 1., 0.);
                }
                if (phase == 2 && ++group == groups) break;
            }
            if (!decided) continue;
            if (phase == 0) {
                nf = cur;
                outers += 1;
                at_max += (nf == A.cf.max);
                at_base += (nf == A.cf.base);
                cur = A.cc.base;
                phase = fine_only ? 2 : 1;
            } else {
                nc = cur;
                phase = 2;
            }
            if (phase == 2) {
                if (fine_only) {
                    small = nf;
                    inner += nf;
                } else if (ep.antithetic) {
                    f_big = nf > nc;
                    big = f_big ? nf : nc;
                    small = f_big ? nc : nf;
                    groups = big / small;
                    inner += big;
                } else {
                    groups = 2;
                    inner += nf + nc;
                }
            }
        }
        if (!fine_only && ep.antithetic) {
            const double phi_big = phi_scalar(mp.phi_type, start + s1_big / (double)big, 1., 0.);
            f_phi = f_big ? phi_big : phi_small;
            c_phi = f_big ? phi_small : phi_big;
        }
        add_moments(&f_phi, 1, f_sums, ep.fine_moments);
        if (!fine_only) {
            const double dphi = f_phi - c_phi;
            add_moments(&dphi, 1, d_sums, ep.diff_moments);
        }
        if (gl == 0) {
            if (A.tr_phi_f) A.tr_phi_f[m] = f_phi;
            if (A.tr_phi_c) A.tr_phi_c[m] = c_phi;
            if (A.tr_nf) A.tr_nf[m] = nf;
            if (A.tr_nc) A.tr_nc[m] = nc;
        }
    }
    if (active && gl == 0) {
        A.states[2 * t] = ss;
        A.states[2 * t + 1] = si;
    }
    // The block's record: the sums of its virtual threads in lane order (wave sums,
    // then wave by wave), its other fields zero.  The model adds one unit of
    // work per inner sample drawn (model_sampler.cpp:67), tests included.
    constexpr int ND = 2 * kMaxMoments + 1, NU = 5;
    __shared__ double pd[4][ND];
    __shared__ uint64_t pu[4][NU];
    const bool leader = active && gl == 0;
    double d[ND] = {f_sums[0], f_sums[1], f_sums[2], f_sums[3], d_sums[0], d_sums[1], d_sums[2], d_sums[3], (double)inner};
    uint64_t u[NU] = {inner, outers, at_max, at_base, randn_count};
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < ND; k++) {
        if constexpr (G < 64) d[k] = wave_sum(leader ? d[k] : 0.);
        if (lane == 0) pd[wave][k] = (G < 64 || leader) ? d[k] : 0.;
    }
#pragma unroll
    for (int k = 0; k < NU; k++) {
        if constexpr (G < 64) u[k] = wave_sum_u64(leader ? u[k] : 0);
        if (lane == 0) pu[wave][k] = (G < 64 || leader) ? u[k] : 0;
    }
    __syncthreads();
    uint64_t* out = reinterpret_cast<uint64_t*>(&A.partials[blockIdx.x]);
    const uint32_t k = threadIdx.x;
    const int fd = k < 4 ? (int)k : (k >= 16 && k < 20) ? (int)k - 12 : k == 32 ? ND - 1 : -1;
    const int fu = k >= 33 && k < 37 ? (int)k - 33 : k == 38 ? 4 : -1;
    uint64_t v = 0;
    if (fd >= 0) v = (uint64_t)__double_as_longlong(((pd[0][fd] + pd[1][fd]) + pd[2][fd]) + pd[3][fd]);
    if (fu >= 0) v = pu[0][fu] + pu[1][fu] + pu[2][fu] + pu[3][fu];
    if (k < (uint32_t)kPartialFields) out[k] = v;
    if constexpr (G == 256) {
        if (A.help) help_others<VAR>(mp, A.help, A.help_base, k0, turn);
    }
}
static_assert(kMaxPhi * kMaxMoments == 16, "word layout of a Partial used above");

template <int VAR>
static hipError_t launch_var(const ModelParityArgs& A, uint32_t G, uint32_t blocks, hipStream_t s) {
    const dim3 grid(blocks), block(256);
    switch (G) {
    case 1: hipLaunchKernelGGL((k_model_parity<VAR, 1>), grid, block, 0, s, A); break;
    case 2: hipLaunchKernelGGL((k_model_parity<VAR, 2>), grid, block, 0, s, A); break;
    case 4: hipLaunchKernelGGL((k_model_parity<VAR, 4>), grid, block, 0, s, A); break;
    case 8: hipLaunchKernelGGL((k_model_parity<VAR, 8>), grid, block, 0, s, A); break;
    case 16: hipLaunchKernelGGL((k_model_parity<VAR, 16>), grid, block, 0, s, A); break;
    case 32: hipLaunchKernelGGL((k_model_parity<VAR, 32>), grid, block, 0, s, A); break;
    case 256: hipLaunchKernelGGL((k_model_parity<VAR, 256>), grid, block, 0, s, A); break;
    default: hipLaunchKernelGGL((k_model_parity<VAR, 64>), grid, block, 0, s, A); break;
    }
    return hipGetLastError();
}

hipError_t launch_model_parity(const ModelParityArgsHost& H, hipStream_t s) {
    ModelParityArgs A;
    A.mp = H.mp;
    A.ep = H.ep;
    A.cf = H.cf;
    A.cc = H.cc;
    A.seed = H.seed;
    A.M = H.M;
    A.T = H.T;
    A.ell = H.ell;
    A.help = H.help;
    A.help_base = H.help_base;
    A.states = H.states;
    A.partials = H.partials;
    A.tr_phi_f = H.tr_phi_f;
    A.tr_phi_c = H.tr_phi_c;
    A.tr_nf = H.tr_nf;
    A.tr_nc = H.tr_nc;
    if (H.mp.variant == MODEL_REF) return launch_var<MODEL_REF>(A, H.G, H.blocks, s);
    return launch_var<MODEL_SHIFT>(A, H.G, H.blocks, s);
}

}  // namespace nmlmc
