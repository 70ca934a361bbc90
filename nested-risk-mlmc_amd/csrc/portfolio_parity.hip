// Plain FP64 form of the portfolio problem with the reference's keying.
//
// kernel_sample<false, portfolio::sampler> (nested_sampler.hpp:369-485) for the
// OpenMP semantics: T virtual threads, thread t owning a sync and an inner
// stream keyed {seed, t} that persist across calls, its libgomp static share
// of [0, M) walked in order.  One wavefront per virtual thread:
//   - the outer draw (portfolio_sampler.cpp:293-311) takes its normals from
//     known positions of the sync stream, one stock per lane, into LDS;
//   - an inner loop with sub-sampling and no Unbiased options draws, for
//     sample k, the method uniform from sync word P_s + k and then 1 (BS) or 3
//     (Exact: option uniform + one Box-Muller pair) inner words; lanes take
//     chunks of 64 samples and find their inner word offsets by a ballot
//     prefix count, so every draw matches the sequential reference;
//   - an inner loop with Unbiased options finds its samples' positions in the two
//     streams by windows of 64 sync words and evaluates them on all lanes
//     (general_inner);
//   - other configurations (no sub-sampling, or a cached inner normal in a book
//     without Unbiased options) run the reference loop on thread 0.
// A virtual thread may take a block of W <= 8 waves (W > 1 only for books whose
// options are all Exact, chosen when few virtual threads have outer samples):
// the outer draw's stocks and the inner loop's samples are then spread over
// the block's lanes.  With every option Exact, sample k draws method 1 from
// sync word P_s + k whatever its value, and its option uniform and Box-Muller
// pair from inner words P_i + 3k .. P_i + 3k + 2, so any lane can take any
// sample; the lanes' sums are added wave by wave in a fixed order.
#include "portfolio.hpp"
#include "portfolio_dev.hpp"

namespace nmlmc {

struct PortfolioParityArgs {
    PortfolioDevice pf;
    EngineParams ep;
    LevelCounts cf, cc;
    uint64_t seed, M;
    uint32_t T, ell;
    double bs_work;
    StreamState* states;
    Partial* partials;  // one per virtual thread (block)
    double* tr_phi_f;
    double* tr_phi_c;
    uint64_t* tr_nf;
    uint64_t* tr_nc;
};

// Waves a virtual thread may take, and the doubles of LDS scratch an inner loop
// needs: the wave sums of a block of up to kMaxW waves (3 each), or thread 0's
// broadcast (11 values).
constexpr uint32_t kMaxW = 8;
constexpr uint32_t kParityRed = 32;
static_assert(3 * kMaxW <= kParityRed && 11 <= kParityRed, "LDS reduction scratch");

struct InnerSums {
    double s1, s2, work;
    uint64_t nu, nn;
};

__device__ __forceinline__ double phi_value(int phi_type, double u, double coeff, double phi) {
    return phi_scalar(phi_type, u, coeff, phi);
}

// Kernel variants by the book's option methods: the general one; sub-sampled
// books of Exact options only (the only books given W > 1), whose kernel holds
// no BS or Unbiased code; books without Unbiased options.  Leaving code out
// keeps a kernel to a fraction of the general one's registers.
enum { PAR_GENERAL = 0, PAR_EXACT = 1, PAR_NO_UNBIASED = 2 };

// The inner loop of a sub-sampled book with Unbiased options, on one wave.  A
// sample's draws depend on its own draws: its method is one sync word and, when
// that is Unbiased, its level the next; its normals are 2 (Exact) or 1 + N
// (Unbiased, N steps at its level) of the inner stream after one word for the
// option, drawn in pairs whose second normal waits for the next sample that needs
// one.  But the words that set these positions are few, so the wave takes the
// samples by windows of 64 sync words:
//   - every lane evaluates its word both as a method and as a level; the samples'
//     first words follow from the mask of Unbiased methods (a word after the
//     method of an Unbiased sample is its level);
//   - lanes that hold a sample get its inner words by a prefix sum (whether a
//     normal waits is the parity of the odd draws before it), and its waiting
//     normal from the words of the last pair drawn before it;
//   - Black-Scholes and Exact samples are then evaluated side by side;
//   - the normals of the Unbiased samples with at most kFlat pairs (levels 0
//     and 1 by default) are computed as one list spread over all lanes, into LDS,
//     and each sample's paths run in its lane;
//   - the longer ones follow one at a time: all lanes compute the path factors of
//     kBatch steps, and six lanes run the six paths on them.
// Draws, and every operation within a sample, are those of the sequence on one
// lane; only the order of the samples' sums differs.
//
// On one lane (63 idle) a sample took some 1500 dependent instructions: the mix of
// the reference's own main (1000 options, levels 0..3, 8192 outer samples at level 0)
// 43 ms a sweep, 4.2 ms this way.
struct GeneralScratch {
    static constexpr uint32_t kFlat = 20;    // pairs of a sample of the flat list
    static constexpr uint32_t kPairs = 384;  // the list's buffer
    static constexpr uint32_t kBatch = 126;  // steps of a long path at a time (rounded down to whole coarse steps)
    double z[2 * kPairs];                    // normals; long paths: dW
    double g[kBatch], gc[kBatch];            // long paths: fine and coarse step factors
    uint8_t owner[kPairs];
};

struct LdsNormals {
    const double* z;
    double first;
    bool has_first;
    __device__ __forceinline__ double randn() {
        if (has_first) {
            has_first = false;
            return first;
        }
        return *z++;
    }
};

__device__ __forceinline__ void lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The long paths of lane ow's sample (level p.L, p.N steps; normals from inner
// word Pn, the first of them the waiting one when sb), over the wave; the owner's p
// gets the values at T and, for Asians, the averages.
__device__ __forceinline__ void long_paths(const PortfolioDevice& pf, uint64_t seed, uint64_t k1, uint32_t ow,
                                           uint64_t Pn, uint32_t sb, double sigma, double T, GeneralScratch& sc,
                                           UnbiasedPath& p) {
    const uint32_t lane = threadIdx.x & 63;
    Pn = bcast_u64(Pn, ow);
    sb = bcast_u32(sb, ow);
    const uint64_t N = bcast_u64(p.N, ow);
    const bool coarse = bcast_u32(p.L, ow) != 0;
    const uint32_t beta = coarse ? pf.dt_beta : 1;
    const double sg = bcast_f64(sigma, ow), t = bcast_f64(T, ow);
    const double mu = pf.r, dt = t / (double)N, sqrt_dt = sqrt(dt), dt_c = t / (double)(N / beta);
    const bool milstein = pf.use_milstein;
    double S = 0., A = 0.;  // lane i < 6: path i
#pragma unroll
    for (int i = 0; i < 6; i++) {
        const double v = bcast_f64(p.S[i], ow);
        if (lane == (uint32_t)i) S = v;
    }
    const uint32_t per = GeneralScratch::kBatch - GeneralScratch::kBatch % beta;
    for (uint64_t s0 = 0; s0 < N; s0 += per) {
        const uint32_t n = (uint32_t)(N - s0 < per ? N - s0 : per);
        // Step s uses normal s + 1 of the sample, number s + 1 - sb of its pairs.
        const uint64_t first = (s0 + 1 - sb) >> 1, last = (s0 + n - sb) >> 1;
        const uint64_t b = first + lane;
        if (b <= last) {  // at most 64 pairs
            double x, y;
            stream_bm_f64(seed, k1, Pn + 2 * b, x, y);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const uint64_t num = 2 * b + e + sb;  // the sample's normal number
                if (num >= s0 + 1 && num <= s0 + n) {
                    const uint32_t k = (uint32_t)(num - 1 - s0);
                    const double dW = sqrt_dt * (e ? y : x);
                    const double m = milstein ? (0.5 * (sg * sg) * (dW * dW - dt)) : 0.;
                    sc.z[k] = dW;
                    sc.g[k] = mu * dt + sg * dW + m;
                }
            }
        }
        lds_fence();
        if (coarse) {
            for (uint32_t c = lane; c < n / beta; c += 64) {
                double dW_c = 0.;
                for (uint32_t i = 0; i < beta; i++) dW_c += sc.z[c * beta + i];
                const double m = milstein ? (0.5 * (sg * sg) * (dW_c * dW_c - dt_c)) : 0.;
                sc.gc[c] = mu * dt_c + sg * dW_c + m;
            }
            lds_fence();
        }
        const double* f = lane < 3 ? sc.g : sc.gc;
        const uint32_t len = lane < 3 ? n : (coarse ? n / beta : 0);
        if (lane < 6)
            for (uint32_t k = 0; k < len; k++) {
                S += S * f[k];
                A += S;
            }
        lds_fence();
    }
#pragma unroll
    for (int i = 0; i < 6; i++) {
        const double v = bcast_f64(S, i), a = bcast_f64(A, i);
        if (lane == ow) {
            p.S[i] = v;
            if (i < 3 || coarse) p.A[i] = a / (double)(i < 3 ? N : N / beta);
        }
    }
}

__device__ __forceinline__ InnerSums general_inner(const PortfolioParityArgs& A, const double* R, uint64_t k1,
                                                   StreamState& ss, StreamState& si, uint64_t count,
                                                   GeneralScratch& sc) {
    const PortfolioDevice& pf = A.pf;
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
    double s1 = 0., s2 = 0., work = 0.;
    uint64_t nu = 0, nn = 0;
    // The waiting normal: known (si.saved), or the second of the pair at word wait_pos.
    uint32_t wait = si.is_saved;
    bool wait_known = true;
    uint64_t wait_pos = 0;
    auto add = [&](double v) {
        s1 += v;
        s2 += v * v;
    };
    for (uint64_t done = 0; done < count;) {
        const double uw = u01_f64(stream_word(A.seed, k1, ss.P + lane));
        const uint32_t method = pick_method(pf, uw * pf.prob_norm);
        const uint32_t level = unbiased_level(pf, uw);
        // Samples whose words all lie in the window, in order, at most those left.
        const uint64_t two = __ballot(method == 2), left = count - done;
        uint64_t starts = 0;
        uint32_t pos = 0, n = 0;
        while (pos < 63 && n < left) {
            const uint64_t rest = two >> pos;
            const uint32_t to2 = rest ? pos + (uint32_t)__builtin_ctzll(rest) : 64u;
            uint32_t run = (to2 < 63 ? to2 : 63) - pos;  // one-word samples before it
            if (run > left - n) run = (uint32_t)(left - n);
            if (run) starts |= (~0ull >> (64 - run)) << pos;
            pos += run;
            n += run;
            if (n < left && pos == to2 && pos < 63) {
                starts |= 1ull << pos;
                pos += 2;
                n++;
            }
        }
        ss.P += pos;
        done += n;
        const bool mine = (starts >> lane) & 1;
        const uint32_t L = (uint32_t)__shfl((int)level, (int)((lane + 1) & 63), 64);
        const bool bs = mine && method == 0, exact = mine && method == 1, unb = mine && method == 2;
        const uint64_t N = unb ? (uint64_t)pf.dt_h0inv * upow(pf.dt_beta, L) : 0;
        // Whether a normal waits before the sample; its inner words.
        const uint64_t odd = __ballot(unb && ((1 + N) & 1));
        const uint32_t sb = wait ^ ((uint32_t)__popcll(odd & below) & 1u);
        const uint64_t pairs = exact ? 1 : unb ? (1 + N - sb + 1) / 2 : 0;
        uint64_t end = mine ? 1 + 2 * pairs : 0;  // inclusive prefix sum of the words
#pragma unroll
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const uint64_t v = __shfl_up((unsigned long long)end, o, 64);
            if (lane >= o) end += v;
        }
        const uint64_t total = bcast_u64(end, 63);
        end += si.P;
        const uint64_t Pn = end - 2 * pairs;  // the sample's first normal's word
        const uint64_t drew = __ballot(pairs != 0);
        const uint64_t before = drew & below;
        const uint32_t prev = before ? 63u - (uint32_t)__clzll((long long)before) : 0u;
        const uint64_t prev_end = __shfl((unsigned long long)end, (int)prev, 64);
        double w = si.saved;
        if ((exact || unb) && sb && (before || !wait_known)) {
            double x;
            stream_bm_any_f64(A.seed, k1, before ? prev_end - 2 : wait_pos, x, w);
        }
        if (mine) {
            nu += unb ? 3 : 2;
            nn += exact ? 2 : unb ? 1 + N : 0;
        }
        uint32_t idx = 0;
        Words3 wd{};
        if (mine) {
            wd = stream_words3(A.seed, k1, Pn - 1);
            idx = pick_in_method(pf, method, u01_f64(wd.w0));
        }
        if (exact) {
            double x, y;
            boxmuller_f64(wd.w2, wd.w1, x, y);
            add(exact_term(pf, idx, R, sb ? w : x, sb ? x : y, work));
        }
        if (bs) {
            const OptionRec o = pf.options[0][idx];
            add(inner_bs_d(pf, o, R, work) / option_prob(pf, o));
        }
        // Unbiased samples of few pairs: their normals as one list.
        const bool flat = unb && pairs <= GeneralScratch::kFlat;
        uint32_t off = flat ? (uint32_t)pairs : 0;  // inclusive prefix sum of the pairs
#pragma unroll
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const uint32_t v = (uint32_t)__shfl_up((int)off, o, 64);
            if (lane >= o) off += v;
        }
        if (flat) off -= (uint32_t)pairs;
        for (uint64_t rem = __ballot(flat); rem;) {
            const uint32_t base = bcast_u32(off, (uint32_t)__builtin_ctzll(rem));
            const bool sel = ((rem >> lane) & 1) && off + (uint32_t)pairs - base <= GeneralScratch::kPairs;
            const uint64_t smask = __ballot(sel);  // the first of rem always fits
            const uint32_t lastl = 63u - (uint32_t)__clzll((long long)smask);
            const uint32_t cnt = bcast_u32(off + (uint32_t)pairs, lastl) - base;
            rem &= ~smask;
            if (sel)
                for (uint32_t k = 0; k < (uint32_t)pairs; k++) sc.owner[off - base + k] = (uint8_t)lane;
            lds_fence();
            for (uint32_t c0 = 0; c0 < cnt; c0 += 64) {
                const uint32_t c = c0 + lane;
                const int o = c < cnt ? (int)sc.owner[c] : (int)lane;
                const uint64_t oP = __shfl((unsigned long long)Pn, o, 64);
                const uint32_t oo = (uint32_t)__shfl((int)off, o, 64) - base;
                if (c < cnt) stream_bm_any_f64(A.seed, k1, oP + 2 * (uint64_t)(c - oo), sc.z[2 * c], sc.z[2 * c + 1]);
            }
            lds_fence();
            if (sel) {
                LdsNormals ln{sc.z + 2 * (off - base), w, sb != 0};
                const OptionRec o = pf.options[2][idx];
                add(inner_unbiased_at(pf, o, R, L, ln, work) / option_prob(pf, o));
            }
            lds_fence();
        }
        // Longer ones, one at a time.
        for (uint64_t rem = __ballot(unb && !flat); rem; rem &= rem - 1) {
            const uint32_t ow = (uint32_t)__builtin_ctzll(rem);
            const bool me = lane == ow;
            UnbiasedPath p;
            p.L = 0;
            p.N = 1;
            double sigma = 0., T = 1.;
            OptionRec o{};
            if (pf.dt_beta > GeneralScratch::kBatch) {  // coarse steps longer than a batch: in the lane
                if (me) {
                    DStream in;
                    in.init(A.seed, k1, 0, Pn, w, sb);
                    o = pf.options[2][idx];
                    add(inner_unbiased_at(pf, o, R, L, in, work) / option_prob(pf, o));
                }
                continue;
            }
            if (me) {
                o = pf.options[2][idx];
                double z = w;
                if (!sb) {
                    double y;
                    stream_bm_f64(A.seed, k1, Pn, z, y);
                }
                unbiased_begin(pf, o, R, L, z, work, p);
                sigma = pf.stocks[o.stock_ind].sigma;
                T = o.maturity - pf.tau;
            }
            long_paths(pf, A.seed, k1, ow, Pn, sb, sigma, T, sc, p);
            if (me) add(unbiased_end(pf, o, R, p) / option_prob(pf, o));
        }
        si.P += total;
        wait ^= (uint32_t)__popcll(odd) & 1u;
        if (drew) {
            wait_known = false;
            wait_pos = bcast_u64(end, 63u - (uint32_t)__clzll((long long)drew)) - 2;
        }
    }
    if (wait && !wait_known) {
        double x, y;
        stream_bm_f64(A.seed, k1, wait_pos, x, y);
        si.saved = y;
    }
    si.is_saved = wait;
    return InnerSums{wave_sum(s1), wave_sum(s2), wave_sum(work), wave_sum_u64(nu), wave_sum_u64(nn)};
}

// inner_sampler::sample_inner (nested_sampler.hpp:131-161) over `count` samples
// from the thread's streams (ss: sync, si: inner), block-uniform result.  red:
// LDS scratch of kParityRed doubles; sc: the general kernel's.
template <uint32_t W, int KIND>
__device__ __forceinline__ InnerSums parity_inner(const PortfolioParityArgs& A, const double* R, uint64_t k1,
                                                  StreamState& ss, StreamState& si, uint64_t count, double* red,
                                                  GeneralScratch* sc) {
    constexpr bool EXACT_ONLY = KIND == PAR_EXACT;
    const PortfolioDevice& pf = A.pf;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    InnerSums r{0., 0., 0., 0, 0};
    const bool fast = pf.subsample != 0 && !(pf.compute_prob[2] > 0) && !si.is_saved;
    if (EXACT_ONLY && fast) {
        // Every option Exact: method 1 for every sample, three inner words each.
        // A lane takes two consecutive samples, six words: three blocks when the
        // stream stands at an even word, four at an odd one, and the parity is the
        // same in all lanes.  (One sample a lane leaves neighbouring lanes at
        // different parities, which costs four blocks a sample.)
        double s1 = 0., s2 = 0., work = 0.;
        auto sample = [&](uint64_t w0, uint64_t w1, uint64_t w2) {
            const uint32_t idx = pick_in_method(pf, 1, u01_f64(w0));
            double x, y;
            boxmuller_f64(w2, w1, x, y);
            const double v = exact_term(pf, idx, R, x, y, work);
            s1 += v;
            s2 += v * v;
        };
        const bool odd = si.P & 1;
        for (uint64_t k = 2 * tid; k < count; k += 128 * W) {
            const uint64_t b = (si.P + 3 * k) >> 1;
            const u64x2 b0 = threefry2x64_20(b, 0, A.seed, k1), b1 = threefry2x64_20(b + 1, 0, A.seed, k1),
                        b2 = threefry2x64_20(b + 2, 0, A.seed, k1);
            uint64_t v0, v1, v2;
            if (!odd) {
                sample(b0.b, b0.a, b1.b);
                v0 = b1.a, v1 = b2.b, v2 = b2.a;
            } else {
                sample(b0.a, b1.b, b1.a);
                v0 = b2.b, v1 = b2.a, v2 = threefry2x64_20(b + 3, 0, A.seed, k1).b;
            }
            if (k + 1 < count) sample(v0, v1, v2);
        }
        const double a = wave_sum(s1), b = wave_sum(s2), c = wave_sum(work);
        if (lane == 0) {
            red[3 * wave] = a;
            red[3 * wave + 1] = b;
            red[3 * wave + 2] = c;
        }
        __syncthreads();
        double t1 = 0., t2 = 0., tw = 0.;
        for (uint32_t w = 0; w < W; w++) {
            t1 += red[3 * w];
            t2 += red[3 * w + 1];
            tw += red[3 * w + 2];
        }
        __syncthreads();  // red is reused by the next call
        ss.P += count;
        si.P += 3 * count;
        return InnerSums{t1, t2, tw, 2 * count, 2 * count};
    }
    if (!EXACT_ONLY && fast) {
        double s1 = 0., s2 = 0., work = 0.;
        uint64_t nn = 0;
        uint64_t base = 0;
        const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
        for (uint64_t c0 = 0; c0 < count; c0 += 64) {
            const uint64_t k = c0 + lane;
            const bool valid = k < count;
            uint32_t method = 0;
            if (valid) method = pick_method(pf, u01_f64(stream_word(A.seed, k1, ss.P + k)) * pf.prob_norm);
            const uint64_t exact = __ballot(valid && method == 1);
            const uint64_t nvalid = count - c0 < 64 ? count - c0 : 64;
            const uint64_t q = si.P + base + (valid ? lane + 2 * __popcll(exact & below) : 0);
            if (valid) {
                const Words3 w = stream_words3(A.seed, k1, q);
                const uint32_t idx = pick_in_method(pf, method, u01_f64(w.w0));
                double v;
                if (method == 1) {
                    double x, y;
                    boxmuller_f64(w.w2, w.w1, x, y);
                    v = exact_term(pf, idx, R, x, y, work);
                    nn += 2;
                } else {
                    const OptionRec o = pf.options[0][idx];
                    v = inner_bs_d(pf, o, R, work) / option_prob(pf, o);
                }
                s1 += v;
                s2 += v * v;
            }
            base += nvalid + 2 * (uint64_t)__popcll(exact);
        }
        r.s1 = wave_sum(s1);
        r.s2 = wave_sum(s2);
        r.work = wave_sum(work);
        r.nn = wave_sum_u64(nn);
        r.nu = 2 * count;
        ss.P += count;
        si.P += base;
        return r;
    }
    if constexpr (KIND == PAR_GENERAL) {
        static_assert(W == 1, "one wave a virtual thread");
        if (pf.subsample != 0) return general_inner(A, R, k1, ss, si, count, *sc);
    }
    // Reference loop on thread 0.
    if (tid == 0) {
        DStream sy, in;
        sy.init(A.seed, k1, 0, ss.P, ss.saved, ss.is_saved);
        in.init(A.seed, k1, 0, si.P, si.saved, si.is_saved);
        double s1 = 0., s2 = 0., work = 0.;
        for (uint64_t i = 0; i < count; i++) {
            double d;
            if constexpr (EXACT_ONLY) {
                // pick_option and the Exact branch of inner_sample_d: the
                // method uniform is drawn, and method 1 is the only one.
                uint32_t method, idx;
                pick_option(pf, sy, in, method, idx);
                const double z0 = in.randn();
                const double z1 = in.randn();
                d = exact_term(pf, idx, R, z0, z1, work);
            } else {
                d = inner_sample_d<KIND != PAR_NO_UNBIASED>(pf, R, sy, in, work);
            }
            s1 += d;
            s2 += d * d;
        }
        r = InnerSums{s1, s2, work, sy.nu + in.nu, sy.nn + in.nn};
        ss.P = sy.P;
        ss.saved = sy.saved;
        ss.is_saved = sy.is_saved;
        si.P = in.P;
        si.saved = in.saved;
        si.is_saved = in.is_saved;
    }
    if (W == 1) {
        r.s1 = __shfl(r.s1, 0, 64);
        r.s2 = __shfl(r.s2, 0, 64);
        r.work = __shfl(r.work, 0, 64);
        r.nu = __shfl(r.nu, 0, 64);
        r.nn = __shfl(r.nn, 0, 64);
        ss.P = __shfl(ss.P, 0, 64);
        ss.saved = __shfl(ss.saved, 0, 64);
        ss.is_saved = __shfl(ss.is_saved, 0, 64);
        si.P = __shfl(si.P, 0, 64);
        si.saved = __shfl(si.saved, 0, 64);
        si.is_saved = __shfl(si.is_saved, 0, 64);
        return r;
    }
    // W > 1: thread 0's results to the whole block through LDS.
    uint64_t* ru = reinterpret_cast<uint64_t*>(red);
    if (tid == 0) {
        red[0] = r.s1;
        red[1] = r.s2;
        red[2] = r.work;
        ru[3] = r.nu;
        ru[4] = r.nn;
        ru[5] = ss.P;
        red[6] = ss.saved;
        ru[7] = ss.is_saved;
        ru[8] = si.P;
        red[9] = si.saved;
        ru[10] = si.is_saved;
    }
    __syncthreads();
    r = InnerSums{red[0], red[1], red[2], ru[3], ru[4]};
    ss.P = ru[5];
    ss.saved = red[6];
    ss.is_saved = (uint32_t)ru[7];
    si.P = ru[8];
    si.saved = red[9];
    si.is_saved = (uint32_t)ru[10];
    __syncthreads();
    return r;
}

// Waves per SIMD the kernels are compiled for: 2.  The Exact-only kernel then keeps its two
// samples a lane in 243 to 248 VGPRs with 96 B of scratch (small book's plain sweep 8.4 ms; at
// 3, 384 B of scratch a lane, 9.3 ms; at 4, 528 B, 10.0 ms); the general one spills 387 VGPRs,
// 704 B a lane, of its window (the reference main's mix 5.7 ms; at 3 6.7 ms).
#ifndef NMLMC_PLAIN_EXACT_WAVES
#define NMLMC_PLAIN_EXACT_WAVES 2
#endif
#ifndef NMLMC_PLAIN_NO_UNBIASED_WAVES
#define NMLMC_PLAIN_NO_UNBIASED_WAVES 2
#endif
#ifndef NMLMC_PLAIN_GENERAL_WAVES
#define NMLMC_PLAIN_GENERAL_WAVES 2
#endif

// Doubles of LDS that the outer draw's normals and the inner loops' scratch take by turns.
__host__ __device__ constexpr uint32_t lds_shared_doubles(bool general, uint32_t d) {
    const uint32_t scratch = kParityRed + (general ? (uint32_t)(sizeof(GeneralScratch) / sizeof(double)) : 0u);
    return d > scratch ? d : scratch;
}
static_assert(sizeof(GeneralScratch) % sizeof(double) == 0, "LDS layout in doubles");

template <uint32_t W, int KIND>
__global__ __launch_bounds__(64 * W, (KIND == PAR_EXACT ? NMLMC_PLAIN_EXACT_WAVES : KIND == PAR_NO_UNBIASED ? NMLMC_PLAIN_NO_UNBIASED_WAVES : NMLMC_PLAIN_GENERAL_WAVES)) void k_portfolio_parity(
    PortfolioParityArgs A) {
    constexpr bool EXACT_ONLY = KIND == PAR_EXACT;
    // The moment sums, which thread 0 keeps (in registers, 32 doubles in every lane,
    // they spilled); the inner loops' scratch, and in its place z[d], the outer draw's
    // normals; R_tau[d].
    extern __shared__ double smem[];
    const PortfolioDevice& pf = A.pf;
    const EngineParams& ep = A.ep;
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    const uint64_t k1 = t;
    const uint32_t d = pf.d;
    double* f_sums = smem;
    double* d_sums = f_sums + kMaxPhi * kMaxMoments;
    double* z = d_sums + kMaxPhi * kMaxMoments;
    double* red = z;
    GeneralScratch* sc = KIND == PAR_GENERAL ? reinterpret_cast<GeneralScratch*>(red + kParityRed) : nullptr;
    double* R = z + lds_shared_doubles(KIND == PAR_GENERAL, d);
    if (tid == 0)
        for (int i = 0; i < kMaxPhi * kMaxMoments; i++) f_sums[i] = d_sums[i] = 0.;

    uint64_t q = A.M / A.T, rr = A.M % A.T;
    if (t < rr) {
        q++;
        rr = 0;
    }
    const uint64_t s0 = q * t + rr, e0 = s0 + q;
    StreamState ss = A.states[2 * t], si = A.states[2 * t + 1];
    uint64_t stats[kStatsExt] = {0, 0, 0, 0, 0, 0, 0, 0};
    double work = 0.;
    const bool fine_only = A.ell == 0;
    const uint32_t ps = pf.phi_size;

    for (uint64_t m = s0; m < e0; m++) {
        // ---- portfolio::sampler::sample_outer ----
        uint64_t used;
        if (pf.chol) {
            for (uint32_t j = tid; j < d; j += 64 * W) z[j] = normal_at_f64(A.seed, k1, ss, j);
            __syncthreads();
            for (uint32_t i = tid; i < d; i += 64 * W) {
                double a = 0.;
                for (uint32_t j = 0; j <= i; j++) a += pf.chol[(size_t)i * d + j] * z[j];
                const StockRec st = pf.stocks[i];
                R[i] = simulate_stock_d(st.S0, st.mu, st.sigma, pf.tau, pf.stau * a);
            }
            used = d;
        } else {
            const double dW_sys = pf.stau * normal_at_f64(A.seed, k1, ss, 0);
            if (d == 1) {
                if (tid == 0) R[0] = simulate_stock_d(pf.stocks[0].S0, pf.stocks[0].mu, pf.stocks[0].sigma, pf.tau, dW_sys);
                used = 1;
            } else {
                for (uint32_t i = tid; i < d; i += 64 * W) {
                    const double dW_ind = pf.stau * normal_at_f64(A.seed, k1, ss, 1 + i);
                    const double Wi = pf.rho * dW_sys + pf.s1_rho2 * dW_ind;
                    const StockRec st = pf.stocks[i];
                    R[i] = simulate_stock_d(st.S0, st.mu, st.sigma, pf.tau, Wi);
                }
                used = 1 + d;
            }
        }
        __syncthreads();
        ss = advance_normals_f64(A.seed, k1, ss, used);
        stats[5] += used;
        // constant = -max_loss - compute_delta_cv() (sequential sum, as the reference).
        double cv = 0.;
        if (pf.use_delta_cv)
            for (uint32_t i = 0; i < d; i++) cv += (R[i] - pf.stocks[i].S0) * pf.delta_coalesce[i];
        const double constant = -pf.max_loss - cv;
        // init_inner_sampler: the pre-summed BS options without sub-sampling.
        double w_det = 0.;
        double start = constant;
        if constexpr (!EXACT_ONLY)
            if (pf.subsample == 0) start += det_bs_sum(pf, R, w_det);

        // The outer sample's draw groups one after another, from one call of the
        // inner loop (inlined at the five places that the reference calls it from,
        // it outgrew the instruction cache and the registers): the test rounds of
        // the fine count (phase 0) and of the coarse one (1), then the finals (2).
        uint64_t nf = 0, nc = 0, cur = A.cf.base;
        uint64_t group = 0, groups = 1, small = 0, big = 0;
        bool f_big = true;
        double f_phi[kMaxPhi] = {}, c_phi[kMaxPhi] = {}, s1_big = 0.;
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
                    stats[0] += cur;
                }
            } else {
                n = (fine_only || ep.antithetic) ? small : group == 0 ? nf : nc;
            }
            if (!decided) {
                const InnerSums s = parity_inner<W, KIND>(A, R, k1, ss, si, n, red, sc);
                work += s.work + A.bs_work;
                stats[4] += s.nu;
                stats[5] += s.nn;
                if (phase < 2) {
                    const double tmp = phase == 0 ? A.cf.tmp : A.cc.tmp;
                    const double out_var = s.s2 / (double)(n - 1) - (s.s1 * s.s1) / (double)(n * (n - 1));
                    const double dist = start + s.s1 / (double)n;
                    const double delta2 = dist * dist / out_var;
                    const double want = A.cf.rule == 1 ? tmp / delta2 : pow(delta2, -ep.adaptive_r / 2) * tmp;
                    if (want <= (double)n) decided = true;
                    else cur *= 2;
                } else if (fine_only) {
                    phi_add(pf, start + s.s1 / (double)nf, 1., f_phi);
                } else if (ep.antithetic) {
                    const double coeff = (double)(1.f / (float)groups);
                    phi_add(pf, start + s.s1 / (double)small, coeff, f_big ? c_phi : f_phi);
                    s1_big += s.s1;
                } else {
                    phi_add(pf, start + s.s1 / (double)n, 1., group == 0 ? f_phi : c_phi);
                }
                if (phase == 2 && ++group == groups) break;
            }
            if (!decided) continue;
            if (phase == 0) {
                nf = cur;
                stats[1] += 1;
                stats[2] += (nf == A.cf.max);
                stats[3] += (nf == A.cf.base);
                cur = A.cc.base;
                phase = fine_only ? 2 : 1;
            } else {
                nc = cur;
                phase = 2;
            }
            if (phase == 2) {
                if (fine_only) {
                    small = nf;
                    stats[0] += nf;
                } else if (ep.antithetic) {
                    f_big = nf > nc;
                    big = f_big ? nf : nc;
                    small = f_big ? nc : nf;
                    groups = big / small;
                    stats[0] += big;
                } else {
                    groups = 2;
                    stats[0] += nf + nc;
                }
            }
        }
        if (!fine_only && ep.antithetic) phi_add(pf, start + s1_big / (double)big, 1., f_big ? f_phi : c_phi);
        if (tid == 0) {
            add_moments(f_phi, ps, f_sums, ep.fine_moments);
            if (!fine_only) {
                double dphi[kMaxPhi];
                for (uint32_t i = 0; i < ps; i++) dphi[i] = f_phi[i] - c_phi[i];
                add_moments(dphi, ps, d_sums, ep.diff_moments);
            }
            if (A.tr_phi_f) A.tr_phi_f[m] = f_phi[0];
            if (A.tr_phi_c) A.tr_phi_c[m] = fine_only ? 0. : c_phi[0];
            if (A.tr_nf) A.tr_nf[m] = nf;
            if (A.tr_nc) A.tr_nc[m] = nc;
        }
        __syncthreads();
    }
    if (tid == 0) {
        A.states[2 * t] = ss;
        A.states[2 * t + 1] = si;
        Partial& p = A.partials[t];
        for (int i = 0; i < kMaxPhi * kMaxMoments; i++) {
            p.f[i] = f_sums[i];
            p.d[i] = d_sums[i];
        }
        p.work = work;
        for (int i = 0; i < kStatsExt; i++) p.stats[i] = stats[i];
    }
}

hipError_t launch_portfolio_parity(const PortfolioParityHost& H, hipStream_t s) {
    PortfolioParityArgs A;
    A.pf = H.pf;
    A.ep = H.ep;
    A.cf = H.cf;
    A.cc = H.cc;
    A.seed = H.seed;
    A.M = H.M;
    A.T = H.T;
    A.ell = H.ell;
    A.bs_work = H.bs_work;
    A.states = H.states;
    A.partials = H.partials;
    A.tr_phi_f = H.tr_phi_f;
    A.tr_phi_c = H.tr_phi_c;
    A.tr_nf = H.tr_nf;
    A.tr_nc = H.tr_nc;
    // Waves per virtual thread: more than one only for books whose options are
    // all Exact, while the virtual threads with outer samples (min(M, T)) are
    // too few to fill the device: up to kMaxW, doubling while they stay within
    // a budget of 6144 waves (the small book's plain sweep takes 9.8 ms at a budget
    // of 1024, 8.8 at 2048, 8.6 at 6144 and 8.6 at 12288).
    // NMLMC_PLAIN_WAVE_BUDGET and NMLMC_PLAIN_WAVES (1, 2, 4 or 8) override it;
    // per-sample results do not depend on it.
    uint32_t W = 1;
    const bool exact_only = H.pf.subsample != 0 && H.pf.nopt[0] == 0 && H.pf.nopt[2] == 0;
    if (exact_only) {
        const uint64_t act = H.M < (uint64_t)H.T ? H.M : (uint64_t)H.T;
        uint64_t budget = 6144;
        if (const char* env = getenv("NMLMC_PLAIN_WAVE_BUDGET")) budget = strtoull(env, nullptr, 10);
        uint32_t wmax = kMaxW;
        if (const char* env = getenv("NMLMC_PLAIN_WAVES_MAX")) wmax = (uint32_t)strtoul(env, nullptr, 10);
        while (W < wmax && W < kMaxW && act * (2 * W) <= budget) W *= 2;
        if (const char* env = getenv("NMLMC_PLAIN_WAVES")) {
            const uint32_t v = (uint32_t)strtoul(env, nullptr, 10);
            W = (v >= 8) ? 8 : (v >= 4) ? 4 : (v >= 2) ? 2 : 1;
        }
    }
    // 16 B a stock and 256 B from some 1100 stocks on: 10224 stocks fill a block's 160 KB.
    const bool general = !exact_only && H.pf.nopt[2] != 0;
    const size_t lds = sizeof(double) * ((size_t)H.pf.d + lds_shared_doubles(general, H.pf.d) + 2 * kMaxPhi * kMaxMoments);
    switch (W) {
    case 8: hipLaunchKernelGGL((k_portfolio_parity<8, PAR_EXACT>), dim3(H.blocks), dim3(512), lds, s, A); break;
    case 4: hipLaunchKernelGGL((k_portfolio_parity<4, PAR_EXACT>), dim3(H.blocks), dim3(256), lds, s, A); break;
    case 2: hipLaunchKernelGGL((k_portfolio_parity<2, PAR_EXACT>), dim3(H.blocks), dim3(128), lds, s, A); break;
    default:
        if (exact_only)
            hipLaunchKernelGGL((k_portfolio_parity<1, PAR_EXACT>), dim3(H.blocks), dim3(64), lds, s, A);
        else if (!general)
            hipLaunchKernelGGL((k_portfolio_parity<1, PAR_NO_UNBIASED>), dim3(H.blocks), dim3(64), lds, s, A);
        else
            hipLaunchKernelGGL((k_portfolio_parity<1, PAR_GENERAL>), dim3(H.blocks), dim3(64), lds, s, A);
        break;
    }
    return hipGetLastError();
}

// sampler::sample_delta_unbiased (portfolio_sampler.cpp:397-444): pathwise
// delta of an Unbiased option from an antithetic pair, dt_h0inv Milstein steps
// (volatility sigma and -sigma) against the exact GBM paths driven by the same
// Brownian increment.
__device__ double delta_unbiased_d(const PortfolioDevice& pf, const OptionRec& o, DStream& in, double& work) {
    const StockRec st = pf.stocks[o.stock_ind];
    const double r = pf.r, sigma = st.sigma;
    const double T = o.maturity - pf.tau;
    const uint64_t N = pf.dt_h0inv;
    const double dW_0_tau = pf.stau * in.randn();
    const double S1 = simulate_stock_d(st.S0, r, sigma, pf.tau, dW_0_tau);
    const double S2 = simulate_stock_d(st.S0, r, sigma, pf.tau, -dW_0_tau);
    double STf[2] = {S1, S2};
    const double sig[2] = {sigma, -sigma};
    const double dt = T / (double)N;
    const double sqrt_dt = sqrt(dt);
    double W = 0.;
    for (uint64_t n = 0; n < N; n++) {
        const double dW = sqrt_dt * in.randn();
        W += dW;
        for (int i = 0; i < 2; i++) {
            const double m = pf.use_milstein ? (0.5 * (sig[i] * sig[i]) * (dW * dW - dt)) : 0.;
            STf[i] += STf[i] * (r * dt + sig[i] * dW + m);
        }
    }
    const double ST0 = simulate_stock_d(S1, r, sigma, T, W);
    const double ST1 = simulate_stock_d(S2, r, sigma, T, -W);
    work += (double)(2 * N) * o.W_est;
    double val = 0.;
    val += derv_from_stock_d(o, STf[0], st.S0, r);
    val += derv_from_stock_d(o, STf[1], st.S0, r);
    val -= derv_from_stock_d(o, ST0, st.S0, r);
    val -= derv_from_stock_d(o, ST1, st.S0, r);
    return val / (2.0 * o.w);
}

// One lane per virtual thread t: its libgomp static share of the M samples, in
// order, from its inner stream {seed, t}; moments and work go to partials[t].
// The work is tiny (dt_h0inv steps per sample), so lanes are independent and no
// lane of a block waits on another.
__global__ __launch_bounds__(64) void k_portfolio_delta(PortfolioDeltaHost A) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= A.T) return;
    uint64_t q = A.M / A.T, rr = A.M % A.T;
    if (t < rr) {
        q++;
        rr = 0;
    }
    const uint64_t s0 = q * t + rr, e0 = s0 + q;
    StreamState si = A.states[2 * t + 1];
    DStream in;
    in.init(A.seed, t, 0, si.P, si.saved, si.is_saved);
    const OptionRec o = A.pf.options[2][A.option_index];
    double f[kMaxMoments] = {0., 0., 0., 0.};
    double work = 0.;
    for (uint64_t m = s0; m < e0; m++) {
        const double dl = delta_unbiased_d(A.pf, o, in, work);
        double p = 1.;
        for (uint32_t j = 0; j < A.moments; j++) {
            p *= dl;
            f[j] += p;
        }
    }
    si.P = in.P;
    si.saved = in.saved;
    si.is_saved = in.is_saved;
    A.states[2 * t + 1] = si;
    Partial& P = A.partials[t];
    for (int i = 0; i < kMaxPhi * kMaxMoments; i++) {
        P.f[i] = i < kMaxMoments ? f[i] : 0.;
        P.d[i] = 0.;
    }
    P.work = work;
    for (int i = 0; i < kStatsExt; i++) P.stats[i] = 0;
}

hipError_t launch_portfolio_delta(const PortfolioDeltaHost& H, hipStream_t s) {
    const uint32_t blocks = (H.T + 63) / 64;
    hipLaunchKernelGGL(k_portfolio_delta, dim3(blocks), dim3(64), 0, s, H);
    return hipGetLastError();
}

}  // namespace nmlmc
