// Counter-based RNG for gfx950: Threefry2x64-20 with the reference's stream
// semantics (Random123 as used by par_omp.hpp:72-121).
//
// A stream is a key {k0, k1} and a position P = number of u64 words already
// handed out.  Word q of a stream is element 1 - (q & 1) of the block
// threefry({q >> 1, 0}, key): random_state::rand() returns cur[1] before cur[0]
// (par_omp.hpp:92-99).  randn() takes two consecutive words (first, second) and
// evaluates boxmuller(u0 = second, u1 = first) - the argument order the
// reference build produces - returning x and caching y.  Because every position
// is a pure function of (key, P), any lane can compute any draw: the reference's
// sequential stream becomes a parallel one.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nmlmc {

struct u64x2 {
    uint64_t a, b;
};

// 64-bit rotate by a compile-time amount as two v_alignbit_b32 funnel shifts
// (one per 32-bit half); a rotate by 32 is a register swap.
template <unsigned N>
__device__ __forceinline__ uint64_t rotl64(uint64_t x) {
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    uint32_t rlo, rhi;
    if constexpr (N == 32) {
        rlo = hi;
        rhi = lo;
    } else if constexpr (N < 32) {
        rhi = __builtin_amdgcn_alignbit(hi, lo, 32 - N);
        rlo = __builtin_amdgcn_alignbit(lo, hi, 32 - N);
    } else {
        rhi = __builtin_amdgcn_alignbit(lo, hi, 64 - N);
        rlo = __builtin_amdgcn_alignbit(hi, lo, 64 - N);
    }
    return ((uint64_t)rhi << 32) | rlo;
}

// Threefry2x64 with 20 rounds (Random123/threefry.h:190-293): Skein rotation
// constants {16,42,12,31,16,32,24,21}, key-schedule parity 0x1BD11BDAA9FC1A22,
// key injection every 4 rounds with the injection count added to word 1.
__device__ __forceinline__ u64x2 threefry2x64_20(uint64_t c0, uint64_t c1, uint64_t k0, uint64_t k1) {
    const uint64_t k2 = 0x1BD11BDAA9FC1A22ULL ^ k0 ^ k1;
    uint64_t x0 = c0 + k0, x1 = c1 + k1;
#define NMLMC_TF_R(R)     \
    x0 += x1;             \
    x1 = rotl64<R>(x1);   \
    x1 ^= x0;
    NMLMC_TF_R(16) NMLMC_TF_R(42) NMLMC_TF_R(12) NMLMC_TF_R(31)
    x0 += k1; x1 += k2 + 1;
    NMLMC_TF_R(16) NMLMC_TF_R(32) NMLMC_TF_R(24) NMLMC_TF_R(21)
    x0 += k2; x1 += k0 + 2;
    NMLMC_TF_R(16) NMLMC_TF_R(42) NMLMC_TF_R(12) NMLMC_TF_R(31)
    x0 += k0; x1 += k1 + 3;
    NMLMC_TF_R(16) NMLMC_TF_R(32) NMLMC_TF_R(24) NMLMC_TF_R(21)
    x0 += k1; x1 += k2 + 4;
    NMLMC_TF_R(16) NMLMC_TF_R(42) NMLMC_TF_R(12) NMLMC_TF_R(31)
    x0 += k2; x1 += k0 + 5;
#undef NMLMC_TF_R
    return {x0, x1};
}

// r123::u01 / uneg11 for W = 64 (Random123/uniform.hpp:144-180).  The scale is
// a power of two, so the product is exact and fused or unfused evaluation
// rounds identically.
__device__ __forceinline__ double u01_f64(uint64_t u) { return (double)u * 0x1p-64 + 0x1p-65; }
__device__ __forceinline__ double uneg11_f64(uint64_t u) {
    return (double)(int64_t)u * 0x1p-63 + 0x1p-64;
}
__device__ __forceinline__ float u01_f32(uint64_t u) { return (float)u * 0x1p-64f + 0x1p-65f; }

// (double)u of a 64-bit integer as one fma of its halves: the same single
// rounding, three instructions.
__device__ __forceinline__ double u64_to_f64(uint64_t u) {
    return __builtin_fma((double)(uint32_t)(u >> 32), 0x1p32, (double)(uint32_t)u);
}
__device__ __forceinline__ double i64_to_f64(uint64_t u) {
    return __builtin_fma((double)(int32_t)(u >> 32), 0x1p32, (double)(uint32_t)u);
}

// The three functions of the FP64 Box-Muller pair on just the arguments it
// meets, in straight-line code.  The reductions are the classical ones (fdlibm's log by
// s = f / (2 + f) and its cosine with the rounding of 1 - t / 2 carried, Cody and Waite's
// two-part constants); the polynomials are minimax fits computed for these ranges, which
// leave less than 2^-57.
//
// log u, u in (0, 1]: u = 2^e m with m in [sqrt(1/2), sqrt 2), f = m - 1,
// s = f / (2 + f), and log m = 2 atanh s = f - s (f - R) with R = s^2 (2/3 +
// 2/5 s^2 + ...), in which f is exact and every rounding is scaled by s < 0.18.
__device__ __forceinline__ double log_unit(double u) {
    int e = __builtin_amdgcn_frexp_exp(u);
    double m = __builtin_amdgcn_frexp_mant(u);
    const bool low = m < 0x1.6a09e667f3bcdp-1;
    m = low ? m + m : m;
    e -= low ? 1 : 0;
    const double f = m - 1., den = m + 1.;
    double y = __builtin_amdgcn_rcp(den);
    y = __builtin_fma(__builtin_fma(-den, y, 1.), y, y);
    double s = f * y;
    s = __builtin_fma(__builtin_fma(-den, s, f), y, s);
    const double t = s * s;
    double p = 0x1.2f0705f170fb3p-3;
    p = __builtin_fma(p, t, 0x1.39a1932baa49ap-3);
    p = __builtin_fma(p, t, 0x1.7466405c577d3p-3);
    p = __builtin_fma(p, t, 0x1.c71c5202b0693p-3);
    p = __builtin_fma(p, t, 0x1.24924941f8d50p-2);
    p = __builtin_fma(p, t, 0x1.999999997fd36p-2);
    p = __builtin_fma(p, t, 0x1.5555555555592p-1);
    const double k = (double)e;
    const double g = __builtin_fma(-t, p, f);
    // ln 2 in two parts, the first of 42 bits: k times it is exact.
    return __builtin_fma(k, 0x1.62e42fefa3800p-1, f - __builtin_fma(s, g, k * -0x1.ef35793c76730p-45));
}

// sqrt v for v = 0 or v >= 2^-1000: the hardware's reciprocal root, one Newton
// step for root and half reciprocal, and the residual's correction.
__device__ __forceinline__ double sqrt_pos(double v) {
    const double y = __builtin_amdgcn_rsq(fmax(v, 0x1p-1000));
    double g = v * y, h = 0.5 * y;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    return __builtin_fma(__builtin_fma(-g, g, v), h, g);
}

// sin p, cos p for |p| <= 4: p = k pi/2 + (f + fl), |f| <= pi/4.
__device__ __forceinline__ void sincos_small(double p, double& sn, double& cs) {
    const double k = __builtin_rint(p * 0x1.45f306dc9c883p-1);
    const double f0 = __builtin_fma(-k, 0x1.921fb54442d18p+0, p);  // exact
    const double f = __builtin_fma(-k, 0x1.1a62633145c07p-54, f0);
    const double fl = __builtin_fma(-k, 0x1.1a62633145c07p-54, f0 - f);
    const double t = f * f;
    double a = 0x1.5d93183f7215ap-33;
    a = __builtin_fma(a, t, -0x1.ae5e6688215c6p-26);
    a = __builtin_fma(a, t, 0x1.71de35781606bp-19);
    a = __builtin_fma(a, t, -0x1.a01a019c1202dp-13);
    a = __builtin_fma(a, t, 0x1.111111110f87dp-7);
    a = __builtin_fma(a, t, -0x1.5555555555549p-3);
    const double s0 = f + __builtin_fma(f * t, a, fl);
    double b = -0x1.8faeb5dfe0cc7p-37;
    b = __builtin_fma(b, t, 0x1.1ee9ec1888c51p-29);
    b = __builtin_fma(b, t, -0x1.27e4f80a33a2dp-22);
    b = __builtin_fma(b, t, 0x1.a01a019cb2169p-16);
    b = __builtin_fma(b, t, -0x1.6c16c16c15181p-10);
    b = __builtin_fma(b, t, 0x1.555555555554cp-5);
    const double w = __builtin_fma(-0.5, t, 1.);
    const double c0 = w + __builtin_fma(t * t, b, __builtin_fma(-0.5, t, 1. - w) - f * fl);
    const int q = (int)k;
    const bool odd = q & 1;
    const double s1 = odd ? c0 : s0, c1 = odd ? s0 : c0;
    sn = __hiloint2double(__double2hiint(s1) ^ (int)((uint32_t)(q & 2) << 30), __double2loint(s1));
    cs = __hiloint2double(__double2hiint(c1) ^ (int)((uint32_t)((q + 1) & 2) << 30), __double2loint(c1));
}

// boxmuller(uint64, uint64) (Random123/boxmuller.hpp:128-137) with the
// sincospi fallback sincos(PI * x) (boxmuller.hpp:104-107).
//
// Bound by FP64 issue (one instruction a slot; the reciprocal and the
// reciprocal root four each).  With the device library's sincos, log and sqrt
// the pair took 199 slots of 64 lanes, most of them scaling, range reduction
// and special cases that these arguments never meet; this way 94 (a Threefry
// block: 116).  The normals' error against extended precision stays what it
// was: over 2^20 pairs, edges included, at most 2.7 (rms 0.52) units of 2^-53 r.
__device__ __forceinline__ void boxmuller_f64(uint64_t u0, uint64_t u1, double& x, double& y) {
    double s, c;
    sincos_small(3.1415926535897932 * __builtin_fma(i64_to_f64(u0), 0x1p-63, 0x1p-64), s, c);
    const double r = sqrt_pos(-2. * log_unit(__builtin_fma(u64_to_f64(u1), 0x1p-64, 0x1p-65)));
    x = s * r;
    y = c * r;
}

// The same pair through the device library's functions; it differs from the one above by
// a last-place rounding in some of its values.  The model's batched FP64 form keeps it: the
// differences of calls on which no outer sample straddles the threshold are nothing but
// rounding residues of means that are equal, and with other roundings they are other
// residues (Engine::residue_segment).
__device__ __forceinline__ void boxmuller_f64_lib(uint64_t u0, uint64_t u1, double& x, double& y) {
    double s, c;
    sincos(3.1415926535897932 * uneg11_f64(u0), &s, &c);
    const double r = sqrt(-2. * log(u01_f64(u1)));
    x = s * r;
    y = c * r;
}

// FP32 Box-Muller for the mixed form: the same words, u1 -> (0,1] in float and
// u0 -> [-1,1], sin/cos(pi x) and log by the hardware's instructions, as the
// polar parts of the pair (r sn, r cs) and r2 = r^2.
//
// The angle goes in revolutions, which is what the instructions take: u0 2^-64 from
// its high word, off by at most 2^-32 for the low word and 2^-26 for the rounding of
// the high word to a float, 2^-23.3 of an angle.  The float of u1 carries a relative
// error of about 2^-24, i.e. an absolute error of that in ln u1; the radius
// r = sqrt(-2 ln u1) then has an error of about 2^-24 / r, which for u1 near 1
// (small r) would reach 100% (a word of u1 >= 2^64 - 2^39 rounds to 1: radius 0
// against an FP64 radius up to 2^-12).  Words with u1 > 1 - 2^-8 (top byte all ones,
// 2^-8 of them) therefore take the radius from q = 1 - u01(u1) = ~u1 2^-64 + 2^-65,
// whose float is accurate to 2^-24 relative: -ln(1 - q) = q (1 + q/2 + q^2/3 + q^3/4),
// truncation below 2^-33 relative for q <= 2^-8.
//
// Error of a normal z = r sn or r cs: at most 2^-19.93 (1 + |z|), from all 2^32 high
// words of either argument (low words 0, 2^31 and 2^32 - 1): sine and cosine off by at
// most 2^-22.33 (2^-23.32 where below 2^-10), the radius by 2^-21.4 below 0.1,
// 2^-22 up to 2, 2^-21 up to 4, and at the largest (2^-32 of the words) 2^-20.3.  rms over random
// words 2^-23.3.
//
// Bound by VALU issue, as the Threefry block before it.  Whole-word conversions
// (a shift, clamp and scaling each), the C functions' denormal steps and the
// correctly rounded root took 85 slots of 64 lanes after a block of 116; this
// way 11, with an error no larger: over 2^20 pairs, edges included, at most 2^-20.5
// against 2^-19.8, rms 2^-23.3 against 2^-22.9.
__device__ __forceinline__ void bm_polar_f32(uint64_t u0, uint64_t u1, float& sn, float& cs, float& r, float& r2) {
    const float h = (float)(int32_t)(u0 >> 32) * 0x1p-32f;
    sn = __builtin_amdgcn_sinf(h);
    cs = __builtin_amdgcn_cosf(h);
    const uint32_t hi = (uint32_t)(u1 >> 32), lo = (uint32_t)u1;
    const float u = __builtin_fmaf((float)hi, 0x1p-32f, __builtin_fmaf((float)lo, 0x1p-64f, 0x1p-65f));
    r2 = __builtin_amdgcn_logf(u) * -0x1.62e43p+0f;  // log2 u times -2 ln 2
    if (hi >= 0xFF000000u) {  // one wave in five meets such a lane
        const float q = __builtin_fmaf((float)~hi, 0x1p-32f, __builtin_fmaf((float)~lo, 0x1p-64f, 0x1p-65f));
        r2 = 2.f * q * (1.f + q * (0.5f + q * (0x1.555556p-2f + q * 0.25f)));
    }
    r = __builtin_amdgcn_sqrtf(r2);
}
__device__ __forceinline__ void boxmuller_f32(uint64_t u0, uint64_t u1, float& x, float& y) {
    float sn, cs, r, r2;
    bm_polar_f32(u0, u1, sn, cs, r, r2);
    x = sn * r;
    y = cs * r;
}

// Word q of the stream keyed {k0, k1}.
__device__ __forceinline__ uint64_t stream_word(uint64_t k0, uint64_t k1, uint64_t q) {
    const u64x2 b = threefry2x64_20(q >> 1, 0, k0, k1);
    return (q & 1) ? b.a : b.b;
}

// The Box-Muller pair built from words (P, P+1) of a stream.
__device__ __forceinline__ void stream_bm_f64(uint64_t k0, uint64_t k1, uint64_t P, double& x,
                                              double& y) {
    uint64_t first, second;
    if ((P & 1) == 0) {
        const u64x2 b = threefry2x64_20(P >> 1, 0, k0, k1);
        first = b.b;
        second = b.a;
    } else {
        first = stream_word(k0, k1, P);
        second = stream_word(k0, k1, P + 1);
    }
    boxmuller_f64(second, first, x, y);
}

// Words q, q + 1, q + 2 of a stream, and the Box-Muller pair of words P, P + 1,
// where the lanes of a wave stand at positions of either parity: always two
// blocks and a select (the branches on the parity would both be taken, three
// blocks a pair and four with a word before it).
struct Words3 {
    uint64_t w0, w1, w2;
};
__device__ __forceinline__ Words3 stream_words3(uint64_t k0, uint64_t k1, uint64_t q) {
    const u64x2 b0 = threefry2x64_20(q >> 1, 0, k0, k1), b1 = threefry2x64_20((q >> 1) + 1, 0, k0, k1);
    return (q & 1) ? Words3{b0.a, b1.b, b1.a} : Words3{b0.b, b0.a, b1.b};
}
__device__ __forceinline__ void stream_bm_any_f64(uint64_t k0, uint64_t k1, uint64_t P, double& x, double& y) {
    const u64x2 b0 = threefry2x64_20(P >> 1, 0, k0, k1), b1 = threefry2x64_20((P + 1) >> 1, 0, k0, k1);
    boxmuller_f64((P & 1) ? b1.b : b0.a, (P & 1) ? b0.a : b0.b, x, y);
}

// A random_state (par_omp.hpp:72-121) positioned on a keyed counter sequence:
// block b of the stream is threefry({b, c1}, {k0, k1}); word q is element
// 1 - (q & 1) of block q >> 1.  c1 = 0 for the reference keying's per-thread
// streams; c1 = (tag << 40) | unit for a batched inner unit.
struct DStream {
    uint64_t k0, k1, c1, P;
    double saved;
    uint32_t is_saved;
    uint64_t blk;
    u64x2 cur;
    uint64_t nu, nn;  // randu / randn calls (inner_stats[4], [5])

    __device__ void init(uint64_t a, uint64_t b, uint64_t c, uint64_t p, double sv, uint32_t iss) {
        k0 = a;
        k1 = b;
        c1 = c;
        P = p;
        saved = sv;
        is_saved = iss;
        blk = ~0ull;
        nu = nn = 0;
    }
    __device__ uint64_t rand() {
        const uint64_t q = P++;
        const uint64_t b = q >> 1;
        if (b != blk) {
            cur = threefry2x64_20(b, c1, k0, k1);
            blk = b;
        }
        return (q & 1) ? cur.a : cur.b;
    }
    __device__ double randn() {
        nn++;
        if (is_saved) {
            is_saved = 0;
            return saved;
        }
        const uint64_t first = rand();
        const uint64_t second = rand();
        double x, y;
        boxmuller_f64(second, first, x, y);
        is_saved = 1;
        saved = y;
        return x;
    }
    __device__ double randu() {
        nu++;
        return u01_f64(rand());
    }
    // Move past the next k normals of a normal-only run of draws (the cached
    // one first, then Box-Muller pairs): the stream is then where k randn()
    // calls leave it, its last pair computed when k ends inside one.
    __device__ void skip_normals(uint64_t k) {
        if (k == 0) return;
        if (is_saved) {
            is_saved = 0;
            k--;
        }
        P += 2 * (k >> 1);
        if (k & 1) (void)randn();
    }
};

// Persistent state of one reference stream between calls: P words handed out,
// plus the cached second normal of the last Box-Muller pair.
struct StreamState {
    uint64_t P;
    double saved;
    uint32_t is_saved;
    uint32_t pad;
};

// Uniform (wave-uniform in practice) sequential draws on a stream state.
__device__ __forceinline__ double st_randn_f64(uint64_t k0, uint64_t k1, StreamState& s) {
    if (s.is_saved) {
        s.is_saved = 0;
        return s.saved;
    }
    double x, y;
    stream_bm_f64(k0, k1, s.P, x, y);
    s.P += 2;
    s.saved = y;
    s.is_saved = 1;
    return x;
}

__device__ __forceinline__ double st_randu_f64(uint64_t k0, uint64_t k1, StreamState& s) {
    return u01_f64(stream_word(k0, k1, s.P++));
}

// Normal number n (0-based) of the normal-only draw sequence that starts at
// state s: normal 0 is the cached one when s.is_saved, the rest come in
// Box-Muller pairs from words P, P+2, ...
__device__ __forceinline__ double normal_at_f64(uint64_t k0, uint64_t k1, const StreamState& s,
                                                uint64_t n) {
    if (s.is_saved) {
        if (n == 0) return s.saved;
        n -= 1;
    }
    double x, y;
    stream_bm_f64(k0, k1, s.P + 2 * (n >> 1), x, y);
    return (n & 1) ? y : x;
}

// State after consuming k normals from s (normal-only consumption).
__device__ __forceinline__ StreamState advance_normals_f64(uint64_t k0, uint64_t k1, StreamState s,
                                                           uint64_t k) {
    if (k == 0) return s;
    if (s.is_saved) {
        s.is_saved = 0;
        k -= 1;
    }
    const uint64_t pairs = (k + 1) >> 1;
    if (k & 1) {
        double x, y;
        stream_bm_f64(k0, k1, s.P + 2 * (pairs - 1), x, y);
        s.saved = y;
        s.is_saved = 1;
    }
    s.P += 2 * pairs;
    return s;
}

}  // namespace nmlmc
