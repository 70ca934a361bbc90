#!/usr/bin/env python3
"""Count the VALU operations used by bench.py's roofline (writes opcount.json).

Builds probe kernels around this package's own device functions (Threefry2x64-20,
FP64 and FP32 Box-Muller, the Exact terms) for gfx950, reads the VALU instructions of
each kernel body from the compiler's assembly listing, subtracts the probe's
load/store scaffolding, and drops the blocks that only run for rare arguments (the
library sine's large-argument reduction; the FP32 radius of the words next to 1; a
stock level next to the strike).  Counts are wave instructions, i.e. lane-ops per lane.

Per-sample algorithmic costs of the shift model (one normal per inner sample,
so half a Threefry block and half a Box-Muller pair):
  fp64  inner = (threefry + bm64_lib) / 2 + 4   (batched form: Y + z, s1 +=, s2 += d*d)
  plain inner = (threefry + bm64) / 2 + 4
  mixed inner = (threefry + polar32) / 2 + 3    (a pair's x + y and radius, each widened and
                                                 added; test rounds one more)
  outer = threefry + bm64_lib                   (one outer normal in FP64)

Per-sample costs of an Exact-GBM inner sample of the sub-sampled portfolio
(two Threefry blocks: the option uniform, then the Box-Muller pair):
  mixed = 2 threefry + bm32 + exact_mix + search + 4
          (exact_mix: the FP32 loss and its error scale from the 16-byte
          record; search: the option uniform to its guide bucket, the path of
          most draws; 4: the term and half a pair's error scale widened and added;
          test rounds some more)
  fp64  = 2 threefry + bm64 + exact_d + search + 1
          (exact_d: the FP64 loss from the 40-byte record, the weight over the
          option's probability in it)
"""
import json
import os
import re
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))

PROBE = r'''
#include "%s/csrc/rng.hpp"
using namespace nmlmc;
extern "C" __global__ void op_base(const uint64_t* in, uint64_t* out) {
    int i = threadIdx.x; out[i] = in[i] ^ in[i + 64] ^ in[i + 128]; out[i + 64] = in[i]; }
extern "C" __global__ void op_threefry(const uint64_t* in, uint64_t* out) {
    int i = threadIdx.x; u64x2 r = threefry2x64_20(in[i], 0, in[i + 64], in[i + 128]);
    out[i] = r.a; out[i + 64] = r.b; }
extern "C" __global__ void op_bm64(const uint64_t* in, double* out) {
    int i = threadIdx.x; double x, y; boxmuller_f64(in[i], in[i + 64], x, y);
    out[i] = x; out[i + 64] = y; }
extern "C" __global__ void op_bm64_lib(const uint64_t* in, double* out) {
    int i = threadIdx.x; double x, y; boxmuller_f64_lib(in[i], in[i + 64], x, y);
    out[i] = x; out[i + 64] = y; }
extern "C" __global__ void op_bm32(const uint64_t* in, float* out) {
    int i = threadIdx.x; float x, y; boxmuller_f32(in[i], in[i + 64], x, y);
    out[i] = x; out[i + 64] = y; }
extern "C" __global__ void op_polar32(const uint64_t* in, float* out) {
    int i = threadIdx.x; float s, c, r, r2; bm_polar_f32(in[i], in[i + 64], s, c, r, r2);
    out[i] = s; out[i + 64] = c; out[i + 128] = r; out[i + 192] = r2; }
'''

PROBE_PF = r'''
#include "%s/csrc/portfolio_dev.hpp"
using namespace nmlmc;
extern "C" __global__ void op_base_mix(const float* f, const uint32_t* u, float* out) {
    int i = threadIdx.x;
    float a = f[i] + f[i + 64] + f[i + 128] + (float)u[i] + f[i + 192] + f[i + 256] + f[i + 320] + f[i + 384]
              + f[i + 448] + f[i + 512] + f[i + 576];
    out[i] = a; out[i + 64] = a; }
extern "C" __global__ void op_exact_mix(const float* f, const uint32_t* u, float* out) {
    int i = threadIdx.x;
    MixRec q{f[i], f[i + 64], f[i + 128], u[i]};
    MixStock st{f[i + 192], f[i + 256], f[i + 320], f[i + 384]};
    float mag;
    float d = inner_exact_mix(q, st, true, true, f[i + 448], f[i + 512], f[i + 576], mag);
    out[i] = d; out[i + 64] = mag; }
extern "C" __global__ void op_base_d(const double* f, const uint32_t* u, double* out) {
    int i = threadIdx.x;
    double a = f[i] + f[i + 64] + f[i + 128] + f[i + 192] + f[i + 256] + f[i + 320] + f[i + 384] + f[i + 448]
               + f[i + 512] + f[i + 576] + f[i + 640] + f[i + 704] + (double)u[i];
    out[i] = a; }
extern "C" __global__ void op_exact_d(const double* f, const uint32_t* u, double* out) {
    int i = threadIdx.x;
    const ExactRec q{f[i], f[i + 64], f[i + 128], f[i + 192], u[i], 0};
    const ExactStock st{f[i + 256], f[i + 320], f[i + 384], f[i + 448], f[i + 512], f[i + 576]};
    out[i] = inner_exact_d(q, st, true, true, f[i + 640], f[i + 704], f[i + 704] * 0.5); }
extern "C" __global__ void op_base_search(const uint64_t* in, const PortfolioDevice pf, uint32_t* out) {
    int i = threadIdx.x; out[i] = (uint32_t)in[i]; }
extern "C" __global__ void op_search(const uint64_t* in, const PortfolioDevice pf, uint32_t* out) {
    int i = threadIdx.x;
    const uint32_t nb = pf.guide_nb[1];
    const double fb = u01_f64(in[i]) * pf.compute_prob[1] * pf.guide_scale[1];
    out[i] = fb < (double)(nb - 1) ? (uint32_t)fb : nb - 1; }
'''


def kernel_bodies(asm):
    res, cur = {}, None
    for line in asm.split("\n"):
        t = line.split(";")[0].strip()
        m = re.match(r"^(op_\w+):$", t)
        if m:
            cur = m.group(1)
            res[cur] = []
            continue
        if cur and t.startswith("s_endpgm"):
            cur = None
            continue
        if cur and t and (t.endswith(":") or not t.startswith((".", "/"))):
            res[cur].append(t)
    return res


def valu_count(body, skip_large_arg=False):
    """VALU instructions; optionally skip the block behind the first divergent branch
    (the rare arguments)."""
    n, skipping, skip_label = 0, False, None
    for i, t in enumerate(body):
        if t.endswith(":"):
            if skipping and t[:-1] == skip_label:
                skipping = False
            continue
        if skip_large_arg and skip_label is None and t.startswith("s_cbranch_execz"):
            skip_label = t.split()[1]
            skipping = True
            continue
        if not skipping and t.startswith("v_"):
            n += 1
    return n


def compile_asm(text):
    with tempfile.TemporaryDirectory() as d:
        src = os.path.join(d, "probe.hip")
        with open(src, "w") as f:
            f.write(text)
        out = os.path.join(d, "probe.s")
        subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17",
                        "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "--cuda-device-only", "-S", src, "-o", out],
                       check=True, stderr=subprocess.DEVNULL)
        return open(out).read()


def main():
    b = kernel_bodies(compile_asm(PROBE % HERE))
    bp = kernel_bodies(compile_asm(PROBE_PF % HERE))
    base = valu_count(b["op_base"])
    tf = valu_count(b["op_threefry"]) - base
    bm64 = valu_count(b["op_bm64"]) - base
    bm64_lib = valu_count(b["op_bm64_lib"], skip_large_arg=True) - base
    bm32 = valu_count(b["op_bm32"], skip_large_arg=True) - base
    polar32 = valu_count(b["op_polar32"], skip_large_arg=True) - base
    # The base probes combine their loads with 11 operations (FP32: 10 adds, a conversion)
    # and 13 (FP64).
    exact_mix = valu_count(bp["op_exact_mix"], skip_large_arg=True) - valu_count(bp["op_base_mix"]) + 11
    exact_d = valu_count(bp["op_exact_d"]) - valu_count(bp["op_base_d"]) + 13
    search = valu_count(bp["op_search"]) - valu_count(bp["op_base_search"])
    res = {
        "isa": "gfx950",
        "unit": "VALU wave instructions (lane-ops per lane)",
        "threefry2x64_20": tf,
        "boxmuller_f64": bm64,
        "boxmuller_f64_lib": bm64_lib,
        "boxmuller_f32": bm32,
        "bm_polar_f32": polar32,
        "shift_model": {
            "plain": {"inner": (tf + bm64) / 2 + 4, "outer": tf + bm64},
            "fp64": {"inner": (tf + bm64_lib) / 2 + 4, "outer": tf + bm64_lib},
            "mixed": {"inner": (tf + polar32) / 2 + 3, "outer": tf + bm64_lib},
        },
        "exact_mix_term": exact_mix,
        "exact_fp64_term": exact_d,
        "option_search_guide_hit": search,
        "portfolio_exact": {
            "mixed": {"inner": 2 * tf + bm32 + exact_mix + search + 4},
            "fp64": {"inner": 2 * tf + bm64 + exact_d + search + 1},
        },
    }
    path = os.path.join(HERE, "opcount.json")
    with open(path, "w") as f:
        json.dump(res, f, indent=1)
    print(json.dumps(res))


if __name__ == "__main__":
    main()
