"""The library's own functions on the device (lib/libnmlmc_probe.so), over random arguments
and the edges of their ranges, against extended precision on the host (x87, 64-bit mantissa;
numpy's longdouble).

Bounds, in units of 2^-53 of the value unless said otherwise:
- log_unit 2: the final sum's rounding, 1, and s (f - R) below 0.18 |f| with a few roundings of
  its own; sqrt_pos 1.1: the correction step's rounding, and its residue;
- sincos_small 1 absolute (half a unit of the last sum, and the rounding of the part below
  0.08) and 2 relative; exp_d 1.25 (the last sum's half unit in the last place, at most 1, and the
  polynomial's last places), one unit in the last place of a subnormal result;
- boxmuller_f64: r = sqrt(-2 log u) within 2 / 2 + 1.1, times the sine within 1, and a rounding:
  (1 + 3.1 |s|) r <= 4.2 r;
- FP32 pairs: 2^-19.5 (1 + |z|).  Over all 2^32 high words of the angle and of the radius (low
  words 0, 2^31 and 2^32 - 1) the sine is off by at most 2^-22.33 (2^-23.32 where it is below
  2^-10), the radius by 2^-20.3, and together 2^-19.93 (1 + |z|);
- mixed sums of a draw group: the refinement's bounds e1 = 2^-19 (sab + n) and
  e2 = 2^-17 (smm + sab) + 2^-36 n, which the FP32 pairs' error above and the FP32 operations
  (2^-23 of mag) leave room for;
- the mixed Exact term: 2^-18 of its error scale, for every draw up to sigma sqrt(T) = 1."""
import ctypes as C
import os

import numpy as np
import pytest

from rng_np import threefry2x64_20

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LOG, SQRT, SINCOS, EXP, PAIR_F64, PAIR_F64_LIB, PAIR_F32 = range(7)
U = 2.0 ** -53
LD = np.longdouble


@pytest.fixture(scope="module")
def probe():
    lib = C.CDLL(os.path.join(ROOT, "nested-risk-mlmc_amd", "lib", "libnmlmc_probe.so"))
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)

    def functions(which, a, b=None):
        a = np.ascontiguousarray(a).view(np.uint64)
        b = a if b is None else np.ascontiguousarray(b).view(np.uint64)
        out = np.zeros((2, len(a)))
        assert lib.probe_functions(which, C.c_uint64(len(a)), ptr(a), ptr(b), ptr(out)) == 0
        return out

    def units(variant, f32, tau, seed, count, Y, m, u0, u1):
        n = len(Y)
        Y, m = np.ascontiguousarray(Y, np.float64), np.ascontiguousarray(m, np.uint64)
        u, out = np.ascontiguousarray([u0, u1], np.uint64), np.zeros((4, n))
        assert lib.probe_units(variant, int(f32), C.c_double(tau), C.c_uint64(seed), C.c_uint64(n),
                               C.c_uint64(count), ptr(Y), ptr(m), ptr(u), ptr(out)) == 0
        return out

    def exact(r, tau, anti, cv, params, words):
        n = params.shape[1]
        params, words, out = np.ascontiguousarray(params), np.ascontiguousarray(words), np.zeros((3, n))
        assert lib.probe_exact(C.c_uint64(n), C.c_double(r), C.c_double(tau), int(anti), int(cv), ptr(params),
                               ptr(words), ptr(out)) == 0
        return out
    return functions, units, exact


def _words(n, seed):
    rs = np.random.RandomState(seed)
    return rs.randint(0, 1 << 32, n, np.uint64) << np.uint64(32) | rs.randint(0, 1 << 32, n, np.uint64)


def _rel(got, want):
    want = np.asarray(want, LD)
    return np.abs((got - want) / np.where(want == 0, 1, want)).astype(np.float64)


def test_log(probe):
    u = np.concatenate([_words(1 << 18, 1).astype(np.float64) * 2.0 ** -64 + 2.0 ** -65,
                        2.0 ** -np.arange(0, 66.0), 1 - 2.0 ** -np.arange(1, 54.0),
                        np.nextafter(2.0 ** -np.arange(0, 60.0), 0), np.nextafter(2.0 ** -np.arange(1, 60.0), 1),
                        np.sqrt(0.5) * (1 + np.arange(-8, 9) * 2.0 ** -52)])
    got = probe[0](LOG, u)[0]
    assert got[u == 1.].max() == 0.
    assert _rel(got, np.log(u.astype(LD))).max() <= 2 * U


def test_sqrt(probe):
    rs = np.random.RandomState(2)
    v = np.concatenate([[0., 2.0 ** -1000, 2.0 ** -52, 91.], np.exp(rs.uniform(-60, 5, 1 << 18)),
                        np.arange(1, 100.) ** 2, 2.0 ** -np.arange(0, 120.)])
    got = probe[0](SQRT, v)[0]
    assert got[0] == 0.
    assert _rel(got, np.sqrt(v.astype(LD))).max() <= 1.1 * U


def test_sincos(probe):
    rs = np.random.RandomState(3)
    near = [np.nextafter(k * np.pi / 4, d) for k in range(-4, 5) for d in (-9, 9)] + [k * np.pi / 4 for k in range(-4, 5)]
    p = np.concatenate([rs.uniform(-np.pi, np.pi, 1 << 18), near, [0., 4., -4.], 2.0 ** -np.arange(0, 80.),
                        -2.0 ** -np.arange(0, 80.), np.pi / 2 * (1 + np.arange(-50, 51) * 2.0 ** -52)])
    s, c = probe[0](SINCOS, p)
    # pi itself to 64 bits is not enough next to its multiples: reduce by three parts of pi / 2.
    k = np.rint(p / (np.pi / 2))
    f = (p.astype(LD) - k * LD(np.pi / 2)) - k * LD(6.123233995736766e-17)
    f = f - k * LD(-1.4973849048591833e-33)
    q = k.astype(int) & 3
    ws = np.choose(q, [np.sin(f), np.cos(f), -np.sin(f), -np.cos(f)])
    wc = np.choose(q, [np.cos(f), -np.sin(f), -np.cos(f), np.sin(f)])
    for got, want in ((s, ws), (c, wc)):
        assert np.abs(got - want).max() <= 1 * U
        assert _rel(got, want).max() <= 2 * U


def test_exp(probe):
    rs = np.random.RandomState(4)
    x = np.concatenate([rs.uniform(-1, 1, 1 << 17), rs.uniform(-708, 709, 1 << 17), [0., -0., 709.78, -708.39],
                        np.log(2.) / 2 * np.arange(-2040, 2040), 2.0 ** -np.arange(0, 80.), -2.0 ** -np.arange(0, 80.)])
    assert _rel(probe[0](EXP, x)[0], np.exp(x.astype(LD))).max() <= 1.25 * U
    tiny = rs.uniform(-745.1, -708.4, 1000)
    assert np.abs(probe[0](EXP, tiny)[0] - np.exp(tiny.astype(LD))).max() <= 2.0 ** -1074
    assert np.all(probe[0](EXP, np.array([-745.2, -800., -1e6, -2.0 ** 29]))[0] == 0.)
    assert np.all(probe[0](EXP, np.array([709.79, 800., 1e6, 2.0 ** 29]))[0] == np.inf)


EDGES0 = np.array([0, 1, 2 ** 32, 2 ** 62 - 1, 2 ** 62, 2 ** 62 + 1, 2 ** 63 - 1, 2 ** 63, 2 ** 63 + 1, 3 * 2 ** 62, 2 ** 64 - 1,
                   2 ** 61, 2 ** 40, 2 ** 64 - 2 ** 40], np.uint64)
EDGES1 = np.array([0, 1, 2 ** 12, 2 ** 32 - 1, 2 ** 32, 2 ** 43, 2 ** 44, 2 ** 45, 2 ** 63, 0xFEFFFFFFFFFFFFFF, 0xFF00000000000000,
                   0xFF00000000000001, 2 ** 64 - 2 ** 39, 2 ** 64 - 2 ** 12, 2 ** 64 - 2, 2 ** 64 - 1], np.uint64)


def _pairs():
    e0, e1 = [g.ravel() for g in np.meshgrid(EDGES0, EDGES1)]
    a, b = _words(1 << 18, 5), _words(1 << 18, 6)
    small = _words(1 << 12, 7) >> np.uint64(44)  # u1 below 2^-44: the largest radii
    top = ~(_words(1 << 12, 8) >> np.uint64(8))  # u1 above 1 - 2^-8: the smallest
    return np.concatenate([e0, a, a[:1 << 12], a[:1 << 12]]), np.concatenate([e1, b, small, top])


def _reference(u0, u1):
    """The pair of the words' doubles in extended precision, and the radius."""
    p = (np.pi * (u0.view(np.int64).astype(np.float64) * 2.0 ** -63 + 2.0 ** -64)).astype(LD)
    u = (u1.astype(np.float64) * 2.0 ** -64 + 2.0 ** -65).astype(LD)
    r = np.sqrt(-2 * np.log(u))
    return np.sin(p) * r, np.cos(p) * r, r


def test_box_muller_f64(probe):
    u0, u1 = _pairs()
    x, y, r = _reference(u0, u1)
    for which in (PAIR_F64, PAIR_F64_LIB):
        got = probe[0](which, u0, u1)
        for g, w in zip(got, (x, y)):
            assert np.all(np.abs(g - w) <= 4.2 * U * r)


def test_box_muller_f32(probe):
    """Against the words' values, which the FP64 pair rounds where u1 is next to 1."""
    u0, u1 = _pairs()
    a = LD(np.pi) * ((u0.view(np.int64)).astype(LD) * LD(2.0) ** -63 + LD(2.0) ** -64)
    q = (~u1).astype(LD) * LD(2.0) ** -64 + LD(2.0) ** -65
    r = np.sqrt(-2 * np.where(u1 >> np.uint64(56) == 255, np.log1p(-q), np.log(u1.astype(LD) * LD(2.0) ** -64 + LD(2.0) ** -65)))
    got = probe[0](PAIR_F32, u0, u1)
    for g, w in zip(got, (np.sin(a) * r, np.cos(a) * r)):
        assert np.all(np.abs(g - w) <= 2.0 ** -19.5 * (1 + np.abs(w)))


@pytest.mark.parametrize("variant, tau", [(1, 0.5), (0, 0.02), (0, 0.5), (0, 0.98)])
@pytest.mark.parametrize("count", [2, 5, 64, 1023])
def test_mixed_sums_within_the_decision_bounds(probe, variant, tau, count):
    rs = np.random.RandomState(count)
    n = 4096
    Y = np.concatenate([rs.standard_normal(n - 6), [0., 9.5, -9.5, 2.0 ** -30, 1., -1.]])
    m, spu = np.arange(n), 2 if variant else 1
    z = np.zeros(n)
    units = (count + spu - 1) // spu
    f = probe[1](variant, True, tau, 11, count, Y, m, z, z + units)
    d = probe[1](variant, False, tau, 11, count, Y, m, z, z + units)
    s1, s2, sab, smm = f
    assert np.all(np.abs(s1 - d[0]) <= 2.0 ** -19 * (sab + count))
    assert np.all(np.abs(s2 - d[1]) <= 2.0 ** -17 * (smm + sab) + 2.0 ** -36 * count)
    assert np.all(sab * (1 + 2.0 ** -20) >= np.abs(d[0])) and np.all(smm * (1 + 2.0 ** -20) >= d[1])


@pytest.mark.parametrize("anti", [True, False])
@pytest.mark.parametrize("cv", [True, False])
@pytest.mark.parametrize("tau", [1.0 / 52, 0.2])
@pytest.mark.parametrize("level", ["fp32", "fp64"])
def test_mixed_exact_term_within_its_scale(probe, anti, cv, tau, level):
    """Vanillas and digitals near and far from the money, strikes within 2^-17 of the level
    among them (the FP64 level of the draw itself, and both sides of the window); outer levels
    that FP32 holds, and any, which the FP32 term rounds first."""
    u0, u1 = _pairs()
    n = len(u0)
    rs = np.random.RandomState(17)
    S0, T = 10.0 ** rs.uniform(-3, 5, n), rs.uniform(0.25, 4, n)
    sigma = rs.uniform(0.05, 1, n) / np.sqrt(T)
    R = np.exp(rs.normal(0, 0.3, n))
    R = R.astype(np.float32).astype(np.float64) if level == "fp32" else R
    typ = rs.choice([1., -1., 2., -2.], n)
    x, y, _ = (v.astype(np.float64) for v in _reference(u0, u1))
    drift = 0.05 - sigma * sigma / 2
    g = np.exp(sigma * np.sqrt(T - tau) * y + drift * (T - tau))
    levels = [R * S0 * g] + [S0 * np.exp(s * sigma * np.sqrt(tau) * x + drift * tau) * g for s in (1, -1)]
    at = np.choose(rs.randint(0, 3, n), levels) * (1 + rs.choice([0, 1, -1], n) * 2.0 ** rs.uniform(-24, -15, n))
    K = np.where(rs.uniform(size=n) < 0.3, at, S0 * np.exp(rs.normal(0, 0.3, n)))
    K = np.clip(K, 1e-6 * S0, 1e6 * S0)
    f, mag, d = probe[2](0.05, tau, anti, cv, np.array([S0, sigma, K, T, rs.standard_t(3, n), R, typ]), np.array([u0, u1]))
    assert np.all(np.isfinite(f)) and np.all(np.abs(f - d) <= 2.0 ** -18 * mag)


def test_error_scale_of_a_long_run(probe):
    """The scale of 2^17 pairs in one lane is that of the same pairs in 2^11 lanes: sums of
    positive FP64 terms, at most 2^17 2^-53 apart."""
    pairs, parts = 1 << 17, 1 << 11
    one = probe[1](1, True, 0.5, 3, 2 * pairs, [0.25], [9], [0], [pairs])
    u = np.arange(parts) * (pairs // parts)
    many = probe[1](1, True, 0.5, 3, 2 * pairs, np.full(parts, 0.25), np.full(parts, 9), u, u + pairs // parts)
    for k in (2, 3):
        assert abs(one[k][0] / many[k].sum() - 1) <= pairs * U
    # And it is sqrt(2) times the radii's sum, to the FP32 radii's error.
    b = np.arange(pairs, dtype=np.uint64)
    w = threefry2x64_20(0, (np.uint64(65) << np.uint64(40)) | b, 3, 9)
    r = np.sqrt(-2 * np.log(w[1].astype(np.float64) * 2.0 ** -64 + 2.0 ** -65))
    assert abs(one[2][0] / (2 * pairs * 0.25 + np.sqrt(2) * r.sum()) - 1) <= 2.0 ** -20
