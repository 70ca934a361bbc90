"""Plain model form, draw groups long enough for the blocks to share: postings.

Per-sample results, counts and the streams after each call against the oracle, as
for any plain model call.  The reference model has one Box-Muller pair an inner
sample, the shift model half of one.  Counts lie at the edge of a posting (32768
pairs, one below), off the segments' multiples, and above 256 of the smallest
segments; one, a few and more virtual threads than outer samples; antithetic
coarse groups of their own; calls one after another on the same postings.
Max with a threshold far below the mean loss: phi is then the mean loss plus 10, on
which the oracle's sum in sequence carries 2^-53 sqrt(n) |mean| < 1e-14 for n up to
2^22 terms of mean below 0.1 (differences of phi, of size 1e-3 and less, carry the
same error and are left out).  Tolerance 1e-12 relative, as elsewhere; a segment
left out or run twice changes phi by 1e-6 and more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _cmp(g, o, values=("phi_f", "phi_c", "fsums")):
    assert np.array_equal(g["stats"], o["stats"]), (g["stats"], o["stats"])
    assert g["work"] == o["work"]
    for k in ("nf", "nc"):
        assert np.array_equal(g[k], o[k])
    for k in values:
        np.testing.assert_allclose(g[k], o[k], rtol=RTOL, atol=1e-300)


@pytest.mark.parametrize("variant,cores,N0,beta,anti,calls", [
    (0, 1, 32767, 2, True, ((0, 2), (1, 1))),
    (0, 3, 32768, 2, True, ((0, 2), (1, 4))),
    (0, 4, 33333, 3, False, ((0, 5), (1, 3), (0, 1))),
    (0, 2, 2097153, 2, True, ((0, 1),)),
    (1, 2, 65535, 2, True, ((0, 3), (1, 2))),
    (1, 5, 65537, 2, True, ((0, 6), (1, 3), (0, 2))),
])
def test_posted_groups_match_oracle(nm, oracle_f64, variant, cores, N0, beta, anti, calls):
    print("case", variant, cores, N0, beta, anti, flush=True)
    tau, ml = (0.02, -10.) if variant == 0 else (0.5, -10.)
    nm.init_nestedmc_sampler(cores, N0, beta, 0.0, anti)
    nm.model_init_ex(nm.MODEL_SHIFT if variant else nm.MODEL_REF, 1, tau, ml, 5)
    orc = oracle_f64.new(cores, N0, beta, 0.0, anti)
    orc.model_init(variant, 1, tau, ml, 5)
    for ell, M in calls:
        _cmp(nm.sample(ell, M, trace=True), orc.sample(ell, M, trace=True))
    nm.cleanup_nestedmc_sampler()


@pytest.mark.parametrize("M", [3, 64, 700])
def test_adaptive_groups_match_a_wave_each(nm, monkeypatch, M):
    """Adaptive counts up to 2^17 pairs, more and fewer blocks than run at a time: the
    posted sums against the same call with 64 lanes a virtual thread, which posts
    nothing (itself held to the oracle elsewhere)."""
    print("case", M, flush=True)
    out = []
    for wide in ("32768", "0"):
        monkeypatch.setenv("NMLMC_PLAIN_WIDE_MAX", wide)
        nm.init_nestedmc_sampler(1024, 32, 4, 1.5, True)
        nm.model_init(0, 0.02, 0.08, 9)
        out.append([nm.sample(6, M, trace=True), nm.sample(6, 2, trace=True)])
        assert nm.last_group_lanes() == (256 if wide != "0" else 64)
        nm.cleanup_nestedmc_sampler()
    for a, b in zip(*out):
        _cmp(a, b, ("phi_f", "phi_c", "fsums", "diffsums"))  # whole numbers: Indicator
