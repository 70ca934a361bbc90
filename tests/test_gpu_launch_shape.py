"""The default launch shape of a batched level call: which segment the rule takes
at either side of its lines, and that the call's outer samples are those of
another split (7 units a segment): the counts and indicators are equal."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=True, use_antithetic_risk=True, phi_type=0, phi_size=1,
            subsample=1)


def _check(nm, monkeypatch, ell, M, segment):
    monkeypatch.setenv("NMLMC_BLOCK_CALLS", "0")
    got = nm.sample(ell, M, outer_offset=0, trace=True)
    assert nm.last_group_lanes() == segment, (ell, M, nm.last_group_lanes())
    monkeypatch.setenv("NMLMC_SEGMENT", "7")
    want = nm.sample(ell, M, outer_offset=0, trace=True)
    monkeypatch.delenv("NMLMC_SEGMENT")
    assert np.array_equal(got["stats"], want["stats"]) and got["work"] == want["work"]
    for k in ("nf", "nc", "phi_f", "phi_c"):
        assert np.array_equal(got[k], want[k]), (ell, M, k)


@pytest.mark.parametrize("form, cap, calls", [
    ("mixed", 6, [(0, 1023, 1), (0, 1024, 2), (0, 4096, 4), (0, 16383, 4), (0, 16384, 16), (3, 2048, 8),
                  (3, 8191, 8), (3, 8192, 16), (3, 32768, 32), (9, 1, 1), (9, 2, 2)]),
    ("mixed", 0, [(0, 1, 16), (1, 4095, 4), (1, 4096, 32), (2, 32767, 16), (2, 32768, 64)]),
    ("batched", 6, [(0, 4095, 1), (0, 4096, 2), (0, 131071, 8), (0, 131072, 16)]),
    ("batched", 0, [(0, 100, 16), (3, 255, 1), (3, 256, 2), (3, 1024, 4), (2, 32768, 64)]),
])
def test_model_segments(nm, monkeypatch, form, cap, calls):
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, True)
    if cap:
        nm.set_adaptive_rule(1, cap)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.model_init_ex(nm.MODEL_SHIFT, 0, 0.5, 2.0, 1)
    for ell, M, segment in calls:
        print(form, cap, ell, M, flush=True)
        _check(nm, monkeypatch, ell, M, segment)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("form, counts, cap, coupled, calls", [
    ("mixed", (0, 40, 0), 2, False, [(0, 255, 1), (0, 256, 2), (1, 512, 4), (2, 1024, 8), (0, 16384, 16)]),
    ("batched", (0, 40, 0), 2, False, [(0, 511, 1), (0, 512, 2), (1, 1024, 4)]),
    ("mixed", (0, 40, 0), 0, False, [(0, 1023, 1), (0, 1024, 2), (0, 4096, 4)]),
    ("mixed", (5, 20, 3), 2, False, [(0, 255, 1), (0, 256, 2), (1, 512, 4)]),
    ("mixed", (5, 20, 3), 2, True, [(0, 255, 1), (1, 512, 2), (1, 2048, 8)]),
])
def test_book_segments(nm, monkeypatch, form, counts, cap, coupled, calls):
    nm.init_nestedmc_sampler(1, 64, 2, 0.0, True)
    if cap:
        nm.set_adaptive_rule(1, cap)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    pf, _, _ = to_library(nm, synthetic(Q=3, counts=counts, digitals=counts[2] == 0, seed=9), **SCAL)
    nm.set_level_coupled_paths(coupled)
    nm.portfolio_init(pf, 3)
    for ell, M, segment in calls:
        print(form, counts, cap, ell, M, flush=True)
        _check(nm, monkeypatch, ell, M, segment)
    nm.set_level_coupled_paths(False)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
