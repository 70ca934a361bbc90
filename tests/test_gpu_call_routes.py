"""Which calls run in one launch, and where whole first groups go to one lane, at either side
of the lines; outer samples and counts are those of the launch sequence at 7 units a segment."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=True, use_antithetic_risk=True, phi_type=0, phi_size=1,
            subsample=1)


def _check(nm, monkeypatch, ell, M, kernel=None, segment=None):
    print(ell, M, flush=True)
    got = nm.sample(ell, M, outer_offset=0, trace=True)
    if kernel:
        assert nm.last_kernel_name() == kernel, (ell, M)
    if segment:
        assert nm.last_group_lanes() == segment, (ell, M, nm.last_group_lanes())
    monkeypatch.setenv("NMLMC_SEGMENT", "7")
    want = nm.sample(ell, M, outer_offset=0, trace=True)
    monkeypatch.delenv("NMLMC_SEGMENT")
    assert nm.last_kernel_name() == "k_b_final"
    assert np.array_equal(got["stats"], want["stats"])
    for k in ("nf", "nc", "phi_f", "phi_c"):
        assert np.array_equal(got[k], want[k]), (ell, M, k)


@pytest.mark.parametrize("form, variant, calls", [
    ("mixed", 1, [(4, 3072, 1), (4, 3073, 0), (5, 1024, 1), (5, 1025, 0), (6, 128, 1), (6, 129, 0), (7, 1, 0)]),
    ("mixed", 0, [(3, 3072, 1), (4, 1024, 1), (4, 1025, 0), (5, 1, 0)]),
    ("batched", 1, [(3, 3072, 1), (3, 3073, 0), (4, 128, 1), (4, 129, 0), (5, 1, 0)]),
    ("batched", 0, [(2, 3072, 1), (2, 3073, 0), (3, 128, 1), (3, 129, 0), (4, 1, 0)]),
])
def test_model_in_one_launch(nm, monkeypatch, form, variant, calls):
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, True)
    nm.set_adaptive_rule(1, 6)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.model_init_ex(variant, 0, 0.5 if variant else 0.02, 2.0 if variant else 0.08, 1)
    for ell, M, block in calls:
        _check(nm, monkeypatch, ell, M, "k_b_block" if block else "k_b_final")
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("form", ["mixed", "batched"])
@pytest.mark.parametrize("Q, correlated, calls", [
    (4, False, [(0, 2048, 1), (0, 2049, 0)]), (5, False, [(0, 1024, 1), (0, 1025, 0)]),
    (24, False, [(1, 1024, 1)]), (25, False, [(1, 1, 0)]), (100, False, [(0, 300, 0)]),
    (100, True, [(0, 2048, 1), (0, 2049, 0)]),
])
def test_book_in_one_launch(nm, monkeypatch, form, Q, correlated, calls):
    """Without a correlation factor a block's first lane draws the stocks one by one."""
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, True)
    nm.set_adaptive_rule(1, 2)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.portfolio_init(to_library(nm, synthetic(Q=Q, counts=(0, 200, 0), seed=9), **SCAL)[0], 3)
    if correlated:
        nm.portfolio_set_correlation(np.linalg.cholesky(0.5 * np.eye(Q) + 0.5))
    for ell, M, block in calls:
        _check(nm, monkeypatch, ell, M, "k_b_block" if block else "k_b_final")
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("form, variant, segment", [("mixed", 0, 4), ("batched", 0, 4), ("batched", 1, 2), ("mixed", 1, 1)])
def test_long_groups(nm, monkeypatch, form, variant, segment):
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, True)
    nm.set_adaptive_rule(1, 6)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.model_init_ex(variant, 0, 0.5 if variant else 0.02, 2.0 if variant else 0.08, 1)
    _check(nm, monkeypatch, 7, 1, "k_b_final", segment)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("form, N0, cap, calls", [
    ("batched", 20, 2, [(32767, 4), (32768, 16)]), ("batched", 50, 2, [(41943, 8), (41944, 16)]), ("batched", 20, 4, [(49151, 4), (49152, 16)]),
    ("batched", 26, 6, [(49151, 4), (49152, 16)]), ("batched", 4, 2, [(65535, 2), (65536, 8)]),
    ("mixed", 4, 2, [(65535, 4), (65536, 16)]), ("mixed", 10, 2, [(32767, 4), (32768, 8)]),
])
def test_segments_of_first_groups(nm, monkeypatch, form, N0, cap, calls):
    nm.init_nestedmc_sampler(1, N0, 2, 0.0, True)
    nm.set_adaptive_rule(1, cap)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.model_init_ex(nm.MODEL_SHIFT, 0, 0.5, 2.0, 1)
    for M, segment in calls:
        _check(nm, monkeypatch, 0, M, segment=segment)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
