"""Small level calls in one launch, a block an outer sample (k_b_block), against the
launch sequence on the same outer samples: counts, work, draw statistics, FP64 rechecks
and redos and indicators are equal; other losses differ by the order of the sums of
at most 2^13 terms, 2^13 2^-53 of their magnitudes (a few times the loss's scale): 1e-11."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=True, use_antithetic_risk=True, phi_size=1, subsample=1)


def _compare(nm, monkeypatch, calls, indicator):
    for ell, M in calls:
        print(ell, M, flush=True)
        res = []
        for block in "10":
            monkeypatch.setenv("NMLMC_BLOCK_CALLS", block)
            res.append((nm.sample(ell, M, outer_offset=5, trace=True), nm.mixed_stats(), nm.last_kernel_name()))
        (g, gs, gk), (w, ws, wk) = res
        assert (gk, wk) == ("k_b_block", "k_b_final")
        assert gs == ws and g["work"] == w["work"] and np.array_equal(g["stats"], w["stats"])
        assert np.array_equal(g["nf"], w["nf"]) and np.array_equal(g["nc"], w["nc"])
        for k in ("phi_f", "phi_c", "fsums", "diffsums"):
            np.testing.assert_allclose(g[k], w[k], rtol=0 if indicator and k[0] == "p" else 1e-11,
                                       atol=0 if indicator and k[0] == "p" else 1e-11)


@pytest.mark.parametrize("redo_all", [False, True])
@pytest.mark.parametrize("N0, cap, r", [(32, 6, 0.0), (6, 2, 0.0), (514, 0, 0.0), (32, 0, 1.5)])
@pytest.mark.parametrize("form, phi, variant", [("mixed", 0, 1), ("batched", 0, 1), ("batched", 1, 1), ("mixed", 0, 0)])
def test_model(nm, monkeypatch, form, phi, variant, N0, cap, r, redo_all):
    """Counts from three units a group (most lanes idle) to ones past a unit a lane, at
    either rule, odd numbers of outer samples and more of them than blocks."""
    if redo_all:
        if form != "mixed":
            pytest.skip("the redo is the mixed form's")
        monkeypatch.setenv("NMLMC_MIXED_REDO_ALL", "1")
    nm.init_nestedmc_sampler(1, N0, 4 if r else 2, r, True)
    if cap:
        nm.set_adaptive_rule(1, cap)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.model_init_ex(variant, phi, 0.5 if variant else 0.02, 2.0 if variant else 0.08, 1)
    _compare(nm, monkeypatch, [(0, 1), (0, 4097), (1, 301), (3, 77)], phi == 0)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("redo_all", [False, True])
@pytest.mark.parametrize("correlated", [False, True])
@pytest.mark.parametrize("form, phi", [("mixed", 0), ("batched", 1)])
def test_book(nm, monkeypatch, form, phi, correlated, redo_all):
    """Books of Exact options, with outer states drawn in the block (one factor) or
    by the kernel before it (a correlation factor)."""
    if redo_all:
        if form != "mixed":
            pytest.skip("the redo is the mixed form's")
        monkeypatch.setenv("NMLMC_MIXED_REDO_ALL", "1")
    nm.init_nestedmc_sampler(1, 16, 2, 0.0, True)
    nm.set_adaptive_rule(1, 3)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    pf, _, _ = to_library(nm, synthetic(Q=19, counts=(0, 300, 0), seed=9), phi_type=phi, **SCAL)
    nm.portfolio_init(pf, 3)
    if correlated:
        nm.portfolio_set_correlation(np.linalg.cholesky(0.5 * np.eye(19) + 0.5))
    _compare(nm, monkeypatch, [(0, 1), (0, 403), (1, 301), (4, 33)], phi == 0)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
