"""A staging that fails half way (NMLMC_TEST_STAGE_FAIL: after the upload into the block of
the staged book): no book is staged after it, and the next one is whole."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=True, use_antithetic_risk=True, phi_type=1, phi_size=1,
            subsample=1)


def _book(nm, n, seed, Q=5):
    return to_library(nm, synthetic(Q=Q, counts=(0, n, 0), seed=seed), **SCAL)[0]


@pytest.mark.parametrize("Q", [5, 300])  # 300: a correlation factor outside the tables' block
def test_no_book_after_a_failure(nm, monkeypatch, Q):
    nm.init_nestedmc_sampler(1, 16, 2, 0.0, True)
    nm.set_form(nm.FORM_BATCHED if Q == 5 else nm.FORM_PLAIN)
    nm.portfolio_init(_book(nm, 40, 3, Q), 5)
    nm.portfolio_set_correlation(np.linalg.cholesky(0.5 * np.eye(Q) + 0.5))
    nm.sample(0, 100)
    other = _book(nm, 30, 4, Q)  # fits the block
    monkeypatch.setenv("NMLMC_TEST_STAGE_FAIL", "1")
    with pytest.raises(nm.NmlmcError, match="portfolio tables"):
        nm.portfolio_update_data(other)
    monkeypatch.delenv("NMLMC_TEST_STAGE_FAIL")
    with pytest.raises(nm.NmlmcError, match="no problem staged"):
        nm.sample(0, 100)
    with pytest.raises(nm.NmlmcError, match="no portfolio staged"):
        nm.portfolio_set_correlation(np.eye(Q))
    nm.portfolio_init(other, 7)
    got = nm.sample(0, 100, trace=True)
    nm.portfolio_cleanup()
    nm.portfolio_init(other, 7)
    want = nm.sample(0, 100, trace=True)
    assert np.array_equal(got["phi_f"], want["phi_f"]) and np.array_equal(got["nf"], want["nf"])
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


def test_a_staged_model_stays(nm, monkeypatch):
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, True)
    nm.set_form(nm.FORM_BATCHED)
    nm.model_init_ex(nm.MODEL_SHIFT, 0, 0.5, 2.0, 1)
    want = nm.sample(1, 200, outer_offset=0)
    monkeypatch.setenv("NMLMC_TEST_STAGE_FAIL", "1")
    with pytest.raises(nm.NmlmcError, match="portfolio tables"):
        nm.portfolio_update_data(_book(nm, 40, 3))
    got = nm.sample(1, 200, outer_offset=0)
    assert got["work"] == want["work"] and np.array_equal(got["fsums"], want["fsums"])
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
