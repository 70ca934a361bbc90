"""The mixed form's FP32 Exact terms take stock levels in units of the stock's S0.  Books
for which that is no unit (a stock at zero or below, a strike out of a float's reach in it)
run their terms in FP64: counts and indicators of the batched FP64 form, as for any book."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=False, use_antithetic_risk=True, phi_type=0, phi_size=1,
            subsample=1)


def _zero(d):
    d["S0"][1] = 0.


def _negative(d):
    d["S0"][0] = -95.


def _strike(d):
    d["strike"][::7] = 1e30
    d["type"][::14] = 2


def _small(d):
    d["S0"][2], d["strike"][::5] = 1e-40, 1e-40


@pytest.mark.parametrize("change", [_zero, _negative, _strike, _small])
@pytest.mark.parametrize("counts", [(0, 60, 0), (5, 50, 5)])
@pytest.mark.parametrize("batch", [False, True])
def test_books_without_the_unit(nm, change, counts, batch):
    if batch and counts[0]:
        pytest.skip("one kind of batch")
    nm.init_nestedmc_sampler(1, 16, 2, 0.0, True)
    nm.set_adaptive_rule(1, 3)
    d = synthetic(Q=3, counts=counts, digitals=not counts[2], seed=8)
    change(d)
    pf = to_library(nm, d, **SCAL)[0]
    if change is _strike:  # the digitals' and calls' payoffs are 0: no loss but from puts of size 1e30
        pf.set_max_loss(-1e25)
    out = []
    for form in (nm.FORM_BATCHED, nm.FORM_MIXED):
        nm.set_form(form)
        if batch:
            other = to_library(nm, synthetic(Q=3, counts=counts, seed=9), **SCAL)[0]
            nm.batch_begin(2)
            nm.batch_stage(0, pf, 3)
            nm.batch_stage(1, other, 3)
            out.append([nm.batch_sample(ell, [M, M]) for ell, M in ((0, 400), (2, 150))])
        else:
            nm.portfolio_init(pf, 3)
            out.append([nm.sample(ell, M, outer_offset=0, trace=True) for ell, M in ((0, 400), (2, 150))])
    for a, b in zip(*out):
        for x, y in zip(a, b) if batch else ((a, b),):
            assert np.array_equal(x["stats"], y["stats"]) and x["work"] == y["work"]
            assert np.array_equal(x["fsums"], y["fsums"]) and np.array_equal(x["diffsums"], y["diffsums"])
            if not batch:
                assert np.array_equal(x["nf"], y["nf"]) and np.array_equal(x["phi_f"], y["phi_f"])
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
