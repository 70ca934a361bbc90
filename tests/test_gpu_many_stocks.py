"""Plain books of many stocks: a block keeps every stock's level in LDS, and the outer
draw's normals where the inner loops have their scratch (16 B a stock and 256 B from some
1100 stocks on).  Books that just fill 64 KB and the 160 KB a block may have, of every kernel;
and correlated ones around the block's widths.  Against the oracle."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library, to_oracle

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=True, use_antithetic_risk=True, phi_type=1, phi_size=1,
            subsample=1)


def _check(nm, orc, Q, counts, calls, chol=None):
    print(Q, counts, flush=True)
    d = synthetic(Q=Q, counts=counts, digitals=counts[2] == 0, seed=Q)
    nm.init_nestedmc_sampler(2, 16, 2, 0.0, True)
    pf, start, delta = to_library(nm, d, **SCAL)
    nm.portfolio_init(pf, 3)
    o = orc.new(2, 16, 2, 0.0, True)
    o.portfolio_init(to_oracle(d, start, delta, **SCAL), 3, chol)
    if chol is not None:
        nm.portfolio_set_correlation(chol)
    rtol = 1e-9 if counts[2] else 1e-12
    for ell, M in calls:
        g, e = nm.sample(ell, M, trace=True), o.sample(ell, M, trace=True)
        assert np.array_equal(g["stats"], e["stats"])
        np.testing.assert_allclose(g["phi_f"], e["phi_f"], rtol=rtol, atol=rtol)
        np.testing.assert_allclose(g["phi_c"], e["phi_c"], rtol=rtol, atol=rtol)
    nm.cleanup_nestedmc_sampler()


@pytest.mark.parametrize("counts", [(0, 30, 0), (10, 20, 0), (5, 20, 5)])
def test_books_at_the_edge(nm, oracle_f64, counts):
    for lds in (65536, 163840):
        _check(nm, oracle_f64, (lds - 256) // 16, counts, ((0, 3), (1, 2)))


@pytest.mark.parametrize("Q", [1, 63, 64, 65, 128, 129, 513])
@pytest.mark.parametrize("counts", [(0, 30, 0), (10, 20, 0)])
def test_correlated_levels(nm, oracle_f64, Q, counts):
    """M = 2 of 2 virtual threads: books of Exact options take 8 waves a thread, 512 rows at a time."""
    rs = np.random.RandomState(Q)
    B = rs.uniform(-0.4, 0.4, (Q, 3))
    C = B @ B.T
    C[np.diag_indices(Q)] = 1.0
    _check(nm, oracle_f64, Q, counts, ((0, 5), (1, 2)), np.linalg.cholesky(C))
