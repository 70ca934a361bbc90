"""Plain form on books with Unbiased options: the wave's windows of sync words, the
waiting normals and the two ways paths are run give the reference's draws.

Per-sample results and the streams after each call (the next call starts there)
against the oracle.  The cases put inner counts at the edges of a window (62 to 66
and several windows), step counts of either parity (an odd number of normals
leaves one waiting), many deep levels (long paths: batches of 126 steps, with a
remainder; coarse steps longer than a batch), uniform sub-sampling and Asians.
Tolerance 1e-9 relative, as for every book with Unbiased options: a last-place
difference of the device's exp, log or sqrt is divided by the level's
probability."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library, to_oracle

pytestmark = pytest.mark.gpu

RTOL = 1e-9


@pytest.mark.parametrize("h0inv,beta,expo,subsample,asian,N0,counts", [
    (8, 4, -1.5, 1, False, 62, (6, 10, 8)),
    (8, 4, -1.5, 1, False, 65, (0, 0, 12)),
    (7, 4, -1.2, 1, False, 33, (3, 5, 9)),
    (3, 3, -1.1, -1, True, 64, (2, 7, 9)),
    (50, 2, -1.1, 1, True, 16, (0, 4, 9)),
    (1, 2, -1.05, 1, False, 200, (4, 0, 5)),
    (4, 150, -0.6, 1, False, 16, (2, 6, 4)),
])
def test_windows_and_paths(nm, oracle_f64, h0inv, beta, expo, subsample, asian, N0, counts):
    print("case", h0inv, beta, expo, subsample, asian, N0, counts, flush=True)
    cores = 3
    d = synthetic(Q=4, counts=counts, digitals=False, seed=7 * h0inv + beta)
    if asian:
        d["type"][sum(counts[:2]):] *= 3
    scal = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=h0inv, dt_beta=beta, dt_prob_expo=expo, max_loss=0.01,
                subsample=subsample, use_delta_cv=True, use_coarse_delta_cv=False, use_antithetic_risk=True,
                use_milstein=True, phi_type=1, phi_size=1)
    nm.init_nestedmc_sampler(cores, N0, 2, 0.0, True)
    nm.set_adaptive_rule(1, 2)
    nm.set_form(nm.FORM_PLAIN)
    pf, start, delta = to_library(nm, d, **scal)
    nm.portfolio_init(pf, 11)
    o = oracle_f64.new(cores, N0, 2, 0.0, True, adapt_rule=1, cap_log2=2)
    o.portfolio_init(to_oracle(d, start, delta, **scal), 11, None)
    for ell, M in ((0, 8), (1, 5), (0, 7)):
        g = nm.sample(ell, M, trace=True)
        e = o.sample(ell, M, trace=True)
        assert np.array_equal(g["stats"], e["stats"]), (g["stats"], e["stats"])
        assert np.array_equal(g["nf"], e["nf"]) and np.array_equal(g["nc"], e["nc"])
        np.testing.assert_allclose(g["work"], e["work"], rtol=1e-12)
        scale = max(1.0, float(np.max(np.abs(e["phi_f"]))))
        np.testing.assert_allclose(g["phi_f"], e["phi_f"], rtol=RTOL, atol=0.1 * RTOL * scale)
        np.testing.assert_allclose(g["phi_c"], e["phi_c"], rtol=RTOL, atol=0.1 * RTOL * scale)
    nm.cleanup_nestedmc_sampler()
