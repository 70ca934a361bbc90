"""Staging of a book on the device: the option-search guides and the Exact
records are built by a kernel from the uploaded options, in one block of memory
that the next book takes over when it fits.

Books whose option counts lie at the edges of the guide's blocks (4 n + 1 entries
in blocks of 256) and of the records' are staged one after another in one
process, growing and shrinking, and sampled against the oracle: every inner
sample's option must be the reference search's, so counts are equal and phi agrees
to rounding: 1e-12 relative, with 1e-13 absolute (the file's other FP64
comparisons); books with Unbiased options 1e-9."""
import numpy as np
import pytest

from portfolio_util import synthetic, to_library, to_oracle

pytestmark = pytest.mark.gpu

SCAL = dict(r=0.05, rho=0.2, tau=0.02, dt_h0inv=8, dt_beta=4, dt_prob_expo=-1.5, use_coarse_delta_cv=False,
            use_milstein=True, max_loss=0.01, use_delta_cv=True, use_antithetic_risk=True, phi_type=1, phi_size=1)


@pytest.mark.parametrize("subsample", [1, -1])
@pytest.mark.parametrize("form", [0, 1])
def test_books_at_block_edges(nm, oracle_f64, form, subsample):
    books = [(0, 1, 0), (0, 63, 0), (1, 64, 0), (0, 1025, 0), (64, 65, 0), (3, 2, 5), (0, 256, 0)]
    nm.init_nestedmc_sampler(4, 16, 2, 0.0, True)
    nm.set_adaptive_rule(1, 2)
    nm.set_form(form)
    for k, counts in enumerate(books):
        print("book", counts, form, subsample, flush=True)
        d = synthetic(Q=3 + k, counts=counts, digitals=counts[2] == 0, seed=50 + k)
        scal = dict(SCAL, subsample=subsample)
        pf, start, delta = to_library(nm, d, **scal)
        nm.portfolio_init(pf, 70 + k)
        o = oracle_f64.new(4, 16, 2, 0.0, True, adapt_rule=1, cap_log2=2)
        o.portfolio_init(to_oracle(d, start, delta, **scal), 70 + k, None)
        rtol = 1e-9 if counts[2] else 1e-12
        for ell, M in ((0, 40), (1, 24)):
            g = nm.sample(ell, M, trace=True)
            e = o.sample(ell, M, keying=form, trace=True)
            assert np.array_equal(g["stats"], e["stats"]), (g["stats"], e["stats"])
            assert np.array_equal(g["nf"], e["nf"]) and np.array_equal(g["nc"], e["nc"])
            np.testing.assert_allclose(g["phi_f"], e["phi_f"], rtol=rtol, atol=0.1 * rtol)
            np.testing.assert_allclose(g["phi_c"], e["phi_c"], rtol=rtol, atol=0.1 * rtol)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


def test_refused_book_leaves_the_staged_one(nm):
    """A book that staging refuses does not touch the staged tables."""
    nm.init_nestedmc_sampler(1, 16, 2, 0.0, True)
    nm.set_form(nm.FORM_BATCHED)
    d = synthetic(counts=(0, 40, 0), seed=3)
    pf, _, _ = to_library(nm, d, **dict(SCAL, subsample=1))
    nm.portfolio_init(pf, 5)
    want = nm.sample(0, 100, outer_offset=0, trace=True)
    bad, _, _ = to_library(nm, d, **dict(SCAL, subsample=1))
    bad.ops["prob"][7] = -1.0
    with pytest.raises(nm.NmlmcError):
        nm.portfolio_update_data(bad)
    got = nm.sample(0, 100, outer_offset=0, trace=True)
    assert np.array_equal(got["phi_f"], want["phi_f"])
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
