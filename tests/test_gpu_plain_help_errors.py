"""Plain model calls with postings after a refused call: an allocation that fails leaves
an error with the runtime, which the next launch's check must not take for its own
(the blocks' counters would then run ahead of the host's copy of them)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_refused_allocation_between_posted_calls(nm, oracle_f64):
    nm.init_nestedmc_sampler(3, 32768, 2, 0.0, True)
    nm.model_init(1, 0.02, -10., 5)
    orc = oracle_f64.new(3, 32768, 2, 0.0, True)
    orc.model_init(0, 1, 0.02, -10., 5)
    lib, out, one = nm.load(), nm.Output(), (ctypes.c_double * 1)()
    for ell, M in ((0, 4), (1, 2), (0, 3)):
        print(ell, M, flush=True)
        # Trace buffers of 2^45 samples: refused before anything is launched.
        rc = lib.nmlmc_sample(0, 1 << 45, (1 << 64) - 1, ctypes.byref(out.c), one, None, None, None)
        assert rc != 0 and lib.nmlmc_last_error() == rc
        g, o = nm.sample(ell, M, trace=True), orc.sample(ell, M, trace=True)
        assert np.array_equal(g["stats"], o["stats"]) and g["work"] == o["work"]
        np.testing.assert_allclose(g["phi_f"], o["phi_f"], rtol=1e-12)
    nm.cleanup_nestedmc_sampler()
