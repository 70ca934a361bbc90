"""The FP64 model's differences at levels where no outer sample straddles the threshold.

With phi = max and antithetic groups they are the last places of the means, set by
the order in which the inner samples were added: part of the call's results, the
same whatever segments and launches other calls take.  Held bit by bit to digests of
phi_fine and phi_coarse (sha256, first 16 digits) and to the difference sums, at the
levels whose groups take at most two waves of the launch sequence (the sum of two is the
same in either order; with more its atomics decide, run by run).  Beyond, small calls are
one launch whose order is the same in every run.  Last: which calls the rule covers."""
import hashlib

import pytest

pytestmark = pytest.mark.gpu


def _setup(nm, phi, anti=True):
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, anti)
    nm.set_form(nm.FORM_BATCHED)
    nm.model_init_ex(nm.MODEL_SHIFT, phi, 0.5, 2.0, 1)


@pytest.mark.parametrize("ell, M, digest, diff", [
    (3, 1000, "87c83513ca07252e", "-0x1.02090ee720240p-3"),
    (4, 300, "8a6b31031c4b6821", "-0x1.cf3a29de2ca00p-9"),
    (5, 200, "9beba855a38d26b4", "0x1.0000000000000p-52"),  # residues alone, as the next two
    (6, 40, "bd6e74484f76fdf0", "0x1.0000000000000p-52"),
    (6, 100, "303e2630c0f20ed7", "0x1.0000000000000p-51"),
])
def test_bits(nm, ell, M, digest, diff):
    _setup(nm, nm.PHI_MAX)
    for _ in range(3):
        o = nm.sample(ell, M, outer_offset=7, trace=True)
        assert hashlib.sha256(o["phi_f"].tobytes() + o["phi_c"].tobytes()).hexdigest()[:16] == digest
        if M == 1000:  # differences of several sizes: their sum depends on its order
            assert abs(o["diffsums"][0] - float.fromhex(diff)) < 1e-15
        else:
            assert float(o["diffsums"][0]).hex() == diff
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("ell, M", [(7, 691), (8, 245), (9, 87)])
def test_same_in_every_run(nm, ell, M):
    _setup(nm, nm.PHI_MAX)
    runs = {(o["phi_f"].tobytes(), o["phi_c"].tobytes())
            for o in (nm.sample(ell, M, outer_offset=7, trace=True) for _ in range(12))}
    assert len(runs) == 1
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)


@pytest.mark.parametrize("phi, anti, ell, M, kernel, segment", [
    ("max", True, 6, 1954, "k_b_final", 4), ("max", True, 6, 40, "k_b_final", 4),
    ("max", True, 7, 691, "k_b_block", 8), ("max", True, 8, 245, "k_b_block", 8),  # more than two waves
    ("max", True, 5, 5525, "k_b_final", 16), ("max", True, 2, 32767, "k_b_final", 16),
    ("max", True, 2, 32768, "k_b_final", 64),          # hundreds straddle
    ("max", True, 0, 300, "k_b_block", 16),            # no differences
    ("indicator", True, 6, 1954, "k_b_block", 8),      # whole numbers
    ("max", False, 6, 300, "k_b_final", 4),            # independent groups: no residues
])
def test_calls_of_the_rule(nm, phi, anti, ell, M, kernel, segment):
    _setup(nm, nm.PHI_MAX if phi == "max" else nm.PHI_INDICATOR, anti)
    nm.sample(ell, M, outer_offset=0)
    assert (nm.last_kernel_name(), nm.last_group_lanes()) == (kernel, segment)
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
