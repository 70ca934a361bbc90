"""A tuned launch shape is the launch sequence's: small calls at a tuned level stay in one
launch, larger ones and those told to take the sequence take it at the tuned segment."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["mixed", "batched"])
def test_small_calls_of_a_tuned_level(nm, monkeypatch, form):
    nm.init_nestedmc_sampler(1, 32, 2, 0.0, True)
    nm.set_adaptive_rule(1, 2)
    nm.set_form(nm.FORM_MIXED if form == "mixed" else nm.FORM_BATCHED)
    nm.model_init_ex(nm.MODEL_SHIFT, 0, 0.5, 2.0, 1)
    untuned = nm.sample(2, 1000, outer_offset=0, trace=True)
    assert nm.last_kernel_name() == "k_b_block"
    S, _, _ = nm.autotune_level(2, 1000)
    small = nm.sample(2, 1000, outer_offset=0, trace=True)
    assert nm.last_kernel_name() == "k_b_block" and nm.last_group_lanes() == S
    nm.sample(2, 20000, outer_offset=0)
    assert nm.last_kernel_name() == "k_b_final" and nm.last_group_lanes() == S
    monkeypatch.setenv("NMLMC_BLOCK_CALLS", "0")
    seq = nm.sample(2, 1000, outer_offset=0, trace=True)
    assert nm.last_kernel_name() == "k_b_final" and nm.last_group_lanes() == S
    monkeypatch.delenv("NMLMC_BLOCK_CALLS")
    monkeypatch.setenv("NMLMC_SEGMENT", "8")
    nm.sample(2, 1000, outer_offset=0)
    assert nm.last_kernel_name() == "k_b_final" and nm.last_group_lanes() == 8
    for o in (small, seq):
        assert np.array_equal(o["stats"], untuned["stats"]) and np.array_equal(o["phi_f"], untuned["phi_f"])
    nm.cleanup_nestedmc_sampler()
    nm.set_form(nm.FORM_PLAIN)
