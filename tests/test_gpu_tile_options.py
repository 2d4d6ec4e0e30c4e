"""The options of a step in blocks other than 2048, on lists long enough for the
tile kernel: fed bits, clipping, the non-finite guard (accepted, rejected and
let through) and grouped launches.  The tests are those of the other modules,
their transformations built with another block size and their trees given
another leaf (test_gpu_long_lists.py); the bars are theirs."""

from __future__ import annotations

import numpy as np
import pytest

import tests.test_gpu_finite as finite
from tests._helpers import to_host
from tests.test_gpu_clip import test_fused_clip_matches_oracle  # noqa: F401
from tests.test_gpu_finite import (  # noqa: F401
    test_guarded_fused_step_matches_oracle,
    test_rejected_step_leaves_state_and_clears_negative_zero,
)
from tests.test_gpu_groups import (  # noqa: F401
    test_grouped_step_equals_groups_one_by_one,
    test_guarded_clipped_grouped_step_equals_separate_passes,
)
from tests.test_gpu_long_lists import lengthen
from tests.test_gpu_step import test_fed_bits_equal_in_kernel_bits  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=[256, 1000, 4096])
def other_blocks(monkeypatch, request):
    if request.function is not test_rejected_update_only_step:
        lengthen(monkeypatch, request.function, block_size=request.param)
    return request.param


def test_rejected_update_only_step(other_blocks):
    """A rejected tx.update: zero updates like the grads, the moments as they
    were (spans of every kind, and a generic list beside them)."""
    import torch

    import rollfast_amd as rf

    _, params = finite._params(4)
    params["big"] = torch.zeros(3400 * 1024 + 77, dtype=torch.bfloat16, device="cuda")
    tx = rf.apply_if_finite(rf.scale_by_adam8(block_size=other_blocks), 3)
    state = tx.init(params)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    for step, poison in enumerate((None, (1, np.nan), (0, np.inf), None)):
        _, grads = finite._grads(30 + step, poison)
        grads["big"] = (torch.randn(params["big"].shape, generator=gen, device="cuda") * 1e-2).to(torch.bfloat16)
        before = {k: [to_host(t).copy() for t in (m.values, m.scales)] for k, m in state.inner_state.mu.items()
                  if isinstance(m, rf.QuantizedBlocks)}
        updates, new = tx.update(grads, state, params)
        torch.cuda.synchronize()
        assert int(new.notfinite_count) == (0 if poison is None else int(state.notfinite_count) + 1)
        for k, (values, scales) in before.items():
            m = new.inner_state.mu[k]
            if poison is None:
                assert (to_host(m.values) != values).any()
            else:
                np.testing.assert_array_equal(to_host(m.values), values)
                np.testing.assert_array_equal(to_host(m.scales), scales)
        for k, u in updates.items():
            assert u.shape == grads[k].shape and bool(to_host(u).any()) == (poison is None)
        state = new
