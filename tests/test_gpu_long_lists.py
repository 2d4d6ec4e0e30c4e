"""The step's edge tests again, on trees long enough for the streaming
kernels.  A short list of full 2048-blocks runs in the generic list, a
workgroup per block, and a short list of other block sizes there too; only
beyond those limits do k_adam8 and the tile kernel take the blocks.  The
trees of the other modules are short.  Here each of them gets one more leaf,
last in leaf order (so that no other leaf's keys move): more 2048-blocks than
the largest limit (16 per compute unit), which is also past the limit of
every other block size.  The bars are those of the tests themselves.
"""

from __future__ import annotations

import pytest

import tests.test_gpu_groups as groups
from tests.test_gpu_clip import test_fused_clip_matches_oracle  # noqa: F401
from tests.test_gpu_dtypes import (  # noqa: F401
    test_adamw8_16_bit_scales_and_f16_params,
    test_adamw8_f16_and_16_bit_scales_other_block_sizes,
    test_adamw8_f16_tree_param_sr_and_clipping,
)
from tests.test_gpu_exact_midpoints import test_exact_mode_at_bf16_midpoints  # noqa: F401
from tests.test_gpu_finite import (  # noqa: F401
    test_guarded_fused_step_matches_oracle,
    test_rejected_step_leaves_state_and_clears_negative_zero,
)
from tests.test_gpu_groups import (  # noqa: F401
    test_grouped_step_equals_groups_one_by_one,
    test_guarded_clipped_grouped_step_equals_separate_passes,
)
from tests.test_gpu_packed_bits import (  # noqa: F401
    test_packed_both_roundings_block_4096,
    test_packed_moment_sr_fused_step,
    test_packed_param_sr_fused_step,
)
from tests.test_gpu_step import (  # noqa: F401
    test_block_size_4096_partial_blocks_by_workgroup,
    test_fast_direction_over_twenty_steps,
    test_fed_bits_equal_in_kernel_bits,
    test_folded_direction_wide_hyperparameters,
    test_folded_step_where_updates_cancel_params,
    test_generic_block_size_256_and_nesterov,
    test_mixed_tree_bf16_f32,
    test_moment_stochastic_rounding_matches_threefry_bits,
    test_non_finite_and_extreme_gradient_blocks,
    test_odd_block_size_and_eps_root,
    test_param_stochastic_rounding_matches_threefry_bits,
    test_weight_decay_schedule,
)
from tests.test_gpu_tile import (  # noqa: F401
    test_tile_block_sizes,
    test_tile_default_direction,
    test_tile_special_blocks,
    test_tile_stochastic_and_nesterov,
)

pytestmark = pytest.mark.gpu

PAD = "zz"


def _blocks():
    import torch

    return 16 * torch.cuda.get_device_properties(0).multi_processor_count + 5


def lengthen(monkeypatch, function, **options):
    """Another leaf in every tree of the test `function`: around rf.adamw8
    (called with `options` too) and rf.adamw8_step (zero grads, not compared),
    and, for grouped trees, in their module's own list of leaves (compared
    like the rest)."""
    import torch

    import rollfast_amd as rf

    shape = (_blocks(), 2048)
    build, step = rf.adamw8, rf.adamw8_step
    if function.__module__ == groups.__name__:
        leaves = groups.LEAVES + [(PAD, shape, "bf16", "base")]
        monkeypatch.setattr(groups, "LEAVES", leaves)
        monkeypatch.setattr(groups, "LABELS", {name: lab for name, _s, _d, lab in leaves})
        monkeypatch.setattr(rf, "adamw8", lambda *args, **kwargs: build(*args, **options, **kwargs))
        return

    pad = torch.full(shape, 0.01, dtype=torch.bfloat16, device="cuda")
    zero = torch.zeros_like(pad)

    def adamw8(*args, **kwargs):
        tx = build(*args, **options, **kwargs)
        return tx._replace(init=lambda params: tx.init({**params, PAD: pad}))

    def adamw8_step(tx, params, grads, state, *args, random_bits=None, **kwargs):
        n = len(params)
        if random_bits is not None:
            words = torch.zeros(pad.numel() + 4096, dtype=torch.int32, device="cuda").view(torch.uint32)
            random_bits = {**random_bits, n: (words, words, words)}
        params, state = step(tx, {**params, PAD: pad}, {**grads, PAD: zero}, state, *args, random_bits=random_bits,
                             **kwargs)
        params.pop(PAD)
        assert len(params) == n
        return params, state

    monkeypatch.setattr(rf, "adamw8", adamw8)
    monkeypatch.setattr(rf, "adamw8_step", adamw8_step)


@pytest.fixture(autouse=True)
def longer_tree(monkeypatch, request):
    lengthen(monkeypatch, request.function)
