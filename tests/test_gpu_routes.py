"""The step on both sides of the list lengths at which full 2048-blocks move
from the generic list (a workgroup per block) to k_adam8 (a wave per block):
6 blocks per CU for 16-bit params and grads rounded to nearest in the hardware
direction, 12 for their update-only form and packed param rounding and for
nearest rounding with f32 params or grads (these a step further where the
generic units would launch apart), 16 otherwise.  Every dtype instance of k_adam8 and each
option runs above its limit, against the CPU oracle (codes, scales and
exact-mode params bit for bit, default-mode params within one ulp)."""

from __future__ import annotations

import pytest

import tests.test_gpu_packed_bits as packed
import tests.test_gpu_step as step

pytestmark = pytest.mark.gpu


def _blocks(per_cu, more):
    import torch

    return per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more


@pytest.mark.parametrize("more", [0, 1])
def test_light_limit(more):
    spec = [((_blocks(6, more) - 3, 2048), "bf16", "bf16"), ((3 * 2048 + 77,), "bf16", "bf16"), ((300,), "bf16", "bf16")]
    step._run(spec, steps=2)


@pytest.mark.parametrize("more", [0, 1])
def test_middle_limit(more):
    n = _blocks(12, more) - 3
    tail = [((3 * 2048 + 77,), "bf16", "bf16"), ((300,), "bf16", "bf16")]
    step._run([((n + 3, 2048), "f32", "f32")], steps=1)  # nothing for the generic list
    step._run([((n, 2048), "f32", "bf16")] + tail, steps=1)
    step._optax_mode([((n, 2048), "bf16", "bf16")] + tail, adamw=False, exact=False)
    packed._run_packed([((n, 2048), "bf16", "bf16")] + tail, steps=1, msr=False, psr=True)


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("pdtype,gdtype,opts", [
    ("f32", "f32", {}),
    ("f32", "bf16", {"nesterov": True, "exact": True}),
    ("bf16", "f32", {"msr": True, "exact": True}),
    ("bf16", "bf16", {"psr": True, "exact": True}),
    ("bf16", "bf16", {"exact": True}),
    ("f32", "f32", {"msr": True, "exact": True}),
])
def test_heavy_limit(more, pdtype, gdtype, opts):
    spec = [((_blocks(16, more) - 3, 2048), pdtype, gdtype), ((3 * 2048 + 77,), pdtype, gdtype), ((300,), "bf16", "bf16")]
    step._run(spec, steps=1, **opts)
