"""GPU parity of the step kernel for block sizes other than 2048 against the
CPU oracle: codes, scales and (exact=True) params bit for bit, default-mode
params within one bf16 ulp.

Block sizes at the edges of the kernel's layouts (powers of two up to 1024 in
1024-element spans; other multiples of 8 below 1024 a wave each; up to 4096 a
workgroup each) and just outside them; leaves of whole spans, of a partial
last block and of a partial group of 8 elements;
zero, tiny and non-finite blocks.
"""

from __future__ import annotations

import numpy as np
import pytest

import tests.test_gpu_step as step
from tests._helpers import bf16_bits, to_device

pytestmark = pytest.mark.gpu

SIZES = [8, 16, 64, 128, 256, 512, 1024, 24, 1000, 2040, 2056, 4096, 8192, 8200]
SPEC = [
    ((4, 2048), "bf16", "bf16"),  # whole tiles
    ((8965,), "bf16", "f32"),     # a partial group of 5 elements
    ((16, 531), "f32", "f32"),    # 8496: whole groups, a partial tile
    ((40,), "bf16", "bf16"),
    ((11,), "f32", "bf16"),
]


@pytest.mark.parametrize("bs", SIZES)
def test_tile_block_sizes(bs):
    step._run(SPEC, steps=2, block_size=bs, min_size=8, exact=True)


@pytest.mark.parametrize("msr,psr,nesterov", [(True, True, False), (False, True, True), (True, False, True)])
@pytest.mark.parametrize("bs", [32, 512, 1000, 4096])
def test_tile_stochastic_and_nesterov(bs, msr, psr, nesterov):
    step._run(SPEC, steps=2, block_size=bs, min_size=8, msr=msr, psr=psr, nesterov=nesterov, exact=True)


@pytest.mark.parametrize("wd,eps_root", [(0.01, 0.0), (0.0, 0.0), (0.01, 1e-9)])
@pytest.mark.parametrize("bs", [256, 1000, 4096])
def test_tile_default_direction(bs, wd, eps_root):
    step._run(SPEC, steps=2, block_size=bs, min_size=8, wd=wd, eps_root=eps_root)


@pytest.mark.parametrize("msr", [False, True])
@pytest.mark.parametrize("bs", [64, 1024, 1000, 4096])
def test_tile_special_blocks(bs, msr, monkeypatch):
    """Zero blocks, blocks whose scale is below the table range, Inf and NaN
    grads beside ordinary blocks; the codes and scales are compared."""

    def grads(spec, seed, std=1e-2):
        rng = np.random.default_rng(seed)
        host, dev = [], {}
        for i, (shape, _pd, gd) in enumerate(spec):
            n = int(np.prod(shape))
            g = (rng.standard_normal(n) * std).astype(np.float32)
            g[: n // 4] *= np.float32(1e-25)
            g[n // 4: n // 2] = 0.0
            if i % 2 == 0:
                g[5 * n // 8] = np.inf
                g[7 * n // 8] = np.nan
            g = bf16_bits(g) if gd == "bf16" else g
            host.append(g)
            dev["l%03d" % i] = to_device(g, gd).reshape(shape)
        return host, dev

    monkeypatch.setattr(step, "_grads", grads)
    monkeypatch.setattr(step, "_compare_params", lambda *a: None)
    step._run(SPEC, steps=2, block_size=bs, min_size=8, msr=msr, exact=True)
