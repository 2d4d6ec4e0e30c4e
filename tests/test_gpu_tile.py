"""GPU parity of the step for block sizes other than 2048 against the CPU
oracle: codes, scales and (exact=True) params bit for bit, default-mode
params within one bf16 ulp.

Block sizes at the edges of the tile kernel's layouts (powers of two below
1024 in 1024-element spans; 1024 and other multiples of 8 below it a wave
each; up to 4096 a workgroup each) and just outside them; leaves of whole
spans, of a partial last block and of a partial group of 8 elements; zero,
tiny and non-finite blocks.

Blocks of up to 2048 elements go to the tile kernel in lists of more than 4
(above 512 elements), 6 (above 128) or 8 blocks per compute unit; SPEC's lists
are shorter (the generic list's kernel; another leaf takes them past the
limit in test_gpu_long_lists.py).  The trees of the second half are long, all
bf16 or of f32 params: the kernel's two dtype instances, its waves' later
spans and later runs, and the chunk prefetched between them.
"""

from __future__ import annotations

import numpy as np
import pytest

import tests.test_gpu_packed_bits as packed
import tests.test_gpu_step as step
from tests._helpers import bf16_bits, bf16_to_f32, to_device, to_host

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


BF16_SIZES = [8, 64, 256, 512, 1000, 1024, 2056, 4096]


def _long(bs, n=3400 * 1024 + 77):
    """More spans than the chip has waves; a short last span and block."""
    return [((n,), "bf16", "bf16"), ((3 * bs + 40,), "bf16", "bf16"), ((300,), "bf16", "bf16")]


@pytest.mark.parametrize("opts", [{"exact": True}, {}, {"wd": 0.0}, {"exact": True, "msr": True, "psr": True},
                                  {"psr": True, "exact": True, "nesterov": True}], ids=str)
@pytest.mark.parametrize("bs", BF16_SIZES)
def test_tile_all_bf16(bs, opts):
    """Trees of bf16 params and grads alone."""
    step._run(_long(bs), steps=1, block_size=bs, min_size=301, **opts)


@pytest.mark.parametrize("bs", [64, 512, 1000, 4096])
def test_tile_all_bf16_packed(bs):
    """Packed draws over several blocks per wave."""
    packed._run_packed(_long(bs), steps=1, msr=True, psr=True, block_size=bs)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("bs", [16, 256, 1000, 2056])
def test_tile_update_only(bs, exact):
    step._optax_mode(_long(bs) + [((5000,), "f32", "bf16")], adamw=True, exact=exact, block_size=bs, cancelling=True)
    step._optax_mode(_long(bs), adamw=False, exact=exact, block_size=bs)


@pytest.mark.parametrize("msr", [False, True])
@pytest.mark.parametrize("pdtype", ["bf16", "f32"])
@pytest.mark.parametrize("bs", [64, 512, 1000])
def test_tile_special_blocks_between_prefetched_spans(bs, pdtype, msr, monkeypatch):
    """Runs of two spans, several per wave, with a span of tiny, zero or
    non-finite blocks here and there: the next span's first chunk is already
    loaded when such a span takes the literal search."""

    def grads(spec, seed, std=1e-2):
        rng = np.random.default_rng(seed)
        host, dev = [], {}
        for i, (shape, _pd, gd) in enumerate(spec):
            g = (rng.standard_normal(int(np.prod(shape)), dtype=np.float32) * np.float32(std)).astype(np.float32)
            blocks = g[: g.size // bs * bs].reshape(-1, bs)
            blocks[3::37] *= np.float32(1e-25)
            blocks[5::41] = 0.0
            blocks[7::43, bs // 3] = np.inf
            blocks[11::47, bs // 2] = np.nan
            g = bf16_bits(g) if gd == "bf16" else g
            host.append(g)
            dev["l%03d" % i] = to_device(g, gd).reshape(shape)
        return host, dev

    def compare(spec, tree, dev_params, exact, what, before):
        for i, ((_shape, pd, _gd), L) in enumerate(zip(spec, tree.leaves)):
            got, want = to_host(dev_params["l%03d" % i]), L["param"]
            gf, wf = (bf16_to_f32(got), bf16_to_f32(want)) if pd == "bf16" else (got, want)
            both_nan = np.isnan(gf) & np.isnan(wf)
            u = np.uint16 if pd == "bf16" else np.uint32
            assert not ((got.view(u) != want.view(u)) & ~both_nan).any(), f"{what} leaf {i}"

    monkeypatch.setattr(step, "_grads", grads)
    monkeypatch.setattr(step, "_compare_params", compare)
    n = 6600 * 1024 + 333
    step._run([((n,), pdtype, "bf16")], steps=2, block_size=bs, msr=msr, exact=True)


def _blocks(per_cu, more):
    import torch

    return per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("bs,per_cu", [(8, 8), (128, 8), (136, 6), (512, 6), (520, 4), (1024, 4), (1032, 4),
                                       (2040, 4)])
def test_short_list_limit(bs, per_cu, more):
    """Both sides of the list length at which blocks move from the generic
    list to the tile kernel."""
    spec = [(((_blocks(per_cu, more) - 3) * bs,), "bf16", "bf16"), ((3 * bs - 5,), "bf16", "bf16")]
    step._run(spec, steps=2, block_size=bs, min_size=8, exact=True)
    step._run(spec, steps=1, block_size=bs, min_size=8, msr=True, psr=True, exact=True)


# ------------------------------------- blocks that no register layout holds --
GENERIC = [((4, 2048), "bf16", "bf16"), ((8965,), "bf16", "f32"), ((20011,), "f32", "f32"), ((40,), "bf16", "bf16"),
           ((11,), "f32", "bf16")]


@pytest.mark.parametrize("opts", [{"exact": True, "msr": True, "psr": True}, {"exact": True, "psr": True,
                                  "nesterov": True}, {}, {"eps_root": 1e-9}, {"nesterov": True}], ids=str)
@pytest.mark.parametrize("bs", [1001, 8192])
def test_generic_blocks(bs, opts):
    """Block sizes that are not a multiple of 8, or beyond a workgroup's
    registers: the two-pass units."""
    step._run(GENERIC, steps=2, block_size=bs, min_size=8, **opts)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("bs", [1001, 8192])
def test_generic_blocks_update_only(bs, exact):
    step._optax_mode(GENERIC, adamw=True, exact=exact, block_size=bs)


@pytest.mark.parametrize("opts", [{"exact": True}, {"exact": True, "msr": True, "psr": True}, {"nesterov": True}, {}],
                         ids=str)
@pytest.mark.parametrize("bs", [2048, 256])
def test_unaligned_leaves_beside_aligned_ones(bs, opts, monkeypatch):
    """Params and grads that are views at element 1 of their buffers (the
    two-pass units) in a tree with aligned leaves: in blocks of 2048 these
    have partial blocks in the same list, which share its workgroup words and
    staged tables."""
    import torch

    def unaligned(arr, dtype, device="cuda"):
        t = to_device(arr, dtype, device)
        if t.numel() % 3 == 0:  # some leaves stay aligned
            return t
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=device)
        buf[1:] = t
        return buf[1:]

    monkeypatch.setattr(step, "to_device", unaligned)
    spec = [((5 * 2048,), "bf16", "bf16"), ((9000,), "bf16", "bf16"), ((3 * 2048 + 77,), "f32", "f32"),
            ((12345,), "bf16", "f32"), ((6000,), "f32", "bf16"), ((100,), "bf16", "bf16")]
    step._run(spec, steps=2, block_size=bs, min_size=4096, **opts)
