"""quantize_blocks over the block sizes of its layouts (powers of two up to
1024 in 1024-element tiles; 2048 in registers; other sizes a wave per block,
by vectors where the size is a multiple of 8 and no short one, a short last
row aside) and dequantize_blocks over its
own (powers of two, other multiples of 4, odd sizes), against the CPU oracle
bit for bit, and on an unaligned input."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as orc
from tests._helpers import bf16_bits, to_device, to_host
from tests.test_gpu_kernels import QUANTIZERS, _edge_values

pytestmark = pytest.mark.gpu

BLOCK_SIZES = [3, 4, 8, 12, 16, 24, 32, 64, 128, 192, 200, 256, 264, 448, 456, 512, 520, 576, 584, 872, 880, 1000, 1024,
               1028, 1032, 2040, 2048, 4096, 5000, 8192]


def _check(x, dtype, bs, quantizer, sr, offset=0):
    import torch

    import rollfast_amd as rf

    if dtype == "bf16":
        bits16 = bf16_bits(x)
        x = (bits16.astype(np.uint32) << 16).view(np.float32)
        xd = to_device(bits16, "bf16")
    else:
        xd = to_device(x, "f32")
    x, xd = x[offset:], xd[offset:]
    key = rf.prng.PRNGKey(5)
    qb = rf.quantize_blocks(xd, block_size=bs, quantizer=quantizer, stochastic_rounding=sr, key=key if sr else None)
    torch.cuda.synchronize()
    nb = max(1, -(-x.size // bs))
    bits = orc.random_bits(key, nb * bs) if sr else None
    codes, scales = orc.quantize(x, bs, QUANTIZERS[quantizer], bits=bits)
    np.testing.assert_array_equal(to_host(qb.scales).view(np.uint32), scales.view(np.uint32))
    np.testing.assert_array_equal(to_host(qb.values).view(np.uint8), codes.reshape(-1).view(np.uint8))
    if np.isfinite(x).all():
        ref = orc.dequantize(codes, scales, x.size, bs, QUANTIZERS[quantizer])
        np.testing.assert_array_equal(to_host(rf.dequantize_blocks(qb)).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("bs", BLOCK_SIZES)
@pytest.mark.parametrize("quantizer", list(QUANTIZERS))
def test_quantize_block_sizes(bs, quantizer):
    rng = np.random.default_rng(bs)
    for size in (1, bs, 5 * bs + 3, 40003):
        for dtype in ("f32", "bf16"):
            for sr in (False, True):
                print(f"quantize {quantizer} {dtype} block {bs} size {size} sr {sr}", flush=True)
                _check(_edge_values(rng, size), dtype, bs, quantizer, sr)


@pytest.mark.parametrize("bs", [64, 2048, 4096])
def test_quantize_unaligned_input(bs):
    rng = np.random.default_rng(bs)
    _check(_edge_values(rng, 20002), "f32", bs, "dynamic_signed", False, offset=1)


@pytest.mark.parametrize("bs", [16, 256, 1024, 2048, 4096])
@pytest.mark.parametrize("quantizer", ["dynamic_signed", "dynamic_unsigned"])
def test_quantize_special_blocks_among_ordinary(bs, quantizer):
    """Zero, tiny, infinite and NaN blocks beside ordinary ones in one wave."""
    x = _edge_values(np.random.default_rng(bs), 12 * bs)
    x[bs: 2 * bs] = 0.0
    x[3 * bs: 4 * bs] *= np.float32(1e-30)
    x[5 * bs + 3] = np.inf
    x[7 * bs + 1] = -np.inf
    x[9 * bs + 2] = np.nan
    _check(x, "f32", bs, quantizer, False)


def test_quantize_waves_of_several_tiles():
    """Enough tiles that each wave walks several, with a partial last one."""
    import torch

    import rollfast_amd as rf

    n = 256 * 32 * 4 * 1024 * 2 + 1024 * 3 + 77
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    x = torch.randn(n, generator=gen, device="cuda")
    a = rf.quantize_blocks(x, block_size=512)
    for lo in (0, n // 1024 // 2 * 1024, (n - 100_000) // 1024 * 1024):
        b = rf.quantize_blocks(x[lo: lo + 100_000].clone(), block_size=512)
        k = min(b.values.shape[0], (n - lo) // 512) - 1
        assert torch.equal(a.values[lo // 512: lo // 512 + k], b.values[:k])
        assert torch.equal(a.scales[lo // 512: lo // 512 + k], b.scales[:k])
    host = x[-(n % 512 + 512 * 9):].cpu().numpy()
    codes, scales = orc.quantize(host, 512, orc.Q_SIGNED)
    assert np.array_equal(a.values[-10:].cpu().numpy().view(np.uint8), codes.view(np.uint8))
    assert np.array_equal(a.scales[-10:].cpu().numpy(), scales)
