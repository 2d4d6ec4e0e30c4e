"""The global-norm pre-pass at the edges of its work units: quarters of 4096
and units of 16384 elements, remainders below 8, unaligned leaves, and the
64-leaf batches of the final sum, against a NumPy restatement (f64 sum of
squares per leaf, rounded to f32, added in f32 in leaf order)."""

from __future__ import annotations

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expected(leaves):
    total = np.float32(0.0)
    for x in leaves:
        total = np.float32(total + np.float32(math.fsum((x.astype(np.float64) ** 2).tolist())))
    return np.sqrt(total)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("sizes,offset", [
    ([1, 7, 8, 9, 511, 512, 4095, 4096, 4097], 0),
    ([16383, 16384, 16385, 40001], 0),
    ([3, 4099, 16384 + 2048, 20480], 1),  # grads at an odd element: the element path
    ([13] * 63, 0), ([5] * 64, 0), ([17] * 65, 0), ([9] * 129, 0),
    ([9] * 4095, 0), ([9] * 4097, 0),     # the sums one LDS load of the final pass takes
    ([16384 * 1100 + 77], 0),             # more than 1024 units of one leaf
])
def test_norm_edges(dtype, sizes, offset):
    import torch

    import rollfast_amd as rf

    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(sizes))
    grads, host = {}, []
    for i, n in enumerate(sizes):
        g = (torch.randn(n + offset, generator=gen, device="cuda") * 0.25).to(dt)[offset:]
        grads["l%04d" % i] = g
        host.append(g.float().cpu().numpy())
    print(f"norm {dtype} {len(sizes)} leaves of up to {max(sizes)} offset {offset}", flush=True)
    stats = torch.zeros(2, device="cuda")
    tx = rf.clip_by_global_norm(1.0)
    tx.update(grads, tx.init(grads), stats=stats)
    norm = stats.cpu().numpy()[1]
    # the f64 sums in another order differ by about 1e-13, which can move one
    # f32 rounding of a leaf's sum or of the total by an ulp
    assert abs(norm - _expected(host)) <= 2.0 ** -23 * norm
