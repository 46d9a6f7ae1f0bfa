"""SiLU-and-mul above the size from which it streams past the last-level cache, against the
same rows in calls below it (bit for bit: each row's arithmetic is the same), with strided
rows and an odd row count."""
from __future__ import annotations

import pytest
import torch

from fastkernels_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,pad", [(3701, 12288, 0), (3501, 12808, 64)])
def test_silu_and_mul_streamed(cuda, rows, d, pad):
    print(f"silu streamed {rows} x {d}", flush=True)
    assert 3 * rows * d * 2 > 256 << 20
    g = torch.Generator(device=cuda).manual_seed(rows)
    x = torch.randn(rows, 2 * d + pad, generator=g, device=cuda, dtype=torch.bfloat16)[:, :2 * d]
    out = torch.full((rows, d + pad), 7.0, device=cuda, dtype=torch.bfloat16)
    want = torch.empty(rows, d, device=cuda, dtype=torch.bfloat16)
    ops.silu_and_mul(out[:, :d], x)
    for a in range(0, rows, 1000):
        ops.silu_and_mul(want[a:a + 1000], x[a:a + 1000])
    torch.cuda.synchronize()
    assert bool(torch.equal(out[:, :d], want))
    assert bool((out[:, d:] == 7.0).all())
