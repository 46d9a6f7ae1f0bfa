"""Ragged prefill launches of up to 64 sequences dispatch their items longest first; larger
batches keep the grid's own order.  The order must only permute the work: the same
sequences followed by enough empty ones to pass 64 (the general path) give the same
bits; each case checks that its two launches take the two orders.  Lengths cover empty sequences, one token, block edges, ties, fewer keys than
queries, and causal pairs beside unpaired blocks."""
from __future__ import annotations

import pytest
import torch

from fastkernels_amd import _native, ops

pytestmark = pytest.mark.gpu

# (label, query lengths, key lengths, query heads, kv heads, head size, causal, window, fp8).
# Enough blocks that both batch sizes run 4-wave work-groups (two or more per CU).
CASES = [
    ("mixed pairs and chunks", [1, 0, 700, 33, 32, 31, 700, 512], [1, 0, 700, 500, 32, 9, 2100, 512],
     32, 8, 128, True, -1, False),
    ("ties", [500] * 5 + [100] * 4, [500] * 5 + [100] * 4, 32, 8, 128, True, -1, False),
    ("equal lengths past the caches", [200] * 64, [1200] * 64, 16, 2, 256, True, -1, False),
    ("fp8, window", [300, 700, 5, 0, 650], [300, 4000, 2000, 40, 651], 32, 8, 128, True, 255, True),
    ("not causal, 64 sequences", [(37 * i) % 400 for i in range(64)],
     [1 + (53 * i) % 1500 for i in range(64)], 16, 16, 80, False, -1, False),
    ("head 64, one query head per kv head", [1300, 3, 900], [1300, 777, 901], 32, 32, 64, True,
     -1, False),
    ("group of 8", [500, 129, 800], [3000, 129, 801], 64, 8, 128, True, -1, False),
    ("one sequence", [4200], [4200], 32, 8, 128, True, -1, False),
]


def _cu(lens):
    return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_order_only_permutes(case):
    label, ql, kl, hq, hk, d, causal, window, fp8 = case
    print(label, flush=True)
    g = torch.Generator(device="cuda").manual_seed(len(ql))

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)

    q = rnd(sum(ql), hq, d)
    scale, outs = d ** -0.5, []
    page = 16
    if causal:
        pages = [-(-k // page) for k in kl]
        kc, vc = rnd(sum(pages) + 1, page, hk, d), rnd(sum(pages) + 1, page, hk, d)
        if fp8:
            kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    else:
        k, v = rnd(sum(kl), hk, d), rnd(sum(kl), hk, d)
    for extra in (0, 65 - min(len(ql), 64)):
        cq, ck = _cu(ql + [0] * extra), _cu(kl + [0] * extra)
        shape = _native.prefill_shape(causal, _native.FK_DTYPE_FP8_E4M3FN if fp8 else
                                      _native.FK_DTYPE_BF16, len(ql) + extra, sum(ql), max(ql),
                                      max(kl), hq, hk, d, d, causal, window)
        assert shape[1:] == (1, 1, 0 if extra else len(ql))
        out = torch.full_like(q, 7.0)
        if causal:
            bt = torch.full((len(ql) + extra, max(pages)), -1, dtype=torch.int32)
            at = 0
            for i, n in enumerate(pages):
                bt[i, :n] = torch.arange(at, at + n)
                at += n
            ops.paged_prefill(out, q, kc, vc, bt.cuda(), cq, ck, max(ql), scale, causal=True,
                              window_left=window, max_seqlen_k=max(kl))
        else:
            ops.varlen_prefill(out, q, k, v, cq, ck, max(ql), scale, causal=False,
                               max_seqlen_k=max(kl))
        torch.cuda.synchronize()
        outs.append(out)
    same = bool(torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16)))
    assert same
