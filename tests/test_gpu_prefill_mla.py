"""MLA's head sizes (query / key 192, value 128) through every kernel the launch rule picks
from: one or two 16-query column blocks a wave (64 or 128 query tokens a work-group), the
keys whole, over the halves of a work-group or in fp32 parts over work-groups; dense keys
with the log-sum-exp and paged ones, causal and not, lengths at the edges of tiles, waves
and blocks.  Each case checks which launch it gets, then compares with float64 over the
same bf16 inputs: atol = rtol = 1e-2 for bf16 rows (P and the row rounded once, 2^-9
each), 1e-5 for the fp32 log-sum-exp."""
from __future__ import annotations

import pytest
import torch

from fastkernels_amd import _native, ops

pytestmark = pytest.mark.gpu

EDGES = [1, 31, 33, 127, 129, 64, 65, 128, 300]
# (query lengths, key lengths, heads, causal, paged, (wg_tokens, key_split, parts))
CASES = [
    (EDGES, EDGES, 2, True, False, (64, 2, 1)),
    (EDGES, EDGES, 2, False, False, (64, 2, 1)),
    ([33, 1, 20] * 11, [33, 1, 20] * 11, 32, True, False, (64, 1, 1)),
    ([600, 40], [2000, 20], 2, True, False, (64, 2, 6)),
    ([64, 1, 33] * 3, [9000, 100, 8000] * 3, 16, True, False, (64, 1, 7)),
    (EDGES * 4, EDGES * 4, 16, True, False, (128, 1, 1)),
    (EDGES * 4, [n + 700 for n in EDGES] * 4, 16, False, False, (128, 1, 1)),
    (EDGES, EDGES, 16, False, False, (128, 2, 1)),
    ([512] * 8, [8192] * 8, 2, False, False, (128, 2, 4)),
    (EDGES, [n + 3000 for n in EDGES], 16, True, False, (128, 1, 2)),
    ([512] * 8, [8192] * 7 + [100], 4, False, False, (128, 1, 4)),
    (EDGES, EDGES, 2, True, True, (64, 2, 1)),
    (EDGES, [n + 3000 for n in EDGES], 16, True, True, (128, 1, 2)),
    (EDGES * 4, EDGES * 4, 16, True, True, (128, 1, 1)),
]


def _cu(lens):
    return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32,
                        device="cuda")


def _reference(q, k, v, ql, kl, scale, causal):
    """float64 rows and log-sum-exp, one sequence after another."""
    out = torch.zeros(q.shape[0], q.shape[1], v.shape[2], dtype=torch.float64, device="cuda")
    lse = torch.full((q.shape[1], q.shape[0]), float("-inf"), dtype=torch.float64, device="cuda")
    a = c = 0
    for n, m in zip(ql, kl):
        qs, ks, vs = (t.double().transpose(0, 1).contiguous()
                      for t in (q[a:a + n], k[c:c + m], v[c:c + m]))
        s = torch.matmul(qs, ks.transpose(1, 2).contiguous()) * scale
        if causal:
            i = torch.arange(n, device="cuda")[:, None] + m - n
            s.masked_fill_(torch.arange(m, device="cuda")[None, :] > i, float("-inf"))
        lse[:, a:a + n] = torch.logsumexp(s, -1)
        out[a:a + n] = torch.matmul(torch.softmax(s, -1).nan_to_num(0.0), vs).transpose(0, 1)
        a, c = a + n, c + m
    return out, lse


@pytest.mark.parametrize("i", range(len(CASES)))
def test_mla_launches_against_float64(cuda, i):
    ql, kl, h, causal, paged, want = CASES[i]
    print(f"mla case {i}: {len(ql)} sequences, {h} heads, causal={causal} paged={paged}",
          flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the expected launches are those of 256 CUs")
    shape = _native.prefill_shape(paged, _native.FK_DTYPE_BF16, len(ql), sum(ql), max(ql),
                                  max(kl), h, h, 192, 128, causal)
    assert shape[:3] == want
    g = torch.Generator(device=cuda).manual_seed(900 + i)

    def rnd(*s):
        return torch.randn(*s, generator=g, device=cuda, dtype=torch.float32).to(torch.bfloat16)

    q, k, v = rnd(sum(ql), h, 192), rnd(sum(kl), h, 192), rnd(sum(kl), h, 128)
    ref, ref_lse = _reference(q, k, v, ql, kl, 192 ** -0.5, causal)
    out = torch.full((sum(ql), h, 128), float("nan"), dtype=torch.bfloat16, device=cuda)
    lse = None
    if paged:
        page = 16
        pages = [-(-m // page) for m in kl]
        kc = torch.full((sum(pages), page, h, 192), float("nan"), dtype=torch.bfloat16,
                        device=cuda)
        vc = torch.full((sum(pages), page, h, 128), float("nan"), dtype=torch.bfloat16,
                        device=cuda)
        bt = torch.full((len(kl), max(pages)), -1, dtype=torch.int32)
        at = c = 0
        for b, (m, n) in enumerate(zip(kl, pages)):
            bt[b, :n] = torch.arange(at, at + n)
            kc[at:at + n].view(-1, h, 192)[:m] = k[c:c + m]
            vc[at:at + n].view(-1, h, 128)[:m] = v[c:c + m]
            at, c = at + n, c + m
        ops.paged_prefill(out, q, kc, vc, bt.to(cuda), _cu(ql), _cu(kl), max(ql), 192 ** -0.5,
                          causal=causal, max_seqlen_k=max(kl))
    else:
        lse = torch.full((h, sum(ql)), float("nan"), dtype=torch.float32, device=cuda)
        ops.varlen_prefill(out, q, k, v, _cu(ql), _cu(kl), max(ql), 192 ** -0.5, causal,
                           max_seqlen_k=max(kl), lse=lse)
    torch.cuda.synchronize()
    torch.testing.assert_close(out.double(), ref, rtol=1e-2, atol=1e-2)
    if lse is not None:
        torch.testing.assert_close(lse.double(), ref_lse, rtol=1e-5, atol=1e-5)
