"""Key parts of prefill chunks over cached keys at the edges of the rule that counts them
(slots = two work-groups per CU): launches that fill one round of the slots, and ones whose
parts run in two, against the same call without parts.  The parts keep O in bf16 before
they are merged (rounded once, 2^-9 relative, beside the result's own rounding), so the two
agree within the bf16 bar of the other prefill tests, atol = rtol = 1e-2."""
from __future__ import annotations

import pytest
import torch

from fastkernels_amd import _native, ops

pytestmark = pytest.mark.gpu

# (query tokens per sequence, cached tokens, fp8, parts expected): 32-token blocks of 8 kv
# heads, 256 CUs, so a launch has 8 x blocks work-groups for 512 slots.
CASES = [
    ([512], 11000, False, 4),     # 128 work-groups: 4 parts, one round
    ([800], 8192, False, 5),      # 200: two rounds of 5 parts
    ([800], 4096, False, 3),      # 200, keys too few for 5 parts
    ([1000], 8192, True, 2),      # 256: one round of 2, fp8 pages
    ([1100], 8192, False, 3),     # 280: two rounds of 3
    ([700, 660], 5000, False, 2),  # 352: two rounds of 2
]


@pytest.mark.parametrize("ql,cached,fp8,parts", CASES)
def test_parts_match_whole_blocks(cuda, ql, cached, fp8, parts):
    print(f"parts {ql} over {cached} fp8={fp8}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the expected parts are those of 256 CUs")
    hq, hk, d, page = 32, 8, 128, 16
    g = torch.Generator(device=cuda).manual_seed(sum(ql))
    kl = [q + cached for q in ql]
    pages = [-(-k // page) for k in kl]

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device=cuda, dtype=torch.float32)

    q = rnd(sum(ql), hq, d).to(torch.bfloat16)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    kc, vc = rnd(sum(pages), page, hk, d).to(dt), rnd(sum(pages), page, hk, d).to(dt)
    bt = torch.full((len(ql), max(pages)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(at, at + n)
        at += n
    bt = bt.to(cuda)

    def cu(lens):
        return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32,
                            device=cuda)

    nbytes = _native.prefill_split_bytes(
        True, _native.FK_DTYPE_FP8_E4M3FN if fp8 else _native.FK_DTYPE_BF16, len(ql), sum(ql),
        max(ql), max(kl), hq, hk, d, d, True)
    per_part = sum(ql) * hq * (d * 2 + 16)
    assert nbytes // per_part == parts
    outs = []
    for split in (True, False):
        ops.PREFILL_SPLIT = split
        try:
            out = torch.full_like(q, float("nan"))
            ops.paged_prefill(out, q, kc, vc, bt, cu(ql), cu(kl), max(ql), d ** -0.5,
                              max_seqlen_k=max(kl))
            torch.cuda.synchronize()
        finally:
            ops.PREFILL_SPLIT = True
        outs.append(out.float())
    assert torch.isfinite(outs[0]).all()
    torch.testing.assert_close(outs[0], outs[1], rtol=1e-2, atol=1e-2)
