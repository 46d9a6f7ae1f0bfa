"""Sliding-window decode launches that give a sequence's whole window to one work-group
(its waves merge in LDS, no merge launch), at the edges of the rule that picks them: one
sequence, as many as fill the chip, windows of one token up to a wave's most tiles, 1, 2, 4
and 8 shares, every head size and query group, several column blocks per kv head, idle
waves, fp8 pages, empty contexts, masked pages, and the fused store.  Each case checks which
launch it gets; a window one tile past the rule takes the balanced schedule.

Against the fixed partitions over the same inputs and against float64.  All paths sum in
fp32 and round P and the row to bf16, so two of them differ by the rounding of P (2^-9
relative each) and of the result: rtol = 2^-7, and atol = 2^-7 of values of N(0, 1) rows
averaged over the window."""
from __future__ import annotations

import pytest
import torch

from fastkernels_amd import _native, ops, workloads

pytestmark = pytest.mark.gpu

# (batch, query heads, kv heads, head size, window_left, fp8, (waves, shares, whole)).  The
# rule counts (window_left + 16) / 16 + 1 tiles, one more than a window that is a multiple of
# 16 touches.
CASES = [
    (1, 64, 8, 64, 127, False, (1, 8, True)),
    (1, 32, 8, 128, 0, False, (1, 8, True)),
    (3, 32, 8, 128, 367, False, (1, 8, True)),     # 24 tiles: the most a few sequences take
    (3, 32, 8, 128, 368, False, (8, 1, False)),
    (5, 16, 2, 256, 175, False, (1, 4, True)),     # 12 tiles, head 256 (at most 4 shares)
    (5, 16, 2, 256, 176, False, (2, 1, False)),
    (40, 64, 8, 64, 128, False, (2, 4, True)),
    (150, 32, 8, 128, 127, True, (8, 1, True)),    # one share per head, 9 tiles
    (150, 32, 8, 128, 128, False, (4, 2, True)),
    (17, 71, 1, 64, 367, False, (1, 8, True)),     # five column blocks of one kv head
    (210, 71, 1, 64, 127, False, (4, 1, True)),    # ... in work-groups of 4: 3 idle waves
    (103, 71, 1, 64, 271, False, (4, 2, True)),    # 18 tiles over 2 shares, 3 idle heads
    (52, 71, 1, 64, 559, False, (2, 4, True)),     # 36 tiles over 4 shares, 1 idle head
    (33, 20, 20, 64, 1135, False, (1, 8, True)),   # 72 tiles over 8 shares
    (33, 20, 20, 64, 1136, False, (8, 1, False)),
    (25, 20, 20, 64, 1135, True, (1, 8, True)),    # fp8: 500 work-groups of 8 shares
    (26, 20, 20, 64, 1135, True, (8, 1, False)),   # 520: past two per CU
    (260, 16, 2, 256, 300, False, (1, 4, True)),
    (130, 8, 1, 128, 300, True, (1, 8, True)),
    (2, 40, 1, 256, 15, True, (1, 4, True)),
]


def _float64(case, bt, lens, window, sinks, fp8):
    """The rows in float64: keys of the window on readable pages, the sink in the sum."""
    hk, d = case.k_cache.shape[2:]
    b, hq = case.q.shape[:2]
    kc, vc = case.k_cache.float(), case.v_cache.float()
    if fp8:
        kc, vc = kc * case.k_scale.view(1, 1, -1, 1), vc * case.v_scale.view(1, 1, -1, 1)
    kc, vc = kc.view(-1, hk, d).double(), vc.view(-1, hk, d).double()
    page = case.k_cache.shape[1]
    out = torch.zeros(b, hq, d, dtype=torch.float64, device=case.q.device)
    for i, n in enumerate(lens):
        if n == 0:
            continue
        pos = torch.arange(max(0, n - 1 - window), n, device=case.q.device)
        pg = bt[i].long()[pos // page]
        slot = (pg * page + pos % page)[pg >= 0]
        k, v = (t[slot].transpose(0, 1).contiguous() for t in (kc, vc))  # [hk, keys, d]
        q = case.q[i].double().view(hk, hq // hk, d)
        s = torch.matmul(q, k.transpose(1, 2).contiguous()) * case.scale
        s = torch.cat([s, sinks.double().view(hk, hq // hk, 1)], -1)
        p = torch.softmax(s, -1)[..., :-1].contiguous()
        out[i] = torch.matmul(p, v).view(hq, d)
    return out


@pytest.mark.parametrize("batch,hq,hk,d,window,fp8,launch", CASES)
def test_whole_windows_match_partitions(cuda, batch, hq, hk, d, window, fp8, launch):
    print(f"windows {batch} {hq}/{hk}/{d} {window} fp8={fp8}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the expected launches are those of 256 CUs")
    plan = _native.plan(batch, hq, hk, d, 1500, 0)
    assert _native.decode_shape(batch, hq, hk, d, _native.FK_DTYPE_FP8_E4M3FN if fp8 else
                                _native.FK_DTYPE_BF16, window, plan[0], plan[1]) == launch
    lens = [(977 * i * i + 31 * i) % 1500 for i in range(batch)]  # 0 first, then mixed
    if batch == 1:
        lens = [1203]
    pool = sum((n + 15) // 16 for n in lens) + 2
    make = workloads.c5_fp8_decode if fp8 else workloads.c3_decode
    case = make(cuda, num_heads=hq, kv_heads=hk, head_dim=d, block_size=16, pool_blocks=pool,
                ctx_lens=lens, seed=batch + window)
    bt = case.block_tables.clone()
    if batch > 2:  # a page inside the last sequences' windows that must not be read
        rows = [b for b in range(batch) if lens[b] > 40][-2:]
        for b in rows:
            bt[b, (lens[b] - 20) // 16] = -1
    sinks = torch.linspace(-3, 3, hq, device=cuda)
    outs = []
    for splits in (0, 4):
        part, parts, nbytes = ops.paged_decode_plan(batch, hq, hk, d, max(lens), splits)
        ws = torch.zeros(max(1, nbytes), dtype=torch.uint8, device=cuda)
        out = torch.full_like(case.q, float("nan"))
        ops.paged_decode(out, case.q, case.k_cache, case.v_cache, bt, case.ctx_lens, case.scale,
                         part, parts, ws, case.k_scale, case.v_scale, window, sinks)
        torch.cuda.synchronize()
        outs.append(out.float())
    assert torch.isfinite(outs[0]).all()
    torch.testing.assert_close(outs[0], outs[1], rtol=2 ** -7, atol=2 ** -7)
    torch.testing.assert_close(outs[0].double(), _float64(case, bt, lens, window, sinks, fp8),
                               rtol=2 ** -7, atol=2 ** -7)
    for b in range(batch):
        if lens[b] == 0:
            assert not outs[0][b].any()
    # The fused store: the same bits as the store, then the decode.
    rows = workloads.decode_step_rows(case)
    kc, vc = case.k_cache.clone(), case.v_cache.clone()
    ops.store_kvcache(rows.key, rows.value, kc, vc, rows.slot_mapping)
    part, parts, nbytes = ops.paged_decode_plan(batch, hq, hk, d, max(lens), 0)
    ws = torch.zeros(max(1, nbytes), dtype=torch.uint8, device=cuda)
    want, got = torch.empty_like(case.q), torch.empty_like(case.q)
    ops.paged_decode(want, case.q, kc, vc, case.block_tables, case.ctx_lens, case.scale, part,
                     parts, ws, case.k_scale, case.v_scale, window, sinks)
    ops.store_paged_decode(got, case.q, rows.key, rows.value, case.k_cache, case.v_cache,
                           rows.slot_mapping, case.block_tables, case.ctx_lens, case.scale, part,
                           parts, ws, case.k_scale, case.v_scale, window, sinks)
    torch.cuda.synchronize()
    assert bool(torch.equal(want.view(torch.int16), got.view(torch.int16)))
    assert bool(torch.equal(kc.view(torch.uint8), case.k_cache.view(torch.uint8)))
    assert bool(torch.equal(vc.view(torch.uint8), case.v_cache.view(torch.uint8)))


@pytest.mark.parametrize("splits", [0, 1, 2])
def test_window_of_a_context_past_2_30(cuda, splits):
    """int32 lengths reach past 2^30 tokens, where a partition count formed as (ctx +
    part - 1) / part wraps.  Pages of 2^16 tokens, all but the last two unmapped; the
    window's 101 keys against float64 over them."""
    print(f"window of a context past 2^30, splits={splits}", flush=True)
    page, hq, hk, d, window, ctx = 1 << 16, 2, 1, 64, 100, (1 << 30) + 37
    g = torch.Generator(device=cuda).manual_seed(3)
    q = torch.randn(1, hq, d, generator=g, device=cuda).to(torch.bfloat16)
    kc, vc = (torch.randn(2, page, hk, d, generator=g, device=cuda).to(torch.bfloat16)
              for _ in range(2))
    pages = -(-ctx // page)
    bt = torch.full((1, pages), -1, dtype=torch.int32, device=cuda)
    bt[0, -2], bt[0, -1] = 1, 0  # the window starts in the page before the last
    part, parts, nbytes = ops.paged_decode_plan(1, hq, hk, d, 1 << 30, splits)
    ws = torch.zeros(max(1, nbytes), dtype=torch.uint8, device=cuda)
    out = torch.full_like(q, float("nan"))
    ops.paged_decode(out, q, kc, vc, bt, torch.tensor([ctx], dtype=torch.int32, device=cuda),
                     d ** -0.5, part, parts, ws, window_left=window)
    torch.cuda.synchronize()
    n = ctx - (pages - 1) * page  # tokens in the last page
    k = torch.cat([kc[1, page - (window + 1 - n):, 0], kc[0, :n, 0]]).double()
    v = torch.cat([vc[1, page - (window + 1 - n):, 0], vc[0, :n, 0]]).double()
    want = torch.softmax(q[0].double() @ k.T * d ** -0.5, -1) @ v
    torch.testing.assert_close(out[0].double(), want, rtol=1e-2, atol=1e-2)
