"""Performance cases of the decode-step operator path, called as a serving engine calls it.

Each case is one pass through the L1 operator classes (``fastkernels_amd.candidate.L1``)
at the sizes a serving engine meets: single decode steps of small and large batches, long
contexts with fp8 pages, sliding windows with sinks, prompts and prompt chunks, the
encoders' dense attention, MLA's chunked prefill, and the row operators of a prompt.

Kinds (``case["kind"]``):

    layer    one decode step of a layer without its matrix products: add + RMSNorm, q/k norm +
             rotary + store, paged decode attention, SiLU-and-mul
    decode   FlashAttnDecode.forward over a paged cache (bf16 or fp8, window, sinks)
    prefill  FlashAttnPrefill.forward over a paged cache (bf16 or fp8, window, sinks)
    varlen   FlashAttnVarlen.forward over dense keys, not causal (the encoders)
    mla      MLA's prefill of new tokens over a cached context: a causal call with its
             log-sum-exp, one over the context chunk with its own, MergeAttnStates
    rows     the row operators at a prompt's token count: add + RMSNorm, q/k norm + rotary +
             store, SiLU-and-mul

Sequence lengths are part of a case (drawn from ``len_seed`` between ``lo`` and ``hi``); the
values come from the seed given to ``prepare``.
"""
from __future__ import annotations

import math
import random

import torch

from fastkernels_amd.candidate.L1.flash_attn_decode import FlashAttnDecode
from fastkernels_amd.candidate.L1.flash_attn_prefill import FlashAttnPrefill
from fastkernels_amd.candidate.L1.flash_attn_varlen import FlashAttnVarlen
from fastkernels_amd.candidate.L1.merge_attn_states import MergeAttnStates
from fastkernels_amd.candidate.L1.rms_norm import RMSNorm
from fastkernels_amd.candidate.L1.rotary_emb import RotaryEmbedding
from fastkernels_amd.candidate.L1.silu_and_mul import SiluAndMul

DEV = "cuda"
_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_FP8 = torch.float8_e4m3fn
MAX_POS = 40960
THETA = 1e6


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _layer(batch, lo, hi, hq=32, hk=8, d=128, hidden=4096, inter=12288, page=16, kv="bf16",
           qk_norm=True, len_seed=1):
    return dict(kind="layer", batch=batch, lo=lo, hi=hi, hq=hq, hk=hk, d=d, hidden=hidden,
                inter=inter, page=page, kv=kv, qk_norm=qk_norm, len_seed=len_seed)


def _decode(batch, lo, hi, hq=32, hk=8, d=128, page=16, kv="bf16", window=-1, sinks=False,
            len_seed=1):
    return dict(kind="decode", batch=batch, lo=lo, hi=hi, hq=hq, hk=hk, d=d, page=page, kv=kv,
                window=window, sinks=sinks, len_seed=len_seed)


def _prefill(batch, qlo, qhi, clo, chi, hq=32, hk=8, d=128, page=16, kv="bf16", window=-1,
             sinks=False, len_seed=1):
    return dict(kind="prefill", batch=batch, qlo=qlo, qhi=qhi, clo=clo, chi=chi, hq=hq, hk=hk,
                d=d, page=page, kv=kv, window=window, sinks=sinks, len_seed=len_seed)


def _varlen(batch, qlo, qhi, heads=16, d=80, len_seed=1):
    return dict(kind="varlen", batch=batch, qlo=qlo, qhi=qhi, heads=heads, d=d,
                len_seed=len_seed)


def _mla(batch, qlo, qhi, clo, chi, heads=16, len_seed=1):
    return dict(kind="mla", batch=batch, qlo=qlo, qhi=qhi, clo=clo, chi=chi, heads=heads,
                len_seed=len_seed)


def _rows(tokens, hidden=4096, inter=12288, hq=32, hk=8, d=128, dtype="bf16", page=16,
          qk_norm=True):
    return dict(kind="rows", tokens=tokens, hidden=hidden, inter=inter, hq=hq, hk=hk, d=d,
                dtype=dtype, page=page, qk_norm=qk_norm)


def listed():
    return [
        # One user's decode step: the smallest calls, four operators, latency and launches.
        dict(_layer(1, 1013, 1013), name="layer_b1"),
        # The same step for a medium batch with an fp8 cache (Llama-3-70B heads, no q/k norm).
        dict(_layer(32, 256, 4096, hq=64, hidden=8192, inter=28672, kv="fp8", qk_norm=False),
             name="layer_b32_fp8"),
        # The headline: Qwen3-8B heads, 64 sequences of 512 to 8192 tokens, 256-token pages.
        dict(_decode(64, 512, 8192, page=256), name="decode_b64"),
        # Long documents on fp8 pages, Llama-3-70B heads, the largest decode.
        dict(_decode(8, 131072, 131072, hq=64, page=256, kv="fp8"), name="decode_long_fp8"),
        # gpt-oss-like sliding-window layers with sinks, a large batch of short windows.
        dict(_decode(128, 300, 6000, hq=64, d=64, window=127, sinks=True),
             name="decode_window_sinks"),
        # One prompt: time to first token.
        dict(_prefill(1, 2048, 2048, 0, 0), name="prefill_1x2048"),
        # Chunks of several prompts over their cached starts (chunked prefill), ragged.
        dict(_prefill(5, 300, 700, 2000, 6000), name="prefill_chunks"),
        # A ragged batch of short prompts on fp8 pages.
        dict(_prefill(13, 70, 1100, 0, 0, kv="fp8"), name="prefill_ragged_fp8"),
        # A long prompt in one call: the largest matrix work.
        dict(_prefill(1, 12288, 12288, 0, 0, page=256), name="prefill_long"),
        # A vision encoder's attention over a few images (Qwen2.5-VL heads).
        dict(_varlen(6, 500, 3000), name="encoder_ragged"),
        # MLA prefill: new tokens of two sequences over their cached contexts.
        dict(_mla(2, 800, 1200, 2500, 4500), name="mla_chunk"),
        # The row operators of an 8192-token prompt step.
        dict(_rows(8192), name="rows_8192"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (query heads, kv heads, head size) of the models whose decode and prompt the path serves.
_DECODE_HEADS = [(32, 8, 128), (32, 8, 128), (64, 8, 128), (16, 2, 256), (20, 20, 64),
                 (64, 8, 64), (8, 1, 128)]


def draw(rng):
    """One more case of the ranges above; sizes spread over their logarithm."""
    kind = rng.choice(["layer", "decode", "decode", "prefill", "prefill", "varlen", "mla", "rows"])
    ls = rng.randrange(1 << 20)
    page = rng.choice([16, 16, 64, 256])
    if kind == "layer":
        batch = _log_int(rng, 1, 96)
        hi = _log_int(rng, 200, 4096)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        if rng.random() < 0.5:
            return _layer(batch, lo, hi, page=page, kv=rng.choice(["bf16", "fp8"]), len_seed=ls)
        return _layer(batch, lo, hi, hq=64, hidden=8192, inter=28672, page=page,
                      kv=rng.choice(["bf16", "fp8"]), qk_norm=False, len_seed=ls)
    if kind == "decode":
        hq, hk, d = rng.choice(_DECODE_HEADS)
        kv = rng.choice(["bf16", "bf16", "fp8"])
        elt = 1 if kv == "fp8" else 2
        batch = _log_int(rng, 1, 160)
        # at most the bytes of decode_long_fp8, and at most its length
        cap = int(2 * (1 << 30) / (2 * hk * d * elt * batch))
        hi = _log_int(rng, 64, max(65, min(131072, cap)))
        lo = max(1, int(hi * rng.uniform(0.05, 1.0)))
        windowed = rng.random() < 0.25
        return _decode(batch, lo, hi, hq=hq, hk=hk, d=d, page=page, kv=kv,
                       window=rng.choice([127, 1023, 4095]) if windowed else -1,
                       sinks=windowed, len_seed=ls)
    if kind == "prefill":
        hq, hk, d = rng.choice([(32, 8, 128), (32, 8, 128), (64, 8, 128), (16, 2, 256),
                                (20, 20, 64), (64, 8, 64)])
        batch = _log_int(rng, 1, 24)
        # matrix work of a batch: at most half of prefill_long's
        pairs = 12288 * 12288 / 4 * (32 * 128) / (hq * d) / batch
        chunked = rng.random() < 0.5
        chi = _log_int(rng, 64, 16384) if chunked else 0
        qcap = int(math.sqrt(chi * chi + 2 * pairs) - chi)  # q (c + q / 2) <= pairs
        qhi = _log_int(rng, 16, max(17, min(8192, qcap)))
        qlo = max(1, int(qhi * rng.uniform(0.1, 1.0)))
        clo = int(chi * rng.uniform(0.3, 1.0))
        windowed = (hq, hk, d) == (64, 8, 64) and rng.random() < 0.5
        return _prefill(batch, qlo, qhi, clo, chi, hq=hq, hk=hk, d=d, page=page,
                        kv=rng.choice(["bf16", "bf16", "fp8"]), window=127 if windowed else -1,
                        sinks=windowed, len_seed=ls)
    if kind == "varlen":
        heads, d = rng.choice([(16, 80), (16, 72), (12, 32), (20, 64)])
        batch = _log_int(rng, 1, 32)
        qhi = _log_int(rng, 50, max(51, int(math.sqrt(12288 * 12288 / 4 / batch))))
        qlo = max(1, int(qhi * rng.uniform(0.2, 1.0)))
        return _varlen(batch, qlo, qhi, heads=heads, d=d, len_seed=ls)
    if kind == "mla":
        batch = _log_int(rng, 1, 4)
        qhi = _log_int(rng, 64, 2048)
        chi = _log_int(rng, 256, 8192)
        return _mla(batch, max(1, int(qhi * rng.uniform(0.3, 1.0))), qhi,
                    int(chi * rng.uniform(0.3, 1.0)), chi, len_seed=ls)
    tokens = _log_int(rng, 1, 8192)
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    if dtype == "f32":
        return _rows(min(tokens, 4096), hidden=1024, inter=4096, dtype="f32", page=page)
    if rng.random() < 0.3:
        return _rows(min(tokens, 3400), hidden=8192, inter=28672, hq=64, dtype=dtype, page=page,
                     qk_norm=False)
    return _rows(tokens, dtype=dtype, page=page)


# ---------------------------------------------------------------------------
# Lengths and sizes
# ---------------------------------------------------------------------------
def _lens(case, n, lo, hi, salt=0):
    """n lengths in [lo, hi], the longest among them (a case costs what its bounds say)."""
    g = random.Random(case["len_seed"] * 7919 + salt)
    out = [g.randint(lo, hi) for _ in range(n)]
    out[g.randrange(n)] = hi
    return out


def _decode_lens(case):
    return _lens(case, case["batch"], case["lo"], case["hi"])


def _chunk_lens(case):
    """(new tokens, cached tokens) per sequence."""
    b = case["batch"]
    return (_lens(case, b, case["qlo"], case["qhi"], 1), _lens(case, b, case["clo"], case["chi"], 2))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _tables(lens, page, g_seed):
    """Non-overlapping pages in random order, -1 padded; returns (tables, pool pages)."""
    pages = [-(-n // page) for n in lens]
    pool = sum(pages) + 8
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(g_seed)).to(torch.int32)
    bt = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
    at = 0
    for i, p in enumerate(pages):
        bt[i, :p] = perm[at:at + p]
        at += p
    return bt.to(DEV), pool


def _quant(g, shape, scale):
    """N(0, 1) values as fp8 e4m3fn codes of x / scale[kv head], saturated; in slices, so that
    a large pool needs no float32 copy of itself."""
    out = torch.empty(shape, dtype=_FP8, device=DEV)
    step = max(1, (1 << 26) // (shape[1] * shape[2] * shape[3]))
    for a in range(0, shape[0], step):
        part = _randn(g, min(step, shape[0] - a), *shape[1:], dtype=torch.float32)
        if scale is not None:
            part = part / scale.view(1, 1, -1, 1)
        out[a:a + step] = part.clamp_(-448.0, 448.0).to(_FP8)
    return out


def _caches(g, pool, page, hk, d, kv, scaled):
    """K and V pages, and the fp8 scales per kv head (None without)."""
    shape = (pool, page, hk, d)
    if kv == "bf16":
        return _randn(g, *shape), _randn(g, *shape), None, None
    ks = vs = None
    if scaled:
        ks = 0.01 + 0.09 * torch.rand(hk, generator=g, device=DEV)
        vs = 0.01 + 0.09 * torch.rand(hk, generator=g, device=DEV)
    return _quant(g, shape, ks), _quant(g, shape, vs), ks, vs


def _cu(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return torch.tensor(cu, dtype=torch.int32, device=DEV)


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def _norm(g, width, dtype):
    m = RMSNorm(width).to(DEV, dtype)
    m.weight.data.copy_(1.0 + 0.1 * torch.randn(width, generator=g, device=DEV))
    return m


def _row_state(case, g, tokens, dtype):
    """What the row operators of a layer take, and the modules that run them."""
    hq, hk, d, hidden, inter = (case[k] for k in ("hq", "hk", "d", "hidden", "inter"))
    s = dict(norm=_norm(g, hidden, dtype), rope=RotaryEmbedding(d, MAX_POS, THETA).to(DEV),
             silu=SiluAndMul(), q_norm=None, k_norm=None)
    if case["qk_norm"]:
        s["q_norm"], s["k_norm"] = _norm(g, d, dtype), _norm(g, d, dtype)
    s["x"] = _randn(g, tokens, hidden, dtype=dtype)
    s["residual"] = _randn(g, tokens, hidden, dtype=dtype)
    qkv = _randn(g, tokens, (hq + 2 * hk) * d, dtype=dtype)
    s["q"], s["k"], s["v"] = qkv.split([hq * d, hk * d, hk * d], dim=-1)
    s["gate_up"] = _randn(g, tokens, 2 * inter, dtype=dtype)
    return s


def _prepare_layer(case, seed):
    g = _gen(seed)
    lens = _decode_lens(case)
    page = case["page"]
    bt, pool = _tables(lens, page, seed)
    s = _row_state(case, g, case["batch"], torch.bfloat16)
    s["kc"], s["vc"], _, _ = _caches(g, pool, page, case["hk"], case["d"], case["kv"], False)
    s["bt"] = bt
    s["ctx"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    last = s["ctx"].to(torch.int64) - 1
    s["pos"] = last
    rows = torch.arange(len(lens), device=DEV)
    s["slots"] = bt[rows, last // page].to(torch.int64) * page + last % page
    s["max_len"] = max(lens)
    s["attn"] = FlashAttnDecode(case["hq"], case["hk"], case["d"])
    s["attn"].preallocate(case["batch"], torch.device(DEV, torch.cuda.current_device()))
    s["scale"] = case["d"] ** -0.5
    # The caches as they are returned: fp8 pages as bytes.
    s["kc_out"], s["vc_out"] = ((s["kc"].view(torch.uint8), s["vc"].view(torch.uint8))
                                if case["kv"] == "fp8" else (s["kc"], s["vc"]))
    return s


def _prepare_decode(case, seed):
    g = _gen(seed)
    lens = _decode_lens(case)
    bt, pool = _tables(lens, case["page"], seed)
    kc, vc, ks, vs = _caches(g, pool, case["page"], case["hk"], case["d"], case["kv"], True)
    s = dict(q=_randn(g, case["batch"], case["hq"], case["d"]), kc=kc, vc=vc, bt=bt,
             ctx=torch.tensor(lens, dtype=torch.int32, device=DEV), max_len=max(lens))
    s["attn"] = FlashAttnDecode(case["hq"], case["hk"], case["d"])
    s["attn"].preallocate(case["batch"], torch.device(DEV, torch.cuda.current_device()))
    s["kw"] = dict(softmax_scale=case["d"] ** -0.5, causal=True)
    if ks is not None:
        s["kw"].update(k_scale=ks, v_scale=vs)
    if case["window"] >= 0:
        s["kw"]["window_size"] = (case["window"], 0)
    s["sinks"] = None
    if case["sinks"]:
        s["kw"]["s_aux"] = s["sinks"] = torch.randn(case["hq"], generator=g, device=DEV)
    return s


def _prepare_prefill(case, seed):
    g = _gen(seed)
    ql, cl = _chunk_lens(case)
    kl = [a + b for a, b in zip(ql, cl)]
    bt, pool = _tables(kl, case["page"], seed)
    kc, vc, ks, vs = _caches(g, pool, case["page"], case["hk"], case["d"], case["kv"], True)
    s = dict(q=_randn(g, sum(ql), case["hq"], case["d"]), kc=kc, vc=vc, cu_q=_cu(ql),
             cu_k=_cu(kl), max_q=max(ql), max_k=max(kl))
    s["attn"] = FlashAttnPrefill(case["hq"], case["hk"], case["d"])
    s["kw"] = dict(softmax_scale=case["d"] ** -0.5, causal=True, block_table=bt)
    if ks is not None:
        s["kw"].update(k_descale=ks, v_descale=vs)
    if case["window"] >= 0:
        s["kw"]["window_size"] = (case["window"], 0)
    s["sinks"] = None
    if case["sinks"]:
        s["kw"]["s_aux"] = s["sinks"] = torch.randn(case["hq"], generator=g, device=DEV)
    return s


def _prepare_varlen(case, seed):
    g = _gen(seed)
    ql = _lens(case, case["batch"], case["qlo"], case["qhi"], 1)
    n, h, d = sum(ql), case["heads"], case["d"]
    # q, k and v are views of the encoder's fused projection.
    qkv = _randn(g, n, 3 * h * d).view(n, 3, h, d)
    cu = _cu(ql)
    return dict(q=qkv[:, 0], k=qkv[:, 1], v=qkv[:, 2], cu=cu, max_q=max(ql), scale=d ** -0.5,
                attn=FlashAttnVarlen())


def _prepare_mla(case, seed):
    g = _gen(seed)
    ql, cl = _chunk_lens(case)
    h, nq, nc = case["heads"], sum(ql), sum(cl)
    return dict(q=_randn(g, nq, h, 192), k=_randn(g, nq, h, 192), v=_randn(g, nq, h, 128),
                kc=_randn(g, nc, h, 192), vc=_randn(g, nc, h, 128), cu_q=_cu(ql), cu_c=_cu(cl),
                max_q=max(ql), max_c=max(cl), scale=192 ** -0.5, attn=FlashAttnVarlen(),
                merge=MergeAttnStates())


def _prepare_rows(case, seed):
    g = _gen(seed)
    t, dtype, page = case["tokens"], _DTYPES[case["dtype"]], case["page"]
    s = _row_state(case, g, t, dtype)
    s["pos"] = torch.arange(t, device=DEV)
    bt, pool = _tables([t], page, seed)
    s["kc"] = torch.zeros(pool, page, case["hk"], case["d"], dtype=dtype, device=DEV)
    s["vc"] = torch.zeros_like(s["kc"])
    s["slots"] = bt[0, s["pos"] // page].to(torch.int64) * page + s["pos"] % page
    return s


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"])


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def _run_layer(s):
    x, residual = s["norm"](s["x"], s["residual"])
    q, k = s["rope"].forward_store(s["pos"], s["q"], s["k"], s["v"], s["kc"], s["vc"], s["slots"],
                                   q_norm=s["q_norm"], k_norm=s["k_norm"])
    o = s["attn"](q, s["kc"], s["vc"], s["ctx"], block_table=s["bt"], softmax_scale=s["scale"],
                  causal=True, max_seq_len=s["max_len"])
    act = s["silu"](s["gate_up"])
    return {"x": x, "residual": residual, "q": q, "k": k, "kc": s["kc_out"], "vc": s["vc_out"],
            "o": o, "act": act}


def _run_decode(s):
    return s["attn"](s["q"], s["kc"], s["vc"], s["ctx"], block_table=s["bt"],
                     max_seq_len=s["max_len"], **s["kw"])


def _run_prefill(s):
    return s["attn"](s["q"], s["kc"], s["vc"], s["cu_q"], s["cu_k"], s["max_q"], s["max_k"],
                     **s["kw"])


def _run_varlen(s):
    return s["attn"](s["q"], s["k"], s["v"], s["cu"], s["cu"], s["max_q"], s["max_q"], s["scale"],
                     causal=False)


def _run_mla(s):
    new, new_lse = s["attn"](s["q"], s["k"], s["v"], s["cu_q"], s["cu_q"], s["max_q"], s["max_q"],
                             s["scale"], causal=True, return_softmax_lse=True)
    old, old_lse = s["attn"](s["q"], s["kc"], s["vc"], s["cu_q"], s["cu_c"], s["max_q"],
                             s["max_c"], s["scale"], causal=False, return_softmax_lse=True)
    out, lse = torch.empty_like(new), torch.empty_like(new_lse)
    s["merge"](out, old, old_lse, new, new_lse, lse)
    return {"out": out, "lse": lse}


def _run_rows(s):
    x, residual = s["norm"](s["x"], s["residual"])
    q, k = s["rope"].forward_store(s["pos"], s["q"], s["k"], s["v"], s["kc"], s["vc"], s["slots"],
                                   q_norm=s["q_norm"], k_norm=s["k_norm"])
    act = s["silu"](s["gate_up"])
    return {"x": x, "residual": residual, "q": q, "k": k, "kc": s["kc"], "vc": s["vc"],
            "act": act}


def run(state):
    return _RUN[state["kind"]](state)


_PREPARE = {"layer": _prepare_layer, "decode": _prepare_decode, "prefill": _prepare_prefill,
            "varlen": _prepare_varlen, "mla": _prepare_mla, "rows": _prepare_rows}
_RUN = {"layer": _run_layer, "decode": _run_decode, "prefill": _run_prefill,
        "varlen": _run_varlen, "mla": _run_mla, "rows": _run_rows}


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _decode_work(case, lens):
    elt = 1 if case["kv"] == "fp8" else 2
    w = case.get("window", -1)
    seen = sum(min(n, w + 1) if w >= 0 else n for n in lens)
    pages = sum(-(-n // case["page"]) for n in lens)
    hq, hk, d = case["hq"], case["hk"], case["d"]
    return (2 * seen * hk * d * elt + 4 * len(lens) * hq * d + 4 * pages + 4 * len(lens),
            4 * seen * hq * d)


def _rows_work(case, t, elt, kv_elt):
    hq, hk, d, hidden, inter = (case[k] for k in ("hq", "hk", "d", "hidden", "inter"))
    norm = 4 * t * hidden * elt + hidden * elt
    # q and k read and written, v read, the cache rows written, slots, positions, cos/sin
    qk = t * d * ((2 * hq + 2 * hk + hk) * elt + 2 * hk * kv_elt) + t * (8 + 8 + 4 * d)
    silu = 3 * t * inter * elt
    return norm + qk + silu, t * (5 * hidden + 6 * (hq + hk) * d + 6 * inter)


def _visible(ql, kl, window, causal=True):
    """Query-key pairs a chunk of ql queries at the end of kl keys sees."""
    if not causal:
        return ql * kl
    off, n = kl - ql, 0
    if window < 0:
        return ql * off + ql * (ql + 1) // 2
    for j in range(ql):
        n += min(off + j + 1, window + 1)
    return n


def work(case):
    kind = case["kind"]
    if kind == "layer":
        b, f = _decode_work(case, _decode_lens(case))
        rb, rf = _rows_work(case, case["batch"], 2, 1 if case["kv"] == "fp8" else 2)
        return {"bytes": b + rb, "flops": f + rf}
    if kind == "decode":
        b, f = _decode_work(case, _decode_lens(case))
        return {"bytes": b, "flops": f}
    if kind == "rows":
        elt = 4 if case["dtype"] == "f32" else 2
        b, f = _rows_work(case, case["tokens"], elt, elt)
        return {"bytes": b, "flops": f}
    if kind == "varlen":
        ql = _lens(case, case["batch"], case["qlo"], case["qhi"], 1)
        h, d = case["heads"], case["d"]
        return {"bytes": 8 * sum(ql) * h * d, "flops": 4 * h * d * sum(n * n for n in ql)}
    ql, cl = _chunk_lens(case)
    kl = [a + b for a, b in zip(ql, cl)]
    nq, nc = sum(ql), sum(cl)
    if kind == "mla":
        h = case["heads"]
        pairs = sum(_visible(a, b, -1) for a, b in zip(ql, kl))
        return {"bytes": 2 * h * (nq * (192 + 192 + 128 + 128) + nc * 320) + 4 * h * nq,
                "flops": 2 * h * 320 * pairs}
    hq, hk, d, w = case["hq"], case["hk"], case["d"], case["window"]
    elt = 1 if case["kv"] == "fp8" else 2
    keys = sum(min(k, q + w) if w >= 0 else k for q, k in zip(ql, kl))
    pairs = sum(_visible(q, k, w) for q, k in zip(ql, kl))
    return {"bytes": 4 * nq * hq * d + 2 * keys * hk * d * elt, "flops": 4 * hq * d * pairs}


# ---------------------------------------------------------------------------
# tolerance: about four times the error against exact() that the path showed over these ranges
# (54 cases: attention rel up to 3.9e-3 and max 7.8e-2 (short rows of a prompt, fp8); row
# operators rel 3.1e-3 / 3.9e-4 / 6.5e-8 and max 2.9e-2 / 1.1e-2 / 3.6e-7 in bf16 / f16 / f32).
# ---------------------------------------------------------------------------
def tolerance(case):
    if case["kind"] == "rows":
        return {"f32": {"rel": 3e-7, "max": 1.5e-6}, "f16": {"rel": 1.6e-3, "max": 4.5e-2},
                "bf16": {"rel": 1.3e-2, "max": 0.12}}[case["dtype"]]
    if case["kind"] == "layer":  # fp8 cache bytes: rows stored from a k on a rounding boundary
        return {"rel": 1.5e-2, "max": 0.12, "differ": 1e-4}
    return {"rel": 1.5e-2, "max": 0.3}


# ---------------------------------------------------------------------------
# exact: the same results in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, scale, offset, causal, window, sinks):
    """Softmax attention of q [n, Hq, D] over k [m, Hk, D], v [m, Hk, Dv] in float64; query j
    sits at position offset + j.  Returns (out, lse [Hq, n])."""
    n, hq, d = q.shape
    m, hk, dv = v.shape
    out = torch.empty(n, hq, dv, dtype=torch.float64, device=q.device)
    lse = torch.empty(hq, n, dtype=torch.float64, device=q.device)
    kpos = torch.arange(m, device=q.device)
    step = max(1, (1 << 27) // max(1, m))
    for h in range(hk):
        kt = k[:, h].double().t().contiguous()
        vh = v[:, h].double().contiguous()
        g = hq // hk
        for a in range(0, n, step):
            qpos = torch.arange(a, min(n, a + step), device=q.device) + offset
            hide = torch.zeros(len(qpos), m, dtype=torch.bool, device=q.device)
            if causal:
                hide |= kpos[None] > qpos[:, None]
                if window >= 0:
                    hide |= kpos[None] < qpos[:, None] - window
            for hh in range(h * g, (h + 1) * g):
                sc = torch.mm(q[a:a + step, hh].double().contiguous(), kt) * scale
                sc.masked_fill_(hide, -math.inf)
                top = sc.amax(dim=1, keepdim=True)
                p = torch.exp(sc - top)
                den = p.sum(dim=1, keepdim=True)
                lse[hh, a:a + step] = (top + den.log())[:, 0]
                if sinks is not None:
                    den = den + torch.exp(sinks[hh].double() - top)
                out[a:a + step, hh] = torch.mm(p, vh) / den
    return out, lse


def _gather(cache, bt_row, n, scale):
    """The first n cached rows of a sequence in float64, dequantised."""
    page = cache.shape[1]
    rows = cache[bt_row[:-(-n // page)].to(torch.int64)] if cache.dtype != _FP8 else \
        cache.view(torch.uint8)[bt_row[:-(-n // page)].to(torch.int64)].view(_FP8)
    rows = rows.reshape(-1, *cache.shape[2:])[:n].double()
    return rows if scale is None else rows * scale.double().view(1, -1, 1)


def _exact_rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _exact_rows(s, d):
    """The row operators' results in float64, and the stored k rows [T, Hk, D]."""
    t = s["x"].shape[0]
    residual = s["x"].double() + s["residual"].double()
    x = _exact_rms(residual, s["norm"].weight.detach())
    q, k = s["q"].double().reshape(t, -1, d), s["k"].double().reshape(t, -1, d)
    if s["q_norm"] is not None:
        q = _exact_rms(q, s["q_norm"].weight.detach())
        k = _exact_rms(k, s["k_norm"].weight.detach())
    cs = s["rope"].cos_sin_cache[s["pos"]].double()
    cos, sin = cs[:, None, :d // 2], cs[:, None, d // 2:]

    def rot(z):
        a, b = z[..., :d // 2], z[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    q, k = rot(q), rot(k)
    gate, up = s["gate_up"].double().chunk(2, dim=-1)
    return x, residual, q, k, gate * torch.sigmoid(gate) * up


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind in ("rows", "layer"):
        d = case["d"]
        t = s["x"].shape[0]
        x, residual, q, k, act = _exact_rows(s, d)
        v = s["v"].reshape(t, -1, d)
        out = {"x": x, "residual": residual, "q": q.reshape(t, -1), "k": k.reshape(t, -1),
               "act": act, "kc": None, "vc": None}
        fp8 = case.get("kv") == "fp8"
        if not fp8:
            for name, new in (("kc", k), ("vc", v)):
                c = s[name].double()
                c.view(-1, *c.shape[2:])[s["slots"]] = new.double()
                out[name] = c
        if kind == "layer":
            rows = torch.empty(t, case["hq"], d, dtype=torch.float64, device=DEV)
            for b, n in enumerate(_decode_lens(case)):
                kk, vv = (_gather(s[c], s["bt"][b], n, None) for c in ("kc", "vc"))
                # (the row the step stores, rounded to the cache's type as any cached row is)
                kk[n - 1] = k[b].to(torch.bfloat16).to(s["kc"].dtype).double()
                vv[n - 1] = v[b].to(s["vc"].dtype).double()
                rows[b] = _attend(q[b:b + 1], kk, vv, s["scale"], n - 1, True, -1, None)[0][0]
            out["o"] = rows
        return out
    if kind == "decode":
        rows = torch.empty(case["batch"], case["hq"], case["d"], dtype=torch.float64, device=DEV)
        for b, n in enumerate(_decode_lens(case)):
            kk, vv = (_gather(s[c], s["bt"][b], n, s["kw"].get(sc))
                      for c, sc in (("kc", "k_scale"), ("vc", "v_scale")))
            rows[b] = _attend(s["q"][b:b + 1], kk, vv, case["d"] ** -0.5, n - 1, True,
                              case["window"], s["sinks"])[0][0]
        return rows
    outs, lses, at, kat = [], [], 0, 0
    if kind == "varlen":
        for n in _lens(case, case["batch"], case["qlo"], case["qhi"], 1):
            sl = slice(at, at + n)
            outs.append(_attend(s["q"][sl], s["k"][sl], s["v"][sl], s["scale"], 0, False, -1,
                                None)[0])
            at += n
        return torch.cat(outs)
    ql, cl = _chunk_lens(case)
    for b, (n, c) in enumerate(zip(ql, cl)):
        q = s["q"][at:at + n]
        if kind == "mla":
            kk = torch.cat([s["kc"][kat:kat + c], s["k"][at:at + n]])
            vv = torch.cat([s["vc"][kat:kat + c], s["v"][at:at + n]])
            o, lse = _attend(q, kk, vv, s["scale"], c, True, -1, None)
            lses.append(lse)
        else:
            bt = s["kw"]["block_table"][b]
            kk, vv = (_gather(s[x], bt, n + c, s["kw"].get(sc))
                      for x, sc in (("kc", "k_descale"), ("vc", "v_descale")))
            o = _attend(q, kk, vv, case["d"] ** -0.5, c, True, case["window"], s["sinks"])[0]
        outs.append(o)
        at, kat = at + n, kat + c
    if kind == "mla":
        return {"out": torch.cat(outs), "lse": torch.cat(lses, dim=1)}
    return torch.cat(outs)
