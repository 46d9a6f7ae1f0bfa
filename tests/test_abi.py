"""The C ABI without a GPU: libfk_amd.so loads, exports every symbol the header
declares, and its host-side logic (planning, argument validation) behaves.

Only calls that return before any HIP launch are made here (argument errors and
the host-only planner), so these tests run on a machine without a GPU.
"""
from __future__ import annotations

import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "fastkernels_amd.h"


@pytest.fixture(scope="module")
def lib():
    from fastkernels_amd import _native, build

    if not _native.LIB_PATH.exists():
        build.build(verbose=False)
    return _native.lib()


def header_symbols() -> list[str]:
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fk_\w+)\s*\(", text)))


def test_header_declares_the_operator_set():
    syms = header_symbols()
    for name in ("fk_rmsnorm", "fk_fused_add_rmsnorm", "fk_rotary_embedding", "fk_store_kvcache",
                 "fk_paged_decode_plan", "fk_paged_decode", "fk_paged_decode_partials",
                 "fk_paged_decode_reduce", "fk_silu_and_mul", "fk_version", "fk_last_error"):
        assert name in syms


def test_library_exports_every_header_symbol(lib):
    from fastkernels_amd import _native

    for name in header_symbols():
        assert hasattr(lib, name), f"{name} declared but not exported"
        assert name in _native.EXPORTED, f"{name} has no ctypes signature"
    if shutil.which("nm"):
        out = subprocess.run(["nm", "-D", "--defined-only", str(_native.LIB_PATH)],
                             capture_output=True, text=True, check=True).stdout
        exported = set(re.findall(r"\sT\s+(fk_\w+)$", out, flags=re.M))
        assert set(header_symbols()) <= exported
        # nothing outside the header leaks as an fk_ entry point
        assert exported <= set(header_symbols())


def test_version_and_clean_error(lib):
    from fastkernels_amd import _native

    # Major version 2: fk_paged_prefill / fk_varlen_prefill took head_size_v, lse and
    # lse_row_stride; the bindings refuse a library of another major version.
    assert lib.fk_version() // 10000 == _native.ABI_MAJOR == 2
    text = HEADER.read_text()
    assert re.search(r"#define FK_VERSION_MAJOR 2\b", text)


def test_prefill_head_sizes_and_lse_arguments(lib):
    """fk_varlen_prefill refuses head-size pairs that are not built (before any launch)
    and names them; the Python layer's table agrees with the C library's."""
    from fastkernels_amd import _native as N
    from fastkernels_amd import ops

    fake = ctypes.c_void_p(0x100000)
    cu = ctypes.c_void_p(0x200000)

    def varlen(d, dv, lse_stride=0):
        return lib.fk_varlen_prefill(fake, 8 * dv, fake, 8 * d, fake, 2 * d, fake, 2 * dv,
                                     cu, cu, 1, 16, 16, 8, 2, d, dv, 0.1, 1, -1, None,
                                     fake if lse_stride else None, lse_stride, None)

    for d, dv in ((48, 48), (128, 64), (192, 192), (512, 512), (80, 72)):
        assert not ops.prefill_heads_supported(d, dv)
        assert varlen(d, dv) == N.FK_ERR_UNSUPPORTED, (d, dv)
        assert "head sizes" in _last_error(lib)
    for d, dv in ((80, 80), (192, 128), (72, 72), (32, 32), (96, 96)):
        assert ops.prefill_heads_supported(d, dv)
    assert not ops.prefill_heads_supported(80, 80, fp8=True)
    assert ops.prefill_heads_supported(128, 128, fp8=True)
    assert varlen(128, 128, lse_stride=-1) == N.FK_ERR_INVALID_ARG


def test_prefill_page_bytes_bound(lib):
    """fk_paged_prefill addresses a page's rows by 32-bit offsets from its first row, so
    it refuses pages of 2^32 bytes or more (before any launch); one byte less per page
    passes that check."""
    from fastkernels_amd import _native as N

    fake = ctypes.c_void_p(0x100000)
    cu = ctypes.c_void_p(0x200000)

    def paged(block_size, hk, d):
        return lib.fk_paged_prefill(fake, 32 * d, fake, 32 * d, fake, fake, N.FK_DTYPE_BF16,
                                    None, None, fake, 4, cu, cu, 1, 0, 0, 32, hk, d, d,
                                    block_size, 1, 0.1, 1, -1, None, None)

    # 2^22 slots of 8 heads x 128 bf16 (2 KiB rows): 2^33 bytes per page
    assert paged(1 << 22, 8, 128) == N.FK_ERR_INVALID_ARG
    assert "2^32" in _last_error(lib)
    # 2^20 slots of 2 KiB rows: 2^31 bytes; max_seqlen_q 0 then returns before launching
    assert paged(1 << 20, 8, 128) == N.FK_OK


def _last_error(lib) -> str:
    return lib.fk_last_error().decode()


def test_plan_host_logic(lib):
    from fastkernels_amd import _native

    part, nparts, ws = _native.plan(64, 32, 8, 128, 8192, 0)
    assert part == 0 and nparts >= 1  # balanced: one range per work-group
    rows = nparts * 2 * 32
    assert ws >= rows * 128 * 4 + rows * 8 + (64 + 2) * 4
    part, nparts, ws = _native.plan(64, 32, 8, 128, 8192, 16)
    assert (part, nparts) == (512, 16)
    part, nparts, _ = _native.plan(8, 64, 8, 128, 131072, 64)
    assert (part, nparts) == (2048, 64)
    part, nparts, _ = _native.plan(4, 32, 8, 128, 100, 3)  # rounds up to 64-token units
    assert part == 64 and nparts == 2
    part, nparts, _ = _native.plan(10000, 32, 8, 128, 4096, 0)  # too many for LDS prefix sums
    assert part > 0
    # head sizes 64 / 256: partial rows of head_size floats
    _, n64, ws64 = _native.plan(64, 32, 8, 64, 8192, 0)
    _, n256, ws256 = _native.plan(64, 32, 8, 256, 8192, 0)
    assert n64 == n256 and ws256 - ws64 >= n64 * 2 * 32 * (256 - 64) * 4
    # Balanced group counts, relative to C3's (8 kv heads: one work-group per CU).
    # Fewer than 8 virtual heads: 4 / Hk work-groups per CU, whatever the group size
    # (a group above 16 query heads takes one wave per 16 query columns).
    _, n_c3, _ = _native.plan(64, 32, 8, 128, 8192, 0)
    _, n_g32, _ = _native.plan(64, 64, 2, 128, 8192, 0)  # 2 kv heads x 2 column blocks
    _, n_g8, _ = _native.plan(64, 16, 2, 128, 8192, 0)   # 2 kv heads x 1 column block
    assert n_g8 == n_g32 == 2 * n_c3
    assert _native.plan(64, 8, 1, 128, 8192, 0)[1] == 4 * n_c3
    assert _native.plan(64, 16, 4, 128, 8192, 0)[1] == n_c3
    # Several full groups of 8 virtual heads: one work-group per CU over all of them;
    # a last group with idle waves keeps one per CU per group.
    assert _native.plan(16, 32, 32, 128, 8192, 0)[1] * 4 == n_c3
    assert _native.plan(64, 20, 20, 64, 8192, 0)[1] == n_c3
    with pytest.raises(_native.FkError, match="head_size"):
        _native.plan(64, 32, 8, 96, 8192, 0)
    with pytest.raises(_native.FkError):
        _native.plan(-1, 32, 8, 128, 10, 0)


def test_decode_work_groups_fit_the_kernel(lib):
    """A work-group of the partition kernel has waves * shares waves of 64 lanes, bounded to
    512 threads; waves is one of the counts the kernels are built for and covers the heads
    (three heads used to run as eight waves in two shares: 1024 threads)."""
    from fastkernels_amd import _native

    shares_seen = set()
    for hk in (1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 20):
        for group in (1, 3, 16, 17, 40):
            for d in (64, 128, 256):
                for batch in (1, 3, 17, 60, 100, 300, 5000):
                    for part, parts, window in ((512, 1, -1), (512, 4, -1), (512, 16, 100),
                                                (0, 256, -1), (0, 256, 0), (0, 256, 127),
                                                (0, 256, 1023), (0, 256, 5000)):
                        for kv in (_native.FK_DTYPE_BF16, _native.FK_DTYPE_FP8_E4M3FN):
                            what = (batch, hk * group, hk, d, kv, window, part, parts)
                            waves, shares, whole = _native.decode_shape(*what)
                            assert waves in (1, 2, 4, 8) and shares in (1, 2, 4, 8), what
                            assert waves * shares <= 8, what
                            assert whole <= (part == 0 and window >= 0), what
                            assert shares == 1 or whole or part > 0, what
                            shares_seen.add((whole, shares))
    assert shares_seen == {(False, 1), (False, 2), (True, 1), (True, 2), (True, 4), (True, 8)}
    # The shape that made the illegal work-group: 3 kv heads, 100 sequences, 4 partitions.
    bf16, fp8 = _native.FK_DTYPE_BF16, _native.FK_DTYPE_FP8_E4M3FN
    assert _native.decode_shape(100, 9, 3, 64, bf16, -1, 512, 4) == (4, 2, False)
    # Eight shares over fp8 pages: up to two work-groups per CU (256 without a GPU).
    assert _native.decode_shape(64, 32, 8, 128, fp8, 1023, 0, 256) == (1, 8, True)
    assert _native.decode_shape(65, 32, 8, 128, fp8, 1023, 0, 256)[2] is False
    assert _native.decode_shape(65, 32, 8, 128, bf16, 1023, 0, 256) == (1, 8, True)


def test_prefill_order_rule(lib):
    """fk_prefill_shape's item order: longest first for ragged launches that hold more
    work-groups than CUs or chunks over long caches, the grid's own for equal or short
    lengths, small launches, more than 64 sequences, and where the search would outweigh the
    items."""
    from fastkernels_amd import _native as N

    def order(batch, max_q, total_q, max_k=0, hq=32, hk=8, d=128, causal=True, window=-1, ws=True):
        return N.prefill_shape(True, N.FK_DTYPE_BF16, batch, total_q, max_q, max_k or max_q, hq,
                               hk, d, d, causal, window, ws)[3]

    assert order(16, 1500, 13000) == 16          # ragged prompts
    assert order(16, 1500, 16 * 1500) == 0       # equal ones
    assert order(65, 1500, 50000) == 0           # past the ordering's 64
    assert order(1, 1500, 1500) == 1             # one sequence: its blocks in order
    assert order(64, 40, 1300) == 0              # short
    assert order(64, 200, 7000) == 0             # many short ones: the search outweighs them
    assert order(5, 200, 600) == 0               # fewer work-groups than CUs
    assert order(16, 300, 3000, max_k=4300) == 16  # ragged chunks over long caches
    assert order(16, 300, 3000, max_k=4300, window=10) == 0  # a short window: few stages
    assert order(64, 200, 64 * 200, max_k=1200) == 64  # equal, keys past the last-level cache
    assert order(64, 200, 64 * 200, max_k=300) == 0
    assert order(64, 600, 64 * 600, hq=16, hk=2, d=256) == 64  # head 256: past the L2s
    assert order(16, 1500, 0, ws=False) == 16    # rows unknown: taken as ragged
    assert order(4, 2000, 7440) == 4             # prompts at 93 % of the longest: long ones
    assert order(4, 2000, 7840) == 0             # 98 %
    assert order(32, 300, 8930) == 0             # 93 %, short ones
    assert order(16, 256, 16 * 256, max_k=4256) == 16  # equal chunks: caches of any lengths
    assert order(16, 256, 16 * 256, max_k=1256) == 0   # over short ones
    assert order(16, 256, 16 * 256, max_k=4256, window=500) == 0
    # Not causal: keys of other lengths than the queries, and keys past the L2s whose heads
    # stay on one XCD each.
    assert order(4, 1200, 4800, max_k=1600, hq=16, hk=16, causal=False) == 4
    assert order(4, 1200, 4800, hq=16, hk=16, causal=False) == 0
    assert order(32, 700, 32 * 700, hq=16, hk=16, d=64, causal=False) == 32
    assert order(32, 700, 32 * 700, hq=20, hk=20, d=64, causal=False) == 0
    assert order(64, 150, 64 * 150, hq=16, hk=16, d=128, causal=False) == 0  # short


def test_argument_errors_return_before_launch(lib):
    from fastkernels_amd import _native as N

    fake = ctypes.c_void_p(0x100000)  # never dereferenced: every call below is rejected first
    stream = ctypes.c_void_p(0)
    rc = lib.fk_store_kvcache(fake, 8, fake, 8, fake, fake, fake, 1, 4, 8, 3, 64, stream)
    assert rc == N.FK_ERR_INVALID_ARG and "elem_bytes" in _last_error(lib)
    rc = lib.fk_store_kvcache(fake, 4, fake, 8, fake, fake, fake, 1, 4, 8, 2, 64, stream)
    assert rc == N.FK_ERR_INVALID_ARG and "stride" in _last_error(lib)
    rc = lib.fk_rmsnorm(fake, 64, fake, 64, fake, 2, 64, 1e-6, 9, stream)
    assert rc == N.FK_ERR_UNSUPPORTED and "dtype" in _last_error(lib)
    rc = lib.fk_fused_add_rmsnorm(fake, 32, fake, 64, fake, 2, 64, 1e-6, N.FK_DTYPE_BF16, stream)
    assert rc == N.FK_ERR_INVALID_ARG
    rc = lib.fk_rotary_embedding(fake, fake, 512, fake, 128, fake, 0, 100, 4, 4, 1, 128, 127, 1,
                                 N.FK_DTYPE_BF16, stream)
    assert rc == N.FK_ERR_INVALID_ARG and "rot_dim" in _last_error(lib)
    rc = lib.fk_silu_and_mul(fake, 4, fake, 4, -1, 2, N.FK_DTYPE_BF16, stream)
    assert rc == N.FK_ERR_INVALID_ARG

    def decode(**kw):
        a = dict(head=128, hq=32, hk=8, bs=256, nb=64, part=512, nparts=4, ws=fake, wsb=1 << 30,
                 kv=N.FK_DTYPE_BF16, window=-1)
        a.update(kw)
        return lib.fk_paged_decode(fake, a["hq"] * 128, fake, a["hq"] * 128, fake, fake, a["kv"],
                                   None, None, fake, 32, fake, 4, a["hq"], a["hk"], a["head"],
                                   a["bs"], a["nb"], 0.088, a["window"], None, a["part"],
                                   a["nparts"], a["ws"], a["wsb"], stream)

    assert decode(head=96) == N.FK_ERR_UNSUPPORTED and "head_size" in _last_error(lib)
    assert decode(head=512) == N.FK_ERR_UNSUPPORTED and "head_size" in _last_error(lib)
    assert decode(hq=30, hk=8) == N.FK_ERR_INVALID_ARG
    assert decode(bs=24) == N.FK_ERR_INVALID_ARG and "block_size" in _last_error(lib)
    assert decode(part=100) == N.FK_ERR_INVALID_ARG and "part_tokens" in _last_error(lib)
    assert decode(kv=N.FK_DTYPE_F32) == N.FK_ERR_INVALID_ARG
    assert decode(nb=0) == N.FK_ERR_INVALID_ARG and "block" in _last_error(lib)
    assert decode(wsb=16) == N.FK_ERR_WORKSPACE and "workspace" in _last_error(lib)
    assert decode(ws=None, part=0, nparts=256) == N.FK_ERR_WORKSPACE
    assert decode(window=-2) == N.FK_ERR_INVALID_ARG and "window_left" in _last_error(lib)


def test_python_layer_fails_loudly_without_gpu(lib):
    """No CPU fallback: CPU tensors are rejected, not computed."""
    import torch

    from fastkernels_amd import ops

    x = torch.zeros(4, 2 * 64, dtype=torch.bfloat16)
    out = torch.empty(4, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="GPU"):
        ops.silu_and_mul(out, x)
    with pytest.raises(RuntimeError, match="GPU"):
        ops.rms_norm(torch.empty(4, 64), torch.zeros(4, 64), torch.ones(64), 1e-6)


@pytest.mark.parametrize("wrong", ["key", "value", "k_cache", "v_cache"])
def test_qk_norm_rope_store_names_the_wrong_dtype(lib, wrong):
    import torch

    from fastkernels_amd import ops

    bf16 = dict(dtype=torch.bfloat16)
    t = dict(query=torch.zeros(2, 256, **bf16), key=torch.zeros(2, 128, **bf16),
             value=torch.zeros(2, 128, **bf16), k_cache=torch.zeros(1, 16, 2, 64, **bf16),
             v_cache=torch.zeros(1, 16, 2, 64, **bf16))
    t[wrong] = t[wrong].float()
    with pytest.raises(TypeError, match=rf"qk_norm_rope_store: {wrong} dtype"):
        ops.qk_norm_rope_store(torch.zeros(2, dtype=torch.int64), t["query"], t["key"], t["value"],
                               t["k_cache"], t["v_cache"], torch.zeros(2, dtype=torch.int64), 64,
                               torch.zeros(8, 64), True)


def test_missing_library_raises(monkeypatch, tmp_path):
    from fastkernels_amd import _native

    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setenv("FASTKERNELS_AMD_LIB", str(tmp_path / "absent.so"))
    with pytest.raises(RuntimeError, match="no fallback"):
        _native.lib()
    monkeypatch.setattr(_native, "_lib", None)
