"""Host-side contract of libdsv3fp8.so: it loads without a GPU, exports every symbol
include/dsv3_fp8.h declares, and validates arguments before touching HIP."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parent.parent
HEADER = ROOT / "include" / "dsv3_fp8.h"


@pytest.fixture(scope="module")
def L():
    from dsv3fp8 import _lib
    return _lib


def test_exports_every_declared_symbol(L):
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    declared = set(re.findall(r"\b(dsv3_[a-z0-9_]+)\s*\(", text))
    assert declared == set(L.EXPORTS), (declared, set(L.EXPORTS))
    for name in declared:
        assert hasattr(L.lib, name)
    assert L.lib.dsv3_version() >= 100


def test_status_strings(L):
    seen = {L.status_string(c) for c in range(8)}
    assert len(seen) == 8 and "ok" in seen
    assert L.status_string(12345) == "unknown status"


A16 = 0x1000  # a fake, 16-byte aligned, non-null address: validation must reject before dereferencing


def test_act_quant_validation(L):
    f = L.lib.dsv3_act_quant
    assert f(None, L.BF16, A16, A16, 128, 128, 128, 0, None) == 1
    assert f(A16, L.BF16, None, A16, 128, 128, 128, 0, None) == 1
    assert f(A16, L.BF16, A16, None, 128, 128, 128, 0, None) == 1
    assert f(A16, L.BF16, A16, A16, 100, 100, 128, 0, None) == 2        # last dim % block (kernel.py:52)
    assert f(A16, L.BF16, A16, A16, -128, 128, 128, 0, None) == 2
    assert f(A16, L.BF16, A16, A16, 384, 256, 128, 0, None) == 2        # numel not a multiple of last dim
    assert f(A16, L.BF16, A16, A16, 128, 128, 100, 0, None) == 2        # any block size, but it must divide the last dim
    assert f(A16, L.BF16, A16, A16, 128, 128, 0, 0, None) == 3
    assert f(A16, L.BF16, A16, A16, 128, 128, -128, 0, None) == 3
    assert f(A16 + 2, L.BF16, A16, A16, 128, 128, 128, 0, None) == 4
    assert f(A16, 9, A16, A16, 128, 128, 128, 0, None) == 5
    assert f(A16, L.BF16, A16, A16, 128, 128, 128, 7, None) == 5
    assert f(None, L.BF16, None, None, 0, 128, 128, 0, None) == 0       # empty input: nothing to do


def test_weight_dequant_validation(L):
    f = L.lib.dsv3_weight_dequant
    assert f(None, A16, A16, L.BF16, 128, 128, 128, None) == 1
    assert f(A16, None, A16, L.BF16, 128, 128, 128, None) == 1
    assert f(A16, A16, None, L.BF16, 128, 128, 128, None) == 1
    assert f(A16, A16, A16, L.BF16, -1, 128, 128, None) == 2
    assert f(A16, A16, A16, L.BF16, 128, 128, 0, None) == 3
    assert f(A16, A16, A16, 5, 128, 128, 128, None) == 5
    assert f(A16, A16, A16 + 1, L.BF16, 128, 128, 128, None) == 4
    assert f(None, None, None, L.BF16, 0, 128, 128, None) == 0


def test_weight_quant_validation(L):
    f = L.lib.dsv3_weight_quant
    assert f(None, L.BF16, A16, A16, 128, 128, 128, 0, None) == 1
    assert f(A16, L.BF16, None, A16, 128, 128, 128, 0, None) == 1
    assert f(A16, L.BF16, A16, None, 128, 128, 128, 0, None) == 1
    assert f(A16, L.BF16, A16, A16, 128, -1, 128, 0, None) == 2
    assert f(A16, L.BF16, A16, A16, 128, 128, 64, 0, None) == 3         # only 128 x 128 blocks exist on disk
    assert f(A16, L.BF16, A16, A16, 128, 128, 128, 5, None) == 5        # unknown scale format
    assert f(A16, 7, A16, A16, 128, 128, 128, 0, None) == 5
    assert f(A16 + 1, L.BF16, A16, A16, 128, 128, 128, 0, None) == 4
    assert f(A16, L.BF16, A16, A16 + 2, 128, 128, 128, 0, None) == 4
    assert f(None, L.BF16, None, None, 0, 128, 128, 0, None) == 0


@pytest.mark.parametrize("entry", ["dsv3_fp8_gemm", "dsv3_fp8_gemm_pow2"])
def test_fp8_gemm_validation(L, entry):
    f = getattr(L.lib, entry)
    ws = L.lib.dsv3_fp8_gemm_workspace_bytes
    assert f(None, A16, A16, A16, A16, L.BF16, 4, 128, 128, None, 0, None) == 1
    assert f(A16, A16, A16, A16, None, L.BF16, 4, 128, 128, None, 0, None) == 1
    assert f(A16, A16, A16, A16, A16, L.BF16, 70000, 128, 100, None, 0, None) == 2    # K % 128 != 0 is served by a fallback whose grid takes m <= 65535
    assert f(A16, A16, A16, A16, A16, L.BF16, -4, 128, 128, None, 0, None) == 2
    assert f(A16 + 8, A16, A16, A16, A16, L.BF16, 4, 128, 128, None, 0, None) == 4
    assert f(A16, A16, A16, A16, A16, 3, 4, 128, 128, None, 0, None) == 5
    assert f(None, None, None, None, None, L.BF16, 0, 128, 128, None, 0, None) == 0
    need = ws(8, 1536, 7168)
    assert need > 0 and ws(4096, 18432, 7168) == 0 and ws(0, 1, 128) == 0 and ws(8, 8, 100) == 0
    assert f(A16, A16, A16, A16, A16, L.BF16, 8, 1536, 7168, None, 0, None) == 6
    assert f(A16, A16, A16, A16, A16, L.BF16, 8, 1536, 7168, A16, need - 1, None) == 6
    assert f(A16, A16, A16, A16, A16, L.BF16, 8, 1536, 7168, A16 + 16, need, None) == 6


def test_fp8_gemm_static_reports_argument_errors_before_the_size_limit(L):
    """The entry point that allocates nothing checks its arguments like dsv3_fp8_gemm and only then the size of its
    scratch array: a malformed call on a large shape reports what is wrong with it, not DSV3_ERR_TOO_LARGE."""
    f = L.lib.dsv3_fp8_gemm_static
    big = (9, 129280, 7168)                                               # 84 MiB of partial sums: beyond the array
    assert L.lib.dsv3_fp8_gemm_workspace_bytes(*big) > L.lib.dsv3_fp8_gemm_static_max_bytes()
    assert f(A16, A16, A16, A16, A16, L.BF16, *big, None) == 8            # well-formed: refused for its size
    assert f(A16, A16, A16, A16, A16, 3, *big, None) == 5                 # bad dtype code
    assert f(None, A16, A16, A16, A16, L.BF16, *big, None) == 1
    assert f(A16 + 8, A16, A16, A16, A16, L.BF16, *big, None) == 4
    assert f(A16, A16, A16, A16, A16, L.BF16, 70000, 129280, 7168 + 64, None) == 2   # K % 128 != 0 with more rows than its fallback takes
    assert f(A16, A16, A16, A16, A16, L.BF16, -9, 129280, 7168, None) == 2
    assert f(None, None, None, None, None, L.BF16, 0, 129280, 7168, None) == 0   # nothing to do


def test_ops_shape_inference_and_no_cpu_fallback():
    import dsv3fp8  # noqa: F401  (registers the ops)
    x = torch.empty(2, 3, 256, device="meta", dtype=torch.bfloat16)
    y, s = torch.ops.dsv3fp8.act_quant(x, 128, 0)
    assert y.shape == (2, 3, 256) and y.dtype == torch.float8_e4m3fn and s.shape == (2, 3, 2) and s.dtype == torch.float32
    w = torch.empty(576, 256, device="meta", dtype=torch.float8_e4m3fn)
    ws = torch.empty(5, 2, device="meta")
    assert torch.ops.dsv3fp8.weight_dequant(w, ws, 128, 0).dtype == torch.bfloat16
    c = torch.ops.dsv3fp8.fp8_gemm(y, s, w, ws, 0)
    assert c.shape == (2, 3, 576) and c.dtype == torch.bfloat16
    with pytest.raises((NotImplementedError, RuntimeError)):
        torch.ops.dsv3fp8.act_quant(torch.zeros(1, 128, dtype=torch.bfloat16), 128, 0)   # CPU tensors: no kernel


def test_python_wrappers_keep_the_reference_asserts():
    import dsv3fp8
    x = torch.empty(4, 100, device="meta", dtype=torch.bfloat16)
    with pytest.raises(AssertionError, match="divisible by block_size"):
        dsv3fp8.act_quant(x)
    with pytest.raises(AssertionError, match="contiguous"):
        dsv3fp8.act_quant(torch.empty(256, 4, device="meta", dtype=torch.bfloat16).t())
    with pytest.raises(AssertionError, match="2 dimensions"):
        dsv3fp8.weight_dequant(torch.empty(2, 4, 4, device="meta", dtype=torch.float8_e4m3fn), torch.empty(1, 1, device="meta"))


def test_grouped_validation(L):
    f = L.lib.dsv3_fp8_gemm_grouped
    assert L.lib.dsv3_fp8_gemm_grouped_tile_rows() > 0
    ok = dict(a=A16, a_s=A16, a_rows=None, an=64, b=A16, b_s=A16, bst=128 * 128, sst=1, c=A16, cd=L.BF16,
              m=64, n=128, k=128, tg=A16, t0=A16, tr=A16, nt=2, st=None)

    def call(**kw):
        v = {**ok, **kw}
        return f(*[v[key] for key in ("a", "a_s", "a_rows", "an", "b", "b_s", "bst", "sst", "c", "cd", "m", "n", "k",
                                      "tg", "t0", "tr", "nt", "st")])
    assert call(a=None) == 1 and call(tg=None) == 1 and call(c=None) == 1
    assert call(k=100) == 2 and call(k=0) == 2 and call(m=-1) == 2 and call(nt=-1) == 2
    assert call(an=1 << 30, k=128 * 64) == 2                 # byte offsets of a beyond 32 bits
    assert call(a=A16 + 4) == 4 and call(bst=100) == 4
    assert call(cd=7) == 5
    assert call(m=0, a=None, tg=None) == 0 and call(nt=0) == 0


def test_grouped_swiglu_validation(L):
    f, fused = L.lib.dsv3_fp8_gemm_grouped_swiglu, L.lib.dsv3_fp8_gemm_grouped_swiglu_fused
    assert fused(4096, 4096, 2048, 7168) and fused(321, 100, 128, 128)
    assert not fused(320, 4096, 2048, 7168)          # few rows in all: the weight-streaming kernel, two calls
    assert not fused(4096, 4096, 2000, 7168) and not fused(4096, 4096, 2048, 7100) and not fused(0, 0, 128, 128)
    ok = dict(a=A16, a_s=A16, a_rows=None, an=4096, b=A16, b_s=A16, bst=256 * 128, sst=2, y=A16, s=A16,
              m=4096, inter=128, k=128, tg=A16, t0=A16, tr=A16, nt=40, blk=128, fmt=0, st=None)

    def call(**kw):
        v = {**ok, **kw}
        return f(*[v[key] for key in ("a", "a_s", "a_rows", "an", "b", "b_s", "bst", "sst", "y", "s", "m", "inter", "k",
                                      "tg", "t0", "tr", "nt", "blk", "fmt", "st")])
    assert call(a=None) == 1 and call(y=None) == 1 and call(s=None) == 1 and call(tr=None) == 1
    assert call(k=100) == 2 and call(inter=100) == 2 and call(m=-1) == 2
    assert call(m=100) == 2                          # below the tile kernel's range: ask ..._fused first
    assert call(blk=64) == 3 and call(fmt=5) == 5
    assert call(a=A16 + 8) == 4 and call(y=A16 + 2) == 4 and call(bst=100) == 4
    assert call(m=0) == 0 and call(nt=0) == 0


def test_group_tiles_validation(L):
    f = L.lib.dsv3_group_tiles
    assert f(None, 4, 8, A16, A16, A16, None) == 1
    assert f(A16, 4, 8, None, A16, A16, None) == 1
    assert f(A16, -1, 8, A16, A16, A16, None) == 2
    assert f(A16, 4, 0, None, None, None, None) == 0


def test_swiglu_quant_validation(L):
    f = L.lib.dsv3_swiglu_quant
    assert f(None, L.BF16, A16, A16, 4, 128, 128, 0, None) == 1
    assert f(A16, L.F32, A16, A16, 4, 128, 128, 0, None) == 5          # bf16 only
    assert f(A16, L.BF16, A16, A16, 4, 128, 64, 0, None) == 3
    assert f(A16, L.BF16, A16, A16, 4, 100, 128, 0, None) == 2
    assert f(A16, L.BF16, A16, A16, 4, 128, 128, 9, None) == 5
    assert f(A16 + 2, L.BF16, A16, A16, 4, 128, 128, 0, None) == 4
    assert f(None, L.BF16, None, None, 0, 128, 128, 0, None) == 0


def test_moe_combine_validation(L):
    f = L.lib.dsv3_moe_combine
    assert f(None, L.BF16, A16, A16, None, A16, 4, 2, 128, None) == 1
    assert f(A16, L.BF16, A16, A16, None, None, 4, 2, 128, None) == 1
    assert f(A16, L.F16, A16, A16, None, A16, 4, 2, 128, None) == 5
    assert f(A16, L.BF16, A16, A16, None, A16, 4, 2, 100, None) == 2
    assert f(A16 + 2, L.BF16, A16, A16, None, A16, 4, 2, 128, None) == 4
    assert f(None, L.BF16, None, None, None, None, 0, 2, 128, None) == 0


def test_moe_route_validation(L):
    f = L.lib.dsv3_moe_route
    #     idx  w    dtype   tok topk exp shared max_tiles scratch a_rows rows w_sorted tile tables    stream
    ok = [A16, A16, L.BF16, 4,  2,   8,  0,     12,       A16,    A16,   A16, A16,     A16, A16, A16, None]

    def call(i=None, v=None):
        a = list(ok)
        if i is not None:
            a[i] = v
        return f(*a)
    assert call(0, None) == 1 and call(8, None) == 1 and call(12, None) == 1
    assert call(2, L.F32) == 5
    assert call(4, 0) == 2 and call(4, 17) == 2 and call(5, 0) == 2 and call(3, -1) == 2
    assert call(0, A16 + 4) == 4


def test_wkv_b_absorb_validation(L):
    f = L.lib.dsv3_wkv_b_absorb
    #     x    ts        hs   w    ws   y    dtype   side tokens heads nope v   kv_rank block stream
    ok = [A16, 128 * 192, 192, A16, A16, A16, L.BF16, 0,   4,     128,  128, 128, 512,   128,  None]

    def call(i=None, v=None):
        a = list(ok)
        if i is not None:
            a[i] = v
        return f(*a)
    assert call(0, None) == 1 and call(3, None) == 1 and call(4, None) == 1 and call(5, None) == 1
    assert call(6, L.F32) == 5
    assert call(13, 64) == 3
    assert call(7, 2) == 2                         # neither side
    assert call(10, 32) == 2 and call(10, 96) == 2  # side Q implements nope_dim 64 and 128
    assert call(12, 500) == 2 and call(11, 100) == 2
    assert call(2, 100) == 2 and call(1, 12) == 2   # head stride shorter than the row / strides not multiples of 8
    assert call(0, A16 + 8) == 4 and call(5, A16 + 2) == 4
    assert call(8, -1) == 2 and call(9, 70000) == 2
    assert call(8, 0) == 0                           # nothing to do: no launch, no dereference
    v = list(ok); v[7] = 1; v[12] = 384
    assert f(*v) == 2                               # side V implements kv_rank 128, 256, 512


def test_gate_route_validation(L):
    f = L.lib.dsv3_gate_route
    #     logits dtype   bias  w    idx  tokens experts topk groups topk_groups func scale stream
    ok = [A16,   L.BF16, None, A16, A16, 4,     256,    8,   8,     4,          1,   2.5,  None]

    def call(i=None, v=None):
        a = list(ok)
        if i is not None:
            a[i] = v
        return f(*a)
    assert call(0, None) == 1 and call(3, None) == 1 and call(4, None) == 1
    assert call(1, L.F32) == 5 and call(10, 2) == 5
    assert call(6, 513) == 2 and call(7, 0) == 2 and call(7, 65) == 2 and call(5, -1) == 2
    assert call(8, 7) == 2                          # experts not divisible by the number of groups
    assert call(9, 9) == 2 and call(9, 0) == 2
    a = list(ok); a[8], a[9], a[7] = 64, 1, 8       # one group of 4 experts cannot supply 8
    assert f(*a) == 2
    assert call(0, A16 + 1) == 4 and call(4, A16 + 4) == 4
    assert call(5, 0) == 0


def test_linear_fp8_validation(L):
    f, fused = L.lib.dsv3_linear_fp8, L.lib.dsv3_linear_fp8_fused
    assert fused(1, 1536, 7168) and fused(2, 7168, 16384) and not fused(16, 7168, 16384) and not fused(17, 1536, 7168)
    # 3+ rows: two calls wherever fp8_gemm takes the activation-streaming kernel (K of 512 and more); one and two rows
    # are always one call
    assert fused(8, 4096, 256) and not fused(8, 24576, 1536) and not fused(8, 7168, 16384)
    assert fused(1, 24576, 1536) and fused(2, 576, 7168) and fused(1, 32768, 512)
    assert not fused(4096, 1536, 7168)
    assert not fused(4, 1536, 7000) and not fused(0, 8, 128)
    #     x    dtype   b    b_s  c    cdtype  m  n     k     block fmt ws    ws_bytes stream
    ok = [A16, L.BF16, A16, A16, A16, L.BF16, 2, 1536, 7168, 128,  0,  A16 * 16, 1 << 30, None]

    def call(i=None, v=None):
        a = list(ok)
        if i is not None:
            a[i] = v
        return f(*a)
    assert call(0, None) == 1 and call(2, None) == 1 and call(3, None) == 1 and call(4, None) == 1
    assert call(1, L.F32) == 5 and call(5, 7) == 5 and call(10, 3) == 5
    assert call(9, 64) == 3
    assert call(8, 7000) == 2 and call(6, 64) == 2          # K not a multiple of 128; too many rows for the fused kernel
    assert call(0, A16 + 2) == 4
    assert call(11, None) == 6 and call(12, 16) == 6         # the split-K workspace is required and checked
    assert call(6, 0) == 0


def test_mla_prefill_validation(L):
    def call(q=A16, kv=A16, pe=A16, w=A16, y=A16, s=A16, mask=None, md=0, b=2, rows=64, pos=64, heads=4, nope=128, rope=64,
             v=128, c=512, kvs=64 * 512, pes=64 * 64, scale=0.1, ws=0x1000, wsb=1 << 40, freqs=A16):
        return L.lib.dsv3_mla_prefill(q, freqs, kv, kvs, pe, pes, w, A16, mask, md, y, s, b, rows, pos, heads, nope, rope, v, c,
                                      scale, ws, wsb, None)
    for name in ("q", "kv", "pe", "w", "y", "s", "freqs"):
        assert call(**{name: None}) == 1
    for bad in ({"nope": 64}, {"rope": 32}, {"v": 64}, {"c": 256}, {"b": -1}, {"rows": -1}, {"pos": 0}, {"heads": 65536},
                {"kvs": 64 * 512 - 8}, {"pes": 64 * 64 + 4}, {"scale": 0.0}, {"scale": float("nan")}):
        assert call(**bad) == 2, bad
    for name in ("q", "kv", "pe", "w", "y"):
        assert call(**{name: A16 + 8}) == 4
    assert call(mask=A16, md=L.F16) == 5 and call(mask=A16 + 1) == 4
    need = L.lib.dsv3_mla_prefill_workspace_bytes(2, 64, 64, 4)
    assert need > 0 and call(ws=None) == 6 and call(wsb=need - 1) == 6 and call(ws=0x1080) == 6
    assert call(b=0, q=None) == 0 and call(rows=0, q=None) == 0
    assert L.lib.dsv3_mla_prefill_workspace_bytes(0, 64, 64, 4) == 0


def test_mla_decode_validation(L):
    def call(q=A16, kv=A16, pe=A16, w=A16, y=A16, mask=None, md=0, b=2, rows=1, pos=64, heads=4, nope=128, rope=64,
             v=128, c=512, kvs=64 * 512, pes=64 * 64, scale=0.1, ws=0x1000, wsb=1 << 40, freqs=A16):
        return L.lib.dsv3_mla_decode(q, freqs, kv, kvs, pe, pes, w, A16, mask, md, y, b, rows, pos, heads, nope, rope, v, c,
                                     scale, ws, wsb, None)
    for name in ("q", "kv", "pe", "w", "y", "freqs"):
        assert call(**{name: None}) == 1
    for bad in ({"nope": 64}, {"c": 256}, {"b": -1}, {"rows": -1}, {"pos": 0}, {"kvs": 64 * 512 - 8}, {"scale": 0.0}):
        assert call(**bad) == 2, bad
    for name in ("q", "kv", "pe", "w", "y"):
        assert call(**{name: A16 + 8}) == 4
    need = L.lib.dsv3_mla_decode_workspace_bytes(2, 1, 64, 4)
    assert need > 0 and call(ws=None) == 6 and call(wsb=need - 1) == 6 and call(ws=0x1080) == 6
    assert call(b=0, q=None) == 0 and L.lib.dsv3_mla_decode_workspace_bytes(2, 0, 64, 4) == 0


def test_mla_decode_quant_validation(L):
    def call(q=A16, kv=A16, pe=A16, w=A16, w_s=A16, y=A16, s=A16, mask=None, md=0, b=2, rows=1, pos=64, heads=4, nope=128, rope=64,
             v=128, c=512, kvs=64 * 512, pes=64 * 64, scale=0.1, ws=0x1000, wsb=1 << 40, freqs=A16):
        return L.lib.dsv3_mla_decode_quant(q, freqs, kv, kvs, pe, pes, w, w_s, mask, md, y, s, b, rows, pos, heads, nope, rope, v, c,
                                           scale, ws, wsb, None)
    for name in ("q", "kv", "pe", "w", "w_s", "y", "s", "freqs"):
        assert call(**{name: None}) == 1
    for bad in ({"nope": 64}, {"v": 64}, {"c": 256}, {"b": -1}, {"rows": -1}, {"pos": 0}, {"kvs": 64 * 512 - 8}, {"scale": 0.0}):
        assert call(**bad) == 2, bad
    for name in ("q", "kv", "pe", "w", "y"):
        assert call(**{name: A16 + 8}) == 4
    assert call(s=A16 + 2) == 4 and call(w_s=A16 + 2) == 4 and call(mask=A16, md=L.F16) == 5
    need = L.lib.dsv3_mla_decode_workspace_bytes(2, 1, 64, 4)
    assert call(ws=None) == 6 and call(wsb=need - 1) == 6 and call(ws=0x1080) == 6
    assert call(b=0, q=None) == 0 and call(rows=0, q=None) == 0


def test_mla_latent_gemm_validation(L):
    def call(x=A16, x_s=A16, w=A16, w_s=A16, k=7168, a=A16, qw=A16, kw=A16, f=A16, kv=A16, kvs=512 * 8, pe=A16, pes=64 * 8, y=A16, s=A16,
             b=2, rows=4, qr=1536, c=512, rope=64, ws=0x1000, wsb=1 << 40):
        return L.lib.dsv3_mla_latent_gemm(x, x_s, w, w_s, k, a, qw, kw, f, kv, kvs, pe, pes, y, s, b, rows, qr, c, rope, 1e-6, 1e-6, ws, wsb, None)
    for name in ("x", "x_s", "w", "w_s", "a", "qw", "kw", "f", "kv", "pe", "y", "s"):
        assert call(**{name: None}) == 1
        assert call(**{name: A16 + 2}) == 4
    for bad in ({"qr": 100}, {"qr": 2176}, {"c": 256}, {"rope": 32}, {"b": -1}, {"rows": -1}, {"kvs": 2040}, {"k": 7000}, {"k": -128}):
        assert call(**bad) == 2, bad
    need = L.lib.dsv3_fp8_gemm_workspace_bytes(8, 2112, 7168)
    assert need > 0 and call(ws=None) == 6 and call(wsb=need - 1) == 6 and call(ws=0x1080) == 6
    assert call(b=0, a=None) == 0 and call(rows=0, x=None) == 0


def test_mla_latent_validation(L):
    def call(a=A16, stride=2112, qw=A16, kw=A16, f=A16, kv=A16, kvs=512 * 8, pe=A16, pes=64 * 8, y=A16, s=A16, b=2, rows=4,
             qr=1536, c=512, rope=64):
        return L.lib.dsv3_mla_latent(a, stride, qw, kw, f, kv, kvs, pe, pes, y, s, b, rows, qr, c, rope, 1e-6, 1e-6, None)
    for name in ("a", "qw", "kw", "f", "kv", "pe", "y", "s"):
        assert call(**{name: None}) == 1
        assert call(**{name: A16 + 2}) == 4
    for bad in ({"qr": 100}, {"qr": 2176}, {"qr": 0}, {"c": 256}, {"rope": 32}, {"stride": 2104}, {"b": -1}, {"kvs": 2040}):
        assert call(**bad) == 2, bad
    assert call(b=0, a=None) == 0 and call(rows=0, a=None) == 0


# The native operator bodies, called on tensors of the host: they must say no before any pointer gets to a kernel (here a
# body that does not look gets as far as asking for the GPU).
def _gpu_body(name, *args):
    from dsv3fp8 import ops  # noqa: F401  (registers torch.ops.dsv3fp8)
    return getattr(torch.ops.dsv3fp8, name).default.redispatch(torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA), *args)


def _operator_args(name):
    z = torch.zeros
    fp8, bf16 = torch.float8_e4m3fn, torch.bfloat16
    if name == "weight_dequant":
        return [z(128, 128, dtype=fp8), z(1, 1), 128, 0]
    if name in ("fp8_gemm", "fp8_gemm_pow2"):
        return [z(2, 128, dtype=fp8), z(2, 1), z(128, 128, dtype=fp8), z(1, 1), 0]
    if name == "linear_fp8":
        return [z(2, 128, dtype=bf16), z(128, 128, dtype=fp8), z(1, 1), 0, 0]
    freqs, kv, pe = z(2, 32, dtype=torch.complex64), z(1, 8, 512, dtype=bf16), z(1, 8, 64, dtype=bf16)
    if name == "mla_latent":
        return [z(1, 2, 128 + 576, dtype=bf16), z(128, dtype=bf16), z(512, dtype=bf16), freqs, kv, pe, 3, 1e-6, 1e-6]
    if name == "mla_query":         # 20 rows: the branch with the projection's slabs
        return [z(1, 20, 256, dtype=bf16), z(128 + 576, 256, dtype=fp8), z(6, 2), z(128, dtype=bf16), z(512, dtype=bf16), z(20, 32, dtype=torch.complex64),
                z(1, 32, 512, dtype=bf16), z(1, 32, 64, dtype=bf16), 3, 1e-6, 1e-6, z(768, 128, dtype=fp8), z(6, 1), 4]
    args = [z(1, 2, 4, 192, dtype=bf16), freqs, kv, pe, z(1024, 512, dtype=fp8), z(8, 4), z(2, 8), 8, 0.1]
    return args + [False, z(256, 512, dtype=fp8), z(2, 4)] if name == "mla_output" else args


OPERATORS = {"weight_dequant": (0, 1), "fp8_gemm": (0, 1, 2, 3), "fp8_gemm_pow2": (0, 1, 2, 3), "linear_fp8": (0, 1, 2),
             "mla_prefill": range(7), "mla_decode": range(7), "mla_decode_quant": range(7), "mla_output": (*range(7), 10, 11), "mla_latent": range(6),
             "mla_query": (*range(8), 11, 12)}


@pytest.mark.parametrize("name", OPERATORS)
def test_operators_refuse_tensors_of_two_devices(name):
    with pytest.raises(RuntimeError, match="on the GPU"):
        _gpu_body(name, *_operator_args(name))
    for at in OPERATORS[name]:
        args = _operator_args(name)
        args[at] = args[at].to("meta")
        with pytest.raises(RuntimeError, match="one device"):
            _gpu_body(name, *args)


@pytest.mark.parametrize("name", ["mla_prefill", "mla_decode", "mla_decode_quant", "mla_output", "mla_latent", "mla_query"])
def test_attention_operators_refuse_what_their_kernels_cannot_read(name):
    f = {"mla_latent": 3, "mla_query": 5}.get(name, 1)  # where the phases stand
    bad = {f: [lambda t: t.conj(), lambda t: t[:1]]}
    if name in ("mla_latent", "mla_query"):
        bad[f + 3] = [lambda t: 13 if name == "mla_query" else 7, lambda t: -1, lambda t: 2 ** 63 - 1]
        bad[f - 1] = [lambda t: t.float(), lambda t: t[:511]]
        bad[f + 1] = [lambda t: t.float(), lambda t: t[:, ::2]]
    else:                                               # scales: too few rows, columns, another type
        bad[5] = [lambda t: t[:7], lambda t: t[:, :3].contiguous(), lambda t: t.bfloat16(), lambda t: t.flatten()]
        bad[3] = [lambda t: t.float()]
        bad[6] = [lambda t: t[:, :7], lambda t: t.half()]
    if name == "mla_query":
        bad[0] = [lambda t: torch.zeros(1, 20, 512, dtype=t.dtype)[:, :, ::2], lambda t: t[0]]
        bad[1] = [lambda t: t[:703], lambda t: t.bfloat16(), lambda t: t[:, :255], lambda t: t[0]]
        bad[2] = [lambda t: t[:5], lambda t: t[:, :1], lambda t: t.half()]
        bad[11] = [lambda t: t[:767], lambda t: t[0]]
    for at, changes in bad.items():
        for change in changes:
            args = _operator_args(name)
            args[at] = change(args[at])
            with pytest.raises(RuntimeError, match=r"mla[^:]*: (?!tensors|all tensors)"):
                _gpu_body(name, *args)


# (rows, columns, K, taken): sizes on both sides of each limit; past one the large-M kernel is measured faster
@pytest.mark.parametrize("m,n,k,taken", [
    (64, 36864, 7168, False), (65, 36864, 7168, True), (224, 36864, 7168, True), (225, 36864, 7168, False), (65, 36864, 7296, False),
    (129, 32768, 3072, False), (160, 30752, 3584, False), (193, 31744, 7168, False), (129, 32769, 3072, True), (192, 32769, 16384, True),
    (193, 32769, 16384, False), (193, 33761, 16384, True), (192, 40960, 2560, True), (193, 40960, 3584, False), (224, 40960, 4096, True),
    (224, 40961, 4096, False), (65, 36864, 16384, True), (65, 36864, 16896, False), (193, 18432, 7168, False),
    (128, 32768, 16384, True), (128, 24576, 1536, True), (129, 24576, 1536, False), (128, 24576, 1024, False), (65, 28672, 16896, False),
    (65, 22400, 1536, False), (65, 22401, 1536, True),
    (448, 1536, 7168, True), (449, 1536, 7168, False), (320, 2112, 7168, True), (321, 2112, 7168, False), (65, 2305, 7168, False),
    (8192, 128, 4096, True), (8193, 128, 4096, False), (65, 576, 3584, False)])
def test_sizes_that_the_tiles_of_one_round_take(L, m, n, k, taken):
    supported = L.lib["_ZN4dsv313mid_supportedElll"]            # dsv3::mid_supported(rows, columns, K)
    supported.restype, supported.argtypes = ctypes.c_bool, [ctypes.c_int64] * 3
    assert supported(m, n, k) == taken


# the window of 129 .. 256 rows: rows, tiles of 128 columns, units that slices and columns fill, blocks a slice, K
@pytest.mark.parametrize("m,n,k,taken", [
    (129, 7168, 16384, True), (256, 7168, 18432, True), (257, 7168, 16384, False), (128, 7168, 16384, False), (161, 7168, 18944, False),
    (160, 4096, 11264, True), (161, 4096, 11264, False), (129, 3968, 16384, False), (160, 16384, 2048, True), (161, 16384, 16384, False), (129, 16512, 2048, False),
    (150, 12288, 16384, False), (150, 7168, 7168, False), (150, 7168, 11264, True), (193, 7168, 11264, False), (205, 7168, 14848, False), (205, 7168, 15360, True),
    (200, 9216, 16384, False), (200, 10240, 16384, True), (150, 8192, 4096, True), (150, 8192, 4224, False)])
def test_sizes_that_the_sliced_tiles_take(L, m, n, k, taken):
    test_sizes_that_the_tiles_of_one_round_take(L, m, n, k, taken)


@pytest.mark.parametrize("knob", ["DSV3_PREFILL_NOSPLIT=1", "DSV3_PREFILL_TILE=128", "DSV3_PREFILL_NOPP=1", "DSV3_PREFILL_NOPP128=1", "OTHER=1"])
def test_knobs_of_the_large_m_kernel_keep_products_there(knob):
    """A knob that says how the large-M kernel runs its dense tiles holds for every size it had when the knob was made; without K slices no
    product of more than 64 rows asks for scratch."""
    import os
    import subprocess
    import sys
    code = """
import ctypes
from dsv3fp8 import _lib
f = _lib.lib["_ZN4dsv313mid_supportedElll"]
f.restype, f.argtypes = ctypes.c_bool, [ctypes.c_int64] * 3
sizes = [(65, 36864, 7168), (128, 24576, 1536), (448, 1536, 7168)]
print([f(*s) for s in sizes], sum(_lib.lib.dsv3_fp8_gemm_workspace_bytes(*s) for s in sizes))
"""
    name, value = knob.split("=")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT / "deepseek-v3_amd", capture_output=True, text=True, env={**os.environ, name: value})
    assert r.returncode == 0, r.stderr
    taken, scratch = r.stdout.strip().rsplit(" ", 1)
    assert taken == str([name == "OTHER"] * 3)
    assert (scratch == "0") == (name == "DSV3_PREFILL_NOSPLIT")


def test_binding_needs_the_c_library_only():
    """_lib.py by itself (without the package, which registers the torch operators) loads where libdsv3torch.so is not
    built; the package says which command builds it."""
    import subprocess
    import sys
    code = """
import importlib.util, pathlib
exists = pathlib.Path.exists
pathlib.Path.exists = lambda path: path.name != "libdsv3torch.so" and exists(path)
spec = importlib.util.spec_from_file_location("binding", "dsv3fp8/_lib.py")
binding = importlib.util.module_from_spec(spec)
spec.loader.exec_module(binding)
assert binding.lib.dsv3_version() >= 100
try:
    import dsv3fp8
except ImportError as e:
    assert "libdsv3torch.so" in str(e) and "build.py" in str(e)
else:
    raise AssertionError("imported")
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT / "deepseek-v3_amd", capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


@pytest.mark.parametrize("name", ["fp8_gemm", "fp8_gemm_pow2", "linear_fp8", "weight_dequant"])
def test_operators_refuse_operands_that_are_too_small(name):
    """Scales of another type, too few of them, a weight of fewer columns, strided operands: all would be read past their end."""
    weight = {"linear_fp8": 1, "weight_dequant": 0}.get(name, 2)
    bad = {weight + 1: [lambda t: t.bfloat16(), lambda t: t[:0]], weight: [lambda t: t.float()]}
    if name != "weight_dequant":
        bad[weight].append(lambda t: t[:, :127].contiguous())
    bad[weight].append(lambda t: torch.zeros(128, 256).to(t.dtype)[:, ::2])
    if name.startswith("fp8_gemm"):
        bad[0], bad[1] = [lambda t: t.float()], [lambda t: t.half(), lambda t: t[:1]]
    elif name == "linear_fp8":
        bad[0] = [lambda t: torch.zeros(2, 256, dtype=t.dtype)[:, ::2]]
    for at, changes in bad.items():
        for change in changes:
            args = _operator_args(name)
            args[at] = change(args[at])
            with pytest.raises(RuntimeError, match="contiguous"):
                _gpu_body(name, *args)


@pytest.mark.parametrize("block", [0, -128, 2 ** 32 + 128, 2 ** 31])
def test_operators_refuse_block_sizes_that_do_not_fit(block):
    x, w = torch.zeros(2, 256, dtype=torch.bfloat16), torch.zeros(128, 128, dtype=torch.float8_e4m3fn)
    for name, *args in (("act_quant", x, block, 0), ("weight_quant", x, block, 0), ("swiglu_quant", x, block, 0),
                        ("weight_dequant", w, torch.zeros(1, 1), block, 0)):
        with pytest.raises(RuntimeError, match="block_size must"):
            _gpu_body(name, *args)


def test_block_size_zero_divides_by_zero():
    from dsv3fp8 import act_quant, weight_quant
    for call in (act_quant, weight_quant):
        with pytest.raises(ZeroDivisionError):
            call(torch.zeros(128, 128), 0)


@pytest.mark.parametrize("source", ["fp8_gemm_skinny.hip", "fp8_gemm_stream.hip", "fp8_gemm_mid.hip", "mla_decode.hip", "mla_prefill.hip"])
def test_build_refuses_spills(source):
    import build
    assert source in build.NO_SPILL_SOURCES and (build.CSRC / source).exists()
    report = "remark: Function Name: _ZN4dsv317{}EvNS_4ArgsE\nremark:     {}: {}\n"
    for kernel in ("mla_decode_kernelILi0E", "mla_fold_kernelILb1E", "fp8_gemm_mid_kernelILi6E", "mla_expand_kernel", "mla_attend_kernelILb0E"):
        build.check_no_spills(source, report.format(kernel, "VGPRs Spill", 0))
        for what in ("VGPRs Spill", "ScratchSize [bytes/lane]", "SGPRs Spill"):
            with pytest.raises(RuntimeError, match="must not spill"):
                build.check_no_spills(source, report.format(kernel, what, 4))
    build.check_no_spills(source, report.format("mla_attend_kernelILb0E", "SGPRs Spill", 2))


@pytest.mark.parametrize("spilled", [1, 2, 4])
@pytest.mark.parametrize("what", ["VGPRs Spill", "ScratchSize [bytes/lane]"])
def test_attention_kernel_may_keep_scalars_in_lanes_but_spill_no_vector_registers(what, spilled):
    import build
    report = f"remark: Function Name: _ZN4dsv317mla_attend_kernelILb1EEvNS_10AttendArgsE\nremark:     {what}: {spilled}\n"
    with pytest.raises(RuntimeError, match="must not spill"):
        build.check_no_spills("mla_prefill.hip", report)


# Which variant of the decode attention (tiles that a workgroup takes side by side) the cost rule picks (sequences, tokens, positions, heads): at one
# tile a wavefront the measured fastest or one within 1 % of it; then the sizes that tests/test_gpu_mla_attention.py has for each variant.
@pytest.mark.parametrize("side,b,s,t,h", [
    (1, 1, 1, 40, 128), (1, 1, 1, 300, 128), (2, 1, 1, 700, 128), (1, 2, 1, 300, 128), (1, 3, 1, 200, 128), (1, 4, 1, 128, 128), (1, 48, 1, 4096, 128),
    (1, 64, 1, 4096, 128), (1, 96, 1, 2000, 128), (2, 12, 1, 4096, 128), (2, 24, 1, 2000, 128), (2, 32, 1, 4096, 128), (2, 64, 1, 1000, 128),
    (4, 1, 1, 1000, 128), (4, 2, 1, 512, 128),
    (1, 4, 1, 64, 16), (1, 8, 1, 128, 64), (1, 1, 2, 700, 16), (1, 4, 1, 300, 16), (1, 1, 1, 700, 32), (4, 1, 5, 2200, 16), (4, 2, 5, 700, 32), (4, 8, 1, 40, 128), (4, 16, 1, 64, 128), (4, 1, 1, 2000, 128), (4, 2, 1, 1000, 128), (4, 8, 1, 2000, 128), (4, 32, 1, 200, 128),
    (4, 1, 5, 700, 128),
    (4, 8, 1, 2030, 128), (4, 1, 9, 900, 30), (4, 2, 9, 200, 128), (4, 3, 13, 200, 24), (2, 12, 2, 900, 128), (2, 30, 3, 300, 128), (2, 64, 1, 1005, 100),
    (2, 5, 11, 2050, 50), (1, 64, 1, 3650, 100), (1, 2, 66, 130, 128), (1, 1, 6, 90, 5)])
def test_tiles_side_by_side_of_the_decode_attention(L, side, b, s, t, h):
    plan = L.lib["_ZN4dsv315mla_decode_sideEllli"]              # dsv3::mla_decode_side(sequences, tokens, positions, heads)
    plan.restype, plan.argtypes = ctypes.c_int, [ctypes.c_int64] * 3 + [ctypes.c_int]
    assert plan(b, s, t, h) == side


# The sizes that the dispatcher sends to the mid-M tiles: both sides of the limits at 33 .. 64 rows, ...
WIDE_33_TO_64 = [(32, 36864, 7168, False), (33, 36864, 7168, True), (64, 36864, 7168, True), (64, 32769, 3072, True), (64, 32769, 2560, False),
                 (33, 24576, 3584, True), (33, 24576, 3072, False), (64, 24576, 10240, True), (64, 24576, 10752, False), (65, 24576, 10752, True),
                 (65, 24576, 1536, True), (64, 22400, 7168, False), (64, 22401, 7168, True), (32, 24576, 7168, False), (64, 24576, 7296, False)]
# ... at 129 .. 256 rows of slices of eight K blocks, ...
SLICES_OF_EIGHT = [(139, 15488, 1536, False), (151, 15419, 1536, False), (147, 16000, 2048, True), (159, 8064, 3584, False), (159, 8064, 4096, True),
                   (145, 10816, 2560, False), (145, 10816, 3072, True), (159, 5376, 5632, False), (159, 5376, 6144, True), (158, 4096, 8192, True),
                   (160, 6400, 5120, True)]
# ... and of the tall tiles of narrow weights: rows, columns, K; slices (none, two, more), their blocks, units, rows a tile; columns in whole fours
TALL = [(256, 2304, 8192, False), (257, 2304, 8192, True), (257, 2305, 8192, False), (449, 1536, 7168, True), (321, 2112, 7168, True), (350, 2112, 7168, True),
        (777, 1536, 7168, True), (700, 1536, 7168, True), (400, 2112, 7168, False), (930, 1536, 7168, False), (1280, 1536, 7168, False),
        (1500, 640, 7168, False), (1500, 641, 7168, True), (1500, 640, 8704, True), (398, 1408, 16384, False), (398, 920, 16384, True),
        (881, 1408, 13312, False), (881, 1407, 13312, True), (423, 2187, 13312, True), (423, 2188, 13312, False),
        (1800, 2112, 7168, True), (1600, 2112, 7168, True), (1600, 2304, 8192, False), (1800, 1536, 7168, False), (2400, 1536, 7168, True),
        (1468, 2176, 6656, False), (2886, 1024, 16384, False), (1948, 1792, 11776, False), (2907, 907, 7680, True), (1844, 1453, 4096, True)]


@pytest.mark.parametrize("m,n,k,taken", WIDE_33_TO_64 + SLICES_OF_EIGHT + TALL)
def test_sizes_that_the_dispatcher_sends_to_the_mid_m_tiles(L, m, n, k, taken):
    takes = L.lib["_ZN4dsv39mid_takesElll"]                     # dsv3::mid_takes(rows, columns, K)
    takes.restype, takes.argtypes = ctypes.c_bool, [ctypes.c_int64] * 3
    assert takes(m, n, k) == taken


@pytest.mark.parametrize("knob", ["DSV3_PREFILL_NOSPLIT=1", "DSV3_PREFILL_TILE=128", "DSV3_PREFILL_NOPP=1", "DSV3_PREFILL_NOPP128=1", "OTHER=1"])
def test_knobs_of_the_large_m_kernel_hold_in_every_window_of_the_mid_m_tiles(knob):
    """33 .. 64 rows, 65 rows and more, slices of one row tile, 64 x 128 tiles, tall tiles: as the dispatcher asks."""
    import os
    import subprocess
    import sys
    code = """
import ctypes
from dsv3fp8 import _lib
f = _lib.lib["_ZN4dsv39mid_takesElll"]
f.restype, f.argtypes = ctypes.c_bool, [ctypes.c_int64] * 3
print([f(*s) for s in [(33, 36864, 7168), (64, 24576, 7168), (65, 36864, 7168), (193, 7168, 16384), (448, 1536, 7168), (777, 1536, 7168), (1800, 2112, 7168)]])
"""
    name, value = knob.split("=")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT / "deepseek-v3_amd", capture_output=True, text=True, env={**os.environ, name: value})
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == str([name == "OTHER"] * 7)


@pytest.mark.parametrize("m,n,k,rows", [
    (1, 576, 7168, 8), (2, 1536, 7168, 8), (1, 2048, 7168, 8), (1, 2049, 7168, 16), (3, 576, 7168, 16), (1, 2048, 512, 8), (2, 2049, 512, 16), (1, 2048, 384, 8),
    (1, 128, 128, 8), (1, 2056, 128, 16), (1, 2112, 3072, 16), (2, 4096, 1024, 16), (1, 32768, 256, 16), (1, 2048, 16384, 16)])
def test_weight_rows_of_a_decode_workgroup(L, m, n, k, rows):
    f = L.lib["_ZN4dsv317skinny_strip_rowsElllPi"]              # dsv3::skinny_strip_rows(rows, columns, K, *wavefronts)
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int64] * 3 + [ctypes.POINTER(ctypes.c_int)]
    assert f(m, n, k, None) == rows
