"""The attention kernels of MLA.forward (torch.ops.dsv3fp8.mla_prefill) against a binary64 evaluation of
inference/model.py:470-497 on the same bf16 inputs, at the edges of their tiles, and MLA.forward on them against the
torch-CPU oracle."""
import pytest
import torch

from oracle import oracle
from test_gpu_mla import M  # noqa: F401  (fixture)
from test_oracle_mla import _freqs, small_mla_params

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
NOPE, ROPE, V, C = 128, 64, 128, 512


@pytest.fixture(scope="module", autouse=True)
def _ops():
    from dsv3fp8 import ops  # noqa: F401  (registers torch.ops.dsv3fp8)


def _inputs(b, s, t, h, seed):
    """Queries, rotary phases, caches (NaN behind position t: it must not be read), wkv_b and its scales, on the GPU."""
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(b, s, h, NOPE + ROPE, generator=g) * 2).bfloat16()
    kv = torch.full((b, t + 3, C), float("nan")).bfloat16()
    pe = torch.full((b, t + 3, ROPE), float("nan")).bfloat16()
    kv[:, :t] = torch.randn(b, t, C, generator=g).bfloat16()
    pe[:, :t] = torch.randn(b, t, ROPE, generator=g).bfloat16()
    ang = torch.rand(s, ROPE // 2, generator=g) * 6.28
    w8 = torch.randn(h * (NOPE + V), C, generator=g).to(FP8)
    ws = torch.rand(h * 2, C // 128, generator=g) * 0.03 + 0.01
    return [x.cuda() for x in (q, torch.polar(torch.ones_like(ang), ang), kv, pe, w8, ws)]


def _mask(kind, s, t, seed):
    if kind is None:
        return None
    if kind.startswith("causal"):
        m = torch.full((s, t), float("-inf")).triu_(1 + t - s)
        return m.cuda() if kind == "causal_f32" else m.bfloat16().cuda()
    if kind.startswith("lowest"):                       # the type's lowest value for -inf; row 1 has nothing else
        dtype = torch.float32 if kind == "lowest_f32" else torch.bfloat16
        m = torch.full((s, t), torch.finfo(dtype).min).triu_(1 + t - s)
        m[1] = torch.finfo(dtype).min
        return m.to(dtype).cuda()
    if kind.startswith("ranked"):                       # values near either end of the type's range still have an order
        m = torch.zeros(s, t)
        m[0, : t // 2], m[0, t // 2:] = -3e38, -1e38    # the second half gets everything
        m[1, ::3], m[1, 1::3], m[1, 2::3] = -2e38, -3e38, -2.5e38
        m[2, 5], m[2, t - 1] = 3e38, 3e38               # these two get everything
        m[3, : t // 2] = -3e38
        return m.to(torch.float32 if kind == "ranked_f32" else torch.bfloat16).cuda()
    g = torch.Generator().manual_seed(seed)             # finite values and holes; row 1 sees nothing
    m = torch.where(torch.rand(s, t, generator=g) < 0.3, float("-inf"), torch.randn(s, t, generator=g))
    m[1] = float("-inf")
    return m.bfloat16().cuda()


def _reference(q, freqs, kv, pe, w8, ws, mask, t, scale):
    """Binary64, with the roundings to bf16 that the kernel has in its inputs: weights, keys, values, rotated query."""
    b, s, h, _ = q.shape
    w = (w8.float() * ws.repeat_interleave(128, 0).repeat_interleave(128, 1)).bfloat16().double().view(h, NOPE + V, C)
    pairs = q[..., NOPE:].float().unflatten(-1, (-1, 2))
    re, im = pairs[..., 0], pairs[..., 1]
    cos, sin = freqs.real.view(1, s, 1, -1), freqs.imag.view(1, s, 1, -1)
    qr = torch.stack((re * cos - im * sin, re * sin + im * cos), -1).flatten(-2).bfloat16().double()
    kv, pe = kv[:, :t].double(), pe[:, :t].double()
    out = torch.empty(b, s, h, V, dtype=torch.float64, device=q.device)
    for i in range(h):
        k, v = (kv @ w[i, :NOPE].t()).bfloat16().double(), (kv @ w[i, NOPE:].t()).bfloat16().double()
        sc = q[:, :, i, :NOPE].double() @ k.transpose(1, 2).contiguous() + qr[:, :, i] @ pe.transpose(1, 2).contiguous()
        sc = sc * scale
        if mask is not None:                             # added in binary32, as the layer's tensor operations do
            sc = (sc.float() + mask.float()).double()
        out[:, :, i] = sc.softmax(-1) @ v
    return out


# one tile and its neighbours in positions (64), wavefronts (32 rows) and workgroups (256 rows); head counts that leave
# XCDs unequally loaded; more positions than rows (a cached prefix)
PREFILL = [(1, 32, 32, 1, "causal"), (1, 33, 63, 3, None), (2, 64, 64, 8, "causal"), (1, 65, 65, 9, "causal"),
           (1, 255, 255, 2, "causal_f32"), (2, 257, 257, 3, "causal"), (1, 40, 500, 4, "causal"), (1, 1, 1, 2, None),
           (2, 100, 163, 4, "holes"), (1, 1100, 1100, 2, "causal"),
           (1, 70, 130, 2, "lowest"), (1, 70, 130, 2, "lowest_f32"), (1, 70, 130, 2, "ranked"), (1, 40, 300, 2, "ranked_f32"), (1, 256, 320, 2, "causal_f32"),
           (1, 600, 600, 128, "causal"), (1, 4200, 4200, 16, "causal")]     # two query tiles a workgroup; 66 tiles of flags


# tiles of 32 positions, workgroups of 128 (token, head) rows, wavefronts of 32; one split and many, uneven last ones, more
# units than compute units
DECODE = [(1, 1, 1, 1, None), (1, 1, 31, 128, None), (2, 1, 33, 128, None), (1, 1, 700, 128, None), (3, 1, 1000, 16, None),
          (70, 1, 97, 128, None), (5, 4, 257, 40, "causal"), (1, 31, 95, 16, "causal_f32"), (2, 3, 200, 9, "holes"),
          (2, 100, 700, 20, "causal"), (1, 40, 500, 128, "causal_f32"),         # many row blocks a sequence
          (1, 5, 130, 2, "lowest"), (1, 5, 130, 2, "lowest_f32"), (1, 5, 130, 2, "ranked"), (2, 4, 300, 2, "ranked_f32"), (1, 1, 9000, 3, None)]


def _decode_reference(q, freqs, kv, pe, w8, ws, mask, t, scale):
    """Binary64 with the absorbed form's roundings to bf16: weights, rotated and folded query, latent sum."""
    b, s, h, _ = q.shape
    w = (w8.float() * ws.repeat_interleave(128, 0).repeat_interleave(128, 1)).bfloat16().double().view(h, NOPE + V, C)
    pairs = q[..., NOPE:].float().unflatten(-1, (-1, 2))
    re, im = pairs[..., 0], pairs[..., 1]
    cos, sin = freqs.real.view(1, s, 1, -1), freqs.imag.view(1, s, 1, -1)
    qr = torch.stack((re * cos - im * sin, re * sin + im * cos), -1).flatten(-2).bfloat16().double()
    kv, pe = kv[:, :t].double(), pe[:, :t].double()
    out = torch.empty(b, s, h, V, dtype=torch.float64, device=q.device)
    for i in range(h):
        ql = (q[:, :, i, :NOPE].double() @ w[i, :NOPE]).bfloat16().double()
        sc = (ql @ kv.transpose(1, 2).contiguous() + qr[:, :, i] @ pe.transpose(1, 2).contiguous()) * scale
        if mask is not None:
            sc = (sc.float() + mask.float()).double()
        out[:, :, i] = (sc.softmax(-1) @ kv).bfloat16().double() @ w[i, NOPE:].t()
    return out


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("b,s,t,h,kind", DECODE)
def test_decode_attention(b, s, t, h, kind, grow):
    q, freqs, kv, pe, w8, ws = _inputs(b, s, t, h, s + t)
    if grow:                    # scores that grow along the positions by far more than 2^64: the running maximum is raised
        if kind is not None:
            pytest.skip("one run per shape without a mask")
        pe[:, :t] *= torch.linspace(0.01, 400, t, device="cuda").bfloat16().view(1, t, 1)
    mask = _mask(kind, s, t, 5)
    scale = 0.08
    got = torch.ops.dsv3fp8.mla_decode(q, freqs, kv, pe, w8, ws, mask, t, scale).view(b, s, h, V).double()
    ref = _decode_reference(q, freqs, kv, pe, w8, ws, mask, t, scale)
    if kind == "holes":
        assert torch.isnan(got[:, 1]).all() and torch.isnan(ref[:, 1]).all()
        keep = torch.arange(s, device="cuda") != 1
        got, ref = got[:, keep], ref[:, keep]
    # the latent sum and the result round to bf16 (2^-9 each), the exponentials too; in the value product of 512 terms these
    # errors average out against a result of the same size: 2^-7 of the row's norm
    assert ((got - ref).norm(dim=-1) <= 2.0 ** -7 * ref.norm(dim=-1)).all()


# Tiles side by side in a workgroup (the cost rule of csrc/mla_decode.hip): four, two and one, with a wavefront's second and later tiles, ranges
# whose last step has fewer tiles than wavefronts, tiles past the end and the range, row blocks with missing rows.
SIDES = [(8, 1, 2030, 128, None), (1, 9, 900, 30, "causal_f32"), (2, 9, 200, 128, "causal"), (3, 13, 200, 24, "holes"),         # four
         (12, 2, 900, 128, "holes"), (30, 3, 300, 128, "causal"), (64, 1, 1005, 100, None), (5, 11, 2050, 50, "lowest_f32"),    # two
         (64, 1, 3650, 100, None), (2, 66, 130, 128, "causal_f32"), (1, 6, 90, 5, "lowest")]                                    # one


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("b,s,t,h,kind", SIDES)
def test_decode_attention_tiles_side_by_side(b, s, t, h, kind, grow):
    test_decode_attention(b, s, t, h, kind, grow)


# A workgroup of the fold takes a head and 4, 8 or 16 tokens at a time: 16 heads and fewer 4 here, 128 heads 4 up to 8 tokens in all, 8 up to 16,
# then 16, and past 128 tokens (1024 / heads groups) several groups, one after another.  One token of a group is shared by eight
# wavefronts, two by four each, three or four by two each, more have one each.  Splits below, at and above a wavefront's 64 lanes (256
# workgroups over the row blocks, 32 positions a tile).
FOLD = [(1, 1, 33, 128, None), (1, 1, 2080, 128, None), (1, 1, 8192, 8, None), (2, 1, 700, 128, None), (3, 1, 5000, 16, None),
        (4, 1, 90, 128, None), (1, 5, 300, 128, None), (8, 1, 1, 128, None), (16, 1, 257, 128, None), (17, 1, 64, 32, None), (3, 13, 200, 24, None),
        (32, 1, 100, 128, None), (37, 1, 70, 128, None),            # groups of 16, the last one of 5
        (131, 1, 40, 128, None),                                    # nine groups over eight workgroups a head: 16 tokens, then 3
        (8, 32, 64, 128, "causal"), (2, 66, 130, 128, "causal_f32"), (2, 9, 200, 128, "holes"), (1, 6, 90, 5, "lowest")]


@pytest.mark.parametrize("b,s,t,h,kind", FOLD)
def test_decode_attention_quantised_is_the_rounded_result_quantised(b, s, t, h, kind):
    from dsv3fp8 import kernel
    q, freqs, kv, pe, w8, ws = _inputs(b, s, t, h, s + t)
    args = (q, freqs, kv, pe, w8, ws, _mask(kind, s, t, 5), t, 0.08)
    y = torch.ops.dsv3fp8.mla_decode(*args)
    ref = _decode_reference(*args)
    got = y.view(b, s, h, V).double()
    nan = torch.isnan(ref).any(-1)                       # (a row that sees nothing)
    assert torch.equal(nan, torch.isnan(got).any(-1)) and nan.any() == (kind == "holes")
    assert ((got - ref).norm(dim=-1) <= 2.0 ** -7 * ref.norm(dim=-1))[~nan].all()   # as in test_decode_attention
    yq, ys = torch.ops.dsv3fp8.mla_decode_quant(*args)
    rq, rs = kernel.act_quant(y)
    assert torch.equal(yq.view(torch.uint8), rq.view(torch.uint8)) and torch.equal(ys.view(torch.int32), rs.view(torch.int32))


@pytest.mark.parametrize("explicit", [False, True])
@pytest.mark.parametrize("b,s,t,h,kind", [(1, 1, 40, 4, None), (3, 1, 500, 128, None), (2, 40, 130, 8, "causal"), (1, 33, 33, 128, "causal_f32"), (2, 36, 70, 4, "holes")])
def test_output_in_one_call_is_its_two_parts(b, s, t, h, kind, explicit):
    """mla_output: the attention in either form, quantised, and the product with wo, bit for bit."""
    from dsv3fp8 import quantize
    args = (*_inputs(b, s, t, h, s + t), _mask(kind, s, t, 5), t, 0.08)
    wo, wo_s = quantize.weight_quant((torch.randn(384, h * V, generator=torch.Generator().manual_seed(h)) * 0.02).bfloat16().cuda())
    y = torch.ops.dsv3fp8.mla_output(*args, explicit, wo, wo_s)
    attention = torch.ops.dsv3fp8.mla_prefill if explicit else torch.ops.dsv3fp8.mla_decode_quant
    ref = torch.ops.dsv3fp8.fp8_gemm(*attention(*args), wo, wo_s, 0)
    assert y.shape == (b, s, 384) and y.dtype == torch.bfloat16
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16)) and torch.isfinite(y[:, 0]).all()


# rows whose projection runs as one launch, in K slices of the streaming kernel, in slices of the tile kernel (up to eight), plain
@pytest.mark.parametrize("b,s", [(1, 1), (3, 1), (17, 1), (1, 64), (5, 13), (1, 200), (2, 400), (1, 3000)])
def test_query_in_one_call_is_its_three_parts(b, s):
    from dsv3fp8 import kernel, quantize
    dim, qr, h, start = 7168, 1536, 2, 3
    g = torch.Generator().manual_seed(b * 1000 + s)
    x = torch.randn(b, s, dim, generator=g).bfloat16().cuda()
    wa, wa_s = quantize.weight_quant((torch.randn(qr + C + ROPE, dim, generator=g) * 0.02).bfloat16().cuda())
    wq, wq_s = quantize.weight_quant((torch.randn(h * 192, qr, generator=g) * 0.02).bfloat16().cuda())
    qn, kn = [(1 + 0.1 * torch.randn(n, generator=g)).bfloat16().cuda() for n in (qr, C)]
    ang = torch.rand(s, ROPE // 2, generator=g) * 6.28
    freqs = torch.polar(torch.ones_like(ang), ang).cuda()
    one, three = [[torch.zeros(b, start + s + 2, n, dtype=torch.bfloat16, device="cuda") for n in (C, ROPE)] for _ in range(2)]
    q = torch.ops.dsv3fp8.mla_query(x, wa, wa_s, qn, kn, freqs, *one, start, 1e-6, 1e-6, wq, wq_s, h)
    a = torch.ops.dsv3fp8.linear_fp8(x, wa, wa_s, 0, 0)
    y, ys = torch.ops.dsv3fp8.mla_latent(a, qn, kn, freqs, *three, start, 1e-6, 1e-6)
    assert torch.equal(q, torch.ops.dsv3fp8.fp8_gemm(y, ys, wq, wq_s, 0).view(b, s, h, 192))
    assert torch.equal(one[0], three[0]) and torch.equal(one[1], three[1]) and one[0][:, start:start + s].any()


@pytest.mark.parametrize("b,s,slabs", [(1, 321, 5), (1, 350, 5), (2, 320, 3), (1, 384, 5)])
def test_query_in_one_call_adds_the_slabs_of_the_tall_tiles(b, s, slabs):
    import ctypes
    from dsv3fp8 import _lib
    assert _lib.lib.dsv3_fp8_gemm_workspace_bytes(b * s, 2112, 7168) >= slabs * b * s * 2112 * 4
    takes = _lib.lib["_ZN4dsv39mid_takesElll"]                  # dsv3::mid_takes(rows, columns, K)
    takes.restype, takes.argtypes = ctypes.c_bool, [ctypes.c_int64] * 3
    assert takes(b * s, 2112, 7168)
    test_query_in_one_call_is_its_three_parts(b, s)


LATENT = [(1, 1, 0, 1536), (3, 1, 7, 1536), (2, 5, 0, 128), (1, 40, 3, 2048), (2, 33, 1, 640)]


@pytest.mark.parametrize("b,s,start,q_rank", LATENT)
def test_latent_rows(b, s, start, q_rank):
    from dsv3fp8 import kernel
    import torch.nn.functional as F
    from dsv3fp8.model import apply_rotary_emb
    g = torch.Generator().manual_seed(q_rank + s)
    a = (torch.randn(b, s, q_rank + C + ROPE, generator=g) * 3).bfloat16().cuda()
    a[0, 0, :q_rank] = 0
    qw, kw = [(1 + 0.1 * torch.randn(n, generator=g)).bfloat16().cuda() for n in (q_rank, C)]
    ang = torch.rand(s, ROPE // 2, generator=g) * 6.28
    freqs = torch.polar(torch.ones_like(ang), ang).cuda()
    kv, pe = (torch.full((b + 1, start + s + 2, n), 7.0, dtype=torch.bfloat16, device="cuda") for n in (C, ROPE))
    y, ys = torch.ops.dsv3fp8.mla_latent(a, qw, kw, freqs, kv, pe, start, 1e-6, 1e-6)
    ref = F.rms_norm(a[..., :q_rank].double(), (q_rank,), qw.double(), 1e-6)
    got = y.double() * ys.double().repeat_interleave(128, -1)
    # one rounding to bf16 and one to e4m3 (2^-4 of the value, or half the smallest step of the block)
    amax = ys.double().repeat_interleave(128, -1) * 448
    assert ((got - ref).abs() <= ref.abs() * (2.0 ** -4 + 2.0 ** -8) + amax / 448 * 2.0 ** -10).all()
    q8, s8 = kernel.act_quant(ref.bfloat16().contiguous(), 128)
    assert (q8.view(torch.uint8) != y.view(torch.uint8)).double().mean() <= 2e-3     # ties of the bf16 rounding only
    lat = F.rms_norm(a[..., q_rank:q_rank + C].double(), (C,), kw.double(), 1e-6)
    assert ((kv[:b, start:start + s].double() - lat).abs() <= lat.abs() * 2.0 ** -8).all()
    assert torch.equal(pe[:b, start:start + s], apply_rotary_emb(a[..., q_rank + C:].unsqueeze(2), freqs).squeeze(2))
    for t in (kv, pe):                                                               # nothing else is written
        t[:b, start:start + s] = 7.0
        assert (t == 7.0).all()


@pytest.mark.parametrize("b,s,t,h,kind", PREFILL)
def test_prefill_attention(b, s, t, h, kind):
    q, freqs, kv, pe, w8, ws = _inputs(b, s, t, h, s + t)
    mask = _mask(kind, s, t, 5)
    scale = 0.08
    y, ys = torch.ops.dsv3fp8.mla_prefill(q, freqs, kv, pe, w8, ws, mask, t, scale)
    got = y.float().view(b, s, h, V).double() * ys.double().unsqueeze(-1)
    ref = _reference(q, freqs, kv, pe, w8, ws, mask, t, scale)
    if kind == "holes":                                  # softmax over nothing is NaN, in this row only
        assert torch.isnan(ys[:, 1]).all() and torch.isnan(ref[:, 1]).all()
        keep = torch.arange(s, device="cuda") != 1
        got, ref, ys = got[:, keep], ref[:, keep], ys[:, keep]
    amax = ref.abs().amax(-1)
    # e4m3 codes: half a step at the top of the range, 16 of 448; in front of them exponentials and result are rounded to
    # bf16, 2^-9 each of values whose errors average out: 2^-7 of the block's largest value holds them
    assert ((got - ref).abs() <= amax.unsqueeze(-1) * (16 / 448 + 2.0 ** -7)).all()
    assert ((ys.double() * 448 - amax).abs() <= 2.0 ** -7 * amax).all()


@pytest.mark.parametrize("b,s,t,h,kind,offset", [(4, 129, 200, 128, "holes", 0), (1, 127, 200, 3, "holes", 1), (4, 130, 202, 128, "causal_f32", 0),
                                                 (1, 128, 128, 5, "causal_f32", 1), (1, 200, 204, 128, "ranked", 0), (2, 385, 388, 4, "ranked_f32", 0)])
def test_prefill_attention_query_tiles_of_128(b, s, t, h, kind, offset):
    """One and two query tiles a workgroup, a second half of the flags' word that has no rows; masks that are read four
    values at a time (whole 4s of positions, aligned) and one by one."""
    q, freqs, kv, pe, w8, ws = _inputs(b, s, t, h, 17 * s + t)
    mask = _mask(kind, s, t, 5)
    if offset:
        mask = torch.cat((mask.new_zeros(offset), mask.flatten()))[offset:].view(s, t)
    y, ys = torch.ops.dsv3fp8.mla_prefill(q, freqs, kv, pe, w8, ws, mask, t, 0.08)
    got = y.float().view(b, s, h, V).double() * ys.double().unsqueeze(-1)
    ref = _reference(q, freqs, kv, pe, w8, ws, mask, t, 0.08)
    keep = torch.arange(s, device="cuda") != (1 if kind == "holes" else -1)             # (row 1 of "holes" is NaN)
    got, ref, ys = got[:, keep], ref[:, keep], ys[:, keep]
    # Exponentials are rounded by up to 2^-9, keys' and values' sums land on the other side of a tie (2^-8) at most, the result is rounded
    # by 2^-9: off by (3 A + amax) 2^-9 with A = sum of p |v|.  With these inputs (scores of standard deviation 1.3, some 30
    # positions that count) A is below 4 amax, 13 / 512 in all; e4m3 codes half a step more.
    amax = ref.abs().amax(-1)
    assert ((got - ref).abs() <= amax.unsqueeze(-1) * (16 / 448 + 13 / 512)).all()
    assert ((ys.double() * 448 - amax).abs() <= 13 / 512 * amax).all()


# Two query tiles of 128 rows a workgroup (512 workgroups of a pair and more): the j-th last and the j-th first, j of 0 .. 4, whose flags are other
# words and other windows of 64 position tiles; a middle tile by itself, a last tile of few rows, cached prefixes, two sequences.
PAIRED = [(1, 800, 800, 128, "causal"), (1, 770, 770, 128, "causal_f32"), (1, 800, 4200, 128, "causal"), (2, 513, 640, 128, "holes"),
          (1, 1030, 1030, 128, None), (1, 900, 903, 128, "causal")]


@pytest.mark.parametrize("b,s,t,h,kind", PAIRED)
def test_prefill_attention_two_query_tiles_a_workgroup(b, s, t, h, kind):
    import ctypes
    from dsv3fp8 import _lib
    paired = _lib.lib["_ZN4dsv318mla_prefill_pairedElli"]       # dsv3::mla_prefill_paired(sequences, rows, heads)
    paired.restype, paired.argtypes = ctypes.c_bool, [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    assert paired(b, s, h) and not paired(1, 600, 128) and not paired(1, 4200, 16)
    # (bound: that of test_prefill_attention_query_tiles_of_128, which holds for rows of few positions; in rows of many the errors average out)
    test_prefill_attention_query_tiles_of_128(b, s, t, h, kind, 0)


def _layer(M, p, dim, heads, q_rank, max_seq):
    args = M.ModelArgs(dim=dim, n_heads=heads, q_lora_rank=q_rank, kv_lora_rank=C, qk_nope_head_dim=NOPE,
                       qk_rope_head_dim=ROPE, v_head_dim=V, max_batch_size=2, max_seq_len=max_seq, original_seq_len=max_seq)
    with torch.device("cuda"):
        layer = M.MLA(args)
    with torch.no_grad():
        for name in ("wq_a", "wq_b", "wkv_a", "wkv_b", "wo"):
            getattr(layer, name).weight.copy_(p[name][0].cuda())
            getattr(layer, name).scale.copy_(p[name][1].cuda())
        layer.q_norm.weight.copy_(p["q_norm"].cuda())
        layer.kv_norm.weight.copy_(p["kv_norm"].cuda())
    return layer


def _rel(got, ref):
    return ((got.float().cpu() - ref.float()).norm() / ref.float().norm()).item()


# Two evaluations differ by roundings in front of quantisers; where such a rounding moves an e4m3 code of wo's input the
# result moves by one step.  Codes carry an error of 2.6 % (rms of the rounding); were every one of them chosen anew the
# two results would be sqrt(2) * 2.6 % = 3.7 % apart.
LAYER_TOL = 4e-2


def test_layer_prefill_vs_oracle(M):
    dim, heads, q_rank, s = 256, 4, 128, 70
    p = small_mla_params(dim, heads, q_rank, C, NOPE, ROPE, V, 31)
    layer = _layer(M, p, dim, heads, q_rank, 96)
    assert s >= layer.explicit_min_tokens
    freqs = _freqs(ROPE, 96)
    g = torch.Generator().manual_seed(32)
    x0, x1 = torch.randn(2, s, dim, generator=g).bfloat16(), torch.randn(2, 1, dim, generator=g).bfloat16()
    mask = torch.full((s, s), float("-inf")).triu_(1)
    kv, pe = torch.zeros(2, 96, C, dtype=torch.bfloat16), torch.zeros(2, 96, ROPE, dtype=torch.bfloat16)
    scale = (NOPE + ROPE) ** -0.5
    ref0 = oracle.mla(x0, 0, freqs[:s], mask, p, kv, pe, heads, NOPE, ROPE, V, C, scale)
    ref1 = oracle.mla(x1, s, freqs[s:s + 1], None, p, kv, pe, heads, NOPE, ROPE, V, C, scale)
    with torch.inference_mode():
        y0 = layer(x0.cuda(), 0, freqs[:s].cuda(), mask.cuda())
        y1 = layer(x1.cuda(), s, freqs[s:s + 1].cuda(), None)
    assert _rel(y0, ref0) <= LAYER_TOL and _rel(y1, ref1) <= LAYER_TOL
    assert _rel(layer.kv_cache, kv) <= 1e-2 and _rel(layer.pe_cache, pe) <= 1e-2
    # with gradients enabled the layer keeps to differentiable-by-parts tensor operations: same result, other kernels
    layer.kv_cache.zero_(); layer.pe_cache.zero_()
    layer.requires_grad_(False)
    z0 = layer(x0.cuda(), 0, freqs[:s].cuda(), mask.cuda())
    assert _rel(z0, ref0) <= LAYER_TOL and _rel(y0, z0.cpu()) <= LAYER_TOL


@pytest.mark.parametrize("s", [1, 40])
def test_step_in_a_captured_graph(M, s):
    """A captured step, replayed on new inputs with eager steps in between, gives the eager step's bits, in its result and
    in the cache rows, which hold something else before each replay."""
    dim, heads, q_rank, t = 256, 4, 128, 40
    layer = _layer(M, small_mla_params(dim, heads, q_rank, C, NOPE, ROPE, V, 31), dim, heads, q_rank, 96)
    freqs = _freqs(ROPE, 96)[t:t + s].cuda()
    mask = torch.full((s, t + s), float("-inf"), device="cuda").triu_(1 + t) if s > 1 else None
    g = torch.Generator().manual_seed(33)
    with torch.inference_mode():
        layer.kv_cache.copy_(torch.randn(layer.kv_cache.shape, generator=g))
        layer.pe_cache.copy_(torch.randn(layer.pe_cache.shape, generator=g))
        x = torch.randn(2, s, dim, generator=g).bfloat16().cuda()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x, t, freqs, mask)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer(x, t, freqs, mask)
        for n in range(3):
            new = torch.randn(2, s, dim, generator=g).bfloat16().cuda()
            ref, kv, pe = [o.clone() for o in (layer(new, t, freqs, mask), layer.kv_cache, layer.pe_cache)]
            layer.kv_cache[:, t:t + s] = n
            layer.pe_cache[:, t:t + s] = n
            torch.cuda.synchronize()
            x.copy_(new)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, ref) and torch.equal(layer.kv_cache, kv) and torch.equal(layer.pe_cache, pe)


@pytest.mark.parametrize("s", [1, 40])
def test_two_streams_at_once(M, s):
    """Layers on two streams, several steps without a wait between them: each stream's results are those of a single one."""
    dim, heads, q_rank = 256, 4, 128
    freqs = _freqs(ROPE, 96)[:s].cuda()
    mask = torch.full((s, s), float("-inf"), device="cuda").triu_(1) if s > 1 else None
    layers = [_layer(M, small_mla_params(dim, heads, q_rank, C, NOPE, ROPE, V, n), dim, heads, q_rank, 96) for n in (31, 32)]
    g = torch.Generator().manual_seed(36)
    xs = [torch.randn(2, s, dim, generator=g).bfloat16().cuda() for _ in range(12)]
    with torch.inference_mode():
        ref = [[layer(x, 0, freqs, mask).clone() for x in xs] for layer in layers]
        torch.cuda.synchronize()
        streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], [[], []]
        for x in xs:
            for n, stream in enumerate(streams):
                with torch.cuda.stream(stream):
                    got[n].append(layers[n](x, 0, freqs, mask))
        torch.cuda.synchronize()
    assert all(torch.equal(a, b) for n in (0, 1) for a, b in zip(got[n], ref[n]))


@pytest.mark.parametrize("op", ["prefill", "decode"])
def test_not_finite_inputs(op):
    """NaN and infinity in a query, a mask or a cached row make NaN of the rows that the reference makes NaN of."""
    b, s, t, h, scale = 2, 40, 130, 3, 0.08
    q, freqs, kv, pe, w8, ws = _inputs(b, s, t, h, 7)
    mask = torch.zeros(s, t, device="cuda")
    q[0, 1, 0, 5], q[0, 2, 1, 140], q[0, 3, 2, 60] = float("nan"), float("inf"), float("-inf")
    mask[5, 7], mask[6, 100] = float("nan"), float("inf")
    mask[7, 20:] = float("-inf")
    kv[1, 90, 3] = float("inf")                         # every row of the second sequence
    args = (q, freqs, kv, pe, w8, ws, mask, t, scale)
    if op == "prefill":
        y, ys = torch.ops.dsv3fp8.mla_prefill(*args)
        got, ref = y.float().view(b, s, h, V).double() * ys.double().unsqueeze(-1), _reference(*args)
    else:
        got, ref = torch.ops.dsv3fp8.mla_decode(*args).view(b, s, h, V).double(), _decode_reference(*args)
    bad = torch.isnan(ref).any(-1)
    expected = torch.zeros(b, s, h, dtype=torch.bool, device="cuda")
    expected[1] = True
    expected[0, 1, 0] = expected[0, 2, 1] = expected[0, 3, 2] = True
    expected[0, 5:7] = True
    assert torch.equal(bad, expected) and torch.equal(torch.isnan(got).any(-1), bad)
    assert ((got - ref).norm(dim=-1) <= 2.0 ** -4 * ref.norm(dim=-1))[~bad].all()       # e4m3 in the prefill's result


@pytest.mark.parametrize("op", ["prefill", "decode"])
def test_caches_of_more_sequences_than_the_call(op):
    b, s, t, h, scale = 2, 33, 70, 2, 0.08
    q, freqs, kv, pe, w8, ws = _inputs(b, s, t, h, 9)
    kv5, pe5 = (torch.full((5, t + 30, c.size(2)), float("nan"), dtype=torch.bfloat16, device="cuda") for c in (kv, pe))
    kv5[:b, :t], pe5[:b, :t] = kv[:, :t], pe[:, :t]
    call = getattr(torch.ops.dsv3fp8, "mla_" + op)
    one, other = call(q, freqs, kv, pe, w8, ws, None, t, scale), call(q, freqs, kv5, pe5, w8, ws, None, t, scale)
    for a, c in zip(one, other) if op == "prefill" else ((one, other),):
        assert torch.equal(a.view(torch.uint8), c.view(torch.uint8)) and torch.isfinite(c.float()).all()


def test_layer_with_parts_on_the_host_raises(M):
    """A cache, a norm weight or the mask that stayed on the host is refused by the tensor operations; no kernel sees it."""
    p = small_mla_params(256, 4, 128, C, NOPE, ROPE, V, 31)
    freqs, x = _freqs(ROPE, 96)[:40].cuda(), torch.ones(2, 40, 256, dtype=torch.bfloat16, device="cuda")
    mask = torch.full((40, 40), float("-inf")).triu_(1)
    for part in ("kv_cache", "pe_cache", "q_norm", "mask"):
        layer = _layer(M, p, 256, 4, 128, 96)
        if part == "q_norm":
            layer.q_norm.cpu()
        elif part != "mask":
            setattr(layer, part, getattr(layer, part).cpu())
        with torch.inference_mode(), pytest.raises(RuntimeError, match="device"):
            layer(x, 0, freqs, mask if part == "mask" else mask.cuda())


class _Wrapped(torch.nn.Module):
    """A module put in a layer's place, with none of its attributes (an adapter, say)."""

    def __init__(self, base):
        super().__init__()
        self.base, self.calls = [base], 0

    def forward(self, x):
        self.calls += 1
        return self.base[0](x)


@pytest.mark.parametrize("s", [1, 40])
def test_exchanged_modules_and_hooks_are_called(M, s):
    p = small_mla_params(256, 4, 128, C, NOPE, ROPE, V, 31)
    freqs = _freqs(ROPE, 96)[:s].cuda()
    x = torch.randn(2, s, 256, generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    mask = torch.full((s, s), float("-inf"), device="cuda").triu_(1)
    with torch.inference_mode():
        ref = _layer(M, p, 256, 4, 128, 96)(x, 0, freqs, mask)
        for name in ("wq_a", "q_norm", "wq_b", "wkv_a", "kv_norm", "wo"):
            for how in ("module", "hook", "forward"):
                layer, seen = _layer(M, p, 256, 4, 128, 96), []
                module = getattr(layer, name)
                if how == "module":
                    setattr(layer, name, _Wrapped(module))
                elif how == "hook":
                    module.register_forward_hook(lambda *a: seen.append(1))
                else:
                    module.forward = lambda x, f=module.forward: (seen.append(1), f(x))[1]
                assert _rel(layer(x, 0, freqs, mask), ref.cpu()) <= LAYER_TOL
                assert (getattr(layer, name).calls if how == "module" else len(seen)) == 1, (name, how)
        seen = []
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: seen.append(type(m).__name__))
        try:
            _layer(M, p, 256, 4, 128, 96)(x, 0, freqs, mask)
        finally:
            handle.remove()
        assert sorted(seen) == ["ColumnParallelLinear", "Linear", "Linear", "MLA", "RMSNorm", "RMSNorm", "RowParallelLinear"]


@pytest.mark.parametrize("what", ["scale", "eps", "strided"])
def test_settings_that_the_kernels_do_not_take_still_run(M, what):
    """A softmax scale below zero, a norm without an eps or with a strided weight: the layer's tensor operations."""
    p = small_mla_params(256, 4, 128, C, NOPE, ROPE, V, 31)
    freqs = _freqs(ROPE, 96)[:5].cuda()
    x = torch.randn(2, 5, 256, generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    layer = _layer(M, p, 256, 4, 128, 96).requires_grad_(False)
    if what == "scale":
        layer.softmax_scale = -layer.softmax_scale
    elif what == "eps":
        layer.q_norm.eps = layer.kv_norm.eps = None
    else:
        layer.kv_norm.weight = torch.nn.Parameter(layer.kv_norm.weight.data.repeat_interleave(2)[::2], requires_grad=False)
    with torch.inference_mode():
        y = layer(x, 0, freqs, None)
    assert torch.isfinite(y).all() and _rel(y, layer(x, 0, freqs, None).cpu()) <= LAYER_TOL    # with gradients: no kernels


@pytest.mark.parametrize("s,start,form", [(5, 30, "decode"), (40, 30, "prefill"), (40, 30, "decode"), (1, 0, "decode")])
def test_layer_on_a_filled_cache_vs_oracle(M, s, start, form):
    """Several new tokens behind a cached prefix, mask [s, start + s], on either side of the forms' line."""
    dim, heads, q_rank = 256, 4, 128
    p = small_mla_params(dim, heads, q_rank, C, NOPE, ROPE, V, 31)
    layer = _layer(M, p, dim, heads, q_rank, 96)
    if s >= 32:
        assert layer._explicit_pays(2, s, start + s)
    if form == "decode":
        layer.explicit_min_tokens = 1000
    freqs = _freqs(ROPE, 96)[start:start + s]
    g = torch.Generator().manual_seed(35)
    x = torch.randn(2, s, dim, generator=g).bfloat16()
    kv, pe = torch.zeros(2, 96, C, dtype=torch.bfloat16), torch.zeros(2, 96, ROPE, dtype=torch.bfloat16)
    kv[:, :start], pe[:, :start] = torch.randn(2, start, C, generator=g), torch.randn(2, start, ROPE, generator=g)
    layer.kv_cache.copy_(kv); layer.pe_cache.copy_(pe)
    mask = torch.full((s, start + s), float("-inf")).triu_(1 + start) if s > 1 else None
    ref = oracle.mla(x, start, freqs, mask, p, kv, pe, heads, NOPE, ROPE, V, C, (NOPE + ROPE) ** -0.5)
    with torch.inference_mode():
        y = layer(x.cuda(), start, freqs.cuda(), mask.cuda() if s > 1 else None)
    assert _rel(y, ref) <= LAYER_TOL
    assert _rel(layer.kv_cache, kv) <= 1e-2 and _rel(layer.pe_cache, pe) <= 1e-2
    assert torch.equal(layer.kv_cache[:, :start].cpu(), kv[:, :start]) and not layer.kv_cache[:, start + s:].any()
