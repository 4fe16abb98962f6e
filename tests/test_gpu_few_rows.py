"""A few query rows over a long history (csrc/sage_attn_few.hip) against the same formula in 64 bits on the INT8 operands of the
public quantiser: rows per KV head around the 16-row tile and at the limit, keys around the 128-key tile and the range split,
every K block size (a maximum per 16 keys, per wavefront, across two and four of them), both layouts, with and without K
smoothing and LSE; and the first row count past the limit, which the tiled kernel takes."""
import math

import pytest
import torch

import baselinebenchmark_amd as sa
from baselinebenchmark_amd import _cabi
from tests.helpers import sageattn_cabi

pytestmark = pytest.mark.gpu


def _reference(q, k, v, layout, BLKQ, BLKK, smooth):
    km = sa.k_mean(k, layout) if smooth else None
    q8, qs, k8, ks = (t.cpu().double() for t in sa.per_block_int8(q, k, km=km, BLKQ=BLKQ, BLKK=BLKK, tensor_layout=layout))
    q, v = q.cpu().double(), v.cpu().half().double()
    if layout == "NHD":
        q8, k8, q, v = (t.transpose(1, 2) for t in (q8, k8, q, v))
    rep = q8.shape[1] // k8.shape[1]
    rows = lambda s, blk, n: s.repeat_interleave(blk, -1)[..., :n, None]  # noqa: E731
    s2 = (q8 * rows(qs, BLKQ, q8.shape[2])) @ (k8 * rows(ks, BLKK, k8.shape[2])).repeat_interleave(rep, 1).transpose(-1, -2)
    out = torch.softmax(s2 * math.log(2.0), -1) @ v.repeat_interleave(rep, 1)
    lse = torch.logsumexp(s2 * math.log(2.0), -1)
    if smooth:
        lse = lse + (q * km.cpu().double().reshape(q.shape[0], -1, 1, q.shape[-1]).repeat_interleave(rep, 1)).sum(-1) * q.shape[-1] ** -0.5
    return (out.transpose(1, 2) if layout == "NHD" else out), lse


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,BLKQ,BLKK,layout,smooth", [
    (1, 1, 1, 1, 1025, 128, 64, "HND", True),      # one row, one key past a tile
    (3, 8, 2, 4, 1152, 128, 128, "NHD", True),     # 16 rows: one whole tile; whole 128-key tiles
    (2, 17, 1, 1, 2111, 64, 32, "HND", True),      # 17 rows: the second tile holds one
    (1, 8, 4, 16, 1537, 16, 16, "NHD", False),     # 32 rows, the limit; 16-row and 16-key blocks, no smoothing
    (2, 2, 2, 29, 1300, 16, 64, "HND", True),      # two Q blocks per head, the last one ragged
    (64, 8, 8, 2, 1100, 32, 128, "HND", True),     # one range per (batch, head), ragged last tile
    (1, 4, 1, 8, 70001, 128, 64, "HND", True),     # many ranges of several tiles
    (1, 4, 2, 3, 900, 128, 64, "HND", True),       # the fewest keys at head_dim 128, one-launch pre-pass at 64
    (16, 8, 8, 1, 515, 128, 64, "NHD", True),      # by the pre-pass's re-reads
    (1, 3, 1, 11, 1200, 128, 64, "NHD", True),     # 33 rows: past the limit
])
def test_few_rows_match_the_formula(dtype, D, B, Hq, Hkv, Sq, Skv, BLKQ, BLKK, layout, smooth):
    g = torch.Generator().manual_seed(Skv + D)
    shape = lambda H, L: (B, L, H, D) if layout == "NHD" else (B, H, L, D)  # noqa: E731
    q, k, v = (torch.randn(shape(H, L), generator=g) for H, L in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    k = k + 2.0 * torch.randn((D,), generator=g)
    q, k, v = (t.to(dtype).cuda() for t in (q * 2.0, k, v))
    out, lse = sa.sageattn(q, k, v, tensor_layout=layout, smooth_k=smooth, pv_mode="fp16", BLKQ=BLKQ, BLKK=BLKK, return_lse=True)
    plain = sa.sageattn(q, k, v, tensor_layout=layout, smooth_k=smooth, pv_mode="fp16", BLKQ=BLKQ, BLKK=BLKK)
    want, want_lse = _reference(q, k, v, layout, BLKQ, BLKK, smooth)
    # P is rounded to 11 bits, the output to 11 (float16) or 8 (bfloat16): a few half ulps of a row's own size
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    rms = want.pow(2).mean().sqrt()
    for got in (out, plain):
        err = (got.cpu().double() - want).abs()
        assert float((err / (want.abs() + rms)).max()) < 2 * unit + 4 * 2.0 ** -11
    # fp32 sums of D products and of Skv probabilities
    assert float((lse.cpu().double() - want_lse).abs().max()) < 2e-5 * max(1.0, float(want_lse.abs().max()))


@pytest.mark.parametrize("smooth", [True, False])
def test_more_batch_entries_and_heads_than_a_grid_axis_of_65535(smooth):
    """Short attentions in great number (B * Hkv = 65552, one more head than the limit would hold): every entry like the same
    entry in a batch of its own size below the limit."""
    g = torch.Generator(device="cuda").manual_seed(9)
    q, k, v = (torch.randn((4097, 16, n, 64), generator=g, device="cuda", dtype=torch.bfloat16) for n in (2, 16, 16))
    kw = dict(smooth_k=smooth, pv_mode="fp16", return_lse=True)
    out, lse = sa.sageattn(q, k, v, **kw)
    for part in (slice(0, 2048), slice(2048, 4097)):
        o, l = sa.sageattn(q[part], k[part], v[part], **kw)
        assert torch.equal(out[part], o) and torch.equal(lse[part], l)
    few = slice(4095, 4097)   # the two entries around the limit, against the formula
    want, want_lse = _reference(q[few], k[few], v[few], "HND", 128, 64, smooth)
    rms = want.pow(2).mean().sqrt()
    assert float(((out[few].cpu().double() - want).abs() / (want.abs() + rms)).max()) < 2 * 2.0 ** -8 + 4 * 2.0 ** -11
    assert float((lse[few].cpu().double() - want_lse).abs().max()) < 2e-5 * max(1.0, float(want_lse.abs().max()))


def test_equal_scores_average_v():
    """Nothing of what lies past the last key of a ragged tile reaches the sums."""
    g = torch.Generator().manual_seed(5)
    k, v = (torch.randn((1, 2, 1500, 128), generator=g).half().cuda() for _ in range(2))
    flat = sa.sageattn(torch.zeros((1, 8, 2, 128)).half().cuda(), k, v, pv_mode="fp16").cpu().double()
    mean = v.cpu().double().mean(2, keepdim=True).repeat_interleave(4, 1)
    assert float((flat - mean).abs().max()) < 2.0 ** -11 * float(mean.abs().max()) + 1e-6   # the output's rounding, fp32 sums


@pytest.mark.parametrize("Sq,Skv", [(22, 3), (23, 7), (23, 8), (28, 47), (28, 48), (32, 79), (32, 80)])
def test_many_heads_of_few_keys(Sq, Skv):
    """Both sides of the line between the two kernels where K and V are short (one query head per KV head, head_dim 128)."""
    g = torch.Generator().manual_seed(Sq + Skv)
    B, H = 4 + (1 << 22) // (32 * Skv * 128), 32   # more elements of K than the one-launch pre-pass takes
    q, k, v = (torch.randn((2, H, n, 128), generator=g).to(torch.bfloat16).cuda() for n in (Sq, Skv, Skv))
    many = lambda t: t.repeat((B + 1) // 2, 1, 1, 1)  # noqa: E731
    out, lse = sa.sageattn(many(q), many(k), many(v), pv_mode="fp16", return_lse=True)
    want, want_lse = _reference(q, k, v, "HND", 128, 64, True)
    rms = want.pow(2).mean().sqrt()
    for i in (0, out.shape[0] // 4 * 2, out.shape[0] - 2):
        assert float(((out[i:i + 2].cpu().double() - want).abs() / (want.abs() + rms)).max()) < 2 * 2.0 ** -8 + 4 * 2.0 ** -11
        assert float((lse[i:i + 2].cpu().double() - want_lse).abs().max()) < 2e-5 * max(1.0, float(want_lse.abs().max()))


def _inputs(seed, B, Hq, Hkv, Sq, Skv, D, dtype):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((B, H, L, D), generator=g) for H, L in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    return tuple(t.to(dtype).cuda() for t in (q, k + 2.0 * torch.randn((D,), generator=g), v))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("smooth", [True, False])
@pytest.mark.parametrize("where,value", [("v", float("inf")), ("v", float("-inf")), ("v", float("nan")), ("k", float("inf")), ("k", float("nan")),
                                         ("q", float("inf")), ("q", float("nan"))])
def test_infinities_and_nan_reach_what_they_reach_in_the_tiled_kernel(dtype, smooth, where, value):
    """The rows of a call with 40 of them per head (the tiled kernel), the first two alone (this one): the same elements are
    NaN, +inf and -inf, in the outputs and the LSE, and none outside the batch entry and KV head that holds the value."""
    q, k, v = _inputs(11, 2, 8, 2, 40, 1100, 128, dtype)
    if where == "q":
        q[0, 5, 1, 3] = value
    else:
        {"k": k, "v": v}[where][0, 1, 1099, 3] = value
    kw = dict(smooth_k=smooth, pv_mode="fp16", BLKQ=16, return_lse=True)
    tiled = sa.sageattn(q, k, v, **kw)
    few = sa.sageattn(q[:, :, :2].contiguous(), k, v, **kw)
    for t, f in zip(tiled, few):
        for kind in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(kind(t[:, :, :2]), kind(f)), kind
        assert torch.isfinite(f[1]).all() and torch.isfinite(f[0, :4]).all()
    if where == "v" or not math.isnan(value):   # (INT8 holds no NaN: the quantiser makes it 0)
        assert not torch.isfinite(few[0][0, 4:]).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,Sq,Skv", [(32, 1, 1, 1025), (2, 2, 32, 2047), (64, 2, 1, 16500), (8, 8, 1, 1100)])
def test_partial_results_stay_inside_the_workspace(D, Hq, Hkv, Sq, Skv):
    """The partial results lie where the V panels of other calls do: with exactly the workspace that the call asks for, nothing
    behind it is written, and the built-in scratch array gives the same bits."""
    q, k, v = _inputs(Skv, 1, Hq, Hkv, Sq, Skv, D, torch.bfloat16)
    need = _cabi.lib().sage_sageattn_workspace_bytes_for(1, Hq, Hkv, Sq, Skv, D, 128, 64, _cabi.PV_FP16, 0, 0, 0, 1, 0, 0)
    ws = torch.full((need + 65536,), 0xA5, device="cuda", dtype=torch.uint8)
    outs = [torch.full_like(q, float("nan")) for _ in range(2)]
    assert sageattn_cabi(q, k, v, outs[0], workspace=ws[:need]) == 0, _cabi.lib().sage_last_error().decode()
    assert sageattn_cabi(q, k, v, outs[1], static=True) == 0, _cabi.lib().sage_last_error().decode()
    torch.cuda.synchronize()
    assert bool((ws[need:] == 0xA5).all())
    assert torch.isfinite(outs[0].float()).all() and torch.equal(outs[0], outs[1])
    assert torch.equal(outs[0], sa.sageattn(q, k, v, pv_mode="fp16"))


def test_captured_call_replays_like_eager():
    shape = (2, 8, 2, 3, 1700, 128, torch.bfloat16)
    q, k, v = _inputs(1, *shape)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        sa.sageattn(q, k, v, pv_mode="fp16")
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sa.sageattn(q, k, v, pv_mode="fp16")
    for seed in (2, 3, 4):
        fresh = _inputs(seed, *shape)
        eager = sa.sageattn(*fresh, pv_mode="fp16")   # the program's own eager work between replays
        torch.cuda.synchronize()
        for t, n in zip((q, k, v), fresh):
            t.copy_(n)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), seed


@pytest.mark.parametrize("Skv", [128 * 512, 128 * 512 + 1])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_mean_of_very_long_histories(Skv, D, dtype):
    """The last number of chunks whose sums the kernel combines, and the first whose mean it finds ready: the same numbers as with keys that
    were smoothed outside (difference rounded to the input type), bit for bit; LSE up to fp32 rounding of q . k_mean (some 2^-24 * 64)."""
    g = torch.Generator(device="cuda").manual_seed(Skv + D)
    q, k, v = (torch.randn((2, h, n, D), generator=g, device="cuda").to(dtype) for h, n in ((4, 3), (2, Skv), (2, Skv)))
    k += 2.0
    km = sa.k_mean(k)
    out, lse = sa.sageattn(q, k, v, return_lse=True)
    want, want_lse = sa.sageattn(q, k - km, v, smooth_k=False, return_lse=True)
    assert torch.equal(out, want)
    shift = (q.double() * km.double().repeat_interleave(2, 1)).sum(-1) * D ** -0.5
    assert float((lse.double() - want_lse.double() - shift).abs().max()) < 1e-4


# one round of the tiled kernel's workgroups and the first head past it, more than 20 rows, the limits of keys and re-reads
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D", [(64, 8, 8, 2, 5, 64), (57, 9, 9, 2, 5, 64), (32, 8, 8, 3, 17, 128), (29, 9, 9, 3, 17, 128),
                                               (33, 8, 8, 20, 17, 128), (33, 8, 8, 21, 17, 128), (65, 8, 4, 8, 33, 64), (130, 8, 8, 9, 7, 64),
                                               (128, 8, 8, 9, 7, 128), (1, 2, 2, 1, 384, 128), (1, 2, 2, 1, 385, 128), (1, 2, 2, 1, 896, 128),
                                               (1, 2, 2, 1, 897, 128), (4, 8, 8, 1, 512, 128), (4, 8, 8, 1, 513, 128)])
def test_both_sides_of_the_rule_for_short_keys(B, Hq, Hkv, Sq, Skv, D, pv):
    g = torch.Generator().manual_seed(Skv + D + Sq)
    q, k, v = (torch.randn((B, h, n, D), generator=g) for h, n in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    q, k, v = q.half().cuda(), (k + 2.0 * torch.randn((D,), generator=g)).half().cuda(), v.half().cuda()
    got = sa.sageattn(q, k, v, pv_mode=pv).cpu().double()
    want, _ = _reference(q, k, v, "HND", 128, 64, True)
    err = float((got - want).norm() / want.norm())
    # P rounded to 11 bits; e4m3 V (3 mantissa bits: 2^-4 / sqrt(3) of a value) and codes of P (0.933 to 1.105, as much once normalised)
    assert err < (2.0 ** -10 if pv == "fp16" else 0.055)


@pytest.mark.parametrize("D,heads,G,Sq", [(64, 2050, 1, 32), (128, 1030, 2, 16)])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
def test_one_range_per_head_and_more_rows_than_one_walk(D, heads, G, Sq, pv):
    """One range per head is normalised 256 / (D / 4) rows to a workgroup by at most 65536 workgroups, which then walk on: the last heads equal
    a call of their own, which one walk covers (the same kernel, so the same numbers)."""
    B, Skv, rows = 16, 100, G * Sq
    assert B * heads * rows * D // 4 > 256 << 16
    if pv == "fp8" and rows > 16:   # (FP8 takes one score tile here: twice the heads of half the rows)
        heads, Sq = 2 * heads, Sq // 2
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn((B, h, n, D), generator=g, device="cuda").half() for h, n in ((heads * G, Sq), (heads, Skv), (heads, Skv)))
    out, lse = sa.sageattn(q, k, v, pv_mode=pv), None
    if pv == "fp16":
        out, lse = sa.sageattn(q, k, v, return_lse=True)
    for at in (0, B - 1):
        part = slice(at, at + 1)
        want, want_lse = sa.sageattn(q[part], k[part], v[part], pv_mode=pv), None
        assert torch.equal(out[part], want)
        if lse is not None:
            want, want_lse = sa.sageattn(q[part], k[part], v[part], return_lse=True)
            assert torch.equal(lse[part], want_lse) and torch.equal(out[part], want)
