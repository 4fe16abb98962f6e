"""FP8 P.V on a few query rows (split keys): the same arithmetic as the tiled kernel in another order."""
import math

import pytest
import torch

import baselinebenchmark_amd as sa
from baselinebenchmark_amd import _cabi

pytestmark = [pytest.mark.gpu, pytest.mark.sage_attention]


def _inputs(B, Hq, Hkv, Sq, Skv, D, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn((B, h, n, D), generator=g, device="cuda") for h, n in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    return q.to(dtype), (k + 2.0 * torch.randn((1, Hkv, 1, D), generator=g, device="cuda")).to(dtype), v.to(dtype)


def _tiled(q, k, v, blkq, **kw):
    """The same rows as part of 48: the others fill scale blocks of their own, so these rows have the same INT8 values, and the call
    takes the tiled kernel."""
    pad = q[:, :, :1].expand(-1, -1, 48 - q.shape[2], -1)
    assert q.shape[2] % blkq == 0 or q.shape[2] < blkq
    keep = blkq if q.shape[2] < blkq else q.shape[2]
    big = torch.cat((q, q[:, :, -1:].expand(-1, -1, keep - q.shape[2], -1), pad[:, :, :48 - keep]), 2).contiguous()
    return sa.sageattn(big, k, v, pv_mode="fp8", BLKQ=blkq, **kw)[:, :, :q.shape[2]]


# ranges of one tile and of several, a ragged last tile of one key, one and two score tiles, grouped query heads
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv", [(1, 8, 2, 1, 1025), (2, 2, 2, 8, 1157), (1, 2, 1, 8, 4097), (16, 32, 32, 1, 129),
                                             (1, 4, 4, 16, 3000), (2, 8, 4, 16, 4200), (1, 2, 2, 1, 33000)])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("blkk,smooth", [(64, True), (16, True), (128, False)])
def test_equals_the_tiled_kernel(B, Hq, Hkv, Sq, Skv, D, dtype, blkk, smooth):
    """Both take each probability from the same 8-bit code unless rounding puts the score on the other side of a code's edge.  The tiled
    kernel takes the accumulators' bias 1.5 * 2^23 off inside an fma whose addend is rounded: up to ulp(1.26e7 * sc) / 2 in the score and
    as much in the row maximum, sc the product of the scales, at most 5e-4 on these inputs (unsmoothed keys with offsets): 2 * 2.4e-4 * 8
    codes, so f = 4e-3 to 8e-3 of the codes differ, by 1/8 each: sqrt(f) / 8 = 8e-3 to 1.1e-2 of a probability if one key dominated the row,
    less averaged over keys.  Without bias rounding (smoothed keys) f is some 1e-3.  bfloat16 outputs add 2^-9."""
    q, k, v = _inputs(B, Hq, Hkv, Sq, Skv, D, dtype)
    kw = dict(BLKK=blkk, smooth_k=smooth)
    got, want = sa.sageattn(q, k, v, pv_mode="fp8", BLKQ=16, **kw).double(), _tiled(q, k, v, 16, **kw).double()
    assert float((got - want).norm() / want.norm()) < (5e-3 if smooth else 1.1e-2)


@pytest.mark.parametrize("D", [64, 128])
def test_a_late_range_far_above_the_first_tile(D):
    """Keys whose scores lie 2^30 above those of the first tile, and a first tile above everything else: probabilities stay coded near
    the top of their tile's range (cosine of the e4m3 format's own error against exact attention)."""
    for late in (True, False):
        q, k, v = _inputs(1, 4, 2, 2, 2500, D, torch.float16, 3)
        q = torch.ones_like(q)
        k[:, :, slice(2000, 2128) if late else slice(0, 128)] += 30.0 * math.log(2.0) / math.sqrt(D)
        got = sa.sageattn(q, k, v, pv_mode="fp8", BLKK=16, smooth_k=False).double()
        want = torch.softmax(q.double() @ k.double().repeat_interleave(2, 1).transpose(-1, -2).contiguous() / math.sqrt(D), -1) @ v.double().repeat_interleave(2, 1)
        assert float(torch.nn.functional.cosine_similarity(got.flatten(), want.flatten(), 0)) > 0.995


@pytest.mark.parametrize("D,Sq,Skv", [(64, 8, 1900), (128, 8, 4100), (128, 4, 1030), (64, 1, 20000)])
def test_workspace_by_need_is_not_exceeded(D, Sq, Skv):
    Hq, Hkv = 8, 2
    q, k, v = _inputs(1, Hq, Hkv, Sq, Skv, D, torch.float16, 1)
    lib, need = _cabi.lib(), 0
    need = lib.sage_sageattn_workspace_bytes_for(1, Hq, Hkv, Sq, Skv, D, 128, 64, _cabi.PV_FP8, 0, 0, 0, 1, 0, 0)
    out, ws = torch.empty_like(q), torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    st = lambda h, n: (h * n * D, n * D, D)
    rc = lib.sage_sageattn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), None, ws.data_ptr(), need, 1, Hq, Hkv, Sq, Skv, D,
                           *st(Hq, Sq), *st(Hkv, Skv), *st(Hkv, Skv), *st(Hq, Sq), 0, 128, 64, float(D ** -0.5), 0, 1, _cabi.PV_FP8, None,
                           None, 0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and bool((ws[need:] == 0x5A).all())
    assert torch.equal(out, sa.sageattn(q, k, v, pv_mode="fp8"))


@pytest.mark.parametrize("what", ["inf", "-inf", "nan", "huge"])
def test_infinities_and_large_values_come_out_as_in_the_tiled_kernel(what):
    """An infinity makes its channel infinite, values near the end of bfloat16's range stay finite: the V scale multiplies the
    merged, normalised output."""
    q, k, v = _inputs(1, 4, 2, 2, 2100, 64, torch.bfloat16, 5)
    if what == "huge":
        v *= 1e35
    else:
        v[0, 1, 1500, 3] = float(what)
    got, want = sa.sageattn(q, k, v, pv_mode="fp8", BLKQ=16), _tiled(q, k, v, 16)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    if what in ("inf", "-inf"):
        assert bool(torch.isinf(got).any())
    elif what == "huge":
        assert bool(torch.isfinite(got).all())


@pytest.mark.parametrize("D,heads", [(128, 33000), (64, 66000)])
@pytest.mark.parametrize("Skv", [1, 2, 3, 4, 5])
def test_a_handful_of_keys_in_very_many_heads(D, heads, Skv):
    """Four bytes of V statistics per channel and chunk outgrow the byte per channel and key of the region they share with the INT8
    keys where there are fewer than four keys.  The first heads alone are few enough elements for the tiled kernel; two e4m3 roundings of
    V and the codes of at most five probabilities lie between the two, and one key has probability one: V rounded once, bit for bit."""
    B = heads // 2
    q, k, v = _inputs(B, 2, 2, 1, Skv, D, torch.float16, Skv)
    got = sa.sageattn(q, k, v, pv_mode="fp8")
    n = 4096
    for at in (0, B // 3, B - n):   # (statistics that run into the scales go wrong in the later heads)
        part = slice(at, at + n)
        want = sa.sageattn(q[part], k[part], v[part], pv_mode="fp8")
        if Skv < 4:
            assert torch.equal(got[part], want), at
        else:
            assert float((got[part].double() - want.double()).norm() / want.double().norm()) < 5e-3, at
    if Skv == 1:   # the abs-maximum of a channel is the one value: code 448, scale |v| / 448
        assert float((got - v).abs().max()) <= float(v.abs().max()) * 2 ** -10


@pytest.mark.parametrize("D,Sq", [(64, 1), (128, 4), (128, 16), (64, 32)])
@pytest.mark.parametrize("binades", [10.3, 20.3, 36.3, 60.3, 100.3])
def test_a_flat_tail_far_below_one_key(D, Sq, binades):
    """One key lies `binades` above all others, and only keys of later tiles have values (those of its own tile lie below the tile's
    codes): the output is their weight alone, n 2^-binades V.  512 heads are one range each, so the key and its tail meet in one accumulator.
    A code is 2^t with a linear mantissa (up to 1.086), shifted by 0.3 of its 8 steps per binade (0.974) and rounded (2^(+-1/16)): 0.933
    to 1.105 of the probability.  Both kernels have the same code; what is left between them is bfloat16 rounding."""
    B, H, Skv = 64, 8, 128 * 15
    a = binades * math.log(2.0) / math.sqrt(D)
    q = torch.ones((B, H, Sq, D), device="cuda", dtype=torch.bfloat16)
    k = torch.zeros((B, H, Skv, D), device="cuda", dtype=torch.bfloat16)
    v = torch.full((B, H, Skv, D), 30000.0, device="cuda", dtype=torch.bfloat16)
    k[:, :, 5], v[:, :, :128] = a, 0.0
    got = sa.sageattn(q, k, v, pv_mode="fp8", BLKQ=16, smooth_k=False).double()
    p = torch.softmax(k[0, 0].double().sum(-1) / math.sqrt(D), 0)
    want = float(p @ v[0, 0, :, 0].double())
    assert float((got / want - 1).abs().max()) < 0.105 + 2 ** -8
    if Sq <= 16:
        tiled = _tiled(q, k, v, 16, smooth_k=False).double()
        assert float((got / tiled - 1).abs().max()) < 2 ** -7
