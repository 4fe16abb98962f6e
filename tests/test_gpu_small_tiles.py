"""Attention in workgroups of 128 query rows (four wavefronts): sequence ends and diagonals at every edge of a 32-key group."""
import pytest
import torch

import baselinebenchmark_amd as sa
from baselinebenchmark_amd import _cabi
from baselinebenchmark_amd import sageattention as S
from oracle import attention as oa
from tests.helpers import randn

pytestmark = [pytest.mark.gpu, pytest.mark.sage_attention]
DEV = "cuda"
EDGES = [1, 31, 32, 33, 64, 65, 96, 97, 127, 128, 129, 160, 161, 255, 256, 257, 384, 385]


def rows_of(call):
    """A call's results and the query rows per workgroup that it took."""
    out = call()
    return out, _cabi.lib().sage_last_tile_rows()


def from_256_rows(q, k, v, qs, ks, blkk, causal, pv, lse, fused_q=False):
    """The [1, H, L, D] call as a packed batch of one sequence, whose plan has q-tiles of 256 rows at every length."""
    Hq, Sq, D = q.shape[1:]
    Hkv, Skv = k.shape[1:3]
    dtype, pv_mode = v.dtype, S._pv(pv)
    cu_q, cu_k = (torch.tensor([0, n], dtype=torch.int32, device=DEV) for n in (Sq, Skv))
    plan, _ = sa.varlen_plan(cu_q, cu_k, Sq, 64, blkk, is_causal=causal)
    panels, v_scale = sa.prepare_v(v, "HND", pv)
    out = torch.empty((1, Hq, Sq, D), device=DEV, dtype=dtype)
    lse2 = torch.empty((1, Hq, Sq), device=DEV, dtype=torch.float32) if lse else None
    p = S._ptr
    shape = (1, Hq, Hkv, Sq, Skv, D, *q.stride()[:3], *k.stride()[:3], *out.stride()[:3], 64, blkk, int(causal), pv_mode, S._dt(dtype),
             p(cu_q), p(cu_k), p(plan), Sq)
    panel_sh = -(-Skv // _cabi.PANEL_ROWS)
    if fused_q:
        rc = lambda: _cabi.lib().sage_attn_fwd_qfused(p(q), S._dt(dtype), 0.0, p(k), p(panels), p(ks), p(v_scale), p(out), p(lse2), *shape,
                                                      ks.shape[2], panel_sh, S._stream(q))
    else:
        rc = lambda: _cabi.lib().sage_attn_fwd(p(q), p(k), p(panels), p(qs), p(ks), p(v_scale), p(out), p(lse2), *shape, qs.shape[2], ks.shape[2],
                                               panel_sh, S._stream(q))
    assert rows_of(lambda: _cabi.check(rc()))[1] == 256
    return out, lse2


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("blkk", [16, 32, 64, 128])
def test_fixed_length_calls_get_the_same_bits_from_128_and_256_rows(blkk, D, pv, causal):
    for Skv in EDGES:
        Sq = Skv if causal else 130
        g = torch.Generator().manual_seed(3 * Skv + D)
        q, k, v = (randn("HND", 1, 2, n, D, torch.float16, g).to(DEV) for n in (Sq, Skv, Skv))
        qi, qs, ki, ks = sa.per_block_int8(q, k, BLKQ=64, BLKK=blkk)
        kw = dict(output_dtype=torch.float16, BLKQ=64, BLKK=blkk, is_causal=causal, pv_mode=pv)
        for lse in (False, True):
            (out, l2), rows = rows_of(lambda: sa.forward(qi, ki, v, qs, ks, return_lse=lse, **kw))
            assert rows == 128
            want, want_l2 = from_256_rows(qi, ki, v, qs, ks, blkk, causal, pv, lse)
            assert torch.equal(out, want) and (not lse or torch.equal(l2, want_l2)), (Skv, lse)
            (out, l2), rows = rows_of(lambda: sa.forward_fused_q(q, ki, v, ks, return_lse=lse, **kw))
            assert rows == 128
            want, want_l2 = from_256_rows(q, ki, v, None, ks, blkk, causal, pv, lse, fused_q=True)
            assert torch.equal(out, want) and (not lse or torch.equal(l2, want_l2)), (Skv, lse)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("blkk", [16, 32])
def test_every_end_of_a_tile_matches_the_formula(blkk, D, pv, causal):
    # tolerances of test_gpu_attention.py: FP16 P.V relative RMSE 2e-3, FP8 5e-2 (e4m3), LSE2 1e-3
    for Skv in EDGES:
        Sq = Skv if causal else 130
        g = torch.Generator().manual_seed(11 * Skv + D)
        q, k, v = (randn("HND", 1, 2, n, D, torch.float16, g) for n in (Sq, Skv, Skv))
        qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV), BLKQ=64, BLKK=blkk)
        ref, ref_lse = oa.sage_reference(qi.cpu(), ki.cpu(), v, qs.cpu(), ks.cpu(), "HND", 64, blkk, is_causal=causal)
        kw = dict(output_dtype=torch.float16, BLKQ=64, BLKK=blkk, is_causal=causal, pv_mode=pv)
        for lse in (False, True):
            out, l2 = sa.forward(qi, ki, v.to(DEV), qs, ks, return_lse=lse, **kw)
            m = oa.metrics(out.cpu().float(), ref)
            assert m["finite"] and m["rel_rmse"] < (2e-3 if pv == "fp16" else 5e-2), (Skv, lse, m)
            if lse:
                assert (l2.cpu().double() - ref_lse).abs().max().item() < 1e-3, Skv
        assert torch.equal(sa.forward_fused_q(q.to(DEV), ki, v.to(DEV), ks, **kw)[0], sa.forward(qi, ki, v.to(DEV), qs, ks, **kw)[0]), Skv


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("blkk", [32, 64, 128])
def test_packed_batches_get_the_same_bits_from_128_and_256_rows(blkk, pv, causal):
    # head_dim 128: a bound on the lengths far above them makes the call take the workgroups of 256 rows
    T, H, D = sum(EDGES), 4, 128
    cu = torch.tensor([sum(EDGES[:i]) for i in range(len(EDGES) + 1)], dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn((T, h, D), generator=g).to(torch.bfloat16).to(DEV) for h in (H, 2, 2))
    kw = dict(is_causal=causal, pv_mode=pv, BLKQ=128, BLKK=blkk)
    small, rows = rows_of(lambda: sa.sageattn_varlen(q, k, v, cu, cu, max(EDGES), max(EDGES), **kw))
    large, more_rows = rows_of(lambda: sa.sageattn_varlen(q, k, v, cu, cu, 8192, 8192, **kw))
    assert (rows, more_rows) == (128, 256)
    assert torch.isfinite(small.float()).all() and torch.equal(small, large)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("blkk", [32, 64, 128])
def test_packed_batches_of_head_dim_64_get_the_bits_of_256_rows(blkk, pv, causal):
    # (they take the workgroups of 128 rows at every length: each sequence is compared with a call of its own from 256 rows)
    T, D = sum(EDGES), 64
    starts = [sum(EDGES[:i]) for i in range(len(EDGES) + 1)]
    cu = torch.tensor(starts, dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn((T, h, D), generator=g).to(torch.bfloat16).to(DEV) for h in (4, 2, 2))
    packed, rows = rows_of(lambda: sa.sageattn_varlen(q, k, v, cu, cu, max(EDGES), max(EDGES), is_causal=causal, pv_mode=pv, smooth_k=False, BLKQ=64, BLKK=blkk))
    assert rows == 128
    for a, b in zip(starts, starts[1:]):
        qq, kk, vv = (t[a:b].transpose(0, 1)[None].contiguous() for t in (q, k, v))
        qi, qs, ki, ks = sa.per_block_int8(qq, kk, BLKQ=64, BLKK=blkk)
        want, _ = from_256_rows(qi, ki, vv, qs, ks, blkk, causal, pv, False)
        assert torch.equal(packed[a:b].transpose(0, 1), want[0]), b - a


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("D", [64, 128])
def test_interleaved_k_scales_match_the_formula_at_every_end_of_a_tile(D, pv, causal):
    for Skv in EDGES:
        Sq = Skv if causal else 130
        g = torch.Generator().manual_seed(7 * Skv + D)
        q, k, v = (randn("HND", 1, 2, n, D, torch.float16, g) for n in (Sq, Skv, Skv))
        qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV), BLKQ=32, BLKK=64, k_interleave=4)
        n = torch.arange(Skv)
        ref, ref_lse = oa.sage_reference(qi.cpu(), ki.cpu(), v, qs.cpu(), ks.cpu()[..., (n // 64) * 4 + (n % 8) // 2], "HND", 32, 1, is_causal=causal)
        for lse in (False, True):
            out, l2 = sa.forward(qi, ki, v.to(DEV), qs, ks, output_dtype=torch.float16, BLKQ=32, BLKK=64, is_causal=causal, pv_mode=pv, k_interleave=4,
                                 return_lse=lse)
            m = oa.metrics(out.cpu().float(), ref)
            assert m["finite"] and m["rel_rmse"] < (2e-3 if pv == "fp16" else 5e-2), (Skv, lse, m)
            assert not lse or (l2.cpu().double() - ref_lse).abs().max().item() < 1e-3, Skv


@pytest.mark.parametrize("pv,lse", [("fp16", False), ("fp16", True), ("fp8", False)])
@pytest.mark.parametrize("D", [64, 128])
def test_interleaved_k_scales_get_the_same_bits_from_128_and_256_rows(D, pv, lse):
    # (160 heads over more than a thousand keys are one round of the chip in q-tiles of 256 rows, 120 leave it unfilled, 300 are two rounds)
    batches = (150 if (D, pv) == (64, "fp8") else 60, 80)
    for Skv in [1280 + n for n in EDGES]:
        g = torch.Generator().manual_seed(Skv + D)
        q, k, v = (randn("HND", 1, 2, n, D, torch.float16, g).to(DEV) for n in (130, Skv, Skv))
        qi, qs, ki, ks = sa.per_block_int8(q, k, BLKQ=32, BLKK=64, k_interleave=4)
        kw = dict(output_dtype=torch.float16, BLKQ=32, BLKK=64, pv_mode=pv, k_interleave=4, return_lse=lse)
        (small, rows), (large, more_rows) = (rows_of(lambda: sa.forward(*(t.repeat(n, 1, 1, 1) for t in (qi, ki, v)), *(t.repeat(n, 1, 1) for t in (qs, ks)), **kw))
                                             for n in batches)
        assert (rows, more_rows) == (128, 256)
        assert torch.equal(small[0][:60], large[0][:60]) and (not lse or torch.equal(small[1][:60], large[1][:60])), Skv




@pytest.mark.parametrize("kind", ["keep", "keep_rows_alike", "bias"])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("D", [64, 128])
def test_masks_get_the_same_bits_from_128_and_256_rows(D, pv, kind):
    # a mask whose keys are not contiguous makes the call take the workgroups of 256 rows; sageattn packs a boolean one into bits
    for Sq, Skv in [(1, 128), (33, 300), (128, 127), (129, 385), (200, 129), (256, 500), (257, 640), (400, 1100)]:
        g = torch.Generator().manual_seed(Sq + Skv)
        q, k, v = (randn("HND", 2, 2, n, D, torch.bfloat16, g).to(DEV) for n in (Sq, Skv, Skv))
        shape = (2, 1, 1 if kind == "keep_rows_alike" else Sq, Skv)
        mask = torch.randn(shape, generator=g).to(DEV) if kind == "bias" else (torch.rand(shape, generator=g) < 0.6).to(DEV)
        spread = torch.zeros((*shape, 2), dtype=mask.dtype, device=DEV)
        spread[..., 0] = mask
        qi, qs, ki, ks = sa.per_block_int8(q, k, BLKQ=64, BLKK=64)
        kw = dict(output_dtype=torch.bfloat16, BLKQ=64, BLKK=64, pv_mode=pv, return_lse=True)
        (small, rows), (large, more_rows) = (rows_of(lambda: sa.forward(qi, ki, v, qs, ks, attn_mask=m, **kw)) for m in (mask, spread[..., 0]))
        assert (rows, more_rows) == (128, 256) or Skv < 128 and kind == "bias" and rows == 256, (Sq, Skv)
        assert torch.equal(small[0], large[0]) and torch.equal(small[1], large[1]), (Sq, Skv)
        if kind != "bias":
            packed, rows = rows_of(lambda: sa.sageattn(q, k, v, attn_mask=mask, smooth_k=False, pv_mode=pv, BLKQ=64, BLKK=64))
            assert rows == 128, (Sq, Skv)
            assert torch.equal(packed, large[0]), (Sq, Skv)


PLAIN, FINE, INTERLEAVED = dict(BLKQ=128, BLKK=64), dict(BLKQ=128, BLKK=16), dict(BLKQ=32, BLKK=64, q_interleave=8, k_interleave=4)


@pytest.mark.parametrize("D,pv,causal,lse,scales,H,L,rows", [
    (128, "fp16", False, False, PLAIN, 75, 1500, 256), (128, "fp16", False, True, PLAIN, 75, 1500, 256), (128, "fp16", False, False, PLAIN, 37, 1700, 128),
    (128, "fp8", False, False, PLAIN, 73, 1700, 256), (128, "fp8", False, False, PLAIN, 47, 2600, 128), (128, "fp8", False, True, PLAIN, 73, 1700, 128),
    (128, "fp16", False, False, INTERLEAVED, 85, 1500, 256), (128, "fp16", True, False, PLAIN, 32, 3500, 256), (128, "fp8", True, False, PLAIN, 73, 3500, 256),
    (128, "fp8", True, False, FINE, 100, 2300, 128), (128, "fp8", True, False, PLAIN, 8, 16000, 256), (64, "fp16", False, False, PLAIN, 32, 3500, 256),
    (64, "fp16", False, False, PLAIN, 18, 4200, 128), (64, "fp16", True, False, PLAIN, 20, 5600, 256), (64, "fp16", True, False, INTERLEAVED, 20, 5600, 128),
    (64, "fp8", False, False, FINE, 14, 8000, 256), (64, "fp8", False, True, FINE, 8, 8000, 256), (64, "fp8", False, False, INTERLEAVED, 85, 1500, 256),
    (64, "fp8", False, False, INTERLEAVED, 10, 2000, 256), (64, "fp8", False, True, INTERLEAVED, 16, 4200, 128), (64, "fp8", True, False, INTERLEAVED, 16, 4200, 128),
])
def test_calls_take_the_size_that_measured_faster(D, pv, causal, lse, scales, H, L, rows):
    q, k, v = (torch.zeros((1, H, L, D), device=DEV, dtype=torch.bfloat16) for _ in range(3))
    assert rows_of(lambda: sa.sageattn(q, k, v, is_causal=causal, pv_mode=pv, return_lse=lse, **scales))[1] == rows


@pytest.mark.parametrize("D,pv,mask,H,L,rows", [
    (64, "fp16", "keep", 24, 2078, 256), (64, "fp16", "keep", 24, 1500, 128), (64, "fp16", "keep", 33, 2078, 128), (64, "fp16", "bias", 24, 2078, 128),
    (64, "fp8", "keep", 24, 2078, 128), (128, "fp16", "keep", 67, 1500, 256), (128, "fp16", "keep", 33, 2078, 128), (128, "fp16", "keep", 32, 1500, 256),
    (128, "fp8", "keep", 67, 1500, 128),
])
def test_masked_calls_take_the_size_that_measured_faster(D, pv, mask, H, L, rows):
    q, k, v = (torch.zeros((1, H, L, D), device=DEV, dtype=torch.bfloat16) for _ in range(3))
    m = torch.ones((1, 1, 1, L), device=DEV, dtype=torch.bool) if mask == "keep" else torch.zeros((1, 1, L, L), device=DEV)
    assert rows_of(lambda: sa.sageattn(q, k, v, attn_mask=m, pv_mode=pv))[1] == rows
