"""Attention in workgroups of 128 query rows (four wavefronts): sequence ends and diagonals at every edge of a 32-key group."""
import pytest
import torch

import baselinebenchmark_amd as sa
from oracle import attention as oa
from tests.helpers import randn

pytestmark = [pytest.mark.gpu, pytest.mark.sage_attention]
DEV = "cuda"
EDGES = [1, 31, 32, 33, 64, 65, 96, 97, 127, 128, 129, 160, 161, 255, 256, 257, 384, 385]


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
    small = sa.sageattn_varlen(q, k, v, cu, cu, max(EDGES), max(EDGES), **kw)
    large = sa.sageattn_varlen(q, k, v, cu, cu, 8192, 8192, **kw)
    assert torch.isfinite(small.float()).all() and torch.equal(small, large)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("D", [64, 128])
def test_interleaved_k_scales_match_the_formula_at_every_end_of_a_tile(D, pv, causal):
    for Skv in EDGES:
        Sq = Skv if causal else 130
        g = torch.Generator().manual_seed(7 * Skv + D)
        q, k, v = (randn("HND", 1, 2, n, D, torch.float16, g) for n in (Sq, Skv, Skv))
        qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV), BLKQ=32, BLKK=64, k_interleave=4)
        out, _ = sa.forward(qi, ki, v.to(DEV), qs, ks, output_dtype=torch.float16, BLKQ=32, BLKK=64, is_causal=causal, pv_mode=pv, k_interleave=4)
        n = torch.arange(Skv)
        ref, _ = oa.sage_reference(qi.cpu(), ki.cpu(), v, qs.cpu(), ks.cpu()[..., (n // 64) * 4 + (n % 8) // 2], "HND", 32, 1, is_causal=causal)
        m = oa.metrics(out.cpu().float(), ref)
        assert m["finite"] and m["rel_rmse"] < (2e-3 if pv == "fp16" else 5e-2), (Skv, m)


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
        small, large = (sa.forward(qi, ki, v, qs, ks, attn_mask=m, **kw) for m in (mask, spread[..., 0]))
        assert torch.equal(small[0], large[0]) and torch.equal(small[1], large[1]), (Sq, Skv)
        if kind != "bias":
            packed = sa.sageattn(q, k, v, attn_mask=mask, smooth_k=False, pv_mode=pv, BLKQ=64, BLKK=64)
            assert torch.equal(packed, large[0]), (Sq, Skv)
