"""GPU parity of the explicit-mask variants of the attention kernel and of the LSE that the one-call
pipeline returns, through the C ABI.

Reference behaviour followed:
  * forward(..., attn_mask=bool | additive) and the LSE2 output: sageattention_triton.py:92-105, :127-129,
    checked as test_sageattention_hip.py:40-58 does (mask[..., ::3] = False / -2.0; relative RMSE < 3e-2,
    |LSE2 error| < 3e-2) on its shapes (129 x 70, 4 query heads, 2 KV heads, D = 128).
  * sageattn(..., attn_mask=, smooth_k=True, return_lse=True): test_sage_attention_mate.py:186-208, :467-492
    against softmax(sm_scale * q k^T + mask) and its natural-log logsumexp (:171-178) with
    atol 1.5e-1 / rtol 3e-2 on the LSE (:347-353).
"""
import math

import pytest
import torch

import baselinebenchmark_amd as sa
from oracle import attention as oa
from tests.helpers import randn

pytestmark = [pytest.mark.gpu, pytest.mark.sage_attention]
DEV = "cuda"


def _masks(kind, B, Hq, Sq, Skv, g):
    if kind == "bool_stride3":
        m = torch.ones((B, Hq, Sq, Skv), dtype=torch.bool)
        m[..., ::3] = False
    elif kind == "additive_stride3":
        m = torch.zeros((B, Hq, Sq, Skv))
        m[..., ::3] = -2.0
    elif kind == "bool_random":
        m = torch.rand((B, Hq, Sq, Skv), generator=g) > 0.4
        m[..., 0] = True      # no empty rows here
    elif kind == "additive_random":
        m = torch.randn((B, Hq, Sq, Skv), generator=g)
    elif kind == "additive_neg_inf":
        m = torch.zeros((B, Hq, Sq, Skv))
        m[torch.rand((B, Hq, Sq, Skv), generator=g) < 0.5] = -float("inf")
        m[..., 1] = 0.0
    else:
        raise AssertionError(kind)
    return m


@pytest.mark.parametrize("kind", ["bool_stride3", "additive_stride3", "bool_random", "additive_random", "additive_neg_inf"])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("shape", [(1, 4, 2, 129, 70, 128), (2, 2, 1, 300, 391, 64)])
def test_forward_with_mask_matches_reference_formula(kind, pv, shape):
    B, Hq, Hkv, Sq, Skv, D = shape
    g = torch.Generator().manual_seed(2026 + D + Sq + Skv)
    q = randn("HND", B, Hq, Sq, D, torch.float16, g)
    k = randn("HND", B, Hkv, Skv, D, torch.float16, g)
    v = randn("HND", B, Hkv, Skv, D, torch.float16, g)
    mask = _masks(kind, B, Hq, Sq, Skv, g)
    qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV))
    out, lse = sa.forward(qi, ki, v.to(DEV), qs, ks, attn_mask=mask.to(DEV), return_lse=True, pv_mode=pv)
    torch.cuda.synchronize()
    ref, ref_lse = oa.sage_reference(qi.cpu(), ki.cpu(), v, qs.cpu(), ks.cpu(), "HND", 128, 64, attn_mask=mask)
    m = oa.metrics(out.cpu().float(), ref)
    assert m["finite"]
    if pv == "fp16":
        assert m["rel_rmse"] < 3e-2              # the reference's bound
        assert m["rel_rmse"] < 2e-3              # what this kernel achieves
        assert (lse.cpu().double() - ref_lse).abs().max().item() < 1e-3
    else:
        assert m["cosine"] >= 0.999 and m["rel_rmse"] < 5e-2
        assert (lse.cpu().double() - ref_lse).abs().max().item() < 3e-2


@pytest.mark.parametrize("kind", ["bool_random", "additive_random", "additive_neg_inf"])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("gran", [(128, 16, 1), (32, 64, 4), (64, 128, 4), (16, 32, 4)])
@pytest.mark.parametrize("shape", [(1, 4, 2, 129, 70, 128), (2, 2, 1, 300, 391, 64)])
def test_forward_with_mask_and_fine_k_scales(kind, pv, gran, shape):
    """An explicit mask together with K scale blocks of 16 keys (the external (128, 16) recipe) and with four interleaved
    K scales per block: against the formula with the scales expanded key by key.  (No counterpart in the reference,
    whose forward has one K granularity: the masked kernels look the scale of every score up, so only the lookup
    changes.)"""
    B, Hq, Hkv, Sq, Skv, D = shape
    blkq, blkk, ki4 = gran
    g = torch.Generator().manual_seed(77 + D + Sq + blkk + ki4)
    q = randn("HND", B, Hq, Sq, D, torch.float16, g)
    k = randn("HND", B, Hkv, Skv, D, torch.float16, g, offset_std=1.0)
    # keys of very different magnitude inside a block, so that a wrong scale lookup shows
    k = k * (1.0 + 3.0 * (torch.arange(Skv) % 7 == 0).to(k.dtype))[None, None, :, None]
    v = randn("HND", B, Hkv, Skv, D, torch.float16, g)
    mask = _masks(kind, B, Hq, Sq, Skv, g)
    qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV), BLKQ=blkq, BLKK=blkk, k_interleave=ki4)
    out, lse = sa.forward(qi, ki, v.to(DEV), qs, ks, attn_mask=mask.to(DEV), return_lse=True, pv_mode=pv, BLKQ=blkq, BLKK=blkk,
                          k_interleave=ki4)
    torch.cuda.synchronize()
    ref, ref_lse = oa.sage_reference(qi.cpu(), ki.cpu(), v, qs.cpu(), ks.cpu(), "HND", blkq, blkk, attn_mask=mask, k_interleave=ki4)
    m = oa.metrics(out.cpu().float(), ref)
    assert m["finite"]
    if pv == "fp16":
        assert m["rel_rmse"] < 2e-3
        assert (lse.cpu().double() - ref_lse).abs().max().item() < 1e-3
    else:
        assert m["cosine"] >= 0.999 and m["rel_rmse"] < 5e-2
        assert (lse.cpu().double() - ref_lse).abs().max().item() < 3e-2
    # the one-call pipeline takes the same combination
    full = sa.sageattn(q.to(DEV), k.to(DEV), v.to(DEV), attn_mask=mask.to(DEV), pv_mode=pv, BLKQ=blkq, BLKK=blkk, k_interleave=ki4)
    torch.cuda.synchronize()
    logits = torch.einsum("bhqd,bhkd->bhqk", q.double(), k.double().repeat_interleave(Hq // Hkv, 1)) * D ** -0.5
    logits = logits.masked_fill(~mask, -float("inf")) if mask.dtype == torch.bool else logits + mask.double()
    exact = torch.softmax(logits, -1) @ v.double().repeat_interleave(Hq // Hkv, 1)
    assert oa.metrics(full.cpu().float(), exact)["cosine"] >= 0.999
    # ... and without K smoothing it is the two steps above, bit for bit: the granularity reaches the pipeline's quantiser
    # (boolean masks; an additive mask is in natural-log units there and in base-2 units for forward)
    if mask.dtype == torch.bool:
        plain = sa.sageattn(q.to(DEV), k.to(DEV), v.to(DEV), attn_mask=mask.to(DEV), pv_mode=pv, BLKQ=blkq, BLKK=blkk,
                            k_interleave=ki4, smooth_k=False)
        assert torch.equal(plain, out)


def test_mask_broadcasts_without_being_materialised_and_accepts_half_bias():
    g = torch.Generator().manual_seed(11)
    B, Hq, Hkv, Sq, Skv, D = 2, 4, 2, 200, 333, 64
    q = randn("NHD", B, Hq, Sq, D, torch.bfloat16, g)
    k = randn("NHD", B, Hkv, Skv, D, torch.bfloat16, g)
    v = randn("NHD", B, Hkv, Skv, D, torch.bfloat16, g)
    qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV), tensor_layout="NHD")
    key_padding = torch.ones((B, 1, 1, Skv), dtype=torch.bool)      # [B, 1, 1, Skv]: strides 0 for heads and rows
    key_padding[0, ..., 250:] = False
    key_padding[1, ..., 100:] = False
    out, _ = sa.forward(qi, ki, v.to(DEV), qs, ks, tensor_layout="NHD", attn_mask=key_padding.to(DEV),
                        output_dtype=torch.bfloat16)
    ref, _ = oa.sage_reference(qi.cpu(), ki.cpu(), v.to(torch.float16), qs.cpu(), ks.cpu(), "NHD", 128, 64,
                               attn_mask=key_padding.expand(B, Hq, Sq, Skv))
    assert oa.metrics(out.cpu().float(), ref)["rel_rmse"] < 1e-2    # bf16 output rounding
    rel_bias = (torch.randn((Sq, Skv), generator=g) * 0.5).to(torch.float16)   # [Sq, Skv] half-precision bias
    out2, _ = sa.forward(qi, ki, v.to(DEV), qs, ks, tensor_layout="NHD", attn_mask=rel_bias.to(DEV))
    ref2, _ = oa.sage_reference(qi.cpu(), ki.cpu(), v.to(torch.float16), qs.cpu(), ks.cpu(), "NHD", 128, 64,
                                attn_mask=rel_bias.float().expand(B, Hq, Sq, Skv))
    assert oa.metrics(out2.cpu().float(), ref2)["rel_rmse"] < 2e-3


def test_rows_without_any_visible_key_give_zero_output_and_minus_inf_lse():
    g = torch.Generator().manual_seed(12)
    q = randn("HND", 1, 2, 70, 64, torch.float16, g)
    k = randn("HND", 1, 2, 150, 64, torch.float16, g)
    v = randn("HND", 1, 2, 150, 64, torch.float16, g)
    mask = torch.ones((1, 2, 70, 150), dtype=torch.bool)
    mask[:, :, 5, :] = False
    mask[:, 1, 33, :] = False
    qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV))
    out, lse = sa.forward(qi, ki, v.to(DEV), qs, ks, attn_mask=mask.to(DEV), return_lse=True)
    out, lse = out.cpu().float(), lse.cpu()
    assert torch.isfinite(out).all()
    assert out[:, :, 5].abs().max() == 0 and out[:, 1, 33].abs().max() == 0
    assert torch.isinf(lse[:, :, 5]).all() and (lse[:, :, 5] < 0).all() and lse[0, 1, 33] == -float("inf")
    assert torch.isfinite(lse[:, 0, 33]).all()
    ref, _ = oa.sage_reference(qi.cpu(), ki.cpu(), v, qs.cpu(), ks.cpu(), "HND", 128, 64, attn_mask=mask)
    keep = torch.ones(70, dtype=torch.bool); keep[5] = False; keep[33] = False
    assert oa.metrics(out[:, :, keep], ref[:, :, keep])["rel_rmse"] < 2e-3


def test_mask_of_ones_equals_no_mask_bitwise():
    g = torch.Generator().manual_seed(13)
    q = randn("HND", 1, 2, 260, 128, torch.float16, g)
    k = randn("HND", 1, 2, 260, 128, torch.float16, g)
    v = randn("HND", 1, 2, 260, 128, torch.float16, g)
    qi, qs, ki, ks = sa.per_block_int8(q.to(DEV), k.to(DEV))
    a, la = sa.forward(qi, ki, v.to(DEV), qs, ks, return_lse=True)
    b, lb = sa.forward(qi, ki, v.to(DEV), qs, ks, return_lse=True,
                       attn_mask=torch.ones((1, 1, 260, 260), dtype=torch.bool, device=DEV))
    c, lc = sa.forward(qi, ki, v.to(DEV), qs, ks, return_lse=True, attn_mask=torch.zeros((260, 260), device=DEV))
    # the masked variants scale the scores before the maximum instead of after: same values up to fp32 rounding
    assert (a.float() - b.float()).abs().max().item() <= 2e-3 and (a.float() - c.float()).abs().max().item() <= 2e-3
    assert (la - lb).abs().max().item() < 1e-4 and (la - lc).abs().max().item() < 1e-4
    assert torch.equal(b, c) and torch.equal(lb, lc)


@pytest.mark.parametrize("mask_kind", [None, "bool", "additive"])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
def test_sageattn_lse_is_that_of_the_original_logits_with_k_smoothing(mask_kind, pv):
    # shapes and masks of test_sage_attention_mate.py:467-487, plus a K with a large per-channel offset so
    # that the smoothing correction (q . k_mean) is far larger than the tolerance
    torch.manual_seed(7)
    q = torch.randn((1, 2, 129, 128), dtype=torch.float16)
    k = torch.randn((1, 1, 70, 128), dtype=torch.float16) + (3.0 * torch.randn((1, 1, 1, 128))).to(torch.float16)
    v = torch.randn((1, 1, 70, 128), dtype=torch.float16)
    mask = None
    if mask_kind == "bool":
        mask = torch.ones((1, 2, 129, 70), dtype=torch.bool); mask[..., ::3] = False
    elif mask_kind == "additive":
        mask = torch.zeros((1, 2, 129, 70)); mask[..., ::3] = -2.0
    out, lse = sa.sageattn(q.to(DEV), k.to(DEV), v.to(DEV), smooth_k=True, return_lse=True, pv_mode=pv,
                           attn_mask=None if mask is None else mask.to(DEV))
    scores = torch.matmul(q.double(), k.double().repeat_interleave(2, dim=1).transpose(-1, -2)) * 128 ** -0.5
    if mask is not None:
        scores = scores.masked_fill(~mask, -float("inf")) if mask.dtype == torch.bool else scores + mask.double()
    ref = torch.matmul(torch.softmax(scores, dim=-1), v.double().repeat_interleave(2, dim=1))
    ref_lse = torch.logsumexp(scores, dim=-1)
    m = oa.metrics(out.cpu().float(), ref)
    assert m["cosine"] >= 0.999
    torch.testing.assert_close(lse.cpu().double(), ref_lse, atol=1.5e-1, rtol=3e-2)     # the reference's bound
    assert (lse.cpu().double() - ref_lse).abs().max().item() < 6e-2                     # measured: INT8 noise on the logits
    # without the correction the LSE is off by sm_scale * q . mean(k): make sure the test can see that
    km = k.double().mean(dim=2, keepdim=True).repeat_interleave(2, dim=1)
    shift = (torch.matmul(q.double(), km.transpose(-1, -2)) * 128 ** -0.5).abs().max().item()
    assert shift > 1.0


def test_sageattn_lse_correction_causal_gqa_nhd_bf16():
    g = torch.Generator().manual_seed(21)
    B, Hq, Hkv, S, D = 2, 8, 2, 700, 128
    q = randn("NHD", B, Hq, S, D, torch.bfloat16, g)
    k = (randn("NHD", B, Hkv, S, D, torch.bfloat16, g).float() + 2.0 * torch.randn((B, 1, Hkv, D), generator=g)).to(torch.bfloat16)
    v = randn("NHD", B, Hkv, S, D, torch.bfloat16, g)
    out, lse = sa.sageattn(q.to(DEV), k.to(DEV), v.to(DEV), tensor_layout="NHD", is_causal=True, return_lse=True,
                           pv_mode="fp8", BLKQ=64, BLKK=128)
    qh, kh = q.transpose(1, 2).double(), k.transpose(1, 2).double().repeat_interleave(Hq // Hkv, dim=1)
    scores = torch.matmul(qh, kh.transpose(-1, -2)) * D ** -0.5
    i = torch.arange(S)
    scores = scores.masked_fill(i[None, :] > i[:, None], -float("inf"))
    assert tuple(lse.shape) == (B, Hq, S)
    assert (lse.cpu().double() - torch.logsumexp(scores, dim=-1)).abs().max().item() < 1e-1
    ref = oa.sdpa_fp32(q, k, v, "NHD", True)
    assert oa.metrics(out.cpu().float(), ref)["cosine"] >= 0.999


def _direct_masked_call(q, k, v, mask, layout, pv, blkq, blkk, out, lse, extra):
    """sage_sageattn_masked with exactly the workspace that the call needs (``extra`` more bytes): with none the mask is read
    where it lies, by the variants that take any strides."""
    import ctypes
    from baselinebenchmark_amd import _cabi
    lib = _cabi.lib()
    lay = (lambda t: (*t.shape, *t.stride()[:3])) if layout == "HND" else (lambda t: (t.shape[0], t.shape[2], t.shape[1], t.shape[3], t.stride(0), t.stride(2), t.stride(1)))
    B, Hq, Sq, D, *qst = lay(q)
    _, Hkv, Skv, _, *kst = lay(k)
    pvm = _cabi.PV_FP8 if pv == "fp8" else _cabi.PV_FP16
    need = lib.sage_sageattn_workspace_bytes_for(B, Hq, Hkv, Sq, Skv, D, blkq, blkk, pvm, 0, 0, 0, 1, 1, 1) + extra
    ws = torch.empty(need, device=q.device, dtype=torch.uint8)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    m = mask.expand(B, Hq, Sq, Skv)
    return lib.sage_sageattn_masked(P(q), P(k), P(v), P(out), P(lse), P(ws), need, B, Hq, Hkv, Sq, Skv, D, *qst, *kst, *lay(v)[4:],
                                    *lay(out)[4:], _cabi.DT_BF16 if q.dtype == torch.bfloat16 else _cabi.DT_F16, blkq, blkk, D ** -0.5, 0, 1, pvm,
                                    None, None, 0, 0, P(m), 1, *m.stride(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))


# sizes around the edges of the 256-row q-tile, the 32-row group and the 128-key tile; strides of every kind
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("kind", ["per_head", "documents", "padding", "last_key_only", "nothing", "everything", "transposed", "every_other_key"])
@pytest.mark.parametrize("shape", [(2, 4, 2, 257, 385, 64, 64), (1, 2, 2, 513, 128, 128, 16), (3, 2, 1, 31, 1029, 128, 128), (1, 1, 1, 1, 1, 64, 32)])
def test_packed_boolean_mask_equals_the_mask_read_in_place(shape, kind, pv):
    B, Hq, Hkv, Sq, Skv, D, blkk = shape
    g = torch.Generator().manual_seed(5 + Sq + Skv)
    q, k, v = (randn("HND", B, h, n, D, torch.float16, g).to(DEV) for h, n in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    if kind == "per_head":
        mask = (torch.rand((B, Hq, Sq, Skv), generator=g) > 0.7).to(DEV)
    elif kind == "documents":
        mask = ((torch.arange(Sq)[:, None] // 100) == (torch.arange(Skv)[None] // 100))[None, None].expand(B, 1, Sq, Skv).contiguous().to(DEV)
    elif kind == "padding":
        mask = (torch.arange(Skv)[None] < torch.tensor([Skv - 7 * i for i in range(B)])[:, None])[:, None, None].to(DEV)
    elif kind == "last_key_only":
        mask = (torch.arange(Skv) == Skv - 1)[None, None, None].to(DEV)
    elif kind == "transposed":
        mask = (torch.rand((B, 1, Skv, Sq), generator=g) > 0.5).to(DEV).transpose(-1, -2)
    elif kind == "every_other_key":
        mask = (torch.rand((1, Hq, Sq, 2 * Skv), generator=g) > 0.5).to(DEV)[..., ::2]
    else:
        mask = torch.full((1, 1, Sq, Skv), kind == "everything", device=DEV)
    out, lse = sa.sageattn(q, k, v, attn_mask=mask, pv_mode=pv, BLKK=blkk, return_lse=True)
    want, want_lse = torch.empty_like(out), torch.empty_like(lse)
    assert _direct_masked_call(q, k, v, mask, "HND", pv, 128, blkk, want, want_lse, 0) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(lse, want_lse * 0.6931471805599453)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("BLKQ,BLKK,causal", [(16, 32, False), (32, 64, True), (64, 128, False), (128, 64, True), (128, 16, False)])
def test_lse_of_smoothed_keys_from_the_attention_prologue(dtype, D, pv, BLKQ, BLKK, causal):
    """LSE against the formula in 64 bits on the quantiser's own INT8 operands plus q . k_mean: grouped heads, rows that end
    inside a wavefront and a q-tile, every K scale granularity that takes its own kernel (blocks of 16: the stand-alone Q pass)."""
    g = torch.Generator().manual_seed(D + BLKK)
    B, Hq, Hkv, Sq, Skv = 2, 6, 2, 333, 301
    q, k, v = (torch.randn((B, H, L, D), generator=g).to(dtype).cuda() for H, L in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    k = k + (3.0 * torch.randn((1, Hkv, 1, D), generator=g)).to(dtype).cuda()
    _, lse = sa.sageattn(q, k, v, is_causal=causal, pv_mode=pv, BLKQ=BLKQ, BLKK=BLKK, return_lse=True)
    km = sa.k_mean(k)
    q8, qs, k8, ks = (t.cpu().double() for t in sa.per_block_int8(q, k, km=km, BLKQ=BLKQ, BLKK=BLKK))
    qd = q8 * qs.repeat_interleave(BLKQ, -1)[..., :Sq, None]
    kd = (k8 * ks.repeat_interleave(BLKK, -1)[..., :Skv, None]).repeat_interleave(Hq // Hkv, 1)
    s = qd @ kd.transpose(-1, -2) * 0.6931471805599453
    if causal:
        s = s.masked_fill(torch.arange(Skv)[None] > torch.arange(Sq)[:, None], float("-inf"))
    want = torch.logsumexp(s, -1) + (q.cpu().double() * km.cpu().double().reshape(B, Hkv, 1, D).repeat_interleave(Hq // Hkv, 1)).sum(-1) * D ** -0.5
    # fp32 sums of D products and of at most Skv probabilities
    assert float((lse.cpu().double() - want).abs().max()) < 2e-5 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("additive", [False, True])
@pytest.mark.parametrize("Sq,Skv,D,BLKK", [(70, 127, 64, 64), (257, 128, 128, 128), (300, 129, 64, 16), (33, 385, 128, 32)])
def test_mask_strides_reach_the_same_result(pv, additive, Sq, Skv, D, BLKK):
    """Masks read in place: with contiguous keys (kernels of their own from one whole 128-key tile on) and with every other
    stride, the same bits."""
    g = torch.Generator().manual_seed(Sq + Skv)
    B, Hq, Hkv = 2, 4, 2
    q, k, v = (randn("HND", B, h, n, D, torch.float16, g).to(DEV) for h, n in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    q8, qs, k8, ks = sa.per_block_int8(q, k, BLKK=BLKK)
    make = lambda *s: (torch.randn(s, generator=g) if additive else torch.rand(s, generator=g) > 0.4).to(DEV)  # noqa: E731
    masks = {"transposed": make(B, 1, Skv, Sq).transpose(-1, -2), "every other key": make(1, Hq, Sq, 2 * Skv)[..., ::2],
             "rows of one value": make(B, Hq, Sq, 1).expand(B, Hq, Sq, Skv), "rows at odd offsets": make(1, 1, Sq, Skv + 1)[..., 1:],
             "one row for all": make(B, 1, 1, Skv)}
    for name, mask in masks.items():
        got = sa.forward(q8, k8, v, qs, ks, attn_mask=mask, pv_mode=pv, BLKK=BLKK, return_lse=True)
        dense = mask.expand(B, Hq, Sq, Skv).contiguous()
        strided = dense.transpose(-1, -2).contiguous().transpose(-1, -2)
        for other in (dense, strided):
            want = sa.forward(q8, k8, v, qs, ks, attn_mask=other, pv_mode=pv, BLKK=BLKK, return_lse=True)
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), name


# around the packing's chunks of 16 keys and batches of rows, the second chunk of 64 key tiles of the tile list, and every K scale kind
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,BLKQ,BLKK,groups", [
    (8, 64, 8, 3, 5, 64, 128, 64, (1, 1)),        # fewer keys than one load of the packing
    (2, 256, 32, 40, 16, 64, 128, 32, (1, 1)),    # exactly one
    (1, 2, 1, 300, 257, 64, 128, 64, (1, 1)),     # one key past it, two q-tiles
    (1, 2, 2, 129, 399, 128, 32, 64, (8, 4)),     # interleaved scales; a row past half a q-tile
    (1, 2, 1, 257, 641, 64, 128, 16, (1, 1)),     # five key tiles and one key
    (1, 1, 1, 256, 8300, 64, 128, 128, (1, 1)),   # 65 key tiles
])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
def test_packed_mask_is_taken_and_changes_no_bit(B, Hq, Hkv, Sq, Skv, D, BLKQ, BLKK, groups, pv):
    lib = __import__("baselinebenchmark_amd._cabi", fromlist=["lib"]).lib()
    g = torch.Generator().manual_seed(Skv)
    q, k, v = (randn("HND", B, h, n, D, torch.bfloat16, g).to(DEV) for h, n in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    flags = (sa.sageattention.BLK_INTERLEAVE8 if groups[0] == 8 else 0, sa.sageattention.BLK_INTERLEAVE4 if groups[1] == 4 else 0)
    rows = torch.arange(Sq)[:, None]
    masks = {"random": torch.rand((B, 1, Sq, Skv), generator=g) > 0.5,
             "band": ((torch.arange(Skv)[None] - rows * Skv // Sq).abs() < 70)[None, None],
             "far tiles": ((torch.arange(Skv)[None] >= Skv - 3) | (torch.arange(Skv)[None] == rows % 2))[None, None],
             "padding": (torch.arange(Skv) < max(1, Skv - 9))[None, None, None]}
    for name, mask in masks.items():
        mask = mask.to(DEV)
        m = mask.expand(B, Hq, Sq, Skv)
        extra = lib.sage_sageattn_mask_bytes(B, Hq, Sq, Skv, 1, *m.stride()[:3])
        assert extra > 0, name
        outs = [torch.empty_like(q) for _ in range(2)]
        lses = [torch.empty((B, Hq, Sq), device=DEV) for _ in range(2)]
        for out, lse, room in zip(outs, lses, (extra, 0)):   # packed, and read in place for want of room
            assert _direct_masked_call(q, k, v, mask, "HND", pv, BLKQ | flags[0], BLKK | flags[1], out, lse, room) == 0
        out, lse = sa.sageattn(q, k, v, attn_mask=mask, pv_mode=pv, BLKQ=BLKQ, BLKK=BLKK, q_interleave=groups[0], k_interleave=groups[1],
                               return_lse=True)
        assert torch.equal(out, outs[0]) and torch.equal(lse, lses[0] * 0.6931471805599453), name
        assert torch.equal(outs[0], outs[1]) and torch.equal(lses[0], lses[1]), name


def test_masks_that_are_not_packed():
    """More key tiles than the tile list holds, and calls too small for the pass: no room asked for, the mask is read in place."""
    lib = __import__("baselinebenchmark_amd._cabi", fromlist=["lib"]).lib()
    assert lib.sage_sageattn_mask_bytes(2, 16, 500, 200, 1, 100000, 0, 200) == 0
    assert lib.sage_sageattn_mask_bytes(1, 2, 500, 500, 2, 250000, 0, 500) == 0   # additive
    Skv = 128 * 2048 + 1
    assert lib.sage_sageattn_mask_bytes(1, 1, 1, Skv - 1, 1, 0, 0, 0) > 0
    assert lib.sage_sageattn_mask_bytes(1, 1, 1, Skv, 1, 0, 0, 0) == 0
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn((1, 1, n, 64), generator=g, device=DEV, dtype=torch.float16) for n in (2, Skv, Skv))
    keep = torch.zeros((1, 1, 1, Skv), dtype=torch.bool, device=DEV)
    keep[..., [0, 129, 70001, Skv - 1]] = True
    seen = keep.flatten().nonzero().flatten()
    out = sa.sageattn(q, k, v, attn_mask=keep, smooth_k=False)
    want = torch.softmax((q.double() @ k[:, :, seen].double().transpose(-1, -2)) / 8.0, -1) @ v[:, :, seen].double()
    # INT8 logits: half a step of 1/127 of the largest |k| and |q| in every product, as in the other comparisons with plain attention
    assert torch.nn.functional.cosine_similarity(out.double().flatten(), want.flatten(), dim=0) > 0.999
