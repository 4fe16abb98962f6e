"""The pre-passes that share launches (statistics and plan first, quantiser and V panels second) against the same call made of
the separate entry points: every intermediate is the same number, so outputs are equal bit for bit."""
import pytest
import torch

import baselinebenchmark_amd as sa
from baselinebenchmark_amd import _cabi
from tests.helpers import randn

pytestmark = [pytest.mark.gpu, pytest.mark.sage_attention]


def _inputs(B, Hq, Hkv, Sq, Skv, D, dtype, layout, seed):
    g = torch.Generator().manual_seed(seed)
    q = randn(layout, B, Hq, Sq, D, dtype, g)
    k = randn(layout, B, Hkv, Skv, D, dtype, g, offset_std=2.0)
    return q.cuda(), k.cuda(), randn(layout, B, Hkv, Skv, D, dtype, g).cuda()


def _steps(q, k, v, layout, pv, blkq, blkk, smooth, mask=None):
    km = sa.k_mean(k, layout) if smooth else None
    q8, qs, k8, ks = sa.per_block_int8(q, k, km=km, BLKQ=blkq, BLKK=blkk, tensor_layout=layout)
    return sa.forward(q8, k8, v, qs, ks, tensor_layout=layout, output_dtype=q.dtype, pv_mode=pv, BLKQ=blkq, BLKK=blkk, attn_mask=mask)[0]


# one chunk of 512 rows and a bit, whole chunks, the last length whose statistics the second launch combines itself (8 chunks)
# and the first that has a launch for it; then grids whose jobs no longer share launches
@pytest.mark.parametrize("B,H,Skv", [(1, 2, 1025), (1, 2, 1536), (2, 1, 1537), (1, 2, 4096), (1, 2, 4097), (2, 64, 4097)])
@pytest.mark.parametrize("D,dtype,layout", [(64, torch.float16, "NHD"), (128, torch.bfloat16, "HND")])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("smooth", [True, False])
def test_one_call_equals_the_separate_passes(B, H, Skv, D, dtype, layout, pv, smooth):
    q, k, v = _inputs(B, H, H, 70, Skv, D, dtype, layout, Skv + D)
    for blkq, blkk in ((128, 64), (64, 128), (32, 16)):
        got = sa.sageattn(q, k, v, tensor_layout=layout, pv_mode=pv, smooth_k=smooth, BLKQ=blkq, BLKK=blkk)
        assert torch.equal(got, _steps(q, k, v, layout, pv, blkq, blkk, smooth)), (blkq, blkk)


@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("blkq,blkk", [(128, 64), (128, 16), (16, 128)])
def test_masked_call_equals_the_separate_passes(pv, blkq, blkk):
    """The Q quantiser and the packing of the mask share the first launch (or, where its rows per wavefront do not suit the K blocks,
    have one of their own)."""
    q, k, v = _inputs(2, 2, 2, 300, 1100, 64, torch.float16, "HND", 5)
    mask = torch.rand((2, 1, 300, 1100), device="cuda") < 0.5
    got = sa.sageattn(q, k, v, pv_mode=pv, BLKQ=blkq, BLKK=blkk, attn_mask=mask)
    assert torch.equal(got, _steps(q, k, v, "HND", pv, blkq, blkk, True, mask))


@pytest.mark.parametrize("Skv", [1500, 4500])
def test_workspace_without_room_for_both_statistics(Skv):
    """FP8 P.V through the C ABI with exactly sage_sageattn_workspace_bytes_for: the statistics run one after the other in the same
    region; nothing is written past the end, and the output is the one of the call with room for both."""
    B, H, S, D = 1, 3, 40, 128
    q, k, v = _inputs(B, H, H, S, Skv, D, torch.bfloat16, "HND", 9)
    lib = _cabi.lib()
    need = lib.sage_sageattn_workspace_bytes_for(B, H, H, S, Skv, D, 128, 64, _cabi.PV_FP8, 0, 0, 0, 1, 0, 0)
    out, ws = torch.empty_like(q), torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
    hd = lambda n: (H * n * D, n * D, D)
    rc = lib.sage_sageattn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), None, ws.data_ptr(), need, B, H, H, S, Skv, D,
                           *hd(S), *hd(Skv), *hd(Skv), *hd(S), 1, 128, 64, float(D ** -0.5), 0, 1, _cabi.PV_FP8, None, None, 0, 0,
                           torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and bool((ws[need:] == 0xA5).all())
    assert torch.equal(out, sa.sageattn(q, k, v, pv_mode="fp8"))


@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("smooth", [True, False])
def test_packed_call_equals_single_sequences(pv, smooth):
    """The plan shares the first launch: lengths of nothing, one row, one chunk, and one sequence past eight chunks."""
    lens = [0, 1, 130, 0, 512, 700, 4200]
    g = torch.Generator().manual_seed(3)
    T = sum(lens)
    q, k, v = (torch.randn((T, h, 64), generator=g).to(torch.float16).cuda() for h in (4, 2, 2))
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
    got = sa.sageattn_varlen(q, k, v, cu, cu, max(lens), max(lens), is_causal=True, pv_mode=pv, smooth_k=smooth)
    for i, n in enumerate(lens):
        if n:
            s = slice(int(cu[i]), int(cu[i]) + n)
            one = sa.sageattn(q[None, s], k[None, s], v[None, s], tensor_layout="NHD", is_causal=True, pv_mode=pv, smooth_k=smooth)
            assert torch.equal(got[s], one[0]), n


@pytest.mark.parametrize("H", [1, 3, 8])
@pytest.mark.parametrize("Skv", [1, 129, 1100, 4700])
@pytest.mark.parametrize("D", [64, 128])
def test_heads_in_a_row_equal_heads_apart(H, Skv, D):
    """[B, L, H, D] and packed tensors are walked heads first, [B, H, L, D] rows first: the same numbers from every pre-pass."""
    q, k, v = _inputs(2, H, H, 70, Skv, D, torch.bfloat16, "NHD", H + Skv)
    t = [x.transpose(1, 2).contiguous() for x in (q, k, v)]
    km, km_t = sa.k_mean(k, "NHD"), sa.k_mean(t[1], "HND")
    assert torch.equal(km.flatten(1), km_t.flatten(1))   # ([B, 1, H, D] and [B, H, 1, D])
    for blkq, blkk in ((128, 64), (32, 16)):
        a = sa.per_block_int8(q, k, km=km, BLKQ=blkq, BLKK=blkk, tensor_layout="NHD")
        b = sa.per_block_int8(t[0], t[1], km=km_t, BLKQ=blkq, BLKK=blkk, tensor_layout="HND")
        assert torch.equal(a[0], b[0].transpose(1, 2)) and torch.equal(a[1], b[1])
        assert torch.equal(a[2], b[2].transpose(1, 2)) and torch.equal(a[3], b[3])
        for pv in ("fp16", "fp8"):
            got = sa.sageattn(q, k, v, tensor_layout="NHD", pv_mode=pv, BLKQ=blkq, BLKK=blkk)
            assert torch.equal(got, sa.sageattn(*t, pv_mode=pv, BLKQ=blkq, BLKK=blkk).transpose(1, 2)), pv


@pytest.mark.parametrize("H,D", [(16, 128), (32, 64), (32, 128), (24, 64)])
@pytest.mark.parametrize("Skv", [129, 1100, 4700])
def test_rows_of_whole_pages_equal_heads_apart(H, D, Skv):
    """Rows a multiple of 4 KiB apart, which the statistics and the V panels walk heads first, and 3 KiB, which they do not."""
    q, k, v = _inputs(1, H, H, 40, Skv, D, torch.float16, "NHD", H + Skv)
    t = [x.transpose(1, 2).contiguous() for x in (q, k, v)]
    assert torch.equal(sa.k_mean(k, "NHD").flatten(1), sa.k_mean(t[1], "HND").flatten(1))
    for pv in ("fp16", "fp8"):
        for a, b in zip(sa.sageattention.prepare_v(v, "NHD", pv), sa.sageattention.prepare_v(t[2], "HND", pv)):
            assert torch.equal(a, b) if a is not None else b is None
        got = sa.sageattn(q, k, v, tensor_layout="NHD", pv_mode=pv)
        assert torch.equal(got, sa.sageattn(*t, pv_mode=pv).transpose(1, 2)), pv


@pytest.mark.parametrize("rows", [65535 * 64, 65535 * 64 + 1])
def test_more_rows_than_the_second_grid_axis_holds(rows):
    """16-row blocks at head_dim 64: 64 rows per workgroup, 65535 workgroups at most beside the heads."""
    k = torch.randn((1, rows, 2, 64), device="cuda", dtype=torch.float16)
    _, _, k8, ks = sa.per_block_int8(k[:, :16], k, BLKQ=16, BLKK=16, tensor_layout="NHD")
    tail = rows - rows // 16 * 16 + 16 * 8
    _, _, t8, ts = sa.per_block_int8(k[:, :16], k[:, -tail:], BLKQ=16, BLKK=16, tensor_layout="NHD")
    assert torch.equal(k8[:, -tail:], t8) and torch.equal(ks[..., -ts.shape[-1]:], ts)


# element reads (whole sequences, once per K workgroup with a mean and V panel with scales) around the limits of the one-launch pre-pass, 24 Mi
# with a mean, 32 Mi with scales and 42 Mi with both, and heads around its 8192: either way the same numbers as from the separate entry points
@pytest.mark.parametrize("B,H,Skv,D,blkk", [(1, 40, 512, 128, 64), (1, 40, 513, 128, 64), (1, 30, 1024, 64, 64), (1, 31, 1024, 64, 64),
                                            (1, 20, 1024, 64, 16), (1, 21, 1024, 64, 16), (64, 128, 3, 64, 64), (64, 129, 3, 64, 64),
                                            (16, 32, 128, 128, 16), (1, 8, 1024, 128, 64), (1, 8, 1025, 128, 64), (1, 56, 512, 128, 64),
                                            (1, 57, 512, 128, 64), (1, 102, 512, 128, 64), (1, 103, 512, 128, 64)])
@pytest.mark.parametrize("pv", ["fp16", "fp8"])
def test_limits_of_the_one_launch_prepass(B, H, Skv, D, blkk, pv):
    q, k, v = _inputs(B, H, H, 40, Skv, D, torch.float16, "HND", Skv + H)
    for smooth in (True, False):
        got = sa.sageattn(q, k, v, pv_mode=pv, smooth_k=smooth, BLKK=blkk)
        assert torch.equal(got, _steps(q, k, v, "HND", pv, 128, blkk, smooth))


@pytest.mark.parametrize("H,D,L", [(24, 64, 5461), (24, 64, 5462), (16, 128, 24575), (16, 128, 24577), (24, 64, 87381), (24, 64, 87382),
                                   (16, 64, 131073)])
def test_quantiser_walks_of_small_and_large_tensors(H, D, L):
    """Around 8 and 128 M elements, where the walk over the heads of a row changes, and rows 4 KiB apart: the same codes as from heads that lie
    apart."""
    g = torch.Generator(device="cuda").manual_seed(L)
    k = torch.randn((1, L, H, D), generator=g, device="cuda", dtype=torch.float16)
    t = k.transpose(1, 2).contiguous()
    _, _, got, scale = sa.per_block_int8(k[:, :16], k, BLKK=64, tensor_layout="NHD")
    _, _, want, want_scale = sa.per_block_int8(t[:, :, :16].contiguous(), t, BLKK=64)
    assert torch.equal(got.transpose(1, 2), want) and torch.equal(scale, want_scale)


def _cu(lens):
    return torch.tensor([0, *lens], dtype=torch.int64).cumsum(0).to(torch.int32).cuda()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("nseq,longest", [(1, 20000), (63, 900), (65, 5000), (1023, 70), (1024, 70), (1025, 70), (5000, 40)])
def test_plan_of_a_one_call_batch_equals_the_plan_on_its_own(nseq, longest, causal):
    """The plan that rides along with the statistics has 256 lanes and keeps 1024 lengths in LDS, the one of varlen_plan 1024 and 4096: the
    same block offsets and tile list, read back from the end of the call's workspace (empty sequences, other key than query lengths)."""
    g = torch.Generator().manual_seed(nseq)
    lq, lk = (torch.randint(0, longest + 1, (nseq,), generator=g).tolist() for _ in range(2))
    lq[0], lk[-1] = longest, longest
    cuq, cuk, Tq, Tk = _cu(lq), _cu(lk), sum(lq), sum(lk)
    q, k, v = (torch.randn((n, 2, 64), device="cuda", dtype=torch.float16) for n in (Tq, Tk, Tk))
    lib = _cabi.lib()
    need = lib.sage_sageattn_workspace_bytes_for(nseq, 2, 2, max(lq), max(lk), 64, 64, 16, _cabi.PV_FP16, Tq, Tk, 1, 1, 0, 0)
    out, ws = torch.empty_like(q), torch.empty(need, dtype=torch.uint8, device="cuda")
    row = (0, 64, 128)
    rc = lib.sage_sageattn(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), None, ws.data_ptr(), need, nseq, 2, 2, max(lq), max(lk),
                           64, *row, *row, *row, *row, 0, 64, 16, 0.125, int(causal), 1, _cabi.PV_FP16, cuq.data_ptr(), cuk.data_ptr(), Tq, Tk,
                           torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want, offs = sa.varlen_plan(cuq, cuk, Tq, 64, 16, is_causal=causal)
    ints = lib.sage_varlen_plan_ints(nseq, Tq)
    at = need - (4 * ints + 255) // 256 * 256   # the last region of a call without LSE
    got = ws[at:at + 4 * ints].view(torch.int32)
    used = offs[4] + int(want[offs[3]])
    assert torch.equal(got[:used], want[:used])


@pytest.mark.parametrize("pv", ["fp16", "fp8"])
@pytest.mark.parametrize("smooth", [True, False])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_packed_call_of_up_to_eight_chunks(D, dtype, pv, smooth):
    """No sequence past 4096 keys: the second launch combines the statistics itself, of nothing, a part of a chunk, one chunk and a row,
    and eight of them side by side; other key than query lengths."""
    lq, lk = [40, 0, 300, 33, 257, 64, 90], [0, 130, 1, 513, 4096, 512, 3500]
    cuq, cuk = _cu(lq), _cu(lk)
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn((n, h, D), generator=g).to(dtype).cuda() for n, h in ((sum(lq), 4), (sum(lk), 2), (sum(lk), 2)))
    k += 1.5
    got = sa.sageattn_varlen(q, k, v, cuq, cuk, max(lq), max(lk), pv_mode=pv, smooth_k=smooth)
    for i, (n, m) in enumerate(zip(lq, lk)):
        rows = slice(int(cuq[i]), int(cuq[i]) + n)
        keys = slice(int(cuk[i]), int(cuk[i]) + m)
        if n and m:
            one = sa.sageattn(q[None, rows], k[None, keys], v[None, keys], tensor_layout="NHD", pv_mode=pv, smooth_k=smooth)
            assert torch.equal(got[rows], one[0]), (n, m)
        else:
            assert not bool(got[rows].any())


@pytest.mark.parametrize("pv", ["fp16", "fp8"])
def test_packed_call_of_more_sequences_than_the_plan_keeps(pv):
    """1300 sequences, some of them empty, keys of other lengths: each kind of sequence equals the batch of its own, bit for bit."""
    g = torch.Generator().manual_seed(11)
    kinds = [(0, 5), (33, 0), (40, 7), (65, 130), (130, 33), (34, 600)]
    pick = torch.randint(0, len(kinds), (1300,), generator=g).tolist()
    lq, lk = [kinds[i][0] for i in pick], [kinds[i][1] for i in pick]
    cuq, cuk = _cu(lq), _cu(lk)
    q, k, v = (torch.randn((n, 2, 64), generator=g).half().cuda() for n in (sum(lq), sum(lk), sum(lk)))
    got = sa.sageattn_varlen(q, k, v, cuq, cuk, max(lq), max(lk), pv_mode=pv)
    for kind, (n, m) in enumerate(kinds):
        members = [i for i, p in enumerate(pick) if p == kind]
        if not n:
            continue
        rows = torch.stack([got[int(cuq[i]):int(cuq[i]) + n] for i in members])
        if not m:
            assert not bool(rows.any())
            continue
        part = lambda x, cu, length: torch.stack([x[int(cu[i]):int(cu[i]) + length] for i in members])  # noqa: E731
        one = sa.sageattn(part(q, cuq, n), part(k, cuk, m), part(v, cuk, m), tensor_layout="NHD", pv_mode=pv)
        assert torch.equal(rows, one), (n, m)
