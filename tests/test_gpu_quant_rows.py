"""The quantiser at the edges of its row partition: a workgroup takes 64 or 128 rows, a wavefront 16 or 32 of them, a pass of a
wavefront 8 or 16 (head_dim 128 / 64), and a scale block spans 1, 2 or 4 wavefronts."""
import numpy as np
import pytest
import torch

import baselinebenchmark_amd as sa
from oracle import quant as oq
from tests.helpers import randn


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("blk", [16, 32, 64, 128])
@pytest.mark.parametrize("dtype,layout", [(torch.float16, "NHD"), (torch.bfloat16, "HND")])
def test_row_partition_edges_bit_exact(D, blk, dtype, layout):
    """One row, one less and one more than a pass, a wavefront, a workgroup and two workgroups: int8 values, scales and K mean equal
    the oracle's bit for bit."""
    for rows in (1, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 257):
        g = torch.Generator().manual_seed(rows * 131 + D + blk)
        q, k = randn(layout, 1, 2, rows, D, dtype, g), randn(layout, 1, 2, rows, D, dtype, g, offset_std=2.0)
        km = oq.k_mean(k, layout)
        kw = dict(BLKQ=blk, BLKK=blk, tensor_layout=layout)
        want = oq.per_block_int8(q, k, km=km, **kw)
        got = sa.per_block_int8(q.cuda(), k.cuda(), km=km.cuda(), **kw)
        for name, a, b in zip(("q_int8", "q_scale", "k_int8", "k_scale"), got, want):
            assert torch.equal(a.cpu(), b), f"{name}, {rows} rows: {(a.cpu() != b).sum().item()} mismatches"


def test_quotient_through_binary64_reciprocal_is_correctly_rounded():
    """The path for divisors that the binary32 correction step does not cover multiplies by RN64(1/s) and narrows once: equal to the
    true binary32 quotient for all-ones significands, for divisors past 1e30 and for every residue class in between."""
    rng = np.random.default_rng(7)
    s = np.concatenate([(rng.integers(60, 250, 4096).astype(np.uint32) << 23 | 0x7FFFFF).view(np.float32),
                        (rng.random(4096) * 1e38 + 1e30).astype(np.float32), np.exp(rng.uniform(-27, 27, 4096)).astype(np.float32)])
    for _ in range(50):
        x = (s.astype(np.float64) * rng.uniform(-127.5, 127.5, s.size)).astype(np.float32)
        with np.errstate(over="ignore"):
            got = (x.astype(np.float64) * (1.0 / s.astype(np.float64))).astype(np.float32)
        normal = np.abs(got) >= np.finfo(np.float32).tiny
        assert np.array_equal(got[normal], (x / s)[normal])
