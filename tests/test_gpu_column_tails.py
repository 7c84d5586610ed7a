"""Widths at which a lane's four (two) columns run past column N: rows of B and C that are aligned to a float only, the
last lane's columns shifted back over its neighbour's, a last slab of one column.  Integer operands, so every path must
equal the oracle bit for bit; C lies between guard floats that nothing may touch."""
import numpy as np
import pytest

from helpers import random_csr

pytestmark = pytest.mark.gpu

GUARD = 64


@pytest.mark.parametrize("N", [1, 2, 3, 5, 6, 7, 15, 17, 31, 33, 47, 63, 65, 67, 101, 127, 129, 131, 191, 255, 257, 259, 514, 1023])
def test_column_tails(cs, orc, torch_cuda, N):
    torch = torch_cuda
    rng = np.random.default_rng(900 + N)
    M, K = 96, 208
    rp, cl, vl = random_csr(rng, M, K, row_nnz=lambda r: 90 if r == 17 else 12 if r < 48 else 2, values="ints", empty_rows=(3, 95))
    B = rng.integers(-3, 4, (K, N)).astype(np.float32)
    ref = orc.spmm_csr(rp, cl, vl, B)
    h = cs.HRPB(M, K, rp, cl, vl)
    dB = torch.from_numpy(B).cuda()
    brick = dict(path=cs.PATH_BRICK, mfma_shape=1)
    plans = [dict(), dict(path=cs.PATH_ROWS), dict(path=cs.PATH_BRICK, mfma_shape=2), dict(brick, brick_groups=1), dict(brick, brick_groups=2),
             dict(brick, pipeline=2), dict(brick, pipeline=2, brick_groups=2), dict(brick, max_chunk_blocks=1), dict(mfma_shape=1, max_row_nnz=4),
             dict(mfma_shape=2, max_row_nnz=4), dict(brick, precision=cs.PREC_BF16X3)]
    for kw in plans:
        buf = torch.full((GUARD + M * N + GUARD,), float("nan"), device="cuda")
        dC = buf[GUARD:GUARD + M * N].view(M, N)
        plan = cs.SPMM_TC(h, N, **kw)
        plan.run(dB, dC)
        torch.cuda.synchronize()
        assert (dC.cpu().numpy() == ref).all(), (N, kw, plan.info)
        assert bool(torch.isnan(buf[:GUARD]).all()) and bool(torch.isnan(buf[GUARD + M * N:]).all()), (N, kw, plan.info)
    dC = torch.full((M, N), float("nan"), device="cuda")
    cs.csr_spmm_dev(2, h, dB, dC)
    assert (dC.cpu().numpy() == ref).all(), N
