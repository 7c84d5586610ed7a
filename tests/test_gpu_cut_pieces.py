"""Panels and strips that were cut: the pieces add themselves up inside the launch (cute_spmm_run, cute_spmm_run_static) or a second
launch does (cute_spmm_run_scratch).  Both add eight consecutive pieces and then the sums of the eights, so they must agree bit for bit,
run after run; on small integers, whose sums are exact in any order, all must equal the oracle."""
import numpy as np
import pytest

from helpers import random_csr

pytestmark = pytest.mark.gpu

BERR = 2e-6


def _plans(cs):
    brick = dict(path=cs.PATH_BRICK, mfma_shape=1)
    quad = dict(path=cs.PATH_BRICK, mfma_shape=2)
    return [dict(quad, max_chunk_blocks=1), dict(brick, max_chunk_blocks=1), dict(brick, max_chunk_blocks=1, brick_groups=1),
            dict(brick, max_chunk_blocks=1, brick_groups=2), dict(brick, max_chunk_blocks=1, pipeline=2),
            dict(brick, max_chunk_blocks=1, precision=cs.PREC_BF16X3), dict(quad, max_chunk_blocks=3),
            dict(mfma_shape=2, max_row_nnz=8, max_chunk_blocks=1), dict(mfma_shape=1, max_row_nnz=8, max_chunk_blocks=1)]


@pytest.mark.parametrize("quad_layout", [1, 2])
@pytest.mark.parametrize("pieces,N", [(1, 64), (2, 33), (8, 64), (9, 4), (16, 130), (17, 1), (64, 47), (65, 128), (130, 70)])
def test_pieces_add_up_alike(cs, orc, torch_cuda, pieces, N, quad_layout):
    torch = torch_cuda
    rng = np.random.default_rng(40 * pieces + N)
    M, K = 80, max(16 * pieces, 48)
    for values in ("normal", "ints"):
        rp, cl, vl = random_csr(rng, M, K, row_nnz=lambda r: 16 * pieces if r in (5, 37) else 3, values=values, empty_rows=(0, 79))
        B = (rng.standard_normal((K, N)) if values == "normal" else rng.integers(-3, 4, (K, N))).astype(np.float32)
        ref = orc.spmm_csr(rp, cl, vl, B)
        dB = torch.from_numpy(B).cuda()
        d = cs.DeviceHRPB(M, K, *(torch.from_numpy(x if x.dtype == np.float32 else x.view(np.int32)).cuda() for x in (rp, cl, vl)), quad_layout=quad_layout)
        for kw in _plans(cs):
            plan = cs.SPMM_TC(d, N, **kw)
            assert pieces < 3 or plan.info["numAtomicChunks"] >= pieces // 3, (kw, plan.info)
            scratch = torch.full((max(plan.scratch_bytes, 16) // 4,), float("nan"), device="cuda")
            outs = []
            for call in (plan.run, plan.run, plan.run_static, plan.run, plan.run_static, lambda b, c: plan.run_scratch(b, c, scratch)):
                dC = torch.full((M, N), float("nan"), device="cuda")
                call(dB, dC)
                outs.append(dC.cpu().numpy())
            assert all(o.tobytes() == outs[0].tobytes() for o in outs), (kw, plan.info)
            if values == "ints":
                assert (outs[0] == ref).all(), (kw, plan.info)
            elif plan.info["precision"] == cs.PREC_FP32:
                assert cs.backward_error(rp, cl, vl, B, ref, outs[0]) <= BERR, (kw, plan.info)


def test_pieces_in_a_graph(cs, torch_cuda):
    """Replays find the counters as the launch before left them, with eager calls between them."""
    torch = torch_cuda
    A = cs.gen_matrix(4, 7, 12, 8, 0)
    N = 48
    plan = cs.SPMM_TC(cs.HRPB(A.M, A.K, A.rowPtr, A.cols, A.vals), N)
    assert plan.info["numAtomicChunks"] > 16
    dB, dC = torch.randn(A.K, N, device="cuda"), torch.empty(A.M, N, device="cuda")
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    plan.run(dB, dC)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        plan.run(dB, dC, stream=stream)
    for _ in range(4):
        dB.normal_()
        eager = torch.empty_like(dC)
        plan.run(dB, eager)
        dC.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(eager, dC)


@pytest.mark.parametrize("pieces,N", [(9, 5), (20, 6), (9, 24), (17, 27), (9, 65), (9, 66), (17, 67), (70, 68), (9, 129), (17, 131), (9, 257)])
def test_vectors_at_the_last_columns(cs, orc, torch_cuda, pieces, N):
    """Tiles travel by vectors of two and four columns.  A vector that would pass the last column is moved back over columns of the lane, the column group
    or the slab before it: only what is its own may be written, or sums that stand in a first tile already count twice."""
    test_pieces_add_up_alike(cs, orc, torch_cuda, pieces, N, 1)
