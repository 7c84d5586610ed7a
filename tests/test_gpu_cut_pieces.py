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


@pytest.mark.parametrize("lg,edges,N", [(15, 11, 96), (16, 7, 80), (16, 9, 100)])
def test_lists_of_two_slabs(cs, orc, torch_cuda, lg, edges, N):
    """Lists of two column slabs are cut by a rule of their own, with up to twelve groups a share (the first two) and beyond."""
    torch = torch_cuda
    A = cs.gen_matrix(4, 5, lg, edges, 0)
    vals = (np.arange(len(A.vals)) % 7 - 3).astype(np.float32)
    plan = cs.SPMM_TC(cs.HRPB(A.M, A.K, A.rowPtr, A.cols, vals), N)
    assert "quad" in plan.kernel_name and plan.info["numAtomicChunks"] >= 500, plan.info
    B = np.random.default_rng(lg).integers(-3, 4, (A.K, N)).astype(np.float32)
    ref, dB = orc.spmm_csr(A.rowPtr, A.cols, vals, B), torch.from_numpy(B).cuda()
    scratch = torch.full((plan.scratch_bytes // 4,), float("nan"), device="cuda")
    for call in (plan.run, plan.run_static, lambda b, c: plan.run_scratch(b, c, scratch)):
        dC = torch.full((A.M, N), float("nan"), device="cuda")
        call(dB, dC)
        assert (dC.cpu().numpy() == ref).all()


def test_coarser_cut_where_the_finer_ones_tiles_do_not_fit(cs, orc, torch_cuda):
    """2 016 panels of 65 list groups, 16 a share: cut at four shares into twos they come in three, of which a limit of 20 groups makes six, 47 MiB of tiles at
    N = 64; cut at six shares the limit alone cuts them, into four, 31.5 MiB, which cute_spmm_run_static takes."""
    torch = torch_cuda
    if torch.cuda.get_device_properties(0).multi_processor_count != 256: pytest.skip("the sizes are those of 256 compute units")
    rng = np.random.default_rng(3)
    panels, groups, N, K = 2016, 65, 64, 4096
    M = 16 * panels
    # a group of a panel's list takes four columns of each quad of rows: the panel's columns all stand in the first row of each quad
    cols = np.stack([np.sort(rng.choice(K, 4 * groups, replace=False)) for _ in range(panels)]).astype(np.uint32)
    lengths = np.where(np.arange(M) % 4 == 0, 4 * groups, 0)
    rp = np.concatenate(([0], np.cumsum(lengths))).astype(np.uint32)
    cl = np.repeat(cols, 4, axis=0).reshape(-1)
    vl = rng.integers(1, 4, len(cl)).astype(np.float32)
    d = cs.DeviceHRPB(M, K, *(torch.from_numpy(x if x.dtype == np.float32 else x.view(np.int32)).cuda() for x in (rp, cl, vl)), quad_layout=1)
    plan = cs.SPMM_TC(d, N, path=cs.PATH_BRICK, mfma_shape=2, max_chunk_blocks=20)
    assert plan.info["numAtomicChunks"] == 4 * panels and plan.scratch_bytes == 4 * panels * 16 * N * 4, plan.info
    B = rng.integers(-3, 4, (K, N)).astype(np.float32)
    dB, dC = torch.from_numpy(B).cuda(), torch.full((M, N), float("nan"), device="cuda")
    plan.run_static(dB, dC)
    assert (dC.cpu().numpy() == orc.spmm_csr(rp, cl, vl, B)).all()
