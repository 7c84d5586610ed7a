"""The brick kernel's slab follows the number of work items (128, 64, 32 or 16 columns): the widths at which each is taken, their
remainders, and the reduced-precision kernel, which has no slab below 64 columns.

Tolerance: |difference| <= 2 * longest row * 2^-24 * sum |a||b| (fp32 in any order); bf16x3 drops at most 2^-15 of each product
on top of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,N,slab,bf16", [
    (56, 64, 16, False), (56, 47, 16, False), (56, 301, 16, False), (400, 47, 16, False), (400, 64, 16, False), (400, 130, 32, False), (400, 200, 16, False),
    (800, 64, 32, False), (800, 66, 32, False), (400, 96, 16, False), (800, 96, 32, False), (400, 256, 64, False),
    (1600, 300, 64, False), (4000, 128, 64, False), (4000, 101, 64, False), (8000, 128, 128, False), (12000, 300, 128, False),
    (400, 64, 64, True), (400, 128, 64, True), (400, 300, 64, True), (8000, 128, 128, True)])
def test_slab_and_product(cs, torch_cuda, size, N, slab, bf16):
    A = cs.gen_matrix(3, 11, size, 60)
    assert (6 * size) % 16 == 0                    # the format takes whole panels
    rp, cl, vl = np.array(A.rowPtr).astype(np.int64), np.array(A.cols), np.array(A.vals)
    rng = np.random.default_rng(N)
    B = rng.standard_normal((A.K, N)).astype(np.float32)
    plan = cs.SPMM_TC(cs.HRPB(A.M, A.K, A.rowPtr, A.cols, A.vals), N, path=cs.PATH_BRICK, mfma_shape=0 if bf16 else 1,
                      precision=cs.PREC_BF16X3 if bf16 else cs.PREC_FP32)
    assert plan.info["mfmaShape"] == 1 and plan.info["slabWidth"] == slab, plan.info
    out = torch_cuda.full((A.M, N), float("nan"), device="cuda")
    plan.run(torch_cuda.from_numpy(B).cuda(), out)
    out = out.cpu().numpy()
    assert np.isfinite(out).all()
    for r in np.unique(np.concatenate([np.arange(0, 40), np.arange(A.M - 40, A.M), rng.integers(0, A.M, 200)])):
        a, b = vl[rp[r]:rp[r + 1]].astype(np.float64), B[cl[rp[r]:rp[r + 1]]].astype(np.float64)
        bound = (2.0 * len(a) * 2.0 ** -24 + (2.0 ** -15 if bf16 else 0.0)) * (np.abs(a) @ np.abs(b))
        assert (np.abs(out[r] - a @ b) <= bound).all(), r


@pytest.mark.parametrize("bf16,N,slab", [(True, 300, 128), (True, 320, 128), (True, 256, 64), (False, 300, 64)])
def test_slab_of_a_graph_beyond_the_cache(cs, torch_cuda, bf16, N, slab):
    """400 panels with one long row each among row panels, operands of more than 256 MB: in bf16x3 the slab stays wide (up to 256 columns
    the operands fit the cache)."""
    M, hubs, per_row, long_row = 131072, 400, 3, 300
    rng = np.random.default_rng(N)
    counts = np.full(M, per_row)
    counts[np.arange(hubs) * 16] = long_row
    rows = np.repeat(np.arange(M), counts)
    key = np.unique(rows * np.int64(M) + rng.integers(0, M, rows.size))
    rows, cl = key // M, (key % M).astype(np.uint32)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=M))]).astype(np.uint32)
    vl = rng.standard_normal(cl.size).astype(np.float32)
    B = rng.standard_normal((M, N), dtype=np.float32)
    plan = cs.SPMM_TC(cs.HRPB(M, M, rp, cl, vl), N, mfma_shape=0 if bf16 else 1, precision=cs.PREC_BF16X3 if bf16 else cs.PREC_FP32)
    assert plan.info["numBrickPanels"] == hubs and plan.info["mfmaShape"] == 1 and plan.info["slabWidth"] == slab, plan.info
    out = torch_cuda.full((M, N), float("nan"), device="cuda")
    plan.run(torch_cuda.from_numpy(B).cuda(), out)
    assert bool(torch_cuda.isfinite(out).all())
    for r in np.unique(np.concatenate([np.arange(0, 40), np.arange(16 * hubs - 20, 16 * hubs + 20), np.arange(M - 20, M)])):
        a, b = vl[rp[r]:rp[r + 1]].astype(np.float64), B[cl[rp[r]:rp[r + 1]]].astype(np.float64)
        bound = (2.0 * max(1, len(a)) * 2.0 ** -24 + (2.0 ** -15 if bf16 else 0.0)) * (np.abs(a) @ np.abs(b))
        assert (np.abs(out[r].cpu().numpy() - a @ b) <= bound + 1e-30).all(), r
