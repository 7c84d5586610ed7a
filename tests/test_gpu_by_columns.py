"""Products whose B rows come from all over B: an XCD owns columns instead of rows (cute_dev::xcd_share), the row kernel walks
slabs of 32 or 64 columns, and the lists keep the panels the planner gives them.  Sizes on both sides of every line of that
rule: remainders of slabs, fewer slabs than XCDs, odd widths, rows of no entries, long and short rows, hub rows.

Tolerance: |difference| <= 2 * longest row * 2^-24 * sum |a||b|, the bound of two orders of one fp32 sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _product(cs, torch, rp, cl, vl, M, K, N, seed, **kw):
    rng = np.random.default_rng(seed)
    B = rng.standard_normal((K, N)).astype(np.float32)
    plan = cs.SPMM_TC(cs.HRPB(M, K, rp, cl, vl), N, **kw)
    out = torch.full((M, N), float("nan"), device="cuda")
    plan.run(torch.from_numpy(B).cuda(), out)
    return B, out.cpu().numpy(), plan


def _check(rp, cl, vl, B, out, M, N, rows, per_product=0.0):
    for r in rows:
        a, b = vl[rp[r]:rp[r + 1]].astype(np.float64), B[cl[rp[r]:rp[r + 1]]].astype(np.float64)
        bound = (2.0 * max(1, len(a)) * 2.0 ** -24 + per_product) * (np.abs(a) @ np.abs(b)) if len(a) else np.zeros(N)
        assert (np.abs(out[r] - (a @ b if len(a) else np.zeros(N))) <= bound + 1e-30).all(), r


def _random(M, K, per_row, seed, empty=0, hubs=0):
    rng = np.random.default_rng(seed)
    counts = np.full(M, per_row)
    if empty:
        counts[rng.integers(0, M, empty)] = 0
    if hubs:
        counts[:hubs] = 700
    rows = np.repeat(np.arange(M), counts)
    cols = rng.integers(0, K, rows.size)
    if hubs:
        cols = np.where(rng.random(rows.size) < 0.5, cols % 256, cols)
    key = np.unique(rows.astype(np.int64) * K + cols)
    rows, cols = key // K, (key % K).astype(np.uint32)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=M))]).astype(np.uint32)
    return rp, cols, rng.standard_normal(cols.size).astype(np.float32)


@pytest.mark.parametrize("M,K,per_row,N,empty,hubs,slabs", [
    (8192, 8192, 7, 256, 0, 0, (0, 8)), (8192, 16384, 5, 288, 500, 0, (0, 9)), (8192, 8192, 7, 301, 0, 0, (0, 5)),
    (8192, 8192, 9, 272, 40, 0, (0, 9)), (16384, 16384, 3, 128, 0, 0, (0, 4)), (16384, 32768, 4, 96, 900, 0, (0, 3)),
    (32768, 32768, 4, 64, 0, 0, (0, 2)), (8192, 8192, 26, 320, 0, 0, (0, 10)), (32768, 40000, 18, 64, 0, 0, (2, 0)),
    (16384, 36864, 17, 512, 0, 0, (16, 0)), (16384, 16384, 20, 299, 0, 0, (5, 0)), (16384, 16384, 6, 256, 100, 64, (4, 4)),
    (16384, 16384, 6, 310, 0, 64, (5, 0)), (131072, 131072, 6, 128, 0, 320, (2, 2)), (2048, 65536, 8, 544, 16, 0, (0, 17)),
    (16384, 16384, 4, 1056, 0, 0, (0, 33)), (8192, 2048, 20, 256, 0, 0, (0, 0))])
def test_every_element_is_written_once_and_right(cs, torch_cuda, M, K, per_row, N, empty, hubs, slabs):
    rp, cl, vl = _random(M, K, per_row, M + N, empty, hubs)
    B, out, plan = _product(cs, torch_cuda, rp, cl, vl, M, K, N, N)
    assert plan.column_slabs == slabs
    assert np.isfinite(out).all()
    rng = np.random.default_rng(1)
    _check(rp, cl, vl, B, out, M, N, np.unique(np.concatenate([[0, 1, 15, 16, M // 8, M // 2 - 1, M - 17, M - 1], rng.integers(0, M, 300)])))
    # every row, by its sum over the columns of B
    total = out.astype(np.float64) @ np.ones(N)
    want = np.zeros(M)
    rows = np.repeat(np.arange(M), np.diff(rp.astype(np.int64)))
    np.add.at(want, rows, vl.astype(np.float64) * (B.astype(np.float64) @ np.ones(N))[cl])
    scale = np.zeros(M)
    np.add.at(scale, rows, np.abs(vl.astype(np.float64)) * (np.abs(B.astype(np.float64)) @ np.ones(N))[cl])
    longest = max(1, int(np.diff(rp.astype(np.int64)).max()))
    assert (np.abs(total - want) <= 2.0 * longest * 2.0 ** -24 * scale + 1e-30).all()


@pytest.mark.parametrize("N", [64, 256, 320])
def test_forced_rows_give_the_bits_of_the_same_rows_in_row_order(cs, torch_cuda, N):
    """The row kernel adds a row up in storage order whatever slab it works on: a matrix whose window is scattered and the same
    rows against a B that repeats a short window give the same bits (the latter runs in row order)."""
    M, K, short = 8192, 32768, 512
    rng = np.random.default_rng(7)
    cl = np.sort(rng.permuted(np.tile(np.arange(short), (M, 1)), axis=1)[:, :9], axis=1).astype(np.uint32)
    far = cl + np.uint32(K - short) * (np.arange(9) >= 5).astype(np.uint32)
    rp, vl = (np.arange(M + 1) * 9).astype(np.uint32), rng.standard_normal(M * 9).astype(np.float32)
    piece = rng.standard_normal((short, N)).astype(np.float32)
    B = np.zeros((K, N), np.float32)
    B[:short] = piece
    B[K - short:] = piece
    outs = []
    for cols in (cl, far):
        plan = cs.SPMM_TC(cs.HRPB(M, K, rp, cols.ravel(), vl), N, path=cs.PATH_ROWS)
        out = torch_cuda.full((M, N), float("nan"), device="cuda")
        plan.run(torch_cuda.from_numpy(B).cuda(), out)
        assert (plan.column_slabs[1] > 0) == (cols is far), plan.column_slabs
        outs.append(out)
    assert torch_cuda.equal(outs[0], outs[1])


ROLLING, PIPELINED, BF16 = dict(mfma_shape=1), dict(mfma_shape=1, pipeline=2), dict(precision=1)


@pytest.mark.parametrize("M,K,per_row,N,hubs,options,kernel,slabs", [
    (8192, 8192, 20, 256, 0, ROLLING, "hrpb_brick_f32_rolling", (4, 0)), (8192, 8192, 20, 301, 0, ROLLING, "hrpb_brick_f32_rolling", (5, 0)),
    (8192, 8192, 20, 256, 0, PIPELINED, "hrpb_brick_f32", (2, 0)), (8192, 8192, 20, 600, 0, PIPELINED, "hrpb_brick_f32", (5, 0)),
    (8192, 16384, 20, 256, 0, BF16, "hrpb_brick_bf16x3", (4, 0)), (8192, 16384, 20, 320, 0, BF16, "hrpb_brick_bf16x3", (5, 0)),
    (16384, 16384, 6, 256, 64, ROLLING, "hrpb_brick_rows_f32", (4, 1)), (16384, 16384, 6, 260, 64, ROLLING, "hrpb_brick_rows_f32", (5, 2)),
    (16384, 16384, 6, 301, 64, ROLLING, "hrpb_brick_rows_f32", (5, 2)), (16384, 16384, 6, 260, 64, PIPELINED, "hrpb_brick_f32", (5, 2)),
    (16384, 16384, 6, 512, 64, BF16, "hrpb_brick_bf16x3", (8, 2)), (8192, 2048, 20, 256, 0, ROLLING, "hrpb_brick_f32_rolling", (0, 0)),
    # two slabs of 128 columns and a remainder: row order, unless an fp32 graph's panels share columns; three whole slabs: by columns
    (32768, 32768, 24, 300, 0, ROLLING, "hrpb_brick_f32_rolling", (0, 0)), (32768, 32768, 24, 300, 0, BF16, "hrpb_brick_bf16x3", (0, 0)),
    (32768, 32768, 24, 256, 0, BF16, "hrpb_brick_bf16x3", (2, 0)), (32768, 32768, 24, 640, 0, ROLLING, "hrpb_brick_f32_rolling", (5, 0)),
    # the rows beside bf16x3 bricks: a slab of 256 columns and a remainder
    (16384, 16384, 6, 260, 64, BF16, "hrpb_brick_bf16x3", (5, 0))])
def test_bricks(cs, torch_cuda, M, K, per_row, N, hubs, options, kernel, slabs):
    """The brick kernels by columns: alone, beside rows in one launch and in two, whole slabs and remainders, and once in row order;
    bf16x3 drops at most 2^-15 of each product on top of the bound."""
    rp, cl, vl = _random(M, K, per_row, M + N, 100 if hubs else 0, hubs)
    B, out, plan = _product(cs, torch_cuda, rp, cl, vl, M, K, N, N, path=cs.PATH_AUTO if hubs else cs.PATH_BRICK, **options)
    assert plan.kernel_name == kernel and plan.column_slabs == slabs, (plan.kernel_name, plan.column_slabs, plan.info)
    assert np.isfinite(out).all()
    rng = np.random.default_rng(1)
    rows = np.unique(np.concatenate([np.arange(80), [M // 8, M // 2 - 1], np.arange(M - 40, M), rng.integers(0, M, 400)]))
    _check(rp, cl, vl, B, out, M, N, rows, 2.0 ** -15 if plan.info["precision"] else 0.0)


@pytest.mark.parametrize("M,per_row,N,kernel,slabs", [
    (20000, 10, 301, "hrpb_quad_f32", (5, 0)), (20000, 10, 600, "csr_rows_batched", (0, 0)), (24000, 4, 264, "hrpb_quad_f32", (0, 0)),
    (30000, 4, 264, "hrpb_quad_f32", (0, 0)), (30000, 4, 301, "csr_rows_batched", (0, 0)), (30000, 20, 257, "hrpb_quad_f32", (0, 0)),
    (30000, 20, 301, "hrpb_quad_f32", (5, 0)), (40000, 10, 496, "hrpb_quad_f32", (0, 0)), (40000, 10, 600, "csr_rows_batched", (0, 0)),
    (65536, 4, 272, "hrpb_quad_f32", (0, 0)), (65536, 4, 296, "csr_rows_batched", (0, 0))])
def test_lists_or_rows_off_the_grid_of_B(cs, torch_cuda, M, per_row, N, kernel, slabs):
    """Widths off 128 bytes, both sides of the lines between the lists and the row kernel (its last walk over few columns), and of
    the remainder that lists by columns take."""
    rp, cl, vl = _random(M, M, per_row, M + N)
    B, out, plan = _product(cs, torch_cuda, rp, cl, vl, M, M, N, N)
    assert (plan.kernel_name, plan.column_slabs) == (kernel, slabs), (plan.kernel_name, plan.column_slabs)
    assert np.isfinite(out).all()
    _check(rp, cl, vl, B, out, M, N, np.unique(np.concatenate([np.arange(40), np.arange(M - 40, M), np.random.default_rng(1).integers(0, M, 300)])))


def test_a_dense_graph_in_row_order_keeps_its_lists(cs, torch_cuda):
    """131 072 nodes: the rule that moves panels with little reuse to the row kernel holds for 24 entries a row only by columns."""
    for per_row, N, many in ((12, 208, False), (12, 256, True), (8, 208, True)):
        A = cs.gen_matrix(4, 5, 17, per_row, 0)
        rp, cl, vl = np.array(A.rowPtr), np.array(A.cols), np.array(A.vals)
        B, out, plan = _product(cs, torch_cuda, rp, cl, vl, A.M, A.K, N, N)
        assert (plan.info["numRowPanelsSparse"] > 5500) == many, (per_row, N, plan.info)
        assert np.isfinite(out).all()
        _check(rp, cl, vl, B, out, A.M, N, np.unique(np.concatenate([np.arange(40), np.random.default_rng(1).integers(0, A.M, 200)])))


@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("M,K,per_row,N,cut", [(32768, 40000, 20, 64, 0), (32768, 40000, 24, 96, 3), (16384, 49152, 28, 288, 0),
                                                (16384, 65536, 32, 512, 2), (32768, 90112, 16, 128, 1)])
def test_lists_on_slabs_of_32_columns(cs, torch_cuda, layout, M, K, per_row, N, cut):
    """Both kinds of list, whole panels and panels cut into pieces; rows of whole multiples of the list unit fill their slots."""
    rng = np.random.default_rng(N)
    cl = np.sort(rng.integers(0, K // per_row, (M, per_row)) + np.arange(per_row) * (K // per_row), axis=1).astype(np.uint32)
    rp, vl = (np.arange(M + 1) * per_row).astype(np.uint32), rng.standard_normal(M * per_row).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    h = cs.HRPB(M, K, rp, cl.ravel(), vl)
    h.upload(quad_layout=layout)
    plan = cs.SPMM_TC(h, N, max_chunk_blocks=cut)
    out, again = (torch_cuda.full((M, N), float("nan"), device="cuda") for _ in range(2))
    dB = torch_cuda.from_numpy(B).cuda()
    plan.run(dB, out)
    plan.run(dB, again)
    assert plan.kernel_name == "hrpb_quad_half_f32" and (plan.info["numAtomicChunks"] > 0) == (cut > 0), plan.info
    assert torch_cuda.equal(out, again)
    _check(rp, cl.ravel(), vl, B, out.cpu().numpy(), M, N, np.unique(np.concatenate([np.arange(40), np.arange(M - 40, M), rng.integers(0, M, 300)])))
