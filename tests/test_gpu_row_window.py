"""Rows whose columns move along with them: their window of B slides through LDS (csr_rows_window).  Sizes around a tile of 1 024 rows,
a slice of 64 and a slab of 8 or 16 columns, windows on both sides of the two rings (2 560 and 5 120 rows of B) and windows that
jump, rows of every length, and rows of B that are not finite.

Whole numbers: the sums are exact whatever their order, so the results are compared bit for bit with the oracle, and with the row
kernel that gathers from memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _band(M, K, counts, reach, seed, start=None):
    """counts[r] distinct columns of row r, within `reach` columns from start[r] on."""
    rng = np.random.default_rng(seed)
    start = np.clip(np.arange(M) - reach // 2, 0, K - reach) if start is None else start
    counts = np.broadcast_to(counts, M)
    step = reach // max(1, counts.max())
    cols = start[:, None] + np.arange(counts.max()) * step + rng.integers(0, step, (M, counts.max()))
    cols[::1024, 0] = start[::1024]                               # the ends of a tile's window are taken
    cols[1023::1024, -1] = start[1023::1024] + reach - 1
    keep = np.arange(counts.max())[None, :] >= counts.max() - counts[:, None]
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    cl = cols[keep].astype(np.uint32)
    return rp, cl, rng.integers(-8, 9, cl.size).astype(np.float32)


def _check(cs, orc, torch, rp, cl, vl, M, K, N, columns, B=None):
    B = np.random.default_rng(N).integers(-8, 9, (K, N)).astype(np.float32) if B is None else B
    h = cs.DeviceHRPB(M, K, *(torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda() for a in (rp, cl, vl)))
    plan = cs.SPMM_TC(h, N, operand_residency=2)
    assert plan.window_columns == columns and plan.info["numChunks"] == 0
    assert plan.kernel_name == ("csr_rows_window" if columns else "csr_rows_batched")
    C = torch.full((M * N + 64,), 7.5, device="cuda")
    out = C[:M * N].view(M, N)
    dB = torch.from_numpy(B).cuda()
    for _ in range(2):                                            # a second pass starts from the first one's LDS
        plan.run(dB, out)
    assert (C[M * N:] == 7.5).all()
    rows = torch.empty(M, N, device="cuda")
    cs.SPMM_TC(h, N, path=cs.PATH_ROWS).run(dB, rows)
    assert np.array_equal(out.cpu().numpy(), rows.cpu().numpy(), equal_nan=True)
    if np.isfinite(B).all():
        assert np.array_equal(out.cpu().numpy(), orc.spmm_csr(rp, cl, vl, B))


@pytest.mark.parametrize("M,per_row,reach,N,columns", [
    (65536, 32, 4097, 256, 8), (65536 + 16, 32, 1500, 256, 16), (60 * 1024 - 16, 31, 1000, 301, 16), (61440 + 64, 30, 3000, 203, 8),
    (131072, 45, 700, 33, 16), (260000, 40, 1200, 16, 16), (400000, 40, 4000, 17, 8), (9 * 1024 + 48, 48, 1537, 1000, 16),
    (65536, 32, 1538, 256, 8), (65536, 32, 4098, 256, 0),
    (163840 + 48, 32, 4097, 301, 8), (200000, 24, 1400, 256, 16)])      # operands of more than 256 MiB, chains of several tiles: B is asked for ahead
def test_whole_numbers(cs, orc, torch_cuda, M, per_row, reach, N, columns):
    rp, cl, vl = _band(M, M, per_row, reach, M + N)
    _check(cs, orc, torch_cuda, rp, cl, vl, M, M, N, columns)


def test_rows_of_every_length(cs, orc, torch_cuda):
    M, N = 81920, 256
    counts = np.repeat(np.tile(np.concatenate([np.arange(20, 49), [0, 48, 47]]), M // 32 // 64 + 1), 64)[:M]
    counts[5::64] = 0
    counts[7::64] -= counts[7::64] // 4                           # rows of a slice differ
    rp, cl, vl = _band(M, M, counts, 1200, 3)
    _check(cs, orc, torch_cuda, rp, cl, vl, M, M, N, 16)


@pytest.mark.parametrize("jump,reach", [(3000, 500), (40000, 1500)])
def test_windows_that_jump_and_rectangles(cs, orc, torch_cuda, jump, reach):
    """Every 8 192 rows the window moves on by `jump` columns, most of which no row reads."""
    M, N = 65536, 256
    K = M + 8 * jump
    start = np.minimum(np.arange(M) // 1024 * 1024 + np.arange(M) // 8192 * jump, K - reach)
    rp, cl, vl = _band(M, K, 32, reach, jump, start)
    _check(cs, orc, torch_cuda, rp, cl, vl, M, K, N, 16)


@pytest.mark.parametrize("empty", [[(0, 2048)], [(30 * 1024, 32 * 1024)], [(79 * 1024 - 300, 81920 + 48)], [(0, 16), (1024, 2064), (5000, 9000), (70000, 80000)]])
def test_tiles_without_entries(cs, orc, torch_cuda, empty):
    """The windows of tiles come from the census, one pair a tile: none of the rows of a tile, or of its panels at either end, may hold an entry."""
    M, N = 81920 + 48, 256
    counts = np.full(M, 40)
    for a, b in empty:
        counts[a:b] = 0
    rp, cl, vl = _band(M, M, counts, 1200, len(empty))
    _check(cs, orc, torch_cuda, rp, cl, vl, M, M, N, 16)


def test_rows_of_b_that_are_not_finite(cs, orc, torch_cuda):
    """An infinity reaches the rows that refer to it and no other: padding is left out, not multiplied by zero."""
    M, N = 65536, 256
    counts = np.full(M, 32)
    counts[3::5] = 29
    rp, cl, vl = _band(M, M, counts, 900, 11)
    vl[vl == 0] = 1.0
    B = np.random.default_rng(1).integers(1, 9, (M, N)).astype(np.float32)
    B[::1000] = np.inf
    B[500::1000, ::3] = np.nan
    _check(cs, orc, torch_cuda, rp, cl, vl, M, M, N, 16, B)


@pytest.mark.parametrize("M,per_row,reach,N,columns", [(65536, 32, 4097, 256, 0), (80000, 30, 400, 101, 0), (200000, 12, 1400, 256, 0), (1048576, 32, 4097, 256, 8)])
def test_a_plan_for_one_product(cs, torch_cuda, M, per_row, reach, N, columns):
    """The lead has to pay for the second form of the entries, unless the caller says that the product runs in a loop."""
    rp, cl, vl = _band(M, M, per_row, reach, M)
    h = cs.DeviceHRPB(M, M, *(torch_cuda.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda() for a in (rp, cl, vl)))
    assert cs.SPMM_TC(h, N).window_columns == columns
    if columns == 0 and M < 200000:
        assert cs.SPMM_TC(h, N, operand_residency=2).window_columns != 0
