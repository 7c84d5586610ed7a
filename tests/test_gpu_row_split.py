"""Products of a few columns: lane groups share a row (csr_rows_split).  Widths of every lane size and of lanes that share columns, rows shorter
than a group, as long as what the groups hold at a time and longer, empty ones; the route, and values that are not finite beside what a row reads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(rng, K, lengths):
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    cl = np.concatenate([np.sort(rng.choice(K, n, replace=False)) for n in lengths]).astype(np.uint32)
    return rp, cl, rng.integers(-4, 5, cl.size).astype(np.float32)


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("lengths,parts", [((24,) * 16, 4), ((27, 28, 29, 28), 8), ((32,) * 4, 8), ((0, 1, 55, 56, 57, 64, 65, 128, 80, 60), 16),
                                           ((16, 17, 18, 90, 40, 0), 8), ((23,) * 8, 1), ((24,) * 9 + (150,), 1)])
def test_against_the_oracle(cs, orc, torch_cuda, lengths, parts, N):
    torch, rng = torch_cuda, np.random.default_rng(N + sum(lengths))
    K, M = 160, 48 * len(lengths)
    rp, cl, vl = _rows(rng, K, lengths * 48)
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    unused = np.setdiff1d(np.arange(K), cl)
    B[unused] = np.inf
    plan = cs.SPMM_TC(cs.HRPB(M, K, rp, cl, vl), N)
    assert plan.row_parts == (parts if N <= 8 else 1), (plan.row_parts, vl.size / M)
    if plan.row_parts > 1:
        assert plan.kernel_name == "csr_rows_split" and plan.info["numChunks"] == 0
    C = torch.full((M, N), float("nan"), device="cuda")
    plan.run(torch.from_numpy(B).cuda(), C)
    assert np.array_equal(C.cpu().numpy(), orc.spmm_csr(rp, cl, vl, B))       # whole numbers: exact in any order


def test_padding_reads_nothing_and_rows_are_written_once(cs, orc, torch_cuda):
    """A row's last turn asks for its last entry again: an infinity there counts once, and the rows beside it stay finite."""
    torch, rng = torch_cuda, np.random.default_rng(1)
    K, M, N = 64, 32, 3
    rp, cl, vl = _rows(rng, K, (30,) * M)
    vl[:] = 1.0
    B = np.ones((K, N), np.float32)
    B[cl[29]] = np.inf                                     # the last column of row 0
    C = torch.full((M, N), float("nan"), device="cuda")
    plan = cs.SPMM_TC(cs.HRPB(M, K, rp, cl, vl), N)
    assert plan.row_parts == 8
    plan.run(torch.from_numpy(B).cuda(), C)
    assert np.array_equal(C.cpu().numpy(), orc.spmm_csr(rp, cl, vl, B))


@pytest.mark.parametrize("kind,rows,per_row,span,N,parts", [(5, 16000, 24, 400, 8, 4), (5, 64000, 24, 400, 8, 1), (5, 64000, 24, 400, 4, 4), (5, 32000, 32, 400, 7, 8), (5, 32000, 32, 2048, 7, 1),
                                                            (5, 64000, 48, 400, 3, 1), (5, 128000, 24, 2048, 4, 1), (5, 64000, 24, 2048, 2, 4), (1, 64000, 32, 0, 1, 1), (1, 16000, 32, 0, 1, 8),
                                                            (5, 128000, 32, 400, 8, 8), (5, 96000, 48, 400, 6, 1),
                                                            (5, 64000, 32, 400, 8, 8), (5, 72000, 30, 800, 4, 8), (1, 64000, 24, 0, 5, 4), (1, 64000, 24, 0, 2, 4)])
def test_the_route_over_the_sizes(cs, orc, torch_cuda, kind, rows, per_row, span, N, parts):
    """Groups share rows while the launch leaves slots free, or from four million entries on; in between it depends on the lanes and on shared columns."""
    torch = torch_cuda
    A = cs.gen_matrix(kind, 5, rows, per_row, span)
    vals = (np.arange(len(A.vals)) % 7 - 3).astype(np.float32)
    plan = cs.SPMM_TC(cs.HRPB(A.M, A.K, A.rowPtr, A.cols, vals), N)
    assert plan.row_parts == parts
    B = np.random.default_rng(N).integers(-4, 5, (A.K, N)).astype(np.float32)
    C = torch.full((A.M, N), float("nan"), device="cuda")
    plan.run(torch.from_numpy(B).cuda(), C)
    assert np.array_equal(C.cpu().numpy(), orc.spmm_csr(A.rowPtr, A.cols, vals, B))
