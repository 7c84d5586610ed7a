"""The row kernel takes a batch of eight entries a round also where a lane group has fewer lanes than that (N <= 16), several
consecutive entries in each lane: rows of every length around a round, the next row's entries never part of a sum.

Whole numbers: the sums are exact, so the results are compared bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 7, 8, 9, 13, 16, 20])
def test_rows_of_every_length_and_values_that_are_not_numbers(cs, torch_cuda, N):
    rng = np.random.default_rng(N)
    K = 256
    counts = np.concatenate([np.arange(0, 34), rng.permutation(np.arange(0, 34)), [63, 64, 65, 128], rng.integers(0, 12, 184)])
    M = counts.size
    assert M == 256
    cols = np.concatenate([np.sort(rng.permutation(K)[:n]) for n in counts]).astype(np.uint32)
    vals = rng.integers(-8, 9, cols.size).astype(np.float32)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    bad = [r for r in range(1, M, 5) if counts[r]]                # rows that start with a NaN or an infinity
    vals[rp[bad]] = np.resize([np.nan, np.inf, -np.inf], len(bad))
    B = rng.integers(1, 9, (K, N)).astype(np.float32)
    plan = cs.SPMM_TC(cs.HRPB(M, K, rp, cols, vals), N, path=cs.PATH_ROWS)
    assert plan.kernel_name == "csr_rows_batched"
    out = torch_cuda.full((M, N), 7.5, device="cuda")
    plan.run(torch_cuda.from_numpy(B).cuda(), out)
    want = np.stack([(vals[rp[r]:rp[r + 1], None] * B[cols[rp[r]:rp[r + 1]]]).sum(0, dtype=np.float32) for r in range(M)])
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)
