"""Panels at the edges of the device builders' kinds: a panel that one work-group holds in LDS (up to 1 024, 2 048 or 4 096 entries,
a column window of up to 131 072), and the entry-parallel path beyond.  Both layouts must equal the host builders word for word,
and every kind must report the same errors."""
import numpy as np
import pytest

from test_device_build import _both_layouts, _check_bricks, _check_quads, _to_gpu

pytestmark = pytest.mark.gpu


def _panels(rng, K, sizes, spans=None, zeros=True):
    """One 16-row panel per entry count; rows of uneven length, columns from a window of `span` columns (all of K: None)."""
    rows = []
    for j, n in enumerate(sizes):
        span = (spans[j] if spans else None) or K
        lo = int(rng.integers(0, K - span + 1))
        left = n
        for r in range(16):
            take = left if r == 15 else min(left, int(rng.integers(0, 2 * (left // (16 - r)) + 2)))
            take = min(take, span)
            c = lo + rng.choice(span, take, replace=False)
            if spans and r == 0 and take >= 2:
                c[0], c[1] = lo, lo + span - 1                # the window is exactly as wide as asked for
                c = np.unique(c)
            rows.append(np.sort(c))
            left -= len(rows[-1])
    rp = np.zeros(len(rows) + 1, np.uint32)
    rp[1:] = np.cumsum([len(c) for c in rows])
    cl = np.concatenate(rows).astype(np.uint32)
    vl = rng.standard_normal(len(cl)).astype(np.float32)
    if zeros:
        vl[rng.random(len(vl)) < 0.1] = 0.0
    return len(rows), rp, cl, vl


@pytest.mark.parametrize("quad_layout", [1, 2])
@pytest.mark.parametrize("sizes", [(1, 0, 16, 255, 256, 257), (1023, 1024, 1025, 0, 3), (2047, 2048, 2049, 5), (4095, 4096, 4097, 8), (0, 9000, 40, 2048, 3000, 0, 4096)])
def test_entry_counts(cs, torch_cuda, sizes, quad_layout):
    K = 4096
    M, rp, cl, vl = _panels(np.random.default_rng(sum(sizes)), K, sizes)
    got = _both_layouts(cs, torch_cuda, M, K, rp, cl, vl, quad_layout).layouts()
    _check_bricks(cs, got, M, K, rp, cl, vl)
    _check_quads(cs, got, M, rp, cl, vl)


@pytest.mark.parametrize("quad_layout", [1, 2])
@pytest.mark.parametrize("sizes,K,spans", [((512, 511, 127, 128, 129, 0), 4096, None), ((512, 0, 1, 513), 4096, None),
                                           ((512, 300, 512), 70000, (65536, 32, 33)), ((512, 300, 700), 400000, (131072, 131073, 40))])
def test_short_panels_and_windows_narrower_than_the_matrix(cs, torch_cuda, sizes, K, spans, quad_layout):
    M, rp, cl, vl = _panels(np.random.default_rng(sum(sizes) + K), K, sizes, spans)
    got = _both_layouts(cs, torch_cuda, M, K, rp, cl, vl, quad_layout).layouts()
    _check_bricks(cs, got, M, K, rp, cl, vl)
    _check_quads(cs, got, M, rp, cl, vl)


@pytest.mark.parametrize("quad_layout", [1, 2])
def test_column_windows(cs, torch_cuda, quad_layout):
    K = 400000
    spans = (31, 32, 33, 131071, 131072, 131073, 400000, 64)
    M, rp, cl, vl = _panels(np.random.default_rng(8), K, (100, 200, 300, 500, 700, 900, 1100, 0), spans)
    got = _both_layouts(cs, torch_cuda, M, K, rp, cl, vl, quad_layout).layouts()
    _check_bricks(cs, got, M, K, rp, cl, vl)
    _check_quads(cs, got, M, rp, cl, vl)


@pytest.mark.parametrize("size,K", [(300, 4096), (3000, 4096), (5000, 4096), (300, 400000)])
def test_errors_of_every_kind(cs, torch_cuda, size, K):
    M, rp, cl, vl = _panels(np.random.default_rng(9), K, (40, size, 40), None, zeros=False)
    r = int(np.argmax(np.diff(rp[16:33].astype(np.int64)))) + 16          # a row of the middle panel
    s, e = int(rp[r]), int(rp[r + 1])
    assert e - s > 4
    swapped, far, first = cl.copy(), cl.copy(), cl.copy()
    swapped[s + 2], swapped[s + 3] = cl[s + 3], cl[s + 2]
    far[e - 1] = K + 7
    first[s] = cl[e - 1]                                                   # the row starts above its end
    for bad, status in ((swapped, -3), (far, -4), (first, -3)):
        with pytest.raises(cs.CuteError) as err:
            cs.DeviceHRPB(M, K, *_to_gpu(torch_cuda, rp, bad, vl))
        assert err.value.status == status


def test_handles_and_plans_come_and_go(cs, orc, torch_cuda):
    """Released memory serves the next handle: products in flight on another stream while handles of the same sizes are freed and made."""
    torch = torch_cuda
    rng = np.random.default_rng(10)
    K, N = 8192, 64
    mats = [_panels(rng, K, (700,) * 200, zeros=False) for _ in range(3)]
    B = torch.from_numpy(rng.integers(-3, 4, (K, N)).astype(np.float32)).cuda()
    dev = [_to_gpu(torch, rp, cl, np.round(vl * 4)) for _, rp, cl, vl in mats]
    refs = [orc.spmm_csr(rp, cl, np.round(vl * 4), B.cpu().numpy()) for _, rp, cl, vl in mats]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    outs = []
    for i in range(12):
        M, C = mats[i % 3][0], torch.full((mats[i % 3][0], N), float("nan"), device="cuda")
        torch.cuda.current_stream().synchronize()
        plan = cs.SPMM_TC(cs.DeviceHRPB(M, K, *dev[i % 3]), N, path=cs.PATH_BRICK, mfma_shape=1 + i % 2)
        plan.run(B, C, stream=side)
        del plan                                                           # its kernel may still run
        outs.append((i % 3, C))
    torch.cuda.synchronize()
    for k, C in outs:
        assert (C.cpu().numpy() == refs[k]).all()


def test_more_panels_than_one_grid_row_holds(cs, torch_cuda):
    """2^28 rows and a panel: 256 threads a panel are more than 2^32 threads in a row of the grid."""
    torch = torch_cuda
    M, K, N = (1 << 28) + 16, 64, 1
    rng = np.random.default_rng(12)
    per = 1 << 22                                                          # panels to a row of the grid
    rows = np.unique(np.concatenate([[0, 15, 16, 16 * per - 1, 16 * per, 32 * per, M - 17, M - 16, M - 1], rng.integers(0, M, 4000)]))
    counts = rng.integers(1, 9, rows.size)
    cl = np.concatenate([np.sort(rng.choice(K, c, replace=False)) for c in counts]).astype(np.int32)
    vl = rng.integers(-4, 5, cl.size).astype(np.float32)
    starts = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).cuda()
    rp = starts[torch.searchsorted(torch.from_numpy(rows).cuda(), torch.arange(M + 1, device="cuda"))]
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    C = torch.full((M, N), float("nan"), device="cuda")
    plan = cs.SPMM_TC(cs.DeviceHRPB(M, K, rp, torch.from_numpy(cl).cuda(), torch.from_numpy(vl).cuda()), N)
    plan.run(torch.from_numpy(B).cuda(), C)
    want = np.zeros((rows.size, N))
    np.add.at(want, np.repeat(np.arange(rows.size), counts), vl[:, None].astype(np.float64) * B[cl])
    assert torch.equal(C[torch.from_numpy(rows).cuda()].cpu(), torch.from_numpy(want).float())       # whole numbers: exact
    C[torch.from_numpy(rows).cuda()] = 0.0
    assert int(torch.count_nonzero(C)) == 0                                # (a NaN counts)
