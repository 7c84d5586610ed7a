"""Panels of more than 4 096 entries: where none holds more than 49 152 or spans more columns than the bitmap takes, one work-group walks
the entries of a panel for the census and of a strip for the strip lists; else all of them, and in any case the brick tiles and
lockstep lists, take the entry-parallel path.  Strips of panels of more than 1 024 go by their own length.  Both layouts must equal the host builders word for word."""
import numpy as np
import pytest

from test_device_build import _both_layouts, _check_bricks, _check_quads
from test_device_build_panels import _panels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quad_layout", [1, 2])
@pytest.mark.parametrize("sizes,spans,K", [
    ((4097, 20, 12000), None, 2048),                       # dense: every column active
    ((30000, 5000, 0, 300), None, 65536),
    ((49152, 4097), None, 60000),                          # the most a panel may hold
    ((49153, 8000), None, 60000),                          # one more: the entry-parallel path for both
    ((40000, 4100), None, 131072),                         # the widest bitmap beside many active columns
    ((49152, 4097), (131072, 5000), 131072),               # the widest bitmap beside the most entries
    ((49153, 5000, 6000), None, 60000),                    # one panel too long among others: all of them take the other path
    ((5000, 6000, 7000), (131072, 131071, 1600), 400000),  # windows at the bitmap's edge and narrow ones
    ((5000, 6000), (131073, 9000), 400000)])
def test_long_panels(cs, torch_cuda, sizes, spans, K, quad_layout):
    M, rp, cl, vl = _panels(np.random.default_rng(sum(sizes) + K), K, sizes, spans)
    got = _both_layouts(cs, torch_cuda, M, K, rp, cl, vl, quad_layout).layouts()
    _check_bricks(cs, got, M, K, rp, cl, vl)
    _check_quads(cs, got, M, rp, cl, vl)


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("strips", [(1023, 2, 0, 0), (0, 1024, 1, 0), (1, 1025, 0, 1024), (1024, 1024, 1024, 1024), (0, 0, 900, 125), (1025, 1, 1026, 1023), (1500, 40, 0, 3000)])
def test_strips_of_panels_beyond_one_work_group(cs, torch_cuda, strips, zeros):
    """Panels of more than 1 024 entries: a strip of up to as many is a work-group's beside the small panels, a longer one big_quads'."""
    rng = np.random.default_rng(sum(strips))
    K, rows = 8192, [np.sort(rng.choice(8192, 5, replace=False)) for _ in range(16)]
    for n in strips:
        a = n // 3
        rows += [np.sort(rng.choice(K, k, replace=False)) for k in (a, 0, n - a - a // 2, a // 2)]
    rows += rows[:16]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    cl = np.concatenate(rows).astype(np.uint32)
    vl = rng.standard_normal(cl.size).astype(np.float32)
    if zeros:
        vl[rng.random(cl.size) < 0.3] = 0.0
    got = _both_layouts(cs, torch_cuda, 48, K, rp, cl, vl, 2).layouts()
    _check_quads(cs, got, 48, rp, cl, vl)


def test_rows_alone_and_products(cs, orc, torch_cuda):
    """One row, the last, or two strips of a long panel hold its entries; the graph's default plan gives the oracle's product."""
    rng = np.random.default_rng(4)
    K = 32768
    rows = [np.zeros(0, np.int64)] * 48
    rows[0] = np.sort(rng.choice(K, 6000, replace=False))
    rows[31] = np.arange(K - 9000, K)
    rows[33], rows[47] = np.sort(rng.choice(K, 5000, replace=False)), np.arange(0, K, 3)
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    cl = np.concatenate(rows).astype(np.uint32)
    vl = rng.integers(-4, 5, cl.size).astype(np.float32)
    got = _both_layouts(cs, torch_cuda, 48, K, rp, cl, vl, 2).layouts()
    _check_bricks(cs, got, 48, K, rp, cl, vl)
    _check_quads(cs, got, 48, rp, cl, vl)
    A = cs.gen_matrix(4, 5, 14, 12)
    vals = np.round(rng.standard_normal(A.nnz) * 2).astype(np.float32)
    B = rng.integers(-4, 5, (A.K, 40)).astype(np.float32)
    h = cs.DeviceHRPB(A.M, A.K, *(torch_cuda.from_numpy(np.array(a).view(np.int32)).cuda() for a in (A.rowPtr, A.cols)), torch_cuda.from_numpy(vals).cuda())
    out = torch_cuda.empty(A.M, 40, device="cuda")
    cs.SPMM_TC(h, 40).run(torch_cuda.from_numpy(B).cuda(), out)
    assert np.array_equal(out.cpu().numpy(), orc.spmm_csr(np.array(A.rowPtr), np.array(A.cols), vals, B))
