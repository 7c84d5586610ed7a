"""The census of new matrices: panels of up to 512 entries that a wavefront holds, where panels are short on average; else a strip's entries held in registers (up to 512) or walked, and the bitmaps of four, two or one strips in LDS
at a time, by the panel's column window.  What it counts decides every place in both layouts, so these must equal the host
builders word for word."""
import numpy as np
import pytest

from test_device_build import _both_layouts, _check_bricks, _check_quads
from test_device_build_panels import _panels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quad_layout", [1, 2])
@pytest.mark.parametrize("K,spans", [
    (65536, (39296, 39297, 65536, 20)),                    # five bitmaps fit, they no longer do, the widest
    (70000, (28000, 28001, 46656, 46657)),                 # beyond 65 536 columns: four strips at a time, two, one
    (131072, (52416, 52417, 87360, 131072))])
def test_windows_by_bitmaps_at_a_time(cs, torch_cuda, K, spans, quad_layout):
    for sizes in ((600, 600, 600, 600), (1900, 40, 2000, 1), (2100, 4000, 5000, 3000)):
        M, rp, cl, vl = _panels(np.random.default_rng(K + sizes[0]), K, sizes, spans)
        got = _both_layouts(cs, torch_cuda, M, K, rp, cl, vl, quad_layout).layouts()
        _check_bricks(cs, got, M, K, rp, cl, vl)
        _check_quads(cs, got, M, rp, cl, vl)


@pytest.mark.parametrize("lengths", [(511, 512, 512, 1), (513, 0, 0, 0), (0, 0, 0, 512), (0, 513, 512, 3), (512, 512, 512, 512)])
def test_strips_held_or_walked(cs, torch_cuda, lengths):
    rng = np.random.default_rng(sum(lengths))
    K = 1024
    rows = []
    for n in lengths:                                      # a strip's entries, cut into its four rows, one of them empty
        cuts = np.sort(rng.integers(0, n + 1, 2))
        rows += [np.sort(rng.choice(K, k, replace=False)) for k in (cuts[0], 0, cuts[1] - cuts[0], n - cuts[1])]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    cl = np.concatenate(rows).astype(np.uint32)
    vl = rng.standard_normal(cl.size).astype(np.float32)
    vl[::5] = 0.0
    got = _both_layouts(cs, torch_cuda, 16, K, rp, cl, vl, 2).layouts()
    _check_bricks(cs, got, 16, K, rp, cl, vl)
    _check_quads(cs, got, 16, rp, cl, vl)
    unsorted = cl.copy()
    for r in range(16):                                    # the last two of every row that has two: seen wherever they stand
        s, e = int(rp[r]), int(rp[r + 1])
        if e - s < 2:
            continue
        unsorted[:] = cl
        unsorted[e - 2:e] = cl[e - 2:e][::-1]
        with pytest.raises(cs.CuteError) as err:
            cs.DeviceHRPB(16, K, *(torch_cuda.from_numpy(x.view(np.int32) if x.dtype == np.uint32 else x).cuda() for x in (rp, unsorted, vl)))
        assert err.value.status == -3


@pytest.mark.parametrize("sizes,spans,K,P", [
    ((0, 1, 63, 64, 65, 511, 512, 513), None, 4096, 9),              # bitmaps only; a panel in front each
    ((512, 512, 300, 512), (9824, 9825, 65536, 2), 65536, 7),        # the last window of five bitmaps, the first of the table
    ((512, 1, 513, 500), (13088, 131072, 131072, 131073), 400000, 9),
    ((512, 513, 5000, 0, 511, 49153, 2, 2000), None, 60000, 1024),   # longer panels; one that is counted entry by entry
    ((512, 513, 5000, 0, 511, 49153, 2, 2000), None, 60000, 1027)])  # four panels to a work-group in front, not a multiple of four
def test_panels_of_a_wavefront(cs, torch_cuda, sizes, spans, K, P):
    rng = np.random.default_rng(P + K)
    more = P - len(sizes)
    sizes = tuple(sizes) + tuple(int(x) for x in rng.integers(0, 40, more))
    M, rp, cl, vl = _panels(rng, K, sizes, spans and tuple(spans) + (500,) * more)
    assert cl.size <= 512 * P                              # short panels on average: this kernel, not the other
    got = _both_layouts(cs, torch_cuda, M, K, rp, cl, vl, 2).layouts()
    _check_bricks(cs, got, M, K, rp, cl, vl)
    _check_quads(cs, got, M, rp, cl, vl)


def test_wavefronts_see_every_unsorted_pair(cs, torch_cuda):
    """Neighbours in a row may stand in two lanes, in two registers of a wavefront, or begin a strip."""
    K, length = 4096, 32
    rng = np.random.default_rng(3)
    rows = [np.sort(rng.choice(K, length, replace=False)) for _ in range(16)]
    rp = (np.arange(17) * length).astype(np.uint32)
    cl, vl = np.concatenate(rows).astype(np.uint32), np.ones(16 * length, np.float32)
    gpu = lambda a: torch_cuda.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda()
    for r in range(16):
        for i in (1, 17, 31):
            bad = cl.copy()
            bad[r * length + i] = bad[r * length + i - 1]
            with pytest.raises(cs.CuteError) as err:
                cs.DeviceHRPB(16, K, gpu(rp), gpu(bad), gpu(vl))
            assert err.value.status == -3
    far = cl.copy()
    far[-1] = K
    with pytest.raises(cs.CuteError) as err:
        cs.DeviceHRPB(16, K, gpu(rp), gpu(far), gpu(vl))
    assert err.value.status == -4
    cs.DeviceHRPB(16, K, gpu(rp), gpu(cl), gpu(vl))


def test_two_threads_build_graphs_at_one_time(cs, torch_cuda):
    """The lists of a graph's long strips are built on a side stream that all threads share: each thread gets the layout that one alone gets."""
    import threading

    def build(seed):
        A = cs.gen_matrix(4, seed, 15, 10, 0)
        dev = [torch_cuda.from_numpy(np.array(x) if x.dtype == np.float32 else np.array(x).view(np.int32)).cuda() for x in (A.rowPtr, A.cols, A.vals)]
        return lambda: cs.DeviceHRPB(A.M, A.K, *dev, quad_layout=2).layouts()

    makers = [build(5), build(6)]
    alone = [make() for make in makers]
    got, barrier = [[], []], threading.Barrier(2)

    def work(i):
        for _ in range(6):
            barrier.wait(timeout=60)
            got[i].append(makers[i]())

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert len(got[i]) == 6
        for one in got[i]:
            assert one.keys() == alone[i].keys()
            assert all(np.array_equal(one[k], alone[i][k], equal_nan=True) if isinstance(one[k], np.ndarray) and one[k].dtype.kind == "f" else
                       np.array_equal(one[k], alone[i][k]) for k in one)
