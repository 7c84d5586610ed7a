"""The census of new matrices: a strip's entries held in registers (up to 512) or walked, and the bitmaps of four, two or one strips in LDS
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
