"""Handles and plans released while other work is under way: a stream being captured, kernels still running."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plan(cs, torch, rows, N):
    A = cs.gen_matrix(1, 3, rows, 16, 0)
    csr = [torch.from_numpy(np.array(a) if a.dtype == np.float32 else np.array(a).view(np.int32)).cuda() for a in (A.rowPtr, A.cols, A.vals)]
    return cs.SPMM_TC(cs.DeviceHRPB(A.M, A.K, *csr), N), torch.randn(A.K, N, device="cuda"), torch.empty(A.M, N, device="cuda")


@pytest.mark.parametrize("rows", [512, 65536])        # blocks below and above the size that is kept for the next handle
def test_release_beside_a_relaxed_capture(cs, torch_cuda, rows):
    torch = torch_cuda
    keep, B, C = _plan(cs, torch, 4096, 32)
    drop, _, _ = _plan(cs, torch, rows, 32)
    want = keep.run(B, C).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(), capture_error_mode="relaxed"):
        keep.run(B, C)
        del drop
        keep.run(B, C)
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)
        assert torch.equal(keep.run(B, C), want)
        torch.cuda.synchronize()


def test_format_from_device_arrays_waits_for_the_device(cs, torch_cuda):
    """cute_hrpb_upload_device_csr promises it, whatever the construction itself has to wait for."""
    torch = torch_cuda
    _plan(cs, torch, 4096, 32)
    side, done = torch.cuda.Stream(), torch.cuda.Event()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(100_000_000)
        done.record()
    rp = torch.arange(0, 513, dtype=torch.int32, device="cuda")
    cl, vl = torch.zeros(512, dtype=torch.int32, device="cuda"), torch.ones(512, device="cuda")
    assert not done.query()
    handle = cs.DeviceHRPB(512, 512, rp, cl, vl)
    assert done.query()
    del handle


def test_release_waits_for_running_kernels(cs, torch_cuda):
    """The block may serve another thread's set-up at once, so a release returns only when every stream is done with it."""
    torch = torch_cuda
    plan, B, C = _plan(cs, torch, 65536, 32)
    side, done = torch.cuda.Stream(), torch.cuda.Event()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(100_000_000)                 # tens of milliseconds
        plan.run(B, C)
        done.record()
    assert not done.query()
    del plan
    assert done.query()


def _free(torch):
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _refused(cs):
    """A Blocked-ELL upload of a tebibyte."""
    index, value = np.zeros(1, np.int32), np.zeros(1, np.float32)
    ell = cs.cute_blocked_ell(1 << 19, 1, 1, 1, 1, index.ctypes.data_as(cs.i32p), value.ctypes.data_as(cs.f32p))
    handle = ctypes.c_void_p()
    assert cs.load_library().cute_blocked_ell_upload(ctypes.byref(ell), ctypes.byref(handle)) == -7 and not handle.value


def test_an_allocation_that_fails_gives_the_kept_blocks_back_first(cs, torch_cuda):
    """A Blocked-ELL upload of a tebibyte is refused whatever the card holds; the memory kept from freed handles has gone back by
    then, and the error is not found again by the next product."""
    torch = torch_cuda
    plan, B, C = _plan(cs, torch, 4096, 32)
    drop, _, _ = _plan(cs, torch, 524288, 32)                  # 64 MiB of entries
    del drop
    before = _free(torch)
    _refused(cs)
    assert _free(torch) - before >= 64 << 20
    plan.run(B, C)
    torch.cuda.synchronize()


def test_a_block_too_large_to_keep_is_as_large_as_asked_for(cs, torch_cuda):
    """131 MiB of entries and row pointers, between two of the sizes that kept blocks are rounded to (128 and 144 MiB), and no
    layout beside them (every panel is the row kernel's)."""
    torch = torch_cuda
    M, per = 1040000, 16
    rp = torch.arange(0, M * per + 1, per, dtype=torch.int32, device="cuda")
    cl = torch.arange(16 * per, dtype=torch.int32, device="cuda").repeat(M // 16)      # the rows of a panel share no column
    vl = torch.ones(M * per, device="cuda")
    _refused(cs)                                       # nothing idle that the construction could take or give back
    before = _free(torch)
    handle = cs.DeviceHRPB(M, 16 * per, rp, cl, vl)
    used, asked = before - _free(torch), handle.device_bytes()
    del handle
    assert 130 << 20 <= asked <= 132 << 20 and abs(used - asked) <= 4 << 20, (used, asked)


def test_idle_memory_is_given_back_on_request(cs, torch_cuda):
    torch = torch_cuda
    keep, B, C = _plan(cs, torch, 65536, 32)
    want = keep.run(B, C).clone()
    drop, _, _ = _plan(cs, torch, 524288, 32)                  # 64 MiB of entries
    del drop
    before = _free(torch)
    cs.release_idle_memory()
    freed = _free(torch) - before
    assert freed >= 64 << 20
    cs.release_idle_memory()
    assert torch.equal(keep.run(B, C.zero_()), want)
    again, B2, C2 = _plan(cs, torch, 65536, 32)
    again.run(B2, C2)
    torch.cuda.synchronize()
