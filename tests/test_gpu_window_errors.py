"""The tables of csr_rows_window: without the memory for them the row kernel takes the rows, and nothing of the failed allocation
is found by a later call; any other failure of the runtime ends the creation of the plan and leaves the handle as it was.

The failures are made on the host: a library loaded in front of the HIP runtime, in a process of its own, answers the calls it is
told to with an error instead of passing them on (a wait is passed on first)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include <dlfcn.h>
#include <cstddef>
struct Dim { unsigned x, y, z; };
static int fail_malloc, fail_host, fail_wait, fail_launch, last;
template <class F> static F real(const char *name)
{
    static void *hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return reinterpret_cast<F>(dlsym(hip, name));
}
extern "C" {
void arm(int malloc_calls, int host_calls, int waits, int launches) { fail_malloc = malloc_calls; fail_host = host_calls; fail_wait = waits; fail_launch = launches; }
int left() { return fail_malloc + fail_host + fail_wait + fail_launch; }
int hipMalloc(void **p, size_t n)
{
    if (n > 4096 && fail_malloc) { --fail_malloc; return last = 2; }
    return real<int (*)(void **, size_t)>("hipMalloc")(p, n);
}
int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    if (fail_host) { --fail_host; return last = 2; }
    return real<int (*)(void **, size_t, unsigned)>("hipHostMalloc")(p, n, flags);
}
int hipStreamSynchronize(void *s)
{
    const int e = real<int (*)(void *)>("hipStreamSynchronize")(s);
    if (fail_wait) { --fail_wait; return last = 999; }
    return e;
}
int hipLaunchKernel(const void *f, Dim g, Dim b, void **args, size_t lds, void *s)
{
    if (fail_launch) { --fail_launch; return last = 9; }
    return real<int (*)(const void *, Dim, Dim, void **, size_t, void *)>("hipLaunchKernel")(f, g, b, args, lds, s);
}
int hipGetLastError()
{
    const int e = last, r = real<int (*)()>("hipGetLastError")();
    last = 0;
    return e ? e : r;
}
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
import numpy as np
import torch
import cutespmm_ae_amd as cs
M, N, per = 65536, 256, 32
rng = np.random.default_rng(3)
cols = (np.clip(np.arange(M) - 400, 0, M - 800)[:, None] + np.arange(per) * 25 + rng.integers(0, 25, (M, per))).astype(np.int32)
csr = [torch.from_numpy(a).cuda() for a in (np.arange(0, M * per + 1, per, dtype=np.int32), cols.ravel(), rng.integers(-8, 9, M * per).astype(np.float32))]
B = torch.randint(-8, 9, (M, N), device="cuda").float()
C = torch.empty(M, N, device="cuda")
want = cs.SPMM_TC(cs.DeviceHRPB(M, M, *csr), N, path=cs.PATH_ROWS).run(B, torch.empty(M, N, device="cuda"))
torch.cuda.synchronize()
for what, calls, fallback in (("device memory", (2, 0, 0, 0), True), ("pinned memory", (0, 1, 0, 0), True), ("launch", (0, 0, 0, 1), False), ("wait", (0, 0, 1, 0), False)):
    print(what, flush=True)
    h = cs.DeviceHRPB(M, M, *csr)
    bytes = h.device_bytes()
    cs.release_idle_memory()             # (so that the tables' memory is asked of the runtime)
    shim.arm(*calls)
    try:
        plan = cs.SPMM_TC(h, N, operand_residency=2)
        assert fallback, what + ": no error"
        assert shim.left() == 0 and plan.window_columns == 0 and plan.kernel_name == "csr_rows_batched"
        assert torch.equal(plan.run(B, C.zero_()), want)
    except cs.CuteError as e:
        assert shim.left() == 0 and not fallback and e.status == -7, (what, e)
    assert h.device_bytes() == bytes
    plan = cs.SPMM_TC(h, N, operand_residency=2)
    assert plan.window_columns == 16 and h.device_bytes() > bytes
    assert torch.equal(plan.run(B, C.zero_()), want)
    torch.cuda.synchronize()
print("done", flush=True)
"""


def test_tables_that_cannot_be_made(torch_cuda, tmp_path):
    (tmp_path / "shim.cpp").write_text(SHIM)
    lib = str(tmp_path / "shim.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", lib, str(tmp_path / "shim.cpp"), "-ldl"], check=True, timeout=60)
    run = subprocess.run([sys.executable, "-c", CHILD, lib], capture_output=True, text=True, timeout=100, env=dict(os.environ, PYTHONPATH=ROOT))
    assert run.returncode == 0 and run.stdout.endswith("done\n"), run.stdout + run.stderr[-3000:]
