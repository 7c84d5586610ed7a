"""Matrices that the host conversion must refuse, one fault at a time: the status is that of the first bad entry in row order,
and nothing past the last entry of the matrix is read on the way (a row pointer that is wrong must not lead there).  A child
process converts them, so that a crash is a failure of this test alone."""
import json
import os
import subprocess
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
M, K, PER_ROW = 1024, 256, 8
RANGE, UNSORTED = -4, -3

CHILD = """
import json, sys
import cutespmm_ae_amd as cs
from test_broken_csr import faults, M, K
out = {}
for name, (rp, cl, vl) in faults().items():
    try:
        cs.HRPB(M, K, rp, cl, vl)
        out[name] = 0
    except cs.CuteError as e:
        out[name] = e.status
    print(name, out[name], file=sys.stderr, flush=True)
print(json.dumps(out))
"""


def faults():
    rng = np.random.default_rng(3)
    cols = np.sort(rng.permuted(np.tile(np.arange(K), (M, 1)), axis=1)[:, :PER_ROW], axis=1).astype(np.uint32)
    rp, vl = (np.arange(M + 1) * PER_ROW).astype(np.uint32), np.ones(M * PER_ROW, np.float32)
    cases = {"sound": (rp, cols.ravel(), vl)}
    # a pointer inside a panel, at a panel's edge, at the edge of a thread's range, in the last panel, just past the last entry
    for row in (1, 5, 16, 17, 512, 1008, 1023):
        for value in (4_000_000_000, 200_000_000, M * PER_ROW + 1, 0):
            broken = rp.copy()
            broken[row] = value
            cases["rowPtr[%d] = %d" % (row, value)] = broken, cols.ravel(), vl
    # rows that hold the fault themselves
    for name, row in (("range before order", [5, 9999, 7]), ("order before range", [9, 7, 9999]), ("range", [5, 7, 256]),
                      ("equal", [5, 5, 7]), ("only out of range", [9999, 5, 7])):
        broken = cols.copy()
        broken[700, :3] = row
        broken[700, 3:] = [100, 101, 102, 103, 104]
        cases[name] = rp, broken.ravel(), vl
    return cases


def first_fault(rp, cl, vl):
    for r in range(M):
        s, e = int(rp[r]), int(rp[r + 1])
        if e < s:
            return RANGE
        for i in range(s, min(e, int(rp[M]))):
            if cl[i] >= K:
                return RANGE
            if i > s and cl[i] <= cl[i - 1]:
                return UNSORTED
        if e > rp[M]:
            return RANGE
    return 0


def test_host_conversion_refuses_broken_matrices_without_leaving_the_arrays():
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]))
    run = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, env=env, timeout=120)
    assert run.returncode == 0, "died after: " + " | ".join(run.stderr.strip().splitlines()[-2:])
    got = json.loads(run.stdout.strip().splitlines()[-1])
    want = {name: first_fault(*m) for name, m in faults().items()}
    assert want["sound"] == 0 and all(v for name, v in want.items() if name != "sound")
    assert got == want
