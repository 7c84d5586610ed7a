"""The products this library is used for, as cases that can be timed and compared.

A case is one sparse-dense product C[M,N] = A[M,K] . B[K,N] through the public entry points, in one of three forms:

  product   the plan is kept (a solver, a layer of a graph network): ``SPMM_TC.run`` on buffers that exist
  device    the matrix is new and already on the GPU (a sampled or re-assembled graph): format, plan and product
  host      the matrix is new and on the host, as the reader leaves it: format, upload, plan and product

``kind`` names the generator of ``cute_gen_matrix`` (uniform, stencil, fem, rmat, banded), ``size``, ``per_row`` and
``span`` its parameters; ``precision`` is fp32 or bf16x3.
"""
import math

import numpy as np
import torch

import cutespmm_ae_amd as cs

KINDS = {"uniform": 1, "stencil": 2, "fem": 3, "rmat": 4, "banded": 5}

# what the largest listed product costs, in entries times columns, and the most entries of a matrix that is new to the call
MOST_TERMS = 33554432 * 256
MOST_NEW_ENTRIES = 2500000


def _case(name, form, kind, size, N, per_row=0, span=0, precision="fp32"):
    c = {"form": form, "kind": kind, "size": size, "per_row": per_row, "span": span, "N": N, "precision": precision}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small layer: the call itself is what costs
        _case("uniform_4096_n32", "product", "uniform", 4096, 32, per_row=16),
        # a 9-point operator on 256 x 256 points applied to a block of 128 vectors
        _case("stencil_256_n128", "product", "stencil", 256, 128),
        # a finite-element matrix of 6 x 6 node blocks, block of 128 vectors
        _case("fem_8000_n128", "product", "fem", 8000, 128, span=200),
        # graph aggregation: power-law graph, 64 features
        _case("rmat_17_n64", "product", "rmat", 17, 64, per_row=10),
        # the largest product: a million rows, 256 columns, 2.4 GB of operands
        _case("banded_1m_n256", "product", "banded", 1048576, 256, per_row=32, span=2048),
        # an odd number of columns (the classes of an output layer) over a graph
        _case("rmat_16_n47", "product", "rmat", 16, 47, per_row=10),
        # an odd number of right-hand sides, an odd grid
        _case("stencil_200_n101", "product", "stencil", 200, 101),
        # short rows at random columns under a wide block of vectors
        _case("uniform_50000_n512", "product", "uniform", 50000, 512, per_row=7),
        # the reduced-precision arithmetic a caller may choose
        _case("fem_8000_n128_bf16x3", "product", "fem", 8000, 128, span=200, precision="bf16x3"),
        # a new graph on the GPU: format, plan, first product
        _case("new_rmat_16_n64", "device", "rmat", 16, 64, per_row=10),
        # a new small operator on the GPU
        _case("new_stencil_128_n32", "device", "stencil", 128, 32),
        # a new matrix from the host, the way the reference's driver uses the library
        _case("host_fem_4000_n128", "host", "fem", 4000, 128, span=200),
    ]


def entries(case):
    """Entries of the case's matrix (exact but for R-MAT graphs)."""
    kind, size, per_row = case["kind"], case["size"], case["per_row"]
    if kind == "stencil":
        return (3 * size - 2) ** 2
    if kind == "fem":
        upper = sum(min(4 if i & 1 else 5, case["span"], size - 1 - i) for i in range(size))
        return 36 * (size + 2 * upper)
    if kind == "rmat":
        # edges in both directions and the diagonal, less the draws that fall together (fitted, within 1 %)
        return int((2 * per_row + 1) * 2 ** size * (1 - 0.282 * (per_row / 10) ** 0.6 * 2 ** (-0.26 * (size - 10))))
    return size * per_row


def rows(case):
    kind, size = case["kind"], case["size"]
    return size * size if kind == "stencil" else 6 * size if kind == "fem" else 2 ** size if kind == "rmat" else size


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any generator, any form, sizes spread over their logarithm, common and odd numbers of columns."""
    while True:
        form = rng.choices(("product", "device", "host"), (5, 2, 1))[0]
        kind = rng.choice(sorted(KINDS))
        N = rng.choice((8, 16, 32, 64, 128, 256, 512)) if rng.random() < 0.5 else _log_int(rng, 1, 600)
        precision = "bf16x3" if form == "product" and rng.random() < 0.15 else "fp32"
        per_row = span = 0
        if kind == "stencil":
            size = 4 * _log_int(rng, 8, 128)            # a multiple of 4: whole panels of 16 rows
        elif kind == "fem":
            size, span = 8 * _log_int(rng, 25, 2000), _log_int(rng, 50, 400)
        elif kind == "rmat":
            size, per_row = rng.randint(10, 17), rng.randint(4, 12)
        elif kind == "uniform":
            size, per_row = 16 * _log_int(rng, 32, 8192), _log_int(rng, 4, 32)
        else:
            size, per_row, span = 16 * _log_int(rng, 32, 32768), _log_int(rng, 8, 48), _log_int(rng, 64, 2048)
        case = _case(None, form, kind, size, N, per_row, span, precision)
        nnz = entries(case)
        if form != "product" and nnz > MOST_NEW_ENTRIES:
            continue
        # rows at random columns, or a graph's, cost more per term than a band's
        if nnz * N * (8 if kind in ("uniform", "rmat") else 1) <= MOST_TERMS and nnz <= 33554432:
            return case


class State:
    """What the caller holds: the matrix (as far as the form of the case keeps it), B, C, and the plan."""


def prepare(case, seed):
    A = cs.gen_matrix(KINDS[case["kind"]], seed, case["size"], *((case["span"],) if case["kind"] == "fem" else (case["per_row"], case["span"])))
    s = State()
    s.M, s.K, s.N, s.form = A.M, A.K, case["N"], case["form"]
    s.precision = cs.PREC_BF16X3 if case["precision"] == "bf16x3" else cs.PREC_FP32
    g = torch.Generator(device="cuda").manual_seed(seed)
    s.B = torch.randn(s.K, s.N, generator=g, device="cuda")
    s.C = torch.empty(s.M, s.N, device="cuda")
    arrays = np.array(A.rowPtr), np.array(A.cols), np.array(A.vals)
    if s.form == "host":
        s.csr = arrays
        return s
    s.csr = tuple(torch.from_numpy(a if a.dtype == np.float32 else a.view(np.int32)).cuda() for a in arrays)
    if s.form == "product":
        s.plan = cs.SPMM_TC(cs.DeviceHRPB(s.M, s.K, *s.csr), s.N, precision=s.precision)
        s.csr = None
    return s


def run(s):
    if s.form == "product":
        return s.plan.run(s.B, s.C)
    make = cs.DeviceHRPB if s.form == "device" else cs.HRPB
    return cs.SPMM_TC(make(s.M, s.K, *s.csr), s.N, precision=s.precision).run(s.B, s.C)


def work(case):
    """CSR arrays and B read once, C written once; a multiplication and an addition per entry and column."""
    nnz, M, N = entries(case), rows(case), case["N"]
    return {"bytes": 8 * nnz + 4 * (M + 1) + 8 * M * N, "flops": 2 * nnz * N}


def tolerance(case):
    """Four times what the same sums differ by in another order, or from their values in 64 bits, on the five kinds of
    matrix: fp32 1.6e-7 of the norm and 2.5e-6 ... 5e-6 of a value (rows of thousands of entries); bf16x3 4.5e-6 and 2.7e-5."""
    return {"rel": 2e-5, "max": 1.2e-4} if case["precision"] == "bf16x3" else {"rel": 6.5e-7, "max": 2e-5}
