"""No kernel of the library spills vector registers: what the compiler reports in the metadata of the built library.

The kernels that walk lists and rows in one launch stand at the 64 registers of eight wavefronts a SIMD, so a value more that
lives across a loop goes to scratch memory, a store and a load a wavefront that no timing of one size shows."""
import re

import cutespmm_ae_amd as cs


def _kernels():
    blob = open(cs.LIB_PATH, "rb").read()
    found = {}
    for m in re.finditer(rb"\.vgpr_spill_count(.)", blob, re.S):
        names = list(re.finditer(rb"\.symbol(?:\xd9.|\xda..|[\xa0-\xbf])(_Z\w+)\.kd", blob[max(0, m.start() - 2048):m.start()], re.S))
        assert names, "a kernel without a symbol"
        found[names[-1].group(1).decode()] = m.group(1)[0]       # a small integer is one byte
    return found


def test_no_kernel_spills_vector_registers():
    kernels = _kernels()
    assert len(kernels) > 100 and any("hrpb_quad_rows_f32" in k for k in kernels), len(kernels)
    assert {k: n for k, n in kernels.items() if n} == {}
