"""No kernel of the library spills vector registers: what the compiler reports in the metadata of the built library.

The kernels that walk lists and rows in one launch stand at the 64 registers of eight wavefronts a SIMD, so a value more that
lives across a loop goes to scratch memory, a store and a load a wavefront that no timing of one size shows."""
import re

import cutespmm_ae_amd as cs


def _kernels(field=b"vgpr_spill_count"):
    blob = open(cs.LIB_PATH, "rb").read()
    found = {}
    for m in re.finditer(rb"\." + field + rb"(.)", blob, re.S):
        names = list(re.finditer(rb"\.symbol(?:\xd9.|\xda..|[\xa0-\xbf])(_Z\w+)\.kd", blob[max(0, m.start() - 2048):m.start()], re.S))
        assert names, "a kernel without a symbol"
        found[names[-1].group(1).decode()] = m.group(1)[0]       # a small integer is one byte
    return found


def test_no_kernel_spills_vector_registers():
    kernels = _kernels()
    assert len(kernels) > 100 and any("hrpb_quad_rows_f32" in k for k in kernels), len(kernels)
    assert {k: n for k, n in kernels.items() if n} == {}


def test_two_work_groups_of_the_hub_kernel_fit_a_compute_unit():
    """Its work-groups are sixteen wavefronts and the launch starts two a compute unit: eight wavefronts a SIMD, 64 registers.  (Off the grid of 64
    columns it has always taken 65.)"""
    hub = {k: n for k, n in _kernels(b"vgpr_count").items() if "hrpb_quad_hub_f32ILb1E" in k}
    assert list(hub.values()) == [64], hub


def test_plans_without_cut_panels_carry_no_registers_for_pieces():
    """The kernels are compiled without the pieces of cut panels as well (the last template argument); 32-column lists take 46 registers that way."""
    half = {k: n for k, n in _kernels(b"vgpr_count").items() if "hrpb_quad_half_f32" in k}
    uncut = [n for k, n in half.items() if re.search(r"ILb[01]ELb0EE", k)]
    assert len(half) == 4 and len(uncut) == 2 and max(uncut) <= 46, half
