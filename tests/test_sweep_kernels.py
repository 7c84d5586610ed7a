"""The sweep tool knows every kernel a plan launches: a profile (written here in the profiler's place) gives the step's time."""
import os
import re

import pytest

from cutespmm_ae_amd import sweep

CSRC = os.path.join(os.path.dirname(sweep.__file__), "csrc")
# kernels of the library's other calls: comparison kernels, the Blocked-ELL product
OTHERS = ("csr_thread_per_element", "csr_wave_scalar", "csr_rows", "blocked_ell_f32")


def _plan_kernels():
    text = open(os.path.join(CSRC, "kernels.hip.hpp")).read()
    names = set(re.findall(r"__global__[^{;]*?\bvoid (\w+)\(", text))
    return sorted(names - set(OTHERS))


def test_the_kernels_are_found():
    names = _plan_kernels()
    assert {"hrpb_quad_f32", "hrpb_brick_f32_rolling", "csr_rows_batched", "csr_rows_window", "reduce_partials"} <= set(names), names


@pytest.mark.parametrize("kernel", _plan_kernels())
def test_kernel_durations_counts_every_kernel_of_a_plan(kernel, tmp_path, monkeypatch):
    prof = tmp_path / "rocprofv3"
    prof.write_text("""#!/bin/sh
while [ "$1" != -d ]; do shift; done
mkdir -p "$2/host"
cat > "$2/host/1_kernel_stats.csv" <<END
"Name","Calls","AverageNs"
"void cute_dev::%s<8, true>(unsigned int)","20","3000.0"
"void cute_dev::csr_rows<4, 5>(unsigned int)","20","9000.0"
"void cute_build::window_entries(unsigned int)","1","70000.0"
END
""" % kernel)
    prof.chmod(0o755)
    monkeypatch.setenv("PATH", "%s:%s" % (tmp_path, os.environ["PATH"]))
    assert sweep.kernel_durations("gen:5", 256, 20) == (3.0, 9.0)
