"""Without a built library every entry point says so at once (there is no fallback)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("call", ["load_library()", "HRPB(16, 16, [0] * 17, [], [])", "gen_matrix(1, 1, 16, 2, 0)"])
def test_missing_library_is_an_error_with_its_message(call, tmp_path):
    env = dict(os.environ, PYTHONPATH=ROOT, CUTESPMM_LIBRARY=str(tmp_path / "libcutespmm.so"))
    code = "import cutespmm_ae_amd as cs\ntry:\n    cs.%s\nexcept cs.CuteError as e:\n    print(e.status, e)" % call
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env, timeout=30)
    assert run.returncode == 0, run.stderr[-2000:]
    assert run.stdout.startswith("-8 ") and "is not built" in run.stdout, run.stdout
