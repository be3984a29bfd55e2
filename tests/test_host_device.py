"""Host compiles of the kernels' address and arithmetic helpers (no GPU needed)."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "ptatin-gene_amd", "csrc")


@pytest.mark.parametrize("name,line", [("test_tile_rows", "tile rows ok"), ("test_row_sums", "row sums ok")])
def test_host_check(tmp_path, name, line):
    exe = str(tmp_path / name)
    subprocess.check_call(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", "-I", CSRC,
                           "-I", os.path.join(REPO, "include"), os.path.join(REPO, "tests", "c", name + ".cpp"),
                           "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr + out.stdout
    assert line in out.stdout
