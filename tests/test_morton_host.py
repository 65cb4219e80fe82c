"""The numbering of blocks centre first: bits of a block's index and of its ranks
along the axes (tests/native/morton_check.cpp, on the host)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_places(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "morton_check")
    src = os.path.join(ROOT, "tests", "native", "morton_check.cpp")
    inc = ["-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "2018_dictionary_tomography_amd", "csrc")]
    res = subprocess.run([HIPCC, "--offload-arch=gfx950", "-x", "hip", "-O2", "-std=c++17", *inc, src, "-o", exe],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    grids, indices = map(int, res.stdout.split())
    assert grids == 680 + 8 and indices > 680
