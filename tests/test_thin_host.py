"""The culls of the Fourier sample planes on long slanted ellipses, by brute
force on the host (tests/native/thin_check.cpp): nothing that holds a sample is
dropped at any axis ratio, and at ordinary ratios most of the rest is."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("thin") / "thin_check")
    src = os.path.join(ROOT, "tests", "native", "thin_check.cpp")
    inc = ["-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "2018_dictionary_tomography_amd", "csrc")]
    res = subprocess.run([HIPCC, "--offload-arch=gfx950", "-x", "hip", "-O2", "-std=c++17", *inc, src, "-o", exe],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return exe


@pytest.mark.parametrize("ratio", [1, 10, 60, 120, 126, 300, 700, 1000, 2000, 3000, 10000])
def test_long_ellipses(check, ratio):
    res = subprocess.run([check, str(ratio), "400"], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    inside, held, kept, rows = map(int, res.stdout.split())
    assert 0 < held <= kept <= rows
    if ratio <= 60:
        assert kept < 0.5 * rows
