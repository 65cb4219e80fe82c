"""Workspace of the Fourier grid evaluation: without a grid, on grids for which
tables of every atom's phases would be far larger than the output, and the
refusal of less (no GPU work)."""
import ctypes

import pytest


def _sizes(gt, n, m):
    L = gt._lib
    lib = L.load()
    a, g = L.gt_atoms(3, n, 0, 1, 1, 1), L.gt_kgrid(3, *m, 1, 1, 1, 1)
    return lib, a, g, lib.gt_ft_workspace(ctypes.byref(a), None), lib.gt_ft_workspace(ctypes.byref(a), ctypes.byref(g))


@pytest.mark.parametrize("n", [1, 300, 16384, 16385])
@pytest.mark.parametrize("m", [(1 << 20, 1, 1), (1, 4, 1 << 20), (128, 128, 128), (4, 4, 4), (1024, 1024, 1024)])
def test_size(gt, n, m):
    lib, a, g, least, need = _sizes(gt, n, m)
    assert least == -(-n * 128 // 256) * 256 * (2 if n <= 16384 else 1)  # records, and their ranked copy
    out = 8 * m[0] * m[1] * m[2]
    assert least == need or need <= max(256 << 20, out)
    # either is enough, less is refused
    less = min(least, need) - 1
    assert lib.gt_ft_eval(ctypes.byref(a), ctypes.byref(g), 256, 256, less, None) == -3
    assert b"workspace" in lib.gt_last_error()
