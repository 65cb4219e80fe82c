"""The Fourier grid evaluation with the workspace of gt_ft_workspace(atoms, NULL):
the kernel without tables, records in radius order, against the FP64 oracle
(tolerance as in test_gpu_fourier_cells: 1.5e-6 of the amplitudes; the hardware
sine and cosine add 1.25e-7)."""
import ctypes
import importlib

import numpy as np
import pytest
import torch

from conftest import f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 40, 257, 1030])
@pytest.mark.parametrize("shape", [(5, 9, 17), (64, 3, 2), (16, 16, 16)])
@pytest.mark.parametrize("order", [1, -1])
def test_without_tables(gt, oracle, cuda, n, shape, order):
    fo = importlib.import_module("2018_dictionary_tomography_amd.fourier")
    lib = gt._lib.load()
    rng = np.random.default_rng(n)
    I, x = rng.uniform(0.5, 1.5, n), rng.uniform(-4, 4, (n, 3))
    r = np.concatenate((rng.uniform(0.2, 0.8, (n, 3)), rng.normal(0, 0.15, (n, 3))), 1)
    k = [(np.arange(m, dtype=float) - m // 2)[::order].copy() for m in shape]
    atoms, grid = fo.FTAtoms(I, x, r, device=cuda), fo.DeviceKGrid(k, cuda)
    a = gt.ops.atoms_struct(atoms)
    ws = torch.empty(lib.gt_ft_workspace(ctypes.byref(a), None), dtype=torch.uint8, device=cuda)
    out = torch.full(shape, float("nan"), dtype=torch.complex64, device=cuda)
    assert lib.gt_ft_eval(ctypes.byref(a), ctypes.byref(grid.struct), out.data_ptr(), ws.data_ptr(), ws.numel(),
                          gt._lib.stream_handle(cuda)) == 0
    ref = oracle.ft_grid(f32(I), f32(x), f32(r), [f32(v) for v in k])
    assert np.abs(out.cpu().numpy() - ref).max() < 1.6e-6 * np.abs(I).sum()
