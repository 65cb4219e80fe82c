"""The Fourier grid on both sides of the line between few atoms (records in radius
order, the phase in FP64) and the phase tables, and at axes around the entries
that one wave tabulates, against the FP64 oracle.

Tolerance as in test_gpu_fourier_cells, 1.5e-6 of the sum of the amplitudes; per
sample the phase alone is better than that of the tables (an FP32 quarter turn and
8.2e-8).
"""
import importlib

import numpy as np
import pytest

from conftest import f32

pytestmark = pytest.mark.gpu


# 64 x 1 x 1 blocks of 8 x 8: few are 131 atoms; 64 x 8 x 8: 197
@pytest.mark.parametrize("shape,n", [((64, 8, 5), 131), ((64, 8, 5), 132), ((64, 57, 60), 197), ((64, 57, 60), 198),
                                     ((65, 57, 60), 20), ((500, 8, 4), 300), ((498, 9, 5), 300), ((3, 4, 1030), 300),
                                     ((9, 1021, 2), 200)])
@pytest.mark.parametrize("iso", [False, True])
def test_paths(gt, oracle, cuda, shape, n, iso):
    fo = importlib.import_module("2018_dictionary_tomography_amd.fourier")
    rng = np.random.default_rng(sum(shape) + n)
    I, x = rng.uniform(0.5, 1.5, n), rng.uniform(-4, 4, (n, 3))
    if iso:
        r = rng.uniform(1.0, 4.0, (n, 1))
    else:
        r = np.concatenate((rng.uniform(0.1, 0.8, (n, 3)), rng.normal(0, 0.1, (n, 3))), 1)
    k = [np.arange(m, dtype=float) - m // 2 for m in shape]
    out = fo.evaluate(fo.FTAtoms(I, x, r, device=cuda), [v.astype(np.float32) for v in k]).cpu().numpy()
    ref = oracle.ft_grid(f32(I), f32(x), f32(r), [f32(v) for v in k], iso=iso)
    assert np.abs(out - ref).max() < 1.5e-6 * np.abs(I).sum()
