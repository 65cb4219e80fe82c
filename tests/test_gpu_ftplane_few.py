"""Fourier sample planes of few atoms on large planes (256-sample tiles, the phase
in FP64) and on both sides of the line to the rectangles, against the FP64
oracle: a term's phase is off by a quarter-turn remainder in FP32 and 8.2e-8, its
profile as in test_gpu_fourier_cells, 1.5e-6 of the amplitudes in all."""
import importlib

import numpy as np
import pytest

from conftest import f32

pytestmark = pytest.mark.gpu


# 16384 samples and 32 + samples / 8192 atoms
@pytest.mark.parametrize("m0,m1,n", [(128, 128, 1), (130, 127, 1), (130, 127, 34), (130, 127, 35), (1031, 17, 5),
                                     (16, 1027, 34)])
@pytest.mark.parametrize("form", ["3d", "2.5d", "grid"])
def test_few_atoms(gt, oracle, cuda, m0, m1, n, form):
    fo = importlib.import_module("2018_dictionary_tomography_amd.fourier")
    rng = np.random.default_rng(m0 + n)
    I = rng.uniform(0.5, 1.5, n)
    k = [np.arange(m, dtype=float) - m // 2 for m in (m0, m1)]
    if form == "grid":
        x = rng.uniform(-3, 3, (n, 2))
        r = np.concatenate((rng.uniform(0.1, 0.8, (n, 2)), rng.normal(0, 0.1, (n, 1))), 1)
        S = (k[0].astype(np.float32), k[1].astype(np.float32))
        K = np.stack(np.meshgrid(*k, indexing="ij"), -1)[None]
        at = [(0, 0), (1, 1), (0, 1)]
    else:
        x = rng.uniform(-3, 3, (n, 3))
        r = np.concatenate((rng.uniform(0.1, 0.8, (n, 3)), rng.normal(0, 0.1, (n, 3))), 1)
        a = np.array([-0.7, 0.1, 0.9])
        w = np.stack((np.cos(a), np.sin(a)), 1)
        w0, w1 = np.concatenate((w, np.zeros((3, 1))), 1), np.tile([0.0, 0.0, 1.0], (3, 1))
        if form == "3d":
            t = rng.normal(size=(3, 3))
            w1 = np.cross(w0, t)
            w1 /= np.linalg.norm(w1, axis=1, keepdims=True)
            w0, w1 = f32(w0), f32(w1)
            S = (k[0].astype(np.float32), k[1].astype(np.float32), w0.astype(np.float32), w1.astype(np.float32))
        else:
            w0 = f32(w0)
            S = (k[0].astype(np.float32), k[1].astype(np.float32), w.astype(np.float32))
        K = k[0][None, :, None, None] * w0[:, None, None] + k[1][None, None, :, None] * w1[:, None, None]
        at = [(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]
    out = fo.evaluate(fo.FTAtoms(I, x, r, device=cuda), S).cpu().numpy().reshape(K.shape[:3])
    ref = np.zeros(K.shape[:3], complex)
    for Ij, xj, rj in zip(f32(I), f32(x), f32(r)):
        M = np.zeros((x.shape[1],) * 2)
        for c, (i, j) in enumerate(at):
            M[i, j] = rj[c]
        q = ((K @ M) ** 2).sum(-1)  # |U^T k|^2
        ref += np.where(q < 30, Ij * np.exp(-0.5 * q) * np.exp(-1j * (K @ xj)), 0)
    assert np.abs(out - ref).max() < 1.5e-6 * np.abs(I).sum()
