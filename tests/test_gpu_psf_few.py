"""The point-spread projector on both sides of the line between few atoms (at most
six, a tile's pixels one by one) and more (whole cells by tabulated rules).

An atom of amplitude 0 takes six atoms over the line and adds exact zeros: the two
kernels agree to the bound of each against the exact integrals (2e-6 of the largest
value or of peak x cell, as derived in test_gpu_psf_project_groups), so to twice
it; seven and twenty atoms are held to that bound against the FP64 oracle at the cell
widths where the number of points per axis changes."""
import importlib

import numpy as np
import pytest

from conftest import f32

pytestmark = pytest.mark.gpu


def _case(gt, rng, n, ratio, det):
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    cell = 2.0 / 65
    axes = [cell * (np.arange(m) - 0.5 * (m - 1)) for m in det]
    T, ortho, _ = W.tilt_series(3, 50.0, axis=(0.1, 1.0, 0.2), det=8)
    space = gt.ProjSpace(orientations=T, ortho=ortho, detector=axes)
    d = ratio / cell / np.sqrt(60) * rng.uniform(0.9, 1.0, (n, 3))
    r = np.concatenate((d, 0.2 * d[:, :1] * rng.uniform(-1, 1, (n, 3))), 1)
    x = rng.uniform(-0.6, 0.6, (n, 3)) * 0.5 * cell * np.array([det[0], det[1], det[1]])
    x[0, 0] = 0.5 * cell * det[0]  # on the edge
    I = rng.uniform(0.5, 1.5, n)
    U = np.zeros((n, 3, 3))
    for k, (i, j) in enumerate([(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]):
        U[:, i, j] = r[:, k]
    peak = max(float((I / np.linalg.norm(U @ t, axis=1)).max()) for t in T) * cell ** 2
    return space, axes, I, x, r, peak


@pytest.mark.parametrize("ratio", [0.45, 0.95, 1.35, 1.9, 2.6])
@pytest.mark.parametrize("det,n", [((7, 5), 7), ((8, 64), 7), ((9, 65), 20), ((17, 130), 7)])
def test_more_than_few(gt, oracle, cuda, ratio, det, n):
    psf = importlib.import_module("2018_dictionary_tomography_amd.psf")
    space, axes, I, x, r, peak = _case(gt, np.random.default_rng(int(100 * ratio) + det[0]), n, ratio, det)
    P = psf.forward(gt.AtomElement(gt.AtomSpace(3, isotropic=False), x, r, I, device=cuda), space).cpu().numpy()
    og = oracle.Geometry(f32(space.orientations), tuple(f32(o) for o in space.ortho), [f32(a) for a in axes])
    want = oracle.psf_radproj(f32(I), f32(x), f32(r), og, 24)
    assert np.abs(P - want).max() <= 2e-6 * max(peak, np.abs(want).max())


@pytest.mark.parametrize("ratio", [0.45, 1.35, 2.6])
@pytest.mark.parametrize("det", [(2, 2), (16, 40), (33, 200)])
def test_across_the_line(gt, cuda, ratio, det):
    psf = importlib.import_module("2018_dictionary_tomography_amd.psf")
    space, _, I, x, r, peak = _case(gt, np.random.default_rng(int(100 * ratio) + det[0]), 7, ratio, det)
    I[3] = 0.0
    aspace, keep = gt.AtomSpace(3, isotropic=False), np.arange(7) != 3
    seven = psf.forward(gt.AtomElement(aspace, x, r, I, device=cuda), space).cpu().numpy()
    six = psf.forward(gt.AtomElement(aspace, x[keep], r[keep], I[keep], device=cuda), space).cpu().numpy()
    assert np.abs(six - seven).max() <= 4e-6 * max(peak, np.abs(six).max())
