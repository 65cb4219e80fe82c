"""The 2D-detector projector at the edges of its work split: lists of one to
nine records (groups of four and a remainder), chunks of 256 records, detectors
that end inside an 8 x 16 rectangle or an 8 x 64 tile, coordinates in ascending
and in no order.  Against the FP64 oracle within the projector's 1e-5."""
import importlib

import numpy as np
import pytest

from conftest import f32, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 255, 257, 515])
@pytest.mark.parametrize("det", [(1, 1), (8, 16), (9, 17), (5, 70), (64, 63)])
def test_forward_groups(gt, oracle, cuda, n, det):
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    rng = np.random.default_rng(n)
    I, x, r, _ = W.draw_aniso3(n, rng, rho=(0.1, 0.3))
    x *= 0.5
    T, ortho, _ = W.tilt_series(3, 60.0, det=8)
    axes = [gt.cell_centres(-1, 1, m) for m in det]
    if n % 2:
        axes = [rng.permutation(a) for a in axes]
    space = gt.ProjSpace(orientations=T, ortho=ortho, detector=axes)
    atoms = gt.AtomElement(gt.AtomSpace(3, isotropic=False), x, r, I, device=cuda)
    R = gt.ops.forward(atoms, space).cpu().numpy()
    g = oracle.Geometry(f32(T), tuple(f32(o) for o in ortho), [f32(a) for a in axes])
    assert relerr(R, oracle.radproj(f32(I), f32(x), f32(r), g)) < 1e-5
