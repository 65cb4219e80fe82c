"""The block fitter with blocks that have nothing to try (an intensity whose
curvature is at most 1e-8: atoms beside the detector, step sizes of 1e12):
groups of any size walk the same blocks, to the same bits as one workgroup."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group", [2, 3, 8])
def test_skipped_blocks(gt, cuda, group):
    F = importlib.import_module("2018_dictionary_tomography_amd.fit")
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    rng = np.random.default_rng(8)
    n, iters = 9, [4, 2]
    I, x, r, _ = W.draw_aniso3(n, rng, rho=(0.03, 0.06))
    x = x * 0.2
    T, ortho, dv = W.tilt_series(24, 60.0, det=33)
    space = gt.ProjSpace(orientations=T, ortho=ortho, detector=[0.25 * np.asarray(d) for d in dv])
    aspace = gt.AtomSpace(3, isotropic=False)
    data = gt.ops.forward(gt.AtomElement(aspace, x, r, I, device=cuda), space)
    x0 = x + rng.normal(0, 0.02, x.shape)
    x0[::2, 1] = 0.97  # the tilt axis: beside the detector at every angle
    start = gt.AtomElement(aspace, x0, r, I * 0.8, device=cuda)
    h = np.full(3 * n, 1e12)
    one, s1 = F.newton_fit(start, space, data, iters, tol=1e-9, group=1, block=True, h=h)
    assert s1.done == 1 and s1.updates > 0
    # an update brings its step size to 1e4 or less: these blocks never had one
    assert (one.h.reshape(3, n)[0].cpu().numpy() == 1e12).tolist() == (np.arange(n) % 2 == 0).tolist()
    req, s = F.newton_fit(start, space, data, iters, tol=1e-9, group=group, block=True, h=h)
    assert (s.done, s.jj, s.accepted, s.updates, s.E) == (s1.done, s1.jj, s1.accepted, s1.updates, s1.E)
    for a, b in ((req.I, one.I), (req.x, one.x), (req.r, one.r), (req.resid, one.resid), (req.h, one.h)):
        assert torch.equal(a, b)
