"""The fitter's pixel passes on detectors whose boxes leave remainders: fewer
rows than a group holds, columns that split a wave unevenly, more columns than
a wave, windows of the row table.  With and without a staging slab the fit is
the same to the bit; its energy is that of the residual it holds, and that
residual the projection of its atoms less the data."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# (the short fits at the larger sizes try and undo proposals only; the long ones accept most of theirs)
@pytest.mark.parametrize("n0,n1,rho,iters", [(5, 3, 0.3, 2), (9, 70, 0.2, 2), (200, 9, 0.3, 2), (33, 64, 0.1, 2),
                                             (17, 22, 0.05, 2), (250, 131, 0.3, 2), (9, 70, 0.2, 12),
                                             (200, 9, 0.3, 12), (12, 33, 0.2, 12)])
def test_boxes(gt, cuda, n0, n1, rho, iters):
    F = importlib.import_module("2018_dictionary_tomography_amd.fit")
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    rng = np.random.default_rng(n0)
    I, x, r, _ = W.draw_aniso3(6, rng, rho=(0.5 * rho, rho))
    x[0] = (0.9, -0.95, 0.9)
    T, ortho, _ = W.tilt_series(5, 60.0, det=9)
    space = gt.ProjSpace(orientations=T, ortho=ortho, detector=[np.linspace(-1, 1, n0), np.linspace(-1, 1, n1)])
    aspace = gt.AtomSpace(3, isotropic=False)
    data = gt.ops.forward(gt.AtomElement(aspace, x, r, I, device=cuda), space)
    start = gt.AtomElement(aspace, x + rng.normal(0, 0.05, x.shape), r, I * 0.7, device=cuda)
    reqs = []
    for stage in (False, True):
        req = F.FitRequest(start, space, data, [iters, 1], tol=1e-9, stage=stage)
        table = torch.as_tensor(np.frombuffer(req.slot_bytes(), dtype=np.uint8).copy(), device=cuda)
        F.run_blocks(table, 1, torch.as_tensor(F.block_table([2]), device=cuda), 2, req.dim, 100)
        reqs.append((req, F.read_slots(table, 1)[0]))
    (req, s), (req2, s2) = reqs
    assert s.done and (s.accepted > 0 or iters == 2)
    assert (s.done, s.jj, s.accepted, s.E) == (s2.done, s2.jj, s2.accepted, s2.E)
    for a, b in ((req.I, req2.I), (req.x, req2.x), (req.r, req2.r), (req.resid, req2.resid)):
        assert torch.equal(a, b)
    # each update's energy change is a sum of terms exact in FP64
    E = 0.5 * float((req.resid.double() ** 2).sum())
    assert abs(s.F - E) <= (s.jj + 1) * data.numel() * 2.0 ** -52 * req.F0
    # an update rounds a pixel once and takes two Gaussians of |exponent| < 64
    now = gt.ops.forward(req, space)
    scale = max(float(data.abs().max()), float(now.abs().max()))
    assert float((req.resid - (now - data)).abs().max()) <= (s.jj + 2) * 128 * 2.0 ** -24 * scale
