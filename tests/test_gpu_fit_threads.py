"""Fits launched together from host threads, each on its own stream: the results
of fits alone, bit for bit."""
import importlib
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_threads(gt, cuda):
    F = importlib.import_module("2018_dictionary_tomography_amd.fit")
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    n, jobs = 6, 5
    T, ortho, dv = W.tilt_series(20, 60.0, det=33)
    space, aspace = gt.ProjSpace(orientations=T, ortho=ortho, detector=dv), gt.AtomSpace(3, isotropic=False)

    def job(k):
        rng = np.random.default_rng(k)
        I, x, r, _ = W.draw_aniso3(n, rng, rho=(0.05, 0.1))
        data = gt.ops.forward(gt.AtomElement(aspace, x, r, I, device=cuda), space)
        start = gt.AtomElement(aspace, x + rng.normal(0, 0.02, x.shape), r, I * 0.8, device=cuda)
        req, s = F.newton_fit(start, space, data, [3, 1])
        return [t.clone() for t in (req.I, req.x, req.r, req.resid)] + [torch.tensor(s.E)]

    alone, got = [job(k) for k in range(jobs)], [None] * jobs
    torch.cuda.synchronize()

    def run(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[k] = job(k)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=run, args=(k,)) for k in range(jobs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        assert all(torch.equal(u, v) for u, v in zip(a, b))
    assert sum(F.workgroups._used.values()) == 0
