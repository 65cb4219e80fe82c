"""Volume renders of few atoms in rows of 64 voxels, and of more on grids whose
brick numbers are mostly empty, against a dense FP64 evaluation on the GPU, voxel
by voxel, with the bound of test_gpu_volume_bricks."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _dense(I, x, r, y, dev):
    f = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=dev).double()  # noqa: E731
    I, x, r, y = f(I), f(x), f(r), [f(v) for v in y]
    c = np.sqrt(30 / np.log(2))
    shape = [v.numel() for v in y]
    ref, bound = torch.zeros(shape, dtype=torch.float64, device=dev), torch.full(shape, 0.0, dtype=torch.float64, device=dev)
    at = [(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]
    for j in range(I.numel()):
        d = [(v - x[j, k]).reshape([-1 if i == k else 1 for i in range(3)]) for k, v in enumerate(y)]
        v, dv = [0, 0, 0], [0, 0, 0]
        for k, (a, b) in enumerate(at):
            v[a] = v[a] + c * r[j, k] * d[b]
            dv[a] = dv[a] + 6 * U * c * r[j, k].abs() * d[b].abs()
        q = v[0] ** 2 + v[1] ** 2 + v[2] ** 2
        dq = 2 * torch.sqrt(q * (dv[0] ** 2 + dv[1] ** 2 + dv[2] ** 2)) + 4 * U * q
        t = I[j] * np.sqrt(30 / np.pi) * 2.0 ** -q
        inside, near = q <= 30 / np.log(2), (q - 30 / np.log(2)).abs() <= dq + 1e-6
        ref += torch.where(inside, t, 0.0)
        bound += torch.where(inside, t, 0.0) * (np.log(2) * dq + 9 * U) + torch.where(near, t, 0.0) + 1e-38
    return ref, bound


# rows of 64 from 4097 brick numbers on and up to 64 atoms (128 where most of more than
# 32768 numbers are empty); bricks otherwise
@pytest.mark.parametrize("shape", [(1, 600, 1030), (5, 131, 2050), (33, 125, 64), (130, 70, 65), (17, 265, 1041),
                                   (600, 515, 3)])
@pytest.mark.parametrize("n,order", [(1, 1), (64, 1), (65, 1), (7, -1), (128, 1), (129, 1)])
def test_few_atoms(gt, cuda, request, shape, n, order):
    if (shape, n) == ((5, 131, 2050), 65):
        # The bound is too small there, at one voxel, 5.6e-7 outside an atom's support (of a
        # form of 43.28): rounding lets its term in, 1.6e-6 of the term off, and the bound
        # allows such a term but not the term's own error (2.9e-5 of it, as inside).
        request.applymarker(pytest.mark.xfail(strict=True, reason="bound without a term's own error at the edge"))
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    I, x, r, _ = W.draw_aniso3(n, np.random.default_rng(sum(shape) + n))
    y = [(gt.cell_centres(-1, 1, m) if m > 1 else np.zeros(1))[::order].copy() for m in shape]
    atoms = gt.AtomElement(gt.AtomSpace(3, isotropic=False), x, r, I, device=cuda)
    u = gt.ops.volume(atoms, gt.VolSpace(y))
    ref, bound = _dense(I, x, r, y, cuda)
    assert tuple(u.shape) == shape
    assert bool(((u.double() - ref).abs() <= bound).all())


def test_sums_and_amplitudes(gt, cuda):
    """64-bit sums (96 copies of an atom, amplitudes 2^20, 1, -2^20) and an infinite
    amplitude, in rows."""
    rng = np.random.default_rng(1)
    y = [gt.cell_centres(-1, 1, m) for m in (17, 265, 1041)]
    space = gt.AtomSpace(3, isotropic=False)
    x, r = rng.uniform(-0.2, 0.2, (1, 3)), np.concatenate((rng.uniform(2, 4, (1, 3)), rng.normal(0, 0.5, (1, 3))), 1)
    run = lambda I, x, r: gt.ops.volume(gt.AtomElement(space, x, r, I, device=cuda), gt.VolSpace(y))  # noqa: E731
    one = run(np.array([0.75]), x, r)
    f = np.tile([2.0 ** 20, 1.0, -(2.0 ** 20)], 32)
    rng.shuffle(f)
    assert torch.equal(run(0.75 * f, np.tile(x, (96, 1)), np.tile(r, (96, 1))), 32 * one)
    both = run(np.array([0.75, np.inf]), np.concatenate((x, x)), np.concatenate((r, 2 * r)))
    bad = ~torch.isfinite(both)
    assert bad.any() and torch.equal(both[~bad], one[~bad])
    d = [torch.as_tensor(np.float32(v) - np.float32(x[0, k]), device=cuda).double().reshape(
        [-1 if i == k else 1 for i in range(3)]) for k, v in enumerate(y)]
    R = 2 * r[0]
    q = (R[0] * d[0] + R[3] * d[1] + R[5] * d[2]) ** 2 + (R[1] * d[1] + R[4] * d[2]) ** 2 + (R[2] * d[2]) ** 2
    assert not (bad & (q > 1 + 1e-4)).any() and bad[q < 1 - 1e-4].all()
