"""Volume render at sizes around the bricks of voxels that a block takes, with
few and many atoms and with coordinates that do not ascend, against a dense
FP64 evaluation, voxel by voxel.

Bound (u = 2^-24): an offset d = (y - x_hi) - x_lo is off by 2 u |d|, a slot of U'
by u, so row i of v = U' d by 6 u sum_k |U'_ik| |d_k|; the exponent -|v|^2 by 2
|v| |dv| + 4 u |v|^2; a term amp 2^-|v|^2 relatively by ln 2 times that plus 4 u
(amplitude, exp2, product); the four-term sums add 4 u of the terms' sum and the
result's rounding u of it.  A term at the cut may fall on either side of it:
e^-30 of its peak.
"""
import importlib

import numpy as np
import pytest

from conftest import f32

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _dense(I, x, r, y, iso):
    """(sum, error bound) per voxel in FP64."""
    c = np.sqrt(30 / np.log(2))
    Y = np.stack(np.meshgrid(*y, indexing="ij"), -1)
    ref, bound = np.zeros(Y.shape[:3]), np.zeros(Y.shape[:3])
    for j in range(I.size):
        M = np.zeros((3, 3))
        at = [(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]
        for k, (a, b) in enumerate(at):
            M[a, b] = c * (r[j, 0] * (k < 3) if iso else r[j, k])
        d = Y - x[j]
        v = d @ M.T
        dv = 6 * U * (np.abs(d) @ np.abs(M).T)
        q = (v * v).sum(-1)
        dq = 2 * np.linalg.norm(v, axis=-1) * np.linalg.norm(dv, axis=-1) + 4 * U * q
        peak = I[j] * np.sqrt(30 / np.pi)
        t = peak * 2.0 ** -q
        inside = q <= 30 / np.log(2)
        ref += np.where(inside, t, 0)
        near = np.abs(q - 30 / np.log(2)) <= dq + 1e-6
        bound += np.where(inside, t, 0) * (np.log(2) * dq + 9 * U) + np.where(near, t, 0) + 1e-38
    return ref, bound


@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 8, 16), (5, 9, 17), (3, 7, 33), (12, 24, 8)])
@pytest.mark.parametrize("n,iso,order", [(1, False, 1), (256, False, 1), (257, True, 1), (700, False, 1), (30, False, -1)])
def test_bricks(gt, cuda, shape, n, iso, order):
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    rng = np.random.default_rng(sum(shape) + n)
    I, x, r, _ = W.draw_aniso3(n, rng)
    if iso:
        r = r[:, :1]
    y = [(gt.cell_centres(-1, 1, m) if m > 1 else np.zeros(1))[::order] for m in shape]
    atoms = gt.AtomElement(gt.AtomSpace(3, isotropic=iso), x, r, I, device=cuda)
    u = gt.ops.volume(atoms, gt.VolSpace([v.copy() for v in y])).cpu().numpy()
    ref, bound = _dense(f32(I), f32(x), f32(r), [f32(v) for v in y], iso)
    assert u.shape == shape
    assert (np.abs(u - ref) <= bound).all()
