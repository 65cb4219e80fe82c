"""An atom whose amplitude is not finite: its samples inside the support are
not finite, every sample outside it is that of the other atoms.

The supports are taken in FP64 and widened by a factor of 1 + 1e-4 in the
form, far above its FP32 rounding at these atoms (axis ratios up to 5).  The
point-spread values may reach the whole cells of the support's bounding box.
Outside, the render with the atom and the one without it add the same terms, in
the same order but for the groups that the atom's place shifts: they agree to 1e-6
of the largest value (the sums' FP32 groups).
"""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BAD = [np.inf, -np.inf, np.nan]


def _atoms(rng, n, bad, at):
    I = rng.uniform(0.5, 1.5, n)
    x = rng.uniform(-0.6, 0.6, (n, 3))
    r = np.concatenate((1.0 / rng.uniform(0.03, 0.1, (n, 3)), rng.normal(0, 4.0, (n, 3))), 1) / np.sqrt(60.0)
    if bad is not None:
        I[at] = bad
    return I, x, r


def _umat(r):
    U = np.zeros((3, 3))
    for k, (i, j) in enumerate([(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]):
        U[i, j] = r[k]
    return U


def _check(with_, without, support, inner):
    """with_, without: outputs with and without the atom; support: where it may
    reach, inner: where it must."""
    with_, without = (t.cpu().numpy() for t in (with_, without))
    bad = ~np.isfinite(with_)
    assert not (bad & ~support).any()
    assert bad[inner].all() and inner.any()
    d = np.abs(with_ - without)[~support]
    assert d.max() < 1e-6 * np.abs(without).max()


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("op", ["GaussTomo", "SingleParticleGaussTomo"])
def test_volume(gt, cuda, op, bad):
    n, at, m = 20, 7, (48, 37, 50)
    I, x, r = _atoms(np.random.default_rng(4), n, bad, at)
    space = gt.AtomSpace(3, isotropic=False)
    y = [gt.cell_centres(-1, 1, k) for k in m]
    T = getattr(gt, op)(space, gt.VolSpace(y), None)
    keep = np.arange(n) != at
    u = T.discretise(gt.AtomElement(space, x, r, I, device=cuda)).data
    v = T.discretise(gt.AtomElement(space, x[keep], r[keep], I[keep], device=cuda)).data
    U = _umat(r[at])
    if op == "GaussTomo":
        d = np.stack(np.meshgrid(*y, indexing="ij"), -1) - x[at]
        q = ((d @ U.T) ** 2).sum(-1)
        _check(u, v, q <= 1 + 1e-4, q <= 1 - 1e-4)
    else:  # the box's half-widths are the rows of U^-1
        hw = np.sqrt((np.linalg.inv(U) ** 2).sum(1))
        box = [np.abs(c - x[at, k]) <= hw[k] * (1 + 1e-4) + (c[1] - c[0]) / 2 for k, c in enumerate(y)]
        core = [np.abs(c - x[at, k]) <= (c[1] - c[0]) / 2 for k, c in enumerate(y)]
        f = lambda b: b[0][:, None, None] & b[1][None, :, None] & b[2]  # noqa: E731
        _check(u, v, f(box), f(core))


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("n0", [64, 9])
def test_point_spread_projection(gt, cuda, bad, n0):
    """Pixels narrower and wider than the atoms."""
    n, at, m = 20, 7, (n0, 50)
    I, x, r = _atoms(np.random.default_rng(4), n, bad, at)
    space = gt.AtomSpace(3, isotropic=False)
    T, ortho = gt.spaces.axis_tilt_geometry(np.linspace(-1, 1, 3), [0, 1, 0], ref=np.array([1.0, 0, 0]))
    det = [gt.cell_centres(-1, 1, k) for k in m]
    P = gt.SingleParticleGaussTomo(space, None, gt.ProjSpace(orientations=T, ortho=ortho, detector=det))
    keep = np.arange(n) != at
    u = P(gt.AtomElement(space, x, r, I, device=cuda)).data
    v = P(gt.AtomElement(space, x[keep], r[keep], I[keep], device=cuda)).data
    C = np.linalg.inv(_umat(r[at]))
    C = C @ C.T  # the support's shadow along w has the half-width sqrt(w C w)
    box, core = np.ones((2, 3) + m, bool)
    for a in range(3):
        for k, w in enumerate(ortho):
            hw, s = np.sqrt(w[a] @ C @ w[a]), (det[k][1] - det[k][0]) / 2
            d = np.abs(det[k] - x[at] @ w[a]).reshape((-1, 1) if k == 0 else (1, -1))
            box[a] &= d <= hw * (1 + 1e-4) + s
            core[a] &= d <= s  # the pixel of the centre
    _check(u, v, box, core)


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("planes,m", [(False, (40, 48, 44)), (False, (70, 66, 40)), (True, (40, 48, 44))])
def test_fourier(gt, cuda, bad, planes, m):
    """Planes; a grid for so few atoms without and one with phase tables."""
    fo = importlib.import_module("2018_dictionary_tomography_amd.fourier")
    rng = np.random.default_rng(6)
    n, at = 20, 7
    I, x = rng.uniform(0.5, 1.5, n), rng.uniform(-0.1, 0.1, (n, 3))
    r = np.concatenate((rng.uniform(0.3, 0.9, (n, 3)), rng.normal(0, 0.1, (n, 3))), 1)
    I[at] = bad
    k = [np.arange(c, dtype=np.float32) - c // 2 for c in m]
    if planes:
        T, ortho = gt.spaces.axis_tilt_geometry(np.linspace(-1, 1, 3), [0, 1, 0], ref=np.array([1.0, 0, 0]))
        S = (k[1], k[2], *ortho)
        K = (k[1][None, :, None, None] * ortho[0][:, None, None, :] + k[2][None, None, :, None] * ortho[1][:, None, None, :])
    else:
        S, K = k, np.stack(np.meshgrid(*k, indexing="ij"), -1)
    keep = np.arange(n) != at
    u = fo.evaluate(fo.FTAtoms(I, x, r, device=cuda), S)
    v = fo.evaluate(fo.FTAtoms(I[keep], x[keep], r[keep], device=cuda), S)
    q = ((K @ _umat(r[at])) ** 2).sum(-1)  # |U^T k|^2
    u, v = torch.view_as_real(u), torch.view_as_real(v)
    q = np.broadcast_to(q[..., None], u.shape)
    inner = q <= 30 * (1 - 1e-4)
    # (at k = 0 the phase's sine is exactly 0: 0 times infinity or 0)
    inner = inner & np.broadcast_to((np.abs(K).sum(-1) > 0)[..., None], u.shape)
    _check(u, v, q <= 30 * (1 + 1e-4), inner)
