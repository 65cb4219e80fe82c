"""The sums over atoms are carried in FP64: 96 copies of one atom, their
amplitudes 2^20, 1 and -2^20 times one value in any order, give 32 times the
output of the one atom (among 95 of amplitude 0), bit for bit.  (A factor of a power of two scales every
term exactly, and the FP64 sum of terms of 24 bits, at most 26 binary places
apart, is exact in any order; a sum in 24 bits is off by a sixteenth of a term at
each step.)
"""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _copies(rng, I, x, r):
    """The 96 copies, and as many of which all but one have amplitude 0."""
    f = np.tile([2.0 ** 20, 1.0, -(2.0 ** 20)], 32)
    rng.shuffle(f)
    return [(I * a, np.tile(x, (96, 1)), np.tile(r, (96, 1))) for a in (f, np.arange(96) == 50)]


def _same(many, one):
    assert torch.isfinite(one).all() and one.abs().max() > 0
    assert torch.equal(many, 32 * one)


# (widths from a few cells to less than one: every rule of the point-spread cells)
@pytest.mark.parametrize("width", [0.3, 0.08, 0.03])
@pytest.mark.parametrize("op,call", [("GaussTomo", "volume"), ("SingleParticleGaussTomo", "volume"),
                                     ("SingleParticleGaussTomo", "projection")])
def test_renders_and_point_spread_projection(gt, cuda, width, op, call):
    rng = np.random.default_rng(3)
    I, x = np.array([0.75]), rng.uniform(-0.2, 0.2, (1, 3))
    r = np.concatenate((1.0 / (width * rng.uniform(0.8, 1.2, (1, 3))), rng.normal(0, 0.5 / width, (1, 3)) / 3), 1)
    r = r / np.sqrt(60.0) * 2
    space = gt.AtomSpace(3, isotropic=False)
    T, ortho = gt.spaces.axis_tilt_geometry(np.linspace(-1, 1, 3), [0, 1, 0], ref=np.array([1.0, 0, 0]))
    P = gt.ProjSpace(orientations=T, ortho=ortho, detector=[gt.cell_centres(-1, 1, m) for m in (40, 37)])
    A = getattr(gt, op)(space, gt.VolSpace([gt.cell_centres(-1, 1, m) for m in (28, 25, 30)]), P)
    run = A.discretise if call == "volume" else A
    _same(*[run(gt.AtomElement(space, xn, rn, In, device=cuda)).data for In, xn, rn in _copies(rng, I, x, r)])


@pytest.mark.parametrize("planes,m", [(False, (24, 27, 30)), (False, (70, 66, 40)), (True, (24, 27, 30))])
def test_fourier(gt, cuda, planes, m):
    """Planes; a grid for so few atoms without and one with phase tables."""
    fo = importlib.import_module("2018_dictionary_tomography_amd.fourier")
    rng = np.random.default_rng(3)
    I, x = np.array([0.75]), rng.uniform(-0.2, 0.2, (1, 3))
    r = np.concatenate((rng.uniform(0.3, 0.9, (1, 3)), rng.normal(0, 0.1, (1, 3))), 1)
    k = [np.arange(c, dtype=np.float32) - c // 2 for c in m]
    S = k
    if planes:
        T, ortho = gt.spaces.axis_tilt_geometry(np.linspace(-1, 1, 3), [0, 1, 0], ref=np.array([1.0, 0, 0]))
        S = (k[1], k[2], *ortho)
    _same(*[torch.view_as_real(fo.evaluate(fo.FTAtoms(In, xn, rn, device=cuda), S))
            for In, xn, rn in _copies(rng, I, x, r)])
