"""l2_loss over the forms of data it takes: the fused residual (float32 data of
the sinogram's shape) and the general expression give the same loss and
gradients.  The residual has the same bits, so the loss differs by the order of
n positive FP64 terms (n eps) and a gradient that is not rescaled by nothing; a
rescaled one also by the general expression's float32 rounding of the scaled
residual, inside the gradients' 1e-5."""
import importlib

import numpy as np
import pytest
import torch
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu


def _case(gt, dev, N=17, iso=False, dtype=torch.float32):
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    rng = np.random.default_rng(4)
    I, x, r, _ = W.draw_aniso3(max(N, 1), rng, rho=(0.06, 0.1))
    T, ortho, det = W.tilt_series(11, 60.0, det=37)
    space = gt.ProjSpace(orientations=T, ortho=ortho, detector=(det[0], gt.cell_centres(-0.9, 0.9, 29)))
    p = [torch.tensor(v[:N], dtype=dtype, device=dev, requires_grad=True) for v in (I, x, r)]
    data = torch.as_tensor(rng.normal(0, 0.1, (11, 37, 29)), dtype=torch.float32, device=dev)
    return p, space, data


def _general(AG, p, space, data):
    d = AG.project(*p, space) - data
    return 0.5 * (d.double() * d.double()).sum()


FORMS = {
    "plain": lambda d: d,
    "strided": lambda d: d.transpose(0, 2).contiguous().transpose(0, 2),
    "offset": lambda d: torch.cat([d.new_zeros(1), d.reshape(-1)])[1:].view(d.shape),
    "negative view": lambda d: torch.complex(d, -d).conj().imag,
    "float64": lambda d: d.double() + 1e-9,
    "one angle": lambda d: d[:1],
    "scalar": lambda d: d[0, 0, 0],
    "cpu scalar": lambda d: d[0, 0, 0].cpu(),
    "half": lambda d: d.half(),
}


@pytest.mark.parametrize("form", FORMS)
def test_forms(gt, cuda, form):
    AG = importlib.import_module("2018_dictionary_tomography_amd.autograd")
    p, space, data = _case(gt, cuda)
    data = FORMS[form](data)
    loss, ref = AG.l2_loss(*p, space, data), _general(AG, p, space, data)
    assert loss.dtype == ref.dtype and loss.shape == ref.shape
    assert abs(loss.item() - ref.item()) <= 11 * 37 * 29 * 2.0 ** -52 * ref.item()
    got = torch.autograd.grad(loss, p, retain_graph=True)
    for a, b in zip(got, torch.autograd.grad(ref, p, retain_graph=True)):
        assert torch.equal(a, b) and a.dtype == b.dtype
    for a, b in zip(got, torch.autograd.grad(loss, p, retain_graph=True)):
        assert torch.equal(a, b)
    for a, b in zip(torch.autograd.grad(-3.7 * loss, p), torch.autograd.grad(-3.7 * ref, p)):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()


@pytest.mark.parametrize("N", [0, 1, 40])
def test_atoms_types_and_hooks(gt, cuda, N):
    AG = importlib.import_module("2018_dictionary_tomography_amd.autograd")
    for dtype in (torch.float32, torch.float64):
        p, space, data = _case(gt, cuda, N=N, dtype=dtype)
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1],
                                                      lambda t: t.to(cuda)):
            loss = AG.l2_loss(*p, space, data)
        assert data.shape in seen
        keep, ref = data.clone(), _general(AG, p, space, data)
        data.zero_()  # the residual is the one of the forward
        got = torch.autograd.grad(loss, p)
        want = torch.autograd.grad(_general(AG, p, space, keep), p)
        assert all(torch.equal(a, b) and a.dtype == dtype for a, b in zip(got, want))
        assert abs(loss.item() - ref.item()) <= 11 * 37 * 29 * 2.0 ** -52 * ref.item()


def test_derivatives_by_the_data(gt, cuda):
    """Reverse and forward mode in the data, as before through the general expression."""
    AG = importlib.import_module("2018_dictionary_tomography_amd.autograd")
    p, space, data = _case(gt, cuda)
    with torch.no_grad():
        d = AG.project(*p, space) - data
    leaf = data.clone().requires_grad_()
    gd, = torch.autograd.grad(AG.l2_loss(*p, space, leaf), leaf)
    assert torch.equal(gd, -d)
    t = torch.ones_like(data)
    with torch.no_grad(), forward_ad.dual_level():
        out = forward_ad.unpack_dual(AG.l2_loss(*p, space, forward_ad.make_dual(data, t)))
        slope = out.tangent.item()
    want = -(d.double()).sum().item()
    assert abs(slope - want) <= 1e-12 * d.double().abs().sum().item()


@pytest.mark.parametrize("det", [(63, 65), (520, 530)])
def test_residual_value(gt, cuda, det):
    """f below and above the number of partial sums that one block adds."""
    W = importlib.import_module("2018_dictionary_tomography_amd.workloads")
    rng = np.random.default_rng(1)
    I, x, r, _ = W.draw_aniso3(5, rng)
    T, ortho, _ = W.tilt_series(50, 60.0, det=16)
    space = gt.ProjSpace(orientations=T, ortho=ortho, detector=[gt.cell_centres(-1, 1, n) for n in det])
    atoms = gt.AtomElement(gt.AtomSpace(3, isotropic=False), x, r, I, device=cuda)
    data = torch.as_tensor(rng.normal(size=(50,) + det), dtype=torch.float32, device=cuda)
    resid, f = gt.ops.residual(atoms, space, data)
    assert torch.equal(resid, gt.ops.forward(atoms, space) - data)
    want = 0.5 * float((resid.double() ** 2).sum())
    assert abs(float(f) - want) <= resid.numel() * 2.0 ** -52 * want
    with pytest.raises(ValueError):
        gt.ops.residual(atoms, space, data.double())
