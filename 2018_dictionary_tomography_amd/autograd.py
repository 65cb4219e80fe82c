"""torch.autograd binding of the projector.

GaussProject.apply(I, x, r, space) returns the sinogram A(theta); its backward
is the hand-written adjoint kernel (gt_derivs in linear mode, order 1), i.e.
the reference's analytic derivative derivs_RadProj / GaussTomo.gradient
(GaussDictCode/bin/NewtonBases.py:954-1069, GaussDictCode/atomFuncs.py:130-144)
applied to the incoming gradient.  Only the atom parameters are saved: the
backward recomputes every per-(atom, angle) detector Gaussian and reduces the
pixel moments again, so no residual x Jacobian intermediates are stored.
"""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import ops


class _Atoms:
    def __init__(self, I, x, r):
        self.I, self.x, self.r = I, x, r


class GaussProject(torch.autograd.Function):
    @staticmethod
    def forward(ctx, I, x, r, space):
        I32, x32, r32 = (t.detach().to(torch.float32).contiguous() for t in (I, x, r))
        R = ops.forward(_Atoms(I32, x32, r32), space)
        ctx.save_for_backward(I32, x32, r32)
        ctx.space = space
        ctx.dtypes = (I.dtype, x.dtype, r.dtype)
        return R

    @staticmethod
    def backward(ctx, grad_R):
        I32, x32, r32 = ctx.saved_tensors
        dim = x32.shape[1]
        _, g, _ = ops.derivs(_Atoms(I32, x32, r32), ctx.space, grad_R.contiguous(), "linear", order=1,
                             want_f=False)
        gI = g[:, 0].to(ctx.dtypes[0])
        gx = g[:, 1:1 + dim].to(ctx.dtypes[1])
        gr = g[:, 1 + dim:].to(ctx.dtypes[2])
        return gI, gx, gr, None


class GaussL2(torch.autograd.Function):
    """1/2 ||A(theta) - data||^2: the forward saves the residual, and since the
    gradient is linear in it, the backward walks it and scales the result.

    5000 atoms, 90 x 256^2: five elementwise passes and a reduction over the
    residual in FP64, with a 47 MB copy of it, become sums in the projection
    kernel (a step 3664 -> 3542 us); 300 atoms, 45 x 96 x 83: 8 launches fewer
    (237 -> 188 us)."""

    @staticmethod
    def forward(ctx, I, x, r, space, data):
        I32, x32, r32 = (t.detach().to(torch.float32).contiguous() for t in (I, x, r))
        resid, f = ops.residual(_Atoms(I32, x32, r32), space, data)
        ctx.save_for_backward(I32, x32, r32, resid)
        ctx.space = space
        ctx.dtypes = (I.dtype, x.dtype, r.dtype)
        return f

    @staticmethod
    def backward(ctx, grad_f):
        I32, x32, r32, resid = ctx.saved_tensors
        dim = x32.shape[1]
        _, g, _ = ops.derivs(_Atoms(I32, x32, r32), ctx.space, resid, "linear", order=1, want_f=False)
        grad_f = grad_f.detach()
        parts = (g[:, 0], g[:, 1:1 + dim], g[:, 1 + dim:])
        return tuple(torch.mul(p, grad_f, out=p.new_empty(p.shape, dtype=d))
                     for p, d in zip(parts, ctx.dtypes)) + (None, None)


def project(I, x, r, space):
    """Differentiable sinogram of atoms (I, x, r) in `space`."""
    return GaussProject.apply(I, x, r, space)


def _plain_float32(data, like):
    """data is a float32 tensor of its own that nothing is differentiated by."""
    return (type(data) is torch.Tensor and data.dtype == torch.float32 and data.device == like.device
            and data.layout == torch.strided and not data.requires_grad
            and forward_ad.unpack_dual(data).tangent is None)


def l2_loss(I, x, r, space, data):
    """1/2 ||A(theta) - data||^2 (transport_loss.l2_squared_loss, :567-585), differentiable."""
    # the residual's sum of squares comes from the projection kernel where
    # R - data is a float32 difference of equal shapes; other types (a float64
    # difference), broadcast data and derivatives by the data go the general way
    if _plain_float32(data, I) and tuple(data.shape) == tuple(ops.device_geometry(space, I.device).shape):
        return GaussL2.apply(I, x, r, space, data.resolve_neg().contiguous())
    R = project(I, x, r, space)
    d = R - data
    return 0.5 * (d.double() * d.double()).sum()
