"""torch.autograd bridge for the fused log-likelihood and its hand-written adjoint.

``rr_lnlike(theta, model, obs, sigma)`` returns lnL per parameter vector for
``theta[npv, 7] = (k, t0, p, a, i, c0, c1)`` (c0, c1: quadratic or power-2
coefficients) and back-propagates through the adjoint computed by the same
kernel launch (``RoadRunnerModel.lnlike``), so the flux is never materialised.
"""
import torch

__all__ = ['RRLogLikelihood', 'rr_lnlike']


class RRLogLikelihood(torch.autograd.Function):
    @staticmethod
    def forward(ctx, theta, model, obs, sigma, e=0.0, w=0.0):
        th = theta.detach().resolve_neg()
        if th.dtype is not torch.float64 or th.device != model.device:
            th = th.to(device=model.device, dtype=torch.float64)
        if th.dim() == 2 and th.shape[1] >= 7:
            lnl, g = model._lnlike_device(None, th[:, None, 5:7], None, None, None, None, obs, sigma, e, w, theta=th)
        else:
            k, t0, p, a, i = (th[:, j] for j in range(5))
            lnl, g = model._lnlike_device(k, th[:, 5:7].reshape(-1, 1, 2), t0, p, a, i, obs, sigma, e, w)
        ctx.save_for_backward(g)
        return lnl if lnl.dtype is theta.dtype else lnl.to(theta.dtype)

    @staticmethod
    def backward(ctx, gout):
        (g,) = ctx.saved_tensors
        if gout.dtype is g.dtype:
            return gout[:, None] * g, None, None, None, None, None
        return (gout.to(g.dtype)[:, None] * g).to(gout.dtype), None, None, None, None, None


def rr_lnlike(theta, model, obs, sigma, e=0.0, w=0.0):
    """Differentiable lnL[npv] of ``theta[npv, 7]`` under ``model`` (a RoadRunnerModel
    with set_data called, 'quadratic' or 'power-2' limb darkening)."""
    return RRLogLikelihood.apply(theta, model, obs, sigma, e, w)
