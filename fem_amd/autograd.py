"""torch.autograd.Function over the engine's C ABI: rho -> C_H with the
element-energy adjoint as backward (fast_fem/FEM3DFun.cpp:222-268 computes
the same dG_ij/dx_e = coef'(x_e) u_i^T K0 u_j for its objective).

Densities on the engine's own device stay there: they are widened to float64 on
the device, and C_H and the gradient are written there
(femh_homogenize_device, femh_gradient_device).  A 128^3 training step spent 6 of
its 23 ms on copies through the host otherwise.  Any other tensor goes through
the host-array entry points."""
import numpy as np
import torch

from .femh import Homogenizer


def _on_device(t, hom):
    return t.is_cuda and t.device.index == hom.opts.device


def _solve(rho, hom):
    """C_H [6,6] of the float64 densities rho (a numpy array, or a device tensor
    of its own that nothing else writes)."""
    if isinstance(rho, np.ndarray):
        C, _ = hom.homogenize(rho)
        C = torch.from_numpy(np.array(C))
    else:
        if rho.numel() != hom.V:
            raise ValueError(f"expected {hom.V} voxels, got {rho.numel()}")
        C = torch.empty((6, 6), dtype=torch.float64, device=rho.device)
        hom.homogenize_device(rho.data_ptr(), C.data_ptr(), torch.cuda.current_stream(rho.device).cuda_stream)
    hom._last_rho = rho
    return C


def _same(a, b):
    if isinstance(a, np.ndarray) or isinstance(b, np.ndarray):
        return isinstance(a, np.ndarray) and isinstance(b, np.ndarray) and np.array_equal(a, b)
    return a is b or (a.shape == b.shape and a.device == b.device and torch.equal(a, b))


class HomogenizeFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rho, hom):
        if _on_device(rho, hom):
            r = rho.detach().to(torch.float64, copy=True).contiguous()
        else:
            r = rho.detach().to("cpu", torch.float64).contiguous().numpy().copy()
        C = _solve(r, hom)
        ctx.hom = hom
        ctx.rho = r
        return C.to(dtype=rho.dtype, device=rho.device)

    @staticmethod
    def backward(ctx, gC):
        hom = ctx.hom
        if getattr(hom, "_last_rho", None) is None or not _same(hom._last_rho, ctx.rho):
            _solve(ctx.rho, hom)  # the context holds the fields of its last solve only
        G = gC.detach().to("cpu", torch.float64).numpy()
        if isinstance(ctx.rho, np.ndarray):
            g = torch.from_numpy(hom.gradient(G))
        else:
            g = torch.empty(hom.shape, dtype=torch.float64, device=ctx.rho.device)
            hom.gradient_device(G, g.data_ptr(), stream_ptr=torch.cuda.current_stream(g.device).cuda_stream)
        return g.to(dtype=gC.dtype, device=gC.device), None


def homogenize(rho: torch.Tensor, hom: Homogenizer) -> torch.Tensor:
    """Differentiable C_H(rho) for a density grid shaped like the context."""
    return HomogenizeFn.apply(rho, hom)
