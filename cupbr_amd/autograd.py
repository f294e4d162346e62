"""torch.autograd wrapper of the heterogeneous-medium renderer and its path-replay adjoint.

    render = GridRender(scene, camera, medium, width, height, spp=16, max_depth=6)
    image = render(density, albedo)           # density [nz, ny, nx], albedo [n_surfaces, 3], CUDA
    loss = ((image - target) ** 2).sum()
    loss.backward()                            # density.grad, albedo.grad from the path-replay adjoint

The forward and backward run the HIP kernels of libcupbr on torch's current stream; nothing
is computed by torch except the loss. The proposal grid that drives the real/null collision
decisions is the density's value at the call (detached), or a fixed grid given to the
constructor, so the gradient is that of the same-seed estimate.
"""
from __future__ import annotations

import torch

from . import Camera, CupbrError, GridMedium, GridRenderer, Scene


def _dense(t):
    """The contiguous float32 tensor that the kernels read for t, None when that is t itself."""
    if t is None or (t.is_contiguous() and t.dtype == torch.float32):
        return None
    return t.detach().contiguous().float()


class _GridRenderFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, density, albedo, renderer: GridRenderer, proposal):
        given = (density, albedo, proposal)  # proposal None: the density itself
        dense = tuple(_dense(t) for t in given)
        rho, alb, prop = (t if c is None else c for t, c in zip(given, dense))
        image = renderer.render(rho, alb, proposal=prop)
        ctx.renderer, ctx.forward_id = renderer, renderer.forward_id()
        # the given tensors for autograd's version check, the converted ones for the adjoint
        ctx.save_for_backward(*given, *dense)
        return image

    @staticmethod
    def backward(ctx, grad_image):
        saved = ctx.saved_tensors
        rho, alb, prop = (t if c is None else c for t, c in zip(saved[:3], saved[3:]))
        # The saved tensors cannot have changed since the forward (autograd checks their versions),
        # so the adjoint may reuse the forward pass's per-path radiance when that render was the
        # last one on the scene (its number says so: equal addresses do not, they may have passed on
        # to another tensor); otherwise every path is replayed once more.
        if ctx.forward_id != 0 and ctx.renderer.forward_id() == ctx.forward_id:
            try:
                gd, ga = ctx.renderer.adjoint(rho, alb, grad_image, proposal=prop, from_forward=True)
                return gd, ga, None, None
            except CupbrError:  # a saved-tensor hook has moved them
                pass
        gd, ga = ctx.renderer.adjoint(rho, alb, grad_image, proposal=prop)
        return gd, ga, None, None


class GridRender(torch.nn.Module):
    """Differentiable render of a voxel-density medium and per-surface albedos."""

    def __init__(self, scene: Scene, camera: Camera, medium: GridMedium, width: int, height: int, spp: int = 16,
                 max_depth: int = 6, frame0: int = 0, proposal: torch.Tensor | None = None):
        super().__init__()
        self.renderer = GridRenderer(scene, camera, medium, width, height, spp=spp, max_depth=max_depth,
                                     frame0=frame0)
        self.proposal = proposal

    def forward(self, density: torch.Tensor, albedo: torch.Tensor) -> torch.Tensor:
        if not (density.is_cuda and albedo.is_cuda):
            raise ValueError("GridRender runs on the GPU: density and albedo must be CUDA tensors")
        if tuple(density.shape) != self.renderer.medium.shape:
            raise ValueError(f"density shape {tuple(density.shape)} != medium grid {self.renderer.medium.shape}")
        return _GridRenderFn.apply(density, albedo, self.renderer, self.proposal)
