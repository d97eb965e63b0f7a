"""Gradients through units saturated near tanh = -1, where 1 - tanh^2 is small: it has to come from
1 / (1 + exp(-2 z)) itself (u - u^2 keeps its leading digits there), not from the rounded tanh, whose
square is off by a float32 rounding of 1.

The last hidden layer's biases are -7, so 1 - tanh^2 is about 3e-6 there and every gradient below the
output layer is proportional to it. Its relative error is that of z, a few float32 roundings of a sum
of size 8 (5e-7 each, 1.5e-6 together); sums over points of both signs can cancel to a tenth of their
terms, so 2e-5 of a block's norm bounds the result (measured: up to 5.4e-6; formed from the rounded
tanh, 1.2e-2 to 2.5e-2).
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import announce, coordinates, packed, require_gpu_extension, upstream
from oracle import torch_ref

pytestmark = pytest.mark.gpu

BLOCKS = ((0, 128), (128, 192), (192, 4288), (4288, 4352), (4352, 8448), (8448, 8512), (8512, 12608),
          (12608, 12672))
BOUND = 2e-5


@pytest.fixture(scope="module", autouse=True)
def _extension():
    return require_gpu_extension()


def _saturated() -> torch.Tensor:
    p = packed(0)
    p[12608:12672] = -7.0
    return p


def _check(got: torch.Tensor, want: torch.Tensor) -> None:
    for lo, hi in BLOCKS:
        error = ((got[lo:hi].double() - want[lo:hi]).norm() / want[lo:hi].norm()).item()
        print(f"parameters [{lo}, {hi}): {error:.2e}")
        assert error < BOUND, f"parameters [{lo}, {hi}): {error:.2e}"


@pytest.mark.parametrize("batch,first", [(1000, 0), (8192, 0), (8193, 0), (16384, 0), (16400, 16384), (70001, 0)])
def test_backward_through_saturated_units(batch: int, first: int) -> None:
    """The small-batch kernel, 64-point tiles, and 16-point tiles past the last whole round (16,400
    points with upstream gradients on the last 16 alone)."""
    announce(f"backward through saturated units, batch={batch}, upstream from point {first}")
    from fused_hoad._extension import fused_forward_laplacian_backward

    p, x = _saturated(), coordinates(batch, seed=5)
    gu, gl = upstream(batch, seed=5)
    gu[:first] = 0.0
    gl[:first] = 0.0
    got, got_x = fused_forward_laplacian_backward(x, p, gu, gl)
    flat = p.double().requires_grad_(True)
    points = x.double().requires_grad_(True)
    outputs = torch_ref.forward_laplacian(flat, points)
    want, want_x = torch.autograd.grad(outputs, (flat, points), (gu.double(), gl.double()))
    _check(got, want)
    assert (got_x.double() - want_x).norm() < BOUND * want_x.norm()


@pytest.mark.parametrize("batch,boundary", [(1000, 0), (1000, 100), (16384, 0), (16384, 1024), (16400, 0), (70001, 0), (70001, 500)])
def test_step_through_saturated_units(batch: int, boundary: int) -> None:
    """The fused step's kernels. With boundary points the source is the network's own Laplacian and
    the boundary term's weight is large, so the gradient is the boundary tiles' alone."""
    announce(f"fused step through saturated units, batch={batch}, boundary={boundary}")
    from fused_hoad import DEFAULT_POISSON_MLP, build_mlp
    from fused_hoad.training import FusedPoissonAdam

    p, x = _saturated(), coordinates(batch, seed=6)
    model = build_mlp(DEFAULT_POISSON_MLP).cuda()
    at = 0
    with torch.no_grad():
        for parameter in model.parameters():
            parameter.copy_(p[at : at + parameter.numel()].view_as(parameter))
            at += parameter.numel()
    flat = p.double().requires_grad_(True)
    _, lap = torch_ref.forward_laplacian(flat, x.double())
    source = (lap.detach() if boundary else lap.detach() + upstream(batch, seed=6)[1]).float()
    loss = (lap - source.double()).square().mean()
    edge, weight = None, 1e4
    if boundary:
        edge = coordinates(boundary, seed=7)
        u, _ = torch_ref.forward_laplacian(flat, edge.double())
        loss = loss + weight * u.square().mean()
    (want,) = torch.autograd.grad(loss, flat)
    trainer = FusedPoissonAdam(model, x, source, boundary=edge, boundary_weight=weight)
    trainer.step()
    _check(trainer.grad, want)
