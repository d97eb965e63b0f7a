"""Accuracy of the hidden products, which run on bf16 matrix cores with operands split into three
parts: against float64 they must be as close as float32 products are.

Each case has its own bound: what the same kernels reached with v_mfma_f32_16x16x4f32 products, over
the same seeds, times 1.03 (the split products reach 0.25 to 1.02 of it). A product of parts left out
shows as 4e-6 or more.

The matrix cores drop low bits of the addends towards minus infinity, which shows where many points'
contributions cancel (random upstream gradients, large batches): parameter gradients were 1.37e-5 off at
262,144 points without the alternating sign of the walk back (walk_sign).
"""

from __future__ import annotations

import math

import pytest
import torch

from gpu_helpers import announce, coordinates, packed, require_gpu_extension, upstream
from oracle import torch_ref

pytestmark = pytest.mark.gpu

SEEDS = range(11, 14)
STEP_SEEDS = range(11, 43)  # a step's error has a part common to its points, which needs more networks
MARGIN = 1.03
HIDDEN = ((192, 4288), (4352, 8448), (8512, 12608))  # the hidden layers' weights

# (batch, scale of the weights): (u, Laplacian). Small-batch kernel, whole tiles, a rest of split tiles.
FORWARD = {
    (1000, 1.0): (5.41e-7, 4.70e-7),
    (1000, 2.0): (4.77e-7, 5.92e-7),
    (8192, 1.0): (5.41e-7, 4.72e-7),
    (8192, 2.0): (4.79e-7, 5.95e-7),
    (16384, 1.0): (5.43e-7, 4.73e-7),
    (16384, 2.0): (4.80e-7, 5.95e-7),
    (16401, 1.0): (5.43e-7, 4.73e-7),
    (16401, 2.0): (4.80e-7, 5.95e-7),
    (65536, 1.0): (5.44e-7, 4.72e-7),
    (65536, 2.0): (4.79e-7, 5.91e-7),
    (70001, 1.0): (5.44e-7, 4.73e-7),
    (70001, 2.0): (4.80e-7, 5.91e-7),
}
# (batch, scale): (all parameters, worst hidden weight block, coordinates).
BACKWARD = {
    (1000, 1.0): (4.74e-7, 4.58e-7, 4.28e-7),
    (1000, 1.5): (4.26e-7, 4.77e-7, 5.49e-7),
    (4096, 1.0): (3.02e-7, 3.21e-7, 4.37e-7),
    (4096, 1.5): (3.15e-7, 3.64e-7, 5.49e-7),
    (8192, 1.0): (4.92e-7, 4.93e-7, 4.32e-7),
    (8192, 1.5): (4.19e-7, 4.53e-7, 5.44e-7),
    (8193, 1.0): (5.66e-7, 6.02e-7, 4.32e-7),
    (8193, 1.5): (6.01e-7, 7.32e-7, 5.48e-7),
    (12289, 1.0): (4.40e-7, 5.23e-7, 4.36e-7),
    (12289, 1.5): (4.32e-7, 5.08e-7, 5.56e-7),
    (65536, 1.0): (5.40e-7, 6.98e-7, 4.37e-7),
    (65536, 1.5): (7.20e-7, 8.58e-7, 5.58e-7),
    (65537, 1.0): (5.17e-7, 6.97e-7, 4.38e-7),
    (65537, 1.5): (5.91e-7, 6.80e-7, 5.57e-7),
    (70001, 1.0): (6.75e-7, 9.71e-7, 4.38e-7),
    (70001, 1.5): (7.80e-7, 9.59e-7, 5.55e-7),
    (262144, 1.0): (1.33e-6, 2.08e-6, 4.38e-7),
    (262144, 1.5): (1.46e-6, 1.85e-6, 5.57e-7),
}
# (batch, boundary, scale): (all parameters, worst hidden weight block). With boundary points the
# interior's residuals vanish and the gradient is the boundary tiles'.
STEP = {
    (1000, 0, 1.0): (8.94e-8, 9.52e-8),
    (1000, 0, 2.0): (1.45e-7, 1.53e-7),
    (8192, 0, 1.0): (9.22e-8, 9.87e-8),
    (8192, 0, 2.0): (1.13e-7, 1.19e-7),
    (16384, 0, 1.0): (9.31e-8, 9.88e-8),
    (16384, 0, 2.0): (1.19e-7, 1.27e-7),
    (16401, 0, 1.0): (9.41e-8, 1.01e-7),
    (16401, 0, 2.0): (1.17e-7, 1.25e-7),
    (70001, 0, 1.0): (8.87e-8, 9.51e-8),
    (70001, 0, 2.0): (1.35e-7, 1.43e-7),
    (1000, 100, 1.0): (1.56e-7, 1.83e-7),
    (1000, 100, 2.0): (1.25e-7, 1.32e-7),
    (4096, 512, 1.0): (1.38e-7, 1.57e-7),
    (4096, 512, 2.0): (1.15e-7, 1.22e-7),
    (16384, 1024, 1.0): (1.30e-7, 1.51e-7),
    (16384, 1024, 2.0): (1.09e-7, 1.16e-7),
    (70001, 500, 1.0): (1.32e-7, 1.54e-7),
    (70001, 500, 2.0): (1.13e-7, 1.20e-7),
}
# (batch, scale), for a source 1 % (of its rms) from the network's own Laplacian, as late in training:
# the forward's own error makes up the gradient's.
FITTED = {
    (1000, 1.0): (1.19e-4, 1.29e-4),
    (1000, 2.0): (1.16e-4, 1.28e-4),
    (8192, 1.0): (3.17e-4, 3.40e-4),
    (8192, 2.0): (2.99e-4, 3.24e-4),
    (16384, 1.0): (4.32e-4, 4.68e-4),
    (16384, 2.0): (4.21e-4, 4.59e-4),
    (16401, 1.0): (4.57e-4, 5.01e-4),
    (16401, 2.0): (4.03e-4, 4.43e-4),
    (70001, 1.0): (9.03e-4, 9.67e-4),
    (70001, 2.0): (7.96e-4, 8.70e-4),
}


@pytest.fixture(scope="module", autouse=True)
def _extension():
    return require_gpu_extension()


def _error(got: torch.Tensor, want: torch.Tensor) -> float:
    return ((got.double() - want).norm() / want.norm()).item()


def _parameter_errors(got: torch.Tensor, want: torch.Tensor) -> list[float]:
    return [_error(got, want), max(_error(got[lo:hi], want[lo:hi]) for lo, hi in HIDDEN)]


def _mean(rows: list[list[float]]) -> list[float]:
    """Geometric means: a network whose u nearly cancels has a large relative error by chance."""
    return [math.exp(sum(math.log(e) for e in column) / len(column)) for column in zip(*rows)]


def forward_errors(batch: int, scale: float) -> list[float]:
    from fused_hoad import fused_forward_laplacian

    rows = []
    for seed in SEEDS:
        p, x = packed(seed, scale), coordinates(batch, seed=seed)
        got = fused_forward_laplacian(x, p)
        rows.append([_error(a, b) for a, b in zip(got, torch_ref.forward_laplacian(p.double(), x.double()))])
    return _mean(rows)


def backward_errors(batch: int, scale: float) -> list[float]:
    from fused_hoad._extension import fused_forward_laplacian_backward

    rows = []
    for seed in SEEDS:
        p, x = packed(seed, scale), coordinates(batch, seed=seed)
        gu, gl = upstream(batch, seed=seed)
        gp, gx = fused_forward_laplacian_backward(x, p, gu, gl)
        flat = p.double().requires_grad_(True)
        points = x.double().requires_grad_(True)
        outputs = torch_ref.forward_laplacian(flat, points)
        want, want_x = torch.autograd.grad(outputs, (flat, points), (gu.double(), gl.double()))
        rows.append([*_parameter_errors(gp, want), _error(gx, want_x)])
    return _mean(rows)


def step_errors(batch: int, boundary: int, scale: float, fitted: bool = False) -> list[float]:
    from fused_hoad import DEFAULT_POISSON_MLP, build_mlp, manufactured_source
    from fused_hoad.training import FusedPoissonAdam

    rows = []
    for seed in STEP_SEEDS:
        p, x = packed(seed, scale), coordinates(batch, seed=seed)
        model = build_mlp(DEFAULT_POISSON_MLP).cuda()
        at = 0
        with torch.no_grad():
            for parameter in model.parameters():
                parameter.copy_(p[at : at + parameter.numel()].view_as(parameter))
                at += parameter.numel()
        flat = p.double().requires_grad_(True)
        _, lap = torch_ref.forward_laplacian(flat, x.double())
        source = lap.detach().float() if boundary else manufactured_source(x)
        if fitted:
            source = (lap.detach() + 0.01 * lap.detach().std() * upstream(batch, seed=seed)[1]).float()
        loss = (lap - source.double()).square().mean()
        edge, weight = None, 1e4
        if boundary:
            edge = coordinates(boundary, seed=seed + 50)
            loss = loss + weight * torch_ref.forward_laplacian(flat, edge.double())[0].square().mean()
        (want,) = torch.autograd.grad(loss, flat)
        trainer = FusedPoissonAdam(model, x, source, boundary=edge, boundary_weight=weight)
        trainer.step()
        rows.append(_parameter_errors(trainer.grad, want))
    return _mean(rows)


def _check(got: list[float], bounds: tuple[float, ...]) -> None:
    print("errors", " ".join(f"{e:.2e}" for e in got), "float32 products", bounds)
    for error, bound in zip(got, bounds, strict=True):
        assert error < MARGIN * bound, (got, bounds)


@pytest.mark.parametrize("batch,scale", FORWARD)
def test_forward_is_as_close_as_float32(batch: int, scale: float) -> None:
    announce(f"forward against float64, batch={batch}, weights x{scale}")
    _check(forward_errors(batch, scale), FORWARD[batch, scale])


@pytest.mark.parametrize("batch,scale", BACKWARD)
def test_cancelling_gradients_are_as_close_as_float32(batch: int, scale: float) -> None:
    announce(f"cancelling gradients against float64, batch={batch}, weights x{scale}")
    _check(backward_errors(batch, scale), BACKWARD[batch, scale])


@pytest.mark.parametrize("batch,boundary,scale", STEP)
def test_step_gradients_are_as_close_as_float32(batch: int, boundary: int, scale: float) -> None:
    announce(f"fused step's gradient against float64, batch={batch}, boundary={boundary}, weights x{scale}")
    _check(step_errors(batch, boundary, scale), STEP[batch, boundary, scale])


@pytest.mark.parametrize("batch,scale", FITTED)
def test_step_gradients_of_a_fitted_network_are_as_close_as_float32(batch: int, scale: float) -> None:
    announce(f"fused step's gradient with small residuals against float64, batch={batch}, weights x{scale}")
    _check(step_errors(batch, 0, scale, fitted=True), FITTED[batch, scale])
