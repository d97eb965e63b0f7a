"""Infinite and NaN values through the kernels, whose split products (three bf16 parts) turn an infinity
into NaN: the forward forms NaN results again from float32 products, so it agrees with a float32
evaluation; a gradient through an infinity is non-finite, and points do not affect each other.
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import announce, coordinates, knobs, packed, require_gpu_extension, upstream
from oracle import torch_ref

pytestmark = pytest.mark.gpu

# Offsets of a weight of hidden layers 1 and 3 (row 5, column 9) and of layer 2's (row 40, column 63).
WEIGHTS = {1: 192 + 5 * 64 + 9, 2: 4352 + 40 * 64 + 63, 3: 8512 + 5 * 64 + 9}


@pytest.fixture(scope="module", autouse=True)
def _extension():
    return require_gpu_extension()


def _forward(x, p):
    from fused_hoad import fused_forward_laplacian

    return fused_forward_laplacian(x, p, 2)


# The small-batch kernel (one and several tiles a workgroup), whole tiles, and split tiles past them.
@pytest.mark.parametrize("batch,split", [(1, None), (1000, None), (20000, "1"), (16384, "0"), (16401, None), (70001, None)])
@pytest.mark.parametrize("layer,value", [(1, float("inf")), (2, float("-inf")), (3, float("inf")), (2, 8.5e37)])
def test_forward_saturates_at_infinite_weights(batch: int, split: str | None, layer: int, value: float) -> None:
    """z is infinite (8.5e37: huge; the kernels' weight 4 W rounds to an infinite bf16), the tanh
    saturates and u stays finite; the Laplacian is NaN where 1 - tanh^2 = 0 meets an infinity."""
    announce(f"forward with weight {value} in layer {layer}, batch={batch}, FUSED_HOAD_FWD_SPLIT={split}")
    p, x = packed(0), coordinates(batch, seed=3)
    p[WEIGHTS[layer]] = value
    with knobs(**({} if split is None else {"FUSED_HOAD_FWD_SPLIT": split})):
        u, lap = _forward(x, p)
    want_u, want_lap = torch_ref.forward_laplacian(p, x)
    assert torch.isfinite(want_u).all()
    torch.testing.assert_close(u, want_u, atol=1e-5, rtol=1e-4)
    torch.testing.assert_close(lap, want_lap, atol=1e-5, rtol=1e-4, equal_nan=True)


@pytest.mark.parametrize("batch", [64, 16401, 65536])
def test_a_nan_point_leaves_the_others_alone(batch: int) -> None:
    """Coordinates of NaN give NaN at their points; every other point's results are bitwise those of a
    batch without them. An infinite coordinate saturates layer 0 and gives finite results."""
    announce(f"forward and backward with NaN and infinite coordinates, batch={batch}")
    from fused_hoad._extension import fused_forward_laplacian_backward

    p, x = packed(0), coordinates(batch, seed=4)
    gu, gl = upstream(batch, seed=4)
    bad = x.clone()
    bad[5, 0] = float("nan")
    bad[batch - 1, 1] = float("nan")
    bad[7, 0] = float("inf")
    rest = torch.ones(batch, dtype=torch.bool, device="cuda")
    rest[[5, 7, batch - 1]] = False
    u, lap = _forward(x, p)
    bu, bl = _forward(bad, p)
    assert torch.equal(u[rest], bu[rest]) and torch.equal(lap[rest], bl[rest])
    assert torch.isnan(bu[[5, batch - 1]]).all() and torch.isnan(bl[[5, batch - 1]]).all()
    want = torch_ref.forward_laplacian(p, bad[7:8])
    torch.testing.assert_close(bu[7:8], want[0], atol=1e-5, rtol=1e-4)
    torch.testing.assert_close(bl[7:8], want[1], atol=1e-5, rtol=1e-4)
    _, gx = fused_forward_laplacian_backward(x, p, gu, gl)
    gp, bx = fused_forward_laplacian_backward(bad, p, gu, gl)
    assert torch.equal(gx[rest], bx[rest])
    assert torch.isnan(bx[5]).all() and not torch.isfinite(gp[:12736]).any()


@pytest.mark.parametrize("batch", [1000, 16401, 65536])
def test_an_infinite_upstream_gradient_is_not_lost(batch: int) -> None:
    """Wherever float32 arithmetic gives a non-finite gradient, so do the kernels (a hidden weight's is
    NaN here, where float32 products can leave an infinity); other points' coordinate gradients are
    bitwise unaffected."""
    announce(f"backward with an infinite upstream gradient, batch={batch}")
    from fused_hoad._extension import fused_forward_laplacian_backward

    p, x = packed(0), coordinates(batch, seed=5)
    gu, gl = upstream(batch, seed=5)
    _, gx = fused_forward_laplacian_backward(x, p, gu, gl)
    gu[11] = float("inf")
    gp, bx = fused_forward_laplacian_backward(x, p, gu, gl)
    want_p, want_x = torch_ref.recompute_backward(p, x, gu, gl)
    assert not torch.isfinite(gp[~torch.isfinite(want_p)]).any()
    assert not torch.isfinite(bx[~torch.isfinite(want_x)]).any()
    rest = torch.arange(batch, device="cuda") != 11
    assert torch.equal(gx[rest], bx[rest])
