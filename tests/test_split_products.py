"""Accuracy of the hidden products, which run on bf16 matrix cores with operands split into three
parts: against float64 they must be at least as close as float32 products are.

The matrix cores truncate as they accumulate, towards minus infinity, which shows where many
points' contributions cancel: sums of 65,536 points with random upstream gradients, over whole
rounds of 64-point tiles, a rest of split 16-point tiles, and the small-batch kernel.

Bound per gradient block, of the block's norm: what products with v_mfma_f32_16x16x4f32 reached over
these cases, 2.44e-6 (parameters, at 262,144 points) and 6.1e-7 (coordinates). The split products
reach 9.6e-7 and 4.6e-7, and 1.37e-5 for the parameters without the alternating sign of the walk
back (walk_sign), which is what the test is for.
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import announce, coordinates, packed, require_gpu_extension, upstream

pytestmark = pytest.mark.gpu

BLOCKS = ((0, 128), (128, 192), (192, 4288), (4288, 4352), (4352, 8448), (8448, 8512), (8512, 12608),
          (12608, 12672), (12672, 12736))


@pytest.mark.parametrize("batch", [4096, 8192, 8193, 12289, 65536, 65537, 70001, 262144])
@pytest.mark.parametrize("scale", [1.0, 1.5])
def test_cancelling_gradients_are_as_close_as_float32(batch: int, scale: float) -> None:
    announce(f"cancelling gradients against float64, batch={batch}, weights x{scale}")
    require_gpu_extension()
    from fused_hoad._extension import fused_forward_laplacian_backward

    from oracle import torch_ref

    p, x = packed(3, scale), coordinates(batch, seed=7)
    gu, gl = upstream(batch, seed=7)
    gp, gx = fused_forward_laplacian_backward(x, p, gu, gl)
    flat = p.double().requires_grad_(True)
    points = x.double().requires_grad_(True)
    u, lap = torch_ref.forward_laplacian(flat, points)
    want, want_x = torch.autograd.grad((u, lap), (flat, points), (gu.double(), gl.double()))
    for lo, hi in BLOCKS:
        error = (gp[lo:hi].double() - want[lo:hi]).norm() / want[lo:hi].norm()
        assert error < 2.44e-6, f"parameters [{lo}, {hi}): {error:.2e}"
    error = (gx.double() - want_x).norm() / want_x.norm()
    assert error < 6.1e-7, f"coordinates: {error:.2e}"
