"""backward="saved" is another name of backward="cuda": the same gradients, bitwise, and nothing more
held between the forward and the backward. (The C pair fhoad_forward_laplacian_saving and
fhoad_forward_laplacian_backward_saved, which checks its buffer and runs the plain kernels, is in
test_c_abi.py.)
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import announce, coordinates, require_gpu_extension

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _extension():
    return require_gpu_extension()


def _model(flatten: bool):
    from fused_hoad import DEFAULT_POISSON_MLP, build_mlp
    from fused_hoad.parameters import flatten_poisson_parameters_

    torch.manual_seed(6)
    model = build_mlp(DEFAULT_POISSON_MLP).cuda()
    if flatten:
        flatten_poisson_parameters_(model)
    return model


@pytest.mark.parametrize("batch", [1, 8192, 8193, 16401, 20000, 65536])
@pytest.mark.parametrize("flatten", [False, True])
@pytest.mark.parametrize("coordinate_grad", [False, True])
def test_saved_mode_gradients_equal_the_cuda_mode(batch: int, flatten: bool, coordinate_grad: bool) -> None:
    """Every parameter's gradient and the coordinate gradient through autograd, for the small-batch
    kernel, 64-point tiles and a rest of split tiles."""
    announce(f"autograd backward='saved' vs 'cuda', batch={batch}, flatten={flatten}, coordinate grad={coordinate_grad}")
    from fused_hoad import manufactured_source
    from fused_hoad.backends.fused import fused_laplacian

    x0 = coordinates(batch, seed=45)
    f = manufactured_source(x0)

    def run(mode: str):
        model = _model(flatten)
        x = x0.clone().requires_grad_(coordinate_grad)
        u, lap = fused_laplacian(model, x, backward=mode)
        ((lap - f).pow(2).mean() + 0.1 * u.pow(2).mean()).backward()
        return [q.grad for q in model.parameters()], x.grad

    want, want_x = run("cuda")
    got, got_x = run("saved")
    torch.cuda.synchronize()
    for index, (a, b) in enumerate(zip(got, want, strict=True)):
        assert torch.equal(a, b), f"parameter {index}"
    if coordinate_grad:
        assert torch.equal(got_x, want_x)


def test_saved_mode_holds_no_layers() -> None:
    """What a forward at 65,536 points leaves allocated until its backward: u and the Laplacian
    (512 KB), as with "cuda", and not 3 KB a point."""
    announce("memory held by backward='saved' and 'cuda', batch=65536")
    from fused_hoad.backends.fused import fused_laplacian

    model, x = _model(True), coordinates(65536, seed=46)

    def held(mode: str) -> int:
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        outputs = fused_laplacian(model, x, backward=mode)
        assert outputs[0].requires_grad
        return torch.cuda.memory_allocated() - before

    assert held("saved") == held("cuda") == 2 * 65536 * 4
