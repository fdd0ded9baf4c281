"""Any subset of a module's gradients: what is asked for is what the pass that computes all of them gives."""

import itertools

import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
RECIPES = ["grouped", "mxfp8", "current", "delayed"]
# Two routes to one 16-bit gradient: FP32 sums in another order, rounded once to bf16 (half an ulp either way, 2e-3 in the
# 2-norm), and for the gate/up side dz rounded to bf16 before (another one).
BOUND = 4e-3


def _poison(*shapes):
    """Leaves NaN behind in the blocks of these sizes that the allocator hands out next."""
    held = [torch.full(shape, float("nan"), device="cuda", dtype=dtype) for shape in shapes for dtype in (torch.float32, torch.bfloat16)]
    del held


def _backward(build, x, dy, wanted, names):
    """Gradients by name of one step of a fresh module in which only `wanted` is trained."""
    torch.manual_seed(7)
    module, x = build(), x.clone().requires_grad_("x" in wanted)
    parameters = dict(module.named_parameters())
    for name in names:
        if name != "x":
            parameters[name].requires_grad_(name in wanted)
    y = module(x)
    _poison(*(p.shape for p in parameters.values()), x.shape)
    y.backward(dy)
    grads = {name: parameters[name].grad for name in names if name != "x"}
    return y.detach(), dict(grads, x=x.grad), module


@pytest.mark.parametrize("rows,n_in,n_out", [(64, 128, 96), (65, 72, 40), (1100, 256, 512), (33, 64, 45)])
@pytest.mark.parametrize("scaling", RECIPES)
def test_linear_every_combination(scaling, rows, n_in, n_out):
    import viola_amd
    torch.manual_seed(rows)
    build = lambda: viola_amd.nn.Linear(n_in, n_out, device="cuda", dtype=torch.bfloat16, scaling=scaling)
    x, dy = torch.randn(rows, n_in, device="cuda").bfloat16(), (torch.randn(rows, n_out, device="cuda") * 1e-2).bfloat16()
    names = ("x", "weight", "bias")
    y, whole, _ = _backward(build, x, dy, names, names)
    assert rel_l2(whole["bias"], dy.double().sum(0)) < 1e-5                       # FP32 gradients by default
    for wanted in itertools.chain.from_iterable(itertools.combinations(names, n) for n in (1, 2)):
        y_part, part, used = _backward(build, x, dy, wanted, names)
        assert torch.equal(y, y_part)
        for name in names:
            assert (part[name] is not None) == (name in wanted), (wanted, name)
            if name in wanted:
                assert rel_l2(part[name], whole[name]) < BOUND, (wanted, name)
        if scaling in ("current", "delayed"):                                    # the gradient quantizer saw this dy, once
            assert used.grad_quantizer.index == 1 and used.grad_quantizer.history[0].item() == dy.abs().max().item()


@pytest.mark.parametrize("rows,n_in,hidden", [(128, 128, 256), (65, 72, 40)])
@pytest.mark.parametrize("scaling", RECIPES)
def test_mlp_every_combination(scaling, rows, n_in, hidden):
    import viola_amd
    torch.manual_seed(hidden)
    build = lambda: viola_amd.nn.MLP(n_in, hidden, device="cuda", dtype=torch.bfloat16, scaling=scaling)
    x, dy = torch.randn(rows, n_in, device="cuda").bfloat16(), (torch.randn(rows, n_in, device="cuda") * 1e-2).bfloat16()
    names = ("x", "gate_up.weight", "gate_up.bias", "down.weight", "down.bias")
    y, whole, _ = _backward(build, x, dy, names, names)
    for wanted in itertools.chain.from_iterable(itertools.combinations(names, n) for n in range(1, len(names))):
        y_part, part, _ = _backward(build, x, dy, wanted, names)
        assert rel_l2(y_part, y) < BOUND
        for name in names:
            assert (part[name] is not None) == (name in wanted), (wanted, name)
            if name in wanted:
                assert rel_l2(part[name], whole[name]) < BOUND, (wanted, name)
