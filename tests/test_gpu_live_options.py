"""Options and quantizer state that change after a module's first call count from the next one on."""

import copy

import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _layer(scaling="current", **options):
    import viola_amd
    torch.manual_seed(4)
    return viola_amd.nn.Linear(256, 192, device="cuda", dtype=torch.bfloat16, scaling=scaling, **options)


def _step(layer, x, dy):
    x = x.clone().requires_grad_()
    layer.weight.grad = None
    y = layer(x)
    y.backward(dy)
    return y.detach(), x.grad, layer.weight.grad


def _data():
    torch.manual_seed(5)
    return torch.randn(96, 256, device="cuda").bfloat16(), (torch.randn(96, 192, device="cuda") * 1e-2).bfloat16()


@pytest.mark.parametrize("first,then", [("current", "delayed"), ("delayed", "current")])
def test_scaling_that_comes_with_a_checkpoint(first, then):
    """The quantizers' extra state names the scaling: loading it after a call is the same as loading it before any."""
    x, dy = _data()
    donor = _layer(then)
    _step(donor, 4 * x, 4 * dy)                                                    # a history above this batch's maximum
    state = copy.deepcopy(donor.state_dict())
    used, fresh = _layer(first), _layer(first)
    _step(used, x, dy)
    used.load_state_dict(state)
    fresh.load_state_dict(state)
    for got, want, other in zip(_step(used, x, dy), _step(fresh, x, dy), _step(donor, x, dy)):
        assert torch.equal(got, want) and torch.equal(got, other)
    assert used.input_quantizer.index == fresh.input_quantizer.index == 2


@pytest.mark.parametrize("name,value", [("accum_dtype", "fp16"), ("saved_input_dtype", "bf16"), ("cache_weight_transpose", True)])
@pytest.mark.parametrize("scaling", ["grouped", "current"])
def test_an_option_changed_after_the_first_call(scaling, name, value):
    x, dy = _data()
    options = dict(weight_dtype="bf16", quantization_limit=8.)                     # sums of 256 products stay within FP16
    used, fresh = _layer(scaling, **options), _layer(scaling, **options)
    before = _step(used, x, dy)
    setattr(used, name, value)
    setattr(fresh, name, value)
    after = _step(used, x, dy)
    for got, want in zip(after, _step(fresh, x, dy)):
        assert torch.equal(got, want)
    if name == "accum_dtype":                                                      # FP16 partial sums are another product
        assert not torch.equal(after[0], before[0]) and rel_l2(after[0], before[0]) < .05


@pytest.mark.parametrize("scaling", ["current", "delayed"])
def test_an_empty_batch_leaves_the_quantizers_alone(scaling):
    """It has no maximum: neither the calls counted nor the history change, and the next batch computes what it would have."""
    x, dy = _data()
    used, fresh = _layer(scaling), _layer(scaling)
    empty = torch.empty(0, 256, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    y = used(empty)
    y.backward(torch.empty(0, 192, device="cuda", dtype=torch.bfloat16))
    assert y.shape == (0, 192) and empty.grad.shape == (0, 256) and used.weight.grad.count_nonzero() == 0 and used.bias.grad.count_nonzero() == 0
    assert [q.index for q in (used.input_quantizer, used.grad_quantizer)] == [0, 0]
    for got, want in zip(_step(used, x, dy), _step(fresh, x, dy)):
        assert torch.equal(got, want)
