"""Weights and scales that are not what a module's constructor made: strided views, the other FP8 format, tensors on the host.
What was multiplied before is multiplied with the same values, the rest is refused before anything is launched."""

import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2
BOUND = 4e-3                                                                       # one bf16 rounding of sums in another order


def _strided(t):
    """The same values, columns contiguous."""
    return t.t().contiguous().t()


def _step(module, x, dy):
    x = x.clone().requires_grad_()
    y = module(x)
    y.backward(dy)
    return [y.detach(), x.grad] + [p.grad for p in module.parameters()]


def _data(rows, n_in, n_out):
    torch.manual_seed(rows)
    return torch.randn(rows, n_in, device="cuda").bfloat16(), (torch.randn(rows, n_out, device="cuda") * 1e-2).bfloat16()


@pytest.mark.parametrize("scaling,storage", [("grouped", "fp8"), ("mxfp8", "fp8"), ("grouped", "bf16"), ("mxfp8", "fp16"), ("current", "bf16"), ("delayed", "fp16")])
def test_linear_takes_a_strided_weight(scaling, storage):
    import viola_amd
    x, dy = _data(96, 128, 192)
    results = []
    for strided in (False, True):
        torch.manual_seed(1)
        module = viola_amd.nn.Linear(128, 192, device="cuda", dtype=torch.bfloat16, scaling=scaling, weight_dtype=storage)
        if strided:
            module.weight.data = _strided(module.weight.data)
            assert not module.weight.is_contiguous()
        results.append(_step(module, x, dy))
    for got, want in zip(*results):
        assert rel_l2(got, want) < BOUND


@pytest.mark.parametrize("scaling", ["grouped", "current"])
def test_mlp_takes_strided_weights(scaling):
    import viola_amd
    x, dy = _data(64, 128, 128)
    results = []
    for strided in (False, True):
        torch.manual_seed(1)
        module = viola_amd.nn.MLP(128, 192, device="cuda", dtype=torch.bfloat16, scaling=scaling, weight_dtype="bf16")
        if strided:
            module.down.weight.data = _strided(module.down.weight.data)
        results.append(_step(module, x, dy))
    for got, want in zip(*results):
        assert rel_l2(got, want) < 2 * BOUND                                       # dz is rounded on the way


def test_strided_codes_of_a_per_tensor_recipe_are_refused():
    import viola_amd
    x, _ = _data(32, 128, 192)
    module = viola_amd.nn.Linear(128, 192, device="cuda", dtype=torch.bfloat16, scaling="current")
    module.weight.data = _strided(module.weight.data)
    with pytest.raises(AssertionError):
        module(x)


@pytest.mark.parametrize("scaling", ["grouped", "current"])
def test_codes_of_the_other_format(scaling):
    """e5m2 codes in a layer whose recipe names e4m3: the product follows the codes' own type."""
    import viola_amd
    x, _ = _data(96, 128, 192)
    torch.manual_seed(1)
    module = viola_amd.nn.Linear(128, 192, bias=False, device="cuda", dtype=torch.bfloat16, scaling=scaling)
    module.weight.data = (torch.randn(192, 128, device="cuda") * 8).to(E5)
    scale = module.weight_scale.float()
    if scaling == "grouped":
        scale = scale.repeat_interleave(32, 0).repeat_interleave(32, 1)
    with torch.no_grad():
        y = module(x)
    assert rel_l2(y, x.float() @ (module.weight.data.float() * scale).T) < .04      # x is rounded to e4m3: 2^-5 on average


def test_scales_of_another_shape_are_refused():
    import viola_amd
    x, _ = _data(32, 128, 192)
    module = viola_amd.nn.Linear(128, 192, device="cuda", dtype=torch.bfloat16, scaling="grouped")
    module.weight_scale = torch.ones(6, 5, device="cuda")
    with pytest.raises(AssertionError):
        module(x)


def test_tensors_on_the_host_are_refused():
    import viola_amd
    x, dy = _data(32, 128, 192)
    module = viola_amd.nn.Linear(128, 192, dtype=torch.bfloat16, scaling="grouped", weight_dtype="bf16", bias=False)
    with pytest.raises(AssertionError):
        module(x)
    module = viola_amd.nn.Linear(128, 192, device="cuda", dtype=torch.bfloat16, scaling="current")
    module.weight_scale = module.weight_scale.cpu()
    with pytest.raises(AssertionError):
        module(x)
    for scaling in ("grouped", "current"):
        module = viola_amd.nn.Linear(128, 192, device="cuda", dtype=torch.bfloat16, scaling=scaling)
        y = module(x.clone().requires_grad_())
        module.cpu()                                                               # between forward and backward
        with pytest.raises(RuntimeError, match="moved or replaced"):
            y.backward(dy)
    experts = viola_amd.nn.GroupedExperts(2, 128, 64, device="cuda")
    experts.weight_scale = experts.weight_scale.cpu()
    with pytest.raises(RuntimeError, match="weight_scale"):
        experts(x, [16, 16])


def test_experts_follow_the_format_of_their_codes():
    import viola_amd
    x, dy = _data(80, 128, 64)
    counts = [33, 0, 47]
    codes = (torch.randn(3, 64, 128, device="cuda") * 8).to(E5)
    scale = torch.full((3, 2, 4), .25, device="cuda")
    weight = torch.nn.Parameter(codes, requires_grad=False)
    x = x.requires_grad_()
    y = viola_amd.nn.grouped_linear(x, weight, scale, counts, forward_dtype="e4m3", grad_dtype=torch.float32)
    y.backward(dy)
    real = codes.float() * .25
    want_y = torch.cat([rows @ w.T for rows, w in zip(x.detach().float().split(counts), real)])
    want_dx = torch.cat([rows @ w for rows, w in zip(dy.float().split(counts), real)])
    assert rel_l2(y, want_y) < .04 and rel_l2(x.grad, want_dx) < .04
    with pytest.raises(RuntimeError, match="weight_scale"):
        viola_amd.nn.grouped_linear(x, weight, scale[:, :, :3].contiguous(), counts, grad_dtype=torch.float32)


class _Double(torch.nn.Module):
    def forward(self, t):
        return 2 * t


@pytest.mark.parametrize("scaling", ["grouped", "mxfp8", "current"])
@pytest.mark.parametrize("native", [True, False])                                  # False: an option of the general path
def test_parametrized_and_pruned_parameters(scaling, native):
    """weight and bias that are attributes computed from other parameters: the products of the values they have (2 w is exact
    in bf16), gradients to what they come from."""
    import viola_amd
    from torch.nn.utils import parametrize, prune
    x, dy = _data(96, 128, 192)
    options = dict(scaling=scaling, weight_dtype="bf16", **({} if native else dict(saved_input_dtype="bf16")))

    def build():
        torch.manual_seed(1)
        return viola_amd.nn.Linear(128, 192, device="cuda", dtype=torch.bfloat16, **options)

    module, plain = build(), build()
    for name in ("weight", "bias"):
        parametrize.register_parametrization(module, name, _Double())
        getattr(plain, name).data.mul_(2)
    y, dx, *grads = _step(module, x, dy)
    want_y, want_dx, dw, db = _step(plain, x, dy)
    assert torch.equal(y, want_y) and torch.equal(dx, want_dx)
    got = {p.dim(): g for p, g in zip(module.parameters(), grads)}
    assert rel_l2(got[2], 2 * dw) < BOUND and rel_l2(got[1], 2 * db) < BOUND          # in the parameter's own 16 bits

    module, plain = build(), build()
    prune.l1_unstructured(module, "weight", .5)
    plain.weight.data.copy_(module.weight.data)
    y, dx, *_ = _step(module, x, dy)
    want = _step(plain, x, dy)
    assert torch.equal(y, want[0]) and torch.equal(dx, want[1])
    assert rel_l2(module.weight_orig.grad, want[2] * module.weight_mask) < BOUND


@pytest.mark.parametrize("kind", ["linear", "mlp"])
@pytest.mark.parametrize("scaling", ["grouped", "current"])
def test_a_strided_bias_keeps_its_gradient(scaling, kind):
    import viola_amd
    x, dy = _data(64, 128, 192 if kind == "linear" else 128)
    results = []
    for strided in (False, True):
        torch.manual_seed(1)
        cls = viola_amd.nn.Linear if kind == "linear" else viola_amd.nn.MLP
        module = cls(128, 192, device="cuda", dtype=torch.bfloat16, scaling=scaling)
        for name, p in module.named_parameters():
            if strided and name.endswith("bias"):
                p.data = torch.stack([p.data, p.data + 1], 1)[:, 0]
        results.append(_step(module, x, dy))
    for got, want in zip(*results):
        assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(got, want)


@pytest.mark.parametrize("up,down", [(dict(scaling="grouped"), dict(scaling="current")), (dict(scaling="current"), dict(scaling="grouped")),
                                     (dict(scaling="mxfp8"), dict(scaling="current")), (dict(scaling="current"), dict(scaling="mxfp8")),
                                     (dict(scaling="mxfp8"), dict(scaling="grouped")), (dict(scaling="mxfp8"), dict(scaling="mxfp8", forward_dtype="e5m2")),
                                     (dict(scaling="mxfp8"), dict(scaling="mxfp8", quantization_limit=64.))])
@pytest.mark.parametrize("rows,train", [(128, True), (128, False), (8, False), (2048, False)])
def test_mlp_with_a_down_projection_of_another_recipe(up, down, rows, train):
    """An MLP one of whose projections was replaced, against the same two Linears with the float activation between them."""
    import viola_amd
    F = torch.nn.functional
    torch.manual_seed(rows)
    mlp = viola_amd.nn.MLP(128, 256, device="cuda", dtype=torch.bfloat16, **up)
    mlp.down = viola_amd.nn.Linear(256, 128, device="cuda", dtype=torch.bfloat16, **down)
    x, dy = _data(rows, 128, 128)

    def composed(t):
        z = mlp.gate_up(t)
        return mlp.down((F.silu(z[..., :256].float()) * z[..., 256:].float()).to(z.dtype))

    if not train:
        with torch.no_grad():
            assert rel_l2(mlp(x), composed(x)) < .025                             # h may round to the neighbouring code
        return
    results = []
    for call in (mlp, composed):
        t = x.clone().requires_grad_()
        mlp.zero_grad()
        y = call(t)
        y.backward(dy)
        results.append([y.detach(), t.grad] + [p.grad for p in mlp.parameters()])
    for got, want in zip(*results):
        assert rel_l2(got, want) < .04                                            # another e5m2 rounding of dz (2^-3 / sqrt(12) of a few elements)
