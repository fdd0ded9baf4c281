"""What autograd, its hooks and the framework's transforms see of the modules' native path."""

import gc

import pytest
import torch

pytestmark = pytest.mark.gpu
RECIPES = ["grouped", "mxfp8", "current", "delayed"]


CASES = [("linear", s, o) for s in RECIPES for o in (dict(), dict(mode="fast"), dict(weight_dtype="bf16", mode="fast"))] + \
    [("mlp", s, {}) for s in RECIPES] + [("experts", "grouped", {})]


def _build(kind, scaling, options):
    import viola_amd
    torch.manual_seed(2)
    if kind == "experts":
        return viola_amd.nn.GroupedExperts(3, 128, 256, device="cuda")
    cls, width = (viola_amd.nn.Linear, 256) if kind == "linear" else (viola_amd.nn.MLP, 192)
    return cls(128, width, device="cuda", dtype=torch.bfloat16, scaling=scaling, **options)


def _inputs(kind):
    torch.manual_seed(3)
    width = 128 if kind == "mlp" else 256
    return torch.randn(200, 128, device="cuda").bfloat16(), (torch.randn(200, width, device="cuda") * 1e-2).bfloat16(), \
        (([70, 0, 130],) if kind == "experts" else ())


def _gradients(module, x):
    return [x.grad] + [p.grad for p in module.parameters()]


@pytest.mark.parametrize("kind,scaling,options", CASES)
def test_hooks_see_what_is_saved(kind, scaling, options):
    """Everything backward needs goes through the hooks: moved to the host and back it gives the same gradients, and x's codes
    are among it (the only thing as large as they are, beside the weight)."""
    results, packed = [], []

    def pack(t):
        packed.append(t.numel() * t.element_size())
        return t.cpu()

    for hooked in (False, True):
        module, (x, dy, extra) = _build(kind, scaling, options), _inputs(kind)
        x.requires_grad_()
        if hooked:
            with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
                y = module(x, *extra)
        else:
            y = module(x, *extra)
        y.backward(dy)
        results.append([y.detach()] + _gradients(module, x))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    weights = [p.numel() * p.element_size() for p in _build(kind, scaling, options).parameters()]
    assert sum(packed) >= sum(n for n in weights if n > 2048) + 200 * 128


def _held_after_forward(kind, scaling, wrap, rows=1 << 14):
    module, (_, _, extra) = _build(kind, scaling, {}), _inputs(kind)
    x = torch.randn(rows, 128, device="cuda").bfloat16().requires_grad_()
    extra = ([rows // 2, 0, rows // 2],) if extra else ()
    call = (lambda x: module(x, *extra)) if wrap is None else (lambda x: wrap(module, x, *extra))
    call(x)                                                                        # warm
    gc.collect()                                                                   # cycles of earlier tests would be freed below
    held = lambda: torch.cuda.memory_stats()["requested_bytes.all.current"]         # not the sizes of the blocks they came from
    before = held()
    y = call(x)
    return held() - before - y.numel() * y.element_size()


@pytest.mark.parametrize("kind,scaling", [("linear", s) for s in RECIPES] + [("mlp", "grouped"), ("mlp", "current"), ("experts", "grouped")])
def test_checkpointed_and_offloaded_modules_hold_nothing_of_the_batch(kind, scaling):
    from torch.utils.checkpoint import checkpoint

    def offload(module, *args):
        with torch.autograd.graph.save_on_cpu():
            return module(*args)

    codes = (1 << 14) * 128
    assert _held_after_forward(kind, scaling, None) >= codes
    assert _held_after_forward(kind, scaling, lambda m, *a: checkpoint(m, *a, use_reentrant=False)) < codes // 4
    assert _held_after_forward(kind, scaling, offload) < codes // 4


@pytest.mark.parametrize("kind,scaling", [("linear", "grouped"), ("linear", "mxfp8"), ("linear", "current"), ("mlp", "grouped"), ("experts", "grouped")])
def test_checkpoint_gives_the_same_gradients(kind, scaling):
    from torch.utils.checkpoint import checkpoint
    results = []
    for wrapped in (False, True):
        module, (x, dy, extra) = _build(kind, scaling, {}), _inputs(kind)
        x.requires_grad_()
        first = torch.ones(1, device="cuda", dtype=torch.bfloat16, requires_grad=True)
        body = lambda t: module(t * first, *extra) * 1.0
        y = checkpoint(body, x, use_reentrant=False) if wrapped else body(x)
        y.backward(dy)
        results.append([y.detach()] + _gradients(module, x))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["linear", "mlp", "experts"])
def test_errors_of_hooks_keep_their_type(kind):
    class Refused(Exception):
        pass

    def refuse(t):
        raise Refused("no")

    module, (x, dy, extra) = _build(kind, "grouped", {}), _inputs(kind)
    with pytest.raises(Refused), torch.autograd.graph.saved_tensors_hooks(refuse, lambda t: t):
        module(x.requires_grad_(), *extra)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, refuse):
        y = module(x, *extra)
    with pytest.raises(Refused):
        y.backward(dy)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.flatten()[:1]):
        y = module(x, *extra)
    with pytest.raises(RuntimeError, match="moved or replaced|came back changed"):
        y.backward(dy)


def test_a_scale_changed_between_forward_and_backward_is_noticed():
    module, (x, dy, _) = _build("linear", "current", {}), _inputs("linear")
    y = module(x.requires_grad_())
    module.refresh_weight(module._master() * 2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy)


@pytest.mark.parametrize("kind,scaling", [("linear", "grouped"), ("linear", "current"), ("mlp", "grouped"), ("experts", "grouped")])
def test_a_graph_is_freed_by_its_first_backward_pass(kind, scaling):
    module, (x, dy, extra) = _build(kind, scaling, {}), _inputs(kind)
    y = module(x.requires_grad_(), *extra)
    y.backward(dy, retain_graph=True)
    first = [g.clone() for g in _gradients(module, x)]
    for t in [x, *module.parameters()]:
        t.grad = None
    y.backward(dy)
    assert all(torch.equal(a, b) for a, b in zip(first, _gradients(module, x)))
    with pytest.raises(RuntimeError, match="second time"):
        y.backward(dy)


SURFACES = [("linear", s) for s in RECIPES] + [("mlp", "grouped"), ("mlp", "current"), ("experts", "grouped")]


@pytest.mark.parametrize("kind,scaling", SURFACES)
def test_forward_mode_is_refused(kind, scaling):
    """The modules have no forward-mode derivative: a dual input must raise, not lose its tangent."""
    import torch.autograd.forward_ad as forward_ad
    module, (x, _, extra) = _build(kind, scaling, {}), _inputs(kind)
    with forward_ad.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):
            module(forward_ad.make_dual(x, torch.ones_like(x)), *extra)


@pytest.mark.parametrize("kind,scaling", SURFACES)
def test_functorch_transforms_are_refused(kind, scaling):
    module, (x, _, extra) = _build(kind, scaling, {}), _inputs(kind)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.func.grad(lambda t: module(t, *extra).float().sum())(x)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.func.vmap(lambda t: module(x, *extra) + t)(torch.ones(2, 1, device="cuda"))


@pytest.mark.parametrize("kind,scaling", SURFACES[:-1])
def test_tracing_is_refused(kind, scaling):
    """torch.jit has no FP8 types: a trace must fail, not record this input's output as a constant."""
    module, (x, _, _) = _build(kind, scaling, {}), _inputs(kind)
    for p in module.parameters():
        p.requires_grad_(False)
    with pytest.raises(RuntimeError):
        torch.jit.trace(module, x, check_trace=False)
