"""GPU: weight gradients of few tiles, which the modules run in parts of k, through nn.Linear and nn.MLP."""

import pytest
import torch

from conftest import rel_l2
from viola_amd import _lib

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2
IN_PARTS = "viola_group_gemm_in_parts"
# FP32 sums of up to 512 scale groups in another order: one rounding per group, 2^-24 of a total that grows like its square root
SUMS = 2e-6


@pytest.fixture(params=["fp32", "bf16", "fp16"])
def gradient_dtype(request):
    import viola_amd
    viola_amd.set_gradient_dtype(request.param)
    yield {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[request.param]
    viola_amd.precision._settings["gradient_dtype"] = None


def _names(fn):
    """What `fn` returns, and the entry points it called."""
    _lib.timeline = []
    try:
        result = fn()
        torch.cuda.synchronize()
        return result, [name for name, _, _ in _lib.timeline]
    finally:
        _lib.timeline = None


def _codes(t, fmt):
    from viola_amd.nn import _grouped_kernels as g
    return g.quantize(t, fmt, (1, 32), transposed=True)


def _weight_gradient(dy, x, out_dtype):
    """Of these transposed codes by the C entry points alone, rows padded to the host path's pitch; no further from their product in
    float64 than the whole product is."""
    rows, pitch, backward = x[0].shape[1], -(-x[0].shape[1] // 128) * 128, dy[0].dtype
    operands = []
    for q, s in (dy, x):
        wide = torch.zeros(q.shape[0], pitch, device="cuda", dtype=torch.uint8)
        wide[:, :rows] = q.view(torch.uint8)
        scales = torch.ones(q.shape[0], pitch // 32, device="cuda")
        scales[:, :s.shape[1]] = s
        operands.append((wide.view(q.dtype), scales))
    (a, sa), (b, sb) = operands
    m, n = a.shape[0], b.shape[0]
    parts = _lib.library().viola_group_gemm_parts(m, n, pitch)
    assert parts > 1
    out, whole = (torch.empty(m, n, device="cuda", dtype=out_dtype) for _ in range(2))
    workspace = torch.empty(parts * (-(-m * n // 4) * 4), device="cuda")
    head = a.data_ptr(), _lib.code(backward), b.data_ptr(), _lib.code(E4), sa.data_ptr(), sb.data_ptr(), m, n, pitch
    _lib.call(IN_PARTS, *head, out.data_ptr(), _lib.code(out_dtype), parts, workspace.data_ptr(), workspace.numel())
    _lib.call("viola_group_gemm", *head, 1, 32, 1, 32, None, 0, whole.data_ptr(), _lib.code(out_dtype))
    exact = (a.double() * sa.double().repeat_interleave(32, 1)) @ (b.double() * sb.double().repeat_interleave(32, 1)).T
    assert rel_l2(out, exact) <= 1.05 * rel_l2(whole, exact) < 4e-3
    return out


def _values(tokens, n_in, n_out, dtype=torch.bfloat16, seed=0):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(torch.randn(tokens, n, device="cuda", generator=generator).to(dtype) for n in (n_in, n_out))


def _linear(n_in, n_out, dtype=torch.bfloat16, **options):
    import viola_amd
    torch.manual_seed(1)
    return viola_amd.nn.Linear(n_in, n_out, device="cuda", dtype=dtype, scaling="grouped", **options)


# token counts that are whole pieces of 128, of 16 and nothing; the count of parts changes with the shape (17, 3, 8 and 20)
@pytest.mark.parametrize("tokens,n_in,n_out,dtype,options", [(8192, 512, 768, torch.bfloat16, dict(backward_dtype="e4m3")), (9850, 768, 3072, torch.float16, {}),
                                                             (8208, 2048, 512, torch.bfloat16, dict(mode="fast")), (16377, 512, 500, torch.float32, dict(bias=False))])
@pytest.mark.parametrize("wanted", ["all", "weight"])
def test_linear_weight_gradient(gradient_dtype, tokens, n_in, n_out, dtype, options, wanted):
    """The gradient is the C entry point's, bit for bit; the pass's other gradients are what they are without it."""
    x, dy = _values(tokens, n_in, n_out, dtype)
    layer = _linear(n_in, n_out, dtype, **options)
    if wanted == "weight":
        for p in layer.parameters():
            p.requires_grad_(p is layer.weight)
    x.requires_grad_(wanted == "all")
    y = layer(x)
    _, calls = _names(lambda: y.backward(dy))
    assert calls.count(IN_PARTS) == 1
    backward = E4 if options.get("backward_dtype") == "e4m3" else E5
    want = _weight_gradient(_codes(dy, backward), _codes(x.detach(), E4), gradient_dtype)
    assert layer.weight.grad.dtype == gradient_dtype and torch.equal(layer.weight.grad, want)
    if wanted == "all":
        other, x2 = _linear(n_in, n_out, dtype, **options), x.detach().clone().requires_grad_()
        other.weight.requires_grad_(False)
        _, calls = _names(lambda: other(x2).backward(dy))
        assert IN_PARTS not in calls and torch.equal(x.grad, x2.grad)
        if layer.bias is not None:
            assert rel_l2(layer.bias.grad, dy.double().sum(0)) < (SUMS if gradient_dtype == torch.float32 else 4e-3)


def test_mlp_weight_gradients(gradient_dtype):
    """Both projections: h goes to the down one as codes, and dz, the up one's dy, is made as codes in its backward."""
    import viola_amd
    from viola_amd.nn import _gated_kernels, _grouped_kernels as g
    torch.manual_seed(2)
    mlp = viola_amd.nn.MLP(512, 384, 448, activation="silu", scaling="grouped", device="cuda", dtype=torch.bfloat16)
    x, dy = _values(8192, 512, 448)
    x.requires_grad_()
    y = mlp(x)
    _, calls = _names(lambda: y.backward(dy))
    assert calls.count(IN_PARTS) == 2
    with torch.no_grad():
        z = mlp.gate_up(x)
    assert torch.equal(mlp.down.weight.grad, _weight_gradient(_codes(dy, E5), g.gated_quantize_dual(z, "silu", E4)[2:], gradient_dtype))
    h = _gated_kernels.gated_forward(z, "silu")[1].requires_grad_()
    mlp.down(h).backward(dy)
    want = _weight_gradient(_codes(_gated_kernels.gated_backward(z, h.grad, "silu"), E5), _codes(x.detach(), E4), gradient_dtype)
    # (this dz is rounded to bf16 on the way to its codes, the pass's is not: by half an ulp, 2^-9, an E5M2 code in 32 is the neighbouring
    # one, a quarter of a value further at most)
    assert rel_l2(mlp.gate_up.weight.grad, want) < .25 / 32 ** .5


def test_saved_codes_that_come_back_out_of_alignment():
    """A saved-tensor hook may hand the codes back anywhere in memory; the product in parts declines what is not 16-byte aligned and
    the whole product takes it, FP32 sums in another order."""
    x, dy = _values(8192, 512, 768)

    def shifted(t):
        if t.dtype != torch.uint8 or t.dim() != 1:
            return t
        place = torch.empty(t.numel() + 4, device="cuda", dtype=torch.uint8)[4:]
        return place.copy_(t)

    layer, other = _linear(512, 768), _linear(512, 768)
    layer(x).backward(dy)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, shifted):
        y = other(x)
    _, calls = _names(lambda: y.backward(dy))
    assert calls.index(IN_PARTS) == calls.index("viola_group_gemm", calls.index(IN_PARTS)) - 1
    assert not torch.equal(other.weight.grad, layer.weight.grad) and rel_l2(other.weight.grad, layer.weight.grad) < SUMS


@pytest.mark.parametrize("tokens", [8192, 8208, 2064])
def test_general_path_adds_in_the_same_order(tokens):
    """A call that the native host path hands on (here for a weight with strided rows) cuts k at the same places and gives
    the same bits where the token count is whole pieces of 16."""
    x, dy = _values(tokens, 512, 768)
    x.requires_grad_()
    results = []
    for strided in (False, True):
        layer = _linear(512, 768)
        if strided:
            layer.weight.data = layer.weight.data.t().contiguous().t()
        x.grad = None
        _, calls = _names(lambda: layer(x).backward(dy))
        results.append((layer.weight.grad, x.grad, layer.bias.grad, calls))
    (dw, dx, db, native), (dw2, dx2, db2, general) = results
    assert "viola_group_gemm" in general and ("viola_codes_transpose_pitched" in native) and ("viola_codes_transpose_pitched" not in general)
    assert native.count(IN_PARTS) == general.count(IN_PARTS) == (tokens > 4096)
    assert torch.equal(dw, dw2) and torch.equal(dx, dx2) and torch.equal(db, db2)
