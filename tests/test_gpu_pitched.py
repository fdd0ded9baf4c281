"""Operands at padded row pitches (zero codes past the matrix), which let every product take the kernels that load whole
16-byte pieces, and the modules on sizes that are multiples of nothing, through the native host path."""

import copy

import pytest
import torch

from conftest import rel_l2
from oracle import grouped as og, linear as ol, tensor as ot

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


def _bytes(t):
    return t.detach().cpu().contiguous().view(torch.uint8)


@pytest.mark.parametrize("native", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,cols,q_pitch,qt_pitch", [(1, 1, 128, 128), (65, 72, 128, 128), (127, 129, 256, 128), (200, 64, 64, 256),
                                                        (64, 130, 130, 64), (33, 1000, 1024, 128), (300, 8, 8, 300)])
def test_dual_quantizer_at_a_pitch(rows, cols, q_pitch, qt_pitch, dtype, native):
    """Codes and scales are the oracle's, everything past the matrix is zero codes; either layout may be left out."""
    from viola_amd import _lib
    torch.manual_seed(rows * 1000 + cols)
    x = (torch.randn(rows, cols) * 3).to(dtype)
    xd = x.cuda()
    kind, fmt = (torch.uint8, 1) if native else (torch.float32, 0)
    groups = lambda n: -(-n // 32)

    def call(rowwise, transposed, sums):
        q = torch.full((rows, q_pitch), 0x55, dtype=torch.uint8, device="cuda")
        s = torch.full((rows, groups(q_pitch)), 9, dtype=kind, device="cuda")
        qt = torch.full((cols, qt_pitch), 0x55, dtype=torch.uint8, device="cuda")
        st = torch.full((cols, groups(qt_pitch)), 9, dtype=kind, device="cuda")
        partial = torch.full((groups(rows), cols), float("nan"), device="cuda")
        keep = lambda t, on: _lib.ptr(t) if on else None
        _lib.call("viola_group_quantize_dual_pitched", _lib.ptr(xd), _lib.code(dtype), rows, cols, keep(q, rowwise), q_pitch, keep(s, rowwise),
                  keep(qt, transposed), qt_pitch, keep(st, transposed), _lib.E4M3, 448.0, keep(partial, sums), fmt)
        return q.cpu(), s.cpu(), qt.cpu(), st.cpu(), partial.cpu()

    eq, es = og.quantize(x, E4, (1, 32), native=native)
    eqt, est = og.quantize(x.T.contiguous(), E4, (1, 32), native=native)
    for rowwise, transposed in ((True, True), (True, False), (False, True)):
        q, s, qt, st, partial = call(rowwise, transposed, transposed)
        if rowwise:
            assert torch.equal(q[:, :cols], _bytes(eq)) and (q[:, cols:] == 0).all() and torch.equal(s[:, :groups(cols)], es)
            assert torch.isfinite(s.float()).all()
        if transposed:
            assert torch.equal(qt[:, :rows], _bytes(eqt)) and (qt[:, rows:] == 0).all() and torch.equal(st[:, :groups(rows)], est)
            assert rel_l2(partial.sum(0), x.float().sum(0)) < 1e-5
        if not rowwise:
            assert (q == 0x55).all()
        if not transposed:
            assert (qt == 0x55).all()


@pytest.mark.parametrize("scale_dtype", [torch.float32, torch.uint8])
@pytest.mark.parametrize("batch,rows,cols,pitch", [(1, 4, 4, 128), (3, 70, 33, 128), (2, 128, 64, 128), (1, 1000, 36, 1024)])
def test_transpose_and_repack_at_a_pitch(batch, rows, cols, pitch, scale_dtype):
    from viola_amd import _lib
    torch.manual_seed(rows)
    blocks = lambda n: -(-n // 32)
    x = torch.randint(0, 256, (batch, rows, cols), dtype=torch.uint8)
    scale = torch.randint(1, 200, (batch, blocks(rows), blocks(cols))).to(scale_dtype)
    partial = torch.randn(37, 75)
    fmt = int(scale_dtype == torch.uint8)
    xd, sd, pd = x.cuda(), scale.cuda(), partial.cuda()
    out = torch.full((batch, cols, pitch), 0x55, dtype=torch.uint8, device="cuda")
    so = torch.full((batch, blocks(cols), blocks(pitch)), 7, dtype=scale_dtype, device="cuda")
    total = torch.empty(75, device="cuda")
    _lib.call("viola_codes_transpose_pitched", _lib.ptr(xd), _lib.ptr(out), batch, rows, cols, pitch, _lib.ptr(sd), _lib.ptr(so), 32, 32, fmt, _lib.ptr(pd), 37, 75,
              _lib.ptr(total), _lib.F32)
    assert torch.equal(out.cpu()[..., :rows], x.transpose(1, 2)) and (out[..., rows:] == 0).all()
    assert torch.equal(so.cpu()[..., :blocks(rows)], scale.transpose(1, 2)) and (so[..., blocks(rows):] == 0).all()
    assert rel_l2(total, partial.sum(0)) < 1e-6
    wide = max(pitch, -(-cols // 128) * 128)
    back = torch.full((batch, rows, wide), 0x55, dtype=torch.uint8, device="cuda")
    sb = torch.full((batch, blocks(rows), blocks(wide)), 7, dtype=scale_dtype, device="cuda")
    _lib.call("viola_codes_repack", _lib.ptr(xd), _lib.ptr(back), batch, rows, cols, wide, _lib.ptr(sd), _lib.ptr(sb), 32, 32, fmt)
    assert torch.equal(back.cpu()[..., :cols], x) and (back[..., cols:] == 0).all()
    assert torch.equal(sb.cpu()[..., :blocks(cols)], scale) and (sb[..., blocks(cols):] == 0).all()


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 8), (100, 264), (4099, 512), (700, 9000)])
def test_tensor_encode_equals_its_parts(rows, cols):
    """One call for amax, scale, history and codes, whichever of its launch plans the size takes; the scale and the history
    are the oracle's on the first call, on a delayed later one, and with column sums from the same read."""
    from viola_amd import _lib
    torch.manual_seed(rows)
    x = torch.randn(rows, cols).bfloat16()
    xd = x.cuda()
    pitch, pitch_t = -(-cols // 128) * 128, -(-rows // 128) * 128
    slices = _lib.library().viola_tensor_encode_slices(_lib.BF16, rows, cols)
    work = torch.empty(1024 + slices * cols, device="cuda")
    for index, delayed, sums in ((0, 0, False), (2, 1, False), (3, 0, cols % 8 == 0)):
        old = torch.arange(4.0) * .25
        history, scale = old.cuda(), torch.empty(1, device="cuda")
        q = torch.full((rows, pitch), 0x55, dtype=torch.uint8, device="cuda")
        qt = torch.full((cols, pitch_t), 0x55, dtype=torch.uint8, device="cuda")
        total = torch.empty(cols, device="cuda")
        _lib.call("viola_tensor_encode", _lib.ptr(xd), _lib.BF16, rows, cols, _lib.ptr(work), work.numel(), _lib.ptr(history), 4, index, delayed, 57344.0,
                  _lib.ptr(scale), _lib.ptr(q), pitch, _lib.ptr(qt), pitch_t, _lib.E5M2, _lib.ptr(total) if sums else None, _lib.F32)
        amax = x.float().abs().max()
        expect = torch.clamp_min(old.max() if delayed and index else amax, 1e-30) / 57344.0
        old[index % 4] = amax
        assert torch.equal(scale.cpu()[0], expect) and torch.equal(history.cpu(), old)
        codes = _bytes(ot.quantize(x, expect.reshape(1), E5))
        assert torch.equal(q.cpu()[:, :cols], codes) and (q[:, cols:] == 0).all()
        assert torch.equal(qt.cpu()[:, :rows], codes.T) and (qt[:, rows:] == 0).all()
        if sums:
            assert rel_l2(total, x.float().sum(0)) < 1e-5


@pytest.fixture
def bf16_gradients():
    import viola_amd
    viola_amd.set_gradient_dtype("bf16")
    yield
    viola_amd.precision._settings["gradient_dtype"] = None


@pytest.mark.parametrize("weight_dtype,mode", [("fp8", "memory"), ("fp8", "fast"), ("bf16", "memory"), ("bf16", "fast")])
@pytest.mark.parametrize("scaling", ["grouped", "mxfp8", "current"])
@pytest.mark.parametrize("tokens,n_in,n_out", [(1, 33, 47), (197, 96, 130), (130, 257, 64), (77, 40, 1000)])
def test_linear_on_sizes_that_are_multiples_of_nothing(bf16_gradients, tokens, n_in, n_out, scaling, weight_dtype, mode):
    import viola_amd
    torch.manual_seed(tokens)
    layer = viola_amd.nn.Linear(n_in, n_out, device="cuda", dtype=torch.bfloat16, scaling=scaling, weight_dtype=weight_dtype, mode=mode, backward_dtype="e4m3")
    x, dy = torch.randn(tokens, n_in).bfloat16(), torch.randn(tokens, n_out).bfloat16()
    xg = x.cuda().requires_grad_()
    y = layer(xg)
    y.backward(dy.cuda())
    bias, weight = layer.bias.detach().cpu(), layer.weight.detach().cpu()
    if scaling == "current":
        one = lambda t: ot.tensor_scale(t, torch.zeros(1), 0)[0]
        sx, sg = one(x), one(dy)
        sw = layer.weight_scale.cpu() if weight_dtype == "fp8" else one(weight)
        qw = weight if weight_dtype == "fp8" else ot.quantize(weight, sw, E4)
        qx, qg = ot.quantize(x, sx, E4), ot.quantize(dy, sg, E4)
        want = dict(y=ot.gemm(qx, qw, sx, sw, bias=bias, out_dtype=torch.bfloat16), dx=ot.gemm(qg, qw.T.contiguous(), sg, sw, out_dtype=torch.bfloat16),
                    dw=ot.gemm(qg.T.contiguous(), qx.T.contiguous(), sg, sx, out_dtype=torch.bfloat16))
    else:
        native = scaling == "mxfp8"
        codes, scale = (weight, layer.weight_scale.cpu()) if weight_dtype == "fp8" else og.quantize(weight, E4, (32, 32), native=native)
        want = ol.linear(x, og.dequantize(codes, og.decode_scale(scale), (32, 32)), bias, dy, native=native)
    for got, key in ((y, "y"), (xg.grad, "dx"), (layer.weight.grad, "dw")):
        assert rel_l2(got, want[key]) < 3e-3, key
    assert rel_l2(layer.bias.grad, dy.float().sum(0)) < 3e-3


@pytest.mark.parametrize("scaling", ["grouped", "mxfp8", "current"])
@pytest.mark.parametrize("tokens,n_in,hidden", [(1, 33, 50), (130, 96, 136), (77, 257, 40)])
def test_mlp_on_sizes_that_are_multiples_of_nothing(bf16_gradients, tokens, n_in, hidden, scaling):
    """The one-node MLP against its own two Linears and the float activation between them."""
    import torch.nn.functional as F
    import viola_amd
    torch.manual_seed(tokens)
    mlp, twin = (viola_amd.nn.MLP(n_in, hidden, device="cuda", dtype=torch.bfloat16, scaling=scaling, backward_dtype="e4m3") for _ in range(2))
    twin.load_state_dict(mlp.state_dict())
    x = torch.randn(2, tokens, n_in, device="cuda").bfloat16().requires_grad_()
    dy = torch.randn(2, tokens, n_in, device="cuda").bfloat16()
    mlp(x).backward(dy)
    got = [x.grad] + [p.grad for p in mlp.parameters()]
    x.grad = None
    z = twin.gate_up(x)
    twin.down((F.silu(z[..., :hidden].float()) * z[..., hidden:].float()).to(z.dtype)).backward(dy)
    for a, b in zip(got, [x.grad] + [p.grad for p in twin.parameters()]):
        assert a.shape == b.shape and a.dtype == b.dtype and rel_l2(a, b) < .025
    with torch.no_grad():
        assert torch.equal(copy.deepcopy(mlp)(x), mlp(x))


@pytest.mark.parametrize("counts,n_in,n_out", [([5, 0, 37, 1], 72, 40), ([64, 33], 257, 96), ([0, 0], 64, 64), ([1] * 70, 96, 33)])
def test_variable_groups_on_sizes_that_are_multiples_of_nothing(bf16_gradients, counts, n_in, n_out):
    import viola_amd
    torch.manual_seed(len(counts))
    experts = viola_amd.nn.GroupedExperts(len(counts), n_in, n_out, device="cuda")
    x = torch.randn(sum(counts), n_in).bfloat16()
    dy = torch.randn(sum(counts), n_out).bfloat16()
    xg = x.cuda().requires_grad_()
    y = experts(xg, counts)
    y.backward(dy.cuda())
    begin = 0
    for g, count in enumerate(counts):
        rows = slice(begin, begin + count)
        begin += count
        if count == 0:
            assert (experts.weight.grad[g] == 0).all()
            continue
        w = og.dequantize(experts.weight[g].detach().cpu(), experts.weight_scale[g].cpu(), (32, 32))
        want = ol.linear(x[rows], w, torch.zeros(n_out), dy[rows])
        for got, key in ((y[rows], "y"), (xg.grad[rows], "dx"), (experts.weight.grad[g], "dw")):
            assert rel_l2(got, want[key]) < 4e-3, (g, key)


@pytest.mark.parametrize("tokens,n_in,n_out", [(500, 512, 512), (1001, 1024, 1024), (3001, 1024, 1024), (2049, 512, 512), (1533, 256, 300)])
def test_step_behind_a_ragged_token_count_differs_by_the_order_of_the_sums(bf16_gradients, tokens, n_in, n_out):
    """A padded pitch takes the weight gradient off the guarded kernel, which adds the 32-k groups in ascending order, to kernels
    that for few tiles and k >= 1024 add two halves of the k range separately (and longer ranges than these, several parts:
    test_gpu_k_parts.py). Below that nothing changes. Above it FP32 sums
    differ by about sqrt(k / 32) 2^-24, a bf16 ulp is 2^-8 of the value: one gradient element in 10^4 rounds the other way
    (measured 0.7 to 2.3e-4), one momentum code in 10^5 (at most 2e-5 over 768 x 3072), by one step in the first step. The
    Newton-Schulz products spread that over the update: 1e-4 of the master's norm, and 0.2 to 0.5 % of the FP8 weights lie
    so near a rounding edge that they take the neighbouring code. Bounds are four times what was measured."""
    from viola_amd import nn, optim
    from viola_amd.nn import _grouped_kernels as g

    def build():
        torch.manual_seed(0)
        module = nn.Linear(n_in, n_out, device="cuda", dtype=torch.bfloat16, scaling="grouped", backward_dtype="e4m3")
        optimizer = optim.bind_optimizer(module, optim.FP8Muon(module.parameters(), lr=1e-3, weight_decay=.01))
        return module, optimizer, next(p for p in optimizer.param_groups[0]["params"] if p.dim() == 2)

    torch.manual_seed(10)
    x, dy = torch.randn(tokens, n_in, device="cuda").bfloat16(), (torch.randn(tokens, n_out, device="cuda") * 1e-2).bfloat16()
    gt, sgt = g.quantize_dual(dy, E4, (1, 32))[2:]
    xt, sxt = g.quantize_dual(x, E4, (1, 32))[2:]
    ascending = g.gemm(gt, xt, sgt, sxt, (1, 32), (1, 32), out_dtype=torch.bfloat16)      # rows of `tokens` codes: the guarded kernel
    (a, opt_a, master_a), (b, opt_b, master_b) = build(), build()
    for module in (a, b):
        module(x).backward(dy)
    gradient = a.weight.grad.clone()
    b.weight.grad = ascending.clone()
    opt_a.step()
    opt_b.step()
    differ = lambda p, q: (p != q).float().mean().item()
    codes = [opt.state[master]["momentum_q"] for opt, master in ((opt_a, master_a), (opt_b, master_b))]
    weights = [m.weight.detach().float() for m in (a, b)]
    real = [m.dequantize_weight() for m in (a, b)]
    if -(-tokens // 128) * 128 < 1024:
        assert torch.equal(gradient, ascending) and torch.equal(*codes) and torch.equal(*weights) and torch.equal(master_a, master_b)
        return
    assert rel_l2(gradient, ascending) < 1e-4 and 0 < differ(gradient, ascending) < 1e-3
    assert differ(*codes) < 1e-4 and (codes[0].int() - codes[1].int()).abs().max().item() <= 1
    assert rel_l2(master_a, master_b) < 5e-4
    assert differ(*weights) < .02 and rel_l2(*real) < 5e-3                                # a code step is 1/8 of a value: sqrt(.005) / 16
