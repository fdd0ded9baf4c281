"""Products, scaled matrices and weight updates of several shapes in one launch against the calls that take one shape each, bit for bit, and
the optimizer step that is made of them against one optimizer per parameter."""

import ctypes

import pytest
import torch

from viola_amd import _lib

pytestmark = pytest.mark.gpu


class Product(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in ("a", "b", "residual", "out", "out_diag")] + [(name, ctypes.c_int64) for name in ("batch", "m", "n", "k")] + \
               [("add_diag", ctypes.c_float)] + [(name, ctypes.c_int) for name in ("transpose_b", "epilogue", "transpose_out")] + \
               [("weights", ctypes.c_void_p), ("keep", ctypes.c_float), ("rate", ctypes.c_float)]


class Matrices(ctypes.Structure):
    _fields_ = [("in_", ctypes.c_void_p), ("out", ctypes.c_void_p)] + [(name, ctypes.c_int64) for name in ("batch", "rows", "cols")]


# (batch, m, n, k, transpose_b, b is a, epilogue, second copy, transposed result): edges and remainders of each tile, all kinds in one launch
SMALL = [(1, 8, 8, 8, 1, 1, 0, 0, 0), (2, 64, 64, 72, 1, 1, 1, 1, 0), (1, 72, 136, 72, 0, 0, 2, 0, 1), (3, 40, 40, 200, 0, 1, 1, 0, 0), (1, 65, 72, 64, 1, 0, 2, 0, 0),
         (2, 120, 56, 8, 0, 0, 0, 1, 0), (1, 64, 128, 1024, 0, 0, 2, 0, 0), (1, 136, 136, 64, 1, 1, 1, 0, 1)]
MIDDLE = [(24, 256, 256, 136, 1, 1, 1, 1, 0), (20, 256, 384, 256, 0, 0, 2, 0, 1), (10, 264, 136, 40, 1, 0, 0, 0, 0)]
WIDE = [(24, 384, 384, 200, 1, 1, 1, 0, 0), (40, 192, 576, 192, 0, 0, 2, 0, 1), (12, 384, 192, 72, 0, 0, 1, 0, 0)]
LARGE = [(100, 384, 1152, 384, 0, 0, 2, 0, 1), (128, 384, 384, 72, 0, 0, 0, 0, 0), (150, 768, 192, 40, 0, 0, 1, 0, 0)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [SMALL, MIDDLE, WIDE, LARGE, SMALL[:1]])
def test_products_in_one_launch_equal_one_launch_each(case, dtype):
    torch.manual_seed(len(case))
    rows, outs, wants, held = (Product * len(case))(), [], [], []
    for i, (batch, m, n, k, transpose_b, same, epilogue, second, transpose_out) in enumerate(case):
        a = (torch.randn(batch, m, k, device="cuda") / k ** .5).to(dtype)
        b = a if same else (torch.randn(batch, *((n, k) if transpose_b else (k, n)), device="cuda")).to(dtype)
        if same and not transpose_b:                                          # a . a, square
            a = (torch.randn(batch, m, m, device="cuda") / m ** .5).to(dtype)
            b, k = a, m
        residual = torch.randn(batch, m, n, device="cuda").to(dtype) if epilogue else None
        shape = (batch, n, m) if transpose_out else (batch, m, n)
        got, want = ([torch.full(shape, float("nan"), device="cuda", dtype=dtype) for _ in range(2 if second else 1)] for _ in range(2))
        _lib.call("viola_ns_gemm", _lib.ptr(a), _lib.ptr(b), _lib.ptr(residual), _lib.ptr(want[0]), _lib.code(dtype), transpose_b, epilogue, batch, m, n, k, 3.4445,
                  _lib.ptr(want[1]) if second else None, transpose_out)
        rows[i] = Product(_lib.ptr(a), _lib.ptr(b), _lib.ptr(residual), _lib.ptr(got[0]), _lib.ptr(got[1]) if second else None, batch, m, n, k, 3.4445, transpose_b,
                          epilogue, transpose_out)
        outs += got; wants += want; held += [a, b, residual]
    _lib.call("viola_ns_gemm_many", ctypes.addressof(rows), len(case), _lib.code(dtype))
    for i, (got, want) in enumerate(zip(outs, wants)):
        assert torch.isfinite(want).all() and torch.equal(got, want), i


# (batch, m, n, k, epilogue, transposed weight): edges and remainders of each tile, with a product that is stored in the same launch; 128 x 64 alone
INTO_WEIGHTS = [[(1, 8, 8, 8, 0, 0), (2, 64, 136, 72, 2, 0), (1, 72, 136, 64, 2, 1), (3, 40, 200, 40, 0, 1)], [(20, 256, 384, 256, 2, 1), (24, 264, 136, 40, 0, 0)],
                [(40, 192, 576, 192, 2, 1), (40, 384, 384, 72, 2, 0), (24, 192, 200, 72, 0, 1)], [(100, 384, 1152, 384, 2, 1), (128, 384, 384, 72, 0, 0), (100, 768, 200, 40, 2, 0)], [(1, 1016, 3080, 1016, 2, 1)]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", INTO_WEIGHTS)
def test_products_into_weights_equal_product_and_update(case, dtype):
    torch.manual_seed(len(case))
    lr, decay, scale = .02, .1, 1.7
    f32 = lambda v: torch.tensor(v, dtype=torch.float32)
    keep, rate = (1.0 - f32(lr) * f32(decay)).item(), (f32(lr) * f32(scale)).item()
    rows, pairs, held = (Product * len(case))(), [], []
    for i, (batch, m, n, k, epilogue, transposed) in enumerate(case):
        a, b = (torch.randn(batch, m, k, device="cuda") / k ** .5).to(dtype), torch.randn(batch, k, n, device="cuda").to(dtype)
        residual = torch.randn(batch, m, n, device="cuda").to(dtype) if epilogue else None
        shape = (n, m) if transposed else (m, n)
        weights = [torch.randn(*shape, device="cuda") for _ in range(batch)]
        update = torch.empty(batch, *shape, device="cuda", dtype=dtype)
        _lib.call("viola_ns_gemm", _lib.ptr(a), _lib.ptr(b), _lib.ptr(residual), _lib.ptr(update), _lib.code(dtype), 0, epilogue, batch, m, n, k, 0.0, None, transposed)
        for w, u in zip(weights, update):
            want = w.clone()
            _lib.call("viola_weight_update", _lib.ptr(want), 0, _lib.ptr(u), _lib.code(dtype), w.numel(), lr, decay, scale, 0, 0, 0, 0)
            pairs.append((w, want))
        addresses = torch.tensor([w.data_ptr() for w in weights], device="cuda")
        rows[i] = Product(_lib.ptr(a), _lib.ptr(b), _lib.ptr(residual), None, None, batch, m, n, k, 0.0, 0, epilogue, transposed, addresses.data_ptr(), keep, rate)
        held += [a, b, residual, addresses]
    stored = torch.full((1, 384, 192), float("nan"), device="cuda", dtype=dtype)
    x, y = torch.randn(1, 384, 64, device="cuda").to(dtype), torch.randn(1, 64, 192, device="cuda").to(dtype)
    if len(case) > 1:
        more = (Product * (len(case) + 1))(*rows, Product(_lib.ptr(x), _lib.ptr(y), None, _lib.ptr(stored), None, 1, 384, 192, 64, 0.0, 0, 0, 0, None, 0, 0))
    else:
        more = rows
    _lib.call("viola_ns_gemm_many", ctypes.addressof(more), len(more), _lib.code(dtype))
    for got, want in pairs:
        assert torch.equal(got, want)
    want = torch.empty_like(stored)
    _lib.call("viola_ns_gemm", _lib.ptr(x), _lib.ptr(y), None, _lib.ptr(want), _lib.code(dtype), 0, 0, 1, 384, 192, 64, 0.0, None, 0)
    assert len(case) == 1 or torch.equal(stored, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_scaled_matrices_of_several_shapes_equal_one_shape_each(dtype):
    shapes = [(2, 8, 8), (3, 96, 160), (1, 160, 96), (2, 33, 72), (1, 72, 8), (1, 1024, 64), (2, 512, 1536), (1, 130, 136)]
    torch.manual_seed(4)
    ins = [torch.randn(*s, device="cuda").bfloat16() for s in shapes]
    ins[1][2, 5, 7] = float("nan")
    ins[3][0, 1, 2] = float("inf")
    ins[4].zero_()
    sums = torch.full((256 * sum(s[0] for s in shapes),), float("nan"), device="cuda")
    outs, rows = [torch.zeros(b, min(r, c), max(r, c), device="cuda", dtype=dtype) for b, r, c in shapes], (Matrices * len(shapes))()
    for i, ((b, r, c), x, out) in enumerate(zip(shapes, ins, outs)):
        rows[i] = Matrices(x.data_ptr(), out.data_ptr(), b, r, c)
    _lib.call("viola_ns_prepare_many", ctypes.addressof(rows), len(shapes), _lib.code(dtype), _lib.ptr(sums), 0)
    for (b, r, c), x, out in zip(shapes, ins, outs):
        want = torch.empty_like(out)
        _lib.call("viola_ns_prepare", _lib.ptr(x), _lib.code(torch.bfloat16), _lib.ptr(want), _lib.code(dtype), b, r, c, _lib.ptr(sums))
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), (b, r, c)


@pytest.mark.parametrize("working", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("grads,tile,rounding", [(torch.float32, 256, 0), (torch.bfloat16, 512, 1), (torch.float16, 1024, 0), (torch.float32, 1024, 1)])
def test_momentum_with_sums_of_squares(grads, tile, rounding, working):
    """State and updates are those of viola_momentum_update, one tensor at a time; the sums those of the updates in float64: at most 2^-24 for each of
    the some 40 additions on the way of a term."""
    torch.manual_seed(tile)
    tiles = [1, 5, 16, 300, 4099]
    table, want, got, held = [], [], [], []
    for i, n in enumerate(tiles):
        g = (torch.randn(n * tile, device="cuda") * 1e-2).to(grads)
        q, s = torch.randint(0, 120, (n * tile,), device="cuda", dtype=torch.uint8), torch.rand(n, device="cuda") * 1e-3
        sides = [(q.clone(), s.clone(), torch.zeros(n * tile, device="cuda", dtype=torch.bfloat16)) for _ in range(2)]
        (wq, ws, wu), (gq, gs, gu) = sides
        _lib.call("viola_momentum_update", _lib.ptr(g), _lib.code(grads), _lib.ptr(wq), _lib.ptr(ws), _lib.ptr(wq), _lib.ptr(ws), _lib.ptr(wu), n * tile, .95, 1.0, 1, 0, tile,
                  1, 1, 1, 1, 1, rounding, 3, 77 + i)
        table.append([g.data_ptr(), gq.data_ptr(), gs.data_ptr(), gq.data_ptr(), gs.data_ptr(), gu.data_ptr(), 77 + i, n])
        want.append((wq, ws, wu)); got.append((gq, gs, gu)); held.append(g)
    rows, sums = torch.tensor(table, device="cuda"), torch.full((len(tiles), 256), float("nan"), device="cuda")
    _lib.call("viola_momentum_update_squares", rows.data_ptr(), len(tiles), max(tiles), _lib.code(grads), tile, .95, 1.0, 1, rounding, 3, _lib.code(working), sums.data_ptr())
    for a, b, row in zip(want, got, sums):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
        exact = a[2].to(working).double().square().sum().item()
        assert abs(row.double().sum().item() - exact) <= 40 * 2.0 ** -24 * exact


def test_calls_that_one_launch_does_not_take_are_refused_before_it():
    x = torch.randn(1, 16, 16, device="cuda").bfloat16()
    out = torch.full_like(x, 7.0)
    sums = torch.zeros(256 * 16, device="cuda")
    good = Product(x.data_ptr(), x.data_ptr(), None, out.data_ptr(), None, 1, 16, 16, 16, 0.0, 1, 0, 0)
    odd = Product(x.data_ptr(), x.data_ptr(), None, out.data_ptr(), None, 1, 15, 15, 15, 0.0, 1, 0, 0)          # rows that are no 16-byte pieces
    address = torch.tensor([out.data_ptr()], device="cuda")
    into = lambda *kinds, m=16: Product(x.data_ptr(), x.data_ptr(), x.data_ptr(), None, kinds[3], 1, m, 16, 16, 0.0, *kinds[:3], address.data_ptr(), 1.0, 1.0)
    refused = [into(1, 0, 0, None), into(0, 1, 0, None), into(0, 2, 0, out.data_ptr()), into(0, 2, 1, None, m=12)]
    for rows in ([good, odd], [good] * 9, *([p] for p in refused)):
        assert _lib.call("viola_ns_gemm_many", ctypes.addressof((Product * len(rows))(*rows)), len(rows), _lib.code(torch.bfloat16), unsupported_ok=True) == -2
    for rows in ([Matrices(x.data_ptr(), out.data_ptr(), 1, 16, 15)], [Matrices(x.data_ptr() + 2, out.data_ptr(), 1, 8, 8)], [Matrices(x.data_ptr(), out.data_ptr(), 1, 16, 16)] * 9):
        assert _lib.call("viola_ns_prepare_many", ctypes.addressof((Matrices * len(rows))(*rows)), len(rows), _lib.code(torch.bfloat16), _lib.ptr(sums), 0, unsupported_ok=True) == -2
    torch.cuda.synchronize()
    assert out.eq(7.0).all()


@pytest.mark.parametrize("method", ["standard", "gram"])
@pytest.mark.parametrize("options", [dict(), dict(tile_size=512, nesterov=False, adjust_lr_fn="match_rms_adamw"), dict(rounding="stochastic", rounding_seed=9, ns_steps=3)])
@pytest.mark.parametrize("batched,dtype", [(True, torch.float32), (False, torch.float32), (False, torch.bfloat16)])
def test_step_of_several_shapes_equals_stepping_each_parameter_alone(method, options, batched, dtype):
    """Sets of shapes that step together, wide, tall and square ones, for three steps: with a parameter of two matrices, whose sums of squares are a pass of
    their own, and without, where they come with the momentum, of FP32 and BF16 gradients."""
    import viola_amd
    shapes = [(192, 64), (64, 192), (64, 64), (192, 64), (2, 32, 64), (256, 64), (96, 128), (64, 64)]
    shapes = [s for s in shapes if batched or len(s) == 2]

    def build(one_each):
        torch.manual_seed(3)
        params = [torch.nn.Parameter(torch.randn(*s, device="cuda") * .05) for s in shapes]
        for p in params:
            p.grad_dtype = dtype
        groups = [dict(params=[p], batched=p.dim() == 3) for p in params]
        make = lambda gs: viola_amd.optim.FP8Muon(gs, lr=2e-3, weight_decay=.01, ns_method=method, **options)
        if not one_each:
            return params, [make(groups)]
        optimizers = [make([g]) for g in groups]
        for i, opt in enumerate(optimizers):
            opt.param_groups[0]["viola_parameter_indices"] = [i]
        return params, optimizers

    (together, one), (apart, each) = build(False), build(True)
    for step in range(3):
        torch.manual_seed(50 + step)
        grads = [(torch.randn(*s, device="cuda") * 1e-2).to(dtype) for s in shapes]
        for params, optimizers in ((together, one), (apart, each)):
            for p, g in zip(params, grads):
                p.grad = g.clone()
            for opt in optimizers:
                opt.step()
    assert not one[0]._streams[together[0].device]                            # no lanes: the set went together
    for i, (a, b) in enumerate(zip(together, apart)):
        assert torch.equal(a, b), i
        for key, value in one[0].state[a].items():
            other = each[i].state[b][key]
            assert torch.equal(value, other) if isinstance(value, torch.Tensor) else value == other == 3
