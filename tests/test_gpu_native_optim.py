"""The native Newton-Schulz chain against the same chain product by product, and the native optimizer step on parameters
that do not fit the table kernels."""

import pytest
import torch

from viola_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [0, 1, 2, 5])
@pytest.mark.parametrize("method", ["standard", "gram"])
@pytest.mark.parametrize("shape", [(64, 64), (3, 96, 160), (2, 160, 96), (33, 70)])
def test_native_chain_equals_the_products_one_by_one(shape, method, steps):
    from viola_amd.optim import _orthogonalize_kernels as nk
    from viola_amd.optim._orthogonalize import METHODS
    torch.manual_seed(steps)
    x = torch.randn(*shape, device="cuda")
    got, want = METHODS[method](x, steps=steps), nk.run(x, steps, method)
    assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(got, want)


@pytest.mark.parametrize("options", [dict(granularity="block", block_shape=(16, 16)), dict(tile_size=64), dict(tile_size=256, rounding="stochastic")])
def test_native_step_equals_stepping_each_parameter_alone(options):
    """Ragged tiles, small tiles and 2-D blocks go through the per-tensor kernels; a batched 3-D group keeps its matrices;
    bf16 weights round on store. Three steps, bit for bit what one optimizer per parameter gives."""
    import viola_amd
    shapes = [(48, 80), (48, 80), (33, 70), (2, 48, 64), (7,), (7,), (129,)]

    def build(one_each):
        torch.manual_seed(3)
        params = [torch.nn.Parameter((torch.randn(*s, device="cuda") * .05).to(torch.bfloat16 if i == 1 else torch.float32)) for i, s in enumerate(shapes)]
        groups = [dict(params=[p], batched=p.dim() == 3) for p in params]
        make = lambda gs: viola_amd.optim.FP8Muon(gs, lr=2e-3, weight_decay=.01, rounding_seed=9, **options)
        if not one_each:
            return params, [make(groups)]
        optimizers = [make([g]) for g in groups]
        for i, opt in enumerate(optimizers):
            opt.param_groups[0]["viola_parameter_indices"] = [i]
        return params, optimizers

    (together, one), (apart, each) = build(False), build(True)
    for step in range(3):
        torch.manual_seed(50 + step)
        grads = [torch.randn(*s, device="cuda") * 1e-2 for s in shapes]
        for params, optimizers in ((together, one), (apart, each)):
            for i, (p, g) in enumerate(zip(params, grads)):
                p.grad = g.to(p.dtype)
            for opt in optimizers:
                opt.step()
    for i, (a, b) in enumerate(zip(together, apart)):
        assert torch.equal(a, b), i
        for key, value in one[0].state[a].items():
            other = each[i].state[b][key]
            assert torch.equal(value, other) if isinstance(value, torch.Tensor) else value == other == 3


@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("tile,n", [(64, 1), (128, 4095), (256, 70001), (512, 66048), (256, 1 << 20)])
def test_wire_round_trip_in_one_pass_equals_pack_then_unpack(tile, n, fp8):
    """Values and packet bytes, with a short last tile, an Inf and a NaN."""
    torch.manual_seed(n)
    x = torch.randn(n, device="cuda") * torch.exp2(torch.randint(-20, 20, (n,), device="cuda").float())
    if n > 4000:
        x[17], x[n - 1] = float("nan"), float("inf")
    groups = -(-n // tile)
    packets = [torch.zeros((groups * (tile + 4) + 15) // 16 * 16, device="cuda", dtype=torch.uint8) for _ in range(2)]
    got, want = x.clone(), x.clone()
    _lib.call("viola_comm_roundtrip", got.data_ptr(), n, packets[0].data_ptr(), groups, tile, _lib.code(fp8))
    _lib.call("viola_comm_pack", x.data_ptr(), n, packets[1].data_ptr(), 1, groups, tile, _lib.code(fp8))
    _lib.call("viola_comm_unpack", packets[1].data_ptr(), want.data_ptr(), n, 1, groups, tile, _lib.code(fp8), 0)
    assert torch.equal(packets[0], packets[1]) and torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("shape,key", [((64, 128), "momentum_q"), ((64, 128), "momentum_scale"), ((96,), "exp_avg"), ((96,), "exp_avg_sq")])
@pytest.mark.parametrize("how", ["host", "short"])
def test_state_that_is_not_where_the_kernels_read_is_refused(shape, key, how):
    """State offloaded to the host, or cut, must be refused before anything is launched: the kernels read it by address."""
    import viola_amd
    params = [torch.nn.Parameter(torch.randn(*shape, device="cuda")) for _ in range(3)]
    opt = viola_amd.optim.FP8Muon(params, lr=1e-3)
    for p in params:
        p.grad = torch.randn_like(p)
    opt.step()
    state = opt.state[params[1]]
    held = state[key]
    state[key] = held.cpu() if how == "host" else held[:held.numel() // 2]
    before = [p.detach().clone() for p in params]
    with pytest.raises(RuntimeError, match="state of a parameter"):
        opt.step()
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(before, params))
    state[key] = held
    opt.step()


@pytest.mark.parametrize("odd", ["gradient off 16 bytes", "gradient of another type", "weight off 16 bytes", "strided gradient"])
def test_buckets_with_a_member_that_does_not_fit_the_table_kernels(odd):
    """Whole tiles of 256, so a bucket takes one launch over pointer tables; with one odd member each goes alone. Either way two
    steps give what the per-tensor operators give, bit for bit."""
    import viola_amd
    from viola_amd.optim import _kernels as k
    from viola_amd.optim._orthogonalize import METHODS
    torch.manual_seed(8)
    shape, count = (48, 64), 48 * 64

    def shifted(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)

    weights = [torch.randn(*shape, device="cuda") * .05 for _ in range(3)]
    if odd == "weight off 16 bytes":
        weights[1] = shifted(weights[1])
        assert weights[1].data_ptr() % 16
    params = [torch.nn.Parameter(w) for w in weights]
    opt = viola_amd.optim.FP8Muon(params, lr=2e-3, weight_decay=.01, rounding="stochastic", rounding_seed=5)
    twins = [w.detach().clone() for w in weights]
    state = [(torch.zeros(count, device="cuda", dtype=torch.uint8), torch.ones(count // 256, device="cuda")) for _ in params]
    for step in range(2):
        grads = [torch.randn(*shape, device="cuda") * 1e-2 for _ in params]
        if odd == "gradient off 16 bytes":
            grads[1] = shifted(grads[1])
        elif odd == "gradient of another type":
            grads[1] = grads[1].bfloat16()
            params[1].grad_dtype = torch.bfloat16
        elif odd == "strided gradient":
            grads[1] = grads[1].t().contiguous().t()
        for p, g in zip(params, grads):
            p.grad = g
        opt.step()
        for i, (w, g, (q, s)) in enumerate(zip(twins, grads, state)):
            out = torch.empty(count, device="cuda", dtype=torch.bfloat16)
            k.momentum_update(g, q, s, q, s, out, beta=.95, rounding="stochastic", rounding_step=step, rounding_key=(5 + i * 0x9E3779B97F4A7C15) & ((1 << 63) - 1))
            k.weight_update(w, METHODS["standard"](out.view(shape), steps=5), 2e-3, .01, update_scale=.2 * 64 ** .5)
    for p, w, (q, s) in zip(params, twins, state):
        assert torch.equal(opt.state[p]["momentum_q"], q) and torch.equal(opt.state[p]["momentum_scale"], s) and torch.equal(p, w)


def test_operators_read_strided_gradients_in_order():
    """A 1-D gradient with a stride: flattening it is no copy."""
    from viola_amd.optim import _kernels as k
    torch.manual_seed(6)
    n = 512
    grad = torch.randn(n, 2, device="cuda")[:, 0]
    assert not grad.is_contiguous()
    results = []
    for g in (grad, grad.contiguous()):
        w, m, v = torch.ones(n, device="cuda"), torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda")
        k.adam_update(w, g, m, v, lr=1e-2, weight_decay=.01, betas=(.9, .95), eps=1e-8, step=1)
        q, s, out = torch.zeros(n, device="cuda", dtype=torch.uint8), torch.ones(n // 256, device="cuda"), torch.empty(n, device="cuda", dtype=torch.bfloat16)
        k.momentum_update(g, q, s, q, s, out, beta=.95)
        w2 = torch.ones(n, device="cuda")
        k.weight_update(w2, g, 1e-2, .01)
        results.append((w, m, v, q, s, out, w2))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("refused", ["strided matrix", "strided vector", "FP8 parameter"])
def test_a_refused_step_changes_nothing(refused):
    """One parameter that FP8Muon does not update, behind others that it does: the step raises before its first launch."""
    import viola_amd
    torch.manual_seed(9)
    shapes = [(64, 128), (64, 128), (128, 64), (96,)]
    params = [torch.nn.Parameter(torch.randn(*s, device="cuda")) for s in shapes]
    if refused == "strided matrix":
        params.append(torch.nn.Parameter(torch.randn(80, 48, device="cuda").t()))
    elif refused == "strided vector":
        params.append(torch.nn.Parameter(torch.randn(96, 2, device="cuda")[:, 0]))
    else:
        params.append(torch.nn.Parameter(torch.randn(64, 64, device="cuda").to(torch.float8_e4m3fn)))
        params[-1].grad_dtype = torch.float32
    opt = viola_amd.optim.FP8Muon(params[:-1], lr=1e-2)
    for p in params:
        p.grad = torch.randn(p.shape, device="cuda")
    opt.step()
    opt.add_param_group(dict(params=[params[-1]]))
    before = [p.detach().clone() for p in params]
    state = [{key: value.clone() if isinstance(value, torch.Tensor) else value for key, value in opt.state[p].items()} for p in params[:-1]]
    with pytest.raises((RuntimeError, AssertionError)):
        opt.step()
    torch.cuda.synchronize()
    for p, old, kept in zip(params, before, state + [{}]):
        assert torch.equal(p.detach().view(torch.uint8) if p.element_size() == 1 else p, old.view(torch.uint8) if p.element_size() == 1 else old)
        for key, value in kept.items():
            assert torch.equal(opt.state[p][key], value) if isinstance(value, torch.Tensor) else opt.state[p][key] == value
