"""GPU parity: the kernel of small Linear products against the quantizers' codes multiplied out in double precision."""

import pytest
import torch

from conftest import rel_l2
from viola_amd import _lib

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


def _skinny(x, sx, w, sw, grouped, native, bias, out_dtype, history=None, scale=None):
    m, k, n = x.shape[0], x.shape[1], w.shape[0]
    out = torch.full((m, n), 7.0, device="cuda", dtype=out_dtype)
    status = _lib.call("viola_skinny_linear", _lib.ptr(x), _lib.code(x.dtype), _lib.ptr(sx), m, k, _lib.ptr(w), _lib.code(w.dtype), _lib.ptr(sw), int(grouped), n,
                       float(torch.finfo(w.dtype).max), int(native), _lib.ptr(history), 3, _lib.ptr(scale), _lib.ptr(bias), _lib.code(bias.dtype), _lib.ptr(out),
                       _lib.code(out_dtype), unsupported_ok=True)
    return out if status == 0 else None


@pytest.mark.parametrize("recipe", ["grouped", "mxfp8", "tensor"])
@pytest.mark.parametrize("m,k,n,dtype,formats", [(1, 16, 1, torch.bfloat16, (E4, E4)), (16, 48, 31, torch.float16, (E5, E5)), (17, 1040, 520, torch.bfloat16, (E4, E4)),
                                                 (32, 2080, 8200, torch.bfloat16, (E5, E4)), (5, 4096, 8192, torch.float16, (E4, E5)), (32, 64, 100, torch.bfloat16, (E4, E4)),
                                                 (50, 528, 1000, torch.bfloat16, (E4, E4)), (300, 192, 410, torch.float16, (E5, E4)), (1000, 1040, 250, torch.bfloat16, (E4, E4))])
def test_small_linear(m, k, n, dtype, formats, recipe):
    """Row and k counts around the tiles (16 or 32 rows and columns, 64 k) in every size of tile, odd scale rows; x as codes in both
    formats, and quantized in the kernel: the same result bit for bit, with an Inf and a NaN in x too."""
    from viola_amd.nn import _grouped_kernels as g, _linear_kernels as lk
    torch.manual_seed(m + k + n)
    native = recipe == "mxfp8"
    x = (torch.randn(m, k, device="cuda") * torch.exp2(torch.randint(-6, 6, (m, 1), device="cuda").float())).to(dtype)
    bias = torch.randn(n, device="cuda")
    groups, blocks = -(-k // 32), -(-n // 32)
    for x_format, w_format in {formats, (formats[1], formats[1])}:
        w = torch.randn(n, k, device="cuda").to(w_format)
        history, scale = torch.zeros(8, device="cuda"), torch.zeros(1, device="cuda")
        if recipe == "tensor":
            sw = torch.full((1,), .37, device="cuda")
            sx = lk.tensor_scale(x, history=torch.zeros(8, device="cuda"), index=0, delayed=False, fp8_dtype=x_format)
            q, _ = lk.quantize(x, sx, fp8_dtype=x_format)
            a, b = q.double() * sx.double(), w.double() * sw.double()
        else:
            sw = torch.randint(120, 130, (blocks, groups), device="cuda", dtype=torch.uint8) if native else torch.rand(blocks, groups, device="cuda") + .5
            q, sx = g.quantize(x, x_format, (1, 32), native=native)
            spell = lambda t, s, rows: t.double() * (torch.exp2(s.double() - 127) if native else s.double()).repeat_interleave(rows, 0)[:t.shape[0]].repeat_interleave(32, 1)[:, :k]
            a, b = spell(q, sx, 1), spell(w, sw, 32)
        coded = _skinny(q, sx, w, sw, recipe != "tensor", native, bias, torch.float32)
        assert rel_l2(coded, a @ b.T + bias.double()) < 2e-5
        assert torch.equal(_skinny(q, sx, w, sw, recipe != "tensor", native, bias, torch.bfloat16), coded.bfloat16())
        if x_format != w_format or m * n > 256 * 16 * 32 and m > 32:
            continue
        assert torch.equal(_skinny(x, None, w, sw, recipe != "tensor", native, bias, torch.float32, history, scale), coded)
        if recipe == "tensor":
            assert scale.item() == sx.item() and history[3].item() == x.abs().max().item() and history.count_nonzero() == 1
        else:
            x2 = x.clone()
            x2[0, 5], x2[m - 1, k - 2] = float("nan"), float("inf")
            q, sx = g.quantize(x2, x_format, (1, 32), native=native)
            bits = [t.nan_to_num(nan=123.0) for t in (_skinny(x2, None, w, sw, True, native, bias, torch.float32), _skinny(q, sx, w, sw, True, native, bias, torch.float32))]
            assert torch.equal(*bits)
    assert _skinny(torch.zeros(m, 24, device="cuda", dtype=dtype), None, w, sw, True, native, bias, torch.float32) is None          # k not whole pieces
    big = torch.zeros(8300, k, device="cuda", dtype=torch.uint8).view(E4)
    assert _skinny(big[:4200], sx, big[:100], sw, recipe != "tensor", native, bias, torch.float32) is None                          # too many tiles
