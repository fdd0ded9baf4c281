"""GPU parity: per-tensor and block-scaled products whose last round of 256 x 256 tiles runs on tiles of 128 x 128. Integer operands and
power-of-two scales, so every element must equal the integer product."""

import pytest
import torch

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2

# one and four full rounds; last rounds of 4, 20, 33, 32 and 64 tiles; small tiles partly and wholly outside of the matrix; k that ends in
# either half of a chunk; tests/test_scaled_form.py holds them to the form that they are here for
LAST_ROUND = [(5000, 3300, 2192, (E4, E4)), (2891, 5760, 3072, (E5, E4)), (4100, 4104, 2064, (E4, E5)), (8192, 8448, 1024, (E4, E4)), (4096, 5120, 2048, (E5, E5))]


@pytest.mark.parametrize("scaling", ["tensor", "mx"])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k,formats", LAST_ROUND)
def test_last_round_on_small_tiles(m, n, k, formats, out_dtype, scaling):
    from viola_amd.nn import _grouped_kernels as g, _linear_kernels as lk
    if scaling == "mx":
        k = -(-k // 128) * 128
    torch.manual_seed(m + n + k)
    a, b = torch.randint(-2, 3, (m, k), device="cuda").float(), torch.randint(-2, 3, (n, k), device="cuda").float()
    bias = torch.randint(-8, 9, (n,), device="cuda").float()
    qa, qb = a.to(formats[0]), b.to(formats[1])
    if scaling == "tensor":
        out = lk.gemm(qa, qb, torch.full((1,), 2.0, device="cuda"), torch.full((1,), .5, device="cuda"), out_dtype=out_dtype, bias=bias)
        want = a @ b.T + bias
    else:
        sa = torch.randint(126, 129, (m, k // 32), device="cuda", dtype=torch.uint8)
        sb = torch.randint(126, 129, (n, k // 32), device="cuda", dtype=torch.uint8)
        spell = lambda t, s: t * torch.exp2(s.float() - 127).repeat_interleave(32, 1)
        out = g.gemm(qa, qb, sa, sb, (1, 32), (1, 32), out_dtype=out_dtype, bias=bias, native=True)
        want = spell(a, sa) @ spell(b, sb).T + bias
    assert torch.equal(out, want.to(out_dtype))
