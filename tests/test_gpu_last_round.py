"""GPU parity: products whose last round of 256 x 256 tiles runs on smaller ones, per-tensor and block-scaled ones on tiles of 128 x 128, grouped
ones on halves or quarters of 256 rows. Integer operands and power-of-two scales, so every element must equal the integer product."""

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


# last rounds of 4, 52 and 64 tiles (quarters), 88, 96 and 128 (halves), 133 (whole); columns that end in a quarter, in front of one, with one;
# k that ends in either half of a chunk
GROUPED_LAST_ROUND = [(5000, 3300, 4112, (E4, E4), torch.bfloat16), (12000, 3072, 768, (E5, E4), torch.float32), (8192, 4608, 1056, (E4, E5), torch.float16),
                      (6100, 6330, 2080, (E4, E4), torch.bfloat16), (8190, 4700, 1040, (E5, E5), torch.float32), (16384, 8704, 400, (E4, E4), torch.bfloat16),
                      (11008, 3840, 2064, (E4, E4), torch.float32)]


@pytest.mark.parametrize("m,n,k,formats,out_dtype", GROUPED_LAST_ROUND)
def test_grouped_last_round(m, n, k, formats, out_dtype):
    from viola_amd.nn import _grouped_kernels as g
    torch.manual_seed(m + n + k)
    a, b, groups = torch.randint(-2, 3, (m, k), device="cuda").float(), torch.randint(-2, 3, (n, k), device="cuda").float(), -(-k // 32)
    scale = lambda rows: torch.exp2(torch.randint(-1, 2, (rows, groups), device="cuda").float())
    sa, sb = scale(m), scale(-(-n // 32))
    bias = torch.randint(-8, 9, (n,), device="cuda").float()
    out = g.gemm(a.to(formats[0]), b.to(formats[1]), sa, sb, (1, 32), (32, 32), out_dtype=out_dtype, bias=bias)
    spell = lambda t, s: t * s.repeat_interleave(32, 1)[:, :k]
    want = spell(a, sa) @ spell(b, sb.repeat_interleave(32, 0)[:n]).T + bias
    assert torch.equal(out, want.to(out_dtype))


# rows of the groups, so that there are four rounds and 16 tiles, two and 96 (halves), five and 8 with empty groups and more of them than 64, one and 44
VARLEN_LAST_ROUND = [([1800] * 14 + [2304, 2100], 2048, 1024), ([4096] * 4 + [1536, 1400], 2048, 2064), ([0, 1] * 33 + [16384, 16200, 0], 2048, 2048),
                     ([5000, 500, 0, 257, 11], 3072, 4096)]


@pytest.mark.parametrize("counts,n,k", VARLEN_LAST_ROUND)
def test_varlen_last_round(counts, n, k):
    import test_gpu_grouped_pingpong as cases
    torch.manual_seed(n + k)
    cases._varlen_products(counts, n, k)
