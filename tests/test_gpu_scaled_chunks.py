"""GPU parity: per-tensor and block-scaled products on the alternating-phase tiles whose chunks are 128 k (256 x 256, 256 x 128, and
128 x 128 alone on its CU). Integer operands and power-of-two scales, so every element must equal the integer product."""

import pytest
import torch

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


# k ends in the first half of a chunk, in its second half, with a chunk, inside and with a block of 512 k of scale bytes; fewer chunks
# than stages; ragged rows and columns
@pytest.mark.parametrize("scaling", ["tensor", "mx"])
@pytest.mark.parametrize("m,n,k,formats", [(4096, 1152, 1296, (E4, E4)), (4090, 1150, 1360, (E5, E4)), (4096, 1152, 128, (E4, E5)), (4000, 1100, 256, (E4, E4)),
                                           (2048, 1152, 4624, (E4, E4)), (2000, 1030, 2064, (E5, E5)), (1920, 1920, 640, (E4, E4)), (1921, 1919, 80, (E4, E4)),
                                           (4096, 4096, 1104, (E4, E5)), (4090, 4000, 2128, (E4, E4)), (4000, 4090, 4608, (E5, E5)), (4096, 4096, 384, (E4, E4)),
                                           (9200, 1150, 2064, (E4, E4)), (1152, 9216, 4160, (E5, E4))])
def test_products_in_chunks_of_128(m, n, k, formats, scaling):
    from viola_amd.nn import _grouped_kernels as g, _linear_kernels as lk
    if scaling == "mx":
        k = -(-k // 128) * 128
    torch.manual_seed(m + n + k)
    a, b = torch.randint(-2, 3, (m, k), device="cuda").float(), torch.randint(-2, 3, (n, k), device="cuda").float()
    bias = torch.randint(-8, 9, (n,), device="cuda").float()
    qa, qb = a.to(formats[0]), b.to(formats[1])
    if scaling == "tensor":
        out = lk.gemm(qa, qb, torch.full((1,), 2.0, device="cuda"), torch.full((1,), .5, device="cuda"), out_dtype=torch.bfloat16, bias=bias)
        want = a @ b.T + bias
    else:
        sa = torch.randint(126, 129, (m, k // 32), device="cuda", dtype=torch.uint8)
        sb = torch.randint(126, 129, (n, k // 32), device="cuda", dtype=torch.uint8)
        spell = lambda t, s: t * torch.exp2(s.float() - 127).repeat_interleave(32, 1)
        out = g.gemm(qa, qb, sa, sb, (1, 32), (1, 32), out_dtype=torch.bfloat16, bias=bias, native=True)
        want = spell(a, sa) @ spell(b, sb).T + bias
    assert torch.equal(out, want.bfloat16())
