"""GPU parity: the large-tile form of the grouped-scale products (256 x 256, row-wise b scales 256 x 128) at its edges.

Integer operands and power-of-two scales throughout, so that the sums are exact in FP32 and every element must equal the integer
product, rounded once where the output is narrower. test_group_form.py holds these shapes to the kernels they are here for."""

import pytest
import torch

from viola_amd import _lib

pytestmark = pytest.mark.gpu
E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


def _integers(*shape):
    return torch.randint(-2, 3, shape, device="cuda").float()


def _scales(*shape):
    return torch.exp2(torch.randint(-1, 2, shape, device="cuda").float())


def _spell(t, s, rows):
    return t * s.repeat_interleave(rows, 0)[:t.shape[0]].repeat_interleave(32, 1)[:, :t.shape[1]]


# rows and columns short of the last tile, columns whose rows of the output are 16-byte aligned or not; k that ends inside a chunk
# of 64, inside a piece of four scales and inside a block of eight
LARGE = [(4090, 4070, 2064, (E4, E4), torch.float32), (4096, 4096, 1536, (E5, E4), torch.bfloat16),
         (4001, 4072, 2272, (E4, E5), torch.float16), (8190, 8180, 2592, (E5, E5), torch.bfloat16)]


@pytest.mark.parametrize("gb", [(32, 32), (1, 32)])
@pytest.mark.parametrize("m,n,k,formats,out_dtype", LARGE)
def test_grouped_products_on_large_tiles(m, n, k, formats, out_dtype, gb):
    from viola_amd.nn import _grouped_kernels as g
    torch.manual_seed(m + n + k)
    a, b, groups = _integers(m, k), _integers(n, k), -(-k // 32)
    sa, sb = _scales(m, groups), _scales(-(-n // gb[0]), groups)
    bias = torch.randint(-8, 9, (n,), device="cuda").float()
    out = g.gemm(a.to(formats[0]), b.to(formats[1]), sa, sb, (1, 32), gb, out_dtype=out_dtype, bias=bias)
    assert torch.equal(out, (_spell(a, sa, 1) @ _spell(b, sb, gb[0]).T + bias).to(out_dtype))


LARGE_LEAK_K = [1568, 1824]                                                  # 49 and 57 groups: one scale in the last piece, and in the last block


@pytest.mark.parametrize("gb", [(32, 32), (1, 32)])
@pytest.mark.parametrize("k", LARGE_LEAK_K)
def test_scales_of_the_next_row_do_not_leak_on_large_tiles(gb, k):
    """The piece that holds a row's last scales reaches into the next row's: a NaN or an Inf there stays in its own row."""
    from viola_amd.nn import _grouped_kernels as g
    torch.manual_seed(k)
    m, n = 4096, 4096
    a, b = _integers(m, k), _integers(n, k)
    sa, sb = _scales(m, k // 32), _scales(n // gb[0], k // 32)
    clean = g.gemm(a.to(E4), b.to(E4), sa, sb, (1, 32), gb, out_dtype=torch.float32)
    bad = [7, 256, 4095]
    sa[bad, 0] = torch.tensor([float("nan"), float("inf"), float("nan")], device="cuda")
    out = g.gemm(a.to(E4), b.to(E4), sa, sb, (1, 32), gb, out_dtype=torch.float32)
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[bad] = False
    assert torch.equal(out[keep], clean[keep]) and not torch.isfinite(out[bad]).all()
    sa[bad, 0] = 1.0
    base = g.gemm(a.to(E4), b.to(E4), sa, sb, (1, 32), gb, out_dtype=torch.float32)
    row = 65
    sb[row, 0] = float("nan")
    out = g.gemm(a.to(E4), b.to(E4), sa, sb, (1, 32), gb, out_dtype=torch.float32)
    inside = torch.arange(n, device="cuda") // gb[0] == row
    assert torch.equal(out[:, ~inside], base[:, ~inside]) and torch.isnan(out[:, inside]).all()


VARLEN_LARGE, VARLEN_LARGE_SIZE = [[7500, 0, 1, 7400, 256, 15843, 0], [1000] * 66], (1000, 2048)


def _varlen_products(counts, n, k):
    """viola_varlen_group_gemm on these groups of rows, every element against the exact product."""
    groups, total = len(counts), sum(counts)
    a, b = _integers(total, k), _integers(groups, n, k)
    offsets = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], device="cuda")
    sa, sb = _scales(total, -(-k // 32)), _scales(groups, -(-n // 32), -(-k // 32))
    out, qa, qb = torch.full((total, n), 7.0, device="cuda"), a.to(E4), b.to(E4)
    _lib.call("viola_varlen_group_gemm", qa.data_ptr(), _lib.code(E4), qb.data_ptr(), _lib.code(E4), sa.data_ptr(), sb.data_ptr(), offsets.data_ptr(),
              groups, total, n, k, 1, 32, 32, 32, n * k, sb[0].numel(), out.data_ptr(), 0)
    row = 0
    for g, c in enumerate(counts):
        assert torch.equal(out[row:row + c], _spell(a[row:row + c], sa[row:row + c], 1) @ _spell(b[g], sb[g], 32).T)
        row += c


@pytest.mark.parametrize("counts", VARLEN_LARGE)
def test_varlen_products_on_large_tiles(counts):
    """Row ranges per group (more groups than a count of 64 covers in the second case), empty ones among them."""
    torch.manual_seed(len(counts))
    _varlen_products(counts, *VARLEN_LARGE_SIZE)


# one round of 256 x 128 tiles in chunks of 128 k: k that ends with a chunk, in each quarter of one and inside a slot of 32; ragged rows and columns
TALL = [(8192, 1024, 2048, torch.bfloat16), (8000, 1000, 2064, torch.float32), (5000, 900, 2144, torch.float16),
        (3000, 2304, 2208, torch.bfloat16), (2304, 2250, 1968, torch.float32), (16384, 512, 1792, torch.bfloat16)]


@pytest.mark.parametrize("m,n,k,out_dtype", TALL)
def test_grouped_products_on_one_round_of_tall_tiles(m, n, k, out_dtype):
    """(with a row's first scale a NaN, which the piece of the row before's last ones reaches into)"""
    from viola_amd.nn import _grouped_kernels as g
    torch.manual_seed(m + n + k)
    a, b, groups = _integers(m, k), _integers(n, k), -(-k // 32)
    sa, sb = _scales(m, groups), _scales(-(-n // 32), groups)
    bias = torch.randint(-8, 9, (n,), device="cuda").float()
    want = _spell(a, sa, 1) @ _spell(b, sb, 32).T + bias
    sa[7, 0], sb[-1, 0] = float("nan"), float("inf")
    out = g.gemm(a.to(E5), b.to(E4), sa, sb, (1, 32), (32, 32), out_dtype=out_dtype, bias=bias)
    rows, columns = torch.arange(m, device="cuda") != 7, (n - 1) // 32 * 32
    assert torch.equal(out[rows, :columns], want[rows, :columns].to(out_dtype)) and torch.isnan(out[7]).all()


# row ranges per group, empty ones among them; k that ends with a chunk, and in its first and third quarter
VARLEN_TALL = [([2900, 0, 1, 3000, 256], 1000, 4192), ([2900, 0, 1, 3000, 256], 900, 4112), ([700, 0, 255, 257, 2884], 1024, 4224)]


@pytest.mark.parametrize("counts,n,k", VARLEN_TALL)
def test_varlen_products_on_one_round_of_tall_tiles(counts, n, k):
    torch.manual_seed(k)
    _varlen_products(counts, n, k)


VARLEN_WGRAD = [0, 2080, 32, 4096, 1952, 0, 2176], 2040, 4000                # slots of the groups, rows and columns of the gradients


def test_varlen_weight_gradient_on_large_tiles():
    """k ranges per group: none, one slot of 32, ranges that end inside a chunk; ragged rows and columns."""
    torch.manual_seed(3)
    slots, n, kout = VARLEN_WGRAD
    offsets = torch.tensor([0, *torch.tensor(slots).cumsum(0).tolist()], device="cuda")
    total = -(-sum(slots) // 128) * 128
    a, b = _integers(n, total), _integers(kout, total)
    sa, sb = _scales(n, total // 32), _scales(kout, total // 32)
    out, qa, qb = torch.full((len(slots), n, kout), 7.0, device="cuda"), a.to(E4), b.to(E5)
    _lib.call("viola_varlen_wgrad_gemm", qa.data_ptr(), _lib.code(E4), qb.data_ptr(), _lib.code(E5), sa.data_ptr(), sb.data_ptr(), offsets.data_ptr(),
              len(slots), total, n, kout, out.data_ptr(), 0)
    a, b, start = _spell(a, sa, 1), _spell(b, sb, 1), 0
    for g, length in enumerate(slots):
        assert torch.equal(out[g], a[:, start:start + length] @ b[:, start:start + length].T)
        start += length


TEAMS = [(4096, 1024, 8192, torch.bfloat16), (2000, 1028, 1536, torch.float32), (1921, 2047, 1552, torch.float16),
         (1500, 1535, 1568, torch.bfloat16), (1536, 1536, 1808, torch.float32), (1536, 1536, 2064, torch.float32)]


@pytest.mark.parametrize("m,n,k,out_dtype", TEAMS)
def test_row_scaled_products_whose_teams_share_the_k_range(m, n, k, out_dtype):
    """129 to 256 tiles of 128 x 128: the teams' ranges of equal and different length, the second ending inside a block of scales (with
    the next row's scale, a NaN, in the piece that holds its last ones), ragged rows and columns."""
    from viola_amd.nn import _grouped_kernels as g
    torch.manual_seed(m + n + k)
    a, b, groups = _integers(m, k), _integers(n, k), -(-k // 32)
    sa, sb = _scales(m, groups), _scales(n, groups)
    bias = torch.randint(-8, 9, (n,), device="cuda").float()
    want = _spell(a, sa, 1) @ _spell(b, sb, 1).T + bias
    sa[7, 0], sb[n - 1, 0] = float("nan"), float("inf")
    out = g.gemm(a.to(E4), b.to(E5), sa, sb, (1, 32), (1, 32), out_dtype=out_dtype, bias=bias)
    rows = torch.arange(m, device="cuda") != 7
    assert torch.equal(out[rows, :n - 1], want[rows, :n - 1].to(out_dtype)) and torch.isnan(out[7]).all()


@pytest.mark.parametrize("m,n,k,parts,out_dtype", [(3072, 768, 9856, 3, torch.bfloat16), (512, 516, 2080, 8, torch.float32), (200, 100, 1040, 64, torch.float16),
                                                   (257, 333, 4112, 5, torch.bfloat16), (1024, 1024, 192, 2, torch.float32), (64, 40, 16, 2, torch.float32)])
def test_product_in_parts_of_k(m, n, k, parts, out_dtype):
    """The k range cut into parts: parts that end inside a chunk and inside a block of scales, fewer chunks than parts, rows of the
    partial products that are not whole pieces, tiles that do not divide over the XCDs."""
    torch.manual_seed(m + n + k)
    a, b, groups = _integers(m, k), _integers(n, k), -(-k // 32)
    sa, sb = _scales(m, groups), _scales(n, groups)
    out, qa, qb = torch.full((m, n), 7.0, device="cuda", dtype=out_dtype), a.to(E4), b.to(E5)
    floats = parts * (-(-m * n // 4) * 4)
    workspace = torch.full((floats + 64,), float("nan"), device="cuda")
    args = lambda size: (qa.data_ptr(), _lib.code(E4), qb.data_ptr(), _lib.code(E5), sa.data_ptr(), sb.data_ptr(), m, n, k, out.data_ptr(), _lib.code(out_dtype), parts,
                         workspace.data_ptr(), size)
    with pytest.raises(RuntimeError):
        _lib.call("viola_group_gemm_in_parts", *args(floats - 1))
    assert (out == 7.0).all()
    _lib.call("viola_group_gemm_in_parts", *args(floats))
    assert torch.equal(out, (_spell(a, sa, 1) @ _spell(b, sb, 1).T).to(out_dtype)) and torch.isnan(workspace[floats:]).all()


def test_linear_weight_gradient_in_parts_against_float64():
    """The C entry point at a shape that the modules run in parts: no further from the float64 product of the very codes than the whole
    product is."""
    from viola_amd.nn import _grouped_kernels as g
    torch.manual_seed(1)
    m, n, k = 768, 512, 8192
    parts = _lib.library().viola_group_gemm_parts(m, n, k)
    assert parts > 1
    (qa, sa), (qb, sb) = (g.quantize(torch.randn(r, k, device="cuda").bfloat16(), E4, (1, 32)) for r in (m, n))
    out, workspace = torch.empty(m, n, device="cuda"), torch.empty(parts * m * n, device="cuda")
    _lib.call("viola_group_gemm_in_parts", qa.data_ptr(), _lib.code(E4), qb.data_ptr(), _lib.code(E4), sa.data_ptr(), sb.data_ptr(), m, n, k, out.data_ptr(), 0, parts,
              workspace.data_ptr(), workspace.numel())
    whole = g.gemm(qa, qb, sa, sb, (1, 32), (1, 32), out_dtype=torch.float32)
    exact = (qa.float() * sa.repeat_interleave(32, 1)).double() @ (qb.float() * sb.repeat_interleave(32, 1)).double().T
    error = lambda t: ((t - exact).norm() / exact.norm()).item()
    assert error(out) <= 1.05 * error(whole)
