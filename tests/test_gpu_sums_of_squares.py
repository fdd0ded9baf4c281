"""Sums of squares of a matrix in one order on every way to Newton-Schulz: its norm is rounded to 16 bits, so that another order would now and
then scale the whole matrix differently when it steps in other company."""

import ctypes

import pytest
import torch

from viola_amd import _lib

pytestmark = pytest.mark.gpu


class Matrices(ctypes.Structure):
    _fields_ = [("in_", ctypes.c_void_p), ("out", ctypes.c_void_p)] + [(name, ctypes.c_int64) for name in ("batch", "rows", "cols")]


def _prepared(x, working):
    """Partial sums that viola_ns_prepare forms for [batch, rows, cols], alone."""
    batch, rows, cols = x.shape
    sums, out = torch.full((batch, 256), float("nan"), device="cuda"), torch.empty(x.numel(), device="cuda", dtype=working)
    _lib.call("viola_ns_prepare", _lib.ptr(x), _lib.code(x.dtype), _lib.ptr(out), _lib.code(working), batch, rows, cols, _lib.ptr(sums))
    return sums


# rows x columns in tiles of 1024: one, a unit of 4096 elements and a tile more, all 256 slots and a tile more, five turns and some (every turn twice)
SHAPES = [(8, 128), (32, 128), (40, 128), (1024, 1024), (1025, 1024), (5 * 1024 + 40, 1024)]


@pytest.mark.parametrize("working", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile", [256, 512, 1024])
@pytest.mark.parametrize("shapes", [SHAPES, SHAPES[:2], SHAPES[-1:]])
def test_sums_beside_the_momentum_are_those_of_a_pass(shapes, tile, working):
    torch.manual_seed(len(shapes))
    table, updates, held = [], [], []
    for i, (rows, cols) in enumerate(shapes):
        n = rows * cols
        g, q = torch.randn(n, device="cuda") * 1e-2, torch.randint(0, 120, (n,), device="cuda", dtype=torch.uint8)
        s, update = torch.rand(n // tile, device="cuda") * 1e-3, torch.empty(1, rows, cols, device="cuda", dtype=torch.bfloat16)
        table.append([g.data_ptr(), q.data_ptr(), s.data_ptr(), q.data_ptr(), s.data_ptr(), update.data_ptr(), 77 + i, n // tile])
        updates.append(update); held.append((g, q, s))
    rows, sums = torch.tensor(table, device="cuda"), torch.full((len(shapes), 256), float("nan"), device="cuda")
    _lib.call("viola_momentum_update_squares", rows.data_ptr(), len(shapes), max(r * c for r, c in shapes) // tile, _lib.F32, tile, .95, 1.0, 1, 0, 3, _lib.code(working),
              sums.data_ptr())
    for i, update in enumerate(updates):
        assert torch.equal(sums[i], _prepared(update, working)[0]), shapes[i]


# in more than 512 blocks each takes half as many wavefronts, with two tiles each: the last of them has one, or none
@pytest.mark.parametrize("grads", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("working", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tiles", [(1, 2, 15, 16, 17, 301, 4098, 4099), (4096, 4096), (3,) * 171, (4096,)])
def test_stochastic_momentum_and_sums_are_those_of_a_tensor_alone(tiles, working, grads):
    torch.manual_seed(len(tiles))
    table, pairs = [], []
    for i, n in enumerate(tiles):
        g, q, s = (torch.randn(256 * n, device="cuda") * 1e-2).to(grads), torch.randint(0, 120, (256 * n,), device="cuda", dtype=torch.uint8), torch.rand(n, device="cuda") * 1e-3
        want, got = [(q.clone(), s.clone(), torch.zeros(1, 32 * n, 8, device="cuda", dtype=torch.bfloat16)) for _ in range(2)]
        _lib.call("viola_momentum_update", _lib.ptr(g), _lib.code(grads), *map(_lib.ptr, (*want[:2], *want)), 256 * n, .95, 1.0, 1, 0, 256, 1, 1, 1, 1, 1, 1, 3, 77 + i)
        table.append([t.data_ptr() for t in (g, *got[:2], *got)] + [77 + i, n])
        pairs.append((want, got, g))
    rows, sums = torch.tensor(table, device="cuda"), torch.full((len(tiles), 256), float("nan"), device="cuda")
    _lib.call("viola_momentum_update_squares", rows.data_ptr(), len(tiles), max(tiles), _lib.code(grads), 256, .95, 1.0, 1, 1, 3, _lib.code(working), sums.data_ptr())
    for i, (want, got, _) in enumerate(pairs):
        assert all(torch.equal(a, b) for a, b in zip(want, got)), tiles[i]
        assert torch.equal(sums[i], _prepared(got[2], working)[0]), tiles[i]


@pytest.mark.parametrize("working", [torch.bfloat16, torch.float16])
def test_sums_of_several_shapes_are_those_of_each_matrix_alone(working):
    """Extents that end within a unit, a chunk and a wavefront; of several matrices one holds infinities and NaN."""
    shapes = [(2, 8, 8), (1, 33, 72), (3, 96, 160), (1, 1024, 1032), (2, 700, 1600), (1, 72, 8)]
    torch.manual_seed(4)
    ins = [torch.randn(*s, device="cuda").bfloat16() for s in shapes]
    ins[2][1, 5, 7], ins[2][2, 0, 0] = float("nan"), float("-inf")
    outs = [torch.empty(x.numel(), device="cuda", dtype=working) for x in ins]
    sums, rows = torch.full((sum(s[0] for s in shapes), 256), float("nan"), device="cuda"), (Matrices * len(shapes))()
    for i, (shape, x, out) in enumerate(zip(shapes, ins, outs)):
        rows[i] = Matrices(x.data_ptr(), out.data_ptr(), *shape)
    _lib.call("viola_ns_prepare_many", ctypes.addressof(rows), len(shapes), _lib.code(working), _lib.ptr(sums), 0)
    at = 0
    for x in ins:
        for matrix in x:
            alone = _prepared(matrix[None], working)[0]
            assert torch.equal(torch.nan_to_num(sums[at], nan=-1.0), torch.nan_to_num(alone, nan=-1.0))
            exact = matrix.to(working).double().square().sum()
            if torch.isfinite(exact):                                         # at most 2^-24 for each of the some 40 additions on the way of a term
                assert abs(alone.double().sum() - exact) <= 40 * 2.0 ** -24 * exact
            else:
                assert not torch.isfinite(alone.sum())
            at += 1
