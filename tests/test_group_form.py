"""Which form a product under the grouped recipe runs in is host arithmetic of the library (viola_group_gemm_form), so it can be
replayed here without a GPU: the shapes of the GPU tests of the large-tile forms have to reach the kernels that they are there for."""

import pytest

import test_gpu_grouped_pingpong as cases
from viola_amd import _lib

BLOCKS, BLOCKS_SPLIT, NARROW, NARROW_SPLIT, LARGE, TALL, TEAMS = range(7)


def form(m, n, k, row_scaled_b=False, row_groups=0, k_groups=0):
    return _lib.library().viola_group_gemm_form(m, n, k, int(row_scaled_b), row_groups, k_groups)


@pytest.mark.parametrize("row_scaled_b", [False, True])
def test_large_tiles(row_scaled_b):
    for m, n, k, *_ in cases.LARGE + [(4096, 4096, k) for k in cases.LARGE_LEAK_K]:
        assert form(m, n, k, row_scaled_b) == LARGE, (m, n, k)


def test_tall_tiles_and_teams():
    for m, n, k, _ in cases.TALL:
        assert form(m, n, k) == TALL, (m, n, k)
    for m, n, k, _ in cases.TEAMS:
        assert form(m, n, k, row_scaled_b=True) == TEAMS, (m, n, k)


def test_variable_groups():
    for counts in cases.VARLEN_LARGE:
        assert form(sum(counts), *cases.VARLEN_LARGE_SIZE, row_groups=len(counts)) == LARGE, counts
    for counts, n, k in cases.VARLEN_TALL:
        assert form(sum(counts), n, k, row_groups=len(counts)) == TALL, (counts, n, k)
    slots, n, kout = cases.VARLEN_WGRAD
    assert form(n, kout, -(-sum(slots) // 128) * 128, row_scaled_b=True, k_groups=len(slots)) == LARGE


# the shapes that the rule's comments quote for the blocks of group_gemm_fast
@pytest.mark.parametrize("m,n,k,row_scaled_b,says", [(6000, 4096, 1024, False, BLOCKS), (4096, 3072, 8192, True, BLOCKS),
                                                     (8192, 1024, 1024, False, BLOCKS), (4096, 1024, 4096, False, BLOCKS_SPLIT),
                                                     (4096, 1024, 1024, False, NARROW), (600, 4096, 1024, False, NARROW), (1024, 1024, 16384, True, NARROW_SPLIT),
                                                     (512, 512, 4096, False, NARROW_SPLIT), (100, 64, 512, False, BLOCKS)])
def test_blocks(m, n, k, row_scaled_b, says):
    assert form(m, n, k, row_scaled_b) == says


def test_what_the_guarded_kernel_takes_is_refused():
    for args in ((1024, 1024, 1000), (0, 64, 64), (64, 64, 0), (64, 1 << 20, 1 << 12), (1 << 24, 64, 64), (64, 64, 64, True, 2, 2), (64, 64, 64, False, 0, 2)):
        assert form(*args) == -1, args
