"""Which form a product runs in is host arithmetic of the library (viola_scaled_gemm_form for per-tensor and block scales, viola_group_gemm_form
for the grouped recipe): the shapes of the GPU tests of a last round on smaller tiles have to reach it."""

import test_gpu_last_round as cases
from viola_amd import _lib

BLOCKS, LARGE, MEDIUM, SMALL, LARGE_THEN_SMALL = range(5)


def form(m, n, k):
    return _lib.library().viola_scaled_gemm_form(m, n, k)


def test_last_round_on_small_tiles():
    for m, n, k, _ in cases.LAST_ROUND:
        for length in (k, -(-k // 128) * 128):
            assert form(m, n, length) == LARGE_THEN_SMALL, (m, n, length)


def test_where_the_line_lies():
    """Full rounds stay as they are, and so does a last round of more than a quarter of the CUs."""
    assert form(4096, 4096, 4096) == form(16384, 4096, 4096) == LARGE                   # 256 and 1024 tiles
    assert form(4096, 4352, 4096) == LARGE_THEN_SMALL                                   # 272
    assert form(4096, 5120, 4096) == LARGE_THEN_SMALL                                   # 320
    assert form(4096, 6400, 4096) == form(5000, 5000, 4096) == LARGE                    # 400
    assert form(1024, 1024, 1024) == BLOCKS and form(8192, 1024, 4096) == MEDIUM and form(2048, 1152, 4608) == SMALL
    assert _lib.library().viola_scaled_gemm_form(0, 1, 1) == -1


def test_grouped_last_round():
    """Large tiles, and a last round of the size that the test says."""
    group_form, large = _lib.library().viola_group_gemm_form, 4
    rests = []
    for m, n, k, *_ in cases.GROUPED_LAST_ROUND:
        assert group_form(m, n, k, 0, 0, 0) == large, (m, n, k)
        rests.append(-(-m // 256) * -(-n // 256) % 256)
    assert rests == [4, 52, 64, 88, 96, 128, 133]
    rests = []
    for counts, n, k in cases.VARLEN_LAST_ROUND:
        assert group_form(sum(counts), n, k, 0, len(counts), 0) == large, (counts, n, k)
        rests.append(sum(-(-c // 256) for c in counts) * -(-n // 256) % 256)
    assert rests == [16, 96, 8, 44]
