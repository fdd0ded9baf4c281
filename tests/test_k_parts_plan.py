"""In how many parts of k a row-wise scaled product runs is host arithmetic of the library (viola_group_gemm_parts), so the rule can
be replayed here without a GPU."""

import pytest

from viola_amd import _lib


def parts(m, n, k):
    return _lib.library().viola_group_gemm_parts(m, n, k)


# the shapes that the rule's comment quotes: what it says of each, next to the count of the fastest run
@pytest.mark.parametrize("m,n,k,says,fastest", [(3072, 768, 9856, 3, 3), (1024, 1024, 16384, 8, 8), (512, 512, 16384, 20, 20), (256, 256, 16384, 32, 32),
                                                (1000, 332, 3200, 10, 8), (1152, 1152, 16384, 5, 5), (4096, 1024, 8192, 1, 1), (1024, 1024, 4096, 1, 1),
                                                (2048, 1024, 8192, 1, 4)])
def test_the_rule_answers_what_its_comment_says(m, n, k, says, fastest):
    assert parts(m, n, k) == says


def test_no_part_is_empty():
    for k in range(1024, 16385, 48):
        chunks = -(-k // 128) * 2                                             # of the padded rows that the modules give it
        for m, n in ((256, 256), (768, 512), (3072, 768), (1536, 1536), (3072, 3072)):
            count = parts(m, n, k)
            length = -(-chunks // count)
            assert count == 1 or (-(-chunks // length) == count and length >= 4), (m, n, k)


def test_products_that_gain_nothing_stay_whole():
    for shape in ((1024, 1024, 1008), (63, 4096, 8192), (4096, 60, 8192), (512, 514, 8192), (0, 64, 8192), (64, 64, 0), (8192, 8192, 8192)):
        assert parts(*shape) == 1, shape


def test_partial_products_stay_within_their_bound():
    """At most 96 MiB of scratch, at most 34 MB up to 256 tiles of 128 x 128 and 16384 tokens."""
    from itertools import product
    widths = (64, 256, 512, 768, 1000, 1536, 2304, 3072, 3584, 4352, 5248, 7680, 8192)
    largest = few = 0
    for m, n, k in product(widths, widths, (1024, 3072, 8192, 9856, 15936, 16384, 65536)):
        count = parts(m, n, k)
        scratch = 0 if count == 1 else count * m * n * 4
        largest = max(largest, scratch)
        if -(-m // 128) * -(-n // 128) <= 256 and k <= 16384:
            few = max(few, scratch)
    assert 64 << 20 < largest <= 96 << 20 and few <= 34e6
    assert parts(3072, 3072, 16384) == 2 and parts(4352, 4224, 16128) == parts(3584, 5248, 16384) == parts(7680, 2304, 15936) == 1


def test_sizes_that_the_product_in_parts_refuses_are_whole():
    for shape in ((512, 512, 1 << 23), (768, 512, 1 << 22), (1 << 40, 1 << 40, 8192), (512, 1 << 62, 8192), (512, 512, 1 << 62)):
        assert parts(*shape) == 1, shape
