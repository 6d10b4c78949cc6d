"""The default attention tile: at either side of each line of its rule."""

import pytest

from newt_amd.workloads import attention_tile


@pytest.mark.parametrize("S,heads,D,causal,want", [
    (4096, 128, 128, True, (256, 8)), (4096, 128, 128, False, (256, 8)),
    # causal, wide heads: 160, 256, 512 and 1024 programs of 256 rows
    (1024, 40, 128, True, (64, 4)), (1024, 41, 128, True, (128, 8)),
    (512, 128, 128, True, (64, 4)), (2048, 32, 128, True, (128, 8)),
    (2048, 33, 128, True, (128, 4)), (2048, 64, 128, True, (256, 8)),
    (2048, 65, 128, True, (128, 4)), (2048, 48, 128, True, (256, 8)), (2048, 128, 128, True, (256, 8)),
    (1024, 256, 128, True, (128, 4)),
    # causal, 64-wide heads: 1024 keys, then 768 programs of 128 rows
    (1024, 256, 64, True, (64, 4)), (2048, 48, 64, True, (64, 4)),
    (2048, 49, 64, True, (128, 4)),
    # not causal: rounds of the 256 CUs
    (256, 256, 128, False, (256, 8)), (256, 129, 128, False, (256, 8)),
    (256, 128, 128, False, (128, 8)), (256, 257, 128, False, (128, 4)),
    (256, 400, 128, False, (256, 8)), (256, 64, 128, False, (64, 4)),
    (1, 1, 128, False, (64, 4)), (1000, 32, 64, False, (128, 4)),
    (1500, 24, 64, False, (64, 4)),
])
def test_tile_rule(S, heads, D, causal, want):
    assert attention_tile(S, heads, D, causal) == want


@pytest.mark.parametrize("S,heads,want", [
    # heads that the 8 XCDs share evenly, around 376, 512 and 1024 programs
    (2048, 40, (128, 4)), (4096, 16, (128, 8)), (2816, 32, (128, 4)), (5888, 16, (128, 4)),
    (6144, 16, (256, 8)), (3000, 32, (256, 8)), (2560, 40, (256, 8)), (3072, 40, (256, 8)),
    (2560, 48, (256, 8)), (4096, 32, (256, 8)), (8192, 16, (256, 8)), (3328, 40, (128, 4)),
    (2048, 72, (128, 4)), (4096, 56, (128, 4)), (2048, 120, (128, 4)), (4096, 64, (256, 8)),
    (2048, 136, (256, 8)),
    # an odd number of heads per XCD, 9 blocks and more
    (2048, 56, (128, 4)), (2304, 56, (128, 4)), (2305, 40, (256, 8)), (4096, 24, (256, 8)),
    # heads that they do not, beside those
    (2048, 47, (128, 4)), (2048, 49, (128, 4)), (2048, 63, (128, 4)), (4096, 31, (128, 4)),
    (2048, 129, (128, 4)), (4096, 65, (128, 4)),
    # shorter sequences
    (2047, 48, (128, 4)), (1024, 128, (128, 4)), (1024, 256, (128, 4)),
])
def test_causal_lines_and_their_neighbours(S, heads, want):
    assert attention_tile(S, heads, 128, True) == want


@pytest.mark.parametrize("S,heads", [(2048, 48), (2560, 40), (2048, 128), (4096, 64)])
def test_wider_heads_keep_four_waves(S, heads):
    assert attention_tile(S, heads, 256, True) == (128, 4)
