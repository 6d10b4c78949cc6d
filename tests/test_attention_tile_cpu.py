"""The default attention tile: at either side of each line of its rule."""

import pytest

from newt_amd.workloads import attention_tile


@pytest.mark.parametrize("S,heads,D,causal,want", [
    (4096, 128, 128, True, (256, 8)), (4096, 128, 128, False, (256, 8)),
    # causal, wide heads: 512 programs of 256 rows, then 512 of 128
    (2048, 64, 128, True, (256, 8)), (2048, 63, 128, True, (128, 8)),
    (2048, 32, 128, True, (128, 8)), (2048, 31, 128, True, (64, 4)),
    # causal, 64-wide heads: 1024 programs of 128 rows
    (2048, 64, 64, True, (128, 4)), (2048, 63, 64, True, (64, 4)),
    # not causal: 193 programs of 256 rows, then 129 to 256 of 128
    (256, 193, 128, False, (256, 8)), (256, 192, 128, False, (64, 4)),
    (256, 128, 128, False, (128, 8)), (256, 65, 128, False, (128, 8)),
    (256, 64, 128, False, (64, 4)), (1, 1, 128, False, (64, 4)),
    (1000, 32, 64, False, (128, 4)), (1500, 24, 64, False, (64, 4)),
])
def test_tile_rule(S, heads, D, causal, want):
    assert attention_tile(S, heads, D, causal) == want
