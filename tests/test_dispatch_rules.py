"""The rules on sizes that choose a kernel, where they are Python."""


def test_tile_group_counts_experts():
    """64-pair groups while the pairs average at most 48 per expert. Without a count (GroupedPairs takes n_experts as an option) the
    tables' bound of 512 must not stand in for it: 24,576 pairs over 8 experts would stream each expert's weights 48 times."""
    from dsv41_amd.hipkern import LIGHT_GROUP, LIGHT_PAIRS, LIGHT_PAIRS_PER_EXPERT as most, TILE_GROUP, tile_group
    for E in (1, 8, 128, 384, 512):
        assert tile_group(most * E, E) == LIGHT_GROUP and tile_group(most * E + 1, E) == TILE_GROUP
    assert tile_group(LIGHT_PAIRS, None) == LIGHT_GROUP
    assert tile_group(LIGHT_PAIRS + 1, None) == tile_group(most * 512, None) == TILE_GROUP
