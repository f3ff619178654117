"""Key splits of a prefill launch: none when the query tiles fill the GPU or the rows are short, two workgroups per CU over
long rows and one over shorter ones, never fewer than two key tiles or more than 64 splits."""
import pytest


@pytest.mark.parametrize("tiles,keys,want", [(64, 4096, 1), (1, 3, 1), (1, 4, 2), (1, 256, 64), (2, 256, 32),
                                             (2, 1024, 64), (8, 255, 8), (8, 256, 16), (16, 64, 4), (63, 1024, 3),
                                             (63, 47, 2)])
def test_prefill_splits(tiles, keys, want):
    from lfm3_kv800_amd import kv800_hip
    assert kv800_hip.prefill_splits(tiles, keys) == want
