"""Which kernels take a query row of a selection: asked of the library, no GPU."""
import pytest

from vlm_training_amd import _lib


@pytest.mark.parametrize("Hq,Hkv,K,longest,listed", [
    # head_dim 128, three and four heads per kv head: rows past 24 K are gathered by the list ...
    (8, 2, 512, 24 * 512, 0), (8, 2, 512, 24 * 512 + 1, 1), (12, 4, 256, 24 * 256 + 1, 1),
    # ... also in segments that are longer, as long as the walk would have too few rows to pay for its launch (a batch may hold such beside a long one),
    (8, 2, 512, 17000, 1), (8, 2, 512, 39000, 1),
    # and all of them where it could never have enough
    (8, 2, 64, 4500, 1), (8, 2, 128, 9000, 1),
    # many heads: the walk from its first long segment on, up to where rows are too thin for it
    (32, 8, 2048, 24 * 2048 + 1, 0), (32, 8, 2048, 131072, 0), (32, 8, 2048, 75 * 2048, 0), (32, 8, 2048, 75 * 2048 + 1, 1), (288, 72, 512, 13000, 0),
    # two heads per kv head: the tiles in the gather's place
    (16, 8, 512, 14000, 0), (16, 8, 512, 150 * 512, 0), (16, 8, 512, 150 * 512 + 1, 1), (16, 8, 64, 4864, 0), (16, 8, 64, 4865, 1), (8, 4, 64, 4865, 1),
])
def test_rows_that_the_list_is_read_for(Hq, Hkv, K, longest, listed):
    lib = _lib.load()
    assert lib.dsa_get_tile_crossover() == 24
    assert lib.dsa_attn_reads_list(Hq, Hkv, 128, K, longest) == listed
    # elsewhere one line, wherever the heads stand
    assert lib.dsa_attn_reads_list(Hq, Hkv, 64, K, longest) == (longest > (24 * K + 255) // 256 * 256)


def test_pairs_of_a_workload_are_counted_where_the_tile_kernels_take_all():
    from vlm_training_amd import workloads as W
    for w in (W.C1, W.C2, W.C3, W.C5):
        assert w.executed_pairs() == (w.pair_counts()[0],) * 2
    assert W.C4.executed_pairs() == (None, None)         # late rows and the key side are the compacted walks'
    few = W.head_shard(W.C4, 8)                          # (one kv head: key tiles cut into pieces, never walked)
    assert few.executed_pairs() == (None, few.pair_counts()[0])
    assert W.C3.executed_pairs(crossover=0) == (None, W.C3.pair_counts()[0])
