"""Which kernels take a query row of a selection: asked of the library, no GPU."""
import pytest

from vlm_training_amd import _lib


@pytest.mark.parametrize("Hq,Hkv,K,longest,listed", [
    # head_dim 128, three and four heads per kv head: segments of more than 32 K have their rows past 24 K gathered by the list where the walk begins
    # later still, for it would have too few rows to pay for its launch (a batch may hold such segments beside a long one),
    (8, 2, 256, 32 * 256, 0), (8, 2, 256, 32 * 256 + 1, 1), (12, 4, 128, 32 * 128, 0), (12, 4, 128, 32 * 128 + 1, 1), (8, 2, 256, 17000, 1),
    # and wherever it could never have enough;
    (8, 2, 64, 2048, 0), (8, 2, 64, 2049, 1), (8, 2, 64, 4500, 1), (8, 2, 128, 9000, 1),
    # segments a little too short for it: the tiles
    (8, 2, 512, 24 * 512 + 1, 0), (8, 2, 512, 17000, 0), (8, 2, 512, 38400, 0), (8, 2, 512, 38401, 1), (12, 4, 256, 24 * 256 + 1, 0),
    # many heads: the walk from its first long segment on, up to where rows are too thin for it
    (32, 8, 2048, 24 * 2048 + 1, 0), (32, 8, 2048, 131072, 0), (32, 8, 2048, 75 * 2048, 0), (32, 8, 2048, 75 * 2048 + 1, 1), (288, 72, 512, 13000, 0),
    # two heads per kv head: the tiles in the gather's place, to 75 K
    (16, 8, 512, 14000, 0), (16, 8, 512, 150 * 512, 0), (16, 8, 512, 150 * 512 + 1, 1), (16, 8, 64, 9728, 0), (16, 8, 64, 9729, 1), (4, 2, 64, 6485, 0),
    (4, 2, 64, 6486, 1), (4, 2, 64, 11000, 1),
])
def test_rows_that_the_list_is_read_for(Hq, Hkv, K, longest, listed):
    lib = _lib.load()
    assert lib.dsa_get_tile_crossover() == 24
    assert lib.dsa_attn_reads_list(Hq, Hkv, 128, K, longest) == listed
    # elsewhere one line, wherever the heads stand
    assert lib.dsa_attn_reads_list(Hq, Hkv, 64, K, longest) == (longest > (24 * K + 255) // 256 * 256)


@pytest.mark.parametrize("Hq,Hkv,K,lens,listed", [
    # segments long enough on average: the batch walks them all, and those a little too short for it stay on the tiles
    (8, 2, 64, (2100,) * 8, 0), (8, 2, 64, (2247,) * 7, 0), (8, 2, 256, (8967,) * 2, 0), (16, 4, 64, (2247,) * 9, 0), (12, 4, 64, (2247,) * 9, 0),
    (64, 16, 16, (500, 430, 405, 400, 295), 0), (64, 16, 16, (513, 430, 405, 400, 295), 0), (4, 1, 128, (5127,) * 4, 0), (4, 1, 128, (6407,) * 3, 0),
    (32, 8, 64, (2567,) + (384,) * 4, 0), (32, 8, 64, (2500,) + (384,) * 4, 0), (32, 8, 64, (2500,), 1),
    # too few tokens for that, too short an average, and rows too thin for the walk
    (8, 2, 64, (2100,) * 4, 1), (8, 2, 64, (2100,) * 8 + (9,) * 10, 1), (8, 2, 64, (4900, 2048) + (1800,) * 8, 1),
    # one segment: its tokens are the batch's
    (8, 2, 256, (12000,), 0), (8, 2, 256, (10000,), 1), (8, 2, 64, (4900,), 1),
])
def test_rows_that_the_list_is_read_for_in_a_batch(Hq, Hkv, K, lens, listed):
    """A batch whose rows are all walked or on tiles writes no list and launches no gather, also where a longer segment alone would need one."""
    lib = _lib.load()
    assert lib.dsa_get_tile_crossover() == 24
    assert lib.dsa_attn_batch_reads_list(Hq, Hkv, 128, K, sum(lens), len(lens), max(lens)) == listed
    assert lib.dsa_attn_reads_list(Hq, Hkv, 128, K, max(lens)) >= listed


def test_pairs_of_a_workload_are_counted_where_the_tile_kernels_take_all():
    from vlm_training_amd import workloads as W
    for w in (W.C1, W.C2, W.C3, W.C5):
        assert w.executed_pairs() == (w.pair_counts()[0],) * 2
    assert W.C4.executed_pairs() == (None, None)         # late rows and the key side are the compacted walks'
    few = W.head_shard(W.C4, 8)                          # (one kv head: key tiles cut into pieces, never walked)
    assert few.executed_pairs() == (None, few.pair_counts()[0])
    assert W.C3.executed_pairs(crossover=0) == (None, W.C3.pair_counts()[0])
