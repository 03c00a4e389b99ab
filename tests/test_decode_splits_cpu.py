"""How a decode step's keys are cut into slices: the number is one for the whole step, its sequences may be of any lengths."""
import pytest

from trapetum_amd.kernels.ops import HipOps


@pytest.mark.parametrize("keys", [64, 129, 500, 1024, 2048, 4096, 8000, 32768])
@pytest.mark.parametrize("n,KV", [(1, 1), (1, 4), (3, 5), (4, 4), (8, 4), (15, 4), (16, 4), (16, 16), (31, 4), (32, 4), (47, 4), (48, 4), (64, 4), (64, 8), (100, 4), (256, 8)])
def test_a_long_sequence_is_cut_whatever_stands_beside_it(n, KV, keys):
    splits, pairs = HipOps.decode_splits(n, KV, 256, keys), n * KV
    assert 1 <= splits <= min(128, -(-keys // 64))
    # a block walks at most two of the bounds, or there are six blocks a CU, or as many slices as the kernel takes
    bound = 320 if pairs < 128 else 512 if pairs < 512 else 1024
    assert keys / splits < 2 * bound or splits == 128 or (pairs < 128 and splits * pairs >= 1536)
    # every CU has a block where there are keys for one
    assert splits * pairs >= 256 or splits >= min(128, keys // 64)


def test_many_slices_are_a_multiple_of_eight():
    for n, KV in ((1, 4), (3, 4), (5, 4), (7, 4), (8, 4), (9, 4), (11, 8), (31, 4)):
        for keys in (2048, 4096, 5000, 8192):
            splits = HipOps.decode_splits(n, KV, 256, keys)
            assert splits <= 8 or splits % 8 == 0 or splits * 128 > keys - 1024, (n, KV, keys, splits)
    assert HipOps.decode_splits(8, 4, 256, 8192) == 16 and HipOps.decode_splits(12, 4, 256, 4096) == 16 and HipOps.decode_splits(28, 4, 256, 1024) == 10


def test_short_sequences_that_fill_the_chip_are_not_cut():
    assert HipOps.decode_splits(64, 4, 256, 80) == 1 and HipOps.decode_splits(32, 8, 128, 128) == 1
    assert HipOps.decode_splits(1, 4, 256, 200) == 4 and HipOps.decode_splits(64, 4, 256, 1024) == 3
