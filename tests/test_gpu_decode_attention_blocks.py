"""lcr_decode_attention's choice of block: as many waves as a split has
64-position tiles (1, 2, 4, 8), one register set up to eight tiles and two
past them, and up to four query heads of a kv head per block from 10 million
key elements over all query heads and 128 such blocks on. Every choice gives the oracle's bits; the sizes are the first and last
of each, for groups of 1, 2, 4 and 8 heads and both head dims."""

import pytest

from test_gpu_kernels import check_decode_attention

pytestmark = pytest.mark.gpu

HEADS = [(32, 8, 64), (16, 8, 128), (16, 2, 64), (8, 8, 128)]


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("heads,kv,hd", HEADS)
def test_block_by_tiles(gpu, lcr, orc, heads, kv, hd, paged):
    for positions in (1, 64, 65, 128, 129, 256, 257, 512, 513):
        print(heads, kv, hd, positions, paged, flush=True)
        check_decode_attention(gpu, lcr, orc, heads, kv, hd, positions, 1, paged, 16)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("heads,kv,hd", HEADS)
def test_block_by_splits(gpu, lcr, orc, heads, kv, hd, paged):
    for positions, splits in ((3840, 15), (16, 16), (4096, 16), (4097, 16), (8192, 16), (8193, 16), (70, 64)):
        print(heads, kv, hd, positions, splits, paged, flush=True)
        check_decode_attention(gpu, lcr, orc, heads, kv, hd, positions, splits, paged, 16)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("heads,kv,hd,cases", [
    (32, 8, 64, [(4882, 16), (4883, 16), (4883, 15), (5000, 20), (8193, 16), (10500, 16)]),
    (16, 8, 128, [(4882, 16), (4883, 16), (4883, 15), (9000, 64)]),
    (16, 2, 64, [(9765, 32), (9766, 32), (9766, 31)]),
    (8, 8, 128, [(9766, 16)])])
def test_shared_heads(gpu, lcr, orc, heads, kv, hd, cases, paged):
    for positions, splits in cases:
        print(heads, kv, hd, positions, splits, paged, flush=True)
        check_decode_attention(gpu, lcr, orc, heads, kv, hd, positions, splits, paged, 16)
