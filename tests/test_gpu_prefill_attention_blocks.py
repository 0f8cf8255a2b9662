"""lcr_prefill_attention's choice of block (32 rows; 16 rows with two or four
key groups) and its ways to a page's table entry (one scalar read per load for
power-of-two pages of eight positions up, per position otherwise), against
the oracle's prefill attention: sizes on both sides of each choice, odd
row-block counts, a first chunk and chunks behind cached positions."""

import ctypes

import numpy as np
import pytest

import oracle
from helpers import expect_close
from test_gpu_kernels import BF16, Cache, NULL, dev, fill_cache, host, ok, p, random_elems, rng, to_f32, zeros_dev

pytestmark = pytest.mark.gpu

# (tokens, start, heads, kv heads, head_dim)
CASES = [
    (2047, 0, 32, 8, 64), (2049, 0, 32, 8, 64),    # 64 blocks of 32 rows a kv head, and one more (16 rows)
    (2015, 40, 32, 8, 64), (2016, 0, 16, 8, 128),  # just below: 16 rows at head_dim 128
    (2048, 0, 16, 8, 128),
    (511, 513, 32, 8, 64), (512, 512, 32, 8, 64), (513, 512, 32, 8, 64),  # four groups up to one block a unit
    (500, 523, 32, 8, 64), (500, 524, 32, 8, 64),  # and from 1024 keys on
    (1, 1023, 32, 8, 64), (17, 2000, 16, 2, 64), (65, 0, 8, 8, 64), (33, 1500, 16, 8, 128),
    # the second resident round in reverse: one to two blocks a unit, runs of several and of less than one kv head,
    # two blocks of four heads a kv head (one of them half empty), empty places at the end of the last XCD
    (1009, 0, 64, 8, 64), (1000, 0, 32, 16, 64), (1024, 0, 16, 16, 64), (700, 0, 32, 4, 64), (530, 9, 48, 8, 64),
    (600, 0, 10, 10, 64),
    # 32 rows from 7/4 blocks a unit on, with one head a kv head only behind cached keys, and again from 7/3 on
    (1761, 0, 32, 8, 64), (1760, 0, 32, 8, 64), (1024, 512, 16, 16, 64), (1024, 511, 16, 16, 64), (1185, 0, 32, 16, 64),
    (1217, 0, 32, 16, 64),
]


@pytest.mark.parametrize("tokens,start,heads,kv,hd", CASES)
def test_blocks(gpu, lcr, orc, tokens, start, heads, kv, hd):
    check(gpu, lcr, orc, tokens, start, heads, kv, hd, None)


@pytest.mark.parametrize("page_size", [1, 4, 7, 8, 16, 64])
@pytest.mark.parametrize("tokens,start,heads,kv,hd", [(100, 1000, 32, 8, 64), (90, 61, 16, 8, 128),
                                                      (2048, 3, 32, 8, 64)])
def test_pages(gpu, lcr, orc, tokens, start, heads, kv, hd, page_size):
    check(gpu, lcr, orc, tokens, start, heads, kv, hd, page_size)


def check(lib, lcr, orc, tokens, start, heads, kv, hd, page_size):
    print(tokens, start, heads, kv, hd, page_size, flush=True)
    r = rng(tokens + 7 * start + hd)
    n = start + tokens
    keys, values = random_elems(r, (n, kv * hd)), random_elems(r, (n, kv * hd))
    q = random_elems(r, (heads, tokens, hd))
    table = None if page_size is None else r.permutation(-(-n // page_size)).astype(np.int32)
    cache = Cache(kv, hd, n, page_size is not None, page_size or 16, table)
    fill_cache(lib, lcr, cache, keys, values, n)
    paged = int(page_size is not None)
    out, v = zeros_dev(tokens * heads * hd), cache.view(lcr)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(hd)))
    ok(lib, lib.lcr_prefill_attention(p(out), p(dev(q)), ctypes.byref(v), heads, heads // kv, tokens, start, scale,
                                      paged, NULL), "prefill attention")
    got = to_f32(host(out)).reshape(tokens, heads * hd)
    # The oracle on the rows of the first, middle and last blocks.
    rows = sorted({t for a in (0, tokens // 2, tokens - 1) for t in range(a - 17, a + 18) if 0 <= t < tokens})
    hv = cache.host_view()
    for first in [t for t in rows if t - 1 not in rows]:
        count = next(c for c in range(1, tokens + 1) if first + c not in rows)
        part = np.ascontiguousarray(q[:, first:first + count])
        exp = np.zeros(count * heads * hd, dtype=np.uint16)
        orc.load().orc_prefill_attention(BF16, exp.ctypes.data, part.ctypes.data, ctypes.byref(hv), heads,
                                         heads // kv, count, start + first, scale, paged)
        expect_close(got[first:first + count].ravel(), to_f32(exp), 3e-2, f"rows {first} .. {first + count - 1}")
