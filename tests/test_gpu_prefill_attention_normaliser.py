"""lcr_prefill_attention's softmax normaliser at scores from 1 to 64000.

Every row's largest score is S and the others lie up to five below it, all of
them exact in fp32 (whole multiples of 1/256 below 2^16), so the weights depend
on the keys' places below S alone and the outputs are compared with float64
ones. An error in a row's normaliser scales the row's outputs by 1 + a; a is
estimated as the projection of the outputs on the exact ones over all heads of
the row, which averages the roundings of weights and outputs: with u the
element type's unit roundoff, an output carries two independent relative errors
within +-u (its own and its weights'), so that over n outputs the estimate has
a standard deviation of at most u sqrt(2 / 3 / n) sqrt(E w^4) / E w^2, where
the last factor is sqrt(3) for normal outputs. Asked for is a root mean square
over the rows of twice that, plus 2^-21 for the fp32 sums. Exponents
that keep the rounding of their own size (92000 at the last score, in steps of
2^-7) measured 6e-4 to 9e-4 there, against bounds of 4.9e-4 or less (bf16) and
6.1e-5 or less (fp16)."""

import ctypes

import numpy as np
import pytest

from helpers import BF16, FP16, dev, host, p, random_elems, rng, zeros_dev
import oracle
from test_gpu_kernels import NULL, Cache, fill_cache, ok

pytestmark = pytest.mark.gpu

# (tokens, start, head_dim): 32 rows; 16 rows with two and four key groups
BLOCKS = [(2048, 0, 64), (700, 0, 64), (300, 1000, 64), (2048, 0, 128), (300, 300, 128)]
# score -> two factors whose product, sixteen times and scaled by 1/8, it is
FACTORS = {1: (1, 0.5), 100: (5, 10), 1000: (20, 25), 16000: (80, 100), 64000: (160, 200)}


@pytest.mark.parametrize("kind,variant", [pytest.param(BF16, "bf16", id="bf16"), pytest.param(FP16, "fp16", id="fp16")])
@pytest.mark.parametrize("tokens,start,hd", BLOCKS)
def test_rows_are_normalised(gpu, lcr, kind, variant, tokens, start, hd):
    lib = lcr.load_library(variant)
    r = rng(tokens + start + hd)
    n, kv, group = start + tokens, 8, 2
    heads = kv * group
    values = random_elems(r, (n, kv * hd), kind=kind)
    v64 = oracle.elems_to_f32(values, kind).astype(np.float64).reshape(n, kv, hd)
    steps = r.integers(-40 * 32, 1, size=(n, kv))  # of 1/256 score
    steps[0] = 0
    for score, (a, b) in FACTORS.items():
        print(f"{variant} {tokens} tokens at {start}, head_dim {hd}, scores of {score}", flush=True)
        q, k = np.zeros((heads, tokens, hd), np.float32), np.zeros((n, kv, hd), np.float32)
        q[:, :, :16], k[:, :, :16] = a, b
        q[:, :, 16], k[:, :, 16] = 1, steps // 32
        q[:, :, 17], k[:, :, 17] = 1 / 32, steps % 32
        cache = Cache(kv, hd, n, False, 16, None)
        fill_cache(lib, lcr, cache, oracle.f32_to_elems(k, kind).reshape(n, kv * hd), values, n)
        qd, out, view = dev(oracle.f32_to_elems(q, kind)), zeros_dev(tokens * heads * hd), cache.view(lcr)
        ok(lib, lib.lcr_prefill_attention(p(out), p(qd), ctypes.byref(view), heads, group, tokens, start, 0.125, 0,
                                          NULL), "prefill attention")
        got = oracle.elems_to_f32(host(out), kind).astype(np.float64).reshape(tokens, kv, group, hd)
        weight = np.exp(steps / 256.0)
        exact = (np.cumsum(weight[:, :, None] * v64, 0) / np.cumsum(weight, 0)[:, :, None])[start:]
        rows = np.arange(tokens) + start >= 64  # enough keys for their roundings to average
        num = np.einsum("tkgd,tkd->t", got, exact) / group
        off = (num / np.einsum("tkd,tkd->t", exact, exact) - 1)[rows]
        unit = 2.0**-8 if kind == BF16 else 2.0**-11
        bound = 2 * unit * np.sqrt(2.0 / 3.0 / (kv * hd)) * np.sqrt(3.0) + 2.0**-21
        rms = np.sqrt(np.mean(off**2))
        print(f"  rms {rms:.2e}, mean {off.mean():+.2e}, bound {bound:.2e}", flush=True)
        assert rms <= bound
