"""The 64 x 128 tile of the prefill GEMM (few tokens) and the plans that use it,
at the tile's edges, unsplit and split over K, through every fused entry.

The plain product is compared with a float64 one; the bound is the fp32
accumulation's: with u = 2^-24, K products summed in at most K + splits
additions err by (K + 16) u sum |x w| (for K = 8192 about 5e-4 of that sum; the
observed error is far below, as roundings cancel), and one rounding to the
16-bit element. The fused entries give the plain product's bits."""

import ctypes

import numpy as np
import pytest

import oracle
from helpers import BF16, FP16, dev, expect_bits_equal, host, p, random_elems, rng, sync, zeros_dev
from test_gpu_kernels import Cache, ok, rope_table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,N,K", [
    # gate/up rows, unsplit: token edges of the tile
    (64, 16384, 2048), (65, 16384, 2048), (127, 16384, 2048), (128, 16384, 2048), (129, 2048, 2048),
    # split plans, and rows that end inside a 64-row tile
    (77, 2048, 8192), (100, 1000, 2048), (66, 2044, 4096), (90, 3001, 2048), (70, 2016, 4096),
    # K not in whole stages of 64: the tile does not apply
    (100, 3072, 2080), (100, 3072, 2056),
    # one slice's worth of K and less
    (80, 16384, 256), (80, 16384, 64)])
@pytest.mark.parametrize("kind,variant", [pytest.param(BF16, "bf16", id="bf16"), pytest.param(FP16, "fp16", id="fp16")])
def test_narrow_tile_products(gpu, lcr, kind, variant, T, N, K):
    lib = lcr.load_library(variant)
    r = rng(T + N + K)
    X, W = random_elems(r, (T, K), kind=kind), random_elems(r, (N, K), 0.05, kind=kind)
    Xd, Wd = dev(X), dev(W)
    X64, W64 = (oracle.elems_to_f32(a, kind).astype(np.float64) for a in (X, W))
    exp = X64 @ W64.T
    bound = (K + 16) * 2.0**-24 * (np.abs(X64) @ np.abs(W64).T) + 1e-30
    unit = 2.0**-8 if kind == BF16 else 2.0**-11
    full = lib.lcr_gemm_workspace_bytes(T, N, K)
    # the preferred plan, one with too small a workspace for it, and unsplit
    for ws_bytes in dict.fromkeys((full, full // 2, 0)):
        print(f"{variant} {T}x{N}x{K} workspace {ws_bytes}", flush=True)
        ws = zeros_dev(max(ws_bytes, 16) // 4, np.float32)
        wsp = p(ws) if ws_bytes else None
        Y, Yb = zeros_dev(T * N, np.float32), zeros_dev(T * N)
        ok(lib, lib.lcr_gemm_ws(p(Y), 1, p(Xd), p(Wd), T, N, K, wsp, ws_bytes, None), "gemm_ws fp32 out")
        ok(lib, lib.lcr_gemm_ws(p(Yb), 0, p(Xd), p(Wd), T, N, K, wsp, ws_bytes, None), "gemm_ws")
        y = host(Y, np.float32).reshape(T, N)
        assert (np.abs(y - exp) <= bound).all(), (np.abs(y - exp) / bound).max()
        yb = oracle.elems_to_f32(host(Yb), kind).reshape(T, N)
        # the 16-bit output is the fp32 one rounded once (2^-25 covers fp16's subnormals)
        assert (np.abs(yb.astype(np.float64) - y) <= unit * np.abs(y) + 2.0**-25).all()
        if N % 32 == 0:
            want, got = zeros_dev(T * N // 2), zeros_dev(T * N // 2)
            ok(lib, lib.lcr_swiglu_strided(p(want), p(Yb), ctypes.c_void_p(Yb.ptr + N), T, N // 2, N, None), "swiglu")
            ok(lib, lib.lcr_gemm_swiglu_ws(p(got), p(Xd), p(Wd), T, N // 2, K, wsp, ws_bytes, None), "gemm_swiglu_ws")
            expect_bits_equal(host(got), host(want), "gemm + swiglu")
        x0, weight = random_elems(r, (T, N), kind=kind), dev(random_elems(r, (N,), 0.5, kind=kind))
        x_want, x_got, want, got, scratch = dev(x0), dev(x0), zeros_dev(T * N), zeros_dev(T * N), zeros_dev(T * N)
        ok(lib, lib.lcr_add_residual_rmsnorm(p(want), p(x_want), p(Yb), p(weight), T, N, 1e-5, None), "norm")
        ok(lib, lib.lcr_gemm_residual_rmsnorm_ws(p(got), p(x_got), p(scratch), p(Xd), p(Wd), p(weight), T, N, K, 1e-5,
                                                 wsp, ws_bytes, None), "gemm_residual_rmsnorm_ws")
        expect_bits_equal(host(got), host(want), "gemm + residual norm")
        expect_bits_equal(host(x_got), host(x_want), "residual")


@pytest.mark.parametrize("T,nh,K,start,paged,shift", [
    # 3072 rows, split: rotated in the reduction
    (64, 32, 2048, 0, False, 0), (65, 32, 2048, 5, True, 0), (128, 32, 2048, 100, True, 0), (500, 32, 2048, 3, True, 0),
    # 16384 rows, 256 tiles of one head each: rotated in the tile's epilogue
    (64, 240, 256, 0, False, 0), (65, 240, 256, 5, True, 0), (128, 240, 320, 100, True, 0),
    # caches 8 bytes past a 16-byte boundary
    (65, 32, 2048, 3, True, 4), (128, 240, 256, 3, False, 4)])
def test_narrow_tile_qkv_rope(gpu, lcr, T, nh, K, start, paged, shift):
    """The q/k/v projection with RoPE and the cache append against the plain
    product, the RoPE of its queries and the append."""
    check_qkv_rope(lcr, T, nh, 64, K, start, paged, shift)


@pytest.mark.parametrize("shift", [0, 4])
@pytest.mark.parametrize("T,nh,hd,K,start,paged", [
    # 4096 rows: 64 x 128 tiles unsplit from 385 tokens on, then wider ones; 128-row heads are two pieces of a tile
    (384, 16, 128, 2048, 0, False), (385, 16, 128, 2048, 3, True), (512, 16, 128, 2048, 0, True),
    (513, 16, 128, 2048, 0, False), (700, 16, 128, 2048, 9, True), (1024, 16, 128, 2048, 0, False),
    (2048, 16, 128, 2048, 0, False), (400, 48, 64, 2048, 5, True),
    # 192-row tiles (one and a half heads of 128), 6144 and 5120 rows
    (1024, 32, 128, 2048, 0, True), (1300, 24, 128, 3072, 0, False),
    # few tokens, odd head counts, K outside the ring stages of 64 and of 32
    (3, 16, 128, 2048, 1, True), (77, 3, 128, 512, 0, False), (300, 16, 128, 2080, 2, False),
    (300, 48, 64, 2056, 2, True), (1500, 16, 128, 2056, 0, False)])
def test_qkv_rope_takes_the_plain_plan(gpu, lcr, T, nh, hd, K, start, paged, shift):
    """Whatever the head size, the cache's alignment and the workspace (its own,
    none, or one that other projections need larger), K is summed in the slices of
    the plain product."""
    check_qkv_rope(lcr, T, nh, hd, K, start, paged, shift, 64 << 20)


def check_qkv_rope(lcr, T, nh, hd, K, start, paged, shift, shared=0):
    lib = lcr.load_library("bf16")
    kv = 8
    N = (nh + 2 * kv) * hd
    r = rng(T + start + shift)
    Xd, Wd = dev(random_elems(r, (T, K))), dev(random_elems(r, (N, K), 0.05))
    freq = dev(rope_table(hd))
    table = zeros_dev((start + T) * hd, np.float32)
    ok(lib, lib.lcr_rope_table(p(table), p(freq), start + T, hd, None), "rope_table")
    full = lib.lcr_gemm_workspace_bytes(T, N, K)
    max_seq = -(-(start + T) // 16) * 16
    pages = r.permutation(max_seq // 16) if paged else None
    for ws_bytes in dict.fromkeys((full, 0, shared)):
        print(f"qkv {T} tokens at {start}, {nh} heads of {hd}, K {K}, paged {paged}, shift {shift}, workspace {ws_bytes}", flush=True)
        ws = zeros_dev(max(ws_bytes, 16) // 4, np.float32)
        wsp = p(ws) if ws_bytes else None
        wc, gc = Cache(kv, hd, max_seq, paged, 16, pages), Cache(kv, hd, max_seq, paged, 16, pages)
        elems = kv * max_seq * hd
        shifted = [zeros_dev(elems + 8) for _ in range(2)]
        qkv, q_want, q_got = zeros_dev(T * N), zeros_dev(nh * T * hd), zeros_dev(nh * T * hd)
        ok(lib, lib.lcr_gemm_ws(p(qkv), 0, p(Xd), p(Wd), T, N, K, wsp, ws_bytes, None), "gemm_ws")
        ok(lib, lib.lcr_rope_q(p(q_want), p(qkv), p(freq), T, start, nh, hd, N, None), "rope_q")
        vw, vg = wc.view(lcr), gc.view(lcr)
        if shift:
            vg.keys, vg.values = (b.ptr + 2 * shift for b in shifted)
        ok(lib, lib.lcr_rope_write_kv(ctypes.byref(vw), ctypes.c_void_p(qkv.ptr + 2 * nh * hd),
                                      ctypes.c_void_p(qkv.ptr + 2 * (nh + kv) * hd), p(freq), T, start,
                                      1 if paged else 0, N, None), "rope_write_kv")
        ok(lib, lib.lcr_gemm_qkv_rope_ws(p(q_got), ctypes.byref(vg), p(Xd), p(Wd), p(table), T, nh, K, start,
                                         1 if paged else 0, wsp, ws_bytes, None), "gemm_qkv_rope_ws")
        sync()
        got = [host(b)[shift:shift + elems] for b in shifted] if shift else [host(gc.keys), host(gc.values)]
        pairs = [(host(q_got), host(q_want), "queries"), (got[0], host(wc.keys), "keys"),
                 (got[1], host(wc.values), "values")]
        for g, w, name in pairs:
            expect_bits_equal(g, w, f"qkv + rope: {name}")
