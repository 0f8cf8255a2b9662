"""Prompt chunks of 2 to 63 tokens run as one pass (kernels/short_prompt.h) and
give every token the bits of decoding it.

Each length is compared with a model that runs its prompt token by token
through the decode step (prefill_via_decode, itself bit-identical to the
oracle elsewhere): the last logits, every layer's keys and values, and the
greedy continuation, bit for bit. The lengths sit at the edges of the
16- and 32-token tiles and at both ends of the range; the starts give the
attention one, two, four and eight waves (64 positions each) and more."""

import json

import numpy as np
import pytest

import oracle
from helpers import expect_bits_equal

pytestmark = pytest.mark.gpu

VOCAB = 4096


def checkpoint(lcr, tmp_path_factory, kv_heads=8, fp16=False):
    d = tmp_path_factory.mktemp(f"short_{kv_heads}_{int(fp16)}")
    cfg = lcr.llama_config(num_hidden_layers=2, vocab_size=VOCAB, num_key_value_heads=kv_heads)
    return lcr.write_synthetic_checkpoint(d, cfg, fp16=fp16)


def compare(lcr, ckpt, variant, kv_heads, paged, cases):
    a = lcr.Model(ckpt, variant=variant, max_seq=700, paged=int(paged))
    b = lcr.Model(ckpt, variant=variant, max_seq=700, paged=int(paged), prefill_via_decode=1)
    for start, count in cases:
        what = f"{variant}, {kv_heads} kv heads, paged {paged}, {count} tokens at {start}"
        print(what, flush=True)
        ids = lcr.synthetic_tokens(start + count, VOCAB, seed=100 * count + start)
        got = []
        for m in (a, b):
            m.reset()
            for t in ids[:start]:
                m.decode(int(t))
            logits = m.logits(m.prefill(ids[start:]))
            assert m.position == start + count
            kv = [m.kv_export(layer, start + count, kv_heads, 64) for layer in range(2)]
            first = m.sample(m.decode(oracle.argmax(logits)), 0.0)
            got.append((logits, kv, [first] + [int(t) for t in m.generate_greedy(first, 2)[0]]))
        expect_bits_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32), f"logits, {what}")
        for layer in range(2):
            for k in range(2):
                expect_bits_equal(got[0][1][layer][k], got[1][1][layer][k], f"layer {layer} cache, {what}")
        assert got[0][2] == got[1][2], what
    a.close()
    b.close()


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("variant", ["bf16", "fp16"])
def test_short_prompt_bits(lcr, tmp_path_factory, variant, paged):
    ckpt = checkpoint(lcr, tmp_path_factory, fp16=variant == "fp16")
    cases = [(0, n) for n in (2, 15, 16, 17, 31, 32, 33, 48, 49, 63)]
    cases += [(1, 63), (62, 2), (100, 20), (190, 63), (300, 33), (600, 40)]
    compare(lcr, ckpt, variant, 8, paged, cases)


@pytest.mark.parametrize("kv_heads", [32, 16, 4])
def test_short_prompt_bits_other_groups(lcr, tmp_path_factory, kv_heads):
    compare(lcr, checkpoint(lcr, tmp_path_factory, kv_heads), "bf16", kv_heads, True, [(0, 2), (0, 37), (130, 63)])


def rewrite(ckpt, edits):
    """Applies edits[name](array of element bits) to tensors of a checkpoint."""
    with open(ckpt / "model.safetensors", "r+b") as f:
        size = int.from_bytes(f.read(8), "little")
        header = json.loads(f.read(size))
        for name, edit in edits.items():
            first, last = header[name]["data_offsets"]
            f.seek(8 + size + first)
            bits = np.frombuffer(f.read(last - first), np.uint16).reshape(header[name]["shape"]).copy()
            edit(bits)
            f.seek(8 + size + first)
            f.write(bits.tobytes())


@pytest.mark.parametrize("variant", ["bf16", "fp16"])
def test_short_prompt_bits_of_extreme_weights(lcr, tmp_path_factory, variant):
    """The projections' matrix instructions round like the decode step's fused
    multiply-adds also where products are denormal, cancel, spread over many
    binades or are infinite. Values of the first kv head of layer 0 come from rows
    of denormal weights, of large ones, of pairs (a, -a) against equal inputs, and
    of magnitudes over 20 to 40 binades; o_proj reads none of them (zero columns),
    so the rest of the model stays in range. Two elements of layer 1's value rows
    are then infinite: its cache holds infinities of both signs, and the logits,
    which they reach, are not compared."""
    kind = oracle.FP16 if variant == "fp16" else oracle.BF16
    ckpt = checkpoint(lcr, tmp_path_factory, fp16=variant == "fp16")
    r = np.random.default_rng(5)

    def elems(x):
        return oracle.f32_to_elems(np.asarray(x, np.float32), kind)

    def equal_pairs(bits):
        bits[..., 1::2] = bits[..., 0::2]

    def values0(bits):
        hidden = bits.shape[1]
        bits[0:16] = r.integers(1, 128 if kind == oracle.BF16 else 1024, (16, hidden)) + 0x8000 * r.integers(0, 2, (16, hidden))
        big = 2.0**100 if kind == oracle.BF16 else 2.0**10  # sums of 2048 products stay in range
        bits[16:32] = elems(r.standard_normal((16, hidden)) * big / 8)
        bits[32:48, 0::2] = elems(r.standard_normal((16, hidden // 2)))
        bits[32:48, 1::2] = bits[32:48, 0::2] ^ 0x8000
        span = (-30, 10) if kind == oracle.BF16 else (-14, 6)
        bits[48:64] = elems(r.standard_normal((16, hidden)) * 2.0**r.integers(*span, (16, hidden)))

    def values1(bits):
        bits[3, 700], bits[70, 1999] = elems([np.inf, -np.inf])

    def no_first_group(bits):
        bits[:, :4 * 64] = 0

    layer0, layer1 = (f"model.layers.{i}.self_attn." for i in (0, 1))
    rewrite(ckpt, {"model.embed_tokens.weight": equal_pairs, layer0 + "v_proj.weight": values0,
                   layer0 + "o_proj.weight": no_first_group, "model.layers.0.input_layernorm.weight": equal_pairs})
    compare(lcr, ckpt, variant, 8, False, [(0, 2), (0, 16), (0, 33), (3, 63)])
    rewrite(ckpt, {layer1 + "v_proj.weight": values1})
    a, b = (lcr.Model(ckpt, variant=variant, max_seq=64, prefill_via_decode=v) for v in (0, 1))
    ids = lcr.synthetic_tokens(40, VOCAB, seed=9)
    caches = []
    for m in (a, b):
        m.prefill(ids)
        caches.append([m.kv_export(layer, len(ids), 8, 64) for layer in (0, 1)])
        m.close()
    for layer in (0, 1):
        for k in (0, 1):
            expect_bits_equal(caches[0][layer][k], caches[1][layer][k], f"layer {layer} cache, {variant}")
    first, last = (oracle.elems_to_f32(caches[0][layer][1], kind) for layer in (0, 1))
    assert (np.isposinf(last).any() and np.isneginf(last).any()) and not np.isnan(last).any()
    head0 = first.reshape(8, -1, 64)[0]
    assert np.isfinite(first).all() and (head0[:, :16] != 0).any() and (np.abs(head0[:, 16:32]) > 2.0**8).any()


def test_short_prompt_leaves_the_step_state(lcr, tmp_path_factory):
    """After a short prompt the greedy sample reads the id its head reduced,
    decode() of that id copies no state, and both equal the oracle's."""
    ckpt = checkpoint(lcr, tmp_path_factory)
    m = lcr.Model(ckpt, max_seq=64)
    o = oracle.OracleModel(ckpt, max_seq=64, multiprocessors=m.stats().multiprocessors)
    prompt = lcr.synthetic_tokens(9, VOCAB, seed=3)
    ptr = m.prefill(prompt)
    lo = o.prefill(prompt, use_decode_path=True)
    expect_bits_equal(m.logits(ptr).view(np.uint32), lo.view(np.uint32), "prompt logits")
    for _ in range(4):
        tok = m.sample(ptr, 0.0)
        assert tok == oracle.argmax(lo)
        ptr, lo = m.decode(tok), o.decode(tok)
        expect_bits_equal(m.logits(ptr).view(np.uint32), lo.view(np.uint32), "step logits")
    ptr = m.prefill(prompt[:5])  # a second short chunk behind the decoded tokens
    for t in prompt[:5]:
        lo = o.decode(int(t))
    expect_bits_equal(m.logits(ptr).view(np.uint32), lo.view(np.uint32), "second chunk's logits")
    m.close()
    o.close()
