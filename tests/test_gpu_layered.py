"""The layered decoder on the device against the float64 oracle: every mechanism alone, prompts, decoding, portions, mixed
batches, reused pages and slots, window edges, long decoding, greedy and sampled generation through the scheduler."""
import ctypes as C
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from helpers import layered_build as B
from helpers import layered_ref as R
from helpers.device import ROOT, dev
from helpers.layered_model import TOL, Model, check, err, feed, greedy, margin

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cai():
    return dev()


BIG = dict(layers=[B.layer(B.delta(heads=6, kv_heads=3, dim=20, vdim=36, conv=3)), B.layer(B.delta(heads=1, dim=70, vdim=130, conv=1), ff=None),
                   B.layer((B.attn(heads=6, kv_heads=2, dim=20, vdim=44, window=11), B.delta(heads=4, kv_heads=2, dim=9, vdim=17, conv=5))),
                   B.layer(B.delta(heads=3, dim=33, vdim=5, conv=2), ff=17)], width=100, vocab=211, loop=dict(start=1, stop=3, times=3))


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    return Model(tmp_path_factory.mktemp("layered"), B.config(**BIG), seed=11)


# ---------------------------------------------------------------- products over bfloat16 weights
@pytest.mark.parametrize("rows, cols", [(37, 50), (64, 64), (131, 520), (700, 1100), (9000, 96)])
def test_bf16_products(cai, rows, cols):
    rng = np.random.default_rng(rows)
    bits, w = B.to_bf16(rng.standard_normal((rows, cols)))
    w = w.reshape(rows, cols); bias = rng.standard_normal(rows).astype(np.float32)
    q = cai.QWeight(cai.BF16, rows, cols, bits, bias)
    assert np.array_equal(q.dequant_rows(3, 5), w[3:8].astype(np.float32))
    for n in (1, 2, 3, 5, 8, 9, 33, 70, 130):
        x = rng.standard_normal((n, cols)).astype(np.float32)
        want = x.astype(np.float64) @ w.T + bias
        if n <= 8:
            assert err(q.gemv(x), want) < 3e-6
            assert err(q.gemv(x, cai.ACT_RELU), np.maximum(want, 0)) < 3e-6
        assert err(q.gemm(x), want) < 3e-6


def bf16_rows(cai, q, x, gated=False):
    """one product over activations rounded to bfloat16, as the sublayers of a bfloat16 decoder run it (rows, or relu(gate) * up of a gated matrix)"""
    x = np.ascontiguousarray(x, np.float32)
    y = np.empty((len(x), q.rows // 2 if gated else q.rows), np.float32)
    cai.check(cai.load().cai_bf16_rows(q.h, C.c_void_p(x.ctypes.data), len(x), int(gated), C.c_void_p(y.ctypes.data)))
    return y


# a last slot of 8 columns (264, 8200), of 64 (2112), whole ones; rows 8 k + 1 to 8 k + 7; fewer tiles than work-groups and more; past 8192 columns (8200) another kernel
@pytest.mark.parametrize("rows, cols", [(9, 64), (66, 40), (1003, 320), (12292, 70), (517, 2112), (62, 264), (71, 8192), (4113, 520), (35, 8200), (2050, 1032)])
def test_products_over_bf16_rows(cai, rows, cols):
    """Every result of 1 to 16 rows, and of tiles of 32 and 64 tokens, against 64 bits.  A sum of 32 products is cut off at 2^-23 of the largest of them at most
    eight times, sums are then rounded to 2^-24 three times: 2^-19 of the sum of absolute products bounds them all."""
    rng = np.random.default_rng(rows)
    bits, w = B.to_bf16(rng.standard_normal((rows, cols)))
    w = w.reshape(rows, cols).astype(np.float64); bias = rng.standard_normal(rows).astype(np.float32)
    q = cai.QWeight(cai.BF16, rows, cols, bits, bias)
    for n in (1, 2, 3, 5, 7, 8, 9, 13, 16, 17, 33, 70):
        x = B.to_bf16(rng.standard_normal((n, cols)))[1].reshape(n, cols).astype(np.float64)
        assert np.all(np.abs(bf16_rows(cai, q, x) - (x @ w.T + bias)) <= 2.0 ** -19 * (np.abs(x) @ np.abs(w).T + np.abs(bias))), n
    q.close()


@pytest.mark.parametrize("rows, cols", [(8193, 72), (8201, 2120), (8198, 4616), (8195, 6160)])
def test_few_rows_of_many_outputs_over_bf16_rows(cai, rows, cols):
    """the same of one to four and sixteen rows where the ring kernel takes every count: one to four slots of a row a wave, with fewer and more tiles than
    work-groups, bounds as above"""
    rng = np.random.default_rng(rows)
    bits, w = B.to_bf16(rng.standard_normal((rows, cols), np.float32))
    w = w.reshape(rows, cols).astype(np.float64)
    q = cai.QWeight(cai.BF16, rows, cols, bits)
    for n in (1, 2, 3, 4, 16):
        x = B.to_bf16(rng.standard_normal((n, cols)))[1].reshape(n, cols).astype(np.float64)
        assert np.all(np.abs(bf16_rows(cai, q, x) - x @ w.T) <= 2.0 ** -19 * (np.abs(x) @ np.abs(w).T)), n
    q.close()


@pytest.mark.parametrize("rows, cols", [(32, 64), (96, 320), (5664, 72), (8224, 72), (2144, 2112), (8288, 2112), (64, 8192), (160, 264), (64, 8200)])
def test_gated_products_over_bf16_rows(cai, rows, cols):
    gated_products(cai, rows, cols, (1, 2, 3, 5, 7, 8, 9, 13, 16, 17, 33, 70))


@pytest.mark.parametrize("rows, cols, tokens", [(2016, 264, 1100), (6208, 136, 2050), (2016, 264, 2000), (6208, 136, 2310)])
def test_gated_products_on_one_round_of_large_tiles(cai, rows, cols, tokens):
    """tiles of 256 x 256 (the second and the last) and of 128 x 128 by sixteen waves (the third), and what fewer tokens take"""
    assert cai.load().cai_bf16_tiles(rows, cols, tokens, 1) == {1100: 1, 2050: 5, 2000: 2, 2310: 5}[tokens]
    gated_products(cai, rows, cols, (tokens,))


def gated_products(cai, rows, cols, tokens):
    """the same of gate and up rows: the bounds of both sums, then one rounding to bfloat16 (2^-8 of the value at most)"""
    rng = np.random.default_rng(rows + cols)
    bits, w = B.to_bf16(rng.standard_normal((rows, cols)))
    w = w.reshape(rows // 32, 2, 16, cols).astype(np.float64)
    gate, up = w[:, 0].reshape(-1, cols), w[:, 1].reshape(-1, cols)
    q = cai.QWeight(cai.BF16, rows, cols, bits)
    for n in tokens:
        x = B.to_bf16(rng.standard_normal((n, cols)))[1].reshape(n, cols).astype(np.float64)
        g, u = x @ gate.T, x @ up.T
        dg, du = 2.0 ** -19 * (np.abs(x) @ np.abs(gate).T), 2.0 ** -19 * (np.abs(x) @ np.abs(up).T)
        want = np.maximum(g, 0) * u
        off = (np.maximum(g, 0) + dg) * du + dg * np.abs(u)
        assert np.all(np.abs(bf16_rows(cai, q, x, True) - want) <= off + 2.0 ** -8 * (np.abs(want) + off)), n
    q.close()


@pytest.mark.parametrize("cols", [320, 1024, 2048, 5632, 8192])
@pytest.mark.parametrize("spread", [0.0, 1.5])
def test_few_bf16_rows_are_as_near_as_the_32_bit_walk(cai, cols, spread):
    """activations of even and of widely differing sizes: what the matrix cores make of five to sixteen rows is as close to 64 bits as the 32-bit walk over the same
    rows (relative errors of 40 rows of 2000 results, squares averaged; one chain of matrix instructions was 1.4 to 2.2 times as far off)"""
    rng = np.random.default_rng(cols)
    bits, w = B.to_bf16(rng.standard_normal((2000, cols)))
    w = w.reshape(2000, cols).astype(np.float64)
    q = cai.QWeight(cai.BF16, 2000, cols, bits)
    off = np.zeros(2)
    for n in (5, 5, 6, 8, 16):
        x = B.to_bf16(rng.standard_normal((n, cols)) * np.exp(spread * rng.standard_normal((n, cols))))[1].reshape(n, cols).astype(np.float64)
        want = x @ w.T
        for i, got in enumerate((bf16_rows(cai, q, x), np.concatenate([q.gemv(x[k:k + 8]) for k in range(0, n, 8)]))):
            off[i] += np.sum(np.linalg.norm(got - want, axis=1) ** 2 / np.linalg.norm(want, axis=1) ** 2)
    assert off[0] <= off[1], np.sqrt(off / 40)
    q.close()


def test_bf16_matrices_stay_out_of_the_other_decoders(cai):
    bits, _ = B.to_bf16(np.zeros((64, 64)))
    q = cai.QWeight(cai.BF16, 64, 64, bits)
    with pytest.raises(cai.CaiError):
        q.ffn_gateup(np.zeros((1, 64), np.float32))


# ---------------------------------------------------------------- each mechanism alone
def only(part):
    def edit(w):
        for n in w:
            if part == "attention" and n.endswith("right.out"):
                w[n] = w[n] * 0
            if part == "channel delta" and n.endswith("left.out"):
                w[n] = w[n] * 0
            if part == "feed-forward" and n.endswith("norm1b"):
                w[n] = w[n] * 0
            if part == "squash" and n.endswith(".alpha"):
                w[n] = w[n] * 3
    return edit


MECHANISMS = {
    "delta": [("delta", B.delta(h, g, d, dv, t)) for h, g, d, dv, t in ((1, 1, 8, 8, 1), (4, 2, 64, 64, 4), (2, 2, 33, 70, 2), (3, 1, 129, 20, 6), (2, 1, 128, 128, 4), (1, 1, 256, 256, 3))],
    "channel delta": [("parallel", (B.attn(), B.delta(h, g, d, dv, t))) for h, g, d, dv, t in ((1, 1, 8, 8, 1), (4, 2, 32, 64, 4), (3, 3, 45, 131, 3), (2, 1, 200, 34, 5))],
    "attention": [("parallel", (B.attn(h, g, d, dv, w), B.delta())) for h, g, d, dv, w in
                  ((1, 1, 8, 8, 1), (4, 4, 24, 40, 2), (6, 2, 48, 96, 64), (8, 1, 130, 70, 65), (10, 2, 256, 256, 33), (2, 1, 64, 20, 1000), (3, 1, 17, 9, 63))],
    "feed-forward": [("delta", B.delta())], "squash": [("parallel", (B.attn(), B.delta()))],
}
CASES = [(m, i) for m, v in MECHANISMS.items() for i in range(len(v))]


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("mech, i", CASES, ids=["%s-%d" % c for c in CASES])
def test_mechanism_alone(cai, tmp_path, mech, i, dt):
    kind, mixer = MECHANISMS[mech][i]
    m = Model(tmp_path, B.config([B.layer(mixer, ff=48 if mech == "feed-forward" else None)], width=40 + 8 * i, vocab=67), seed=i, edit=only(mech), rank_a=3 + 9 * i, rank_g=20)
    tok = m.tokens(90, i)
    dec = m.open(cai, 128, 1, dt)
    check(feed(dec, tok, [90]), m.ref(tok), dt)
    dec.reset()
    check(feed(dec, tok, [70, 1]), m.ref(tok), dt)
    dec.close()


# Heads at the edges of what a lane and a quad have requested ahead: one and two channels a lane, low-rank rows of one piece, of all four, and of one more; more
# rows than quads have places for (128 channels and 128 gates are 256 of 416)
@pytest.mark.parametrize("h, g, d, dv, ra, rg", [(4, 2, 64, 64, 7, 11), (2, 1, 128, 128, 128, 127), (2, 2, 128, 128, 129, 33), (3, 1, 65, 70, 32, 128), (2, 1, 20, 126, 40, 8), (2, 1, 128, 130, 16, 16)])
@pytest.mark.parametrize("mech", ["delta", "channel delta"])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_single_tokens(cai, tmp_path, mech, h, g, d, dv, ra, rg, dt):
    """tokens one by one from the first on, where the convolutions reach in front of the text and the state is what an earlier sequence left"""
    mixer = B.delta(h, g, d, dv, 4)
    m = Model(tmp_path, B.config([B.layer(mixer if mech == "delta" else (B.attn(), mixer))], width=72, vocab=67), seed=d, edit=only(mech), rank_a=ra, rank_g=rg)
    tok = m.tokens(24, dv)
    dec = m.open(cai, 64, 1, dt)
    feed(dec, m.tokens(9, 1), [9])
    dec.reset()
    check(feed(dec, tok, [1] * 7 + [9] + [1] * 8), m.ref(tok), dt)
    dec.close()


# Numbers of chunks of 16 that leave the walk's loop over three at each of its places, last chunks whole and ragged; key widths of 4, 8 and 16
# tiles, value widths of whole and of ragged slices
@pytest.mark.parametrize("n", [32, 33, 47, 48, 49, 64, 81])
@pytest.mark.parametrize("h, g, d, dv", [(8, 4, 64, 48), (2, 1, 72, 22), (2, 2, 136, 16)])
@pytest.mark.parametrize("mech", ["delta", "channel delta"])
def test_chunks_of_a_portion(cai, tmp_path, mech, h, g, d, dv, n):
    mixer = B.delta(h, g, d, dv, 4)
    m = Model(tmp_path, B.config([B.layer(mixer if mech == "delta" else (B.attn(), mixer))], width=72, vocab=67), seed=n, edit=only(mech), rank_a=9, rank_g=20)
    tok = m.tokens(n + 13, d)              # (the second portion: eight rows together behind what the ring holds, and five one by one)
    dec = m.open(cai, 192, 1, "f32")
    check(feed(dec, tok, [n, 13]), m.ref(tok), "f32")
    dec.close()


def test_dynamic_tanh_is_as_near_as_the_library_s(cai, tmp_path):
    """The identity as vocabulary matrix and a layer that adds a constant a channel: the logits are the final norm of known 32-bit values.  tanhf is 2.43 * 2^-24 of its
    value from 64 bits at most below 1, and 1.25 * 2^-24 from there on (measured); what takes its place may not be further off.  Half of the arguments lie
    around 1, where forms of a tanh meet."""
    n, rng = 1024, np.random.default_rng(5)

    def edit(w):
        w["l0.mix.o"] = w["l0.mix.o"] * 0
        w["l0.norm1b.b"] = np.exp(rng.uniform(np.log(2.0 ** -22), np.log(2.0 ** -7), n))
        w["embed"] = np.exp(rng.uniform(np.log(0.02), np.log(9.5), (n, n))) * rng.choice([-1, 1], (n, n))
        w["embed"][::2] = 1.0 + rng.integers(-5, 3, (n // 2, n)) / 256.0
        w["head"], w["final.norm"], w["final.norm.b"], w["final.norm.alpha"] = np.eye(n), np.ones(n), np.zeros(n), np.asarray(1.0)

    m = Model(tmp_path, B.config([B.layer(B.delta(1, 1, 8, 8, 2), ff=None)], width=n, vocab=n), edit=edit)
    dec = m.open(cai, 1024, 1, "f32")
    got = feed(dec, list(range(n)), [n]).astype(np.float64)
    dec.close()
    x = (m.w["embed"].astype(np.float32) + m.w["l0.norm1b.b"].astype(np.float32)).astype(np.float64)
    want = np.tanh(x)
    off = np.abs(got - want) / np.abs(want) * 2.0 ** 24
    assert off[np.abs(x) < 1].max() < 2.45 and off[np.abs(x) >= 1].max() < 1.27, (off[np.abs(x) < 1].max(), off[np.abs(x) >= 1].max())


@pytest.mark.parametrize("counts", [(30001,), (20000, 6400, 40, 1), (585 * 16, 17)])
@pytest.mark.parametrize("mech", ["delta", "channel delta"])
def test_long_steps_walk_their_records_in_passes(cai, tmp_path, mech, counts):
    """Records of 64 heads are 896 KB a chunk, so 585 chunks lie side by side: steps of three passes, of passes that an entry ends before, in or at the end of, and of one chunk more than
    a pass holds.  The sequences are those of portions that are one pass each, from the same chunks (32-bit products by other tiles are the only difference), and what a
    step of 30001 rows takes on the device is less than its records alone would be (1.72 GB)."""
    import torch
    mixer = B.delta(64, 64, 8, 8, 4)
    m = Model(tmp_path, B.config([B.layer(mixer if mech == "delta" else (B.attn(), mixer))], width=72, vocab=67), seed=len(counts), edit=only(mech), rank_a=9, rank_g=20)
    toks = [m.tokens(n, n) for n in counts]
    rows = [sorted({n // 2, max(n - 2, 0), n - 1}) for n in counts]
    want = []
    dec = m.open(cai, sum(-(-n // 64) + 1 for n in counts) * 64, len(counts), "f32")
    for e, (t, w) in enumerate(zip(toks, rows)):
        for i in range(0, len(t), 4096):
            here = [k - i for k in w if i <= k < i + 4096]
            got = dec.step_batch([(e, t[i:i + 4096], here)])[1]
            want += list(got) if here else []
    dec.close()
    dec = m.open(cai, sum(-(-n // 64) + 1 for n in counts) * 64, len(counts), "f32")
    before = torch.cuda.mem_get_info()[0]
    got = dec.step_batch([(e, t, w) for e, (t, w) in enumerate(zip(toks, rows))])[1]
    taken = before - torch.cuda.mem_get_info()[0]
    assert err(np.asarray(got, np.float64), np.asarray(want, np.float64)) < 1e-5
    after = dec.step_batch([(e, [5], [0]) for e in range(len(counts))])[1]      # (from the states they left)
    dec.close()
    assert np.isfinite(after).all()
    if counts == (30001,) and mech == "delta":
        assert taken < 1.6e9, taken


@pytest.mark.parametrize("tokens, ff", [(129, 16400), (257, 8208), (300, 12000), (129, 16000), (257, 8000), (300, 8100)])
def test_products_on_tiles_of_256_tokens(cai, tmp_path, tokens, ff):
    """gate | up matrices whose products fill the chip with large tiles, of 256 x 128 (the first and the last three), 128 x 128 (the second) and 256 x 256: tokens one past half a tile, one past a tile and inside a second
    one, rows that end inside a tile; one and a half steps of depth"""
    assert cai.load().cai_bf16_tiles(2 * ff, 72, tokens, 1) == {8208: 3, 12000: 5}.get(ff, 4)
    m = Model(tmp_path, B.config([B.layer(B.delta(), ff=ff)], width=72, vocab=67), seed=tokens, edit=only("feed-forward"), rank_a=3, rank_g=20)
    tok = m.tokens(tokens, 1)
    dec = m.open(cai, 320, 1, "bf16")
    check(feed(dec, tok, [tokens]), m.ref(tok), "bf16")
    dec.close()


@pytest.mark.parametrize("tokens, ff, width", [(300, 12000, 448), (700, 12000, 320), (129, 16400, 448), (600, 5632, 320), (300, 8100, 448)])
def test_products_on_large_tiles_of_many_steps(cai, tmp_path, tokens, ff, width):
    """the same products seven and five steps of 64 deep, so that every slot of the tiles' rings is filled again and the last fill lies in another
    slot than the first: tiles of 256 x 256 (the first), 128 x 128 (the fourth) and 256 x 128"""
    assert cai.load().cai_bf16_tiles(2 * ff, width, tokens, 1) == {(300, 12000): 5, (600, 5632): 3}.get((tokens, ff), 4)
    m = Model(tmp_path, B.config([B.layer(B.delta(), ff=ff)], width=width, vocab=67), seed=tokens, edit=only("feed-forward"), rank_a=3, rank_g=20)
    tok = m.tokens(tokens, 1)
    dec = m.open(cai, 768, 1, "bf16")
    check(feed(dec, tok, [tokens]), m.ref(tok), "bf16")
    dec.close()


@pytest.mark.parametrize("rows, cols, tokens, tiles", [(2041, 264, 1100, 1), (4300, 72, 513, 1), (16300, 320, 130, 4), (6200, 328, 2050, 4), (4104, 72, 2100, 4),
                                                      (2041, 264, 2000, 2), (4300, 72, 890, 2), (16300, 320, 193, 2), (16300, 1096, 130, 2), (6200, 328, 2310, 5), (4104, 72, 3810, 5), (4104, 776, 2310, 5)])
def test_one_round_of_large_tiles(cai, rows, cols, tokens, tiles):
    """Tiles of 128 x 128 by sixteen waves (2: one round of them) and of 256 x 256 (5: one round instead of two of smaller ones), one to eighteen steps of 64 deep, rows and
    tokens that end inside a tile; and what sizes a little below them take (1: 64 x 64, 4: 256 x 128).  The bound is that of
    test_products_over_bf16_rows."""
    assert cai.load().cai_bf16_tiles(rows, cols, tokens, 0) == tiles
    rng = np.random.default_rng(rows)
    bits, w = B.to_bf16(rng.standard_normal((rows, cols)))
    w = w.reshape(rows, cols).astype(np.float64); bias = rng.standard_normal(rows).astype(np.float32)
    q = cai.QWeight(cai.BF16, rows, cols, bits, bias)
    x = B.to_bf16(rng.standard_normal((tokens, cols)))[1].reshape(tokens, cols).astype(np.float64)
    assert np.all(np.abs(bf16_rows(cai, q, x) - (x @ w.T + bias)) <= 2.0 ** -19 * (np.abs(x) @ np.abs(w).T + np.abs(bias)))
    q.close()


@pytest.mark.parametrize("width, tokens, ff", [(2056, 1100, 72), (4104, 2050, 72), (2054, 1090, 72), (2056, 1100, 1032), (4104, 2310, 776), (2054, 1090, 1032)])
def test_residuals_of_large_tiles(cai, tmp_path, width, tokens, ff):
    """the stream's update and the norms around it behind tiles of 128 x 128 by sixteen waves and of 256 x 256 (ff of 1032 and of 776, depths at which they are taken), and behind
    the tiles of shallow products; a width that is no whole fours"""
    if ff > 72:
        assert cai.load().cai_bf16_tiles(width, ff, tokens, 0) == (5 if ff == 776 else 2)
    m = Model(tmp_path, B.config([B.layer(B.delta(1, 1, 8, 8, 2), ff=ff)], width=width, vocab=67), seed=width, rank_a=3, rank_g=20)
    tok = m.tokens(tokens, 1)
    dec = m.open(cai, 2368, 1, "bf16")
    check(feed(dec, tok, [tokens]), m.ref(tok), "bf16")
    dec.close()


@pytest.mark.parametrize("width, ff, vocab", [(72, 17, 61), (192, 300, 131), (264, 520, 9), (776, 1100, 1003), (2056, 2120, 67), (328, 4200, 67), (72, 8192, 67), (72, 8200, 67)])
def test_streamed_bf16_products(cai, tmp_path, width, ff, vocab):
    """One to sixteen rows: one partial slot of 256 columns, a last slot of 8 to 200 columns, one to four waves of a row with and without work, two
    to four slots a wave, widths of 8192 columns and past them (another kernel); rows that end inside a tile; fewer tiles than work-groups and more."""
    m = Model(tmp_path, B.config([B.layer(B.delta(), ff=ff)], width=width, vocab=vocab), seed=width, edit=only("feed-forward"), rank_a=3, rank_g=20)
    tok = m.tokens(40, 1)
    dec = m.open(cai, 64, 1, "bf16")
    for cuts in ([1], [2, 3, 5, 7, 8], [9, 16, 15]):
        check(feed(dec, tok, cuts), m.ref(tok), "bf16")
        dec.reset()
    dec.close()


@pytest.mark.parametrize("width, ff, vocab", [(64, 17, 61), (72, 130, 131), (192, 300, 520), (320, 390, 67), (384, 448, 67), (448, 1100, 67), (264, 8200, 67)])
def test_small_tiles_of_few_steps(cai, tmp_path, width, ff, vocab):
    """Tiles of 32 and 64 tokens whose copies run five and two steps ahead: products of one to eight steps, and of many; a token past a tile."""
    m = Model(tmp_path, B.config([B.layer(B.delta(), ff=ff)], width=width, vocab=vocab), seed=width, edit=only("feed-forward"), rank_a=3, rank_g=20)
    tok = m.tokens(130, 1)
    dec = m.open(cai, 192, 1, "bf16")
    for cuts in ([17, 33, 80], [32, 65, 33], [130]):
        check(feed(dec, tok, cuts), m.ref(tok), "bf16")
        dec.reset()
    dec.close()


# ---------------------------------------------------------------- whole models
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("cuts", [[300], [1], [2], [3, 2, 65, 1, 1, 16, 17, 2], [64], [130, 1], [5, 9, 7]], ids=str)
def test_portions_and_decoding_agree_with_the_whole(cai, model, cuts, dt):
    tok = model.tokens(150, 3)
    dec = model.open(cai, 192, 1, dt)
    check(feed(dec, tok, cuts), model.ref(tok), dt)
    assert dec.len() == 150 and dec.cache_rows() <= 128
    dec.close()


@pytest.mark.parametrize("loop", [None, (0, 3, 2), (2, 3, 3), (0, 1, 4), (1, 1, 5), (1, 2, 1), (0, 2, 2)], ids=str)
def test_repeated_layers(cai, tmp_path, loop):
    """stretches at the start, in the middle, at the end, of one layer, empty and run once: each pass has cache and state of its own"""
    cfg = B.config([B.layer(B.delta()), B.layer((B.attn(window=5), B.delta(dim=12)), ff=None), B.layer((B.attn(heads=2, window=70), B.delta()))],
                   loop=loop and dict(start=loop[0], stop=loop[1], times=loop[2]))
    if loop is None:
        del cfg["loop"]
    m = Model(tmp_path, cfg, seed=4)
    tok = m.tokens(100, 1)
    dec = m.open(cai, 128)
    for cuts in ([100], [40, 1], [33, 2, 5]):
        dec.reset()
        check(feed(dec, tok, cuts), m.ref(tok), "f32")
    dec.close()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("dim", [128, 136, 256])
def test_scores_of_single_tokens_add_columns_half_a_row_apart_first(cai, tmp_path, dim, dt):
    """Keys whose 2^25 and -2^25 lie 64 columns apart, beside two ones 8 columns behind each: a score of 2 (the oracle's) where these are the first that meet, of 0 where neighbouring
    groups of eight do, since 2^25 + 1 has no place in 32 bits.  Token 1's key is the negative of the others'."""
    cfg = B.config([B.layer((B.attn(heads=2, kv_heads=1, dim=dim, vdim=24, window=64, scale=1.0), B.delta()), ff=None)], width=64, vocab=40)

    def edit(w):
        w["embed"][:, 0] = 4.0; w["embed"][1::2, 0] = -4.0; w["embed"][:, 1] = 4.0
        w["l0.norm1.alpha"] = np.asarray(8.0); w["l0.norm1"][:2] = 1.0; w["l0.norm1.b"][:2] = 0.0        # tanh(32) = 1 in 32 bits
        p = "l0.mix.left."
        for n, col in (("q", 1), ("k", 0)):
            w[p + n][:] = 0.0; w[p + n][:, col] = 1.0
        w[p + "q.norm"][:] = 1.0; w[p + "k.norm"][:] = 0.0
        w[p + "k.norm"][[0, 64, 8, 72]] = [2.0 ** 25, -2.0 ** 25, 1.0, 1.0]
    m = Model(tmp_path, cfg, seed=dim, edit=edit)
    t = [1 + i % 2 for i in range(24)]
    want, flat = m.ref(t), {n: a.copy() for n, a in m.w.items()}
    flat["l0.mix.left.k.norm"][[8, 72]] = 0.0
    assert err(R.forward(cfg, flat, np.array(t))[4:], want[4:]) > 0.1           # (scores of 0 are seen)
    dec = m.open(cai, 64, 1, dt)
    check(feed(dec, t, [1]), want, dt)
    dec.close()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_a_window_wider_than_the_pool(cai, tmp_path, dt):
    m = Model(tmp_path, B.config([B.layer((B.attn(heads=3, kv_heads=1, dim=40, vdim=72, window=1 << 29), B.delta()))]), seed=6)
    tok = m.tokens(384, 2)
    dec = m.open(cai, 384, 1, dt)
    for cuts in ([384], [300, 1]):
        dec.reset()
        check(feed(dec, tok, cuts), m.ref(tok), dt)
    dec.close()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_first_tokens(cai, model, dt):
    dec = model.open(cai, 64, 1, dt)
    for n in range(1, 7):
        tok = model.tokens(n, 40 + n)
        dec.reset()
        check(feed(dec, tok, [n]), model.ref(tok), dt)
        dec.reset()
        check(feed(dec, tok, [1]), model.ref(tok), dt)
    dec.close()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_mixed_batches_with_reused_slots_and_pages(cai, model, dt):
    """eight requests over three slots; portions of some beside single tokens of others; a pool that the live ones nearly fill"""
    rng = np.random.default_rng(5)
    lens = [70, 9, 131, 1, 64, 33, 90, 200]
    reqs = [model.tokens(n, 100 + i) for i, n in enumerate(lens)]
    dec = model.open(cai, 320, 3, dt)
    todo, live, free = list(range(8)), {}, [0, 1, 2]
    got = {i: [] for i in todo}
    while todo or live:
        while free and todo:
            live[todo.pop(0)] = [free.pop(int(rng.integers(len(free)))), 0]
        pick = [i for i in live if rng.random() < 0.8] or list(live)
        rng.shuffle(pick)
        entries, where = [], []
        for i in pick:
            slot, at = live[i]
            n = min(int(rng.choice([1, 1, 1, 2, 3, 17, 40, 64])), lens[i] - at)
            entries.append((slot, reqs[i][at:at + n], range(n))); where.append((i, n))
        lg = dec.step_batch(entries)[1]
        r0 = 0
        for i, n in where:
            got[i].append(lg[r0:r0 + n]); r0 += n
            live[i][1] += n
            if live[i][1] == lens[i]:
                slot = live.pop(i)[0]
                dec.reset(slot); free.append(slot)
    for i in got:
        check(np.concatenate(got[i]), model.ref(reqs[i]), dt)
    assert dec.room(0) == 320                     # every page came back
    dec.close()


def test_batches_agree_with_each_request_alone_to_rounding(cai, model):
    reqs = [model.tokens(n, 60 + n) for n in (21, 90, 2, 1)]
    dec = model.open(cai, 512, 4)
    alone = []
    for r in reqs:
        alone.append(feed(dec, r, [len(r)])); dec.reset()
    lg = dec.step_batch([(3 - i, r, range(len(r))) for i, r in enumerate(reqs)])[1]
    assert err(lg.astype(np.float64), np.concatenate(alone).astype(np.float64)) < 4e-6
    dec.close()


# ---------------------------------------------------------------- window edges
def pointed(window, heads=2):
    """token 400 + t asks for token t: keys carry a sign vector in the first half of the width, askers the same one in the second,
    W_k reads the first half and W_q the second, so that one score stands far above all others"""
    cfg = B.config([B.layer((B.attn(heads=heads, kv_heads=1, dim=64, vdim=24, window=window, scale=0.15), B.delta()), ff=None)], width=128, vocab=800)

    def edit(w):
        sign = np.sign(np.random.default_rng(77).standard_normal((400, 64)))
        w["embed"] = np.zeros((800, 128)); w["embed"][:400, :64] = sign; w["embed"][400:, 64:] = sign
        w["l0.norm1"] = np.ones(128); w["l0.norm1.b"] = np.zeros(128)
        w["l0.mix.left.k"] = np.eye(64, 128); w["l0.mix.left.q"] = np.concatenate([np.eye(64, 128, 64)] * heads)
        w["l0.mix.left.q.norm"] = np.full(64, 1.0); w["l0.mix.left.k.norm"] = np.full(64, 1.5)
        w["l0.mix.right.out"] = w["l0.mix.right.out"] * 0
    return cfg, edit


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("window", [2, 3, 63, 64, 65, 128, 200, 257])
def test_window_edges(cai, tmp_path, window, dt):
    """a key that outweighs all others, just inside and just outside the window of the token that asks for it: in a prompt, in
    portions and decoded, at page borders and elsewhere"""
    cfg, edit = pointed(window)
    m = Model(tmp_path, cfg, seed=window, edit=edit)
    T = 330
    keys = np.random.default_rng(window).permutation(400)[:T]
    places = [p for p in (0, 5, 59, 63, 64, 70, 127, 128) if p + window < T]
    if window == 2:
        places = places[:-1]
    inside, outside = keys.copy(), keys.copy()
    for p in places:
        inside[p + window - 1] = 400 + keys[p]; outside[p + window] = 400 + keys[p]
    # the oracle tells the edge apart: seen from the last place of the window, not from the next one
    wider = json.loads(json.dumps(cfg)); wider["layers"][0]["mixer"]["left"]["mask"]["size"] = window + 1
    rows = [p + window for p in places if not (outside[p] >= 400)]
    apart = np.abs(R.forward(wider, m.w, outside) - m.ref(outside))[rows].max(1)
    assert apart.min() > 0.1
    dec = m.open(cai, 384, 1, dt)
    for tok in (inside, outside):
        for cuts in ([T], [60, 1], [2, 100, 3], [65, 63, 20, 1, 1, 40]):
            dec.reset()
            check(feed(dec, tok.tolist(), cuts), m.ref(tok), dt)
    dec.close()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_a_far_token_is_kept_by_the_state(cai, tmp_path, dt):
    """slow decay and full-strength writes: what the first tokens wrote is read hundreds of tokens later"""
    cfg = B.config([B.layer(B.delta(heads=2, kv_heads=2, dim=48, vdim=24, conv=1), ff=None)], width=96, vocab=97)

    def edit(w):
        w["l0.mix.dt_bias"] = np.full(2, -9.0); w["l0.mix.k"] = w["l0.mix.q"]; w["l0.mix.b"] = w["l0.mix.b"] * 0.05
    m = Model(tmp_path, cfg, seed=2, edit=edit)
    tok = np.random.default_rng(9).integers(10, 97, 500)
    tok[2] = 5; tok[450:] = np.where(tok[450:] == 5, 11, tok[450:]); tok[490] = 5
    want = m.ref(tok)
    lost = tok.copy(); lost[2] = 6
    assert err(R.forward(cfg, m.w, lost)[490:491], want[490:491]) > 5 * TOL["f32"]
    dec = m.open(cai, 64, 1, dt)
    for cuts in ([500], [470, 1], [33, 2]):
        dec.reset()
        check(feed(dec, tok.tolist(), cuts)[480:], want[480:], dt)
    dec.close()


# ---------------------------------------------------------------- long decoding, generation, scheduler
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_long_decoding_in_a_small_pool(cai, model, dt):
    """a pool of two pages carries 420 tokens: pages behind the window come back while the sequence runs on"""
    tok = model.tokens(420, 8)
    dec = model.open(cai, 128, 1, dt)
    check(feed(dec, tok, [1]), model.ref(tok), dt)
    assert dec.cache_rows() <= 128
    dec.close()


def dec_tail(model, tokens, n):
    out = []
    for _ in range(n):
        out.append(int(model.ref(tokens + out)[-1].argmax()))
    return out


def test_sampled_requests_do_not_depend_on_their_company(cai, model):
    prompts = [model.tokens(n, 20 + n) for n in (8, 40, 21)]
    dec = model.open(cai, 256, 3)
    sched = cai.Scheduler(dec)
    alone = []
    for k, p in enumerate(prompts):
        i = sched.submit(p, 25, temperature=1.3, top_k=12, seed=k + 1); sched.run(); alone.append(sched.result(i)[0])
    ids = [sched.submit(p, 25, temperature=1.3, top_k=12, seed=k + 1) for k, p in enumerate(prompts)]
    sched.run()
    assert [sched.result(i)[0] for i in ids] == alone
    assert len(set(map(tuple, alone))) == 3 and any(a != greedy_of(dec, p) for a, p in zip(alone, prompts))
    # a drawn token is one of the most probable ones
    lg = model.ref(prompts[0] + alone[0][:-1])[len(prompts[0]) - 1:]
    for row, t in zip(lg, alone[0]):
        assert t in np.argsort(row)[-14:]
    sched.close(); dec.close()


def greedy_of(dec, p):
    dec.reset()
    return greedy(dec, p, 25)


def test_the_scheduler_serves_the_uniform_decoders_too(cai):
    from helpers.fixtures_io import ref_path
    dec = cai.Decoder.load(ref_path("tiny_llama_f32.gguf"), 32, 2, cai.DTYPE_F32)
    prompts = [[1, 5, 2, 7], [3, 0, 6], [4, 4, 1, 2, 3, 5, 6, 7, 0, 1, 2]]
    want = []
    for p in prompts:
        dec.reset()
        out = [dec.prefill(p)[0]]
        while len(out) < 6:
            out.append(int(dec.step([out[-1]], [len(p) + len(out) - 1])[0][0]))
        want.append(out)
    sched = cai.Scheduler(dec, portion=5)
    ids = [sched.submit(p, 6) for p in prompts]
    sched.run()
    assert [sched.result(i)[0] for i in ids] == want
    # inner rows of a long entry
    dec.reset()
    lg = dec.step_batch([(0, prompts[2], [0, 5, 10])])[1]
    dec.reset()
    one = np.array([dec.step([t], [p])[1][0] for p, t in enumerate(prompts[2])])
    assert err(lg, one[[0, 5, 10]]) < 1e-5
    sched.close(); dec.close()


# ---------------------------------------------------------------- sessions
def test_snapshot_restore_fork_and_hidden_state(cai, model):
    tok = model.tokens(120, 31)
    dec = model.open(cai, 384, 2)
    feed(dec, tok[:80], [80])
    snap = dec.snapshot()
    dec.fork(0, 1)
    a = feed(dec, tok[80:], [7], 0)
    b = feed(dec, tok[80:], [1], 1)
    check(a, model.ref(tok)[80:], "f32"); check(b, model.ref(tok)[80:], "f32")
    dec.reset(1)
    dec.restore(snap, 1)
    assert dec.len(1) == 80
    check(feed(dec, tok[80:], [40], 1), model.ref(tok)[80:], "f32")
    h = dec.hidden_state(39)
    check((R.linear(model.w["head"], h.astype(np.float64)))[None], model.ref(tok)[-1:], "f32")
    t, p = dec.candidates(5, row=39)
    assert t.tolist() == np.argsort(-model.ref(tok)[-1])[:5].tolist()
    with pytest.raises(cai.CaiError):
        dec.truncate(100, 1)                      # recurrent state cannot be taken back
    dec.truncate(0, 1)
    assert dec.len(1) == 0
    cai.load().cai_kv_snap_destroy(snap)
    dec.close()


def test_a_full_pool_refuses_a_step_and_changes_nothing(cai, tmp_path):
    m = Model(tmp_path, B.config([B.layer((B.attn(window=500), B.delta()))]), seed=3)
    tok = m.tokens(140, 4)
    dec = m.open(cai, 128, 2)
    a = feed(dec, tok[:60], [60], 0)
    feed(dec, tok[:50], [50], 1)
    with pytest.raises(cai.CaiError):
        dec.step_batch([(0, tok[60:70], [9]), (1, tok[50:60], [9])])
    assert dec.len(0) == 60 and dec.len(1) == 50 and dec.room(0) == 4
    b = feed(dec, tok[60:64], [2], 0)
    dec.reset(1)
    c = feed(dec, tok[64:128], [64], 0)
    check(np.concatenate([a, b, c]), m.ref(tok[:128]), "f32")
    with pytest.raises(cai.CaiError):
        dec.step_batch([(0, tok[128:129], [0])])
    for bad in ([(0, [999], [0])], [(2, [1], [0])], [(0, [1], []), (0, [1], [])]):
        with pytest.raises(cai.CaiError):
            dec.step_batch(bad)
    for f in (lambda: dec.set_eviction(1, 2), lambda: dec.set_rope_scaling(1, 2.0), lambda: dec.profile(1)):
        with pytest.raises(cai.CaiError):
            f()
    sched = cai.Scheduler(dec)
    with pytest.raises(cai.CaiError):
        sched.submit(tok, 10)
    sched.close(); dec.close()


@pytest.mark.parametrize("name, change", [
    ("heads", lambda c, w: c["layers"][0]["mixer"].update(heads=3, kv_heads=2)), ("type", lambda c, w: c["layers"][0].update(type="other")),
    ("mlp.gate", lambda c, w: c["layers"][0]["mlp"].update(ff=57)), ("kind", lambda c, w: c["layers"][0]["mlp"].update(kind="other")),
    ("head", lambda c, w: w.pop("head")), ("dim", lambda c, w: c["layers"][0]["mixer"].pop("dim")), ("loop.stop", lambda c, w: c["loop"].update(stop=9)),
    ("alpha", lambda c, w: w.pop("l0.norm2.alpha")), ("eps", lambda c, w: c["norm"].clear())])
def test_loader_names_what_is_wrong(cai, tmp_path, name, change):
    cfg = B.config([B.layer(B.delta())])
    w = B.weights(cfg)
    change(cfg, w)
    B.write(str(tmp_path), cfg, w)
    with pytest.raises(cai.CaiError) as e:
        cai.Decoder.load(str(tmp_path), 64)
    assert name in str(e.value)


# ---------------------------------------------------------------- programs
def test_command_line_generation(cai, model):
    prompts = [model.tokens(9, 1), model.tokens(20, 2)]
    dec = model.open(cai, 128)
    want = []
    for p in prompts:
        want.append(greedy(dec, p, 7)); dec.reset()
    dec.close()
    exe = os.path.join(ROOT, "neural-api_amd", "host", "caihip_run")
    one = subprocess.run([exe, model.folder, "7", "--dtype", "float32"] + [str(t) for t in prompts[0]], capture_output=True, text=True, timeout=100)
    assert one.returncode == 0 and [int(t) for t in one.stdout.splitlines()[0].split()] == want[0], one.stdout + one.stderr
    both = subprocess.run([exe, model.folder, "7", "--dtype", "float32", "--portion", "4"] + [str(t) for t in prompts[0]] + ["--"] + [str(t) for t in prompts[1]],
                          capture_output=True, text=True, timeout=100)
    assert [[int(t) for t in s.split()] for s in both.stdout.splitlines()] == want, both.stdout + both.stderr


@pytest.mark.parametrize("dt, name", [("f32", "float32"), ("bf16", "bfloat16")])
def test_trace_replay(cai, model, tmp_path, dt, name):
    a, b = model.tokens(50, 6), model.tokens(30, 7)
    steps = [dict(step=0, entries=[dict(id="x", tokens=a[:40], want=[39, 0])], end=[]), dict(step=1, entries=[dict(id="y", tokens=b[:2], want=[])], end=[]),
             dict(step=2, entries=[dict(id="y", tokens=b[2:], want=[27]), dict(id="x", tokens=a[40:41], want=[0])], end=["y"]),
             dict(step=3, entries=[dict(id="z", tokens=b, want=[29]), dict(id="x", tokens=a[41:], want=[8, 7])], end=["x", "z"])]
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", model.folder, "--dtype", name, "--out", str(tmp_path), "--max-tokens", "128"],
                       input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and [x for x in r.stdout.splitlines() if x.startswith("done")] == ["done %d" % i for i in range(4)], r.stderr
    got = lambda i: np.fromfile(tmp_path / ("%d.f32" % i), "<f4").reshape(-1, model.cfg["vocab"])
    check(got(0), model.ref(a)[[39, 0]], dt)
    assert not os.path.exists(tmp_path / "1.f32")
    check(got(2), np.stack([model.ref(b)[29], model.ref(a)[40]]), dt)
    check(got(3), np.stack([model.ref(b)[29], model.ref(a)[49], model.ref(a)[48]]), dt)
