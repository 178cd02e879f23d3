"""Multi-position attention on the f32 matrix cores (attn_mm.hip) against single decode steps, bit for bit, where its
tiles and units can go wrong: every group size and tiles-per-split count (rounds of four tiles included), lengths
around tile edges, unit counts around 16, cache rows past the length that hold infinities and NaNs, and a K/V row of
the block itself that overflows fp16 (it must not reach the positions before it)."""
import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def model(heads, kv_heads, layers=2, wdtype=moert.F32, seed=5):
    cfg = moert.Config(hidden=256, inter=128, layers=layers, heads=heads, kv_heads=kv_heads, head_dim=64, vocab=97,
                       experts=4, top_k=2, embedding_multiplier=2.0, residual_multiplier=0.5,
                       attention_multiplier=0.25, logits_scaling=4.0)
    return moert.SynthModel(cfg, seed=seed, wdtype=wdtype, embed_dtype=moert.F32, std=0.1)


def steps(g, toks, pos0):
    g.set_position(pos0)
    for t in toks:
        lg = g.step(int(t))[0]
    n = pos0 + len(toks)
    return lg, [tuple(a[:, pos0:n].copy() for a in g.read_kv(l, n)) for l in range(g.cfg.layers)]


def block(g, toks, pos0):
    g.set_position(pos0)
    lg, _ = g.prefill(toks)
    n = pos0 + len(toks)
    return lg, [tuple(a[:, pos0:n].copy() for a in g.read_kv(l, n)) for l in range(g.cfg.layers)]


def same(a, b, label):
    assert np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32)), label
    for l, (x, y) in enumerate(zip(a[1], b[1])):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), (label, l)


@pytest.mark.parametrize("heads,kv_heads", [(4, 4), (4, 2), (4, 1)])
@pytest.mark.parametrize("tps", [1, 2, 3, 4, 5, 9])
def test_blocks_equal_single_steps(gpu, heads, kv_heads, tps):
    m = model(heads, kv_heads)
    max_len = 576  # 9 tiles
    g = moert.GpuModel(m, max_len, attn_splits=-(-9 // tps))
    rng = np.random.default_rng(heads * 100 + tps)
    for l in range(m.cfg.layers):
        k = rng.standard_normal((kv_heads, max_len, 64)).astype(np.float16)
        v = rng.standard_normal((kv_heads, max_len, 64)).astype(np.float16)
        g.kv_prefill(l, k.view(np.uint16), v.view(np.uint16))
    for pos0, n in ((0, 1), (59, 6), (63, 5), (64, 17), (300, 32), (543, 33)):
        print(f"[case] heads {heads}/{kv_heads} tps {tps} pos {pos0} n {n}", flush=True)
        toks = rng.integers(0, m.cfg.vocab, n)
        same(block(g, toks, pos0), steps(g, toks, pos0), (pos0, n))
    g.close()


def test_rows_past_the_length_are_never_read_into_a_sum(gpu):
    m = model(8, 2)
    g = moert.GpuModel(m, 128, attn_splits=2)
    c = moert.GpuModel(m, 128, attn_splits=2)
    rng = np.random.default_rng(3)
    for l in range(m.cfg.layers):
        k = rng.standard_normal((2, 128, 64)).astype(np.float16)
        v = rng.standard_normal((2, 128, 64)).astype(np.float16)
        c.kv_prefill(l, k.view(np.uint16), v.view(np.uint16))
        k[:, 40:], v[:, 40:] = np.inf, np.nan
        g.kv_prefill(l, k.view(np.uint16), v.view(np.uint16))
    toks = rng.integers(0, m.cfg.vocab, 21)
    same(block(g, toks, 40), steps(c, toks, 40), "stale rows")
    g.close()
    c.close()


def test_an_overflowing_row_of_the_block_leaves_the_positions_before_it_alone(gpu):
    m = model(8, 2)
    # some V elements of layer 0 overflow fp16, at some positions only
    m.arrays["0.v"] = (m.arrays["0.v"].reshape(128, 256) * np.where(np.arange(128) % 64 == 7, 2e4, 1.0)[:, None]
                       ).astype(np.float32).reshape(-1)
    g = moert.GpuModel(m, 128, attn_splits=2)
    rng = np.random.default_rng(8)
    seen = 0
    for trial in range(8):
        toks = rng.integers(0, m.cfg.vocab, 24)
        got, want = block(g, toks, 0), steps(g, toks, 0)
        v = want[1][0][1].view(np.float16)
        bad = np.flatnonzero(~np.isfinite(v).all(axis=(0, 2)))
        first = int(bad[0]) if bad.size else len(toks)
        seen += 0 < first < len(toks)
        for l in range(m.cfg.layers):
            for a, b in zip(got[1][l], want[1][l]):
                assert np.array_equal(a[:, :first], b[:, :first]), (trial, first, l)
        assert np.array_equal(got[1][0][1], want[1][0][1])  # layer 0's rows, the infinities included
    assert seen > 0
    g.close()
