"""Prompts read in large blocks (moert_prefill) against single decode steps, bit for bit: the row products' tiles of 16
and 32 positions with remainders, experts with none, few and many members, every weight type and row length of the two
model shapes, one pass and several, buffers that grow from one prompt to the next; in mode 1 against steps of 32."""
import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def run(g, toks, pos0, batched):
    g.set_position(pos0)
    if batched:
        lg, am = g.prefill(toks)
    else:
        for t in toks:
            lg, _, _, am = g.step(int(t))
    n = pos0 + len(toks)
    return lg, am, g.hidden(), [tuple(a[:, pos0:n].copy() for a in g.read_kv(l, n)) for l in range(g.cfg.layers)]


def same(a, b, label):
    assert np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32)), label
    assert a[1] == b[1], label
    assert np.array_equal(a[2].view(np.uint32), b[2].view(np.uint32)), label
    for l, (x, y) in enumerate(zip(a[3], b[3])):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), (label, l)


@pytest.mark.parametrize("wdtype", [moert.Q8_0, moert.Q4_0, moert.F32])
@pytest.mark.parametrize("shape", ["1b", "3b", "tiny"])
def test_prompts_equal_single_steps(gpu, shape, wdtype):
    base = {"1b": moert.GRANITE_1B, "3b": moert.GRANITE_3B, "tiny": moert.TINY}[shape]
    cfg = moert.Config(**{**base, "layers": 2, "vocab": 211})
    m = moert.SynthModel(cfg, seed=17, wdtype=wdtype, embed_dtype=moert.Q8_0, std=0.05,
                         zipf_s=1.1 if shape == "3b" else None)
    g = moert.GpuModel(m, 1152, attn_splits=8)
    rng = np.random.default_rng(wdtype + 29)
    for pos0, n in ((0, 1), (3, 33), (36, 16), (52, 257), (0, 530), (530, 81)):
        print(f"[case] {shape} dtype {wdtype} pos {pos0} n {n}", flush=True)
        toks = rng.integers(0, cfg.vocab, n)
        want = run(g, toks, pos0, False)
        same(run(g, toks, pos0, True), want, (pos0, n))
    g.close()


def test_mode_1_prompts_equal_steps_of_32(gpu):
    cfg = moert.Config(**{**moert.GRANITE_1B, "layers": 2, "vocab": 211})
    m = moert.SynthModel(cfg, seed=18, std=0.05)
    g = moert.GpuModel(m, 256, attn_splits=8)
    g.batched_mode(1)
    toks = np.random.default_rng(4).integers(0, cfg.vocab, 107)
    got = run(g, toks, 0, True)
    g.set_position(0)
    for i in range(0, len(toks), 32):
        lg, am = g.step_batched(toks[i:i + 32])
    want = lg, am, g.hidden(), [tuple(a.copy() for a in g.read_kv(l, len(toks))) for l in range(cfg.layers)]
    same(got, want, "mode 1")
    g.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_generate_equals_steps_for_every_prompt_length(gpu, mode):
    """moert_generate reads a prompt of more than a few tokens in passes: the tokens and gaps of prompts of 1 to 6 and
    of 40 tokens equal those of a loop of single steps, whatever the model's mode of its own multi-position steps."""
    cfg = moert.Config(**{**moert.GRANITE_1B, "layers": 2, "vocab": 211})
    m = moert.SynthModel(cfg, seed=19, std=0.05)
    g = moert.GpuModel(m, 128, attn_splits=8)
    g.batched_mode(mode)
    rng = np.random.default_rng(6)
    pos = 0
    for n in (1, 2, 3, 4, 5, 6, 40):
        prompt = rng.integers(0, cfg.vocab, n)
        g.set_position(pos)
        out, gaps = g.generate(prompt, 4, gaps=True)
        end, lg = g.position(), g.read_logits()
        g.set_position(pos)
        want, feed = [], list(prompt)
        for t in feed:
            slg, _, _, am = g.step(int(t))
        wgaps = []
        for i in range(4):
            s = np.sort(slg)
            want.append(am)
            wgaps.append(np.float32(s[-1] - s[-2]))
            if i < 3:
                slg, _, _, am = g.step(am)
        assert out.tolist() == want and np.array_equal(gaps, np.array(wgaps, np.float32)), n
        assert end == pos + n + 3 and np.array_equal(lg.view(np.uint32), slg.view(np.uint32)), n
        pos += 3
    g.close()
