"""Multi-position steps of few positions (few.hip) against single decode steps, bit for bit: every weight type and the
two model shapes, position counts around the staged group of 8 positions and around the rule's lines (8 positions of
quantised weights, 14 of f32), from the start of a cache and across a tile edge of it, and a step behind a long one on
the same buffers."""
import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def run(g, toks, pos0, batched):
    g.set_position(pos0)
    if batched:
        lg, am = g.step_batched(toks)
    else:
        for t in toks:
            lg, _, _, am = g.step(int(t))
    n = pos0 + len(toks)
    return [lg.view(np.uint32), am, g.hidden().view(np.uint32), g.position()] + [
        a[:, pos0:] for l in range(g.cfg.layers) for a in g.read_kv(l, n)]


@pytest.mark.parametrize("wdtype", [moert.Q8_0, moert.Q4_0, moert.F32])
@pytest.mark.parametrize("shape", ["1b", "3b", "tiny"])
def test_few_positions_equal_single_steps(gpu, shape, wdtype):
    base = {"1b": moert.GRANITE_1B, "3b": moert.GRANITE_3B, "tiny": moert.TINY}[shape]
    cfg = moert.Config(**{**base, "layers": 2, "vocab": 211})
    m = moert.SynthModel(cfg, seed=31, wdtype=wdtype, embed_dtype=moert.Q8_0, std=0.05,
                         zipf_s=1.1 if shape == "3b" else None)
    g = moert.GpuModel(m, 320, attn_splits=4)
    rng = np.random.default_rng(wdtype + 41)
    for pos0, n in ((0, 2), (2, 1), (61, 3), (60, 8), (120, 7), (121, 9), (0, 32), (30, 5), (190, 13), (50, 14), (64, 15)):
        print(f"[case] {shape} dtype {wdtype} pos {pos0} n {n}", flush=True)
        toks = rng.integers(0, cfg.vocab, n)
        for a, b in zip(run(g, toks, pos0, True), run(g, toks, pos0, False)):
            assert np.array_equal(a, b), (pos0, n)
    # one token at every position: every expert of it has all positions as members
    toks = np.full(8, 17)
    for a, b in zip(run(g, toks, 100, True), run(g, toks, 100, False)):
        assert np.array_equal(a, b)
    g.close()
