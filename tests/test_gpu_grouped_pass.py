"""Grouped mode (mode 1): prompts read in passes against the same tokens in steps of 32 positions, bit for bit, on both
row lengths: a short prompt, then one of more than a pass (530 tokens: two unequal passes on a boundary of steps, the
last step partial) on grown buffers, then continuations from positions that are no multiple of 32, the last step of one,
16, 17 and 31 positions."""
import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def state(g, pos0, n):
    return [g.hidden().view(np.uint32), g.position()] + [
        a[:, pos0:] for l in range(g.cfg.layers) for a in g.read_kv(l, pos0 + n)]


@pytest.mark.parametrize("shape,zipf", [("1b", None), ("3b", None), ("3b", 1.1)])
def test_grouped_passes_equal_steps_of_32(gpu, shape, zipf):
    base = {"1b": moert.GRANITE_1B, "3b": moert.GRANITE_3B}[shape]
    cfg = moert.Config(**{**base, "layers": 2, "vocab": 211})
    m = moert.SynthModel(cfg, seed=47, std=0.05, zipf_s=zipf)
    g, ref = (moert.GpuModel(m, 1216, attn_splits=8) for _ in range(2))
    g.batched_mode(1)
    ref.batched_mode(1)
    rng = np.random.default_rng(9)
    for pos0, n in ((0, 20), (0, 530), (530, 33), (7, 48), (563, 49), (612, 95), (1, 1100)):
        print(f"[case] {shape} zipf {zipf} pos {pos0} n {n}", flush=True)
        toks = rng.integers(0, cfg.vocab, n)
        g.set_position(pos0)
        lg, am = g.prefill(toks)
        ref.set_position(pos0)
        for i in range(0, n, 32):
            rlg, ram = ref.step_batched(toks[i:i + 32])
        assert np.array_equal(lg.view(np.uint32), rlg.view(np.uint32)) and am == ram, (pos0, n)
        for a, b in zip(state(g, pos0, n), state(ref, pos0, n)):
            assert np.array_equal(a, b), (pos0, n)
    g.close()
    ref.close()
