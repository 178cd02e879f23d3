"""Prompts on a device that has no memory for the buffers of a large pass, forced from the host
(moert_pass_limit_inject: the request is one that no device can serve): smaller passes, single steps where there is
memory for none, the same results bit for bit, and a model that stays usable."""
import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def model(seed=23):
    cfg = moert.Config(**{**moert.GRANITE_1B, "layers": 2, "vocab": 211})
    return cfg, moert.SynthModel(cfg, seed=seed, std=0.05)


def read(g, toks, pos0):
    g.set_position(pos0)
    lg, am = g.prefill(toks)
    n = pos0 + len(toks)
    return [lg.view(np.uint32), am, g.hidden().view(np.uint32), g.position()] + [
        a[:, pos0:] for l in range(g.cfg.layers) for a in g.read_kv(l, n)]


def same(a, b, label):
    for x, y in zip(a, b):
        assert np.array_equal(x, y), label


def test_prompts_in_smaller_passes_and_in_steps(gpu):
    cfg, m = model()
    g, ref = (moert.GpuModel(m, 640, attn_splits=8) for _ in range(2))
    rng = np.random.default_rng(2)
    # nothing, then 32 and 96 -> 64 positions, with a prompt that asks for more than that, then all that it asks for
    for limit, n in ((0, 40), (0, 1), (32, 70), (96, 300), (96, 530), (-1, 530)):
        print(f"[case] limit {limit} prompt {n}", flush=True)
        toks = rng.integers(0, cfg.vocab, n)
        g.pass_limit_inject(limit)
        same(read(g, toks, 7), read(ref, toks, 7), (limit, n))
    g.close()
    ref.close()


def test_generate_without_memory_for_a_pass(gpu):
    cfg, m = model()
    g, ref = (moert.GpuModel(m, 128, attn_splits=8) for _ in range(2))
    prompt = np.random.default_rng(3).integers(0, cfg.vocab, 40)
    want, wgaps = ref.generate(prompt, 5, gaps=True)
    for limit in (0, 32, -1):
        g.pass_limit_inject(limit)
        g.reset()
        out, gaps = g.generate(prompt, 5, gaps=True)
        assert np.array_equal(out, want) and np.array_equal(gaps, wgaps), limit
        assert g.position() == ref.position()
    g.close()
    ref.close()


def test_grouped_prompts_in_smaller_passes(gpu):
    """Mode 1 keeps the buffers of a step of 32 positions from the mode's start; without memory for those the mode is a
    device error, as any allocation of a model that fails."""
    cfg, m = model()
    g, ref = (moert.GpuModel(m, 640, attn_splits=8) for _ in range(2))
    g.batched_mode(1)
    ref.batched_mode(1)
    rng = np.random.default_rng(4)
    for limit, n in ((32, 107), (64, 530), (-1, 530)):
        print(f"[case] grouped limit {limit} prompt {n}", flush=True)
        toks = rng.integers(0, cfg.vocab, n)
        g.pass_limit_inject(limit)
        same(read(g, toks, 5), read(ref, toks, 5), (limit, n))
    g.close()
    ref.close()
    h = moert.GpuModel(m, 64, attn_splits=1)
    h.pass_limit_inject(0)
    with pytest.raises(moert.MoertError) as e:
        h.batched_mode(1)
    assert e.value.code == -1
    h.close()
