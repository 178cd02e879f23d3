"""Results and inputs of a model call through its pinned buffer: what the public entry points refuse."""
import ctypes

import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def tiny(layers=2):
    cfg = moert.Config(hidden=256, inter=128, layers=layers, heads=4, kv_heads=2, head_dim=64, vocab=97, experts=8,
                       top_k=2)
    return cfg, moert.SynthModel(cfg, seed=13, std=0.1)


def test_null_outputs_are_errors(gpu):
    """A null hidden state is a reported device error that leaves the handle unusable, as a failed copy does; the
    entry points that check their outputs refuse a null one before that."""
    cfg, m = tiny()
    g = moert.GpuModel(m, 64, attn_splits=1)
    g.step(3)
    null, n = ctypes.c_void_p(None), ctypes.c_int(2)
    lib = moert.lib()
    assert lib.moert_read_logits(g.h, null) == -2
    assert lib.moert_read_kv_fp16(g.h, 0, null, null, n) == -5
    assert np.isfinite(g.hidden()).all()
    assert lib.moert_read_hidden(g.h, null) == -1
    assert lib.moert_read_hidden(g.h, null) == -3
    g.close()
