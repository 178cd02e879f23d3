"""Metrics while moert_generate reads a long prompt in passes: the progress through the prompt is published, and the
speed of the new tokens does not count the prompt's."""
import threading
import time

import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


def test_progress_and_speeds_of_a_prompt_read_in_passes(gpu, tmp_path):
    """1500 prompt tokens (three passes) and 300 new ones, every read-back published; a thread reads the file
    throughout. A read-back waits behind the steps queued before it, so each publication stands for milliseconds.
    Prompt tokens cost about a tenth of a new one's step: a window that counted them as new tokens would show a decode
    speed far above the request's."""
    cfg = moert.Config(**{**moert.GRANITE_1B, "layers": 8, "vocab": 211})
    m = moert.SynthModel(cfg, seed=3, std=0.05)
    g = moert.GpuModel(m, 1856, attn_splits=8)
    path = tmp_path / "metrics.json"
    mx = moert.Metrics(path)
    g.attach_metrics(mx, 0)
    prompt = np.random.default_rng(8).integers(0, cfg.vocab, 1500)
    g.generate(prompt, 8)  # the passes' buffers
    g.reset()
    seen, stop = [], threading.Event()

    def watch():
        while not stop.is_set():
            kind, s = moert.read_metrics(path)
            if kind == "live":
                seen.append((s["state"], s["speed"]))
            time.sleep(0.0001)

    t = threading.Thread(target=watch)
    t.start()
    try:
        g.generate(prompt, 300)
    finally:
        stop.set()
        t.join()
    request = moert.read_metrics(path)[1]["requests"][0]
    distinct = []
    for s in seen:
        if not distinct or distinct[-1] != s:
            distinct.append(s)
    print(request, *distinct, sep="\n")
    g.attach_metrics(None)
    g.close()
    mx.close()
    assert (request["prompt_tokens"], request["output_tokens"]) == (1500, 300)
    reading = [s for s, _ in distinct if s["kind"] == "reading"]
    assert any(0 < s["done"] < 1500 for s in reading), reading
    now = [sp["decode_now"] for s, sp in distinct if s["kind"] == "generating"]
    assert now and max(now) < 4 * request["decode_tok_s"], (now, request)
