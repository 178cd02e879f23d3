"""Metrics while moert_generate reads a long prompt in passes: the progress through the prompt is published, and the
speed of the new tokens does not count the prompt's."""
import threading
import time

import numpy as np
import pytest

import moert

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(gpu):
    cfg = moert.Config(**{**moert.GRANITE_1B, "layers": 16, "vocab": 211})
    return moert.SynthModel(cfg, seed=3, std=0.05)


def generate(m, path, n_new, gaps):
    """1500 prompt tokens (three passes) and n_new new ones, every read-back published: the (state, speed) pairs that a
    thread reading the file throughout saw, and the request."""
    g = moert.GpuModel(m, 2560, attn_splits=8)
    mx = moert.Metrics(path)
    g.attach_metrics(mx, 0)
    prompt = np.random.default_rng(8).integers(0, m.cfg.vocab, 1500)
    g.generate(prompt, 8)  # the passes' buffers
    g.reset()
    seen, stop = [], threading.Event()

    def watch():
        while not stop.is_set():
            kind, s = moert.read_metrics(path)
            if kind == "live" and (not seen or seen[-1] != (s["state"], s["speed"])):
                seen.append((s["state"], s["speed"]))
            time.sleep(0.0001)

    t = threading.Thread(target=watch)
    t.start()
    try:
        g.generate(prompt, n_new, gaps=gaps)
    finally:
        stop.set()
        t.join()
    request = moert.read_metrics(path)[1]["requests"][0]
    print(request, *seen[:20], sep="\n")
    g.attach_metrics(None)
    g.close()
    mx.close()
    assert (request["prompt_tokens"], request["output_tokens"]) == (1500, n_new)
    return seen, request


def test_progress_through_a_prompt_read_in_passes(model, tmp_path):
    """The first pass's read-back is complete milliseconds before the last of 1000 steps is launched, and the next one
    waits behind everything launched by then: the prompt's progress stands in the file for that long."""
    seen, _ = generate(model, tmp_path / "metrics.json", 1000, False)
    done = [s["done"] for s, _ in seen if s["kind"] == "reading"]
    assert any(0 < d < 1500 for d in done), done


def test_the_decode_speed_does_not_count_the_prompt(model, tmp_path):
    """With gaps every step is waited for, so read-backs follow one another through the new tokens, the first of them
    behind the prompt. A window that counted the prompt's tokens as new ones would show hundreds of times the decode
    speed of the request."""
    seen, request = generate(model, tmp_path / "metrics.json", 60, True)
    now = [sp["decode_now"] for s, sp in seen if s["kind"] == "generating"]
    assert len(now) > 2 and max(now) < 4 * request["decode_tok_s"], (now, request)
