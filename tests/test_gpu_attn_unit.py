"""Decode attention of one length in one or two launches against the oracle, bit for bit: every group size and count of
tiles of the one-launch form (lengths up to 256) with splits of one tile to more tiles than the length has, the first
lengths of the two-launch form, and poison in the rows past the length."""
import numpy as np
import pytest

import moert
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads", [(2, 2), (4, 2), (6, 2), (8, 2), (24, 8)])
def test_short_lengths_equal_the_oracle(gpu, heads, kv_heads):
    max_len = 512
    q = moert.synth_normal(91, heads, heads * 64)
    kf = moert.synth_normal(92, heads, kv_heads * max_len * 64)
    vf = moert.synth_normal(93, heads, kv_heads * max_len * 64)
    for length in (1, 63, 64, 65, 127, 130, 192, 193, 255, 256, 257, 320, 321):
        kc = oracle.f2h(kf).reshape(kv_heads, max_len, 64).copy()
        vc = oracle.f2h(vf).reshape(kv_heads, max_len, 64).copy()
        kc[:, length:] = 0x7E00
        vc[:, length:] = 0xFC00
        for tps in (1, 2, 3, 4, 5, 8):
            print(f"[case] heads {heads}/{kv_heads} len {length} tiles/split {tps}", flush=True)
            got = moert.attn_decode(q, kc.reshape(-1), vc.reshape(-1), heads, kv_heads, max_len, length, 0.125, tps)
            want = oracle.attention(q, kc.reshape(-1), vc.reshape(-1), heads, kv_heads, max_len, length, 0.125, tps)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (length, tps)
