"""The hybrid model's prompt-chunk kernels (causal conv, delta rule, norms) at
the edges of their tiles, bit for bit against the oracle: chunk lengths around
the token groups they stage (and up to four tokens, where equal key and value
heads take the fused mixer), every key width, value widths that leave column
groups ragged, conv rings longer than a chunk."""
import numpy as np
import pytest

import synth35
from test_gpu_qwen35 import Pair, tiny

pytestmark = pytest.mark.gpu

SHAPES = [  # key_dim, value_dim, key_heads, value_heads, conv_kernel
    (16, 8, 2, 4, 4), (32, 130, 2, 4, 3), (64, 72, 1, 2, 8), (128, 128, 2, 2, 4), (128, 40, 1, 1, 2),
    (16, 12, 2, 2, 4), (32, 130, 4, 4, 3), (64, 256, 1, 1, 4), (128, 200, 1, 1, 4)]


@pytest.mark.parametrize("shape", SHAPES)
def test_chunks_match_oracle(shape):
    kd, vd, kh, vh, k = shape
    cfg = tiny(layers=2, pattern="LF", key_dim=kd, value_dim=vd, key_heads=kh, value_heads=vh, conv_kernel=k)
    c, t = synth35.in_memory(cfg, seed=kd + vd)
    p = Pair(c, t, max_lanes=4, max_rows=128, max_seqs=4, max_context=200)
    rng = np.random.default_rng(7)
    seqs = [p.alloc() for _ in range(4)]
    for lengths in ((5, 8, 17, 1), (4, 1, 3, 2), (9, 33, 2, 16), (1, 7, 64, 3), (1, 1, 1, 1)):
        print(f"case: hybrid chunks {shape} {lengths}", flush=True)
        p.step([(s, [int(v) for v in rng.integers(0, c["vocabulary"], n)]) for s, n in zip(seqs, lengths)])
        for s in seqs:
            p.check_state(s)
