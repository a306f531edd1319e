"""The hybrid model's f64 sums under wide exponent ranges.

The exact hybrid step adds the f32 products and squares of its linears, norms,
gates and delta rule in f64 as the reference does, but as trees and split sums
where the reference runs one chain.  The two can differ only where a partial
sum rounds, which needs terms about 29 binades apart, and then only when the
f64 value sits within that difference of an f32 rounding boundary.

N(0, 0.02) weights never get there.  Here every matrix row, norm weight and
conv tap is scaled by 2^U[-6, 5].  A 300-token and a 90-token prompt are
stepped in chunks beside each other, then decoded, with the packed-prefill
regime off; every sampled row's logits and at the end the whole state are
compared with the oracle, and the number of differing bits is printed."""
import numpy as np
import pytest

import orc
import synth35
from test_gpu_qwen35 import make_q35, tiny
from test_gpu_qwen35_order import edit

pytestmark = pytest.mark.gpu


def spread(t, seed):
    rng = np.random.default_rng(seed)
    for name in list(t):
        if name.endswith(("A_log", "dt_bias")):
            continue

        def scaled(f):
            e = np.exp2(rng.integers(-6, 6, f.shape[:1] + (1,) * (f.ndim - 1))).astype(np.float32)
            if f.ndim == 1 and not name.endswith("linear_attn.norm.weight"):
                return (f + 1) * e - 1  # zero-centred norms scale by w + 1
            return f * e

        edit(t, name, scaled)


@pytest.mark.parametrize("heads,key_dim,value_dim", [(2, 32, 32), (2, 128, 64)])
def test_wide_exponent_range_matches_oracle(heads, key_dim, value_dim):
    print(f"case: hybrid wide exponent range, {heads} heads of {key_dim} keys x {value_dim}", flush=True)
    cfg = tiny(layers=4, pattern="LLLF", hidden=320, intermediate=448, heads=4, kv_heads=2, key_heads=heads,
               value_heads=heads, key_dim=key_dim, value_dim=value_dim, context=512)
    cfg, t = synth35.in_memory(cfg, seed=31, tied=False)
    spread(t, 32)
    m = make_q35(cfg, t, False, max_lanes=2, max_rows=128, max_seqs=2, max_context=400)
    o = orc.Qwen35Model(cfg, t, threads=8)
    rng = np.random.default_rng(33)
    tokens = [[int(v) for v in rng.integers(0, cfg["vocabulary"], n)] for n in (312, 102)]
    seqs, sess = [m.seq_alloc() for _ in tokens], [o.session(400) for _ in tokens]
    plan = [(60, 45)] * 2 + [(60, 0)] * 3 + [(1, 1)] * 12
    at, differing, compared, worst, top = [0, 0], 0, 0, 0.0, 0.0
    for step, lens in enumerate(plan):
        live = [i for i in range(2) if lens[i]]
        res = m.step([dict(seq=seqs[i], tokens=tokens[i][at[i]:at[i] + lens[i]], logits=True) for i in live])
        for i, r in zip(live, res):
            assert r["status"] == 0, (step, i)
            for tok in tokens[i][at[i]:at[i] + lens[i]]:
                assert not any(o.forward_batch([sess[i]], [tok]))
            at[i] += lens[i]
            want = sess[i].logits()
            differing += int((r["logits"].view(np.uint32) != want.view(np.uint32)).sum())
            compared += want.size
            top = max(top, float(np.abs(want).max()))
            worst = max(worst, float(np.abs(r["logits"].astype(np.float64) - want).max()))
            assert r["argmax"] == int(np.argmax(want)), (step, i)
    words = bad = 0
    for i in range(2):
        for layer, full in enumerate(cfg["full"]):
            for which in ((0, 1) if full else (2, 3)):
                got, want = m.read_state(seqs[i], layer, which), sess[i].state(layer, which).reshape(-1)
                words += got.size
                bad += int((got.view(np.uint32) != want.view(np.uint32)).sum())
    print(f"{differing} of {compared} logits (up to {top:.3g}, max-abs {worst:.3g}) and "
          f"{bad} of {words} state words differ in bits", flush=True)
    assert differing == 0 and bad == 0
