"""Whole steps on the kernel instances that wide matrices and many rows pick,
bit for bit against the oracle: several batch tiles per workgroup in the exact
F16, K-quant and hybrid linears, each split of K over waves, and the combine
with several heads per workgroup (the last group not full)."""
import numpy as np
import pytest

import cohx
import orc
import synth
import synth35
from test_gpu_kquant import model_dtypes
from test_gpu_qwen35 import Pair, tiny
from test_gpu_step import build

pytestmark = pytest.mark.gpu


def check(c, m, o, plan, context, seed=3):
    """Steps of the given tokens per lane (0: the lane sits out): every lane's
    logits and greedy id, and at the end every K/V row."""
    rng = np.random.default_rng(seed)
    n = max(len(lens) for lens in plan)
    seqs, sess = [m.seq_alloc() for _ in range(n)], [o.session(context) for _ in range(n)]
    used = set()
    for step, lens in enumerate(plan):
        live = [i for i, k in enumerate(lens) if k]
        used.update(live)
        toks = {i: [int(v) for v in rng.integers(0, c["vocabulary"], lens[i])] for i in live}
        res = m.step([dict(seq=seqs[i], tokens=toks[i], logits=True) for i in live])
        for j in range(max(lens)):
            unit = [i for i in live if j < lens[i]]
            for u in range(0, len(unit), 16):  # the oracle's units of at most 16 lanes
                part = unit[u:u + 16]
                assert not o.forward_batch([sess[i] for i in part], [toks[i][j] for i in part]).any()
        bad = 0
        for i, r in zip(live, res):
            assert r["status"] == 0, (step, i)
            want = sess[i].logits()
            bad += int((r["logits"].view(np.uint32) != want.view(np.uint32)).sum())
            assert r["argmax"] == orc.Sampler().sample(want)[1], (step, i)
        print(f"step {step}, {sum(lens)} rows: {bad} logits differ in bits", flush=True)
        assert bad == 0, step
    for i in sorted(used):
        for layer in range(c["layers"]):
            for values in (False, True):
                assert np.array_equal(m.seq_read_kv(seqs[i], layer, values), sess[i].kv(layer, values)), (i, layer)


@pytest.mark.parametrize("vocabulary", [9000, 13000, 25000])
def test_f16_wide_head_and_gate_up(vocabulary):
    """Heads of 563, 813 and 1,563 tiles at 17 and 49 lanes; 304 gate and up
    tile pairs at 56, 70 and 100 rows."""
    print(f"case: F16 head of {vocabulary} rows, gate+up of 4864", flush=True)
    cfg = synth.config(layers=1, hidden=64, intermediate=4864, heads=2, kv_heads=1, vocabulary=vocabulary,
                       context=160)
    c, _, m, o = build("f16", 8, cfg, max_lanes=49, max_rows=100, max_seqs=49, max_context=160)
    check(c, m, o, [(1,) * 17, (1,) * 49, (20, 36), (30, 40), (1, 40, 1, 58)], 160)


def test_f16_wide_qkv():
    """96 qkv tile pairs at 176, 256 and 352 rows, the packed-prefill regime off."""
    print("case: F16 qkv of 3072 rows", flush=True)
    cfg = synth.config(layers=1, hidden=1024, intermediate=32, heads=32, kv_heads=32, vocabulary=64, context=256)
    c, _, m, o = build("f16", 9, cfg, exact=True, max_lanes=8, max_rows=352, max_seqs=8, max_context=200)
    check(c, m, o, [(44,) * 4, (32,) * 8, (44,) * 8], 256)


@pytest.mark.parametrize("hidden,heads,kv_heads", [(384, 6, 3), (384, 3, 3)])
def test_f16_combine_of_several_heads(hidden, heads, kv_heads):
    """8,192 (row, head) pairs and more: four heads of 64 elements a workgroup
    (six heads: 4 + 2) and two of 128 (three heads: 2 + 1), the regime off."""
    print(f"case: F16 combine, {heads} heads of {hidden // heads}", flush=True)
    cfg = synth.config(layers=1, hidden=hidden, intermediate=64, heads=heads, kv_heads=kv_heads, vocabulary=64,
                       context=512)
    rows = (8192 + heads - 1) // heads
    lanes = 16
    c, _, m, o = build("f16", 10, cfg, exact=True, max_lanes=lanes, max_rows=rows + lanes, max_seqs=lanes,
                       max_context=256)
    check(c, m, o, [((rows + lanes - 1) // lanes,) * lanes], 256)


@pytest.mark.parametrize("hidden,intermediate,heads,plan", [
    (1024, 4096, 16, ((9,), (20,), (30, 40), (10, 33, 50, 37), (1,) * 70, (1,) * 130)),
    (4096, 256, 64, ((1,) * 20, (1,) * 130))])
def test_kquant_wide_steps(hidden, intermediate, heads, plan):
    """All matrices K-quants, prompt and decode steps of 9 to 130 rows: 64
    output tiles with a long K (down at 1,024, the head at 4,096) and a short
    one, and 256 gate and up pairs, which take one, two and three batch tiles a
    workgroup."""
    print(f"case: K-quant steps, hidden {hidden}", flush=True)
    cfg = synth.config(layers=1, hidden=hidden, intermediate=intermediate, heads=heads, kv_heads=heads // 8,
                       vocabulary=1011, context=256)
    c, t = synth.in_memory(cfg, "q4_k_m", seed=11)
    print("dtypes:", model_dtypes(t), flush=True)
    m = cohx.Model(c, t, max_lanes=130, max_rows=130, max_seqs=130, max_context=128)
    o = orc.Model(c, t, threads=8)
    check(c, m, o, plan, 128)


@pytest.mark.parametrize("hidden", [64, 72])
def test_hybrid_wide_linears(hidden):
    """514 mix tiles, 513 gate and up tile pairs at 120 rows and a head of 4,125
    tiles at 12 lanes, whole and ragged K, the regime off."""
    print(f"case: hybrid hidden {hidden}, wide mix, gate+up and head", flush=True)
    cfg = tiny(layers=2, pattern="LF", hidden=hidden, intermediate=8200, vocabulary=66000, key_heads=16,
               value_heads=16, key_dim=128, value_dim=128)
    c, t = synth35.in_memory(cfg, seed=12)
    p = Pair(c, t, max_lanes=12, max_rows=120, max_seqs=12, max_context=32)
    rng = np.random.default_rng(13)
    seqs = [p.alloc() for _ in range(12)]
    for n in (10, 1):
        p.step([(s, [int(v) for v in rng.integers(0, c["vocabulary"], n)]) for s in seqs])
    for s in seqs[::5]:
        p.check_state(s)


@pytest.mark.parametrize("value_dim", [16, 18])
def test_hybrid_wide_residuals(value_dim):
    """512 output tiles of the residual linears at 120 rows, whole and ragged K."""
    print(f"case: hybrid hidden 8192, out projection of {4 * value_dim}", flush=True)
    cfg = tiny(layers=2, pattern="LF", hidden=8192, intermediate=4 * value_dim, vocabulary=300, key_dim=16,
               value_dim=value_dim, heads=2, kv_heads=1, head_dim=2 * value_dim, rotary_dim=16)
    c, t = synth35.in_memory(cfg, seed=14)
    p = Pair(c, t, max_lanes=12, max_rows=120, max_seqs=12, max_context=32)
    rng = np.random.default_rng(15)
    seqs = [p.alloc() for _ in range(12)]
    for n in (10, 1):
        p.step([(s, [int(v) for v in rng.integers(0, c["vocabulary"], n)]) for s in seqs])
    for s in seqs[::5]:
        p.check_state(s)
