"""The exact hybrid step does not depend on the batch: chunked, token by token,
alone or beside other lanes, every logit and state word is the same.

Its f64 sums (linears, gates, delta rule, head norm) are split over lanes and
waves, in an order that the model's shape fixes.  The inputs here make any
difference visible: large terms that cancel exactly, with small ones between
them that round at the large terms' last bit, so two orders give different f32
results.  (On ordinary weights the orders agree, and these sums equal the
oracle's one chain.)"""
import numpy as np
import pytest

import gguf
import synth35
from test_gpu_qwen35 import make_q35, tiny

pytestmark = pytest.mark.gpu


def edit(t, name, fn):
    """Replaces tensor `name` by fn(its float32 values, [rows][width])."""
    o = t[name]
    v = o.data.view(np.uint16) if o.dtype == synth35.BF16 else o.data.view(np.float32)
    f = synth35.bf16_to_f32(v) if o.dtype == synth35.BF16 else v.copy()
    f = f.reshape(-1, o.shape[0]) if len(o.shape) > 1 else f
    f = fn(f).astype(np.float32)
    data = (synth35.to_bf16(f) if o.dtype == synth35.BF16 else f).view(np.uint8).reshape(-1)
    t[name] = gguf.Tensor(o.name, o.shape, o.dtype, data)


def schedules(cfg, t, lengths, decode):
    """Bits of every lane's logits after its prompt and after each decode step,
    and of its recurrent state, with all lanes in one batch and with each
    sequence alone, token by token."""
    rng = np.random.default_rng(5)
    prompts = [[int(v) for v in rng.integers(0, cfg["vocabulary"], n)] for n in lengths]
    tails = [[int(v) for v in rng.integers(0, cfg["vocabulary"], decode)] for _ in lengths]
    n = len(lengths)
    out = []
    for together in (True, False):
        m = make_q35(cfg, t, False, max_lanes=n, max_rows=max(sum(lengths), n), max_seqs=n, max_context=64)
        seqs = [m.seq_alloc() for _ in lengths]
        steps = []
        if together:
            plan = [list(prompts)] + [[[tl[k]] for tl in tails] for k in range(decode)]
            for chunk in plan:
                res = m.step([dict(seq=s, tokens=c, logits=True) for s, c in zip(seqs, chunk)])
                assert all(r["status"] == 0 for r in res)
                steps.append(np.stack([r["logits"].view(np.uint32) for r in res]))
        else:
            per = []
            for s, p, tl in zip(seqs, prompts, tails):
                logits = []
                for tok in p + tl:
                    (r,) = m.step([dict(seq=s, tokens=[tok], logits=True)])
                    assert r["status"] == 0
                    logits.append(r["logits"].view(np.uint32))
                per.append(np.stack(logits[len(p) - 1:]))
            steps = list(np.stack(per, axis=1))
        state = [m.read_state(s, layer, which).view(np.uint32)
                 for s in seqs for layer, full in enumerate(cfg["full"]) for which in ((0, 1) if full else (2, 3))]
        out.append((np.stack(steps), state))
    (la, sa), (lb, sb) = out
    bad = int((la != lb).sum())
    bad_state = sum(int((a != b).sum()) for a, b in zip(sa, sb))
    print(f"{bad} of {la.size} logits and {bad_state} state words differ between the schedules", flush=True)
    return bad + bad_state


LENGTHS = (9, 5, 12, 7, 6, 8, 11, 5, 5, 10, 9, 6, 7, 5, 8, 12)


def test_hybrid_linears_do_not_depend_on_the_batch():
    print("case: hybrid, 16 lanes in one batch against each alone; linears with cancelling inputs", flush=True)
    H = 512
    cfg = tiny(layers=2, pattern="LF", hidden=H, intermediate=480, vocabulary=2304, key_heads=4, value_heads=4,
               key_dim=64, value_dim=64, heads=4, kv_heads=2)
    cfg, t = synth35.in_memory(cfg, seed=21, tied=False)
    pairs = ((3, 300), (70, 450), (200, 500), (20, 333))

    def mirror(f):  # the inputs of a pair are equal ...
        for a, b in pairs:
            f[..., b] = f[..., a]
        return f

    def cancel(f):  # ... and their weights +-2^28
        for a, b in pairs:
            f[:, a], f[:, b] = 2.0 ** 28, -2.0 ** 28
        return f

    for name in list(t):
        if name.endswith(("embed_tokens.weight", "layernorm.weight", "language_model.norm.weight")):
            edit(t, name, mirror)
        elif name.endswith(("out_proj.weight", "o_proj.weight", "down_proj.weight")):
            edit(t, name, lambda f: mirror(f.T).T)
        elif name.endswith(("lm_head.weight", "gate_proj.weight", "up_proj.weight")) or "in_proj" in name or \
                name.endswith(("q_proj.weight", "k_proj.weight", "v_proj.weight")):
            edit(t, name, cancel)
    assert schedules(cfg, t, LENGTHS, 3) == 0


@pytest.mark.parametrize("key_dim,value_dim", [(32, 40), (64, 64), (128, 128), (128, 200)])
def test_hybrid_mixer_does_not_depend_on_the_chunking(key_dim, value_dim):
    """Chunks of five tokens and more run the mixer's separate kernels, one
    token the fused one.  Query channels a and b of a head are negated copies
    (their taps are small enough that SiLU halves them exactly) and the key
    channels equal ones, so cells a and b cancel in the head's read sum."""
    print(f"case: hybrid mixer, chunks against single tokens, {key_dim} keys x {value_dim}", flush=True)
    heads = 2
    cfg = tiny(layers=2, pattern="LF", hidden=128, vocabulary=300, key_heads=heads, value_heads=heads,
               key_dim=key_dim, value_dim=value_dim)
    cfg, t = synth35.in_memory(cfg, seed=key_dim + value_dim)
    keys = heads * key_dim
    rng = np.random.default_rng(key_dim)
    pairs = [(h * key_dim + a, h * key_dim + b) for h in range(heads)
             for a, b in rng.permutation(key_dim)[:key_dim // 4 * 2].reshape(-1, 2)]
    pa, pb = (np.array(v) for v in zip(*pairs))
    lone = np.setdiff1d(np.arange(keys), np.concatenate([pa, pb]))
    p = "model.language_model.layers.0.linear_attn"

    def rows(f):
        f[pb], f[keys + pb] = f[pa], f[keys + pa]
        return f

    def taps(f):
        f = f.reshape(-1, cfg["conv_kernel"])
        f[:keys] *= 2.0 ** -28
        f[pb], f[keys + pb] = -f[pa], f[keys + pa]
        f[lone] *= 2.0 ** -32
        return f.reshape(-1)

    edit(t, f"{p}.in_proj_qkv.weight", rows)
    edit(t, f"{p}.conv1d.weight", taps)
    edit(t, f"{p}.out_proj.weight", lambda f: f * 2.0 ** 50)
    assert schedules(cfg, t, (9, 5, 12, 7), 3) == 0
