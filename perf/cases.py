"""Workloads of the continuous-batching step, timed through its public entry
points (cohx.Model / cohx.Qwen35: seq_*, step, step_decode).

Each case is one pass over a batch of sequences of the Qwen2.5-0.5B shape (or
the Qwen3.5-0.8B hybrid shape) with random weights.  A pass of a paged (Qwen2)
case rewinds its sequences to where they stood, runs one ragged step (decode
rows and prompt chunks) that also returns the logits of the lanes that sample
from them, and then goes on greedily for `steps - 1` decode steps.  A pass of a
hybrid case works on fresh sequences or on forks, since recurrent state cannot
be rewound.  A model's weights are the same for every seed (a server loads them
once); the sequences' lengths, cached rows and tokens are the seed's.

Lengths are spread evenly over their declared range and dealt out by the seed,
so every seed of a case is the same amount of work.
"""
import math
import os
import sys
import zlib

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "coheryn-ai-studio_amd"))
import cohx  # noqa: E402
import gguf  # noqa: E402
import synth  # noqa: E402
import synth35  # noqa: E402

DEV = "cuda"
CONTEXT = 4096      # rows per paged sequence
CONTEXT35 = 1096    # rows per hybrid sequence (prompts to 1024, 64 generated)
PREFIX = 256        # tokens that a group of 16 lanes shares
STATES = 5          # states that may be alive at once
SAMPLED = 4         # lanes of a wide batch that want their logits
PIECE35 = 96        # packed rows per step when a hybrid prompt is cached


def _case(name, weights, lanes=0, kv=(0, 0), prompts=0, rows=(0, 0), past=(0, 0), steps=1, layers=24,
          shared=False):
    c = {"name": name, "weights": weights, "layers": layers, "lanes": lanes, "kv_lo": kv[0],
         "kv_hi": kv[1], "prompts": prompts, "rows_lo": rows[0], "rows_hi": rows[1],
         "past_lo": past[0], "past_hi": past[1], "shared": shared, "steps": steps}
    return c


def listed():
    return [
        # one person chatting with the model: the smallest call, step latency
        _case("q8_0 decode 1", "q8_0", 1, (700, 700), steps=8),
        # the headline metric: ragged Q8_0 decode at 32 and 128 sequences
        _case("q8_0 decode 32", "q8_0", 32, (64, 2048), steps=8),
        _case("q8_0 decode 128", "q8_0", 128, (64, 2048), steps=8),
        # four F16 requests from their prompts on (prompt rows below the wide regime)
        _case("f16 four requests", "f16", prompts=4, rows=(9, 37), steps=8),
        # a busy F16 server between prompts
        _case("f16 decode 56", "f16", 56, (256, 4080), steps=4),
        # agents behind common system prompts: 8 groups of 16 lanes share 256 tokens
        _case("q4_0 shared decode 128", "q4_0", 128, (PREFIX, 3500), steps=4, shared=True),
        # the publisher's mixed file (Q5_0, Q8_0, Q4_K, Q6_K matrices), served
        _case("q4_k_m decode 32", "q4_k_m", 32, (64, 2048), steps=8),
        # and a document given to it
        _case("q4_k_m prompt", "q4_k_m", prompts=1, rows=(387, 387)),
        # continuous batching: eight prompt chunks beside 56 decoding lanes
        _case("f16 mixed", "f16", 56, (256, 4080), prompts=8, rows=(128, 512), past=(0, 1024)),
        # the same on Q8_0, two layers deep: the operands' int8 rounding turns a
        # last-bit difference into whole steps, and more layers into noise
        _case("q8_0 mixed", "q8_0", 56, (256, 4080), prompts=8, rows=(128, 512), past=(0, 1024), layers=2),
        # the hybrid model: sixteen cached conversations go on, sixteen prompts come in
        _case("qwen3.5 decode 16", "bf16", 16, (32, 448), steps=4),
        _case("qwen3.5 prompts", "bf16", prompts=16, rows=(64, 449)),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "mixed", "hybrid decode", "hybrid prompts"])
    if kind == "decode":
        w = rng.choice(["q8_0", "q8_0", "q4_0", "f16", "q4_k_m"])
        lo = rng.randint(1, 600)
        hi = lo + _log(rng, 1, 3300)
        shared = w != "f16" and rng.random() < 0.25
        lanes = _log(rng, 1, 56 if w == "f16" else 128)
        c = _case("", w, lanes, (lo + PREFIX if shared else lo, hi + PREFIX if shared else hi),
                  steps=rng.randint(1, 4), shared=shared)
    elif kind == "prompt":
        w = rng.choice(["q8_0", "q4_0", "f16", "q4_k_m"])
        n, hi = rng.randint(1, 4), _log(rng, 4, 96 if w == "q4_k_m" else 500)
        lo = rng.randint(max(1, hi // 3), hi)
        past = rng.choice([0, rng.randint(1, 900)])
        c = _case("", w, prompts=n, rows=(lo, hi), past=(past, past + 64 if past else 0), steps=rng.randint(1, 2))
    elif kind == "mixed":
        w = rng.choice(["q8_0", "q4_0", "f16"])
        lo = rng.randint(40, 200)
        c = _case("", w, _log(rng, 1, 56), (rng.randint(2, 300), rng.randint(400, 4000)),
                  prompts=rng.randint(1, 8), rows=(lo, lo + rng.randint(1, 300)), past=(0, rng.randint(1, 1500)))
    elif kind == "hybrid decode":
        lo = rng.randint(2, 60)
        c = _case("", "bf16", _log(rng, 1, 16), (lo, lo + rng.randint(1, 380)), steps=rng.randint(1, 4))
    else:
        hi = _log(rng, 5, 440)
        c = _case("", "bf16", prompts=_log(rng, 1, 16), rows=(rng.randint(1, hi), hi))
    if not _exact_bits(c):
        c["steps"] = 1
        if c["weights"] in ("q8_0", "q4_0"):
            c["layers"] = 2
    del c["name"]
    return c


# ---- sizes ------------------------------------------------------------------


def _spread(lo, hi, n):
    return [int(lo + (hi - lo) * (i + 0.5) / n) if n else lo for i in range(n)]


def _lengths(case):
    """(cached rows of the decode lanes, rows of the prompts, rows before them)"""
    return (_spread(case["kv_lo"], case["kv_hi"] + 1, case["lanes"]),
            _spread(case["rows_lo"], case["rows_hi"] + 1, case["prompts"]),
            _spread(case["past_lo"], case["past_hi"] + 1, case["prompts"]))


def _rows(case):
    return case["lanes"] + sum(_lengths(case)[1])


def _exact_bits(case):
    """Steps that the framework computes in the reference's own order, bit for
    bit: everything but wide steps with prompt rows."""
    return case["weights"] == "q4_k_m" or not case["prompts"] or _rows(case) < 128


def _sampled(case):
    """Lanes of the first step whose logits are wanted: prompts first."""
    n = case["prompts"] + case["lanes"]
    return list(range(n)) if n <= 4 else sorted(set(_spread(0, max(case["prompts"], 1), SAMPLED) if case["prompts"]
                                                    else _spread(0, n, SAMPLED)) | ({n - 1} if case["lanes"] else set()))


def _config(case):
    return synth.config(layers=case["layers"])


def work(case):
    kv, rows, past = _lengths(case)
    steps, R = case["steps"], _rows(case)
    lanes = case["lanes"] + case["prompts"]
    first = [k + 1 for k in kv] + [p + r for p, r in zip(past, rows)]  # rows a lane attends to in the first step
    pairs = sum(k + 1 for k in kv) + sum(r * p + r * (r + 1) // 2 for p, r in zip(past, rows))
    if case["weights"] == "bf16":
        c = synth35.config()
        H, F, V, D = c["hidden"], c["intermediate"], c["vocabulary"], c["head_dim"]
        keys, vals = c["key_heads"] * c["key_dim"], c["value_heads"] * c["value_dim"]
        full, lin = sum(c["full"]), c["layers"] - sum(c["full"])
        kvw, qw = c["kv_heads"] * D, c["heads"] * D
        lin_w = H * (2 * keys + 2 * vals + 2 * c["value_heads"]) + vals * H
        full_w = H * (2 * qw + 2 * kvw) + qw * H
        weights = lin * lin_w + full * full_w + c["layers"] * 3 * H * F
        state = 4 * lin * ((2 * keys + vals) * c["conv_kernel"] + vals * c["key_dim"])
        cells = vals * c["key_dim"]
        b = steps * 2.0 * (weights + V * H) + steps * lanes * 2 * state
        f = 2.0 * weights * (R + (steps - 1) * lanes) + 2.0 * V * H * lanes * steps
        f += lin * 6.0 * cells * (R + (steps - 1) * lanes) + full * 4.0 * qw * pairs
        for i in range(steps):
            b += full * 8.0 * kvw * sum(n + i for n in first) + full * 8.0 * kvw * (R if i == 0 else lanes)
            f += full * 4.0 * qw * sum(n + i for n in first) * (i > 0)
        return {"bytes": b + 4.0 * V * len(_sampled(case)), "flops": f}
    c = _config(case)
    L, H, F, V = c["layers"], c["hidden"], c["intermediate"], c["vocabulary"]
    kvd = c["kv_heads"] * c["head_dim"]
    block = sum(n * k for n, k in ((H + 2 * kvd, H), (H, H), (2 * F, H), (H, F))) * L
    w_bytes = sum(_tensor_bytes(case, c, n, r, k) for n, r, k in _matrices(c, case["weights"] == "q4_k_m"))
    per_row = L * kvd * 8.0
    once = 0
    if case["shared"]:  # a group's prefix is read once for its lanes
        groups = (case["lanes"] + 15) // 16
        once = (case["lanes"] - groups) * PREFIX
    b = f = 0.0
    for i in range(steps):
        b += w_bytes + per_row * (sum(n + i for n in first) - once + (R if i == 0 else lanes))
        f += 2.0 * block * (R if i == 0 else lanes) + 2.0 * V * H * lanes
        f += L * 4.0 * H * (pairs if i == 0 else sum(n + i for n in first))
    return {"bytes": b + 4.0 * V * len(_sampled(case)), "flops": f}


def tolerance(case):
    # Exact steps follow the reference's order of operations and are the same
    # bits whatever the kernel.  The wide prompt regime sums binary16 (bfloat16)
    # products in f32; between it and the exact kernels the logits of these
    # cases differ by 1.2e-3 to 3.0e-3 on F16 (max 1.5e-2 of their rms), by
    # 6e-5 to 9e-5 (max 4e-4) on the hybrid model, and by 1.6e-2 to 2.1e-2
    # (max 1.1e-1) on two layers of Q8_0 or Q4_0 (1.1e-2 to 1.5e-2 on one
    # layer, 2.4e-2 to 2.9e-2 on four), whose inputs are rounded to int8 again
    # before every linear.
    if _exact_bits(case):
        return "exact"
    if case["weights"] == "bf16":
        return {"rel": 3.5e-4, "max": 2e-3}
    if case["weights"] == "f16":
        return {"rel": 1.2e-2, "max": 6e-2}
    return {"rel": 3e-2, "max": 2e-1}


# ---- random weights, made on the GPU ------------------------------------------


def _gen(*key):
    g = torch.Generator(device=DEV)
    g.manual_seed(zlib.crc32(repr(key).encode()))
    return g


def _normal(key, *shape):
    return torch.randn(*shape, generator=_gen("weights", *key), device=DEV, dtype=torch.float32)


def _f16_bytes(x):
    return x.to(torch.float16).contiguous().view(torch.uint8)


def _q_blocks(x, levels, signed_max):
    """32-value blocks of x, their scale in binary16 and the signed value that sets it."""
    b = x.reshape(x.shape[0], -1, 32)
    at = b.abs().argmax(-1, keepdim=True)
    m = b.gather(-1, at)
    d = (m.abs() if not signed_max else -m) / levels
    return b, torch.where(d == 0, 0.0, 1.0 / d), d.to(torch.float16)


def _q8_0(x):
    b, inv, d = _q_blocks(x, 127.0, False)
    q = torch.round(b * inv).clamp(-127, 127)
    pay = torch.cat([_f16_bytes(d), q.to(torch.int8).view(torch.uint8)], -1)
    return pay.reshape(-1), (q.double() * d.double()).reshape(x.shape)


def _q4_0(x):
    b, inv, d = _q_blocks(x, 8.0, True)
    q = torch.floor(b * inv + 8.5).clamp(0, 15).to(torch.uint8)
    pay = torch.cat([_f16_bytes(d), q[..., :16] | (q[..., 16:] << 4)], -1)
    return pay.reshape(-1), ((q.double() - 8) * d.double()).reshape(x.shape)


def _q5_0(x):
    b, inv, d = _q_blocks(x, 16.0, True)
    q = torch.floor(b * inv + 16.5).clamp(0, 31).to(torch.int32)
    bits = ((q >> 4).reshape(*q.shape[:-1], 4, 8) << torch.arange(8, device=DEV, dtype=torch.int32)).sum(-1)
    nib = (q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)
    pay = torch.cat([_f16_bytes(d), bits.to(torch.uint8), nib.to(torch.uint8)], -1)
    return pay.reshape(-1), ((q.double() - 16) * d.double()).reshape(x.shape)


def _q4_k(x):
    g = x.reshape(x.shape[0], -1, 8, 32)
    lo = g.amin(-1).clamp(max=0.0)
    scale = (g.amax(-1) - lo) / 15.0
    d = (scale.amax(-1, keepdim=True) / 63.0).to(torch.float16)
    dm = ((-lo).amax(-1, keepdim=True) / 63.0).to(torch.float16)
    sc = torch.round(scale / d.float()).clamp(0, 63).to(torch.int32)
    mn = torch.round(-lo / dm.float()).clamp(0, 63).to(torch.int32)
    step = (d.float() * sc).unsqueeze(-1)
    q = torch.where(step > 0, torch.round((g + (dm.float() * mn).unsqueeze(-1)) / step), 0.0).clamp(0, 15)
    n = q.to(torch.int32)
    head = torch.cat([(sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6), (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6),
                      (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1).to(torch.uint8)
    nib = (n[..., 0::2, :] | (n[..., 1::2, :] << 4)).to(torch.uint8)
    pay = torch.cat([_f16_bytes(d), _f16_bytes(dm), head, nib.flatten(-2)], -1)
    val = d.double().unsqueeze(-1) * sc.double().unsqueeze(-1) * q.double() - dm.double().unsqueeze(-1) * mn.double().unsqueeze(-1)
    return pay.reshape(-1), val.reshape(x.shape)


def _q6_k(x):
    g = x.reshape(x.shape[0], -1, 16, 16)
    scale = g.abs().amax(-1) / 31.0
    d = (scale.amax(-1, keepdim=True) / 127.0).to(torch.float16)
    sc = torch.round(scale / d.float()).clamp(-128, 127)
    step = (d.float() * sc).unsqueeze(-1)
    q = torch.where(step > 0, torch.round(g / step), 0.0).clamp(-32, 31)
    v = (q.to(torch.int32) + 32).reshape(*g.shape[:2], 2, 4, 32)  # [half][group of 32][value]
    low = torch.stack([(v[..., 0, :] & 15) | ((v[..., 2, :] & 15) << 4),
                       (v[..., 1, :] & 15) | ((v[..., 3, :] & 15) << 4)], -2)
    high = sum((v[..., k, :] >> 4) << (2 * k) for k in range(4))
    pay = torch.cat([low.flatten(-3).to(torch.uint8), high.flatten(-2).to(torch.uint8),
                     sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], -1)
    return pay.reshape(-1), (d.double().unsqueeze(-1) * sc.double().unsqueeze(-1) * q.double()).reshape(x.shape)


def _f16(x):
    h = x.to(torch.float16)
    return _f16_bytes(h).reshape(-1), h.double()


FORMATS = {1: _f16, 2: _q4_0, 6: _q5_0, 8: _q8_0, 12: _q4_k, 14: _q6_k}
ROW_BYTES = {1: lambda k: 2 * k, 2: lambda k: k // 32 * 18, 6: lambda k: k // 32 * 22, 8: lambda k: k // 32 * 34,
             12: lambda k: k // 256 * 144, 14: lambda k: k // 256 * 210}


def _dtype(case, c, name, width):
    if case["weights"] != "q4_k_m":
        return synth.DTYPES[case["weights"]]
    layer = int(name.split(".")[1]) if name.startswith("blk.") else None
    return synth.q4_k_m_dtype(name.split(".", 2)[2] if layer is not None else name, width, layer, c["layers"])


def _matrices(c, untied):
    """(name, rows, width) of every matrix that a step reads."""
    H, F, V, kvd = c["hidden"], c["intermediate"], c["vocabulary"], c["kv_heads"] * c["head_dim"]
    out = [("output.weight" if untied else "token_embd.weight", V, H)]
    for i in range(c["layers"]):
        p = f"blk.{i}."
        out += [(p + "attn_q.weight", H, H), (p + "attn_k.weight", kvd, H), (p + "attn_v.weight", kvd, H),
                (p + "attn_output.weight", H, H), (p + "ffn_gate.weight", F, H), (p + "ffn_up.weight", F, H),
                (p + "ffn_down.weight", H, F)]
    return out


def _tensor_bytes(case, c, name, rows, width):
    return rows * ROW_BYTES[_dtype(case, c, name, width)](width)


def _matrix(case, c, name, rows, width):
    """(GGUF payload, values in 64 bits) of one random matrix, on the GPU."""
    return FORMATS[_dtype(case, c, name, width)](0.02 * _normal((name, case["weights"]), rows, width))


def _vector(c, name, n):
    v = _normal((name,), n)
    return 1.0 + 0.1 * v if "norm" in name else 0.02 * v


def _weights35(name, kind, shape, vocab):
    """One hybrid tensor as float32 on the GPU (matrices already rounded to bfloat16)."""
    n = int(np.prod(shape))
    v = _normal((name, "hybrid"), n)
    if kind == synth35.BF16:
        return (0.02 * v).to(torch.bfloat16).float().reshape(shape[1], shape[0])
    if name.endswith("A_log"):
        return torch.log(1.0 + 15.0 * torch.special.ndtr(v))
    if name.endswith("dt_bias"):
        return 1.0 + 0.1 * v
    if name.endswith("conv1d.weight"):
        return 0.25 * v
    return (1.0 if name.endswith("linear_attn.norm.weight") else 0.0) + 0.02 * v


_models = {}


def _model(case):
    key = (case["weights"], case["layers"])
    if key in _models:
        return _models[key]
    if case["weights"] == "bf16":
        c = dict(synth35.config(), tied=True)
        tensors = {}
        for name, kind, shape, _ in synth35._plan(c, True):
            v = _weights35(name, kind, shape, c["vocabulary"])
            raw = v.to(torch.bfloat16) if kind == synth35.BF16 else v
            tensors[name] = gguf.Tensor(name, shape, kind, raw.contiguous().view(torch.uint8).reshape(-1).cpu().numpy())
        m = cohx.Qwen35(c, tensors, max_lanes=16, max_rows=16 * 449, max_seqs=16 * (STATES + 1), max_context=CONTEXT35)
    else:
        c, untied = _config(case), case["weights"] == "q4_k_m"
        c["eos_token_id"] = c["vocabulary"] - 1
        H, V, kvd = c["hidden"], c["vocabulary"], c["kv_heads"] * c["head_dim"]
        tensors = {}
        mats = _matrices(c, untied) + ([("token_embd.weight", V, H)] if untied else [])
        for name, rows, width in mats:
            pay = _matrix(case, c, name, rows, width)[0].cpu().numpy()
            tensors[name] = gguf.Tensor(name, (width, rows), _dtype(case, c, name, width), pay)
        vecs = [("output_norm.weight", H)]
        for i in range(c["layers"]):
            p = f"blk.{i}."
            vecs += [(p + "attn_norm.weight", H), (p + "ffn_norm.weight", H), (p + "attn_q.bias", H),
                     (p + "attn_k.bias", kvd), (p + "attn_v.bias", kvd)]
        for name, n in vecs:
            tensors[name] = gguf.Tensor(name, (n,), 0, _vector(c, name, n).view(torch.uint8).cpu().numpy())
        m = cohx.Model(c, tensors, max_lanes=128, max_rows=64 + 8 * 512, max_seqs=136 * STATES, max_context=CONTEXT,
                       kv_pages=STATES * 128 * 1800 // 16)
    _models[key] = m
    return m


# ---- a pass -------------------------------------------------------------------


def _draws(case, seed):
    """The seed's deal of the lengths, and its tokens."""
    rng = np.random.default_rng(seed)
    kv, rows, past = _lengths(case)
    rng.shuffle(kv)
    rng.shuffle(rows)
    rng.shuffle(past)
    V = synth35.QWEN35_08B["vocabulary"] if case["weights"] == "bf16" else synth.QWEN25_05B["vocabulary"]
    prompts = [rng.integers(0, V, n).astype(np.uint32) for n in rows]
    tokens = rng.integers(0, V, case["lanes"]).astype(np.uint32)
    cached = [rng.integers(0, V, n).astype(np.uint32) for n in kv] if case["weights"] == "bf16" else None
    return kv, past, prompts, tokens, cached


class State:
    """A batch's sequences in the model's pool; given back when it is dropped."""

    def __init__(self, case, model):
        self.case, self.model, self.seqs, self.start = case, model, [], []

    def __del__(self):
        if getattr(self.model, "h", None):
            for s in self.seqs:
                self.model.seq_free(s)


def prepare(case, seed):
    m = _model(case)
    st = State(case, m)
    kv, past, prompts, tokens, cached = _draws(case, seed)
    sampled = set(_sampled(case))
    if case["weights"] == "bf16":
        if case["prompts"]:
            st.lanes = [dict(tokens=p, logits=i in sampled) for i, p in enumerate(prompts)]
            return st
        st.seqs = [m.seq_alloc() for _ in kv]
        done = [0] * len(kv)
        per = PIECE35 // len(kv)
        while any(d < n for d, n in zip(done, kv)):
            go = [i for i in range(len(kv)) if done[i] < kv[i]]
            m.step([dict(seq=st.seqs[i], tokens=cached[i][done[i]:done[i] + per], skip_head=True) for i in go])
            for i in go:
                done[i] = min(kv[i], done[i] + per)
        st.start = list(kv)
        st.lanes = [dict(tokens=tokens[i:i + 1], logits=i in sampled) for i in range(len(kv))]
        return st
    for i, n in enumerate(past):
        s = m.seq_alloc()
        st.seqs.append(s)
        st.start.append(n)
        if n:
            m.seq_fill_synthetic(s, n, seed, 10000 + i)
    base = None
    for i, n in enumerate(kv):
        if case["shared"]:
            if i % 16 == 0:
                base = m.seq_alloc()
                m.seq_fill_synthetic(base, PREFIX, seed, 20000 + i // 16)
            s = m.seq_fork(base, PREFIX)
            if i % 16 == 15 or i + 1 == len(kv):
                m.seq_free(base)
        else:
            s = m.seq_alloc()
        st.seqs.append(s)
        st.start.append(n)
        m.seq_fill_synthetic(s, n, seed, i)
    toks = prompts + [tokens[i:i + 1] for i in range(len(kv))]
    st.lanes = [dict(seq=s, tokens=t, logits=i in sampled) for i, (s, t) in enumerate(zip(st.seqs, toks))]
    st.ids = np.asarray(st.seqs, np.uint32)
    return st


def run(st):
    m, case = st.model, st.case
    if case["weights"] == "bf16":
        if st.seqs:
            seqs = [m.seq_fork(s, n) for s, n in zip(st.seqs, st.start)]
        else:
            seqs = [m.seq_alloc() for _ in st.lanes]
        ids = np.asarray(seqs, np.uint32)
        lanes = [dict(ln, seq=s) for ln, s in zip(st.lanes, seqs)]
    else:
        for s, n in zip(st.seqs, st.start):
            m.seq_truncate(s, n)
        ids, lanes = st.ids, st.lanes
    res = m.step(lanes)
    if any(r["status"] for r in res):
        raise RuntimeError("a lane failed")
    logits = [r["logits"] for r in res if r["logits"] is not None]
    tokens = [np.asarray([r["argmax"] for r in res], np.int64)]
    for _ in range(case["steps"] - 1):
        status, tok = m.step_decode(ids, tokens[-1])
        if status.any():
            raise RuntimeError("a lane failed")
        tokens.append(tok.astype(np.int64))
    if case["weights"] == "bf16":
        for s in seqs:
            m.seq_free(s)
    # a wide prompt step is held to a tolerance: its logits say all, and a tie
    # in them may fall either way
    return {"logits": logits, "tokens": tokens} if _exact_bits(case) else {"logits": logits}


# ---- the same in 64 bits ---------------------------------------------------------


def _signed(v):
    return v - (1 << 64) if v >= 1 << 63 else v


def _shr(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _mix64(z):
    z = z + _signed(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _cached_rows(seed, stream, layer, which, first, end, width):
    """Rows [first, end) that cohx_seq_fill_synthetic writes."""
    at = torch.tensor([(stream << 32) | (layer << 1) | which], device=DEV, dtype=torch.int64)
    pos = torch.arange(first, end, device=DEV, dtype=torch.int64)[:, None]
    e = torch.arange(width, device=DEV, dtype=torch.int64)[None, :]
    h = _mix64((_mix64(at) ^ _signed(seed)) ^ ((pos << 16) | e))
    return (_shr(h, 40) - (1 << 23)).double() * 2.0 ** -23


def _operand(x, dtype):
    """A linear's input as its format defines it: rounded to binary16 for F16,
    Q8_0 blocks of 32 (scale in binary16) or Q8_K blocks of 256 for the others."""
    if dtype == 1:
        return x.to(torch.float16).double()
    if dtype in (12, 14):
        b = x.reshape(x.shape[0], -1, 256)
        d = -b.gather(-1, b.abs().argmax(-1, keepdim=True)) / 127.0
        return (torch.round(b / torch.where(d == 0, 1.0, d)).clamp(max=127) * d).reshape(x.shape)
    b = x.reshape(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    q = torch.round(b / torch.where(d == 0, 1.0, d))
    return (q * d.to(torch.float16).double()).reshape(x.shape)


def _rope(x, pos, base, n):
    """NeoX rotation of the first n elements of x [rows, heads, D]."""
    half = n // 2
    ang = pos.double()[:, None] * base ** (-2.0 * torch.arange(half, device=DEV, dtype=torch.float64) / n)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :half], x[..., half:n]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., n:]], -1)


def _attend(q, k, v, start):
    """Causal softmax(q k / sqrt(D)) v: q [T, NH, D] at positions start.., k and v [N, NKV, D]."""
    T, NH, D = q.shape
    rep = NH // k.shape[1]
    k, v = k.repeat_interleave(rep, 1).permute(1, 2, 0).contiguous(), v.repeat_interleave(rep, 1).permute(1, 0, 2).contiguous()
    s = torch.matmul(q.permute(1, 0, 2).contiguous(), k) / math.sqrt(D)
    late = torch.arange(k.shape[2], device=DEV)[None, :] > start + torch.arange(T, device=DEV)[:, None]
    p = torch.softmax(s.masked_fill(late, -math.inf), -1)
    return torch.matmul(p, v).permute(1, 0, 2).reshape(T, NH * D)


def _exact_paged(case, seed):
    c = _config(case)
    H, F, V, L = c["hidden"], c["intermediate"], c["vocabulary"], c["layers"]
    NH, NKV, D = c["heads"], c["kv_heads"], c["head_dim"]
    kvd = NKV * D
    kv, past, prompts, tokens, _ = _draws(case, seed)
    n_pr = len(prompts)
    lanes = []  # (tokens, start, [(stream, first, end)])
    for i in _sampled(case):
        if i < n_pr:
            lanes.append((prompts[i], past[i], [(10000 + i, 0, past[i])]))
        else:
            j = i - n_pr
            spans = [(20000 + j // 16, 0, PREFIX), (j, PREFIX, kv[j])] if case["shared"] else [(j, 0, kv[j])]
            lanes.append((tokens[j:j + 1], kv[j], spans))
    ids = torch.from_numpy(np.concatenate([t for t, _, _ in lanes]).astype(np.int64)).to(DEV)
    pos = torch.cat([torch.arange(s, s + len(t), device=DEV) for t, s, _ in lanes])
    cut = np.cumsum([0] + [len(t) for t, _, _ in lanes])

    def norm(x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + c["norm_epsilon"]) * _vector(c, name, H).double()

    def mat(name, rows, width):
        return _matrix(case, c, name, rows, width)[1], _dtype(case, c, name, width)

    def linear(x, w):
        return _operand(x, w[1]) @ w[0].t()

    x = mat("token_embd.weight", V, H)[0][ids].clone()
    for i in range(L):
        p = f"blk.{i}."
        h = norm(x, p + "attn_norm.weight")
        q, k, v = (linear(h, mat(p + f"attn_{n}.weight", r, H)) + _vector(c, p + f"attn_{n}.bias", r).double()
                   for n, r in (("q", H), ("k", kvd), ("v", kvd)))
        q = _rope(q.reshape(-1, NH, D), pos, c["rope_base"], D)
        k = _rope(k.reshape(-1, NKV, D), pos, c["rope_base"], D)
        v = v.reshape(-1, NKV, D)
        outs = []
        for n, (_, start, spans) in enumerate(lanes):
            a, b = cut[n], cut[n + 1]
            old = [torch.cat([_cached_rows(seed, s, i, w, f, e, kvd) for s, f, e in spans]).reshape(-1, NKV, D)
                   for w in (0, 1)]
            outs.append(_attend(q[a:b], torch.cat([old[0], k[a:b]]), torch.cat([old[1], v[a:b]]), start))
        x = x + linear(torch.cat(outs), mat(p + "attn_output.weight", H, H))
        h = norm(x, p + "ffn_norm.weight")
        g, u = linear(h, mat(p + "ffn_gate.weight", F, H)), linear(h, mat(p + "ffn_up.weight", F, H))
        x = x + linear(torch.nn.functional.silu(g) * u, mat(p + "ffn_down.weight", H, F))
    last = norm(x[torch.as_tensor(cut[1:] - 1, device=DEV)], "output_norm.weight")
    head = mat("output.weight" if case["weights"] == "q4_k_m" else "token_embd.weight", V, H)
    return linear(last, head)


def _exact_hybrid(case, seed):
    c = synth35.config()
    _, _, prompts, tokens, cached = _draws(case, seed)
    seqs = prompts if case["prompts"] else [np.append(a, t) for a, t in zip(cached, tokens)]
    seqs = [seqs[i] for i in _sampled(case)]
    plan = {n: (kind, shape) for n, kind, shape, _ in synth35._plan(c, True)}
    n = [len(s) for s in seqs]
    B, T = len(seqs), max(n)
    ids = torch.zeros(B, T, dtype=torch.int64)  # lanes padded at their end: nothing there reaches a lane's last row
    for i, s in enumerate(seqs):
        ids[i, :n[i]] = torch.from_numpy(s.astype(np.int64))
    eps, D, NH, NKV = c["epsilon"], c["head_dim"], c["heads"], c["kv_heads"]
    KH, VH, KD, VD, K = c["key_heads"], c["value_heads"], c["key_dim"], c["value_dim"], c["conv_kernel"]
    keys, rep = KH * KD, VH // KH
    pos = torch.arange(T, device=DEV)

    def w(name):
        return _weights35(name, *plan[name], c["vocabulary"]).double()

    def rms(x, weight):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight

    silu = torch.nn.functional.silu
    x = w("model.language_model.embed_tokens.weight")[ids.to(DEV)]
    for i, full in enumerate(c["full"]):
        p = f"model.language_model.layers.{i}."
        h = rms(x, 1.0 + w(p + "input_layernorm.weight"))
        if full:
            a = p + "self_attn."
            qg = (h @ w(a + "q_proj.weight").t()).reshape(B, T, NH, 2 * D)
            k = (h @ w(a + "k_proj.weight").t()).reshape(B, T, NKV, D)
            v = (h @ w(a + "v_proj.weight").t()).reshape(B, T, NKV, D)
            q, gate = rms(qg[..., :D], 1.0 + w(a + "q_norm.weight")), qg[..., D:].reshape(B, T, NH * D)
            k = rms(k, 1.0 + w(a + "k_norm.weight"))
            o = torch.stack([_attend(_rope(q[b], pos, c["rope_base"], c["rotary_dim"]),
                                     _rope(k[b], pos, c["rope_base"], c["rotary_dim"]), v[b], 0) for b in range(B)])
            x = x + (o * torch.sigmoid(gate)) @ w(a + "o_proj.weight").t()
        else:
            a = p + "linear_attn."
            mix = (h @ w(a + "in_proj_qkv.weight").t()).transpose(1, 2)
            taps = w(a + "conv1d.weight").reshape(-1, K)
            pad = torch.nn.functional.pad(mix, (K - 1, 0))
            conv = silu(sum(pad[..., j:j + T] * taps[None, :, j:j + 1] for j in range(K))).transpose(1, 2)
            q = conv[..., :keys].reshape(B, T, KH, KD).repeat_interleave(rep, 2)
            k = conv[..., keys:2 * keys].reshape(B, T, KH, KD).repeat_interleave(rep, 2)
            v = conv[..., 2 * keys:].reshape(B, T, VH, VD)
            q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) / math.sqrt(KD)
            k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            dt = torch.nn.functional.softplus(h @ w(a + "in_proj_a.weight").t() + w(a + "dt_bias"), threshold=1e9)
            decay = torch.exp(-torch.exp(w(a + "A_log")) * dt)[..., None, None]
            beta = torch.sigmoid(h @ w(a + "in_proj_b.weight").t())[..., None]
            S = torch.zeros(B, VH, KD, VD, device=DEV, dtype=torch.float64)
            o = torch.empty(B, T, VH, VD, device=DEV, dtype=torch.float64)
            for t in range(T):
                S *= decay[:, t]
                corr = beta[:, t] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
                S += k[:, t, :, :, None] * corr[:, :, None, :]
                o[:, t] = (S * q[:, t, :, :, None]).sum(2)
            z = (h @ w(a + "in_proj_z.weight").t()).reshape(B, T, VH, VD)
            o = rms(o, w(a + "norm.weight")) * silu(z)
            x = x + o.reshape(B, T, VH * VD) @ w(a + "out_proj.weight").t()
        h = rms(x, 1.0 + w(p + "post_attention_layernorm.weight"))
        x = x + (silu(h @ w(p + "mlp.gate_proj.weight").t()) * (h @ w(p + "mlp.up_proj.weight").t())) @ \
            w(p + "mlp.down_proj.weight").t()
    last = x[torch.arange(B, device=DEV), torch.as_tensor(n, device=DEV) - 1]
    last = rms(last, 1.0 + w("model.language_model.norm.weight"))
    return last @ w("model.language_model.embed_tokens.weight").t()


def exact(case, seed):
    """The first step's logits in 64 bits, with the formats' own rounding of the
    linears' inputs (it is part of what they compute).  The greedy tokens follow
    from every step before them and have no value of their own."""
    logits = (_exact_hybrid if case["weights"] == "bf16" else _exact_paged)(case, seed).cpu().numpy()
    out = {"logits": list(logits)}
    if _exact_bits(case):
        out["tokens"] = None
    return out
