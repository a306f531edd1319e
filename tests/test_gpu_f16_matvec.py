"""GPU parity of the exact F16 kernels at the edges of their tiles: one matrix
against a few and many rows, and whole steps whose qkv, gate+up and head tiles
end ragged.

Every product of two binary16 values is a multiple of 2^-48, so a dot whose
partial sums stay below 2^5 is exact in f64 in any order: the expected bits are
those of the sequential f64 sum, with no tolerance."""
import numpy as np
import pytest

import cohx
import orc
import synth
from test_gpu_kquant import host_model
from test_gpu_step import build

pytestmark = pytest.mark.gpu

F16 = 1


@pytest.mark.parametrize("rows,K", [(1, 32), (15, 96), (17, 160), (40, 72), (130, 896), (64, 4864)])
def test_f16_matvec_edges(rows, K):
    m = host_model()
    rng = np.random.default_rng(rows * K)
    w = (rng.standard_normal((rows, K)) * 0.02).astype(np.float16)
    w[0, ::3] = 0
    for n in (1, 4, 5, 11, 16, 17, 31, 64, 70):
        print(f"case: f16 matvec {rows} x {K}, {n} inputs", flush=True)
        x = rng.standard_normal((n, K)).astype(np.float32)
        x[0] *= np.float32(2.0 ** -18)  # subnormal binary16 operands
        out, _, st, _ = m.matvec(F16, rows, K, w.view(np.uint8), x)
        assert not st.any()
        p = w.astype(np.float32)[None] * x.astype(np.float16).astype(np.float32)[:, None]
        sums = np.cumsum(p.astype(np.float64), axis=-1)
        assert np.abs(sums).max() < 32
        assert np.array_equal(out.view(np.uint32), sums[..., -1].astype(np.float32).view(np.uint32)), n


@pytest.mark.parametrize("K", [32, 96, 128, 160])
def test_f16_matvec_keeps_the_sign_of_zero(K):
    """A dot of -0 terms alone is -0, also where K is not whole chunks."""
    m = host_model()
    w = np.zeros((9, K), np.float16)
    w[1] = -0.0
    for n in (4, 16, 20):
        print(f"case: f16 zero rows of {K}, {n} inputs", flush=True)
        x = -np.arange(1, n * K + 1, dtype=np.float32).reshape(n, K) / (n * K)
        out, _, st, _ = m.matvec(F16, 9, K, w.view(np.uint8), x)
        assert not st.any()
        want = np.full((n, 9), 0x80000000, np.uint32)  # +0 weights: -0 products
        want[:, 1] = 0
        assert np.array_equal(out.view(np.uint32), want), n


@pytest.mark.parametrize("hidden,heads,kv_heads,vocabulary", [(128, 4, 2, 300), (128, 2, 1, 259), (256, 2, 2, 65)])
@pytest.mark.parametrize("lengths", [(1,), (2, 1, 1), (4, 3, 9), (5, 12, 20), (40, 33, 7)])
def test_f16_steps_match_oracle(hidden, heads, kv_heads, vocabulary, lengths):
    print(f"case: f16 steps {hidden}/{heads}/{kv_heads} {lengths}", flush=True)
    cfg = synth.config(layers=2, hidden=hidden, intermediate=224, heads=heads, kv_heads=kv_heads,
                       vocabulary=vocabulary, context=256)
    c, _, m, o = build("f16", 5, cfg, max_rows=96)
    rng = np.random.default_rng(len(lengths))
    seqs, sess = [m.seq_alloc() for _ in lengths], [o.session(128) for _ in lengths]
    for plan in (lengths, (1,) * len(lengths)):
        toks = [[int(v) for v in rng.integers(0, vocabulary, n)] for n in plan]
        res = m.step([dict(seq=s, tokens=t, logits=True) for s, t in zip(seqs, toks)])
        for i, r in enumerate(res):
            assert r["status"] == 0
            for t in toks[i]:
                assert o.forward_batch([sess[i]], [t])[0] == 0
            assert np.array_equal(r["logits"].view(np.uint32), sess[i].logits().view(np.uint32)), (plan, i)
            assert r["argmax"] == orc.Sampler().sample(sess[i].logits())[1]
    for i, s in enumerate(seqs):
        for layer in range(c["layers"]):
            for values in (False, True):
                assert np.array_equal(m.seq_read_kv(s, layer, values), sess[i].kv(layer, values)), (i, layer)


def test_f16_matvec_reports_non_finite_inputs():
    m = host_model()
    w = np.ones((20, 64), np.float16)
    x = np.ones((3, 64), np.float32)
    x[1, 7] = 1e6  # past binary16
    out, _, st, _ = m.matvec(F16, 20, 64, w.view(np.uint8), x)
    assert list(st) == [cohx.OK, cohx.INVALID_GGUF, cohx.OK] and np.all(out[[0, 2]] == 64)
