"""GPU parity of the K-quant matvec where a workgroup takes one, two and three
batch tiles: every dot bit for bit against the oracle, with a last group that
is not full."""
import numpy as np
import pytest

import synth
from test_gpu_kquant import NAMES, host_model, oracle_dots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,encode", [(12, synth.quantize_q4_k), (14, synth.quantize_q6_k)])
@pytest.mark.parametrize("rows,K,n", [(19, 768, 113), (19, 768, 130), (907, 768, 70), (907, 1536, 33),
                                      (907, 4096, 150)])
def test_kquant_many_inputs_match_oracle(dtype, encode, rows, K, n):
    """19 rows and 907 of a long K take one tile at 113 to 130 and at 33
    inputs, 907 rows two at 70 (5 tiles) and three at 150 (10 tiles)."""
    print(f"case: {NAMES[dtype]}, {rows} x {K} against {n} inputs", flush=True)
    rng = np.random.default_rng(n + dtype)
    w = encode(rng.standard_normal((rows, K)).astype(np.float32) * np.float32(0.05))
    x = rng.standard_normal((n, K)).astype(np.float32)
    out, _, st, _ = host_model().matvec(dtype, rows, K, w.reshape(-1), x)
    want, rcs = oracle_dots(list(w), dtype, K, x)
    assert not st.any() and not rcs.any()
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
