"""GPU parity of the K-quant matvec where a workgroup takes several batch
tiles (eight or more of them): every dot bit for bit against the oracle, with
a last group that is not full."""
import numpy as np
import pytest

import synth
from test_gpu_kquant import NAMES, host_model, oracle_dots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,encode", [(12, synth.quantize_q4_k), (14, synth.quantize_q6_k)])
@pytest.mark.parametrize("n", [113, 130])
def test_kquant_many_inputs_match_oracle(dtype, encode, n):
    print(f"case: {NAMES[dtype]} against {n} inputs", flush=True)
    rng = np.random.default_rng(n + dtype)
    rows = encode(rng.standard_normal((19, 768)).astype(np.float32) * np.float32(0.05))
    x = rng.standard_normal((n, 768)).astype(np.float32)
    out, _, st, _ = host_model().matvec(dtype, 19, 768, rows.reshape(-1), x)
    want, rcs = oracle_dots(list(rows), dtype, 768, x)
    assert not st.any() and not rcs.any()
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
