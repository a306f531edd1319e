"""The order of the exact F16 dots' f64 sums does not depend on the batch.

The exact F16 kernels split a dot over lanes and waves.  Which products meet in
which order is fixed by the matrix and the side of 16 rows, never by the number
of rows.  The inputs here make any difference visible: large products that
cancel exactly, with small ones between them that round at the large ones' last
bit, so two orders give different f32 results.  (On ordinary weights the orders
agree, and these sums equal the oracle's one chain.)"""
import numpy as np
import pytest

from test_gpu_kquant import host_model

pytestmark = pytest.mark.gpu

F16 = 1


@pytest.mark.parametrize("rows", [300, 6400, 9600])
def test_f16_dots_do_not_depend_on_the_batch(rows):
    """300, 6,400 and 9,600 rows cross the dispatch's lines on grid size at
    17 to 129 inputs."""
    print(f"case: F16 dots of {rows} rows among 1 to 129 inputs", flush=True)
    rng = np.random.default_rng(rows)
    K = 512
    m = host_model()
    w = (rng.standard_normal((rows, K)) * 2.0 ** -14).astype(np.float16)
    x = (rng.standard_normal((129, K)) * 2.0 ** -10).astype(np.float16)
    big = rng.permutation(K)[:16].reshape(8, 2)  # eight pairs of +-2^30
    for a, b in big:
        w[:, a] = rng.uniform(2.0 ** 14, 2.0 ** 15, rows).astype(np.float16)
        w[:, b] = -w[:, a]
        x[:, a] = x[:, b] = rng.uniform(2.0 ** 14, 2.0 ** 15, 129).astype(np.float16)
    x = x.astype(np.float32)
    got = {}
    for n in (1, 4, 5, 11, 16, 17, 33, 65, 97, 129):
        out, _, st, _ = m.matvec(F16, rows, K, w.view(np.uint8), x[:n])
        assert not st.any()
        got[n] = out.view(np.uint32)
    for n in (1, 4, 5, 11):
        assert np.array_equal(got[n], got[16][:n]), n
    for n in (17, 33, 65, 97):
        assert np.array_equal(got[n], got[129][:n]), n
