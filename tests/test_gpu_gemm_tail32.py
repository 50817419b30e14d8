"""FP32 products whose last round of 128x128 tiles is shared by several workgroups, against NumPy in FP64: the sizes
of tests/test_gpu_gemm_tail.py, whose map of tiles and parts is the same."""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_gemm_tail import SHAPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trans", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("M,N,K", SHAPES + [(6460, 6460, 330)])
def test_gemm_tail_fp32(ctx, trans, M, N, K):
    rng = np.random.default_rng(M * 5 + N * 3 + K)
    A = rng.normal(size=(K, M) if trans[0] == "T" else (M, K))
    B = rng.normal(size=(N, K) if trans[1] == "T" else (K, N))
    C0 = rng.normal(size=(M, N))
    ref = 0.7 * ((A.T if trans[0] == "T" else A) @ (B.T if trans[1] == "T" else B)) - 1.3 * C0
    out = ctx.gemm_test(1, trans[0], trans[1], 0.7, A, B, -1.3, C0)
    # inputs rounded to FP32 and a K-term sum of independent terms, whose rounding grows as sqrt(K) at most
    assert rel_err(out, ref) < 2e-5 * max(1.0, np.sqrt(K) / 4)
    assert np.array_equal(out, ctx.gemm_test(1, trans[0], trans[1], 0.7, A, B, -1.3, C0))  # fixed order
