"""FP64 products whose last round of 128x128 tiles is shared by several workgroups, against NumPy: sizes with and
without tiles past the edge of M, of N and of both, with whole tiles before the shared ones and without, and
contractions that 16 does not divide."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

SHAPES = [(253, 8911, 2911), (256, 4992, 5040), (400, 2000, 10000), (210, 5050, 5050), (2500, 2500, 1999),
          (2432, 2432, 2000), (3082, 3082, 1600), (3073, 2945, 2001), (129, 9000, 7000)]


@pytest.mark.parametrize("trans", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_tail(ctx, trans, M, N, K):
    rng = np.random.default_rng(M * 5 + N * 3 + K)
    A = rng.normal(size=(K, M) if trans[0] == "T" else (M, K))
    B = rng.normal(size=(N, K) if trans[1] == "T" else (K, N))
    C0 = rng.normal(size=(M, N))
    ref = 0.7 * ((A.T if trans[0] == "T" else A) @ (B.T if trans[1] == "T" else B)) - 1.3 * C0
    out = ctx.gemm_test(0, trans[0], trans[1], 0.7, A, B, -1.3, C0)
    # the rounding of a K-term sum of independent terms grows as sqrt(K) at most
    assert rel_err(out, ref) < 1e-13 * max(1.0, np.sqrt(K) / 4)
    assert np.array_equal(out, ctx.gemm_test(0, trans[0], trans[1], 0.7, A, B, -1.3, C0))  # fixed order
