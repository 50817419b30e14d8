"""Products that take each form of the GEMM dispatch (direct, 64x64, 128x128, short, tall; split and
unsplit contractions), at the edges of their tiles, against NumPy."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

# (M, N, K): vectors, blocks below one 16x16 MFMA block, one past a tile edge, K tails of 1 and 15, long
# contractions split over workgroups, and mid-sized squares around the 32 / 64 / 128 tiles
SHAPES = [(1, 2000, 2000), (360, 1, 2000), (1, 1, 5000), (5, 5, 1805), (16, 17, 15), (17, 16, 31), (33, 31, 129),
          (95, 95, 95), (65, 64, 1025), (129, 127, 700), (20, 20, 70001), (120, 1000, 2850), (500, 499, 501),
          (1125, 1123, 300), (20, 9001, 100), (9001, 20, 96), (640, 641, 1280)]


@pytest.mark.parametrize("prec,tol", [(0, 1e-13), (1, 2e-5)])
@pytest.mark.parametrize("trans", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_forms(ctx, prec, tol, trans, M, N, K):
    rng = np.random.default_rng(M * 5 + N * 3 + K)
    A = rng.normal(size=(K, M) if trans[0] == "T" else (M, K))
    B = rng.normal(size=(N, K) if trans[1] == "T" else (K, N))
    C0 = rng.normal(size=(M, N))
    ref = 0.7 * ((A.T if trans[0] == "T" else A) @ (B.T if trans[1] == "T" else B)) - 1.3 * C0
    out = ctx.gemm_test(prec, trans[0], trans[1], 0.7, A, B, -1.3, C0)
    # the rounding of a K-term sum of independent terms grows as sqrt(K) at most
    assert rel_err(out, ref) < tol * max(1.0, np.sqrt(K) / 4)
    assert np.array_equal(out, ctx.gemm_test(prec, trans[0], trans[1], 0.7, A, B, -1.3, C0))  # fixed order


@pytest.mark.parametrize("prec,tol", [(0, 1e-13), (1, 2e-5)])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("M0,N0,K0,M1,N1,K1", [(15, 15, 190, 10, 10, 171), (120, 120, 2850, 105, 105, 2775),
                                               (210, 5050, 210, 190, 4950, 190), (276, 276, 9045, 253, 253, 8911)])
def test_gemm_pair_forms(ctx, prec, tol, trans, M0, N0, K0, M1, N1, K1):
    rng = np.random.default_rng(M0 + K1)
    A0, A1 = rng.normal(size=(M0, K0)), rng.normal(size=(M1, K1))
    B0, B1 = (rng.normal(size=(n, k) if trans == "T" else (k, n)) for n, k in ((N0, K0), (N1, K1)))
    C0, C1 = rng.normal(size=(M0, N0)), rng.normal(size=(M1, N1))
    X0, X1 = ctx.gemm_pair_test(prec, trans, 0.5, A0, B0, C0, A1, B1, C1, 1.0)
    for X, A, B, C, K in ((X0, A0, B0, C0, K0), (X1, A1, B1, C1, K1)):
        assert rel_err(X, 0.5 * (A @ (B.T if trans == "T" else B)) + C) < tol * max(1.0, np.sqrt(K) / 4)
