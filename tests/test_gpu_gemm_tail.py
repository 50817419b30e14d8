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


@pytest.mark.parametrize("prec,tol", [(0, 1e-13), (1, 2e-5)])
@pytest.mark.parametrize("M,N,K", [(400, 2000, 10000), (2500, 2490, 1999)])
def test_gemm_tail_leading_dimensions(ctx, prec, tol, M, N, K):
    """Odd leading dimensions above the sizes; what lies past M in C's columns is left alone."""
    from jues._lib import ptr
    rng = np.random.default_rng(M + N)
    A = np.asfortranarray(rng.normal(size=(M + 3, K)))
    B = np.asfortranarray(rng.normal(size=(K + 5, N)))
    C = np.asfortranarray(rng.normal(size=(M + 7, N)))
    C0 = C.copy()
    ctx.check(ctx.lib.jues_gemm_test(ctx.h, prec, b"N", b"N", M, N, K, 0.7, ptr(A), M + 3, ptr(B), K + 5, -1.3, ptr(C),
                                     M + 7))
    ref = 0.7 * (A[:M] @ B[:K]) - 1.3 * C0[:M]
    # as above and as in the FP32 test: inputs rounded once, a sum's rounding grows as sqrt(K) at most
    assert rel_err(C[:M], ref) < tol * max(1.0, np.sqrt(K) / 4)
    left = C0[M:] if prec == 0 else C0[M:].astype(np.float32)  # an FP32 product returns its FP32 copy of C
    assert np.array_equal(C[M:], left)
