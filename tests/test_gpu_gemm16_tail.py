"""Split-FP16 products whose last round of 256x128 tiles is shared by several workgroups, and tiles past the edge of M
and of N, against NumPy by the normwise error of tests/test_gpu_gemm16.py: with and without whole tiles before the
shared ones."""
import numpy as np
import pytest

from test_gpu_gemm16 import FP16X3, _normwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(595, 18145, 2048), (561, 9000, 4096), (6460, 6460, 1100), (256, 128, 3000),
                                   (4100, 4100, 1500), (300, 33000, 1060), (2561, 2689, 1056), (49, 20000, 2080)])
def test_gemm16_tail(ctx, M, N, K):
    rng = np.random.default_rng(M + N + K)
    A, B, C0 = rng.normal(size=(K, M)), rng.normal(size=(K, N)), rng.normal(size=(M, N))
    ref = 0.5 * (A.T @ B) + 0.25 * C0
    out = ctx.gemm_test(FP16X3, "T", "N", 0.5, A, B, 0.25, C0)
    assert _normwise(out, ref, A, B, 0.5, 0.25, C0) < 4e-6
    assert np.array_equal(out, ctx.gemm_test(FP16X3, "T", "N", 0.5, A, B, 0.25, C0))  # fixed order
