"""The error of long FP32 products: whatever form a product takes, an accumulator sums no more of k than the chunk given
here before it is added to others in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,chunk", [(1000, 1000, 8192, 1024), (500, 3000, 8192, 1024), (2048, 512, 16384, 1024),
                                         (800, 800, 20000, 1056), (2800, 1500, 33600, 2240), (4200, 1500, 33600, 6720)])
def test_chain_length(ctx, M, N, K, chunk):
    rng = np.random.default_rng(M + K)
    A = rng.normal(size=(M, K)).astype(np.float32).astype(np.float64)
    B = rng.normal(size=(K, N)).astype(np.float32).astype(np.float64)
    rows = slice(0, M, M // 50)
    d = ctx.gemm_test(1, "N", "N", 1.0, A, B, 0.0, np.zeros((M, N)))[rows] - A[rows] @ B
    # a sum of L products of unit variance: step j rounds a partial sum of size sqrt(j), by u / sqrt(3) of it with
    # u = 2^-24, so its error has the root mean square u / sqrt(3) L / sqrt(2); K / L such sums are independent
    bound = 2.0 ** -24 / np.sqrt(6.0) * np.sqrt(K * chunk)
    assert float(np.sqrt(np.mean(d * d))) < bound
