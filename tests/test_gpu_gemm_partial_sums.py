"""FP32 products over a long contraction whose partial sums come from several workgroups or wavefronts: the partial
sums, and beta C, are added in FP64 and rounded once.  Each of the three products that are not zero lies in a partial sum
of its own, exact in FP32, and the large ones cancel: added in FP32 the small one would be lost."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 60 tiles of 128 x 128 shared by workgroups; the same with tiles past the edges; tiles of 16 x 16 shared by wavefronts
@pytest.mark.parametrize("M,N,K", [(640, 1536, 20000), (600, 1500, 20000), (200, 200, 4096)])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_partial_sums_in_fp64(ctx, M, N, K, beta):
    big, mid = 4096.0, K // 2 + 16
    A, B = np.zeros((M, K)), np.zeros((K, N))
    A[:, 0], B[0] = big, big                                # 2^24
    A[:, mid], B[mid] = 1.0 + 2.0 * (np.arange(M) % 4), 1.0   # odd: 2^24 + it has no FP32 value
    want = np.broadcast_to(A[:, mid:mid + 1], (M, N))
    C0 = np.full((M, N), -big * big)
    if beta == 0.0:
        A[:, K - 1], B[K - 1] = -big, big
    assert np.array_equal(ctx.gemm_test(1, "N", "N", 1.0, A, B, beta, C0), want)
