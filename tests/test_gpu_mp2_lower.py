"""MP2 energy and adjoint from the lower triangle of (ia|jb) = L L^T (factored integrals, FP64) against the oracle:
fewer rows than a 128x128 tile, rows that 128 divides and does not, several bands of tiles, and the occupied counts at
and past the ends of the range that takes it."""
import numpy as np
import pytest

import jues_oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


def _system(o, v, naux, seed):
    rng = np.random.default_rng(seed)
    n = o + v
    B = rng.normal(size=(n, n, naux)) * 0.05
    B = np.asfortranarray(B + B.transpose(1, 0, 2) + 0.01 * rng.normal(size=B.shape))  # not symmetric
    C = np.asfortranarray(np.linalg.qr(rng.normal(size=(n, n)))[0])
    eps = np.concatenate([np.sort(rng.uniform(-1.5, -0.5, o)), np.sort(rng.uniform(0.5, 3.0, v))])
    return B, C, eps


@pytest.mark.parametrize("o,v,naux", [(15, 20, 30), (16, 3, 40), (16, 64, 70), (17, 41, 50), (40, 61, 130), (65, 40, 90),
                                      (88, 21, 60), (89, 11, 60)])
def test_mp2_lower_triangle(o, v, naux):
    from jues import MollerPlesset
    from jues.Wavefunction import Wfn, FactoredERI
    B, C, eps = _system(o, v, naux, 100 * o + v)
    w = Wfn.from_orbitals(C, eps, o, FactoredERI(B))
    E0, dC0 = O.rmp2_grad_factors(B, C, eps, o)
    K = O.mo_from_factors(B, C[:, :o], C[:, o:], C[:, :o], C[:, o:])
    de0 = O.rmp2_grad_eps(K, eps, o)
    # rounding of sums of naux and (ov)^2 terms
    assert abs(MollerPlesset.do_rmp2(w) - E0) < 1e-12 * abs(E0)
    E, dC, dg, de = MollerPlesset.rmp2_grad(w)
    assert dg is None and abs(E - E0) < 1e-12 * abs(E0)
    assert rel_err(dC, dC0) < 1e-11 and rel_err(de, de0) < 1e-11
