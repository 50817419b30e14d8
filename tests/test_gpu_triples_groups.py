"""(T) where the occupied triples are taken in several groups (their W exceed the group's 192 MB), the last
one short, and where the virtual dimension is just past a tile edge, against the oracle."""
import numpy as np
import pytest

import jues_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,prec,tol", [(5, 110, "fp64", 1e-12), (5, 120, "fp32_mixed", 2e-5), (6, 65, "fp64", 1e-12)])
def test_triples_in_groups(o, v, prec, tol):
    from jues import CoupledCluster as CC
    rng = np.random.default_rng(o * 1000 + v)
    n, naux = o + v, 30
    L = rng.normal(scale=0.1, size=(n, n, naux))
    L = L + L.transpose(1, 0, 2)
    Vvvvo, Vvooo, Vvovo = O.pt_integrals(lambda *C: O.mo_from_factors(L, *C), np.eye(n)[:, :o], np.eye(n)[:, o:])
    T1, T2 = rng.normal(size=(o, v)), rng.normal(size=(o, o, v, v))
    T2 = T2 + T2.transpose(1, 0, 3, 2)
    fo, fv = -1.5 + np.arange(o) / o, 0.3 + np.arange(v) / v
    ref = O.compute_pT(T1, T2, Vvvvo, Vvooo, Vvovo, fo, fv)
    E = CC.PerturbativeTriples.compute_pT(T1=T1, T2=T2, Vvvvo=Vvvvo, Vvooo=Vvooo, Vvovo=Vvovo, fo=fo, fv=fv, prec=prec)
    # the same bounds as the single-group (T) tests: the sum's rounding does not depend on the grouping
    assert abs(E - ref) < tol * abs(ref)
