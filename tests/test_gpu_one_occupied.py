"""One occupied orbital and as many virtual ones as the small system's launches (forced here) index V+ with 32 bits for
(303), and one more: the stored ladder, whose V+ has 46056 and 46360 rows and columns there, against the recomputed one,
which has no V+."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["rccd", "rccsd"])
@pytest.mark.parametrize("v", [303, 304])
def test_stored_ladder_equals_recomputed(v, method, monkeypatch):
    monkeypatch.setenv("JUES_SMALL_MAX_OV", "504")
    from jues import synthetic
    from jues.CoupledCluster import Solver
    from jues.Wavefunction import Wfn, FactoredERI
    s = synthetic.make_system(v + 1, 1, v, 40, v)
    w = Wfn.from_orbitals(s.C, s.eps, 1, FactoredERI(np.asfortranarray(0.1 * s.B)))
    got = []
    for ladder in ("stored", "recompute"):
        sv = Solver(w, method=method, prec="fp64", guess="mp2", diis=False, ladder=ladder)
        sv.iterate(2, "fp64")
        got.append(sv.result())
        del sv
    # sums of v^2 products in another order: their rounding grows as the root, v, times 1.1e-16
    scale = np.max(np.abs(got[0][-1]))
    assert float(np.max(np.abs(got[0][-1] - got[1][-1]))) < 32 * v * 1.2e-16 * scale
    assert abs(got[0][0] - got[1][0]) < 32 * v * 1.2e-16 * abs(got[0][0])
