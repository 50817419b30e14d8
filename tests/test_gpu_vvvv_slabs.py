"""The packed (vv|vv) integrals, cut to the pairs e <= f and packed through LDS, at virtual counts around the 16-wide
tiles and with one to several slabs of the cut product: CCD steps from factored integrals, with the ladder stored and
recomputed, against those from the dense integrals, whose (vv|vv) is transformed whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v", [(2, 2), (2, 15), (3, 16), (3, 17), (2, 33), (11, 40), (3, 70)])
def test_vvvv_slabs(o, v):
    from jues import synthetic
    from jues.CoupledCluster import Solver
    from jues.Wavefunction import FactoredERI, Wfn
    s = synthetic.make_system(o + v, o, v, 2 * (o + v), 70 + v, name="vvvv")

    def steps(eri, ladder):
        sol = Solver(Wfn.from_orbitals(s.C, s.eps, s.o, eri), method="rccd", prec="fp64", guess="mp2", diis=False,
                     ladder=ladder)
        sol.iterate(2, "fp64")
        return sol.result()

    ref = steps(s.ao_eri(), "stored")
    for ladder in ("stored", "recompute"):
        got = steps(FactoredERI(s.B), ladder)
        # two steps from the same start differ by rounding, relative to the largest amplitude (as in the ladder's tests)
        assert abs(got[0] - ref[0]) < 1e-12 * max(1.0, abs(ref[0]))
        assert np.max(np.abs(got[-1] - ref[-1])) < 1e-12 * np.max(np.abs(ref[-1]))
