"""One CCD / CCSD update of random amplitudes where the small system's launches evaluate the residual, and just
past their limit, against the oracle's restatements: blocks below, at and past one 16 x 16 tile, o > v, one occupied
or one virtual orbital, contractions cut into partial outputs, dense and factored integrals, both CCSD equation
sets, FP64 and FP32."""
import numpy as np
import pytest

import jues_oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 6), (5, 2), (3, 1), (4, 4), (2, 9), (8, 6), (5, 19), (12, 28), (9, 38), (17, 30)]


@pytest.mark.parametrize("dense", [True, False])
@pytest.mark.parametrize("o,v", SIZES)
def test_one_update(o, v, dense):
    from jues import CoupledCluster as CC
    from jues import synthetic
    from jues.Wavefunction import Wfn
    n = o + v
    s = synthetic.make_system(n, o, v, 3 * n, n)
    s.B = s.B * np.sqrt(0.1)
    g, w = s.ao_eri(), Wfn.from_synthetic(s, dense=dense)
    rng = np.random.default_rng(n)
    T1, T2 = 0.1 * rng.normal(size=(o, v)), 0.1 * rng.normal(size=(o, o, v, v))
    T2 = T2 + T2.transpose(1, 0, 3, 2)
    D1, D2 = O.form_Dia(s.eps, o, v), O.form_Dijab(s.eps, o, v)
    want = {"ccd": (O.rccd_step(T2, O.make_rccd_integrals(g, s.Co, s.Cv), D2),)}
    X = O.make_rccsd15_integrals(lambda *C: O.tei_transform(g, *C), s.Co, s.Cv)
    want["RCCSD"] = [r / d for r, d in zip(O.rccsd15_update(T1, T2, X), (D1, D2))]
    want["mRCCSD"] = [r / d for r, d in zip(O.rccsd_update(T1, T2, O.make_rccsd_integrals(g, s.Co, s.Cv)), (D1, D2))]
    # sums of at most o v^2 products: FP64 rounding well below 1e-12 of the largest element, FP32 (unit roundoff
    # 6e-8) below 2e-5 of it
    for prec, tol in (("fp64", 1e-12), ("fp32_mixed", 2e-5)):
        kw = dict(T2=T2, maxit=1, refine_maxit=0, check_convergence=False, prec=prec, diis=False)
        got = {"ccd": CC.RCCD.do_rccd(w, return_T2=True, **kw)[1:],
               "RCCSD": CC.RCCSD.do_rccsd(w, T1=T1, return_T=True, **kw)[1:],
               "mRCCSD": CC.mRCCSD.do_rccsd(w, T1=T1, return_T=True, **kw)[1:]}
        for name in want:
            for a, b in zip(got[name], want[name]):
                assert np.max(np.abs(a - b)) <= tol * np.max(np.abs(b)), (name, prec)
