"""One CCD / CCSD update of random amplitudes with many occupied and few virtual orbitals, against the oracle's
restatements: below and past the 77 (FP64) and 110 (FP32) occupied orbitals up to which the update kernel symmetrises
the ring terms itself, at products o v where a system of fewer occupied orbitals takes the small system's launches, by
default (up to 40 and 60) or forced (JUES_SMALL_MAX_OV)."""
import numpy as np
import pytest

import jues_oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(77, 4, False), (78, 2, False), (78, 2, True), (84, 4, False), (84, 6, False), (100, 5, False), (110, 3, False),
         (111, 2, False), (111, 3, False)]


def check_one_update(o, v, dense):
    from jues import CoupledCluster as CC
    from jues import synthetic
    from jues.Wavefunction import Wfn
    n = o + v
    s = synthetic.make_system(n, o, v, 40, n)
    s.B = s.B * np.sqrt(0.1)
    w = Wfn.from_synthetic(s, dense=dense)
    rng = np.random.default_rng(n)
    T1, T2 = 0.1 * rng.normal(size=(o, v)), 0.1 * rng.normal(size=(o, o, v, v))
    T2 = T2 + T2.transpose(1, 0, 3, 2)
    D1, D2 = O.form_Dia(s.eps, o, v), O.form_Dijab(s.eps, o, v)
    ccd = O.rccd_step(T2, O.rccd_integrals_from_factors(s.B, s.Co, s.Cv), D2)
    ccsd = [r / d for r, d in zip(O.rccsd_update(T1, T2, O.rccsd_integrals_from_factors(s.B, s.Co, s.Cv)), (D1, D2))]
    # the longest sums have o^2 products: rounding grows as their root, o, times the unit roundoff; 64 for the number
    # of such terms and the size of the largest intermediates
    for prec, u in (("fp64", 1.2e-16), ("fp32_mixed", 6e-8)):
        kw = dict(T2=T2, maxit=1, refine_maxit=0, check_convergence=False, prec=prec, diis=False)
        got = [CC.RCCD.do_rccd(w, return_T2=True, **kw)[1], *CC.mRCCSD.do_rccsd(w, T1=T1, return_T=True, **kw)[1:]]
        for name, a, b in zip(("CCD T2", "CCSD T1", "CCSD T2"), got, (ccd, *ccsd)):
            err, bound = float(np.max(np.abs(a - b))), 64 * o * u * float(np.max(np.abs(b)))
            assert err <= bound, (name, prec)


@pytest.mark.parametrize("o,v,dense", SIZES + [(40, 4, False), (41, 4, False), (60, 3, False), (60, 4, True), (61, 3, False)])
def test_one_update(o, v, dense):
    check_one_update(o, v, dense)


@pytest.mark.parametrize("o,v,dense", SIZES)
def test_one_update_forced(o, v, dense, monkeypatch):
    monkeypatch.setenv("JUES_SMALL_MAX_OV", "504")
    check_one_update(o, v, dense)


@pytest.mark.parametrize("o", [78, 111])
def test_one_virtual_orbital(o):
    """No pairs a < b: the antisymmetric part of Z = tau (mf|ae) is empty.  Twice, so that the second run's buffers are
    the first one's blocks with what they were left with."""
    for _ in range(2):
        check_one_update(o, 1, False)
