"""A defect correction asked for in split FP16 whose system is too small for split products (they run in FP32) stops its
inner solves where the FP32 form does: the two take the same iterations."""
import pytest

pytestmark = pytest.mark.gpu


def test_fp32_products_take_the_fp32_target(cfg1):
    from jues import CoupledCluster as CC
    from jues.Wavefunction import Wfn
    w = Wfn.from_synthetic(cfg1, dense=False)
    runs = []
    for prec in ("fp32_mixed", "fp16x3"):
        hist = []
        E = CC.mRCCD.do_rccd(w, prec=prec, refine="defect", cc_e_conv=1e-11, cc_max_rms=1e-11, maxit=300,
                             callback=hist.append)
        runs.append((E, [(h["stage"] == 0, h["energy"], h["rnorm"]) for h in hist]))
    assert runs[0] == runs[1]
