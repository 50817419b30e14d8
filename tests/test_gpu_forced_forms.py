"""The tests of the split-FP16 stage, of the recomputed ladder, of released FP64 blocks, of the defect correction and of
the packed pairs' edges once more with the general residual and split products forced (JUES_SMALL_MAX_OV,
JUES_SPLIT_MIN_OV): by size, their systems take the small system's launches and FP32 products."""
import numpy as np
import pytest

from test_auto_rccsd import non_hf, test_gpu_auto_non_hf, water  # noqa: F401
from test_df import cfg1_df, cfg1_df_ref, test_gpu_df_rccd_fast_forms  # noqa: F401
from test_gpu_defect import (e_ccd, test_defect_solve_reaches_fp64_fixed_point,  # noqa: F401
                             test_defect_solve_with_frozen_core_and_continuation,
                             test_defect_solve_with_released_fp64_blocks, test_fast_correction_error_scales_with_d,
                             test_fp64_inner_reproduces_jacobi_steps)
from test_gpu_failures import test_identical_solves_are_bitwise_identical  # noqa: F401
from test_gpu_fp16x3 import (test_cfg1_rccd_converges_to_fp64, test_cfg1_rccsd_converges_to_fp64,  # noqa: F401
                             test_split_steps_track_fp64, test_water_known_answers_fp16x3)
from test_gpu_ladder import (small_slabs, test_recompute_converges_to_golden,  # noqa: F401
                             test_recompute_steps_match_stored)
from test_gpu_pair_edges import test_rccd_pair_edges, test_rccsd_pair_edges  # noqa: F401
from test_gpu_thin import refs, test_thin_fast_forms_converge, test_thin_stage_switches, thin  # noqa: F401
from test_known_answers import test_gpu_rccd_known_answer_defect_correction, water_psi4  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def forced(monkeypatch):
    monkeypatch.setenv("JUES_SMALL_MAX_OV", "0")
    monkeypatch.setenv("JUES_SPLIT_MIN_OV", "0")


def test_forms_are_forced(cfg1, monkeypatch):
    """One fp16x3 update at n = 24: FP32 products by size, other ones when the split is forced."""
    from jues.CoupledCluster import Solver
    from jues.Wavefunction import Wfn

    def step(prec):
        sv = Solver(Wfn.from_synthetic(cfg1, dense=False), method="rccd", prec=prec, guess="mp2", diis=False)
        sv.iterate(1, prec)
        return sv.result()[1]

    split, general = step("fp16x3"), step("fp32_mixed")
    assert not np.array_equal(split, general)
    monkeypatch.delenv("JUES_SPLIT_MIN_OV")
    assert np.array_equal(step("fp16x3"), general)
    monkeypatch.delenv("JUES_SMALL_MAX_OV")
    small = step("fp32_mixed")
    assert not np.array_equal(small, general) and np.array_equal(step("fp16x3"), small)
