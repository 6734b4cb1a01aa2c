"""The kernels launched one by one and the captured graphs on grids that would
run resident, with the resident solver tuned off (TL_TUNE_RESIDENT 0): the tests
of those kernels' remainders, buffers and graph captures over again, which compare
their one-step and two-step forms, a solve with the same solve on a fresh chunk,
and either with the oracle.

Beside them the two-step kernels against the one-step ones on a grid beyond the
resident solver, with grouped tile columns and partial tiles, bitwise.
"""
import numpy as np
import pytest

from _pairs import setup
from tealeaf_opencl_amd import decks
from test_gpu_decks import (test_cheby_native_iteration_cap, test_cheby_two_iterations_per_launch_bitwise,  # noqa: F401
                            test_config1_cg_diag_512, test_dropin_and_native_agree, test_kat1_jacobi,
                            test_kat6_ppcg_halo4, test_ppcg_fresh_z, test_ppcg_two_steps_per_launch_bitwise,
                            test_solvers_small)
from test_gpu_refine import (test_cg_and_ppcg_on_one_chunk, test_deck_summary_vs_oracle,  # noqa: F401
                             test_deterministic_and_reentrant, test_iteration_cap,
                             test_mixed_iterations_close_to_fp64, test_ppcg_deck_summary, test_ppcg_true_residual,
                             test_reinit_with_new_operator, test_stalls_at_rounding_floor, test_true_residual)
from test_gpu_refine import test_ppcg_two_steps_per_launch_bitwise as test_refined_ppcg_two_steps_bitwise  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def launched(hiplib):
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, 0)
    yield
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, 1)


def test_tuned_off(hiplib, tmp_path):
    """Kernel times are sampled only where kernels are launched one by one."""
    deck = decks.write_deck(str(tmp_path / "t.in"), 130, 90, decks.seeded_states(2, 2, True), max_iters=90, eps=1e-300)
    off = hiplib.bench_deck(deck, warmup=0, steps=1)
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, 1)
    on = hiplib.bench_deck(deck, warmup=0, steps=1)
    assert off["k_samples"] > 0 and on["k_samples"] == 0
    assert off["iterations"] == on["iterations"] and off["final_summary"] == on["final_summary"]
    for value in (-3, 1001):
        with pytest.raises(hiplib.TealeafError):
            hiplib.set_tuning(hiplib.TUNE_RESIDENT, value)


WIDE = (3001, 1601)  # 47 tile columns in eight groups, partial in both directions


@pytest.mark.parametrize("solver,key", [("tl_use_ppcg", "TUNE_PPCG_STEPS_PER_LAUNCH"),
                                        ("tl_use_chebyshev", "TUNE_CHEBY_STEPS_PER_LAUNCH")])
@pytest.mark.parametrize("prec", ["none", "jac_block"])
def test_two_steps_on_grouped_columns(hiplib, tmp_path, solver, key, prec):
    deck = decks.write_deck(str(tmp_path / "w.in"), *WIDE, decks.seeded_states(2, 2, True), solver=solver,
                            preconditioner=prec, end_step=1, eps=1e-300, max_iters=41,
                            extra=["tl_ppcg_inner_steps=7", "tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"])
    out = []
    try:
        for per in (1, 2):
            hiplib.set_tuning(getattr(hiplib, key), per)
            out.append(hiplib.run_deck(deck, tmp_path / ("%d.log" % per)))
    finally:
        hiplib.set_tuning(getattr(hiplib, key), 2)
    assert out[0]["summary"] == out[1]["summary"]
    assert np.array_equal(np.array(out[0]["solve"], float), np.array(out[1]["solve"], float), equal_nan=True)
    assert out[0]["solve"][0][1] == 41


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("prec,inner", [(1, 6), (3, 7)])
def test_refined_two_steps_on_grouped_columns(hiplib, prec, inner, precision):
    out = []
    for per in (1, 2):
        c = hiplib.Chunk(*WIDE, 1, prec)
        setup(c, seed=2, coef=2)
        hiplib.set_tuning(hiplib.TUNE_PPCG_STEPS_PER_LAUNCH, per, chunk=c)
        res = c.solve_refined_ppcg(precision, tol=1e-300, max_iters=41, presteps=20, inner_steps=inner)
        out.append((res["iterations"], res["updates"], res["rel_residual"], c.get_field("u")))
        c.close()
    assert out[0][:3] == out[1][:3] and out[0][0] == 41
    assert np.array_equal(out[0][3], out[1][3])
