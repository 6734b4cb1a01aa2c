"""PPCG solves of the resident solver that end at tl_max_iters, with more
smoothing steps than one launch holds several outer steps of: a launch makes
1024 / (inner + 2) outer steps, rounded down (at least one), so that a capped
solve takes more launches than its smoothing steps alone would need. The same
iterations launched one by one (a profiler_on run) end at the same cap, bitwise
alike."""
import pytest

from test_gpu_resident import both

pytestmark = pytest.mark.gpu


# 128 smoothing steps (the deck reader's default at 1024^2): 7 outer steps per
# launch; 600: one. The long timestep keeps the residual from reaching zero.
@pytest.mark.parametrize("nx,ny,inner,cap", [(200, 148, 128, 1000), (130, 70, 600, 700)])
def test_ppcg_ends_at_the_cap(hiplib, tmp_path, nx, ny, inner, cap):
    log = both(hiplib, tmp_path, nx, ny, "tl_use_ppcg", "jac_diag", cap, steps=1, eps=1e-300, dt=4e3,
               coefficient="tl_coefficient_inverse_density",
               extra=["tl_ppcg_inner_steps=%d" % inner, "tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"])
    assert log["solve"][0][1] == cap
