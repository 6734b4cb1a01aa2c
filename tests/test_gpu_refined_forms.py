"""Refined resident phases, every form, against the same phases launched kernel by
kernel (TL_TUNE_RESIDENT 0): capped solves, so that forms whose solve takes long
are run too (PPCG without a preconditioner), on the edges of flat and tall blocks.

The two sum p.w in different orders (by bands of rows where launched), so they
agree to rounding. With n cells a sum of positive terms differs by at most n 2^-53
relative, and so do alpha and beta; the timestep is short (rx, ry <= 0.2 and faces of
at most 10: A's eigenvalues lie in [1, 17]), so that an iteration does not enlarge
what comes in by more than that, and after k iterations or smoothing steps the
increment d of the solution differs by at most 20 k n 2^-53 of its largest value. FP32
inner vectors are rounded in every step, where a difference may fall on either side:
20 k 2^-24."""
import numpy as np
import pytest

from _pairs import setup

pytestmark = pytest.mark.gpu

GRIDS = [(64, 16), (65, 17), (63, 130), (515, 509), (4160, 64), (1024, 1024), (1100, 1000), (16001, 100), (1500, 1401),
         (130, 20001), (2048, 2048)]


def solve(hiplib, nx, ny, prec, precision, inner, resident):
    c = hiplib.Chunk(nx, ny, 1, prec)
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, resident, chunk=c)
    setup(c, seed=2, coef=1, dt=0.2 * (10.0 / max(nx, ny)) ** 2)
    if inner:
        res = c.solve_refined_ppcg(precision, tol=1e-300, max_iters=9, presteps=6, inner_steps=inner)
    else:
        res = c.solve_refined(precision, tol=1e-300, max_iters=9)
    u, u0 = c.interior(c.get_field("u")), c.interior(c.get_field("u0"))
    c.close()
    assert not (resident and res["k_samples"])
    return res, u, u - u0


@pytest.mark.parametrize("inner", [0, 5])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("prec", [1, 2, 3])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_capped(hiplib, nx, ny, prec, precision, inner):
    (a, ua, da), (b, ub, db) = (solve(hiplib, nx, ny, prec, precision, inner, r) for r in (1, 0))
    assert a["iterations"] == b["iterations"] == 9
    assert a["inner_iterations"] == b["inner_iterations"]
    k = 9 + a["inner_iterations"]
    tol = 20 * k * (nx * ny * 2.0 ** -53 if precision == 0 else 2.0 ** -24)
    assert np.abs(ua - ub).max() <= tol * np.abs(db).max(), (np.abs(ua - ub).max() / np.abs(db).max(), tol)
    assert a["initial_residual"] == b["initial_residual"]
