"""The resident solver on tall blocks (tl_resident.h: grids of more than a
million cells, faces formed anew in every pass) against the same iterations
launched one by one, as a profiler_on run does: the same operations in the same
order, so bitwise the same summaries, iteration counts and residuals. Only
Chebyshev's residual norms differ, in the order of at most 2^22 positive terms:
1e-10 relative.

Grids: blocks of 32, 48 and 64 strips of rows, with the last block's wavefronts,
strips, rows and columns partly or wholly outside the grid, one row of blocks,
and the largest grid that fits.
"""
import pytest

from _pairs import setup
from test_gpu_resident import both

pytestmark = pytest.mark.gpu

GRIDS = [(1100, 1000), (16001, 100), (1500, 1401), (2001, 1503), (130, 20001), (2048, 2048)]
PRECS = ["none", "jac_diag", "jac_block"]


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_cg(hiplib, tmp_path, nx, ny, prec):
    both(hiplib, tmp_path, nx, ny, "tl_use_cg", prec, 40)


def test_cg_several_launches(hiplib, tmp_path):
    log = both(hiplib, tmp_path, 1100, 1000, "tl_use_cg", "jac_diag", 1300, steps=1, eps=1e-15,
               coefficient="tl_coefficient_inverse_density")
    assert log["solve"][0][1] > 1024


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_cheby(hiplib, tmp_path, nx, ny, prec):
    both(hiplib, tmp_path, nx, ny, "tl_use_chebyshev", prec, 61,
         extra=["tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"], norm=1e-10)


@pytest.mark.parametrize("inner", [1, 7])
@pytest.mark.parametrize("prec", PRECS + ["jac_block-fresh"])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_ppcg(hiplib, tmp_path, nx, ny, prec, inner):
    parts = prec.split("-")
    extra = ["tl_ppcg_inner_steps=%d" % inner, "tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"]
    both(hiplib, tmp_path, nx, ny, "tl_use_ppcg", parts[0], 30, steps=1,
         extra=extra + ["tl_ppcg_fresh_z"] * (len(parts) - 1))


def test_ppcg_several_launches(hiplib, tmp_path):
    log = both(hiplib, tmp_path, 1100, 1000, "tl_use_ppcg", "jac_diag", 120, steps=1, eps=1e-300,
               extra=["tl_ppcg_inner_steps=10", "tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"])
    assert log["solve"][0][1] == 120


@pytest.mark.parametrize("inner", [0, 6])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("prec", [1, 2, 3])
@pytest.mark.parametrize("nx,ny", [(1100, 1000), (1500, 1401), (2048, 2048)])
def test_refined(hiplib, nx, ny, prec, precision, inner):
    """The solution's true residual, formed by the library's own residual and
    norm kernels, meets the tolerance that the solve claims (1 % for the norms'
    rounding) and agrees with the one it reports."""
    if inner and prec == 1:
        pytest.skip("PPCG without a preconditioner takes up to more than 20000 steps on these grids")
    c = hiplib.Chunk(nx, ny, 1, prec)
    setup(c, seed=2, coef=2)
    c.calc_residual()
    r0 = c.calc_2norm(1) ** 0.5
    if inner:
        res = c.solve_refined_ppcg(precision, tol=1e-10, max_iters=20000, presteps=20, inner_steps=inner)
    else:
        res = c.solve_refined(precision, tol=1e-10, max_iters=20000)
    assert res["converged"], res
    c.calc_residual()
    r = c.calc_2norm(1) ** 0.5
    assert r <= 1.01e-10 * r0, (r / r0, res)
    assert abs(res["rel_residual"] - r / r0) <= 1e-2 * 1e-10
    c.close()
