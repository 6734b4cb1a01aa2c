"""The resident solver (tl_resident.h: the driver's iteration loops with the
whole state in registers, one launch per phase) against the same iterations
launched one by one, which a profiler_on run does. Both form every value with
the same operations and sum in the same order, so the field summaries, the
iteration counts and the residuals that end the solves are bitwise the same:
no tolerance.

Grids: one block (with partial strips and columns), the edges of a block's 64
columns and 16, 32 or 64 rows, a grid of one block per column or row of tiles,
the largest that fits, and solves of more iterations than one launch makes.
"""
import numpy as np
import pytest

from tealeaf_opencl_amd import decks

pytestmark = pytest.mark.gpu

GRIDS = [(10, 10), (64, 16), (65, 17), (63, 130), (200, 148), (515, 509), (64, 4096), (4160, 64), (1000, 701),
         (1024, 1024)]


def both(hiplib, tmp_path, nx, ny, solver, prec, max_iters, steps=2, eps=1e-13, extra=(), **kw):
    out = []
    for name, more in (("resident", []), ("launched", ["profiler_on"])):
        deck = decks.write_deck(str(tmp_path / (name + ".in")), nx, ny, decks.seeded_states(2, 2, True), solver=solver,
                                preconditioner=prec, end_step=steps, eps=eps, max_iters=max_iters,
                                extra=list(extra) + more, **kw)
        out.append(hiplib.run_deck(deck, str(tmp_path / (name + ".log"))))
    a, b = out
    assert a["summary"] == b["summary"]
    assert np.array_equal(np.array(a["solve"], float), np.array(b["solve"], float), equal_nan=True)
    return a


@pytest.mark.parametrize("prec", ["none", "jac_diag", "jac_block"])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_cg(hiplib, tmp_path, nx, ny, prec):
    both(hiplib, tmp_path, nx, ny, "tl_use_cg", prec, 90)


def test_cg_several_launches(hiplib, tmp_path):
    log = both(hiplib, tmp_path, 1024, 1024, "tl_use_cg", "jac_diag", 1300, steps=1, eps=1e-15,
               coefficient="tl_coefficient_inverse_density")
    assert log["solve"][0][1] > 1024
