"""The start of the resident solver's launches: block 0 stores the solver state
at a launch's end, and every block reads it at the start, so a launch of few
Chebyshev iterations, whose blocks exchange with their neighbours only, has to
wait until every block has begun. Long grids (blocks up to 250 apart) with one
to five iterations after the switch, or in the second launch, alone and while
another stream keeps the compute units busy, bitwise the same iterations launched
one by one (a profiler_on run). 1e-10 for the norms: the order of at most 2^21
positive terms."""
import pytest
import torch

from test_gpu_resident import both

pytestmark = pytest.mark.gpu


def cheby(hiplib, tmp_path, nx, ny, prec, cap):
    log = both(hiplib, tmp_path, nx, ny, "tl_use_chebyshev", prec, cap, steps=1, eps=1e-300, norm=1e-10, dt=4e3,
               coefficient="tl_coefficient_inverse_density",
               extra=["tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"])
    assert log["solve"][0][1] == cap


@pytest.mark.parametrize("prec", ["none", "jac_block"])
@pytest.mark.parametrize("cap", [21, 22, 25, 20 + 1024 + 1])
@pytest.mark.parametrize("nx,ny", [(4160, 64), (64, 4096), (16001, 100), (130, 16001)])
def test_short_chebyshev(hiplib, tmp_path, nx, ny, cap, prec):
    cheby(hiplib, tmp_path, nx, ny, prec, cap)


@pytest.mark.parametrize("nx,ny", [(4160, 64), (16001, 100)])
def test_short_chebyshev_beside_another_stream(hiplib, tmp_path, nx, ny):
    a = torch.ones(4096, 4096, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(40):
            b = a @ a
    cheby(hiplib, tmp_path, nx, ny, "jac_diag", 22)
    s.synchronize()
    assert float(b[0, 0]) == 4096.0
