"""Resident launches that the device refuses, or that are given up because not all
of their blocks came onto the device: the solve goes on from where it stands with
the kernels launched one by one, at the start of a phase or between two launches
of one, and gives bitwise what it gives otherwise (Chebyshev's residual norms
within 1e-10, the order of at most 2^21 positive terms). The host closes the
launches before they begin, or has them wait for a millisecond only beside another
stream. Launches that end in the middle, for want of a block, return an
error, and the chunk solves again afterwards."""
import os
import subprocess
import sys
import textwrap

import numpy as np
import pytest
import torch

from _pairs import setup
from tealeaf_opencl_amd import decks

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def tuning(hiplib):
    yield
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, 1)


CASES = [  # grid, solver, preconditioner, presteps, smoothing steps, cap
    (10, 10, "cg", "jac_diag", 6, 1, 30),  # one block: a grid of none is refused
    (515, 509, "cg", "jac_block", 20, 1, 1300),
    (1100, 1000, "cg", "jac_diag", 20, 1, 1100),
    (200, 148, "jacobi", "none", 20, 1, 1501),
    (515, 509, "chebyshev", "none", 20, 1, 20 + 1024 + 101),
    (515, 509, "chebyshev", "jac_block", 21, 1, 20 + 1024 + 102),
    (1100, 1000, "chebyshev", "jac_diag", 20, 1, 20 + 1024 + 30),
    (515, 509, "ppcg", "jac_diag", 20, 10, 20 + 85 + 20),
    (1100, 1000, "ppcg", "jac_block", 20, 7, 20 + 113 + 11),
]


@pytest.mark.parametrize("at", [1, 2, 3])
@pytest.mark.parametrize("nx,ny,solver,prec,presteps,inner,cap", CASES)
def test_launch_left(hiplib, tmp_path, nx, ny, solver, prec, presteps, inner, cap, at):
    """`at`: the first launch that is left, of the deck's two timesteps."""
    deck = decks.write_deck(str(tmp_path / "t.in"), nx, ny, decks.seeded_states(2, 2, True),
                            solver="tl_use_" + solver, preconditioner=prec, end_step=2, eps=1e-300, max_iters=cap,
                            dt=4e3, coefficient="tl_coefficient_inverse_density",
                            extra=["tl_ppcg_inner_steps=%d" % inner, "tl_ch_cg_presteps=%d" % presteps,
                                   "tl_ch_cg_epslim=1.0e300", "end_time=1.0e9"])
    ran = hiplib.run_deck(deck, tmp_path / "ran.log")
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, at + 1)
    left = hiplib.run_deck(deck, tmp_path / "left.log")
    assert left["summary"] == ran["summary"]
    a, b = np.array(left["solve"], float), np.array(ran["solve"], float)
    assert np.array_equal(np.delete(a, 2, 1), np.delete(b, 2, 1), equal_nan=True), (a, b)
    tol = 1e-10 if solver == "chebyshev" else 0.0
    assert np.array_equal(np.isnan(a[:, 2]), np.isnan(b[:, 2]))
    assert not np.any(np.abs(a[:, 2] - b[:, 2]) > tol * b[:, 2]), (a, b)
    assert [x[1] for x in left["solve"]] == [cap] * 2


@pytest.mark.parametrize("nx,ny,solver,prec,presteps,inner,cap", CASES[1:])
def test_short_wait_beside_another_stream(hiplib, tmp_path, nx, ny, solver, prec, presteps, inner, cap):
    """Matrix products of some 10 ms each hold the device while launches wait
    for a millisecond: whether a launch begins in time or is left, the deck
    gives the same."""
    deck = decks.write_deck(str(tmp_path / "t.in"), nx, ny, decks.seeded_states(2, 2, True),
                            solver="tl_use_" + solver, preconditioner=prec, end_step=2, eps=1e-300, max_iters=cap,
                            dt=4e3, coefficient="tl_coefficient_inverse_density",
                            extra=["tl_ppcg_inner_steps=%d" % inner, "tl_ch_cg_presteps=%d" % presteps,
                                   "tl_ch_cg_epslim=1.0e300", "end_time=1.0e9"])
    ran = hiplib.run_deck(deck, tmp_path / "ran.log")
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, -2)
    a = torch.ones(8192, 8192, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(8):
            b = a @ a
    left = hiplib.run_deck(deck, tmp_path / "left.log")
    s.synchronize()
    assert float(b[0, 0]) == 8192.0
    assert left["summary"] == ran["summary"]
    assert [x[1] for x in left["solve"]] == [x[1] for x in ran["solve"]]


def test_left_for_good(hiplib, tmp_path):
    """After a launch was left the kernels are launched one by one (and their
    times sampled), until the key is set again."""
    c = hiplib.Chunk(515, 509, 1, 3)
    setup(c, seed=2, coef=2)
    samples = []
    for value in (2, None, 1):
        if value is not None:
            hiplib.set_tuning(hiplib.TUNE_RESIDENT, value, chunk=c)
        c.set_field()
        c.common_init(2, 0.004)
        res = c.solve_refined(0, tol=1e-10, max_iters=5000)
        assert res["converged"]
        samples.append(res["k_samples"])
    assert samples[0] > 0 and samples[1] > 0 and samples[2] == 0
    c.close()


@pytest.mark.parametrize("at", [1, 2, 3])
@pytest.mark.parametrize("inner", [0, 6])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", [(515, 509), (1100, 1000)])
def test_refined_left(hiplib, nx, ny, precision, inner, at):
    """The refined solves meet their tolerance, by the library's own residual and
    norm kernels (1 % for the norms' rounding)."""
    c = hiplib.Chunk(nx, ny, 1, 3)
    setup(c, seed=2, coef=2)
    c.calc_residual()
    r0 = c.calc_2norm(1) ** 0.5
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, at + 1, chunk=c)
    if inner:
        res = c.solve_refined_ppcg(precision, tol=1e-10, max_iters=20000, presteps=20, inner_steps=inner)
    else:
        res = c.solve_refined(precision, tol=1e-10, max_iters=20000)
    assert res["converged"], res
    c.calc_residual()
    r = c.calc_2norm(1) ** 0.5
    assert r <= 1.01e-10 * r0, (r / r0, res)
    assert abs(res["rel_residual"] - r / r0) <= 1e-2 * 1e-10
    if inner:
        assert res["inner_iterations"] == inner * (res["iterations"] - 20)
    c.close()


@pytest.mark.parametrize("solver", ["cg", "jacobi", "chebyshev", "ppcg"])
@pytest.mark.parametrize("nx,ny", [(515, 509), (1100, 1000)])
def test_stuck(hiplib, tmp_path, nx, ny, solver):
    if solver == "jacobi" and nx > 1024:
        pytest.skip("no Jacobi on tall blocks")
    deck = decks.write_deck(str(tmp_path / "t.in"), nx, ny, decks.seeded_states(2, 2, True),
                            solver="tl_use_" + solver, end_step=1, eps=1e-300, max_iters=40,
                            extra=["tl_ppcg_inner_steps=4", "tl_ch_cg_presteps=20", "tl_ch_cg_epslim=1.0e300"])
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, -1)
    with pytest.raises(hiplib.TealeafError, match="waited too long"):
        hiplib.run_deck(deck, tmp_path / "t.log")


@pytest.mark.parametrize("inner", [0, 6])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny", [(515, 509), (1100, 1000)])
def test_stuck_and_again(hiplib, nx, ny, precision, inner):
    def solve(c):
        setup(c, seed=2, coef=2)
        if inner:
            c.solve_refined_ppcg(precision, tol=1e-10, max_iters=5000, presteps=20, inner_steps=inner)
        else:
            c.solve_refined(precision, tol=1e-10, max_iters=5000)
        return c.get_field("u")

    c, fresh = hiplib.Chunk(nx, ny, 1, 3), hiplib.Chunk(nx, ny, 1, 3)
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, -1, chunk=c)
    with pytest.raises(hiplib.TealeafError, match="waited too long"):
        solve(c)
    hiplib.set_tuning(hiplib.TUNE_RESIDENT, 1, chunk=c)
    assert np.array_equal(solve(c), solve(fresh))
    c.close()
    fresh.close()


def test_two_processes(hiplib, tmp_path):
    """Two processes that solve on the one GPU at the same time, each launch of
    which holds every compute unit, give what each gives alone."""
    code = textwrap.dedent("""
        import sys
        import numpy as np
        import tealeaf_opencl_amd as tl
        from tealeaf_opencl_amd import decks
        deck = decks.write_deck(sys.argv[1] + ".in", 1024, 1024, decks.seeded_states(2, 2, True), end_step=20,
                                eps=1e-300, max_iters=200, preconditioner="jac_diag")
        print("ready", flush=True)
        sys.stdin.readline()
        print(repr(tl.run_deck(deck, sys.argv[1] + ".log")["summary"]), flush=True)
    """)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    procs = [subprocess.Popen([sys.executable, "-c", code, str(tmp_path / str(k))], stdin=subprocess.PIPE,
                              stdout=subprocess.PIPE, text=True, cwd=root) for k in range(2)]
    for p in procs:
        assert p.stdout.readline() == "ready\n"
    for p in procs:
        p.stdin.write("\n")
        p.stdin.flush()
    out = [p.communicate(timeout=100)[0] for p in procs]
    assert [p.returncode for p in procs] == [0, 0]
    deck = decks.write_deck(str(tmp_path / "alone.in"), 1024, 1024, decks.seeded_states(2, 2, True), end_step=20,
                            eps=1e-300, max_iters=200, preconditioner="jac_diag")
    alone = repr(hiplib.run_deck(deck, tmp_path / "alone.log")["summary"])
    assert [o.strip() for o in out] == [alone, alone]
