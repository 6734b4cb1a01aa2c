"""Grids beyond the resident solver whose tile columns go in groups, one per
XCD (make_ext): every tile is visited once. The field summary and the dot
products against numpy, over grids with whole groups, a column short of them, a
partly filled last column and tile row, and one column too many for groups
(row by row). All sums run over n positive terms of at most n roundings, hence
n * 2^-53 relative."""
import numpy as np
import pytest

from _pairs import setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2048, 2100), (3001, 2999), (2945, 1601), (4096, 1040), (4097, 1040), (500, 9000)])
def test_every_tile_once(hiplib, nx, ny):
    c = hiplib.Chunk(nx, ny, 1, 1)
    setup(c, seed=2, coef=2)
    rng = np.random.default_rng(3)
    a = rng.uniform(0.5, 1.5, (ny + 2, nx + 2))
    c.put_field("r", a)
    r = a[1:-1, 1:-1]
    n = nx * ny
    assert abs(c.calc_2norm(1) - float((r * r).sum())) <= n * 2.0 ** -53 * float((r * r).sum())
    rho = c.interior(c.get_field("density"))
    vol, mass = c.field_summary()[:2]
    area = c.interior(c.get_field("volume"))
    for got, want in ((vol, area.sum()), (mass, (area * rho).sum())):
        assert abs(got - want) <= n * 2.0 ** -53 * want
    c.close()
