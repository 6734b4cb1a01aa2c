"""Field transfers (tl_field_set / tl_field_get), which cross through pinned
slots of 2^17 values: the image comes back bit for bit, whole slots, remainders
and images of less than a slot, with rows across the slots' edges, and no other
field changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,hd", [(1, 1, 1), (10, 10, 2), (254, 510, 1), (254, 1022, 1), (255, 1022, 1),
                                      (1000, 701, 2), (70000, 5, 1), (3, 60000, 1)])
def test_round_trip(hiplib, nx, ny, hd):
    c = hiplib.Chunk(nx, ny, hd, 1)
    rng = np.random.default_rng(5)
    a = rng.standard_normal((ny + 2 * hd, nx + 2 * hd))
    b = rng.standard_normal(a.shape)
    c.put_field("density", a)
    c.put_field("energy1", b)
    assert np.array_equal(c.get_field("density"), a)
    assert np.array_equal(c.get_field("energy1"), b)
    assert not c.get_field("u").any()
    c.put_field("density", b)
    assert np.array_equal(c.get_field("density"), b)
    c.close()
