"""Prefix sums at the edges of their forms (one launch up to 16 tiles of 2,048
elements, two up to 2,048 tiles, three beyond), through the bucket build, whose
counts are one a cell and one for the ghosts."""
import numpy as np
import pytest

from mps_amd import capi, configs
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


# cells: one element below, at and above a tile; 16 tiles; 2,048 tiles
@pytest.mark.parametrize("nx,ny", [(31, 66), (23, 89), (32, 64), (217, 151), (128, 256), (2047, 2049), (2048, 2048)])
def test_bucket_lists(nx, ny):
    l0 = 0.01
    rng = np.random.default_rng(nx)
    s = configs.dambreak_settings(l0, 1e-4, 1.0)
    length = max(s.ratio_pressure, s.ratio_viscosity, s.ratio_surface) * l0
    size = np.array([(nx - 2.5) * length, (ny - 2.5) * length])
    s.domain_x, s.domain_y = (0.0, float(size[0])), (0.0, float(size[1]))
    n = 20000
    pos = np.zeros((n, 3))
    pos[:, :2] = rng.uniform(0.0, 1.0, (n, 2)) * size
    pos[:4, :2] = np.array([[0, 0], [1, 0], [0, 1], [1, 1]]) * size * 0.999999
    sc = configs.Scene(np.full(n, configs.FLUID, np.int8), pos, np.zeros((n, 3)))
    o, g = Oracle(s, sc), capi.Simulation(s, sc)
    o.set_neighbors()
    want, got = o.bucket(), g.bucket()
    g.close()
    assert tuple(got["dims"]) == (3 * nx * ny, nx, ny, 3)  # the empty layers of a plane are not counted
    for k in ("dims", "first", "last", "next"):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
