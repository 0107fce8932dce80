"""Downloads through the pinned staging: a state in one go, and a large one in
turns of 2 MiB pieces copied out by several threads."""
import ctypes

import numpy as np
import pytest

from mps_amd import capi, configs

pytestmark = pytest.mark.gpu


def _sim(nx, ny):
    l0 = 0.01
    tank = (2 * nx * l0, (ny + 8) * l0)
    sc = configs.lattice_2d(l0, tank, (0.0, nx * l0), (0.0, ny * l0), 2, 2)
    s = configs.dambreak_settings(l0, 4e-4, 1.0)
    s.domain_x, s.domain_y = (-0.1, tank[0] + 0.1), (-0.1, tank[1] + 0.1)
    vel = np.zeros_like(sc.pos)
    fluid = sc.type == configs.FLUID
    vel[fluid, :2] = 0.05 * np.random.default_rng(nx).standard_normal((int(fluid.sum()), 2))
    sim = capi.Simulation(s, configs.Scene(sc.type, sc.pos, vel))
    sim.set_solver(precision=capi.MPS_PREC_MIXED, tolerance=1e-6, preconditioner=capi.MPS_PRECOND_MULTIGRID)
    sim.load_initial_state()
    sim.step(is_export=True)
    return sim


def _slot(sim):
    """The same state through the export slot's own pinned buffers."""
    n = sim.n
    out = [ctypes.c_void_p() for _ in range(6)]
    sim._check(sim.L.mps_snapshot_begin(sim.h, 0))
    sim._check(sim.L.mps_snapshot_end(sim.h, 0, *[ctypes.byref(o) for o in out]))

    def arr(p, t, shape):
        c = np.prod(shape) * np.dtype(t).itemsize
        return np.frombuffer((ctypes.c_char * int(c)).from_address(p.value), t).reshape(shape).copy()

    return dict(type=arr(out[0], np.int8, (n,)), pos=arr(out[1], np.float64, (n, 3)),
                vel=arr(out[2], np.float64, (n, 3)), p=arr(out[3], np.float64, (n,)),
                ndr=arr(out[4], np.float64, (n,)), bc=arr(out[5], np.int8, (n,)))


# a few particles; either side of 2 MiB in all (31,775 particles); one slot of
# the staging; more pieces than slots with a ragged last one
@pytest.mark.parametrize("nx,ny", [(9, 7), (155, 180), (160, 185), (333, 301), (701, 611)])
def test_state_is_the_export_slots(nx, ny):
    sim = _sim(nx, ny)
    want = _slot(sim)
    for _ in range(2):
        got = sim.state()
        for k, v in want.items():
            assert (got[k] == v).all(), k
    sim.close()


def test_arrays_one_at_a_time():
    sim = _sim(160, 185)
    want = _slot(sim)
    for k, (at, shape) in dict(type=(0, ()), pos=(1, (3,)), vel=(2, (3,)), p=(3, ()), ndr=(4, ()), bc=(5, ())).items():
        got = np.zeros((sim.n,) + shape, want[k].dtype)
        args = [None] * 6
        args[at] = got.ctypes.data_as(ctypes.c_void_p)
        sim._check(sim.L.mps_download(sim.h, *args))
        assert (got == want[k]).all(), k
    sim.close()


# either side of 4 MiB in all (63,550 particles): one copy, several threads
@pytest.mark.parametrize("nx,ny,large", [(225, 264, False), (225, 265, True)])
def test_state_where_the_threads_start(nx, ny, large):
    sim = _sim(nx, ny)
    assert (66 * sim.n >= 4 << 20) == large
    want = _slot(sim)
    for _ in range(2):
        got = sim.state()
        for k, v in want.items():
            assert (got[k] == v).all(), k
    sim.close()
