"""The coarse levels of the multigrid cycle as one launch (k_mg_coarse).

It computes each level with the arithmetic of the launch-a-level kernels, so
whatever levels, block sizes and tails it takes, and whether it ran or gave
up, a run must give the same bits as with MPS_AMD_MG_COARSE=0.
"""
import threading

import numpy as np
import pytest

from mps_amd import capi, configs

pytestmark = pytest.mark.gpu

FIELDS = ("type", "pos", "vel", "p", "ndr", "bc", "pmin")
FP64, MIXED = capi.MPS_PREC_FP64, capi.MPS_PREC_MIXED


def _scene(dim, *n):
    l0 = 0.01 if dim == 2 else 0.02
    if dim == 2:
        nx, ny = n
        tank = (2 * nx * l0, (ny + 8) * l0)
        sc = configs.lattice_2d(l0, tank, (0.0, nx * l0), (0.0, ny * l0), 2, 2)
        s = configs.dambreak_settings(l0, 4e-4, 1.0)
    else:
        nx, ny, nz = n
        tank = (2 * nx * l0, (ny + 6) * l0, nz * l0)
        sc = configs.lattice_3d(l0, tank, (0.0, nx * l0), (0.0, ny * l0), (0.0, nz * l0), 2, 2)
        s = configs.dambreak_settings(l0, 2e-4, 1.0, dim=3)
        s.domain_z = (-0.1, tank[2] + 0.1)
    s.domain_x, s.domain_y = (-0.1, tank[0] + 0.1), (-0.1, tank[1] + 0.1)
    vel = np.zeros_like(sc.pos)
    fluid = sc.type == configs.FLUID
    vel[fluid, :2] = 0.05 * np.random.default_rng(sum(n)).standard_normal((int(fluid.sum()), 2))
    return s, configs.Scene(sc.type, sc.pos, vel)


def _run(members, precision, monkeypatch, coarse, steps=3, fine=None, **opt):
    monkeypatch.delenv("MPS_AMD_MG_COARSE", raising=False)
    monkeypatch.delenv("MPS_AMD_MG_FINE", raising=False)
    if coarse is not None:
        monkeypatch.setenv("MPS_AMD_MG_COARSE", coarse)
    if fine:
        monkeypatch.setenv("MPS_AMD_MG_FINE", fine)
    sim = capi.Simulation(members) if len(members) > 1 else capi.Simulation(*members[0])
    sim.set_solver(precision=precision, tolerance=1e-12, warm_start=True, preconditioner=capi.MPS_PRECOND_MULTIGRID,
                   **opt)
    sim.load_initial_state()
    its = []
    for _ in range(steps):
        sim.step()
        its.append(sim.solver_stats()["iterations"])
    st = sim.state()
    sim.close()
    return its, st


def _same(a, b):
    assert a[0] == b[0]
    for k in FIELDS:
        assert (a[1][k] == b[1][k]).all(), k


# rows just above the preconditioner's least, three to five coarse levels;
# caps of workgroups that leave the finest levels to launches (12: the last
# two alone) or give a block more rows
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("dim,n", [(2, (110, 80)), (2, (251, 139)), (2, (502, 403)), (3, (22, 20, 21)),
                                   (3, (41, 30, 33))])
def test_same_bits_as_a_launch_a_level(dim, n, precision, monkeypatch):
    m = [_scene(dim, *n)]
    want = _run(m, precision, monkeypatch, "0")
    assert max(want[0]) > 0
    for coarse in (None, "60", "12"):
        _same(_run(m, precision, monkeypatch, coarse), want)


@pytest.mark.parametrize("opt", [dict(fine="additive"), dict(use_graph=False)], ids=["additive", "no_graph"])
def test_same_bits_with_options(opt, monkeypatch):
    m = [_scene(2, 251, 139)]
    _same(_run(m, MIXED, monkeypatch, None, **opt), _run(m, MIXED, monkeypatch, "0", **opt))


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_ensemble(precision, monkeypatch):
    """Scenes of different sizes, one of a few rows: their levels share rows
    of the coarse matrices' arrays, never entries."""
    m = [_scene(2, 120, 90), _scene(2, 60, 61), _scene(2, 9, 7)]
    _same(_run(m, precision, monkeypatch, None), _run(m, precision, monkeypatch, "0"))


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_a_wait_given_up_solves_by_launches(precision, monkeypatch):
    """A wait of one poll fails at once: the launch ends, marks the solve, and
    the solve is done over a launch a level."""
    m = [_scene(2, 110, 80)]
    _same(_run(m, precision, monkeypatch, "256,1"), _run(m, precision, monkeypatch, "0"))


def test_handles_in_threads(monkeypatch):
    """Handles that together ask for more workgroups than run at once: those
    that do not get them solve by launches."""
    m = [_scene(2, 251, 139)]
    want = _run(m, MIXED, monkeypatch, "0", steps=4)
    monkeypatch.delenv("MPS_AMD_MG_COARSE", raising=False)
    got, sims = [None] * 4, []
    for k in range(4):
        sim = capi.Simulation(*m[0])
        sim.set_solver(precision=MIXED, tolerance=1e-12, warm_start=True,
                       preconditioner=capi.MPS_PRECOND_MULTIGRID)
        sim.load_initial_state()
        sims.append(sim)

    def work(k):
        its = []
        for _ in range(4):
            sims[k].step()
            its.append(sims[k].solver_stats()["iterations"])
        got[k] = its, sims[k].state()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for sim, g in zip(sims, got):
        _same(g, want)
        sim.close()
