"""Which launches a solve took.  The tests that compare a launch's bits with
those of the launches it replaces would pass as well if it never ran, so the
same scenes are run here for their counters."""
import threading

import numpy as np
import pytest

from mps_amd import capi, configs
from test_gpu_coarse import FIELDS, FP64, MIXED, _run, _same, _scene
from test_gpu_resident import SCENES, _scene_2d, _scene_3d

pytestmark = pytest.mark.gpu

PRECISIONS = pytest.mark.parametrize("precision", [FP64, MIXED])
ENV = ("MPS_AMD_MG_COARSE", "MPS_AMD_MG_FINE", "MPS_AMD_CG_RESIDENT", "MPS_AMD_CG_RESIDENT_HALO")


def _sim(members, precision, multigrid, monkeypatch, env=None, **opt):
    for k in ENV:
        monkeypatch.delenv(k, raising=False)
    for k, v in (env or {}).items():
        monkeypatch.setenv(k, v)
    sim = capi.Simulation(members) if len(members) > 1 else capi.Simulation(*members[0])
    pre = capi.MPS_PRECOND_MULTIGRID if multigrid else capi.MPS_PRECOND_JACOBI
    sim.set_solver(precision=precision, tolerance=1e-12, warm_start=True, preconditioner=pre, **opt)
    sim.load_initial_state()
    return sim


def _counts(*args, steps=2, **kw):
    sim = _sim(*args, **kw)
    for _ in range(steps):
        sim.step()
    c = sim.debug_counters()
    sim.close()
    return c


# ---- the coarse launch of the multigrid cycle


@PRECISIONS
@pytest.mark.parametrize("coarse", [None, "60", "12"])
@pytest.mark.parametrize("dim,n", [(2, (110, 80)), (2, (251, 139)), (2, (502, 403)), (3, (22, 20, 21)),
                                   (3, (41, 30, 33))])
def test_coarse_launch_runs(dim, n, coarse, precision, monkeypatch):
    c = _counts([_scene(dim, *n)], precision, True, monkeypatch, {"MPS_AMD_MG_COARSE": coarse} if coarse else None)
    assert c["coarse_cycles"] == c["cg_launched"] > 0 and c["coarse_gave_up"] == c["refused"] == 0, c


@PRECISIONS
def test_coarse_launch_runs_with_options_and_scenes(precision, monkeypatch):
    one, three = [_scene(2, 251, 139)], [_scene(2, 120, 90), _scene(2, 60, 61), _scene(2, 9, 7)]
    for c in (_counts(one, precision, True, monkeypatch, {"MPS_AMD_MG_FINE": "additive"}),
              _counts(one, precision, True, monkeypatch, use_graph=False),
              _counts(three, precision, True, monkeypatch)):
        assert c["coarse_cycles"] == c["cg_launched"] > 0, c
    c = _counts(one, precision, True, monkeypatch, {"MPS_AMD_MG_COARSE": "0"})
    assert c["coarse_cycles"] == 0 < c["cg_launched"], c


@PRECISIONS
def test_coarse_launch_gives_up(precision, monkeypatch):
    c = _counts([_scene(2, 110, 80)], precision, True, monkeypatch, {"MPS_AMD_MG_COARSE": "256,1"})
    assert c["coarse_gave_up"] == 1, c


@PRECISIONS
@pytest.mark.parametrize("dim,n,fits", [(2, (203, 207), True), (2, (420, 330), False), (3, (27, 25, 26), True)])
def test_fine_level_in_the_coarse_launch(dim, n, fits, precision, monkeypatch):
    c = _counts([_scene(dim, *n)], precision, True, monkeypatch)
    if dim == 3 and precision == MIXED:
        fits = False  # its fine level stays with its own launches
    assert c["coarse_fine_cycles"] == (c["coarse_cycles"] if fits else 0), c
    assert c["coarse_cycles"] > 0


# the fewest rows but two that take the multigrid cycle (8,192); rows that
# end at a wavefront
@PRECISIONS
@pytest.mark.parametrize("n,rows", [((85, 92), 8194), ((86, 96), 8640)])
def test_fine_level_of_the_fewest_rows(n, rows, precision, monkeypatch):
    m = [_scene(2, *n)]
    sim = _sim(m, precision, True, monkeypatch)
    sim.step()
    assert sim.solver_stats()["rows"] == rows
    sim.step()
    c = sim.debug_counters()
    sim.close()
    assert c["coarse_fine_cycles"] == c["cg_launched"] > 0, c
    _same(_run(m, precision, monkeypatch, None), _run(m, precision, monkeypatch, "0"))


@PRECISIONS
def test_fine_level_with_rows_wider_than_it_keeps(precision, monkeypatch):
    s, sc = _scene(2, 140, 120)
    c = (sc.pos[:, 0] < 0.25) & (sc.pos[:, 1] < 0.25) & (sc.type == 0)
    sc.pos[c, 0] *= 0.8
    sim = _sim([(s, sc)], precision, True, monkeypatch)
    sim.set_snapshot(True)
    sim.step()
    widest = int(np.diff(sim.pressure_system()["row_ptr"]).max())
    counts = sim.debug_counters()
    sim.close()
    assert widest > 16 and counts["coarse_fine_cycles"] == counts["cg_launched"] > 0, (widest, counts)


def test_fine_level_while_the_rows_change(monkeypatch):
    sim = _sim([_scene(2, 130, 101)], MIXED, True, monkeypatch)
    rows = set()
    for _ in range(12):
        sim.step()
        rows.add(sim.solver_stats()["rows"])
    c = sim.debug_counters()
    sim.close()
    assert len(rows) > 1 and c["coarse_fine_cycles"] == c["cg_launched"] > 0, (rows, c)


def test_coarse_launch_is_tried_again_after_it_gave_up(monkeypatch):
    """Waits of one poll: the launch gives up, and again 256 solves later."""
    m = [_scene(2, 110, 80)]
    off = _sim(m, MIXED, True, monkeypatch, {"MPS_AMD_MG_COARSE": "0"})
    sim = _sim(m, MIXED, True, monkeypatch, {"MPS_AMD_MG_COARSE": "256,1"})
    for s in (off, sim):
        s.run_steps(256)
    assert sim.debug_counters()["coarse_gave_up"] == 1
    for s in (off, sim):
        s.step()
    assert sim.debug_counters()["coarse_gave_up"] == 2
    a, b = sim.state(), off.state()
    sim.close()
    off.close()
    for k in FIELDS:
        assert (a[k] == b[k]).all(), k


def test_coarse_launch_comes_back_after_a_refusal(monkeypatch):
    """A handle whose workgroups another one holds solves by a launch a level
    then, and takes the coarse launch again once they are free."""
    m = [_scene(2, 251, 139)]
    off = _sim(m, MIXED, True, monkeypatch, {"MPS_AMD_MG_COARSE": "0"})
    sims = [_sim(m, MIXED, True, monkeypatch) for _ in range(2)]
    ts = [threading.Thread(target=s.run_steps, args=(60,)) for s in sims]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    off.run_steps(62)
    want = off.state()
    off.close()
    refused = 0
    for s in sims:
        before = s.debug_counters()
        s.run_steps(2)
        after = s.debug_counters()
        got = s.state()
        s.close()
        refused += before["refused"]
        assert after["refused"] == before["refused"] and after["coarse_gave_up"] == 0, after
        assert after["coarse_cycles"] - before["coarse_cycles"] == after["cg_launched"] - before["cg_launched"] > 0
        for k in FIELDS:
            assert (got[k] == want[k]).all(), k
    assert refused > 0


# ---- resident solves


@PRECISIONS
@pytest.mark.parametrize("name", sorted(SCENES))
def test_resident_solve_runs(name, precision, monkeypatch):
    c = _counts([SCENES[name]()], precision, False, monkeypatch)
    assert c["resident_solves"] == 2 and c["resident_gave_up"] == c["refused"] == 0, c


@PRECISIONS
def test_resident_solve_runs_with_options_and_scenes(precision, monkeypatch):
    seven = [(m[0], m[1]) for m in configs.ensemble_members(seed=7, count=7, l0_choices=(0.02, 0.015, 0.01))]
    wide = [_scene_2d(41, 53, 3.1)]
    for c in (_counts(seven, precision, False, monkeypatch),
              _counts(seven, precision, False, monkeypatch, use_graph=False),
              _counts(wide, precision, False, monkeypatch, max_iterations=7)):
        assert c["resident_solves"] == 2 and c["resident_gave_up"] == 0, c


@PRECISIONS
@pytest.mark.parametrize("halo", ["0", "150"])
def test_resident_solve_gives_up(halo, precision, monkeypatch):
    c = _counts([_scene_2d(41, 53, 2.1)], precision, False, monkeypatch, {"MPS_AMD_CG_RESIDENT_HALO": halo})
    assert c["resident_solves"] == 0 < c["resident_gave_up"], c


# 184 and 247 blocks of the 256 that a launch may take
@PRECISIONS
@pytest.mark.parametrize("n,radius", [((431, 209), 2.1), ((500, 245), 3.1)])
def test_resident_solve_of_many_blocks(n, radius, precision, monkeypatch):
    m = [_scene_2d(*n, radius)]
    got = []
    for env in ({}, {"MPS_AMD_CG_RESIDENT": "0"}):
        sim = _sim(m, precision, False, monkeypatch, env)
        sim.run_steps(2)
        got.append((sim.state(), sim.solver_stats(), sim.debug_counters()["resident_solves"]))
        sim.close()
    assert got[0][2] == 2 and got[1][2] == 0 and got[0][1] == got[1][1]
    assert got[0][1]["rows"] > 150 * 512
    for k in FIELDS:
        assert (got[0][0][k] == got[1][0][k]).all(), k


def _wide(dim, n, radius):
    s, sc = _scene_2d(*n, radius) if dim == 2 else _scene_3d(*n)
    s.ratio_pressure = s.ratio_surface = radius
    return [(s, sc)]


# rows wider than the 36 entries a thread holds: split blocks, whole ones
@PRECISIONS
@pytest.mark.parametrize("dim,n,radius", [(3, (27, 12, 12), 3.1), (2, (70, 50), 5.1), (3, (27, 16, 18), 2.9),
                                          (2, (120, 90), 5.1)])
def test_rows_wider_than_a_thread_holds(dim, n, radius, precision, monkeypatch):
    m = _wide(dim, n, radius)
    got = []
    for env in ({}, {"MPS_AMD_CG_RESIDENT": "0"}):
        sim = _sim(m, precision, False, monkeypatch, env)
        sim.set_snapshot(True)
        sim.run_steps(3)
        got.append((sim.state(), sim.solver_stats(), sim.debug_counters()["resident_solves"]))
        rp = sim.pressure_system()["row_ptr"]
        sim.close()
    assert got[0][2] == 3 and got[1][2] == 0
    assert rp[-1] > 36 * got[0][1]["rows"]
    assert got[0][1] == got[1][1]
    for k in FIELDS:
        assert (got[0][0][k] == got[1][0][k]).all(), k


# rows wider than pays (93 entries; 3D, split blocks of 4,096 rows or more 144);
# more bytes than the L2s keep in FP64 (56 entries a row are read again), not in
# mixed precision
@pytest.mark.parametrize("dim,n,radius,taken", [(2, (120, 90), 6.6, (0, 0)), (2, (70, 50), 6.6, (0, 0)),
                                                (3, (9, 11, 8), 3.1, (0, 0)), (3, (27, 16, 18), 3.1, (0, 0)),
                                                (3, (44, 28, 28), 2.9, (0, 2))])
def test_rows_too_wide_are_left_to_the_kernels(dim, n, radius, taken, monkeypatch):
    for precision, want in zip((FP64, MIXED), taken):
        c = _counts(_wide(dim, n, radius), precision, False, monkeypatch)
        assert c["resident_solves"] == want and c["resident_gave_up"] == 0, (precision, c)


def test_resident_solve_is_tried_again_after_it_gave_up(monkeypatch):
    """No halo fits: the launch gives up, and again 257 solves later."""
    m = [_scene_2d(41, 53, 2.1)]
    off = _sim(m, FP64, False, monkeypatch, {"MPS_AMD_CG_RESIDENT": "0"})
    sim = _sim(m, FP64, False, monkeypatch, {"MPS_AMD_CG_RESIDENT_HALO": "0"})
    for s in (off, sim):
        s.run_steps(257)
    assert sim.debug_counters()["resident_gave_up"] == 1
    for s in (off, sim):
        s.step()
    assert sim.debug_counters()["resident_gave_up"] == 2
    a, b = sim.state(), off.state()
    sim.close()
    off.close()
    for k in FIELDS:
        assert (a[k] == b[k]).all(), k


def test_handles_that_ask_for_more_than_the_chip(monkeypatch):
    """Two handles of 149 workgroups each step at the same time: one is
    refused at least once, and no launch gives up."""
    sims = [_sim([_scene_2d(301, 253, 2.1)], FP64, False, monkeypatch) for _ in range(2)]
    ts = [threading.Thread(target=sim.run_steps, args=(12,)) for sim in sims]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    cs = [sim.debug_counters() for sim in sims]
    for sim in sims:
        sim.close()
    assert sum(c["refused"] for c in cs) > 0, cs
    assert all(c["resident_solves"] + c["refused"] == 12 and c["resident_gave_up"] == 0 for c in cs), cs
