"""The resident CG (the whole Jacobi-scaled solve of a small or middle system
in one launch) gives the bits of the launch-per-kernel CG: it takes the same
rows per block, the same sums in the same order.  So every comparison here is
exact."""
import numpy as np
import pytest

from mps_amd import capi, configs

pytestmark = pytest.mark.gpu

FIELDS = ("type", "pos", "vel", "p", "ndr", "bc", "pmin")


def _flow(sc, seed):
    rng = np.random.default_rng(seed)
    vel = np.zeros_like(sc.pos)
    fl = sc.type == configs.FLUID
    vel[fl, :2] = 0.05 * rng.standard_normal((int(fl.sum()), 2))
    return configs.Scene(sc.type, sc.pos, vel)


def _scene_2d(nx, ny, radius, tank=None):
    l0 = 0.01
    tank = tank or (2 * nx * l0, (ny + 8) * l0)
    sc = configs.lattice_2d(l0, tank, (0.0, nx * l0), (0.0, ny * l0), 2, 2)
    s = configs.dambreak_settings(l0, 4e-4, 1.0)
    s.domain_x, s.domain_y = (-0.1, tank[0] + 0.1), (-0.1, tank[1] + 0.1)
    s.ratio_pressure = s.ratio_surface = radius
    return s, _flow(sc, nx + ny)


def _scene_3d(nx, ny, nz):
    l0 = 0.02
    tank = (2 * nx * l0, (ny + 6) * l0, nz * l0)
    sc = configs.lattice_3d(l0, tank, (0.0, nx * l0), (0.0, ny * l0), (0.0, nz * l0), 2, 2)
    s = configs.dambreak_settings(l0, 2e-4, 1.0, dim=3)
    s.domain_x, s.domain_y, s.domain_z = (-0.1, tank[0] + 0.1), (-0.1, tank[1] + 0.1), (-0.1, tank[2] + 0.1)
    return s, _flow(sc, nx + ny + nz)


def _run(members, monkeypatch, env, steps=4, precision=capi.MPS_PREC_FP64, tol=1e-12, **opt):
    for k in ("MPS_AMD_CG_RESIDENT", "MPS_AMD_CG_RESIDENT_HALO"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    sim = capi.Simulation(members) if isinstance(members, list) else capi.Simulation(*members)
    sim.set_solver(precision=precision, tolerance=tol, **opt)
    sim.load_initial_state()
    its = []
    for _ in range(steps):
        sim.step()
        its.append(sim.solver_stats())
    st, counters = sim.state(), sim.debug_counters()
    sim.close()
    return st, its, counters


def _same(a, b):
    for k in FIELDS:
        assert (a[0][k] == b[0][k]).all(), k
    assert a[1] == b[1]


# one block with few rows; one full block and a little more; the tile edge
# from below; several blocks at both row widths; 3D anchors; one row of cells
# wider than a block
SCENES = {
    "tiny": lambda: _scene_2d(6, 7, 2.1),
    "one_block": lambda: _scene_2d(17, 26, 2.1),
    "two_blocks": lambda: _scene_2d(20, 30, 2.1),
    "wide_rows": lambda: _scene_2d(41, 53, 3.1),
    "long_row": lambda: _scene_2d(900, 9, 2.1),
    "many_blocks": lambda: _scene_2d(151, 203, 2.1),
    "3d": lambda: _scene_3d(9, 11, 8),
    "3d_blocks": lambda: _scene_3d(23, 19, 21),
}


@pytest.mark.parametrize("precision", [capi.MPS_PREC_FP64, capi.MPS_PREC_MIXED])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_resident_matches_launches(name, precision, monkeypatch):
    scene = SCENES[name]()
    on = _run(scene, monkeypatch, {}, precision=precision, warm_start=True)
    off = _run(scene, monkeypatch, {"MPS_AMD_CG_RESIDENT": "0"}, precision=precision, warm_start=True)
    _same(on, off)
    # the resident path ran: it enqueues no iteration past convergence, the
    # chunks round up to even lengths
    assert on[2]["cg_launched"] == sum(x["iterations"] for x in on[1])
    assert off[2]["cg_launched"] > on[2]["cg_launched"]


@pytest.mark.parametrize("precision", [capi.MPS_PREC_FP64, capi.MPS_PREC_MIXED])
def test_resident_ensemble_and_direct_launch(precision, monkeypatch):
    members = [(m[0], m[1]) for m in configs.ensemble_members(seed=7, count=7, l0_choices=(0.02, 0.015, 0.01))]
    on = _run(members, monkeypatch, {}, precision=precision)
    direct = _run(members, monkeypatch, {}, precision=precision, use_graph=False)
    off = _run(members, monkeypatch, {"MPS_AMD_CG_RESIDENT": "0"}, precision=precision)
    _same(on, off)
    _same(on, direct)


def test_resident_at_machine_epsilon_and_under_a_cap(monkeypatch):
    """Restarts from the iterate (machine epsilon) and an iteration cap."""
    scene = _scene_2d(41, 53, 3.1)
    for opt in (dict(tol=float(np.finfo(float).eps)), dict(tol=1e-12, max_iterations=7)):
        on = _run(scene, monkeypatch, {}, **opt)
        off = _run(scene, monkeypatch, {"MPS_AMD_CG_RESIDENT": "0"}, **opt)
        _same(on, off)


@pytest.mark.parametrize("precision", [capi.MPS_PREC_FP64, capi.MPS_PREC_MIXED])
@pytest.mark.parametrize("halo", ["0", "150"])
def test_resident_gives_up_and_the_launches_take_over(halo, precision, monkeypatch):
    """Blocks whose halo exceeds the limit leave at once, tell the others, and
    the solve starts again by launches (at 150 only some blocks exceed it)."""
    scene = _scene_2d(41, 53, 2.1)
    gave_up = _run(scene, monkeypatch, {"MPS_AMD_CG_RESIDENT_HALO": halo}, precision=precision, warm_start=2)
    off = _run(scene, monkeypatch, {"MPS_AMD_CG_RESIDENT": "0"}, precision=precision, warm_start=2)
    _same(gave_up, off)


def test_two_handles_share_the_chip(monkeypatch):
    """Handles stepped from two threads: launches that together exceed the
    chip run by kernels, and every trajectory keeps its solo bits."""
    import threading

    scene = _scene_2d(301, 253, 2.1)  # 149 blocks each
    want = _run(scene, monkeypatch, {"MPS_AMD_CG_RESIDENT": "0"}, steps=3)
    monkeypatch.delenv("MPS_AMD_CG_RESIDENT", raising=False)
    out = [None, None]

    def work(i):
        sim = capi.Simulation(*scene)
        sim.set_solver(tolerance=1e-12)
        sim.load_initial_state()
        sim.run_steps(3)
        out[i] = sim.state()
        sim.close()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for st in out:
        for k in FIELDS:
            assert (st[k] == want[0][k]).all(), k
