"""The fine level of the multigrid cycle in the coarse launch: the bits of a
launch a level, whichever of its rows, workgroups and entries it takes."""
import pytest

from mps_amd import capi
from test_gpu_coarse import FP64, MIXED, _run, _same, _scene

pytestmark = pytest.mark.gpu


# the fewest rows with a level above the tail; rows that end inside and at a
# wavefront; several scenes; 3D; rows too many for the launch to hold
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("dim,n", [(2, (90, 71)), (2, (96, 64)), (2, (203, 207)), (2, (350, 262)), (2, (420, 330)),
                                   (3, (27, 25, 26))])
def test_same_bits(dim, n, precision, monkeypatch):
    m = [_scene(dim, *n)]
    want = _run(m, precision, monkeypatch, "0")
    assert max(want[0]) > 0
    for coarse in (None, "150"):
        _same(_run(m, precision, monkeypatch, coarse), want)


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_wide_rows(precision, monkeypatch):
    """Some slices hold more entries a row than the launch keeps: a cluster of
    particles pressed together in a scene of ordinary rows."""
    s, sc = _scene(2, 140, 120)
    c = (sc.pos[:, 0] < 0.25) & (sc.pos[:, 1] < 0.25) & (sc.type == 0)
    sc.pos[c, 0] *= 0.8
    m = [(s, sc)]
    _same(_run(m, precision, monkeypatch, None), _run(m, precision, monkeypatch, "0"))


def test_grows(monkeypatch):
    """One handle whose row count changes from step to step."""
    m = [_scene(2, 130, 101)]
    a = _run(m, MIXED, monkeypatch, None, steps=12)
    _same(a, _run(m, MIXED, monkeypatch, "0", steps=12))
