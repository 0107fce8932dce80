"""The build compiles again when its flags change, and refuses kernels that
must not spill scalar registers and do (the compiler is stood in for)."""
import types

import pytest

from mps_amd import build

REMARKS = """resident.hip:1:1: remark: Function Name: _Z16k_solve_resident{0} [-Rpass-analysis=kernel-resource-usage]
resident.hip:1:1: remark:     TotalSGPRs: 106 [-Rpass-analysis=kernel-resource-usage]
resident.hip:1:1: remark:     SGPRs Spill: {1} [-Rpass-analysis=kernel-resource-usage]
resident.hip:9:1: remark: Function Name: _Z7k_other [-Rpass-analysis=kernel-resource-usage]
resident.hip:9:1: remark:     SGPRs Spill: 7 [-Rpass-analysis=kernel-resource-usage]
"""


@pytest.fixture
def compiler(tmp_path, monkeypatch):
    ran = []

    def run(cmd, **kw):
        ran.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return types.SimpleNamespace(returncode=0, stdout="", stderr=ran_stderr[0])

    ran_stderr = [REMARKS.format("Id", 0)]
    monkeypatch.setattr(build, "BUILD", str(tmp_path))
    monkeypatch.setattr(build.subprocess, "run", run)
    return ran, ran_stderr


def test_changed_flags_compile_again(compiler, monkeypatch):
    ran, _ = compiler
    for _ in range(2):
        assert build._compile("grid.hip", False)[1] is None
    assert len(ran) == 1
    monkeypatch.setattr(build, "FLAGS", build.FLAGS + ["-O2"])
    for _ in range(2):
        assert build._compile("grid.hip", False)[1] is None
    assert len(ran) == 2 and "-O2" in ran[1]


def test_scalar_spills_fail_the_build(compiler):
    ran, stderr = compiler
    assert build._compile("resident.hip", False)[1] is None
    for text in (REMARKS.format("Id", 2), REMARKS.format("Id", 0) + REMARKS.format("If", 12), "", "warning: x"):
        stderr[0] = text
        assert "k_solve_resident" in build._compile("resident.hip", True)[1]
        assert "k_solve_resident" in build._compile("resident.hip", False)[1], "a refused object stays refused"
    stderr[0] = REMARKS.format("Id", 0)
    assert build._compile("resident.hip", False)[1] is None
