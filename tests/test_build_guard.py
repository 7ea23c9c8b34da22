"""The build refuses a matrix-core kernel that spills vector registers."""
import pytest

from fringe_amd import build

REPORT = """solve.hpp:740:0: remark: Function Name: {0} [-Rpass-analysis=kernel-resource-usage]
solve.hpp:740:0: remark:     VGPRs: 128 [-Rpass-analysis=kernel-resource-usage]
solve.hpp:740:0: remark:     SGPRs Spill: 40 [-Rpass-analysis=kernel-resource-usage]
solve.hpp:740:0: remark:     VGPRs Spill: {1} [-Rpass-analysis=kernel-resource-usage]
"""


def test_report_of_spills():
    report = REPORT.format("first", 0) + REPORT.format("second", 3) + REPORT.format("third", 0)
    assert build.spilling_kernels(report) == ([("second", 3)], 3)
    with pytest.raises(RuntimeError):
        build.spilling_kernels(report + "remark: Function Name: fourth\n")


@pytest.mark.parametrize("spilled,stderr", [(True, REPORT.format("kernel", 2)), (True, ""), (False, REPORT.format("kernel", 0))])
def test_build_fails_on_a_spill(monkeypatch, spilled, stderr):
    """Also when the compiler reports no kernel at all; sources without matrix-core
    kernels are not looked at."""
    calls = []

    class Done:
        returncode, stdout = 0, ""

    def run(cmd, **kw):
        calls.append(cmd)
        d = Done()
        d.stderr = stderr
        return d

    monkeypatch.setattr(build.subprocess, "run", run)
    for name in build.NO_SPILL:
        if spilled:
            with pytest.raises(RuntimeError):
                build._compile(f"csrc/{name}")
        else:
            build._compile(f"csrc/{name}")
        assert build.RESOURCES[0] in calls[-1]
    build._compile("csrc/solvers.hip")
    assert build.RESOURCES[0] not in calls[-1]


def test_guarded_sources_exist():
    names = {s.rsplit("/", 1)[-1] for s in build.sources()}
    assert set(build.NO_SPILL) <= names
