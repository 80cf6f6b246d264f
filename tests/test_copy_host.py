"""Large downloads where something is refused (CPU only): the control flow of
spade_amd/csrc/host_copy.hpp with a host buffer for the device."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("copy") / "copy_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", os.path.join(HERE, "native", "copy_check.cpp"), "-o", exe],
                   check=True)

    def go(scenario, nbytes):
        r = subprocess.run([exe, scenario, str(nbytes)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stderr[-300:])
        result, *numbers = r.stdout.split()
        return (result, *map(int, numbers))
    return go


@pytest.mark.parametrize("nbytes", [1, (4 << 20) + 3, (20 << 20) + 5, 67 << 20])
@pytest.mark.parametrize("scenario", ["all", "no_thread", "one_thread", "no_memory"])
def test_threads_refused(run, scenario, nbytes):
    """Whatever refuses a thread, every piece arrives and the running threads end."""
    result, equal, pieces, *_ = run(scenario, nbytes)
    assert result == "all" and equal and pieces >= 1


def test_failing_piece_is_reported(run):
    result, _, pieces, *_ = run("failing_piece", 67 << 20)
    assert result == "failed" and pieces < 17


def test_no_pinned_memory(run):
    """Refused pinned memory copies nothing and says so: the caller goes on with
    the pageable copy."""
    result, equal, pieces, *_ = run("no_slots", 20 << 20)
    assert (result, equal, pieces) == ("no_slots", 0, 0)


@pytest.mark.parametrize("scenario, helpers", [("all", 3), ("one_thread", 1), ("no_thread", 0)])
def test_the_callers_device_stays(run, scenario, helpers):
    """Helper threads set the context's device, the caller's thread keeps its own
    (another context's, where a program drives several devices), also where it
    copies a refused thread's pieces."""
    result, equal, _, entered, callers = run(scenario, 20 << 20)
    assert result == "all" and equal
    assert (entered, callers) == (helpers, 0)
