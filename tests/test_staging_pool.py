"""The buffers that calls keep (openradioss_amd/csrc/or_staging.h) on the CPU, with a counting allocator:
large workspaces push out no host buffers, limits hold, memory running out gives the idle buffers
up, and a buffer belongs to one call at a time.  The
threads that share a transfer: a helper without a buffer leaves its share to the others.  Built here from tests/stage_check.cpp with g++."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stage") / "libstage_check.so")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Werror", "-fPIC", "-shared", "-pthread",
                           os.path.join(HERE, "stage_check.cpp"), "-o", out])
    return C.CDLL(out)


@pytest.mark.parametrize("case", ["pool_keeps_host_buffers_beside_workspaces", "pool_limit_drops_the_oldest",
                                  "pool_frees_idle_buffers_when_memory_runs_out"])
def test_pool(check, case):
    line = getattr(check, case)()
    assert line == 0, f"stage_check.cpp:{line}"


def test_pool_with_threads(check):
    line = check.pool_threads(8, 2000)
    assert line == 0, f"stage_check.cpp:{line}"


@pytest.mark.parametrize("threads,items", [(1, 0), (1, 3), (6, 1), (6, 5), (6, 400)])
def test_team_takes_every_item_once(check, threads, items):
    line = check.team_takes_every_item_once(threads, items)
    assert line == 0, f"stage_check.cpp:{line}"


def test_team_reports_errors(check):
    line = check.team_reports_errors()
    assert line == 0, f"stage_check.cpp:{line}"
