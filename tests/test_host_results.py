"""The host side of results on their way to the caller, without a GPU."""
import os
import subprocess

import pytest

from tests.cpp import build_cpp


@pytest.fixture(scope="module")
def probe():
    exe = build_cpp.build_host_results_probe()

    def run(*args, **kw):
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60, **kw)
        assert out.returncode == 0, out.stdout + out.stderr
        return out.stdout

    return run


def test_a_process_ends_after_the_threads_that_bring_results(probe):
    assert probe("exit") == "ended 1\n"


@pytest.mark.parametrize("wanted", [1, 2, 3])
def test_no_more_threads_bring_results_than_are_wanted(probe, wanted):
    assert 1 <= int(probe("threads", env=dict(os.environ, ND_HOST_THREADS=str(wanted)))) <= wanted


@pytest.mark.parametrize("files,groups,cpus", [
    ({}, "", "inf"),
    ({"cpu.max": "max 100000"}, "0::/\n", "inf"),
    ({"cpu.max": "1600000 100000"}, "0::/\n", "16"),
    # a group inside another: the smaller of the two
    ({"cpu.max": "max 100000", "a/cpu.max": "250000 100000", "a/b/cpu.max": "400000 100000"}, "0::/a/b\n", "2.5"),
    # the older layout, the controllers listed by name
    ({"cpu/cpu.cfs_quota_us": "-1", "cpu/cpu.cfs_period_us": "100000"}, "1:cpu:/\n", "inf"),
    ({"cpu/x/cpu.cfs_quota_us": "50000", "cpu/x/cpu.cfs_period_us": "100000"}, "3:cpuset:/y\n1:cpu,cpuacct:/x\n", "0.5"),
])
def test_the_control_groups_share_is_counted(probe, tmp_path, files, groups, cpus):
    root = tmp_path / "cgroup"
    root.mkdir()
    for name, text in files.items():
        (root / name).parent.mkdir(parents=True, exist_ok=True)
        (root / name).write_text(text + "\n")
    (tmp_path / "groups").write_text(groups)
    assert probe("cpus", root, tmp_path / "groups").strip() == cpus


def test_as_many_arrays_wait_for_their_next_use_as_there_are_kinds_of_result(probe):
    mb16 = 16 << 20
    assert [int(x) for x in probe("pool").split()] == [2 * mb16, mb16, 2 * mb16, 3 * mb16, 4 * mb16, 0, 1000, 0]


def test_a_forked_child_does_not_wait_for_threads_it_does_not_have(probe):
    assert "child ended 1\n" in probe("fork")
