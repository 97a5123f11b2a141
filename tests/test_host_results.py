"""The host side of results on their way to the caller, without a GPU."""
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
