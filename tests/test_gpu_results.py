"""Results on their way to the host: the packed transfer against the words it starts from, and the arrays
a caller is given, which stay what they were when later results are fetched."""
import os
import subprocess

import numpy as np
import pytest

import nextdoor_amd as nd
from tests import graphs
from tests.cpp.build_cpp import RESULT_PROBE

pytestmark = pytest.mark.gpu


def test_packed_transfer_gives_back_the_words_on_the_device():
    assert os.path.exists(RESULT_PROBE), "tests/cpp/result_stream_probe is built by __graft_entry__.build()"
    out = subprocess.run([RESULT_PROBE], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("all equal\n"), out.stdout[-300:] + out.stderr[-300:]


# 1.1 MB: copied as it is; 8.8 MB: packed (12 bits, the ids and INVALID); 36 MB of 16 and 17 bits
@pytest.mark.parametrize("n", [1000, 4095, 32767, 32768])
def test_arrays_stay_the_callers(oracle, n):
    g = graphs.random_graph(n=n, mean_degree=6, seed=n, isolated_every=3)
    s = nd.Sampler("KHop", g, seed=42)
    d = oracle.app_desc(oracle.KHOP, 2, [25, 10])
    want, _ = oracle.sample_individual(graphs.oracle_view(g), d, 42, s.initial_contents)
    held = []
    for turn in range(12):  # more than any pool of the library's keeps
        print("n", n, "turn", turn, flush=True)
        s.do_transit_parallel()
        got = s.final_samples()
        assert np.array_equal(got, want)
        got[:] = -turn
        if turn % 3 != 2:
            held.append((turn, got))
        del got
    s.close()
    for turn, got in held:
        assert np.all(got == -turn)
