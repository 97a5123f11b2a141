"""Results on their way to the host: the packed transfer against the words it starts from, and the arrays
a caller is given, which stay what they were when later results are fetched."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import nextdoor_amd as nd
from tests import graphs
from tests.cpp.build_cpp import RESULT_PROBE, ROWS_AHEAD_PROBE

pytestmark = pytest.mark.gpu


def test_packed_transfer_gives_back_the_words_on_the_device():
    assert os.path.exists(RESULT_PROBE), "tests/cpp/result_stream_probe is built by __graft_entry__.build()"
    out = subprocess.run([RESULT_PROBE], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("all equal\n"), out.stdout[-300:] + out.stderr[-300:]


def test_what_is_asked_for_before_rows_that_are_on_their_way():
    """States fetched while rows are on their way do not take the news of a failed transfer with them: the rows are
    then fetched anew, not given out unfilled."""
    assert os.path.exists(ROWS_AHEAD_PROBE), "tests/cpp/rows_ahead_probe is built by __graft_entry__.build()"
    out = subprocess.run([ROWS_AHEAD_PROBE], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("all as they should be\n"), out.stdout[-300:] + out.stderr[-300:]


# 1.1 MB: copied as it is; 4.5 MB: packed (12 bits, the ids and INVALID); 36 MB of 15 and 16 bits
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


def mapping_flags(address):
    """The kernel's flags of the mapping an address is in (/proc/self/smaps)."""
    inside = False
    for line in open("/proc/self/smaps"):
        first = line.split()[0]
        if not first.endswith(":"):
            lo, hi = (int(x, 16) for x in first.split("-"))
            inside = lo <= address < hi
        elif inside and first == "VmFlags:":
            return line.split()[1:]


@pytest.mark.parametrize("n", [300, 2711, 4095, 9000])  # 0.3 and 3 MB, 4.5 MB, 9.9 MB
def test_arrays_are_ordinary_memory(n):
    """What a forked child inherits and system calls may pin, as any other array of the caller's."""
    s = nd.Sampler("KHop", graphs.random_graph(n=n, mean_degree=6, seed=n), seed=42)
    for _ in range(3):
        s.do_transit_parallel()
        got = s.final_samples()
        for address in (got.ctypes.data, got.ctypes.data + got.nbytes - 1):
            flags = mapping_flags(address)
            # dc: left out in a child; io, pf: a device's pages; sh: shared with a child that writes to it
            assert flags and not {"dc", "io", "pf", "sh"} & set(flags), flags
    s.close()


# fewer walks than are split into ranges, two ranges, and more than the device holds at once
@pytest.mark.parametrize("n", [98303, 196609, 1000003])
def test_rows_that_leave_before_the_pass_is_over(oracle, n):
    g = graphs.random_graph(n=n, mean_degree=4, seed=n, isolated_every=3)
    s = nd.Sampler("UniformRandomWalk8", g, seed=42)
    d = oracle.app_desc(oracle.UNIFORM_WALK, s.steps, [s.step_size(k) for k in range(s.steps)])
    want, _ = oracle.sample_individual(graphs.oracle_view(g), d, 42, s.initial_contents)
    step = lambda name: print("n", n, name, flush=True)
    rows = []
    for turn in range(3):  # from the second pass on the engine expects the rows to be fetched
        step("pass")
        s.do_transit_parallel()
        rows.append(s.final_samples())
        assert np.array_equal(rows[-1], want)
    step("a pass whose rows nobody fetches, and one more")
    s.do_transit_parallel()
    s.do_transit_parallel()
    assert np.array_equal(s.final_samples(), want)
    assert all(np.array_equal(r, want) for r in rows)
    step("rows changed after the pass")
    s.do_transit_parallel()
    s.distinct()
    changed = s.final_samples()
    assert np.array_equal(changed, want)  # one id a segment: each is distinct
    step("closed with rows on their way")
    s.do_transit_parallel()
    s.close()
    assert all(np.array_equal(r, want) for r in rows)


# rows of one launch: as many as the ring of what is on its way holds (64 MB of ids), a few more, and more than that by a whole launch
@pytest.mark.parametrize("n", [167772, 167801, 190003])
def test_rows_behind_a_pass_around_what_the_ring_holds(oracle, n):
    g = graphs.random_graph(n=n, mean_degree=4, seed=n, isolated_every=3)
    s = nd.Sampler("UniformRandomWalk", g, seed=42)
    d = oracle.app_desc(oracle.UNIFORM_WALK, s.steps, [s.step_size(k) for k in range(s.steps)])
    want, _ = oracle.sample_individual(graphs.oracle_view(g), d, 42, s.initial_contents)
    for turn in range(4):  # fetched after the first pass, behind the others
        print("n", n, "turn", turn, flush=True)
        s.do_transit_parallel()
        assert np.array_equal(s.final_samples(), want)
    s.do_transit_parallel()
    s.close()  # with rows on their way


def device_memory_left():
    hip = ctypes.CDLL("libamdhip64.so")
    left, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
    return left.value


def test_walks_take_device_memory_for_what_they_run():
    """Neither the buffers of an inversion nor the edges as walk records are there before a pass uses them."""
    n, walk = 400009, 100
    src = np.arange(n)
    g = nd.Graph.from_edges(np.repeat(src, 22), (np.repeat(src, 22) * 31 + np.tile(np.arange(22), n)) % n, n_vertices=n)
    rows, pairs, records = 4 * n * walk, 4 * n, 16 * g.n_edges
    assert 4 * g.n_edges > 32 << 20  # enough for the records to pay
    # What is left counts whole pages, and the runtime keeps blocks that earlier samplers of the process gave back: small
    # allocations may come from those.  32 MB is several times all small ones of a sampler, a fifth of any that matters here.
    held = 32 << 20
    before = device_memory_left()
    step = lambda name: print(name, before - device_memory_left(), flush=True)
    s = nd.Sampler("UniformRandomWalk", g, seed=42)
    try:
        step("allocated")
        s.set_inversion_period(1)
        s.do_transit_parallel()
        step("inverted")
        want = s.final_samples()
        inverted = device_memory_left()
        assert before - inverted >= 2 * rows - held
        s.set_inversion_period(0)
        s.do_transit_parallel()
        step("with records")
        assert inverted - device_memory_left() >= records - held  # no sampler that only inverts has them
        assert np.array_equal(s.final_samples(), want)
        s.close()
        s = nd.Sampler("UniformRandomWalk", g, seed=42)
        s.do_transit_parallel()
        step("not inverted")
        # the graph, the rows, the records: and neither the results by step nor pairs to sort (allocations round up)
        assert before - device_memory_left() <= 8 * g.n_edges + 8 * n + rows + records + 8 * pairs + (64 << 20)
        assert np.array_equal(s.final_samples(), want)
        s.set_inversion_period(1)
        s.do_transit_parallel()
        assert np.array_equal(s.final_samples(), want)
    finally:
        s.close()


# the forms a walk has: its state in registers, in memory (and transits of its own), the edges as walk records; each in one launch
# whose rows leave by stretch, from the least number of walks on (1), and below it by the range, in so many launches (0: one, at
# whose end they all leave); and walks whose state is in memory with rows that are stored by lines
@pytest.mark.parametrize("app,kind,n,mean_degree,launches", [
    ("WeightedNode2Vec8", "WEIGHTED_NODE2VEC", 360007, 3, 2),
    ("WeightedNode2Vec8", "WEIGHTED_NODE2VEC", 1523713, 3, 1),
    ("MultiRW4x6", "MULTIRW", 300007, 3, 4),
    ("MultiRW4x6", "MULTIRW", 812647, 3, 1),
    ("MultiRW", "MULTIRW", 65537, 6, 0),
    ("MultiRW", "MULTIRW", 100003, 6, 2),
    ("MultiRW", "MULTIRW", 196608, 6, 1),
    ("WeightedNode2Vec8", "WEIGHTED_NODE2VEC", 120011, 3, 0),
    ("UniformRandomWalk8", "UNIFORM_WALK", 600011, 15, 4),
    ("UniformRandomWalk8", "UNIFORM_WALK", 1777663, 2, 6),
    ("UniformRandomWalk8", "UNIFORM_WALK", 1777664, 2, 1),
    ("DeepWalkPerVertex", "DEEPWALK", 350003, 12, 3),
    ("DeepWalkPerVertex", "DEEPWALK", 500009, 9, 1),
])
@pytest.mark.parametrize("mode", ["transit", "sample"])
def test_rows_of_every_kind_of_walk_leave_before_the_pass_is_over(oracle, app, kind, n, mean_degree, launches, mode):
    g = graphs.random_graph(n=n, mean_degree=mean_degree, seed=n, isolated_every=5)
    og = graphs.oracle_view(g)
    s = nd.Sampler(app, g, seed=42)
    try:
        states_of = lambda: s.sample_states().view(np.int32).reshape(s.num_samples, -1)
        alive = slice(None)
        if kind == "MULTIRW":
            want, walkers, last, _ = oracle.sample_multirw(og, 42, states_of()[:, :-1], s.steps)
            want_states = np.concatenate([walkers, last[:, None]], axis=1)
        else:
            d = oracle.app_desc(getattr(oracle, kind), s.steps, [s.step_size(k) for k in range(s.steps)], p=2.0, q=0.5)
            want, want_states = oracle.sample_individual(og, d, 42, s.initial_contents)
            if kind == "WEIGHTED_NODE2VEC":
                alive = want_states != -1
                want_states = want_states.reshape(s.num_samples, -1)
            else:
                want_states = None
        run = s.do_transit_parallel if mode == "transit" else s.do_sample_parallel
        early = []
        for turn, states_first in enumerate([False, False, True, True]):
            print("app", app, "mode", mode, "turn", turn, flush=True)
            run()
            assert s.phase_times()["flat_launches"] == (max(launches, 1) if turn else 1)
            if states_first and want_states is not None:
                assert np.array_equal(states_of()[alive], want_states[alive])
            assert np.array_equal(s.final_samples(), want)
            if want_states is not None:
                assert np.array_equal(states_of()[alive], want_states[alive])
            # from the second pass on some are sent while others are still being walked (as far as the host keeps up)
            early.append(s.counter(10))
            print("parts that left early", early[-1], flush=True)
        assert early[0] == 0 and (max(early) > 0) == (launches > 0)
        run()
        s.set_profiling(True)  # rows stay until they are asked for
        run()
        assert s.counter(10) == 0 and np.array_equal(s.final_samples(), want)
    finally:
        s.close()


# rows as lines of memory: one walk more than are stored by fours, rows that end within a line and share it with the next,
# walks that end after a step, a stretch of one walk, and as many walks as leave by range or by stretch
@pytest.mark.parametrize("app,kind,n,isolated_every", [
    ("UniformRandomWalk", "UNIFORM_WALK", 65536, 7),
    ("UniformRandomWalk", "UNIFORM_WALK", 65537, 2),
    ("PPRPerVertex", "PPR", 458752, 3),
    ("WeightedNode2Vec", "WEIGHTED_NODE2VEC", 98304, 0),
    ("WeightedNode2Vec", "WEIGHTED_NODE2VEC", 98305, 3),
])
def test_rows_that_are_stored_by_lines(oracle, app, kind, n, isolated_every):
    g = graphs.random_graph(n=n, mean_degree=3, seed=n, isolated_every=isolated_every)
    s = nd.Sampler(app, g, seed=42)
    try:
        d = oracle.app_desc(getattr(oracle, kind), s.steps, [s.step_size(k) for k in range(s.steps)], p=2.0, q=0.5)
        want, _ = oracle.sample_individual(graphs.oracle_view(g), d, 42, s.initial_contents)
        for turn in range(3):
            print("app", app, "n", n, "turn", turn, flush=True)
            s.do_transit_parallel()
            assert np.array_equal(s.final_samples(), want)
    finally:
        s.close()


# rows enough for a quarter of the samples to be sampled first (96 MB), in the rows themselves and regrouped at the end
@pytest.mark.parametrize("app,n", [("KHop", 92003), ("Layer", 97001)])
def test_rows_of_hops_that_leave_before_the_pass_is_over(oracle, app, n):
    g = graphs.random_graph(n=n, mean_degree=5, seed=n, isolated_every=7)
    s = nd.Sampler(app, g, seed=42)
    steps = [s.step_size(k) for k in range(s.steps)]
    want, _ = oracle.sample_individual(graphs.oracle_view(g), oracle.app_desc(oracle.KHOP, 2, steps), 42, s.initial_contents)
    counts = None
    for turn in range(6):  # from the second pass on the rows are expected, but after one whose rows were made distinct first
        print("n", n, "turn", turn, flush=True)
        s.do_transit_parallel(load_balancing=turn % 2 == 0)
        if turn == 3:
            counts = s.distinct()  # with the rows as they were on their way
            changed = s.final_samples()
            assert changed.shape == want.shape and not np.array_equal(changed, want)
            continue
        rows = s.final_samples()
        assert np.array_equal(rows, want)
        del rows
    assert np.array_equal(s.distinct(), counts)
    s.do_sample_parallel()
    assert np.array_equal(s.final_samples(), want)
    s.do_transit_parallel()
    s.close()  # with rows on their way


# walks whose rows follow their one launch, and leave by range, with states; weighted walks with a state that travels
@pytest.mark.parametrize("app,n", [("MultiRW4x6", 3001), ("MultiRW4x6", 90001), ("WeightedNode2Vec8", 300007)])
def test_states_that_leave_with_the_rows(app, n):
    g = graphs.random_graph(n=n, mean_degree=5, seed=n, isolated_every=7)
    s = nd.Sampler(app, g, seed=42)
    s.do_transit_parallel()
    want, states = s.final_samples(), s.sample_states()  # fetched after the pass
    for turn in range(8):
        print("app", app, "n", n, "turn", turn, flush=True)
        s.do_transit_parallel()
        if turn == 2:
            assert np.array_equal(s.sample_states(), states)  # asked for first
            assert np.array_equal(s.final_samples(), want)
        elif turn == 3:
            assert np.array_equal(s.final_samples(), want)  # and not asked for
        elif turn == 5:
            continue  # nor the rows
        else:
            assert np.array_equal(s.final_samples(), want)
            assert np.array_equal(s.sample_states(), states)
    s.close()


# lists that follow the pass, and that leave as they are written (64 MB of rows and columns)
@pytest.mark.parametrize("n,degree", [(4004, 6), (60004, 24), (60020, 24)])
def test_edge_lists_that_leave_with_the_pass(n, degree):
    g = graphs.random_graph(n=n, mean_degree=degree, seed=n, isolated_every=7)
    s = nd.Sampler("MVS", g, seed=42)
    s.do_transit_parallel()
    want = s.adjacency()  # fetched after the pass
    assert n < 5000 or want[0].nbytes + want[1].nbytes > 64 << 20
    print("edges of the first quarter, from a group of eight on", want[2][s.num_samples // 4] % 8, flush=True)
    held = []
    for turn in range(6):
        print("n", n, "turn", turn, flush=True)
        s.do_transit_parallel()
        if turn == 1:
            continue
        if turn == 3:
            assert s.final_samples().shape[0] == s.num_samples  # asked for while the lists are on their way
        held.append(s.adjacency())
        if turn == 4:
            again = s.adjacency()
            assert all(np.array_equal(a, b) for a, b in zip(want, again))
    for lists in held:
        assert all(np.array_equal(a, b) for a, b in zip(want, lists))
    s.do_transit_parallel()
    s.close()  # with lists on their way


@pytest.mark.parametrize("app", ["FastGCNImportance3x16", "LADIESImportance3x16"])
def test_layer_rows_that_follow_the_pass(app):
    s = nd.Sampler(app, graphs.random_graph(n=4000, mean_degree=9, seed=5, isolated_every=7, hub=3), seed=42)
    s.do_transit_parallel()
    want = s.final_samples()  # fetched after the pass
    for turn in range(6):
        s.do_transit_parallel()
        if turn == 2:
            continue  # nobody asks
        got = s.final_samples()
        assert np.array_equal(got, want)
        if turn == 4:
            assert np.array_equal(s.final_samples(), want)
    s.do_transit_parallel()
    s.close()  # with rows on their way
