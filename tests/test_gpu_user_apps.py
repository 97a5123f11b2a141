"""Applications that are not compiled into the library.  tests/cpp/user_apps.hip holds two App
structs written on the contract the way a user of the reference writes them, built by hipcc
into a shared object of its own that registers them when it loads (ND_REGISTER_APP); what the
engine samples with them is the oracle's bytes.  Then the per-app Python module surface
(src/nextDoorPythonModule.cu:40-102) end to end on a binary edge-list file."""
import os

import numpy as np
import pytest

import nextdoor_amd as nd
from tests import graphs, oracle_binding as ob
from tests.cpp.build_cpp import USER_APPS_LIB

SEED = 42


@pytest.mark.gpu
@pytest.mark.parametrize("gname", ["sparse", "hub"])
@pytest.mark.parametrize("app,kind,sizes", [("UserThreeHop", "KHOP", [5, 3, 2]),
                                            ("UserShortDeepWalk", "DEEPWALK", [1] * 7)])
def test_apps_registered_from_their_own_shared_object_match_the_oracle(app, kind, sizes, gname):
    assert os.path.exists(USER_APPS_LIB), "tests/cpp/libuser_apps.so is built by __graft_entry__.build()"
    nd.load_app_library(USER_APPS_LIB)
    assert app in nd.app_names()
    g = graphs.random_graph(**{"sparse": dict(n=300, mean_degree=3, seed=1, isolated_every=7),
                               "hub": dict(n=400, mean_degree=10, seed=2, hub=5)}[gname])
    og = graphs.oracle_view(g)
    s = nd.Sampler(app, g, seed=SEED)
    try:
        assert [s.step_size(k) for k in range(s.steps)] == sizes
        assert s.num_samples == (g.n_vertices if kind == "KHOP" else 3 * g.n_vertices)
        if kind == "DEEPWALK":
            assert np.array_equal(s.initial_contents, np.arange(s.num_samples, dtype=np.int32) % g.n_vertices)
        d = ob.app_desc(getattr(ob, kind), s.steps, sizes)
        want, _ = ob.sample_individual(og, d, SEED, s.initial_contents)
        for lb in (False, True):
            print("app", app, "graph", gname, "lb", lb, flush=True)
            s.do_transit_parallel(load_balancing=lb)
            assert np.array_equal(s.final_samples(), want)
            assert s.check_results() == (True, "")
        s.do_sample_parallel()
        assert np.array_equal(s.final_samples(), want)
    finally:
        s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("gname", ["sparse", "hub"])
def test_an_app_with_explicit_transits_and_several_transits_per_sample(gname):
    """stepTransits decides the next step's transits (src/nextdoor.cu:279-289) for an app that is
    not a walk: four transits per sample, step sizes 2, 3, 2; every schedule gives the oracle's bytes."""
    nd.load_app_library(USER_APPS_LIB)
    g = graphs.random_graph(**{"sparse": dict(n=300, mean_degree=3, seed=1, isolated_every=7),
                               "hub": dict(n=1200, mean_degree=10, seed=2, hub=5)}[gname])
    og = graphs.oracle_view(g)
    s = nd.Sampler("UserAnchorHop", g, seed=SEED)
    try:
        assert (s.steps, s.initial_sample_size, s.final_sample_size) == (3, 4, 8 + 24 + 48)
        anchors = s.initial_contents.reshape(-1, 4)
        assert np.array_equal(anchors, np.stack([(np.arange(g.n_vertices) * 7 + i * 13) % g.n_vertices
                                                 for i in range(4)], axis=1))
        want, _ = ob.sample_anchor_hop(og, SEED, anchors, [2, 3, 2])
        for mode in (False, True, "sample_parallel", True):
            print("UserAnchorHop", gname, mode, flush=True)
            if mode == "sample_parallel":
                s.do_sample_parallel()
            else:
                s.do_transit_parallel(load_balancing=mode)
            assert np.array_equal(s.final_samples(), want)
        with pytest.raises(nd.NextDoorError):  # explicit transits: the library has no validator
            s.check_results()
    finally:
        s.close()


# neighbourhoods ranked in LDS (of fewer vertices than a layer takes, and of more), and larger ones, with keys that tell the
# vertices apart and with equal ones
@pytest.mark.gpu
@pytest.mark.parametrize("n,mean_degree,weight", [(2000, 0.5, "any"), (2000, 10, "any"), (6000, 700, "any"), (6000, 700, "tiny")])
def test_a_ranked_layer_hands_over_as_many_vertices_as_it_takes(n, mean_degree, weight):
    """numEdges of the LADIES form is a function of the graph and the roots: the layer's size, or all that there are."""
    nd.load_app_library(USER_APPS_LIB)
    rng = np.random.default_rng(5)
    src, dst = rng.integers(0, n, (2, int(n * mean_degree)))
    w = rng.uniform(1.0, 2.0, len(src)).astype(np.float32)
    if weight == "tiny":  # terms of 0, but for one edge of each row
        w[:] = 1e-9
        src, dst, w = np.append(src, np.arange(n)), np.append(dst, rng.integers(0, n, n)), np.append(w, np.ones(n, np.float32))
    g = nd.Graph.from_edges(src, dst, w, n_vertices=n)
    s = nd.Sampler("UserRankedCount", g, seed=SEED)
    try:
        roots = s.initial_contents.reshape(s.num_samples, -1)
        distinct = [len(np.unique(np.concatenate([g.col[g.row_ptr[r]:g.row_ptr[r + 1]] for r in row]))) for row in roots]
        want = np.minimum(distinct, s.step_size(0))
        print("UserRankedCount", n, mean_degree, weight, "least and most vertices", min(distinct), max(distinct), flush=True)
        for _ in range(3):
            s.do_transit_parallel()
            got = s.final_samples()
            assert np.array_equal(got[:, 0], want)
            assert np.array_equal((got[:, 1:] != s.invalid_vertex).sum(axis=1), np.maximum(want - 1, 0))
    finally:
        s.close()


# rows that follow their one launch and rows that leave by range, all states together a whole number of words and not
@pytest.mark.gpu
@pytest.mark.parametrize("n", [3002, 3001, 90002])
@pytest.mark.parametrize("app,fields", [("UserSumWalk", 1), ("UserTallyWalk", 3)])
def test_states_of_no_whole_number_of_words(oracle, app, fields, n):
    """States of 2 and 6 bytes are those of the pass, also where rows and states were taken after the passes before."""
    nd.load_app_library(USER_APPS_LIB)
    g = graphs.random_graph(n=n, mean_degree=5, seed=n, isolated_every=7)
    s = nd.Sampler(app, g, seed=SEED)
    d = ob.app_desc(ob.UNIFORM_WALK, s.steps, [1] * s.steps)
    want, _ = ob.sample_individual(graphs.oracle_view(g), d, SEED, s.initial_contents)
    visited = want != s.invalid_vertex
    steps = visited.sum(axis=1)
    notes = [np.where(visited, want, 0).sum(axis=1), want[np.arange(n), np.maximum(steps, 1) - 1] * (steps > 0), steps]
    notes = np.stack(notes[:fields], axis=1).astype(np.uint16)
    try:
        for turn in range(6):
            print("app", app, "n", n, "turn", turn, flush=True)
            s.set_inversion_period(1 if turn == 4 else 0)
            s.do_transit_parallel()
            assert np.array_equal(s.final_samples(), want)
            states = s.sample_states()
            assert states.size == 2 * n * fields
            assert np.array_equal(np.frombuffer(states.tobytes(), np.uint16).reshape(n, fields), notes)
    finally:
        s.close()


def write_binary_edge_list(path, src, dst, weight):
    """The reference's binary edge list: 12-byte records (int32 src, int32 dst, float32 weight),
    src/graph.hpp:42-75."""
    rec = np.zeros(len(src), dtype=[("s", "<i4"), ("d", "<i4"), ("w", "<f4")])
    rec["s"], rec["d"], rec["w"] = src, dst, weight
    rec.tofile(path)


def edges_of(g):
    src = np.repeat(np.arange(g.n_vertices, dtype=np.int32), np.diff(g.row_ptr))
    return src, g.col.copy(), g.weight.copy()


@pytest.mark.gpu
def test_sampling_module_functions_end_to_end(tmp_path):
    """initSampling -> sample -> finalSampleLength -> finalSamplesArray -> freeDeviceMemory on a
    written file, a second initSampling on another graph and app, and the calls before
    initSampling (the sequence of src/apps/khop/KHopSamplingPy3 users, nextDoorPythonModule.cu)."""
    lib = nd._capi.lib()
    lib.nd_free_device_memory()
    module = nd.SamplingModule("KHop", seed=SEED)
    with pytest.raises(nd.NextDoorError, match="before initSampling"):
        module.sample()
    with pytest.raises(nd.NextDoorError, match="before initSampling"):
        module.finalSamplesArray()
    assert module.finalSampleLength() == 0
    with pytest.raises(nd.NextDoorError):
        module.initSampling(tmp_path / "missing.data")

    cases = [("KHop", ob.KHOP, graphs.random_graph(n=500, mean_degree=8, seed=11, hub=2)),
             ("DeepWalk", ob.DEEPWALK, graphs.random_graph(n=300, mean_degree=4, seed=12, isolated_every=5))]
    for i, (app, kind, g) in enumerate(cases):
        path = tmp_path / f"graph{i}.data"
        write_binary_edge_list(path, *edges_of(g))
        loaded = nd.Graph.load(str(path), "edge-list", "binary")
        assert np.array_equal(loaded.row_ptr, g.row_ptr) and np.array_equal(loaded.col, g.col)
        og = graphs.oracle_view(loaded)
        reference = nd.Sampler(app, loaded, seed=SEED)  # only for the shape and the roots
        steps, sizes, roots = reference.steps, [reference.step_size(k) for k in range(reference.steps)], reference.initial_contents.copy()
        final = reference.final_sample_size
        reference.close()
        want, _ = ob.sample_individual(og, ob.app_desc(kind, steps, sizes), SEED, roots)

        print("SamplingModule", app, flush=True)
        module = nd.SamplingModule(app, seed=SEED)
        module.initSampling(path)  # the second pass replaces the first module state
        for _ in range(2):  # sample() may be called again, as in the reference
            module.sample()
            assert module.finalSampleLength() == want.size
            got = module.finalSamplesArray()
            assert got.dtype == np.int32 and np.array_equal(got.reshape(-1, final), want)
        assert module.finalSamples()[:final] == want[0].tolist()
    # the same sampler from CSR arrays in memory
    app, kind, g = cases[0]
    module = nd.SamplingModule(app, seed=SEED)
    module.initSamplingFromCSR(g.row_ptr, g.col, g.weight)
    module.sample()
    reference = nd.Sampler(app, g, seed=SEED)
    want, _ = ob.sample_individual(graphs.oracle_view(g), ob.app_desc(kind, reference.steps, [reference.step_size(k) for k in range(reference.steps)]),
                                   SEED, reference.initial_contents.copy())
    reference.close()
    assert np.array_equal(module.finalSamplesArray().reshape(want.shape), want)
    module.freeDeviceMemory()
    assert module.finalSampleLength() == 0
    with pytest.raises(nd.NextDoorError, match="before initSampling"):
        module.sample()
    module.freeDeviceMemory()  # twice is harmless
