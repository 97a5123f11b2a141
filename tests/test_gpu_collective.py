"""GPU parity of the layer-wise (CollectiveNeighborhood) engine against the CPU oracle:
collective-neighbourhood build, the reference's FastGCN/LADIES app (vertices, recorded
adjacency-matrix entries, the reference's validator) and the importance sampler."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

import nextdoor_amd as nd
from tests import graphs
from tests.cpp.build_cpp import LONG_NEIGHBOURHOOD_PROBE

pytestmark = pytest.mark.gpu

SEED = 42


def test_collective_neighborhood_matches_oracle(oracle):
    g = graphs.random_graph(n=400, mean_degree=5, seed=11, isolated_every=6, hub=9)
    og = graphs.oracle_view(g)
    rng = np.random.default_rng(0)
    S, B = 37, 300  # more transits than one scan chunk of 256
    transits = rng.integers(0, g.n_vertices + 1, (S, B)).astype(np.int32)  # includes INVALID (= n_vertices)
    transits[3] = g.n_vertices  # a sample with nothing but INVALID transits
    sizes, offsets, cols, weights, rows = nd.collective_neighborhood(g, transits, B, g.n_vertices, 1 << 22)
    assert offsets[0] == 0 and np.array_equal(np.cumsum(sizes), offsets[1:])
    for s in range(S):
        wc, ww, wr = oracle.collective_neighborhood(og, transits[s], g.n_vertices)
        assert sizes[s] == len(wc)
        assert np.array_equal(cols[offsets[s]:offsets[s + 1]], wc)
        assert np.array_equal(weights[offsets[s]:offsets[s + 1]], ww)
        assert np.array_equal(rows[s], wr)
    assert sizes[3] == 0


def device_memory_left():
    hip = ctypes.CDLL("libamdhip64.so")
    left, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
    return left.value


def layer_desc(oracle, s, kind):
    return oracle.app_desc(kind, s.steps, [s.step_size(k) for k in range(s.steps)],
                           initial_size=s.initial_sample_size)


@pytest.mark.parametrize("app,layers,batch", [("LayerLiteral2x8", 2, 8), ("LayerLiteral3x16", 3, 16)])
def test_layer_literal_matches_oracle(oracle, app, layers, batch):
    g = graphs.random_graph(n=300, mean_degree=8, seed=5, hub=2)
    og = graphs.oracle_view(g)
    s = nd.Sampler(app, g, seed=SEED)
    d = layer_desc(oracle, s, oracle.LAYER_LITERAL)
    roots = s.initial_contents
    assert np.array_equal(roots, np.arange(s.num_samples * batch) % g.n_vertices)  # fastgcnSampling.cu:75-85
    want, want_rows, want_cols = oracle.sample_layer_literal(og, d, SEED, roots)
    for lb in (False, True):
        print("app", app, "lb", lb, flush=True)
        s.do_transit_parallel(lb)
        got = s.final_samples()
        assert np.array_equal(got, want)
        # LayerSampleT: int len[L]; int row[L][B*B]; int col[L][B*B]; int val[L][B*B]
        st = s.sample_states().view(np.int32).reshape(s.num_samples, -1)
        bb = batch * batch
        assert st.shape[1] == layers + 3 * layers * bb
        got_rows = st[:, layers:layers + layers * bb].reshape(-1, layers, bb)
        got_cols = st[:, layers + layers * bb:layers + 2 * layers * bb].reshape(-1, layers, bb)
        assert np.array_equal(got_rows, want_rows) and np.array_equal(got_cols, want_cols)
        assert np.all(st[:, :layers] == 0)
    # the reference's own validator on the GPU result
    assert oracle.check_adjacency_matrix(og, d, roots, got, got_rows, got_cols, s.invalid_vertex)
    assert s.check_results() == (True, "")  # and the library's
    print("app", app, "sample parallel", flush=True)
    s.do_sample_parallel()
    assert np.array_equal(s.final_samples(), want)
    s.close()


@pytest.mark.parametrize("app", ["FastGCNImportance2x8", "FastGCNImportance3x16"])
@pytest.mark.parametrize("gname", ["sparse", "hub"])
def test_fastgcn_importance_matches_oracle(oracle, app, gname):
    g = (graphs.random_graph(n=300, mean_degree=3, seed=1, isolated_every=4) if gname == "sparse"
         else graphs.random_graph(n=2000, mean_degree=12, seed=2, hub=5))
    og = graphs.oracle_view(g)
    s = nd.Sampler(app, g, seed=SEED)
    d = layer_desc(oracle, s, oracle.FASTGCN_IMPORTANCE)
    roots = s.initial_contents
    assert roots.min() >= 0 and roots.max() < g.n_vertices
    want = oracle.sample_fastgcn_importance(og, d, SEED, roots)
    print("app", app, "graph", gname, flush=True)
    s.do_transit_parallel(True)
    got = s.final_samples()
    assert np.array_equal(got, want)
    # every drawn vertex is a neighbour of some vertex of the previous layer
    B = s.step_size(0)
    for row, init in list(zip(got, roots.reshape(-1, s.initial_sample_size)))[:40]:
        prev = init
        for k in range(s.steps):
            cur = row[k * B:(k + 1) * B]
            for v in cur[cur != s.invalid_vertex]:
                assert any(p != s.invalid_vertex and oracle.lib().ndo_has_edge(og.struct, int(p), int(v)) for p in prev)
            prev = cur
    s.do_transit_parallel(True)
    assert np.array_equal(s.final_samples(), want)
    assert s.check_results() == (True, "")
    s.close()


@pytest.mark.parametrize("app", ["FastGCNImportance2x8", "FastGCNImportance3x16", "LADIESImportance2x8",
                                 "LADIESImportance3x16"])
def test_importance_sampling_with_ready_made_hub_pieces(oracle, app, monkeypatch):
    """Vertices with many edges into one stretch of the vertex range contribute a piece built
    once per graph (a bitmap, or the importance sums) instead of their entries: same samples,
    with or without."""
    g = graphs.random_graph(n=2000, mean_degree=12, seed=2, hub=5)
    og = graphs.oracle_view(g)
    monkeypatch.setenv("ND_DENSE_PIECE_ENTRIES", "0")
    s = nd.Sampler(app, g, seed=SEED)
    assert s.counter(3) == 0
    ladies = app.startswith("LADIES")
    d = layer_desc(oracle, s, oracle.LADIES_IMPORTANCE if ladies else oracle.FASTGCN_IMPORTANCE)
    want = (oracle.sample_ladies_importance if ladies else oracle.sample_fastgcn_importance)(
        og, d, SEED, s.initial_contents)
    s.do_transit_parallel(True)
    assert np.array_equal(s.final_samples(), want)
    s.close()
    for entries in ("4", "16", "400"):
        monkeypatch.setenv("ND_DENSE_PIECE_ENTRIES", entries)
        s = nd.Sampler(app, g, seed=SEED)
        print("app", app, "pieces from", entries, "entries:", s.counter(3), flush=True)
        assert s.counter(3) > 0
        s.do_transit_parallel(True)
        assert np.array_equal(s.final_samples(), want)
        s.do_transit_parallel(True)
        assert np.array_equal(s.final_samples(), want)
        s.close()


@pytest.mark.parametrize("app", ["FastGCNImportance3x16", "LADIESImportance3x16"])
@pytest.mark.parametrize("pieces", ["default", "8", "0"])
def test_importance_sampling_over_several_stretches(oracle, app, pieces, monkeypatch):
    """130,000 vertices: two stretches of the FastGCN form, 19 of the LADIES form (two
    workgroups per sample), a hub with edges into all of them."""
    if pieces != "default":
        monkeypatch.setenv("ND_DENSE_PIECE_ENTRIES", pieces)
    g = graphs.random_graph(n=130000, mean_degree=3, seed=5, hub=8, isolated_every=6)
    og = graphs.oracle_view(g)
    s = nd.Sampler(app, g, seed=SEED)
    ladies = app.startswith("LADIES")
    d = layer_desc(oracle, s, oracle.LADIES_IMPORTANCE if ladies else oracle.FASTGCN_IMPORTANCE)
    want = (oracle.sample_ladies_importance if ladies else oracle.sample_fastgcn_importance)(
        og, d, SEED, s.initial_contents)
    print("app", app, "pieces", pieces, "built", s.counter(3), flush=True)
    # without pieces the hub's 260,000 edges go through the entry-by-entry path (and the
    # attempt to take a workgroup's stretches at once gives up on their number)
    assert (s.counter(3) > 0) == (pieces != "0")
    s.do_transit_parallel(True)
    assert np.array_equal(s.final_samples(), want)
    s.close()


def test_distinct_is_refused_for_layer_apps():
    g = graphs.random_graph(n=100, mean_degree=4, seed=1)
    s = nd.Sampler("LayerLiteral2x8", g, seed=SEED)
    s.do_transit_parallel(True)
    with pytest.raises(nd.NextDoorError):
        s.distinct()
    s.close()


@pytest.mark.parametrize("app", ["LADIESImportance2x8", "LADIESImportance3x16"])
@pytest.mark.parametrize("gname", ["sparse", "hub"])
def test_ladies_importance_matches_oracle(oracle, app, gname):
    g = (graphs.random_graph(n=300, mean_degree=3, seed=1, isolated_every=4) if gname == "sparse"
         else graphs.random_graph(n=2000, mean_degree=12, seed=2, hub=5))
    og = graphs.oracle_view(g)
    s = nd.Sampler(app, g, seed=SEED)
    d = layer_desc(oracle, s, oracle.LADIES_IMPORTANCE)
    roots = s.initial_contents
    want = oracle.sample_ladies_importance(og, d, SEED, roots)
    print("app", app, "graph", gname, flush=True)
    s.do_transit_parallel(True)
    got = s.final_samples()
    assert np.array_equal(got, want)
    # without replacement: no vertex twice inside a layer segment
    B = s.step_size(0)
    for row in got[:100]:
        for k in range(s.steps):
            seg = row[k * B:(k + 1) * B]
            seg = seg[seg != s.invalid_vertex]
            assert len(set(seg.tolist())) == len(seg)
    assert s.check_results() == (True, "")
    s.close()


@pytest.mark.parametrize("weights", ["equal_keys", "later_is_better", "one_of_all"])
@pytest.mark.parametrize("pieces", ["0", "default"])
def test_ladies_keys_that_are_hard_to_tell_apart(oracle, weights, pieces, monkeypatch):
    """What a workgroup keeps of a sample: nearly all keys equal (terms below 2^-53: importance 0, told apart by vertex;
    more of them in one stretch than a workgroup begins the next with), every stretch's keys better than the last one's,
    and one vertex far better than all others."""
    if pieces != "default":
        monkeypatch.setenv("ND_DENSE_PIECE_ENTRIES", pieces)
    n, hubs = 60000, 24
    rng = np.random.default_rng(3)
    src = np.concatenate([np.repeat(np.arange(hubs), n), np.arange(n)])  # the hubs know everyone, everyone knows a hub
    dst = np.concatenate([np.tile(np.arange(n), hubs), rng.integers(0, hubs, n)])
    w = np.ones(len(src), np.float32)
    if weights == "equal_keys":
        w[:hubs * n] = 1e-9
        w[np.arange(hubs) * n + rng.integers(0, n, hubs)] = 1.0
    elif weights == "later_is_better":
        w[:hubs * n] = np.tile(np.exp2(np.arange(n) / 3000.0), hubs)
    else:
        w[np.arange(hubs) * n + 4321] = 1e6
    g = nd.Graph.from_edges(src, dst, w, n_vertices=n)
    s = nd.Sampler("LADIESImportance2x8", g, seed=SEED)
    want = oracle.sample_ladies_importance(graphs.oracle_view(g), layer_desc(oracle, s, oracle.LADIES_IMPORTANCE), SEED,
                                           s.initial_contents)
    print("weights", weights, "pieces", pieces, "built", s.counter(3), flush=True)
    for _ in range(2):
        s.do_transit_parallel(True)
        assert np.array_equal(s.final_samples(), want)
    assert s.counter(2) == s.steps  # one chunk a layer
    s.close()
    monkeypatch.setenv("ND_LAYER_CHUNK_ENTRIES", str(20 * n))
    s = nd.Sampler("LADIESImportance2x8", g, seed=SEED)
    for _ in range(2):
        s.do_transit_parallel(True)
        assert np.array_equal(s.final_samples(), want)
    assert s.counter(2) > 3 * s.steps
    s.close()


def test_what_is_kept_of_a_sample_is_no_more_than_there_are_vertices(oracle):
    """1024 samples over 2000 vertices: 16 MB for what is kept of them, where room for a workgroup's stretches is 100."""
    g = graphs.random_graph(n=2000, mean_degree=60, seed=6, hub=5)  # 512 roots have 30000 neighbours: ranked in parts
    before = device_memory_left()
    s = nd.Sampler("LADIESImportance", g, seed=SEED)
    try:
        s.do_transit_parallel(True)
        taken = before - device_memory_left()
        print("taken", taken, flush=True)
        assert taken < 64 << 20
        want = oracle.sample_ladies_importance(graphs.oracle_view(g), layer_desc(oracle, s, oracle.LADIES_IMPORTANCE), SEED,
                                               s.initial_contents)
        assert np.array_equal(s.final_samples(), want)
    finally:
        s.close()


@pytest.mark.parametrize("app,kind_name", [("FastGCNImportance3x16", "FASTGCN_IMPORTANCE"),
                                           ("LADIESImportance3x16", "LADIES_IMPORTANCE"),
                                           ("LayerLiteral3x16", "LAYER_LITERAL")])
def test_chunked_processing_gives_the_same_samples(oracle, app, kind_name, monkeypatch):
    g = graphs.random_graph(n=2000, mean_degree=12, seed=2, hub=5)
    s = nd.Sampler(app, g, seed=SEED)
    s.do_transit_parallel(True)
    whole = s.final_samples()
    assert s.counter(2) == s.steps  # one chunk per layer
    s.close()
    monkeypatch.setenv("ND_LAYER_CHUNK_ENTRIES", "3000")  # a few samples per chunk
    s = nd.Sampler(app, g, seed=SEED)
    s.do_transit_parallel(True)
    assert s.counter(2) > 3 * s.steps
    assert np.array_equal(s.final_samples(), whole)
    s.close()


@pytest.mark.parametrize("app", ["FastGCNImportance2x8", "LADIESImportance2x8", "LayerLiteral2x8"])
def test_progress_is_reported_for_every_layer(app, monkeypatch, capfd):
    monkeypatch.setenv("ND_PROGRESS", "1")
    s = nd.Sampler(app, graphs.random_graph(n=400, mean_degree=8, seed=3, hub=2), seed=SEED)
    try:
        for _ in range(2):
            capfd.readouterr()
            s.do_transit_parallel()
            lines = re.findall(r"\[nextdoor\] layer (\d+): samples (\d+) of (\d+) done, (\d+) ", capfd.readouterr().err)
            assert [int(l[0]) for l in lines] == list(range(s.steps))  # a chunk a layer
            assert all(int(l[1]) == int(l[2]) == s.num_samples for l in lines)
            assert int(lines[-1][3]) == s.counter(0) > int(lines[0][3]) > 0
    finally:
        s.close()


def test_neighbourhoods_that_are_too_long_are_worked_on_by_nobody():
    """A neighbourhood of 2^31 entries is refused before its layer, as far as any kernel is concerned, and the layers after
    it work on none; the pass reports it when it is over."""
    assert os.path.exists(LONG_NEIGHBOURHOOD_PROBE), "tests/cpp/long_neighbourhood_probe is built by __graft_entry__.build()"
    out = subprocess.run([LONG_NEIGHBOURHOOD_PROBE], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("all as they should be\n"), out.stdout[-300:] + out.stderr[-300:]


# eight transits of this many neighbours each: up to 8192 pairs are ranked in LDS, whose table is fullest then
@pytest.mark.parametrize("degree", [1, 8, 9, 257, 1023, 1024, 1025])
@pytest.mark.parametrize("weights", ["random", "equal_keys", "few_vertices"])
def test_ladies_neighbourhoods_at_the_edge_of_what_is_ranked_in_lds(oracle, degree, weights):
    """All neighbours different; nearly all keys equal (more than there is room for in order); and many pairs on few vertices."""
    n = 9001
    rng = np.random.default_rng(degree)
    v = np.repeat(np.arange(n), degree)
    i = np.tile(np.arange(degree), n)
    dst = (v * 1024 + i * (7 if weights == "few_vertices" else 1)) % (1100 if weights == "few_vertices" else n)
    w = (rng.random(len(v)) * 4 + 1).astype(np.float32)
    if weights == "equal_keys":
        w[i != 0] = 1e-9  # the terms of all but one are below 2^-53
    g = nd.Graph.from_edges(v, dst, w, n_vertices=n)
    s = nd.Sampler("LADIESImportance2x8", g, seed=SEED)
    want = oracle.sample_ladies_importance(graphs.oracle_view(g), layer_desc(oracle, s, oracle.LADIES_IMPORTANCE), SEED,
                                           s.initial_contents)
    for _ in range(2):
        s.do_transit_parallel(True)
        assert np.array_equal(s.final_samples(), want)
    s.close()


# Neighbourhoods too large to be ranked in LDS (8192 pairs), so that they are marked by stretches of 7168 vertices: every transit has `low`
# neighbours in the first stretch and `high` in the second.  Wavefronts take 256 pairs a round: transits that start with a
# round, one before it and one behind, rounds of one transit, and of more than the 63 starts that a round takes.
@pytest.mark.parametrize("app,low,high", [("LADIESImportance2x8", low, high) for low in (255, 256, 257, 512) for high in (900, 1024)] +
                         [("LADIESImportanceB8", low, high) for low, high in ((1, 17), (2, 15), (4, 16), (5, 64))])
def test_ladies_transits_that_start_at_the_edges_of_a_round(oracle, app, low, high):
    n = 9001
    v = np.repeat(np.arange(n), low + high)
    i = np.tile(np.arange(low + high), n)
    dst = np.where(i < low, (v * 37 + i * 11) % 7168, 7168 + (v * 41 + i * 7) % (n - 7168))  # all of a transit's are different
    w = (np.random.default_rng(low).random(len(v)) * 4 + 1).astype(np.float32)
    g = nd.Graph.from_edges(v, dst, w, n_vertices=n)
    s = nd.Sampler(app, g, seed=SEED)
    want = oracle.sample_ladies_importance(graphs.oracle_view(g), layer_desc(oracle, s, oracle.LADIES_IMPORTANCE), SEED,
                                           s.initial_contents)
    s.do_transit_parallel(True)
    assert np.array_equal(s.final_samples(), want)
    s.close()
