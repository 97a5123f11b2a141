"""The work that users of the sampling engine have it do, as cases that can be timed.

A case is one graph, one application and one way of running it.  What a program keeps (the graph,
the sampler with its device buffers) is prepared once; a pass is what such a program does per epoch:
run the sampling and take the samples, as host arrays, with whatever else the application leaves
(distinct counts, walker states, edge lists).
"""
import math

import nextdoor_amd as nd

# ---- the cases ---------------------------------------------------------------------------------
# graph: "rmat" (scale, edge_factor, symmetrised or not) or "chung_lu" (vertices, edges, exponent).
# run:   "transit" (transit-parallel with load balancing, the default of every caller), or "sample"
#        (the sample-parallel mode, what the reference's module function sample() runs).
# period: how often walks invert the map: 1 is the default, 0 leaves it to the engine.


def rmat(scale, edge_factor, symmetrise):
    return {"graph": "rmat", "scale": scale, "edge_factor": edge_factor, "symmetrise": symmetrise}


def chung_lu(vertices, edges, exponent):
    return {"graph": "chung_lu", "vertices": vertices, "edges": edges, "exponent": exponent}


def case(name, app, graph, run="transit", period=1):
    out = {"name": name, "app": app, "run": run, "period": period}
    out.update(graph)
    return out


def listed():
    return [
        # a citation-network sized graph: what a notebook or a unit of a pipeline calls, all latency
        case("walk_small", "UniformRandomWalk", chung_lu(2711, 21000, 2.3)),
        # the uniform walk of the benchmark (one walk per vertex of a protein-network sized graph)
        case("walk_57k", "UniformRandomWalk", chung_lu(56944, 818000, 2.1)),
        # DeepWalk corpora: a hundred weighted walks from every vertex, many walks share a transit
        case("deepwalk_100_per_vertex", "DeepWalk", chung_lu(10007, 300000, 2.2)),
        # personalised PageRank walks, which end early, over a larger graph, in the sample-parallel mode
        case("ppr_sample_parallel", "PPRPerVertex", chung_lu(262139, 4000000, 2.2), run="sample"),
        # the benchmark's headline: weighted node2vec over R-MAT 22, one walk per vertex
        case("node2vec_rmat22", "WeightedNode2Vec", rmat(22, 16, True)),
        # the same walk on an odd-sized sparser graph, the inversion period left to the engine
        case("node2vec_engine_period", "WeightedNode2Vec", chung_lu(700001, 9000000, 2.2), period=0),
        # multi-dimensional random walk: explicit transits, the walkers' states are part of the result
        case("multi_walk", "MultiRW", chung_lu(100003, 1500000, 2.2)),
        # GraphSAGE mini-batch neighbourhoods over every vertex of a large directed graph
        case("khop_rmat20", "KHop", rmat(20, 32, False)),
        # the same for a small graph, every hop made distinct afterwards
        case("khop_distinct", "KHop", chung_lu(60013, 1200000, 2.2), run="transit_distinct"),
        # FastGCN importance sampling, 4096 batches of 64, two layers
        case("fastgcn_rmat20", "FastGCNImportance", rmat(20, 16, True)),
        # LADIES importance sampling, 1024 batches of 512, two layers
        case("ladies_500k", "LADIESImportance", chung_lu(500009, 12000000, 2.0)),
        # minimal-variance sampling: every edge that leaves a batch of 32 vertices, as edge lists
        case("mvs_edge_lists", "MVS", chung_lu(150004, 2600000, 2.2)),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    app, lo, hi, mean_degree = rng.choice([
        ("UniformRandomWalk", 2000, 1500000, (4, 20)),
        ("DeepWalk", 1000, 10000, (8, 40)),
        ("DeepWalkPerVertex", 20000, 1000000, (8, 20)),
        ("PPRPerVertex", 20000, 1000000, (8, 20)),
        ("WeightedNode2Vec", 10000, 1500000, (6, 24)),
        ("MultiRW", 5000, 200000, (8, 24)),
        ("KHop", 3000, 800000, (8, 40)),
        ("Layer", 3000, 500000, (8, 40)),
        ("FastGCNImportance", 50000, 1000000, (8, 24)),
        ("LADIESImportance", 50000, 500000, (8, 24)),
        ("MVS", 10000, 300000, (8, 24)),
    ])
    if rng.random() < 0.25:
        scale = rng.randint(math.ceil(math.log2(lo)), math.floor(math.log2(hi)))
        symmetrise = rng.random() < 0.5
        degree = max(2, int(rng.uniform(*mean_degree)) // (2 if symmetrise else 1))
        graph = rmat(scale, degree, symmetrise)
    else:
        vertices = _spread(rng, lo, hi) | 1
        if app == "MVS":
            vertices += 3  # a multiple of 4: every vertex is in the same number of batches
            vertices -= vertices % 4
        graph = chung_lu(vertices, int(vertices * rng.uniform(*mean_degree)) | 1, round(rng.uniform(2.0, 2.5), 2))
    run, period = "transit", 1
    if app in ("KHop", "Layer"):
        run = rng.choice(["transit", "transit", "transit_distinct"])
    elif "Walk" in app or "PPR" in app or "2Vec" in app:
        run = rng.choice(["transit", "transit", "transit", "sample"])
        period = rng.choice([1, 1, 0])
    out = case("", app, graph, run, period)
    del out["name"]
    return out


# ---- running them ------------------------------------------------------------------------------

class _State:
    pass


def prepare(case, seed):
    state = _State()
    if case["graph"] == "rmat":
        state.graph = nd.Graph.rmat(case["scale"], case["edge_factor"], seed=seed, symmetrise=case["symmetrise"])
    else:
        state.graph = nd.Graph.chung_lu(case["vertices"], case["edges"], case["exponent"], seed=seed)
    state.sampler = nd.Sampler(case["app"], state.graph, seed=seed)
    if case["period"] != 1:
        state.sampler.set_inversion_period(case["period"])
    state.mode = case["run"]
    state.with_states = case["app"] == "MultiRW"
    state.with_edges = case["app"] == "MVS"
    return state


def run(state):
    sampler = state.sampler
    out = {}
    if state.mode == "sample":
        sampler.do_sample_parallel()
    else:
        sampler.do_transit_parallel(load_balancing=True)
    if state.mode == "transit_distinct":
        out["distinct_counts"] = sampler.distinct()
    if state.with_edges:
        out["rows"], out["cols"], out["list_start"] = sampler.adjacency()
        return out  # this application samples no vertices
    out["samples"] = sampler.final_samples()
    if state.with_states:
        out["states"] = sampler.sample_states()
    return out


# ---- what a pass cannot do without --------------------------------------------------------------

def _shape(case):
    """(vertices, edges, samples, outputs per sample, draws per sample)"""
    if case["graph"] == "rmat":
        vertices = 1 << case["scale"]
        edges = vertices * case["edge_factor"] * (2 if case["symmetrise"] else 1)
    else:
        vertices, edges = case["vertices"], case["edges"]
    app = case["app"]
    if app == "KHop":
        return vertices, edges, vertices, 25 + 25 * 10, 275
    if app == "Layer":
        return vertices, edges, vertices, 10 + 10 * 25, 260
    if app == "FastGCNImportance":
        return vertices, edges, 4096, 2 * 64, 2 * 64
    if app == "LADIESImportance":
        return vertices, edges, 1024, 2 * 512, 2 * 512
    if app == "MVS":
        # eight times every vertex, hence every edge; two words an edge, one a sample
        samples = -(-vertices * 8 // 32)
        return vertices, edges, samples, 1 + 2 * 8 * edges / samples, 0
    if app == "DeepWalk":
        return vertices, edges, vertices * (100 if vertices < 256 * 1024 else 1), 100, 100
    return vertices, edges, vertices, 100, 100


def work(case):
    """Each input read once and each output written once.  Per-transit sampling reads at most the
    whole graph and at least, per draw, a row's extent and one edge; layer-wise sampling builds the
    neighbourhood of every batch and is charged the graph once."""
    vertices, edges, samples, outputs, draws = _shape(case)
    weighted = case["app"] not in ("UniformRandomWalk", "KHop", "Layer", "MultiRW", "FastGCNImportance", "MVS")
    edge_bytes = 8 if weighted else 4
    whole_graph = 4 * (vertices + 1) + edge_bytes * edges
    touched = samples * draws * (8 + edge_bytes)
    layer_wise = case["app"] in ("FastGCNImportance", "LADIESImportance", "MVS")
    read = whole_graph if layer_wise else min(whole_graph, touched)
    written = 4 * samples * outputs
    if case["app"] == "MultiRW":
        read += 404 * samples      # the walkers and the one that moves next, per sample
        written += 404 * samples
    if case["run"] == "transit_distinct":
        written += 8 * samples
    return {"bytes": float(read + written), "flops": 0.0}


def tolerance(case):
    # vertex ids, counts, states and edge lists: whole numbers, fixed by the graph and the seed
    return "exact"
