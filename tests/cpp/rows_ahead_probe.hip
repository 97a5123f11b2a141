// Rows of walks that are sent to the host while the pass is still going on (Engine::rows_ahead), and what else may be
// asked for before they are: the engine is instantiated here, so that a transfer can be made to fail.  Prints the case
// before it runs, "all as they should be" at the end.
#include "../../nextdoor_amd/csrc/nd_apps_walks.hpp"
#include "../../nextdoor_amd/csrc/nd_graph.hpp"
#include "../../nextdoor_amd/csrc/nd_sharded_engine.hpp"

#include <stdio.h>
#include <sys/resource.h>

#include <thread>

#define CHECK(expr)                                           \
  do {                                                        \
    if (!(expr)) { printf("not so: %s\n", #expr); return 1; } \
  } while (0)
#define STEP(text) printf("%s\n", text), fflush(stdout)

// Leaves the process `bytes` of private memory more than it has, or lifts that again (0).
static bool leave_memory(size_t bytes) {
  static rlim_t before = 0;
  rlimit limit;
  if (getrlimit(RLIMIT_DATA, &limit) != 0) return false;
  if (bytes) {
    size_t used_kb = 0;
    char line[256];
    FILE* f = fopen("/proc/self/status", "r");
    if (!f) return false;
    while (fgets(line, sizeof(line), f))
      if (sscanf(line, "VmData: %zu kB", &used_kb) == 1) break;
    fclose(f);
    before = limit.rlim_cur;
    limit.rlim_cur = used_kb * 1024 + bytes;
  } else {
    limit.rlim_cur = before;
  }
  return setrlimit(RLIMIT_DATA, &limit) == 0;
}

static bool make_graph(CSR& graph, int32_t vertices) {
  std::vector<int32_t> src, dst;
  std::vector<float> weight;
  for (int32_t v = 0; v < vertices; ++v)
    for (int32_t k = 0; k < v % 4; ++k) {
      src.push_back(v);
      dst.push_back((int32_t)(((int64_t)v * 7919 + k * 104729 + 1) % vertices));
      weight.push_back(1.0f + (float)(k + v % 3));
    }
  std::string error;
  return nd::csr_from_edges(graph, vertices, src.size(), src.data(), dst.data(), weight.data(), &error) == 0;
}

typedef nd::ShardedEngine<Node2VecSample, WeightedNode2VecAppT<8>> Walks;

// Passes of samplers of the same seed over each of the graphs, a thread each, whose rows leave ahead at the same time.
static int beside_each_other(const std::vector<const CSR*>& graphs) {
  std::vector<std::vector<VertexID_t>> want(graphs.size());
  for (size_t g = 0; g < graphs.size(); ++g) {
    Walks sampler("walks");
    nd::EngineBase& base = sampler;
    CHECK(base.set_graph(graphs[g]) == 0 && base.alloc(42) == 0);
    CHECK(base.sample(nd::kTransitParallelLoadBalanced) == 0 && base.fetch_final_samples() == 0);
    want[g].assign(base.hFinalSamples.data(), base.hFinalSamples.data() + base.hFinalSamples.size());
  }
  std::vector<int> wrong(graphs.size(), -1);
  std::vector<std::thread> threads;
  for (size_t g = 0; g < graphs.size(); ++g)
    threads.emplace_back([&, g] {
      Walks sampler("walks");
      nd::EngineBase& base = sampler;
      if (base.set_graph(graphs[g]) != 0 || base.alloc(42) != 0) return;
      int differ = 0;
      for (int pass = 0; pass < 12; ++pass) {
        if (base.sample(nd::kTransitParallelLoadBalanced) != 0 || base.fetch_final_samples() != 0) return;
        differ += memcmp(base.hFinalSamples.data(), want[g].data(), want[g].size() * sizeof(VertexID_t)) != 0;
        delete base.hFinalSamples.detach();
      }
      wrong[g] = differ;
    });
  for (auto& t : threads) t.join();
  for (int w : wrong) CHECK(w == 0);
  return 0;
}

// more states than are copied without the result stream, and walks enough for their rows to leave by stretch; and for ranges
static const int32_t kVertices = 1600007, kFewer = 400003, kFewest = 90001;

int main() {
  CSR graph;
  CHECK(make_graph(graph, kVertices));
  nd::Engine<Node2VecSample, WeightedNode2VecAppT<8>> engine("walks");
  CHECK(engine.set_graph(&graph) == 0 && engine.alloc(42) == 0);
  const size_t n = (size_t)kVertices * 8;
  CHECK(engine.sample_state_bytes() > nd::kDirectResultBytes);
  STEP("a pass whose rows nobody expects");
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0 && !engine.finish_rows_ahead());
  std::vector<VertexID_t> want(n), got(n, -7);
  std::vector<char> states(engine.sample_state_bytes()), want_states(states.size());
  CHECK(engine.fetch_final_samples_into(want.data()) == 0);
  CHECK(engine.fetch_sample_states(want_states.data(), want_states.size()) == 0);

  STEP("rows ahead");
  engine.rows_ahead = got.data();
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0 && engine.finish_rows_ahead());
  CHECK(got == want && !engine.finish_rows_ahead());

  STEP("states asked for before rows");
  std::fill(got.begin(), got.end(), -7);
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0);
  CHECK(engine.fetch_sample_states(states.data(), states.size()) == 0 && states == want_states);
  CHECK(engine.finish_rows_ahead() && got == want);

  uint32_t* sign = nullptr;  // what has arrived, and what never does
  CHECK(hipHostMalloc((void**)&sign, 2 * sizeof(uint32_t), hipHostMallocDefault) == hipSuccess);
  sign[0] = 1, sign[1] = 0;
  for (int form = 0; form < 6; ++form) {
    // all at once; by range; by stretch, with copies under way
    const int with_states = form % 2, parts = form / 2;
    printf("rows whose transfer fails, states asked for %d, parts %d\n", with_states, parts);
    fflush(stdout);
    std::fill(got.begin(), got.end(), -7);
    CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0);
    // in the place of the rows' transfer one that waits for no event at all, which the runtime refuses
    CHECK(engine.result_stream->finish() == hipSuccess);
    std::fill(got.begin(), got.end(), -7);
    int32_t* words = nullptr;
    CHECK(hipMalloc(&words, n * sizeof(int32_t)) == hipSuccess);
    std::vector<nd::ResultStream::Ready> ready{{n, nullptr}};
    if (parts == 1) ready.insert(ready.begin(), {n / 2, nullptr});
    if (parts == 2) ready = {{n / 2, nullptr, sign, 1}, {n, nullptr, sign + 1, 1}};
    CHECK(engine.result_stream->begin(words, n, 32, 0, got.data(), nullptr, ready) == hipSuccess);
    if (with_states) {
      std::fill(states.begin(), states.end(), 0);
      CHECK(engine.fetch_sample_states(states.data(), states.size()) == 0 && states == want_states);
    }
    CHECK(!engine.finish_rows_ahead());  // they did not get there
    CHECK(engine.fetch_final_samples_into(got.data()) == 0 && got == want);
    CHECK(hipFree(words) == hipSuccess);
  }

  CHECK(hipHostFree(sign) == hipSuccess);
  STEP("and the next pass's");
  std::fill(got.begin(), got.end(), -7);
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0 && engine.finish_rows_ahead() && got == want);
  STEP("freed with rows on their way");
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0);
  engine.free_device();
  STEP("what a sampler holds, given back");
  for (const char* ranges : {"1", "2"}) {
    setenv("ND_SAMPLE_RANGES", ranges, 1);
    Walks sampler("walks");
    nd::EngineBase& base = sampler;
    CHECK(base.set_graph(&graph) == 0 && base.alloc(42) == 0);
    for (int pass = 0; pass < 2; ++pass) {
      CHECK(base.sample(nd::kTransitParallelLoadBalanced) == 0 && base.fetch_final_samples() == 0);
      CHECK(memcmp(base.hFinalSamples.data(), want.data(), n * sizeof(VertexID_t)) == 0);
      delete base.hFinalSamples.detach();  // so that the next pass sends its rows ahead
    }
    CHECK(base.result_stream->page_locked_bytes() > 0);
    base.free_device();  // what nd_sampler_free_device does
    base.result_stream->release();
    CHECK(base.result_stream->page_locked_bytes() == 0);
  }
  unsetenv("ND_SAMPLE_RANGES");
  STEP("no host memory for rows that nobody has asked for yet");
  {
    Walks sampler("walks");
    nd::EngineBase& base = sampler;
    CHECK(base.set_graph(&graph) == 0 && base.alloc(42) == 0);
    CHECK(base.sample(nd::kTransitParallelLoadBalanced) == 0 && base.fetch_final_samples() == 0);
    nd::HostLease* held = base.hFinalSamples.detach();
    CHECK(leave_memory(n * sizeof(VertexID_t) / 2));
    int rc = -1;
    try {
      rc = base.sample(nd::kTransitParallelLoadBalanced);
    } catch (const std::bad_alloc&) {
    }
    CHECK(leave_memory(0));
    CHECK(rc == 0 && base.fetch_final_samples() == 0);
    CHECK(memcmp(base.hFinalSamples.data(), want.data(), n * sizeof(VertexID_t)) == 0);
    delete held;
  }
  STEP("samplers beside each other");
  CSR fewer, fewest;
  CHECK(make_graph(fewer, kFewer) && make_graph(fewest, kFewest));
  if (beside_each_other({&graph, &fewer, &fewest, &graph, &fewest}) != 0) return 1;
  printf("all as they should be\n");
  return 0;
}
