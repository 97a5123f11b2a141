// Rows of walks that are sent to the host while the pass is still going on (Engine::rows_ahead), and what else may be
// asked for before they are: the engine is instantiated here, so that a transfer can be made to fail.  Prints the case
// before it runs, "all as they should be" at the end.
#include "../../nextdoor_amd/csrc/nd_apps_walks.hpp"
#include "../../nextdoor_amd/csrc/nd_graph.hpp"
#include "../../nextdoor_amd/csrc/nd_sharded_engine.hpp"

#include <stdio.h>
#include <sys/resource.h>

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

// more states than are copied without the result stream, and two ranges of walks
static const int32_t kVertices = 1200007;

int main() {
  CSR graph;
  std::string error;
  {
    std::vector<int32_t> src, dst;
    std::vector<float> weight;
    for (int32_t v = 0; v < kVertices; ++v)
      for (int32_t k = 0; k < v % 4; ++k) {
        src.push_back(v);
        dst.push_back((int32_t)(((int64_t)v * 7919 + k * 104729 + 1) % kVertices));
        weight.push_back(1.0f + (float)(k + v % 3));
      }
    CHECK(nd::csr_from_edges(graph, kVertices, src.size(), src.data(), dst.data(), weight.data(), &error) == 0);
  }
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

  for (int with_states = 0; with_states < 2; ++with_states) {
    printf("rows whose transfer fails, states asked for %d\n", with_states);
    fflush(stdout);
    std::fill(got.begin(), got.end(), -7);
    CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0);
    // in the place of the rows' transfer one that waits for no event at all, which the runtime refuses
    CHECK(engine.result_stream->finish() == hipSuccess);
    std::fill(got.begin(), got.end(), -7);
    int32_t* words = nullptr;
    CHECK(hipMalloc(&words, n * sizeof(int32_t)) == hipSuccess);
    CHECK(engine.result_stream->begin(words, n, 32, 0, got.data(), nullptr, {{n, nullptr}}) == hipSuccess);
    if (with_states) {
      std::fill(states.begin(), states.end(), 0);
      CHECK(engine.fetch_sample_states(states.data(), states.size()) == 0 && states == want_states);
    }
    CHECK(!engine.finish_rows_ahead());  // they did not get there
    CHECK(engine.fetch_final_samples_into(got.data()) == 0 && got == want);
    CHECK(hipFree(words) == hipSuccess);
  }

  STEP("and the next pass's");
  std::fill(got.begin(), got.end(), -7);
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0 && engine.finish_rows_ahead() && got == want);
  STEP("freed with rows on their way");
  CHECK(engine.sample(nd::kTransitParallelLoadBalanced) == 0);
  engine.free_device();
  STEP("what a sampler holds, given back");
  for (const char* ranges : {"1", "2"}) {
    setenv("ND_SAMPLE_RANGES", ranges, 1);
    nd::ShardedEngine<Node2VecSample, WeightedNode2VecAppT<8>> sampler("walks");
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
  STEP("no host memory for rows that nobody has asked for yet");
  {
    nd::ShardedEngine<Node2VecSample, WeightedNode2VecAppT<8>> sampler("walks");
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
  printf("all as they should be\n");
  return 0;
}
