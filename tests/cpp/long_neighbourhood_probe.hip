// Neighbourhoods of 2^31 entries and more: what the kernels that look at a layer's samples first make of them.  The graph has
// row extents only - they read nothing else - and the samples of the next layer come after a refusal.  Prints the case
// before it runs, "all as they should be" at the end.
#include "../../nextdoor_amd/csrc/nd_layer_engine.hpp"

#include <stdio.h>

#define TRY(expr)                                                              \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess) { printf("%s\n", hipGetErrorString(e_)); return 1; } \
  } while (0)
#define CHECK(expr)                                            \
  do {                                                         \
    if (!(expr)) { printf("not so: %s\n", #expr); return 1; } \
  } while (0)

template <class T>
static hipError_t to_device(T** out, const std::vector<T>& v) {
  const hipError_t e = hipMalloc((void**)out, v.size() * sizeof(T));
  return e != hipSuccess ? e : hipMemcpy(*out, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
}

int main() {
  // vertices with 2^30, no, 5, 5000 and 2^30 - 1 edges
  const int32_t big = 1 << 30;
  const std::vector<EdgePos_t> rows = {0, big, big, big + 5, big + 5005, 2147483647};
  const int32_t invalid = 5;
  // two transits a sample: 10 entries; 2^31; 2^30 + 5000; 10,000; 2^31 - 1 less 5005 and no vertex; none
  const std::vector<int32_t> transits = {2, 2, 0, 0, 0, 3, 3, 3, 4, invalid, -1, 1};
  const uint32_t n = 6;
  const uint32_t size_of[2][6] = {{10, 0, (1u << 30) + 5000, 10000, 2147483647u - big - 5005, 0}, {0, 0, 0, 0, 0, 0}};
  CSRPartition csr{};
  nd::MarkedSamples marked{};
  nd::TransitView tv{};
  uint32_t *sizes, *merged_sizes, *distinct, *too_long;
  EdgePos_t* d_rows;
  int32_t* d_transits;
  TRY(to_device(&d_rows, rows));
  TRY(to_device(&d_transits, transits));
  TRY(to_device(&sizes, std::vector<uint32_t>(n, 77u)));
  TRY(to_device(&merged_sizes, std::vector<uint32_t>(n, 77u)));
  TRY(to_device(&distinct, std::vector<uint32_t>(n, 77u)));
  TRY(to_device(&marked.count, std::vector<uint32_t>(2, 0u)));
  TRY(to_device(&marked.sample, std::vector<uint32_t>(n, 77u)));
  TRY(to_device(&marked.transits, std::vector<int32_t>(2 * n, 77)));
  TRY(to_device(&marked.transit_count, std::vector<uint2>(n)));
  TRY(hipHostMalloc((void**)&too_long, sizeof(uint32_t), hipHostMallocDefault));
  marked.stride = 2;
  csr.row_ptr = d_rows;
  csr.n_vertices = invalid;
  tv.base = d_transits;
  tv.stride = tv.count = 2;
  nd::MergedEdges merged{};
  merged.row_ptr = d_rows;
  for (int form = 0; form < 2; ++form) {
    TRY(hipMemset(marked.count, 0, 2 * sizeof(uint32_t)));
    *too_long = 0;
    for (int layer = 0; layer < 2; ++layer) {
      printf("form %d layer %d\n", form, layer);
      fflush(stdout);
      TRY(hipMemset(marked.count, 0, sizeof(uint32_t)));
      const dim3 grid((n + nd::kSortOutThreads / 64 - 1) / (nd::kSortOutThreads / 64)), block(nd::kSortOutThreads);
      if (form == 0)
        nd::sort_out_samples<<<grid, block>>>(csr, tv, n, invalid, nullptr, sizes, distinct, marked, too_long);
      else
        nd::sort_out_ranked<<<grid, block>>>(csr, merged, tv, n, invalid, sizes, merged_sizes, marked.count, marked.sample, too_long);
      TRY(hipGetLastError());
      TRY(hipDeviceSynchronize());
      CHECK(*too_long == 1);
      std::vector<uint32_t> got(n), count(2), listed(n);
      TRY(hipMemcpy(count.data(), marked.count, 2 * sizeof(uint32_t), hipMemcpyDeviceToHost));
      TRY(hipMemcpy(listed.data(), marked.sample, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
      CHECK(count[1] == 1);
      CHECK(layer == 0 ? count[0] <= 3 : count[0] == 0);
      for (uint32_t i = 0; i < count[0]; ++i) CHECK(listed[i] >= 2 && listed[i] <= 4);  // not the refused one
      for (int which = 0; which <= form; ++which) {
        TRY(hipMemcpy(got.data(), which ? merged_sizes : sizes, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
        // samples looked at while the refusal is found may count as empty already
        for (uint32_t i = 0; i < n; ++i) CHECK(got[i] == size_of[layer][i] || got[i] == 0);
      }
    }
  }
  printf("all as they should be\n");
  return 0;
}
