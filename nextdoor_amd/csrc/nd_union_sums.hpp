// The distinct vertices of a sample's collective neighbourhood weighted by degree^2, and draws from them
// (nd::apps::kDistinctByDegreeSquared).
//
// A draw is "the first distinct vertex, ascending, whose running sum of degree^2 exceeds a target".  Two ways
// there, chosen by the number of entries of the sample's neighbourhood:
//
//  * up to kSortedEntries: the entries are sorted in LDS (sorted_layer_kernel), repeats are neighbours then, and the
//    draws search the running sums.  Such a sample never leaves its workgroup.
//  * more: a bit per vertex (union_parts).  The vertex range is cut into parts of 16,384 vertices; a wavefront has the
//    2 KB of one sample's part in its registers.  What a vertex with many edges into a part contributes to it is the
//    same for every sample that holds the vertex, so it is a ready-made piece of 2 KB, built once per graph, that is
//    read and OR-ed in.  degree^2 of the marked vertices is summed over groups of 256 vertices by the matrix cores:
//    bits (16 samples x 256 vertices) times the 7-bit limbs of degree^2 (256 vertices x 9), a row of ones counting
//    the marked vertices on the way.  All of it is exact: i8 products, i32 sums of at most 256 * 127.
//
// R-MAT 20 (1 M vertices, 33 M edges), 4096 samples: see the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <string>

#include "nd_contract.hpp"
#include "nd_device_scan.hpp"

namespace nd {

// transits of sample s: base[s * stride + i], i < count
struct TransitView {
  const int32_t* base;
  uint32_t stride;
  uint32_t count;
};

constexpr uint32_t kMaxLayerTransits = 1024;  // transits of a sample

constexpr uint32_t kGroupWords = 8;                                // a group: 256 vertices
constexpr uint32_t kGroupsPerPart = 64;
constexpr uint32_t kPartWords = kGroupWords * kGroupsPerPart;      // 512: 8 per lane
constexpr uint32_t kPartVertices = kPartWords * 32u;               // 16,384
constexpr uint32_t kNoPiece = 0xFFFFFFFFu;

// ---- what is known of a graph's hubs ---------------------------------------------------------

// Vertices with kHubDegree edges or more have a row of cuts: where their (ascending) adjacency passes from part to
// part.  Where kPieceEntries of it or more lie in one part, the part's bits are there as a piece of kPartWords words.
// (A piece is 2 KB and two loads per lane; as many entries are 512 B, a load and an LDS atomic for every
// 64 of them.  R-MAT 20 with pieces from 128: 56 MB of them, 976 uses and 65 K entries a sample in its second layer;
// from 256: 27 MB, 870 and 90 K.)
constexpr uint32_t kHubDegree = 128, kPieceEntries = 128;
constexpr size_t kPieceBudgetBytes = (size_t)2 << 30, kCutBudgetBytes = (size_t)1 << 30;

// A hub and a part: the hub's first edge into the part or beyond, and its piece (kNoPiece: go through the entries).
// A row has one more for the end of the last part.
struct HubCut {
  EdgePos_t from;
  uint32_t piece;
};
struct HubTables {
  const int32_t* row_of;   // [vertices], -1: none
  const HubCut* cuts;      // [rows][parts + 1]
  const uint32_t* pieces;  // [.][kPartWords]
};

__device__ __forceinline__ EdgePos_t first_edge_from(const VertexID* __restrict__ edges, EdgePos_t lo, EdgePos_t hi,
                                                     uint32_t vertex) {
  while (lo < hi) {
    const EdgePos_t mid = lo + (hi - lo) / 2;
    if ((uint32_t)edges[mid] < vertex) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(256) void number_hubs(CSRPartition csr, uint32_t from_degree, int32_t* row_of,
                                                   int32_t* vertex_of, uint32_t* rows) {
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  const bool hub = v < (uint32_t)csr.n_vertices && (uint32_t)(csr.row_ptr[v + 1] - csr.row_ptr[v]) >= from_degree;
  const uint64_t mask = __ballot(hub);
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t base = 0;
  if (lane == 0 && mask) base = atomicAdd(rows, (uint32_t)__popcll(mask));
  base = __shfl(base, 0, kWave);
  const uint32_t row = base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
  if (v < (uint32_t)csr.n_vertices && row_of) row_of[v] = hub ? (int32_t)row : -1;
  if (hub && vertex_of) vertex_of[row] = (int32_t)v;
}

__global__ __launch_bounds__(256) void cut_hubs(CSRPartition csr, const int32_t* vertex_of, uint32_t rows,
                                                uint32_t parts, uint32_t part_vertices, HubCut* cuts) {
  const uint32_t row = blockIdx.x * 256u + threadIdx.x, part = blockIdx.y;
  if (row >= rows) return;
  const int32_t v = vertex_of[row];
  const EdgePos_t begin = csr.row_ptr[v], end = csr.row_ptr[v + 1];
  cuts[(size_t)row * (parts + 1) + part] =
      HubCut{part == parts ? end : first_edge_from(csr.edges, begin, end, part * part_vertices), kNoPiece};
}

// Numbers the pieces (those beyond `most` are left out), or, without place_of, only counts them.
__global__ __launch_bounds__(256) void number_pieces(HubCut* cuts, uint32_t rows, uint32_t parts, uint32_t from_entries,
                                                     uint32_t most, uint2* place_of, uint32_t* pieces) {
  const uint32_t row = blockIdx.x * 256u + threadIdx.x, part = blockIdx.y;
  HubCut* cut = cuts + (size_t)row * (parts + 1) + part;
  const bool dense = row < rows && (uint32_t)(cut[1].from - cut[0].from) >= from_entries;
  const uint64_t mask = __ballot(dense);
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t base = 0;
  if (lane == 0 && mask) base = atomicAdd(pieces, (uint32_t)__popcll(mask));
  const uint32_t piece = __shfl(base, 0, kWave) + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
  if (!dense || piece >= most || !place_of) return;
  cut->piece = piece;
  place_of[piece] = make_uint2(part, row);
}

__global__ __launch_bounds__(256) void fill_pieces(CSRPartition csr, const HubCut* cuts, uint32_t parts,
                                                   const uint2* place_of, uint32_t* pieces) {
  __shared__ uint32_t s_bits[kPartWords];
  for (uint32_t i = threadIdx.x; i < kPartWords; i += 256) s_bits[i] = 0;
  __syncthreads();
  const uint2 place = place_of[blockIdx.x];
  const HubCut* cut = cuts + (size_t)place.y * (parts + 1) + place.x;
  for (EdgePos_t e = cut[0].from + (EdgePos_t)threadIdx.x; e < cut[1].from; e += 256) {
    const uint32_t local = (uint32_t)csr.edges[e] - place.x * kPartVertices;
    atomicOr(&s_bits[local >> 5], 1u << (local & 31u));
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kPartWords; i += 256) pieces[(size_t)blockIdx.x * kPartWords + i] = s_bits[i];
}

// degree^2 as the matrix cores take it: for every group of 256 vertices four operands of 16 x 64 bytes, row 0 ones, row
// m the (m - 1)-th 7-bit limb; only the `rows` that the largest degree needs are stored (5 limbs up to 131 K edges).
// The 16 bytes of row m for quarter q of operand k are those of the vertices of word 2 q + k / 2 of the group in the order in
// which union_parts takes the word apart: byte b of dword d is bit 8 b + 4 (k & 1) + d.
constexpr uint32_t kMostSquareRows = 10;
__global__ __launch_bounds__(256) void square_limbs(CSRPartition csr, uint32_t rows, uint32_t* __restrict__ out) {
  const uint32_t group = blockIdx.x, k = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint32_t m = lane & 15u, q = lane >> 4;
  if (m >= rows) return;
  uint32_t dwords[4];
#pragma unroll
  for (uint32_t d = 0; d < 4; ++d) {
    dwords[d] = 0;
    for (uint32_t b = 0; b < 4; ++b) {
      const uint32_t v = group * 256u + (2u * q + (k >> 1)) * 32u + 8u * b + 4u * (k & 1u) + d;
      uint64_t degree = 0;
      if (v < (uint32_t)csr.n_vertices) degree = (uint64_t)(csr.row_ptr[v + 1] - csr.row_ptr[v]);
      const uint32_t byte = m == 0 ? 1u : (uint32_t)(degree * degree >> (7u * (m - 1u))) & 127u;
      dwords[d] |= byte << (8u * b);
    }
  }
  *(uint4*)(out + ((size_t)((group * 4u + k) * 4u + q) * rows + m) * 4u) = make_uint4(dwords[0], dwords[1], dwords[2], dwords[3]);
}

__global__ __launch_bounds__(256) void largest_degree(CSRPartition csr, uint32_t* largest) {
  uint32_t mine = 0;
  for (uint32_t v = blockIdx.x * 256u + threadIdx.x; v < (uint32_t)csr.n_vertices; v += gridDim.x * 256u)
    mine = max(mine, (uint32_t)(csr.row_ptr[v + 1] - csr.row_ptr[v]));
  for (int d = 32; d > 0; d >>= 1) mine = max(mine, (uint32_t)__shfl_xor(mine, d, kWave));
  if ((threadIdx.x & 63u) == 0) atomicMax(largest, mine);
}

// The tables of one graph.
class UnionTables {
 public:
  UnionTables() = default;
  UnionTables(const UnionTables&) = delete;
  UnionTables& operator=(const UnionTables&) = delete;
  ~UnionTables() { release(); }

  HubTables hubs{};
  const uint32_t* squares = nullptr;
  uint32_t square_rows = kMostSquareRows;
  uint32_t parts = 0;
  size_t pieces = 0;

  hipError_t build(const CSRPartition& csr, uint32_t words_per_sample) {
    release();
    parts = words_per_sample / kPartWords;
    const uint32_t V = (uint32_t)csr.n_vertices;
    uint32_t* counts = nullptr;
    hipError_t e = hipMalloc((void**)&counts, 2 * sizeof(uint32_t));
    if (e == hipSuccess) e = build_hubs(csr, V, counts);
    uint32_t largest = 0;
    if (e == hipSuccess) e = hipMemset(counts, 0, sizeof(uint32_t));
    if (e == hipSuccess) {
      largest_degree<<<dim3(256), dim3(256)>>>(csr, counts);
      e = hipMemcpy(&largest, counts, sizeof(largest), hipMemcpyDeviceToHost);
    }
    if (counts) (void)hipFree(counts);
    square_rows = 2;
    while (square_rows < kMostSquareRows && (uint64_t)largest * largest >> (7u * (square_rows - 1u)) != 0) square_rows++;
    if (e == hipSuccess) e = hipMalloc((void**)&d_squares_, (size_t)parts * kPartVertices * square_rows);
    if (e == hipSuccess) {
      square_limbs<<<dim3(parts * kGroupsPerPart), dim3(256)>>>(csr, square_rows, d_squares_);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) release();
    else squares = d_squares_;
    return e;
  }

  void release() {
    for (void* p : {(void*)d_row_of_, (void*)d_cuts_, (void*)d_pieces_, (void*)d_squares_})
      if (p) (void)hipFree(p);
    d_row_of_ = nullptr;
    d_cuts_ = nullptr;
    d_pieces_ = d_squares_ = nullptr;
    hubs = HubTables{};
    squares = nullptr;
    pieces = 0;
  }

 private:
  hipError_t build_hubs(const CSRPartition& csr, uint32_t V, uint32_t* counts) {
    uint32_t hub_degree = kHubDegree, piece_entries = kPieceEntries;
    if (const char* env = getenv("ND_DENSE_PIECE_ENTRIES")) {  // 0: no pieces; small: to exercise them on small graphs
      const long long v = atoll(env);
      piece_entries = v > 0 ? (uint32_t)v : kNoPiece;
      hub_degree = std::min(hub_degree, piece_entries);
    }
    uint32_t rows = 0;
    const dim3 over_vertices((V + 255u) / 256u);
    for (;; hub_degree *= 2) {  // fewer rows where the cuts of all of them would take too much
      hipError_t e = hipMemset(counts, 0, 2 * sizeof(uint32_t));
      if (e != hipSuccess) return e;
      number_hubs<<<over_vertices, dim3(256)>>>(csr, hub_degree, nullptr, nullptr, counts);
      e = hipMemcpy(&rows, counts, sizeof(rows), hipMemcpyDeviceToHost);
      if (e != hipSuccess) return e;
      if ((size_t)rows * (parts + 1) * sizeof(HubCut) <= kCutBudgetBytes) break;
    }
    if (rows == 0) return hipSuccess;
    int32_t* vertex_of = nullptr;
    uint2* place_of = nullptr;
    hipError_t e = hipMalloc((void**)&d_row_of_, sizeof(int32_t) * V);
    if (e == hipSuccess) e = hipMalloc((void**)&vertex_of, sizeof(int32_t) * rows);
    if (e == hipSuccess) e = hipMalloc((void**)&d_cuts_, sizeof(HubCut) * (size_t)rows * (parts + 1));
    if (e == hipSuccess) e = hipMemset(counts, 0, 2 * sizeof(uint32_t));
    if (e == hipSuccess) {
      number_hubs<<<over_vertices, dim3(256)>>>(csr, hub_degree, d_row_of_, vertex_of, counts);
      cut_hubs<<<dim3((rows + 255) / 256, parts + 1), dim3(256)>>>(csr, vertex_of, rows, parts, kPartVertices, d_cuts_);
      number_pieces<<<dim3((rows + 255) / 256, parts), dim3(256)>>>(d_cuts_, rows, parts, piece_entries, 0u, nullptr, counts + 1);
      uint32_t found = 0;
      e = hipMemcpy(&found, counts + 1, sizeof(found), hipMemcpyDeviceToHost);
      const uint32_t most = (uint32_t)std::min<size_t>(found, kPieceBudgetBytes / (sizeof(uint32_t) * kPartWords));
      if (e == hipSuccess && most > 0) e = hipMalloc((void**)&d_pieces_, sizeof(uint32_t) * kPartWords * (size_t)most);
      if (e == hipSuccess) e = hipMalloc((void**)&place_of, sizeof(uint2) * std::max(1u, most));
      if (e == hipSuccess) e = hipMemset(counts, 0, 2 * sizeof(uint32_t));
      if (e == hipSuccess) {
        number_pieces<<<dim3((rows + 255) / 256, parts), dim3(256)>>>(d_cuts_, rows, parts, piece_entries, most, place_of, counts + 1);
        if (most > 0) fill_pieces<<<dim3(most), dim3(256)>>>(csr, d_cuts_, parts, place_of, d_pieces_);
        e = hipGetLastError();
      }
      if (e == hipSuccess) e = hipDeviceSynchronize();
      pieces = most;
    }
    if (vertex_of) (void)hipFree(vertex_of);
    if (place_of) (void)hipFree(place_of);
    if (e == hipSuccess) hubs = HubTables{d_row_of_, d_cuts_, d_pieces_};
    return e;
  }

  int32_t* d_row_of_ = nullptr;
  HubCut* d_cuts_ = nullptr;
  uint32_t *d_pieces_ = nullptr, *d_squares_ = nullptr;
};

// ---- the samples of a layer, by the size of their neighbourhoods ------------------------------

// Entries a sample may have to be sorted in LDS.
constexpr uint32_t kSortedEntries = 4096;

// The samples with more, in whatever order they are found, and their transits without repeats: the first occurrences
// of hubs (as rows of the tables) from the front of the sample's stretch of `transits`, others from its back.
// A layer drawn with replacement by degree^2 repeats its hubs (34 distinct transits of 64 over R-MAT 20), and a vertex
// marks the same bits however often it is there.
struct MarkedSamples {
  uint32_t* count;      // and, next to it, whether a neighbourhood of this pass was too long (entries_or_refused)
  uint32_t* sample;     // [n]
  int32_t* transits;    // [n][stride]
  uint2* transit_count; // [n]: hubs, others
  uint32_t stride;
};

// What a sample's neighbourhood of `entries` counts for.  One of 2^31 entries or more is refused, and the pass with it: the host
// hears of it at the end (*too_long, host memory), and until then nobody works on it - it counts as empty, and so does
// every neighbourhood of the layers that follow (*refused).
__device__ __forceinline__ uint32_t entries_or_refused(uint64_t entries, uint32_t* refused, uint32_t* too_long) {
  const bool before = __hip_atomic_load(refused, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  if (entries >= (1ull << 31)) {
    *too_long = 1;
    __hip_atomic_store(refused, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  return before || entries >= (1ull << 31) ? 0u : (uint32_t)entries;
}

// A wavefront per sample: sizes[s] = entries of its neighbourhood, and which way it goes.  One atomic for the
// 16 samples of a workgroup: atomics on one address follow each other at 10 ns (4096 of them 41 us).
constexpr uint32_t kSortOutThreads = 1024;
__global__ __launch_bounds__(kSortOutThreads) void sort_out_samples(CSRPartition csr, TransitView tv, uint32_t n_samples,
                                                        int32_t invalid, const int32_t* __restrict__ row_of,
                                                        uint32_t* __restrict__ sizes, uint32_t* __restrict__ distinct,
                                                        MarkedSamples marked, uint32_t* __restrict__ too_long) {
  __shared__ uint32_t s_taken, s_base;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t s = blockIdx.x * (kSortOutThreads / 64u) + (threadIdx.x >> 6);
  if (threadIdx.x == 0) s_taken = 0;
  __syncthreads();
  const int32_t* transits = tv.base + (size_t)s * tv.stride;
  uint64_t sum = 0;
  for (uint32_t i = lane; i < tv.count && s < n_samples; i += 64u) {
    const int32_t t = transits[i];
    if (t != invalid && t != -1) sum += (uint64_t)(csr.row_ptr[t + 1] - csr.row_ptr[t]);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)sum, d, kWave), hi = __shfl_xor((uint32_t)(sum >> 32), d, kWave);
    sum += ((uint64_t)hi << 32) | lo;
  }
  // one lane asks, since the answer may change meanwhile
  const uint32_t size = (uint32_t)__shfl((int)(lane == 0 ? entries_or_refused(sum, marked.count + 1, too_long) : 0u), 0, kWave);
  uint32_t at = 0;
  if (lane == 0 && s < n_samples) {
    sizes[s] = size;
    distinct[s] = 0;
    if (size > kSortedEntries) at = atomicAdd(&s_taken, 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_taken) s_base = atomicAdd(marked.count, s_taken);
  __syncthreads();
  if (size <= kSortedEntries) return;  // the same for the whole wavefront
  at = s_base + __shfl(at, 0, kWave);
  if (lane == 0) marked.sample[at] = s;
  int32_t* mine = marked.transits + (size_t)at * marked.stride;
  uint32_t hubs = 0, others = 0;
  for (uint32_t c = 0; c < tv.count; c += 64u) {
    const uint32_t i = c + lane;
    const int32_t t = i < tv.count ? transits[i] : -1;
    bool first = t != invalid && t != -1;
    for (uint32_t before = 0; before <= c; before += 64u) {
      const int32_t others = before == c ? t : transits[before + lane];
      for (uint32_t j = 0; j < 64u; ++j)
        if (__builtin_amdgcn_readlane(others, (int)j) == t && before + j < i) first = false;
    }
    const int32_t row = first && row_of ? row_of[t] : -1;
    const uint64_t hub_mask = __ballot(first && row >= 0), other_mask = __ballot(first && row < 0);
    const uint64_t below = (1ull << lane) - 1ull;
    if (first && row >= 0) mine[hubs + (uint32_t)__popcll(hub_mask & below)] = row;
    if (first && row < 0) mine[marked.stride - 1u - (others + (uint32_t)__popcll(other_mask & below))] = t;
    hubs += (uint32_t)__popcll(hub_mask);
    others += (uint32_t)__popcll(other_mask);
  }
  if (lane == 0) marked.transit_count[at] = make_uint2(hubs, others);
}

// ---- small neighbourhoods: sorted in LDS ---------------------------------------------------

constexpr uint32_t kSortedThreads = 512, kSortedWaves = kSortedThreads / 64;
constexpr uint32_t kSortedChunk = 8;  // ids a running sum is kept for

// What next() receives as transitEdges there.
struct SortedByDegreeSquared {
  const uint32_t* ids;      // ascending, with repeats
  const uint64_t* through;  // degree^2 of the distinct ids of chunks 0..c
  uint32_t chunks;
  const EdgePos_t* row_ptr;

  __device__ __forceinline__ uint64_t total() const { return through[chunks - 1]; }

  // the smallest distinct id whose running sum of degree^2 exceeds target; target < total()
  __device__ inline VertexID first_exceeding(uint64_t target) const {
    uint32_t lo = 0, hi = chunks - 1;
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (through[mid] > target) hi = mid; else lo = mid + 1;
    }
    uint64_t running = lo ? through[lo - 1] : 0ull;
    uint32_t before = lo ? ids[lo * kSortedChunk - 1] : 0xFFFFFFFFu;
    for (uint32_t k = 0; k < kSortedChunk; ++k) {
      const uint32_t v = ids[lo * kSortedChunk + k];
      if (v == 0xFFFFFFFFu) break;
      if (v != before) {
        const uint64_t d = (uint64_t)(row_ptr[v + 1] - row_ptr[v]);
        running += d * d;
        if (running > target) return (VertexID)v;
      }
      before = v;
    }
    return -1;
  }
};

// The n ids at `ids` in ascending order, by passes over 7 bits, least significant first; returns where they are, there or in `other`.  A wavefront takes a stretch of the ids, 64 at a time: lanes with equal digits find each other by
// ballots, and what came before them is in the wavefront's counters.  (A bitonic sort, 78 stages of LDS reads and writes for
// 4096 ids, took 0.36 ms for the 4096 samples of R-MAT 20's first layer.)
constexpr uint32_t kSortedDigitBits = 7, kSortedDigits = 1u << kSortedDigitBits;
__device__ __forceinline__ uint32_t* sort_ids(uint32_t* ids, uint32_t* other, uint32_t (*s_count)[kSortedDigits],
                                              uint32_t* s_wave_count, uint32_t n, uint32_t bits) {
  constexpr uint32_t kThreads = kSortedThreads, kWaves = kSortedWaves;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t stretch = ((n + kWaves - 1) / kWaves + 63u) & ~63u;
  const uint32_t begin = wave * stretch, end = begin + stretch < n ? begin + stretch : n;
  for (uint32_t shift = 0; shift < bits; shift += kSortedDigitBits) {
    for (uint32_t i = threadIdx.x; i < kWaves * kSortedDigits; i += kThreads) (&s_count[0][0])[i] = 0;
    __syncthreads();
    for (uint32_t i = begin + lane; i < end; i += 64u) atomicAdd(&s_count[wave][ids[i] >> shift & (kSortedDigits - 1u)], 1u);
    __syncthreads();
    // starts: by digit, then by wavefront; lane t has two counters that follow each other in that order
    const uint32_t digit = threadIdx.x / (kWaves / 2u), of = threadIdx.x % (kWaves / 2u) * 2u;
    const uint32_t a = s_count[of][digit], b = s_count[of + 1u][digit];
    const uint32_t through = wave_inclusive_scan(a + b);
    if (lane == 63) s_wave_count[wave] = through;
    __syncthreads();
    uint32_t before = through - a - b;
    for (uint32_t w = 0; w < wave; ++w) before += s_wave_count[w];
    s_count[of][digit] = before;
    s_count[of + 1u][digit] = before + a;
    __syncthreads();
    for (uint32_t i0 = begin; i0 < end; i0 += 64u) {
      const bool here = i0 + lane < end;
      const uint32_t id = here ? ids[i0 + lane] : 0u, d = id >> shift & (kSortedDigits - 1u);
      uint64_t same = __ballot(here);
#pragma unroll
      for (uint32_t bit = 0; bit < kSortedDigitBits; ++bit) {
        const bool set = d >> bit & 1u;
        const uint64_t with = __ballot(set);
        same &= set ? with : ~with;
      }
      if (here) {
        const uint32_t rank = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        const uint32_t to = s_count[wave][d] + rank;
        other[to] = id;
        if (rank == 0) s_count[wave][d] = to + (uint32_t)__popcll(same);
      }
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t* const sorted = other;
    other = ids;
    ids = sorted;
  }
  return ids;
}

// A workgroup per sample: fetches the entries, sorts them, adds degree^2 up over the distinct ones and draws.
template <class Draw>
__device__ __forceinline__ void sorted_layer(const CSRPartition& csr, const int32_t* transits, uint32_t n_transits,
                                             int32_t invalid, uint32_t size, uint32_t* __restrict__ distinct_out, Draw draw) {
  __shared__ uint32_t s_buffers[2][kSortedEntries];
  __shared__ uint32_t s_count[kSortedWaves][kSortedDigits];
  __shared__ uint64_t s_through[kSortedEntries / kSortedChunk];
  __shared__ uint64_t s_wave_sum[kSortedThreads / 64];
  __shared__ uint32_t s_wave_count[kSortedThreads / 64];
  static_assert(kSortedEntries >= 2 * kMaxLayerTransits, "room for the transits");
  uint32_t* s_start = s_buffers[1];  // of the transits; until the sort needs the room
  EdgePos_t* s_edge = (EdgePos_t*)s_start + kMaxLayerTransits;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t carry = 0;
  for (uint32_t c = 0; c < n_transits; c += kSortedThreads) {
    const uint32_t i = c + threadIdx.x;
    const int32_t t = i < n_transits ? transits[i] : -1;
    EdgePos_t begin = 0;
    uint32_t degree = 0;
    if (t != invalid && t != -1) {
      begin = csr.row_ptr[t];
      degree = (uint32_t)(csr.row_ptr[t + 1] - begin);
    }
    const uint32_t through = wave_inclusive_scan(degree);
    if (lane == 63) s_wave_count[wave] = through;
    __syncthreads();
    uint32_t before = carry;
    for (uint32_t w = 0; w < kSortedThreads / 64; ++w) {
      if (w < wave) before += s_wave_count[w];
      carry += s_wave_count[w];
    }
    if (i < n_transits) {
      s_start[i] = before + through - degree;
      s_edge[i] = begin;
    }
    __syncthreads();
  }
  for (uint32_t e = threadIdx.x; e < size; e += kSortedThreads) {
    uint32_t lo = 0, hi = n_transits;  // the last transit that starts at e or before (empty ones start where the next does)
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (s_start[mid] <= e) lo = mid; else hi = mid;
    }
    s_buffers[0][e] = (uint32_t)csr.edges[s_edge[lo] + (EdgePos_t)(e - s_start[lo])];
  }
  __syncthreads();
  uint32_t* s_ids = sort_ids(s_buffers[0], s_buffers[1], s_count, s_wave_count, size, 32u - (uint32_t)__clz(csr.n_vertices));
  const uint32_t chunks = size ? (size + kSortedChunk - 1) / kSortedChunk : 1u;
  if (size + threadIdx.x < chunks * kSortedChunk) s_ids[size + threadIdx.x] = 0xFFFFFFFFu;
  __syncthreads();
  // a chunk a lane
  static_assert(kSortedEntries == kSortedThreads * kSortedChunk, "a lane per chunk");
  uint64_t sum = 0;
  uint32_t count = 0;
  if (threadIdx.x < chunks) {
    uint32_t before = threadIdx.x ? s_ids[threadIdx.x * kSortedChunk - 1] : 0xFFFFFFFFu;
#pragma unroll
    for (uint32_t i = 0; i < kSortedChunk; ++i) {
      const uint32_t v = s_ids[threadIdx.x * kSortedChunk + i];
      if (v != 0xFFFFFFFFu && v != before) {
        const uint64_t d = (uint64_t)(csr.row_ptr[v + 1] - csr.row_ptr[v]);
        sum += d * d;
        count++;
      }
      before = v;
    }
  }
  const uint64_t through = wave_inclusive_scan_u64(sum);
  for (int d = 32; d > 0; d >>= 1) count += __shfl_xor(count, d, kWave);
  if (lane == 63) {
    s_wave_sum[wave] = through;
    s_wave_count[wave] = count;
  }
  __syncthreads();
  uint64_t before = through;
  uint32_t distinct = 0;
  for (uint32_t w = 0; w < kSortedWaves; ++w) {
    if (w < wave) before += s_wave_sum[w];
    distinct += s_wave_count[w];
  }
  s_through[threadIdx.x] = before;
  __syncthreads();
  if (threadIdx.x == 0) *distinct_out = distinct;
  SortedByDegreeSquared view{s_ids, s_through, chunks, csr.row_ptr};
  draw(view, distinct);
}

// ---- large neighbourhoods: a bit per vertex ---------------------------------------------------

constexpr uint32_t kXcdCount = 8;
constexpr uint32_t kUnionThreads = 256, kUnionWaves = kUnionThreads / 64;
constexpr uint32_t kUnionSlices = 256;                   // workgroups that share the samples of a part
// degree^2 is summed over halves of parts, so that two workgroups are on a compute unit and one works while the other waits at a barrier.
constexpr uint32_t kHalvesOfPart = 2, kGroupsPerHalf = kGroupsPerPart / kHalvesOfPart, kHalfWords = kPartWords / kHalvesOfPart;
constexpr uint32_t kSumThreads = 512, kSumWaves = kSumThreads / 64;
constexpr uint32_t kSumSamples = 16;                     // the columns of a matrix product
constexpr uint32_t kSumGroups = kGroupsPerHalf / kSumWaves;  // of a wavefront
constexpr uint32_t kSumPitch = kHalfWords + 8;           // words between samples in LDS: spreads them over the banks
constexpr uint32_t kSumSlices = 16;                      // workgroups that share the samples of a half
static_assert(kSumSamples == 2 * kSumWaves && kHalfWords == 4 * 64 && kGroupsPerHalf == 32, "two samples a wavefront");

typedef int32_t IntVector4 __attribute__((ext_vector_type(4)));

// Lanes of `mask`: their pieces into this lane's eight words, four pieces' loads under way at a time (a lane
// that stands in where fewer than four are left repeats one: OR does not mind).
__device__ __forceinline__ void or_pieces(uint64_t mask, uint32_t piece, const uint32_t* __restrict__ pieces, uint32_t lane,
                                          uint4& low, uint4& high) {
  while (mask) {
    const uint4* from[4];  // the same for every lane
    uint32_t at = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      if (mask) {
        at = (uint32_t)__builtin_ctzll(mask);
        mask &= mask - 1ull;
      }
      const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)piece, (int)at);
      from[k] = (const uint4*)(pieces + (size_t)p * kPartWords);
    }
    uint4 a[4], b[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      a[k] = from[k][2u * lane];
      b[k] = from[k][2u * lane + 1u];
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      low.x |= a[k].x; low.y |= a[k].y; low.z |= a[k].z; low.w |= a[k].w;
      high.x |= b[k].x; high.y |= b[k].y; high.z |= b[k].z; high.w |= b[k].w;
    }
  }
}

// Every lane's entries [from, from + length) into the wavefront's bits, eight lanes' at a time.
__device__ __forceinline__ void mark_entries(const VertexID* __restrict__ edges, EdgePos_t from, uint32_t length, uint32_t lane,
                                             uint32_t* bits) {
  uint64_t mask = __ballot(length != 0);
  while (mask) {
    EdgePos_t first[8];
    uint32_t count[8], v[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
      first[k] = 0;
      count[k] = 0;
      if (mask) {
        const int at = __builtin_ctzll(mask);
        mask &= mask - 1ull;
        first[k] = (EdgePos_t)__builtin_amdgcn_readlane((int)from, at);
        count[k] = (uint32_t)__builtin_amdgcn_readlane((int)length, at);
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) v[k] = lane < count[k] ? (uint32_t)(edges + first[k])[lane] : 0u;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k)
      if (lane < count[k]) atomicOr(&bits[(v[k] % kPartVertices) >> 5], 1u << (v[k] & 31u));
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k)
      for (uint32_t e = lane + 64u; e < count[k]; e += 64u) {
        const uint32_t more = (uint32_t)(edges + first[k])[e];
        atomicOr(&bits[(more % kPartVertices) >> 5], 1u << (more & 31u));
      }
  }
}

// The bits of the marked samples: bitmap[at * words_per_sample + ...], at = the sample's place among them.  A wavefront
// takes one part of one sample after the other, what is known of the next one's transits on its way meanwhile: pieces are
// OR-ed into registers, entries marked in 2 KB of LDS.  Bound by what L2 gives a compute unit (R-MAT 20, second layer: 9 GB of
// pieces and entries).  A die's L2 has the pieces of the parts its own workgroups are at: blockIdx % 8, the die
// a workgroup is put on, chooses the part (0.9 MB of pieces a part); every eight parts one die's turn starts at another
// of them, since how full a part is goes by the bits of its number (R-MAT).
__global__ __launch_bounds__(kUnionThreads, 6) void union_parts(CSRPartition csr, HubTables hubs, uint32_t parts,
                                                                MarkedSamples marked, uint32_t words_per_sample,
                                                                uint32_t* __restrict__ bitmap) {
  __shared__ __align__(16) uint32_t s_bits[kUnionWaves][kPartWords];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t turn = blockIdx.x / kXcdCount, eight = turn / kUnionSlices, slice = turn % kUnionSlices;
  const uint32_t part = kXcdCount * eight + (blockIdx.x + 3u * eight) % kXcdCount;
  if (part >= parts) return;
  const uint32_t n = *marked.count;
  uint32_t* mine = s_bits[wave];
  uint4* my_lines = (uint4*)mine + 2u * lane;
  // hub c + lane of sample at: its piece, or its entries
  auto look_up = [&](uint32_t at, uint32_t c, uint32_t hubs_here, uint32_t* piece, EdgePos_t* from, uint32_t* length) {
    *piece = kNoPiece;
    *length = 0;
    *from = 0;
    if (c + lane >= hubs_here) return;
    const uint32_t row = (uint32_t)marked.transits[(size_t)at * marked.stride + c + lane];
    const HubCut* cut = hubs.cuts + (size_t)row * (parts + 1) + part;
    const HubCut here = cut[0], next = cut[1];
    *piece = here.piece;
    *from = here.from;
    *length = here.piece == kNoPiece ? (uint32_t)(next.from - here.from) : 0u;
  };
  constexpr uint32_t kStride = kUnionSlices * kUnionWaves;
  uint32_t at = slice * kUnionWaves + wave;
  uint2 counts = at < n ? marked.transit_count[at] : make_uint2(0u, 0u);
  uint32_t piece, length;
  EdgePos_t from;
  look_up(at, 0, counts.x, &piece, &from, &length);
  while (at < n) {
    const uint32_t next_at = at + kStride;
    const uint2 next_counts = next_at < n ? marked.transit_count[next_at] : make_uint2(0u, 0u);
    uint32_t next_piece, next_length;
    EdgePos_t next_from;
    look_up(next_at, 0, next_counts.x, &next_piece, &next_from, &next_length);
    uint4 low = make_uint4(0u, 0u, 0u, 0u), high = low;
    my_lines[0] = low;
    my_lines[1] = high;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t c = 0;;) {
      mark_entries(csr.edges, from, length, lane, mine);
      or_pieces(__ballot(piece != kNoPiece), piece, hubs.pieces, lane, low, high);
      c += 64u;
      if (c >= counts.x) break;
      look_up(at, c, counts.x, &piece, &from, &length);
    }
    for (uint32_t c = 0; c < counts.y; c += 64u) {
      uint32_t more = 0;
      EdgePos_t first = 0;
      if (c + lane < counts.y) {
        const int32_t v = marked.transits[(size_t)at * marked.stride + marked.stride - 1u - (c + lane)];
        const EdgePos_t end = csr.row_ptr[v + 1];
        first = first_edge_from(csr.edges, csr.row_ptr[v], end, part * kPartVertices);
        more = (uint32_t)(first_edge_from(csr.edges, first, end, (part + 1) * kPartVertices) - first);
      }
      mark_entries(csr.edges, first, more, lane, mine);
    }
    __builtin_amdgcn_wave_barrier();
    const uint4 a = my_lines[0], b = my_lines[1];
    uint4* out = (uint4*)(bitmap + (size_t)at * words_per_sample + (size_t)part * kPartWords) + 2u * lane;
    out[0] = make_uint4(low.x | a.x, low.y | a.y, low.z | a.z, low.w | a.w);
    out[1] = make_uint4(high.x | b.x, high.y | b.y, high.z | b.z, high.w | b.w);
    at = next_at;
    counts = next_counts;
    piece = next_piece;
    from = next_from;
    length = next_length;
  }
}

// degree^2 over the bits: a workgroup has half of a part, a wavefront four of its 32 groups, whose operands stay in its registers
// while the samples go past them, 16 at a time.
//   group_through[(at * halves + half) * 32 + g]         degree^2 of the marked vertices of groups 0..g of the half
//   half_total[at * halves + half]                       of the whole half
//   distinct[sample] += marked vertices
// Bound by instructions (taking the bits apart is half of them) and the two barriers of a block of samples: second layer of 4096
// samples over R-MAT 20 (0.5 GB of bits) 0.196 ms, over 0.9 M vertices 0.182; with a whole part a workgroup of 1024, one to a
// compute unit, 0.244 and 0.243.
__global__ __launch_bounds__(kSumThreads, 4) void union_sums(const uint32_t* __restrict__ squares, uint32_t square_rows,
                                                             uint32_t halves, MarkedSamples marked,
                                                             uint32_t words_per_sample,
                                                             const uint32_t* __restrict__ bitmap,
                                                             uint64_t* __restrict__ group_through,
                                                             uint64_t* __restrict__ half_total,
                                                             uint32_t* __restrict__ distinct) {
  __shared__ __align__(16) uint32_t s_bits[2][kSumSamples * kSumPitch];
  __shared__ uint64_t s_sums[2][2][kSumSamples * (kGroupsPerHalf + 1)];
  __shared__ uint32_t s_top[2][kSumSamples * (kGroupsPerHalf + 1)];
  __shared__ uint32_t s_marked[2][kSumSamples];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t half = blockIdx.x / kSumSlices, slice = blockIdx.x % kSumSlices;
  const uint32_t n = *marked.count;
  const uint32_t blocks = (n + kSumSamples - 1) / kSumSamples;
  const uint32_t column = lane & 15u, q = lane >> 4;
  IntVector4 limbs[kSumGroups][4];  // this lane's row is `column`
#pragma unroll
  for (uint32_t g = 0; g < kSumGroups; ++g)
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      limbs[g][k] = IntVector4{0, 0, 0, 0};
      if (column < square_rows && slice < blocks)
        limbs[g][k] = *((const IntVector4*)squares +
                        ((size_t)(half * kGroupsPerHalf + wave * kSumGroups + g) * 16u + 4u * k + q) * square_rows + column);
    }
  if (threadIdx.x < 2 * kSumSamples) (&s_marked[0][0])[threadIdx.x] = 0;
  __syncthreads();
  // A wavefront brings the bits of two samples into LDS, 1 KB each; those of the next two blocks are on their way while one is worked
  // on.
  const uint4* lines = (const uint4*)(bitmap + (size_t)half * kHalfWords) + lane;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  uint4 one[2] = {zero, zero}, two[2] = {zero, zero};
  auto fetch = [&](uint32_t block, uint4& a, uint4& b) {
    const uint32_t at = block * kSumSamples + 2u * wave;
    // what the lane had is no less of a sample: nobody reads its sums
    if (at < n) a = lines[(size_t)at * (words_per_sample / 4u)];
    if (at + 1u < n) b = lines[(size_t)(at + 1u) * (words_per_sample / 4u)];
  };
  fetch(slice, one[0], two[0]);
  fetch(slice + kSumSlices, one[1], two[1]);
  for (uint32_t block0 = slice; block0 < blocks; block0 += 2u * kSumSlices)
#pragma unroll
  for (uint32_t turn = 0; turn < 2; ++turn) {
    const uint32_t block = block0 + turn * kSumSlices;
    if (block >= blocks) break;
    ((uint4*)(s_bits[turn] + 2u * wave * kSumPitch))[lane] = one[turn];
    ((uint4*)(s_bits[turn] + (2u * wave + 1u) * kSumPitch))[lane] = two[turn];
    fetch(block + 2u * kSumSlices, one[turn], two[turn]);
    __syncthreads();
    uint2 now[kSumGroups];
#pragma unroll
    for (uint32_t g = 0; g < kSumGroups; ++g)
      now[g] = *(const uint2*)(s_bits[turn] + column * kSumPitch + (wave * kSumGroups + g) * kGroupWords + 2u * q);
    uint32_t count = 0;
#pragma unroll
    for (uint32_t g = 0; g < kSumGroups; ++g) {
      IntVector4 sums = {0, 0, 0, 0};
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t word = (k < 2 ? now[g].x : now[g].y) >> (4u * (k & 1u));
        const IntVector4 bits = {(int32_t)(word & 0x01010101u), (int32_t)(word >> 1 & 0x01010101u),
                                 (int32_t)(word >> 2 & 0x01010101u), (int32_t)(word >> 3 & 0x01010101u)};
        sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(limbs[g][k], bits, sums, 0, 0, 0);
      }
      // this lane: rows 4 q .. 4 q + 3 of sample `column`; row 0 the count, row m limb m - 1, none above 256 * 127.  What
      // it adds up to (for q = 0, 128 times that) lies side by side with the shares of the other lanes of the sample.
      const uint32_t first = q == 0 ? 0u : (uint32_t)sums[0];
      count += (uint32_t)sums[0];
      const uint64_t share = (uint64_t)(uint32_t)sums[3] * (1u << 21) + (first + ((uint32_t)sums[1] << 7) + ((uint32_t)sums[2] << 14));
      const uint32_t to = column * (kGroupsPerHalf + 1) + wave * kSumGroups + g;
      if (q < 2) s_sums[turn][q][to] = share;
      if (q == 2 && square_rows > 8) s_top[turn][to] = (uint32_t)sums[0] + ((uint32_t)sums[1] << 7);
    }
    if (q == 0 && count) atomicAdd(&s_marked[turn][column], count);
    __syncthreads();
    // half of the wavefront has one sample, half the other
    const uint32_t sample = 2u * wave + (lane >> 5), group = lane & 31u, at = block * kSumSamples + sample;
    const uint32_t of = sample * (kGroupsPerHalf + 1) + group;
    uint64_t sum = (s_sums[turn][0][of] >> 7) + (s_sums[turn][1][of] << 21);
    if (square_rows > 8) sum += (uint64_t)s_top[turn][of] << 49;
    uint64_t through = wave_inclusive_scan_u64(sum);
    const uint64_t others = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(through >> 32), 31) << 32 |
                            (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)through, 31);
    if (lane >= 32) through -= others;
    if (at < n) {
      const size_t place = (size_t)at * halves + half;
      group_through[place * kGroupsPerHalf + group] = through;
      if (group == kGroupsPerHalf - 1u) half_total[place] = through;
      if (group == 0 && s_marked[turn][sample]) atomicAdd(&distinct[marked.sample[at]], s_marked[turn][sample]);
    }
    if (group == 0) s_marked[turn][sample] = 0;
  }
}

// One wavefront per marked sample: half_before[at * (halves + 1) + p] = degree^2 of the marked vertices
// of the sample's halves before p; entry `halves` is the sample's total.
__global__ __launch_bounds__(64) void sample_half_sums(const uint64_t* __restrict__ half_total, uint32_t halves,
                                                       const uint32_t* __restrict__ n_marked,
                                                       uint64_t* __restrict__ half_before) {
  const uint32_t s = blockIdx.x, lane = threadIdx.x;
  if (s >= *n_marked) return;
  uint64_t carry = 0;
  for (uint32_t p0 = 0; p0 < halves; p0 += 64) {
    const uint32_t p = p0 + lane;
    const uint64_t mine = p < halves ? half_total[(size_t)s * halves + p] : 0ull;
    const uint64_t through = wave_inclusive_scan_u64(mine);
    if (p < halves) half_before[(size_t)s * (halves + 1) + p] = carry + through - mine;
    const uint32_t lo = __shfl((uint32_t)through, 63, kWave), hi = __shfl((uint32_t)(through >> 32), 63, kWave);
    carry += ((uint64_t)hi << 32) | lo;
  }
  if (lane == 0) half_before[(size_t)s * (halves + 1) + halves] = carry;
}

// What next() receives as transitEdges for a marked sample.  A lane searches for itself: 64 draws' misses are then under
// way in a wavefront (R-MAT 20, 262 K draws: 0.058 ms; a wavefront to a draw, its lanes searching together: 0.198).
struct MarkedByDegreeSquared {
  const uint32_t* bits;           // the sample's bitmap
  const uint64_t* half_before;    // the sample's halves + 1 entries
  const uint64_t* group_through;  // the sample's halves * 32 entries
  const EdgePos_t* row_ptr;
  uint32_t halves;

  __device__ __forceinline__ uint64_t total() const { return half_before[halves]; }

  // the smallest marked vertex whose running sum of degree^2 (marked vertices ascending) exceeds target;
  // target < total()
  __device__ inline VertexID first_exceeding(uint64_t target) const {
    uint32_t half = 0, end = halves;  // the last half whose sum-before is <= target
    while (end - half > 1) {
      const uint32_t mid = half + (end - half) / 2;
      if (half_before[mid] <= target) half = mid; else end = mid;
    }
    target -= half_before[half];
    const uint64_t* through = group_through + (size_t)half * kGroupsPerHalf;
    uint32_t group = 0, last = kGroupsPerHalf - 1;  // the first group whose sum-through exceeds it
    while (group < last) {
      const uint32_t mid = group + (last - group) / 2;
      if (through[mid] > target) last = mid; else group = mid + 1;
    }
    if (group) target -= through[group - 1];
    const uint32_t first_word = half * kHalfWords + group * kGroupWords;
    uint64_t running = 0;
    for (uint32_t k = 0; k < kGroupWords; ++k)
      for (uint32_t word = bits[first_word + k]; word; word &= word - 1u) {
        const uint32_t v = (first_word + k) * 32u + (uint32_t)__builtin_ctz(word);
        const uint64_t d = (uint64_t)(row_ptr[v + 1] - row_ptr[v]);
        running += d * d;
        if (running > target) return (VertexID)v;
      }
    return -1;
  }
};

}  // namespace nd
