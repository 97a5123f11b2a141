// Layer-wise (CollectiveNeighborhood) sampling engine for one MI355X (gfx950, wave64).
//
// Reference behaviour this covers (file:line in the reference tree):
//   collective branch of doTransitParallelSampling   src/nextdoor.cu:2402-2453, 2475-2496, 2900-2923
//   collectiveNeighbrsSize                           src/nextdoor.cu:1206-1246  -> collective_sizes
//   collectiveNeighborhood                           src/nextdoor.cu:1248-1283  -> collective_build
//   sampleParallelKernel, Collective branch          src/nextdoor.cu:1394-1446, 1485-1487 -> layer_execute_kernel
//
// Per layer k, for every sample s: its transits are the initial vertices (k = 0) or the
// layer k-1 segment of its result row; the collective neighbourhood is the concatenation
// of the transits' adjacencies; next() runs once per (sample, nbr < stepSize(k)) and its
// result goes to final[s * F + stepSizeAtStep(k-1) + nbr].
//
// Differences that are deliberate:
//  * The reference sizes the neighbourhood with a global atomic (offsets in arrival order),
//    cudaMallocs it inside the step loop and never hands it to next() (transitEdges is
//    nullptr, nextdoor.cu:1441-1446).  Here offsets are an exclusive scan over samples
//    (deterministic), the buffers are grown once and reused, and next() receives the
//    neighbourhood in the form the app declares (nd::apps::NeighborhoodForm).
//  * The importance forms never store the concatenation.  kDistinctByDegreeSquared (nd_union_sums.hpp): small
//    neighbourhoods are sorted in LDS; of the others every part of the vertex range becomes bits, OR-ed from the
//    hubs' ready-made pieces and marked entry by entry, whose degree^2 the matrix cores sum by group; a draw searches
//    the sums.
//  * kRankedByLadiesImportance: each entry carries (weight * (1 / rowsum(transit)))^2 as a 2^53 fixed-point integer,
//    worked out once per graph with parallel edges merged.  Small neighbourhoods are summed, keyed
//    (Efraimidis-Spirakis) and sorted in LDS by one workgroup.  Of the others the terms of a vertex are summed in LDS
//    stretch by stretch, its key is formed from the sum as it leaves LDS (the only thing stored per sample and
//    vertex), a radix select keeps the few entries that can be among the sample's first picks, and stable sorts
//    order those by descending key.
//  * Samples are processed in chunks whose concatenated neighbourhoods fit a fixed budget
//    of entries, so a layer whose frontier sits on hubs cannot outgrow memory.
//  * Random numbers: Philox keyed by the output slot s * stepSize(k) + nbr and the layer.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <type_traits>
#include <vector>

#include "nd_apps_layer.hpp"
#include "nd_contract.hpp"
#include "nd_device_graph.hpp"
#include "nd_engine.hpp"
#include "nd_radix_sort.hpp"
#include "nd_union_sums.hpp"

namespace nd {

// One wave per sample: sum of the degrees of its valid transits.
__global__ __launch_bounds__(256) void collective_sizes(CSRPartition csr, TransitView tv, uint32_t n_samples,
                                                        int32_t invalid, uint32_t* __restrict__ sizes) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t s = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (s >= n_samples) return;
  const int32_t* transits = tv.base + (size_t)s * tv.stride;
  uint64_t sum = 0;
  for (uint32_t i = lane; i < tv.count; i += 64u) {
    const int32_t t = transits[i];
    if (t != invalid && t != -1) sum += (uint64_t)(csr.row_ptr[t + 1] - csr.row_ptr[t]);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint32_t lo = __shfl_down((uint32_t)sum, d, 64);
    const uint32_t hi = __shfl_down((uint32_t)(sum >> 32), d, 64);
    sum += ((uint64_t)hi << 32) | lo;
  }
  // sizes are 32-bit; a neighbourhood that does not fit saturates and the host refuses it
  if (lane == 0) sizes[s] = sum > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)sum;
}

// Entries of a sample's concatenation one workgroup of collective_build copies; samples
// with longer neighbourhoods are spread over several workgroups.
constexpr uint32_t kBuildItemEntries = 8192;

// Copies the adjacencies of every sample's transits, in transit order, to
// cols[offsets[s] ...] (and weights).
// Work items: item_start[s] = number of items of the samples before s (exclusive scan of
// ceil(size_s / kBuildItemEntries), with the total at [n_samples]); workgroup b serves the
// sample whose item range holds b and the b - item_start[s]-th stretch of its entries.
__global__ __launch_bounds__(256) void collective_build(CSRPartition csr, TransitView tv, int32_t invalid,
                                                        const uint32_t* __restrict__ offsets,
                                                        const uint32_t* __restrict__ item_start, uint32_t n_samples,
                                                        int32_t* __restrict__ cols, float* __restrict__ weights,
                                                        uint32_t* __restrict__ row_offsets) {
  __shared__ uint32_t s_start[kMaxLayerTransits + 1];  // start of transit i inside the sample's concatenation
  __shared__ uint32_t s_scan_tmp[4];
  // sample of this work item: last s with item_start[s] <= blockIdx.x
  uint32_t lo_s = 0, hi_s = n_samples;
  while (hi_s - lo_s > 1) {
    const uint32_t mid = lo_s + (hi_s - lo_s) / 2;
    if (item_start[mid] <= blockIdx.x) lo_s = mid; else hi_s = mid;
  }
  const uint32_t s = lo_s;
  const uint32_t item = blockIdx.x - item_start[s];
  const int32_t* transits = tv.base + (size_t)s * tv.stride;
  uint32_t carry = 0;
  for (uint32_t chunk = 0; chunk < tv.count; chunk += 256) {
    const uint32_t i = chunk + threadIdx.x;
    uint32_t deg = 0;
    if (i < tv.count) {
      const int32_t t = transits[i];
      if (t != invalid && t != -1) deg = (uint32_t)(csr.row_ptr[t + 1] - csr.row_ptr[t]);
    }
    uint32_t total;
    const uint32_t excl = block_exclusive_scan_256(deg, s_scan_tmp, &total);
    if (i < tv.count) s_start[i] = carry + excl;
    carry += total;
  }
  if (threadIdx.x == 0) s_start[tv.count] = carry;
  __syncthreads();
  const uint32_t base = offsets[s];
  const uint32_t size = s_start[tv.count];
  if (row_offsets && item == 0)
    for (uint32_t i = threadIdx.x; i < tv.count; i += 256) row_offsets[(size_t)s * tv.count + i] = s_start[i];
  const uint32_t first = item * kBuildItemEntries;
  const uint32_t last = first + kBuildItemEntries < size ? first + kBuildItemEntries : size;
  uint32_t cur = 0;  // transit of the previous entry this lane copied: the next one is usually the same
  for (uint32_t e = first + threadIdx.x; e < last; e += 256) {
    if (!(s_start[cur] <= e && e < s_start[cur + 1])) {
      // transit whose range holds e: last i with s_start[i] <= e
      uint32_t lo = 0, hi = tv.count;
      while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (s_start[mid] <= e) lo = mid; else hi = mid;
      }
      cur = lo;
    }
    const int32_t t = transits[cur];
    const EdgePos_t src = csr.row_ptr[t] + (EdgePos_t)(e - s_start[cur]);
    cols[base + e] = csr.edges[src];
    if (weights) weights[base + e] = csr.weights[src];
  }
}

// (weight * (1 / rowsum))^2 as a 2^53 fixed-point integer, truncated: sums of up to 1024 of
// them fit 64 bits and, unlike float sums, do not depend on the order of the additions.
// A float in (0, 1) is (2^23 + m) * 2^(e - 150) with exponent field e and mantissa m, so the
// product with 2^53 is the 24-bit mantissa shifted by e - 97; the same integer as
// (unsigned long long)(term * 2^53f), without a float -> 64-bit conversion.
__host__ __device__ __forceinline__ unsigned long long importance_term_fixed(float term) {
  uint32_t bits;
  __builtin_memcpy(&bits, &term, sizeof(bits));
  if ((int32_t)bits <= 0) return 0ull;  // zero or negative
  if (bits >= 0x3F800000u) return bits > 0x7F800000u ? 0ull : 1ull << 53;  // >= 1 (NaN: 0)
  const uint32_t e = bits >> 23;
  const uint32_t mantissa = (bits & 0x7FFFFFu) | (e ? 0x800000u : 0u);
  const int shift = (int)e - 97;
  if (shift >= 0) return (unsigned long long)mantissa << shift;
  return shift > -24 ? (unsigned long long)(mantissa >> -shift) : 0ull;
}

// ---- LADIES form: the importance sums of a collective neighbourhood, stretch by stretch ----
//
// What an entry (u, v) contributes to v does not depend on the sample: (weight * inverse_row_sum[u])^2 as a 2^53
// fixed-point integer.  So the terms are worked out once per graph, and parallel edges (hub pairs are joined by
// thousands: 4.5 M entries of a sample's second layer over 500 K vertices are 1.5 M pairs) are one entry with the sum of
// theirs - integers, to which the order of the additions does not matter.
struct MergedEdges {
  const EdgePos_t* row_ptr;          // [vertices + 1]
  const VertexID* ids;               // ascending and without repeats in every row
  const unsigned long long* terms;
  bool zero_terms;                   // some are 0: a vertex can be there with the sum 0
  // Vertices with kCutDegree neighbours or more: where their rows pass from stretch to stretch (a search of a hub's row
  // is twenty dependent loads, and a workgroup waits for its slowest lane's in every stretch).
  const int32_t* cut_row_of;         // [vertices], -1: none
  const HubCut* cuts;                // [rows][stretches + 1]; no pieces in it
};
constexpr uint32_t kCutDegree = 32;

__global__ __launch_bounds__(256) void first_of_parallel_edges(CSRPartition csr, uint32_t* __restrict__ is_first) {
  const size_t e = (size_t)blockIdx.x * 256u + threadIdx.x;
  if (e > (size_t)csr.n_edges) return;
  if (e == (size_t)csr.n_edges) {
    is_first[e] = 0;
    return;
  }
  const VertexID u = source_of_edge(csr.row_ptr, csr.n_vertices, (EdgePos_t)e);
  is_first[e] = (EdgePos_t)e == csr.row_ptr[u] || csr.edges[e - 1] != csr.edges[e] ? 1u : 0u;
}

// at[e] = how many first edges there are before e
__global__ __launch_bounds__(256) void merge_rows(CSRPartition csr, const uint32_t* __restrict__ at, EdgePos_t* __restrict__ row_ptr) {
  const size_t v = (size_t)blockIdx.x * 256u + threadIdx.x;
  if (v <= (size_t)csr.n_vertices) row_ptr[v] = (EdgePos_t)at[csr.row_ptr[v]];
}

__global__ __launch_bounds__(256) void merge_edges(CSRPartition csr, const float* __restrict__ inverse_row_sums,
                                                   const uint32_t* __restrict__ at, VertexID* __restrict__ ids,
                                                   unsigned long long* __restrict__ terms, uint32_t* zero_terms) {
  const size_t e = (size_t)blockIdx.x * 256u + threadIdx.x;
  if (e >= (size_t)csr.n_edges || at[e + 1] == at[e]) return;
  const float inverse = inverse_row_sums[source_of_edge(csr.row_ptr, csr.n_vertices, (EdgePos_t)e)];
  unsigned long long sum = 0;
  for (size_t i = e;;) {  // to the next first edge
    const float p = csr.weights[i] * inverse;
    sum += importance_term_fixed(p * p);
    ++i;
    if (i >= (size_t)csr.n_edges || at[i + 1] != at[i]) break;
  }
  ids[at[e]] = csr.edges[e];
  terms[at[e]] = sum;
  if (sum == 0) *zero_terms = 1;
}

constexpr uint32_t kBitmapTileWords = 2048;  // bitmaps are padded to whole tiles of 65536 vertices (4 parts)

// log2 of a positive normal float from exponent extraction and an atanh series; every step
// is a single IEEE operation so that host and device agree bit for bit.
__host__ __device__ __forceinline__ float det_log2(float x) {
  uint32_t bits;
#if defined(__HIP_DEVICE_COMPILE__)
  bits = __float_as_uint(x);
#else
  memcpy(&bits, &x, sizeof(bits));
#endif
  int e = (int)(bits >> 23) - 127;
  const uint32_t mbits = (bits & 0x7FFFFFu) | 0x3F800000u;
  float m;
#if defined(__HIP_DEVICE_COMPILE__)
  m = __uint_as_float(mbits);
#else
  memcpy(&m, &mbits, sizeof(m));
#endif
  if (m > 1.41421354f) { m = m * 0.5f; e += 1; }
  const float z = (m - 1.0f) / (m + 1.0f);
  const float z2 = z * z;
  float poly = z2 * 0.142857149f;
  poly = poly + 0.2f;
  poly = poly * z2;
  poly = poly + 0.333333343f;
  poly = poly * z2;
  poly = poly + 1.0f;
  float ln_m = z * poly;
  ln_m = ln_m * 2.0f;
  return (float)e + ln_m * 1.44269502f;
}

// Efraimidis-Spirakis key of (sample, vertex): log2(u) / importance, importance the fixed-point
// sum of the vertex's terms (the common 2^53 scale does not change the order of the keys), u
// from Philox: the pair's index is P = sample * (|V| rounded up to a multiple of 4) + vertex,
// its uniform comes from word P & 3 of the block with counter P >> 2 - four consecutive
// vertices of a sample share a block, so a lane that handles four of them pays for one (the
// ten rounds of multiplications are what the key pass of a dense layer is bound by).  As
// sortable bits, inverted so that an ascending sort yields descending keys.  No key is
// 0xFFFFFFFF (it would be a negative NaN): kAbsentKey marks the vertices a sample's
// neighbourhood does not hold.
constexpr uint32_t kAbsentKey = 0xFFFFFFFFu;
// importance sums stay below 2^63 (at most 1024 transits, each adding at most 2^53)
constexpr unsigned long long kAbsentSum = ~0ull;
__host__ __device__ __forceinline__ uint64_t ladies_pair_index(uint64_t sample, uint32_t n_vertices, uint32_t v) {
  return sample * (uint64_t)((n_vertices + 3u) & ~3u) + v;
}
__device__ __forceinline__ PhiloxBlock ladies_block(uint64_t pair, uint32_t step, uint64_t seed) {
  const uint64_t block = pair >> 2;
  return philox4x32_10((uint32_t)block, (uint32_t)(block >> 32), step, 0, (uint32_t)seed, (uint32_t)(seed >> 32));
}
__device__ __forceinline__ uint32_t ladies_key_from_word(unsigned long long importance_fixed, uint32_t word) {
  const float importance = (float)importance_fixed;
  const float u = ((float)(word >> 8) + 0.5f) * 5.9604644775390625e-08f;
  float key = -__builtin_inff();
  if (importance > 0.0f) key = det_log2(u) / importance;
  uint32_t b = __float_as_uint(key);
  b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ~b;
}
// one pair on its own
__device__ __forceinline__ uint32_t ladies_key_bits(unsigned long long importance_fixed, uint64_t pair, uint32_t step,
                                                    uint64_t seed) {
  const PhiloxBlock blk = ladies_block(pair, step, seed);
  const uint32_t which = (uint32_t)pair & 3u;
  uint32_t word = blk.w[0];
  word = which == 1 ? blk.w[1] : word;
  word = which == 2 ? blk.w[2] : word;
  word = which == 3 ? blk.w[3] : word;
  return ladies_key_from_word(importance_fixed, word);
}

// ---- wave-wide data movement on the VALU (DPP), no LDS traffic ----
// The value of the lane `shift` below inside the lane's row of 16; lanes without one get `fill`.
template <int kShift>
__device__ __forceinline__ uint32_t row_shift_up(uint32_t fill, uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)x, 0x110 | kShift, 0xF, 0xF, false);
}
// One workgroup per (sample, some consecutive stretches of 7168 vertices), the sums of one stretch in LDS at a time.
// Adjacencies are sorted by destination, so the part of a transit's adjacency that falls into a stretch is one
// sub-range; the workgroup streams the sub-ranges of all the sample's transits, adds in LDS, and writes the stretch
// out once - plain stores that cover the whole map, so nothing is cleared beforehand and no atomic reaches memory
// (global atomics stop at ~24 G/s on this part).  Every wavefront walks a contiguous part of the stretch's entries,
// which lets a lane step from one sub-range to the next instead of searching the table for every entry.
constexpr uint32_t kBinThreads = 1024;
constexpr uint32_t kBinWaves = kBinThreads / 64;
constexpr uint32_t kBinAhead = 4;             // entries a lane fetches before it works on the first
constexpr uint32_t kBinsPerGroup = 16;        // consecutive stretches of a sample one workgroup takes
constexpr uint32_t kBinVertices = 7168;       // 56 KB of 64-bit sums + 896 B of bits
constexpr uint32_t kBinWords = kBinVertices / 32u;

// Dense pieces.  What a hub contributes to a stretch can be thousands of entries (a layer drawn by importance sits on
// the hubs), and it is the same for every sample that holds the hub.  Where a vertex has kDensePieceEntries or more
// neighbours in one stretch, the stretch's piece of that vertex is built once per graph - the importance sum of every
// vertex of the stretch (7168 64-bit integers, kAbsentSum where there is no edge) - and a sample adds the piece on the
// stretch's way out of LDS instead of going through the entries.  hub_row[v] = row of v in piece_of or -1;
// piece_of[row * stretches + stretch] = piece index or kNoPiece.
constexpr uint32_t kDensePieceEntries = 2048;
constexpr size_t kDensePieceBudgetBytes = (size_t)2 << 30;
struct DensePieces {
  const int32_t* hub_row = nullptr;  // nullptr: the graph has none
  const uint32_t* piece_of = nullptr;
  const unsigned long long* sums = nullptr;
};

// LADIES form: the marking kernel turns the importance sums into sampling keys itself where a
// stretch leaves LDS (a lane takes four consecutive vertices and pays for one Philox block) and
// writes those, 4 bytes per vertex and sample.  Writing the sums instead and forming the keys in
// the selection's pass cost 8 + 8 + 4 bytes per vertex and sample of traffic, and 3.4 ms more
// per pass at full size.
struct KeysOnTheWayOut {
  uint32_t* keys = nullptr;
  uint64_t seed = 0;
  uint64_t first_sample = 0;
  uint32_t step = 0;
  uint32_t n_vertices = 0;
};

// 32-bit words of one sample's presence map: a bit per vertex, padded to whole tiles.
inline uint32_t bitmap_words_for(uint32_t n_vertices) {
  return ((n_vertices + 31u) / 32u + kBitmapTileWords - 1) / kBitmapTileWords * kBitmapTileWords;
}

// The workgroup's sub-ranges, a lane each (lanes of a wavefront without a transit: length 0), into the tables: those that
// hold entries in lane order, starts[k] = first entry of sub-range k, starts[kept] = all entries, edge[k] its first edge.
// A length with kPieceFlag set stands for a transit whose entries reach the stretch as a ready-made piece: its index
// joins the list `pieces`.  Two barriers; every lane gets the three counts.
constexpr uint32_t kPieceFlag = 0x80000000u;
struct Subranges {
  uint32_t ranges, pieces, entries;
};
__device__ __forceinline__ Subranges list_subranges(uint32_t raw, EdgePos_t first, uint32_t n_transits, uint32_t* starts,
                                                    EdgePos_t* edge, uint32_t* pieces, uint4* s_wave) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = (n_transits + 63u) / 64u;
  const bool is_piece = (raw & kPieceFlag) != 0;
  const uint32_t len = is_piece ? 0u : raw;
  const uint64_t holds = __ballot(len != 0), ready = __ballot(is_piece), below = (1ull << lane) - 1ull;
  const uint32_t through = wave < waves ? wave_inclusive_scan(len) : 0u;
  if (lane == 63 && wave < waves) s_wave[wave] = make_uint4((uint32_t)__popcll(holds), (uint32_t)__popcll(ready), through, 0u);
  __syncthreads();
  Subranges all{0, 0, 0}, mine{0, 0, 0};
  for (uint32_t w = 0; w < waves; ++w) {
    const uint4 t = s_wave[w];
    if (w == wave) mine = all;
    all.ranges += t.x;
    all.pieces += t.y;
    all.entries += t.z;
  }
  if (len != 0) {
    const uint32_t k = mine.ranges + (uint32_t)__popcll(holds & below);
    starts[k] = mine.entries + through - len;
    edge[k] = first;
  }
  if (is_piece) pieces[mine.pieces + (uint32_t)__popcll(ready & below)] = raw & ~kPieceFlag;
  if (threadIdx.x == 0) starts[all.ranges] = all.entries;
  __syncthreads();
  return all;
}

// A sample without hubs among its transits and with at most this many entries in a workgroup's stretches (a layer whose
// transits are drawn uniformly) adds them all up at once, in an LDS table of twice as many slots.
constexpr uint32_t kSparseGroupEntries = 2048;

// The samples that are not ranked in LDS (ranked_layer): the keys of sample `at` of them go to keys + at * keys_per_sample.
// Two workgroups of 16 wavefronts share a compute unit only at 8 wavefronts per SIMD, which the kernel's attributes ask
// the compiler for.
// 500 K vertices, 12 M edges, second layer of 1024 samples of 512 (1.5 M pairs a sample): see the engine's rank_by_keys.
__global__ __launch_bounds__(kBinThreads, 8) __attribute__((amdgpu_num_vgpr(56))) void collective_mark_binned(
    MergedEdges merged, TransitView tv, int32_t invalid, uint32_t n_samples, const uint32_t* __restrict__ n_marked,
    const uint32_t* __restrict__ marked, uint32_t bins_per_sample, uint32_t keys_per_sample, DensePieces dense,
    KeysOnTheWayOut keys_out) {
  __shared__ __align__(16) uint32_t s_bits[kBinWords];  // where some terms are 0
  __shared__ __align__(16) unsigned long long s_acc[kBinVertices];
  // the sub-ranges that hold entries, in transit order
  __shared__ uint32_t s_start[kMaxLayerTransits + 1];  // first entry of sub-range k among the stretch's entries
  __shared__ EdgePos_t s_edge[kMaxLayerTransits];      // its first edge
  __shared__ uint32_t s_piece[kMaxLayerTransits];      // the stretch's dense pieces
  __shared__ uint4 s_wave[kBinWaves];
  // A workgroup takes kBinsPerGroup consecutive stretches of one sample, one after the other: where a transit's sub-range
  // ends in one stretch it begins in the next, and the end is then only a short gallop away instead of a search of the
  // whole adjacency.  The low stretches hold the hubs and take longest: all samples' first groups start first.
  const uint32_t group = blockIdx.x / n_samples;
  const uint32_t at = blockIdx.x - group * n_samples;
  if (at >= *n_marked) return;
  const uint32_t s = marked[at];
  const uint32_t first_bin = group * kBinsPerGroup;
  const int32_t* transits = tv.base + (size_t)s * tv.stride;
  uint32_t* my_keys = keys_out.keys + (size_t)at * keys_per_sample;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = threadIdx.x >> 6;
  // tv.count <= kBinThreads: lane i keeps transit i's adjacency and how far the stretches before this one reach into it
  EdgePos_t my_end = 0, my_reach = 0;
  uint32_t my_next = 0xFFFFFFFFu;  // destination of edge my_reach; none left: above every vertex
  int32_t my_hub = -1, my_cut_row = -1;
  int32_t my_transit = -1;
  if (threadIdx.x < tv.count) {
    my_transit = transits[threadIdx.x];
    if (my_transit == invalid) my_transit = -1;
    if (my_transit != -1 && dense.hub_row) my_hub = dense.hub_row[my_transit];
    if (my_transit != -1 && merged.cut_row_of) my_cut_row = merged.cut_row_of[my_transit];
  }
  const bool hubs_among_transits = __syncthreads_or(my_hub >= 0) != 0;
  const HubCut* my_cuts = merged.cuts + (my_cut_row < 0 ? 0 : (size_t)my_cut_row * (bins_per_sample + 1));
  if (my_transit != -1) {
    my_end = merged.row_ptr[my_transit + 1];
    my_reach = my_cut_row >= 0 ? my_cuts[first_bin].from
                               : first_edge_from(merged.ids, merged.row_ptr[my_transit], my_end, first_bin * kBinVertices);
    if (my_cut_row < 0 && my_reach < my_end) my_next = (uint32_t)merged.ids[my_reach];
  }
  if (!hubs_among_transits) {
    // The stretches of the workgroup as one: the sums are gathered in an LDS table hashed by vertex (in the room of the
    // per-vertex sums), the keys of the whole range are written as absent, and the table's vertices then get theirs.
    // Stretch by stretch, 16 chains of searches, tables and barriers cost a workgroup 130 us for a few hundred entries.
    const uint32_t group_bins = first_bin + kBinsPerGroup < bins_per_sample ? kBinsPerGroup : bins_per_sample - first_bin;
    const uint32_t v_lo = first_bin * kBinVertices, v_hi = v_lo + group_bins * kBinVertices;
    EdgePos_t stop = my_reach;
    if (my_cut_row >= 0) stop = my_cuts[first_bin + group_bins].from;
    else if (my_next < v_hi) stop = first_edge_from(merged.ids, my_reach, my_end, v_hi);
    const Subranges all = list_subranges((uint32_t)(stop - my_reach), my_reach, tv.count, s_start, s_edge, s_piece, s_wave);
    const uint32_t ranges = all.ranges, size = all.entries;
    if (size <= kSparseGroupEntries) {
      constexpr uint32_t kSlots = 2u * kSparseGroupEntries;  // a power of two
      unsigned long long* slot_sum = s_acc;
      uint32_t* slot_vertex = (uint32_t*)(s_acc + kSlots);
      for (uint32_t i = threadIdx.x; i < kSlots; i += kBinThreads) {
        slot_vertex[i] = 0xFFFFFFFFu;
        slot_sum[i] = 0;
      }
      uint32_t* out_keys = my_keys + v_lo;
      for (uint32_t i = threadIdx.x; i < group_bins * kBinVertices; i += kBinThreads) out_keys[i] = kAbsentKey;
      __syncthreads();
      for (uint32_t e = threadIdx.x; e < size; e += kBinThreads) {
        uint32_t lo = 0, hi = ranges;  // the sub-range that holds entry e
        while (hi - lo > 1) {
          const uint32_t mid = lo + (hi - lo) / 2;
          if (s_start[mid] <= e) lo = mid; else hi = mid;
        }
        const EdgePos_t src = s_edge[lo] + (EdgePos_t)(e - s_start[lo]);
        const uint32_t local = (uint32_t)merged.ids[src] - v_lo;
        uint32_t slot = (local * 2654435761u) >> 20 & (kSlots - 1u);
        for (;;) {  // at most half of the slots are ever taken
          const uint32_t before = atomicCAS(&slot_vertex[slot], 0xFFFFFFFFu, local);
          if (before == 0xFFFFFFFFu || before == local) break;
          slot = (slot + 1u) & (kSlots - 1u);
        }
        atomicAdd(&slot_sum[slot], merged.terms[src]);
      }
      __syncthreads();  // the table is complete, and the absent keys have been written
      for (uint32_t i = threadIdx.x; i < kSlots; i += kBinThreads) {
        const uint32_t local = slot_vertex[i];
        if (local == 0xFFFFFFFFu) continue;
        out_keys[local] = ladies_key_bits(slot_sum[i], ladies_pair_index(keys_out.first_sample + s, keys_out.n_vertices, v_lo + local),
                                          keys_out.step, keys_out.seed);
      }
      return;
    }
    // too many entries for that: stretch by stretch
    __syncthreads();
  }
  EdgePos_t cut_after = my_cut_row >= 0 ? my_cuts[first_bin + 1].from : 0;  // the end of the coming stretch, fetched one stretch ahead
  for (uint32_t bin = first_bin; bin < first_bin + kBinsPerGroup && bin < bins_per_sample; ++bin) {
    const uint32_t v_lo = bin * kBinVertices;
    if (merged.zero_terms)
      for (uint32_t i = threadIdx.x; i < kBinWords; i += kBinThreads) s_bits[i] = 0;
    for (uint32_t i = threadIdx.x; i < kBinVertices; i += kBinThreads) s_acc[i] = 0;
    uint32_t length = 0;
    const EdgePos_t my_from = my_reach;
    if (my_transit != -1) {
      const uint32_t v_hi = v_lo + kBinVertices;
      if (my_cut_row >= 0) {
        my_reach = cut_after;
        if (bin + 2 <= bins_per_sample) cut_after = my_cuts[bin + 2].from;
      } else if (my_next < v_hi) {  // nothing is fetched where the next edge already lies beyond the stretch
        my_reach = first_edge_from(merged.ids, my_from, my_end, v_hi);
        my_next = my_reach < my_end ? (uint32_t)merged.ids[my_reach] : 0xFFFFFFFFu;
      }
      length = (uint32_t)(my_reach - my_from);
      if (my_hub >= 0 && length != 0) {
        const uint32_t piece = dense.piece_of[(size_t)my_hub * bins_per_sample + bin];
        if (piece != kNoPiece) length = kPieceFlag | piece;  // these entries reach the stretch ready-made
      }
    }
    const Subranges all = list_subranges(length, my_from, tv.count, s_start, s_edge, s_piece, s_wave);
    const uint32_t ranges = all.ranges, size = all.entries;
    // every wavefront walks a contiguous part of the entries, 64 * kBinAhead per round
    constexpr uint32_t kRound = 64u * kBinAhead;
    const uint32_t part = (size + kBinWaves * kRound - 1) / (kBinWaves * kRound) * kRound;
    const uint32_t part_begin = wave * part;
    const uint32_t part_end = part_begin + part < size ? part_begin + part : size;
    uint32_t cur = 0, cur_begin = 0, cur_end = 0;
    EdgePos_t cur_edges = 0;
    if (part_begin + lane < part_end) {  // the sub-range of the lane's first entry
      const uint32_t e = part_begin + lane;
      uint32_t lo = 0, hi = ranges;
      while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (s_start[mid] <= e) lo = mid; else hi = mid;
      }
      cur = lo;
      cur_begin = s_start[lo];
      cur_end = s_start[lo + 1];
      cur_edges = s_edge[lo];
    }
    for (uint32_t e0 = part_begin; e0 < part_end; e0 += kRound) {
      uint32_t locals[kBinAhead];  // vertex - v_lo
      unsigned long long terms[kBinAhead];
#pragma unroll
      for (uint32_t a = 0; a < kBinAhead; ++a) {
        const uint32_t e = e0 + a * 64u + lane;
        locals[a] = 0xFFFFFFFFu;
        terms[a] = 0;
        if (e < part_end) {
          if (e >= cur_end) {
            do {  // no sub-range is empty
              ++cur;
              cur_begin = cur_end;
              cur_end = s_start[cur + 1];
            } while (e >= cur_end);
            cur_edges = s_edge[cur];
          }
          const EdgePos_t src = cur_edges + (EdgePos_t)(e - cur_begin);
          locals[a] = (uint32_t)merged.ids[src] - v_lo;
          terms[a] = merged.terms[src];
        }
      }
#pragma unroll
      for (uint32_t a = 0; a < kBinAhead; ++a) {
        if (locals[a] == 0xFFFFFFFFu) continue;
        atomicAdd(&s_acc[locals[a]], terms[a]);
        if (merged.zero_terms) atomicOr(&s_bits[locals[a] >> 5], 1u << (locals[a] & 31u));
      }
    }
    __syncthreads();
    // What leaves the workgroup is the sampling key of every vertex of the stretch (kAbsentKey where the neighbourhood
    // does not hold the vertex).  A lane takes four consecutive vertices: 16-byte accesses to LDS, to the pieces and to
    // the output, and one Philox block where it forms keys.
    const uint32_t n_pieces = all.pieces;
    for (uint32_t q = threadIdx.x; q < kBinVertices / 4u; q += kBinThreads) {
      const uint32_t i = 4u * q;
      const ulonglong2 low = ((const ulonglong2*)s_acc)[2u * q], high = ((const ulonglong2*)s_acc)[2u * q + 1u];
      unsigned long long sum[4] = {low.x, low.y, high.x, high.y};  // 0 where nothing was added
      const uint32_t bits = merged.zero_terms ? (s_bits[i >> 5] >> (i & 31u)) & 15u : 0u;
      bool present[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) present[k] = sum[k] != 0 || (bits >> k & 1u) != 0;
#pragma unroll 4
      for (uint32_t p = 0; p < n_pieces; ++p) {
        const ulonglong2* piece = (const ulonglong2*)(dense.sums + (size_t)s_piece[p] * kBinVertices + i);
        const ulonglong2 a = piece[0], b = piece[1];
        const unsigned long long ready[4] = {a.x, a.y, b.x, b.y};
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
          if (ready[k] != kAbsentSum) {
            sum[k] += ready[k];
            present[k] = true;
          }
      }
      uint32_t key[4] = {kAbsentKey, kAbsentKey, kAbsentKey, kAbsentKey};
      if (present[0] || present[1] || present[2] || present[3]) {
        const PhiloxBlock blk = ladies_block(ladies_pair_index(keys_out.first_sample + s, keys_out.n_vertices, v_lo + i),
                                             keys_out.step, keys_out.seed);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
          if (present[k]) key[k] = ladies_key_from_word(sum[k], blk.w[k]);
      }
      *(uint4*)(my_keys + v_lo + i) = make_uint4(key[0], key[1], key[2], key[3]);
    }
    __syncthreads();  // the next stretch clears what this one has just read
  }
}

// ---- LADIES form: small neighbourhoods, ranked in LDS -------------------------------------

// Entries (pairs) of a sample's neighbourhood up to which it is ranked by one workgroup in LDS; the others, in whatever
// order they are found, are listed.
constexpr uint32_t kRankedEntries = 8192;
constexpr uint32_t kRankedThreads = 1024;

// A wavefront per sample: sizes[s] = entries of its neighbourhood, parallel edges and all, merged_sizes[s] = without.
__global__ __launch_bounds__(kSortOutThreads) void sort_out_ranked(CSRPartition csr, MergedEdges merged, TransitView tv,
                                                                   uint32_t n_samples, int32_t invalid,
                                                                   uint32_t* __restrict__ sizes,
                                                                   uint32_t* __restrict__ merged_sizes,
                                                                   uint32_t* n_marked, uint32_t* __restrict__ marked,
                                                                   uint32_t* __restrict__ too_long) {
  __shared__ uint32_t s_taken, s_base;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t s = blockIdx.x * (kSortOutThreads / 64u) + (threadIdx.x >> 6);
  if (threadIdx.x == 0) s_taken = 0;
  __syncthreads();
  uint64_t both = 0, pairs = 0;
  for (uint32_t i = lane; i < tv.count && s < n_samples; i += 64u) {
    const int32_t t = tv.base[(size_t)s * tv.stride + i];
    if (t == invalid || t == -1) continue;
    both += (uint64_t)(csr.row_ptr[t + 1] - csr.row_ptr[t]);
    pairs += (uint64_t)(merged.row_ptr[t + 1] - merged.row_ptr[t]);
  }
  both = __shfl(wave_inclusive_scan_u64(both), 63, kWave);
  pairs = __shfl(wave_inclusive_scan_u64(pairs), 63, kWave);
  uint32_t at = 0;
  if (lane == 0 && s < n_samples) {
    const uint32_t size = entries_or_refused(both, n_marked + 1, too_long);
    if (size == 0) pairs = 0;
    sizes[s] = size;
    merged_sizes[s] = (uint32_t)pairs;
    if (pairs > kRankedEntries) at = atomicAdd(&s_taken, 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_taken) s_base = atomicAdd(n_marked, s_taken);
  __syncthreads();
  if (lane == 0 && s < n_samples && pairs > kRankedEntries) marked[s_base + at] = s;
}

// A workgroup per sample: fetches the entries, sorts them by vertex, adds their terms up, forms the keys and sorts the
// vertices by them (equal keys by vertex, as the sorts are stable).  Marked stretch by stretch, a layer of 1024 such samples
// over 500 K vertices wrote and read 4 GB of keys, most of them absent.
template <class Draw>
__device__ __forceinline__ void ranked_layer(const MergedEdges& merged, uint32_t n_vertices, const int32_t* transits,
                                             uint32_t n_transits, int32_t invalid, uint32_t size, uint64_t sample,
                                             uint32_t step, uint64_t seed, uint32_t* __restrict__ distinct_out, Draw draw) {
  constexpr uint32_t kEach = kRankedEntries / kRankedThreads;
  // two buffers of ids with one for the kept ids between them: next to whichever the sort leaves free it makes the sums' room
  __shared__ __align__(16) uint32_t s_words[3 * kRankedEntries];
  __shared__ uint16_t s_payload[2][kRankedEntries];
  __shared__ uint32_t s_start[kMaxLayerTransits];
  __shared__ EdgePos_t s_edge[kMaxLayerTransits];
  __shared__ uint32_t s_count[kRankedThreads / 64][kSortedDigits];
  __shared__ uint32_t s_wave_count[kRankedThreads / 64];
  static_assert(kMaxLayerTransits <= kRankedThreads && kRankedEntries <= 65536, "a lane a transit; 16 bits an entry");
  uint32_t* const kept = s_words + kRankedEntries;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  auto before_wave = [&](uint32_t through, uint32_t* all) {  // exclusive prefix of a wavefront's total
    if (lane == 63) s_wave_count[wave] = through;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t w = 0; w < kRankedThreads / 64; ++w) {
      if (w < wave) before += s_wave_count[w];
      total += s_wave_count[w];
    }
    __syncthreads();
    *all = total;
    return before;
  };
  uint32_t total;
  {
    const int32_t t = threadIdx.x < n_transits ? transits[threadIdx.x] : -1;
    EdgePos_t begin = 0;
    uint32_t degree = 0;
    if (t != invalid && t != -1) {
      begin = merged.row_ptr[t];
      degree = (uint32_t)(merged.row_ptr[t + 1] - begin);
    }
    const uint32_t through = wave_inclusive_scan(degree);
    const uint32_t before = before_wave(through, &total);
    if (threadIdx.x < n_transits) {
      s_start[threadIdx.x] = before + through - degree;
      s_edge[threadIdx.x] = begin;
    }
    __syncthreads();
  }
  auto edge_of = [&](uint32_t e) {
    uint32_t lo = 0, hi = n_transits;  // the last transit that starts at e or before (empty ones start where the next does)
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (s_start[mid] <= e) lo = mid; else hi = mid;
    }
    return s_edge[lo] + (EdgePos_t)(e - s_start[lo]);
  };
  for (uint32_t e = threadIdx.x; e < size; e += kRankedThreads) {
    s_words[e] = (uint32_t)merged.ids[edge_of(e)];
    s_payload[0][e] = (uint16_t)e;
  }
  __syncthreads();
  SortedIds sorted{s_words, s_words + 2 * kRankedEntries, s_payload[0], s_payload[1]};
  sorted = sort_ids<kRankedThreads, true>(sorted, s_count, s_wave_count, size, 32u - (uint32_t)__clz((int)n_vertices));
  // which of a lane's entries are a vertex's first, and how many vertices come before
  unsigned long long* sums = (unsigned long long*)(sorted.other == s_words ? s_words : kept);
  for (uint32_t i = threadIdx.x; i < kRankedEntries; i += kRankedThreads) sums[i] = 0;
  uint32_t id[kEach], firsts = 0;
  uint32_t last = threadIdx.x != 0 && threadIdx.x * kEach <= size ? sorted.ids[threadIdx.x * kEach - 1] : 0xFFFFFFFFu;
#pragma unroll
  for (uint32_t k = 0; k < kEach; ++k) {
    const uint32_t i = threadIdx.x * kEach + k;
    id[k] = i < size ? sorted.ids[i] : 0xFFFFFFFFu;
    if (i < size && id[k] != last) firsts |= 1u << k;
    last = id[k];
  }
  const uint32_t through = wave_inclusive_scan((uint32_t)__popc(firsts));
  uint32_t distinct;
  const uint32_t rank0 = before_wave(through, &distinct) + through - (uint32_t)__popc(firsts);  // the sums are clear now
#pragma unroll
  for (uint32_t k = 0; k < kEach; ++k) {
    const uint32_t i = threadIdx.x * kEach + k;
    if (i >= size) continue;
    const uint32_t rank = rank0 + (uint32_t)__popc(firsts & ((2u << k) - 1u)) - 1u;
    atomicAdd(&sums[rank], merged.terms[edge_of(sorted.payload[i])]);
  }
  __syncthreads();
  uint32_t key[kEach];
#pragma unroll
  for (uint32_t k = 0; k < kEach; ++k) {
    key[k] = 0;
    if (firsts >> k & 1u)
      key[k] = ladies_key_bits(sums[rank0 + (uint32_t)__popc(firsts & ((1u << k) - 1u))], ladies_pair_index(sample, n_vertices, id[k]),
                               step, seed);
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kEach; ++k) {
    if (!(firsts >> k & 1u)) continue;
    const uint32_t rank = rank0 + (uint32_t)__popc(firsts & ((1u << k) - 1u));
    s_words[rank] = key[k];
    kept[rank] = id[k];
    s_payload[0][rank] = (uint16_t)rank;
  }
  __syncthreads();
  sorted = SortedIds{s_words, s_words + 2 * kRankedEntries, s_payload[0], s_payload[1]};
  sorted = sort_ids<kRankedThreads, true>(sorted, s_count, s_wave_count, distinct, 32);
  for (uint32_t i = threadIdx.x; i < distinct; i += kRankedThreads) sorted.other[i] = kept[sorted.payload[i]];
  __syncthreads();
  if (threadIdx.x == 0) *distinct_out = distinct;
  draw((const CSR::Edge*)sorted.other, distinct);
}

// item_count[s] = work items of sample s (at least one, so that row offsets get written)
__global__ void build_item_counts(const uint32_t* __restrict__ sizes, uint32_t n, uint32_t* __restrict__ item_count) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) {
    const uint32_t items = (sizes[s] + kBuildItemEntries - 1) / kBuildItemEntries;
    item_count[s] = items ? items : 1u;
  } else if (s == n) {
    item_count[s] = 0;
  }
}

__global__ void gather_u32(const uint32_t* __restrict__ table, const uint32_t* __restrict__ index, size_t n,
                           uint32_t* __restrict__ out, uint32_t* __restrict__ index_copy) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = index[i];
  out[i] = table[p];
  if (index_copy) index_copy[i] = p;
}

__global__ void fill_u32(uint32_t* dst, size_t n, uint32_t value) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = value;
}

// ---- the best m keys of every sample, without sorting everything ----
//
// Only the first stepSize ranked vertices of a sample are ever read, out of up to millions of
// distinct ones.  A radix select on the upper 14 bits of the sort key finds, per sample, the
// smallest prefix T such that at least m keys have a prefix <= T; the entries with a prefix
// <= T (m and some more) are copied out and only those are sorted.
// The keys of a chunk are dense: keys[s * keys_per_sample + v] for every vertex v (kAbsentKey
// where sample s does not hold v), so position tells sample and vertex and no list of the
// distinct pairs is ever written.

// One workgroup per sample, one pass over its keys: counts the present ones by their upper
// kSelectBits bits in an LDS
// histogram and picks the bin that holds the wanted-th smallest key: threshold[s] = that bin,
// kept[s] = keys up to and including it (a sample with fewer keys than wanted keeps them all),
// distinct[its number] = all its keys.  A sample's whole histogram stays in the workgroup: no atomic
// reaches memory, and no second pass over the keys refines the threshold (two levels of 8 bits,
// counted by a workgroup per tile of 8192 keys, read every key twice).
constexpr uint32_t kSelectBits = 14;
constexpr uint32_t kSelectBins = 1u << kSelectBits;
constexpr uint32_t kSelectThreads = 1024;
// The pass also notes, for every stretch of 256 consecutive keys (what a wavefront handles at a
// time, four keys per lane), the smallest prefix in it: the copying of the kept entries then
// reads only the stretches that hold one (a few hundred of a sample's 12,000).
constexpr uint32_t kCollectStretch = 256;
__device__ __forceinline__ void note_best_of_stretch(const uint32_t (&key)[4], uint32_t quad, uint32_t lane,
                                                     uint16_t* __restrict__ best_of) {
  uint32_t a = key[0] < key[1] ? key[0] : key[1], b = key[2] < key[3] ? key[2] : key[3];
  uint32_t best = (a < b ? a : b) >> (32u - kSelectBits);  // kAbsentKey: the largest prefix
  // minimum of the wavefront into lane 63, on the VALU (DPP): along the rows of 16 lanes, then
  // the last lane of a row into the next row, then lane 31 into the upper half
  const uint32_t none = 0xFFFFFFFFu;
  uint32_t other = row_shift_up<1>(none, best);
  best = other < best ? other : best;
  other = row_shift_up<2>(none, best);
  best = other < best ? other : best;
  other = row_shift_up<4>(none, best);
  best = other < best ? other : best;
  other = row_shift_up<8>(none, best);
  best = other < best ? other : best;
  other = (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)best, 0x142, 0xA, 0xF, false);  // row_bcast:15
  best = other < best ? other : best;
  other = (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)best, 0x143, 0xC, 0xF, false);  // row_bcast:31
  best = other < best ? other : best;
  if (lane == 63) best_of[quad / 64u] = (uint16_t)best;
}
__global__ __launch_bounds__(kSelectThreads, 8) __attribute__((amdgpu_num_vgpr(56))) void select_threshold(
    const uint32_t* __restrict__ keys, uint32_t keys_per_sample, uint32_t wanted, const uint32_t* __restrict__ n_marked,
    const uint32_t* __restrict__ marked, uint32_t* __restrict__ threshold, uint32_t* __restrict__ kept,
    uint32_t* __restrict__ claimed, uint32_t* __restrict__ distinct, uint16_t* __restrict__ stretch_best) {
  __shared__ uint32_t s_hist[kSelectBins];
  __shared__ uint32_t s_wave_total[kSelectThreads / 64];
  const uint32_t s = blockIdx.x;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) claimed[s] = 0;  // for select_collect
  if (s >= *n_marked) {
    if (threadIdx.x == 0) kept[s] = 0;
    return;
  }
  for (uint32_t i = threadIdx.x; i < kSelectBins; i += kSelectThreads) s_hist[i] = 0;
  __syncthreads();
  const uint32_t* mine = keys + (size_t)s * keys_per_sample;
  uint16_t* my_best = stretch_best + (size_t)s * (keys_per_sample / kCollectStretch);
  {
    const uint4* my_keys = (const uint4*)mine;
    for (uint32_t q0 = 0; q0 < keys_per_sample / 4u; q0 += 4 * kSelectThreads) {
      uint4 batch[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t q = q0 + k * kSelectThreads + threadIdx.x;
        batch[k] = q < keys_per_sample / 4u ? my_keys[q] : make_uint4(kAbsentKey, kAbsentKey, kAbsentKey, kAbsentKey);
      }
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t q = q0 + k * kSelectThreads + threadIdx.x;
        if (q >= keys_per_sample / 4u) continue;  // whole wavefronts: the sample holds a multiple of 256 keys
        const uint32_t key[4] = {batch[k].x, batch[k].y, batch[k].z, batch[k].w};
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
          if (key[i] != kAbsentKey) atomicAdd(&s_hist[key[i] >> (32u - kSelectBits)], 1u);
        note_best_of_stretch(key, q, lane, my_best);
      }
    }
  }
  __syncthreads();
  // lane t owns bins [16 t, 16 t + 16): the bin in which the running count reaches `wanted`
  constexpr uint32_t kOwn = kSelectBins / kSelectThreads;
  uint32_t own = 0;
#pragma unroll
  for (uint32_t b = 0; b < kOwn; ++b) own += s_hist[threadIdx.x * kOwn + b];
  const uint32_t through_wave = wave_inclusive_scan(own);
  if (lane == 63) s_wave_total[wave] = through_wave;
  __syncthreads();
  uint32_t before = through_wave - own, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < kSelectThreads / 64; ++w) {
    const uint32_t t = s_wave_total[w];
    if (w < wave) before += t;
    total += t;
  }
  if (threadIdx.x == 0) distinct[marked[s]] = total;
  if (total < wanted) {  // everything stays
    if (threadIdx.x == 0) {
      threshold[s] = kSelectBins - 1u;
      kept[s] = total;
    }
  } else if (before < wanted && before + own >= wanted) {  // exactly one lane
    uint32_t running = before;
    for (uint32_t b = 0; b < kOwn; ++b) {
      running += s_hist[threadIdx.x * kOwn + b];
      if (running >= wanted) {
        threshold[s] = threadIdx.x * kOwn + b;
        kept[s] = running;
        break;
      }
    }
  }
}

__device__ __forceinline__ bool select_keeps(uint32_t key, uint32_t threshold) {
  return key != kAbsentKey && (key >> (32u - kSelectBits)) <= threshold;
}

// Copies the kept entries of sample s into its part [ranked_start[s], ranked_start[s + 1]) of
// kept_key / kept_id, in whatever order the wavefronts get there (a wavefront claims room for
// the entries of a round with one atomic).  A few hundred of a sample's millions of keys stay:
// one workgroup per sample, whose wavefronts look at the best prefix of each stretch of 256 keys
// first and read only those that hold a kept key.  The sorts that follow fix the order.
__global__ __launch_bounds__(kSelectThreads) void select_collect(const uint32_t* __restrict__ keys,
                                                                 uint32_t keys_per_sample,
                                                                 const uint16_t* __restrict__ stretch_best,
                                                      const uint32_t* __restrict__ threshold_of,
                                                      const uint32_t* __restrict__ ranked_start,
                                                      uint32_t* __restrict__ claimed, uint32_t* __restrict__ kept_key,
                                                      uint32_t* __restrict__ kept_sample, int32_t* __restrict__ kept_id) {
  const uint32_t s = blockIdx.x;
  const uint32_t* mine = keys + (size_t)s * keys_per_sample;
  const uint32_t stretches = keys_per_sample / kCollectStretch;
  const uint16_t* best_of = stretch_best + (size_t)s * stretches;
  const uint32_t threshold = threshold_of[s];
  const uint32_t first = ranked_start[s];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  // a wavefront looks at 64 stretches at a time: lane i knows whether stretch i holds a kept key
  for (uint32_t stretch_begin = wave * 64u; stretch_begin < stretches; stretch_begin += (kSelectThreads / 64u) * 64u) {
    const uint32_t my_stretch = stretch_begin + lane;
    const bool holds = my_stretch < stretches && best_of[my_stretch] <= threshold;
    uint64_t todo = __ballot(holds);
    while (todo) {  // the same for every lane
      const uint32_t stretch = stretch_begin + (uint32_t)__ffsll((long long)todo) - 1u;
      todo &= todo - 1ull;
      const uint32_t v0 = stretch * kCollectStretch + lane * 4u;
      const uint4 four = *(const uint4*)(mine + v0);
      const uint32_t key[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const bool stays = select_keeps(key[i], threshold);
        const uint64_t mask = __ballot(stays);
        if (mask == 0) continue;
        uint32_t base = 0;
        if (lane == (uint32_t)__ffsll((long long)mask) - 1u) base = atomicAdd(&claimed[s], (uint32_t)__popcll(mask));
        base = __shfl(base, __ffsll((long long)mask) - 1, kWave);
        if (stays) {
          const uint32_t at = first + base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
          kept_key[at] = key[i];
          kept_sample[at] = s;
          kept_id[at] = (int32_t)(v0 + i);
        }
      }
    }
  }
}

struct LayerParams {
  CSRPartition csr;
  TransitView transits;   // base already points at the first sample of the chunk
  int step;
  uint32_t step_size;
  uint32_t chunk_samples; // samples in this launch
  uint32_t sample_begin;  // index of the chunk's first sample
  uint32_t final_size;
  uint32_t out_base;      // stepSizeAtStep(step - 1)
  int32_t invalid;
  uint64_t seed;
  uint64_t first_sample;  // index of the device's first sample (multi-device offset)
  int32_t* final_samples;
  void* samples;
  // kConcatenated: offsets are relative to the chunk
  const uint32_t* offsets;
  const int32_t* nbr_cols;
  const float* nbr_weights;
  // kRankedByLadiesImportance: the kept ids of sample ls in descending key order are
  // ranked_ids[ranked_start[at] .. ranked_start[at + 1]) for marked[at] == ls, at < n_marked
  const uint32_t* ranked_start;
  const int32_t* ranked_ids;
  const uint32_t* marked;
  uint32_t n_marked;
};

template <class SampleType, class App>
__global__ __launch_bounds__(256) void layer_execute_kernel(LayerParams P) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  constexpr bool ranked_form = apps::neighborhood_form_of<App>::value == apps::kRankedByLadiesImportance;
  if (i >= (uint64_t)(ranked_form ? P.n_marked : P.chunk_samples) * P.step_size) return;
  const uint32_t at = (uint32_t)(i / P.step_size);
  const uint32_t nbr = (uint32_t)(i - (uint64_t)at * P.step_size);
  const uint32_t ls = ranked_form ? P.marked[at] : at;  // sample inside the chunk
  const uint32_t s = P.sample_begin + ls;
  CSRPartition csr = P.csr;
  const int32_t* transits = P.transits.base + (size_t)ls * P.transits.stride;
  SampleType local_state;
  SampleType* state = std::is_empty<SampleType>::value ? &local_state : (SampleType*)P.samples + s;
  curandState rng;
  rng.reset(P.seed, (P.first_sample + s) * P.step_size + nbr, (uint32_t)P.step);
  const VertexID sample_id = (VertexID)(P.first_sample + s);
  VertexID neighbor = P.invalid;
  if constexpr (apps::neighborhood_form_of<App>::value == apps::kConcatenated) {
    // only the first transit decides whether next() runs (nextdoor.cu:1421)
    if (transits[0] != P.invalid && transits[0] != -1) {
      const uint32_t begin = P.offsets[ls];
      const CSR::Edge* edges = P.nbr_cols + begin;
      const float* weights = P.nbr_weights + begin;
      const VertexID r = App().template next<SampleType, const CSR::Edge*, const float*>(
          P.step, &csr, transits, sample_id, state, 0.0f, edges, weights, (EdgePos_t)(P.offsets[ls + 1] - begin),
          (VertexID_t)nbr, &rng);
      neighbor = r == -1 ? P.invalid : r;
    }
  } else {
    const uint32_t begin = P.ranked_start[at];
    const CSR::Edge* ranked = P.ranked_ids + begin;
    const float* no_weights = nullptr;
    const VertexID r = App().template next<SampleType, const CSR::Edge*, const float*>(
        P.step, &csr, transits, sample_id, state, 0.0f, ranked, no_weights,
        (EdgePos_t)(P.ranked_start[at + 1] - begin), (VertexID_t)nbr, &rng);
    neighbor = r == -1 ? P.invalid : r;
  }
  P.final_samples[(size_t)s * P.final_size + P.out_base + nbr] = neighbor;
}

// next() for output nbr of sample ls of the chunk, with what it takes for transitEdges.
template <class SampleType, class App, class Distinct>
__device__ __forceinline__ void draw_from(const LayerParams& P, uint32_t ls, uint32_t nbr, Distinct& distinct,
                                               uint32_t n_distinct) {
  const uint32_t s = P.sample_begin + ls;
  CSRPartition csr = P.csr;
  SampleType local_state;
  SampleType* state = std::is_empty<SampleType>::value ? &local_state : (SampleType*)P.samples + s;
  curandState rng;
  rng.reset(P.seed, (P.first_sample + s) * P.step_size + nbr, (uint32_t)P.step);
  const float* no_weights = nullptr;
  const VertexID r = App().template next<SampleType, Distinct, const float*>(
      P.step, &csr, P.transits.base + (size_t)ls * P.transits.stride, (VertexID)(P.first_sample + s), state, 0.0f, distinct,
      no_weights, (EdgePos_t)n_distinct, (VertexID_t)nbr, &rng);
  P.final_samples[(size_t)s * P.final_size + P.out_base + nbr] = r == -1 ? P.invalid : r;
}

template <class SampleType, class App>
__global__ __launch_bounds__(kSortedThreads) void sorted_layer_kernel(LayerParams P, const uint32_t* __restrict__ sizes,
                                                                      uint32_t* __restrict__ distinct) {
  const uint32_t ls = blockIdx.x, size = sizes[ls];
  if (size > kSortedEntries) return;
  sorted_layer(P.csr, P.transits.base + (size_t)ls * P.transits.stride, P.transits.count, P.invalid, size, distinct + ls,
               [&](SortedByDegreeSquared& view, uint32_t n_distinct) {
                 for (uint32_t nbr = threadIdx.x; nbr < P.step_size; nbr += kSortedThreads)
                   draw_from<SampleType, App>(P, ls, nbr, view, n_distinct);
               });
}

template <class SampleType, class App>
__global__ __launch_bounds__(kRankedThreads) void ranked_layer_kernel(LayerParams P, MergedEdges merged,
                                                                      const uint32_t* __restrict__ merged_sizes,
                                                                      uint32_t* __restrict__ distinct) {
  const uint32_t ls = blockIdx.x, size = merged_sizes[ls];
  if (size > kRankedEntries) return;
  ranked_layer(merged, (uint32_t)P.csr.n_vertices, P.transits.base + (size_t)ls * P.transits.stride, P.transits.count, P.invalid,
               size, P.first_sample + P.sample_begin + ls, (uint32_t)P.step, P.seed, distinct + ls,
               [&](const CSR::Edge* ranked, uint32_t n_distinct) {
                 for (uint32_t nbr = threadIdx.x; nbr < P.step_size; nbr += kRankedThreads)
                   draw_from<SampleType, App>(P, ls, nbr, ranked, n_distinct);
               });
}

// The draws of the marked samples, a lane each, the workgroups of the grid in turn.
template <class SampleType, class App>
__global__ __launch_bounds__(256) void marked_layer_kernel(LayerParams P, MarkedSamples marked,
                                                           const uint32_t* __restrict__ distinct,
                                                           const uint32_t* __restrict__ bitmap, uint32_t words_per_sample,
                                                           const uint64_t* __restrict__ part_before,
                                                           const uint64_t* __restrict__ group_through, uint32_t parts) {
  const uint64_t draws = (uint64_t)*marked.count * P.step_size;
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < draws; i += gridDim.x * 256ull) {
    const uint32_t at = (uint32_t)(i / P.step_size), nbr = (uint32_t)(i - (uint64_t)at * P.step_size);
    const uint32_t ls = marked.sample[at];
    MarkedByDegreeSquared mine{bitmap + (size_t)at * words_per_sample, part_before + (size_t)at * (parts + 1),
                               group_through + (size_t)at * parts * kGroupsPerPart, P.csr.row_ptr, parts};
    draw_from<SampleType, App>(P, ls, nbr, mine, distinct[ls]);
  }
}

// Entries of concatenated neighbourhood one chunk of samples may hold (about 70 bytes of
// device memory per entry across all work arrays).
constexpr uint64_t kLayerChunkEntries = 96ull << 20;
// Importance forms: nothing is stored per entry, so a chunk is bounded by the memory of its
// presence maps (and accumulators) and by the number of marking work items (entries / kBuildItemEntries) of one launch.
constexpr uint64_t kBitmapBudgetBytes = 48ull << 30;
constexpr uint64_t kBitmapChunkEntries = 1ull << 40;

template <class SampleType, class App>
class LayerEngine : public EngineBase {
 public:
  explicit LayerEngine(const char* name) : name_(name) {}
  ~LayerEngine() override { free_device(); }

  const char* app_name() const override { return name_; }
  int64_t num_samples() const override { return n_samples_; }
  int final_sample_size() const override { return nd::final_sample_size<App>(); }
  int steps() const override { return App().steps(); }
  int step_size(int k) const override { return App().stepSize(k); }
  int initial_sample_size() const override { return App().initialSampleSize(nullptr); }
  int sampling_type() const override { return App().samplingType(); }
  int32_t invalid_vertex() const override { return invalid_; }
  int max_bits() const override { return max_bits_; }
  size_t sample_state_bytes() const override {
    return std::is_empty<SampleType>::value ? 0 : sizeof(SampleType) * (size_t)n_samples_;
  }

  int set_graph(const CSR* graph) override {
    free_run_buffers();  // sized against the previous graph: alloc() is due again
    graph_ = nullptr;
    if (!dgraph_.upload(graph, false, app_uses_edge_lookup<App>::value, &last_error)) return -1;
    if (apps::neighborhood_form_of<App>::value == apps::kRankedByLadiesImportance) {
      // 1 / (weights of every vertex summed in edge order, sequential float adds)
      const size_t V = (size_t)graph->get_n_vertices();
      std::vector<float> sums(V);
      for (size_t v = 0; v < V; ++v) {
        float acc = 0.0f;
        for (EdgePos_t x = graph->row_ptr[v]; x < graph->row_ptr[v + 1]; ++x) acc = acc + graph->weight[x];
        sums[v] = 1.0f / acc;  // the kernels multiply by the inverse
      }
      int rc = merge_parallel_edges(sums);
      if (rc == 0) rc = build_dense_pieces(graph, sums.data());
      if (rc != 0) return rc;
    }
    if (apps::neighborhood_form_of<App>::value == apps::kDistinctByDegreeSquared) {
      ND_HIP_TRY(union_.build(dgraph_.view, bitmap_words_for((uint32_t)graph->get_n_vertices())));
      dense_pieces_ = union_.pieces;
    }
    graph_ = graph;
    return 0;
  }

  int alloc(uint64_t seed) override {
    if (!graph_) { last_error = "alloc before set_graph"; return -1; }
    free_run_buffers();
    seed_ = seed;
    CSR* csr = const_cast<CSR*>(graph_);
    App app;
    if (!is_collective<App>()) { last_error = "not a CollectiveNeighborhood app"; return -2; }
    if (app.hasExplicitTransits()) { last_error = "apps with explicit transits are not supported"; return -2; }
    const int n_steps = app.steps();
    if (n_steps < 1 || n_steps > kMaxSteps) { last_error = "steps() must be in [1, 128]"; return -2; }
    n_samples_ = app.numSamples(csr);
    init_size_ = app.initialSampleSize(csr);
    if (n_samples_ <= 0 || init_size_ <= 0) { last_error = "app yields no samples"; return -2; }
    if (n_samples_ >= (1ll << 31)) { last_error = "too many samples"; return -2; }
    uint32_t widest = (uint32_t)init_size_;
    for (int k = 0; k < n_steps; ++k) {
      if (app.stepSize(k) <= 0) { last_error = "stepSize must be positive"; return -2; }
      if ((uint32_t)app.stepSize(k) > widest) widest = (uint32_t)app.stepSize(k);
    }
    if (widest > kMaxLayerTransits) { last_error = "more than 1024 transits per sample"; return -2; }
    invalid_ = graph_->get_n_vertices();
    max_bits_ = 0;
    while ((invalid_ >> max_bits_) != 0) max_bits_++;

    samples_.clear();
    initialContents.clear();
    samples_.reserve((size_t)n_samples_);
    for (int64_t s = 0; s < n_samples_; ++s) {
      samples_.push_back(app.template initializeSample<SampleType>(csr, (VertexID_t)s));
      std::vector<VertexID_t> roots = app.initialSample((int)s, csr, samples_.back());
      if ((EdgePos_t)roots.size() != init_size_) {
        last_error = "initialSample size differs from initialSampleSize";
        return -2;
      }
      if (!roots_are_vertices(roots, graph_->get_n_vertices())) {
        last_error = "initialSample returned a root that is not a vertex of the graph";
        return -2;
      }
      initialContents.insert(initialContents.end(), roots.begin(), roots.end());
    }
    const size_t F = (size_t)final_sample_size();
    hFinalSamples.assign((size_t)n_samples_ * F, invalid_);
    h_sizes_.resize((size_t)n_samples_);
    chunk_entries_ = kLayerChunkEntries;
    bitmap_chunk_entries_ = kBitmapChunkEntries;
    progress_ = getenv("ND_PROGRESS") != nullptr;  // a line on stderr per chunk
    if (const char* env = getenv("ND_LAYER_CHUNK_ENTRIES")) {  // smaller chunks, e.g. to exercise chunking
      const long long v = atoll(env);
      if (v > 0) chunk_entries_ = bitmap_chunk_entries_ = (uint64_t)v;
    }
    // one byte per vertex for the LADIES form, one bit for the FastGCN form
    bitmap_words_ = bitmap_words_for((uint32_t)invalid_);
    // bytes a sample of a chunk holds: its bitmap (FastGCN form) or one key per vertex, padded
    // to whole stretches (LADIES form)
    uint64_t bytes_per_sample = (uint64_t)bitmap_words_ * sizeof(uint32_t);
    if (apps::neighborhood_form_of<App>::value == apps::kRankedByLadiesImportance) {
      bytes_per_sample = (uint64_t)((bitmap_words_ + kBinWords - 1) / kBinWords) * kBinVertices * sizeof(uint32_t);
    }
    const uint64_t fit = kBitmapBudgetBytes / bytes_per_sample;
    bitmap_chunk_samples_ = fit < 1 ? 1u : fit > (uint64_t)n_samples_ ? (uint32_t)n_samples_ : (uint32_t)fit;
    // the selection kernels of the LADIES form index the samples of a chunk by blockIdx.y
    if (apps::neighborhood_form_of<App>::value == apps::kRankedByLadiesImportance && bitmap_chunk_samples_ > 65535u)
      bitmap_chunk_samples_ = 65535u;

    ND_HIP_TRY(hipStreamCreate(&stream_));
    ND_HIP_TRY(hipEventCreate(&ev_begin_));
    ND_HIP_TRY(hipEventCreate(&ev_end_));
    ND_HIP_TRY(hipEventCreate(&ev_a_));
    ND_HIP_TRY(hipEventCreate(&ev_b_));
    allocated_ = true;
    ND_HIP_TRY(hipMalloc(&d_initial_, sizeof(VertexID_t) * initialContents.size()));
    ND_HIP_TRY(hipMemcpy(d_initial_, initialContents.data(), sizeof(VertexID_t) * initialContents.size(),
                         hipMemcpyHostToDevice));
    if (!std::is_empty<SampleType>::value) {
      ND_HIP_TRY(hipMalloc(&d_samples_, sizeof(SampleType) * (size_t)n_samples_));
      ND_HIP_TRY(hipMalloc(&d_samples_init_, sizeof(SampleType) * (size_t)n_samples_));
      ND_HIP_TRY(hipMemcpy(d_samples_init_, samples_.data(), sizeof(SampleType) * (size_t)n_samples_,
                           hipMemcpyHostToDevice));
      // what fetch_sample_states gives before the first run
      ND_HIP_TRY(hipMemcpy(d_samples_, d_samples_init_, sizeof(SampleType) * (size_t)n_samples_,
                           hipMemcpyDeviceToDevice));
      std::vector<SampleType>().swap(samples_);  // the pristine copy now lives on the device
    }
    ND_HIP_TRY(hipMalloc(&d_final_, sizeof(VertexID_t) * (size_t)n_samples_ * F));
    ND_HIP_TRY(hipMalloc(&d_sizes_, sizeof(uint32_t) * ((size_t)n_samples_ + 1)));
    ND_HIP_TRY(hipMemset(d_sizes_, 0, sizeof(uint32_t) * ((size_t)n_samples_ + 1)));
    ND_HIP_TRY(hipMalloc(&d_offsets_, sizeof(uint32_t) * ((size_t)n_samples_ + 1)));
    ND_HIP_TRY(hipMalloc(&d_item_count_, sizeof(uint32_t) * ((size_t)n_samples_ + 1)));
    ND_HIP_TRY(hipMalloc(&d_item_start_, sizeof(uint32_t) * ((size_t)n_samples_ + 1)));
    ND_HIP_TRY(hipMalloc(&d_row_offsets_, sizeof(uint32_t) * (size_t)n_samples_ * widest));
    ND_HIP_TRY(hipMalloc(&d_small_scratch_, sizeof(uint32_t) * scan_scratch_elems((size_t)n_samples_ + 1)));
    if (apps::neighborhood_form_of<App>::value != apps::kConcatenated) {
      ND_HIP_TRY(hipMalloc(&d_layer_counts_, sizeof(uint32_t) * 2 * (size_t)n_samples_ * n_steps));
      ND_HIP_TRY(hipHostMalloc((void**)&h_too_long_, 3 * sizeof(uint32_t), hipHostMallocDefault));
      *h_too_long_ = 0;
      ND_HIP_TRY(hipMalloc(&marked_.count, 2 * sizeof(uint32_t)));
      ND_HIP_TRY(hipMalloc(&marked_.sample, sizeof(uint32_t) * (size_t)n_samples_));
    }
    if (apps::neighborhood_form_of<App>::value == apps::kDistinctByDegreeSquared) {
      marked_.stride = widest;
      ND_HIP_TRY(hipMalloc(&marked_.transits, sizeof(int32_t) * (size_t)n_samples_ * widest));
      ND_HIP_TRY(hipMalloc(&marked_.transit_count, sizeof(uint2) * (size_t)n_samples_));
    }
    if (apps::neighborhood_form_of<App>::value == apps::kRankedByLadiesImportance) {
      const size_t per_sample = sizeof(uint32_t) * ((size_t)n_samples_ + 1);
      ND_HIP_TRY(hipMalloc(&d_ranked_start_, per_sample));
      ND_HIP_TRY(hipMalloc(&d_select_kept_, per_sample));
      ND_HIP_TRY(hipMalloc(&d_select_threshold_, per_sample));
      ND_HIP_TRY(hipMalloc(&d_select_claimed_, per_sample));
      ND_HIP_TRY(hipMalloc(&d_merged_sizes_, per_sample));
    }
    return 0;
  }

  int sample(int) override {
    if (!allocated_) { last_error = "sample before alloc"; return -1; }
    App app;
    const int n_steps = app.steps();
    const size_t F = (size_t)final_sample_size();
    times = PhaseTimes();
    neighborhood_total_ = 0;
    distinct_total_ = 0;
    chunks_run_ = 0;
    counted_ = true;
    if (h_too_long_) {
      *h_too_long_ = 0;
      ND_HIP_TRY(hipMemsetAsync(marked_.count + 1, 0, sizeof(uint32_t), stream_));
    }
    if (!std::is_empty<SampleType>::value) {
      ND_HIP_TRY(hipMemcpyAsync(d_samples_, d_samples_init_, sizeof(SampleType) * (size_t)n_samples_,
                                hipMemcpyDeviceToDevice, stream_));
    }
    ND_HIP_TRY(hipStreamSynchronize(stream_));
    ND_HIP_TRY(hipEventRecord(ev_begin_, stream_));
    const uint32_t S = (uint32_t)n_samples_;
    for (int step = 0; step < n_steps; ++step) {
      TransitView all;
      if (step == 0) {
        all.base = d_initial_;
        all.stride = (uint32_t)init_size_;
        all.count = (uint32_t)init_size_;
      } else {
        all.base = d_final_ + step_size_at_step<App>(step - 2);
        all.stride = (uint32_t)F;
        all.count = (uint32_t)app.stepSize(step - 1);
      }
      constexpr int form = apps::neighborhood_form_of<App>::value;
      if (form != apps::kConcatenated && bitmap_chunk_entries_ == kBitmapChunkEntries) {
        // chunks of as many samples as there is memory for bitmaps of: nothing the host has to know first
        for (uint32_t s0 = 0, s1; s0 < S; s0 = s1) {
          s1 = std::min(S, s0 + bitmap_chunk_samples_);
          if (run_chunk(step, all, s0, s1, 0) != 0) return -1;
          chunks_run_++;
          if (progress_ && report_progress(step, s1, /*on_device=*/true) != 0) return -1;
        }
        continue;
      }
      // size of every sample's collective neighbourhood, then chunks of samples that fit the budget
      collective_sizes<<<dim3((S + 3) / 4), dim3(256), 0, stream_>>>(dgraph_.view, all, S, invalid_, d_sizes_);
      ND_HIP_TRY(hipMemcpyAsync(h_sizes_.data(), d_sizes_, sizeof(uint32_t) * S, hipMemcpyDeviceToHost, stream_));
      ND_HIP_TRY(hipStreamSynchronize(stream_));
      // chunk limits: entries of concatenation the work arrays hold, or (bitmap form) bitmaps
      // that fit the budget and a grid of marking work items that fits 31 bits
      constexpr bool by_bitmap = form != apps::kConcatenated;
      const uint64_t entry_budget = by_bitmap ? bitmap_chunk_entries_ : chunk_entries_;
      const uint32_t sample_budget = by_bitmap ? bitmap_chunk_samples_ : S;
      for (uint32_t s = 0; s < S; ++s)
        if (h_sizes_[s] >= (1u << 31)) { last_error = kTooLong; return -2; }
      uint32_t s0 = 0;
      while (s0 < S) {
        uint64_t total = h_sizes_[s0];
        uint32_t s1 = s0 + 1;
        while (s1 < S && s1 - s0 < sample_budget && total + h_sizes_[s1] <= entry_budget) total += h_sizes_[s1++];
        if (run_chunk(step, all, s0, s1, total) != 0) return -1;
        neighborhood_total_ += total;
        chunks_run_++;
        if (progress_ && report_progress(step, s1, /*on_device=*/false) != 0) return -1;
        s0 = s1;
      }
    }
    ND_HIP_TRY(hipEventRecord(ev_end_, stream_));
    ND_HIP_TRY(hipStreamSynchronize(stream_));
    ND_HIP_TRY(hipEventElapsedTime(&times.end_to_end, ev_begin_, ev_end_));
    if (h_too_long_ && *h_too_long_) { last_error = kTooLong; return -2; }
    counted_ = apps::neighborhood_form_of<App>::value == apps::kConcatenated;
    return 0;
  }

  int fetch_final_samples() override {
    if (!allocated_) { last_error = "no device data"; return -1; }
    hFinalSamples.resize((size_t)n_samples_ * (size_t)final_sample_size());
    return fetch_to_host(hFinalSamples.data(), d_final_, sizeof(VertexID_t) * hFinalSamples.size(), (uint32_t)max_bits(),
                         invalid_, stream_);
  }

  int fetch_sample_states(void* dst, size_t bytes) override {
    if (!allocated_ || std::is_empty<SampleType>::value) { last_error = "no sample state"; return -1; }
    if (bytes != sample_state_bytes()) { last_error = "sample state size mismatch"; return -1; }
    return states_to_host(dst, d_samples_, bytes, stream_);
  }

  int distinct() override {
    last_error = "distinct applies to IndividualNeighborhood results";
    return -2;
  }

  // sizes of the last run, for the algorithmic-bytes figure
  int64_t counter(int which) const override {
    if (!counted_ && (which == 0 || which == 1)) {  // the last pass left them on the device
      std::vector<uint32_t> all(2 * (size_t)n_samples_ * (size_t)App().steps());
      if (hipMemcpy(all.data(), d_layer_counts_, sizeof(uint32_t) * all.size(), hipMemcpyDeviceToHost) != hipSuccess) return 0;
      neighborhood_total_ = distinct_total_ = 0;
      for (size_t i = 0; i < all.size(); ++i) (i < all.size() / 2 ? neighborhood_total_ : distinct_total_) += all[i];
      counted_ = true;
    }
    return which == 0 ? (int64_t)neighborhood_total_ : which == 1 ? (int64_t)distinct_total_
           : which == 2 ? (int64_t)chunks_run_ : which == 3 ? (int64_t)dense_pieces_ : 0;
  }

  void free_device() override {
    free_run_buffers();
    release_merged();
    release_dense_pieces();
    union_.release();
    dgraph_.release();
    graph_ = nullptr;
  }

 private:
  template <class T>
  static void release(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
  }

  // The graph's edges with their terms, parallel ones as one (MergedEdges).
  int merge_parallel_edges(const std::vector<float>& inverse_row_sums) {
    release_merged();
    const size_t E = (size_t)graph_edges(), V = inverse_row_sums.size();
    float* d_inverse = nullptr;
    uint32_t *d_at = nullptr, *d_zero = nullptr, *d_scratch = nullptr;
    uint32_t pairs = 0, zero = 0;
    hipError_t e = hipMalloc(&d_inverse, sizeof(float) * V);
    if (e == hipSuccess) e = hipMemcpy(d_inverse, inverse_row_sums.data(), sizeof(float) * V, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMalloc(&d_at, sizeof(uint32_t) * (E + 1));
    if (e == hipSuccess) e = hipMalloc(&d_scratch, sizeof(uint32_t) * scan_scratch_elems(E + 1));
    if (e == hipSuccess) e = hipMalloc(&d_zero, sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemset(d_zero, 0, sizeof(uint32_t));
    const dim3 over_edges((unsigned)((E + 256) / 256));
    if (e == hipSuccess) {
      first_of_parallel_edges<<<over_edges, dim3(256)>>>(dgraph_.view, d_at);
      e = exclusive_scan_u32(d_at, d_at, E + 1, d_scratch, nullptr);
    }
    if (e == hipSuccess) e = hipMemcpy(&pairs, d_at + E, sizeof(pairs), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMalloc(&d_merged_rows_, sizeof(EdgePos_t) * (V + 1));
    if (e == hipSuccess) e = hipMalloc(&d_merged_ids_, sizeof(VertexID) * std::max<size_t>(1, pairs));
    if (e == hipSuccess) e = hipMalloc(&d_merged_terms_, sizeof(unsigned long long) * std::max<size_t>(1, pairs));
    if (e == hipSuccess) {
      merge_rows<<<dim3((unsigned)((V + 256) / 256)), dim3(256)>>>(dgraph_.view, d_at, d_merged_rows_);
      merge_edges<<<over_edges, dim3(256)>>>(dgraph_.view, d_inverse, d_at, d_merged_ids_, d_merged_terms_, d_zero);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&zero, d_zero, sizeof(zero), hipMemcpyDeviceToHost);
    release(d_inverse); release(d_at); release(d_zero); release(d_scratch);
    if (e != hipSuccess) {
      release_merged();
      last_error = std::string("merging parallel edges: ") + hipGetErrorString(e);
      return -1;
    }
    merged_ = MergedEdges{d_merged_rows_, d_merged_ids_, d_merged_terms_, zero != 0, nullptr, nullptr};
    return cut_merged_rows();
  }
  int cut_merged_rows() {
    CSRPartition view = dgraph_.view;
    view.row_ptr = d_merged_rows_;
    view.edges = d_merged_ids_;
    const uint32_t V = (uint32_t)view.n_vertices, stretches = (bitmap_words_for(V) + kBinWords - 1) / kBinWords;
    uint32_t *d_rows = nullptr, rows = 0;
    int32_t* d_vertex_of = nullptr;
    const dim3 over_vertices((V + 255u) / 256u);
    hipError_t e = hipMalloc(&d_rows, sizeof(uint32_t));
    uint32_t from_degree = kCutDegree;
    for (; e == hipSuccess; from_degree *= 2) {  // fewer rows where the cuts of all of them would take too much
      e = hipMemset(d_rows, 0, sizeof(uint32_t));
      if (e != hipSuccess) break;
      number_hubs<<<over_vertices, dim3(256)>>>(view, from_degree, nullptr, nullptr, d_rows);
      e = hipMemcpy(&rows, d_rows, sizeof(rows), hipMemcpyDeviceToHost);
      if (e != hipSuccess || (size_t)rows * (stretches + 1) * sizeof(HubCut) <= kCutBudgetBytes) break;
    }
    if (e == hipSuccess && rows > 0) {
      e = hipMalloc(&d_cut_row_of_, sizeof(int32_t) * V);
      if (e == hipSuccess) e = hipMalloc(&d_vertex_of, sizeof(int32_t) * rows);
      if (e == hipSuccess) e = hipMalloc(&d_cuts_, sizeof(HubCut) * (size_t)rows * (stretches + 1));
      if (e == hipSuccess) e = hipMemset(d_rows, 0, sizeof(uint32_t));
      if (e == hipSuccess) {
        number_hubs<<<over_vertices, dim3(256)>>>(view, from_degree, d_cut_row_of_, d_vertex_of, d_rows);
        cut_hubs<<<dim3((rows + 255) / 256, stretches + 1), dim3(256)>>>(view, d_vertex_of, rows, stretches, kBinVertices, d_cuts_);
        e = hipGetLastError();
      }
      if (e == hipSuccess) e = hipDeviceSynchronize();
    }
    release(d_rows); release(d_vertex_of);
    if (e != hipSuccess) {
      release_merged();
      last_error = std::string("cutting rows: ") + hipGetErrorString(e);
      return -1;
    }
    merged_.cut_row_of = d_cut_row_of_;
    merged_.cuts = d_cuts_;
    return 0;
  }
  size_t graph_edges() const { return (size_t)dgraph_.view.n_edges; }
  void release_merged() {
    release(d_merged_rows_); release(d_merged_ids_); release(d_merged_terms_);
    release(d_cut_row_of_); release(d_cuts_);
    merged_ = MergedEdges{};
  }

  // What the vertices with many neighbours in one stretch contribute to it, built once per graph (see DensePieces).
  int build_dense_pieces(const CSR* graph, const float* inverse_row_sums) {
    release_dense_pieces();
    uint32_t threshold = kDensePieceEntries;
    if (const char* env = getenv("ND_DENSE_PIECE_ENTRIES")) {  // 0: no pieces; small: to exercise them on small graphs
      const long long v = atoll(env);
      if (v <= 0) return 0;
      threshold = (uint32_t)v;
    }
    const uint32_t V = (uint32_t)graph->get_n_vertices();
    const uint32_t stretches = (bitmap_words_for(V) + kBinWords - 1) / kBinWords;
    const size_t most_pieces = kDensePieceBudgetBytes / (sizeof(uint64_t) * kBinVertices);
    std::vector<int32_t> hub_row(V, -1);
    std::vector<uint32_t> piece_of;
    std::vector<unsigned long long> sums;
    size_t n_hubs = 0, n_pieces = 0;
    for (uint32_t v = 0; v < V; ++v) {
      const int32_t* const row = graph->col.data() + graph->row_ptr[v];
      const int32_t* first = row;
      const int32_t* last = graph->col.data() + graph->row_ptr[v + 1];
      if ((size_t)(last - first) < threshold) continue;
      while (first < last) {  // one sub-range of the sorted adjacency per stretch
        const uint32_t b = (uint32_t)*first / kBinVertices;
        const uint32_t limit = (b + 1) * kBinVertices;
        const int32_t* stop = std::partition_point(first, last, [limit](int32_t c) { return (uint32_t)c < limit; });
        size_t neighbours = (size_t)(stop - first);
        if (neighbours >= threshold) {  // without the repeats
          neighbours = 1;
          for (const int32_t* c = first + 1; c < stop; ++c) neighbours += c[0] != c[-1];
        }
        if (neighbours >= threshold && n_pieces < most_pieces) {
          if (hub_row[v] < 0) {
            hub_row[v] = (int32_t)n_hubs++;
            piece_of.resize(n_hubs * stretches, kNoPiece);
          }
          piece_of[(size_t)hub_row[v] * stretches + b] = (uint32_t)n_pieces;
          sums.resize((n_pieces + 1) * kBinVertices, kAbsentSum);
          unsigned long long* of = sums.data() + n_pieces * kBinVertices;
          for (const int32_t* c = first; c < stop; ++c) {
            // the term of this edge, in the arithmetic of merge_edges
            const float p = graph->weight[(size_t)graph->row_ptr[v] + (size_t)(c - row)] * inverse_row_sums[v];
            unsigned long long& sum = of[(uint32_t)*c - b * kBinVertices];
            sum = (sum == kAbsentSum ? 0 : sum) + importance_term_fixed(p * p);
          }
          ++n_pieces;
        }
        first = stop;
      }
    }
    if (n_pieces == 0) return 0;
    ND_HIP_TRY(hipMalloc(&d_hub_row_, sizeof(int32_t) * V));
    ND_HIP_TRY(hipMalloc(&d_piece_of_, sizeof(uint32_t) * piece_of.size()));
    ND_HIP_TRY(hipMalloc(&d_piece_sums_, sizeof(uint64_t) * sums.size()));
    ND_HIP_TRY(hipMemcpy(d_hub_row_, hub_row.data(), sizeof(int32_t) * V, hipMemcpyHostToDevice));
    ND_HIP_TRY(hipMemcpy(d_piece_of_, piece_of.data(), sizeof(uint32_t) * piece_of.size(), hipMemcpyHostToDevice));
    ND_HIP_TRY(hipMemcpy(d_piece_sums_, sums.data(), sizeof(uint64_t) * sums.size(), hipMemcpyHostToDevice));
    dense_.hub_row = d_hub_row_;
    dense_.piece_of = d_piece_of_;
    dense_.sums = d_piece_sums_;
    dense_pieces_ = n_pieces;
    return 0;
  }

  void release_dense_pieces() {
    release(d_hub_row_);
    release(d_piece_of_);
    release(d_piece_sums_);
    dense_ = DensePieces();
    dense_pieces_ = 0;
  }


  static constexpr uint32_t kDrawBlocks = 4096;
  static constexpr const char* kTooLong = "collective neighbourhood of one sample has 2^31 or more entries";

  // A line on stderr when a chunk of a layer is done.  on_device: the sizes of its neighbourhoods were not needed here, and are
  // there, layer after layer.
  int report_progress(int step, uint32_t samples_done, bool on_device) {
    ND_HIP_TRY(hipStreamSynchronize(stream_));
    uint64_t entries = neighborhood_total_;
    if (on_device) {
      std::vector<uint32_t> sizes((size_t)n_samples_ * step + samples_done);
      ND_HIP_TRY(hipMemcpy(sizes.data(), d_layer_counts_, sizeof(uint32_t) * sizes.size(), hipMemcpyDeviceToHost));
      for (uint32_t n : sizes) entries += n;
    }
    fprintf(stderr, "[nextdoor] layer %d: samples %u of %u done, %llu neighbourhood entries so far\n", step, samples_done,
            (uint32_t)n_samples_, (unsigned long long)entries);
    fflush(stderr);
    return 0;
  }

  // events around the neighbourhood kernel when profiling is on
  void tick() {
    if (profiling) (void)hipEventRecord(ev_a_, stream_);
  }
  void tock() {
    if (!profiling) return;
    (void)hipEventRecord(ev_b_, stream_);
    (void)hipEventSynchronize(ev_b_);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, ev_a_, ev_b_);
    times.neighborhood += ms;
    times.neighborhood_launches++;
  }

  // One chunk of samples [s0, s1) of one layer: concatenate, post-process in the form the
  // app asks for, run next() for every (sample, nbr).
  int run_chunk(int step, const TransitView& all, uint32_t s0, uint32_t s1, uint64_t total) {
    App app;
    const uint32_t n = s1 - s0;
    const size_t F = (size_t)final_sample_size();
    constexpr int form = apps::neighborhood_form_of<App>::value;
    TransitView tv = all;
    tv.base = all.base + (size_t)s0 * all.stride;
    if (form == apps::kConcatenated) {
      // work items of the build: long neighbourhoods are spread over several workgroups
      uint64_t n_items = 0;
      for (uint32_t s = s0; s < s1; ++s) {
        const uint64_t items = ((uint64_t)h_sizes_[s] + kBuildItemEntries - 1) / kBuildItemEntries;
        n_items += items ? items : 1;
      }
      if (n_items >= (1ull << 31)) { last_error = "a chunk needs 2^31 or more work items"; return -2; }
      build_item_counts<<<dim3((n + 1 + 255) / 256), dim3(256), 0, stream_>>>(d_sizes_ + s0, n, d_item_count_);
      ND_HIP_TRY(exclusive_scan_u32(d_item_count_, d_item_start_, (size_t)n + 1, d_small_scratch_, stream_));
      if (ensure_neighborhood_capacity((uint32_t)total) != 0) return -1;
      // offsets of the chunk's samples, relative to the chunk (element n = total)
      ND_HIP_TRY(exclusive_scan_u32(d_sizes_ + s0, d_offsets_, (size_t)n + 1, d_small_scratch_, stream_));
      tick();
      collective_build<<<dim3((unsigned)n_items), dim3(256), 0, stream_>>>(
          dgraph_.view, tv, invalid_, d_offsets_, d_item_start_, n, d_nbr_cols_, d_nbr_weights_,
          d_row_offsets_ + (size_t)s0 * all.count);
      tock();
      ND_HIP_TRY(hipGetLastError());
    }

    LayerParams P{};
    P.csr = dgraph_.view;
    P.transits = tv;
    P.step = step;
    P.step_size = (uint32_t)app.stepSize(step);
    P.chunk_samples = n;
    P.sample_begin = s0;
    P.final_size = (uint32_t)F;
    P.out_base = (uint32_t)step_size_at_step<App>(step - 1);
    P.invalid = invalid_;
    P.seed = seed_;
    P.first_sample = 0;
    P.final_samples = d_final_;
    P.samples = d_samples_;
    P.offsets = d_offsets_;
    P.nbr_cols = d_nbr_cols_;
    P.nbr_weights = d_nbr_weights_;
    if constexpr (form == apps::kDistinctByDegreeSquared) {
      return run_by_degree(P, step);
    } else if constexpr (form == apps::kRankedByLadiesImportance) {
      return run_ranked(P, step);
    } else {
      const uint64_t outputs = (uint64_t)n * P.step_size;
      layer_execute_kernel<SampleType, App><<<dim3((unsigned)((outputs + 255) / 256)), dim3(256), 0, stream_>>>(P);
      ND_HIP_TRY(hipGetLastError());
      return 0;
    }
  }

  // kDistinctByDegreeSquared: the samples of the chunk by the size of their neighbourhoods, and their draws.
  int run_by_degree(const LayerParams& P, int step) {
    const uint32_t n = P.chunk_samples, parts = union_.parts;
    const size_t n_parts = (size_t)n * parts;
    if (n > bitmap_samples_) {
      release(d_bitmap_); release(d_group_through_); release(d_part_total_); release(d_part_before_);
      ND_HIP_TRY(hipMalloc(&d_bitmap_, sizeof(uint32_t) * (size_t)n * bitmap_words_));
      ND_HIP_TRY(hipMalloc(&d_group_through_, sizeof(uint64_t) * n_parts * kGroupsPerPart));
      ND_HIP_TRY(hipMalloc(&d_part_total_, sizeof(uint64_t) * n_parts));
      ND_HIP_TRY(hipMalloc(&d_part_before_, sizeof(uint64_t) * (size_t)n * (parts + 1)));
      bitmap_samples_ = n;
    }
    const size_t S = (size_t)n_samples_;
    uint32_t* sizes = d_layer_counts_ + S * step + P.sample_begin;
    uint32_t* distinct = sizes + S * App().steps();
    ND_HIP_TRY(hipMemsetAsync(marked_.count, 0, sizeof(uint32_t), stream_));
    sort_out_samples<<<dim3((n + 15) / 16), dim3(kSortOutThreads), 0, stream_>>>(P.csr, P.transits, n, invalid_, union_.hubs.row_of, sizes,
                                                                   distinct, marked_, h_too_long_);
    tick();
    sorted_layer_kernel<SampleType, App><<<dim3(n), dim3(kSortedThreads), 0, stream_>>>(P, sizes, distinct);
    const uint32_t turns = (parts + kXcdCount - 1) / kXcdCount * kUnionSlices;
    union_parts<<<dim3(turns * kXcdCount), dim3(kUnionThreads), 0, stream_>>>(P.csr, union_.hubs, parts, marked_, bitmap_words_,
                                                                              d_bitmap_);
    union_sums<<<dim3(parts * kSumSlices), dim3(kSumThreads), 0, stream_>>>(
        union_.squares, union_.square_rows, parts, marked_, bitmap_words_, d_bitmap_, d_group_through_, d_part_total_, distinct);
    tock();
    sample_part_sums<<<dim3(n), dim3(64), 0, stream_>>>(d_part_total_, parts, marked_.count, d_part_before_);
    marked_layer_kernel<SampleType, App><<<dim3(kDrawBlocks), dim3(256), 0, stream_>>>(
        P, marked_, distinct, d_bitmap_, bitmap_words_, d_part_before_, d_group_through_, parts);
    ND_HIP_TRY(hipGetLastError());
    return 0;
  }

  // LADIES form: small neighbourhoods are ranked by a workgroup each.  The others leave one sampling key per (sample,
  // vertex); per sample, the vertices that can be among its first `wanted` in key order are picked by a radix select on the
  // upper 14 bits of the key and ordered by descending key.  Their distinct pairs (2.4 M per batch at full size) are
  // never listed.
  int run_ranked(LayerParams P, int step) {
    const uint32_t n = P.chunk_samples;
    const uint32_t bins = (bitmap_words_ + kBinWords - 1) / kBinWords, groups = (bins + kBinsPerGroup - 1) / kBinsPerGroup;
    if ((uint64_t)n * groups >= (1ull << 31)) { last_error = "a chunk needs 2^31 or more workgroups"; return -1; }
    const uint32_t keys_per_sample = bins * kBinVertices;
    if (n > bitmap_samples_) {
      release(d_keys_dense_); release(d_stretch_best_);
      ND_HIP_TRY(hipMalloc(&d_keys_dense_, sizeof(uint32_t) * (size_t)n * keys_per_sample));
      ND_HIP_TRY(hipMalloc(&d_stretch_best_, sizeof(uint16_t) * (size_t)n * (keys_per_sample / kCollectStretch)));
      bitmap_samples_ = n;
    }
    const size_t S = (size_t)n_samples_;
    uint32_t* sizes = d_layer_counts_ + S * step + P.sample_begin;
    uint32_t* distinct = sizes + S * App().steps();
    ND_HIP_TRY(hipMemsetAsync(marked_.count, 0, sizeof(uint32_t), stream_));
    sort_out_ranked<<<dim3((n + 15) / 16), dim3(kSortOutThreads), 0, stream_>>>(
        P.csr, merged_, P.transits, n, invalid_, sizes, d_merged_sizes_, marked_.count, marked_.sample, h_too_long_);
    tick();
    ranked_layer_kernel<SampleType, App><<<dim3(n), dim3(kRankedThreads), 0, stream_>>>(P, merged_, d_merged_sizes_, distinct);
    KeysOnTheWayOut keys_out;
    keys_out.keys = d_keys_dense_;
    keys_out.seed = seed_;
    keys_out.first_sample = P.first_sample + P.sample_begin;
    keys_out.step = (uint32_t)step;
    keys_out.n_vertices = (uint32_t)invalid_;
    collective_mark_binned<<<dim3(n * groups), dim3(kBinThreads), 0, stream_>>>(
        merged_, P.transits, invalid_, n, marked_.count, marked_.sample, bins, keys_per_sample, dense_, keys_out);
    tock();
    const uint32_t wanted = (uint32_t)App().stepSize(step);
    select_threshold<<<dim3(n), dim3(kSelectThreads), 0, stream_>>>(d_keys_dense_, keys_per_sample, wanted, marked_.count,
                                                                    marked_.sample, d_select_threshold_, d_select_kept_,
                                                                    d_select_claimed_, distinct, d_stretch_best_);
    // where every sample's ranked list starts: exclusive scan of the kept counts
    fill_u32<<<dim3(1), dim3(1), 0, stream_>>>(d_select_kept_ + n, 1, 0u);
    ND_HIP_TRY(exclusive_scan_u32(d_select_kept_, d_ranked_start_, (size_t)n + 1, d_small_scratch_, stream_));
    ND_HIP_TRY(hipMemcpyAsync(h_too_long_ + 1, marked_.count, sizeof(uint32_t), hipMemcpyDeviceToHost, stream_));
    ND_HIP_TRY(hipMemcpyAsync(h_too_long_ + 2, d_small_scratch_ + scan_num_tiles((size_t)n + 1), sizeof(uint32_t),
                              hipMemcpyDeviceToHost, stream_));
    ND_HIP_TRY(hipStreamSynchronize(stream_));
    const uint32_t n_marked = h_too_long_[1], n_kept = h_too_long_[2];
    if (n_marked == 0) return 0;
    if (ensure_distinct_capacity(n_kept) != 0) return -1;
    select_collect<<<dim3(n_marked), dim3(kSelectThreads), 0, stream_>>>(
        d_keys_dense_, keys_per_sample, d_stretch_best_, d_select_threshold_, d_ranked_start_, d_select_claimed_, d_kept_key_,
        d_kept_sample_, d_kept_id_);
    // order the kept vertices of every sample by descending key, equal keys by ascending
    // vertex id: stable sorts by vertex, then by key, then by sample
    if (n_kept > 0) {
      int chunk_bits = 1;
      while (((uint64_t)n >> chunk_bits) != 0) chunk_bits++;
      const unsigned blocks = (n_kept + 255) / 256;
      const SortPlan by_vertex = make_sort_plan(n_kept, max_bits_);
      uint32_t *k2 = nullptr, *j2 = nullptr;
      ND_HIP_TRY(radix_sort_pairs(by_vertex, (const uint32_t*)d_kept_id_, nullptr, d_keys_a_, d_vals_a_, d_keys_b_,
                                  d_vals_b_, d_hist_, d_scratch_, stream_, &k2, &j2));
      gather_u32<<<dim3(blocks), dim3(256), 0, stream_>>>(d_kept_key_, j2, n_kept, d_key2_, d_index2_);
      const SortPlan by_key = make_sort_plan(n_kept, 32);
      uint32_t *k3 = nullptr, *j3 = nullptr;
      ND_HIP_TRY(radix_sort_pairs(by_key, d_key2_, d_index2_, d_keys_a_, d_vals_a_, d_keys_b_, d_vals_b_, d_hist_,
                                  d_scratch_, stream_, &k3, &j3));
      gather_u32<<<dim3(blocks), dim3(256), 0, stream_>>>(d_kept_sample_, j3, n_kept, d_key2_, d_index2_);
      const SortPlan by_sample = make_sort_plan(n_kept, chunk_bits);
      uint32_t *k4 = nullptr, *j4 = nullptr;
      ND_HIP_TRY(radix_sort_pairs(by_sample, d_key2_, d_index2_, d_keys_a_, d_vals_a_, d_keys_b_, d_vals_b_, d_hist_,
                                  d_scratch_, stream_, &k4, &j4));
      gather_u32<<<dim3(blocks), dim3(256), 0, stream_>>>((const uint32_t*)d_kept_id_, j4, n_kept,
                                                          (uint32_t*)d_ranked_ids_, nullptr);
    }
    P.ranked_start = d_ranked_start_;
    P.ranked_ids = d_ranked_ids_;
    P.marked = marked_.sample;
    P.n_marked = n_marked;
    const uint64_t outputs = (uint64_t)n_marked * P.step_size;
    layer_execute_kernel<SampleType, App><<<dim3((unsigned)((outputs + 255) / 256)), dim3(256), 0, stream_>>>(P);
    ND_HIP_TRY(hipGetLastError());
    return 0;
  }

  // Arrays with one entry per listed (sample, vertex) pair of a chunk: the distinct pairs
  // (FastGCN form) or the pairs the selection keeps (LADIES form).
  int ensure_distinct_capacity(uint32_t n_distinct) {
    if (n_distinct <= distinct_capacity_ && distinct_capacity_ > 0) return 0;
    constexpr int form = apps::neighborhood_form_of<App>::value;
    const size_t cap = (size_t)n_distinct + n_distinct / 8 + 1024;
    release_distinct_buffers();
    if (form == apps::kRankedByLadiesImportance) {
      ND_HIP_TRY(hipMalloc(&d_ranked_ids_, sizeof(int32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_kept_key_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_kept_sample_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_kept_id_, sizeof(int32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_keys_a_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_vals_a_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_keys_b_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_vals_b_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_key2_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_index2_, sizeof(uint32_t) * cap));
      ND_HIP_TRY(hipMalloc(&d_hist_, sizeof(uint32_t) * sort_hist_capacity(cap)));
      size_t scratch = make_sort_plan(cap, 32).scratch_elems;
      ND_HIP_TRY(hipMalloc(&d_scratch_, sizeof(uint32_t) * scratch));
    }
    distinct_capacity_ = cap;
    return 0;
  }

  // The concatenated neighbourhood itself (kConcatenated form).
  int ensure_neighborhood_capacity(uint32_t total) {
    if (total <= capacity_ && capacity_ > 0) return 0;
    const size_t cap = (size_t)total + total / 8 + 1024;
    release(d_nbr_cols_); release(d_nbr_weights_);
    ND_HIP_TRY(hipMalloc(&d_nbr_cols_, sizeof(int32_t) * cap));
    ND_HIP_TRY(hipMalloc(&d_nbr_weights_, sizeof(float) * cap));
    capacity_ = cap;
    return 0;
  }

  void release_distinct_buffers() {
    release(d_ranked_ids_);
    release(d_keys_a_); release(d_vals_a_); release(d_keys_b_); release(d_vals_b_);
    release(d_key2_); release(d_index2_); release(d_hist_); release(d_scratch_);
    release(d_kept_key_); release(d_kept_sample_); release(d_kept_id_);
    distinct_capacity_ = 0;
  }

  void release_neighborhood_buffers() {
    release(d_nbr_cols_); release(d_nbr_weights_);
    release(d_bitmap_); release(d_keys_dense_); release(d_stretch_best_);
    release(d_group_through_); release(d_part_total_); release(d_part_before_);
    release_distinct_buffers();
    capacity_ = 0;
    bitmap_samples_ = 0;
  }

  void free_run_buffers() {
    release(d_initial_); release(d_samples_); release(d_samples_init_); release(d_final_);
    release(d_sizes_); release(d_offsets_); release(d_row_offsets_); release(d_small_scratch_);
    release(d_item_count_); release(d_item_start_);
    release(d_layer_counts_);
    if (h_too_long_) (void)hipHostFree(h_too_long_);
    h_too_long_ = nullptr;
    release(marked_.count); release(marked_.sample); release(marked_.transits); release(marked_.transit_count);
    release(d_ranked_start_); release(d_select_kept_);
    release(d_select_threshold_); release(d_select_claimed_); release(d_merged_sizes_);
    release_neighborhood_buffers();
    // whatever exists, also after an alloc that failed half way
    for (hipEvent_t* ev : {&ev_a_, &ev_b_, &ev_begin_, &ev_end_}) {
      if (*ev) (void)hipEventDestroy(*ev);
      *ev = nullptr;
    }
    if (stream_) (void)hipStreamDestroy(stream_);
    stream_ = nullptr;
    allocated_ = false;
  }

  const char* name_;
  const CSR* graph_ = nullptr;
  DeviceGraph dgraph_;
  int32_t* d_hub_row_ = nullptr;       // dense pieces of the graph (LADIES form)
  uint32_t* d_piece_of_ = nullptr;
  unsigned long long* d_piece_sums_ = nullptr;
  DensePieces dense_;
  size_t dense_pieces_ = 0;
  std::vector<SampleType> samples_;
  std::vector<uint32_t> h_sizes_;
  int64_t n_samples_ = 0;
  int init_size_ = 0;
  int32_t invalid_ = 0;
  int max_bits_ = 0;
  uint64_t seed_ = 0;
  bool allocated_ = false;
  size_t capacity_ = 0;
  uint32_t bitmap_words_ = 0;          // 32-bit words of one sample's presence map (a multiple of kBitmapTileWords)
  uint32_t bitmap_chunk_samples_ = 0;  // samples whose bitmaps fit the budget
  uint64_t bitmap_chunk_entries_ = 0;
  uint32_t bitmap_samples_ = 0;        // samples the allocated bitmaps hold
  size_t distinct_capacity_ = 0;
  uint32_t* d_bitmap_ = nullptr;
  // LADIES form: importance sums and sampling keys, [sample][vertex, padded to whole stretches]
  uint32_t* d_keys_dense_ = nullptr;
  uint16_t* d_stretch_best_ = nullptr;  // LADIES form: best key prefix of every 256 keys of every sample
  mutable uint64_t neighborhood_total_ = 0, distinct_total_ = 0;
  uint64_t chunks_run_ = 0;
  mutable bool counted_ = true;  // those two are the last pass's
  uint64_t chunk_entries_ = kLayerChunkEntries;
  bool progress_ = false;

  hipStream_t stream_ = nullptr;
  hipEvent_t ev_begin_ = nullptr, ev_end_ = nullptr, ev_a_ = nullptr, ev_b_ = nullptr;
  VertexID_t* d_initial_ = nullptr;
  SampleType* d_samples_ = nullptr;
  SampleType* d_samples_init_ = nullptr;
  VertexID_t* d_final_ = nullptr;
  uint32_t *d_sizes_ = nullptr, *d_offsets_ = nullptr, *d_row_offsets_ = nullptr, *d_small_scratch_ = nullptr;
  uint32_t *d_item_count_ = nullptr, *d_item_start_ = nullptr;
  // LADIES form: the selection of the best keys per sample
  uint32_t *d_ranked_start_ = nullptr, *d_select_kept_ = nullptr, *d_select_threshold_ = nullptr;
  uint32_t* d_select_claimed_ = nullptr;  // entries of a sample that have been given room
  uint32_t* d_merged_sizes_ = nullptr;    // pairs of a sample's neighbourhood
  EdgePos_t* d_merged_rows_ = nullptr;    // the graph without parallel edges
  VertexID* d_merged_ids_ = nullptr;
  unsigned long long* d_merged_terms_ = nullptr;
  int32_t* d_cut_row_of_ = nullptr;
  HubCut* d_cuts_ = nullptr;
  MergedEdges merged_{};
  uint32_t *d_kept_key_ = nullptr, *d_kept_sample_ = nullptr;
  int32_t* d_kept_id_ = nullptr;
  int32_t* d_nbr_cols_ = nullptr;
  float* d_nbr_weights_ = nullptr;
  uint32_t *d_keys_a_ = nullptr, *d_vals_a_ = nullptr, *d_keys_b_ = nullptr, *d_vals_b_ = nullptr;
  uint32_t *d_key2_ = nullptr, *d_index2_ = nullptr, *d_hist_ = nullptr, *d_scratch_ = nullptr;
  // FastGCN form: degree^2 of the marked vertices, by group inside a part, by part, by sample
  uint64_t *d_group_through_ = nullptr, *d_part_total_ = nullptr, *d_part_before_ = nullptr;
  UnionTables union_;                  // of the graph
  MarkedSamples marked_{};
  uint32_t* d_layer_counts_ = nullptr;  // entries of every layer and sample's neighbourhood, then its distinct vertices
  uint32_t* h_too_long_ = nullptr;      // whether a neighbourhood was too long, and two counts the LADIES form waits for
  int32_t* d_ranked_ids_ = nullptr;
};

}  // namespace nd
