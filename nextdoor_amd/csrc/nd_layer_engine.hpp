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
//    stretch by stretch, and of the keys formed from the sums as they leave LDS those that can be among the sample's
//    first picks are kept (the only thing stored); one more workgroup a sample puts them in order.
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
__host__ __device__ __forceinline__ uint64_t ladies_pair_index(uint64_t sample, uint32_t n_vertices, uint32_t v) {
  return sample * (uint64_t)((n_vertices + 3u) & ~3u) + v;
}
__device__ __forceinline__ PhiloxBlock ladies_block(uint64_t pair, uint32_t step, uint64_t seed) {
  const uint64_t block = pair >> 2;
  // (the key opaque, as in grouped_first_block_scalar_seed: the round keys as they come, not twenty of them in registers)
  uint32_t k0 = __builtin_amdgcn_readfirstlane((uint32_t)seed), k1 = __builtin_amdgcn_readfirstlane((uint32_t)(seed >> 32));
  asm volatile("" : "+s"(k0), "+s"(k1));
  return philox4x32_10((uint32_t)block, (uint32_t)(block >> 32), step, 0, k0, k1);
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
// Whether ladies_key_from_word of the same can be at or below the bound that `reach` belongs to (Keeper::reach): the word's
// upper 24 bits against the least that can be, with 4 for what the float of 2^24 and the uniform itself are rounded by.
__device__ __forceinline__ bool key_may_be_within(float reach, unsigned long long importance_fixed, uint32_t word) {
  const float least = __builtin_fmaf((float)((uint32_t)(importance_fixed >> 32) + 1u), -reach, 16777212.0f);
  return (word >> 8) >= (uint32_t)least;  // (negative and NaN: 0)
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

// One workgroup per (sample, some consecutive stretches of 7168 vertices), the sums of one stretch in LDS at a time.
// Adjacencies are sorted by destination, so the part of a transit's adjacency that falls into a stretch is one
// sub-range; the workgroup streams the sub-ranges of all the sample's transits and adds in LDS, and no atomic reaches
// memory (global atomics stop at ~24 G/s on this part).  Every wavefront walks a contiguous part of the stretch's entries,
// a few of each lane at a time, and finds the sub-range of each from bits that say where the next ones start.
constexpr uint32_t kBinThreads = 1024;
constexpr uint32_t kBinWaves = kBinThreads / 64;
constexpr uint32_t kBinAhead = 4;             // entries a lane fetches before it works on the first
constexpr uint32_t kBinsPerGroup = 16;        // consecutive stretches of a sample one workgroup takes
constexpr uint32_t kBinVertices = 7168;       // 56 KB of 64-bit sums + 896 B of bits
constexpr uint32_t kBinWords = kBinVertices / 32u;

// Dense pieces.  What a hub contributes to a stretch can be thousands of entries (a layer drawn by importance sits on
// the hubs), and it is the same for every sample that holds the hub.  Where a vertex has kDensePieceEntries or more
// neighbours in one stretch, the stretch's piece of that vertex is built once per graph - the importance sum of every
// vertex of the stretch (7168 64-bit integers, 0 where there is no edge; there is no piece where an edge's sum is 0) - and a
// sample adds the piece on the stretch's way out of LDS instead of going through the entries.  hub_row[v] = row of v in piece_of or -1;
// piece_of[row * stretches + stretch] = piece index or kNoPiece.
constexpr uint32_t kDensePieceEntries = 2048;
constexpr size_t kDensePieceBudgetBytes = (size_t)2 << 30;
struct DensePieces {
  const int32_t* hub_row = nullptr;  // nullptr: the graph has none
  const uint32_t* piece_of = nullptr;
  const unsigned long long* sums = nullptr;
};

// ---- the best keys of a sample ----
//
// Only the first stepSize vertices of a sample in key order are ever read, out of up to millions: `wanted` of them.  A
// workgroup forms the keys of its stretches where the sums leave LDS and keeps those that can still be among them: it
// counts what it has kept by the upper bits of the keys, and once `wanted` keys lie at or below an edge between two counts
// (the bound) nothing above that edge can be.  A bound is good for the whole sample, and workgroups that start later begin
// with it.  (One key for every vertex of a sample, written to memory, selected from and sorted by the radix sort's launches:
// 2 GB written and read and 50 launches a layer over 500 K vertices.)
// By float exponent and two bits of the mantissa: an edge lets at most a quarter too many through.
constexpr uint32_t kBoundBins = 1024;
constexpr uint32_t kNoBound = 0xFFFFFFFEu;  // below kAbsentKey
// a key is the bit pattern of a negative float, or of +0 (the best there is) as 0x7FFFFFFF
__device__ __forceinline__ uint32_t bin_of_key(uint32_t key) { return (int32_t)key >= 0 ? 0u : key >> 21 & (kBoundBins - 1u); }
__device__ __forceinline__ uint32_t last_key_of_bin(uint32_t bin) { return 0x80000000u | bin << 21 | 0x1FFFFFu; }

// What a workgroup keeps at most: room for everything a stretch can add to what it may begin the stretch with.
constexpr uint32_t kKeptEntries = 12288;
struct KeptKeys {
  uint2* kept;          // (key, vertex), [workgroup of the chunk][room]
  uint32_t room;        // kKeptEntries, or as many as there are vertices
  uint32_t* n_kept;     // [workgroup of the chunk]
  uint32_t* bound;      // [marked sample]; kNoBound before the layer
  uint32_t* distinct;   // [sample of the chunk]; 0 before the layer
  uint64_t seed;
  uint64_t first_sample;
  uint32_t step;
  uint32_t n_vertices;
  uint32_t wanted;
};

// 32-bit words of one sample's presence map: a bit per vertex, padded to whole tiles.
inline uint32_t bitmap_words_for(uint32_t n_vertices) {
  return ((n_vertices + 31u) / 32u + kBitmapTileWords - 1) / kBitmapTileWords * kBitmapTileWords;
}

// The workgroup's sub-ranges, a lane each (lanes of a wavefront without a transit: length 0), into the tables: those that
// hold entries in lane order, starts[k] = first entry of sub-range k, starts[kept] = all entries, shift[k] = its first edge
// less that (entry e of it is edge e + shift[k]).
// A length with kPieceFlag set stands for a transit whose entries reach the stretch as a ready-made piece: its index
// joins the list `pieces`.  Two barriers; every lane gets the three counts.
constexpr uint32_t kPieceFlag = 0x80000000u;
struct Subranges {
  uint32_t ranges, pieces, entries;
};
__device__ __forceinline__ Subranges list_subranges(uint32_t raw, EdgePos_t first, uint32_t n_transits, uint32_t* starts,
                                                    EdgePos_t* shift, uint32_t* pieces, uint4* s_wave) {
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
    shift[k] = first - (EdgePos_t)starts[k];
  }
  if (is_piece) pieces[mine.pieces + (uint32_t)__popcll(ready & below)] = raw & ~kPieceFlag;
  if (threadIdx.x == 0) starts[all.ranges] = all.entries;
  __syncthreads();
  return all;
}

// The rank-th smallest (from 1) of the values each(f) hands to f, all of them different; each() is called by the whole
// workgroup, every value handed out by one lane, and there are at least `rank`.  Eight bits a turn.
struct PickScratch {
  uint32_t count[256];
  uint32_t digit, rank;
};
template <class Each>
__device__ __forceinline__ uint64_t nth_smallest(Each each, uint32_t rank, PickScratch& scratch) {
  uint64_t prefix = 0, known = 0;
  for (int shift = 56; shift >= 0; shift -= 8) {
    __syncthreads();
    if (threadIdx.x < 256) scratch.count[threadIdx.x] = 0;
    __syncthreads();
    each([&](uint64_t value) {
      if ((value & known) == prefix) atomicAdd(&scratch.count[value >> shift & 255u], 1u);
    });
    __syncthreads();
    if (threadIdx.x < 64) {
      uint32_t own = 0;
      for (uint32_t d = 0; d < 4; ++d) own += scratch.count[threadIdx.x * 4u + d];
      const uint32_t through = wave_inclusive_scan(own);
      uint32_t before = through - own;
      if (before < rank && through >= rank) {  // one lane
        uint32_t d = threadIdx.x * 4u;
        while (before + scratch.count[d] < rank) before += scratch.count[d++];
        scratch.digit = d;
        scratch.rank = rank - before;
      }
    }
    __syncthreads();
    prefix |= (uint64_t)scratch.digit << shift;
    known |= 255ull << shift;
    rank = scratch.rank;
  }
  return prefix;
}
// keys in ascending order, equal ones by vertex
__device__ __forceinline__ uint64_t rank_value(uint2 kept) { return (uint64_t)kept.x << 32 | kept.y; }

// What a workgroup of collective_mark_binned knows of the keys it has kept; in LDS, set before use by begin().
struct Keeper {
  uint32_t counts[kBoundBins];  // of the keys at or below the bound of their time
  uint32_t wave_total[kBinThreads / 64];
  uint32_t bound, fresh, n;     // no key above it is wanted; keys since it was looked for; keys kept
  PickScratch pick;

  __device__ __forceinline__ void begin(uint32_t sample_bound) {  // the caller's next barrier ends it
    for (uint32_t i = threadIdx.x; i < kBoundBins; i += kBinThreads) counts[i] = 0;
    if (threadIdx.x == 0) {
      bound = sample_bound;
      fresh = n = 0;
    }
  }
  // How far from 1 a uniform may be without its key being above the bound for certain, in units of 2^-24, for an importance of
  // 2^32: -log2(u) is at least (1 - u) / ln 2, and 0.69325 for ln 2 leaves 1.5e-4 to what the two sides are rounded by (every
  // operation by 6e-8).  NaN, and then everything may, without a bound.
  __device__ __forceinline__ float reach() const {
    return __uint_as_float(bound & 0x7FFFFFFFu) * (0.69325f * 4294967296.0f * 16777216.0f);
  }
  // A key that was formed: kAbsentKey where it is above the bound, else counted.
  __device__ __forceinline__ uint32_t count(uint32_t key) {
    if (key > bound) return kAbsentKey;
    atomicAdd(&counts[bin_of_key(key)], 1u);
    return key;
  }
  // When every lane has counted what it has of a stretch, `here` keys a wavefront: lowers the bound as far as it goes.
  __device__ __forceinline__ void lower_bound_to(uint32_t wanted, uint32_t here, uint32_t* sample_bound) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0 && here != 0) atomicAdd(&fresh, here);
    __syncthreads();
    if (fresh * 4u < wanted) return;  // not worth another look yet
    static_assert(kBoundBins == kBinThreads, "a lane per count");
    const uint32_t own = counts[threadIdx.x], through = wave_inclusive_scan(own);
    if (lane == 63) wave_total[wave] = through;
    __syncthreads();
    uint32_t before = through - own;
    for (uint32_t w = 0; w < wave; ++w) before += wave_total[w];
    if (before < wanted && before + own >= wanted) {  // at most one lane
      const uint32_t edge = last_key_of_bin(threadIdx.x);
      if (edge < bound) {
        bound = edge;
        atomicMin(sample_bound, edge);
      }
    }
    if (threadIdx.x == 0) fresh = 0;
    __syncthreads();
  }
  // Then: a key of the lane's, if it is within the bound.  kept has room.
  __device__ __forceinline__ void keep(uint32_t key, uint32_t vertex, uint2* kept) {
    const bool stays = key <= bound;
    const uint64_t mask = __ballot(stays);
    if (mask == 0) return;
    const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
    uint32_t base = 0;
    if (stays && below == 0) base = atomicAdd(&n, (uint32_t)__popcll(mask));
    base = __shfl(base, __ffsll((unsigned long long)mask) - 1, kWave);
    if (stays) kept[base + below] = make_uint2(key, vertex);
  }
  // Only the best `wanted` stay (there are more).  For the whole workgroup, between barriers.
  __device__ __forceinline__ void drop_all_but(uint32_t wanted, uint2* kept, uint32_t* sample_bound) {
    const uint32_t had = n;
    const uint64_t last = nth_smallest(
        [&](auto f) {
          for (uint32_t i = threadIdx.x; i < had; i += kBinThreads) f(rank_value(kept[i]));
        },
        wanted, pick);
    if (threadIdx.x == 0) {
      n = 0;
      const uint32_t edge = (uint32_t)(last >> 32);
      if (edge < bound) {
        bound = edge;
        atomicMin(sample_bound, edge);
      }
    }
    for (uint32_t from = 0; from < had; from += kBinThreads) {
      const uint32_t i = from + threadIdx.x;
      const uint2 mine = i < had ? kept[i] : make_uint2(0xFFFFFFFFu, 0xFFFFFFFFu);
      __syncthreads();  // what is written goes where everything has been read
      if (rank_value(mine) <= last) kept[atomicAdd(&n, 1u)] = mine;
    }
    __syncthreads();
  }
};

// The best `wanted` of a sample's keys (those each(f) hands to f, as for nth_smallest), and mostly a few more, in order: an edge
// between counts of their upper bits first; where more are at or below it than there is room for (many equal keys), the
// wanted ones are picked out exactly.  Returns how many; their vertices are in `ids`.  For a workgroup of kBinThreads; begins and ends
// with a barrier.
constexpr uint32_t kBestEntries = 2048;
struct BestRoom {
  uint64_t best[kBestEntries];
  int32_t ids[kBestEntries];
};
struct BestScratch {
  uint32_t counts[kBoundBins];
  uint32_t wave_total[kBinWaves];
  uint64_t last;
  uint32_t through, n;
  PickScratch pick;
};
template <class Each>
__device__ __forceinline__ uint32_t best_in_order(Each each, uint32_t wanted, BestRoom& room, BestScratch& scratch) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  static_assert(kBoundBins == kBinThreads, "a lane per count");
  scratch.counts[threadIdx.x] = 0;
  if (threadIdx.x == 0) scratch.n = 0;
  __syncthreads();
  each([&](uint64_t value) { atomicAdd(&scratch.counts[bin_of_key((uint32_t)(value >> 32))], 1u); });
  __syncthreads();
  const uint32_t own = scratch.counts[threadIdx.x], through_wave = wave_inclusive_scan(own);
  if (lane == 63) scratch.wave_total[wave] = through_wave;
  __syncthreads();
  uint32_t through = through_wave;
  for (uint32_t w = 0; w < wave; ++w) through += scratch.wave_total[w];
  if (threadIdx.x == kBinThreads - 1 && through < wanted) {  // all of them
    scratch.last = ~0ull;
    scratch.through = through;
  }
  if (through - own < wanted && through >= wanted) {  // else one lane
    scratch.last = (uint64_t)last_key_of_bin(threadIdx.x) << 32 | 0xFFFFFFFFu;
    scratch.through = through;
  }
  __syncthreads();
  uint64_t last = scratch.last;
  uint32_t n = scratch.through;
  if (n > kBestEntries) {
    last = nth_smallest(each, wanted, scratch.pick);
    n = wanted;
  }
  each([&](uint64_t value) {
    if (value <= last) room.best[atomicAdd(&scratch.n, 1u)] = value;
  });
  uint32_t padded = 64;
  while (padded < n) padded *= 2u;
  __syncthreads();
  for (uint32_t i = n + threadIdx.x; i < padded; i += kBinThreads) room.best[i] = ~0ull;
  __syncthreads();
  for (uint32_t size = 2; size <= padded; size *= 2u) {
    for (uint32_t stride = size / 2u; stride != 0; stride /= 2u) {
      for (uint32_t i = threadIdx.x; i < padded / 2u; i += kBinThreads) {
        const uint32_t a = (i / stride) * 2u * stride + i % stride, b = a + stride;
        const uint64_t x = room.best[a], y = room.best[b];
        if ((x > y) == ((a & size) == 0)) {
          room.best[a] = y;
          room.best[b] = x;
        }
      }
      __syncthreads();
    }
  }
  for (uint32_t i = threadIdx.x; i < n; i += kBinThreads) room.ids[i] = (int32_t)(uint32_t)room.best[i];
  __syncthreads();
  return n;
}

// A sample without hubs among its transits and with at most this many entries in a workgroup's stretches (a layer whose
// transits are drawn uniformly) adds them all up at once, in an LDS table of twice as many slots.
constexpr uint32_t kSparseGroupEntries = 2048;

// The samples that are not ranked in LDS (ranked_layer).
// Two workgroups of 16 wavefronts share a compute unit only at 8 wavefronts per SIMD, which the kernel's attributes ask
// the compiler for.
// 500 K vertices, 12 M edges, second layer of 1024 samples of 512 (1.5 M pairs and 136 pieces a sample): 2.42 ms.  Writing a
// key for every vertex it took 3.42, and the selection, the collecting and the sorts 1.1 more, where kept_layer_kernel takes
// 0.04; forming only keys that may be within the bound 3.17, the ids of all of a round's entries under way before the first
// is used 2.86, starts as bits 2.59 (2.52 when it was last measured before the next two), those counted by mbcnt and full rounds without
// masks 2.42.  What bounds it now: vector instructions take 63 % of the issue slots (0.94 G of them at four clocks; 1.08 G before those
// two), the rest is the phases of a stretch waiting for each other, and registers that do not fit.
__global__ __launch_bounds__(kBinThreads, 8) __attribute__((amdgpu_num_vgpr(56))) void collective_mark_binned(
    MergedEdges merged, TransitView tv, int32_t invalid, uint32_t n_samples, const uint32_t* __restrict__ n_marked,
    const uint32_t* __restrict__ marked, uint32_t bins_per_sample, DensePieces dense, KeptKeys out) {
  __shared__ __align__(16) uint32_t s_bits[kBinWords];  // where some terms are 0
  __shared__ __align__(16) unsigned long long s_acc[kBinVertices];
  // the sub-ranges that hold entries, in transit order
  __shared__ uint32_t s_start[kMaxLayerTransits + 1];  // first entry of sub-range k among the stretch's entries
  __shared__ EdgePos_t s_shift[kMaxLayerTransits];     // its first edge less that
  __shared__ uint32_t s_piece[kMaxLayerTransits];      // the stretch's dense pieces
  __shared__ uint4 s_wave[kBinWaves];
  __shared__ uint32_t s_starts_here[kBinWaves][2 * kBinAhead];  // where sub-ranges start among a round's entries
  __shared__ Keeper s_keeper;
  // A workgroup takes kBinsPerGroup consecutive stretches of one sample, one after the other: where a transit's sub-range
  // ends in one stretch it begins in the next, and the end is then only a short gallop away instead of a search of the
  // whole adjacency.  The low stretches hold the hubs and take longest: all samples' first groups start first.
  const uint32_t group = blockIdx.x / n_samples;
  const uint32_t at = blockIdx.x - group * n_samples;
  if (at >= *n_marked) return;
  const uint32_t s = marked[at];
  const uint32_t first_bin = group * kBinsPerGroup;
  const int32_t* transits = tv.base + (size_t)s * tv.stride;
  const uint32_t listing = at * (gridDim.x / n_samples) + group;
  uint2* const kept = out.kept + (size_t)listing * out.room;
  uint32_t* const sample_bound = out.bound + at;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = threadIdx.x >> 6;
  s_keeper.begin(__hip_atomic_load(sample_bound, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  uint32_t n_present = 0;  // of the wavefront
  // tv.count <= kBinThreads: lane i keeps transit i and how far the stretches before this one reach into its adjacency
  int32_t my_transit = -1, my_hub = -1, my_cut_row = -1;
  EdgePos_t my_reach = 0;
  // rows that are cut: the end of the coming stretch, fetched one stretch ahead; the others: the destination of edge
  // my_reach, none left: above every vertex
  uint32_t my_next = 0xFFFFFFFFu;
  if (threadIdx.x < tv.count) {
    my_transit = transits[threadIdx.x];
    if (my_transit == invalid) my_transit = -1;
    if (my_transit != -1 && dense.hub_row) my_hub = dense.hub_row[my_transit];
    if (my_transit != -1 && merged.cut_row_of) my_cut_row = merged.cut_row_of[my_transit];
  }
  const bool hubs_among_transits = __syncthreads_or(my_hub >= 0) != 0;
  auto my_cut = [&](uint32_t bin) { return merged.cuts[(size_t)my_cut_row * (bins_per_sample + 1) + bin].from; };
  if (my_transit != -1) {
    if (my_cut_row >= 0) {
      my_reach = my_cut(first_bin);
    } else {
      const EdgePos_t end = merged.row_ptr[my_transit + 1];
      my_reach = first_edge_from(merged.ids, merged.row_ptr[my_transit], end, first_bin * kBinVertices);
      if (my_reach < end) my_next = (uint32_t)merged.ids[my_reach];
    }
  }
  if (!hubs_among_transits) {
    // The stretches of the workgroup as one: the sums are gathered in an LDS table hashed by vertex (in the room of the
    // per-vertex sums).  Stretch by stretch, 16 chains of searches, tables and barriers cost a workgroup 130 us for a few
    // hundred entries.
    const uint32_t group_bins = first_bin + kBinsPerGroup < bins_per_sample ? kBinsPerGroup : bins_per_sample - first_bin;
    const uint32_t v_lo = first_bin * kBinVertices, v_hi = v_lo + group_bins * kBinVertices;
    EdgePos_t stop = my_reach;
    if (my_cut_row >= 0) stop = my_cut(first_bin + group_bins);
    else if (my_next < v_hi) stop = first_edge_from(merged.ids, my_reach, merged.row_ptr[my_transit + 1], v_hi);
    const Subranges all = list_subranges((uint32_t)(stop - my_reach), my_reach, tv.count, s_start, s_shift, s_piece, s_wave);
    const uint32_t ranges = all.ranges, size = all.entries;
    if (size <= kSparseGroupEntries) {
      constexpr uint32_t kSlots = 2u * kSparseGroupEntries;  // a power of two
      unsigned long long* slot_sum = s_acc;
      uint32_t* slot_vertex = (uint32_t*)(s_acc + kSlots);
      for (uint32_t i = threadIdx.x; i < kSlots; i += kBinThreads) {
        slot_vertex[i] = 0xFFFFFFFFu;
        slot_sum[i] = 0;
      }
      __syncthreads();
      for (uint32_t e = threadIdx.x; e < size; e += kBinThreads) {
        uint32_t lo = 0, hi = ranges;  // the sub-range that holds entry e
        while (hi - lo > 1) {
          const uint32_t mid = lo + (hi - lo) / 2;
          if (s_start[mid] <= e) lo = mid; else hi = mid;
        }
        const EdgePos_t src = (EdgePos_t)e + s_shift[lo];
        const uint32_t local = (uint32_t)merged.ids[src] - v_lo;
        uint32_t slot = (local * 2654435761u) >> 20 & (kSlots - 1u);
        for (;;) {  // at most half of the slots are ever taken
          const uint32_t before = atomicCAS(&slot_vertex[slot], 0xFFFFFFFFu, local);
          if (before == 0xFFFFFFFFu || before == local) break;
          slot = (slot + 1u) & (kSlots - 1u);
        }
        atomicAdd(&slot_sum[slot], merged.terms[src]);
      }
      __syncthreads();  // the table is complete
      uint32_t here = 0;
      for (uint32_t i = threadIdx.x; i < kSlots; i += kBinThreads) {
        const uint32_t local = slot_vertex[i];
        n_present += (uint32_t)__popcll(__ballot(local != 0xFFFFFFFFu));
        uint32_t key = kAbsentKey;
        if (local != 0xFFFFFFFFu)
          key = s_keeper.count(ladies_key_bits(slot_sum[i], ladies_pair_index(out.first_sample + s, out.n_vertices, v_lo + local),
                                               out.step, out.seed));
        here += (uint32_t)__popcll(__ballot(key != kAbsentKey));
        slot_sum[i] = key;
      }
      s_keeper.lower_bound_to(out.wanted, here, sample_bound);
      for (uint32_t i = threadIdx.x; i < kSlots; i += kBinThreads)
        s_keeper.keep((uint32_t)slot_sum[i], v_lo + slot_vertex[i], kept);
      if (lane == 0 && n_present != 0) atomicAdd(out.distinct + s, n_present);
      __syncthreads();
      if (threadIdx.x == 0) out.n_kept[listing] = s_keeper.n;
      return;
    }
    // too many entries for that: stretch by stretch
    __syncthreads();
  }
  if (my_cut_row >= 0) my_next = (uint32_t)my_cut(first_bin + 1);
  uint32_t my_piece = my_hub >= 0 ? dense.piece_of[(size_t)my_hub * bins_per_sample + first_bin] : kNoPiece;
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
        my_reach = (EdgePos_t)my_next;
        if (bin + 2 <= bins_per_sample) my_next = (uint32_t)my_cut(bin + 2);
      } else if (my_next < v_hi) {  // nothing is fetched where the next edge already lies beyond the stretch
        const EdgePos_t end = merged.row_ptr[my_transit + 1];
        my_reach = first_edge_from(merged.ids, my_from, end, v_hi);
        my_next = my_reach < end ? (uint32_t)merged.ids[my_reach] : 0xFFFFFFFFu;
      }
      length = (uint32_t)(my_reach - my_from);
      // (fetched one stretch ahead)
      if (my_hub >= 0) {
        if (length != 0 && my_piece != kNoPiece) length = kPieceFlag | my_piece;  // these entries reach the stretch ready-made
        if (bin + 1 < bins_per_sample) my_piece = dense.piece_of[(size_t)my_hub * bins_per_sample + bin + 1];
      }
    }
    const Subranges all = list_subranges(length, my_from, tv.count, s_start, s_shift, s_piece, s_wave);
    if (s_keeper.n > kKeptEntries - kBinVertices) s_keeper.drop_all_but(out.wanted, kept, sample_bound);
    const uint32_t ranges = all.ranges, size = all.entries;
    // Every wavefront walks a contiguous part of the entries, 64 * kBinAhead per round.  Which sub-range an entry is in: the
    // starts that fall into a round, at most 63 (a round ends early for more), become bits, each at the entry before its own, and the
    // bits below an entry are counted: two instructions, which also add what came before (by masks of the bits up to a lane's: four, and two
    // registers more; a pass over 500 K vertices 3.26 ms instead of 3.18).  (A lane that stepped from sub-range to sub-range for itself took five turns an entry for the slowest of 64, each
    // a trip to LDS: 2.80 ms instead of 2.59 where collective_mark_binned gives its figures.)
    constexpr uint32_t kRound = 64u * kBinAhead;
    const uint32_t uniform_wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave);
    const uint32_t part = (size + kBinWaves * kRound - 1) / (kBinWaves * kRound) * kRound;
    uint32_t e0 = uniform_wave * part;
    const uint32_t part_end = e0 + part < size ? e0 + part : size;
    uint32_t before = 0;  // the sub-range that holds e0, or the one before it where one starts there
    if (e0 < part_end) {
      uint32_t hi = ranges;
      while (hi - before > 1) {
        const uint32_t mid = before + (hi - before) / 2;
        if (s_start[mid] <= e0) before = mid; else hi = mid;
      }
      before = (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
    }
    while (e0 < part_end) {
      const uint32_t start = before + 1u + lane < ranges ? s_start[before + 1u + lane] : 0xFFFFFFFFu;
      uint32_t end = e0 + kRound < part_end ? e0 + kRound : part_end;
      const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)start, 63);
      end = last < end ? last : end;
      const bool falls_here = start < end;
      if (lane < kRound / 32u) s_starts_here[wave][lane] = 0;
      __builtin_amdgcn_wave_barrier();
      if (falls_here && start != e0) atomicOr(&s_starts_here[wave][(start - e0 - 1u) >> 5], 1u << ((start - e0 - 1u) & 31u));
      __builtin_amdgcn_wave_barrier();
      // (nothing may be worked out from an id before the last is asked for: the compiler waits for it where that is done)
      // all: every lane has an entry every time, as in most rounds, so that none is masked out (500 K vertices: 3.18 -> 3.12 ms a pass)
      auto add_up = [&](auto all) {
        constexpr bool kAll = decltype(all)::value;
        uint32_t ids[kBinAhead];
        unsigned long long terms[kBinAhead];
        uint32_t of = before + ((uint32_t)__builtin_amdgcn_readfirstlane((int)start) == e0 ? 1u : 0u);  // only the first can
#pragma unroll
        for (uint32_t a = 0; a < kBinAhead; ++a) {
          const uint32_t low = s_starts_here[wave][2u * a], high = s_starts_here[wave][2u * a + 1u];
          const uint32_t e = e0 + a * 64u + lane;
          const uint32_t mine = __builtin_amdgcn_mbcnt_hi(high, __builtin_amdgcn_mbcnt_lo(low, of));
          of += (uint32_t)__popc(low) + (uint32_t)__popc(high);
          if (!kAll) {
            ids[a] = 0;
            terms[a] = 0;
            if (e >= end) continue;
          }
          const uint32_t src = e + (uint32_t)s_shift[mine];  // an edge: not negative
          ids[a] = (uint32_t)merged.ids[src];
          terms[a] = merged.terms[src];
        }
#pragma unroll
        for (uint32_t a = 0; a < kBinAhead; ++a) {
          if (!kAll && e0 + a * 64u + lane >= end) continue;
          const uint32_t local = ids[a] - v_lo;
          atomicAdd(&s_acc[local], terms[a]);
          if (merged.zero_terms) atomicOr(&s_bits[local >> 5], 1u << (local & 31u));
        }
      };
      if (end - e0 == kRound) add_up(std::true_type());
      else add_up(std::false_type());
      before += (uint32_t)__popcll(__ballot(falls_here));
      e0 = end;
    }
    __syncthreads();
    // The keys of the stretch's vertices.  A lane takes four consecutive vertices: 16-byte accesses to LDS and to the pieces,
    // and one Philox block where it forms keys.  Most vertices' uniforms are too far from 1 for any importance like theirs:
    // the two divisions and the logarithm are for the few others.
    const uint32_t n_pieces = all.pieces;
    const float reach = s_keeper.reach();
    uint32_t here = 0, with_keys = 0;  // keys of the wavefront, and in which turns there were any
    for (uint32_t q = threadIdx.x; q < kBinVertices / 4u; q += kBinThreads) {  // whole wavefronts
      const uint32_t i = 4u * q;
      const ulonglong2 low = ((const ulonglong2*)s_acc)[2u * q], high = ((const ulonglong2*)s_acc)[2u * q + 1u];
      unsigned long long sum[4] = {low.x, low.y, high.x, high.y};  // 0 where nothing was added
      const uint32_t bits = merged.zero_terms ? (s_bits[i >> 5] >> (i & 31u)) & 15u : 0u;
      // two pieces under way before the first is used
      const ulonglong2* const pieces = (const ulonglong2*)(dense.sums + i);
      uint32_t p = 0;
      for (; p + 1 < n_pieces; p += 2) {
        const ulonglong2* one = pieces + (size_t)s_piece[p] * (kBinVertices / 2u);
        const ulonglong2* two = pieces + (size_t)s_piece[p + 1] * (kBinVertices / 2u);
        const ulonglong2 a = one[0], b = one[1], c = two[0], d = two[1];
        sum[0] += a.x + c.x;
        sum[1] += a.y + c.y;
        sum[2] += b.x + d.x;
        sum[3] += b.y + d.y;
      }
      if (p < n_pieces) {
        const ulonglong2* one = pieces + (size_t)s_piece[p] * (kBinVertices / 2u);
        const ulonglong2 a = one[0], b = one[1];
        sum[0] += a.x;
        sum[1] += a.y;
        sum[2] += b.x;
        sum[3] += b.y;
      }
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) n_present += (uint32_t)__popcll(__ballot(sum[k] != 0 || (bits >> k & 1u) != 0));
      const PhiloxBlock blk = ladies_block(ladies_pair_index(out.first_sample + s, out.n_vertices, v_lo + i), out.step, out.seed);
      bool may[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) may[k] = key_may_be_within(reach, sum[k], blk.w[k]);
      uint32_t key[4] = {kAbsentKey, kAbsentKey, kAbsentKey, kAbsentKey};
      if (may[0] || may[1] || may[2] || may[3]) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
          if (may[k] && (sum[k] != 0 || (bits >> k & 1u) != 0)) key[k] = s_keeper.count(ladies_key_from_word(sum[k], blk.w[k]));
      }
      uint32_t keys_here = 0;
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) keys_here += (uint32_t)__popcll(__ballot(key[k] != kAbsentKey));
      here += keys_here;
      if (keys_here != 0) ((uint4*)s_acc)[2u * q] = make_uint4(key[0], key[1], key[2], key[3]);  // in the sums' room
      with_keys |= (keys_here != 0 ? 1u : 0u) << q / kBinThreads;
    }
    s_keeper.lower_bound_to(out.wanted, here, sample_bound);
    if (with_keys != 0)
      for (uint32_t q = threadIdx.x; q < kBinVertices / 4u; q += kBinThreads) {
        if ((with_keys >> q / kBinThreads & 1u) == 0) continue;
        const uint4 key = ((const uint4*)s_acc)[2u * q];
        const uint32_t v = v_lo + 4u * q;
        s_keeper.keep(key.x, v, kept);
        s_keeper.keep(key.y, v + 1u, kept);
        s_keeper.keep(key.z, v + 2u, kept);
        s_keeper.keep(key.w, v + 3u, kept);
      }
    __syncthreads();  // the next stretch clears what this one has just read
  }
  if (lane == 0 && n_present != 0) atomicAdd(out.distinct + s, n_present);
  __syncthreads();
  if (threadIdx.x == 0) out.n_kept[listing] = s_keeper.n;
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
                                                                   uint32_t* __restrict__ too_long,
                                                                   uint32_t* __restrict__ distinct = nullptr,
                                                                   uint32_t* __restrict__ bound = nullptr) {
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
  if (lane == 0 && s < n_samples && pairs > kRankedEntries) {
    marked[s_base + at] = s;
    if (bound) bound[s_base + at] = kNoBound;
    if (distinct) distinct[s] = 0;
  }
}

// A workgroup per sample: fetches the pairs, adds their terms up in an LDS table hashed by vertex, forms the keys of the vertices
// there and puts the best of them in order (equal keys by vertex).  Marked stretch by stretch, a layer of 1024 such samples
// over 500 K vertices wrote and read 4 GB of keys, most of them absent.
// Bound by round trips to LDS, of which one workgroup fills a compute unit.  806 samples of the first layer over 500 K vertices
// 0.140 ms, 1024 over 114 K 0.084; by two sorts in LDS, of the pairs by vertex and of the vertices by key, and with the terms fetched
// in the first one's order, 0.317 and 0.190.
template <class Draw>
__device__ __forceinline__ void ranked_layer(const MergedEdges& merged, uint32_t n_vertices, const int32_t* transits,
                                             uint32_t n_transits, int32_t invalid, uint32_t size, uint64_t sample,
                                             uint32_t step, uint64_t seed, uint32_t wanted, uint32_t* __restrict__ distinct_out,
                                             Draw draw) {
  constexpr uint32_t kEach = kRankedEntries / kRankedThreads;
  constexpr uint32_t kSlots = kRankedEntries + kRankedEntries / 2;  // at most two thirds of them are ever taken
  constexpr uint32_t kNobody = 0xFFFFFFFFu;
  __shared__ __align__(16) unsigned long long s_sum[kSlots];  // then key and vertex, all ones where there is none
  __shared__ union { uint32_t vertex[kSlots]; BestRoom best; } s_table;
  __shared__ uint32_t s_start[kMaxLayerTransits];
  __shared__ EdgePos_t s_edge[kMaxLayerTransits];
  __shared__ BestScratch s_scratch;
  __shared__ uint32_t s_distinct;
  static_assert(kMaxLayerTransits <= kRankedThreads && kRankedThreads == kBinThreads, "a lane a transit");
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t slots = (size + size / 2u + 63u) & ~63u;  // of them in use: fewer to clear and to look through
  static_assert(kSlots % 64 == 0, "as many as there are");
  for (uint32_t i = threadIdx.x; i < slots; i += kRankedThreads) {
    s_sum[i] = 0;
    s_table.vertex[i] = kNobody;
  }
  if (threadIdx.x == 0) s_distinct = 0;
  {
    const int32_t t = threadIdx.x < n_transits ? transits[threadIdx.x] : -1;
    EdgePos_t begin = 0;
    uint32_t degree = 0;
    if (t != invalid && t != -1) {
      begin = merged.row_ptr[t];
      degree = (uint32_t)(merged.row_ptr[t + 1] - begin);
    }
    const uint32_t through = wave_inclusive_scan(degree);
    if (lane == 63) s_scratch.wave_total[wave] = through;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += s_scratch.wave_total[w];
    if (threadIdx.x < n_transits) {
      s_start[threadIdx.x] = before + through - degree;
      s_edge[threadIdx.x] = begin;
    }
    __syncthreads();
  }
  uint32_t id[kEach];
  unsigned long long term[kEach];
#pragma unroll
  for (uint32_t k = 0; k < kEach; ++k) {
    const uint32_t e = k * kRankedThreads + threadIdx.x;
    id[k] = kNobody;
    term[k] = 0;
    if (e >= size) continue;
    uint32_t lo = 0, hi = n_transits;  // the last transit that starts at e or before (empty ones start where the next does)
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (s_start[mid] <= e) lo = mid; else hi = mid;
    }
    const EdgePos_t at = s_edge[lo] + (EdgePos_t)(e - s_start[lo]);
    id[k] = (uint32_t)merged.ids[at];
    term[k] = merged.terms[at];
  }
#pragma unroll
  for (uint32_t k = 0; k < kEach; ++k) {
    if (id[k] == kNobody) continue;
    uint32_t slot = __umulhi(id[k] * 2654435761u, slots);
    for (;;) {
      const uint32_t before = atomicCAS(&s_table.vertex[slot], kNobody, id[k]);
      if (before == kNobody || before == id[k]) break;
      slot = slot + 1u == slots ? 0u : slot + 1u;
    }
    atomicAdd(&s_sum[slot], term[k]);
  }
  __syncthreads();
  uint32_t distinct = 0;  // of the wavefront
  for (uint32_t i = threadIdx.x; i < slots; i += kRankedThreads) {  // whole wavefronts
    const uint32_t v = s_table.vertex[i];
    distinct += (uint32_t)__popcll(__ballot(v != kNobody));
    unsigned long long value = ~0ull;
    if (v != kNobody) value = rank_value(make_uint2(ladies_key_bits(s_sum[i], ladies_pair_index(sample, n_vertices, v), step, seed), v));
    s_sum[i] = value;
  }
  if (lane == 0 && distinct != 0) atomicAdd(&s_distinct, distinct);
  // (the barrier it begins with: nobody needs s_table.vertex any more)
  const uint32_t n = best_in_order(
      [&](auto f) {
        for (uint32_t i = threadIdx.x; i < slots; i += kRankedThreads)
          if (s_sum[i] != ~0ull) f(s_sum[i]);
      },
      wanted, s_table.best, s_scratch);
  if (threadIdx.x == 0) *distinct_out = s_distinct;
  draw((const CSR::Edge*)s_table.best.ids, n);
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
};

// The draws of kConcatenated.
template <class SampleType, class App>
__global__ __launch_bounds__(256) void layer_execute_kernel(LayerParams P) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint64_t)P.chunk_samples * P.step_size) return;
  const uint32_t ls = (uint32_t)(i / P.step_size);  // sample inside the chunk
  const uint32_t nbr = (uint32_t)(i - (uint64_t)ls * P.step_size);
  const uint32_t s = P.sample_begin + ls;
  CSRPartition csr = P.csr;
  const int32_t* transits = P.transits.base + (size_t)ls * P.transits.stride;
  SampleType local_state;
  SampleType* state = std::is_empty<SampleType>::value ? &local_state : (SampleType*)P.samples + s;
  curandState rng;
  rng.reset(P.seed, (P.first_sample + s) * P.step_size + nbr, (uint32_t)P.step);
  const VertexID sample_id = (VertexID)(P.first_sample + s);
  VertexID neighbor = P.invalid;
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
               size, P.first_sample + P.sample_begin + ls, (uint32_t)P.step, P.seed, P.step_size, distinct + ls,
               [&](const CSR::Edge* ranked, uint32_t n) {
                 const uint32_t n_first = n < P.step_size ? n : P.step_size;
                 for (uint32_t nbr = threadIdx.x; nbr < P.step_size; nbr += kRankedThreads)
                   draw_from<SampleType, App>(P, ls, nbr, ranked, n_first);
               });
}

// A workgroup per marked sample: the best of what the workgroups of collective_mark_binned have kept of it, in order, and the
// draws.  1024 samples of 512, five workgroups' keys each (500 K vertices): 0.044 ms; 27 workgroups' (3.07 M vertices): 0.08.
template <class SampleType, class App>
__global__ __launch_bounds__(kBinThreads) void kept_layer_kernel(LayerParams P, const uint32_t* __restrict__ n_marked,
                                                                 const uint32_t* __restrict__ marked, uint32_t groups,
                                                                 KeptKeys in) {
  __shared__ BestRoom s_best;
  __shared__ BestScratch s_scratch;
  const uint32_t at = blockIdx.x;
  if (at >= *n_marked) return;
  const uint32_t bound = in.bound[at];
  auto each = [&](auto f) {
    for (uint32_t g = 0; g < groups; ++g) {
      const uint32_t listing = at * groups + g, n = in.n_kept[listing];
      const uint2* kept = in.kept + (size_t)listing * in.room;
      for (uint32_t i = threadIdx.x; i < n; i += kBinThreads) {
        const uint2 mine = kept[i];
        if (mine.x <= bound) f(rank_value(mine));
      }
    }
  };
  const uint32_t n = best_in_order(each, in.wanted, s_best, s_scratch);
  const CSR::Edge* ranked = (const CSR::Edge*)s_best.ids;
  // (how many more there are here depends on what the workgroups knew of each other's bounds)
  const uint32_t n_first = n < P.step_size ? n : P.step_size;
  for (uint32_t nbr = threadIdx.x; nbr < P.step_size; nbr += kBinThreads) draw_from<SampleType, App>(P, marked[at], nbr, ranked, n_first);
}

// The draws of the marked samples, a lane each, the workgroups of the grid in turn.
template <class SampleType, class App>
__global__ __launch_bounds__(256) void marked_layer_kernel(LayerParams P, MarkedSamples marked,
                                                           const uint32_t* __restrict__ distinct,
                                                           const uint32_t* __restrict__ bitmap, uint32_t words_per_sample,
                                                           const uint64_t* __restrict__ half_before,
                                                           const uint64_t* __restrict__ group_through, uint32_t halves) {
  const uint64_t draws = (uint64_t)*marked.count * P.step_size;
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < draws; i += gridDim.x * 256ull) {
    const uint32_t at = (uint32_t)(i / P.step_size), nbr = (uint32_t)(i - (uint64_t)at * P.step_size);
    const uint32_t ls = marked.sample[at];
    MarkedByDegreeSquared mine{bitmap + (size_t)at * words_per_sample, half_before + (size_t)at * (halves + 1),
                               group_through + (size_t)at * halves * kGroupsPerHalf, P.csr.row_ptr, halves};
    draw_from<SampleType, App>(P, ls, nbr, mine, distinct[ls]);
  }
}

// Entries of concatenated neighbourhood one chunk of samples may hold (about 70 bytes of
// device memory per entry across all work arrays).
constexpr uint64_t kLayerChunkEntries = 96ull << 20;
// Importance forms: nothing is stored per entry, so a chunk is bounded by the memory of its presence maps or of the keys
// that are kept.
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
    bitmap_words_ = bitmap_words_for((uint32_t)invalid_);
    // bytes a sample of a chunk holds: its bitmap (FastGCN form), or what its workgroups keep (LADIES form)
    uint64_t bytes_per_sample = (uint64_t)bitmap_words_ * sizeof(uint32_t);
    if (apps::neighborhood_form_of<App>::value == apps::kRankedByLadiesImportance) {
      bytes_per_sample = (uint64_t)ladies_groups() * kept_room() * sizeof(uint2);
    }
    const uint64_t fit = kBitmapBudgetBytes / bytes_per_sample;
    bitmap_chunk_samples_ = fit < 1 ? 1u : fit > (uint64_t)n_samples_ ? (uint32_t)n_samples_ : (uint32_t)fit;

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
      ND_HIP_TRY(hipHostMalloc((void**)&h_too_long_, sizeof(uint32_t), hipHostMallocDefault));
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
    drop_rows_ahead();  // nobody asked for them
    // a caller who took the last pass's rows, array and all, is expected to take this one's as well
    const bool rows_expected = rows_fetched_ && hFinalSamples.taken() && !profiling;
    rows_fetched_ = false;
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
    if (rows_expected) send_rows();
    ND_HIP_TRY(hipEventSynchronize(ev_end_));
    if (rows_ahead_) result_stream->words_are_there();
    ND_HIP_TRY(hipEventElapsedTime(&times.end_to_end, ev_begin_, ev_end_));
    if (h_too_long_ && *h_too_long_) {
      drop_rows_ahead();
      last_error = kTooLong;
      return -2;
    }
    counted_ = apps::neighborhood_form_of<App>::value == apps::kConcatenated;
    return 0;
  }

  int fetch_final_samples() override {
    if (!allocated_) { last_error = "no device data"; return -1; }
    rows_fetched_ = true;
    settle_rows_ahead();
    if (rows_ahead_) {
      rows_ahead_ = false;
      return 0;
    }
    hFinalSamples.resize((size_t)n_samples_ * (size_t)final_sample_size());
    return fetch_to_host(hFinalSamples.data(), d_final_, sizeof(VertexID_t) * hFinalSamples.size(), (uint32_t)max_bits(),
                         invalid_, stream_);
  }

  int fetch_sample_states(void* dst, size_t bytes) override {
    if (!allocated_ || std::is_empty<SampleType>::value) { last_error = "no sample state"; return -1; }
    if (bytes != sample_state_bytes()) { last_error = "sample state size mismatch"; return -1; }
    settle_rows_ahead();
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
    std::vector<unsigned long long> sums, piece(kBinVertices);
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
          std::fill(piece.begin(), piece.end(), 0ull);
          for (const int32_t* c = first; c < stop; ++c) {
            // the term of this edge, in the arithmetic of merge_edges
            const float p = graph->weight[(size_t)graph->row_ptr[v] + (size_t)(c - row)] * inverse_row_sums[v];
            piece[(uint32_t)*c - b * kBinVertices] += importance_term_fixed(p * p);
          }
          if (std::all_of(first, stop, [&](int32_t c) { return piece[(uint32_t)c - b * kBinVertices] != 0; })) {
            if (hub_row[v] < 0) {
              hub_row[v] = (int32_t)n_hubs++;
              piece_of.resize(n_hubs * stretches, kNoPiece);
            }
            piece_of[(size_t)hub_row[v] * stretches + b] = (uint32_t)n_pieces++;
            sums.insert(sums.end(), piece.begin(), piece.end());
          }
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
    const uint32_t n = P.chunk_samples, parts = union_.parts, halves = parts * kHalvesOfPart;
    if (n > bitmap_samples_) {
      release(d_bitmap_); release(d_group_through_); release(d_half_total_); release(d_half_before_);
      ND_HIP_TRY(hipMalloc(&d_bitmap_, sizeof(uint32_t) * (size_t)n * bitmap_words_));
      ND_HIP_TRY(hipMalloc(&d_group_through_, sizeof(uint64_t) * (size_t)n * parts * kGroupsPerPart));
      ND_HIP_TRY(hipMalloc(&d_half_total_, sizeof(uint64_t) * (size_t)n * halves));
      ND_HIP_TRY(hipMalloc(&d_half_before_, sizeof(uint64_t) * (size_t)n * (halves + 1)));
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
    union_sums<<<dim3(halves * kSumSlices), dim3(kSumThreads), 0, stream_>>>(
        union_.squares, union_.square_rows, halves, marked_, bitmap_words_, d_bitmap_, d_group_through_, d_half_total_, distinct);
    tock();
    sample_half_sums<<<dim3(n), dim3(64), 0, stream_>>>(d_half_total_, halves, marked_.count, d_half_before_);
    marked_layer_kernel<SampleType, App><<<dim3(kDrawBlocks), dim3(256), 0, stream_>>>(
        P, marked_, distinct, d_bitmap_, bitmap_words_, d_half_before_, d_group_through_, halves);
    ND_HIP_TRY(hipGetLastError());
    return 0;
  }

  // LADIES form: small neighbourhoods are ranked by a workgroup each, in LDS.  Of the others every workgroup of the marking
  // keeps the keys that can be among the sample's first, and one more workgroup a sample puts those together.
  int run_ranked(LayerParams P, int step) {
    const uint32_t n = P.chunk_samples;
    const uint32_t bins = ladies_bins(), groups = ladies_groups();
    if ((uint64_t)n * groups >= (1ull << 31)) { last_error = "a chunk needs 2^31 or more workgroups"; return -1; }
    if (n > bitmap_samples_) {
      release(d_kept_); release(d_n_kept_); release(d_bound_);
      ND_HIP_TRY(hipMalloc(&d_kept_, sizeof(uint2) * kept_room() * (size_t)n * groups));
      ND_HIP_TRY(hipMalloc(&d_n_kept_, sizeof(uint32_t) * (size_t)n * groups));
      ND_HIP_TRY(hipMalloc(&d_bound_, sizeof(uint32_t) * (size_t)n));
      bitmap_samples_ = n;
    }
    const size_t S = (size_t)n_samples_;
    uint32_t* sizes = d_layer_counts_ + S * step + P.sample_begin;
    uint32_t* distinct = sizes + S * App().steps();
    ND_HIP_TRY(hipMemsetAsync(marked_.count, 0, sizeof(uint32_t), stream_));
    sort_out_ranked<<<dim3((n + 15) / 16), dim3(kSortOutThreads), 0, stream_>>>(
        P.csr, merged_, P.transits, n, invalid_, sizes, d_merged_sizes_, marked_.count, marked_.sample, h_too_long_,
        distinct, d_bound_);
    tick();
    ranked_layer_kernel<SampleType, App><<<dim3(n), dim3(kRankedThreads), 0, stream_>>>(P, merged_, d_merged_sizes_, distinct);
    KeptKeys kept;
    kept.kept = d_kept_;
    kept.room = kept_room();
    kept.n_kept = d_n_kept_;
    kept.bound = d_bound_;
    kept.distinct = distinct;
    kept.seed = seed_;
    kept.first_sample = P.first_sample + P.sample_begin;
    kept.step = (uint32_t)step;
    kept.n_vertices = (uint32_t)invalid_;
    kept.wanted = P.step_size;
    collective_mark_binned<<<dim3(n * groups), dim3(kBinThreads), 0, stream_>>>(
        merged_, P.transits, invalid_, n, marked_.count, marked_.sample, bins, dense_, kept);
    tock();
    kept_layer_kernel<SampleType, App><<<dim3(n), dim3(kBinThreads), 0, stream_>>>(P, marked_.count, marked_.sample, groups, kept);
    ND_HIP_TRY(hipGetLastError());
    return 0;
  }
  uint32_t ladies_bins() const { return (bitmap_words_ + kBinWords - 1) / kBinWords; }
  uint32_t ladies_groups() const { return (ladies_bins() + kBinsPerGroup - 1) / kBinsPerGroup; }
  uint32_t kept_room() const { return std::max(1u, std::min(kKeptEntries, (uint32_t)invalid_)); }  // no vertex is kept twice

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

  void release_neighborhood_buffers() {
    release(d_nbr_cols_); release(d_nbr_weights_);
    release(d_bitmap_); release(d_kept_); release(d_n_kept_); release(d_bound_);
    release(d_group_through_); release(d_half_total_); release(d_half_before_);
    capacity_ = 0;
    bitmap_samples_ = 0;
  }

  // The rows of the pass that is enqueued, directly behind it; fetched when they are asked for if they cannot be sent now.
  void send_rows() {
    try {
      hFinalSamples.resize((size_t)n_samples_ * (size_t)final_sample_size());
      rows_ahead_ = result_stream->begin(d_final_, hFinalSamples.size(), (uint32_t)max_bits(), invalid_, hFinalSamples.data(),
                                         stream_, {}, /*follows=*/true) == hipSuccess;
    } catch (const std::bad_alloc&) {
      rows_ahead_ = false;
    }
    if (!rows_ahead_) (void)hipGetLastError();
  }
  // The result stream carries one transfer at a time: rows on their way are waited for where it is known whose they are.
  void settle_rows_ahead() {
    if (rows_ahead_ && result_stream->finish() != hipSuccess) rows_ahead_ = false;
  }
  void drop_rows_ahead() {
    if (rows_ahead_) result_stream->abandon();
    rows_ahead_ = false;
  }

  void free_run_buffers() {
    drop_rows_ahead();
    rows_fetched_ = false;
    release(d_initial_); release(d_samples_); release(d_samples_init_); release(d_final_);
    release(d_sizes_); release(d_offsets_); release(d_row_offsets_); release(d_small_scratch_);
    release(d_item_count_); release(d_item_start_);
    release(d_layer_counts_);
    if (h_too_long_) (void)hipHostFree(h_too_long_);
    h_too_long_ = nullptr;
    release(marked_.count); release(marked_.sample); release(marked_.transits); release(marked_.transit_count);
    release(d_merged_sizes_);
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
  bool rows_fetched_ = false;  // since the last pass
  bool rows_ahead_ = false;    // rows are on their way to hFinalSamples
  bool allocated_ = false;
  size_t capacity_ = 0;
  uint32_t bitmap_words_ = 0;          // 32-bit words of one sample's presence map (a multiple of kBitmapTileWords)
  uint32_t bitmap_chunk_samples_ = 0;  // samples whose bitmaps fit the budget
  uint64_t bitmap_chunk_entries_ = 0;
  uint32_t bitmap_samples_ = 0;        // samples the allocated bitmaps hold
  uint32_t* d_bitmap_ = nullptr;
  // LADIES form: what the workgroups of the marking keep (KeptKeys)
  uint2* d_kept_ = nullptr;
  uint32_t *d_n_kept_ = nullptr, *d_bound_ = nullptr;
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
  uint32_t* d_merged_sizes_ = nullptr;    // pairs of a sample's neighbourhood
  EdgePos_t* d_merged_rows_ = nullptr;    // the graph without parallel edges
  VertexID* d_merged_ids_ = nullptr;
  unsigned long long* d_merged_terms_ = nullptr;
  int32_t* d_cut_row_of_ = nullptr;
  HubCut* d_cuts_ = nullptr;
  MergedEdges merged_{};
  int32_t* d_nbr_cols_ = nullptr;
  float* d_nbr_weights_ = nullptr;
  // FastGCN form: degree^2 of the marked vertices, by group inside half a part, by half, by sample
  uint64_t *d_group_through_ = nullptr, *d_half_total_ = nullptr, *d_half_before_ = nullptr;
  UnionTables union_;                  // of the graph
  MarkedSamples marked_{};
  uint32_t* d_layer_counts_ = nullptr;  // entries of every layer and sample's neighbourhood, then its distinct vertices
  uint32_t* h_too_long_ = nullptr;      // whether a neighbourhood was too long
};

}  // namespace nd
