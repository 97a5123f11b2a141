// Results on their way to the host, and the host memory they land in.
//
// A pass leaves gigabytes of 4-byte vertex ids in device memory and the caller wants them in
// host memory: of 4.2 M node2vec walks (1.68 GB, 34 ms to sample) the copy took 29 ms at the bus's
// 57 GB/s, and another 118 ms went into handing the caller an array of their own.  Three things
// are done about it here:
//
//  * What crosses the bus is packed (pack_results): ids take as many bits as the largest one, the
//    number of vertices, needs (23 instead of 32 for R-MAT 22), and groups of eight consecutive
//    ids that are all INVALID - walks that have ended, samples without neighbours - are left out.
//    The kernel writes its output straight into page-locked memory (54.7 GB/s, as fast as the copy
//    engine's 57, without a launch and a copy per piece), and host threads unpack a piece
//    while the next one crosses.  The host side is not what bounds it: eight threads write 170 GB/s of
//    unpacked ids on the 16-core share of a GPU's host, four 147.
//  * The arrays results land in come from a small pool per sampler and keep their pages: a first
//    touch costs 0.1-0.4 s per GB, more than the sampling.
//  * Such an array can be given to the caller (HostLease) instead of being copied for them; it goes
//    back to the pool when the caller lets go of it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <functional>
#include <list>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

namespace nd {

// ---- host threads ------------------------------------------------------------------------

// A few threads of the process that help whoever calls run(); they sleep otherwise.  They live
// until the process ends (no destructor: a thread must not outlast what it waits on).
class HostWorkers {
 public:
  // More do not help: unpacking is bound by memory from four threads on.
  static constexpr unsigned kMost = 7;

  static HostWorkers& get() {
    static HostWorkers* workers = new HostWorkers;
    return *workers;
  }

  // Runs body() on this thread and, as far as threads are free, on up to `helpers` others.  Returns
  // when every body() that started has returned.  body() has to be able to do all the work
  // alone, and must not throw.
  void run(unsigned helpers, const std::function<void()>& body, const std::function<void()>& caller_body) {
    helpers = std::min(helpers, limit());
    Job job{&body, helpers, 0};
    if (helpers > 0) {
      std::lock_guard<std::mutex> lock(mutex_);
      grow(helpers);
      jobs_.push_back(&job);
    }
    if (helpers > 0) wake_.notify_all();
    caller_body();
    if (helpers == 0) return;
    std::unique_lock<std::mutex> lock(mutex_);
    jobs_.remove(&job);  // nobody starts on it any more
    ended_.wait(lock, [&] { return job.running == 0; });
  }
  void run(unsigned helpers, const std::function<void()>& body) { run(helpers, body, body); }

 private:
  struct Job {
    const std::function<void()>* body;
    unsigned wanted, running;
  };

  HostWorkers() = default;

  static unsigned limit() {
    const unsigned hw = std::thread::hardware_concurrency();
    return hw > 1 ? std::min(hw / 2, kMost) : 0;
  }

  void grow(unsigned helpers) {
    while (threads_ < helpers) {
      try {
        std::thread([this] { work(); }).detach();
      } catch (...) {
        return;  // fewer threads, or none: the caller does the work
      }
      threads_++;
    }
  }

  void work() {
    std::unique_lock<std::mutex> lock(mutex_);
    for (;;) {
      Job* job = nullptr;
      for (Job* j : jobs_)
        if (j->wanted > 0) { job = j; break; }
      if (!job) {
        wake_.wait(lock);
        continue;
      }
      job->wanted--;
      job->running++;
      lock.unlock();
      (*job->body)();
      lock.lock();
      if (--job->running == 0) ended_.notify_all();
    }
  }

  std::mutex mutex_;
  std::condition_variable wake_, ended_;
  std::list<Job*> jobs_;
  unsigned threads_ = 0;
};

// ---- host memory ---------------------------------------------------------------------------

struct HostBlock {
  enum Kind { kNone, kPinned, kPages, kHeap };
  void* p = nullptr;
  size_t bytes = 0;
  Kind kind = kNone;
};

// Results up to this size are copied by the copy engine straight into page-locked memory; above it
// they are packed and streamed (ResultStream).
constexpr size_t kDirectResultBytes = 4u << 20;

// The host arrays of one sampler.  At most kKeep of them wait for their next use; all of those are
// freed when the sampler goes, the others when their holders let go of them.
class HostPool {
 public:
  HostPool() = default;
  HostPool(const HostPool&) = delete;
  HostPool& operator=(const HostPool&) = delete;
  ~HostPool() { close(); }

  HostBlock take(size_t bytes) {
    bool pinned = bytes <= kDirectResultBytes;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (size_t i = 0; i < free_.size(); ++i)
        if (free_[i].bytes >= bytes && free_[i].bytes / 2 <= bytes) {
          const HostBlock b = free_[i];
          free_.erase(free_.begin() + (ptrdiff_t)i);
          return b;
        }
      // page-locked memory is for what is in use, not for arrays a caller collects
      pinned = pinned && pinned_ < kMostPinned;
      if (pinned) pinned_++;
    }
    HostBlock b;
    if (pinned) {
      if (hipHostMalloc(&b.p, bytes, hipHostMallocDefault) == hipSuccess && b.p) {
        b.bytes = bytes;
        b.kind = HostBlock::kPinned;
        return b;
      }
      (void)hipGetLastError();  // the refusal is not an error of a later call
      b.p = nullptr;
      std::lock_guard<std::mutex> lock(mutex_);
      pinned_--;
    }
    if (bytes > kDirectResultBytes) {
      // 2 MB pages: a two-thousandth of the faults
      const size_t whole = (bytes + kPage - 1) / kPage * kPage;
      char* raw = (char*)mmap(nullptr, whole + kPage, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
      if (raw != (char*)MAP_FAILED) {
        char* at = (char*)(((uintptr_t)raw + kPage - 1) / kPage * kPage);
        if (at != raw) munmap(raw, (size_t)(at - raw));
        munmap(at + whole, kPage - (size_t)(at - raw));
        (void)madvise(at, whole, MADV_HUGEPAGE);
        b.p = at;
        b.bytes = whole;
        b.kind = HostBlock::kPages;
        return b;
      }
    }
    b.p = malloc(bytes);
    if (!b.p) throw std::bad_alloc();
    b.bytes = bytes;
    b.kind = HostBlock::kHeap;
    return b;
  }

  void give(HostBlock b) {
    HostBlock drop = b;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (open_ && b.kind != HostBlock::kHeap) {
        free_.push_back(b);
        drop = HostBlock();
        if (free_.size() > kKeep) {
          drop = free_.front();  // the one that has waited longest
          free_.erase(free_.begin());
        }
      }
      if (drop.kind == HostBlock::kPinned) pinned_--;
    }
    release(drop);
  }

  void close() {
    std::vector<HostBlock> all;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      open_ = false;
      all.swap(free_);
    }
    for (const HostBlock& b : all) release(b);
  }

 private:
  // two arrays of a loop that holds the last result while it makes the next, for each of two results
  static constexpr size_t kKeep = 4;
  static constexpr int kMostPinned = 8;
  static constexpr size_t kPage = 2u << 20;

  static void release(const HostBlock& b) {
    if (b.kind == HostBlock::kPinned) (void)hipHostFree(b.p);
    else if (b.kind == HostBlock::kPages) munmap(b.p, b.bytes);
    else if (b.kind == HostBlock::kHeap) free(b.p);
  }

  std::mutex mutex_;
  std::vector<HostBlock> free_;
  int pinned_ = 0;
  bool open_ = true;
};

// An array that belongs to a caller: gives its memory back when it is deleted.
struct HostLease {
  std::shared_ptr<HostPool> pool;
  HostBlock block;
  ~HostLease() { pool->give(block); }
};

// A host array out of a pool.  Its contents are not set when it is made.
template <class T>
class HostArray {
 public:
  explicit HostArray(std::shared_ptr<HostPool> pool) : pool_(std::move(pool)) {}
  HostArray(const HostArray&) = delete;
  HostArray& operator=(const HostArray&) = delete;
  ~HostArray() { clear(); }
  T* data() { return (T*)block_.p; }
  const T* data() const { return (const T*)block_.p; }
  size_t size() const { return size_; }
  bool empty() const { return size_ == 0; }
  bool page_locked() const { return block_.kind == HostBlock::kPinned; }

  void resize(size_t n) {
    if (n == size_ && (n == 0 || block_.p)) return;
    clear();
    if (n) block_ = pool_->take(n * sizeof(T));
    size_ = n;
  }
  // n elements, every one `value` (and every page touched: by several threads where there are many)
  void assign(size_t n, T value) {
    resize(n);
    constexpr size_t kPiece = (4u << 20) / sizeof(T);
    std::atomic<size_t> next(0);
    auto fill = [&] {
      for (size_t at; (at = next.fetch_add(kPiece)) < n;) std::fill_n(data() + at, std::min(kPiece, n - at), value);
    };
    if (n <= 2 * kPiece) fill();
    else HostWorkers::get().run(HostWorkers::kMost, fill);
  }
  // Hands the memory over.  size() stays what it was: the next resize() takes other memory.
  HostLease* detach() {
    if (!block_.p) return nullptr;
    HostLease* lease = new HostLease{pool_, block_};
    block_ = HostBlock();
    return lease;
  }
  void clear() {
    if (block_.p) pool_->give(block_);
    block_ = HostBlock();
    size_ = 0;
  }

 private:
  std::shared_ptr<HostPool> pool_;
  HostBlock block_;
  size_t size_ = 0;
};

// ---- packing -------------------------------------------------------------------------------

constexpr uint32_t kPackThreads = 256;
constexpr uint32_t kPackGroup = 8;                               // ids of a group: b bits each, b bytes together
constexpr uint32_t kPackChunkGroups = 512;                       // groups of a chunk, a workgroup's work
constexpr uint32_t kPackChunk = kPackGroup * kPackChunkGroups;   // ids of a chunk: 16 KB of results
constexpr uint32_t kPackMostBits = 25;                           // wider ids travel as whole words

// What a chunk's groups are: which of them hold anything but `fill` (bit g of word g / 64), and whether an id
// did not fit its bits.
struct PackHeader {
  uint64_t live[kPackChunkGroups / 64];
  uint64_t overflow;
  uint64_t pad[7];
};

// Packs ids [chunk * kPackChunk, ...) of src into out[chunk * kPackChunkGroups * bits ...): the groups of
// eight that are not all `fill`, back to back, `bits` bytes each.  out and headers are host memory, and the
// stores to it are what takes the time (54.7 GB/s of packed bytes; packing the 1.68 GB of R-MAT 22 walks into
// device memory instead would take a twentieth of it), hence whole chunks through LDS and 16-byte stores by
// consecutive lanes; nothing else here is tuned.
__global__ __launch_bounds__(kPackThreads) void pack_results(const int32_t* __restrict__ src, size_t n, uint32_t bits,
                                                             int32_t fill, uint8_t* __restrict__ out,
                                                             PackHeader* __restrict__ headers) {
  __shared__ __align__(16) uint8_t s_packed[kPackChunk * sizeof(int32_t)];
  __shared__ uint64_t s_live[kPackChunkGroups / 64];
  constexpr uint32_t kRounds = kPackChunkGroups / kPackThreads;
  const size_t first = (size_t)blockIdx.x * kPackChunk;
  const uint32_t lane = threadIdx.x & 63u;
  int32_t ids[kRounds][kPackGroup];
  bool live[kRounds];
  bool overflow = false;
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) {
    const size_t at = first + (size_t)(r * kPackThreads + threadIdx.x) * kPackGroup;
    if (at + kPackGroup <= n) {
      const int4 lo = *reinterpret_cast<const int4*>(src + at), hi = *reinterpret_cast<const int4*>(src + at + 4);
      ids[r][0] = lo.x; ids[r][1] = lo.y; ids[r][2] = lo.z; ids[r][3] = lo.w;
      ids[r][4] = hi.x; ids[r][5] = hi.y; ids[r][6] = hi.z; ids[r][7] = hi.w;
    } else {
#pragma unroll
      for (uint32_t i = 0; i < kPackGroup; ++i) ids[r][i] = at + i < n ? src[at + i] : fill;
    }
    live[r] = false;
#pragma unroll
    for (uint32_t i = 0; i < kPackGroup; ++i) live[r] = live[r] || ids[r][i] != fill;
    const uint64_t mask = __ballot(live[r]);
    if (lane == 0) s_live[(r * kPackThreads + threadIdx.x) / 64u] = mask;
    if (bits < 32 && live[r]) {
#pragma unroll
      for (uint32_t i = 0; i < kPackGroup; ++i) overflow = overflow || ((uint32_t)ids[r][i] >> bits) != 0;
    }
  }
  const int any_overflow = __syncthreads_or(overflow ? 1 : 0);
  uint32_t total = 0;
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) {
    const uint32_t word = (r * kPackThreads + threadIdx.x) / 64u;
    uint32_t before = 0;
    total = 0;
    for (uint32_t w = 0; w < kPackChunkGroups / 64; ++w) {
      const uint32_t here = (uint32_t)__popcll(s_live[w]);
      if (w < word) before += here;
      total += here;
    }
    if (!live[r]) continue;
    before += (uint32_t)__popcll(s_live[word] & ((1ull << lane) - 1ull));
    uint8_t* dst = s_packed + before * bits;
    uint64_t acc = 0;
    uint32_t held = 0;
#pragma unroll
    for (uint32_t i = 0; i < kPackGroup; ++i) {
      acc |= (uint64_t)(uint32_t)ids[r][i] << held;
      held += bits;
      while (held >= 8) {
        *dst++ = (uint8_t)acc;
        acc >>= 8;
        held -= 8;
      }
    }
  }
  __syncthreads();
  uint8_t* chunk_out = out + (size_t)blockIdx.x * kPackChunkGroups * bits;
  const uint32_t words = (total * bits + 15u) / 16u;
  for (uint32_t i = threadIdx.x; i < words; i += kPackThreads)
    reinterpret_cast<uint4*>(chunk_out)[i] = reinterpret_cast<const uint4*>(s_packed)[i];
  if (threadIdx.x < kPackChunkGroups / 64) headers[blockIdx.x].live[threadIdx.x] = s_live[threadIdx.x];
  if (threadIdx.x == kPackChunkGroups / 64) headers[blockIdx.x].overflow = (uint64_t)any_overflow;
}

// ---- unpacking -----------------------------------------------------------------------------

// How eight `bits`-bit ids come out of `bits` bytes: ids 0-3 out of the 16 bytes at 0, ids 4-7 out of the 16 bytes
// at high_at; id i is the little-endian word at the bytes its shuffle names, shifted right and masked.
struct UnpackPlan {
  uint32_t bits = 32;
  uint32_t high_at = 0;
  int8_t shuffle[32];
  int32_t shift[8];
  uint32_t mask = 0xffffffffu;

  explicit UnpackPlan(uint32_t b) : bits(b) {
    if (b > kPackMostBits) return;
    mask = (1u << b) - 1u;
    high_at = (4 * b) >> 3;
    for (uint32_t i = 0; i < 8; ++i) {
      const uint32_t bit = i < 4 ? i * b : i * b - 8 * high_at;
      for (uint32_t k = 0; k < 4; ++k) shuffle[4 * i + k] = (int8_t)((bit >> 3) + k);
      shift[i] = (int32_t)(bit & 7u);
    }
  }
};

// Bytes the unpacking may read past the last group of a chunk.
constexpr size_t kUnpackOverread = 32;

inline void unpack_groups_plain(const UnpackPlan& plan, const uint8_t* src, int32_t* dst, size_t groups) {
  for (size_t g = 0; g < groups; ++g, src += plan.bits, dst += kPackGroup) {
    if (plan.bits > kPackMostBits) {
      memcpy(dst, src, kPackGroup * sizeof(int32_t));
      continue;
    }
    for (uint32_t i = 0; i < kPackGroup; ++i) {
      uint64_t word;
      memcpy(&word, src + ((i * plan.bits) >> 3), sizeof(word));
      dst[i] = (int32_t)((uint32_t)(word >> ((i * plan.bits) & 7u)) & plan.mask);
    }
  }
}

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
// Streaming stores (dst is a multiple of 32 bytes): the result is written once and read by nobody here, and a line
// that is not fetched before it is overwritten is half the memory traffic.
__attribute__((target("avx2"))) inline void unpack_groups_avx2(const UnpackPlan& plan, const uint8_t* src, int32_t* dst,
                                                               size_t groups) {
  if (plan.bits > kPackMostBits) {
    for (size_t g = 0; g < groups; ++g)
      _mm256_stream_si256((__m256i*)(dst + g * kPackGroup), _mm256_loadu_si256((const __m256i*)(src + g * 32)));
    return;
  }
  const __m256i shuffle = _mm256_loadu_si256((const __m256i*)plan.shuffle);
  const __m256i shift = _mm256_loadu_si256((const __m256i*)plan.shift);
  const __m256i mask = _mm256_set1_epi32((int)plan.mask);
  for (size_t g = 0; g < groups; ++g, src += plan.bits) {
    const __m128i lo = _mm_loadu_si128((const __m128i*)src);
    const __m128i hi = _mm_loadu_si128((const __m128i*)(src + plan.high_at));
    const __m256i both = _mm256_inserti128_si256(_mm256_castsi128_si256(lo), hi, 1);
    const __m256i ids = _mm256_and_si256(_mm256_srlv_epi32(_mm256_shuffle_epi8(both, shuffle), shift), mask);
    _mm256_stream_si256((__m256i*)(dst + g * kPackGroup), ids);
  }
}
__attribute__((target("avx2"))) inline void fill_groups_avx2(int32_t fill, int32_t* dst, size_t groups) {
  const __m256i ids = _mm256_set1_epi32(fill);
  for (size_t g = 0; g < groups; ++g) _mm256_stream_si256((__m256i*)(dst + g * kPackGroup), ids);
}
inline bool unpack_has_avx2() { return __builtin_cpu_supports("avx2"); }
inline void unpack_fence() { _mm_sfence(); }
inline void spin_pause() { _mm_pause(); }
#else
inline void unpack_groups_avx2(const UnpackPlan&, const uint8_t*, int32_t*, size_t) {}
inline void fill_groups_avx2(int32_t, int32_t*, size_t) {}
inline bool unpack_has_avx2() { return false; }
inline void unpack_fence() {}
inline void spin_pause() {}
#endif

// One chunk: count ids (at most kPackChunk) to dst.
inline void unpack_chunk(const UnpackPlan& plan, const PackHeader& header, const uint8_t* src, int32_t fill,
                         int32_t* dst, size_t count) {
  alignas(32) int32_t whole[kPackChunk];
  const bool direct = count == kPackChunk;
  int32_t* at = direct ? dst : whole;
  const bool streams = ((uintptr_t)at & 31u) == 0 && unpack_has_avx2();
  for (uint32_t w = 0; w < kPackChunkGroups / 64; ++w) {
    uint64_t live = header.live[w];
    for (uint32_t g = 0; g < 64;) {
      // a run of groups of one kind
      const bool is_live = live & 1u;
      const uint64_t ends = is_live ? ~live : live;
      uint32_t run = ends ? (uint32_t)__builtin_ctzll(ends) : 64u;
      run = std::min(run, 64u - g);
      if (is_live) {
        if (streams) unpack_groups_avx2(plan, src, at, run);
        else unpack_groups_plain(plan, src, at, run);
        src += (size_t)run * plan.bits;
      } else if (streams) {
        fill_groups_avx2(fill, at, run);
      } else {
        std::fill_n(at, (size_t)run * kPackGroup, fill);
      }
      at += (size_t)run * kPackGroup;
      g += run;
      live = run < 64 ? live >> run : 0;
    }
  }
  if (!direct) memcpy(dst, whole, count * sizeof(int32_t));
}

// ---- the stream ----------------------------------------------------------------------------

// Brings words of device memory to the host, packed on the way.  One caller at a time.
class ResultStream {
 public:
  ResultStream() = default;
  ResultStream(const ResultStream&) = delete;
  ResultStream& operator=(const ResultStream&) = delete;
  ~ResultStream() { release(); }

  // n words at src (aligned to 16 bytes) to dst, in stream order.  Words that are `fill` in groups of eight cost
  // nothing; words are expected to fit `bits` bits (one that does not makes the whole transfer start again with
  // 32).  Large transfers only: it pays from a few megabytes on.
  hipError_t fetch(const int32_t* src, size_t n, uint32_t bits, int32_t fill, int32_t* dst, hipStream_t stream) {
    if (bits > kPackMostBits) bits = 32;
    bool overflow = false;
    hipError_t e = transfer(src, n, bits, fill, dst, stream, &overflow);
    if (e == hipSuccess && overflow) e = transfer(src, n, 32, fill, dst, stream, &overflow);
    return e;
  }

  void release() {
    for (Slot& s : slots_) {
      if (s.done) (void)hipEventDestroy(s.done);
      s.done = nullptr;
    }
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
    ring_bytes_ = 0;
  }

 private:
  static constexpr int kSlots = 8;
  // Chunks of a piece: at most 8 MB of results (0.1 ms on the bus, long against a launch and an event; with pieces of
  // 16 MB the ring no longer stays in the last-level cache between the bus and the threads: 1.68 GB in 16 instead of 14
  // ms), at least 1 MB, else a sixth of the whole (23 MB: 265 us, with a sixteenth 352).
  static constexpr size_t kMostChunks = 512, kLeastChunks = 64, kPieces = 6;
  static constexpr size_t kChunksAtOnce = 4;  // what a thread takes
  static constexpr int kSpins = 4000;  // tens of microseconds; none: 1.68 GB in 19 instead of 13 ms, 23 MB in 527 instead of 290 us

  struct Slot {
    hipEvent_t done = nullptr;
  };

  hipError_t prepare(size_t slot_bytes) {
    for (Slot& s : slots_)
      if (!s.done) {
        const hipError_t e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming | hipEventReleaseToSystem);
        if (e != hipSuccess) return e;
      }
    if (ring_bytes_ >= slot_bytes * kSlots) return hipSuccess;
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
    ring_bytes_ = 0;
    const hipError_t e = hipHostMalloc((void**)&ring_, slot_bytes * kSlots, hipHostMallocDefault);
    if (e == hipSuccess) ring_bytes_ = slot_bytes * kSlots;
    return e;
  }

  hipError_t transfer(const int32_t* src, size_t n, uint32_t bits, int32_t fill, int32_t* dst, hipStream_t stream,
                      bool* overflow) {
    *overflow = false;
    if (n == 0) return hipSuccess;
    const size_t chunks = (n + kPackChunk - 1) / kPackChunk;
    size_t per_piece = (chunks + kPieces - 1) / kPieces;
    per_piece = std::min(kMostChunks, std::max(kLeastChunks, per_piece));
    per_piece = (per_piece + kChunksAtOnce - 1) / kChunksAtOnce * kChunksAtOnce;
    const size_t pieces = (chunks + per_piece - 1) / per_piece;
    const size_t chunk_bytes = (size_t)kPackChunkGroups * bits;
    const size_t packed_at = sizeof(PackHeader) * per_piece;
    const size_t slot_bytes = (packed_at + chunk_bytes * per_piece + kUnpackOverread + 255) / 256 * 256;
    hipError_t error = prepare(slot_bytes);
    if (error != hipSuccess) return error;
    const UnpackPlan plan(bits);

    struct Shared {
      std::atomic<size_t> next{0};       // chunk to take
      std::atomic<size_t> arrived{0};    // pieces whose bytes are here
      std::atomic<bool> stop{false}, overflow{false};
      std::mutex mutex;
      std::condition_variable more;
      unsigned sleepers = 0;
    } shared;
    // A piece comes every 20-200 us: worth a short wait awake (a thread that sleeps is back 50 us later, and
    // waking all of them costs the driving thread as much), but not more than that.
    auto await = [&](size_t piece) {
      for (int spin = 0; spin < kSpins; ++spin) {
        if (shared.arrived.load(std::memory_order_acquire) > piece || shared.stop.load()) return;
        spin_pause();
      }
      std::unique_lock<std::mutex> lock(shared.mutex);
      shared.sleepers++;
      shared.more.wait(lock, [&] { return shared.arrived.load(std::memory_order_acquire) > piece || shared.stop.load(); });
      shared.sleepers--;
    };
    auto announce = [&](size_t arrived, bool stop) {
      bool asleep;
      {
        std::lock_guard<std::mutex> lock(shared.mutex);
        if (stop) shared.stop.store(true);
        else shared.arrived.store(arrived, std::memory_order_release);
        asleep = shared.sleepers > 0;
      }
      if (asleep) shared.more.notify_all();
    };
    std::vector<std::atomic<size_t>> left(pieces);  // chunks of a piece that are not unpacked yet
    for (size_t p = 0; p < pieces; ++p) left[p].store(std::min(per_piece, chunks - p * per_piece));

    auto slot = [&](size_t piece) { return ring_ + (piece % kSlots) * slot_bytes; };
    auto launch = [&](size_t piece) -> hipError_t {
      const size_t first = piece * per_piece * kPackChunk;
      const size_t here = std::min(n - first, per_piece * kPackChunk);
      uint8_t* at = slot(piece);
      pack_results<<<dim3((unsigned)((here + kPackChunk - 1) / kPackChunk)), dim3(kPackThreads), 0, stream>>>(
          src + first, here, bits, fill, at + packed_at, (PackHeader*)at);
      const hipError_t e = hipGetLastError();
      return e != hipSuccess ? e : hipEventRecord(slots_[piece % kSlots].done, stream);
    };
    // unpacks the chunks [c, end) of a piece that is here
    auto unpack = [&](size_t c, size_t end) {
      const size_t piece = c / per_piece;
      const uint8_t* at = slot(piece);
      for (size_t i = c; i < end; ++i) {
        const size_t in_piece = i - piece * per_piece;
        const PackHeader& header = ((const PackHeader*)at)[in_piece];
        if (header.overflow) shared.overflow.store(true, std::memory_order_relaxed);
        const size_t first = i * kPackChunk;
        unpack_chunk(plan, header, at + packed_at + in_piece * chunk_bytes, fill, dst + first,
                     std::min<size_t>(kPackChunk, n - first));
      }
      unpack_fence();
      left[piece].fetch_sub(end - c, std::memory_order_release);
    };
    auto work = [&] {
      for (;;) {
        const size_t c = shared.next.fetch_add(kChunksAtOnce);
        if (c >= chunks) return;
        const size_t piece = c / per_piece;
        await(piece);
        if (shared.stop.load()) return;
        unpack(c, std::min(c + kChunksAtOnce, std::min(chunks, (piece + 1) * per_piece)));
      }
    };
    auto drive = [&] {
      size_t launched = 0;
      for (; launched < pieces && launched < kSlots && error == hipSuccess; ++launched) error = launch(launched);
      for (size_t p = 0; p < pieces && error == hipSuccess; ++p) {
        // the slot of piece p - 1 is free for piece p - 1 + kSlots once it is unpacked; kSlots - 1 pieces are
        // under way meanwhile
        if (p > 0 && launched < pieces) {
          while (left[p - 1].load(std::memory_order_acquire) != 0) {
            const size_t c = shared.next.load();
            size_t mine = c;
            if (c < p * per_piece && shared.next.compare_exchange_strong(mine, c + kChunksAtOnce))
              unpack(c, std::min(c + kChunksAtOnce, std::min(chunks, (c / per_piece + 1) * per_piece)));
            else
              std::this_thread::yield();
          }
          error = launch(launched);
          if (error != hipSuccess) break;
          launched++;
        }
        error = hipEventSynchronize(slots_[p % kSlots].done);
        if (error != hipSuccess) break;
        announce(p + 1, false);
      }
      if (error != hipSuccess) {
        announce(0, true);
        return;
      }
      work();
    };
    HostWorkers::get().run(HostWorkers::kMost, work, drive);
    if (error != hipSuccess) {
      (void)hipStreamSynchronize(stream);  // nothing writes to the ring after this
      return error;
    }
    *overflow = shared.overflow.load();
    return hipSuccess;
  }

  uint8_t* ring_ = nullptr;
  size_t ring_bytes_ = 0;
  Slot slots_[kSlots];
};

}  // namespace nd
