// Results on their way to the host, and the host memory they land in.
//
// A pass leaves gigabytes of 4-byte vertex ids in device memory and the caller wants them in
// host memory: of 4.2 M node2vec walks (1.68 GB, 34 ms to sample) the copy took 29 ms at the bus's
// 57 GB/s, and another 118 ms went into handing the caller an array of their own.  Four things
// are done about it here:
//
//  * What crosses the bus is packed (pack_results): ids take as many bits as the largest one, the
//    number of vertices, needs (23 instead of 32 for R-MAT 22), and groups of eight consecutive
//    ids that are all INVALID - walks that have ended, samples without neighbours - are left out.
//    The kernel writes its output straight into page-locked memory (54.7 GB/s, as fast as the copy
//    engine's 57, without a copy per piece) and stamps every chunk that is there, and host threads unpack
//    a chunk while the next ones cross.  Twelve threads write 220 GB/s of unpacked ids on the 16-core share of a
//    GPU's host, 140 while the bus writes to the same memory at its full rate.
//  * Results whose first words are final while later ones are still being computed (walks) can leave then already
//    (ResultStream::begin, with what to wait for).  They are packed into device memory and the copy engine takes them
//    from there: stores of a kernel that wait for the bus stand in the way of all others, and the computation took as much
//    longer as the transfer saved (R-MAT 22 walks 24.1 ms alone, 26.9 with 32 such workgroups beside it, 34 with 512; 24.3
//    with the copy engine at 55 GB/s).
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
#include <unistd.h>
#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <functional>
#include <list>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "nd_host_threads.hpp"

namespace nd {

// ---- host threads ------------------------------------------------------------------------

// A few threads of the process that help whoever calls run(); they sleep otherwise.  They live
// until the process ends (no destructor: a thread must not outlast what it waits on), and the process does not
// end while one of them is at work: a thread inside the HIP runtime while that is being taken down does not come to a good end.
class HostWorkers {
 public:
  // PPR walks over 262 K vertices, most groups dead: 1.33 ms with seven, 1.18 with eleven.
  static constexpr unsigned kMost = 11;

  static HostWorkers& get() {
    static HostWorkers* workers = [] {
      HostWorkers* w = new HostWorkers;
      // what was registered last is done first: the runtime, which was there before any work for these threads, is still whole
      (void)std::atexit([] { (void)get().rest(); });
      return w;
    }();
    return *workers;
  }

  // Work that several threads may take part in: each calls body() once, and the body() of whoever calls join() has to be able to
  // do all of it alone.  It must not throw.  A Job stays where it is from start() to join().
  struct Job {
    std::function<void()> body;
    unsigned wanted = 0, running = 0;
  };

  // Has up to `helpers` threads call body(), as far as threads are free.
  void start(Job& job, unsigned helpers) {
    job.wanted = std::min(helpers, limit());
    job.running = 0;
    if (job.wanted == 0) return;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      grow(job.wanted);
      jobs_.push_back(&job);
    }
    wake_.notify_all();
  }

  // The same again, for a job that has been started: for threads whose body() returned because there was nothing to do yet.
  void more(Job& job, unsigned helpers) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      job.wanted += helpers;
    }
    wake_.notify_all();
  }

  // Nobody starts on it any more; returns when every body() that started has returned.
  void join(Job& job) {
    std::unique_lock<std::mutex> lock(mutex_);
    jobs_.remove(&job);
    ended_.wait(lock, [&] { return job.running == 0; });
  }

  // For the end of the process: no thread starts on anything any more; returns whether none is at work.  What they work on
  // ends by itself, within tens of milliseconds; if something else is amiss the process still ends.  (A forked child
  // has none of the threads, but a copy of what they were at, and of who held the lock.)
  bool rest() {
    if (getpid() != process_) return false;
    std::unique_lock<std::mutex> lock(mutex_);
    resting_ = true;
    return ended_.wait_for(lock, std::chrono::seconds(10), [&] { return at_work_ == 0; });
  }

  // body() on this thread and on up to `helpers` others.
  void run(unsigned helpers, const std::function<void()>& body) {
    Job job;
    job.body = body;
    start(job, helpers);
    body();
    join(job);
  }

 private:
  HostWorkers() = default;

  // besides the thread that calls
  static unsigned limit() {
    if (const unsigned wanted = host_threads_wanted()) return std::min(wanted - 1, kMost);
    const unsigned cpus = host_cpus();
    return cpus > 1 ? std::min(cpus * 3 / 4, kMost) : 0;
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
        if (j->wanted > 0 && !resting_) { job = j; break; }
      if (!job) {
        wake_.wait(lock);
        continue;
      }
      job->wanted--;
      job->running++;
      at_work_++;
      lock.unlock();
      job->body();
      lock.lock();
      at_work_--;
      if (--job->running == 0) ended_.notify_all();
    }
  }

  std::mutex mutex_;
  std::condition_variable wake_, ended_;
  std::list<Job*> jobs_;
  const pid_t process_ = getpid();
  unsigned threads_ = 0, at_work_ = 0;
  bool resting_ = false;
};

// ---- host memory ---------------------------------------------------------------------------

struct HostBlock {
  void* p = nullptr;
  size_t bytes = 0;
  bool mapped = false;  // by mmap, else from the heap
};

// Results up to this size are unpacked by the thread that asks for them, and into the caches: other threads are awake 50 us
// later (64 KB to 2 MB in 31 to 118 us by the copy engine and memcpy(), which also waited for the bus before it began; walks
// over 2.7 K vertices, 1.1 MB, whose packing follows them: 0.121 ms a pass instead of 0.147).
constexpr size_t kDirectResultBytes = 2u << 20;

// The host arrays of one sampler.  A few of them (keep()) wait for their next use; all of those are freed with the
// sampler's device memory and when it goes, the others when their holders let go of them.
// They are ordinary private memory, since callers do with them what they do with any array: page-locked memory
// of the runtime's is not there in a forked child (a data loader's worker that touches it dies), nor may system calls
// that pin pages use it.  (The copy engine writing into it directly would save 1.1 MB of results 39 of 67 us.)
class HostPool {
 public:
  HostPool() = default;
  HostPool(const HostPool&) = delete;
  HostPool& operator=(const HostPool&) = delete;
  ~HostPool() { close(); }

  HostBlock take(size_t bytes) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (size_t i = 0; i < free_.size(); ++i)
        if (free_[i].bytes >= bytes && free_[i].bytes / 2 <= bytes) {
          const HostBlock b = free_[i];
          free_.erase(free_.begin() + (ptrdiff_t)i);
          return b;
        }
    }
    HostBlock b;
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
        b.mapped = true;
        return b;
      }
    }
    b.p = malloc(bytes);
    if (!b.p) throw std::bad_alloc();
    b.bytes = bytes;
    return b;
  }

  void give(HostBlock b) {
    HostBlock drop = b;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (open_) {
        free_.push_back(b);
        drop = HostBlock();
        if (free_.size() > keep_) {
          drop = free_.front();  // the one that has waited longest
          free_.erase(free_.begin());
        }
      }
    }
    release(drop);
  }

  // How many wait at most.  A loop that holds its last results while it makes the next leaves one array of each kind
  // of result waiting at a time.
  void keep(size_t kinds) {
    trim();
    std::lock_guard<std::mutex> lock(mutex_);
    keep_ = kinds;
  }
  // frees those that wait
  void trim() { drop_waiting(true); }
  // ... and keeps none from here on
  void close() { drop_waiting(false); }

  size_t waiting_bytes() {
    std::lock_guard<std::mutex> lock(mutex_);
    size_t sum = 0;
    for (const HostBlock& b : free_) sum += b.bytes;
    return sum;
  }

 private:
  void drop_waiting(bool open) {
    std::vector<HostBlock> all;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      open_ = open_ && open;
      all.swap(free_);
    }
    for (const HostBlock& b : all) release(b);
  }
  static constexpr size_t kPage = 2u << 20;

  static void release(const HostBlock& b) {
    if (b.mapped) munmap(b.p, b.bytes);
    else free(b.p);
  }

  std::mutex mutex_;
  std::vector<HostBlock> free_;
  size_t keep_ = 2;
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

  void resize(size_t n) {
    if (n == size_ && (n == 0 || block_.p)) return;
    clear();
    if (n) block_ = pool_->take(n * sizeof(T));
    size_ = n;
  }
  // The same where the memory is only good to have: false, and empty, if there is none.
  bool try_resize(size_t n) {
    try {
      resize(n);
      return true;
    } catch (const std::bad_alloc&) {
      return false;
    }
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
  // its memory was handed over, and not taken anew since
  bool taken() const { return size_ != 0 && !block_.p; }
  void swap(HostArray& other) {
    std::swap(pool_, other.pool_);
    std::swap(block_, other.block_);
    std::swap(size_, other.size_);
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

// What a chunk's groups are: which of them hold anything but `fill` (bit g of word g / 64), how many bits an id of
// theirs takes, counted from the smallest (all ones: `fill`; 32: the words as they are), and whether that is more than there is room for.
struct PackHeader {
  uint64_t live[kPackChunkGroups / 64];
  uint64_t overflow;
  uint64_t at;  // of its bytes among the piece's, if staged
  uint32_t bits, base;
  uint64_t stamp;  // straight to the host: the transfer's number and the chunk's, once all else of the chunk is there
  uint64_t pad[4];
};
static_assert(sizeof(PackHeader) == 128, "a line of memory");

// Where the chunks' bytes go: chunk after chunk, each as far from the last as a whole one takes, round a ring (a power of two chunks, or
// more than there are), or (staged) one directly after another, in whatever order the workgroups get there, for a copy that is to
// take no more than there is.
struct PackedOut {
  uint8_t* bytes;
  PackHeader* headers;
  // straight
  uint32_t first = 0, ring_mask = 0xffffffffu;  // of the launch's first chunk
  uint64_t stamp = 0;                           // its
  // staged
  uint32_t* cursor = nullptr;    // 16 bytes each; 0 before the launch and after it
  uint32_t* finished = nullptr;  // workgroups; likewise
  uint32_t* total = nullptr;     // host memory: what cursor was at the end
};

// Bits for the numbers 0 .. range and one more, all of them ones.
__host__ __device__ inline uint32_t bits_for_range(uint32_t range) {
  uint32_t bits = 1;
  while (bits <= kPackMostBits && range >= (1u << bits) - 1u) bits++;
  return bits <= kPackMostBits ? bits : 32u;
}

__device__ __forceinline__ void store_past_caches(uint4* at, uint4 v) {
  typedef uint32_t Four __attribute__((ext_vector_type(4)));
  const Four x = {v.x, v.y, v.z, v.w};
  // (two wait states before its registers are written again, as the compiler would have them)
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" : : "v"(at), "v"(x) : "memory");
}

// Packs ids [chunk * kPackChunk, ...) of src: the groups of eight that are not all `fill`, back to back, at most `bits` bits an
// id.  Where out is host memory the stores to it are what takes the time (54.7 GB/s of packed bytes; packing the 1.68 GB of
// R-MAT 22 walks into device memory instead takes a twentieth of it), hence whole chunks through LDS and 16-byte stores by
// consecutive lanes.  Such a chunk is stamped when its bytes have been acknowledged: the threads that unpack it look for that,
// so that any number of chunks is one launch (uniform walks 57 K, whose rows were nine launches with an event and
// 5.6 us between each and the next: 225 us from the first to the last, now 180).  Ids are counted from the chunk's
// smallest: two in five bits of what MVS lists (rows of 32 batches of consecutive vertices: 9 bits instead of 18) and, with
// `fill` all ones, one of the 21 that 2^20 vertices and INVALID would take.  (kStaged is the kernel's and not the launch's: with both
// forms' loads in one kernel those of a chunk wait for each other, and MultiRW 100 K took 1.59 ms instead of 1.55, KHop over
// R-MAT 20 11.7 instead of 11.4.)
template <bool kStaged>
__global__ __launch_bounds__(kPackThreads) void pack_results(const int32_t* __restrict__ src, size_t n, uint32_t most_bits,
                                                             int32_t fill, PackedOut out, uint32_t n_chunks) {
  __shared__ __align__(16) uint8_t s_packed[kPackChunk * sizeof(int32_t)];
  __shared__ uint64_t s_live[kPackChunkGroups / 64];
  __shared__ uint32_t s_least[kPackThreads / 64], s_largest[kPackThreads / 64];
  __shared__ uint32_t s_at;
  constexpr uint32_t kRounds = kPackChunkGroups / kPackThreads;
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t chunk = blockIdx.x; chunk < n_chunks; chunk += gridDim.x) {
    const size_t first = (size_t)chunk * kPackChunk;
    int32_t ids[kRounds][kPackGroup];
    bool live[kRounds];
    uint32_t least = 0xffffffffu, largest = 0;  // of those that are not `fill`
#pragma unroll
    for (uint32_t r = 0; r < kRounds; ++r) {
      const size_t at = first + (size_t)(r * kPackThreads + threadIdx.x) * kPackGroup;
      if (at + kPackGroup <= n) {
        int4 lo, hi;
        if (kStaged) {
          // Words of a kernel that is still running, which stored them past its caches: they are read past this one's.  (A fence
          // that empties the caches would empty them for that kernel too: DeepWalk, a million walks, 2.3 -> 3.1 ms.)
          const uint64_t* from = reinterpret_cast<const uint64_t*>(src + at);
          uint64_t two[4];
#pragma unroll
          for (uint32_t i = 0; i < 4; ++i) two[i] = __hip_atomic_load(from + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          lo = make_int4((int)two[0], (int)(two[0] >> 32), (int)two[1], (int)(two[1] >> 32));
          hi = make_int4((int)two[2], (int)(two[2] >> 32), (int)two[3], (int)(two[3] >> 32));
        } else {
          lo = *reinterpret_cast<const int4*>(src + at);
          hi = *reinterpret_cast<const int4*>(src + at + 4);
        }
        ids[r][0] = lo.x; ids[r][1] = lo.y; ids[r][2] = lo.z; ids[r][3] = lo.w;
        ids[r][4] = hi.x; ids[r][5] = hi.y; ids[r][6] = hi.z; ids[r][7] = hi.w;
      } else {
#pragma unroll
        for (uint32_t i = 0; i < kPackGroup; ++i)
          ids[r][i] = at + i >= n ? fill : kStaged ? __hip_atomic_load(src + at + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) : src[at + i];
      }
    }
#pragma unroll
    for (uint32_t r = 0; r < kRounds; ++r) {
      live[r] = false;
#pragma unroll
      for (uint32_t i = 0; i < kPackGroup; ++i) {
        const bool counts = ids[r][i] != fill;
        live[r] = live[r] || counts;
        least = counts && (uint32_t)ids[r][i] < least ? (uint32_t)ids[r][i] : least;
        largest = counts && (uint32_t)ids[r][i] > largest ? (uint32_t)ids[r][i] : largest;
      }
      const uint64_t mask = __ballot(live[r]);
      if (lane == 0) s_live[(r * kPackThreads + threadIdx.x) / 64u] = mask;
    }
    for (int d = 32; d > 0; d >>= 1) {
      const uint32_t a = (uint32_t)__shfl_xor((int)least, d, 64), b = (uint32_t)__shfl_xor((int)largest, d, 64);
      least = a < least ? a : least;
      largest = b > largest ? b : largest;
    }
    if (lane == 0) s_least[threadIdx.x / 64u] = least, s_largest[threadIdx.x / 64u] = largest;
    __syncthreads();
#pragma unroll
    for (uint32_t w = 0; w < kPackThreads / 64; ++w) {
      least = s_least[w] < least ? s_least[w] : least;
      largest = s_largest[w] > largest ? s_largest[w] : largest;
    }
    const bool any = least <= largest;
    const uint32_t bits = any ? bits_for_range(largest - least) : 1u;
    const bool overflow = bits > most_bits;
    const uint32_t base = bits == 32 || !any ? 0u : least, none = bits == 32 ? (uint32_t)fill : (1u << bits) - 1u;
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
        acc |= (uint64_t)(ids[r][i] == fill ? none : (uint32_t)ids[r][i] - base) << held;
        held += bits;
        while (held >= 8) {
          *dst++ = (uint8_t)acc;
          acc >>= 8;
          held -= 8;
        }
      }
    }
    const uint32_t words = overflow ? 0u : (total * bits + 15u) / 16u;
    if (kStaged && threadIdx.x == 0) s_at = atomicAdd(out.cursor, words);
    __syncthreads();
    const uint32_t place = kStaged ? chunk : (out.first + chunk) & out.ring_mask;
    const size_t at = kStaged ? (size_t)s_at * 16u : (size_t)place * kPackChunkGroups * most_bits;
    uint4* chunk_out = reinterpret_cast<uint4*>(out.bytes + at);
    PackHeader* header = out.headers + place;
    for (uint32_t i = threadIdx.x; i < words; i += kPackThreads) {
      const uint4 v = reinterpret_cast<const uint4*>(s_packed)[i];
      if (kStaged) chunk_out[i] = v;
      else store_past_caches(chunk_out + i, v);
    }
    constexpr uint32_t kLiveWords = kPackChunkGroups / 64;
    if (threadIdx.x < kLiveWords + 3) {
      const uint64_t v = threadIdx.x < kLiveWords ? s_live[threadIdx.x % kLiveWords] : threadIdx.x == kLiveWords ? (uint64_t)overflow
                         : threadIdx.x == kLiveWords + 1 ? (uint64_t)at : (uint64_t)bits | (uint64_t)base << 32;
      uint64_t* to = reinterpret_cast<uint64_t*>(header) + threadIdx.x;
      if (kStaged) *to = v;
      else __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (!kStaged) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wavefront's part of the chunk is in host memory
    __syncthreads();  // ... and the others'; the next chunk overwrites what has just been read
    if (!kStaged && threadIdx.x == 0) __hip_atomic_store(&header->stamp, out.stamp + chunk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (kStaged && threadIdx.x == 0 && atomicAdd(out.finished, 1u) == gridDim.x - 1) {
    // the last workgroup: the others' claims were answered before they counted themselves
    __hip_atomic_store(out.total, atomicAdd(out.cursor, 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    *out.cursor = 0;
    *out.finished = 0;
  }
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
  static const UnpackPlan& of(uint32_t bits) {
    static const std::vector<UnpackPlan> plans = [] {
      std::vector<UnpackPlan> made;
      for (uint32_t b = 0; b <= kPackMostBits + 1; ++b) made.emplace_back(b <= kPackMostBits ? b : 32u);
      return made;
    }();
    return plans[std::min(bits, kPackMostBits + 1)];
  }
};

// Bytes the unpacking may read past the last group of a chunk.
constexpr size_t kUnpackOverread = 32;

// One chunk to dst (kPackChunk ids).
inline void unpack_chunk_plain(const PackHeader& header, const uint8_t* src, int32_t fill, int32_t* dst) {
  const UnpackPlan& plan = UnpackPlan::of(header.bits);
  const bool whole = plan.bits > kPackMostBits;
  for (uint32_t g = 0; g < kPackChunkGroups; ++g, dst += kPackGroup) {
    if (!(header.live[g / 64] >> (g % 64) & 1u)) {
      std::fill_n(dst, kPackGroup, fill);
      continue;
    }
    for (uint32_t i = 0; i < kPackGroup; ++i) {
      uint64_t word = 0;
      memcpy(&word, src + ((i * plan.bits) >> 3), whole ? sizeof(uint32_t) : sizeof(word));
      const uint32_t code = (uint32_t)(word >> ((i * plan.bits) & 7u)) & plan.mask;
      dst[i] = whole ? (int32_t)code : code == plan.mask ? fill : (int32_t)(code + header.base);
    }
    src += plan.bits;
  }
}

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
// The same.  kStreaming (dst a multiple of 32 bytes), for results larger than the caches: the result is written once and read by nobody here, and
// a line that is not fetched before it is overwritten is half the memory traffic.  Words of 64 live groups, and of 64
// dead ones, have loops of their own; in a mixed word every group is unpacked from where the next live one
// starts and replaced by `fill` if it is not live itself - no branch to mispredict where walks end at random.
// Eight threads: 200 GB/s of ids (76-100 with a call for every run of groups of one kind).
template <bool kStreaming>
__attribute__((target("avx2"))) inline void unpack_chunk_avx2(const PackHeader& header, const uint8_t* src, int32_t fill,
                                                              int32_t* dst) {
  const UnpackPlan& plan = UnpackPlan::of(header.bits);
  const bool whole = plan.bits > kPackMostBits;
  const size_t bits = plan.bits;
  const __m256i shuffle = _mm256_loadu_si256((const __m256i*)plan.shuffle);
  const __m256i shift = _mm256_loadu_si256((const __m256i*)plan.shift);
  const __m256i mask = _mm256_set1_epi32((int)plan.mask), dead = _mm256_set1_epi32(fill);
  const __m256i base = _mm256_set1_epi32((int)header.base);
  const size_t high_at = plan.high_at;
#define ND_STORE_GROUP(group)                                        \
  do {                                                               \
    const __m256i stored = (group);                                  \
    if (kStreaming) _mm256_stream_si256((__m256i*)dst, stored);      \
    else _mm256_storeu_si256((__m256i*)dst, stored);                 \
  } while (0)
#define ND_UNPACKED_CODES                                                                                          \
  _mm256_and_si256(                                                                                                \
      _mm256_srlv_epi32(_mm256_shuffle_epi8(_mm256_inserti128_si256(                                               \
                                                _mm256_castsi128_si256(_mm_loadu_si128((const __m128i*)src)),      \
                                                _mm_loadu_si128((const __m128i*)(src + high_at)), 1),              \
                                            shuffle),                                                              \
                        shift),                                                                                    \
      mask)
  for (uint32_t w = 0; w < kPackChunkGroups / 64; ++w) {
    uint64_t live = header.live[w];
    if (live == 0) {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup) ND_STORE_GROUP(dead);
    } else if (whole) {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup, live >>= 1) {
        const __m256i here = _mm256_set1_epi32(-(int)(live & 1u));
        ND_STORE_GROUP(_mm256_blendv_epi8(dead, _mm256_loadu_si256((const __m256i*)src), here));
        src += bits & (0 - (size_t)(live & 1u));
      }
    } else if (~live == 0) {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup, src += bits) {
        const __m256i codes = ND_UNPACKED_CODES;
        ND_STORE_GROUP(_mm256_blendv_epi8(_mm256_add_epi32(codes, base), dead, _mm256_cmpeq_epi32(codes, mask)));
      }
    } else {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup, live >>= 1) {
        const __m256i codes = ND_UNPACKED_CODES, gone = _mm256_set1_epi32((int)(live & 1u) - 1);
        ND_STORE_GROUP(_mm256_blendv_epi8(_mm256_add_epi32(codes, base), dead,
                                          _mm256_or_si256(gone, _mm256_cmpeq_epi32(codes, mask))));
        src += bits & (0 - (size_t)(live & 1u));
      }
    }
  }
#undef ND_UNPACKED_CODES
#undef ND_STORE_GROUP
}
inline bool unpack_has_avx2() { return __builtin_cpu_supports("avx2"); }
inline void unpack_fence() { _mm_sfence(); }
inline void spin_pause() { _mm_pause(); }
#else
template <bool kStreaming>
inline void unpack_chunk_avx2(const PackHeader&, const uint8_t*, int32_t, int32_t*) {}
inline bool unpack_has_avx2() { return false; }
inline void unpack_fence() {}
inline void spin_pause() {}
#endif

// The first count ids (at most kPackChunk) of a chunk to dst; streaming: past the caches.
inline void unpack_chunk(const PackHeader& header, const uint8_t* src, int32_t fill, int32_t* dst, size_t count, bool streaming) {
  alignas(32) int32_t part[kPackChunk];
  int32_t* at = count == kPackChunk ? dst : part;
  if (!unpack_has_avx2()) unpack_chunk_plain(header, src, fill, at);
  else if (streaming && at != part && ((uintptr_t)at & 31u) == 0) unpack_chunk_avx2<true>(header, src, fill, at);
  else unpack_chunk_avx2<false>(header, src, fill, at);
  if (at == part) memcpy(dst, part, count * sizeof(int32_t));
}

// Makes a device this thread's current one for as long as it lives.
class OnDevice {
 public:
  explicit OnDevice(int device) {
    error = hipGetDevice(&before_);
    if (error != hipSuccess || before_ == device) return;
    error = hipSetDevice(device);
    moved_ = error == hipSuccess;
  }
  OnDevice(const OnDevice&) = delete;
  OnDevice& operator=(const OnDevice&) = delete;
  ~OnDevice() { if (moved_) (void)hipSetDevice(before_); }
  hipError_t error;

 private:
  int before_ = 0;
  bool moved_ = false;
};

// The device of a stream; of the default stream: the current one.
inline hipError_t device_of(hipStream_t stream, int* device) {
  return stream ? hipStreamGetDevice(stream, device) : hipGetDevice(device);
}

// The streams results cross the bus on while something else is computed: two per device (which has to be the current one) and process, each on
// a hardware queue of its own, which a stream with a mask of compute units (here: all) gets.  (Ordinary streams share
// four; where the computation's lands on the same one, nothing overlaps.)  All the samplers of the process share them, so nothing on
// them ever waits for a computation: what others put there would wait as well.  They are destroyed when the process ends, while
// the runtime and whatever watches it are still there: left to the runtime, their queues outlive a profiler's
// bookkeeping of them, and a profiled process ended in a segmentation fault.
inline std::vector<hipStream_t>& transfer_streams() {
  static std::vector<hipStream_t>* streams = [] {
    auto* made = new std::vector<hipStream_t>;
    (void)std::atexit([] {
      if (!HostWorkers::get().rest()) return;  // somebody may still use them
      for (hipStream_t& s : transfer_streams())
        if (s) (void)hipStreamDestroy(s), s = nullptr;
    });
    return made;
  }();
  return *streams;
}
constexpr size_t kTransferStreams = 2;  // of a device
inline hipStream_t transfer_stream(int device, size_t which) {
  static std::mutex mutex;
  std::vector<hipStream_t>* streams = &transfer_streams();
  std::lock_guard<std::mutex> lock(mutex);
  const size_t at = kTransferStreams * (size_t)device + which;
  if (streams->size() <= at) streams->resize(at + 1, nullptr);
  hipStream_t& stream = (*streams)[at];
  if (!stream) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) return nullptr;
    std::vector<uint32_t> every_cu((size_t)(cus + 31) / 32, 0xffffffffu);
    if (cus % 32 != 0) every_cu.back() = (1u << (cus % 32)) - 1u;
    if (hipExtStreamCreateWithCUMask(&stream, (uint32_t)every_cu.size(), every_cu.data()) != hipSuccess) {
      (void)hipGetLastError();
      stream = nullptr;
    }
  }
  return stream;
}

// ---- the stream ----------------------------------------------------------------------------

// Brings words of device memory to the host, packed on the way.  One caller at a time.  Everything happens on the device of the
// stream that is given, whatever the calling thread's current device is, and leaves that as it was.
class ResultStream {
 public:
  ResultStream() = default;
  ResultStream(const ResultStream&) = delete;
  ResultStream& operator=(const ResultStream&) = delete;
  ~ResultStream() { release(); }

  // Words of device memory that go together.  Those that are `fill` in groups of eight cost nothing; they are expected to fit `bits`
  // bits (one that does not makes the whole transfer start again with 32).  src is aligned to 16 bytes.
  struct Part {
    const int32_t* src;
    size_t n;
    uint32_t bits;
    int32_t fill;
    int32_t* dst;
    bool sparse = false;  // such groups are to be expected anywhere (rows of walks, which end)
  };

  // The first `words` words of a transfer's parts are on the device once `event` has happened, or, if there is a `sign` (all of a
  // transfer's have one or none has; page-locked memory a kernel that is still running writes to, after the words), once that is
  // `value`.
  struct Ready {
    size_t words;
    hipEvent_t event;
    const uint32_t* sign = nullptr;
    uint32_t value = 0;
  };

  // Takes, on the current device and ahead of the first, what a fetch() of n words needs.
  hipError_t reserve(size_t n, uint32_t bits) {
    hipError_t e = finish();
    if (e == hipSuccess) e = come_to_device_of(nullptr);
    if (e != hipSuccess || n == 0) return e;
    if (!transfer_) transfer_.reset(new Transfer);
    transfer_->set({{nullptr, n, bits, 0, nullptr}}, {});
    e = prepare(*transfer_);
    // its pages are mapped when they are first touched: 0.8 ms of 2 MB
    if (e == hipSuccess) memset(ring_, 0, transfer_->chunk_bytes * transfer_->ring_chunks);
    return e;
  }

  // bytes at src to dst as they are, in stream order, complete on return.  For what is not words.
  hipError_t copy(const void* src, size_t bytes, void* dst, hipStream_t stream) {
    hipError_t e = finish();  // an earlier one that nobody waited for
    if (e == hipSuccess) e = come_to_device_of(stream);
    if (e != hipSuccess || bytes == 0) return e;
    const OnDevice on(device_);
    e = on.error != hipSuccess ? on.error : make_ring(kDirectResultBytes);
    for (size_t at = 0; at < bytes && e == hipSuccess; at += kDirectResultBytes) {
      const size_t here = std::min(bytes - at, kDirectResultBytes);
      e = hipMemcpyAsync(ring_, (const char*)src + at, here, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e == hipSuccess) memcpy((char*)dst + at, ring_, here);
    }
    return e;
  }

  // Parts to where they belong, in stream order.
  hipError_t fetch(std::vector<Part> parts, hipStream_t stream) {
    const hipError_t e = begin(std::move(parts), stream, {});
    return e == hipSuccess ? finish() : e;
  }
  hipError_t fetch(const int32_t* src, size_t n, uint32_t bits, int32_t fill, int32_t* dst, hipStream_t stream) {
    return fetch({{src, n, bits, fill, dst}}, stream);
  }
  hipError_t begin(const int32_t* src, size_t n, uint32_t bits, int32_t fill, int32_t* dst, hipStream_t stream,
                   std::vector<Ready> ready, bool follows = false) {
    return begin({{src, n, bits, fill, dst}}, stream, std::move(ready), follows);
  }

  // The same as a begin() that returns at once, other threads taking it from there, and a finish() that takes part
  // and returns when the words are at dst.  `ready` (words ascending, the last all of them; with a sign, of a single part): what has to have
  // happened before words may be read, while other work of the caller's is still going on; empty: stream order, and `follows` where what the
  // words follow there takes a while: the threads then look for none until the caller, who waits for that anyway, says words_are_there().
  // (A thread that asked for the event meanwhile would get no answer: hipEventSynchronize() holds the event until it returns, and a
  // query of 13.9 ms was over 13 to 36 us after that.)  What is given has to stay until finish().
  hipError_t begin(std::vector<Part> parts, hipStream_t stream, std::vector<Ready> ready, bool follows = false) {
    hipError_t e = finish();  // an earlier one that nobody waited for
    parts.erase(std::remove_if(parts.begin(), parts.end(), [](const Part& p) { return p.n == 0; }), parts.end());
    if (e != hipSuccess || parts.empty()) return e;
    if (!transfer_) transfer_.reset(new Transfer);
    Transfer& t = *transfer_;
    e = come_to_device_of(stream);
    if (e != hipSuccess) return e;
    t.device = device_;
    const OnDevice on(t.device);
    if (on.error != hipSuccess) return on.error;
    t.set(std::move(parts), std::move(ready));
    e = prepare(t);
    if (e == hipSuccess && t.staged) e = prepare_staging(t.slot_bytes);
    if (e != hipSuccess) return e;
    t.number = ++transfers_;
    t.streams[0] = t.streams[1] = transfer_stream(t.device, 0);
    if (t.staged || !t.ready.empty()) t.streams[t.staged ? 0 : 1] = transfer_stream(t.device, 1);
    if (!t.ready.empty()) ahead_.store(0, std::memory_order_relaxed);
    size_t helpers = HostWorkers::kMost;
    if (t.ready.empty()) {
      t.streams[0] = stream;
      t.follows = follows;
      if (t.chunks <= t.ring_chunks) t.streams[1] = stream;
      else e = hipEventRecord(begun_, stream);
      // (all on the given stream: the other one is not only ours, and what is computed before this may take long)
      while (e == hipSuccess && t.sent < t.ring_chunks)
        e = launch(std::min(t.part_ends[t.part_of(t.sent)], t.ring_chunks), blocks_in_order(), stream);
      if (e != hipSuccess) {
        (void)hipStreamSynchronize(stream);  // nothing writes to the ring after this
        return e;
      }
      // few chunks are unpacked before a thread is awake, unless it is woken while they are computed
      if (t.chunks <= kFewChunks) helpers = follows ? t.chunks / kChunksAHelper : 0;
      if (!follows) announce(t.sent);
    }
    job_.body = [this] { take_part(/*stays=*/false); };
    under_way_ = true;
    helped_ = false;
    try {
      if (helpers) HostWorkers::get().start(job_, (unsigned)helpers), helped_ = true;
    } catch (const std::bad_alloc&) {  // nobody has begun on it: finish() does all of it
    }
    return hipSuccess;
  }

  // What the words of the last begin() follow is done.
  void words_are_there() {
    if (!under_way_ || !transfer_->follows) return;
    transfer_->follows = false;
    announce(transfer_->sent);  // (nobody sends more before that)
  }

  hipError_t finish() {
    if (!under_way_) return hipSuccess;
    Transfer& t = *transfer_;
    words_are_there();  // or will be: who looks for a chunk waits until it comes
    take_part(/*stays=*/true);
    if (helped_) HostWorkers::get().join(job_);
    under_way_ = false;
    if (t.error != hipSuccess) {
      const OnDevice on(t.device);
      for (hipStream_t s : t.streams) (void)hipStreamSynchronize(s);  // nothing writes to the ring after this
      return t.error;
    }
    if (!t.overflow.load()) return hipSuccess;
    misfit_ = true;
    const OnDevice on(t.device);  // the stream may be the default one
    std::vector<Part> parts = t.parts;
    for (Part& p : parts) p.bits = 32;
    return fetch(std::move(parts), t.ready.empty() ? t.streams[0] : transfer_stream(t.device, 0));
  }

  // Nobody wants the words any more.
  void abandon() {
    if (under_way_) transfer_->fail(hipErrorUnknown);
    (void)finish();
  }

  // whether a word has ever not fitted
  bool misfit() const { return misfit_; }
  // launches of the last begin() that was given a `ready` which set out before all of that had happened
  size_t parts_ahead() const { return ahead_.load(std::memory_order_relaxed); }
  // of what it owns through a pointer (nd::engine_abi)
  static constexpr size_t transfer_bytes() { return sizeof(Transfer); }
  // page-locked memory it holds until release()
  size_t page_locked_bytes() const { return ring_bytes_ + headers_held_ * sizeof(PackHeader); }

  void release() {
    (void)finish();
    release_device();
  }

 private:
  void release_device() {
    for (hipEvent_t& ev : packed_)
      if (ev) (void)hipEventDestroy(ev), ev = nullptr;
    release_staging();
    if (begun_) (void)hipEventDestroy(begun_);
    begun_ = nullptr;
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
    ring_bytes_ = 0;
    if (headers_) (void)hipHostFree(headers_);
    headers_ = nullptr;
    headers_held_ = 0;
  }

  // Straight to the host: a ring of as many chunks as there are, or of kRingChunks (64 MB of ids; with twice that the ring no longer stays in the
  // last-level cache between the bus and the threads: 1.68 GB in 16 instead of 14 ms), into which launches of up to
  // kMostChunks go as the threads make room.
  static constexpr size_t kRingChunks = 4096, kMostChunks = 512;
  // Packed in device memory first: pieces in slots; the copy engine rests 8 us between two.  The first one is 1 MB and each of the
  // next twice as long, so that the threads have something to do soon, and none is more than a third of what is left, so that
  // little is left to do when the last one arrives.
  static constexpr size_t kSlots = 8, kMostStagedChunks = 1024;
  static constexpr size_t kBlock = 64;          // chunks that are counted, as they are unpacked, together
  static constexpr size_t kChunksAtOnce = 4;    // what a thread takes; kBlock is a multiple
  static constexpr size_t kFewChunks = kDirectResultBytes / (kPackChunk * sizeof(int32_t)), kChunksAHelper = 32;
  // Workgroups of a launch of pack_results that goes straight to the ring, and launches under way, while something else is
  // computed: stores that wait for the bus stand in the way of that something's own.
  static constexpr uint32_t kGentleBlocks = 32;
  // ... and of one that has the device to itself: enough to keep the bus busy, and no more, so that chunks arrive in about the order the
  // threads look for them in, and not all of them at the end; of more chunks than the ring holds that leave while others are computed
  // (OfMany: the last three) the gaps between launches matter more.  Passes with their rows by workgroups, ms (a workgroup a chunk: walks
  // 0.47, distinct 1.11):
  //                                     32     64     96    128    256
  //     uniform walks 57 K           0.347  0.302  0.336  0.350  0.391
  //     KHop 60 K, distinct          0.951  0.798  0.876  0.913  0.950
  //     MVS 150 K                    1.774  1.739  1.728  1.730  1.785
  //     uniform walks 250 K          1.020  0.984  0.992  1.009  1.048
  //     KHop R-MAT 20 (17 rings)     9.96   9.71   9.65   9.60   9.72
  static constexpr uint32_t kBusBlocks = 64, kBusBlocksOfMany = 128;
  // More chunks in stream order than the ring holds: the ring is filled by one launch, and what is launched beside that takes its part of
  // the bus for chunks that nobody looks for yet.  So the next launch sets out when no more than kChunksAhead are on their way.  Rows
  // of walks keep to kBusBlocks: where many groups are left out it is the threads that take the time, and they want chunks in their
  // order.  Passes with their rows, and (fetch) rows alone, ms, by workgroups (Chung-Lu graphs, a third of the walks' groups left out); with
  // 128 and launches as far ahead as the ring has room; in pieces on two streams, an event for each, as it was before chunks had stamps:
  //                                     64     80     96    128    far ahead   in pieces
  //     uniform walks 170 K          0.762  0.828  0.846  0.872        0.894       0.785
  //                   190 K          0.842  0.908  0.931  0.954        0.963       0.867
  //     DeepWalk 180 K               1.024  1.089  1.102  1.122        1.151       1.043
  //     weighted node2vec 170 K      1.481  1.556  1.558  1.583        1.609       1.480
  //                       230 K      1.788  1.849  1.866  1.891        1.915       1.814
  //     KHop 65 K                    0.959  0.942  0.945  0.972        0.978
  //          85 K                    1.286  1.261  1.244  1.249        1.235       1.327
  //     Layer 85 K                   1.373  1.339  1.325  1.330        1.319       1.410
  //     fetch: KHop 62 K             0.758  0.753  0.759  0.799        0.805       0.770
  //                300 K             3.629  3.599  3.625  3.673        3.768       3.664
  //            MVS 90 K              0.788  0.778  0.787  0.783        0.860
  //            PPR 262 K             0.694  0.698  0.728  0.789        0.826       0.903
  static constexpr uint32_t kBusBlocksInOrder = 96;
  static constexpr size_t kChunksAhead = 1024;
  static constexpr size_t kGentleAhead = 2;
  static constexpr size_t kPackedAhead = 3;     // pieces packed before the copy engine has come to them
  static constexpr int kSignsPerQuery = 1024;   // looks at a sign for one at the event beside it: some 20 us
  static constexpr int kSpins = 4000;  // tens of microseconds; none: 1.68 GB in 19 instead of 13 ms, 23 MB in 527 instead of 290 us

  hipError_t come_to_device_of(hipStream_t stream) {
    int device = 0;
    const hipError_t e = device_of(stream, &device);
    if (e != hipSuccess || device == device_) return e;
    release_device();  // events of one device are not recorded on another's streams
    device_ = device;
    return hipSuccess;
  }

  hipError_t make_ring(size_t bytes) {
    if (ring_bytes_ >= bytes) return hipSuccess;
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
    ring_bytes_ = 0;
    const hipError_t e = hipHostMalloc((void**)&ring_, bytes, hipHostMallocDefault);
    if (e == hipSuccess) ring_bytes_ = bytes;
    return e;
  }

  // Headers have memory of their own: nothing but a stamp is ever where a stamp is looked for.
  hipError_t make_headers(size_t chunks) {
    if (headers_held_ >= chunks) return hipSuccess;
    if (headers_) (void)hipHostFree(headers_);
    headers_ = nullptr;
    headers_held_ = 0;
    const hipError_t e = hipHostMalloc((void**)&headers_, chunks * sizeof(PackHeader), hipHostMallocDefault);
    if (e != hipSuccess) return e;
    memset((void*)headers_, 0, chunks * sizeof(PackHeader));  // the number of no transfer
    headers_held_ = chunks;
    return hipSuccess;
  }

  struct Transfer;
  hipError_t prepare(const Transfer& t) {
    for (hipEvent_t& ev : packed_)
      if (!ev) {
        const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming | hipEventReleaseToSystem);
        if (e != hipSuccess) return e;
      }
    if (!begun_) {
      const hipError_t e = hipEventCreateWithFlags(&begun_, hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    if (t.staged) return make_ring(t.slot_bytes * kSlots);
    // Room for a few chunks more, or for more bits, so that a sampler's other results do not need another ring: to touch one for the
    // first time takes 0.4 ms a MB (MultiRW, rows of 2,442 chunks and states of 2,466: a first pass of 9.5 ms instead of 3.5).
    size_t held = 16;
    while (held < t.ring_chunks) held *= 2;
    const hipError_t e = make_headers(held);
    return e != hipSuccess ? e : make_ring((size_t)kPackChunkGroups * std::max(t.bits, kPackMostBits) * held + kUnpackOverread);
  }

  // What pieces that are packed in device memory take.
  hipError_t prepare_staging(size_t slot_bytes) {
    for (hipEvent_t& ev : copied_)
      if (!ev) {
        const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) return e;
      }
    hipError_t e = hipSuccess;
    if (!totals_) e = hipHostMalloc((void**)&totals_, kSlots * sizeof(uint32_t), hipHostMallocDefault);
    if (e == hipSuccess && !counts_) {
      e = hipMalloc(&counts_, 2 * kSlots * kWordsPerLine * sizeof(uint32_t));
      // on a stream that waits for no computation
      const hipStream_t stream = transfer_stream(device_, 0);
      if (e == hipSuccess) e = hipMemsetAsync(counts_, 0, 2 * kSlots * kWordsPerLine * sizeof(uint32_t), stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
    }
    if (e == hipSuccess && staging_bytes_ < slot_bytes * kSlots) {
      if (staging_) (void)hipFree(staging_);
      staging_ = nullptr;
      staging_bytes_ = 0;
      e = hipMalloc(&staging_, slot_bytes * kSlots);
      if (e == hipSuccess) staging_bytes_ = slot_bytes * kSlots;
    }
    if (e != hipSuccess) release_staging();
    return e;
  }
  void release_staging() {
    for (hipEvent_t& ev : copied_)
      if (ev) (void)hipEventDestroy(ev), ev = nullptr;
    if (totals_) (void)hipHostFree(totals_);
    totals_ = nullptr;
    if (counts_) (void)hipFree(counts_);
    counts_ = nullptr;
    if (staging_) (void)hipFree(staging_);
    staging_ = nullptr;
    staging_bytes_ = 0;
  }

  struct Transfer {
    std::vector<Part> parts;
    std::vector<size_t> part_ends;     // chunks; a chunk is of one part
    uint32_t bits = 0;                 // the most of any part
    bool streaming = false;            // results larger than the caches
    bool sparse = false;               // a part is
    hipStream_t streams[2];
    std::vector<Ready> ready;
    std::vector<size_t> ready_chunks;  // that are there once a `ready` has happened
    bool follows = false;  // and the caller has not said that they are there
    bool staged = false;  // pieces are packed in device memory, for the copy engine, while something else is computed
    int device = 0;

    size_t chunks, chunk_bytes;
    size_t happened;                   // of `ready`
    bool computed;                     // all of it
    // straight
    size_t ring_chunks = 0;
    uint64_t number = 0;
    size_t sent = 0, launches = 0;     // chunks, and what they were sent with
    size_t unpacked_to = 0;            // blocks
    // staged
    size_t pieces = 0, packed_at = 0, slot_bytes = 0;
    std::vector<size_t> begins;        // first chunk of every piece, and the end of the last
    std::vector<uint32_t> piece_of;    // of every block

    std::atomic<bool> driven{false};   // a thread has taken the launching on
    std::atomic<size_t> next{0};       // chunk to take
    std::atomic<size_t> there{0};      // chunks that have been sent (straight), or whose bytes are here (staged)
    std::atomic<bool> stop{false}, overflow{false};
    hipError_t error = hipSuccess;     // the first one
    std::mutex mutex;
    std::condition_variable more;
    unsigned sleepers = 0, gone = 0;   // threads that wait for chunks, and that went back for want of them
    std::vector<std::atomic<size_t>> left;  // chunks of a block that are not unpacked yet

    void set(std::vector<Part> parts_, std::vector<Ready> ready_) {
      parts = std::move(parts_), ready = std::move(ready_);
      staged = !ready.empty() && ready.front().sign != nullptr;
      follows = false;
      happened = 0;
      computed = false;
      chunks = 0;
      bits = 0;
      sparse = false;
      part_ends.clear();
      size_t words = 0;
      for (const Part& p : parts) {
        words += p.n;
        sparse = sparse || p.sparse;
        part_ends.push_back(chunks += (p.n + kPackChunk - 1) / kPackChunk);
        bits = std::max(bits, p.bits > kPackMostBits ? 32 : p.bits);
      }
      streaming = words * sizeof(int32_t) > kDirectResultBytes;
      ready_chunks.clear();
      for (const Ready& r : ready) ready_chunks.push_back(chunks_of(r.words));
      chunk_bytes = (size_t)kPackChunkGroups * bits;
      ring_chunks = std::min(chunks, kRingChunks);
      sent = launches = unpacked_to = 0;
      begins.clear();
      piece_of.clear();
      if (staged) {
        size_t most = kBlock, longest = 0;
        for (size_t at = 0; at < chunks; most = std::min(kMostStagedChunks, most * 2)) {
          const size_t third = ((chunks - at) / 3 + kBlock - 1) / kBlock * kBlock;
          const size_t here = std::max(kBlock, std::min(most, third));
          piece_of.insert(piece_of.end(), here / kBlock, (uint32_t)begins.size());
          begins.push_back(at);
          longest = std::max(longest, here);
          at += here;
        }
        pieces = begins.size();
        begins.push_back(chunks);
        packed_at = sizeof(PackHeader) * longest;
        slot_bytes = (packed_at + chunk_bytes * longest + kUnpackOverread + 255) / 256 * 256;
      }
      driven = false, next = 0, there = 0, stop = false, overflow = false, error = hipSuccess, gone = 0;
      const size_t blocks = (chunks + kBlock - 1) / kBlock;
      left = std::vector<std::atomic<size_t>>(blocks);
      for (size_t b = 0; b < blocks; ++b) left[b].store(std::min(kBlock, chunks - b * kBlock));
    }

    // whole chunks among the first words
    size_t chunks_of(size_t words) const {
      for (size_t p = 0; p < parts.size(); ++p) {
        if (words < parts[p].n) return part_begin(p) + words / kPackChunk;
        words -= parts[p].n;
      }
      return chunks;
    }
    size_t part_begin(size_t p) const { return p == 0 ? 0 : part_ends[p - 1]; }
    size_t part_of(size_t chunk) const {
      size_t p = 0;
      while (part_ends[p] <= chunk) p++;
      return p;
    }

    // (no other chunk's that was or will be where this one is)
    uint64_t stamp(size_t chunk) const { return (number << 32) + chunk; }

    bool here(size_t chunk) const { return there.load(std::memory_order_acquire) > chunk || stop.load(); }
    // Words come every 20-200 us: worth a short wait awake (a thread that sleeps is back 50 us later, and
    // waking all of them costs the driving thread as much), but not more than that.
    bool comes_soon(size_t chunk) const {
      for (int spin = 0; spin < kSpins; ++spin) {
        if (here(chunk)) return true;
        spin_pause();
      }
      return false;
    }
    void await(size_t chunk) {
      if (comes_soon(chunk)) return;
      std::unique_lock<std::mutex> lock(mutex);
      sleepers++;
      more.wait(lock, [&] { return here(chunk); });
      sleepers--;
    }
    // False: it is not here, and who announces the next ones calls a thread back for this one.
    bool here_or_gone(size_t chunk) {
      if (comes_soon(chunk)) return true;
      std::lock_guard<std::mutex> lock(mutex);
      if (here(chunk)) return true;
      gone++;
      return false;
    }
    // Returns how many threads to call back.
    unsigned announce(size_t chunks_there) {
      bool asleep;
      unsigned back;
      {
        std::lock_guard<std::mutex> lock(mutex);
        there.store(chunks_there, std::memory_order_release);
        asleep = sleepers > 0;
        back = gone;
        gone = 0;
      }
      if (asleep) more.notify_all();
      return back;
    }
    void fail(hipError_t e) {
      {
        std::lock_guard<std::mutex> lock(mutex);
        if (error == hipSuccess) error = e;
        stop.store(true);
      }
      (void)hipGetLastError();  // reported by finish(), not to this thread's next launch
      more.notify_all();
    }
  };

  void announce(size_t chunks_there) {
    if (const unsigned back = transfer_->announce(chunks_there)) HostWorkers::get().more(job_, back);
  }

  uint8_t* slot(size_t piece) const { return ring_ + (piece % kSlots) * transfer_->slot_bytes; }

  // (hipEventSynchronize() keeps whoever uses the event's stream otherwise, another transfer's begin() for one, until it has happened.)
  static hipError_t wait_for(hipEvent_t event) {
    hipError_t e;
    while ((e = hipEventQuery(event)) == hipErrorNotReady)
      for (int pause = 0; pause < 32; ++pause) spin_pause();
    return e;
  }

  // Whether the first chunks may be read, or, with `waits`, until they may.
  bool readable(size_t chunks, bool waits, hipError_t* error) {
    Transfer& t = *transfer_;
    while (t.happened < t.ready.size() && (t.happened == 0 || t.ready_chunks[t.happened - 1] < chunks)) {
      const Ready& next = t.ready[t.happened];
      hipError_t e = hipErrorNotReady;
      if (!next.sign) {
        e = waits ? wait_for(next.event) : hipEventQuery(next.event);
      } else {
        for (;;) {
          if (__atomic_load_n(next.sign, __ATOMIC_ACQUIRE) == next.value) e = hipSuccess;
          else if (looks_++ % kSignsPerQuery == 0) e = hipEventQuery(next.event);  // the kernel may have ended, or failed
          if (e != hipErrorNotReady || !waits) break;
          spin_pause();
        }
      }
      if (e == hipErrorNotReady) return false;
      if (e != hipSuccess) {
        *error = e;
        return false;
      }
      t.happened++;
    }
    return true;
  }

  // Whether nothing is being computed any more that the transfer could be in the way of, or ahead of.
  bool computed() {
    Transfer& t = *transfer_;
    if (!t.computed) t.computed = t.ready.empty() || hipEventQuery(t.ready.back().event) == hipSuccess;
    return t.computed;
  }

  uint32_t bus_blocks() const { return transfer_->chunks > transfer_->ring_chunks ? kBusBlocksOfMany : kBusBlocks; }
  uint32_t blocks_in_order() const {
    return transfer_->chunks > transfer_->ring_chunks && !transfer_->sparse ? kBusBlocksInOrder : kBusBlocks;
  }

  // Straight: the chunks from t.sent on, up to `end`, all of one part.
  hipError_t launch(size_t end, uint32_t most_blocks, hipStream_t on) {
    Transfer& t = *transfer_;
    const size_t part = t.part_of(t.sent), first = (t.sent - t.part_begin(part)) * kPackChunk;
    const Part& p = t.parts[part];
    const uint32_t n_chunks = (uint32_t)(end - t.sent);
    const size_t here = std::min(p.n - first, n_chunks * (size_t)kPackChunk);
    PackedOut out{ring_, headers_};
    out.first = (uint32_t)(t.sent % t.ring_chunks);
    out.ring_mask = t.chunks > t.ring_chunks ? (uint32_t)t.ring_chunks - 1u : UINT32_MAX;
    static_assert((kRingChunks & (kRingChunks - 1)) == 0, "a ring that is gone round");
    out.stamp = t.stamp(t.sent);
    pack_results<false><<<dim3(std::min(n_chunks, most_blocks)), dim3(kPackThreads), 0, on>>>(
        p.src + first, here, t.bits, p.fill, out, n_chunks);
    t.launches++;
    t.sent = end;
    return hipGetLastError();
  }

  // Staged: a piece.
  hipError_t launch_piece(size_t piece) {
    const Transfer& t = *transfer_;
    const Part& p = t.parts[0];
    const size_t first = t.begins[piece] * kPackChunk;
    const size_t here = std::min(p.n, t.begins[piece + 1] * kPackChunk) - first, slot_of = piece % kSlots;
    uint8_t* at = staging_ + slot_of * t.slot_bytes;
    const uint32_t n_chunks = (uint32_t)((here + kPackChunk - 1) / kPackChunk);
    PackedOut out{at + t.packed_at, (PackHeader*)at};
    out.cursor = counts_ + 2 * slot_of * kWordsPerLine;
    out.finished = out.cursor + kWordsPerLine;
    out.total = totals_ + slot_of;
    pack_results<true><<<dim3(n_chunks), dim3(kPackThreads), 0, t.streams[0]>>>(p.src + first, here, t.bits, p.fill, out, n_chunks);
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : hipEventRecord(packed_[slot_of], t.streams[0]);
  }

  // Sends a piece that is packed in device memory on its way.
  hipError_t copy_piece(size_t piece) {
    const Transfer& t = *transfer_;
    const size_t slot_of = piece % kSlots;
    const hipStream_t stream = t.streams[1];
    const size_t bytes = t.packed_at + 16 * (size_t)__atomic_load_n(totals_ + slot_of, __ATOMIC_RELAXED);
    const hipError_t e = hipMemcpyAsync(slot(piece), staging_ + slot_of * t.slot_bytes, bytes, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipEventRecord(copied_[slot_of], stream);
  }

  // Straight: waits for a chunk that has been sent.  False: it does not come, or the transfer has failed otherwise.
  bool await_stamp(const PackHeader& header, size_t chunk) {
    Transfer& t = *transfer_;
    const uint64_t stamp = t.stamp(chunk);
    for (int spin = 1;; ++spin) {
      if (__atomic_load_n(&header.stamp, __ATOMIC_ACQUIRE) == stamp) return true;
      if (t.stop.load(std::memory_order_relaxed)) return false;
      if (spin < kSpins) {
        spin_pause();
        continue;
      }
      // long in coming: others are before it on its stream, or the kernel has failed
      const OnDevice on(t.device);
      hipError_t e = on.error;
      for (hipStream_t s : t.streams)
        if (e == hipSuccess) e = hipStreamQuery(s);
      if (e == hipSuccess && __atomic_load_n(&header.stamp, __ATOMIC_ACQUIRE) != stamp) e = hipErrorUnknown;
      if (e != hipSuccess && e != hipErrorNotReady) {
        t.fail(e);
        return false;
      }
      std::this_thread::sleep_for(std::chrono::microseconds(20));
    }
  }

  // Unpacks the chunks [c, end) of a block, which have been sent, or (staged) are here.
  void unpack(size_t c, size_t end) {
    Transfer& t = *transfer_;
    const size_t piece = t.staged ? t.piece_of[c / kBlock] : 0;
    const PackHeader* headers = t.staged ? (const PackHeader*)slot(piece) + (c - t.begins[piece]) : headers_ + c % t.ring_chunks;
    const uint8_t* bytes = t.staged ? slot(piece) + t.packed_at : ring_ + (c % t.ring_chunks) * t.chunk_bytes;
    // Where a chunk's bytes are is read for all of them first, and only if it has to be: to wait for a header that has just
    // crossed the bus before every chunk cost 4 % of KHop's rows over R-MAT 20.
    size_t bytes_at[kChunksAtOnce];
    for (size_t i = 0; i < end - c; ++i) bytes_at[i] = t.staged ? headers[i].at : i * t.chunk_bytes;
    for (size_t i = 0; i < end - c; ++i) {
      if (!t.staged && !await_stamp(headers[i], c + i)) return;
      if (headers[i].overflow) {
        t.overflow.store(true, std::memory_order_relaxed);
        continue;
      }
      const size_t part = t.part_of(c + i), first = (c + i - t.part_begin(part)) * kPackChunk;
      const Part& p = t.parts[part];
      unpack_chunk(headers[i], bytes + bytes_at[i], p.fill, p.dst + first, std::min<size_t>(kPackChunk, p.n - first), t.streaming);
    }
    unpack_fence();
    t.left[c / kBlock].fetch_sub(end - c, std::memory_order_release);
  }

  // Has all of it packed, if nobody does yet, and unpacks what is there.  A thread that does not stay holds no chunk that is not, and is
  // free for other transfers until there are some: a pass may take long, and there are no more than kMost threads for all samplers.
  void take_part(bool stays) {
    Transfer& t = *transfer_;
    for (;;) {
      // (what follows something has nothing to be driven before it is there)
      if (!t.driven.load(std::memory_order_relaxed) && (!t.ready.empty() || t.there.load() != 0) && !t.driven.exchange(true)) drive();
      const size_t c = t.next.load();
      if (c >= t.chunks || t.stop.load()) return;
      if (unpack_some()) continue;
      const size_t last = std::min(c + kChunksAtOnce, t.chunks) - 1;
      if (stays) t.await(last);
      else if (!t.here_or_gone(last)) return;
    }
  }

  // Some of what is there, if anything is that nobody has taken.
  bool unpack_some() {
    Transfer& t = *transfer_;
    size_t c = t.next.load(), end;
    do {
      end = std::min(c + kChunksAtOnce, t.chunks);
      if (c >= t.chunks || t.there.load(std::memory_order_acquire) < end) return false;
    } while (!t.next.compare_exchange_weak(c, c + kChunksAtOnce));
    unpack(c, end);
    return true;
  }

  // Has all of it packed and announces it as it sets out, or arrives.
  void drive() {
    Transfer& t = *transfer_;
    const OnDevice on(t.device);
    hipError_t error = on.error;
    if (error == hipSuccess) error = t.staged ? drive_staged() : drive_straight();
    if (error != hipSuccess) t.fail(error);
  }

  // Launches one after another as words become readable and the threads make room in the ring; few, and of few workgroups, while
  // something is computed.
  hipError_t drive_straight() {
    Transfer& t = *transfer_;
    hipError_t error = hipSuccess;
    bool gently = !t.ready.empty(), ordered = gently;
    size_t gentle = 0, gone = 0;  // launches of those, and how many of them have ended
    while (t.sent < t.chunks && error == hipSuccess && !t.stop.load(std::memory_order_relaxed)) {
      gently = gently && !computed();
      while (gone < gentle && (error = hipEventQuery(packed_[gone % kSlots])) == hipSuccess) gone++;
      if (error == hipErrorNotReady) error = hipSuccess;
      if (error != hipSuccess) break;
      while (t.unpacked_to < t.left.size() && t.left[t.unpacked_to].load(std::memory_order_acquire) == 0) t.unpacked_to++;
      const bool in_order = t.ready.empty();
      const size_t unpacked = std::min(t.chunks, t.unpacked_to * kBlock), room = std::min(t.chunks, unpacked + t.ring_chunks);
      // up to the end of what may be read, if that is known, else a piece at a time
      size_t end = std::min(t.chunks, t.sent + kMostChunks);
      if (!in_order) {
        if (!readable(t.sent + 1, /*waits=*/t.next.load() >= t.sent && gone == gentle, &error)) {
          if (error == hipSuccess && !unpack_some()) spin_pause();
          continue;
        }
        end = std::min(t.ready_chunks[t.happened - 1], gently || t.chunks > t.ring_chunks ? t.sent + kMostChunks : t.chunks);
      }
      end = std::min(end, t.part_ends[t.part_of(t.sent)]);
      if (end > room || (gently && gentle - gone >= kGentleAhead) || (in_order && t.sent > unpacked + kChunksAhead)) {
        if (!unpack_some()) std::this_thread::yield();
        continue;
      }
      // Two streams, so that the bus is not idle between two launches.  Words in stream order are there by now, as chunks behind them
      // have arrived: nobody waits for that event.
      if (!ordered && (error = hipStreamWaitEvent(t.streams[1], begun_, 0)) != hipSuccess) break;
      ordered = true;
      if (gently) ahead_.fetch_add(1, std::memory_order_relaxed);
      const hipStream_t stream = t.streams[t.launches % 2];
      error = launch(end, gently ? kGentleBlocks : in_order ? blocks_in_order() : bus_blocks(), stream);
      if (error == hipSuccess && gently) error = hipEventRecord(packed_[gentle++ % kSlots], stream);
      if (error == hipSuccess) announce(t.sent);
    }
    return error;
  }

  // A few pieces packed ahead of the copy engine, as they become readable and as slots become free.
  hipError_t drive_staged() {
    Transfer& t = *transfer_;
    size_t launched = 0, sent = 0, here = 0;
    while (here < t.pieces && !t.stop.load(std::memory_order_relaxed)) {
      hipError_t e = hipSuccess;
      bool moved = false;
      if (launched < t.pieces && launched < sent + kPackedAhead && readable(t.begins[launched + 1], /*waits=*/here == launched, &e) &&
          slot_is_free(launched)) {
        if (!computed()) ahead_.fetch_add(1, std::memory_order_relaxed);
        e = launch_piece(launched++);
        moved = true;
      }
      if (e != hipSuccess) return e;
      if (sent < launched && (e = hipEventQuery(packed_[sent % kSlots])) != hipErrorNotReady) {
        if (e == hipSuccess) e = copy_piece(sent++);
        if (e != hipSuccess) return e;
        moved = true;
      }
      if (here < sent && (e = hipEventQuery(copied_[here % kSlots])) != hipErrorNotReady) {
        if (e != hipSuccess) return e;
        announce(t.begins[++here]);
        moved = true;
      }
      if (!moved) spin_pause();
    }
    return hipSuccess;
  }

  // Whether a piece's slot is free: the piece before it there is unpacked.  If not, does some of that.
  bool slot_is_free(size_t piece) {
    Transfer& t = *transfer_;
    if (piece < kSlots) return true;
    for (size_t b = t.begins[piece - kSlots] / kBlock; b * kBlock < t.begins[piece - kSlots + 1]; ++b)
      if (t.left[b].load(std::memory_order_acquire) != 0) {
        if (!unpack_some()) std::this_thread::yield();
        return false;
      }
    return true;
  }

  std::unique_ptr<Transfer> transfer_;
  HostWorkers::Job job_;
  bool under_way_ = false, helped_ = false, misfit_ = false;
  int device_ = -1;  // of the events and the ring
  uint32_t looks_ = 0;
  std::atomic<size_t> ahead_{0};  // parts_ahead()
  uint64_t transfers_ = 0;
  uint8_t* ring_ = nullptr;
  size_t ring_bytes_ = 0;
  PackHeader* headers_ = nullptr;  // straight
  size_t headers_held_ = 0;
  hipEvent_t packed_[kSlots] = {}, begun_ = nullptr;
  // of pieces that are packed in device memory
  static constexpr size_t kWordsPerLine = 32;
  hipEvent_t copied_[kSlots] = {};
  uint8_t* staging_ = nullptr;
  size_t staging_bytes_ = 0;
  uint32_t *counts_ = nullptr, *totals_ = nullptr;
};

}  // namespace nd
