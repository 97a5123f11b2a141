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
//    engine's 57, without a launch and a copy per piece), and host threads unpack a piece
//    while the next one crosses.  Twelve threads write 220 GB/s of unpacked ids on the 16-core share of a
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

  // Work that several threads may take part in: each calls body() once, and every body() has to be able to
  // do all of it alone, and must not throw.  A Job stays where it is from start() to join().
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

// Results up to this size go through page-locked memory by the copy engine and one thread, above it they are packed and
// streamed by several.  Copied / streamed with ids of 12 and of 32 bits, us: 0.5 MB 31 / 75, 82; 1.1 MB 67 / 95, 105;
// 1.5 MB 92 / 100, 116; 2 MB 118 / 110, 128; 3 MB 169 / 121, 155; 4 MB 220 / 113, 158.
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

// What a chunk's groups are: which of them hold anything but `fill` (bit g of word g / 64), and whether an id
// did not fit its bits.
struct PackHeader {
  uint64_t live[kPackChunkGroups / 64];
  uint64_t overflow;
  uint64_t at;  // of its bytes among the piece's, if staged
  uint64_t pad[6];
};

// Where the chunks' bytes go: chunk after chunk, each as far from the last as a whole one takes, or (staged) one directly
// after another, in whatever order the workgroups get there, for a copy that is to take no more than there is.
struct PackedOut {
  uint8_t* bytes;
  PackHeader* headers;
  // staged
  uint32_t* cursor = nullptr;    // 16 bytes each; 0 before the launch and after it
  uint32_t* finished = nullptr;  // workgroups; likewise
  uint32_t* total = nullptr;     // host memory: what cursor was at the end
};

// Packs ids [chunk * kPackChunk, ...) of src into out[chunk * kPackChunkGroups * bits ...): the groups of
// eight that are not all `fill`, back to back, `bits` bytes each.  Where out is host memory the
// stores to it are what takes the time (54.7 GB/s of packed bytes; packing the 1.68 GB of R-MAT 22 walks into
// device memory instead takes a twentieth of it), hence whole chunks through LDS and 16-byte stores by
// consecutive lanes; nothing else here is tuned.  (kStaged is the kernel's and not the launch's: with both forms' loads in one
// kernel those of a chunk wait for each other, and MultiRW 100 K took 1.59 ms instead of 1.55, KHop over R-MAT 20 11.7 instead
// of 11.4.)
template <bool kStaged>
__global__ __launch_bounds__(kPackThreads) void pack_results(const int32_t* __restrict__ src, size_t n, uint32_t bits,
                                                             int32_t fill, PackedOut out, uint32_t n_chunks) {
  __shared__ __align__(16) uint8_t s_packed[kPackChunk * sizeof(int32_t)];
  __shared__ uint64_t s_live[kPackChunkGroups / 64];
  __shared__ uint32_t s_at;
  constexpr uint32_t kRounds = kPackChunkGroups / kPackThreads;
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t chunk = blockIdx.x; chunk < n_chunks; chunk += gridDim.x) {
    const size_t first = (size_t)chunk * kPackChunk;
    int32_t ids[kRounds][kPackGroup];
    bool live[kRounds];
    bool overflow = false;
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
      live[r] = false;
#pragma unroll
      for (uint32_t i = 0; i < kPackGroup; ++i) live[r] = live[r] || ids[r][i] != fill;
      const uint64_t mask = __ballot(live[r]);
      if (lane == 0) s_live[(r * kPackThreads + threadIdx.x) / 64u] = mask;
      if (bits < 32 && live[r]) {
        if (at + kPackGroup > n)  // what fills the last group up need not fit
#pragma unroll
          for (uint32_t i = 0; i < kPackGroup; ++i) ids[r][i] = at + i < n ? ids[r][i] : 0;
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
    const uint32_t words = (total * bits + 15u) / 16u;
    if (kStaged && threadIdx.x == 0) s_at = atomicAdd(out.cursor, words);
    __syncthreads();
    const size_t at = kStaged ? (size_t)s_at * 16u : (size_t)chunk * kPackChunkGroups * bits;
    uint8_t* chunk_out = out.bytes + at;
    for (uint32_t i = threadIdx.x; i < words; i += kPackThreads)
      reinterpret_cast<uint4*>(chunk_out)[i] = reinterpret_cast<const uint4*>(s_packed)[i];
    if (threadIdx.x < kPackChunkGroups / 64) out.headers[chunk].live[threadIdx.x] = s_live[threadIdx.x];
    if (threadIdx.x == kPackChunkGroups / 64) {
      out.headers[chunk].overflow = (uint64_t)any_overflow;
      if (kStaged) out.headers[chunk].at = at;
    }
    __syncthreads();  // the next chunk overwrites what has just been read
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
};

// Bytes the unpacking may read past the last group of a chunk.
constexpr size_t kUnpackOverread = 32;

// One chunk to dst (kPackChunk ids).
inline void unpack_chunk_plain(const UnpackPlan& plan, const PackHeader& header, const uint8_t* src, int32_t fill,
                               int32_t* dst) {
  for (uint32_t g = 0; g < kPackChunkGroups; ++g, dst += kPackGroup) {
    if (!(header.live[g / 64] >> (g % 64) & 1u)) {
      std::fill_n(dst, kPackGroup, fill);
      continue;
    }
    for (uint32_t i = 0; i < kPackGroup; ++i) {
      uint64_t word = 0;
      memcpy(&word, src + ((i * plan.bits) >> 3), plan.bits > kPackMostBits ? sizeof(uint32_t) : sizeof(word));
      dst[i] = (int32_t)((uint32_t)(word >> ((i * plan.bits) & 7u)) & plan.mask);
    }
    src += plan.bits;
  }
}

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
// The same with dst a multiple of 32 bytes.  Streaming stores: the result is written once and read by nobody here, and
// a line that is not fetched before it is overwritten is half the memory traffic.  Words of 64 live groups, and of 64
// dead ones, have loops of their own; in a mixed word every group is unpacked from where the next live one
// starts and replaced by `fill` if it is not live itself - no branch to mispredict where walks end at random.
// Eight threads: 200 GB/s of ids (76-100 with a call for every run of groups of one kind).
__attribute__((target("avx2"))) inline void unpack_chunk_avx2(const UnpackPlan& plan, const PackHeader& header,
                                                              const uint8_t* src, int32_t fill, int32_t* dst) {
  const bool whole = plan.bits > kPackMostBits;
  const size_t bits = plan.bits;
  const __m256i shuffle = _mm256_loadu_si256((const __m256i*)plan.shuffle);
  const __m256i shift = _mm256_loadu_si256((const __m256i*)plan.shift);
  const __m256i mask = _mm256_set1_epi32((int)plan.mask), dead = _mm256_set1_epi32(fill);
  const size_t high_at = plan.high_at;
#define ND_UNPACKED_GROUP                                                                                          \
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
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup) _mm256_stream_si256((__m256i*)dst, dead);
    } else if (whole) {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup, live >>= 1) {
        const __m256i here = _mm256_set1_epi32(-(int)(live & 1u));
        _mm256_stream_si256((__m256i*)dst, _mm256_blendv_epi8(dead, _mm256_loadu_si256((const __m256i*)src), here));
        src += bits & (0 - (size_t)(live & 1u));
      }
    } else if (~live == 0) {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup, src += bits)
        _mm256_stream_si256((__m256i*)dst, ND_UNPACKED_GROUP);
    } else {
      for (uint32_t g = 0; g < 64; ++g, dst += kPackGroup, live >>= 1) {
        const __m256i here = _mm256_set1_epi32(-(int)(live & 1u));
        _mm256_stream_si256((__m256i*)dst, _mm256_blendv_epi8(dead, ND_UNPACKED_GROUP, here));
        src += bits & (0 - (size_t)(live & 1u));
      }
    }
  }
#undef ND_UNPACKED_GROUP
}
inline bool unpack_has_avx2() { return __builtin_cpu_supports("avx2"); }
inline void unpack_fence() { _mm_sfence(); }
inline void spin_pause() { _mm_pause(); }
#else
inline void unpack_chunk_avx2(const UnpackPlan&, const PackHeader&, const uint8_t*, int32_t, int32_t*) {}
inline bool unpack_has_avx2() { return false; }
inline void unpack_fence() {}
inline void spin_pause() {}
#endif

// The first count ids (at most kPackChunk) of a chunk to dst.
inline void unpack_chunk(const UnpackPlan& plan, const PackHeader& header, const uint8_t* src, int32_t fill,
                         int32_t* dst, size_t count) {
  alignas(32) int32_t part[kPackChunk];
  int32_t* at = count == kPackChunk ? dst : part;
  if (((uintptr_t)at & 31u) == 0 && unpack_has_avx2()) unpack_chunk_avx2(plan, header, src, fill, at);
  else unpack_chunk_plain(plan, header, src, fill, at);
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

// The streams results cross the bus on while something else is computed: two or three per device (which has to be the current one) and process, each on
// a hardware queue of its own, which a stream with a mask of compute units (here: all) gets.  (Ordinary streams share
// four; where the computation's lands on the same one, nothing overlaps.)  What each is for: StreamUse.  They are destroyed when the process ends, while
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
constexpr size_t kTransferStreams = 3;  // of a device, at most
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

// What a transfer may use besides the first of its device's streams, on which nothing ever waits for a computation: all the
// samplers of the process share it, and what others put there would wait as well.  The second is either one transfer's that
// has it wait for its computation, or packs pieces for any number that do not; who wants to pack while somebody waits
// there does so on a third.  (Not a stream for each from the start: uniform walks 57 K, whose rows wait for them, 0.35 ms, 0.40
// on the third such stream of a process.)
class StreamUse {
 public:
  StreamUse() = default;
  StreamUse(const StreamUse&) = delete;
  StreamUse& operator=(const StreamUse&) = delete;
  ~StreamUse() { give_back(); }

  // the second one, for waiting: false if it is in use
  bool wait(int device) {
    give_back();
    int nobody = 0;
    if ((unsigned)device >= kDevices || !users(device).compare_exchange_strong(nobody, -1)) return false;
    device_ = device, held_ = -1;
    return true;
  }
  // the one to pack on
  size_t pack(int device) {
    give_back();
    if ((unsigned)device >= kDevices) return 1;  // nobody waits there
    for (int now = users(device).load();;) {
      if (now < 0) return 2;
      if (users(device).compare_exchange_weak(now, now + 1)) break;
    }
    device_ = device, held_ = 1;
    return 1;
  }
  // nothing of the transfer is on it any more
  void give_back() {
    if (held_ != 0) users(device_).fetch_sub(held_);
    held_ = 0;
  }

 private:
  static constexpr unsigned kDevices = 64;
  static std::atomic<int>& users(int device) {  // of the second stream; -1: one that waits
    static std::atomic<int> all[kDevices] = {};
    return all[device];
  }
  int device_ = 0, held_ = 0;
};

// Brings words of device memory to the host, packed on the way.  One caller at a time.  Everything happens on the device of the
// stream that is given, whatever the calling thread's current device is, and leaves that as it was.
class ResultStream {
 public:
  ResultStream() = default;
  ResultStream(const ResultStream&) = delete;
  ResultStream& operator=(const ResultStream&) = delete;
  ~ResultStream() { release(); }

  // The first `words` words of a result are on the device once `event` has happened, or, if there is a `sign` (all of a
  // transfer's have one or none has; page-locked memory a kernel that is still running writes to, after the words), once that is
  // `value`.
  struct Ready {
    size_t words;
    hipEvent_t event;
    const uint32_t* sign = nullptr;
    uint32_t value = 0;
  };

  // Takes, on the current device and ahead of the first, what a copy() or a fetch() of n words needs.
  hipError_t reserve(size_t n, uint32_t bits) {
    hipError_t e = finish();
    if (e == hipSuccess) e = come_to_device_of(nullptr);
    if (e != hipSuccess) return e;
    if (n * sizeof(int32_t) <= kDirectResultBytes) {
      e = make_ring(kDirectResultBytes);
    } else {
      if (!transfer_) transfer_.reset(new Transfer);
      transfer_->set(nullptr, n, bits > kPackMostBits ? 32 : bits, 0, nullptr, {});
      e = prepare(transfer_->slot_bytes);
    }
    if (e == hipSuccess) memset(ring_, 0, ring_bytes_);  // its pages are mapped when they are first touched: 0.8 ms of 2 MB
    return e;
  }

  // bytes at src to dst as they are, in stream order, complete on return.  For few of them, and for what is not words.
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

  // n words at src (aligned to 16 bytes) to dst, in stream order.  Words that are `fill` in groups of eight cost
  // nothing; words are expected to fit `bits` bits (one that does not makes the whole transfer start again with
  // 32).  Large transfers only: it pays from a few megabytes on.
  hipError_t fetch(const int32_t* src, size_t n, uint32_t bits, int32_t fill, int32_t* dst, hipStream_t stream) {
    const hipError_t e = begin(src, n, bits, fill, dst, stream, {});
    return e == hipSuccess ? finish() : e;
  }

  // The same as a begin() that returns at once, other threads taking it from there, and a finish() that takes part
  // and returns when the words are at dst.  `ready` (words ascending, the last n): what has to have
  // happened before words may be read, while other work of the caller's is still going on; empty: stream order.  What is given has to stay until finish().
  hipError_t begin(const int32_t* src, size_t n, uint32_t bits, int32_t fill, int32_t* dst, hipStream_t stream,
                   std::vector<Ready> ready) {
    hipError_t e = finish();  // an earlier one that nobody waited for
    use_.give_back();
    if (e != hipSuccess || n == 0) return e;
    if (!transfer_) transfer_.reset(new Transfer);
    Transfer& t = *transfer_;
    e = come_to_device_of(stream);
    if (e != hipSuccess) return e;
    t.device = device_;
    const OnDevice on(t.device);
    if (on.error != hipSuccess) return on.error;
    t.set(src, n, bits > kPackMostBits ? 32 : bits, fill, dst, std::move(ready));
    e = prepare(t.slot_bytes);
    if (e == hipSuccess && t.staged) e = prepare_staging(t.slot_bytes);
    if (e != hipSuccess) return e;
    t.streams[0] = t.streams[1] = transfer_stream(t.device, 0);
    // all words at once: the device waits for them, without a way over a thread, if it can
    t.device_waits = t.ready.size() == 1 && !t.staged && use_.wait(t.device);
    if (t.device_waits) t.streams[0] = t.streams[1] = transfer_stream(t.device, 1);
    if (t.staged) t.streams[0] = transfer_stream(t.device, use_.pack(t.device));
    if (t.ready.empty()) {
      // pieces alternate between two streams, so that the bus is not idle between two of them
      t.streams[0] = stream;
      e = hipEventRecord(begun_, stream);
      if (e == hipSuccess) e = hipStreamWaitEvent(t.streams[1], begun_, 0);
      if (e != hipSuccess) return e;
    }
    if (!t.ready.empty()) ahead_.store(0, std::memory_order_relaxed);
    job_.body = [this] { take_part(); };
    HostWorkers::get().start(job_, HostWorkers::kMost);
    under_way_ = true;  // (not if start() throws: nobody has begun on it then)
    return hipSuccess;
  }

  hipError_t finish() {
    if (!under_way_) return hipSuccess;
    Transfer& t = *transfer_;
    take_part();
    HostWorkers::get().join(job_);
    under_way_ = false;
    if (t.error != hipSuccess) {
      const OnDevice on(t.device);
      for (hipStream_t s : t.streams) (void)hipStreamSynchronize(s);  // nothing writes to the ring after this
    }
    use_.give_back();
    if (t.error != hipSuccess) return t.error;
    if (!t.overflow.load()) return hipSuccess;
    misfit_ = true;
    const OnDevice on(t.device);  // the stream may be the default one
    return fetch(t.src, t.n, 32, t.fill, t.dst, t.ready.empty() ? t.streams[0] : transfer_stream(t.device, 0));
  }

  // whether a word has ever not fitted
  bool misfit() const { return misfit_; }
  // pieces of the last begin() that was given a `ready` which set out before all of that had happened
  size_t parts_ahead() const { return ahead_.load(std::memory_order_relaxed); }
  // of what it owns through a pointer (nd::engine_abi)
  static constexpr size_t transfer_bytes() { return sizeof(Transfer); }
  // page-locked memory it holds until release()
  size_t page_locked_bytes() const { return ring_bytes_; }

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
  }

  static constexpr size_t kSlots = 8;
  // Chunks of a piece: at most 8 MB of results (0.1 ms on the bus, long against a launch and an event; with pieces of
  // 16 MB the ring no longer stays in the last-level cache between the bus and the threads: 1.68 GB in 16 instead of 14
  // ms; the copy engine, which rests 8 us between two copies, gets 16 MB all the same).  The first one is 1 MB and each of the next twice as long, so that the threads have something to do soon, and
  // none is more than a third of what is left, so that little is left to do when the last one arrives.
  static constexpr size_t kMostChunks = 512, kMostStagedChunks = 1024, kLeastChunks = 64;
  static constexpr size_t kChunksAtOnce = 4;  // what a thread takes; kLeastChunks is a multiple
  // Workgroups of a launch of pack_results that goes straight to the ring, and launches under way, while something else is
  // computed: stores that wait for the bus stand in the way of that something's own.
  static constexpr uint32_t kGentleBlocks = 32;
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

  hipError_t prepare(size_t slot_bytes) {
    for (hipEvent_t& ev : packed_)
      if (!ev) {
        const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming | hipEventReleaseToSystem);
        if (e != hipSuccess) return e;
      }
    if (!begun_) {
      const hipError_t e = hipEventCreateWithFlags(&begun_, hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    return make_ring(slot_bytes * kSlots);
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
    const int32_t* src;
    size_t n;
    uint32_t bits;
    int32_t fill;
    int32_t* dst;
    hipStream_t streams[2];
    std::vector<Ready> ready;
    bool staged = false;  // pieces are packed in device memory, for the copy engine, while something else is computed
    bool device_waits = false;
    int device = 0;

    size_t chunks, pieces, chunk_bytes, packed_at, slot_bytes;
    std::vector<size_t> begins;        // first chunk of every piece, and the end of the last
    std::vector<uint32_t> piece_of;    // of every kLeastChunks chunks
    size_t happened;                   // of `ready`
    bool computed;                     // all of it
    UnpackPlan plan{32};
    std::atomic<bool> driven{false};   // a thread has taken the launching on
    std::atomic<size_t> next{0};       // chunk to take
    std::atomic<size_t> arrived{0};    // pieces whose bytes are here
    std::atomic<bool> stop{false}, overflow{false};
    hipError_t error = hipSuccess;     // the driving thread's
    std::mutex mutex;
    std::condition_variable more;
    unsigned sleepers = 0;
    std::vector<std::atomic<size_t>> left;  // chunks of a piece that are not unpacked yet

    void set(const int32_t* src_, size_t n_, uint32_t bits_, int32_t fill_, int32_t* dst_, std::vector<Ready> ready_) {
      src = src_, n = n_, bits = bits_, fill = fill_, dst = dst_, ready = std::move(ready_);
      staged = !ready.empty() && ready.front().sign != nullptr;
      happened = 0;
      computed = false;
      chunks = (n + kPackChunk - 1) / kPackChunk;
      begins.clear();
      piece_of.clear();
      size_t most = kLeastChunks, longest = 0;
      for (size_t at = 0; at < chunks; most = std::min(staged ? kMostStagedChunks : kMostChunks, most * 2)) {
        const size_t third = ((chunks - at) / 3 + kLeastChunks - 1) / kLeastChunks * kLeastChunks;
        const size_t here = std::max(kLeastChunks, std::min(most, third));
        piece_of.insert(piece_of.end(), here / kLeastChunks, (uint32_t)begins.size());
        begins.push_back(at);
        longest = std::max(longest, here);
        at += here;
      }
      pieces = begins.size();
      begins.push_back(chunks);
      chunk_bytes = (size_t)kPackChunkGroups * bits;
      packed_at = sizeof(PackHeader) * longest;
      slot_bytes = (packed_at + chunk_bytes * longest + kUnpackOverread + 255) / 256 * 256;
      plan = UnpackPlan(bits);
      driven = false, next = 0, arrived = 0, stop = false, overflow = false, error = hipSuccess;
      left = std::vector<std::atomic<size_t>>(pieces);
      for (size_t p = 0; p < pieces; ++p) left[p].store(begins[p + 1] - begins[p]);
    }

    // A piece comes every 20-200 us: worth a short wait awake (a thread that sleeps is back 50 us later, and
    // waking all of them costs the driving thread as much), but not more than that.
    void await(size_t piece) {
      for (int spin = 0; spin < kSpins; ++spin) {
        if (arrived.load(std::memory_order_acquire) > piece || stop.load()) return;
        spin_pause();
      }
      std::unique_lock<std::mutex> lock(mutex);
      sleepers++;
      more.wait(lock, [&] { return arrived.load(std::memory_order_acquire) > piece || stop.load(); });
      sleepers--;
    }
    void announce(size_t pieces_here, bool stops) {
      bool asleep;
      {
        std::lock_guard<std::mutex> lock(mutex);
        if (stops) stop.store(true);
        else arrived.store(pieces_here, std::memory_order_release);
        asleep = sleepers > 0;
      }
      if (asleep) more.notify_all();
    }
  };

  uint8_t* slot(size_t piece) const { return ring_ + (piece % kSlots) * transfer_->slot_bytes; }
  size_t piece_end(size_t piece) const {
    return std::min(transfer_->n, transfer_->begins[piece + 1] * kPackChunk);
  }

  // Whether piece may be read, or, with `waits`, until it may.
  bool readable(size_t piece, bool waits, hipError_t* error) {
    Transfer& t = *transfer_;
    while (t.happened < t.ready.size() && (t.happened == 0 || t.ready[t.happened - 1].words < piece_end(piece))) {
      const Ready& next = t.ready[t.happened];
      hipError_t e = hipErrorNotReady;
      if (!next.sign) {
        e = waits ? hipEventSynchronize(next.event) : hipEventQuery(next.event);
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

  hipError_t launch(size_t piece, uint32_t most_blocks = UINT32_MAX) {
    const Transfer& t = *transfer_;
    const size_t first = t.begins[piece] * kPackChunk;
    const size_t here = piece_end(piece) - first, slot_of = piece % kSlots;
    uint8_t* at = t.staged ? staging_ + slot_of * t.slot_bytes : slot(piece);
    const uint32_t n_chunks = (uint32_t)((here + kPackChunk - 1) / kPackChunk);
    const hipStream_t stream = t.streams[t.staged ? 0 : piece % 2];  // (a copy on it would be waited for)
    PackedOut out{at + t.packed_at, (PackHeader*)at};
    if (t.staged) {
      out.cursor = counts_ + 2 * slot_of * kWordsPerLine;
      out.finished = out.cursor + kWordsPerLine;
      out.total = totals_ + slot_of;
    }
    const dim3 grid(std::min(n_chunks, most_blocks)), block(kPackThreads);
    if (t.staged) pack_results<true><<<grid, block, 0, stream>>>(t.src + first, here, t.bits, t.fill, out, n_chunks);
    else pack_results<false><<<grid, block, 0, stream>>>(t.src + first, here, t.bits, t.fill, out, n_chunks);
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : hipEventRecord(packed_[slot_of], stream);
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

  // unpacks the chunks [c, end) of a piece that is here
  void unpack(size_t c, size_t end) {
    Transfer& t = *transfer_;
    const size_t piece = t.piece_of[c / kLeastChunks];
    const uint8_t* at = slot(piece);
    const PackHeader* headers = (const PackHeader*)at + (c - t.begins[piece]);
    // Where a chunk's bytes are is read for all of them first, and only if it has to be: to wait for a header that has just
    // crossed the bus before every chunk cost 4 % of KHop's rows over R-MAT 20.
    size_t bytes_at[kChunksAtOnce];
    for (size_t i = 0; i < end - c; ++i) bytes_at[i] = t.staged ? headers[i].at : (c - t.begins[piece] + i) * t.chunk_bytes;
    for (size_t i = 0; i < end - c; ++i) {
      if (headers[i].overflow) t.overflow.store(true, std::memory_order_relaxed);
      const size_t first = (c + i) * kPackChunk;
      unpack_chunk(t.plan, headers[i], at + t.packed_at + bytes_at[i], t.fill, t.dst + first, std::min<size_t>(kPackChunk, t.n - first));
    }
    unpack_fence();
    t.left[piece].fetch_sub(end - c, std::memory_order_release);
  }

  void take_part() {
    Transfer& t = *transfer_;
    if (!t.driven.exchange(true)) drive();
    for (;;) {
      const size_t c = t.next.fetch_add(kChunksAtOnce);
      if (c >= t.chunks) return;
      const size_t piece = t.piece_of[c / kLeastChunks];
      t.await(piece);
      if (t.stop.load()) return;
      unpack(c, std::min(c + kChunksAtOnce, t.chunks));
    }
  }

  // Whether a piece's slot is free: the piece before it there is unpacked.  If not, does some of that (of pieces that are here).
  bool slot_is_free(size_t piece, size_t here) {
    Transfer& t = *transfer_;
    if (piece < kSlots || t.left[piece - kSlots].load(std::memory_order_acquire) == 0) return true;
    size_t c = t.next.load();
    if (c < t.begins[here] && t.next.compare_exchange_strong(c, c + kChunksAtOnce)) unpack(c, std::min(c + kChunksAtOnce, t.chunks));
    else std::this_thread::yield();
    return false;
  }

  // Has all pieces packed and announces them as they arrive.
  void drive() {
    Transfer& t = *transfer_;
    const OnDevice on(t.device);
    hipError_t error = on.error;
    if (error == hipSuccess) error = t.staged ? drive_staged() : drive_straight();
    if (error != hipSuccess) {
      t.error = error;
      (void)hipGetLastError();  // reported by finish(), not to this thread's next launch
      t.announce(0, true);
    }
  }

  // Up to kSlots pieces under way at a time, straight to the ring; few, and of few workgroups, while something is computed.
  hipError_t drive_straight() {
    Transfer& t = *transfer_;
    hipError_t error = hipSuccess;
    size_t launched = 0;
    bool gently = !t.ready.empty();
    if (t.device_waits) {
      error = hipStreamWaitEvent(t.streams[0], t.ready[0].event, 0);
      t.happened = 1;
      gently = false;
    }
    for (size_t p = 0; p < t.pieces && error == hipSuccess; ++p) {
      while (launched < t.pieces && error == hipSuccess && readable(launched, /*waits=*/launched == p, &error)) {
        gently = gently && !computed();
        if (launched >= p + (gently ? kGentleAhead : kSlots)) break;
        while (!slot_is_free(launched, p)) {}
        if (gently) ahead_.fetch_add(1, std::memory_order_relaxed);
        error = launch(launched++, gently ? kGentleBlocks : UINT32_MAX);
      }
      if (error == hipSuccess) error = hipEventSynchronize(packed_[p % kSlots]);
      if (error == hipSuccess) t.announce(p + 1, false);
    }
    return error;
  }

  // A few pieces packed ahead of the copy engine, as they become readable and as slots become free.
  hipError_t drive_staged() {
    Transfer& t = *transfer_;
    size_t launched = 0, sent = 0, here = 0;
    while (here < t.pieces) {
      hipError_t e = hipSuccess;
      bool moved = false;
      if (launched < t.pieces && launched < sent + kPackedAhead && readable(launched, /*waits=*/here == launched, &e) &&
          slot_is_free(launched, here)) {
        if (!computed()) ahead_.fetch_add(1, std::memory_order_relaxed);
        e = launch(launched++);
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
        t.announce(++here, false);
        moved = true;
      }
      if (!moved) spin_pause();
    }
    return hipSuccess;
  }

  std::unique_ptr<Transfer> transfer_;
  HostWorkers::Job job_;
  StreamUse use_;
  bool under_way_ = false, misfit_ = false;
  int device_ = -1;  // of the events and the ring
  uint32_t looks_ = 0;
  std::atomic<size_t> ahead_{0};  // parts_ahead()
  uint8_t* ring_ = nullptr;
  size_t ring_bytes_ = 0;
  hipEvent_t packed_[kSlots] = {}, begun_ = nullptr;
  // of pieces that are packed in device memory
  static constexpr size_t kWordsPerLine = 32;
  hipEvent_t copied_[kSlots] = {};
  uint8_t* staging_ = nullptr;
  size_t staging_bytes_ = 0;
  uint32_t *counts_ = nullptr, *totals_ = nullptr;
};

}  // namespace nd
