// Results brought to the host by ResultStream (nd_host_results.hpp), against the words that were put on the device:
// every width, sizes around a group, a chunk, a piece and the ring, dead groups, chunks of few different ids, ids that do not fit
// their width, targets that are no multiple of 32 bytes; straight to the host, and packed on the device as words that come while others are still
// computed are, with a sign that is there and with one that never comes.  Prints the case before it runs, "all equal" at the end.
#include "../../nextdoor_amd/csrc/nd_host_results.hpp"

#include <stdio.h>

#include <chrono>
#include <thread>

#define TRY(expr)                                                              \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess) { printf("%s\n", hipGetErrorString(e_)); return 1; } \
  } while (0)

// Words on one device brought home by a thread whose current device is another (or, where there is only one, the same):
// the words are right and the thread's device stays what it was.
static int on_other_devices() {
  int devices = 0;
  TRY(hipGetDeviceCount(&devices));
  const size_t n = (size_t)70 * nd::kPackChunk;
  std::vector<int32_t> want(n), got(n);
  for (size_t i = 0; i < n; ++i) want[i] = (int32_t)(i & 0xfff);
  nd::ResultStream results;
  for (int home = 0; home < std::min(devices, 2); ++home) {
    TRY(hipSetDevice(home));
    int32_t* d = nullptr;
    hipStream_t stream;
    hipEvent_t done;
    TRY(hipMalloc(&d, n * sizeof(int32_t)));
    TRY(hipStreamCreate(&stream));
    TRY(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    TRY(hipMemcpyAsync(d, want.data(), n * sizeof(int32_t), hipMemcpyHostToDevice, stream));
    TRY(hipEventRecord(done, stream));
    for (int away = 0; away < std::min(devices, 2); ++away) {
      for (int ahead = 0; ahead < 2; ++ahead) {
        printf("words on device %d, thread on %d, ahead %d\n", home, away, ahead);
        fflush(stdout);
        TRY(hipSetDevice(away));
        std::fill(got.begin(), got.end(), -1);
        std::vector<nd::ResultStream::Ready> ready;
        if (ahead) ready.push_back({n, done});
        TRY(results.begin(d, n, 12, 0, got.data(), stream, ready));
        TRY(results.finish());
        int now = -1;
        TRY(hipGetDevice(&now));
        if (now != away || got != want) { printf("device %d, or other words\n", now); return 1; }
      }
    }
    TRY(hipSetDevice(home));
    TRY(hipEventDestroy(done));
    TRY(hipStreamDestroy(stream));
    TRY(hipFree(d));
  }
  TRY(hipSetDevice(0));
  return 0;
}

// Some 70 ms of one wavefront; it ends by itself.
__global__ void take_a_while() {
  for (uint32_t i = 0; i < 20000; ++i) __builtin_amdgcn_s_sleep(127);
}
__global__ void write_words(int32_t* words, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) words[i] = (int32_t)(i & 0xfff);
}

// Two transfers whose words come at the end of a long computation, and others whose words are there: those do not wait for it.
static int beside_one_that_waits() {
  const size_t n = (size_t)300 * nd::kPackChunk;
  std::vector<int32_t> want(n), late(n), later(n), got(n);
  for (size_t i = 0; i < n; ++i) want[i] = (int32_t)(i & 0xfff);
  int32_t *d = nullptr, *d_late = nullptr;
  uint32_t* sign = nullptr;
  hipStream_t busy, stream;
  hipEvent_t there, computed;
  TRY(hipMalloc(&d, n * sizeof(int32_t)));
  TRY(hipMalloc(&d_late, n * sizeof(int32_t)));
  TRY(hipHostMalloc((void**)&sign, sizeof(uint32_t), hipHostMallocDefault));
  *sign = 7;
  TRY(hipStreamCreate(&stream));
  TRY(hipStreamCreate(&busy));
  TRY(hipEventCreateWithFlags(&there, hipEventDisableTiming));
  TRY(hipEventCreateWithFlags(&computed, hipEventDisableTiming));
  TRY(hipMemcpyAsync(d, want.data(), n * sizeof(int32_t), hipMemcpyHostToDevice, stream));
  TRY(hipEventRecord(there, stream));
  TRY(hipStreamSynchronize(stream));
  nd::ResultStream first, second, other;
  for (int turn = 0; turn < 3; ++turn) {  // the first one takes the memory
    TRY(hipMemset(d_late, 0, n * sizeof(int32_t)));
    TRY(hipDeviceSynchronize());
    if (turn) take_a_while<<<dim3(1), dim3(64), 0, busy>>>();
    write_words<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, busy>>>(d_late, n);
    TRY(hipGetLastError());
    TRY(hipEventRecord(computed, busy));
    std::fill(late.begin(), late.end(), -1);
    std::fill(later.begin(), later.end(), -1);
    TRY(first.begin(d_late, n, 12, 0, late.data(), busy, {{n, computed}}));
    TRY(second.begin(d_late, n, 12, 0, later.data(), busy, {{n, computed}}));
    std::this_thread::sleep_for(std::chrono::milliseconds(5));  // other threads take them on
    for (int form = 0; form < 3; ++form) {
      printf("beside one that waits: turn %d form %d\n", turn, form);
      fflush(stdout);
      std::vector<nd::ResultStream::Ready> ready{{n, there}};
      if (form == 1) ready.insert(ready.begin(), {n / 2, there});
      if (form == 2) ready = {{n / 3, there, sign, 7u}, {n, there, sign, 7u}};
      std::fill(got.begin(), got.end(), -1);
      TRY(other.begin(d, n, 12, 0, got.data(), stream, ready));
      TRY(other.finish());
      const bool before = hipEventQuery(computed) == hipErrorNotReady;
      (void)hipGetLastError();
      if (got != want) { printf("other words\n"); return 1; }
      if (turn && !before) { printf("held up until the other computation was over\n"); return 1; }
    }
    TRY(first.finish());
    TRY(second.finish());
    if (late != want || later != want) { printf("words from before they were there\n"); return 1; }
  }
  first.release();
  second.release();
  other.release();
  TRY(hipEventDestroy(there));
  TRY(hipEventDestroy(computed));
  TRY(hipStreamDestroy(stream));
  TRY(hipStreamDestroy(busy));
  TRY(hipHostFree(sign));
  TRY(hipFree(d));
  TRY(hipFree(d_late));
  return 0;
}

// One in stream order behind a long computation, of more chunks than the ring holds, and others whose words are there: those do not wait
// for it.
static int beside_one_that_follows() {
  const size_t many = (size_t)4200 * nd::kPackChunk, n = (size_t)300 * nd::kPackChunk;
  std::vector<int32_t> want(many), late(many), got(n);
  for (size_t i = 0; i < many; ++i) want[i] = (int32_t)(i & 0xfff);
  int32_t *d = nullptr, *d_late = nullptr;
  uint32_t* sign = nullptr;
  hipStream_t busy, stream;
  hipEvent_t there, computed;
  TRY(hipMalloc(&d, n * sizeof(int32_t)));
  TRY(hipMalloc(&d_late, many * sizeof(int32_t)));
  TRY(hipHostMalloc((void**)&sign, sizeof(uint32_t), hipHostMallocDefault));
  *sign = 7;
  TRY(hipStreamCreate(&stream));
  TRY(hipStreamCreate(&busy));
  TRY(hipEventCreateWithFlags(&there, hipEventDisableTiming));
  TRY(hipEventCreateWithFlags(&computed, hipEventDisableTiming));
  TRY(hipMemcpyAsync(d, want.data(), n * sizeof(int32_t), hipMemcpyHostToDevice, stream));
  TRY(hipEventRecord(there, stream));
  TRY(hipStreamSynchronize(stream));
  nd::ResultStream first, other;
  for (int turn = 0; turn < 3; ++turn) {  // the first one takes the memory
    TRY(hipMemset(d_late, 0, many * sizeof(int32_t)));
    TRY(hipDeviceSynchronize());
    if (turn) take_a_while<<<dim3(1), dim3(64), 0, busy>>>();
    write_words<<<dim3((unsigned)((many + 255) / 256)), dim3(256), 0, busy>>>(d_late, many);
    TRY(hipGetLastError());
    TRY(hipEventRecord(computed, busy));
    std::fill(late.begin(), late.end(), -1);
    TRY(first.begin(d_late, many, 12, 0, late.data(), busy, {}, /*follows=*/turn < 2));
    std::this_thread::sleep_for(std::chrono::milliseconds(5));  // other threads take it on
    for (int form = 0; form < 3; ++form) {
      printf("beside one that follows: turn %d form %d\n", turn, form);
      fflush(stdout);
      std::vector<nd::ResultStream::Ready> ready{{n, there}};
      if (form == 1) ready.insert(ready.begin(), {n / 2, there});
      if (form == 2) ready = {{n / 3, there, sign, 7u}, {n, there, sign, 7u}};
      std::fill(got.begin(), got.end(), -1);
      TRY(other.begin(d, n, 12, 0, got.data(), stream, ready));
      TRY(other.finish());
      const bool before = hipEventQuery(computed) == hipErrorNotReady;
      (void)hipGetLastError();
      if (!std::equal(got.begin(), got.end(), want.begin())) { printf("other words\n"); return 1; }
      if (turn && !before) { printf("held up until the other computation was over\n"); return 1; }
    }
    if (turn == 1) {  // else finish() goes on without
      TRY(hipEventSynchronize(computed));
      first.words_are_there();
    }
    TRY(first.finish());
    if (late != want) { printf("words from before they were there\n"); return 1; }
  }
  first.release();
  other.release();
  TRY(hipEventDestroy(there));
  TRY(hipEventDestroy(computed));
  TRY(hipStreamDestroy(stream));
  TRY(hipStreamDestroy(busy));
  TRY(hipHostFree(sign));
  TRY(hipFree(d));
  TRY(hipFree(d_late));
  return 0;
}

// Threads that take part in work that is asked for now, within 10 ms.
static unsigned threads_that_are_free() {
  std::atomic<unsigned> here{0};
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(10);
  nd::HostWorkers::get().run(nd::HostWorkers::kMost, [&] {
    if (std::chrono::steady_clock::now() < until) here++;  // else one of them comes again
    while (std::chrono::steady_clock::now() < until) std::this_thread::yield();
  });
  return here.load();
}

// While a transfer waits for its words, at most one thread does: one that asks for them, unless they follow a computation.
static int threads_beside_one_that_waits() {
  const size_t n = (size_t)300 * nd::kPackChunk;
  std::vector<int32_t> want(n), late(n);
  for (size_t i = 0; i < n; ++i) want[i] = (int32_t)(i & 0xfff);
  int32_t* d_late = nullptr;
  uint32_t* sign = nullptr;
  hipStream_t busy;
  hipEvent_t computed;
  TRY(hipMalloc(&d_late, n * sizeof(int32_t)));
  TRY(hipHostMalloc((void**)&sign, sizeof(uint32_t), hipHostMallocDefault));
  *sign = 0;
  TRY(hipStreamCreate(&busy));
  TRY(hipEventCreateWithFlags(&computed, hipEventDisableTiming));
  nd::ResultStream first;
  const unsigned all = threads_that_are_free();
  for (int turn = 0; turn < 2; ++turn)  // the first one takes the memory
    for (int form = 0; form < 3; ++form) {
      TRY(hipMemset(d_late, 0, n * sizeof(int32_t)));
      TRY(hipDeviceSynchronize());
      if (turn) take_a_while<<<dim3(1), dim3(64), 0, busy>>>();
      write_words<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, busy>>>(d_late, n);
      TRY(hipGetLastError());
      TRY(hipEventRecord(computed, busy));
      std::vector<nd::ResultStream::Ready> ready{{n, computed}};
      if (form == 0) ready.clear();
      if (form == 2) ready = {{n / 3, computed, sign, 7u}, {n, computed, sign, 7u}};
      std::fill(late.begin(), late.end(), -1);
      TRY(first.begin(d_late, n, 12, 0, late.data(), busy, ready, /*follows=*/form == 0));
      std::this_thread::sleep_for(std::chrono::milliseconds(5));  // other threads take it on
      unsigned now = threads_that_are_free();
      for (int again = 0; again < 2 && now < all; ++again) now = std::max(now, threads_that_are_free());  // one was slow to wake
      const bool before = hipEventQuery(computed) == hipErrorNotReady;
      (void)hipGetLastError();
      printf("threads beside one that waits: turn %d form %d: %u of %u\n", turn, form, now, all);
      fflush(stdout);
      if (turn && !before) { printf("the computation was over\n"); return 1; }
      if (turn && now + (form == 0 ? 0 : 1) < all) { printf("threads are kept\n"); return 1; }
      TRY(first.finish());
      if (late != want) { printf("words from before they were there\n"); return 1; }
    }
  first.release();
  TRY(hipEventDestroy(computed));
  TRY(hipStreamDestroy(busy));
  TRY(hipHostFree(sign));
  TRY(hipFree(d_late));
  return 0;
}

int main() {
  if (on_other_devices() != 0) return 1;
  if (beside_one_that_waits() != 0) return 1;
  if (beside_one_that_follows() != 0) return 1;
  if (threads_beside_one_that_waits() != 0) return 1;
  const size_t piece = (size_t)64 * nd::kPackChunk;  // the smallest piece
  const size_t sizes[] = {1, 7, 8, 9, nd::kPackChunk - 1, nd::kPackChunk, nd::kPackChunk + 1, piece, piece + 9, 13 * piece + 4097,
                          (size_t)4200 * nd::kPackChunk + 5, (size_t)9000 * nd::kPackChunk + 5};
  nd::ResultStream stream;
  uint32_t* sign = nullptr;  // what has arrived, and what never does
  hipEvent_t done;
  TRY(hipHostMalloc((void**)&sign, 2 * sizeof(uint32_t), hipHostMallocDefault));
  sign[0] = 3, sign[1] = 0;
  TRY(hipEventCreateWithFlags(&done, hipEventDisableTiming));
  for (size_t n : sizes) {
    int32_t* d = nullptr;
    TRY(hipMalloc(&d, n * sizeof(int32_t)));
    for (uint32_t bits : {1u, 2u, 7u, 8u, 9u, 12u, 16u, 17u, 23u, 24u, 25u, 26u, 31u, 32u}) {
      if (n > piece + 9 && bits != 12 && bits != 23 && bits != 32) continue;
      if (n > 14 * piece && bits == 23) continue;
      if (n > 70 * piece && bits != 12) continue;
      for (int misfit = 0; misfit < 2; ++misfit) {
        printf("n %zu bits %u misfit %d\n", n, bits, misfit);
        fflush(stdout);
        const uint32_t mask = bits == 32 ? 0xffffffffu : (1u << bits) - 1u;
        const int32_t fill = (int32_t)mask;
        std::vector<int32_t> want(n), got(n + 2, 77);
        for (size_t i = 0; i < n; ++i)
          want[i] = (i / 11) % 3 == 0 || (i / 700) % 4 == 1 ? fill : (int32_t)(((uint32_t)i * 2654435761u) & mask);
        for (size_t i = 0; i < n; ++i)  // every third chunk: ids next to each other, one of them the largest there is
          if (i / nd::kPackChunk % 3 == 1 && want[i] != fill) want[i] = (int32_t)(mask - 1u - ((uint32_t)want[i] & mask & 9u));
        if (misfit) want[n / 2] = -5;
        TRY(hipMemcpy(d, want.data(), n * sizeof(int32_t), hipMemcpyHostToDevice));
        for (int shift = 0; shift < 2; ++shift) {
          if (bits == 32) {  // as bytes, the last word not whole
            const size_t bytes = n * sizeof(int32_t) - (size_t)shift;
            TRY(stream.copy(d, bytes, got.data() + shift, nullptr));
            if (memcmp(got.data() + shift, want.data(), bytes) != 0) { printf("bytes differ\n"); return 1; }
          }
          TRY(stream.fetch({{d, n, bits, fill, got.data() + shift, /*sparse=*/shift == 1}}, nullptr));
          if (memcmp(got.data() + shift, want.data(), n * sizeof(int32_t)) != 0 || got[n + 1] != 77) {
            printf("differs at shift %d\n", shift);
            return 1;
          }
        }
        TRY(hipEventRecord(done, nullptr));
        TRY(hipEventSynchronize(done));
        for (int comes = 0; comes < 2; ++comes) {
          const uint32_t* word = sign + 1 - comes;
          std::vector<nd::ResultStream::Ready> ready{{n, done, word, 3}};
          if (n > 1) ready.insert(ready.begin(), {n / 2, done, word, 3});
          std::fill(got.begin(), got.end(), 77);
          TRY(stream.begin(d, n, bits, fill, got.data() + comes, nullptr, ready));
          TRY(stream.finish());
          if (memcmp(got.data() + comes, want.data(), n * sizeof(int32_t)) != 0 || got[n + 1] != 77) {
            printf("differs where the sign comes %d\n", comes);
            return 1;
          }
        }
      }
    }
    TRY(hipFree(d));
  }
  stream.release();
  TRY(hipHostFree(sign));
  TRY(hipEventDestroy(done));
  printf("all equal\n");
  return 0;
}
