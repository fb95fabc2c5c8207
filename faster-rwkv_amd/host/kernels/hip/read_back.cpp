// Large results (the logits of every position of a text) from the device into the caller's memory as fp32.
//
// A blocking copy into fresh pageable memory, which is what Copy(x, kCPU) is, runs at 4 GB/s: the driver stages it in
// small pieces, and every page of the destination is faulted in and cleared by the one thread that copies.  Here the
// data cross the bus into a small pinned ring and a few threads carry them on, each faulting its own pages.
//
// Logits are binary16 values: they cross as such, and the threads widen them (exact).  256 x 50277 logits cross at 53 GB/s,
// 0.48 ms instead of 0.96 as fp32; a chunk is 2 MB because each costs the thread that issues copies about 35 us (the copy,
// its event, the wait), as long as 2 MB take on the bus.  The whole call, 12 layers of 768 included: 2.6 -> 1.75 ms, against
// chunks of 1 MB of fp32.
#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "kernels/hip/context.h"
#include "kernels/hip/hip_model.h"

namespace rwkv {
namespace hip {

namespace {

void widen_plain(const float16 *src, float *dst, size_t n) {
  for (size_t i = 0; i < n; i++) dst[i] = static_cast<float>(src[i]);
}

#if defined(__x86_64__)
// The destination is not read again soon: stores past the caches, no line of it is read in first.
__attribute__((target("avx,f16c"))) void widen_f16c(const float16 *src, float *dst, size_t n) {
  size_t i = 0;
  while (i < n && reinterpret_cast<uintptr_t>(dst + i) % 32 != 0) {
    dst[i] = static_cast<float>(src[i]);
    i++;
  }
  for (; i + 8 <= n; i += 8)
    _mm256_stream_ps(dst + i, _mm256_cvtph_ps(_mm_loadu_si128(reinterpret_cast<const __m128i *>(src + i))));
  widen_plain(src + i, dst + i, n - i);
  _mm_sfence();
}

void widen(const float16 *src, float *dst, size_t n) {
  static const bool fast = __builtin_cpu_supports("avx") && __builtin_cpu_supports("f16c");
  fast ? widen_f16c(src, dst, n) : widen_plain(src, dst, n);
}
#else
void widen(const float16 *src, float *dst, size_t n) { widen_plain(src, dst, n); }
#endif

}  // namespace

struct ReadBack {
  static constexpr size_t kChunk = 2u << 20, kSlots = 6;
  void *ring = nullptr;  // pinned, kSlots chunks; lives and dies with the model
  frhip_event landed[kSlots] = {};
  ReadBack() {
    FRHIP_CHECK(frhip_host_malloc(&ring, kChunk * kSlots));
    for (auto &e : landed) FRHIP_CHECK(frhip_event_create(&e));
  }
  ~ReadBack() {
    frhip_stream_sync(stream());  // a call that failed may have left copies on their way
    for (auto e : landed)
      if (e) frhip_event_destroy(e);
    if (ring) frhip_host_free(ring);
  }
};

void read_to_host(ModelExtra &ex, const Tensor &src, float *dst) {
  using RB = ReadBack;
  RV_CHECK(src.dtype() == DType::kFloat16 || src.dtype() == DType::kFloat32);
  const bool half = src.dtype() == DType::kFloat16;
  const size_t n = src.nbytes(), count = static_cast<size_t>(src.numel()), size = src.elem_size();
  // `bytes` bytes of the source that have arrived at `from`, beginning with byte `at` of it
  auto place = [&](const char *from, size_t at, size_t bytes) {
    if (half)
      widen(reinterpret_cast<const float16 *>(from), dst + at / size, bytes / size);
    else
      std::memcpy(dst + at / size, from, bytes);
  };
  if (count * sizeof(float) <= (3u << 20)) {  // a ring has nothing to overlap
    FRHIP_CHECK(frhip_stream_sync(stream()));
    if (half) {
      std::vector<char> tmp(n);
      FRHIP_CHECK(frhip_memcpy(tmp.data(), src.data_ptr(), n, FRHIP_D2H));
      place(tmp.data(), 0, n);
    } else {
      FRHIP_CHECK(frhip_memcpy(dst, src.data_ptr(), n, FRHIP_D2H));
    }
    return;
  }
  if (!ex.read_back) ex.read_back = std::make_shared<RB>();
  RB &rb = *ex.read_back;
  const size_t chunks = (n + RB::kChunk - 1) / RB::kChunk;
  const char *from = static_cast<const char *>(src.data_ptr());
  char *ring = static_cast<char *>(rb.ring);
  auto len = [&](size_t i) { return std::min(RB::kChunk, n - i * RB::kChunk); };
  auto issue = [&](size_t i) {
    const size_t s = i % RB::kSlots;
    FRHIP_CHECK(frhip_memcpy_async(ring + s * RB::kChunk, from + i * RB::kChunk, len(i), FRHIP_D2H, stream()));
    FRHIP_CHECK(frhip_event_record(rb.landed[s], stream()));
  };
  // a thread takes a piece of a chunk at a time, so that the last chunk is not one thread's work
  constexpr size_t kPiece = 256u << 10, kPieces = RB::kChunk / kPiece;
  const size_t pieces = (n + kPiece - 1) / kPiece;
  auto carry = [&](size_t p) {
    place(ring + p / kPieces % RB::kSlots * RB::kChunk + p % kPieces * kPiece, p * kPiece, std::min(kPiece, n - p * kPiece));
  };

  std::mutex mu;
  std::condition_variable cv, freed;  // pieces to take; a chunk is out of the ring
  size_t ready = 0, taken = 0;  // pieces [0, ready) are in the ring or beyond; [0, taken) have a thread
  bool stop = false;
  std::vector<size_t> left(chunks);  // pieces of a chunk still in the ring
  for (size_t i = 0; i < chunks; i++) left[i] = (len(i) + kPiece - 1) / kPiece;
  auto work = [&]() {
    std::unique_lock<std::mutex> lock(mu);
    for (;;) {
      cv.wait(lock, [&] { return stop || taken < ready; });
      if (taken >= ready) return;  // stopped, nothing left
      const size_t p = taken++;
      lock.unlock();
      carry(p);
      lock.lock();
      if (--left[p / kPieces] == 0) freed.notify_all();
    }
  };
  struct Crew {
    std::vector<std::thread> threads;
    std::mutex &mu;
    std::condition_variable &cv;
    bool &stop;
    ~Crew() {  // also when a device call below throws
      {
        std::lock_guard<std::mutex> lock(mu);
        stop = true;
      }
      cv.notify_all();
      for (auto &t : threads) t.join();
    }
  } crew{{}, mu, cv, stop};
  const size_t hands = std::min<size_t>({8, std::max(1u, std::thread::hardware_concurrency()), pieces});
  constexpr size_t kAhead = RB::kSlots / 2;
  for (size_t i = 0; i < std::min(kAhead, chunks); i++) issue(i);
  try {
    for (size_t t = 0; t < hands; t++) crew.threads.emplace_back(work);
  } catch (const std::exception &) {  // as many as the system gives; with none this thread carries
  }
  for (size_t j = 0; j < chunks; j++) {
    FRHIP_CHECK(frhip_event_sync(rb.landed[j % RB::kSlots]));
    if (crew.threads.empty()) {
      for (size_t p = j * kPieces; p < std::min(pieces, (j + 1) * kPieces); p++) carry(p);
    } else {
      std::unique_lock<std::mutex> lock(mu);
      ready = std::min(pieces, (j + 1) * kPieces);
      cv.notify_all();
      // chunk j + kAhead goes into the slot of chunk j - kAhead
      if (j >= kAhead && j + kAhead < chunks) freed.wait(lock, [&] { return left[j - kAhead] == 0; });
    }
    if (j + kAhead < chunks) issue(j + kAhead);
  }
}  // the crew finishes what is in the ring

}  // namespace hip
}  // namespace rwkv
