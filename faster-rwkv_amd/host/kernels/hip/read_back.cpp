// Large results (the logits of every position of a text) from the device into the caller's memory.
//
// A blocking copy into fresh pageable memory, which is what Copy(x, kCPU) is, runs at 4 GB/s: the driver stages it in
// small pieces, and every page of the destination is faulted in and cleared by the one thread that copies.  Here the
// data cross the bus into a small pinned ring and a few threads carry them on, each faulting its own pages.
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

struct ReadBack {
  static constexpr size_t kChunk = 1u << 20, kSlots = 8;
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

void read_to_host(ModelExtra &ex, const Tensor &src, void *dst) {
  using RB = ReadBack;
  const size_t n = src.nbytes(), chunks = (n + RB::kChunk - 1) / RB::kChunk;
  if (chunks < 4) {  // a ring has nothing to overlap
    FRHIP_CHECK(frhip_stream_sync(stream()));
    FRHIP_CHECK(frhip_memcpy(dst, src.data_ptr(), n, FRHIP_D2H));
    return;
  }
  if (!ex.read_back) ex.read_back = std::make_shared<RB>();
  RB &rb = *ex.read_back;
  const char *from = static_cast<const char *>(src.data_ptr());
  char *ring = static_cast<char *>(rb.ring), *to = static_cast<char *>(dst);
  auto len = [&](size_t i) { return std::min(RB::kChunk, n - i * RB::kChunk); };
  auto issue = [&](size_t i) {
    const size_t s = i % RB::kSlots;
    FRHIP_CHECK(frhip_memcpy_async(ring + s * RB::kChunk, from + i * RB::kChunk, len(i), FRHIP_D2H, stream()));
    FRHIP_CHECK(frhip_event_record(rb.landed[s], stream()));
  };
  auto carry = [&](size_t i) { std::memcpy(to + i * RB::kChunk, ring + (i % RB::kSlots) * RB::kChunk, len(i)); };

  std::mutex mu;
  std::condition_variable cv;
  size_t ready = 0, taken = 0;  // chunks [0, ready) are in the ring or beyond; [0, taken) have a thread
  bool stop = false;
  std::vector<char> done(chunks, 0);
  auto work = [&]() {
    std::unique_lock<std::mutex> lock(mu);
    for (;;) {
      cv.wait(lock, [&] { return stop || taken < ready; });
      if (taken >= ready) return;  // stopped, nothing left
      const size_t i = taken++;
      lock.unlock();
      carry(i);
      lock.lock();
      done[i] = 1;
      cv.notify_all();
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
  const size_t hands = std::min<size_t>({8, std::max(1u, std::thread::hardware_concurrency()), chunks / 2});
  try {
    for (size_t t = 0; t < hands; t++) crew.threads.emplace_back(work);
  } catch (const std::exception &) {  // as many as the system gives; with none this thread carries
  }
  constexpr size_t kAhead = RB::kSlots / 2;
  for (size_t i = 0; i < std::min(kAhead, chunks); i++) issue(i);
  for (size_t j = 0; j < chunks; j++) {
    FRHIP_CHECK(frhip_event_sync(rb.landed[j % RB::kSlots]));
    if (crew.threads.empty()) {
      carry(j);
    } else {
      std::unique_lock<std::mutex> lock(mu);
      ready = j + 1;
      cv.notify_all();
      // chunk j + kAhead goes into the slot of chunk j - kAhead
      if (j >= kAhead) cv.wait(lock, [&] { return done[j - kAhead] != 0; });
    }
    if (j + kAhead < chunks) issue(j + kAhead);
  }
}  // the crew finishes what is in the ring

}  // namespace hip
}  // namespace rwkv
