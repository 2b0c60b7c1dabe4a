// The host side of a request's transfers: threads that copy its inputs into
// pinned memory piece by piece (ordinary or pinned, the caller's arrays are read
// once), while compute units pull the pieces that are ready over PCIe
// (mi355x_copy_segments), and the way back for its outputs.
#ifndef GLOW_MI355X_HOST_STAGING_H
#define GLOW_MI355X_HOST_STAGING_H

#include "glow_mi355x.h"

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace glow_mi355x {

// One piece of a request's input on its way into pinned memory.
struct StagePiece {
  const uint8_t *src = nullptr; // the caller's memory
  size_t bytes = 0;
  enum { Bytes, Indices64, Lengths, Quantized } form = Bytes; // Indices64: travel as 2, 2.5, 3 or
                                // 4 bytes each where they fit; Lengths: bag lengths, as a byte each
                                // where they fit; Quantized: float values, as int8 (scale, offset)
  float scale = 1.0f, offset = 0.0f;
  size_t at = 0;                // where in the staging buffer
  mi355x_copy_segment seg{};    // what the device does with it (src and, for indices and lengths, op set here)
};

// Up to five helper threads that work on the pieces of one request together
// with the thread that runs it: as many as a third of the CPUs this process may use.
// After a request they stay awake for half a millisecond, no more of them over all the
// pools of a process than that third, and sleep then.
class StagingPool {
public:
  StagingPool();
  ~StagingPool();
  StagingPool(const StagingPool &) = delete;
  StagingPool &operator=(const StagingPool &) = delete;

  int helpers() const { return (int)threads_.size(); }
  // Stages `pieces` into `buffer` and calls launch(first, last) on this thread for
  // every run of finished pieces as it gets long enough, in order; stops at the
  // first launch that does not return MI355X_OK and returns its status.
  template <typename Launch>
  int run(std::vector<StagePiece> &pieces, uint8_t *buffer, Launch launch);

private:
  void loop();
  void work(); // takes pieces until none is left
  static void stage(StagePiece &p, uint8_t *buffer);
  void open(std::vector<StagePiece> &pieces, uint8_t *buffer, bool wake);
  void close();

  std::vector<std::thread> threads_;
  std::mutex mu_;
  std::condition_variable cv_;
  std::atomic<uint64_t> generation_{0};
  std::atomic<bool> stopping_{false};
  std::atomic<int> active_{0};
  bool openJob_ = false;
  StagePiece *pieces_ = nullptr;
  uint8_t *buffer_ = nullptr;
  size_t count_ = 0;
  std::atomic<size_t> next_{0};
  std::unique_ptr<std::atomic<uint8_t>[]> done_;
  size_t room_ = 0; // entries of done_
};

// Source bytes of a piece (but for what has to stay whole), and how many staged
// bytes are ready before the device is told to pull them. Pieces of 128 KiB take a
// thread 4 to 8 us; a launch per megabyte (the first at half of it) keeps the link
// busy, 20 us a megabyte, without the last one waiting long for its bytes (one per
// 0.5, 1, 3 or 6 MB: 398, 382, 385, 421 us for a ranking request of 8.5 MB).
constexpr size_t kStagePiece = 128 << 10;
constexpr size_t kStageGroup = 1 << 20;
// A request with less than this is staged by its own thread alone.
constexpr size_t kStageAlone = 256 << 10;

template <typename Launch>
int StagingPool::run(std::vector<StagePiece> &pieces, uint8_t *buffer, Launch launch) {
  size_t total = 0;
  for (const auto &p : pieces) total += p.bytes;
  open(pieces, buffer, total > kStageAlone && !threads_.empty());
  size_t ready = 0, sent = 0, ready_bytes = 0;
  int rc = MI355X_OK;
  const size_t n = pieces.size();
  while (ready < n) {
    const size_t i = next_.load(std::memory_order_relaxed) < n
                         ? next_.fetch_add(1, std::memory_order_relaxed)
                         : n;
    if (i < n) {
      stage(pieces[i], buffer);
      done_[i].store(1, std::memory_order_release);
    }
    while (ready < n && done_[ready].load(std::memory_order_acquire))
      ready_bytes += pieces[ready++].seg.bytes;
    if (rc == MI355X_OK && ready > sent && (ready == n || ready_bytes >= (sent == 0 ? kStageGroup / 2 : kStageGroup))) {
      rc = launch(sent, ready);
      sent = ready;
      ready_bytes = 0;
    }
  }
  close();
  return rc;
}

} // namespace glow_mi355x
#endif
