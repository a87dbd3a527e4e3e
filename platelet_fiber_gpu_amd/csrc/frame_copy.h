/*
 * frame_copy.h -- the host's half of a frame: a few threads that copy lists
 * of segments, and the loop over half buffers.  Nothing here allocates once
 * the first half is being written, and nothing throws: a buffer given back
 * while a kernel still writes it would hand that kernel's bytes to another
 * call.
 */
#ifndef PFG_FRAME_COPY_H
#define PFG_FRAME_COPY_H

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <thread>

namespace pfg {

constexpr int PACK_MAX = 12;    /* arrays per launch, segments per list */
constexpr int COPIERS_MAX = 8;  /* threads of a copy, the caller's included */

struct Segment { /* bytes of a half buffer and where they go */
  char *dst;
  const char *src;
  size_t bytes;
};

struct SegmentList {
  Segment s[PACK_MAX];
  int n = 0;
  void add(char *dst, const char *src, size_t bytes) { s[n++] = {dst, src, bytes}; }
};

/* Copies lists of segments with a few threads that live for one call. */
class Copiers {
 public:
  explicit Copiers(int n) noexcept {
    for (int t = 1; t < std::min(n, COPIERS_MAX); ++t) {
      try {
        threads_[t - 1] = std::thread([this, t] { work(t); });
      } catch (const std::exception &) {
        break; /* no thread or no memory for one: fewer do it as well */
      }
      ++n_;
    }
    sized_.store(true, std::memory_order_release);
  }
  ~Copiers() {
    stop_.store(true, std::memory_order_release);
    for (int t = 1; t < n_; ++t) threads_[t - 1].join();
  }
  Copiers(const Copiers &) = delete;
  Copiers &operator=(const Copiers &) = delete;
  int count() const { return n_; }
  void copy(const SegmentList &list) noexcept {
    list_ = &list;
    left_.store(n_ - 1, std::memory_order_relaxed);
    epoch_.fetch_add(1, std::memory_order_release);
    share(0);
    while (left_.load(std::memory_order_acquire) > 0) sched_yield();
  }

 private:
  void work(int t) noexcept {
    int seen = 0;
    while (!sized_.load(std::memory_order_acquire)) sched_yield();
    for (;;) {
      while (epoch_.load(std::memory_order_acquire) == seen) {
        if (stop_.load(std::memory_order_acquire)) return;
        sched_yield();
      }
      ++seen;
      share(t);
      left_.fetch_sub(1, std::memory_order_release);
    }
  }
  /* the t-th of n_ equal shares of the list's bytes */
  void share(int t) const noexcept {
    size_t total = 0;
    for (int k = 0; k < list_->n; ++k) total += list_->s[k].bytes;
    const size_t lo = total / n_ * t, hi = t == n_ - 1 ? total : total / n_ * (t + 1);
    size_t at = 0;
    for (int k = 0; k < list_->n; ++k) {
      const Segment &s = list_->s[k];
      const size_t a = std::max(lo, at), b = std::min(hi, at + s.bytes);
      if (a < b) std::memcpy(s.dst + (a - at), s.src + (a - at), b - a);
      at += s.bytes;
    }
  }
  std::thread threads_[COPIERS_MAX - 1];
  const SegmentList *list_ = nullptr;
  int n_ = 1;
  std::atomic<int> epoch_{0}, left_{0};
  std::atomic<bool> stop_{false}, sized_{false};
};

/* Batches 0 .. nb-1 through two halves in turn.  write(b) enqueues the kernel
 * of batch b, written(b) waits for it, list(b, out) says where its bytes go,
 * drain() waits for all that is enqueued, also after an error: no kernel
 * writes the halves once this returns.  Results are error codes, 0 for
 * success; the first error ends the loop. */
template <class Err, class Write, class Written, class List, class Drain>
Err copy_halves(int nb, Copiers &copiers, Write write, Written written, List list, Drain drain) {
  SegmentList segs;
  Err e = write(0);
  for (int b = 0; b < nb && e == Err(0); ++b) {
    if (b + 1 < nb) e = write(b + 1);
    if (e == Err(0)) e = written(b);
    if (e != Err(0)) break;
    segs.n = 0;
    list(b, segs);
    copiers.copy(segs);
  }
  const Err d = drain();
  return e == Err(0) ? d : e;
}

}  // namespace pfg

#endif
