/*
 * frames.hip -- what leaves the device: frames of markers, fields and bonds,
 * and the step report (sem_copyGPUKernel semLB.cu:979, fiber_copy_GPUKernel
 * semLB.cu:669, fluid_initGPUKernel(aFlag=0) semLB.cu:154).
 *
 * A frame is written by a kernel straight into pinned host memory (one launch
 * for all its arrays, coalesced writes over PCIe) and copied from there into
 * the caller's arrays by a few host threads, half a buffer at a time, the next
 * half being written meanwhile.  Bound by PCIe (53 GB/s) and by the page
 * faults of the caller's new arrays, which one thread takes at 7-9 GB/s.
 * Against a copy per array from pageable memory (us): report of a step 44 ->
 * 13, markers of 256 elements 205 -> 27, of 520 000 1000 -> 530, of 2.08 M
 * 9300 -> 4300; fields of 201x99x75 cells 1430 -> 680-1400, of 128^3
 * 4540 -> 1840, of 320x128x128 9390 -> 2780.  6 to 16 threads and halves of 4
 * to 16 MiB measured the same.
 */
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "pfg_internal.h"

namespace pfg {

namespace {

/* ---------------- pinned buffers ---------------- */

/* Two sizes of pinned buffers, shared by all handles of the process: small
 * ones for reports and small frames, large ones in two halves.  A call holds
 * one buffer; at most KEEP of a size stay allocated between calls, and none
 * once the last handle is destroyed. */
constexpr size_t SMALL_BYTES = (size_t)1 << 20, HALF_BYTES = (size_t)8 << 20;
constexpr size_t KEEP = 4;

std::mutex g_mu;
int g_handles = 0;
std::vector<void *> g_free[2]; /* 0: small, 1: large */

size_t size_of(int kind) { return kind == 0 ? SMALL_BYTES : 2 * HALF_BYTES; }

void *take_buffer(int kind) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_free[kind].empty()) {
      void *p = g_free[kind].back();
      g_free[kind].pop_back();
      return p;
    }
  }
  void *p = nullptr;
  return hipHostMalloc(&p, size_of(kind), hipHostMallocPortable) == hipSuccess ? p : nullptr;
}

void give_buffer(int kind, void *p) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_handles > 0 && g_free[kind].size() < KEEP) {
      g_free[kind].push_back(p); /* capacity reserved by frames_ref */
      return;
    }
  }
  hipHostFree(p);
}

struct Buffer {
  int kind;
  void *host = nullptr;
  explicit Buffer(int k) : kind(k), host(take_buffer(k)) {}
  ~Buffer() {
    if (host) give_buffer(kind, host);
  }
  Buffer(const Buffer &) = delete;
  Buffer &operator=(const Buffer &) = delete;
};

/* ---------------- host threads ---------------- */

struct Segment { /* bytes of a half buffer and where they go */
  char *dst;
  const char *src;
  size_t bytes;
};

/* Copies lists of segments with a few threads that live for one call. */
class Copiers {
 public:
  explicit Copiers(int n) {
    for (int t = 1; t < n; ++t) {
      try {
        threads_.emplace_back([this, t] { work(t); });
      } catch (const std::system_error &) {
        break; /* fewer threads do it as well */
      }
    }
    n_ = 1 + (int)threads_.size();
    sized_.store(true, std::memory_order_release);
  }
  ~Copiers() {
    stop_.store(true, std::memory_order_release);
    for (std::thread &t : threads_) t.join();
  }
  void copy(const std::vector<Segment> &list) {
    list_ = &list;
    left_.store(n_ - 1, std::memory_order_relaxed);
    epoch_.fetch_add(1, std::memory_order_release);
    share(0);
    while (left_.load(std::memory_order_acquire) > 0) sched_yield();
  }

 private:
  void work(int t) {
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
  void share(int t) const {
    size_t total = 0;
    for (const Segment &s : *list_) total += s.bytes;
    size_t lo = total / n_ * t, hi = t == n_ - 1 ? total : total / n_ * (t + 1), at = 0;
    for (const Segment &s : *list_) {
      const size_t a = std::max(lo, at), b = std::min(hi, at + s.bytes);
      if (a < b) std::memcpy(s.dst + (a - at), s.src + (a - at), b - a);
      at += s.bytes;
    }
  }
  std::vector<std::thread> threads_;
  const std::vector<Segment> *list_ = nullptr;
  int n_ = 1;
  std::atomic<int> epoch_{0}, left_{0};
  std::atomic<bool> stop_{false}, sized_{false};
};

/* One thread per 2 MiB, at most 8 and half of the CPUs the process may use. */
int copier_count(size_t bytes) {
  cpu_set_t set;
  int cpus = 2;
  if (sched_getaffinity(0, sizeof(set), &set) == 0) cpus = CPU_COUNT(&set);
  const size_t n = std::min<size_t>({bytes / ((size_t)2 << 20), 8, (size_t)cpus / 2});
  return (int)std::max<size_t>(n, 1);
}

/* ---------------- the pipeline ---------------- */

/* Writes batches 0 .. nb-1 into the buffer's halves in turn (fill(b, device
 * pointer) enqueues the kernel) and copies each out (list(b, host pointer,
 * out) says where its bytes go) while the next one is written. */
template <class Fill, class List>
hipError_t run_batches(pfg_handle *h, size_t total, int nb, Fill fill, List list) {
  const int kind = total <= SMALL_BYTES && nb == 1 ? 0 : 1;
  Buffer buf(kind);
  if (!buf.host) return hipErrorOutOfMemory;
  void *dev = nullptr;
  hipError_t e = hipHostGetDevicePointer(&dev, buf.host, 0);
  if (e != hipSuccess) return e;
  std::vector<Segment> segs;
  if (nb == 1) {
    e = fill(0, (char *)dev);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return e;
    list(0, (const char *)buf.host, segs);
    Copiers(copier_count(total)).copy(segs);
    return hipSuccess;
  }
  hipEvent_t ev[2] = {nullptr, nullptr};
  for (int k = 0; k < 2 && e == hipSuccess; ++k)
    e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
  {
    Copiers copiers(copier_count(total));
    auto start = [&](int b) {
      hipError_t r = fill(b, (char *)dev + (size_t)(b & 1) * HALF_BYTES);
      return r == hipSuccess ? hipEventRecord(ev[b & 1], h->stream) : r;
    };
    if (e == hipSuccess) e = start(0);
    for (int b = 0; b < nb && e == hipSuccess; ++b) {
      if (b + 1 < nb) e = start(b + 1);
      if (e == hipSuccess) e = hipEventSynchronize(ev[b & 1]);
      if (e != hipSuccess) break;
      segs.clear();
      list(b, (const char *)buf.host + (size_t)(b & 1) * HALF_BYTES, segs);
      copiers.copy(segs);
    }
  }
  /* no kernel writes the buffer once it is given back */
  const hipError_t e2 = hipStreamSynchronize(h->stream);
  for (hipEvent_t x : ev)
    if (x) hipEventDestroy(x);
  return e == hipSuccess ? e2 : e;
}

/* ---------------- kernels ---------------- */

constexpr int PACK_MAX = 12; /* arrays per launch */

struct PackArgs {
  const uint32_t *src[PACK_MAX];
  uint32_t *dst[PACK_MAX];
  uint32_t words[PACK_MAX];
};

/* blockIdx.y: the array; its words by the blocks along x */
__global__ __launch_bounds__(256) void pack_kernel(PackArgs a) {
  const uint32_t *src = a.src[blockIdx.y];
  uint32_t *dst = a.dst[blockIdx.y];
  const uint32_t n = a.words[blockIdx.y];
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) dst[i] = src[i];
}

__global__ void report_kernel(const int64_t *counters, const int64_t *detach_step,
                              const int64_t *d_step, int64_t *out) {
  const int t = threadIdx.x;
  if (t < N_COUNTERS) out[t] = counters[t];
  if (t == N_COUNTERS) out[t] = *detach_step;
  if (t == N_COUNTERS + 1) out[t] = *d_step;
}

}  // namespace

void frames_ref() {
  std::lock_guard<std::mutex> lk(g_mu);
  ++g_handles;
  for (auto &f : g_free) f.reserve(KEEP);
}

void frames_unref() {
  std::vector<void *> drop;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_handles > 0) return;
    for (auto &f : g_free) {
      drop.insert(drop.end(), f.begin(), f.end());
      f.clear();
    }
  }
  for (void *p : drop) hipHostFree(p);
}

hipError_t fetch_pieces(pfg_handle *h, const Piece *pieces, int n) {
  /* whole words of each array, in batches of half a buffer */
  struct Part {
    int piece;
    size_t off, bytes; /* within the piece */
  };
  std::vector<std::vector<Part>> batches(1);
  size_t total = 0, room = HALF_BYTES;
  for (int k = 0; k < n; ++k) {
    if (pieces[k].bytes % 4 != 0) return hipErrorInvalidValue;
    for (size_t off = 0; off < pieces[k].bytes;) {
      if (room == 0 || batches.back().size() == PACK_MAX) {
        batches.emplace_back();
        room = HALF_BYTES;
      }
      const size_t b = std::min(room, pieces[k].bytes - off);
      batches.back().push_back({k, off, b});
      off += b;
      room -= b;
      total += b;
    }
  }
  if (total == 0) return hipSuccess;
  auto fill = [&](int b, char *dev) {
    PackArgs a;
    uint32_t most = 0;
    const std::vector<Part> &parts = batches[(size_t)b];
    for (size_t q = 0; q < parts.size(); ++q) {
      a.src[q] = (const uint32_t *)((const char *)pieces[parts[q].piece].src + parts[q].off);
      a.dst[q] = (uint32_t *)dev;
      a.words[q] = (uint32_t)(parts[q].bytes / 4);
      dev += parts[q].bytes;
      most = std::max(most, a.words[q]);
    }
    const unsigned gx = std::min(1024u, (most + 255u) / 256u);
    hipLaunchKernelGGL(pack_kernel, dim3(gx, (unsigned)parts.size()), dim3(256), 0, h->stream, a);
    return hipGetLastError();
  };
  auto list = [&](int b, const char *host, std::vector<Segment> &out) {
    for (const Part &q : batches[(size_t)b]) {
      out.push_back({(char *)pieces[q.piece].dst + q.off, host, q.bytes});
      host += q.bytes;
    }
  };
  return run_batches(h, total, (int)batches.size(), fill, list);
}

hipError_t fetch_fields(pfg_handle *h, int k, float *const host[4]) {
  const int64_t n = h->inst[(size_t)k].N;
  int nf = 0;
  for (int c = 0; c < 4; ++c) nf += host[c] != nullptr;
  if (nf == 0) return hipSuccess;
  const size_t total = sizeof(float) * (size_t)n * nf;
  /* cells per batch: whole blocks of 64 */
  const int64_t room = (int64_t)(HALF_BYTES / (sizeof(float) * nf)) / XBLOCK * XBLOCK;
  const int nb = (int)((n + room - 1) / room);
  auto fill = [&](int b, char *dev) {
    const int64_t lo = room * b, hi = std::min(n, lo + room);
    float *win[4], *at = (float *)dev;
    for (int c = 0; c < 4; ++c) {
      win[c] = host[c] ? at : nullptr;
      if (host[c]) at += hi - lo;
    }
    return launch_lb_fields_window(h, k, (uint32_t)lo, (uint32_t)hi, win);
  };
  auto list = [&](int b, const char *src, std::vector<Segment> &out) {
    const int64_t lo = room * b, hi = std::min(n, lo + room);
    const size_t bytes = sizeof(float) * (size_t)(hi - lo);
    for (int c = 0; c < 4; ++c) {
      if (!host[c]) continue;
      out.push_back({(char *)(host[c] + lo), src, bytes});
      src += bytes;
    }
  };
  return run_batches(h, total, nb, fill, list);
}

hipError_t fetch_report(pfg_handle *h, int64_t out[N_COUNTERS + 2]) {
  Buffer buf(0);
  if (!buf.host) return hipErrorOutOfMemory;
  void *dev = nullptr;
  hipError_t e = hipHostGetDevicePointer(&dev, buf.host, 0);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(report_kernel, dim3(1), dim3(64), 0, h->stream, h->m.counters,
                     h->m.detach_step, h->m.d_step, (int64_t *)dev);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  if (e == hipSuccess) std::memcpy(out, buf.host, sizeof(int64_t) * (N_COUNTERS + 2));
  return e;
}

}  // namespace pfg
