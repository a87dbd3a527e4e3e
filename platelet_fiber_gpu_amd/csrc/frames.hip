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
 * 13-15, markers of 256 elements 205 -> 26-30, of 520 000 1000 -> 530-570, of
 * 2.08 M 9300 -> 4300; fields into new arrays of 201x99x75 cells
 * 1430 -> 1220-1510, of 128^3 4540 -> 1510-1760, of 320x128x128
 * 9390 -> 2620-2960 (by host).  6 to 16 threads and halves of 4 to 16 MiB
 * measured the same.
 */
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "frame_copy.h"
#include "pfg_internal.h"

namespace pfg {

namespace {

/* ---------------- pinned buffers ---------------- */

/* Two sizes of pinned buffers, shared by all handles of the process: small
 * ones for reports and small frames, large ones in two halves.  A call holds
 * one buffer; at most KEEP of a size stay allocated between calls, and none
 * once the last handle is destroyed. */
constexpr size_t SMALL_BYTES = (size_t)1 << 20, HALF_BYTES = (size_t)8 << 20;
constexpr int KEEP = 4;

std::mutex g_mu;
int g_handles = 0;
void *g_free[2][KEEP]; /* 0: small, 1: large */
int g_nfree[2];

size_t size_of(int kind) { return kind == 0 ? SMALL_BYTES : 2 * HALF_BYTES; }

void *take_buffer(int kind) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_nfree[kind] > 0) return g_free[kind][--g_nfree[kind]];
  }
  /* coherent by request, not by the environment's default: a half is read
   * after an event, which publishes no other kind of host memory (frames
   * measured the same with and without) */
  void *p = nullptr;
  return hipHostMalloc(&p, size_of(kind), hipHostMallocPortable | hipHostMallocCoherent) ==
                 hipSuccess
             ? p
             : nullptr;
}

void give_buffer(int kind, void *p) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_handles > 0 && g_nfree[kind] < KEEP) {
      g_free[kind][g_nfree[kind]++] = p;
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

/* One thread per 2 MiB, at most COPIERS_MAX and half of the CPUs the process may use. */
int copier_count(size_t bytes) {
  cpu_set_t set;
  int cpus = 2;
  if (sched_getaffinity(0, sizeof(set), &set) == 0) cpus = CPU_COUNT(&set);
  const size_t n = std::min<size_t>({bytes / ((size_t)2 << 20), COPIERS_MAX, (size_t)cpus / 2});
  return (int)std::max<size_t>(n, 1);
}

/* ---------------- the pipeline ---------------- */

struct Events {
  hipEvent_t e[2] = {nullptr, nullptr};
  hipError_t create() {
    hipError_t r = hipSuccess;
    for (int k = 0; k < 2 && r == hipSuccess; ++k)
      r = hipEventCreateWithFlags(&e[k], hipEventDisableTiming);
    return r;
  }
  ~Events() {
    for (hipEvent_t x : e)
      if (x) hipEventDestroy(x);
  }
};

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
  if (nb == 1) {
    e = fill(0, (char *)dev);
    const hipError_t e2 = hipStreamSynchronize(h->stream);
    if (e == hipSuccess) e = e2;
    if (e != hipSuccess) return e;
    SegmentList segs;
    list(0, (const char *)buf.host, segs);
    Copiers(copier_count(total)).copy(segs);
    return hipSuccess;
  }
  Events ev;
  e = ev.create();
  if (e != hipSuccess) return e;
  Copiers copiers(copier_count(total));
  return copy_halves<hipError_t>(
      nb, copiers,
      [&](int b) {
        const hipError_t r = fill(b, (char *)dev + (size_t)(b & 1) * HALF_BYTES);
        return r == hipSuccess ? hipEventRecord(ev.e[b & 1], h->stream) : r;
      },
      [&](int b) { return hipEventSynchronize(ev.e[b & 1]); },
      [&](int b, SegmentList &out) {
        list(b, (const char *)buf.host + (size_t)(b & 1) * HALF_BYTES, out);
      },
      [&] { return hipStreamSynchronize(h->stream); });
}

/* ---------------- kernels ---------------- */

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
}

void frames_unref() {
  void *drop[2 * KEEP];
  int n = 0;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_handles > 0) return;
    for (int kind = 0; kind < 2; ++kind)
      while (g_nfree[kind] > 0) drop[n++] = g_free[kind][--g_nfree[kind]];
  }
  for (int k = 0; k < n; ++k) hipHostFree(drop[k]);
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
      if (room == 0 || batches.back().size() == (size_t)PACK_MAX) {
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
  auto list = [&](int b, const char *host, SegmentList &out) {
    for (const Part &q : batches[(size_t)b]) {
      out.add((char *)pieces[q.piece].dst + q.off, host, q.bytes);
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
  auto list = [&](int b, const char *src, SegmentList &out) {
    const int64_t lo = room * b, hi = std::min(n, lo + room);
    const size_t bytes = sizeof(float) * (size_t)(hi - lo);
    for (int c = 0; c < 4; ++c) {
      if (!host[c]) continue;
      out.add((char *)(host[c] + lo), src, bytes);
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
