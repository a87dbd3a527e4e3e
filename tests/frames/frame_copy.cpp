/* The host's half of a frame (csrc/frame_copy.h) without a device: memory that
 * runs out at any allocation, and errors at any call. */
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "frame_copy.h"

static std::atomic<long> g_left{-1}; /* allocations until they fail; -1: never */
static std::atomic<long> g_count{0};

void *operator new(size_t n) {
  ++g_count;
  long l = g_left.load();
  while (l > 0 && !g_left.compare_exchange_weak(l, l - 1)) {}
  void *p = l == 0 ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

#define CHECK(c)                                            \
  do {                                                      \
    if (!(c)) {                                             \
      std::printf("line %d: %s\n", __LINE__, #c);           \
      std::exit(1);                                         \
    }                                                       \
  } while (0)

using namespace pfg;

/* threads that cannot be made are done without; the bytes arrive all the same */
static void out_of_memory(int threads, long allocations) {
  std::vector<char> src(1000003), dst(src.size(), 0);
  for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(i * 31 + i / 257);
  SegmentList l;
  const size_t cut[] = {0, 1, 77777, 77777, 500000, src.size()};
  for (int k = 0; k < 5; ++k) l.add(dst.data() + cut[k], src.data() + cut[k], cut[k + 1] - cut[k]);
  g_left = allocations;
  {
    Copiers c(threads);
    CHECK(c.count() >= 1 && c.count() <= COPIERS_MAX);
    CHECK(allocations != 0 || c.count() == 1);
    for (int r = 0; r < 3; ++r) c.copy(l);
  }
  g_left = -1;
  CHECK(src == dst);
}

/* nb batches, the call-th call failing (-1: none): what was copied is right,
 * nothing is in flight afterwards, nothing is allocated on the way */
static void halves(int nb, int fail) {
  constexpr size_t HALF = 4096;
  std::vector<char> half[2] = {std::vector<char>(HALF), std::vector<char>(HALF)};
  std::vector<char> dst(HALF * (size_t)nb, 0);
  std::vector<int> state((size_t)nb, 0); /* 1 enqueued, 2 written, 3 copied */
  int call = 0, drained = 0;
  Copiers copiers(3);
  const long before = g_count;
  const int e = copy_halves<int>(
      nb, copiers,
      [&](int b) {
        if (call++ == fail) return 7;
        CHECK(state[(size_t)b] == 0 && (b < 2 || state[(size_t)b - 2] == 3));
        state[(size_t)b] = 1;
        return 0;
      },
      [&](int b) {
        if (call++ == fail) return 7;
        CHECK(state[(size_t)b] == 1);
        for (size_t i = 0; i < HALF; ++i) half[b & 1][i] = (char)(b * 5 + 1 + i % 3);
        state[(size_t)b] = 2;
        return 0;
      },
      [&](int b, SegmentList &out) {
        CHECK(state[(size_t)b] == 2 && out.n == 0);
        state[(size_t)b] = 3;
        for (int k = 0; k < PACK_MAX; ++k) {
          const size_t lo = HALF * k / PACK_MAX, hi = HALF * (k + 1) / PACK_MAX;
          out.add(dst.data() + HALF * b + lo, half[b & 1].data() + lo, hi - lo);
        }
      },
      [&] {
        ++drained;
        return call++ == fail ? 7 : 0;
      });
  CHECK(g_count == before);
  CHECK(drained == 1); /* also after an error */
  CHECK(e == (fail >= 0 && fail < call ? 7 : 0));
  for (int b = 0; b < nb; ++b)
    for (size_t i = 0; i < HALF; ++i)
      CHECK(dst[HALF * b + i] == (state[(size_t)b] == 3 ? (char)(b * 5 + 1 + i % 3) : 0));
  CHECK(fail >= 0 || state.back() == 3);
}

int main() {
  for (int threads : {1, 2, 8, 20})
    for (long n = -1; n < 9; ++n) out_of_memory(threads, n);
  for (int nb : {1, 2, 3, 7})
    for (int fail = -1; fail <= 2 * nb + 1; ++fail) halves(nb, fail);
  std::printf("ok\n");
  return 0;
}
