// Results to host memory and graphs from it.
//
// Callers hand over ordinary (pageable) host memory.  The runtime copies such
// memory in 1 MB pieces through a buffer of its own, one after the other with
// a synchronisation each (16 MB of levels of an R-MAT 22 graph: 1.0 ms, 64 MB
// of a 4096 x 4096 grid in fresh pages 6 ms, against a search of 0.25 and 7.5
// ms).  Here the pieces go through a ring of pinned buffers, so that the card
// writes one piece while the host moves others; large copies are moved by
// several threads, whole pieces each (fresh memory costs more than the copy:
// the kernel zeroes it 2 MB at a time, and threads that share such a page
// wait for one of them, so a piece is one page of host memory); and levels
// cross the bus as one byte per vertex (two from 255 levels on) and are
// widened on arrival.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>

#include "bfsx_internal.hpp"

namespace bfsx {

namespace {

constexpr size_t PIECE = RING_PIECE_BYTES;  // host bytes of a piece; a slot holds one
// Copies of up to SMALL host bytes go through the ring whole, as one transfer
// and a wait (to / from the card, us: 16 KB 12 / 12, 128 KB 11 / 14, 512 KB 24
// / 30; the runtime's copy of pageable memory takes 18 / 26, 59 / 61 and 35 /
// 32 until some 16 MB have warmed its buffers, 12 / 12 to 26 / 30 then).  They
// wait for the stream; after a search for an event, which takes 7 us more
// from 32 KB on but leaves the bookkeeping of the search's launches, some 20
// us, to a later call (R-MAT-like graph of 10^4 edges, levels: 131 -> 110).
constexpr size_t SMALL = PIECE / 4;
constexpr int MAX_HELPERS = 3;              // threads that move pieces beside the caller's
constexpr uint64_t HELP_PIECES = 3;         // copies of fewer pieces: the caller's thread alone

// out[i] = level + 1 (0: unreached), as T; eight levels per thread.
template <class T>
__global__ __launch_bounds__(256) void k_narrow_levels(const int32_t *levels, uint32_t n, T *out) {
  const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (i + 8 <= n) {
    const int4 a = *reinterpret_cast<const int4 *>(levels + i);
    const int4 b = *reinterpret_cast<const int4 *>(levels + i + 4);
    const uint32_t x[8] = {(uint32_t)a.x + 1, (uint32_t)a.y + 1, (uint32_t)a.z + 1,
                           (uint32_t)a.w + 1, (uint32_t)b.x + 1, (uint32_t)b.y + 1,
                           (uint32_t)b.z + 1, (uint32_t)b.w + 1};
    if (sizeof(T) == 1) {
      uint2 o;
      o.x = x[0] | x[1] << 8 | x[2] << 16 | x[3] << 24;
      o.y = x[4] | x[5] << 8 | x[6] << 16 | x[7] << 24;
      *reinterpret_cast<uint2 *>(out + i) = o;
    } else {
      uint4 o;
      o.x = x[0] | x[1] << 16;
      o.y = x[2] | x[3] << 16;
      o.z = x[4] | x[5] << 16;
      o.w = x[6] | x[7] << 16;
      *reinterpret_cast<uint4 *>(out + i) = o;
    }
  } else {
    for (uint32_t k = i; k < n; k++) out[k] = (T)(uint32_t)(levels[k] + 1);
  }
}

template <class T> inline void widen_loop(const T *src, int32_t *dst, size_t n) {
  for (size_t i = 0; i < n; i++) dst[i] = (int32_t)src[i] - 1;
}
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
__attribute__((target("avx2"))) void widen8_avx2(const uint8_t *src, int32_t *dst, size_t n) {
  for (size_t i = 0; i < n; i++) dst[i] = (int32_t)src[i] - 1;
}
__attribute__((target("avx2"))) void widen16_avx2(const uint16_t *src, int32_t *dst, size_t n) {
  for (size_t i = 0; i < n; i++) dst[i] = (int32_t)src[i] - 1;
}
bool have_avx2() {
  static const bool ok = __builtin_cpu_supports("avx2");
  return ok;
}
#else
void widen8_avx2(const uint8_t *src, int32_t *dst, size_t n) { widen_loop(src, dst, n); }
void widen16_avx2(const uint16_t *src, int32_t *dst, size_t n) { widen_loop(src, dst, n); }
bool have_avx2() { return false; }
#endif

void widen(const void *src, int32_t *dst, size_t n, int width) {
  if (width == 1) {
    if (have_avx2()) widen8_avx2(static_cast<const uint8_t *>(src), dst, n);
    else widen_loop(static_cast<const uint8_t *>(src), dst, n);
  } else {
    if (have_avx2()) widen16_avx2(static_cast<const uint16_t *>(src), dst, n);
    else widen_loop(static_cast<const uint16_t *>(src), dst, n);
  }
}

inline void pause() {
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
  __builtin_ia32_pause();
#endif
}

// Runs piece(k) for k = 0 .. pieces - 1, each once, in the caller's thread and,
// for large copies, helpers beside it: whoever is free takes the next one (a
// helper takes some 50 us to start, in which the caller's thread has moved
// its first pieces).  turn(k) waits until the piece `RING_SLOTS` before k, the
// last user of its slot, has been through pass(k).  The first failure stops
// the others and is thrown here, after every helper has ended.
class Crew {
 public:
  template <class F> static void run(bfsx_ctx *ctx, uint64_t pieces, F piece) {
    Crew c;
    auto work = [&c, pieces, &piece] {
      try {
        for (uint64_t k; !c.stop_.load(std::memory_order_relaxed) &&
                         (k = c.next_.fetch_add(1)) < pieces;)
          piece(c, k);
      } catch (...) {
        if (!c.stop_.exchange(true)) c.error_ = std::current_exception();
      }
    };
    std::thread helpers[MAX_HELPERS];
    const int want = pieces < HELP_PIECES ? 0 : (int)std::min<uint64_t>(pieces - 1, MAX_HELPERS);
    int n = 0;
    try {
      for (; n < want; n++)
        helpers[n] = std::thread([ctx, work] {
          if (hipSetDevice(ctx->device) == hipSuccess) work();  // (else the others take its share)
        });
    } catch (...) {  // no more threads: those there take all pieces
    }
    work();
    for (int w = 0; w < n; w++) helpers[w].join();
    if (c.error_) std::rethrow_exception(c.error_);
  }
  void turn(uint64_t k) {
    while (k >= RING_SLOTS && passed_[k % RING_SLOTS].load(std::memory_order_acquire) < k) {
      if (stop_.load(std::memory_order_relaxed)) throw Error{BFSX_ERR_DEVICE, "copy stopped"};
      pause();
    }
  }
  void pass(uint64_t k) { passed_[k % RING_SLOTS].store(k + RING_SLOTS, std::memory_order_release); }

 private:
  std::atomic<uint64_t> next_{0}, passed_[RING_SLOTS] = {};
  std::atomic<bool> stop_{false};
  std::exception_ptr error_;
};

// A closed context's ring, one per device, kept for the next context (a second
// one is freed): pinning 16 MB and the first touches of its pages cost a
// program that makes a context per graph 1 to 3 ms for each.  Context, upload,
// search and close, us: 5 K vertices and 30 K edges 1500-1740 -> 700-890, 700 K
// and 4 M 4200-4500 -> 1900-3400 (the spread is the driver's: device memory
// freed just before is slow to come back).
constexpr int RING_DEVICES = 64;
std::mutex spare_mu;
uint8_t *spare_ring[RING_DEVICES];

// Pieces of `items` items of `width` bytes each at host address p: whole
// PIECE-sized pages of it (cut at multiples of 64 items).
struct Pieces {
  uint64_t items, head, per, n;
  Pieces(const void *p, uint64_t items_, size_t width) : items(items_), per(PIECE / width) {
    head = (PIECE - reinterpret_cast<uintptr_t>(p) % PIECE) / width / 64 * 64;
    n = items <= head ? (items ? 1 : 0) : 1 + (items - head + per - 1) / per;
  }
  uint64_t first(uint64_t k) const { return k == 0 ? 0 : head + (k - 1) * per; }
  uint64_t count(uint64_t k) const { return std::min(items, head + k * per) - first(k); }
};

// Whether p is memory that the runtime knows (pinned, managed, device): such
// copies go straight.
bool known_memory(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// Copies `items` items, `width` bytes each at dst, from the card through the
// ring, `ring_width` bytes each there: issue(first, count, offset in the
// ring) queues some, take(first, count, ring pointer) moves some to the
// caller's memory.  The card's side works in batches of whole pieces, about
// four per copy, at least a piece and at most what a slot holds (a launch and
// its event cost some 8 us of the caller's time: with one per piece the 16 MB
// of an R-MAT 22 search's levels took 215 us instead of 150).
template <class Issue, class Take>
void stream_out(bfsx_ctx *ctx, const void *dst, uint64_t items, size_t width, size_t ring_width,
                bool after_search, Issue issue, Take take) {
  if (items * width <= SMALL) {
    issue(0, items, 0);
    if (after_search) {
      BFSX_HIP(hipEventRecord(ctx->ring_ev[0], ctx->stream));
      BFSX_HIP(hipEventSynchronize(ctx->ring_ev[0]));
    } else {
      BFSX_HIP(hipStreamSynchronize(ctx->stream));
    }
    take(0, items, ctx->ring);
    return;
  }
  const Pieces P(dst, items, width);
  const uint64_t B = std::max<uint64_t>(1, std::min<uint64_t>(P.n / 4, width / ring_width));
  const uint64_t batches = (P.n + B - 1) / B;
  auto at = [](uint64_t j) { return (size_t)(j % RING_SLOTS) * PIECE; };
  auto first = [&](uint64_t j) { return P.first(j * B); };
  auto end = [&](uint64_t j) {
    const uint64_t k = std::min(P.n, (j + 1) * B) - 1;
    return P.first(k) + P.count(k);
  };
  auto queue = [&](uint64_t j) {
    if (end(j) > first(j)) issue(first(j), end(j) - first(j), at(j));
    BFSX_HIP(hipEventRecord(ctx->ring_ev[j % RING_SLOTS], ctx->stream));
  };
  std::atomic<uint64_t> taken[RING_SLOTS] = {};
  for (uint64_t j = 0; j < batches && j < RING_SLOTS; j++) queue(j);
  Crew::run(ctx, P.n, [&](Crew &c, uint64_t k) {
    const uint64_t j = k / B;
    c.turn(j);  // (a batch is queued by whoever moved the last piece of its slot's last one)
    BFSX_HIP(hipEventSynchronize(ctx->ring_ev[j % RING_SLOTS]));
    if (P.count(k))
      take(P.first(k), P.count(k), ctx->ring + at(j) + (P.first(k) - first(j)) * ring_width);
    const uint64_t of = std::min(P.n, (j + 1) * B) - j * B;
    if (taken[j % RING_SLOTS].fetch_add(1, std::memory_order_acq_rel) + 1 < of) return;
    taken[j % RING_SLOTS].store(0, std::memory_order_relaxed);
    if (j + RING_SLOTS < batches) queue(j + RING_SLOTS);
    c.pass(j);
  });
}

}  // namespace

void take_ring(bfsx_ctx *ctx) {
  uint8_t *p = nullptr;
  if (ctx->device < RING_DEVICES) {
    std::lock_guard<std::mutex> g(spare_mu);
    std::swap(p, spare_ring[ctx->device]);
  }
  // (a device reset in between has taken it away)
  if (p && !known_memory(p)) p = nullptr;
  if (!p) BFSX_HIP(hipHostMalloc((void **)&p, RING_PIECE_BYTES * RING_SLOTS, hipHostMallocMapped));
  ctx->ring = p;
  BFSX_HIP(hipHostGetDevicePointer((void **)&ctx->ring_dev, p, 0));
}

void give_ring(bfsx_ctx *ctx) {
  uint8_t *p = ctx->ring;
  ctx->ring = ctx->ring_dev = nullptr;
  if (p && ctx->device < RING_DEVICES) {
    std::lock_guard<std::mutex> g(spare_mu);
    if (!spare_ring[ctx->device]) std::swap(p, spare_ring[ctx->device]);
  }
  if (p) (void)hipHostFree(p);
}

void copy_out(bfsx_ctx *ctx, void *dst, const void *src, size_t bytes, bool after_search) {
  if (bytes == 0) return;
  if (known_memory(dst)) {
    BFSX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    BFSX_HIP(hipStreamSynchronize(ctx->stream));
    return;
  }
  stream_out(
      ctx, dst, bytes, 1, 1, after_search,
      [&](uint64_t first, uint64_t n, size_t at) {
        BFSX_HIP(hipMemcpyAsync(ctx->ring + at, static_cast<const uint8_t *>(src) + first, n,
                                hipMemcpyDeviceToHost, ctx->stream));
      },
      [&](uint64_t first, uint64_t n, const uint8_t *slot) {
        std::memcpy(static_cast<uint8_t *>(dst) + first, slot, n);
      });
}

void copy_levels_out(bfsx_ctx *ctx, int32_t *dst, const int32_t *levels, uint32_t n,
                     uint32_t max_level) {
  const int width = max_level < 255 ? 1 : max_level < 65535 ? 2 : 4;
  if (width == 4 || known_memory(dst)) {
    copy_out(ctx, dst, levels, sizeof(int32_t) * (size_t)n, true);
    return;
  }
  stream_out(
      ctx, dst, n, sizeof(int32_t), width, true,
      [&](uint64_t first, uint64_t k, size_t at) {
        const dim3 grid((unsigned)((k + 2047) / 2048)), block(256);
        if (width == 1)
          hipLaunchKernelGGL(k_narrow_levels<uint8_t>, grid, block, 0, ctx->stream,
                             levels + first, (uint32_t)k, ctx->ring_dev + at);
        else
          hipLaunchKernelGGL(k_narrow_levels<uint16_t>, grid, block, 0, ctx->stream,
                             levels + first, (uint32_t)k, reinterpret_cast<uint16_t *>(ctx->ring_dev + at));
        BFSX_HIP(hipGetLastError());
      },
      [&](uint64_t first, uint64_t k, const uint8_t *slot) {
        widen(slot, dst + first, k, width);
      });
}

// A copy of known memory, or of up to SMALL bytes through slot `at` of the
// ring, is queued here; the caller waits for it.
static bool queue_in(bfsx_ctx *ctx, void *dst, const void *src, size_t bytes, int at) {
  const void *from = src;
  if (!known_memory(src)) {
    if (bytes > SMALL) return false;
    from = std::memcpy(ctx->ring + at * PIECE, src, bytes);
  }
  BFSX_HIP(hipMemcpyAsync(dst, from, bytes, hipMemcpyHostToDevice, ctx->stream));
  return true;
}

void copy_in_both(bfsx_ctx *ctx, void *dst0, const void *src0, size_t bytes0, void *dst1,
                  const void *src1, size_t bytes1) {
  if (bytes0 && !queue_in(ctx, dst0, src0, bytes0, 0)) copy_in(ctx, dst0, src0, bytes0);
  const bool queued = !bytes1 || queue_in(ctx, dst1, src1, bytes1, 1);
  BFSX_HIP(hipStreamSynchronize(ctx->stream));  // (before the ring is used again)
  if (!queued) copy_in(ctx, dst1, src1, bytes1);
}

void copy_in(bfsx_ctx *ctx, void *dst, const void *src, size_t bytes) {
  if (bytes == 0) return;
  if (queue_in(ctx, dst, src, bytes, 0)) {
    BFSX_HIP(hipStreamSynchronize(ctx->stream));
    return;
  }
  const Pieces P(src, bytes, 1);
  Crew::run(ctx, P.n, [&](Crew &c, uint64_t k) {
    uint8_t *slot = ctx->ring + (k % RING_SLOTS) * PIECE;
    c.turn(k);
    if (k >= RING_SLOTS) BFSX_HIP(hipEventSynchronize(ctx->ring_ev[k % RING_SLOTS]));
    std::memcpy(slot, static_cast<const uint8_t *>(src) + P.first(k), P.count(k));
    if (P.count(k))
      BFSX_HIP(hipMemcpyAsync(static_cast<uint8_t *>(dst) + P.first(k), slot, P.count(k),
                              hipMemcpyHostToDevice, ctx->stream));
    BFSX_HIP(hipEventRecord(ctx->ring_ev[k % RING_SLOTS], ctx->stream));
    c.pass(k);
  });
  BFSX_HIP(hipStreamSynchronize(ctx->stream));
}

}  // namespace bfsx
