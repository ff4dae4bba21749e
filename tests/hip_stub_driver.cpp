// The engine's host side (libbfsx.so) on the CPU, over a stand-in for the HIP
// runtime: device memory is host memory behind a limit, copies and fills run
// at once, kernel launches do nothing but are counted.  The executable's
// definitions come before the runtime library's.  For what happens before and
// between kernels: what a refused call has touched, and which memory is held
// when an allocation fails.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "bfsx_internal.hpp"

// ---- the stand-in --------------------------------------------------------------
static std::mutex mu;
static std::map<void *, size_t> blocks;  // device memory
static size_t live = 0, limit = 1u << 30, launches = 0;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> g(mu);
  if (n > limit || live > limit - n) return hipErrorOutOfMemory;
  *p = calloc(n, 1);
  if (!*p) return hipErrorOutOfMemory;
  blocks[*p] = n;
  live += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> g(mu);
  auto it = blocks.find(p);
  if (it == blocks.end()) return p ? hipErrorInvalidValue : hipSuccess;
  live -= it->second;
  blocks.erase(it);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = calloc(n, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) {
  return hipErrorInvalidValue;  // no pointer of the callers is the runtime's
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {  // (the header's versioned name)
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 65536;
  p->warpSize = 64;
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
  *g = *b = dim3(1);
  *m = 0;
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  launches++;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(&launches); }
void __hipRegisterFunction(void **, const void *, char *, const char *, int, void *, void *, void *,
                           void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}

// ---- the checks ----------------------------------------------------------------
static bfsx_ctx *ctx;

#define CHECK(x)                                                                  \
  do {                                                                            \
    if (!(x)) {                                                                   \
      fprintf(stderr, "line %d: %s (last error: %s)\n", __LINE__, #x, bfsx_last_error(ctx)); \
      exit(1);                                                                    \
    }                                                                             \
  } while (0)

static bool says(const char *text) { return strstr(bfsx_last_error(ctx), text) != nullptr; }

// n bytes that end where the process may not read on
static void *fenced(size_t n) {
  const size_t page = 4096, room = (n + page - 1) / page * page;
  char *p = static_cast<char *>(
      mmap(nullptr, room + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
  mprotect(p + room, page, PROT_NONE);
  return p + room - n;
}

// n vertices with k entries each: the k vertices that follow
template <class P> struct Cycle {
  std::vector<P> cp;
  std::vector<uint32_t> ri;
  explicit Cycle(uint32_t n, uint32_t k = 1) : cp(n + 1), ri((size_t)n * k) {
    for (uint32_t i = 0; i <= n; i++) cp[i] = (P)i * k;
    for (size_t i = 0; i < ri.size(); i++) ri[i] = (uint32_t)((i / k + i % k + 1) % n);
  }
  int upload() {
    const uint32_t n = (uint32_t)cp.size() - 1;
    return bfsx_upload_csc(ctx, n, n, cp.data(), sizeof(P), ri.data(), ri.size(), 0);
  }
  // whether this is the resident graph
  bool resident() {
    std::vector<P> c(cp.size());
    std::vector<uint32_t> r(ri.size());
    bfsx_graph_info g;
    return bfsx_graph_info_get(ctx, &g) == BFSX_OK && g.nnz == ri.size() &&
           g.col_ptr_bytes == (int)sizeof(P) &&
           bfsx_download_csc(ctx, c.data(), r.data()) == BFSX_OK && c == cp && r == ri;
  }
};

static void reset() {
  limit = (size_t)1 << 30;
  bfsx_destroy(ctx);
  if (bfsx_create(0, &ctx) != BFSX_OK) exit(2);
}

// A caller's nnz above col_ptr's end: refused before row_idx is read, with
// room for the arrays and without.
template <class P> static void wrong_nnz() {
  Cycle<P> old(100);
  for (uint32_t n : {1u, 5u, 1000u, 300000u}) {
    P *cp = static_cast<P *>(fenced(sizeof(P) * (n + 1)));
    uint32_t *ri = static_cast<uint32_t *>(fenced(4 * (size_t)n));
    const Cycle<P> g(n);
    memcpy(cp, g.cp.data(), sizeof(P) * (n + 1));
    memcpy(ri, g.ri.data(), 4 * (size_t)n);
    for (uint64_t nnz : {(uint64_t)n + 1, (uint64_t)n + 70000, (uint64_t)n + (3u << 20),
                         (uint64_t)1 << 45, ((uint64_t)1 << 62) + n})
      for (size_t room : {(size_t)1 << 30, (size_t)0}) {
        limit = 1u << 30;
        CHECK(old.upload() == BFSX_OK);
        limit = room ? room : live;
        CHECK(bfsx_upload_csc(ctx, n, n, cp, sizeof(P), ri, nnz, 0) == BFSX_ERR_ARG);
        CHECK(says("col_ptr end does not match nnz"));
        CHECK(old.resident());
      }
    limit = 1u << 30;
    CHECK(bfsx_upload_csc(ctx, n, n, cp, sizeof(P), ri, n, 0) == BFSX_OK);
  }
}

// A graph that replaces another needs room for both graphs' arrays at most
// until it is accepted, not beside its own search state.
template <class P> static void replace() {
  Cycle<P> old(1000, 8000), next(4000000);  // many entries; many vertices
  CHECK(next.upload() == BFSX_OK);
  const size_t alone = live;
  reset();
  CHECK(old.upload() == BFSX_OK);
  const size_t margin = alone / 8, arrays = sizeof(P) * next.cp.size() + 4 * next.ri.size();
  CHECK(live + arrays < alone + margin);  // both graphs fit while it is checked
  limit = alone + margin;
  CHECK(next.upload() == BFSX_OK);
  CHECK(next.resident());
}

// Memory that ends at any of the allocations of a new graph's search state:
// afterwards there is no graph, and no call launches anything on one.
static void state_oom() {
  Cycle<uint32_t> old(100), next(500000);
  CHECK(next.upload() == BFSX_OK);
  const size_t alone = live;
  int failed = 0;
  for (size_t room = 1 << 20; room < alone + (alone >> 2); room += 100000) {
    reset();
    CHECK(old.upload() == BFSX_OK);
    limit = room > live ? room : live;
    const int rc = next.upload();
    if (rc == BFSX_OK) {
      CHECK(next.resident());
      continue;
    }
    CHECK(rc == BFSX_ERR_NOMEM);
    bfsx_graph_info g;
    if (bfsx_graph_info_get(ctx, &g) == BFSX_OK) {  // (failed before the old one was given up)
      CHECK(old.resident());
      continue;
    }
    failed++;
    const size_t before = launches;
    std::vector<int32_t> lev(next.ri.size());
    bfsx_run_stats st;
    for (int strategy : {BFSX_LLB, BFSX_GLB, BFSX_LEARNED, BFSX_BEAMER})
      CHECK(bfsx_run(ctx, 0, strategy, 0, lev.data(), nullptr, &st) == BFSX_ERR_STATE);
    CHECK(bfsx_order_adjacency(ctx, BFSX_ORDER_PULL_HUB_FIRST) == BFSX_ERR_STATE);
    CHECK(launches == before);
    limit = (size_t)1 << 30;
    CHECK(next.upload() == BFSX_OK);
    CHECK(next.resident());
  }
  CHECK(failed > 5);
}

// Memory held by the context's arrays, without its spare buffers (which it
// gives back when an allocation fails).
static size_t held() {
  limit = live;
  double ms;
  CHECK(bfsx_stream_copy(ctx, 1 << 26, 1, &ms) == BFSX_ERR_NOMEM);
  return live;
}

// An ordering that fails on its way leaves nothing of the bottom-up copy.
static void order_oom() {
  Cycle<uint32_t> g(200000, 3);
  CHECK(g.upload() == BFSX_OK);
  const size_t plain = held();
  int failed = 0;
  for (size_t room = 0; room < 12u << 20; room += 250000) {
    reset();
    CHECK(g.upload() == BFSX_OK);
    CHECK(held() == plain);
    limit = live + room;
    // (also with memory to spare: the kernels do nothing here, so that the
    // copy's counts do not agree)
    CHECK(bfsx_order_adjacency(ctx, BFSX_ORDER_PULL_HUB_FIRST) != BFSX_OK);
    failed += says("hipMalloc");
    bfsx_graph_info i;
    CHECK(bfsx_graph_info_get(ctx, &i) == BFSX_OK);
    CHECK(!(i.flags & BFSX_GRAPH_PULL_COPY) && i.pull_hubs == 0 && i.hot_vertices == 0);
    limit = (size_t)1 << 30;
    CHECK(g.resident());
    CHECK(held() <= plain + (1 << 16));  // (the checks' scratch)
  }
  CHECK(failed > 5);
}

// Tiles shared by groups: every part the rule wants while they fit a launch.
static void launch_size() {
  for (uint32_t wg = 64; wg <= 1024; wg *= 2)
    for (uint64_t F : {1ull, 255ull, 1ull << 20, 1000000007ull, 1100000000ull, 2147483647ull,
                       2147483649ull, 4294967295ull - 1024})
      for (uint32_t parts : {1u, 2u, 3u, 4u, 5u, 63u, 64u}) {
        const uint32_t tiles = (uint32_t)((F + wg - 1) / wg);
        const uint32_t got = bfsx::launch_parts(parts, tiles, wg);
        const uint64_t tile_threads = (uint64_t)tiles * wg;
        CHECK(got >= 1 && got <= parts);
        CHECK(got * tile_threads < 1ull << 32);
        CHECK(got == parts || (got + 1) * tile_threads >= 1ull << 32);
      }
}

// No room for a graph beside the resident one: it is checked on the host,
// refused with the resident one kept, or takes its place.
template <class P> static void no_room() {
  Cycle<P> old(300000, 20);
  const Cycle<P> good(250000, 22);
  CHECK(old.upload() == BFSX_OK);
  limit = live + (1u << 16);
  auto refused = [&](Cycle<P> g, const char *text) {
    CHECK(g.upload() == BFSX_ERR_ARG);
    CHECK(says(text));
    CHECK(old.resident());
  };
  for (uint32_t at : {1u, 125000u, 249999u}) {
    Cycle<P> g(good);
    g.cp[at] = (P)g.ri.size() + 5;
    refused(g, "col_ptr is not monotone");
    g = good;
    g.ri[at] = 250000;
    refused(g, "row_idx entry >= n_cols");
  }
  Cycle<P> g(good);
  g.ri.back() = 0xFFFFFFFFu;
  refused(g, "row_idx entry >= n_cols");
  g = good;
  g.ri.pop_back();
  refused(g, "col_ptr end does not match nnz");
  g = good;
  CHECK(g.upload() == BFSX_OK);
  CHECK(g.resident());
}

// Memory that ends anywhere in a call that makes temporaries: they are given
// back, and with the context everything is.
static void leaks() {
  const size_t empty = held();
  int failed = 0;
  for (size_t room = 0; room < 8u << 20; room += 150000) {
    reset();
    CHECK(held() == empty);
    uint64_t nnz;
    uint32_t off[3], roots[4];
    double ms;
    const int scales[2] = {9, 12}, factors[2] = {8, 8};
    const uint64_t seeds[2] = {1, 2};
    std::vector<float> X(8 * 4000), W(BFSX_SCHED_PARAMS), Y(4 * 4000);
    for (int call = 0; call < 6; call++) {
      limit = live + room;
      int rc = BFSX_OK;
      if (call == 0) rc = bfsx_generate_rmat(ctx, 13, 8, 0.57, 0.19, 0.19, 1, 2, 4, &nnz);
      if (call == 1) rc = bfsx_generate_grid(ctx, 150, 0.05, 9, 1, 8, &nnz);
      if (call == 2)
        rc = bfsx_generate_rmat_union(ctx, 2, scales, factors, seeds, seeds, 4, off, &nnz);
      if (call == 3) rc = bfsx_mlp_forward(ctx, X.data(), 4000, W.data(), Y.data());
      if (call == 4) rc = bfsx_stream_copy(ctx, 1 << 20, 1, &ms);
      if (call == 5) rc = bfsx_pick_roots(ctx, 4, 1, 2, roots, nullptr);
      failed += rc == BFSX_ERR_NOMEM;
      bfsx_graph_info g;
      if (bfsx_graph_info_get(ctx, &g) != BFSX_OK)  // (what a graph holds is not a leak)
        CHECK(held() <= empty + (2 << 20));  // (state that the next graph takes over)
    }
    limit = (size_t)1 << 30;
  }
  CHECK(failed > 20);
}

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (bfsx_create(0, &ctx) != BFSX_OK) return 2;
  if (what == "wrong_nnz") {
    wrong_nnz<uint32_t>();
    wrong_nnz<uint64_t>();
  } else if (what == "replace") {
    replace<uint32_t>();
    reset();
    replace<uint64_t>();
  } else if (what == "state_oom") {
    state_oom();
  } else if (what == "order_oom") {
    order_oom();
  } else if (what == "launch_size") {
    launch_size();
  } else if (what == "no_room") {
    no_room<uint32_t>();
    reset();
    no_room<uint64_t>();
  } else if (what == "leaks") {
    leaks();
  } else {
    return 2;
  }
  bfsx_destroy(ctx);
  ctx = nullptr;
  if (live != 0) {
    fprintf(stderr, "%zu bytes of device memory left\n", live);
    return 1;
  }
  printf("%s ok\n", what.c_str());
  return 0;
}
