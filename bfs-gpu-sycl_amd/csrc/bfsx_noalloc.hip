// Allocation-free single-source search: bfsx_run_noalloc.
//
// A variant of bfsx_run for callers that cannot allocate device memory.  The
// caller holds the CSC graph and the level array in device memory; the
// search state -- the visited bitmap, the two frontier queues and their
// counters -- lives in `scratch`, a fixed device array of this file (one copy
// per GPU, held until the process ends).  Host code never passes the array's
// name to a kernel: its device address is looked up once per device with
// hipGetSymbolAddress and kept in na_base[].  No call here allocates.
//
// The level loop runs on the device: the host queues, for a few levels at a
// time, an expansion (k_na_expand), a compaction (k_na_compact) and the level
// end, which goes on to run tiny levels by itself (k_na_tiny), all reading
// the frontier's size, edge count and level from the counters, and then
// copies the counters once.  A level's work is shared by edges (the groups
// of k_na_expand take slices of tiles of 256 frontier entries).  Levels with
// few edges discover exact-once (an atomicOr on the visited bitmap elects the
// lane that writes the level and appends the vertex, one atomicAdd per
// work-group and round for the slots); heavy ones store a mark byte for every
// edge whose target was unvisited at the level's start (all writers store the
// same value, no atomic), and the compaction turns marks into levels, visited
// bits and the next queue.  The marks (one byte per vertex, zero between
// levels) lie at the end of the buffer of the queue being expanded, which a
// frontier reaches only on graphs of more than 3.3 M vertices, most of them
// in one level; the levels after such a one discover exact-once.  The state is
// re-initialised by every call (visited bitmap, counters, root), so calls do
// not depend on what an earlier call left in the array; calls that overlap
// on one GPU race on it.
#include <mutex>
#include <string>

#include "bfsx_internal.hpp"

namespace bfsx {
namespace {

constexpr uint32_t NA_MAX = BFSX_NOALLOC_MAX_VERTICES;
constexpr size_t NA_CTL_BYTES = 256;                          // counters
constexpr size_t NA_VIS_BYTES = (size_t)NA_MAX / 8;           // visited bitmap
constexpr size_t NA_Q_BYTES = ((size_t)(NA_MAX + 1) * 4 + 255) / 256 * 256;  // one queue
constexpr size_t NA_BYTES = NA_CTL_BYTES + NA_VIS_BYTES + 2 * NA_Q_BYTES;
static_assert(NA_BYTES == BFSX_NOALLOC_SCRATCH_BYTES, "scratch size in bfsx.h");

__device__ __align__(256) uint8_t scratch[NA_BYTES];

struct NaCtl {
  uint32_t count[2];            // entries in queue 0 / 1
  uint32_t bad;                 // a col_ptr or row_idx entry out of range was seen
  uint32_t level;               // levels expanded so far
  uint32_t cur;                 // queue holding the frontier
  uint32_t done;                // the frontier is empty
  uint32_t dirty;               // a queue ran into its marks: no marking any more
  unsigned long long visited_edges;  // of all frontiers so far, the current one included
  uint32_t pad_[22];
  unsigned long long edges[2];  // out-degree sums of queue 0 / 1 (atomics: a line of their own)
};
static_assert(sizeof(NaCtl) <= NA_CTL_BYTES, "counters");

template <typename PtrT> struct NaGraph {
  const PtrT *col_ptr;
  const uint32_t *row_idx;
  uint64_t nnz;
  uint32_t n_rows, n_cols;
  int32_t *levels;
};

struct NaState {
  NaCtl *ctl;
  uint32_t *vis;
  uint32_t *q[2];
  uint4 *mark[2];   // n_cols bytes at the end of each queue's buffer
  uint32_t q_free;  // entries of a queue in front of its marks
};

constexpr int NA_MAX_DEVICES = 64;
std::mutex na_mu;
void *na_base[NA_MAX_DEVICES];  // device address of scratch, per device

__device__ __forceinline__ uint32_t na_lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

constexpr int NA_EPT = 4;              // edges per lane and round
constexpr uint32_t NA_WG = 256;        // frontier entries per tile
constexpr uint32_t NA_ROUND = NA_WG * NA_EPT;
constexpr uint32_t NA_PART_ROUNDS = 4, NA_MAX_PARTS = 64;
constexpr uint32_t NA_TINY_WG = 1024, NA_TINY_EDGES = 2048, NA_TINY_LEVELS = 4096;
constexpr uint32_t NA_COMPACT_VERTICES = 8192;  // per work-group of the compaction

// List of vertex v; an entry pair outside the graph (col_ptr beyond nnz or
// decreasing) is flagged and cut to the part inside.
template <typename PtrT>
__device__ __forceinline__ void na_list(const NaGraph<PtrT> &g, uint32_t v, uint32_t *bad,
                                        uint64_t &b, uint64_t &deg) {
  b = (uint64_t)g.col_ptr[v];
  uint64_t e = (uint64_t)g.col_ptr[v + 1];
  if (e > g.nnz || b > e) {
    atomicOr(bad, 1u);
    e = e > g.nnz ? g.nnz : e;
    b = b > e ? e : b;
  }
  deg = e - b;
}

// Which levels mark and compact: the engine's rule with its default ratio
// (from n * 4 / 1024 edges on with at least 8 per frontier vertex, from n/16
// in any case).
__device__ __forceinline__ bool na_marks(const NaCtl *ctl, unsigned long long EF, uint32_t F,
                                         uint32_t n) {
  if (ctl->dirty) return false;
  const unsigned long long lo = ((unsigned long long)n * 4 + 1023) / 1024;
  const unsigned long long hi = ((unsigned long long)n + 15) / 16;
  return EF >= (lo > hi ? lo : hi) || (EF >= lo && EF >= 8ull * F);
}

template <class T> __device__ __forceinline__ T na_wave_scan(T x) {
  const int l = __lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T y = __shfl_up(x, d, 64);
    if (l >= d) x += y;
  }
  return x;
}

// Exclusive scan over a work-group of N threads; s holds N / 64 + 1 entries
// and is free again after the next barrier.
template <int N, class T>
__device__ __forceinline__ T na_block_scan(T x, T &total, T *s) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const T inc = na_wave_scan(x);
  if (l == 63) s[w] = inc;
  __syncthreads();
  if (w == 0) {
    const T v = l < N / 64 ? s[l] : T(0);
    const T vi = na_wave_scan(v);
    if (l < N / 64) s[l] = vi - v;
    if (l == N / 64 - 1) s[N / 64] = vi;
  }
  __syncthreads();
  total = s[N / 64];
  return s[w] + inc - x;
}

// levels -1 except the root (0), visited = {root}, queue 0 = {root}
template <typename PtrT>
__global__ __launch_bounds__(256) void k_na_init(NaGraph<PtrT> g, NaState s, uint32_t root,
                                                 uint32_t n_words, int vec) {
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t n4 = vec ? g.n_cols / 4 : 0;  // (vec: levels 16-byte aligned)
  for (uint32_t i = t0; i < n4; i += stride) {
    const uint32_t d = root - i * 4;
    reinterpret_cast<int4 *>(g.levels)[i] =
        make_int4(d == 0 ? 0 : -1, d == 1 ? 0 : -1, d == 2 ? 0 : -1, d == 3 ? 0 : -1);
  }
  for (uint32_t i = n4 * 4 + t0; i < g.n_cols; i += stride) g.levels[i] = i == root ? 0 : -1;
  for (uint32_t w = t0; w < n_words; w += stride)
    s.vis[w] = w == (root >> 5) ? 1u << (root & 31) : 0u;
  const uint32_t n16 = (g.n_cols + 15) / 16;
  for (uint32_t i = t0; i < n16; i += stride)
    s.mark[0][i] = s.mark[1][i] = make_uint4(0, 0, 0, 0);
  if (t0 == 0) {
    s.q[0][0] = root;
    s.ctl->bad = 0;
    uint64_t b, deg = 0;
    if (root < g.n_rows) na_list(g, root, &s.ctl->bad, b, deg);
    s.ctl->count[0] = 1;
    s.ctl->count[1] = 0;
    s.ctl->level = s.ctl->cur = s.ctl->done = s.ctl->dirty = 0;
    s.ctl->edges[0] = deg;
    s.ctl->edges[1] = 0;
    s.ctl->visited_edges = deg;
  }
}

// Expands the frontier: a tile of NA_WG entries is scanned by each of the
// groups that share it, and every group takes a slice of its edges, NA_EPT
// consecutive ones per lane and round.  Entries outside the graph are
// skipped and flagged, never dereferenced.  What bounds a heavy level is the
// rate of random reads (the visited word of every edge, and, where many
// edges lead to each new vertex, its mark, which saves most of the stores):
// R-MAT 22, 130 M edges, whole call 15.5 -> 1.12 ms against one wave per
// frontier vertex with an atomic per new edge and a host round trip a level
// (marking in the 4-byte levels instead of mark bytes: 1.33 ms).
template <typename PtrT>
__global__ __launch_bounds__(NA_WG) void k_na_expand(NaGraph<PtrT> g, NaState s) {
  __shared__ uint64_t s_start[NA_WG], s_scan[NA_WG], s_wave[NA_WG / 64 + 1];
  __shared__ uint32_t s_wave32[NA_WG / 64 + 1];
  __shared__ uint32_t s_base;
  __shared__ unsigned long long s_edges;
  NaCtl *ctl = s.ctl;
  const uint32_t t = threadIdx.x, cur = ctl->cur;
  const uint32_t F = ctl->count[cur];
  const unsigned long long EF = ctl->edges[cur];
  if (ctl->done || F == 0) return;  // (uniform over the launch)
  if (t == 0) s_edges = 0;          // (barriers follow)
  const int32_t next_level = (int32_t)ctl->level + 1;
  const bool mark = na_marks(ctl, EF, F, g.n_cols);
  uint8_t *marks = reinterpret_cast<uint8_t *>(s.mark[cur]);
  const bool probe = g.n_cols >= (1u << 21) && EF >= 8ull * g.n_cols &&
                     (ctl->visited_edges - EF) * 4 < g.nnz;
  const uint32_t *q_in = s.q[cur];
  uint32_t *q_out = s.q[cur ^ 1];
  const uint32_t n_tiles = (F + NA_WG - 1) / NA_WG;
  const unsigned long long per_part = (unsigned long long)NA_ROUND * NA_PART_ROUNDS * n_tiles;
  const unsigned long long want = (EF + per_part - 1) / per_part;
  const uint32_t parts = want < 1 ? 1u : want > NA_MAX_PARTS ? NA_MAX_PARTS : (uint32_t)want;
  unsigned long long dacc = 0;
  for (uint32_t i = blockIdx.x; i < n_tiles * parts; i += gridDim.x) {
    const uint32_t tile = i % n_tiles, part = i / n_tiles;
    const uint32_t idx = tile * NA_WG + t;
    uint64_t st = 0, deg = 0;
    if (idx < F) {
      const uint32_t v = q_in[idx];
      if (v < g.n_rows) na_list(g, v, &ctl->bad, st, deg);
    }
    __syncthreads();  // the previous tile's arrays are no longer read
    uint64_t total;
    const uint64_t ex = na_block_scan<NA_WG>(deg, total, s_wave);
    s_start[t] = st;
    s_scan[t] = ex;
    __syncthreads();
    uint64_t per = total / parts + 1;
    per = per < NA_ROUND ? NA_ROUND : (per + NA_EPT - 1) / NA_EPT * NA_EPT;
    const uint64_t lo = part * per < total ? part * per : total;
    const uint64_t hi = total - lo > per ? lo + per : total;
    for (uint64_t r0 = lo; r0 < hi; r0 += NA_ROUND) {
      const uint64_t base = r0 + t * NA_EPT;
      uint32_t j = 0;
#pragma unroll
      for (uint32_t step = NA_WG / 2; step > 0; step >>= 1)
        if (s_scan[j + step] <= base) j += step;
      uint32_t n[NA_EPT], word[NA_EPT];
      uint64_t at[NA_EPT];
      bool cand[NA_EPT];
#pragma unroll
      for (int k = 0; k < NA_EPT; k++) {
        const uint64_t e = base + k;
        cand[k] = e < hi;
        while (cand[k] && j + 1 < NA_WG && s_scan[j + 1] <= e) j++;
        at[k] = cand[k] ? s_start[j] + (e - s_scan[j]) : 0;
      }
#pragma unroll
      for (int k = 0; k < NA_EPT; k++) n[k] = g.row_idx[at[k]];  // (hi > lo: nnz > 0)
#pragma unroll
      for (int k = 0; k < NA_EPT; k++) {
        if (cand[k] && n[k] >= g.n_cols) {
          atomicOr(&ctl->bad, 1u);
          cand[k] = false;
        }
        n[k] = cand[k] ? n[k] : 0u;
      }
#pragma unroll
      for (int k = 0; k < NA_EPT; k++) word[k] = s.vis[n[k] >> 5];
#pragma unroll
      for (int k = 0; k < NA_EPT; k++) cand[k] = cand[k] && !((word[k] >> (n[k] & 31)) & 1u);
      if (mark) {
        uint8_t seen[NA_EPT];
#pragma unroll
        for (int k = 0; k < NA_EPT; k++) seen[k] = 0;
        if (probe) {  // (uniform)
#pragma unroll
          for (int k = 0; k < NA_EPT; k++) seen[k] = marks[cand[k] ? n[k] : 0u];
        }
#pragma unroll
        for (int k = 0; k < NA_EPT; k++)
          if (cand[k] && !seen[k]) marks[n[k]] = 1;
        continue;
      }
      uint32_t cnt = 0;
      bool any = false;
#pragma unroll
      for (int k = 0; k < NA_EPT; k++) any = any || cand[k];
      if (any) {
        uint32_t old[NA_EPT];
#pragma unroll
        for (int k = 0; k < NA_EPT; k++)
          old[k] = atomicOr(&s.vis[n[k] >> 5], cand[k] ? 1u << (n[k] & 31) : 0u);
#pragma unroll
        for (int k = 0; k < NA_EPT; k++) {
          cand[k] = cand[k] && !((old[k] >> (n[k] & 31)) & 1u);
          if (cand[k]) {
            g.levels[n[k]] = next_level;
            cnt++;
            if (n[k] < g.n_rows) {
              uint64_t b, d;
              na_list(g, n[k], &ctl->bad, b, d);
              dacc += d;
            }
          }
        }
      }
      uint32_t found;
      const uint32_t slot = na_block_scan<NA_WG>(cnt, found, s_wave32);
      if (t == 0 && found) s_base = atomicAdd(&ctl->count[cur ^ 1], found);
      __syncthreads();
      if (cnt) {
        uint32_t p = s_base + slot;
#pragma unroll
        for (int k = 0; k < NA_EPT; k++)
          if (cand[k]) q_out[p++] = n[k];
      }
      __syncthreads();  // s_base and s_wave32 are rewritten by the next round
    }
  }
  if (mark) return;  // (uniform; the compaction adds up the degrees)
  dacc = na_wave_scan(dacc);
  if ((t & 63) == 63 && dacc) atomicAdd(&s_edges, dacc);
  __syncthreads();
  if (t == 0 && s_edges) atomicAdd(&ctl->edges[cur ^ 1], s_edges);
}

// 4-bit mask of the non-zero bytes (0 or 1 each) of w.
__device__ __forceinline__ uint32_t na_nibble(uint32_t w) {
  return (w & 1u) | ((w >> 7) & 2u) | ((w >> 14) & 4u) | ((w >> 21) & 8u);
}

// After a marking level: marks into levels, visited bits and the next queue,
// and cleared.  A work-group owns 8192 vertices (whole bitmap words), a lane
// 16 consecutive ones at a time; one atomic per group for the slots and one
// for the edge count, on different lines.
template <typename PtrT>
__global__ __launch_bounds__(256) void k_na_compact(NaGraph<PtrT> g, NaState s) {
  __shared__ uint32_t s_bits[NA_COMPACT_VERTICES / 32];
  __shared__ uint32_t s_wave32[5];
  __shared__ uint32_t s_base;
  __shared__ unsigned long long s_edges;
  static_assert(NA_COMPACT_VERTICES / 32 == 256, "a word per thread");
  NaCtl *ctl = s.ctl;
  const uint32_t t = threadIdx.x, cur = ctl->cur;
  const uint32_t F = ctl->count[cur];
  if (ctl->done || F == 0 || !na_marks(ctl, ctl->edges[cur], F, g.n_cols)) return;
  const int32_t next_level = (int32_t)ctl->level + 1;
  const uint32_t v0 = blockIdx.x * NA_COMPACT_VERTICES;
  const uint32_t n16 = (g.n_cols + 15) / 16;
  uint16_t *s_half = reinterpret_cast<uint16_t *>(s_bits);
  if (t == 0) s_edges = 0;
  uint32_t m[NA_COMPACT_VERTICES / 4096];
  unsigned long long dacc = 0;
#pragma unroll
  for (uint32_t r = 0; r < NA_COMPACT_VERTICES / 4096; r++) {
    const uint32_t i = v0 / 16 + r * 256 + t;
    const uint4 x = s.mark[cur][i < n16 ? i : 0u];
    m[r] = i < n16 ? na_nibble(x.x) | (na_nibble(x.y) << 4) | (na_nibble(x.z) << 8) |
                         (na_nibble(x.w) << 12)
                   : 0u;
  }
#pragma unroll
  for (uint32_t r = 0; r < NA_COMPACT_VERTICES / 4096; r++) {
    const uint32_t i = v0 / 16 + r * 256 + t;
    s_half[r * 256 + t] = (uint16_t)m[r];
    if (m[r]) s.mark[cur][i] = make_uint4(0, 0, 0, 0);
    for (uint32_t b = m[r]; b; b &= b - 1) {
      const uint32_t v = i * 16 + (__ffs(b) - 1);
      g.levels[v] = next_level;
      if (v < g.n_rows) {
        uint64_t st, d;
        na_list(g, v, &ctl->bad, st, d);
        dacc += d;
      }
    }
  }
  dacc = na_wave_scan(dacc);
  __syncthreads();
  if ((t & 63) == 63 && dacc) atomicAdd(&s_edges, dacc);
  const uint32_t bits = s_bits[t];
  uint32_t found;
  const uint32_t slot = na_block_scan<256>((uint32_t)__popc(bits), found, s_wave32);
  if (!found) return;  // (uniform)
  if (t == 0) s_base = atomicAdd(&ctl->count[cur ^ 1], found);
  if (t == 64 && s_edges) atomicAdd(&ctl->edges[cur ^ 1], s_edges);
  if (bits) s.vis[v0 / 32 + t] |= bits;
  __syncthreads();
  uint32_t p = s_base + slot;
  uint32_t *q_out = s.q[cur ^ 1];
  for (uint32_t b = bits; b; b &= b - 1) q_out[p++] = v0 + t * 32 + (__ffs(b) - 1);
}

// The end of a level that k_na_expand ran (`after`), then tiny levels, one
// work-group: up to NA_TINY_EDGES edges each, the counters and the next
// frontier's lists in LDS, the visited bits set with work-group-scope
// atomics (no other group runs).  A level costs its chain of dependent reads
// (list, visited word, atomic beside col_ptr), not launches.
template <typename PtrT>
__global__ __launch_bounds__(NA_TINY_WG) void k_na_tiny(NaGraph<PtrT> g, NaState s, int after) {
  __shared__ uint64_t s_nstart[NA_TINY_WG], s_start[NA_TINY_WG];
  __shared__ uint32_t s_ndeg[NA_TINY_WG], s_scan[NA_TINY_WG];
  __shared__ uint32_t s_wave[NA_TINY_WG / 64 + 1];
  __shared__ uint32_t s_count;
  __shared__ unsigned long long s_edges;
  NaCtl *ctl = s.ctl;
  const uint32_t t = threadIdx.x, lane = t & 63;
  if (ctl->done) return;  // (uniform, as is all that the loop tests)
  uint32_t cur = ctl->cur, level = ctl->level;
  uint32_t F = ctl->count[cur];
  unsigned long long EF = ctl->edges[cur], VE = ctl->visited_edges;
  uint32_t dirty = ctl->dirty;
  if (after && F) {  // the frontier has been expanded into the other queue
    cur ^= 1;
    level++;
    F = ctl->count[cur];
    EF = ctl->edges[cur];
    VE += EF;
    if (F > s.q_free) dirty = 1;
  }
  // this thread's entry of the frontier's first tile
  uint64_t st = 0;
  uint32_t deg = 0;
  auto load = [&](uint32_t i) {
    deg = 0;
    if (i < F) {
      const uint32_t v = s.q[cur][i];
      uint64_t d;
      if (v < g.n_rows) {
        na_list(g, v, &ctl->bad, st, d);
        deg = (uint32_t)d;  // (at most EF)
      }
    }
  };
  if (F <= NA_TINY_EDGES && EF <= NA_TINY_EDGES) load(t);
  for (uint32_t it = 0; it < NA_TINY_LEVELS; it++) {
    if (F == 0 || F > NA_TINY_EDGES || EF > NA_TINY_EDGES) break;
    uint32_t *q_out = s.q[cur ^ 1];
    if (t == 0) {
      s_count = 0;
      s_edges = 0;
    }
    unsigned long long dacc = 0;
    for (uint32_t e0 = 0; e0 < F; e0 += NA_TINY_WG) {
      if (e0 > 0) load(e0 + t);
      uint32_t total;
      const uint32_t ex = na_block_scan<NA_TINY_WG>(deg, total, s_wave);
      s_scan[t] = ex;
      s_start[t] = st;
      __syncthreads();
      // (at most NA_TINY_EDGES edges: two per thread)
      for (uint32_t r0 = 0; r0 < total; r0 += NA_TINY_WG) {
        const uint32_t e = r0 + t;
        uint32_t j = 0;
#pragma unroll
        for (uint32_t step = NA_TINY_WG / 2; step > 0; step >>= 1)
          if (s_scan[j + step] <= e) j += step;
        bool isnew = e < total;
        uint32_t n = g.row_idx[isnew ? s_start[j] + (e - s_scan[j]) : 0];
        if (isnew && n >= g.n_cols) {
          atomicOr(&ctl->bad, 1u);
          isnew = false;
        }
        n = isnew ? n : 0u;
        const uint32_t bit = 1u << (n & 31);
        isnew = isnew && !(s.vis[n >> 5] & bit);
        uint64_t nst = 0, nd = 0;
        if (isnew) {
          const uint32_t old = __hip_atomic_fetch_or(&s.vis[n >> 5], bit, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_WORKGROUP);
          if (n < g.n_rows) na_list(g, n, &ctl->bad, nst, nd);
          isnew = !(old & bit);
        }
        if (isnew) {
          g.levels[n] = (int32_t)level + 1;
          dacc += nd;
        }
        const unsigned long long m = __ballot(isnew);
        uint32_t slot = 0;
        if (lane == 0 && m) slot = atomicAdd(&s_count, (uint32_t)__popcll(m));
        slot = __shfl(slot, 0, 64) + na_lanes_below(m);
        if (isnew) {
          q_out[slot] = n;
          if (slot < NA_TINY_WG) {
            s_nstart[slot] = nst;
            s_ndeg[slot] = nd > NA_TINY_EDGES ? NA_TINY_EDGES : (uint32_t)nd;  // (not used then)
          }
        }
      }
      __syncthreads();  // this tile's arrays are no longer read
    }
    dacc = na_wave_scan(dacc);
    if (lane == 63 && dacc) atomicAdd(&s_edges, dacc);
    __syncthreads();
    F = s_count;
    EF = s_edges;
    VE += EF;
    deg = 0;
    if (t < F) {
      st = s_nstart[t];
      deg = s_ndeg[t];
    }
    __syncthreads();  // the counters are zeroed by the next level
    cur ^= 1;
    level++;
  }
  if (t == 0) {
    ctl->cur = cur;
    ctl->level = level;
    ctl->count[cur] = F;
    ctl->edges[cur] = EF;
    ctl->count[cur ^ 1] = 0;
    ctl->edges[cur ^ 1] = 0;
    ctl->visited_edges = VE;
    ctl->dirty = dirty;
    ctl->done = F == 0;
  }
}

// Device address of this GPU's scratch array (looked up once per device,
// with that device current).
void *na_scratch(int device) {
  std::lock_guard<std::mutex> g(na_mu);
  if (!na_base[device]) {
    void *p = nullptr;
    BFSX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) fail(BFSX_ERR_DEVICE, "scratch array has no device address");
    na_base[device] = p;
  }
  return na_base[device];
}

template <typename PtrT>
uint32_t na_search(uint8_t *base, hipStream_t s, const PtrT *col_ptr, const uint32_t *row_idx,
                   uint64_t nnz, uint32_t n_cols, uint32_t n_rows, uint32_t root,
                   int32_t *levels, int cus) {
  const NaGraph<PtrT> g{col_ptr, row_idx, nnz, n_rows, n_cols, levels};
  const size_t mark_bytes = ((size_t)n_cols + 15) / 16 * 16;
  static_assert(NA_Q_BYTES % 16 == 0, "marks are 16-byte aligned");
  uint8_t *q0 = base + NA_CTL_BYTES + NA_VIS_BYTES, *q1 = q0 + NA_Q_BYTES;
  const NaState st{reinterpret_cast<NaCtl *>(base),
                   reinterpret_cast<uint32_t *>(base + NA_CTL_BYTES),
                   {reinterpret_cast<uint32_t *>(q0), reinterpret_cast<uint32_t *>(q1)},
                   {reinterpret_cast<uint4 *>(q0 + NA_Q_BYTES - mark_bytes),
                    reinterpret_cast<uint4 *>(q1 + NA_Q_BYTES - mark_bytes)},
                   (uint32_t)((NA_Q_BYTES - mark_bytes) / 4)};
  const uint32_t n_words = (n_cols + 31) / 32;
  const int vec = (reinterpret_cast<uintptr_t>(levels) & 15) == 0;
  const unsigned cap = (unsigned)cus * 8;
  const unsigned want = (n_cols + 1023) / 1024;
  hipLaunchKernelGGL(k_na_init<PtrT>, dim3(want < cap ? want : cap), dim3(256), 0, s, g, st, root,
                     n_words, vec);
  hipLaunchKernelGGL(k_na_tiny<PtrT>, dim3(1), dim3(NA_TINY_WG), 0, s, g, st, 0);
  BFSX_HIP(hipGetLastError());
  const unsigned compact = (n_cols + NA_COMPACT_VERTICES - 1) / NA_COMPACT_VERTICES;
  // Levels queued per copy of the counters: an R-MAT search has three or
  // four levels that are not tiny; a search that needs more gets longer
  // batches (a level after the end costs its empty launches, about 10 us, a
  // copy about 20 us).
  uint32_t batch = 4;
  for (;;) {
    for (uint32_t k = 0; k < batch; k++) {
      hipLaunchKernelGGL(k_na_expand<PtrT>, dim3(cap), dim3(NA_WG), 0, s, g, st);
      hipLaunchKernelGGL(k_na_compact<PtrT>, dim3(compact), dim3(256), 0, s, g, st);
      hipLaunchKernelGGL(k_na_tiny<PtrT>, dim3(1), dim3(NA_TINY_WG), 0, s, g, st, 1);
    }
    BFSX_HIP(hipGetLastError());
    NaCtl c;
    BFSX_HIP(hipMemcpyAsync(&c, st.ctl, sizeof(c), hipMemcpyDeviceToHost, s));
    BFSX_HIP(hipStreamSynchronize(s));
    if (c.done) {
      if (c.bad) fail(BFSX_ERR_ARG, "col_ptr or row_idx entry out of range");
      return c.level;
    }
    if (c.level > n_cols) fail(BFSX_ERR_DEVICE, "level loop did not terminate");
    batch = batch < 16 ? batch * 2 : batch;
  }
}

thread_local std::string na_error;

}  // namespace

const char *noalloc_last_error() { return na_error.c_str(); }

}  // namespace bfsx

extern "C" int bfsx_run_noalloc(int device, void *stream, const void *col_ptr, int col_ptr_bytes,
                                const uint32_t *row_idx, uint32_t n_cols, uint32_t n_rows,
                                uint64_t nnz, uint32_t root, int32_t *levels,
                                uint32_t *n_levels) {
  using namespace bfsx;
  int old = -1;
  try {
    if (!col_ptr || !levels || (nnz && !row_idx)) fail(BFSX_ERR_ARG, "null device pointer");
    if (col_ptr_bytes != 4 && col_ptr_bytes != 8) fail(BFSX_ERR_ARG, "col_ptr_bytes must be 4 or 8");
    if (n_cols == 0 || n_cols > NA_MAX)
      fail(BFSX_ERR_ARG, "n_cols must be in [1, BFSX_NOALLOC_MAX_VERTICES = " +
                             std::to_string(NA_MAX) + "]");
    if (n_rows > n_cols) fail(BFSX_ERR_ARG, "n_rows > n_cols");
    if (root >= n_cols) fail(BFSX_ERR_ARG, "root out of range");
    if (col_ptr_bytes == 4 && nnz > 0xFFFFFFFFull) fail(BFSX_ERR_ARG, "nnz does not fit 4-byte col_ptr");
    int n_dev = 0;
    if (hipGetDeviceCount(&n_dev) != hipSuccess || n_dev == 0) fail(BFSX_ERR_DEVICE, "no HIP device visible");
    if (device < 0 || device >= n_dev || device >= NA_MAX_DEVICES) fail(BFSX_ERR_ARG, "device index out of range");
    BFSX_HIP(hipGetDevice(&old));
    BFSX_HIP(hipSetDevice(device));
    int cus = 0;
    BFSX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    uint8_t *base = static_cast<uint8_t *>(na_scratch(device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t nl =
        col_ptr_bytes == 8
            ? na_search<uint64_t>(base, s, static_cast<const uint64_t *>(col_ptr), row_idx, nnz,
                                  n_cols, n_rows, root, levels, cus)
            : na_search<uint32_t>(base, s, static_cast<const uint32_t *>(col_ptr), row_idx, nnz,
                                  n_cols, n_rows, root, levels, cus);
    if (n_levels) *n_levels = nl;
    (void)hipSetDevice(old);
    na_error.clear();
    return BFSX_OK;
  } catch (const Error &e) {
    if (old >= 0) (void)hipSetDevice(old);
    na_error = e.msg;
    return e.status;
  } catch (...) {
    if (old >= 0) (void)hipSetDevice(old);
    na_error = "unknown failure";
    return BFSX_ERR_DEVICE;
  }
}
