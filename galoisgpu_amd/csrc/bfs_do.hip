// Direction-optimising BFS on gfx950, and the reverse CSR it needs.
//
// The levels are the reference's (apps/bfs/kernel.cu:20-32,312-334,380-393):
// level[src] = 0, first hop LEVEL 1, INF = INT_MAX for unreachable vertices.
// BFS levels are unique, so how a level is discovered does not change them.
// All levels run in one persistent launch with a grid barrier between them.
// A level is either
//   top-down:  the previous level's vertices -- queued when they were found, the
//              heavy ones as chunks of edges -- have their out-edges flattened
//              over each wavefront, and an unvisited destination is claimed with
//              an atomicMin on its level; or
//   bottom-up: every unvisited vertex scans its in-edges and stops at the
//              first parent that was visited before the level.
// The barrier leader picks the direction of the next level from the
// frontier's size and edge count (Beamer, Asanovic and Patterson's rule:
// bottom-up once the frontier's edges exceed 1/alpha of the unexplored edges,
// top-down again once the frontier holds fewer than 1/beta of the vertices;
// here also 1/gamma of all edges).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>

#include "engine.h"
#include "lsg_internal.h"
#include "runtime.h"
#include "scan_dev.h"
#include "wave_dev.h"

namespace lsg {

constexpr uint32_t kAlpha = 14, kBeta = 24, kGamma = 16;

// ---- reverse CSR by a stable radix sort ------------------------------------------
//
// The forward CSR lists edges by source, so sorting the (destination, source,
// weight) triples by destination with a stable sort gives each reverse row
// in ascending source order: the reverse CSR is the same on every call (a
// PageRank sum over in-edges has one order) and a bottom-up search meets low
// source ids first.  LSD radix sort, at most 8 bits per pass (the destination's
// bits spread evenly over the passes); each pass is a per-tile digit histogram,
// a prefix sum over (digit, tile), and a stable scatter.  No atomics on global
// memory: the atomic-counter version serialised on the in-degree counters of
// the hubs (RMAT-20: 4.3 ms).
//
// The scatter is bound by memory: 24 bytes per edge and pass.  A block ranks
// its tile's elements by digit (ballots within a wavefront, counters per
// wavefront), puts them in digit order through LDS and writes each digit's
// run, kRadixTile / 256 = 32 elements on average, as one (writing every element
// to its place as it was ranked: 1.27 ms per pass on RMAT-22, now 0.40: 3.9 TB/s).  The
// first pass finds the sources from the row starts, 64 rows at a time in the
// wavefront's lanes, instead of reading them from an array written before
// (0.81 ms).

constexpr int kRadixBlock = 512;
constexpr uint32_t kRadixTile = 8192;                        // elements per block
constexpr uint32_t kRadixPer = kRadixTile / kRadixBlock;     // per thread
constexpr uint32_t kRadixWave = kWave * kRadixPer;           // per wavefront, consecutive

struct RadixArgs {
  const uint32_t *row_start;               // first pass: forward row starts
  const uint32_t *key, *v1, *v2;           // v1 null: first pass; v2 null: zeros
  uint32_t *key_out, *v1_out, *v2_out;
  uint32_t *hist;                          // [256][ntiles] counts, then places within a scan tile
  const uint32_t *hist_tiles;              // the scan's tile offsets
  uint32_t n, V, shift, mask, ntiles;
};

// hist[d * ntiles + b] = elements of tile b whose digit is d.
__global__ __launch_bounds__(kRadixBlock) void radix_hist_kernel(RadixArgs a) {
  __shared__ uint32_t h[256];
  if (threadIdx.x < 256) h[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t base = blockIdx.x * kRadixTile, count = min(a.n - base, kRadixTile);
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    const uint32_t i = it * kRadixBlock + threadIdx.x;
    if (i < count) atomicAdd(&h[(a.key[base + i] >> a.shift) & a.mask], 1u);
  }
  __syncthreads();
  if (threadIdx.x <= a.mask) a.hist[(size_t)threadIdx.x * a.ntiles + blockIdx.x] = h[threadIdx.x];
}

// Writes the tile's values x[] (element of thread and step) in digit order:
// LDS place lp[], global place of thread i's p-th element in that order gp[].
__device__ __forceinline__ void radix_write(uint32_t *buf, const uint32_t (&x)[kRadixPer],
                                            const uint32_t (&lp)[kRadixPer], const uint32_t (&gp)[kRadixPer],
                                            uint32_t count, uint32_t *out) {
  __syncthreads();
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it)
    if (lp[it] < kRadixTile) buf[lp[it]] = x[it];
  __syncthreads();
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    const uint32_t p = it * kRadixBlock + threadIdx.x;
    if (p < count) out[gp[it]] = buf[p];
  }
}

// Stable scatter of tile b: the elements of digit d go to its place for (d, b)
// on, in tile order.
template <bool kFirst>
__global__ __launch_bounds__(kRadixBlock) void radix_scatter_kernel(RadixArgs a) {
  constexpr uint32_t NW = kRadixBlock / kWave;
  __shared__ uint32_t buf[kRadixTile];
  __shared__ uint32_t wcnt[NW][256];  // per wavefront: count, then LDS place of its first element of the digit
  __shared__ uint32_t goff[256];      // global place of a digit's run, less its LDS place
  __shared__ uint32_t wsum[4];
  const uint32_t lane = lane_id(), wv = threadIdx.x / kWave;
  const uint32_t base = blockIdx.x * kRadixTile, count = min(a.n - base, kRadixTile);
  const uint32_t first = wv * kRadixWave;  // this wavefront's elements in the tile
  for (uint32_t d = lane; d < 256; d += kWave) wcnt[wv][d] = 0;
  uint32_t k[kRadixPer], lp[kRadixPer], gp[kRadixPer];
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    const uint32_t i = first + it * kWave + lane;
    k[it] = a.key[base + min(i, count - 1)];
  }
  // rank within the wavefront's elements of the same digit
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    const bool valid = first + it * kWave + lane < count;
    const uint32_t d = (k[it] >> a.shift) & a.mask;
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (uint32_t bit = 0; bit < 8; ++bit) {
      const uint64_t m = __ballot((d >> bit) & 1u);
      peers &= ((d >> bit) & 1u) ? m : ~m;
    }
    const uint32_t below = lanes_below(peers), before = wcnt[wv][d];
    __builtin_amdgcn_wave_barrier();
    if (valid && below == 0) wcnt[wv][d] = before + (uint32_t)__builtin_popcountll(peers);
    __builtin_amdgcn_wave_barrier();
    lp[it] = valid ? before + below : kRadixTile;
  }
  __syncthreads();
  // per digit: the wavefronts' counts become offsets, the digits' totals places
  uint32_t total = 0, incl = 0;
  if (threadIdx.x < 256) {
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) {
      const uint32_t c = wcnt[w][threadIdx.x];
      wcnt[w][threadIdx.x] = total;
      total += c;
    }
    incl = total;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
      const uint32_t y = __shfl_up(incl, s);
      if (lane >= (uint32_t)s) incl += y;
    }
    if (lane == kWave - 1) wsum[wv] = incl;
  }
  __syncthreads();
  if (threadIdx.x < 256) {
    uint32_t start = incl - total;
    for (uint32_t w = 0; w < wv; ++w) start += wsum[w];
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) wcnt[w][threadIdx.x] += start;
    const size_t e = (size_t)threadIdx.x * a.ntiles + blockIdx.x;
    if (threadIdx.x <= a.mask) goff[threadIdx.x] = a.hist[e] + a.hist_tiles[e / kScanTile] - start;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    if (lp[it] < kRadixTile) {
      lp[it] += wcnt[wv][(k[it] >> a.shift) & a.mask];
      buf[lp[it]] = k[it];
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    const uint32_t p = it * kRadixBlock + threadIdx.x;
    gp[it] = 0;
    if (p < count) {
      const uint32_t x = buf[p];
      gp[it] = goff[(x >> a.shift) & a.mask] + p;
      a.key_out[gp[it]] = x;
    }
  }
  uint32_t x[kRadixPer];
  if (kFirst) {
    uint32_t u0 = 0, re = 0;  // 64 rows: the first, and the end of each
#pragma unroll
    for (uint32_t it = 0; it < kRadixPer; ++it) {
      const uint32_t i = base + first + it * kWave + lane;
      bool todo = lp[it] < kRadixTile;
      x[it] = 0;
      for (uint64_t m = __ballot(todo); m; m = __ballot(todo)) {
        const uint32_t e = readlane(i, (uint32_t)__builtin_ctzll(m));
        if (readlane(re, kWave - 1) <= e) {
          u0 = wave_row_near(a.row_start, a.V, e);
          re = glb(a.row_start)[min(u0 + lane, a.V - 1) + 1];
        }
        uint32_t pos = 0;  // rows that end at or before edge i
#pragma unroll
        for (uint32_t s = kWave / 2; s >= 1; s >>= 1)
          if (__shfl(re, pos + s - 1) <= i) pos += s;
        if (todo && i < readlane(re, kWave - 1)) {
          x[it] = u0 + pos;
          todo = false;
        }
      }
    }
  } else {
#pragma unroll
    for (uint32_t it = 0; it < kRadixPer; ++it) {
      const uint32_t i = first + it * kWave + lane;
      x[it] = a.v1[base + min(i, count - 1)];
    }
  }
  radix_write(buf, x, lp, gp, count, a.v1_out);
#pragma unroll
  for (uint32_t it = 0; it < kRadixPer; ++it) {
    const uint32_t i = first + it * kWave + lane;
    x[it] = a.v2 ? a.v2[base + min(i, count - 1)] : 0u;
  }
  radix_write(buf, x, lp, gp, count, a.v2_out);
}

// Row starts of the reverse CSR from the sorted destinations: the first
// position of each destination value, E for the vertices after the last.
__global__ void row_bounds_kernel(const uint32_t *dst, uint32_t E, uint32_t V, uint32_t *row) {
  const size_t nt = (size_t)gridDim.x * blockDim.x;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i <= E; i += nt) {
    const uint64_t first = i == 0 ? 0ull : (uint64_t)dst[i - 1] + 1;  // vertices whose row starts here
    const uint64_t last = i < E ? (uint64_t)dst[i] : (uint64_t)V;        // ... through this one
    for (uint64_t v = first; v <= last; ++v) row[v] = (uint32_t)i;
  }
}

// ---- the persistent traversal -------------------------------------------------
//
// All levels run in one co-resident launch, in the rounds of the wavefront
// kernels (wave_dev.h).  What bounds a level: the few large ones of a skewed
// graph, the random looks at levels and bitmaps; the many small ones of a road
// network, the chain of round trips between two barriers.
//   - A level is exact when it is found (an atomicMin on the level array whose
//     old value is INF), so no vertex is queued twice.  The row bounds of what
//     a wavefront found are read together at the end of the level: they give the
//     frontier's edges, which the direction rule needs, and take heavy vertices
//     apart into chunks, so that their edges are expanded with their level.
//   - Bottom-up levels read one bitmap of the visited vertices through the
//     caches and write the next (two take turns; while the caches' lines are
//     dropped once per block and level).  Any visited parent is a parent of the
//     last level: had it an earlier one, the vertex would be visited.  The
//     unvisited vertices of a few words are dealt one to a lane, 64 a step; when
//     few lanes still search, the wavefront takes their long rows in turn.
//     (64 consecutive vertices a step, visited or not: RMAT-22 0.33 ms, now 0.20.)
//     The words of a unit lie as far apart as there are units: hubs that follow
//     each other are many wavefronts' (10^6 leaves of 1000 hubs, words in a row /
//     apart: 0.85 / 0.40 ms, bottom-up only 10.6 / 1.2; RMAT-22 so 1.84 / 1.63).
//   - The first top-down level after those reads its frontier from the bitmaps.
//   - Small top-down levels are run by one block, as in wave.hip.
// Kernel ms (with a bitmap per level in place of queues, read through to the
// coherence point, and every block at each barrier -> now): RMAT-16 0.088 ->
// 0.061, RMAT-18 0.097 -> 0.070, RMAT-20 0.140 -> 0.105, RMAT-22 0.274 -> 0.195,
// top-down only 2.84 -> 0.67; road-like 512^2 1.70 -> 0.77, 2048^2 2.84 -> 1.58.
// Where RMAT-22 spends it: 45 us on the hub's chunks, 80 on the first bottom-up
// level, 20 on the second, 23 on two small levels, 30 on the initialisation.

constexpr int kDoBlock = 256;
constexpr uint32_t kDoHeavy = 256;     // out-degree from which a vertex's edges become chunks of that many
constexpr uint32_t kDoPush = 256;      // staged vertices per wavefront
constexpr uint32_t kDoHeavyBuf = 64;   // staged heavy vertices per wavefront, one a lane
constexpr uint32_t kDoLocalCap = 1024; // entries of a pile in LDS
constexpr uint32_t kDoWords = 16;      // most words of 64 vertices in a bottom-up unit
constexpr uint32_t kDoAlone = 8;       // lanes that still search, from which on rows of more than kDoLong edges
constexpr uint32_t kDoLong = 64;       // are taken in turn
constexpr int kDoFlight = 4;           // edges in flight per lane

// A round's WaveRound: round = its level, phase = how it is found, steps = the
// unexplored edges, cut = bottom-up levels before it, roles = in-queue | bitmap
// << 1.
enum DoMode : uint32_t { kDoQueue = 0, kDoUp = 1, kDoBits = 2 };

struct DoArgs : WaveArgs {
  const uint32_t *in_row, *in_src;  // reverse CSR
  uint64_t *bits[2];                // visited vertices
  uint64_t *in_any;                 // vertices with in-edges
  uint64_t *hchunk[2];              // chunks: edges << 32 | first edge
  uint32_t words;                   // of 64 vertices
  uint32_t direction;
};

struct DoHeavy {
  uint32_t first, deg;
};

template <int BS>
struct DoShared {
  static constexpr int NW = BS / kWave;
  uint32_t push[NW][kDoPush];
  DoHeavy heavy[NW][kDoHeavyBuf];
  uint32_t count[NW][4];  // end of a level: queued, chunks, found, their edges
  uint32_t base[2];
  uint64_t hits[NW][kDoWords];  // bottom-up: found in the unit
  WaveRound r;
  uint32_t gen;
  // levels of one block
  Entry pile[2][kDoLocalCap];
  uint32_t pile_n[2];
  uint32_t spill_n, chunk_n;  // handed to the queue and as chunks
  uint32_t stop;              // a heavy vertex was found
  uint32_t edges, last;       // of the vertices found; of those found last
  unsigned long long items;
};

// A wavefront's view of the level.
struct DoLane {
  uint32_t level;
  uint32_t *q, *tail;
  uint64_t *hq;
  uint32_t *htail;
  uint32_t *bits;  // visited, or null
  uint32_t *pbuf;
  DoHeavy *hbuf;
  uint32_t n, settled;       // staged vertices; the first `settled` have been counted (wave-uniform)
  uint32_t hn;               // staged heavy vertices (wave-uniform)
  uint32_t cnt, deg;         // found, and their edges (per lane)
};

// Writes the staged heavy vertices' chunks, counted in `end`, from slot `base` on.
__device__ __forceinline__ void do_store_heavy(const DoArgs &a, DoLane &w, uint32_t end, uint32_t base) {
  chunk_each(end, [&](uint32_t f, uint32_t item, uint32_t k) {
    const uint32_t pos = base + f, skip = k * kDoHeavy;
    const DoHeavy h = w.hbuf[item];
    if (pos < a.hcap) st_coh64(w.hq + pos, (uint64_t)min(h.deg - skip, kDoHeavy) << 32 | (h.first + skip));
    else st_coh(&a.ctrl->abort, kAbortCapacity);
  });
  w.hn = 0;
}
__device__ __forceinline__ uint32_t do_heavy_ends(const DoLane &w) {
  return chunk_ends(w.hn, lane_id() < w.hn ? w.hbuf[lane_id()].deg : 0u, kDoHeavy);
}

// Takes the lanes with `found` into account: vertex v, edges first to first +
// deg.  True for those to be queued, which are not heavy.
__device__ __forceinline__ bool do_found(const DoArgs &a, DoLane &w, bool found, uint32_t first, uint32_t deg) {
  if (found) {
    w.cnt += 1;
    w.deg += deg;
  }
  const bool heavy = found && deg >= kDoHeavy;
  const uint64_t m = __ballot(heavy);
  if (m) {
    const uint32_t c = (uint32_t)__builtin_popcountll(m);
    if (w.hn + c > kDoHeavyBuf) {
      const uint32_t end = do_heavy_ends(w);
      uint32_t base = 0;
      if (lane_id() == 0) base = atomic_add(w.htail, readlane(end, kWave - 1));
      do_store_heavy(a, w, end, readlane(base, 0));
    }
    if (heavy) w.hbuf[w.hn + lanes_below(m)] = DoHeavy{first, deg};
    w.hn += c;
  }
  return found && !heavy;
}

// Row bounds, bitmap and heavy vertices of what was staged since the last call;
// the others close up.
__device__ __forceinline__ void do_settle(const DoArgs &a, DoLane &w) {
  uint32_t out = w.settled;
  for (uint32_t i0 = w.settled; i0 < w.n; i0 += kWave) {
    const bool valid = i0 + lane_id() < w.n;
    const uint32_t v = valid ? w.pbuf[i0 + lane_id()] : 0u;
    const uint64_t rb = ld_pair(a.row_start + v);
    if (valid && w.bits) __hip_atomic_fetch_or(glb(w.bits + (v >> 5)), 1u << (v & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool keep = do_found(a, w, valid, (uint32_t)rb, (uint32_t)(rb >> 32) - (uint32_t)rb);
    const uint64_t m = __ballot(keep);
    if (keep) w.pbuf[out + lanes_below(m)] = v;
    out += (uint32_t)__builtin_popcountll(m);
  }
  w.n = w.settled = out;
}

__device__ __forceinline__ void do_store(const DoArgs &a, DoLane &w, uint32_t base) {
  for (uint32_t i = lane_id(); i < w.n; i += kWave) {
    const uint32_t pos = base + i;
    if (pos < a.qcap) st_coh(w.q + pos, w.pbuf[i]);
    else st_coh(&a.ctrl->abort, kAbortCapacity);
  }
  w.n = w.settled = 0;
}

// Stages v from every lane with `pred` (whole wavefront).
__device__ __forceinline__ void do_stage(const DoArgs &a, DoLane &w, bool pred, uint32_t v) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const uint32_t c = (uint32_t)__builtin_popcountll(m);
  if (w.n + c > kDoPush) {
    do_settle(a, w);
    uint32_t base = 0;
    if (lane_id() == 0 && w.n) base = atomic_add(w.tail, w.n);
    do_store(a, w, readlane(base, 0));
  }
  if (pred) w.pbuf[w.n + lanes_below(m)] = v;
  w.n += c;
}

// Top-down: visits the destinations of edges e[k] of the lanes with act[k]
// (e[k] names some edge in every lane).  `direct`: without a look at the level.
__device__ __forceinline__ void do_visit(const DoArgs &a, DoLane &w, const uint32_t (&e)[kDoFlight],
                                         const bool (&act)[kDoFlight], bool direct) {
  uint32_t v[kDoFlight], lv[kDoFlight], old[kDoFlight];
  bool any = false;
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) v[k] = glb(a.edge_dst)[e[k]];
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) lv[k] = kInf;
  if (!direct) {
    // through the caches: an old value is INF, and the atomicMin finds out
#pragma unroll
    for (int k = 0; k < kDoFlight; ++k) lv[k] = glb(a.dist)[v[k]];
  }
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) any |= act[k] && lv[k] == kInf;
  if (__ballot(any) == 0) return;
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) old[k] = act[k] && lv[k] == kInf ? atomic_min(a.dist + v[k], w.level) : 0u;
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) asm volatile("" : "+v"(old[k]));
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) do_stage(a, w, old[k] == kInf, v[k]);
}

// The edges first to first + deg of each lane, flattened over the wavefront.
__device__ __forceinline__ void do_expand(const DoArgs &a, DoLane &w, uint32_t first, uint32_t deg, bool direct) {
  const uint32_t lane = lane_id();
  uint32_t end = deg;  // inclusive prefix over the lanes
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = __shfl_up(end, d);
    if (lane >= (uint32_t)d) end += y;
  }
  const uint32_t total = readlane(end, kWave - 1);
  const uint32_t base = first - (end - deg);
  direct = direct && total <= 2 * kWave;
  for (uint32_t b0 = 0; b0 < total; b0 += kDoFlight * kWave) {
    uint32_t e[kDoFlight];
    bool act[kDoFlight];
#pragma unroll
    for (int k = 0; k < kDoFlight; ++k) {
      const uint32_t f = min(b0 + k * kWave + lane, total - 1);
      act[k] = b0 + k * kWave + lane < total;
      uint32_t pos = 0;  // lanes whose edges end at or before f
#pragma unroll
      for (uint32_t d = kWave / 2; d >= 1; d >>= 1)
        if ((uint32_t)__shfl(end, pos + d - 1) <= f) pos += d;
      e[k] = (uint32_t)__shfl(base, pos) + f;
    }
    do_visit(a, w, e, act, direct);
  }
}

// Up to 64 in-queue vertices, one per lane below n.
__device__ __forceinline__ void do_items(const DoArgs &a, DoLane &w, const uint32_t *in, uint32_t n, bool direct) {
  const uint32_t lane = lane_id();
  const uint32_t u = lane < n ? ld_coh(in + lane) : 0u;
  const uint64_t rb = ld_pair(a.row_start + u);
  do_expand(a, w, (uint32_t)rb, lane < n ? (uint32_t)(rb >> 32) - (uint32_t)rb : 0u, direct);
}

// One chunk of a heavy vertex.
__device__ __forceinline__ void do_chunk(const DoArgs &a, DoLane &w, const uint64_t *ent) {
  const uint64_t x = ld_coh64(ent);
  const uint32_t first = __builtin_amdgcn_readfirstlane((uint32_t)x), n = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  if (n == 0 || n > kDoHeavy || (uint64_t)first + n > a.nedges) return;
  static_assert(kDoHeavy == kDoFlight * kWave, "a chunk is one step");
  uint32_t e[kDoFlight];
  bool act[kDoFlight];
#pragma unroll
  for (int k = 0; k < kDoFlight; ++k) {
    const uint32_t f = k * kWave + lane_id();
    act[k] = f < n;
    e[k] = first + min(f, n - 1);
  }
  do_visit(a, w, e, act, false);
}

// Top-down from the bitmaps: the vertices of 64 words of 32, one word per lane,
// that `now` has and `before` has not.  (now also gets this level's vertices
// meanwhile, told apart by their level.)  Heavy ones come as chunks.
__device__ __forceinline__ void do_bit_items(const DoArgs &a, DoLane &w, const uint32_t *now, const uint32_t *before,
                                             uint32_t w0) {
  const uint32_t wi = w0 + lane_id();
  uint32_t b = 0;
  if (wi < 2 * a.words) b = ld_coh(now + wi) & ~ld_coh(before + wi);
  while (__ballot(b != 0)) {
    const uint32_t u = b ? wi * 32 + (uint32_t)__builtin_ctz(b) : 0u;
    const bool some = b != 0;
    b &= b - 1;
    const uint32_t lv = ld_coh(a.dist + u);
    const uint64_t rb = ld_pair(a.row_start + u);
    uint32_t deg = (uint32_t)(rb >> 32) - (uint32_t)rb;
    if (!some || lv != w.level - 1 || deg >= kDoHeavy) deg = 0;
    do_expand(a, w, (uint32_t)rb, deg, false);
  }
}

// The position of the n-th set bit of x (n < popcount).
__device__ __forceinline__ uint32_t nth_bit(uint64_t x, uint32_t n) {
  uint32_t pos = 0, w = (uint32_t)x;
  const uint32_t lo = (uint32_t)__builtin_popcount(w);
  if (n >= lo) {
    n -= lo;
    pos = 32;
    w = (uint32_t)(x >> 32);
  }
#pragma unroll
  for (uint32_t h = 16; h >= 1; h >>= 1) {
    const uint32_t c = (uint32_t)__builtin_popcount(w & ((1u << h) - 1));
    if (n >= c) {
      n -= c;
      pos += h;
      w >>= h;
    }
  }
  return pos;
}

// Bottom-up: the unvisited vertices with in-edges of up to kDoWords words (word0
// and every stride-th after it), one per lane and step.
__device__ __forceinline__ void do_up(const DoArgs &a, DoLane &w, const uint64_t *prev, uint64_t *next, uint32_t word0,
                                      uint32_t stride, uint64_t *hits) {
  const uint32_t lane = lane_id();
  const uint32_t own_word = word0 + lane * stride;
  const bool mine = lane < kDoWords && own_word < a.words;
  uint64_t seen = 0, open = 0;
  if (mine) {
    seen = ((const LSG_GLOBAL uint64_t *)prev)[own_word];
    open = ((const LSG_GLOBAL uint64_t *)a.in_any)[own_word] & ~seen;
  }
  uint32_t end = (uint32_t)__builtin_popcountll(open);  // inclusive prefix over the words
  const uint32_t own = end;
#pragma unroll
  for (int d = 1; d < (int)kDoWords; d <<= 1) {
    const uint32_t y = __shfl_up(end, d);
    if (lane >= (uint32_t)d) end += y;
  }
  const uint32_t total = readlane(end, kDoWords - 1);
  if (lane < kDoWords) hits[lane] = 0;
  // Bit 0: whether u was visited.  By a buffer load, which gives 0 for a source beyond
  // the bitmap (of a reverse graph that was changed after it was wrapped) at no cost:
  // tested with instructions RMAT-22 took 204 us, so 190.
  const __amdgpu_buffer_rsrc_t bitmap = __builtin_amdgcn_make_buffer_rsrc((void *)prev, 0, (int)(a.words * 8), 0x00027000);
  auto visited = [&](uint32_t u) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(bitmap, (int)((u >> 5) << 2), 0, 0) >> (u & 31);
  };
  for (uint32_t b0 = 0; b0 < total; b0 += kWave) {
    const uint32_t f = b0 + lane;
    uint32_t wd = 0;  // words that end at or before f
#pragma unroll
    for (uint32_t d = kDoWords / 2; d >= 1; d >>= 1)
      if ((uint32_t)__shfl(end, wd + d - 1) <= f) wd += d;
    const uint64_t bits = (uint64_t)(uint32_t)__shfl((uint32_t)(open >> 32), wd) << 32 | (uint32_t)__shfl((uint32_t)open, wd);
    const uint32_t before = (uint32_t)__shfl(end - own, wd);
    const bool valid = f < total;
    const uint32_t bit = valid ? nth_bit(bits, f - before) : 0u;
    const uint32_t v = valid ? (word0 + wd * stride) * kWave + bit : 0u;
    const uint64_t in = ld_pair(a.in_row + v), rb = ld_pair(a.row_start + v);
    uint32_t e = (uint32_t)in, e1 = valid ? (uint32_t)(in >> 32) : e;
    bool found = false;
    for (;;) {
      const uint64_t m = __ballot(e < e1);
      if (m == 0) break;
      uint64_t lone = __ballot(e1 - e > kDoLong);
      if (lone && (uint32_t)__builtin_popcountll(m) <= kDoAlone) {
        // few rows left: the wavefront takes the long ones in turn
        for (; lone; lone &= lone - 1) {
          const uint32_t l = (uint32_t)__builtin_ctzll(lone), hi = readlane(e1, l);
          bool hit = false;
          for (uint32_t p = readlane(e, l); p < hi && !hit; p += kDoFlight * kWave) {
            uint32_t u[kDoFlight], x[kDoFlight];
#pragma unroll
            for (int k = 0; k < kDoFlight; ++k) u[k] = glb(a.in_src)[min(p + k * kWave + lane, hi - 1)];
#pragma unroll
            for (int k = 0; k < kDoFlight; ++k) x[k] = visited(u[k]);
            uint32_t any = 0;
#pragma unroll
            for (int k = 0; k < kDoFlight; ++k) any |= x[k];
            hit = __ballot(any & 1u) != 0;
          }
          if (lane == l) {
            found = hit;
            e = e1;
          }
        }
        continue;
      }
      uint32_t u[kDoFlight], x[kDoFlight];
#pragma unroll
      for (int k = 0; k < kDoFlight; ++k) u[k] = glb(a.in_src)[e < e1 ? min(e + k, e1 - 1) : 0u];
#pragma unroll
      for (int k = 0; k < kDoFlight; ++k) x[k] = visited(u[k]);
      uint32_t any = 0;
#pragma unroll
      for (int k = 0; k < kDoFlight; ++k) any |= x[k];
      const bool hit = e < e1 && (any & 1u);
      found = found || hit;
      e = hit || e1 - e <= kDoFlight ? e1 : e + kDoFlight;
    }
    if (found) {
      st_coh(a.dist + v, w.level);
      atomicOr((unsigned long long *)&hits[wd], 1ull << bit);
    }
    if (__ballot(found)) do_found(a, w, found, (uint32_t)rb, (uint32_t)(rb >> 32) - (uint32_t)rb);
  }
  if (mine) st_coh64(next + own_word, seen | hits[lane]);
}

// Bottom-up once the frontier's edges exceed 1/kAlpha of the unexplored ones,
// and 1/kGamma of all: the tail of a road network meets the first test with a
// few vertices, whose top-down level costs its fixed round trips (road-like
// 2048^2: 15 of 147 levels bottom-up, 1.90 ms, without them 1.58).
__device__ __forceinline__ bool do_goes_up(const DoArgs &a, uint32_t edges, uint32_t unexplored) {
  return (uint64_t)edges * kAlpha > unexplored && (uint64_t)edges * kGamma > a.nedges;
}

// ---- levels of one block ----------------------------------------------------------

// The visits of such a level: what is found goes to the next pile in LDS, or,
// where that is full, to the queue or as chunks.
template <int BS>
struct DoLocal {
  const DoArgs &a;
  DoShared<BS> &sh;
  uint32_t nxt, level;
  uint32_t *q, *bits;
  uint64_t *hq;
  uint32_t &edges;
  __device__ __forceinline__ bool stopped() const { return false; }
  __device__ __forceinline__ void operator()(const KArgs &, const uint32_t (&v)[kInFlight],
                                             const uint32_t (&)[kInFlight], const bool (&act)[kInFlight]) const {
    uint32_t old[kInFlight];
    uint64_t rb[kInFlight], m[kInFlight];
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      old[k] = act[k] ? atomic_min(a.dist + v[k], level) : 0u;
      rb[k] = ld_pair(a.row_start + v[k]);
    }
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) asm volatile("" : "+v"(old[k]));
    uint32_t t = 0;
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      m[k] = __ballot(old[k] == kInf);
      t += (uint32_t)__builtin_popcountll(m[k]);
    }
    if (t == 0) return;
    uint32_t pos = 0;
    if (lane_id() == 0) pos = atomicAdd(&sh.pile_n[nxt], t);
    pos = readlane(pos, 0);
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      if (old[k] == kInf) {
        const uint32_t p = pos + lanes_below(m[k]);
        const Entry x{v[k], level, (uint32_t)rb[k], (uint32_t)(rb[k] >> 32)};
        edges += x.re - x.rs;
        if (x.re - x.rs >= kDoHeavy) sh.stop = 1;
        if (bits) __hip_atomic_fetch_or(glb(bits + (v[k] >> 5)), 1u << (v[k] & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (p < kDoLocalCap) sh.pile[nxt][p] = x;
        else spill(x);
      }
      pos += (uint32_t)__builtin_popcountll(m[k]);
    }
  }
  // A vertex that this mode hands on.
  __device__ __forceinline__ void spill(const Entry &x) const {
    const uint32_t deg = x.re - x.rs;
    if (deg < kDoHeavy) {
      const uint32_t pos = atomicAdd(&sh.spill_n, 1u);
      if (pos < a.qcap) st_coh(q + pos, x.v);
      else st_coh(&a.ctrl->abort, kAbortCapacity);
      return;
    }
    const uint32_t nch = (deg - 1) / kDoHeavy + 1, base = atomicAdd(&sh.chunk_n, nch);
    for (uint32_t k = 0; k < nch; ++k) {
      const uint32_t skip = k * kDoHeavy;
      if (base + k < a.hcap) st_coh64(hq + base + k, (uint64_t)min(deg - skip, kDoHeavy) << 32 | (x.rs + skip));
      else st_coh(&a.ctrl->abort, kAbortCapacity);
    }
  }
};

// Called by every thread of the block that leads, with the next level in sh.r
// (top-down, at most a.local_max vertices, no chunks): runs it and the levels
// that follow while they are small, and leaves in sh.r the level that the whole
// grid runs next, its chunks in hq.
template <int BS>
__device__ __forceinline__ void do_local(const DoArgs &a, DoShared<BS> &sh, uint64_t *hq) {
  WaveRound r = sh.r;
  if (threadIdx.x == 0) {
    sh.stop = sh.chunk_n = sh.edges = sh.last = 0;
    sh.items = 0;
  }
  uint32_t cur = 0, n = r.items, before = 0, edges = 0, popped = 0, levels = 0;
  const uint32_t *const in = a.q[r.roles & 1];
  uint32_t *const out = a.q[(r.roles & 1) ^ 1];
  uint32_t *const bits = a.direction == 0 ? (uint32_t *)a.bits[r.roles >> 1] : nullptr;
  for (uint32_t i = threadIdx.x; i < n; i += BS) {
    const uint32_t v = ld_coh(in + i);
    const uint64_t rb = ld_pair(a.row_start + v);
    sh.pile[0][i] = Entry{v, r.round - 1, (uint32_t)rb, (uint32_t)(rb >> 32)};
  }
  for (;;) {
    if (threadIdx.x == 0) {
      sh.pile_n[cur ^ 1] = 0;
      sh.spill_n = 0;
    }
    __syncthreads();
    before = edges;
    const DoLocal<BS> relax{a, sh, cur ^ 1, r.round, out, bits, hq, edges};
    expand_entries<Algo::BFS, kLdsAS, BS, true>(a, (EntryPtr<kLdsAS>)sh.pile[cur], n, relax, &sh.items);
    __syncthreads();  // every push of the level is in
    popped += n;
    ++levels;
    r.round += 1;
    const uint32_t found = sh.pile_n[cur ^ 1];
    if (threadIdx.x == 0) st_coh(&a.ctrl->progress, r.round);
    if (found > a.local_max || sh.stop) {
      for (uint32_t i = threadIdx.x; i < min(found, kDoLocalCap); i += BS) relax.spill(sh.pile[cur ^ 1][i]);
      break;
    }
    if (found == 0) {
      r.flags |= kWaveDone;
      break;
    }
    cur ^= 1;
    n = found;
    // (the next level's first barrier separates the reads of sh above from its writes)
  }
  if (edges) atomicAdd(&sh.edges, edges);
  if (edges - before) atomicAdd(&sh.last, edges - before);
  order_release();
  __syncthreads();
  if (threadIdx.x == 0) {
    r.items = r.flags & kWaveDone ? 0u : sh.spill_n;
    r.heavy = sh.chunk_n;
    r.roles ^= 1u;
    const uint32_t left = r.steps - min(r.steps, sh.edges - sh.last);
    // the rule of do_kernel's leader
    if (a.direction == 0 && !(r.flags & kWaveDone) && do_goes_up(a, sh.last, left)) {
      r.phase = kDoUp;
      r.heavy = 0;
    }
    r.steps = left - min(left, sh.last);
    sh.r = r;
    __hip_atomic_fetch_add(&a.ctrl->stat_items, (uint64_t)popped, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_add(&a.ctrl->stat_rounds, (uint64_t)levels, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
}

// ---- the kernel ---------------------------------------------------------------------

template <int BS>
__global__ __launch_bounds__(BS, 4) void do_kernel(DoArgs a) {
  constexpr uint32_t NW = BS / kWave;
  __shared__ DoShared<BS> sh;
  Ctrl *const c = a.ctrl;
  WaveCtrl *const wc = a.wc;
  const uint32_t nb = gridDim.x, wv = threadIdx.x / kWave;
  const uint32_t wave = blockIdx.x * NW + wv, nwaves = nb * NW;
  const uint32_t ngroups = min(kTicketGroups, nb), g = blockIdx.x % ngroups;
  const uint32_t gblocks = (nb + ngroups - 1 - g) / ngroups;  // blocks of this group
  if (!residency_handshake(c, nb, a.residency_limit)) return;
  if (threadIdx.x == 0) {
    // the first level, written before this launch
    WaveRound x;
    memset(&x, 0, sizeof x);
    x.items = c->s.in_count;
    x.heavy = c->s.heavy_count;
    x.round = 1;
    x.phase = c->s.aux[0];
    x.steps = c->s.aux[3];
    sh.r = x;
    sh.gen = 0;
  }
  __syncthreads();
  DoLane w;
  w.pbuf = sh.push[wv];
  w.hbuf = sh.heavy[wv];
  w.n = w.settled = w.hn = 0;
  for (;;) {
    const WaveRound r = sh.r;
    const uint32_t gen = sh.gen;
    if (r.flags & kWaveDone) break;
    WaveCtrl::Slot *const slot = &wc->slot[gen % 3];
    const uint32_t qi = r.roles & 1, bi = r.roles >> 1;
    w.level = r.round;
    w.q = qi ? a.q[0] : a.q[1];
    w.tail = &slot->near_tail.n;
    w.hq = gen & 1 ? a.hchunk[1] : a.hchunk[0];
    w.htail = &slot->heavy_tail.n;
    uint64_t *const now = bi ? a.bits[1] : a.bits[0], *const other = bi ? a.bits[0] : a.bits[1];
    w.bits = a.direction == 0 ? (uint32_t *)now : nullptr;
    w.cnt = w.deg = 0;
    // Units: bottom-up, up to kDoWords words, dealt in turn.  Top-down, in-queue items
    // (`per` at a time) or bitmap words, then chunks: as in wave_kernel.
    const bool up = r.phase == kDoUp;
    const uint32_t per = min((uint32_t)kWave, max(a.unit_min, (r.items + nwaves - 1) / nwaves));
    const uint32_t upw = min(kDoWords, (a.words + nwaves - 1) / nwaves);
    const uint32_t nitem = up ? (a.words + upw - 1) / upw : r.phase == kDoBits ? (2 * a.words + kWave - 1) / kWave : (r.items + per - 1) / per;
    const uint32_t nunits = nitem + (up ? 0u : r.heavy);
    const bool many = nunits > nwaves;
    if (up) {
      for (uint32_t i = wave; i < nunits; i += nwaves) do_up(a, w, now, other, i, nunits, sh.hits[wv]);
    } else {
      const uint32_t *const in = qi ? a.q[1] : a.q[0];
      const uint64_t *const hin = gen & 1 ? a.hchunk[0] : a.hchunk[1];
      const bool direct = r.items <= kDirectMax;
      uint32_t unit = many ? (blockIdx.x / ngroups * NW + wv) * ngroups + g : wave;
      while (unit < nunits) {
        uint32_t t = 0;
        if (many && lane_id() == 0) t = atomic_add(&slot->ticket[g].n, 1u);
        if (unit >= nitem) do_chunk(a, w, hin + (unit - nitem));
        else if (r.phase == kDoBits) do_bit_items(a, w, (const uint32_t *)now, (const uint32_t *)other, unit * kWave);
        else do_items(a, w, in + (size_t)unit * per, min(per, r.items - unit * per), direct);
        if (!many) break;
        unit = (gblocks * NW + readlane(t, 0)) * ngroups + g;
      }
      do_settle(a, w);
    }
    uint32_t cnt = w.cnt, deg = w.deg;
#pragma unroll
    for (int k = kWave / 2; k >= 1; k >>= 1) {
      cnt += __shfl_xor(cnt, k);
      deg += __shfl_xor(deg, k);
    }
    // The block's vertices and chunks get their places with one atomic each.
    const uint32_t hend = w.hn ? do_heavy_ends(w) : 0u;
    order_release();
    if (lane_id() == kWave - 1) {
      sh.count[wv][0] = w.n;
      sh.count[wv][1] = hend;
      sh.count[wv][2] = cnt;
      sh.count[wv][3] = deg;
    }
    __syncthreads();
    uint32_t tot[4] = {0, 0, 0, 0}, off[2] = {0, 0};
#pragma unroll
    for (uint32_t i = 0; i < NW; ++i)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        if (p < 2 && i < wv) off[p] += sh.count[i][p];
        tot[p] += sh.count[i][p];
      }
    if (tot[2]) {
      if (threadIdx.x < 2) {
        const uint32_t n = threadIdx.x == 0 ? tot[0] : tot[1];
        sh.base[threadIdx.x] = n ? atomic_add(threadIdx.x == 0 ? w.tail : w.htail, n) : 0u;
      } else if (threadIdx.x == 2) {
        __hip_atomic_fetch_add(reinterpret_cast<uint64_t *>(&slot->sum[g]), (uint64_t)tot[3] << 32 | tot[2],
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (w.n) do_store(a, w, sh.base[0] + off[0]);
      if (w.hn) do_store_heavy(a, w, hend, sh.base[1] + off[1]);
      order_release();
      __syncthreads();
    }
    // The barrier, as in wave_kernel.
    if (wv == 0) {
      const uint32_t active = many ? nb : (nunits + NW - 1) / NW;
      const uint32_t parties = active + (r.lead >= active ? 1u : 0u);
      const uint32_t seat = blockIdx.x < active ? blockIdx.x : blockIdx.x == r.lead ? active : parties;
      const uint32_t lane = lane_id();
      if (seat < parties && wave_arrive(slot, seat, parties)) {
        order_acquire();
        WaveRound x = r;
        uint64_t sum = lane < ngroups ? ld_coh64(reinterpret_cast<const uint64_t *>(&slot->sum[lane])) : 0ull;
        const uint32_t word = ld_coh(lane == 0 ? w.tail : lane == 1 ? w.htail : &c->abort);
#pragma unroll
        for (int k = kTicketGroups / 2; k >= 1; k >>= 1) sum += __shfl_xor((unsigned long long)sum, k);
        const uint32_t found = readlane((uint32_t)sum, 0), edges = readlane((uint32_t)(sum >> 32), 0);
        const uint32_t queued = readlane(word, 0), chunks = readlane(word, 1), ab = readlane(word, 2);
        // (the slot of the round before the last: no block reads it any more)
        WaveCtrl::Slot *const next = &wc->slot[(gen + 2) % 3];
        const uint32_t nclear = offsetof(WaveCtrl::Slot, arrive) / sizeof(WaveCtrl::Line) + (nb + kBarGroup - 1) / kBarGroup;
        for (uint32_t i = lane; i < nclear; i += kWave)
          st_coh64(reinterpret_cast<uint64_t *>(reinterpret_cast<WaveCtrl::Line *>(next) + i), 0ull);
        const bool full = queued > a.qcap || chunks > a.hcap;
        if (full) st_coh(&c->abort, kAbortCapacity);
        const bool done = full || ab != kAbortNone || found == 0;
        // top-down again below 1/kBeta of the vertices
        const bool small = chunks == 0 && queued <= a.local_max;
        bool next_up = up;
        if (a.direction == 0) {
          if (!up && !small && do_goes_up(a, edges, r.steps)) next_up = true;
          else if (up && (uint64_t)found * kBeta < a.nnodes) next_up = false;
        }
        x.steps = r.steps - min(r.steps, edges);
        x.cut = r.cut + (up ? 1u : 0u);
        x.round = r.round + 1;
        x.lead = blockIdx.x;
        x.phase = next_up ? kDoUp : up ? kDoBits : kDoQueue;
        x.items = up ? found : queued;
        x.heavy = next_up ? 0u : chunks;
        x.roles = (qi ^ 1) | (up ? bi ^ 1 : bi) << 1;
        x.flags = kWaveLead | (done ? kWaveDone : x.phase == kDoQueue && chunks == 0 && queued <= a.local_max / 2 ? kWaveLocal : 0u);
        if (lane == 0) {
          __hip_atomic_fetch_add(&c->stat_items, (uint64_t)r.items, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_fetch_add(&c->stat_rounds, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          sh.r = x;
          sh.gen = gen + 1;
        }
      } else {
        WaveRound x = r;
        const uint32_t tag = wave_wait(a, gen, x);
        if (lane == 0) {
          sh.r = x;
          sh.gen = tag;
        }
      }
    }
    __syncthreads();
    if (sh.r.flags & kWaveLead) {
      if (sh.r.flags & kWaveLocal) do_local<BS>(a, sh, w.hq);
      if (wv == 0) {
        const WaveRound x = sh.r;
        wave_publish(wc, gen + 1, x);
        if ((x.flags & kWaveDone) && lane_id() == 0) {
          c->s.done = 1;
          c->s.round = x.round;
          c->s.phase = x.cut;
        }
      }
    }
    // the bitmap was written by every block: no line read before is kept
    if (!(sh.r.flags & kWaveDone) && sh.r.phase == kDoUp) {
      if (wv == 0) acquire_agent();
      __syncthreads();
    }
  }
}

// level = INF except src = 0; bitmap 0 = {src}; the control words and the first
// level: src, or its chunks if it is heavy.
__global__ void do_init_kernel(DoArgs a, uint32_t src) {
  const uint32_t nt = gridDim.x * blockDim.x, t = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t v = t; v < a.nnodes; v += nt) glb(a.dist)[v] = v == src ? 0u : kInf;
  const uint32_t span = a.words * kWave;
  for (uint32_t v = t; v < span; v += nt) {
    const bool in = v < a.nnodes && a.in_row[v + 1] != a.in_row[v];
    const uint64_t m = __ballot(in);
    if (lane_id() == 0) {
      a.in_any[v / kWave] = m;
      a.bits[0][v / kWave] = v / kWave == src / kWave ? 1ull << (src % kWave) : 0ull;
    }
  }
  const uint32_t rs = a.row_start[src], deg = a.row_start[src + 1] - rs;
  const uint32_t nch = deg >= kDoHeavy ? (deg - 1) / kDoHeavy + 1 : 0u;
  for (uint32_t k = t; k < nch; k += nt)
    a.hchunk[1][k] = (uint64_t)min(deg - k * kDoHeavy, kDoHeavy) << 32 | (rs + k * kDoHeavy);
  Ctrl *c = a.ctrl;
  ctrl_reset_barrier(c, t, nt);
  if (blockIdx.x == 0) wave_reset(a.wc, threadIdx.x, blockDim.x);
  if (t == 0) {
    c->abort = kAbortNone;
    c->checkin = 0;
    c->resident_seen = 0;
    c->progress = 0;
    c->stat_items = c->stat_rounds = c->stat_heavy = c->stat_phases = c->stat_edges = 0;
    a.q[0][0] = src;
    Sched s;
    memset(&s, 0, sizeof s);
    s.round = 1;
    s.in_count = nch ? 0u : 1u;
    s.heavy_count = nch;
    const bool up = a.direction == 2 || (a.direction == 0 && (uint64_t)deg * kAlpha > a.nedges);
    s.aux[0] = up ? kDoUp : kDoQueue;
    s.aux[3] = (uint32_t)a.nedges - deg;
    c->s = s;
  }
}

static int check_device_graph(const lsg_graph *g, const char *what) {
  if (!g || g->device_graph == 0 || !g->row_start || (g->nedges && !g->edge_dst))
    return fail(LSG_ERR_ARG, "%s: expected a device graph (copy_to_gpu first)", what);
  return LSG_OK;
}

}  // namespace lsg

using namespace lsg;

extern "C" {

int lsg_graph_transpose(const lsg_graph *g, lsg_graph *gt) {
  clear_error();
  int rc = check_device_graph(g, "transpose");
  if (rc) return rc;
  if (!gt) return fail(LSG_ERR_ARG, "transpose: NULL output graph");
  Workspace *w;
  if ((rc = get_workspace(g->device, &w))) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  HIPCHK(hipSetDevice(w->device));
  const uint32_t V = g->nnodes, E = g->nedges;
  // (destination, source, weight) triples sorted by destination; pass p writes
  // slot (P - p) & 1, so the last pass lands in slot 1, the output arrays.
  uint32_t bits = 0;
  while (bits < 32 && (V > 1 ? (uint64_t)(V - 1) >> bits : 0) != 0) ++bits;
  const uint32_t P = std::max<uint32_t>(1, (bits + 7) / 8);
  const size_t ne4 = (size_t)(E ? E : 1) * 4;
  const uint32_t ntiles = (uint32_t)(((uint64_t)E + kRadixTile - 1) / kRadixTile);
  const uint64_t nh = 256ull * std::max<uint32_t>(ntiles, 1);
  const uint32_t hscan = (uint32_t)((nh + 1 + kScanTile - 1) / kScanTile);
  void *tbuf, *hbuf;
  if ((rc = ws_buffer(w, kBufTranspose, 4 * ne4, &tbuf)) ||
      (rc = ws_buffer(w, kBufSeedList, (nh + 1 + hscan + 64) * 4, &hbuf)))
    return rc;
  lsg_graph t;
  memset(&t, 0, sizeof t);
  if (hipMalloc(&t.row_start, ((size_t)V + 1) * 4) != hipSuccess || hipMalloc(&t.edge_dst, ne4) != hipSuccess ||
      hipMalloc(&t.edge_data, ne4) != hipSuccess || hipMalloc(&t.node_data, (size_t)V * 4) != hipSuccess) {
    (void)hipFree(t.row_start);
    (void)hipFree(t.edge_dst);
    (void)hipFree(t.edge_data);
    (void)hipFree(t.node_data);
    return fail(LSG_ERR_NOMEM, "transpose: device allocation failed");
  }
  uint32_t *key[2] = {(uint32_t *)tbuf, (uint32_t *)((char *)tbuf + ne4)};
  uint32_t *vs[2] = {(uint32_t *)((char *)tbuf + 2 * ne4), t.edge_dst};
  uint32_t *vw[2] = {(uint32_t *)((char *)tbuf + 3 * ne4), (uint32_t *)t.edge_data};
  uint32_t *hist = (uint32_t *)hbuf, *htiles = hist + nh + 1, *htotal = htiles + hscan;
  if (E) {
    RadixArgs a;
    a.row_start = g->row_start;
    a.key = g->edge_dst;
    a.v1 = nullptr;
    a.v2 = (const uint32_t *)g->edge_data;  // (null for an unweighted graph: its reverse weights are 0)
    a.hist = hist;
    a.hist_tiles = htiles;
    a.n = E;
    a.V = V;
    a.shift = 0;
    a.ntiles = ntiles;
    for (uint32_t p = 0; p < P; ++p) {
      const uint32_t o = (P - p) & 1, width = (bits - a.shift + (P - p) - 1) / (P - p);
      a.mask = (1u << width) - 1;
      a.key_out = key[o];
      a.v1_out = vs[o];
      a.v2_out = vw[o];
      const uint64_t n = ((uint64_t)a.mask + 1) * ntiles;
      const uint32_t nscan = (uint32_t)((n + kScanTile - 1) / kScanTile);
      hipLaunchKernelGGL(radix_hist_kernel, dim3(ntiles), dim3(kRadixBlock), 0, w->stream, a);
      hipLaunchKernelGGL(scan_tile_kernel, dim3(nscan), dim3(kScanBlock), 0, w->stream, hist, (uint32_t)n, hist, htiles);
      hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(kScanBlock), 0, w->stream, htiles, nscan, htotal);
      if (p == 0) hipLaunchKernelGGL(radix_scatter_kernel<true>, dim3(ntiles), dim3(kRadixBlock), 0, w->stream, a);
      else hipLaunchKernelGGL(radix_scatter_kernel<false>, dim3(ntiles), dim3(kRadixBlock), 0, w->stream, a);
      a.key = key[o];
      a.v1 = vs[o];
      a.v2 = vw[o];
      a.shift += width;
    }
  }
  const uint32_t rgrid = (uint32_t)std::min<uint64_t>(((uint64_t)E + 256) / 256, 16ull * w->cus);
  hipLaunchKernelGGL(row_bounds_kernel, dim3(rgrid), dim3(256), 0, w->stream, (const uint32_t *)key[1], E, V,
                     t.row_start);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(w->stream));
  t.nnodes = V;
  t.nedges = E;
  t.device_graph = 1;
  t.device = g->device;
  *gt = t;
  return LSG_OK;
}

int lsg_bfs_do(const lsg_graph *g, const lsg_graph *gt, uint32_t src, int direction, int32_t *level_dev,
               lsg_stats *stats) {
  clear_error();
  auto t0 = std::chrono::steady_clock::now();
  int rc = check_device_graph(g, "bfs_do");
  if (rc) return rc;
  if ((rc = check_device_graph(gt, "bfs_do (reverse graph)"))) return rc;
  if (gt->nnodes != g->nnodes || gt->nedges != g->nedges || gt->device != g->device)
    return fail(LSG_ERR_ARG, "bfs_do: the reverse graph does not match the graph (lsg_graph_transpose)");
  if (src >= g->nnodes) return fail(LSG_ERR_ARG, "source %u out of range [0, %u)", src, g->nnodes);
  if (direction < 0 || direction > 2) return fail(LSG_ERR_ARG, "bad direction %d", direction);
  if (!level_dev) return fail(LSG_ERR_ARG, "NULL level array");
  Workspace *w;
  if ((rc = get_workspace(g->device, &w))) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  HIPCHK(hipSetDevice(w->device));
  const uint32_t V = g->nnodes;
  const uint32_t words = (uint32_t)(((uint64_t)V + kWave - 1) / kWave);
  // every vertex is found once, so all chunks over the whole traversal fit:
  // sum of ceil(deg / kDoHeavy) over heavy vertices <= 2 E / kDoHeavy
  const uint64_t hcap64 = 2ull * g->nedges / kDoHeavy + 64;
  if (hcap64 > UINT32_MAX) return fail(LSG_ERR_ARG, "bfs_do: graph too large");
  const uint32_t hcap = (uint32_t)hcap64;
  constexpr int kBs = kDoBlock;
  const void *fn = (const void *)do_kernel<kBs>;
  int grid = 0;
  if ((rc = resident_grid(w, fn, kBs, &grid))) return rc;
  // Blocks per CU: small levels want few at the barrier, the large ones of a
  // large graph many wavefronts (ms at 1 / 2 / 4: RMAT-16 0.061 / 0.068 / 0.087,
  // RMAT-18 0.070 / 0.076 / 0.097, RMAT-20 0.108 / 0.105 / 0.121, RMAT-22 0.247 /
  // 0.195 / 0.193; road-like 2048^2 1.58 / 1.65 / 1.77).  Bottom-up only, every level
  // looks at every word (10^6 vertices: uniform out-degree 4 0.48 / 0.38 / 0.42, a
  // random tree 0.58 / 0.51 / 0.60, 100^3 grid 6.7 / 5.5 / 5.8; RMAT-18 0.116 / 0.103 /
  // 0.122, uniform of 10^5 0.136 / 0.148 / 0.201).
  const int per_cu = direction == 2 ? (V < (1u << 18) ? 1 : 2) : low_degree(V, g->nedges) || g->nedges < (1u << 23) ? 1 : 2;
  grid = std::min<int>(grid, per_cu * (int)w->cus);
  void *qbuf, *hbuf, *bbuf, *wbuf;
  if ((rc = ws_buffer(w, kBufQueues, 2ull * V * 4, &qbuf)) || (rc = ws_buffer(w, kBufHeavy, 2ull * hcap * 8, &hbuf)) ||
      (rc = ws_buffer(w, kBufStamps, 3ull * words * 8, &bbuf)) || (rc = ws_buffer(w, kBufWave, sizeof(WaveCtrl), &wbuf)))
    return rc;
  DoArgs a;
  memset((void *)&a, 0, sizeof a);
  a.row_start = g->row_start;
  a.edge_dst = g->edge_dst;
  a.nedges = g->nedges;
  a.in_row = gt->row_start;
  a.in_src = gt->edge_dst;
  a.dist = (uint32_t *)level_dev;
  for (int i = 0; i < 2; ++i) {
    a.q[i] = (uint32_t *)qbuf + (size_t)i * V;
    a.hchunk[i] = (uint64_t *)hbuf + (size_t)i * hcap;
    a.bits[i] = (uint64_t *)bbuf + (size_t)i * words;
  }
  a.in_any = (uint64_t *)bbuf + 2ull * words;
  a.ctrl = w->ctrl;
  a.wc = (WaveCtrl *)wbuf;
  a.nnodes = a.qcap = V;
  a.words = words;
  a.hcap = hcap;
  a.heavy_deg = kDoHeavy;
  a.direction = (uint32_t)direction;
  a.unit_min = low_degree(V, g->nedges) ? 16 : 8;
  a.local_max = direction == 2 ? 0 : wave_local_max(V, g->nedges);
  a.spin_limit = spin_limit_ticks(w);
  a.residency_limit = residency_limit_ticks(w);
  const uint32_t igrid = (uint32_t)std::min<uint64_t>(((uint64_t)V + 255) / 256, 8ull * w->cus);
  Ctrl hc;
  float ms = 0;
  for (int attempt = 0;; ++attempt) {
    HIPCHK(hipEventRecord(w->ev0, w->stream));
    hipLaunchKernelGGL(do_init_kernel, dim3(igrid), dim3(256), 0, w->stream, a, src);
    hipLaunchKernelGGL(do_kernel<kBs>, dim3(grid), dim3(kBs), 0, w->stream, a);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(w->ev1, w->stream));
    HIPCHK(hipMemcpyAsync(&hc, w->ctrl, kCtrlHostBytes, hipMemcpyDeviceToHost, w->stream));
    HIPCHK(hipStreamSynchronize(w->stream));
    HIPCHK(hipEventElapsedTime(&ms, w->ev0, w->ev1));
    if (hc.abort != kAbortResidency) break;
    if (attempt > 0 || hc.resident_seen == 0 || hc.resident_seen >= (uint32_t)grid)
      return fail(LSG_ERR_HIP, "bfs_do: persistent grid of %d x %d blocks is not co-resident (%u were)", grid, kBs,
                  hc.resident_seen);
    grid = (int)hc.resident_seen;
    record_resident_grid(w, fn, kBs, grid);
  }
  if (hc.abort == kAbortTimeout)
    return fail(LSG_ERR_TIMEOUT, "bfs_do: grid barrier timed out at level %u; levels are incomplete", wave_last(a.wc).round);
  if (hc.abort == kAbortCapacity) return fail(LSG_ERR_CAPACITY, "bfs_do: chunk queue capacity exceeded");
  if (stats) {
    memset(stats, 0, sizeof *stats);
    stats->ms_kernel = ms;
    stats->iterations = hc.s.round - 2;  // levels with a vertex (the last level finds nothing)
    stats->near_iters = hc.s.phase;      // bottom-up levels
    stats->grid_blocks = grid;
    stats->block_size = kBs;
    stats->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  return LSG_OK;
}

}  // extern "C"
