// PageRank on gfx950: pull-based Jacobi iteration over the reverse CSR.
//
// Reference: apps/pr/kernel.cu -- ALPHA 0.85 and EPSILON 1e-6 (:19-20),
// p = 1 - ALPHA initially (:38), residual push until no residual exceeds
// EPSILON (:110-236), "PR took %d iterations" (:387); apps/pr/support.cu --
// options -n -t -x (:15-42), "sum: %f (%d)" and one "%d %f" line per node
// (:56-97).  Both methods converge to the fixpoint
//     p[v] = (1 - ALPHA) + ALPHA * sum over in-edges (u, v) of p[u] / outdeg(u)
// (vertices without out-edges pass nothing on).  The reference pushes
// residuals with float atomics in a data-driven order; here every iteration
// recomputes every vertex from its in-neighbours' contributions
// c[u] = p[u] / outdeg(u) -- no atomics, a deterministic summation order --
// and stops when no rank moved by more than epsilon relative to itself
// (every rank is at least 1 - ALPHA; an absolute test would wait on the
// float rounding of the largest ranks).
//
// Layout.  The iterations gather one contribution per in-edge from an array of
// V floats, and at RMAT-22's 16 MB that array, four times an XCD's L2, bounds
// them.  So a call first renumbers the vertices by in-degree, largest first
// (a stable counting sort; in-degrees from kHeavyDeg on, or less on small
// graphs, are one class): the contributions read most lie together, and
// vertices of one in-degree are neighbours.  In that order
//   positions [0, heavy)     in-degree >= kHeavyDeg: in-edges cut into chunks of
//     kChunk; one wavefront sums a chunk, and where a vertex has several, one
//     lane then adds their partials in chunk order (one wavefront per vertex
//     left the sweep waiting on the largest in-degree, ~97 K edges on RMAT-22);
//   positions [heavy, live)  the others with in-edges, in slices of 64, one lane
//     per vertex: a slice's sources are stored transposed, slot k of the 64
//     lanes consecutive, as many slots as its largest vertex has in-edges;
//     slots past a vertex's last one name a contribution that is 0;
//   positions [live, V)      no in-edges: rank 1 - alpha from the start.
// Without heavy vertices the sort is by in-degree within tiles of kPrTile
// vertices only (heavy = 0, live = V): there is no hub to bring together, and
// neighbours of a road network stay near (2048^2 road-like: 60 us per
// iteration, sorted as a whole 187; with flags on lines of their own 29).
// Ranks, out-degrees and both contribution arrays are kept in that order and
// the ranks put back at the end.  Per iteration, against lanes that walked the
// reverse CSR in vertex order: RMAT-22 514 -> 245 us, 2^20 vertices of uniform
// degrees 145 -> 88, road-like 74 -> 29; preparing takes 1.1 ms on RMAT-22.
//
// The convergence test stays on the device: the host enqueues iterations in
// batches of one or two launches each; a block in which some rank moved by
// more than epsilon raises one of kFlags flags, and the iteration's last block
// counts the iteration and sets a done flag when none was raised; the kernels
// of later iterations return at once when they find it set.  Iterations stay
// separate launches: the launch boundary makes one iteration's contributions
// visible to every XCD's L2 for the next iteration's gathers, which a
// persistent kernel would have to buy with an L2 invalidate in every block at
// every iteration.
//
// Why pull Jacobi and not the reference's residual push: a push sweep adds
// to its out-neighbours' residuals with one float atomic per edge (measured
// on gfx950: ~27 G random 4-byte atomics/s, against ~90 G gathers/s of the
// pull sweep here), and float atomics make every sum's order, and so the
// ranks' last bits, depend on the schedule; the pull sweep has no atomics and
// one summation order.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>

#include "engine.h"
#include "lsg_internal.h"
#include "runtime.h"
#include "scan_dev.h"

namespace lsg {

constexpr uint32_t kHeavyDeg = 255;  // in-degree from which a vertex is summed in chunks
constexpr uint32_t kWideDeg = 32;    // slices of at least as many slots take a wavefront each, others kSlices
constexpr int kSlices = 4;
// Contributions that pr_sweep_kernel<true> keeps in LDS (one block of kTabBlock
// threads per CU); it is used on graphs of at least kTabEdges edges of which
// at least one in kTabShare leaves those vertices.  A CU's L1 has about 64
// misses in flight, ~290 clocks each from the L2 (counters: 51 M L2 requests
// in 0.40 ms), so gathers that LDS answers are what makes the sweep faster.
// us per iteration without / with it: RMAT-22 (56% of the edges) 400 / 261, of
// ef 8 221 / 141, RMAT-21 179 / 107, RMAT-20 88 / 67, 8 M edges 47 / 49, 4 M 28 / 43.
// 16384 entries and twice the wavefronts: 320 on RMAT-22; 32768: 273.
// Without skew -- the positions' share of the edges less than twice their share of
// the vertices -- the L2 answers as well (100,000 vertices of in-degree 300 11.4 ms with,
// 10.0 without).
constexpr uint32_t kTabSize = 40448, kTabBlock = 1024, kTabEdges = 10000000, kTabShare = 4;
// Index arrays of this many edges and more outgrow the memory-side cache
// (256 MB), which then holds nothing of the last iteration when the next one
// begins where that one began: odd iterations take the units backwards
// (RMAT-22, 261 MB: 261 -> 242 us; 197 MB: 172 -> 166; 64 MB: 67 -> 83, the
// longest units coming last).
constexpr uint32_t kTurnEdges = 48000000;
constexpr uint32_t kPrGroups = 16;  // groups of blocks with work tickets of their own
// Below this many edges vertices of kWideDeg in-edges are heavy already: a wide
// slice is a chain of up to 32 steps, which a small graph has nothing to hide
// behind (whole call, kHeavyDeg / kWideDeg: 120 K edges 1.58 / 1.12 ms, 228 K
// 1.29 / 1.30, 679 K 1.74 / 2.27, 3.9 M 2.8 / 5.5).
constexpr uint32_t kSmallEdges = 200000;
// So are those of kMidDeg on graphs of few slices or where nearly every vertex is
// heavy: the slices' chains would be what an iteration waits for (kHeavyDeg /
// kMidDeg: 10,000 vertices of in-degree 200 2.03 / 1.24 ms, 20,000 2.08 / 1.77, of 300
// 30,000 4.27 / 3.20, 100,000 12.4 / 11.4; 40,000 of 200 2.49 / 3.20, RMAT-22 19.2 / 23.5).
constexpr uint32_t kMidDeg = 128, kMidV = 32768;
constexpr uint32_t kChunk = 4096;    // in-edges per wavefront-sized partial sum
constexpr int kUnrollPr = 8;         // in-edges per lane in flight
constexpr uint32_t kPrBlock = 256;
// Vertices per block of the counting sort, which takes them 256 at a time (4096 /
// 512, whole call: 20,000 vertices of out-degree 4 0.89 / 0.83 ms, 4 x 10^6 18.3 /
// 16.7, small world of 10^6 1.87 / 1.58, road-like 2048^2 2.61 / 2.55, RMAT-22 alike).
constexpr uint32_t kPrTile = 512;
// Sweeps of at most this many blocks end the iteration themselves (every block
// arrives on one word, ~12 ns each); larger ones leave it to pr_finish_kernel's
// launch, ~5 us (road-like 128^2, whole call: 0.88 -> 0.75 ms).
constexpr uint32_t kFusedBlocks = 256;
constexpr uint32_t kFlags = 64;      // "some rank moved" flags, spread over as many words
constexpr uint32_t kIterBatch = 8;   // iterations enqueued per host check

struct PrArgs {
  const uint32_t *row_start;        // forward CSR (out-degrees)
  const uint32_t *in_row, *in_src;  // reverse CSR
  uint32_t *hist;                   // [256][tiles] class counts, then places
  const uint32_t *hist_tiles;       // their scan's tile offsets
  uint32_t *pos_of;                 // [V] position of a vertex
  uint32_t *rs, *deg, *od;          // by position: first in-edge, in-degree, out-degree
  float *p, *c[2];                  // by position; c[.][V] = 0
  uint32_t *shape;                  // scanned: heavy in-degrees | chunks | slots of a slice (nh + 1, nh + 1, ns + 1 entries)
  const uint32_t *shape_tiles;
  uint4 *chunk;                     // a chunk: heavy vertex, in-edges, where they lie in idx (two words)
  float *part;                      // a chunk's sum
  uint32_t *hbase;                  // [heavy + 1] a heavy vertex's first chunk
  uint32_t *slice;                  // [slices + 1] a slice's first slot in idx, past slots, / 64
  uint32_t *idx;                    // source positions: heavy vertices' edges, then the slices
  uint32_t *ctl;
  size_t slots;                     // where the slices begin in idx
  uint32_t V, tiles, nh, ns;        // nh, ns: bounds of the numbers of heavy vertices and slices
  uint32_t heavy, live, nchunks, wide, nslices;  // wide: slices taken one per wavefront
  uint32_t units;                   // of the sweep
  uint32_t turn;                    // odd iterations take the units backwards
  uint32_t hdeg;                    // in-degree from which a vertex is heavy
  uint32_t fused;                   // the sweep also ends the iteration
  uint32_t local;                   // sorted within tiles
  float alpha, epsilon;
};

// control words; the flags of an iteration are those of its parity, so that
// the next iteration's can be cleared while they are read
constexpr int kCtlMax = 0, kCtlDone = 1, kCtlIters = 2, kCtlArrive = 3, kCtlHeavy = 4, kCtlWide = 5, kCtlLive = 6,
              kCtlChunks = 7, kCtlEdges = 8, kCtlHot = 9, kCtlSlots = 10, kCtlFlags = 32, kCtlTickets = kCtlFlags + 2 * 32 * (int)kFlags, kCtlWords = kCtlTickets + 32 * (int)kPrGroups;

__device__ __forceinline__ uint32_t pr_class(const PrArgs &a, uint32_t indeg) { return a.hdeg - min(indeg, a.hdeg); }

// Entry of class d and tile b in the order of the sort.
__device__ __forceinline__ size_t pr_entry(const PrArgs &a, uint32_t d, uint32_t b) {
  return a.local ? (size_t)b * 256 + d : (size_t)d * a.tiles + b;
}

__global__ void pr_clear_kernel(PrArgs a) {
  for (uint32_t i = threadIdx.x; i < (uint32_t)kCtlWords; i += blockDim.x) a.ctl[i] = 0;
}

// The largest in-degree.
__global__ __launch_bounds__(kPrBlock) void pr_max_kernel(PrArgs a) {
  __shared__ uint32_t s_m;
  if (threadIdx.x == 0) s_m = 0;
  __syncthreads();
  uint32_t m = 0;
  for (size_t v = blockIdx.x * (size_t)kPrBlock + threadIdx.x; v < a.V; v += (size_t)gridDim.x * kPrBlock)
    m = max(m, a.in_row[v + 1] - a.in_row[v]);
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) m = max(m, (uint32_t)__shfl_xor(m, d));
  if (lane_id() == 0) atomicMax(&s_m, m);
  __syncthreads();
  // (most blocks find a larger one there already)
  if (threadIdx.x == 0 && s_m > ld_coh(a.ctl + kCtlMax))
    __hip_atomic_fetch_max(glb(a.ctl + kCtlMax), s_m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// hist: vertices of every class and tile.
__global__ __launch_bounds__(kPrBlock) void pr_hist_kernel(PrArgs a) {
  __shared__ uint32_t h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kPrTile;
  for (uint32_t i = threadIdx.x; i < kPrTile && base + i < a.V; i += kPrBlock)
    atomicAdd(&h[pr_class(a, a.in_row[base + i + 1] - a.in_row[base + i])], 1u);
  __syncthreads();
  a.hist[pr_entry(a, threadIdx.x, blockIdx.x)] = h[threadIdx.x];
}

// Exclusive prefix over the classes and tiles at entry i.
__device__ __forceinline__ uint32_t pr_place(const PrArgs &a, size_t i) { return a.hist[i] + a.hist_tiles[i / kScanTile]; }

// Every vertex to its position, stable within a class, with its first rank
// and contribution (lanes of one class are ranked by ballots over its 8 bits).
__global__ __launch_bounds__(kPrBlock) void pr_place_kernel(PrArgs a) {
  constexpr uint32_t NW = kPrBlock / kWave;
  __shared__ uint32_t run[256], wcnt[NW][256], hot;
  const uint32_t lane = lane_id(), wv = threadIdx.x / kWave;
  run[threadIdx.x] = pr_place(a, pr_entry(a, threadIdx.x, blockIdx.x));
  for (uint32_t w = 0; w < NW; ++w) wcnt[w][threadIdx.x] = 0;
  if (threadIdx.x == 0) hot = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const bool whole = !a.local;
    a.ctl[kCtlHeavy] = whole ? pr_place(a, (size_t)a.tiles) : 0u;
    a.ctl[kCtlWide] = whole ? pr_place(a, (size_t)(a.hdeg - kWideDeg + 1) * a.tiles) : 0u;
    a.ctl[kCtlLive] = whole ? pr_place(a, (size_t)a.hdeg * a.tiles) : a.V;
    a.c[0][a.V] = a.c[1][a.V] = 0.0f;
  }
  __syncthreads();
  const float p0 = 1.0f - a.alpha;  // apps/pr/kernel.cu:38
  for (uint32_t it = 0; it < kPrTile / kPrBlock; ++it) {
    const uint64_t v = (uint64_t)blockIdx.x * kPrTile + it * kPrBlock + threadIdx.x;
    const bool valid = v < a.V;
    uint32_t e0 = 0, dg = 0, od = 0, d = 0;
    if (valid) {
      e0 = a.in_row[v];
      dg = a.in_row[v + 1] - e0;
      od = a.row_start[v + 1] - a.row_start[v];
      d = pr_class(a, dg);
    }
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (uint32_t bit = 0; bit < 8; ++bit) {
      const uint64_t m = __ballot((d >> bit) & 1u);
      peers &= ((d >> bit) & 1u) ? m : ~m;
    }
    const uint32_t rank = lanes_below(peers);
    if (valid && rank == 0) wcnt[wv][d] = (uint32_t)__builtin_popcountll(peers);
    __syncthreads();
    if (valid) {
      uint32_t pos = run[d] + rank;
      for (uint32_t w = 0; w < wv; ++w) pos += wcnt[w][d];
      a.pos_of[v] = pos;
      a.rs[pos] = e0;
      a.deg[pos] = dg;
      a.od[pos] = od;
      if (pos < kTabSize) atomicAdd(&hot, od);
      a.p[pos] = p0;
      a.c[0][pos] = a.c[1][pos] = od ? p0 / (float)od : 0.0f;
    }
    __syncthreads();
    uint32_t sum = 0;
    for (uint32_t w = 0; w < NW; ++w) {
      sum += wcnt[w][threadIdx.x];
      wcnt[w][threadIdx.x] = 0;
    }
    run[threadIdx.x] += sum;
    __syncthreads();
  }
  if (threadIdx.x == 0 && hot) atomic_add(a.ctl + kCtlHot, hot);
}

// The unscanned shape: in-degrees and chunk counts of the heavy vertices, slots
// per lane of the slices (a slice's largest in-degree is its first vertex's,
// or, where a tile ends in it, the first one of the next tile's).
__global__ void pr_shape_kernel(PrArgs a) {
  const uint32_t heavy = a.ctl[kCtlHeavy], live = a.ctl[kCtlLive];
  const size_t n = 2 * ((size_t)a.nh + 1) + a.ns + 1;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    uint32_t x = 0;
    if (i < a.nh + 1) {
      if (i < heavy) x = a.deg[i];
    } else if (i < 2 * ((size_t)a.nh + 1)) {
      const size_t k = i - (a.nh + 1);
      if (k < heavy) x = (a.deg[k] + kChunk - 1) / kChunk;
    } else {
      const uint64_t pos = heavy + (uint64_t)(i - 2 * ((size_t)a.nh + 1)) * kWave;
      if (pos < live) x = a.deg[pos];  // kPrTile is a multiple of 64: no slice crosses a tile
    }
    a.shape[i] = x;
  }
}

__device__ __forceinline__ uint32_t pr_shape_at(const PrArgs &a, size_t i) {
  return a.shape[i] + a.shape_tiles[i / kScanTile];
}
// From the shape's scan (each part from 0 on; u32 differences are exact
// whatever wraps): the heavy vertices' first chunks, the chunks, the slices.
__global__ void pr_chunks_kernel(PrArgs a) {
  const uint32_t heavy = a.ctl[kCtlHeavy], live = a.ctl[kCtlLive], lane = lane_id();
  const size_t c0 = a.nh + 1, s0 = 2 * c0;
  const uint32_t first = pr_shape_at(a, c0), first_slot = pr_shape_at(a, s0);
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x;
  for (size_t i = tid / kWave; i < heavy; i += nt / kWave) {
    const uint32_t b = pr_shape_at(a, c0 + i) - first, e = pr_shape_at(a, c0 + i + 1) - first, dg = a.deg[i];
    const uint64_t at = pr_shape_at(a, i);
    if (lane == 0) a.hbase[i] = b;
    for (uint32_t k = b + lane; k < e; k += kWave) {
      const uint32_t lo = (k - b) * kChunk;
      a.chunk[k] = make_uint4((uint32_t)i, min(dg - lo, kChunk), (uint32_t)(at + lo), (uint32_t)((at + lo) >> 32));
    }
  }
  const size_t nsl = ((size_t)live - heavy + kWave - 1) / kWave;
  for (size_t k = tid; k <= nsl; k += nt) a.slice[k] = pr_shape_at(a, s0 + k) - first_slot;
  if (tid == 0) {
    a.ctl[kCtlChunks] = a.hbase[heavy] = pr_shape_at(a, c0 + heavy) - first;
    a.ctl[kCtlEdges] = pr_shape_at(a, heavy);
    a.ctl[kCtlSlots] = pr_shape_at(a, s0 + nsl) - first_slot;
  }
}

// idx: the position of every in-edge's source, one wavefront per chunk or slice.
__global__ __launch_bounds__(kPrBlock) void pr_layout_kernel(PrArgs a) {
  const uint32_t lane = lane_id();
  const uint32_t units = a.nchunks + a.nslices;
  const uint32_t waves = gridDim.x * (kPrBlock / kWave);
  for (uint32_t k = blockIdx.x * (kPrBlock / kWave) + threadIdx.x / kWave; k < units; k += waves) {
    if (k < a.nchunks) {
      const uint4 x = a.chunk[k];
      const uint32_t *src = a.in_src + a.rs[x.x] + (size_t)(k - a.hbase[x.x]) * kChunk;
      uint32_t *const idx = a.idx + ((uint64_t)x.w << 32 | x.z);
      for (uint32_t e = lane; e < x.y; e += kWave) idx[e] = a.pos_of[src[e]];
    } else {
      const uint32_t sl = k - a.nchunks, at = a.slice[sl], w = a.slice[sl + 1] - at;
      uint32_t *const idx = a.idx + a.slots + (size_t)at * kWave + lane;
      const uint64_t pos = a.heavy + (uint64_t)sl * kWave + lane;
      const uint32_t dg = pos < a.live ? a.deg[pos] : 0u;
      const uint32_t *src = a.in_src + (pos < a.live ? a.rs[pos] : 0u);
      for (uint32_t q = 0; q < w; ++q) idx[(size_t)q * kWave] = q < dg ? a.pos_of[src[q]] : a.V;
    }
  }
}

// Whether an earlier iteration converged (written in an earlier launch, so a plain load sees it).
__device__ __forceinline__ bool pr_done(const PrArgs &a) { return a.ctl[kCtlDone] != 0; }

// The vertex at `pos`, whose rank was pc: its new rank and contribution from
// the sum of its in-neighbours' contributions; whether the rank moved.
__device__ __forceinline__ bool pr_store(const PrArgs &a, float *c_next, size_t pos, float sum, float pc, uint32_t od) {
  const float pn = (1.0f - a.alpha) + a.alpha * sum;
  a.p[pos] = pn;
  c_next[pos] = od ? pn / (float)od : 0.0f;
  return fabsf(pn - pc) / pn > a.epsilon;  // pn >= 1 - alpha > 0
}

// Flag f of iteration `it`, on a line of its own: stores to one line from all
// XCDs are performed one at a time (2500 blocks, 10,000 vertices of in-degree 300:
// 36 us an iteration, now 18).
__device__ __forceinline__ uint32_t *pr_flag(const PrArgs &a, uint32_t it, uint32_t f) {
  return a.ctl + kCtlFlags + ((it & 1) * kFlags + f) * 32;
}

// Raises the block's flag if some lane's rank moved.
__device__ __forceinline__ void pr_raise(const PrArgs &a, uint32_t it, bool moved) {
  if (__syncthreads_or(moved) && threadIdx.x == 0) st_coh(pr_flag(a, it, blockIdx.x % kFlags), 1u);
}

// A contribution.  kTab: those of the first kTabSize positions are in LDS, and
// their lanes read the 0 at c[V] instead (one line for all of them).
template <bool kTab>
__device__ __forceinline__ float pr_c(const PrArgs &a, const float *tab, const float *c, uint32_t u) {
  if (!kTab) return glb(c)[u];
  const bool hot = u < kTabSize;
  return tab[hot ? u : kTabSize] + glb(c)[hot ? a.V : u];
}

// The iteration's end, called by every thread of every block of its last
// launch: the last block to get here counts the iteration and decides whether
// it was the last.
__device__ __forceinline__ void pr_end(const PrArgs &a, uint32_t it) {
  __shared__ uint32_t last;
  if (threadIdx.x == 0) {
    order_release();
    last = atomic_add(a.ctl + kCtlArrive, 1u) + 1 == gridDim.x;
  }
  __syncthreads();
  if (!last) return;
  const bool some = threadIdx.x < kFlags && ld_coh(pr_flag(a, it, threadIdx.x)) != 0;
  if (threadIdx.x < kFlags) *pr_flag(a, it + 1, threadIdx.x) = 0;
  if (threadIdx.x < kPrGroups) a.ctl[kCtlTickets + threadIdx.x * 32] = 0;
  const bool go_on = __syncthreads_or(some);
  if (threadIdx.x == 0) {
    a.ctl[kCtlIters] = it + 1;
    a.ctl[kCtlDone] = !go_on;
    a.ctl[kCtlArrive] = 0;
  }
}

// One unit of the sweep; whether some rank moved.
template <bool kTab>
__device__ __forceinline__ bool pr_unit(const PrArgs &a, const float *tab, const float *c, float *c_next, uint32_t k) {
  const uint32_t lane = lane_id();
  bool moved = false;
  if (k < a.nchunks) {
    const uint4 x = a.chunk[k];
    const uint32_t n = __builtin_amdgcn_readfirstlane(x.y);
    const uint32_t *idx = a.idx + ((uint64_t)x.w << 32 | x.z);
    const bool whole = a.deg[x.x] <= kChunk;  // the vertex has no other chunk
    const float pc = a.p[x.x];
    const uint32_t od = a.od[x.x];
    // Every lane loads (past the chunk's end it reloads the last edge and adds
    // 0): loads under per-lane conditions make the compiler wait for the whole
    // memory queue at each, one round trip per load.
    float sum = 0.0f;
    for (uint32_t e = 0; e < n; e += kUnrollPr * kWave) {
      uint32_t u[kUnrollPr];
      float x8[kUnrollPr];
#pragma unroll
      for (int q = 0; q < kUnrollPr; ++q) u[q] = glb(idx)[min(e + q * kWave + lane, n - 1)];
#pragma unroll
      for (int q = 0; q < kUnrollPr; ++q) x8[q] = pr_c<kTab>(a, tab, c, u[q]);
#pragma unroll
      for (int q = 0; q < kUnrollPr; ++q) sum += e + q * kWave + lane < n ? x8[q] : 0.0f;
    }
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) sum += __shfl_xor(sum, d);
    if (lane == 0) {
      if (whole) moved = pr_store(a, c_next, x.x, sum, pc, od);
      else a.part[k] = sum;
    }
  } else if ((k -= a.nchunks) < a.wide) {
    const uint32_t at = a.slice[k], w = __builtin_amdgcn_readfirstlane(a.slice[k + 1] - at);
    const uint32_t *idx = a.idx + a.slots + (size_t)at * kWave + lane;
    const uint64_t pos = min(a.heavy + (uint64_t)k * kWave + lane, (uint64_t)a.live - 1);
    const float pc = a.p[pos];
    const uint32_t od = a.od[pos];
    float sum[kUnrollPr];
#pragma unroll
    for (int q = 0; q < kUnrollPr; ++q) sum[q] = 0.0f;
    for (uint32_t q0 = 0; q0 < w; q0 += kUnrollPr) {
      uint32_t u[kUnrollPr];
      float x8[kUnrollPr];
#pragma unroll
      for (int q = 0; q < kUnrollPr; ++q) u[q] = glb(idx)[(size_t)min(q0 + q, w - 1) * kWave];
#pragma unroll
      for (int q = 0; q < kUnrollPr; ++q) x8[q] = pr_c<kTab>(a, tab, c, u[q]);
#pragma unroll
      for (int q = 0; q < kUnrollPr; ++q) sum[q] += q0 + q < w ? x8[q] : 0.0f;
    }
    if (a.heavy + (uint64_t)k * kWave + lane < a.live)
      moved |= pr_store(a, c_next, pos, ((sum[0] + sum[1]) + (sum[2] + sum[3])) + ((sum[4] + sum[5]) + (sum[6] + sum[7])),
                       pc, od);
  } else if ((k = a.wide + (k - a.wide) * kSlices) < a.nslices) {
    uint32_t at[kSlices + 1], w[kSlices], od[kSlices], wmax = 0;
    float pc[kSlices], sum[kSlices];
    const uint64_t pos = a.heavy + (uint64_t)k * kWave + lane;
#pragma unroll
    for (int j = 0; j <= kSlices; ++j)
      at[j] = __builtin_amdgcn_readfirstlane(a.slice[min(k + j, a.nslices)]);
#pragma unroll
    for (int j = 0; j < kSlices; ++j) {
      w[j] = at[j + 1] - at[j];
      wmax = max(wmax, w[j]);
      const uint64_t x = min(pos + (uint64_t)j * kWave, (uint64_t)a.live - 1);
      pc[j] = a.p[x];
      od[j] = a.od[x];
      sum[j] = 0.0f;
    }
    const uint32_t *idx = a.idx + a.slots + lane;
    constexpr int kSlots = kUnrollPr / kSlices;
    for (uint32_t q0 = 0; q0 < wmax; q0 += kSlots) {
      uint32_t u[kSlices][kSlots];
      float x[kSlices][kSlots];
#pragma unroll
      for (int j = 0; j < kSlices; ++j)
#pragma unroll
        for (int q = 0; q < kSlots; ++q) u[j][q] = q0 + q < w[j] ? glb(idx)[(at[j] + (size_t)(q0 + q)) * kWave] : a.V;
#pragma unroll
      for (int j = 0; j < kSlices; ++j)
#pragma unroll
        for (int q = 0; q < kSlots; ++q) x[j][q] = pr_c<kTab>(a, tab, c, u[j][q]);
#pragma unroll
      for (int j = 0; j < kSlices; ++j)
#pragma unroll
        for (int q = 0; q < kSlots; ++q) sum[j] += x[j][q];
    }
#pragma unroll
    for (int j = 0; j < kSlices; ++j)
      if (pos + (uint64_t)j * kWave < a.live) moved |= pr_store(a, c_next, pos + j * kWave, sum[j], pc[j], od[j]);
  }
  return moved;
}

// One iteration's sums.  Wavefront units: the chunks, the wide slices, then the
// others kSlices at a time (few slots each: their loads go out together).
// Every sum is taken in in-edge order, a wide slice's (32 and more in-edges)
// in eight sums added pairwise, a chunk's per lane and then over the lanes.
template <bool kTab>
__global__ __launch_bounds__(kTab ? kTabBlock : kPrBlock) void pr_sweep_kernel(PrArgs a, uint32_t it) {
  if (pr_done(a)) return;
  constexpr uint32_t kBlock = kTab ? kTabBlock : kPrBlock;
  __shared__ float tab[kTab ? kTabSize + 1 : 1];
  const uint32_t lane = lane_id();
  const float *const c = a.c[it & 1];
  if (kTab) {
    for (uint32_t i = threadIdx.x; i <= kTabSize; i += kBlock) tab[i] = i < kTabSize ? c[i] : 0.0f;
    __syncthreads();
  }
  float *const c_next = a.c[(it & 1) ^ 1];
  const uint32_t wave = threadIdx.x / kWave;
  uint32_t unit, g = 0;
  if (kTab) {
    // Unit j * kPrGroups + g belongs to the blocks b with b % kPrGroups == g: a
    // wavefront takes one, then one per ticket, fetched a unit ahead.
    g = blockIdx.x % kPrGroups;
    unit = (blockIdx.x / kPrGroups * (kBlock / kWave) + wave) * kPrGroups + g;
  } else {
    // One unit per wavefront.  Sorted within tiles, neighbours are near: every
    // XCD takes one contiguous eighth of the units.  (Sorted as a whole the
    // longest units come first and are dealt to all XCDs.)
    const uint32_t b = a.local ? blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    unit = b * (kBlock / kWave) + wave;
  }
  bool moved = false;
  while (unit < a.units) {
    uint32_t t = 0;
    if (kTab && lane == 0) t = atomic_add(a.ctl + kCtlTickets + g * 32, 1u);
    moved |= pr_unit<kTab>(a, tab, c, c_next, a.turn && (it & 1) ? a.units - 1 - unit : unit);
    if (!kTab) break;
    const uint32_t first = (gridDim.x + kPrGroups - 1 - g) / kPrGroups * (kBlock / kWave);
    unit = (first + readlane(t, 0)) * kPrGroups + g;
  }
  pr_raise(a, it, moved);
  if (!kTab && a.fused) pr_end(a, it);
}

// One lane per heavy vertex of several chunks: its partials added in chunk
// order; the iteration's end.
__global__ __launch_bounds__(kPrBlock) void pr_finish_kernel(PrArgs a, uint32_t it) {
  if (pr_done(a)) return;
  const uint32_t i = blockIdx.x * kPrBlock + threadIdx.x;
  bool moved = false;
  if (i < a.heavy) {
    const uint32_t b = a.hbase[i], e = a.hbase[i + 1];
    if (e - b > 1) {
      const float pc = a.p[i];
      const uint32_t od = a.od[i];
      float sum = 0.0f;
      for (uint32_t k = b; k < e; ++k) sum += a.part[k];
      moved = pr_store(a, a.c[(it & 1) ^ 1], i, sum, pc, od);
    }
  }
  pr_raise(a, it, moved);
  pr_end(a, it);
}

// The ranks in vertex order.
__global__ void pr_ranks_kernel(PrArgs a, float *rank) {
  for (size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x; v < a.V; v += (size_t)gridDim.x * blockDim.x)
    rank[v] = a.p[a.pos_of[v]];
}

}  // namespace lsg

using namespace lsg;

extern "C" {

int lsg_pagerank(const lsg_graph *g, const lsg_graph *gt, float alpha, float epsilon, int32_t max_iterations,
                 float *rank_dev, lsg_stats *stats) {
  clear_error();
  auto t0 = std::chrono::steady_clock::now();
  if (!g || g->device_graph == 0 || !g->row_start || !gt || gt->device_graph == 0 || !gt->row_start)
    return fail(LSG_ERR_ARG, "pagerank: expected a device graph and its reverse (lsg_graph_transpose)");
  if (gt->nnodes != g->nnodes || gt->nedges != g->nedges || gt->device != g->device)
    return fail(LSG_ERR_ARG, "pagerank: the reverse graph does not match the graph");
  if (!rank_dev) return fail(LSG_ERR_ARG, "pagerank: NULL rank array");
  if (!(alpha > 0.0f && alpha < 1.0f)) return fail(LSG_ERR_ARG, "pagerank: alpha must be in (0, 1)");
  if (!(epsilon > 0.0f)) return fail(LSG_ERR_ARG, "pagerank: epsilon must be > 0");
  if (max_iterations <= 0) return fail(LSG_ERR_ARG, "pagerank: max_iterations must be > 0");
  Workspace *w;
  int rc = get_workspace(g->device, &w);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  HIPCHK(hipSetDevice(w->device));
  const uint32_t V = g->nnodes;
  const uint64_t E = g->nedges;
  const uint32_t tiles = (uint32_t)(((uint64_t)V + kPrTile - 1) / kPrTile);
  PrArgs a;
  memset(&a, 0, sizeof a);
  a.V = V;
  a.tiles = tiles;
  a.nh = (uint32_t)std::min<uint64_t>(V, E / kWideDeg);
  a.ns = V / kWave + 1;
  const uint64_t nhist = 256ull * tiles, hscan = (nhist + kScanTile - 1) / kScanTile;
  const uint64_t nshape = 2 * (a.nh + 1ull) + a.ns + 1, sscan = (nshape + kScanTile - 1) / kScanTile;
  const uint64_t maxchunks = a.nh + E / kChunk + 1;
  void *buf, *ibuf;
  if ((rc = ws_buffer(w, kBufQueues,
                      (7ull * V + 2 + nhist + hscan + nshape + sscan + (a.nh + 1ull) + (a.ns + 1ull) + 5 * maxchunks +
                       kCtlWords + 2) * 4 + 16, &buf)))
    return rc;
  uint32_t *at = (uint32_t *)buf;
  auto take = [&](uint64_t n) {
    uint32_t *const x = at;
    at += n;
    return x;
  };
  a.pos_of = take(V);
  a.rs = take(V);
  a.deg = take(V);
  a.od = take(V);
  a.p = (float *)take(V);
  a.c[0] = (float *)take(V + 1ull);
  a.c[1] = (float *)take(V + 1ull);
  a.hist = take(nhist);
  uint32_t *const hist_tiles = take(hscan);
  a.hist_tiles = hist_tiles;
  a.shape = take(nshape);
  uint32_t *const shape_tiles = take(sscan);
  a.shape_tiles = shape_tiles;
  a.hbase = take(a.nh + 1ull);
  a.slice = take(a.ns + 1ull);
  a.part = (float *)take(maxchunks);
  a.ctl = take(kCtlWords);
  uint32_t *const total = take(2);
  a.chunk = (uint4 *)(((uintptr_t)at + 15) & ~(uintptr_t)15);
  a.row_start = g->row_start;
  a.in_row = gt->row_start;
  a.in_src = gt->edge_dst;
  a.alpha = alpha;
  a.epsilon = epsilon;
  const uint32_t vgrid = (uint32_t)std::min<uint64_t>(((uint64_t)V + 255) / 256, 16ull * w->cus);
  HIPCHK(hipEventRecord(w->ev0, w->stream));
  uint32_t *hc = w->pinned;
  hipLaunchKernelGGL(pr_clear_kernel, dim3(1), dim3(256), 0, w->stream, a);
  hipLaunchKernelGGL(pr_max_kernel, dim3(std::min<uint32_t>(vgrid, 4u * w->cus)), dim3(kPrBlock), 0, w->stream, a);
  HIPCHK(hipMemcpyAsync(hc, a.ctl, 16 * 4, hipMemcpyDeviceToHost, w->stream));
  HIPCHK(hipStreamSynchronize(w->stream));
  const uint32_t maxdeg = hc[kCtlMax];
  a.local = maxdeg < kWideDeg;
  a.hdeg = E < kSmallEdges ? kWideDeg : V <= kMidV || E >= (uint64_t)kHeavyDeg * V ? kMidDeg : kHeavyDeg;
  hipLaunchKernelGGL(pr_hist_kernel, dim3(tiles), dim3(kPrBlock), 0, w->stream, a);
  hipLaunchKernelGGL(scan_tile_kernel, dim3((uint32_t)hscan), dim3(kScanBlock), 0, w->stream, a.hist, (uint32_t)nhist,
                     a.hist, hist_tiles);
  hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(kScanBlock), 0, w->stream, hist_tiles, (uint32_t)hscan, total);
  hipLaunchKernelGGL(pr_place_kernel, dim3(tiles), dim3(kPrBlock), 0, w->stream, a);
  hipLaunchKernelGGL(pr_shape_kernel, dim3(vgrid), dim3(256), 0, w->stream, a);
  hipLaunchKernelGGL(scan_tile_kernel, dim3((uint32_t)sscan), dim3(kScanBlock), 0, w->stream, a.shape,
                     (uint32_t)nshape, a.shape, shape_tiles);
  hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(kScanBlock), 0, w->stream, shape_tiles, (uint32_t)sscan, total);
  // (a wavefront per heavy vertex: 10,000 of them over 160 wavefronts took 39 us)
  const uint32_t kgrid = std::max(vgrid, (uint32_t)std::min<uint64_t>(a.nh / 4 + 1ull, 8ull * w->cus));
  hipLaunchKernelGGL(pr_chunks_kernel, dim3(kgrid), dim3(256), 0, w->stream, a);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(hc, a.ctl, 16 * 4, hipMemcpyDeviceToHost, w->stream));
  HIPCHK(hipStreamSynchronize(w->stream));
  const uint32_t nheavy = hc[kCtlHeavy];
  a.heavy = nheavy;
  a.live = hc[kCtlLive];
  a.nchunks = hc[kCtlChunks];
  a.nslices = (a.live - a.heavy + kWave - 1) / kWave;
  a.wide = std::min(a.nslices, (hc[kCtlWide] - nheavy * (a.local ? 0u : 1u) + kWave - 1) / kWave);
  a.slots = ((size_t)hc[kCtlEdges] + kWave - 1) / kWave * kWave;
  const uint64_t nidx = a.slots + (uint64_t)kWave * hc[kCtlSlots];
  if (nheavy > a.nh || a.nchunks > maxchunks || a.nslices > a.ns)
    return fail(LSG_ERR_CAPACITY, "pagerank: the reverse graph's degrees exceed its edge count");
  if ((rc = ws_buffer(w, kBufUnion, std::max<uint64_t>(nidx, 1) * 4, &ibuf))) return rc;
  a.idx = (uint32_t *)ibuf;
  hipLaunchKernelGGL(pr_layout_kernel, dim3(8u * w->cus), dim3(kPrBlock), 0, w->stream, a);
  a.units = (uint32_t)((uint64_t)a.nchunks + a.wide + (a.nslices - a.wide + kSlices - 1) / kSlices);
  const bool tab = V >= kTabSize && E >= kTabEdges && hc[kCtlHot] >= E / kTabShare &&
                   (uint64_t)hc[kCtlHot] * V >= 2 * E * kTabSize;
  a.turn = E >= kTurnEdges;
  const uint32_t sgrid = tab ? (uint32_t)w->cus : ((a.units + kPrBlock / kWave - 1) / (kPrBlock / kWave) + 7) / 8 * 8;
  a.fused = maxdeg <= kChunk && !tab && sgrid && sgrid <= kFusedBlocks;
  const uint32_t fgrid = std::max(1u, maxdeg <= kChunk ? 1u : (nheavy + kPrBlock - 1) / kPrBlock);
  for (uint32_t it = 0; it < (uint32_t)max_iterations;) {
    const uint32_t end = std::min<uint32_t>((uint32_t)max_iterations, it + kIterBatch);
    for (; it < end; ++it) {
      if (tab) hipLaunchKernelGGL(pr_sweep_kernel<true>, dim3(sgrid), dim3(kTabBlock), 0, w->stream, a, it);
      else if (sgrid) hipLaunchKernelGGL(pr_sweep_kernel<false>, dim3(sgrid), dim3(kPrBlock), 0, w->stream, a, it);
      if (!a.fused) hipLaunchKernelGGL(pr_finish_kernel, dim3(fgrid), dim3(kPrBlock), 0, w->stream, a, it);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(hc, a.ctl, 16 * 4, hipMemcpyDeviceToHost, w->stream));
    HIPCHK(hipStreamSynchronize(w->stream));
    if (hc[kCtlDone]) break;
  }
  const int iters = (int)hc[kCtlIters];
  hipLaunchKernelGGL(pr_ranks_kernel, dim3(vgrid), dim3(256), 0, w->stream, a, rank_dev);
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(w->ev1, w->stream));
  HIPCHK(hipEventSynchronize(w->ev1));
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, w->ev0, w->ev1));
  if (stats) {
    memset(stats, 0, sizeof *stats);
    stats->ms_kernel = ms;
    stats->iterations = (uint64_t)iters;
    stats->items = nheavy;
    stats->grid_blocks = (int32_t)sgrid;
    stats->block_size = (int32_t)(tab ? kTabBlock : kPrBlock);
    stats->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  return LSG_OK;
}

}  // extern "C"
