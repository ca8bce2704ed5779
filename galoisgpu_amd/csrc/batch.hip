// Batched SSSP on gfx950: up to 64 sources on one graph in one persistent
// launch, vertex-major.
//
// No reference counterpart: the reference runs one source per process
// (apps/sssp/kernel.cu:455-480).  Each source follows exactly the plain
// method's rules -- fixed-delta near/far piles, curdelta += DELTA per phase
// (apps/sssp/kernel.cu:129-144,355-391) -- so its distances are identical to a
// single-source run; what changes is that all sources share every round.
//
// Layout in HBM: D[v][s] (u32, row stride S <= 64): the 64 lanes of a
// wavefront carry the 64 sources, so relaxing edge u->v for every source is one
// coalesced row load of D[v] and masked atomicMin on the same row, and the
// edge's column and weight are read once for all sources.  Per-vertex 64-bit
// masks say which sources must expand a vertex: nmask[2][V] for the near pile
// (indexed by round parity: written in round r, consumed in round r+1) and
// fmask[2][V] for the far pile (phase parity).  A vertex enters a pile's queue
// when its mask goes from 0 to non-zero, so each queue holds a vertex once.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <chrono>
#include <climits>
#include <cstring>
#include <vector>

#include "engine.h"
#include "lsg_internal.h"
#include "runtime.h"
#include "sched_mlp.h"

namespace lsg {

// Flattened path (items of degree < kLongDeg): row loads issued ahead per
// wavefront and frontier items per ticket.  Measured on RMAT-22 x 64 sources
// when every item took this path (ms per launch): 16 / 16 at 4 waves/SIMD
// 65-66; 8 / 8 at 5 waves 68; 8 / 8 at 6 waves 68-69; 4 / 8 at 6 waves 69-70.
constexpr int kUnroll = 16;
// Frontier items a wavefront takes per ticket: their masks, row bounds and
// distance rows are loaded together and their edges relaxed as one list.
constexpr int kItems = 16;
static_assert(kItems >= 1 && kItems <= kWave, "items per ticket");
// Waves per SIMD the register allocation must allow: 4 (128 VGPRs).  5 or 6
// spill and were slower (42 vs 34 ms on the item-major path).
constexpr int kMultiWaves = 4;

// ---- edge filter ------------------------------------------------------------
//
// Nine of ten edge expansions of a batched run improve no source (RMAT-22 x 64
// sources: 42 M of 463 M), and each costs a row access, whose rate bounds the
// kernel.  From a few rounds on, one 4-byte bound per vertex tells most of
// them apart.  With an offset off[s] per source, let
//     bound[v] = max over s of (D[v][s] - off[s]).
// An expansion of u for the sources in A can improve v over an edge of weight
// w only if  min over s in A of (D[u][s] - off[s]) + w < bound[v].
// This holds for any offsets and for bounds taken at any earlier time
// (distances only fall).  The offsets make the test sharp: off[s] = D[h][s]
// for the vertex h of largest out-degree, because on a skewed graph most
// shortest paths run through the hubs, so D[v][s] - D[h][s] is nearly the same for every s
// (a model of the rounds on RMAT-19: 5.67 E expansions, of which 0.58 E
// improve; 5.1 E pass the test without offsets, 1.54 E with them).
// A source that has not reached h yet is left out of the bounds, and an
// expansion for such a source always passes.
//
// The bounds come from up to kSweeps sweeps over D inside the launch, each
// with the offsets of its time and into an array of its own, so that bounds
// read through the caches are never of other offsets; the arrays share no
// cache line (the last bounds of one sweep read beside the first of the next
// array would leave those in the caches as an earlier call left them).  A sweep
// reads V rows in order; it follows once E/2 edges were expanded since the
// last one.
constexpr int kSweeps = 3;
// The test needs a hub that most paths share: it is used where the largest
// out-degree is at least kHubRatio times the mean.  Without / with the test
// (ms, 64 sources unless said): RMAT-21, ratio 4035, 13.4 / 10.2; RMAT of 32768
// vertices 1.44 / 1.42 (2 sources 0.75 / 0.72); 2^20 vertices of skewed
// degrees, ratio 50, 16.8 / 16.3; uniform degrees, ratio 2.5, 16.8 / 17.3;
// road-like 700x700 14.2 / 14.6.
constexpr uint32_t kHubRatio = 16;
constexpr int32_t kNoBound = 0x7FFFFFFF;         // bound of a vertex that some source has not reached
constexpr int32_t kPass = -0x7FFFFFFF - 1;       // lowest distance of an item that takes no test

struct Filter {
  uint64_t incl;        // sources whose offset is set
  uint64_t last_edges;  // edges expanded when the last sweep was ordered
  uint32_t hub;         // vertex of largest out-degree
  uint32_t on;          // the graph has such a hub
  int32_t off[64];
};

// Pace of the near/far threshold (fixed delta, reference far pile): it moves by
// `step` deltas.  A round of a batch costs some 20 us however small, and the far
// pile, expanded as a whole every phase, is mostly work done again: with 64
// sources the rounds of one wide phase expand a vertex for many of them at
// once.  On graphs with a hub, of few hops, the step begins at kHubStep: at 16 and
// less the cost of the first phases, whose frontiers grow by factors, says that
// a wider step does not pay, and the climb stays where vertices are expanded most
// often.  It is climbed from there, or from 1 on other graphs, while the threshold
// then moves further per us of modelled cost, or while rounds are nearly empty;
// else one step back, and two phases later the next trial.  Distances do not
// depend on it.
// Ms at steps of 1 -> from 16 on hubs, 1 elsewhere (delta 32): RMAT of 16400 vertices
// x 5 sources 1.84 -> 0.78, 100003 x 9 3.9 -> 1.37, 262900 x 64 12.0 -> 2.9; grid
// 64^2 x 5 6.0 -> 2.6, road-like 300^2 x 64 at 10000 13 -> 6.9.  Hubs from 16 -> from
// kHubStep: RMAT of 2^20 x 64 at 1 15.4 -> 4.6 (steps of 1: 8.6), 2^18, weights to
// 10000, x 64 at 32 22.0 -> 4.4 (19.9), x 24 9.9 -> 2.8 (13.5), 2^16 of 32 edges x 64
// at 1 9.3 -> 2.7 (5.1); slower only where the hub is no way across: grid 300^2 with
// 1000 edges more at a corner, x 64 at 32, 21.4 -> 28.8 (101).
struct Pace {
  uint32_t step;    // deltas that the threshold moves by
  uint32_t hold;    // phases until the next trial; 0: this phase is one
  float best;       // deltas per us before the trial
  uint32_t rounds;  // before this phase
  uint64_t edges;   // expanded before this phase
};
constexpr uint32_t kMaxMultiStep = 1u << 16, kHubStep = kMaxMultiStep;
constexpr float kRoundUs = 20, kEdgesPerUs = 30000;

// Work tickets and round totals are kept per group of blocks (block b: group
// b % kGroups), each on a line of its own: atomics on one word are performed
// one at a time, ~12 ns each, and a word that all 4096 wavefronts share
// bounds the launch (RMAT-22 x 64 sources: 0.44 M tickets, 5 ms).
constexpr uint32_t kGroups = 16;
struct alignas(128) TicketGroup {
  uint32_t ticket;
};
// Counters the leader turns into trace records and scheduler features.
struct alignas(128) MultiCounters {
  uint64_t lane_items;   // sum over expanded items of active sources
  uint64_t edges;        // edges expanded (per vertex, shared by its sources)
  uint64_t improved;     // rows in which at least one lane improved
};
// One wavefront's share in a round: lane_items and edges per lane, improved wave-uniform.
struct RoundCounters {
  uint32_t lane_items, edges;
  uint64_t improved;
};

struct MArgs {
  const uint32_t *row_start;
  const uint32_t *edge_dst;
  const uint32_t *edge_data;
  uint32_t *D;          // [V][S]
  uint64_t *nmask[2];   // near masks by round parity
  uint64_t *fmask[2];   // far masks by phase parity
  uint32_t *q[3];       // item queues (vertex ids)
  uint64_t *hq[2];      // heavy chunks: two u64 words each: (k << 32 | u), mask
  const uint32_t *srcs; // S source vertices
  Ctrl *ctrl;
  uint32_t nnodes, S, qcap, hcap, delta, heavy_deg;
  uint64_t spin_limit, residency_limit;
  lsg_round_trace *trace;
  uint32_t trace_cap;
  uint32_t sched;       // 1 = learned delta per phase
  const float *mlp;     // scheduler weights (sched_mlp.h layout)
  uint64_t nedges;
  uint32_t far_mode;    // initial far-pile mode (LSG_FAR_*)
  float *feat;          // per-phase feature records [kMaxForced][kFeatRec], or null
  uint32_t *fmin;       // [2][64] smallest pending far distance per source, by phase parity
  uint32_t *thr;        // [64] per-source near/far threshold of the current phase (bucket mode)
  uint32_t *qstamp;     // [V] last round whose in-queue holds the vertex
  Filter *flt;          // edge filter state
  Pace *pace;           // threshold pace, or null (steps of delta)
  TicketGroup *tickets; // [kGroups]
  MultiCounters *tot;   // [kGroups]
  uint64_t *hubs;       // multi_init's largest (out-degree << 32 | ~vertex) of each block
  uint32_t ninit;       // blocks of multi_init
  int32_t *bound[kSweeps];  // [V] each: the vertices' bounds, one array per sweep
};

// Pushes are staged per wavefront in LDS, kPushBuf items per pile, and
// written out with one queue-tail atomic per flush: one atomic per push
// on a tail that every wavefront of the grid shares serialises at the
// memory-side atomic unit (~12 ns each on gfx950).  512 entries measured
// faster than 256 (26.0 vs 26.5 ms on RMAT-22 x 64 sources).
constexpr uint32_t kPushBuf = 512;

// Heavy items are staged the same way (one atomic on the chunk count per
// heavy item, ~0.4 M on RMAT-22 x 64 sources, cost ~5 ms and kept the chunks large).
constexpr uint32_t kHeavyBuf = 64;
struct HeavyItem {
  uint32_t u, nch;
  uint64_t mask;
};

// Per-round, per-lane view of the schedule used by the edge loop.
struct LaneSched {
  uint32_t thr;   // near/far threshold of this lane's source
  bool bucket;    // per-source thresholds (LSG_FAR_BUCKET phase)
  uint32_t fmin;  // smallest distance this lane pushed to the far pile this round
  uint32_t thr32; // threshold of this lane as u32: a candidate nd goes near iff nd <= thr32
  uint32_t *pb;   // this wavefront's LDS push buffers: [0, kPushBuf) near, [kPushBuf, 2 kPushBuf) far
  uint32_t pbn[2];  // items staged per pile (wave-uniform)
  HeavyItem *hb;    // this wavefront's LDS buffer of heavy items, kHeavyBuf entries
  uint32_t hn, hchunks;  // staged heavy items and their chunks (wave-uniform)
  const int32_t *bound;  // the last sweep's bounds, or null (no test)
  int32_t off;      // this lane's source: offset, and whether the bounds include it
  bool incl;
};

// Writes pile `which`'s staged items to its queue (one atomic for all).
__device__ __forceinline__ void push_flush(const MArgs &a, const Sched &s, LaneSched &ls, int which) {
  const uint32_t n = ls.pbn[which];
  if (n == 0) return;
  const uint32_t qi = which ? s.far_q : s.near_q;
  uint32_t base = 0;
  if (lane_id() == 0) base = atomic_add(&a.ctrl->qcount[qi], n);
  base = readlane(base, 0);
  const uint32_t *buf = ls.pb + which * kPushBuf;
  for (uint32_t i = lane_id(); i < n; i += kWave) {
    const uint32_t pos = base + i;
    if (pos < a.qcap) st_coh(a.q[qi] + pos, buf[i]);
    else st_coh(&a.ctrl->abort, kAbortCapacity);
  }
  ls.pbn[which] = 0;
}

// Pushes `item` from every lane with `pred` onto pile `which` (0 near, 1 far).
__device__ __forceinline__ void pile_push(const MArgs &a, const Sched &s, LaneSched &ls, int which, bool pred,
                                          uint32_t item) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const uint32_t n = (uint32_t)__builtin_popcountll(m);
  if (ls.pbn[which] + n > kPushBuf) push_flush(a, s, ls, which);
  if (pred) ls.pb[which * kPushBuf + ls.pbn[which] + lanes_below(m)] = item;
  ls.pbn[which] += n;
}

__device__ __forceinline__ uint64_t bcast64(uint64_t x, uint32_t l) {
  uint32_t lo = readlane((uint32_t)x, l), hi = readlane((uint32_t)(x >> 32), l);
  return ((uint64_t)hi << 32) | lo;
}

// Near-pile push admission: a vertex joins the next round's queue at most
// once (a pop that took its next-round bits leaves it queued while its mask
// is empty again).
__device__ __forceinline__ bool near_admit(const MArgs &a, const Sched &s, uint32_t v) {
  return __hip_atomic_fetch_max(glb(a.qstamp + v), s.round + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < s.round + 1;
}

// Whether v has out-edges.  A vertex without any is never expanded, so an
// improvement of it needs no mask and no queue (RMAT-22 x 64 sources: 14.0 ->
// 11.7 M items popped, 13.9 -> 13.5 ms).
__device__ __forceinline__ bool has_edges(const MArgs &a, uint32_t v) {
  return glb(a.row_start)[v] != glb(a.row_start)[v + 1];
}

// Distance rows of the items a wavefront is expanding: dl[slot][lane] is the
// item's distance for source `lane`, INF where that source does not expand it.
// Each lane only reads its own column, so this is per-lane indexed storage.
typedef uint32_t DistSlots[kItems][kWave];

// Relaxes a batch of n <= 64 edges held one per lane: lane j has edge j's
// destination ev, weight ew and the slot ek of the item it leaves.  The row
// loads of a group of kUnroll edges are all issued before any is used, then
// the group's atomicMins; lane j collects edge j's near / far source bits, and
// the masks of the n destinations are updated with one vector atomic each.
__device__ __forceinline__ void relax_batch(const MArgs &a, const Sched &s, LaneSched &ls, const DistSlots &dl,
                                            uint32_t n, uint32_t ev, uint32_t ew, uint32_t ek,
                                            uint64_t *improved_rows) {
  const uint32_t lane = lane_id();
  // Near/far threshold of this lane: the shared curdelta (apps/sssp/kernel.cu:134)
  // or, in a bucket phase, the lane's own source threshold.
  const int64_t thr = ls.bucket ? (int64_t)ls.thr : s.curdelta();
  // Column this lane loads: its own source, or for lanes >= S (no source, no
  // candidate) the row's last word, so that every load stays inside row v.
  const uint32_t col = min(lane, a.S - 1);
  uint64_t my_nb = 0, my_fb = 0;
  for (uint32_t j0 = 0; j0 < n; j0 += kUnroll) {
    uint32_t v[kUnroll], nd[kUnroll], cur[kUnroll], old[kUnroll];
    bool want[kUnroll];
    // Candidates first (LDS and register work only) ...
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const uint32_t j = min(j0 + k, n - 1);  // a tail slot repeats the batch's last edge, with no candidate
      v[k] = readlane(ev, j);
      const uint32_t du = dl[readlane(ek, j)][lane];
      nd[k] = du == kInf || j0 + k >= n ? kInf : du + readlane(ew, j);
    }
    // ... then the group's row loads, unconditional so that none waits on a
    // branch: every lane loads a word of D[v], whose row (S words) is fetched
    // anyway when any lane needs it.
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) cur[k] = ld_coh(a.D + (size_t)v[k] * a.S + col);
    // every atomicMin of the group is issued before any result is used
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      want[k] = nd[k] < cur[k];
      old[k] = want[k] ? atomic_min(a.D + (size_t)v[k] * a.S + lane, nd[k]) : kInf;
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      bool imp = want[k] && nd[k] < old[k];
      bool nearl = imp && (int64_t)nd[k] <= thr;
      if (imp && !nearl) ls.fmin = min(ls.fmin, nd[k]);
      uint64_t nb = __ballot(nearl), fb = __ballot(imp && !nearl);
      if (nb | fb) *improved_rows += 1;
      if (lane == j0 + k) {
        my_nb = nb;
        my_fb = fb;
      }
    }
  }
  // Two edges of a batch may share a destination; only the lane whose OR
  // finds the mask empty queues it.
  const bool live = has_edges(a, ev);
  if (!live) my_nb = my_fb = 0;
  bool pn = my_nb != 0 && atomic_or64(a.nmask[s.round & 1] + ev, my_nb) == 0 && near_admit(a, s, ev);
  bool pf = my_fb != 0 && atomic_or64(a.fmask[s.phase & 1] + ev, my_fb) == 0;
  pile_push(a, s, ls, 0, pn, ev);
  pile_push(a, s, ls, 1, pf, ev);
}

// ---- item-major relaxation ------------------------------------------------
//
// Items of degree >= kLongDeg and heavy chunks are relaxed one item at a time:
// the item's distance for this lane's source stays in a register, its edges
// come kGroup at a time through the scalar cache (one s_load_dwordx8 for the
// destinations, one for the weights), and each edge costs one row load, an
// add and a compare per wavefront -- no lane shuffles.  Window width,
// measured on RMAT-22 x 64 sources: 8 wide and software-pipelined 33.6 ms,
// 16 wide 34.2 (pipelined or not; pipelined it spills).  Improvements are
// collected in a per-wavefront list and the destinations' masks are updated
// 64 at a time.
constexpr int kGroup = 8;
// Heavy chunks taken as one unit hold at most kChunkUnit edges (and kItems
// chunks): their distance rows are loaded when the unit starts, and a unit
// that runs for long relaxes from old distances (RMAT-22 x 64 sources, chunks
// of 256 edges: 14.6 ms at 256 to 512 edges a unit, 15.0 at 1024, 18.3 at 4096).
constexpr uint32_t kChunkUnit = 512;
// A work ticket covers kSpan units (28.0 -> 27.2 ms from 1 to 2; 4 was
// slower, 29.1 ms, from load imbalance).
constexpr uint32_t kSpan = 2;
constexpr uint32_t kLongDeg = kGroup;  // a relax window must fit inside the item

typedef uint32_t U32xG __attribute__((ext_vector_type(kGroup), aligned(4)));
typedef const __attribute__((address_space(4))) U32xG ScalarXG;
typedef const __attribute__((address_space(4))) uint32_t ScalarU32;

// Words [e, e + kGroup) of a CSR array that the launch never writes, loaded
// into scalar registers with one instruction (e is wave-uniform).
__device__ __forceinline__ U32xG scalar_window(const uint32_t *arr, uint32_t e) {
  return *(ScalarXG *)(arr + e);
}

// Improved edges since the last flush: lane i holds the destination of the
// i-th and the sources for which it must join the near / far pile.
struct Pending {
  uint32_t v, nb_lo, nb_hi, fb_lo, fb_hi;
  uint32_t n;  // wave-uniform
};
// The same for packed rows: in LDS, 64 entries a wavefront.
struct PackedEntry {
  uint32_t v, nb, fb;
};
struct PackedPending {
  PackedEntry *buf;
  uint32_t n;  // wave-uniform
};


// Sets the pending destinations' mask bits; a destination whose mask was
// empty joins the pile's queue (two entries for one destination: only the
// lane whose OR finds the mask empty pushes it).
__device__ __forceinline__ void flush_pending(const MArgs &a, const Sched &s, LaneSched &ls, Pending &p) {
  if (p.n == 0) return;
  order_release();
  const bool act = lane_id() < p.n && has_edges(a, lane_id() < p.n ? p.v : 0u);
  const uint64_t nb = ((uint64_t)p.nb_hi << 32) | p.nb_lo, fb = ((uint64_t)p.fb_hi << 32) | p.fb_lo;
  const bool pn = act && nb != 0 && atomic_or64(a.nmask[s.round & 1] + p.v, nb) == 0 && near_admit(a, s, p.v);
  const bool pf = act && fb != 0 && atomic_or64(a.fmask[s.phase & 1] + p.v, fb) == 0;
  pile_push(a, s, ls, 0, pn, p.v);
  pile_push(a, s, ls, 1, pf, p.v);
  p.n = 0;
}

// Takes a window of kGroup edges whose row loads are in flight (candidate
// cand(k) for row v[k], loaded distance val[k]): issues the atomicMins of the
// lanes whose candidate is lower and lists the improved edges.  Whether a lane
// improved is decided by the loaded distance, so no atomic returns a value
// (a lane that loses a race is expanded once more, for nothing); flush_pending
// waits for the atomics before it publishes their sources.
template <class Cand>
__device__ __forceinline__ void window_take(const MArgs &a, LaneSched &ls, const uint32_t (&v)[kGroup],
                                            const Cand &cand, const uint32_t (&val)[kGroup], uint32_t col, Pending &p,
                                            uint64_t &improved) {
  const uint32_t lane = lane_id();
#pragma unroll
  for (int k = 0; k < kGroup; ++k) {
    const uint32_t nd = cand(k);
    const bool imp = nd < val[k];
    const uint64_t im = __ballot(imp);
    if (im == 0) continue;
    if (imp) atomic_min(a.D + (size_t)v[k] * a.S + col, nd);
    const bool nearl = imp && nd <= ls.thr32;
    const uint64_t nb = __ballot(nearl), fb = im & ~nb;
    if (fb && imp && !nearl) ls.fmin = min(ls.fmin, nd);
    improved += 1;
    if (lane == p.n) {
      p.v = v[k];
      p.nb_lo = (uint32_t)nb;
      p.nb_hi = (uint32_t)(nb >> 32);
      p.fb_lo = (uint32_t)fb;
      p.fb_hi = (uint32_t)(fb >> 32);
    }
    p.n += 1;
  }
}

// Relaxes edges [lo, hi) of one item with at least kGroup edges (distance du
// for this lane's source), kGroup at a time.  The last window is shifted back to end
// at hi, so every window lies inside the item's edges, and its slots that
// the previous window covered are skipped.  Software-pipelined: while a
// window's row loads are in flight the next window's edges are fetched and
// the previous window's atomic results are taken, so a window costs about one
// memory round trip instead of three.
__device__ __forceinline__ void relax_edges(const MArgs &a, const Sched &s, LaneSched &ls, uint32_t du, uint32_t lo,
                                            uint32_t hi, Pending &p, uint64_t &improved) {
  const uint32_t lane = lane_id();
  // lanes >= S have no source and du = INF: they load the row's last word
  // and never issue an atomic
  const uint32_t col = min(lane, a.S - 1);
  // the bounds are wave-uniform; say so, so that they stay in scalar registers
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  uint32_t v[kGroup], nd[kGroup], val[kGroup], nv[kGroup], nnd[kGroup], nval[kGroup];
  // window of edges from e on: slots below e (relaxed already) carry no candidate
  auto load = [&](uint32_t e, uint32_t(&vv)[kGroup], uint32_t(&x)[kGroup], uint32_t(&c)[kGroup]) {
    const uint32_t w0 = min(e, hi - kGroup);
    const U32xG dst = scalar_window(a.edge_dst, w0), w = scalar_window(a.edge_data, w0);
#pragma unroll
    for (int k = 0; k < kGroup; ++k) {
      vv[k] = dst[k];
      c[k] = ld_coh(a.D + (size_t)dst[k] * a.S + col);
      // du + w never wraps (du <= INF, w <= INT_MAX); INF + w and a skipped
      // slot's du + 2^31 both exceed every stored distance
      x[k] = du + (w0 + k < e ? 0x80000000u : w[k]);
    }
  };
  load(lo, v, nd, val);
  for (uint32_t e = lo;;) {
    const uint32_t en = e + kGroup;
    const bool more = en < hi;
    if (more) load(en, nv, nnd, nval);
    if (p.n > (uint32_t)(kWave - kGroup)) flush_pending(a, s, ls, p);
    window_take(a, ls, v, [&](int k) { return nd[k]; }, val, col, p, improved);
    if (!more) break;
    e = en;
#pragma unroll
    for (int k = 0; k < kGroup; ++k) {
      v[k] = nv[k];
      nd[k] = nnd[k];
      val[k] = nval[k];
    }
  }
}

// ---- filtered relaxation ----------------------------------------------------

// Minimum / maximum over the wavefront's 64 lanes (DPP row shifts and
// broadcasts: no LDS round trips).
template <bool kMax>
__device__ __forceinline__ int32_t wave_extreme(int32_t x) {
  constexpr int32_t id = kMax ? -0x7FFFFFFF - 1 : 0x7FFFFFFF;
#define LSG_DPP_STEP(ctrl, rows)                                                    \
  {                                                                                 \
    const int32_t y = __builtin_amdgcn_update_dpp(id, x, ctrl, rows, 0xf, false);   \
    x = kMax ? max(x, y) : min(x, y);                                               \
  }
  LSG_DPP_STEP(0x111, 0xf)  // row_shr:1
  LSG_DPP_STEP(0x112, 0xf)  // row_shr:2
  LSG_DPP_STEP(0x114, 0xf)  // row_shr:4
  LSG_DPP_STEP(0x118, 0xf)  // row_shr:8
  LSG_DPP_STEP(0x142, 0xa)  // row_bcast:15
  LSG_DPP_STEP(0x143, 0xc)  // row_bcast:31
#undef LSG_DPP_STEP
  return __builtin_amdgcn_readlane(x, kWave - 1);
}

// Lowest offset distance of an item over the lanes with `act` (distance du).
__device__ __forceinline__ int32_t item_lowest(const LaneSched &ls, bool act, uint32_t du) {
  const int32_t x = !act ? kNoBound : ls.incl ? (int32_t)du - ls.off : kPass;
  return wave_extreme<false>(x);
}

// The bounds of every vertex with the offsets in a.flt: 64 consecutive rows
// per wavefront and step, kSweepRows row loads in flight.
constexpr int kSweepRows = 16;
__device__ __forceinline__ void sweep_bounds(const MArgs &a, const LaneSched &ls, int32_t *bound, uint32_t wave,
                                             uint32_t nwaves) {
  const uint32_t lane = lane_id(), col = min(lane, a.S - 1);
  for (uint64_t v0 = (uint64_t)wave * kWave; v0 < a.nnodes; v0 += (uint64_t)nwaves * kWave) {
    int32_t mine = 0;
    for (uint32_t r0 = 0; r0 < (uint32_t)kWave; r0 += kSweepRows) {
      uint32_t d[kSweepRows];
#pragma unroll
      for (int k = 0; k < kSweepRows; ++k) {
        const uint64_t v = v0 + r0 + k;
        d[k] = ld_coh(a.D + (size_t)(v < a.nnodes ? v : a.nnodes - 1) * a.S + col);
      }
#pragma unroll
      for (int k = 0; k < kSweepRows; ++k) {
        const int32_t x = !ls.incl ? -kNoBound : d[k] == kInf ? kNoBound : (int32_t)d[k] - ls.off;
        const int32_t m = wave_extreme<true>(x);
        if (lane == r0 + k) mine = m;
      }
    }
    if (v0 + lane < a.nnodes) st_coh((uint32_t *)bound + v0 + lane, (uint32_t)mine);
  }
}

// Relaxes the first n <= 64 listed edges (lane i: destination pv, weight pw,
// item slot pk), kGroup at a time, software-pipelined as relax_edges.
__device__ __forceinline__ void relax_listed(const MArgs &a, const Sched &s, LaneSched &ls, const DistSlots &dl,
                                             uint32_t pv, uint32_t pw, uint32_t pk, uint32_t n, Pending &p,
                                             uint64_t &improved) {
  const uint32_t lane = lane_id();
  const uint32_t col = min(lane, a.S - 1);
  uint32_t v[kGroup], val[kGroup], nv[kGroup], nval[kGroup];
  auto load = [&](uint32_t i, uint32_t(&vv)[kGroup], uint32_t(&x)[kGroup]) {
#pragma unroll
    for (int k = 0; k < kGroup; ++k) {
      vv[k] = readlane(pv, min(i + k, n - 1));  // a slot past the list repeats its last edge, with no candidate
      x[k] = ld_coh(a.D + (size_t)vv[k] * a.S + col);
    }
  };
  load(0, v, val);
  for (uint32_t i = 0; i < n; i += kGroup) {
    if (i + kGroup < n) load(i + kGroup, nv, nval);
    if (p.n > (uint32_t)(kWave - kGroup)) flush_pending(a, s, ls, p);
    auto cand = [&](int k) {
      const uint32_t j = min(i + k, n - 1);
      return dl[readlane(pk, j)][lane] + (i + k < n ? readlane(pw, j) : 0x80000000u);
    };
    window_take(a, ls, v, cand, val, col, p, improved);
#pragma unroll
    for (int k = 0; k < kGroup; ++k) {
      v[k] = nv[k];
      val[k] = nval[k];
    }
  }
}

// Up to kItems items' edges as one flattened list [0, total): lane k's item
// owns [end - degree, end), its edge f is CSR edge base + f, and its lowest
// offset distance is low.
struct Flat {
  uint32_t total, end, base;
  int32_t low;
};

// 64 edges of a flattened list, one per lane: destination, weight, item slot
// and the item's lowest offset distance (lanes past the list repeat its last edge).
struct FlatBatch {
  uint32_t v, w, k;
  int32_t low;
};
__device__ __forceinline__ void flat_load(const MArgs &a, const Flat &t, uint32_t b0, FlatBatch &x) {
  const uint32_t f = min(b0 + lane_id(), t.total - 1);
  uint32_t item = 0;  // the items that end at or before f
#pragma unroll
  for (int k = 0; k < kItems - 1; ++k) item += readlane(t.end, k) <= f ? 1u : 0u;
  const uint32_t e = __shfl(t.base, item) + f;
  x.v = glb(a.edge_dst)[e];
  x.w = glb(a.edge_data)[e];
  x.low = __shfl(t.low, item);
  x.k = item;
}

// ---- packed rows ------------------------------------------------------------
//
// With up to 32 (16) sources a row fills half (a quarter) of a wavefront or less:
// P = 2 (4) edges are relaxed side by side, lanes sub * kWave / P on for the
// sub-th.  A window is kSlots row accesses, P edges each, and its edges come from
// the lanes: long items are flattened too.  Ms with one row an access -> packed
// (learned schedule): RMAT of 16400 vertices x 5 sources 0.87 -> 0.70, 40000 x 20
// 1.49 -> 1.14, 500000 x 12 2.79 -> 2.03, 2^20 x 20 3.52 -> 2.82, 2^22 x 16 9.2 ->
// 7.7; fixed delta 100003 x 9 1.35 -> 1.28, 262900 x 3 1.85 -> 1.87.  (kSlots of 8 / 2:
// 2^20 x 20 3.09 / 2.9 at P = 2; 8 spilled 109 registers.  P = 8 up to 8 sources: 4
// to 8 % better with the learned schedule, 0 to 12 % worse without.)
template <int P>
struct Packing {
  static constexpr uint32_t kRow = kWave / P;  // lanes of an edge
  static constexpr int kSlots = 4;
  static constexpr uint32_t kWindow = kSlots * P;
};

// The source of this lane's column.
template <int P>
__device__ __forceinline__ uint32_t lane_source() {
  return P == 1 ? lane_id() : lane_id() % Packing<P>::kRow;
}

template <int P>
__device__ __forceinline__ void flush_packed(const MArgs &a, const Sched &s, LaneSched &ls, PackedPending &p) {
  if (p.n == 0) return;
  order_release();
  const bool in = lane_id() < p.n;
  const PackedEntry e = p.buf[in ? lane_id() : 0u];
  const bool act = in && has_edges(a, in ? e.v : 0u);
  const bool pn = act && e.nb != 0 && atomic_or64(a.nmask[s.round & 1] + e.v, e.nb) == 0 && near_admit(a, s, e.v);
  const bool pf = act && e.fb != 0 && atomic_or64(a.fmask[s.phase & 1] + e.v, e.fb) == 0;
  pile_push(a, s, ls, 0, pn, e.v);
  pile_push(a, s, ls, 1, pf, e.v);
  p.n = 0;
}

// window_take for packed rows.
template <int P, int N>
__device__ __forceinline__ void packed_take(const MArgs &a, LaneSched &ls, const uint32_t (&v)[N], const uint32_t (&nd)[N],
                                            const uint32_t (&val)[N], PackedPending &p, uint64_t &improved) {
  constexpr uint32_t kRow = Packing<P>::kRow;
  constexpr uint32_t kMask = (uint32_t)((1ull << kRow) - 1);
  const uint32_t col = lane_id() % kRow, shift = lane_id() / kRow * kRow;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const bool imp = nd[k] < val[k];
    const uint64_t im = __ballot(imp);
    if (im == 0) continue;
    if (imp) atomic_min(a.D + (size_t)v[k] * a.S + col, nd[k]);
    const bool nearl = imp && nd[k] <= ls.thr32;
    const uint64_t nb = __ballot(nearl);
    if (imp && !nearl) ls.fmin = min(ls.fmin, nd[k]);
    const uint32_t mine = (uint32_t)(im >> shift) & kMask, near = (uint32_t)(nb >> shift) & kMask;
    const bool lead = col == 0 && mine != 0;
    const uint64_t lm = __ballot(lead);
    if (lead) p.buf[p.n + lanes_below(lm)] = PackedEntry{v[k], near, mine & ~near};
    const uint32_t c = (uint32_t)__builtin_popcountll(lm);
    p.n += c;
    improved += c;
  }
}

// relax_listed for packed rows.
template <int P>
__device__ __forceinline__ void relax_listed_packed(const MArgs &a, const Sched &s, LaneSched &ls, const DistSlots &dl,
                                                    uint32_t pv, uint32_t pw, uint32_t pk, uint32_t n, PackedPending &p,
                                                    uint64_t &improved) {
  using K = Packing<P>;
  const uint32_t col = lane_id() % K::kRow, sub = lane_id() / K::kRow, colc = min(col, a.S - 1);
  for (uint32_t i = 0; i < n; i += K::kWindow) {
    uint32_t v[K::kSlots], nd[K::kSlots], val[K::kSlots];
#pragma unroll
    for (int k = 0; k < K::kSlots; ++k) {
      const uint32_t at = i + (uint32_t)k * P + sub, j = min(at, n - 1);
      v[k] = (uint32_t)__shfl(pv, j);
      const uint32_t wt = (uint32_t)__shfl(pw, j), item = (uint32_t)__shfl(pk, j);  // by every lane
      val[k] = ld_coh(a.D + (size_t)v[k] * a.S + colc);
      // (an edge past the list repeats its last one, with no candidate)
      nd[k] = dl[item][col] + (at < n ? wt : 0x80000000u);
    }
    if (p.n > (uint32_t)kWave - K::kWindow) flush_packed<P>(a, s, ls, p);
    packed_take<P, K::kSlots>(a, ls, v, nd, val, p, improved);
  }
}

// A flattened list without the test: 64 edges at a time.
template <int P>
__device__ __forceinline__ void relax_packed(const MArgs &a, const Sched &s, LaneSched &ls, const DistSlots &dl,
                                             const Flat &t, PackedPending &p, uint64_t &improved) {
  if (t.total == 0) return;
  FlatBatch x, y;
  flat_load(a, t, 0, x);
  for (uint32_t b0 = 0; b0 < t.total; b0 += kWave) {
    flat_load(a, t, b0 + kWave, y);
    relax_listed_packed<P>(a, s, ls, dl, x.v, x.w, x.k, min((uint32_t)kWave, t.total - b0), p, improved);
    x = y;
  }
}

// Relaxes a flattened list (total > 0).  The lanes take one edge each and test
// it against its destination's bound; the edges that pass are collected in a
// list of up to 64, one per lane, and relaxed from there.  Three batches of 64
// are in flight: while one is tested and relaxed, the next one's bounds and
// the edges of the one after it are being loaded.
template <int P, class Pend>
__device__ __forceinline__ void relax_filtered(const MArgs &a, const Sched &s, LaneSched &ls, const DistSlots &dl,
                                               const Flat &t, Pend &p, uint64_t &improved) {
  const uint32_t lane = lane_id();
  uint32_t pv = 0, pw = 0, pk = 0, n = 0;
  FlatBatch x0, x1, x2;
  flat_load(a, t, 0, x0);
  flat_load(a, t, kWave, x1);
  int32_t bd0 = glb(ls.bound)[x0.v], bd1;
  for (uint32_t b0 = 0;; b0 += kWave) {
    uint64_t m = 0;
    uint32_t c = 0;
    if (b0 < t.total) {
      flat_load(a, t, b0 + 2 * kWave, x2);
      bd1 = glb(ls.bound)[x1.v];
      // the saturated sum is below a bound exactly when the sum is
      m = __ballot(b0 + lane < t.total && (x0.low == kPass || bd0 == kNoBound ||
                                           __builtin_elementwise_add_sat(x0.low, (int32_t)x0.w) < bd0));
      c = (uint32_t)__builtin_popcountll(m);
    }
    if (n && (b0 >= t.total || n + c > (uint32_t)kWave)) {
      if constexpr (P > 1) relax_listed_packed<P>(a, s, ls, dl, pv, pw, pk, n, p, improved);
      else relax_listed(a, s, ls, dl, pv, pw, pk, n, p, improved);
      n = 0;
    }
    if (b0 >= t.total) break;
    if (c) {
      // a permutation of the lanes: passing edges to n, n + 1, ..., the others behind them
      const uint32_t to = ((m >> lane) & 1 ? n + lanes_below(m) : n + c + lanes_below(~m)) % kWave * 4;
      const uint32_t tv = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)x0.v);
      const uint32_t tw = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)x0.w);
      const uint32_t tk = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)x0.k);
      if (lane >= n && lane < n + c) {
        pv = tv;
        pw = tw;
        pk = tk;
      }
      n += c;
    }
    x0 = x1;
    x1 = x2;
    bd0 = bd1;
  }
}

// Writes the staged heavy items' chunks to the next round's chunk queue, from
// slot `base` on (reserved for ls.hchunks chunks).
__device__ __forceinline__ void heavy_write(const MArgs &a, const Sched &s, LaneSched &ls, uint32_t base) {
  uint64_t *const hq = a.hq[1u - s.heavy_in];
  for (uint32_t i = 0; i < ls.hn; ++i) {
    const HeavyItem h = ls.hb[i];
    const uint32_t nch = __builtin_amdgcn_readfirstlane(h.nch);
    for (uint32_t k = lane_id(); k < nch; k += kWave) {
      const uint32_t pos = base + k;
      if (pos < a.hcap) {
        st_coh64(hq + 2ull * pos, ((uint64_t)k << 32) | h.u);
        st_coh64(hq + 2ull * pos + 1, h.mask);
      } else {
        st_coh(&a.ctrl->abort, kAbortCapacity);
      }
    }
    base += nch;
  }
  ls.hn = ls.hchunks = 0;
}

// Queues heavy vertex u (edges [rs, re)) as chunks of heavy_deg edges, each
// expanded by a wavefront in the next round with the sources active now.
__device__ __forceinline__ void queue_heavy(const MArgs &a, const Sched &s, LaneSched &ls, uint32_t u, uint32_t rs,
                                            uint32_t re, uint64_t am) {
  if (ls.hn == kHeavyBuf) {
    uint32_t base = 0;
    if (lane_id() == 0) base = atomic_add(&a.ctrl->hcount[1u - s.heavy_in], ls.hchunks);
    heavy_write(a, s, ls, readlane(base, 0));
  }
  const uint32_t nch = (re - rs + a.heavy_deg - 1) / a.heavy_deg;
  if (lane_id() == 0) ls.hb[ls.hn] = HeavyItem{u, nch, am};
  ls.hn += 1;
  ls.hchunks += nch;
}

// One work unit, up to kItems items: frontier items [base, base + cnt), cnt <=
// per, or, with `chunks`, that many of the round's heavy chunks (heavy_deg
// edges of a vertex, for the sources recorded with the chunk).  Lane k consumes
// item k's mask and loads its row bounds; the distance rows of all the items
// are then loaded together and parked in dl.  Heavy items are queued as
// chunks for the next round; the others are relaxed (items of kLongDeg edges
// and more one by one, the rest as one flattened list, 64 edges per batch) or,
// with kFilter, returned as one flattened list.
template <bool kFilter, int P, class Pend>
__device__ __forceinline__ Flat process_unit(const MArgs &a, const Sched &s, LaneSched &ls, bool chunks, uint32_t base,
                                             uint32_t per, DistSlots &dl, RoundCounters &mc, Pend &p) {
  const uint32_t lane = lane_id();
  const uint32_t cnt = min(per, (chunks ? s.heavy_count : s.in_count) - base);
  uint32_t u = a.nnodes;
  uint64_t m = 0;
  uint32_t rs = 0, re = 0;
  if (chunks) {
    uint32_t ck = 0;
    if (lane < cnt) {
      const uint64_t *const ent = a.hq[s.heavy_in] + 2ull * (base + lane);
      const uint64_t uk = ld_coh64(ent);
      m = ld_coh64(ent + 1);
      u = (uint32_t)uk;
      ck = (uint32_t)(uk >> 32);
    }
    if (u < a.nnodes) {
      rs = glb(a.row_start)[u] + ck * a.heavy_deg;
      re = min(glb(a.row_start)[u + 1], rs + a.heavy_deg);
    } else {
      m = 0;
    }
  } else {
    uint64_t *mp = s.aux[0] ? a.fmask[(s.phase - 1) & 1] : a.nmask[(s.round - 1) & 1];
    if (lane < cnt) u = ld_coh(a.q[s.in_q] + base + lane);
    if (u < a.nnodes) {
      m = atomic_exch64(mp + u, 0ull);
      // Gauss-Seidel pop: the bits set for the next round so far are expanded
      // now, with the distances that set them; u stays queued for the next round.
      m |= atomic_exch64(a.nmask[s.round & 1] + u, 0ull);
      rs = glb(a.row_start)[u];
      re = glb(a.row_start)[u + 1];
    }
  }
  // The row loads depend on the exchanged masks, so each reads a distance at
  // least as new as the improvements that set the consumed bits.
  uint32_t du[kItems];
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const uint64_t mk = bcast64(m, k);
    const uint32_t uk = readlane(u, k);
    du[k] = lane < a.S && ((mk >> lane) & 1) ? ld_coh(a.D + (size_t)uk * a.S + lane) : kInf;
  }
  uint64_t am = 0;         // lane k: sources that expand item k
  int32_t low = kNoBound;  // lane k: item k's lowest offset distance (filtered rounds)
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    dl[k][lane] = du[k];
    const uint64_t b = __ballot(du[k] != kInf);
    int32_t x = 0;
    if (kFilter) x = item_lowest(ls, du[k] != kInf, du[k]);
    if (lane == (uint32_t)k) {
      am = b;
      low = x;
    }
  }
  if (s.aux[0] && s.aux[1] && !chunks) {
    // Split / bucket far pile: a source whose distance is still above this
    // phase's threshold (shared, or its own in a bucket phase) waits for a
    // later phase instead of expanding early.
    for (uint32_t k = 0; k < cnt; ++k) {
      const uint32_t d = dl[k][lane];
      const bool defer = d != kInf && (ls.bucket ? d > ls.thr : (int64_t)d > s.curdelta());
      const uint64_t dm = __ballot(defer);
      if (dm == 0) continue;
      const uint32_t uk = readlane(u, k);
      bool push = false;
      if (lane == 0) push = atomic_or64(a.fmask[s.phase & 1] + uk, dm) == 0;
      pile_push(a, s, ls, 1, push, uk);
      if (defer) {
        ls.fmin = min(ls.fmin, d);
        dl[k][lane] = kInf;
      }
      int32_t x = 0;
      if (kFilter) x = item_lowest(ls, d != kInf && !defer, d);
      if (lane == k) {
        am &= ~dm;
        low = x;
      }
    }
  }
  const uint32_t deg = am ? re - rs : 0u;  // lane k: edges of item k
  const bool heavy = !chunks && deg >= a.heavy_deg;
  for (uint64_t hm = __ballot(heavy); hm; hm &= hm - 1) {
    const uint32_t k = (uint32_t)__builtin_ctzll(hm);
    queue_heavy(a, s, ls, readlane(u, k), readlane(rs, k), readlane(re, k), bcast64(am, k));
  }
  const uint32_t now = heavy ? 0u : deg;  // relaxed in this round
  if (now) {
    mc.lane_items += __builtin_popcountll(am);
    mc.edges += now;
  }
  // items relaxed one by one (degree >= kLongDeg); the others as a flattened list
  const uint32_t longm = kFilter || P > 1 ? 0u : (uint32_t)__ballot(now >= kLongDeg);
  const uint32_t mydeg = kFilter || P > 1 || now < kLongDeg ? now : 0u;
  // Inclusive prefix of the items' edge counts over lanes 0..kItems-1: item k
  // owns flattened edges [end_k - deg_k, end_k).
  uint32_t end = mydeg;
#pragma unroll
  for (int d = 1; d < kItems; d <<= 1) {
    const uint32_t t = __shfl_up(end, d);
    if (lane >= (uint32_t)d) end += t;
  }
  const uint32_t total = readlane(end, kItems - 1);
  const uint32_t first = end - mydeg;
  if (kFilter) return Flat{total, end, rs - first, low};
  if constexpr (P > 1) {
    relax_packed<P>(a, s, ls, dl, Flat{total, end, rs - first, 0}, p, mc.improved);
  } else {
  for (uint32_t b0 = 0; b0 < total; b0 += kWave) {
    const uint32_t f = b0 + lane;
    // the item holding flattened edge f is the number of items ending at or before f
    uint32_t item = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) item += readlane(end, k) <= f;
    const uint32_t e = __shfl(rs, item) + (f - __shfl(first, item));
    uint32_t ev = 0, ew = 0;
    if (f < total) {
      ev = glb(a.edge_dst)[e];
      ew = glb(a.edge_data)[e];
    }
    relax_batch(a, s, ls, dl, min((uint32_t)kWave, total - b0), ev, ew, item, &mc.improved);
  }
  for (uint32_t lm = longm; lm; lm &= lm - 1) {
    const uint32_t k = (uint32_t)__builtin_ctz(lm);
    relax_edges(a, s, ls, dl[k][lane], readlane(rs, k), readlane(re, k), p, mc.improved);
  }
  }
  return Flat{0, 0, 0, 0};
}

// Leader step, run by every thread of the last block to reach the barrier:
// the pile rotation of apps/sssp/kernel.cu:363-384 for all sources at once,
// plus, at each phase boundary, the learned scheduler's choice of the next
// phase's delta width and far-pile mode.  Schedule words: aux[0] = the
// in-queue is the far pile, aux[1] = far mode of this phase (LSG_FAR_*).
__device__ __forceinline__ void multi_leader(const MArgs &a) {
  __shared__ Sched s;
  __shared__ SchedFeatures f;
  __shared__ MlpScratch sc;
  __shared__ uint32_t phase_end, consumed;
  __shared__ uint64_t phases_seen;
  __shared__ uint64_t edges_now;
  Ctrl *c = a.ctrl;
  const uint32_t t = threadIdx.x;
  // the hub's distances, for the filter's offsets (beside the loads below)
  const uint32_t hub_d = t < a.S && ld_coh(&a.flt->on) ? ld_coh(a.D + (size_t)ld_coh(&a.flt->hub) * a.S + t) : kInf;
  // every wavefront has left the round's item loops: restart the tickets
  if (t < kGroups) st_coh(&a.tickets[t].ticket, 0u);
  if (t == 0) {
    // every control word of the step in one batch of loads (the schedule to
    // registers first, so that the other loads need not wait for LDS stores)
    Sched sr;
    sched_load(sr, &c->s);
    CtrlCounts k;
    counts_load(k, c);
    uint64_t tot_lane_items = 0, tot_edges = 0;
#pragma unroll
    for (uint32_t g = 0; g < kGroups; ++g) {
      tot_lane_items += ld_coh64(&a.tot[g].lane_items);
      tot_edges += ld_coh64(&a.tot[g].edges);
    }
    s = sr;
    s.aux[3] = 0;
    edges_now = tot_edges;
    const uint32_t nnear = k.q(s.near_q), nfar = k.q(s.far_q), nheavy = k.h(1u - s.heavy_in);
    phase_end = 0;
    phases_seen = k.phases;
    if (nnear > a.qcap || nfar > a.qcap || nheavy > a.hcap) {
      st_coh(&c->abort, kAbortCapacity);
      s.done = 1;
    } else {
      st_coh64(&c->stat_items, k.items + s.in_count);
      st_coh64(&c->stat_heavy, k.heavy + s.heavy_count);
      st_coh64(&c->stat_rounds, k.rounds + 1);
      if (a.trace && s.round - 1 < a.trace_cap) {
        lsg_round_trace &r = a.trace[s.round - 1];
        r.round = s.round;
        r.phase = s.phase;
        r.in_items = s.in_count;
        r.heavy_chunks = s.heavy_count;
        r.near_out = nnear;
        r.far_out = nfar;
        r.heavy_out = nheavy;
        r.curdelta_lo = s.curdelta_lo;
        r.curdelta_hi = s.curdelta_hi;
        r.delta = s.delta;
        r.t_end = wall_clock64();
      }
      consumed = s.in_q;
      st_coh(&c->hcount[s.heavy_in], 0u);
      s.heavy_in = 1u - s.heavy_in;
      s.heavy_count = nheavy;
      if (nnear > 0 || nheavy > 0) {
        s.in_q = s.near_q;
        s.in_count = nnear;
        s.near_q = consumed;
        st_coh(&c->qcount[consumed], 0u);
        s.aux[0] = 0;
        s.round += 1;
      } else if (nfar > 0) {
        phase_end = 1;
        f.in_items = nfar;
        f.phase = s.phase;
        f.round = s.round;
        f.curdelta = (float)s.curdelta();
        f.base_delta = a.delta;
        f.prev_delta = s.delta;
        f.lane_items = (float)tot_lane_items;
        f.edges = (float)tot_edges;
        f.nnodes = a.nnodes;
        f.nedges = (float)a.nedges;
        f.nsrc = a.S;
      } else {
        s.done = 1;
        st_coh64(&c->stat_phases, k.phases + 1);
      }
    }
  }
  __syncthreads();
  // Another sweep, once three quarters of the sources have reached the hub:
  // the next round begins with it, with the hub's distances as offsets.
  if (t < (uint32_t)kWave && s.aux[2] < (uint32_t)kSweeps) {
    const uint64_t fin = __ballot(hub_d != kInf);
    if (4u * (uint32_t)__builtin_popcountll(fin) >= 3u * a.S &&
        edges_now - ld_coh64(&a.flt->last_edges) >= a.nedges / 2) {
      st_coh((uint32_t *)&a.flt->off[t], hub_d != kInf ? hub_d : 0u);
      if (t == 0) {
        st_coh64(&a.flt->incl, fin);
        st_coh64(&a.flt->last_edges, edges_now);
        s.aux[2] += 1;
        s.aux[3] = 1;
      }
    }
  }
  __syncthreads();
  if (!phase_end) {
    if (t == 0) sched_store(&c->s, s);
    return;
  }
  __shared__ int act_sh;
  int act = -1;
  if (a.sched) act = mlp_block_action(a.mlp, f, sc);
  if (t == 0 && a.pace) {
    Pace &p = *a.pace;  // touched by leaders only, ordered by the barrier
    uint32_t step = ld_coh(&p.step), hold = ld_coh(&p.hold);
    float best = __uint_as_float(ld_coh((uint32_t *)&p.best));
    const float rounds = (float)(s.round - ld_coh(&p.rounds)), edges = (float)(edges_now - ld_coh64(&p.edges));
    const float cost = kRoundUs * rounds + edges / kEdgesPerUs, rate = (float)step / cost;
    if (s.phase == 0) {  // the sources alone
      step = ld_coh(&a.flt->on) ? kHubStep : 1u;
    } else if (hold == 0 || cost < 1.25f * kRoundUs * rounds) {
      hold = 0;
      if (rate > 1.02f * best || cost < 1.25f * kRoundUs * rounds) {
        best = rate;
        step = min(step * 2, kMaxMultiStep);
      } else {
        step = max(step / 2, 1u);
        hold = 2;
      }
    } else if (--hold == 0) {
      best = rate;
      step = min(step * 2, kMaxMultiStep);
    }
    st_coh(&p.step, step);
    st_coh(&p.hold, hold);
    st_coh((uint32_t *)&p.best, __float_as_uint(best));
    st_coh(&p.rounds, s.round);
    st_coh64(&p.edges, edges_now);
    s.delta = (uint32_t)min((uint64_t)step * a.delta, (uint64_t)kInf);
  }
  if (t == 0) {
    if (act >= 0) {
      s.delta = action_delta(a.mlp, act, a.delta);
      s.aux[1] = (uint32_t)a.mlp[kOffFarMode + act];
    }
    act_sh = act;
  }
  __syncthreads();
  // Per-source thresholds of the next phase: smallest pending far distance
  // of each source + delta - 1; the recorded minima of the phase after start
  // empty.  (Tracked in every phase so any phase can switch to bucket mode.)
  if (t < a.S) {
    uint32_t m = ld_coh(a.fmin + (s.phase & 1) * 64 + t);
    uint64_t th = m == kInf ? (uint64_t)kInf : (uint64_t)m + s.delta - 1;
    st_coh(a.thr + t, (uint32_t)min(th, (uint64_t)kInf - 1));
    st_coh(a.fmin + ((s.phase + 1) & 1) * 64 + t, kInf);
  }
  if (t == 0) {
    act = act_sh;
    if (a.feat && s.phase < (uint32_t)kMaxForced) {
      float *rec = a.feat + (size_t)s.phase * kFeatRec;
      sched_featurize(f, rec);
      rec[kFeat] = (float)act;
      rec[kFeat + 1] = (float)s.delta;
      rec[kFeat + 2] = (float)s.aux[1];
      rec[kFeat + 3] = (float)(s.round + 1);  // first round of the phase being started
    }
    s.in_q = s.far_q;
    s.in_count = f.in_items;
    s.far_q = consumed;
    st_coh(&c->qcount[consumed], 0u);
    s.aux[0] = 1;
    s.set_curdelta(s.curdelta() + s.delta);
    s.phase += 1;
    s.round += 1;
    st_coh64(&c->stat_phases, phases_seen + 1);
    sched_store(&c->s, s);
  }
}

__device__ __forceinline__ uint64_t wave_sum(uint64_t x) {
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) x += __shfl_xor((unsigned long long)x, d);
  return x;
}

// Blocks of group g in a grid of nb.
__device__ __forceinline__ uint32_t group_blocks(uint32_t nb, uint32_t g) { return (nb + kGroups - 1 - g) / kGroups; }

// kFilter: the rounds from the first sweep on, whose edges are all tested
// against the bounds; the other variant runs the rounds before, and returns
// when a sweep has been ordered.  (One kernel with both edge loops spilled
// 170 VGPRs.)
template <int BS, bool kFilter, int P>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(kMultiWaves, kMultiWaves)))
void multi_kernel(MArgs a) {
  __shared__ Sched ss;
  __shared__ uint32_t quit;
  __shared__ unsigned long long blk[3];
  __shared__ DistSlots dls[BS / kWave];
  __shared__ uint32_t pushbuf[BS / kWave][2 * kPushBuf];
  __shared__ HeavyItem heavybuf[BS / kWave][kHeavyBuf];
  __shared__ uint32_t drain_n[BS / kWave][3], drain_base[3];  // near, far, heavy chunks
  __shared__ PackedEntry pend[P > 1 ? BS / kWave : 1][P > 1 ? kWave : 1];
  Ctrl *c = a.ctrl;
  const uint32_t nb = gridDim.x;
  if (!residency_handshake(c, nb, a.residency_limit)) return;
  const uint32_t wpb = BS / kWave;
  const uint32_t wave = blockIdx.x * wpb + threadIdx.x / kWave;
  const uint32_t nwaves = nb * wpb;
  for (;;) {
    if (threadIdx.x == 0) {
      Sched s;
      sched_load(s, &c->s);
      ss = s;
      quit = s.done || (!kFilter && s.aux[3]) || ld_coh(&c->abort) != kAbortNone;
      blk[0] = blk[1] = blk[2] = 0;
    }
    __syncthreads();
    if (quit) break;
    const Sched s = ss;
    RoundCounters mc = {0, 0, 0};
    LaneSched ls;
    ls.bucket = s.aux[1] == LSG_FAR_BUCKET;
    ls.thr = ls.bucket && lane_source<P>() < a.S ? ld_coh(a.thr + lane_source<P>()) : 0u;
    ls.thr32 = ls.bucket ? ls.thr : (uint32_t)min(s.curdelta(), (int64_t)UINT32_MAX);
    ls.fmin = kInf;
    ls.pb = &pushbuf[threadIdx.x / kWave][0];
    ls.pbn[0] = ls.pbn[1] = 0;
    ls.hb = heavybuf[threadIdx.x / kWave];
    ls.hn = ls.hchunks = 0;
    ls.bound = nullptr;
    ls.off = 0;
    ls.incl = false;
    if (kFilter) {
      int32_t *const bound = s.aux[2] == 1 ? a.bound[0] : s.aux[2] == 2 ? a.bound[1] : a.bound[2];
      ls.bound = bound;
      ls.off = (int32_t)ld_coh((const uint32_t *)&a.flt->off[lane_id()]);
      ls.incl = (ld_coh64(&a.flt->incl) >> lane_id()) & 1;
      if (s.aux[3]) {
        sweep_bounds(a, ls, bound, wave, nwaves);
        grid_barrier_block(c, nb, a.spin_limit, [] {});
        acquire_agent();  // no line of the bounds that was read before is kept
      }
    }
    typename std::conditional<(P > 1), PackedPending, Pending>::type p;
    p.n = 0;
    if constexpr (P > 1) p.buf = pend[threadIdx.x / kWave];
    else p.v = p.nb_lo = p.nb_hi = p.fb_lo = p.fb_hi = 0;
    DistSlots &dl = dls[threadIdx.x / kWave];
    // Work units: first the in-queue's items, `per` at a time (fewer than
    // kItems where that would leave wavefronts idle), then the heavy chunks.
    // Where each wavefront has one at most, the unit of its number; else unit j
    // * kGroups + g belongs to group g, whose wavefronts take one each, then
    // kSpan per ticket (the next ticket is fetched while the last unit of the
    // current one is processed), and at the end help other groups.
    const uint32_t per = min((uint32_t)kItems, max(1u, (s.in_count + nwaves - 1) / nwaves));
    const uint32_t hper = min(min((uint32_t)kItems, max(1u, kChunkUnit / a.heavy_deg)),
                              max(1u, (s.heavy_count + nwaves - 1) / nwaves));
    const uint32_t nitems = (s.in_count + per - 1) / per;
    const uint32_t nunits = nitems + (s.heavy_count + hper - 1) / hper;
    const bool few = nunits <= nwaves;
    uint32_t g = blockIdx.x % kGroups;
    uint32_t j = blockIdx.x / kGroups * wpb + threadIdx.x / kWave, jend = j + 1;
    for (;;) {
      const uint32_t u = few ? wave : j * kGroups + g;
      if (u < nunits) {
        const bool last = j + 1 >= jend && !few;
        uint32_t t = 0;
        if (last && lane_id() == 0) t = atomic_add(&a.tickets[g].ticket, 1u);
        const bool chunks = u >= nitems;
        const Flat f = process_unit<kFilter, P>(a, s, ls, chunks, chunks ? (u - nitems) * hper : u * per,
                                             chunks ? hper : per, dl, mc, p);
        if (kFilter && f.total) relax_filtered<P>(a, s, ls, dl, f, p, mc.improved);
        if (last) {
          j = group_blocks(nb, g) * wpb + readlane(t, 0) * kSpan;
          jend = j + kSpan;
        } else {
          ++j;
          if (few) break;
        }
        continue;
      }
      if (few) break;
      // this group's units are taken: the next group that has some left
      const uint32_t og = (g + 1 + lane_id()) % kGroups;
      const uint32_t oj = group_blocks(nb, og) * wpb + ld_coh(&a.tickets[og].ticket) * kSpan;
      const uint64_t left = __ballot(lane_id() < kGroups && oj * kGroups + og < nunits);
      if (left == 0) break;
      g = (g + 1 + (uint32_t)__builtin_ctzll(left)) % kGroups;
      uint32_t t = 0;
      if (lane_id() == 0) t = atomic_add(&a.tickets[g].ticket, 1u);
      j = group_blocks(nb, g) * wpb + readlane(t, 0) * kSpan;
      jend = j + kSpan;
    }
    if constexpr (P > 1) flush_packed<P>(a, s, ls, p);
    else flush_pending(a, s, ls, p);
    dl[0][lane_id()] = ls.fmin;  // (the items' distances are no longer needed)
    const uint32_t wv = threadIdx.x / kWave;
    const uint64_t lane_items = wave_sum(mc.lane_items), edges = wave_sum(mc.edges);
    if (lane_id() == 0) {
      drain_n[wv][0] = ls.pbn[0];
      drain_n[wv][1] = ls.pbn[1];
      drain_n[wv][2] = ls.hchunks;
      if (lane_items | edges) {
        atomicAdd(&blk[0], (unsigned long long)lane_items);
        atomicAdd(&blk[1], (unsigned long long)edges);
        atomicAdd(&blk[2], (unsigned long long)mc.improved);
      }
    }
    __syncthreads();
    // The block's staged pushes get their places with one queue-tail atomic
    // per pile (one per wavefront, 4096 on one tail, serialise for ~50 us at
    // the memory-side atomic unit every round).
    if (threadIdx.x < 3) {
      const uint32_t which = threadIdx.x;
      uint32_t tot_n = 0;
      for (uint32_t w = 0; w < BS / kWave; ++w) {
        const uint32_t n = drain_n[w][which];
        drain_n[w][which] = tot_n;  // becomes the wavefront's offset
        tot_n += n;
      }
      uint32_t *const tail = which == 2 ? &c->hcount[1u - s.heavy_in] : &c->qcount[which ? s.far_q : s.near_q];
      drain_base[which] = tot_n ? atomic_add(tail, tot_n) : 0u;
    }
    // The block's smallest far push per source -> phase minimum.  One atomic per
    // wavefront and lane, 64 words that every wavefront meets at (with packed rows
    // the same word 2 or 4 times over), took most of a wide round that defers: ms, 16
    // sources, 300,000 vertices of out-degree 4 6.4 -> 2.0, grid 500^2 at 1000 28.7
    // -> 23.6; RMAT of 2^18 vertices, weights to 10000, x 24 19.0 -> 9.9; smallest
    // distances as thresholds, road-like 300^2 x 16 at 32 1905 -> 843.
    if (threadIdx.x >= BS - kWave) {
      uint32_t m = kInf;
      for (uint32_t w = 0; w < BS / kWave; ++w) m = min(m, dls[w][0][lane_id()]);
#pragma unroll
      for (uint32_t d = kWave / P; d < kWave; d *= 2) m = min(m, (uint32_t)__shfl_xor(m, d));
      if (m != kInf && lane_id() < kWave / P) atomic_min(a.fmin + (s.phase & 1) * 64 + lane_id(), m);
    }
    if (threadIdx.x == 0 && (blk[0] | blk[1])) {
      MultiCounters *const tot = a.tot + blockIdx.x % kGroups;
      __hip_atomic_fetch_add(&tot->lane_items, (uint64_t)blk[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_add(&tot->edges, (uint64_t)blk[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_add(&tot->improved, (uint64_t)blk[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      const uint32_t n = ls.pbn[which];
      if (n == 0) continue;
      const uint32_t qi = which ? s.far_q : s.near_q;
      const uint32_t base = drain_base[which] + drain_n[wv][which];
      const uint32_t *buf = ls.pb + which * kPushBuf;
      for (uint32_t i = lane_id(); i < n; i += kWave) {
        const uint32_t pos = base + i;
        if (pos < a.qcap) st_coh(a.q[qi] + pos, buf[i]);
        else st_coh(&a.ctrl->abort, kAbortCapacity);
      }
    }
    if (ls.hn) heavy_write(a, s, ls, drain_base[2] + drain_n[wv][2]);
    grid_barrier_block(c, nb, a.spin_limit, [&] { multi_leader(a); });
  }
}

// D[v][s] = INF, masks cleared.
__global__ void multi_init(MArgs a) {
  size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x;
  size_t cells = (size_t)a.nnodes * a.S;
  for (size_t i = tid; i < cells; i += nt) a.D[i] = kInf;
  for (size_t v = tid; v < a.nnodes; v += nt) {
    a.nmask[0][v] = 0;
    a.nmask[1][v] = 0;
    a.fmask[0][v] = 0;
    a.fmask[1][v] = 0;
    a.qstamp[v] = 0;
  }
  if (tid < kGroups) {
    a.tot[tid] = MultiCounters{0, 0, 0};
    a.tickets[tid].ticket = 0;
  }
  // the block's vertex of largest out-degree (lowest id on ties)
  __shared__ unsigned long long best;
  if (threadIdx.x == 0) best = 0;
  __syncthreads();
  uint64_t mine = 0;
  for (size_t v = tid; v < a.nnodes; v += nt) {
    const uint64_t x = (uint64_t)(a.row_start[v + 1] - a.row_start[v]) << 32 | (uint32_t)~(uint32_t)v;
    mine = x > mine ? x : mine;
  }
  atomicMax(&best, (unsigned long long)mine);
  __syncthreads();
  if (threadIdx.x == 0) a.hubs[blockIdx.x] = best;
}

// Seeds every source (apps/sssp/kernel.cu:33,476-477) and the control block.
// One wavefront; lane s seeds source s.
__global__ void multi_seed(MArgs a) {
  const uint32_t lane = threadIdx.x;
  bool act = lane < a.S;
  uint32_t src = act ? a.srcs[lane] : 0u;
  bool push = false;
  if (act) {
    a.D[(size_t)src * a.S + lane] = 0u;
    push = atomic_or64(a.nmask[0] + src, 1ull << lane) == 0;
    a.qstamp[src] = 1u;  // in round 1's queue
  }
  uint64_t pm = __ballot(push);
  if (push) a.q[0][lanes_below(pm)] = src;
  ctrl_reset_barrier(a.ctrl, lane, kWave);
  uint64_t hub = 0;
  for (uint32_t i = lane; i < a.ninit; i += kWave) hub = a.hubs[i] > hub ? a.hubs[i] : hub;
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) {
    const uint64_t x = __shfl_xor((unsigned long long)hub, d);
    hub = x > hub ? x : hub;
  }
  if (lane == 0) {
    a.flt->hub = ~(uint32_t)hub;
    a.flt->on = (hub >> 32) * a.nnodes >= (uint64_t)kHubRatio * a.nedges && a.nedges;
    a.flt->incl = a.flt->last_edges = 0;
    if (a.pace) *a.pace = Pace{1, 0, 0.0f, 0, 0};
    Ctrl *c = a.ctrl;
    c->qcount[0] = (uint32_t)__builtin_popcountll(pm);
    c->qcount[1] = 0;
    c->qcount[2] = 0;
    c->hcount[0] = 0;
    c->hcount[1] = 0;
    c->abort = kAbortNone;
    c->checkin = 0;
    c->resident_seen = 0;
    Sched s;
    memset(&s, 0, sizeof s);
    s.in_q = 0;
    s.near_q = 1;
    s.far_q = 2;
    s.in_count = (uint32_t)__builtin_popcountll(pm);
    s.round = 1;
    s.set_curdelta(0);
    s.delta = a.delta;
    s.aux[1] = a.far_mode;
    c->s = s;
    for (int k = 0; k < 64; ++k) {
      a.fmin[k] = kInf;
      a.fmin[64 + k] = kInf;
      a.thr[k] = 0u;  // phase 0: threshold 0, as curdelta starts at 0 (apps/sssp/kernel.cu:472)
    }
    c->stat_items = c->stat_rounds = c->stat_heavy = c->stat_phases = c->stat_edges = 0;
  }
}

// out[k][v] = D[v][k] for the units of one launch (per-source arrays).
__global__ void multi_scatter(const uint32_t *D, uint32_t S, uint32_t nnodes, int32_t *const *outs) {
  size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x;
  size_t cells = (size_t)nnodes * S;
  for (size_t i = tid; i < cells; i += nt) {
    uint32_t v = (uint32_t)(i / S), k = (uint32_t)(i % S);
    outs[k][v] = (int32_t)D[i];
  }
}

// Out-degree of each source (deg[i] for srcs[i]).
__global__ void source_degree_kernel(const uint32_t *row_start, const uint32_t *srcs, uint32_t n, uint32_t *deg) {
  if (threadIdx.x < n) deg[threadIdx.x] = row_start[srcs[threadIdx.x] + 1] - row_start[srcs[threadIdx.x]];
}

// D [V][S] from the compact Dc [V][Sc] of the sources that have out-edges:
// column s is Dc's column col[s], or, for a source without out-edges, INF
// except 0 at the source itself.  One wavefront per row, lane = column (8
// rows per wavefront step measured slower: 0.63 vs 0.48 ms on RMAT-22).
__global__ void multi_expand(const uint32_t *Dc, uint32_t Sc, const int32_t *col, const uint32_t *srcs, uint32_t S,
                             uint32_t V, uint32_t *D) {
  const uint32_t lane = lane_id();
  const size_t nwaves = (size_t)gridDim.x * blockDim.x / kWave;
  const int32_t c = lane < S ? col[lane] : -1;
  const uint32_t sv = lane < S ? srcs[lane] : 0u;
  for (size_t v = (blockIdx.x * (size_t)blockDim.x + threadIdx.x) / kWave; v < V; v += nwaves)
    if (lane < S) D[v * S + lane] = c >= 0 ? Dc[v * Sc + (uint32_t)c] : (v == sv ? 0u : kInf);
}

using MultiFn = void (*)(MArgs);

template <bool kFilter, int P>
static MultiFn pick_multi(int bs) {
  switch (bs) {
    case 256: return multi_kernel<256, kFilter, P>;
    case 1024: return multi_kernel<1024, kFilter, P>;
    default: return multi_kernel<512, kFilter, P>;
  }
}
template <bool kFilter>
static MultiFn pick_multi(int bs, uint32_t nsrc) {
  return nsrc <= 16 ? pick_multi<kFilter, 4>(bs) : nsrc <= 32 ? pick_multi<kFilter, 2>(bs) : pick_multi<kFilter, 1>(bs);
}

// Between the two kernels: the barrier and residency words start again.
__global__ void multi_switch(Ctrl *c) {
  ctrl_reset_barrier(c, threadIdx.x, blockDim.x);
  if (threadIdx.x == 0) c->checkin = 0;
}

struct MultiRun {
  double ms_kernel = 0;
  uint64_t rounds = 0, phases = 0, items = 0, heavy = 0, lane_items = 0, edges = 0, improved = 0;
  int grid = 0, bs = 0;
};

// Words of one sweep's bounds: whole wavefronts of a sweep, whole cache lines.
static uint64_t bound_words(uint32_t V) { return ((uint64_t)V + kWave - 1) / kWave * kWave; }

// Runs one vertex-major launch: S = nsrc <= 64 sources of `g` into D [V][S].
static int run_multi(Workspace *w, const lsg_graph *g, const uint32_t *srcs_host, uint32_t nsrc, const lsg_opts &o,
                     uint32_t *D, MultiRun *out) {
  int rc;
  int bs = o.block_size ? o.block_size : 512;
  if (bs != 256 && bs != 512 && bs != 1024) return fail(LSG_ERR_ARG, "block_size must be 256, 512 or 1024");
  // Default chunk size: short chunks spread a small graph's edges over the
  // wavefronts, long ones cost a large graph fewer units (ms at 64 / 256 / 512
  // edges: RMAT of 131072 vertices x 64 sources 2.2 / 2.6 / 2.8, 2^19 3.6 /
  // 3.6 / 4.8, 2^20 4.8 / 4.7 / 4.9, 2^21 8.2 / 7.9 / 7.7, 2^22 15.6 / 13.5 / 13.7;
  // 524288 x 33 at delta 32 14.7 / 16.9 / 23.1).
  uint32_t heavy_deg = o.heavy_deg > 0 ? (uint32_t)o.heavy_deg : g->nedges < (1u << 24) ? 64u : 256u;
  if (heavy_deg < kLongDeg) return fail(LSG_ERR_ARG, "heavy_deg must be >= %u for batched runs", kLongDeg);
  uint32_t V = g->nnodes;
  uint64_t hcap64 = 2ull * g->nedges / heavy_deg + 64;
  uint32_t hcap = (uint32_t)std::min<uint64_t>(hcap64, UINT32_MAX / 4);
  void *qbuf, *hbuf, *mbuf, *sbuf;
  if ((rc = ws_buffer(w, kBufQueues, 3ull * V * 4, &qbuf)) || (rc = ws_buffer(w, kBufHeavy, 2ull * hcap * 16, &hbuf)) ||
      (rc = ws_buffer(w, kBufMasks, (4ull * 8 + 4) * V + kSweeps * bound_words(V) * 4 + 16ull * w->cus * 8 + 512, &mbuf)) || (rc = ws_buffer(w, kBufSeeds, 2048 + kGroups * (sizeof(TicketGroup) + sizeof(MultiCounters)), &sbuf)))
    return rc;
  MArgs a;
  memset(&a, 0, sizeof a);
  a.row_start = g->row_start;
  a.edge_dst = g->edge_dst;
  a.edge_data = (const uint32_t *)g->edge_data;
  a.D = D;
  uint64_t *masks = (uint64_t *)mbuf;
  a.nmask[0] = masks;
  a.nmask[1] = masks + V;
  a.fmask[0] = masks + 2ull * V;
  a.fmask[1] = masks + 3ull * V;
  a.qstamp = (uint32_t *)(masks + 4ull * V);
  int32_t *const bounds = (int32_t *)(((uintptr_t)(a.qstamp + V) + 255) & ~(uintptr_t)255);
  for (int i = 0; i < kSweeps; ++i) a.bound[i] = bounds + i * bound_words(V);
  a.hubs = (uint64_t *)(bounds + kSweeps * bound_words(V));
  a.ninit = (uint32_t)std::min<uint64_t>(((uint64_t)V * nsrc + 255) / 256, 16ull * w->cus);
  for (int i = 0; i < 3; ++i) a.q[i] = (uint32_t *)qbuf + (size_t)i * V;
  a.hq[0] = (uint64_t *)hbuf;
  a.hq[1] = (uint64_t *)hbuf + 2ull * hcap;
  a.srcs = (const uint32_t *)sbuf;
  a.ctrl = w->ctrl;
  a.nnodes = V;
  a.S = nsrc;
  a.qcap = V;
  a.hcap = hcap;
  a.delta = (uint32_t)o.delta;
  a.heavy_deg = heavy_deg;
  a.spin_limit = spin_limit_ticks(w);
  a.residency_limit = residency_limit_ticks(w);
  a.nedges = g->nedges;
  a.fmin = (uint32_t *)((char *)sbuf + 512);
  a.thr = (uint32_t *)((char *)sbuf + 1024);
  a.flt = (Filter *)((char *)sbuf + 1280);
  static_assert(1280 + sizeof(Filter) <= 1792 && 1792 + sizeof(Pace) <= 2048, "the words before the tickets");
  if (!o.sched && !o.trace && o.far_mode == LSG_FAR_REFERENCE) a.pace = (Pace *)((char *)sbuf + 1792);
  a.tickets = (TicketGroup *)((char *)sbuf + 2048);
  a.tot = (MultiCounters *)(a.tickets + kGroups);
  if (o.sched) {
    a.sched = 1;
    a.mlp = sched_model_device(w->device, LSG_SCHED_BATCHED);
    if (!a.mlp)
      return fail(LSG_ERR_ARG, "learned scheduler requested but no batched-kernel model is loaded (lsg_sched_set_model)");
  }
  if (o.far_mode != LSG_FAR_REFERENCE && o.far_mode != LSG_FAR_SPLIT && o.far_mode != LSG_FAR_BUCKET)
    return fail(LSG_ERR_ARG, "bad far_mode %d", o.far_mode);
  a.far_mode = (uint32_t)o.far_mode;
  if (o.trace) {
    void *tbuf;
    size_t tbytes = (1u << 16) * sizeof(lsg_round_trace);
    if ((rc = ws_buffer(w, kBufTrace, tbytes + kMaxForced * kFeatRec * sizeof(float), &tbuf))) return rc;
    a.trace = (lsg_round_trace *)tbuf;
    a.trace_cap = 1u << 16;
    a.feat = (float *)((char *)tbuf + tbytes);
  }
  HIPCHK(hipMemcpyAsync(sbuf, srcs_host, nsrc * 4, hipMemcpyHostToDevice, w->stream));
  const MultiFn fn = pick_multi<false>(bs, nsrc), ffn = pick_multi<true>(bs, nsrc);
  int grid = 0, fgrid = 0;
  if ((rc = resident_grid(w, (const void *)fn, bs, &grid)) || (rc = resident_grid(w, (const void *)ffn, bs, &fgrid)))
    return rc;
  grid = std::min(grid, fgrid);
  if (o.grid_blocks > 0) grid = std::min(o.grid_blocks, grid);
  Ctrl hc;
  float ms = 0;
  for (int attempt = 0;; ++attempt) {
    auto enqueue = [&]() -> int {
      hipLaunchKernelGGL(multi_init, dim3(a.ninit), dim3(256), 0, w->stream, a);
      hipLaunchKernelGGL(multi_seed, dim3(1), dim3(64), 0, w->stream, a);
      hipLaunchKernelGGL(fn, dim3(grid), dim3(bs), 0, w->stream, a);
      hipLaunchKernelGGL(multi_switch, dim3(1), dim3(128), 0, w->stream, w->ctrl);
      hipLaunchKernelGGL(ffn, dim3(grid), dim3(bs), 0, w->stream, a);
      HIPCHK(hipGetLastError());
      return LSG_OK;
    };
    HIPCHK(hipEventRecord(w->ev0, w->stream));
    if (o.graph_launch) {
      std::vector<uint8_t> key;
      key_append(key, a);
      key_append(key, grid);
      key_append(key, bs);
      if ((rc = launch_captured(w, key, enqueue))) return rc;
    } else if ((rc = enqueue())) {
      return rc;
    }
    HIPCHK(hipEventRecord(w->ev1, w->stream));
    HIPCHK(hipMemcpyAsync(&hc, w->ctrl, kCtrlHostBytes, hipMemcpyDeviceToHost, w->stream));
    HIPCHK(hipStreamSynchronize(w->stream));
    HIPCHK(hipEventElapsedTime(&ms, w->ev0, w->ev1));
    if (hc.abort != kAbortResidency) break;
    if (attempt > 0 || hc.resident_seen == 0 || hc.resident_seen >= (uint32_t)grid)
      return fail(LSG_ERR_HIP, "persistent grid of %d x %d blocks is not co-resident (%u were)", grid, bs,
                  hc.resident_seen);
    grid = (int)hc.resident_seen;
    record_resident_grid(w, (const void *)fn, bs, grid);
    record_resident_grid(w, (const void *)ffn, bs, grid);
  }
  if (hc.abort == kAbortTimeout)
    return fail(LSG_ERR_TIMEOUT, "grid barrier timed out (grid %d x %d) at round %u; distances are incomplete",
                grid, bs, hc.s.round);
  if (hc.abort == kAbortCapacity) return fail(LSG_ERR_CAPACITY, "device queue capacity exceeded");
  MultiCounters tg[kGroups], ht = {0, 0, 0};
  HIPCHK(hipMemcpy(tg, a.tot, sizeof tg, hipMemcpyDeviceToHost));
  for (const MultiCounters &t : tg) {
    ht.lane_items += t.lane_items;
    ht.edges += t.edges;
    ht.improved += t.improved;
  }
  if (o.trace) {
    uint32_t n = (uint32_t)std::min<uint64_t>(hc.stat_rounds, a.trace_cap);
    w->last_trace.resize(n);
    if (n) HIPCHK(hipMemcpy(w->last_trace.data(), a.trace, n * sizeof(lsg_round_trace), hipMemcpyDeviceToHost));
    // one record per phase boundary: phase p -> p + 1 is record p
    uint32_t np = std::min<uint32_t>(hc.s.phase, kMaxForced);
    w->last_feat.resize((size_t)np * kFeatRec);
    if (np) HIPCHK(hipMemcpy(w->last_feat.data(), a.feat, w->last_feat.size() * sizeof(float), hipMemcpyDeviceToHost));
  }
  out->ms_kernel = ms;
  out->rounds = hc.stat_rounds;
  out->phases = hc.stat_phases;
  out->items = hc.stat_items;
  out->heavy = hc.stat_heavy;
  out->lane_items = ht.lane_items;
  out->edges = ht.edges;
  out->improved = ht.improved;
  out->grid = grid;
  out->bs = bs;
  return LSG_OK;
}

// Runs nsrc <= 64 sources into D [V][nsrc].  A source without out-edges
// reaches only itself, so it gets no lane: the launch runs the other sources
// into a compact matrix (rows of fewer words: on RMAT-22, where half the
// vertices have no out-edges, 64 random sources leave 33 lanes and rows of
// 132 instead of 256 bytes, 25.5 -> 23.6 ms), which is then expanded.
static int run_multi_live(Workspace *w, const lsg_graph *g, const uint32_t *srcs, uint32_t nsrc, const lsg_opts &o,
                          uint32_t *D, MultiRun *out) {
  int rc;
  void *lbuf;
  if ((rc = ws_buffer(w, kBufSeedList, 4 * 64 * 4, &lbuf))) return rc;
  uint32_t *d_srcs = (uint32_t *)lbuf, *d_deg = d_srcs + 64, *d_col = d_srcs + 128;
  uint32_t deg[64];
  HIPCHK(hipMemcpyAsync(d_srcs, srcs, nsrc * 4, hipMemcpyHostToDevice, w->stream));
  hipLaunchKernelGGL(source_degree_kernel, dim3(1), dim3(64), 0, w->stream, g->row_start, (const uint32_t *)d_srcs,
                     nsrc, d_deg);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(deg, d_deg, nsrc * 4, hipMemcpyDeviceToHost, w->stream));
  HIPCHK(hipStreamSynchronize(w->stream));
  uint32_t live[64];
  int32_t col[64];
  uint32_t nlive = 0;
  for (uint32_t i = 0; i < nsrc; ++i) {
    col[i] = deg[i] ? (int32_t)nlive : -1;
    if (deg[i]) live[nlive++] = srcs[i];
  }
  if (nlive == nsrc) return run_multi(w, g, srcs, nsrc, o, D, out);
  const uint32_t V = g->nnodes;
  void *cbuf = nullptr;
  if (nlive) {
    if ((rc = ws_buffer(w, kBufTranspose, (size_t)V * nlive * 4, &cbuf))) return rc;
    if ((rc = run_multi(w, g, live, nlive, o, (uint32_t *)cbuf, out))) return rc;
  } else {
    *out = MultiRun();
    w->last_trace.clear();
    w->last_feat.clear();
  }
  HIPCHK(hipMemcpyAsync(d_col, col, nsrc * 4, hipMemcpyHostToDevice, w->stream));
  const uint32_t blocks = (uint32_t)std::min<uint64_t>(((uint64_t)V * kWave + 255) / 256, 16ull * w->cus);
  hipLaunchKernelGGL(multi_expand, dim3(blocks), dim3(256), 0, w->stream, (const uint32_t *)cbuf, nlive,
                     (const int32_t *)d_col, (const uint32_t *)d_srcs, nsrc, V, D);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(w->stream));
  return LSG_OK;
}

static int check_multi_args(const lsg_graph *g, const uint32_t *srcs, uint32_t nsrc, const lsg_opts &o) {
  if (!g || !g->device_graph) return fail(LSG_ERR_ARG, "expected a device graph (copy_to_gpu first)");
  if (!srcs || nsrc == 0) return fail(LSG_ERR_ARG, "no sources");
  if (o.delta <= 0) return fail(LSG_ERR_ARG, "delta must be > 0 (got %d)", o.delta);
  for (uint32_t i = 0; i < nsrc; ++i)
    if (srcs[i] >= g->nnodes) return fail(LSG_ERR_ARG, "source %u = %u out of range [0, %u)", i, srcs[i], g->nnodes);
  return LSG_OK;
}

static void fill_stats(lsg_batch_stats *st, const MultiRun &r, int launches) {
  st->ms_kernel += r.ms_kernel;
  st->rounds += r.rounds;
  st->phases += r.phases;
  st->items += r.items;
  st->heavy_chunks += r.heavy;
  st->lane_items += r.lane_items;
  st->edges_expanded += r.edges;
  st->improved_rows += r.improved;
  st->grid_blocks = r.grid;
  st->block_size = r.bs;
  st->launches = launches;
}

}  // namespace lsg

using namespace lsg;

extern "C" {

int lsg_sssp_multi(const lsg_graph *g, const uint32_t *srcs, uint32_t nsrc, const lsg_opts *opts, int32_t *dist_vs,
                   lsg_batch_stats *stats) {
  clear_error();
  auto t0 = std::chrono::steady_clock::now();
  lsg_opts o;
  if (opts) o = *opts;
  else lsg_opts_default(&o);
  int rc = check_multi_args(g, srcs, nsrc, o);
  if (rc) return rc;
  if (nsrc > 64) return fail(LSG_ERR_ARG, "lsg_sssp_multi takes at most 64 sources (got %u)", nsrc);
  if (!dist_vs) return fail(LSG_ERR_ARG, "NULL distance matrix");
  Workspace *w;
  if ((rc = get_workspace(g->device, &w))) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  HIPCHK(hipSetDevice(w->device));
  MultiRun r;
  if ((rc = run_multi_live(w, g, srcs, nsrc, o, (uint32_t *)dist_vs, &r))) return rc;
  if (stats) {
    memset(stats, 0, sizeof *stats);
    fill_stats(stats, r, 1);
    stats->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  return LSG_OK;
}

int lsg_last_features(int device, float *out, uint32_t cap_phases, uint32_t *nphases) {
  Workspace *w;
  int rc = get_workspace(device, &w);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  uint32_t np = (uint32_t)(w->last_feat.size() / kFeatRec);
  uint32_t m = std::min(np, cap_phases);
  if (out && m) memcpy(out, w->last_feat.data(), (size_t)m * kFeatRec * sizeof(float));
  if (nphases) *nphases = np;
  return LSG_OK;
}

int lsg_sssp_batch(const lsg_graph *g, const uint32_t *srcs, uint32_t nsrc, const lsg_opts *opts,
                   int32_t *const *dist_out, lsg_batch_stats *stats) {
  clear_error();
  auto t0 = std::chrono::steady_clock::now();
  lsg_opts o;
  if (opts) o = *opts;
  else lsg_opts_default(&o);
  int rc = check_multi_args(g, srcs, nsrc, o);
  if (rc) return rc;
  if (!dist_out) return fail(LSG_ERR_ARG, "NULL output array list");
  for (uint32_t i = 0; i < nsrc; ++i)
    if (!dist_out[i]) return fail(LSG_ERR_ARG, "output %u is NULL", i);
  Workspace *w;
  if ((rc = get_workspace(g->device, &w))) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  HIPCHK(hipSetDevice(w->device));
  uint32_t S = std::min<uint32_t>(nsrc, 64);
  void *dbuf, *pbuf;
  if ((rc = ws_buffer(w, kBufUnion, (size_t)g->nnodes * S * 4 + 64 * sizeof(void *), &dbuf))) return rc;
  pbuf = (char *)dbuf + (size_t)g->nnodes * S * 4;
  if (stats) memset(stats, 0, sizeof *stats);
  int launches = 0;
  for (uint32_t base = 0; base < nsrc; base += 64) {
    uint32_t n = std::min<uint32_t>(64, nsrc - base);
    MultiRun r;
    if ((rc = run_multi_live(w, g, srcs + base, n, o, (uint32_t *)dbuf, &r))) return rc;
    ++launches;
    HIPCHK(hipMemcpyAsync(pbuf, dist_out + base, n * sizeof(void *), hipMemcpyHostToDevice, w->stream));
    uint32_t blocks = (uint32_t)std::min<uint64_t>(((uint64_t)g->nnodes * n + 255) / 256, 16ull * w->cus);
    hipLaunchKernelGGL(multi_scatter, dim3(blocks), dim3(256), 0, w->stream, (const uint32_t *)dbuf, n, g->nnodes,
                       (int32_t *const *)pbuf);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(w->stream));
    if (stats) fill_stats(stats, r, launches);
  }
  if (stats)
    stats->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return LSG_OK;
}

}  // extern "C"
