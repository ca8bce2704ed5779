// Single-source SSSP and BFS in one persistent launch, by wavefronts.
//
// The rounds, piles and phases are the reference's (apps/sssp/kernel.cu:355-391
// near/far piles, curdelta += DELTA per phase -- here a multiple of it, see
// WavePace -- the whole far pile becoming the next phase;
// apps/bfs/kernel.cu:312-334 levels), as in persistent_kernel
// (sssp_dev.h), which remains for what this kernel does not take: split and
// bucket far piles, degree-binned expansion, the learned scheduler, round
// traces, the -l sweep and the no-allocation entry point.
//
// What bounds a traversal differs: on a skewed graph (RMAT-20, ~20 rounds) the
// random distance loads of some 65 M edge relaxations, on a road network or a
// grid (hundreds of rounds of a few hundred to a few thousand vertices) the
// chain of dependent round trips of a round.
//
//   - Work units belong to wavefronts: up to 64 in-queue items whose edges are
//     flattened over the lanes, or one chunk of a heavy vertex.  No block
//     barrier inside a round, and a wavefront goes on to its next unit while
//     others wait for memory.  (Tiles of a block waited for their slowest
//     wavefront at every ticket.)
//   - Pushes and heavy items are staged per wavefront in LDS and placed with
//     one atomic per pile and block at the end of the round.
//   - Only blocks that had a unit arrive at the barrier (36 units: 9 blocks, one
//     counter), and its message is the round: the last block to arrive
//     publishes the next round's counts and roles as words that carry the
//     generation, so that the waiting blocks read everything with the poll that
//     sees it, and nothing has to be ordered before it.  Tails, tickets and
//     arrival counts are used in turn by generation and cleared two rounds
//     ahead.  A round of 600 low-degree items: 9.2 -> 7.5 us with the arrival
//     of all 256 blocks and the look at d[v] before the atomicMin taken out.
//   - What was expanded already is not expanded again: items of the far pile
//     that came below the last threshold meanwhile were near items then
//     (RMAT-20: most of 505,060, 145 -> 87 us), and chunks of a vertex that was
//     lowered since it was popped are left to its next pop.
//   - Small rounds (at most local_max items, no heavy vertex) are run by the
//     last block alone, with entries in LDS as in the one-workgroup kernel
//     (block.hip): two or three round trips and two block barriers a round
//     while the others stay parked.  The looks at d[v] and at stamps whose
//     older value only costs work are at workgroup scope (64^2 grid 0.85 ->
//     0.79 ms).  The block leaves
//     this mode when the round it would run next is too large, and hands the
//     vertices over through the near queue; it is entered at half that size (a
//     pile counts a vertex as often as it is pushed: 256^2 grid 3.60 -> 3.37 ms,
//     512^2 8.2 -> 7.8).  (Limits of 128 / 256 / 384 / 512
//     items: 64^2 grid SSSP 0.62 / 0.53 / 0.52 / 0.49 ms, 256^2 3.7 / 3.4 / 3.5
//     / 3.6, 512^2 BFS 6.0 / 5.2 / 4.9 / 4.8, road-like 1023 x 777 BFS 0.86 /
//     0.85 / 0.84 / 0.84.)
//
// Ms in persistent_kernel -> here: SSSP RMAT-18 0.72 -> 0.45, RMAT-20 1.60 ->
// 0.87, RMAT-22 5.1 -> 2.07, grid 256^2 8.2 -> 2.57, road-like 2048^2 4.4 -> 2.04;
// BFS RMAT-18 0.205 -> 0.143, RMAT-20 0.447 -> 0.278, road-like 2048^2 1.99 ->
// 1.11.

#include <hip/hip_runtime.h>

#include "wave_dev.h"

namespace lsg {

// The entries of a pile in LDS, of a round that one block runs alone (its pushes
// are not deduplicated in there).
constexpr uint32_t kLocalCap = 1024;
constexpr uint32_t kWavePush = 256;   // staged items per wavefront and pile
constexpr uint32_t kWaveHeavy = 64;   // staged heavy items per wavefront, one a lane
constexpr uint32_t kHopEdges = 256;  // see wave_items
constexpr uint32_t kMaxStep = 1u << 16;
struct WaveHeavy {
  uint32_t u, d, first, deg;
};

// Pace of the near/far threshold on graphs of low degree (low_degree).  There nearly every round is bound by its fixed
// cost, so a wider phase, with its fewer and larger rounds, is faster until
// the vertices that are expanded more than once cost more than the rounds
// saved; how wide depends on the graph, the weights and where the frontier is
// (best multiple of the call's delta: 64^2 grid at 32: 64, 256^2: 16, road-like
// 1000^2 at 10000: 16, 2048^2: 6).  So the threshold moves by `step` deltas,
// and step is climbed: it is doubled while the threshold then moves further per
// us of modelled round cost, or while rounds are nearly empty; else one step
// back, and two phases later the next trial.  Distances do not depend on it.
// Ms with step 1 -> here: grid 64^2 0.80 -> 0.50, 256^2 5.7 -> 3.8, 1000^2 30 ->
// 20, road-like 1000^2 2.67 -> 1.90, 2048^2 3.83 -> 2.88, 2048^2 at delta 2000
// 6.9 -> 3.0.  On RMAT graphs of 8 and more edges a vertex, whose rounds are
// few and large, it gains nothing and loses up to 17 % from random sources.
struct WavePace {
  uint32_t step;    // deltas that the threshold moves by
  uint32_t hold;    // phases until the next trial; 0: this phase is one
  float best;       // deltas per us before the trial
  float cost;       // of the phase so far, us: fitted to both kinds of rounds
  uint32_t rounds;  // of the phase so far
  __device__ void round(uint32_t items, bool local) {
    cost += local ? 3.0f + (float)items * (1.0f / 80) : 6.0f + (float)items * (1.0f / 6000);
    rounds += 1;
  }
  // The step to the threshold of the phase after `phase`.
  __device__ uint32_t next(uint32_t phase, uint32_t flags, bool forest) {
    // (see WaveGrowth)
    if (flags & kWaveSplit || (flags & kWaveWide && forest)) {
      cost = 0;
      rounds = 0;
      step = 1;
      return flags & kWaveSplit ? 1u : kMaxStep;
    }
    const float rate = (float)step / cost;
    const bool empty = cost < 4.0f * (float)rounds;
    cost = 0;
    rounds = 0;
    if (hold == 0 || empty) {
      hold = 0;
      if (rate > 1.02f * best || empty) {
        if (phase > 0) best = rate;  // (phase 0 is the source alone)
        step = min(step * 2, kMaxStep);
      } else {
        step = max(step / 2, 1u);
        hold = 2;
      }
    } else if (--hold == 0) {
      best = rate;
      step = min(step * 2, kMaxStep);
    }
    return step;
  }
};

// Growth of the rounds on graphs of low degree.  Few edges a vertex do not make a
// graph deep: on a random graph or an RMAT graph of 4 edges a vertex the frontier
// grows by factors, the traversal is a few dozen rounds, and what pays on a grid
// does not.  From a round of more than kWideItems items that is more than three times
// the largest so far (a grid's frontier, which grows by a ring a round, never is;
// at twice road-like 2048^2 took 2.55 ms, with it or without the rule 2.03)
// the next kWideRounds rounds -- all that such a graph has -- are wide:
//   - wavefronts go on with what they pushed only in rounds of more than kWideItems
//     and at most kWideHops items: larger ones are bound by work, and what is
//     expanded at a distance that falls later is work done twice; in smaller ones
//     few wavefronts would go on with what all can take;
//   - units are of one item where there are wavefronts enough: a vertex may have many
//     edges;
//   - where vertices of heavy_deg edges are found too (kWaveSplit), the rounds are
//     those of skewed graphs: no going on, vertices of kWaveSplitDeg edges split
//     when they are pushed, the threshold moved by the call's delta;
//   - on graphs of at most 2 edges a vertex (forests: one way to each vertex) the
//     next phase is all that is left.
// A chunk counts as heavy_deg items: it may push so many.  A round that one block
// leaves to the grid because of a vertex's edges (kLocalDeg) is wide by itself.
// Kernel us without / with, delta 10000 where the delta is not said: 5 edges a vertex
// RMAT-like, 32,000 vertices 347 / 207, 100,000 455 / 255, 10^6 1040 / 700, delta 32
// 916 / 622; uniform out-degree 4, 10^6 1028 / 853, BFS 451 / 311, 4 x 10^6 2734 /
// 2381, BFS 1250 / 897; random trees of 10^5 delta 32 388 / 260; 4 x 10^6 leaves of
// 1000 hubs, delta 32 1576 / 1158.  Grids and road-like graphs alike.
constexpr uint32_t kWideItems = 512, kWideRounds = 48;
template <Algo A>
constexpr uint32_t kWideHops = A == Algo::SSSP ? 16384 : 8192;
constexpr uint32_t kWideChunks = 4;  // chunks of a round that say that the graph is skewed
struct WaveGrowth {
  uint32_t peak;   // items of the largest round so far
  uint32_t until;  // rounds before this one are wide
  // The flags of round `round`, of n items, after a round with flags `before`;
  // `heavy`: it took vertices apart.
  __device__ uint32_t flags(uint32_t round, uint32_t n, bool heavy, uint32_t before) {
    if (n > kWideItems && n / 3 > peak) until = round + kWideRounds;
    peak = max(peak, n);
    return round >= until ? 0u : heavy ? kWaveWide | kWaveSplit : kWaveWide | (before & kWaveSplit);
  }
};

template <int BS>
struct WaveShared {
  static constexpr int NW = BS / kWave;
  uint32_t push[NW][2][kWavePush];  // near, far
  WaveHeavy heavy[NW][kWaveHeavy];
  uint32_t count[NW][3];            // end of a round: near, far, heavy chunks
  uint32_t base[3];
  WaveRound r;
  uint32_t gen;
  WavePace pace;
  WaveGrowth growth;
  // rounds of one block
  Entry pile[2][kLocalCap];
  uint32_t pile_n[2];
  uint32_t far_n;    // the far queue's length
  uint32_t spill_n;  // vertices handed to the near queue
  uint32_t stop;     // a vertex of too many edges for this mode was pushed
  unsigned long long items;
};

// A wavefront's view of the round.
struct WaveLane {
  uint32_t near_stamp, far_stamp;  // this round's and phase's stamps
  uint32_t thr;                    // a candidate is near iff it is at most this
  int64_t cut;                     // items at most this far are skipped
  bool direct;
  uint32_t *nq, *fq, *ntail, *ftail;
  WaveChunk *hq;
  uint32_t *htail;
  uint32_t *pbuf[2];
  WaveHeavy *hbuf;
  uint32_t n[2], hn;  // staged: items per pile, heavy items (wave-uniform)
  uint32_t settled;   // see wave_settle
  uint32_t hopped;    // vertices popped in hops, per lane
  uint32_t hops;      // this round's WaveArgs::hops
  bool split;         // vertices of kWaveSplitDeg edges are taken apart when they are pushed
};

__device__ __forceinline__ uint32_t *wave_queue(const WaveArgs &a, uint32_t i) {
  uint32_t *const q0 = a.q[0], *const q1 = a.q[1], *const q2 = a.q[2];
  return i == 0 ? q0 : i == 1 ? q1 : q2;
}

// ---- pushes -------------------------------------------------------------------

// Writes pile `which`'s staged items to its queue from `base` on.
__device__ __forceinline__ void wave_store(const WaveArgs &a, WaveLane &w, int which, uint32_t base) {
  uint32_t *const q = which ? w.fq : w.nq;
  for (uint32_t i = lane_id(); i < w.n[which]; i += kWave) {
    const uint32_t pos = base + i;
    if (pos < a.qcap) st_coh(q + pos, w.pbuf[which][i]);
    else st_coh(&a.ctrl->abort, kAbortCapacity);
  }
  w.n[which] = 0;
  if (which == 0) w.settled = 0;
}

// Writes the staged heavy items' chunks, counted in `end`, from slot `base` on.
__device__ __forceinline__ void wave_store_heavy(const WaveArgs &a, WaveLane &w, uint32_t end, uint32_t base) {
  chunk_each(end, [&](uint32_t f, uint32_t item, uint32_t k) {
    const uint32_t pos = base + f, skip = k * a.heavy_deg;
    const WaveHeavy h = w.hbuf[item];
    if (pos < a.hcap) {
      uint64_t *const p = reinterpret_cast<uint64_t *>(w.hq + pos);
      st_coh64(p, (uint64_t)h.d << 32 | h.u);
      st_coh64(p + 1, (uint64_t)min(h.deg - skip, a.heavy_deg) << 32 | (h.first + skip));
    } else {
      st_coh(&a.ctrl->abort, kAbortCapacity);
    }
  });
  w.hn = 0;
}
__device__ __forceinline__ uint32_t wave_heavy_ends(const WaveArgs &a, const WaveLane &w) {
  return chunk_ends(w.hn, lane_id() < w.hn ? w.hbuf[lane_id()].deg : 0u, a.heavy_deg);
}

// Queues the vertices u of the lanes with `heavy` (at distance d; edges first
// to first + deg) as chunks of heavy_deg edges, expanded in the next round.
__device__ __forceinline__ void wave_heavy(const WaveArgs &a, WaveLane &w, bool heavy, uint32_t u, uint32_t d,
                                           uint32_t first, uint32_t deg) {
  const uint64_t m = __ballot(heavy);
  if (m == 0) return;
  const uint32_t c = (uint32_t)__builtin_popcountll(m);
  if (w.hn + c > kWaveHeavy) {
    const uint32_t end = wave_heavy_ends(a, w);
    uint32_t base = 0;
    if (lane_id() == 0) base = atomic_add(w.htail, readlane(end, kWave - 1));
    wave_store_heavy(a, w, end, readlane(base, 0));
  }
  if (heavy) w.hbuf[w.hn + lanes_below(m)] = WaveHeavy{u, d, first, deg};
  w.hn += c;
}

// The near items staged since the last call: those of kWaveSplitDeg edges and more
// become chunks of the next round, read with the distance of that time; the
// others close up.
__device__ __forceinline__ void wave_settle(const WaveArgs &a, WaveLane &w) {
  uint32_t out = w.settled;
  for (uint32_t i0 = w.settled; i0 < w.n[0]; i0 += kWave) {
    const bool valid = i0 + lane_id() < w.n[0];
    const uint32_t v = valid ? w.pbuf[0][i0 + lane_id()] : 0u;
    const uint64_t rb = ld_pair(a.row_start + v);
    const uint32_t rs = (uint32_t)rb, deg = (uint32_t)(rb >> 32) - rs;
    const bool split = valid && deg >= kWaveSplitDeg;
    wave_heavy(a, w, split, v, kInf, rs, deg);
    const uint64_t m = __ballot(valid && !split);
    if (valid && !split) w.pbuf[0][out + lanes_below(m)] = v;
    out += (uint32_t)__builtin_popcountll(m);
  }
  w.n[0] = w.settled = out;
}

// Pushes `item` from every lane with `pred` (whole wavefront).
__device__ __forceinline__ void wave_stage(const WaveArgs &a, WaveLane &w, int which, bool pred, uint32_t item) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const uint32_t c = (uint32_t)__builtin_popcountll(m);
  if (w.n[which] + c > kWavePush) {
    if (which == 0 && w.split) wave_settle(a, w);
    uint32_t base = 0;
    if (lane_id() == 0 && w.n[which]) base = atomic_add(which ? w.ftail : w.ntail, w.n[which]);
    wave_store(a, w, which, readlane(base, 0));
  }
  if (pred) w.pbuf[which][w.n[which] + lanes_below(m)] = item;
  w.n[which] += c;
}

// ---- relaxation ----------------------------------------------------------------

// Relaxes edges e[k], k < U, leaving vertices at distance du[k], of the lanes
// with act[k] (e[k] names some edge in every lane): the tests, atomics and
// pushes of relax_edges in sssp_dev.h.
template <Algo A, int U>
__device__ __forceinline__ void wave_relax(const WaveArgs &a, WaveLane &w, const uint32_t (&e)[U],
                                           const uint32_t (&du)[U], const bool (&act)[U], bool direct) {
  uint32_t v[U], nd[U], dv[U], old[U], seen[U], got[U];
  bool near[U], cand[U], any = false;
#pragma unroll
  for (int k = 0; k < U; ++k) {
    v[k] = glb(a.edge_dst)[e[k]];
    nd[k] = A == Algo::SSSP ? du[k] + glb(a.edge_data)[e[k]] : du[k] + 1u;
  }
  // through the caches: a stale distance is only ever larger
#pragma unroll
  for (int k = 0; k < U; ++k) dv[k] = kInf;
  if (!direct) {
#pragma unroll
    for (int k = 0; k < U; ++k) dv[k] = glb(a.dist)[v[k]];
  }
#pragma unroll
  for (int k = 0; k < U; ++k) {
    cand[k] = act[k] && nd[k] < dv[k];
    any |= cand[k];
  }
  if (__ballot(any) == 0) return;
  uint32_t *const ns = a.near_stamp, *const fs = a.far_stamp;
#pragma unroll
  for (int k = 0; k < U; ++k) {
    near[k] = A == Algo::BFS || nd[k] <= w.thr;
    seen[k] = glb(near[k] ? ns : fs)[cand[k] ? v[k] : 0u];
    old[k] = cand[k] ? atomic_min(a.dist + v[k], nd[k]) : 0u;
  }
  // results are taken only here (left to itself the compiler tests each
  // result inside its atomic's branch, waiting for the whole memory queue)
#pragma unroll
  for (int k = 0; k < U; ++k) asm volatile("" : "+v"(old[k]));
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const uint32_t stamp = near[k] ? w.near_stamp : w.far_stamp;
    const bool want = nd[k] < old[k] && (seen[k] != stamp || (w.hops && near[k]));
    got[k] = want ? atomic_exch((near[k] ? ns : fs) + v[k], stamp) : stamp;
  }
#pragma unroll
  for (int k = 0; k < U; ++k) asm volatile("" : "+v"(got[k]));
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const bool push = nd[k] < old[k] && got[k] != (near[k] ? w.near_stamp : w.far_stamp);
    wave_stage(a, w, 0, push && near[k], v[k]);
    if (A == Algo::SSSP) wave_stage(a, w, 1, push && !near[k], v[k]);
  }
}

constexpr int kWaveU = 4;

// The vertices u of the lanes below n, with `deg` edges from rs on (0: none to
// expand): heavy ones are queued as chunks, the others' edges flattened over the
// wavefront.  Returns their number.
template <Algo A>
__device__ __forceinline__ uint32_t wave_vertices(const WaveArgs &a, WaveLane &w, int64_t cut, uint32_t u, uint32_t n,
                                                  uint32_t rs, uint32_t deg) {
  const uint32_t lane = lane_id();
  const uint32_t du = lane < n ? ld_coh(a.dist + u) : kInf;
  if (du == kInf || (int64_t)du <= cut) deg = 0;
  const bool heavy = deg >= a.heavy_deg;
  wave_heavy(a, w, heavy, u, du, rs, deg);
  if (heavy) deg = 0;
  uint32_t end = deg;  // inclusive prefix over the lanes
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = __shfl_up(end, d);
    if (lane >= (uint32_t)d) end += y;
  }
  const uint32_t total = readlane(end, kWave - 1);
  const uint32_t base = rs - (end - deg);
  const bool direct = w.direct && total <= 2 * kWave;
  for (uint32_t b0 = 0; b0 < total; b0 += kWaveU * kWave) {
    uint32_t e[kWaveU], d0[kWaveU];
    bool act[kWaveU];
#pragma unroll
    for (int k = 0; k < kWaveU; ++k) {
      const uint32_t f = min(b0 + k * kWave + lane, total - 1);
      act[k] = b0 + k * kWave + lane < total;
      uint32_t pos = 0;  // items that end at or before f
#pragma unroll
      for (uint32_t d = kWave / 2; d >= 1; d >>= 1)
        if ((uint32_t)__shfl(end, pos + d - 1) <= f) pos += d;
      e[k] = (uint32_t)__shfl(base, pos) + f;
      d0[k] = (uint32_t)__shfl(du, pos);
    }
    wave_relax<A, kWaveU>(a, w, e, d0, act, direct);
  }
  return total;
}

// A unit of n in-queue items, and then, w.hops times, what the wavefront itself has
// just pushed near (64 at most), without waiting for the round's end.  A vertex
// taken so loses its stamp before its distance is read, and pushes go by the
// exchange alone (a stamp read ahead of it may be gone): whoever lowers the vertex
// later queues it again.  A heavy vertex is not taken: the chunk queue holds one
// set of chunks per vertex and round (in-queue items are distinct: at most 2 E /
// heavy_deg chunks), and a hub that many light vertices lower within a round would
// be taken apart each time (1000 vertices of 257 edges with a leaf an edge, 16
// blocks: 6440 chunks in a round, room for 4079).  It gets its stamp again and
// stays among the pushes, unless it was pushed by another wavefront meanwhile.
// Distances and levels are lowered until nothing changes,
// so the order is free; a hop costs three round trips, a round ten.  Not for units
// of more than kHopEdges edges, where what the other wavefronts would have lowered
// meanwhile is expanded twice: skewed graphs (RMAT of 2^18 vertices and 4 edges
// each 0.56 ms, 1.04 with 4 hops and no limit, 0.57 with it).  Ms at 0 / 1 / 2 / 4 /
// 6 hops: SSSP road-like 400^2 1.18 / 0.96 / 0.83 / 0.78 / 0.77, 1000^2 1.78 / 1.40 /
// 1.28 / 1.18 / 1.18, 2048^2 2.81 / 2.32 / 2.19 / 2.18 / 2.19, grid 256^2 3.46 / 2.93 /
// 2.73 / 2.58 / 2.54, 512^2 8.1 / 6.7 / 6.0 / 5.6 / 5.3; BFS road-like 1023 x 777 0.87 /
// 0.68 / 0.61 / 0.55 / 0.54, 2048^2 1.50 / 1.25 / 1.17 / 1.13 / 1.17.
template <Algo A>
__device__ __forceinline__ void wave_items(const WaveArgs &a, WaveLane &w, const uint32_t *in, uint32_t n) {
  const uint32_t lane = lane_id();
  uint32_t kept = w.n[0], u = lane < n ? ld_coh(in + lane) : 0u;
  uint64_t rb = ld_pair(a.row_start + u);
  int64_t cut = w.cut;
  for (uint32_t h = 0;; ++h) {
    const uint32_t rs = (uint32_t)rb, deg = lane < n ? (uint32_t)(rb >> 32) - rs : 0u;
    const uint32_t total = wave_vertices<A>(a, w, cut, u, n, rs, deg);
    if (h == w.hops || total > kHopEdges) break;
    if (w.n[0] < kept) kept = 0;  // written out meanwhile
    n = min((uint32_t)kWave, w.n[0] - kept);
    if (n == 0) break;
    w.n[0] = kept = w.n[0] - n;
    u = lane < n ? w.pbuf[0][kept + lane] : 0u;
    rb = ld_pair(a.row_start + u);
    if (lane < n) (void)atomic_exch(a.near_stamp + u, 0u);
    order_release();  // the stamp is gone before the distance is read
    const bool heavy = lane < n && (uint32_t)(rb >> 32) - (uint32_t)rb >= a.heavy_deg;
    w.hopped += lane < n && !heavy ? 1u : 0u;
    if (__ballot(heavy)) {
      const bool back = heavy && atomic_exch(a.near_stamp + u, w.near_stamp) != w.near_stamp;
      const uint64_t m = __ballot(back);
      if (back) w.pbuf[0][kept + lanes_below(m)] = u;
      w.n[0] = kept = kept + (uint32_t)__builtin_popcountll(m);
      if (heavy) rb = 0;
    }
    cut = -1;
  }
}

// One chunk of a heavy vertex.  Where the vertex has come nearer since it was
// popped it is queued again, and the chunk is left to that.
template <Algo A>
__device__ __forceinline__ void wave_chunk(const WaveArgs &a, WaveLane &w, const WaveChunk *ent) {
  const uint32_t lane = lane_id();
  const uint64_t *const p = reinterpret_cast<const uint64_t *>(ent);
  const uint64_t x = ld_coh64(p), y = ld_coh64(p + 1);
  const uint32_t u = __builtin_amdgcn_readfirstlane((uint32_t)x), d = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  const uint32_t rs = __builtin_amdgcn_readfirstlane((uint32_t)y), n = __builtin_amdgcn_readfirstlane((uint32_t)(y >> 32));
  if (u >= a.nnodes || n == 0 || (uint64_t)rs + n > a.nedges) return;
  const uint32_t du = ld_coh(a.dist + u);
  if (d != kInf && du < d) return;
  for (uint32_t b0 = 0; b0 < n; b0 += kWaveU * kWave) {
    uint32_t e[kWaveU], d0[kWaveU];
    bool act[kWaveU];
#pragma unroll
    for (int k = 0; k < kWaveU; ++k) {
      const uint32_t f = b0 + k * kWave + lane;
      act[k] = f < n;
      e[k] = rs + min(f, n - 1);
      d0[k] = du;
    }
    wave_relax<A, kWaveU>(a, w, e, d0, act, false);
  }
}

// ---- rounds of one block --------------------------------------------------------

// The relaxation of such a round: improved neighbours are appended to the next
// pile in LDS with the row bounds loaded beside the atomicMin, or, beyond the
// threshold, to the far queue.
template <Algo A, int BS>
struct LocalRelax {
  const WaveArgs &a;
  WaveShared<BS> &sh;
  uint32_t nxt, thr, near_stamp, far_stamp;
  uint32_t *nq, *fq;
  __device__ __forceinline__ bool stopped() const { return false; }
  __device__ __forceinline__ void operator()(const KArgs &, const uint32_t (&v)[kInFlight],
                                             const uint32_t (&nd)[kInFlight], const bool (&act)[kInFlight]) const {
    uint32_t old[kInFlight], seen[kInFlight], got[kInFlight];
    uint64_t rb[kInFlight];
    bool near[kInFlight];
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      near[k] = A == Algo::BFS || nd[k] <= thr;
      old[k] = act[k] ? atomic_min(a.dist + v[k], nd[k]) : 0u;
      rb[k] = ld_pair(a.row_start + v[k]);
      seen[k] = A == Algo::SSSP ? ld_wg(a.far_stamp + (act[k] && !near[k] ? v[k] : 0u)) : 0u;
    }
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) asm volatile("" : "+v"(old[k]));
    if (A == Algo::SSSP) {
#pragma unroll
      for (int k = 0; k < kInFlight; ++k) {
        const bool want = act[k] && nd[k] < old[k] && !near[k] && seen[k] != far_stamp;
        got[k] = want ? atomic_exch(a.far_stamp + v[k], far_stamp) : far_stamp;
      }
    }
    // near: one reservation per wavefront
    uint64_t m[kInFlight];
    uint32_t t = 0;
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      m[k] = __ballot(act[k] && nd[k] < old[k] && near[k]);
      t += (uint32_t)__builtin_popcountll(m[k]);
    }
    if (t) {
      uint32_t pos = 0;
      if (lane_id() == 0) pos = atomicAdd(&sh.pile_n[nxt], t);
      pos = readlane(pos, 0);
#pragma unroll
      for (int k = 0; k < kInFlight; ++k) {
        if ((m[k] >> lane_id()) & 1) {
          const uint32_t p = pos + lanes_below(m[k]);
          const uint32_t rs = (uint32_t)rb[k], re = (uint32_t)(rb[k] >> 32);
          if (re - rs >= kLocalDeg) sh.stop = 1;
          if (p < kLocalCap) sh.pile[nxt][p] = Entry{v[k], nd[k], rs, re};
          else spill(v[k]);
        }
        pos += (uint32_t)__builtin_popcountll(m[k]);
      }
    }
    if (A == Algo::SSSP) {
#pragma unroll
      for (int k = 0; k < kInFlight; ++k) asm volatile("" : "+v"(got[k]));
      t = 0;
#pragma unroll
      for (int k = 0; k < kInFlight; ++k) {
        m[k] = __ballot(act[k] && nd[k] < old[k] && !near[k] && got[k] != far_stamp);
        t += (uint32_t)__builtin_popcountll(m[k]);
      }
      if (t) {
        uint32_t pos = 0;
        if (lane_id() == 0) pos = atomicAdd(&sh.far_n, t);
        pos = readlane(pos, 0);
#pragma unroll
        for (int k = 0; k < kInFlight; ++k) {
          if ((m[k] >> lane_id()) & 1) put(fq, pos + lanes_below(m[k]), v[k]);
          pos += (uint32_t)__builtin_popcountll(m[k]);
        }
      }
    }
  }
  __device__ __forceinline__ void put(uint32_t *q, uint32_t pos, uint32_t v) const {
    if (pos < a.qcap) st_coh(q + pos, v);
    else st_coh(&a.ctrl->abort, kAbortCapacity);
  }
  // A vertex that this mode hands on: once to the near queue.
  __device__ __forceinline__ void spill(uint32_t v) const {
    if (atomic_exch(a.near_stamp + v, near_stamp) != near_stamp) put(nq, atomicAdd(&sh.spill_n, 1u), v);
  }
};

__device__ __forceinline__ uint32_t wave_threshold(const WaveArgs &a, int64_t cd0, uint32_t steps) {
  const int64_t cd = cd0 + (int64_t)steps * a.delta;
  return (uint32_t)min(cd, (int64_t)0xFFFFFFFFll);
}

// Called by every thread of the block that leads, with the next round in sh.r
// (at most a.local_max items, no heavy chunks): runs it and the rounds that
// follow for as long as they are small, and leaves in sh.r the round that the
// whole grid runs next.  Every wavefront's memory operations are complete on
// return.
template <Algo A, int BS>
__device__ __forceinline__ void wave_local(const WaveArgs &a, WaveShared<BS> &sh, int64_t cd0) {
  WaveRound r = sh.r;
  WavePace pace = sh.pace;
  WaveGrowth growth = sh.growth;
  const uint32_t far_in = A == Algo::SSSP ? ld_coh(&a.wc->far_tail[r.far_q()].n) : 0u;
  if (threadIdx.x == 0) {
    sh.far_n = far_in;
    sh.stop = 0;
    sh.items = 0;
  }
  uint32_t rounds = 0, cur = 0, n = r.items;
  bool load = true;  // the round's items are still in queue in_q
  unsigned long long popped = 0;
  const auto grow = [&]() {
    const uint32_t f = growth.flags(r.round, n, false, r.flags);
    r.flags = (r.flags & ~(kWaveWide | kWaveSplit)) | f;
  };
  for (;;) {
    if (load) {
      const uint32_t *const in = wave_queue(a, r.in_q());
      const int64_t cut = r.flags & kWaveCut ? (int64_t)wave_threshold(a, cd0, r.cut) : -1;
      bool big = false;
      for (uint32_t i = threadIdx.x; i < n; i += BS) {
        const uint32_t v = ld_coh(in + i);
        const uint32_t d = ld_coh(a.dist + v);
        const uint64_t rb = ld_pair(a.row_start + v);
        const uint32_t rs = (uint32_t)rb, re = (int64_t)d <= cut ? rs : (uint32_t)(rb >> 32);
        sh.pile[cur][i] = Entry{v, d, rs, re};
        big |= re - rs >= kLocalDeg;
      }
      // a vertex of many edges among them: the grid runs this round, as a wide one
      if (__syncthreads_or(big)) {
        if (a.hops) r.flags |= kWaveWide;
        break;
      }
      load = false;
    }
    if (threadIdx.x == 0) {
      sh.pile_n[cur ^ 1] = 0;
      sh.spill_n = 0;
    }
    __syncthreads();
    const LocalRelax<A, BS> relax{a,           sh, cur ^ 1, wave_threshold(a, cd0, r.steps), r.round + 1, r.phase + 1,
                                  wave_queue(a, r.near_q()), wave_queue(a, r.far_q())};
    expand_entries<A, kLdsAS, BS, true>(a, (EntryPtr<kLdsAS>)sh.pile[cur], n, relax, &sh.items);
    __syncthreads();  // every push of the round is in
    popped += n;
    ++rounds;
    if (A == Algo::SSSP) pace.round(n, true);
    r.round += 1;
    r.flags &= ~kWaveCut;
    const uint32_t near = sh.pile_n[cur ^ 1], far = sh.far_n;
    if (threadIdx.x == 0) st_coh(&a.ctrl->progress, r.round);
    if (near > a.local_max || sh.stop) {
      // hand over: what spilled already, and the pile
      for (uint32_t i = threadIdx.x; i < min(near, kLocalCap); i += BS) relax.spill(sh.pile[cur ^ 1][i].v);
      __syncthreads();
      n = sh.spill_n;
      r.roles = wave_roles(r.near_q(), r.in_q(), r.far_q());
      if (a.hops) grow();
      if (a.hops && sh.stop) r.flags |= kWaveWide;
      break;
    }
    if (near) {
      cur ^= 1;
      n = near;
      growth.peak = max(growth.peak, n);
    } else if (far) {
      // the whole far pile is the next phase's input (apps/sssp/kernel.cu:374-383)
      r.roles = wave_roles(r.far_q(), r.near_q(), r.in_q());
      r.phase += 1;
      r.flags |= kWaveCut;
      r.cut = r.steps;
      r.steps += a.pace ? pace.next(r.phase - 1, r.flags, a.nedges <= 2ull * a.nnodes) : 1u;
      n = far;
      order_release();  // this wavefront's far pushes have landed
      __syncthreads();  // and every other's; far_n has been read
      if (threadIdx.x == 0) sh.far_n = 0;
      if (n > a.local_max) {
        if (a.hops) grow();
        break;
      }
      growth.peak = max(growth.peak, n);
      load = true;
    } else {
      r.flags |= kWaveDone;
      n = 0;
      break;
    }
    // (the next round's first barrier separates the reads of sh above from its writes)
  }
  order_release();
  __syncthreads();
  if (threadIdx.x == 0) {
    r.items = n;
    r.heavy = 0;
    sh.r = r;
    sh.pace = pace;
    sh.growth = growth;
    if (A == Algo::SSSP) {
      st_coh(&a.wc->far_tail[r.far_q()].n, sh.far_n);
      if (r.far_q() != 0) st_coh(&a.wc->far_tail[0].n, 0u);
      if (r.far_q() != 1) st_coh(&a.wc->far_tail[1].n, 0u);
      if (r.far_q() != 2) st_coh(&a.wc->far_tail[2].n, 0u);
    }
    __hip_atomic_fetch_add(&a.ctrl->stat_items, (uint64_t)popped, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_add(&a.ctrl->stat_rounds, (uint64_t)rounds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  order_release();
  __syncthreads();
}

// ---- the kernel -------------------------------------------------------------------

template <Algo A, int BS>
__global__ __launch_bounds__(BS, 4) void wave_kernel(WaveArgs a) {
  constexpr uint32_t NW = BS / kWave;
  __shared__ WaveShared<BS> sh;
  Ctrl *const c = a.ctrl;
  WaveCtrl *const wc = a.wc;
  const uint32_t nb = gridDim.x, wv = threadIdx.x / kWave;
  const uint32_t wave = blockIdx.x * NW + wv, nwaves = nb * NW;
  const uint32_t ngroups = min(kTicketGroups, nb), g = blockIdx.x % ngroups;
  const uint32_t gblocks = (nb + ngroups - 1 - g) / ngroups;  // blocks of this group
  if (!residency_handshake(c, nb, a.residency_limit)) return;
  const int64_t cd0 = c->s.curdelta();  // written before this launch, as is the first round
  if (threadIdx.x == 0) {
    WaveRound x;
    memset(&x, 0, sizeof x);
    x.items = c->s.in_count;
    x.round = 1;
    x.roles = wave_roles(0, 1, 2);
    x.flags = a.wide ? kWaveWide : 0u;
    sh.r = x;
    sh.gen = 0;
  }
  __syncthreads();
  WaveLane w;
  w.pbuf[0] = sh.push[wv][0];
  w.pbuf[1] = sh.push[wv][1];
  w.hbuf = sh.heavy[wv];
  w.n[0] = w.n[1] = w.hn = w.settled = w.hopped = 0;
  for (;;) {
    const WaveRound r = sh.r;
    const uint32_t gen = sh.gen;
    if (r.flags & kWaveDone) break;
    WaveCtrl::Slot *const slot = &wc->slot[gen % 3];
    w.near_stamp = r.round + 1;
    w.far_stamp = r.phase + 1;
    w.thr = wave_threshold(a, cd0, r.steps);
    w.cut = r.flags & kWaveCut ? (int64_t)wave_threshold(a, cd0, r.cut) : -1;
    w.direct = r.items <= kDirectMax;
    w.nq = wave_queue(a, r.near_q());
    w.fq = wave_queue(a, r.far_q());
    w.ntail = &slot->near_tail.n;
    w.ftail = &wc->far_tail[r.far_q()].n;
    w.htail = &slot->heavy_tail.n;
    w.hq = gen & 1 ? a.chunk[1] : a.chunk[0];
    // (BFS's first round stays one level: levels that mix there mix in every round)
    w.hops = (A == Algo::BFS && r.round == 1) || r.flags & kWaveSplit ||
                     (r.flags & kWaveWide && (r.items > kWideHops<A> || r.items <= kWideItems))
                 ? 0u
                 : a.hops;
    w.split = a.split || r.flags & kWaveSplit;
    // Units: in-queue items, `per` at a time, then heavy chunks.  A wavefront
    // takes the unit of its number; where there are more units than
    // wavefronts, unit j * ngroups + g belongs to the blocks b with b % ngroups
    // == g, whose wavefronts draw tickets of their group (one word for all
    // wavefronts serialises, ~12 ns a ticket).
    const uint32_t *const in = wave_queue(a, r.in_q());
    const WaveChunk *const hin = gen & 1 ? a.chunk[0] : a.chunk[1];
    const uint32_t per = min((uint32_t)kWave, max(r.flags & kWaveWide ? 1u : a.unit_min, (r.items + nwaves - 1) / nwaves));
    const uint32_t nitem = (r.items + per - 1) / per, nunits = nitem + r.heavy;
    const bool many = nunits > nwaves;
    uint32_t unit = many ? (blockIdx.x / ngroups * NW + wv) * ngroups + g : wave;
    while (unit < nunits) {
      uint32_t t = 0;
      if (many && lane_id() == 0) t = atomic_add(&slot->ticket[g].n, 1u);
      if (unit < nitem) wave_items<A>(a, w, in + (size_t)unit * per, min(per, r.items - unit * per));
      else wave_chunk<A>(a, w, hin + (unit - nitem));
      if (!many) break;
      unit = (gblocks * NW + readlane(t, 0)) * ngroups + g;
    }
    // The block's pushes get their places with one atomic per pile.
    if (w.split) wave_settle(a, w);
    const uint32_t hend = w.hn ? wave_heavy_ends(a, w) : 0u;
    order_release();
    if (lane_id() == kWave - 1) {
      sh.count[wv][0] = w.n[0];
      sh.count[wv][1] = w.n[1];
      sh.count[wv][2] = hend;
    }
    __syncthreads();
    uint32_t tot[3] = {0, 0, 0}, off[3] = {0, 0, 0};
#pragma unroll
    for (uint32_t i = 0; i < NW; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        if (i < wv) off[p] += sh.count[i][p];
        tot[p] += sh.count[i][p];
      }
    if (tot[0] | tot[1] | tot[2]) {
      if (threadIdx.x < 3) {
        const uint32_t n = threadIdx.x == 0 ? tot[0] : threadIdx.x == 1 ? tot[1] : tot[2];
        uint32_t *const tail = threadIdx.x == 0 ? w.ntail : threadIdx.x == 1 ? w.ftail : w.htail;
        sh.base[threadIdx.x] = n ? atomic_add(tail, n) : 0u;
      }
      __syncthreads();
      if (w.n[0]) wave_store(a, w, 0, sh.base[0] + off[0]);
      if (w.n[1]) wave_store(a, w, 1, sh.base[1] + off[1]);
      if (w.hn) wave_store_heavy(a, w, hend, sh.base[2] + off[2]);
      order_release();
      __syncthreads();
    }
    // The barrier: wavefront 0.  The blocks with a unit arrive, and the one that
    // led the last round, so that what it cleared then is clear by now; the
    // others only wait for a message of a later generation, and may miss rounds
    // that they had no part in.  The last to arrive finds the next round.
    if (wv == 0) {
      const uint32_t active = many ? nb : (nunits + NW - 1) / NW;
      const uint32_t parties = active + (r.lead >= active ? 1u : 0u);
      const uint32_t seat = blockIdx.x < active ? blockIdx.x : blockIdx.x == r.lead ? active : parties;
      if (seat < parties && wave_arrive(slot, seat, parties)) {
        order_acquire();
        WaveRound x = r;
        // every word that the step needs in one load
        const uint32_t lane = lane_id();
        const uint32_t *p = lane == 0 ? &slot->near_tail.n : lane == 1 ? &slot->heavy_tail.n : lane == 2 ? &c->abort
                            : lane < 10 ? &wc->pace[lane - 3] : &wc->far_tail[r.far_q()].n;
        const uint32_t word = ld_coh(p);
        const uint32_t nnear = readlane(word, 0), nheavy = readlane(word, 1), ab = readlane(word, 2);
        const uint32_t nfar = A == Algo::SSSP ? readlane(word, 10) : 0u;
        WavePace pace{max(readlane(word, 3), 1u), readlane(word, 4), __uint_as_float(readlane(word, 5)),
                      __uint_as_float(readlane(word, 6)), readlane(word, 7)};
        WaveGrowth growth{max(readlane(word, 8), r.items), readlane(word, 9)};
        if (A == Algo::SSSP) pace.round(r.items, false);
        // (the slot of the round before the last: no block reads it any more)
        WaveCtrl::Slot *const next = &wc->slot[(gen + 2) % 3];
        const uint32_t nclear = offsetof(WaveCtrl::Slot, arrive) / sizeof(WaveCtrl::Line) + (nb + kBarGroup - 1) / kBarGroup;
        for (uint32_t i = lane; i < nclear; i += kWave) st_coh(&reinterpret_cast<WaveCtrl::Line *>(next)[i].n, 0u);
        const bool full = nnear > a.qcap || nfar > a.qcap || nheavy > a.hcap;
        if (full) st_coh(&c->abort, kAbortCapacity);
        const bool within = nnear > 0 || nheavy > 0, phase = A == Algo::SSSP && !within && nfar > 0;
        const bool done = full || ab != kAbortNone || !(within || phase);
        x.round = r.round + 1;
        x.lead = blockIdx.x;
        x.heavy = nheavy;
        x.items = phase ? nfar : nnear;
        x.roles = wave_roles(r.near_q(), r.in_q(), r.far_q());
        if (phase) {
          // the whole far pile is the next phase's input (apps/sssp/kernel.cu:374-383)
          x.roles = wave_roles(r.far_q(), r.near_q(), r.in_q());
          x.phase = r.phase + 1;
          x.cut = r.steps;
          x.steps = r.steps + (a.pace ? pace.next(r.phase, r.flags, a.nedges <= 2ull * a.nnodes) : 1u);
          if (lane == 0) st_coh(&wc->far_tail[r.far_q()].n, 0u);
        }
        x.flags = kWaveLead | (done ? kWaveDone : x.heavy == 0 && x.items <= a.local_max / 2 ? kWaveLocal : 0u) |
                  (phase ? kWaveCut : 0u) | (a.hops ? growth.flags(x.round, x.items + a.heavy_deg * nheavy, nheavy >= kWideChunks, r.flags) : 0u);
        if (lane == 0) {
          __hip_atomic_fetch_add(&c->stat_items, (uint64_t)r.items, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_fetch_add(&c->stat_heavy, (uint64_t)r.heavy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_fetch_add(&c->stat_rounds, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          sh.pace = pace;
          sh.growth = growth;
          sh.r = x;
          sh.gen = gen + 1;
        }
      } else {
        WaveRound x = r;
        const uint32_t tag = wave_wait(a, gen, x);
        if (lane_id() == 0) {
          sh.r = x;
          sh.gen = tag;
        }
      }
    }
    __syncthreads();
    if (sh.r.flags & kWaveLead) {
      if (sh.r.flags & kWaveLocal) wave_local<A, BS>(a, sh, cd0);
      if (wv == 0) {
        const uint32_t lane = lane_id();
        const WaveRound x = sh.r;
        wave_publish(wc, gen + 1, x);
        if (a.hops && lane < 7) {
          const WavePace p = sh.pace;
          st_coh(&wc->pace[lane], lane == 0 ? p.step : lane == 1 ? p.hold : lane == 2 ? __float_as_uint(p.best)
                                  : lane == 3 ? __float_as_uint(p.cost) : lane == 4 ? p.rounds
                                  : lane == 5 ? sh.growth.peak : sh.growth.until);
        }
        if ((x.flags & kWaveDone) && lane == 0) {
          c->s.done = 1;
          c->s.round = x.round;
          c->s.phase = x.phase;
          c->s.set_curdelta(cd0 + (int64_t)x.steps * a.delta);
          c->stat_phases = x.phase + 1ull;
        }
      }
    }
  }
  if (!a.hops) return;
  uint32_t hopped = w.hopped;
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) hopped += __shfl_xor(hopped, d);
  if (lane_id() == 0 && hopped)
    __hip_atomic_fetch_add(&c->hop_items[wave % kHopGroups][0], (uint64_t)hopped, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- launch -------------------------------------------------------------------------

__global__ void wave_reset_kernel(WaveCtrl *wc, uint32_t wide) {
  wave_reset(wc, threadIdx.x, blockDim.x);
  __syncthreads();
  if (threadIdx.x == 0 && wide) wc->pace[6] = kWideRounds;  // WaveGrowth::until
}

// Distances, stamps, control words and the one seed (apps/sssp/kernel.cu:23-35,469,476-477).
__global__ void wave_init_kernel(WaveArgs a, uint32_t seed) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
  for (uint32_t v = tid; v < a.nnodes; v += nt) {
    glb(a.dist)[v] = v == seed ? 0u : kInf;
    glb(a.near_stamp)[v] = 0u;
    glb(a.far_stamp)[v] = 0u;
  }
  ctrl_init(a, a.delta, 0, tid, nt);
  if (blockIdx.x == 0) wave_reset(a.wc, threadIdx.x, blockDim.x);
  if (tid == 0) {
    a.q[0][0] = seed;
    a.ctrl->s.in_count = 1;
  }
}

// The deepest level, to aux[3].
__global__ void wave_levels_kernel(const uint32_t *level, uint32_t n, Ctrl *c) {
  uint32_t deep = 0;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    const uint32_t l = glb(level)[v];
    deep = max(deep, l == kInf ? 0u : l);
  }
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) deep = max(deep, (uint32_t)__shfl_xor(deep, d));
  if (lane_id() == 0 && deep) __hip_atomic_fetch_max(glb(&c->s.aux[3]), deep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

using WaveFn = void (*)(WaveArgs);
template <Algo A>
static WaveFn pick_wave(int bs) {
  return bs == 256 ? wave_kernel<A, 256> : bs == 1024 ? wave_kernel<A, 1024> : wave_kernel<A, 512>;
}
static WaveFn pick_wave(Algo algo, int bs) {
  return algo == Algo::SSSP ? pick_wave<Algo::SSSP>(bs) : pick_wave<Algo::BFS>(bs);
}

const void *wave_kernel_fn(Algo algo, int bs) { return (const void *)pick_wave(algo, bs); }

int wave_enqueue(Algo algo, int bs, int grid, const WaveArgs &a, uint32_t seed, const uint32_t *seeds, uint32_t nseeds,
                 const Resume *resume, int cus, hipStream_t stream) {
  const uint32_t blocks = std::min<uint32_t>((a.nnodes + 255) / 256, 8u * cus);
  if (resume || seeds) {
    const KArgs &k = a;
    if (resume) {
      hipLaunchKernelGGL(resume_init_kernel, dim3(blocks), dim3(256), 0, stream, k, a.delta, resume->curdelta);
      hipLaunchKernelGGL(resume_seed_kernel, dim3(blocks), dim3(256), 0, stream, k, resume->lo, resume->hi);
    } else {
      hipLaunchKernelGGL(init_kernel, dim3(blocks), dim3(256), 0, stream, k, a.delta);
      hipLaunchKernelGGL(seed_kernel, dim3(1), dim3(256), 0, stream, k, seeds, nseeds);
    }
    hipLaunchKernelGGL(wave_reset_kernel, dim3(1), dim3(256), 0, stream, a.wc, a.wide);
  } else {
    hipLaunchKernelGGL(wave_init_kernel, dim3(blocks), dim3(256), 0, stream, a, seed);
  }
  hipLaunchKernelGGL(pick_wave(algo, bs), dim3(grid), dim3(bs), 0, stream, a);
  if (a.levels)
    hipLaunchKernelGGL(wave_levels_kernel, dim3(std::min<uint32_t>(blocks, (uint32_t)cus)), dim3(256), 0, stream,
                       (const uint32_t *)a.dist, a.nnodes, a.ctrl);
  HIPCHK(hipGetLastError());
  return LSG_OK;
}

}  // namespace lsg
