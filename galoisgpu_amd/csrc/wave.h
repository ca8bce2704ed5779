// Single-source traversal by wavefronts (wave.hip): what its host side needs.
#pragma once

#include "sssp_dev.h"

namespace lsg {

constexpr int kWaveMsg = 7;
constexpr uint32_t kTicketGroups = 16;

// Words of the wavefront kernel beside the control block, each group of words
// that one atomic unit serves on a line of its own.
struct WaveCtrl {
  // The state of the next round, published by the last block to reach the
  // barrier: value << 32 | generation, so that a word is valid by itself and
  // a waiting block needs no second load and the publisher no ordering.
  uint64_t msg[kWaveMsg];
  uint64_t _p0[16 - kWaveMsg];
  // How far the next phase moves the threshold, and how the rounds grow (WavePace,
  // WaveGrowth); between leading blocks only.
  uint32_t pace[7];
  uint32_t _p1[25];
  struct alignas(8) Line {
    uint32_t n;
    uint32_t _p[31];
  };
  Line far_tail[3];  // by queue
  // By generation mod 3: the leader of one round clears the words of the one
  // after the next.
  struct Slot {
    Line near_tail, heavy_tail, ticket[kTicketGroups], top;
    Line sum[kTicketGroups];  // u64: edges of the vertices found << 32 | vertices found (bfs_do.hip)
    Line arrive[kMaxBarGroups];
  } slot[3];
};

// Up to heavy_deg edges of a heavy vertex: popped at distance d, or INF.
struct WaveChunk {
  uint32_t u, d, first, n;
};

struct WaveArgs : KArgs {
  WaveChunk *chunk[2] = {nullptr, nullptr};  // in place of KArgs::hq
  WaveCtrl *wc = nullptr;
  uint32_t pace = 0;      // the threshold's steps are paced (WavePace)
  uint32_t unit_min = 0;  // fewest items of a unit
  uint32_t local_max = 0; // largest round that one block runs alone
  uint32_t hops = 0;      // times that a wavefront goes on with what it pushed near
  uint32_t wide = 0;      // the first rounds are wide (WaveGrowth)
  uint32_t levels = 0;    // BFS: the deepest level is looked up at the end
  uint32_t _pad = 0;
  uint32_t split = 0;     // vertices of kWaveSplitDeg edges are queued as chunks when they are pushed, else of heavy_deg when popped
};

// Blocks per CU, of 256 threads, where the call leaves the launch shape open.
// Blocks without a unit stay out of a round's barrier, so more of them cost a
// small round little; each wavefront fewer makes the large rounds longer, and a
// graph has to be large to have such rounds.  Ms at 1 / 2 / 3 blocks: RMAT-17
// SSSP 0.358 / 0.359 / 0.369, RMAT-18 0.464 / 0.448 / 0.463, RMAT-19 0.67 / 0.62
// / 0.63, RMAT-20 1.10 / 0.90 / 0.87, RMAT-21 1.81 / 1.35 / 1.26, RMAT-22 3.1 /
// 2.3 / 2.1; BFS RMAT-17 0.117 / 0.117 / 0.132, RMAT-19 0.223 / 0.198 / 0.202, RMAT-20 0.385 /
// 0.293 / 0.278; road-like SSSP 1000^2 1.18 / 1.14 / 1.15, 1500^2 1.77 / 1.73 /
// 1.77, 2048^2 2.17 / 2.05 / 2.03, BFS 0.62 / 0.63 / 0.64, 0.88 / 0.84 / 0.86, 1.13 /
// 1.12 / 1.10; grid 1500^2 SSSP 18.65 / 18.74 / 18.80.  The same wavefronts in blocks
// of 512: RMAT-19 0.71, RMAT-20 0.98, 2048^2 2.08; 1024 worse still.
constexpr int kWaveBlock = 256;
inline int wave_blocks_per_cu(uint64_t nnodes, uint64_t nedges) {
  if (low_degree(nnodes, nedges)) return nedges < 6'000'000 ? 1 : 2;
  return nedges < 3'000'000 ? 1 : nedges < 12'000'000 ? 2 : 3;
}
// Largest round, in items, that one block runs alone: some 2048 edges (limits
// of 512 / 128 items on RMAT: 2^14 vertices 0.256 / 0.245 ms, 2^20 1.00 / 0.98).
inline uint32_t wave_local_max(uint64_t nnodes, uint64_t nedges) {
  return (uint32_t)(nedges <= 4 * nnodes ? 512 : 2048 * nnodes / nedges);
}
// A round with a vertex of this many edges is the whole grid's, on low-degree graphs
// one item a unit: in a round of one block a lane has its edges four at a time, or a
// wavefront several such vertices one after another, and of units of 16 items as few
// wavefronts would have any.  BFS kernel us where it is left at 256 (heavy_deg) / 32 /
// 16 edges: 100,000 vertices of 1000 hubs 391 / 122 / 124, a tree of degree 64 224 / 86
// / 86, of degree 30 117 / 105 / 99, a random tree 202 / 205 / 188; SSSP delta 32 at 256
// / 32 / 16 / 8: uniform out-degree 32, 1000 vertices 259 / 186 / 185 / 186, 10,000 484 /
// 334 / 324 / 327, out-degree 16 378 / 377 / 339 / 335, out-degree 7 280 / 282 / 280 /
// 293, RMAT of 16,384 vertices and 8 edges 196 / 192 / 191 / 197; grids and road-like
// graphs alike, also with vertices of 20 and 40 edges among them.
constexpr uint32_t kLocalDeg = 16;
// A chunk of a heavy vertex is the edges that a wavefront holds in flight
// (kWaveU a lane); 512 and 1024: equal to 5 % slower on RMAT graphs.
constexpr int kWaveHeavyDeg = 256;
// On graphs that are not low_degree, vertices of this many edges are taken apart
// when they are pushed: a round earlier than when they are popped, and no
// item has many edges, so that the units of a round take alike.  The row bounds
// are one more round trip, which the narrow rounds of low-degree graphs would
// feel.  Ms when popped / at 128 / 64 / 32 edges: RMAT-14 (8 edges a vertex) SSSP
// 0.25 / 0.21 / 0.19 / 0.18, RMAT-16 0.37 / 0.30 / 0.27 / 0.30, RMAT-18 0.50 / 0.45 /
// 0.44 / 0.45, RMAT-20 0.97 / 0.86 / 0.88 / 0.90, RMAT-22 2.22 / 2.04 / 2.05 / 2.21;
// BFS RMAT-14 0.072 / 0.069 / 0.067 / 0.067, RMAT-18 0.148 / 0.157 / 0.141 / 0.146,
// RMAT-20 0.285 / 0.283 / 0.288 / 0.297, from random sources 0.340 / 0.286 / 0.303 /
// 0.315.
constexpr uint32_t kWaveSplitDeg = 64;
constexpr uint32_t kWaveHops = 4;  // on low-degree graphs

// Block sizes 256, 512 and 1024.
const void *wave_kernel_fn(Algo algo, int bs);
// Enqueues initialisation and traversal: from one seed (seeds null), from
// several, or, with `resume`, from the distances in a.dist.
int wave_enqueue(Algo algo, int bs, int grid, const WaveArgs &a, uint32_t seed, const uint32_t *seeds, uint32_t nseeds,
                 const Resume *resume, int cus, hipStream_t stream);

// The last round that was published, for the text of an error: the control block
// does not follow the rounds.  (A launch starts with round 1, unpublished.)
struct WaveLast {
  uint32_t round = 1, phase = 0, generation = 0;
};
inline WaveLast wave_last(const WaveCtrl *wc) {
  uint64_t m[kWaveMsg];
  WaveLast l;
  if (hipMemcpy(m, wc->msg, sizeof m, hipMemcpyDeviceToHost) != hipSuccess || m[0] == 0) return l;
  l.round = (uint32_t)(m[2] >> 32);
  l.phase = (uint32_t)(m[3] >> 32);
  l.generation = (uint32_t)m[0];
  return l;
}

}  // namespace lsg
