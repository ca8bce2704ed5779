// Connected components on gfx950: hooking and pointer jumping over a device CSR.
//
// Reference: apps/cc/kernel.cu -- init (:18-29) labels every node with its
// own id, hook_init/hook_high_to_low/hook_low_to_high (:249-336) point the
// root of one endpoint of every edge at the other's, p_jump (:338-369)
// shortcuts parents, count_components (:449-462) counts roots, and gg_main
// (:630-723) iterates until no hook succeeds.  Edges are taken without
// direction (weakly connected components of a directed graph).  The
// reference's hooks are plain racing stores, so which id ends up as a
// component's label depends on the schedule; here a hook is a compare-and-swap
// of the larger root's parent to the smaller root, so every vertex ends labelled
// with the smallest id of its component -- the same partition, with one
// deterministic label per component.
//
// Layout: label u32[V] (the parent pointer, node_data; a parent's id is never
// above its child's) and one control word, the component count.  The reference
// repeats hook and jump passes until no hook succeeds; here every edge is
// looked at once:
//   cc_init_kernel      label[v] = v's first out-neighbour if that is smaller, else v;
//   cc_flatten_kernel   every vertex to the root of that forest;
//   cc_persistent_kernel  joins the trees of every edge's ends (compare-and-swap on
//     the larger root, again from what it found if it lost), a grid barrier, then
//     every vertex to its root.
// An edge whose ends already have the same label needs nothing else, and after
// the first two kernels that is nearly every edge of a skewed graph (a row's
// first neighbour is a hub), so the edge pass is one gather per edge, read
// through the caches: a stale label is an earlier ancestor, which only sends
// the edge on to the coherent loads of cc_join.  RMAT-22 4.5 -> 0.97 ms
// (hook and jump passes until nothing hooked: three passes of 1.4 ms), 2048^2
// road-like 1.5-2.6 -> 0.35 ms.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>

#include "engine.h"
#include "lsg_internal.h"
#include "runtime.h"

namespace lsg {

// control word of the component count
constexpr int kCtlCount = 1;
constexpr uint32_t kCcBlock = 256;
// Consecutive edges per wavefront and step of the edge pass, and label gathers
// in flight per lane.
constexpr uint32_t kCcTile = 1024;
constexpr int kCcFlight = 4;

struct CcArgs {
  const uint32_t *row_start, *edge_dst;
  uint32_t *label, *ctl;
  Ctrl *ctrl;
  uint32_t V, E;
  uint32_t tile;  // vertices per block step of cc_init_kernel
  uint64_t spin_limit, residency_limit;
};

// First labels (tiles of a.tile <= kCcInitTile consecutive vertices per block),
// the count and the control block.  A vertex takes the largest of its first four
// neighbours that is smaller than itself and in its tile, or else its first
// neighbour if that is smaller, or else itself; the tile's trees are then
// flattened in LDS.  Neighbours in the tile make a grid's rows trees of their
// own, flattened at LDS speed (the smallest neighbour alone makes every
// column a chain: 2048^2 road-like 2.9 instead of 0.33 ms); on a skewed graph nearly every
// vertex takes its first neighbour, a hub.
constexpr uint32_t kCcInitTile = 4096;
__global__ __launch_bounds__(kCcBlock) void cc_init_kernel(CcArgs a) {
  __shared__ uint32_t lab[kCcInitTile];
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x;
  const uint32_t ntiles = a.V / a.tile + (a.V % a.tile != 0);
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const uint32_t base = t * a.tile, n = min(a.V - base, a.tile);
    for (uint32_t i = threadIdx.x; i < n; i += kCcBlock) {
      const uint32_t v = base + i, e0 = a.row_start[v], e1 = a.row_start[v + 1];
      uint32_t l = v;
      if (e0 < e1) {
        uint32_t d[4], in = v;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) d[k] = a.edge_dst[min(e0 + k, e1 - 1)];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
          if (d[k] >= base && d[k] < v && (in == v || d[k] > in)) in = d[k];
        l = in != v ? in : min(v, d[0]);
      }
      lab[i] = l;
    }
    __syncthreads();
    // a root with an in-edge from a vertex of the tile (of at most four edges) takes its source
    for (uint32_t i = threadIdx.x; i < n; i += kCcBlock) {
      const uint32_t v = base + i, e0 = a.row_start[v], e1 = a.row_start[v + 1];
      if (e1 - e0 > 4) continue;
      for (uint32_t e = e0; e < e1; ++e) {
        const uint32_t d = a.edge_dst[e];
        if (d > v && d - base < n && lab[d - base] == d) lab[d - base] = v;
      }
    }
    __syncthreads();
    bool more = true;
    while (more) {
      bool changed = false;
      for (uint32_t i = threadIdx.x; i < n; i += kCcBlock) {
        const uint32_t l = lab[i];
        if (l < base) continue;
        const uint32_t up = lab[l - base];
        if (up != l) {
          lab[i] = up;
          changed = true;
        }
      }
      more = __syncthreads_or(changed);
    }
    for (uint32_t i = threadIdx.x; i < n; i += kCcBlock) a.label[base + i] = lab[i];
    __syncthreads();  // lab is read before the next tile's labels replace it
  }
  ctrl_reset_barrier(a.ctrl, tid, nt);
  if (tid == 0) {
    a.ctl[kCtlCount] = 0;
    Ctrl *c = a.ctrl;
    c->abort = kAbortNone;
    c->checkin = 0;
    c->resident_seen = 0;
    c->progress = 0;
    Sched s;
    memset(&s, 0, sizeof s);
    c->s = s;
  }
}

// Moves v's label from its ancestor p to the root of its tree.  Only v's own
// label is written, step by step, so that walks through v get shorter while
// this one goes on (pointer jumping: the steps double when every vertex of a
// deep tree does the same) and no other thread can set v's final label back.
__device__ __forceinline__ void cc_climb(uint32_t *label, uint32_t v, uint32_t p) {
  for (;;) {
    const uint32_t q = ld_coh(label + p);
    if (q == p) return;
    p = q;
    st_coh(label + v, p);
  }
}

// Every vertex to the root of the first forest.  Two steps are read through
// the caches (most trees of a skewed graph are that shallow); the grid takes
// the vertices in ascending order, so a deep tree (a column of a grid) is
// short above the vertices already done.
__global__ __launch_bounds__(kCcBlock) void cc_flatten_kernel(CcArgs a) {
  for (size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x; v < a.V; v += (size_t)gridDim.x * blockDim.x) {
    const uint32_t p = glb(a.label)[v], q = glb(a.label)[p];
    if (q == p) continue;
    st_coh(a.label + v, q);
    cc_climb(a.label, (uint32_t)v, q);
  }
}

// One step towards joining the trees that hold a and b (a != b): hooks the
// larger under the smaller if it is a root, otherwise replaces it by an
// ancestor.  a == b afterwards: joined.
__device__ __forceinline__ void cc_join(uint32_t *label, uint32_t &a, uint32_t &b) {
  const uint32_t hi = max(a, b), lo = min(a, b);
  b = lo;
  const uint32_t p = ld_coh(label + hi);
  if (p != hi) {
    const uint32_t q = ld_coh(label + p);
    if (q != p) st_coh(label + hi, q);
    a = q;
    return;
  }
  uint32_t seen = hi;
  const bool hooked = __hip_atomic_compare_exchange_strong(glb(label + hi), &seen, lo, __ATOMIC_RELAXED,
                                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  a = hooked ? lo : seen;
}

// Joins the listed pairs, lane i's px and py for i < n.
__device__ __forceinline__ void cc_join_listed(uint32_t *label, uint32_t n, uint32_t px, uint32_t py) {
  if (lane_id() >= n) px = py;
  while (__ballot(px != py))
    if (px != py) cc_join(label, px, py);
}

// Joins the trees of every edge's ends.  Edge-balanced: a wavefront takes
// kCcTile edges and holds 64 rows (ends and labels), in which each lane looks
// up its edge's source with six shuffles.  The pairs of unequal labels (2% of
// RMAT-19's edges, so most steps of 256 edges have a few) are listed and
// joined 64 at a time: a join is two or three dependent round trips however
// few lanes take part (RMAT-22 1.29 -> 0.91 ms).  What is left is one label
// gather per edge, 80 G/s from a 16 MB array.
__device__ void cc_edge_pass(const CcArgs &a) {
  const uint32_t lane = lane_id();
  uint32_t px = 0, py = 0, n = 0;  // listed pairs, one per lane below n
  const uint32_t waves = gridDim.x * (kCcBlock / kWave);
  const uint32_t ntiles = a.E / kCcTile + (a.E % kCcTile != 0);
  for (uint32_t t = blockIdx.x * (kCcBlock / kWave) + threadIdx.x / kWave; t < ntiles; t += waves) {
    uint32_t e = t * kCcTile;
    const uint32_t left = a.E - e, tile_end = e + min(left, kCcTile);
    while (e < tile_end) {
      const uint32_t u0 = wave_row_near(a.row_start, a.V, e);
      const uint32_t re = glb(a.row_start)[min(u0 + lane, a.V - 1) + 1];
      const uint32_t lab = glb(a.label)[min(u0 + lane, a.V - 1)];
      const uint32_t end = min(tile_end, readlane(re, kWave - 1));  // > e
      for (; e < end; e += min(end - e, (uint32_t)(kCcFlight * kWave))) {
        uint32_t lu[kCcFlight], lv[kCcFlight];
#pragma unroll
        for (int k = 0; k < kCcFlight; ++k) {
          const uint32_t i = e + min(k * kWave + lane, end - 1 - e);  // past the end: the last edge again
          lv[k] = glb(a.edge_dst)[i];
          uint32_t pos = 0;  // rows that end at or before edge i
#pragma unroll
          for (uint32_t d = kWave / 2; d >= 1; d >>= 1)
            if (__shfl(re, pos + d - 1) <= i) pos += d;
          lu[k] = __shfl(lab, pos);
        }
#pragma unroll
        for (int k = 0; k < kCcFlight; ++k) lv[k] = glb(a.label)[lv[k]];
#pragma unroll
        for (int k = 0; k < kCcFlight; ++k) {
          const uint64_t m = __ballot(e + k * kWave + lane < end && lu[k] != lv[k]);
          const uint32_t c = (uint32_t)__builtin_popcountll(m);
          if (c == 0) continue;
          if (n + c > (uint32_t)kWave) {
            cc_join_listed(a.label, n, px, py);
            n = 0;
          }
          // a permutation of the lanes: unequal pairs to n, n + 1, ..., the others behind them
          const uint32_t to = ((m >> lane) & 1 ? n + lanes_below(m) : n + c + lanes_below(~m)) % kWave * 4;
          const uint32_t tx = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)lu[k]);
          const uint32_t ty = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)lv[k]);
          if (lane >= n && lane < n + c) {
            px = tx;
            py = ty;
          }
          n += c;
        }
      }
    }
  }
  cc_join_listed(a.label, n, px, py);
}

__global__ __launch_bounds__(kCcBlock) void cc_persistent_kernel(CcArgs a) {
  __shared__ uint32_t s_n, quit;
  Ctrl *c = a.ctrl;
  const uint32_t nb = gridDim.x;
  if (!residency_handshake(c, nb, a.residency_limit)) return;
  if (threadIdx.x == 0) s_n = 0;
  cc_edge_pass(a);
  grid_barrier_block(c, nb, a.spin_limit, [&] {
    if (threadIdx.x == 0) st_coh(&c->s.done, 1u);
  });
  if (threadIdx.x == 0) quit = ld_coh(&c->abort) != kAbortNone;
  __syncthreads();
  if (quit) return;
  // no tree changes any more: every vertex to its root
  uint32_t n = 0;
  for (size_t v = blockIdx.x * (size_t)kCcBlock + threadIdx.x; v < a.V; v += (size_t)nb * kCcBlock) {
    const uint32_t p = ld_coh(a.label + v);
    n += p == v;
    if (p != v) cc_climb(a.label, (uint32_t)v, p);
  }
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) n += __shfl_xor(n, d);
  if (lane_id() == 0 && n) atomicAdd(&s_n, n);
  __syncthreads();
  if (threadIdx.x == 0 && s_n) atomic_add(a.ctl + kCtlCount, s_n);
}

}  // namespace lsg

using namespace lsg;

extern "C" {

int lsg_cc(const lsg_graph *g, int32_t *label_dev, uint32_t *ncomponents, lsg_stats *stats) {
  clear_error();
  auto t0 = std::chrono::steady_clock::now();
  if (!g || g->device_graph == 0 || !g->row_start || (g->nedges && !g->edge_dst))
    return fail(LSG_ERR_ARG, "cc: expected a device graph (copy_to_gpu first)");
  if (!label_dev) return fail(LSG_ERR_ARG, "cc: NULL label array");
  Workspace *w;
  int rc = get_workspace(g->device, &w);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(w->mu);
  HIPCHK(hipSetDevice(w->device));
  void *cbuf;
  if ((rc = ws_buffer(w, kBufSeeds, 2048, &cbuf))) return rc;
  uint32_t *ctl = (uint32_t *)cbuf;
  const uint32_t V = g->nnodes, E = g->nedges;
  uint32_t *label = (uint32_t *)label_dev;
  const uint32_t vgrid = (uint32_t)std::min<uint64_t>(((uint64_t)V + 255) / 256, 16ull * w->cus);
  const void *fn = (const void *)cc_persistent_kernel;
  int grid = 0;
  if ((rc = resident_grid(w, fn, kCcBlock, &grid))) return rc;
  // no more blocks than the edge tiles or the vertices keep busy
  grid = (int)std::min<uint64_t>(grid, std::max<uint64_t>({64, E / (kCcTile * (kCcBlock / kWave)) + 1, vgrid}));
  CcArgs a;
  a.row_start = g->row_start;
  a.edge_dst = g->edge_dst;
  a.label = label;
  a.ctl = ctl;
  a.ctrl = w->ctrl;
  a.V = V;
  a.E = E;
  // four tiles per CU where that keeps them below the LDS array (16384 vertices: whole call 81 -> 52 us)
  const uint32_t per = V / (4 * w->cus) / 256 * 256 + 256;
  a.tile = std::min(kCcInitTile, per);
  const uint32_t igrid = (uint32_t)std::min<uint64_t>(V / a.tile + 1, 8ull * w->cus);
  a.spin_limit = spin_limit_ticks(w);
  a.residency_limit = residency_limit_ticks(w);
  Ctrl hc;
  float ms = 0;
  uint32_t *c = w->pinned;
  for (int attempt = 0;; ++attempt) {
    HIPCHK(hipEventRecord(w->ev0, w->stream));
    hipLaunchKernelGGL(cc_init_kernel, dim3(igrid), dim3(kCcBlock), 0, w->stream, a);
    hipLaunchKernelGGL(cc_flatten_kernel, dim3(vgrid), dim3(kCcBlock), 0, w->stream, a);
    hipLaunchKernelGGL(cc_persistent_kernel, dim3(grid), dim3(kCcBlock), 0, w->stream, a);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(w->ev1, w->stream));
    HIPCHK(hipMemcpyAsync(&hc, w->ctrl, kCtrlHostBytes, hipMemcpyDeviceToHost, w->stream));
    HIPCHK(hipMemcpyAsync(c, ctl, 16, hipMemcpyDeviceToHost, w->stream));
    HIPCHK(hipStreamSynchronize(w->stream));
    HIPCHK(hipEventElapsedTime(&ms, w->ev0, w->ev1));
    if (hc.abort != kAbortResidency) break;
    if (attempt > 0 || hc.resident_seen == 0 || hc.resident_seen >= (uint32_t)grid)
      return fail(LSG_ERR_HIP, "cc: persistent grid of %d x %d blocks is not co-resident (%u were)", grid,
                  (int)kCcBlock, hc.resident_seen);
    grid = (int)hc.resident_seen;
    record_resident_grid(w, fn, kCcBlock, grid);
  }
  if (hc.abort != kAbortNone || !hc.s.done)
    return fail(LSG_ERR_TIMEOUT, "cc: the grid barrier after the edge pass timed out");
  if (ncomponents) *ncomponents = c[kCtlCount];
  if (stats) {
    memset(stats, 0, sizeof *stats);
    stats->ms_kernel = ms;
    stats->iterations = 1;
    stats->items = c[kCtlCount];
    stats->grid_blocks = grid;
    stats->block_size = kCcBlock;
    stats->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  return LSG_OK;
}

int lsg_cc_gg_main(lsg_graph *hg, lsg_graph *gg, lsg_stats *stats) {
  (void)hg;
  if (!gg || !gg->node_data) return fail(LSG_ERR_ARG, "cc gg_main: device graph without node_data");
  return lsg_cc(gg, gg->node_data, nullptr, stats);
}

}  // extern "C"
