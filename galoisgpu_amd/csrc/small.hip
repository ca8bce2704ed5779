// Single-source SSSP and BFS of a small low-degree graph in one workgroup, the
// distances in LDS.
//
// A grid or road network of a few thousand vertices is hundreds of rounds of a
// few dozen vertices each.  Even where one block runs them (wave.hip) a round is
// three round trips to the coherence point (edges, atomicMin, stamp), some 3.3
// us.  Here the atomicMins, the sets of queued and far vertices and the round's
// lists are all LDS operations, and what remains of a round is the row bounds
// and the edges, from the L2: 1.2 to 1.5 us.
//
// The phases are near/far phases (apps/sssp/kernel.cu:355-391), the far vertices
// a bitmap.  At the end of a phase the threshold moves by DELTA, then by twice
// as much and so on until kSmallTarget vertices are near (a round costs the same
// up to the workgroup's size), and in later phases by as much at once; rounds
// beyond the workgroup's size halve it again.  Vertices whose distance came below
// the last threshold since they were set were near vertices then, and are dropped.
//
// Used up to kSmallV vertices (128 KB of the CU's 160) of low degree.  A frontier
// of many vertices is faster over the whole GPU: a round of more than kSmallList,
// or, above kSmallSkewV vertices, one that met a vertex of kSmallHub edges (the
// mark of a skewed graph) is left to the wavefront kernel, which goes on from the
// distances reached.  Call us with the persistent kernel / with all rounds here /
// now, delta 10000: uniform out-degree 4, 16384 vertices 260 / 271 / 190, 32768 260 /
// 352 / 194; RMAT-like of 5 edges, 32768 vertices 267 / 857 / 240; 50 hubs and 32768
// vertices 171 / 597 / 198; a tree of degree 16 111 / 260 / 133.  At most 8192
// vertices of a hub's are as fast here.  Kernel ms in wave.hip ->
// here: SSSP grid 64^2 0.52 -> 0.22, 100^2 0.93 -> 0.36, 181^2 1.74 -> 0.75, 40 x
// 500 2.7 -> 1.3, road-like 181^2 0.63 -> 0.44; BFS grid 64^2 0.26 -> 0.16, 181^2
// 0.90 -> 0.45, road-like 181^2 0.39 -> 0.19.
//
// There are no spin waits: every wait is a workgroup barrier.

#include <hip/hip_runtime.h>

#include <cstring>

#include "sssp_dev.h"

namespace lsg {

constexpr uint32_t kSmallThreads = 1024;  // (512 / 256: road-like 181^2 0.44 -> 0.53 / 0.77 ms, grids alike)
constexpr uint32_t kSmallList = 4096;    // listed vertices of a round; with more, the whole grid goes on
constexpr uint32_t kSmallTarget = 256;   // vertices that a phase begins with, if there are so many
constexpr uint32_t kSmallHeavy = 32;     // vertices of more edges are expanded by their wavefront
constexpr uint32_t kSmallHub = 256, kSmallSkewV = 8192;
constexpr uint32_t kSmallWords = kSmallV / 32;

// What the host reads at the end: written to host memory, as a copy back after
// the kernel costs some 8 us of a call.
struct SmallResult {
  uint64_t items, rounds, phases;
  int64_t curdelta;
  uint32_t handed;  // the rounds go on over the whole grid
};
static_assert(sizeof(SmallResult) <= 256, "the workspace's pinned words");

struct SmallArgs {
  const uint32_t *row_start, *edge_dst, *edge_data;
  uint32_t *dist;
  SmallResult *res;
  uint64_t nedges;
  uint32_t nnodes, seed, delta;
  uint32_t hub;  // edges from which a vertex ends the rounds here
};

struct SmallShared {
  uint32_t dist[kSmallV];
  uint32_t queued[kSmallWords];  // vertices on the next round's list, or of this round's not yet expanded
  uint32_t far[kSmallWords];
  uint16_t list[2][kSmallList];
  uint32_t n[3];        // vertices pushed, by round mod 3
  uint32_t left;        // far vertices above the threshold
};

// Lists v in the lanes with `push` for the next round (whole wavefront).
__device__ __forceinline__ void small_list(SmallShared &sh, uint32_t nxt, uint32_t *count, const uint64_t (&m)[kInFlight],
                                           const uint32_t (&v)[kInFlight]) {
  uint32_t t = 0;
#pragma unroll
  for (int k = 0; k < kInFlight; ++k) t += (uint32_t)__builtin_popcountll(m[k]);
  if (t == 0) return;
  uint32_t pos = 0;
  if (lane_id() == 0) pos = atomicAdd(count, t);
  pos = readlane(pos, 0);
#pragma unroll
  for (int k = 0; k < kInFlight; ++k) {
    const uint32_t p = pos + lanes_below(m[k]);
    if (((m[k] >> lane_id()) & 1) && p < kSmallList) sh.list[nxt][p] = (uint16_t)v[k];
    pos += (uint32_t)__builtin_popcountll(m[k]);
  }
}

// Relaxes kInFlight edges per lane to v[k] with candidate nd[k], where act[k].
template <Algo A>
__device__ __forceinline__ void small_relax(SmallShared &sh, uint32_t nxt, uint32_t *count, uint32_t thr, const uint32_t (&v)[kInFlight],
                                            const uint32_t (&nd)[kInFlight], const bool (&act)[kInFlight]) {
  uint32_t old[kInFlight], was[kInFlight];
  uint64_t m[kInFlight];
#pragma unroll
  for (int k = 0; k < kInFlight; ++k) old[k] = act[k] ? atomicMin(&sh.dist[v[k]], nd[k]) : 0u;
#pragma unroll
  for (int k = 0; k < kInFlight; ++k) {
    const uint32_t bit = 1u << (v[k] & 31);
    was[k] = bit;
    if (act[k] && nd[k] < old[k]) {
      if (A == Algo::BFS || nd[k] <= thr) was[k] = atomicOr(&sh.queued[v[k] >> 5], bit) & bit;
      else atomicOr(&sh.far[v[k] >> 5], bit);
    }
  }
#pragma unroll
  for (int k = 0; k < kInFlight; ++k) m[k] = __ballot(was[k] == 0);
  small_list(sh, nxt, count, m, v);
}

// Expands v in the lanes with `valid` (whole wavefront).  Its queued bit goes
// first: a lowering that finds it still set is seen by the read of the distance
// behind it, one that does not lists v again.
template <Algo A>
__device__ __forceinline__ void small_expand(const SmallArgs &a, SmallShared &sh, uint32_t nxt, uint32_t *count, uint32_t thr,
                                             bool valid, uint32_t v) {
  uint32_t d = kInf;
  if (valid) {
    atomicAnd(&sh.queued[v >> 5], ~(1u << (v & 31)));
    asm volatile("" ::: "memory");
    d = *(volatile uint32_t *)&sh.dist[v];
  } else {
    v = 0;
  }
  const uint64_t rb = ld_pair(a.row_start + v);
  const uint32_t rs = (uint32_t)rb, deg = valid ? (uint32_t)(rb >> 32) - rs : 0u;
  const bool heavy = deg > kSmallHeavy;
  const uint32_t ldeg = heavy ? 0u : deg;
  for (uint32_t j = 0; __ballot(j < ldeg); j += kInFlight) {
    uint32_t u[kInFlight], nd[kInFlight];
    bool act[kInFlight];
    const uint32_t base = j < ldeg ? rs + j : 0u;
    if (base + kInFlight <= a.nedges) {
      const uint4 dq = ld_quad(a.edge_dst + base);
      u[0] = dq.x, u[1] = dq.y, u[2] = dq.z, u[3] = dq.w;
      if (A == Algo::SSSP) {
        const uint4 wq = ld_quad(a.edge_data + base);
        nd[0] = d + wq.x, nd[1] = d + wq.y, nd[2] = d + wq.z, nd[3] = d + wq.w;
      }
    } else {  // the last edges of the array
#pragma unroll
      for (int k = 0; k < kInFlight; ++k) {
        const uint32_t e = (uint32_t)min<uint64_t>(base + k, a.nedges - 1);
        u[k] = glb(a.edge_dst)[e];
        if (A == Algo::SSSP) nd[k] = d + glb(a.edge_data)[e];
      }
    }
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      if (A == Algo::BFS) nd[k] = d + 1u;
      act[k] = j + k < ldeg;
    }
    small_relax<A>(sh, nxt, count, thr, u, nd, act);
  }
  for (uint64_t hm = __ballot(heavy); hm; hm &= hm - 1) {
    const uint32_t l = (uint32_t)__builtin_ctzll(hm);
    const uint32_t hd = readlane(d, l), hrs = readlane(rs, l), hre = hrs + readlane(deg, l);
    if (hre - hrs >= a.hub && lane_id() == 0) atomicAdd(count, kSmallV);  // more than a list holds
    for (uint32_t j = hrs; j < hre; j += kWave * kInFlight) {
      uint32_t u[kInFlight], nd[kInFlight];
      bool act[kInFlight];
#pragma unroll
      for (int k = 0; k < kInFlight; ++k) {
        const uint32_t e = j + (uint32_t)k * kWave + lane_id();
        act[k] = e < hre;
        u[k] = glb(a.edge_dst)[act[k] ? e : hrs];
        nd[k] = hd + (A == Algo::SSSP ? glb(a.edge_data)[act[k] ? e : hrs] : 1u);
      }
      small_relax<A>(sh, nxt, count, thr, u, nd, act);
    }
  }
}

template <Algo A>
__global__ __launch_bounds__(kSmallThreads) void small_kernel(SmallArgs a) {
  __shared__ SmallShared sh;
  const uint32_t tid = threadIdx.x, words = (a.nnodes + 31) / 32;
  for (uint32_t v = tid; v < a.nnodes; v += kSmallThreads) sh.dist[v] = v == a.seed ? 0u : kInf;
  for (uint32_t i = tid; i < words; i += kSmallThreads) {
    sh.queued[i] = i == a.seed / 32 ? 1u << (a.seed % 32) : 0u;
    sh.far[i] = 0;
  }
  const uint64_t seed_row = ld_pair(a.row_start + a.seed);
  if (tid == 0) {
    const uint32_t deg = (uint32_t)(seed_row >> 32) - (uint32_t)seed_row;
    sh.list[0][0] = (uint16_t)a.seed;
    sh.n[1] = sh.n[2] = 0;
    sh.n[0] = deg >= a.hub || deg > kSmallList ? kSmallV : 1u;
  }
  // list cur, count of the round to come in n[slot], of the one after in n[slot + 1]
  uint32_t cur = 0, slot = 0, n, rounds = 0, phases = 0, in_phase = 0, since = 0;
  int64_t cd = 0, step = a.delta;
  unsigned long long items = 0;
  bool handed = false;
  __syncthreads();
  n = *(volatile uint32_t *)&sh.n[0];
  for (;;) {
    handed = n > kSmallList;
    if (handed) break;
    const uint32_t thr = (uint32_t)min(cd, (int64_t)0xFFFFFFFFll);
    slot = slot == 2 ? 0 : slot + 1;
    uint32_t *const count = &sh.n[slot];
    for (uint32_t i0 = 0; i0 < n; i0 += kSmallThreads) {
      const uint32_t i = i0 + tid;
      if (__ballot(i < n)) small_expand<A>(a, sh, cur ^ 1, count, thr, i < n, i < n ? sh.list[cur][i] : 0u);
    }
    ++rounds;
    ++since;
    in_phase += n;
    items += n;
    __syncthreads();  // every push of the round is in, and every thread has the round's count
    cur ^= 1;
    n = *(volatile uint32_t *)count;
    if (tid == 0) sh.n[slot == 0 ? 2 : slot - 1] = 0;  // of the round before: for the one after the next
    if (n == 0) {
      if (A == Algo::BFS) break;
      // Rounds of more than the workgroup: narrower phases.
      if (in_phase > since * kSmallThreads) step = max(step / 2, (int64_t)a.delta);
      in_phase = since = 0;
      const uint32_t cut = thr;
      uint32_t left;
      for (;;) {
        __syncthreads();  // n and left have been read
        if (tid == 0) sh.left = 0;
        __syncthreads();
        cd += step;
        const uint32_t t = (uint32_t)min(cd, (int64_t)0xFFFFFFFFll);
        for (uint32_t i = tid; __ballot(i < words); i += kSmallThreads) {
          uint32_t w = i < words ? sh.far[i] : 0u, keep = 0;
          while (__ballot(w != 0)) {
            const bool valid = w != 0;
            const uint32_t b = valid ? (uint32_t)__builtin_ctz(w) : 0u, v = valid ? i * 32 + b : 0u;
            w &= w - 1;
            const uint32_t d = sh.dist[v];
            const bool sel = valid && d > cut && d <= t;
            if (valid && d > t) keep |= 1u << b;
            if (sel) atomicOr(&sh.queued[v >> 5], 1u << b);
            const uint64_t m[kInFlight] = {__ballot(sel), 0, 0, 0};
            const uint32_t vv[kInFlight] = {v, 0, 0, 0};
            small_list(sh, cur, count, m, vv);
          }
          if (i < words) sh.far[i] = keep;
          if (keep) atomicAdd(&sh.left, (uint32_t)__builtin_popcount(keep));
        }
        __syncthreads();
        n = *(volatile uint32_t *)count;
        left = sh.left;
        if (n < kSmallTarget) step *= 2;
        if (left == 0 || n >= kSmallTarget) break;
      }
      if (n == 0) break;
      ++phases;
    }
  }
  for (uint32_t v = tid; v < a.nnodes; v += kSmallThreads) glb(a.dist)[v] = sh.dist[v];
  if (tid == 0) {
    SmallResult *r = a.res;
    r->items = items;
    r->rounds = rounds;
    r->phases = phases + 1ull;
    r->curdelta = cd;
    r->handed = handed;
  }
}

template <Algo A>
static int run_small(Workspace *w, const CsrView &g, uint32_t seed, const lsg_opts &o, uint32_t *dist, lsg_stats *st,
                     Resume *resume) {
  const SmallArgs a{g.row, g.dst, g.w, dist, (SmallResult *)w->pinned, g.nedges, g.nnodes, seed, A == Algo::SSSP ? (uint32_t)o.delta : 1u,
                    g.nnodes > kSmallSkewV ? kSmallHub : UINT32_MAX};
  HIPCHK(hipEventRecord(w->ev0, w->stream));
  hipLaunchKernelGGL(small_kernel<A>, dim3(1), dim3(kSmallThreads), 0, w->stream, a);
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(w->ev1, w->stream));
  HIPCHK(hipStreamSynchronize(w->stream));
  const SmallResult r = *(const SmallResult *)w->pinned;
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, w->ev0, w->ev1));
  if (st) {
    memset(st, 0, sizeof *st);
    st->ms_kernel = ms;
    st->items = r.items;
    st->near_iters = r.rounds;
    st->iterations = A == Algo::SSSP ? r.phases : r.rounds;
    st->last_delta = (int32_t)std::min<int64_t>(r.curdelta, INT32_MAX);
    st->grid_blocks = 1;
    st->block_size = (int32_t)kSmallThreads;
  }
  // (BFS's rounds are its levels: the next one's vertices are of that level)
  const uint32_t level = (uint32_t)r.rounds;
  if (A == Algo::SSSP) *resume = Resume{r.curdelta, 0u, kInf - 1u, true};
  else *resume = Resume{0, level, level, true};
  return r.handed ? kBlockFallback : LSG_OK;
}

int run_small_single(int algo, Workspace *w, const CsrView &g, uint32_t seed, const lsg_opts &o, uint32_t *dist,
                     lsg_stats *st, Resume *resume) {
  return algo == (int)Algo::SSSP ? run_small<Algo::SSSP>(w, g, seed, o, dist, st, resume)
                                 : run_small<Algo::BFS>(w, g, seed, o, dist, st, resume);
}

}  // namespace lsg
