// Rounds of the wavefront kernels (wave.hip, bfs_do.hip): the state of a round,
// the barrier between rounds and the message that starts the next.
#pragma once

#include "wave.h"

namespace lsg {

// Rounds of at most this many items go straight to the atomicMins where a unit
// has few edges: one round trip less, and few enough atomics.
constexpr uint32_t kDirectMax = 4096;

// Roles of the three queues and the state of a round.
struct WaveRound {
  uint32_t items, heavy, round, phase;
  uint32_t steps;  // the near/far threshold, in steps of delta
  uint32_t cut;    // kWaveCut: the previous phase's
  uint32_t lead;   // the block that published the round
  uint32_t roles;  // in | near << 2 | far << 4
  uint32_t flags;
  __device__ uint32_t in_q() const { return roles & 3u; }
  __device__ uint32_t near_q() const { return roles >> 2 & 3u; }
  __device__ uint32_t far_q() const { return roles >> 4 & 3u; }
};
// kWaveCut: the round's input is the far pile; what has come below the previous
// threshold since it was pushed has been expanded as a near item already.
// kWaveWide, kWaveSplit: see WaveGrowth.
constexpr uint32_t kWaveDone = 1, kWaveCut = 2, kWaveLead = 4, kWaveLocal = 8, kWaveWide = 16, kWaveSplit = 32;
__device__ __forceinline__ uint32_t wave_roles(uint32_t in, uint32_t near, uint32_t far) {
  return in | near << 2 | far << 4;
}

// The chunks of up to 64 staged heavy items (lane i < n: degree deg of item i),
// counted along the lanes: the chunks up to and including item i's.
__device__ __forceinline__ uint32_t chunk_ends(uint32_t n, uint32_t deg, uint32_t chunk) {
  uint32_t end = lane_id() < n ? (deg - 1) / chunk + 1 : 0u;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = __shfl_up(end, d);
    if (lane_id() >= (uint32_t)d) end += y;
  }
  return end;
}

// put(f, item, k) for every chunk f in one lane: the k-th of its item.
template <class Put>
__device__ __forceinline__ void chunk_each(uint32_t end, const Put &put) {
  const uint32_t total = readlane(end, kWave - 1), prev = (uint32_t)__shfl_up(end, 1);
  const uint32_t start = lane_id() == 0 ? 0u : prev;
  for (uint32_t f0 = 0; f0 < total; f0 += kWave) {
    const uint32_t f = f0 + lane_id();
    uint32_t item = 0;  // items whose chunks end at or before f
#pragma unroll
    for (uint32_t d = kWave / 2; d >= 1; d >>= 1)
      if ((uint32_t)__shfl(end, item + d - 1) <= f) item += d;
    const uint32_t k = f - (uint32_t)__shfl(start, item);
    if (f < total) put(f, item, k);
  }
}

// Clears the words that the kernels share (tid / nt: the caller's place in one block).
__device__ __forceinline__ void wave_reset(WaveCtrl *wc, uint32_t tid, uint32_t nt) {
  uint32_t *const p = reinterpret_cast<uint32_t *>(wc);
  for (uint32_t i = tid; i < sizeof(WaveCtrl) / 4; i += nt) p[i] = 0;
}

// ---- between rounds -------------------------------------------------------------

// Wavefront 0 of the block with number `seat` of `parties` arrives; true in the
// last.  In groups of kBarGroup, as barrier_arrive; one level where one group
// is enough.
__device__ __forceinline__ bool wave_arrive(WaveCtrl::Slot *slot, uint32_t seat, uint32_t parties) {
  uint32_t last = 0;
  if (lane_id() == 0) {
    const uint32_t grp = seat / kBarGroup, size = min(kBarGroup, parties - grp * kBarGroup);
    last = atomic_add(&slot->arrive[grp].n, 1u) + 1 == size;
    if (last && parties > kBarGroup)
      last = atomic_add(&slot->top.n, 1u) + 1 == (parties + kBarGroup - 1) / kBarGroup;
  }
  return readlane(last, 0) != 0;
}

// Wavefront 0 waits for the message of a generation after `gen` (bounded by
// spin_limit without progress): the round in x, and its generation.
__device__ __forceinline__ uint32_t wave_wait(const WaveArgs &a, uint32_t gen, WaveRound &x) {
  const uint32_t lane = lane_id();
  const uint64_t *const p =
      lane < kWaveMsg ? &a.wc->msg[lane] : reinterpret_cast<const uint64_t *>(&a.ctrl->abort);  // abort, checkin
  uint64_t t0 = wall_clock64();
  uint32_t seen = ld_coh(&a.ctrl->progress), tag;
  uint32_t hi, flags = kWaveDone;
  for (;;) {
    const uint64_t m = ld_coh64(p);
    const uint32_t lo = (uint32_t)m;
    hi = (uint32_t)(m >> 32);
    tag = readlane(lo, 0);
    if (tag != gen && __ballot(lane < kWaveMsg && lo != tag) == 0) {
      flags = (readlane(hi, 6) >> 6 & (kWaveDone | kWaveCut)) | (readlane(hi, 6) >> 26 & (kWaveWide | kWaveSplit));
      break;
    }
    if (readlane(lo, kWaveMsg) != kAbortNone) break;
    if (wall_clock64() - t0 > a.spin_limit) {
      // the leading block may be running rounds on its own
      const uint32_t now = ld_coh(&a.ctrl->progress);
      if (now == seen) {
        st_coh(&a.ctrl->abort, kAbortTimeout);
        break;
      }
      seen = now;
      t0 = wall_clock64();
    }
    __builtin_amdgcn_s_sleep(1);
  }
  x.items = readlane(hi, 0);
  x.heavy = readlane(hi, 1);
  x.round = readlane(hi, 2);
  x.phase = readlane(hi, 3);
  x.steps = readlane(hi, 4);
  x.cut = readlane(hi, 5);
  x.roles = readlane(hi, 6) & 0x3fu;
  x.lead = readlane(hi, 6) >> 8 & 0x3fffffu;
  x.flags = flags;
  order_acquire();
  return tag;
}

// Wavefront 0 publishes round x as generation `tag`.
__device__ __forceinline__ void wave_publish(WaveCtrl *wc, uint32_t tag, const WaveRound &x) {
  const uint32_t m[kWaveMsg] = {x.items, x.heavy, x.round, x.phase, x.steps, x.cut,
                                (x.flags & (kWaveWide | kWaveSplit)) << 26 | x.lead << 8 |
                                    (x.flags & (kWaveDone | kWaveCut)) << 6 | x.roles};
  uint32_t v = 0;
#pragma unroll
  for (int i = 0; i < kWaveMsg; ++i)
    if (lane_id() == (uint32_t)i) v = m[i];
  if (lane_id() < kWaveMsg) st_coh64(&wc->msg[lane_id()], (uint64_t)v << 32 | tag);
}

}  // namespace lsg
