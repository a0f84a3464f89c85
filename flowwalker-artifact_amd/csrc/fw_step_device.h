// Device pieces of a walk step that the task-table kernels (fw_walk_kernel.hip) and the table walk
// (fw_table_walk.hip) share: the streams of a step's draws, a lane's own queue of Philox words and node2vec's
// acceptance test.
#pragma once

#include "fw_device_util.h"
#include "fw_internal.h"

namespace {

constexpr uint32_t kStreamWave = 0x40000000u;  // workgroup-level combine draw
constexpr uint32_t kStreamStop = 0x80000000u;  // PPR stop draw
constexpr uint32_t kStreamAccept = 0x10000000u;  // node2vec acceptance draw of a trial
constexpr uint32_t kMaxTrials = 16384u;          // node2vec: trials per step (the trial index travels in 14 bits)
constexpr int kGroupQuartets = 4;              // quartets per lane per group (part of the sampler's definition)

// ---- node2vec: two-stage step -----------------------------------------------------------------------
// The reference evaluates the bias w * f of every neighbour (f = 1/p for the return edge, 1 for a common neighbour
// of prev and cur, 1/q otherwise: include/app.cuh:108-123), one binary search each.  Here a trial proposes a
// neighbour with probability w_i / sum w through the sampler every application shares -- no adjacency test, and
// walkers that stand on the same vertex can share the pass over its list -- and accepts it with probability
// f_i / F, F = max(1, 1/p, 1/q): ONE search in N(prev) (include/gpu_graph.cuh:97-112).  A rejected trial is
// followed by another with draws of its own (streams offset by trial << 8).  The accepted neighbour has the
// reference's law, w_i f_i / sum_j w_j f_j.

// is `target` in the ascending arr[0, size)?  (one lane on its own: the hub batch kernel, where every lane serves
// another walker)
__device__ __forceinline__ bool sorted_contains(const int32_t* __restrict__ arr, int32_t size, int32_t target) {
  int32_t l = 0, r = size - 1;
  while (l <= r) {
    const int32_t m = l + ((r - l) >> 1);
    const int32_t x = arr[m];
    if (x == target) return true;
    if (x < target) l = m + 1; else r = m - 1;
  }
  return false;
}

// Sum of the weights of the entries of the ascending list adj[0, size) that equal `target`, added in list order
// (0 when there is none): the return edges of a node2vec step.
__device__ __forceinline__ float return_weight(const int32_t* __restrict__ adj, const float* __restrict__ w, uint32_t size,
                                               int32_t target) {
  uint32_t lo = 0u, hi = size;  // first entry that is not smaller
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (adj[mid] < target) lo = mid + 1u; else hi = mid;
  }
  float sum = 0.0f;
  while (lo < size && adj[lo] == target) {
    sum = sum + w[lo];
    ++lo;
  }
  return sum;
}

// The acceptance test u * F < f of trial `trial` at (walker, step) in two halves, so that the search for the proposal
// in N(prev) is only made when its answer matters: f is 1/p for the return edge, else 1 (common neighbour) or 1/q, so a
// threshold u * F below both is accepted and one that reaches both is rejected whichever it is.  F = max(1, 1/q).
// When 1/p is larger than that (a.n2v_extra = 1/p - F > 0) the return edge's excess is a component of its own: with T
// the list's total as the sampler added it up and w_ret the weights of the entries that lead back to prev, the trial
// takes the return edge outright when u0 (F T + extra w_ret) < extra w_ret (take_prev), and otherwise the return
// edge among the proposals is always accepted.  The number of trials then does not depend on p.
struct N2vTest {
  float uF;          // u * F
  bool decided;      // no search needed
  bool accept;       // the decision when decided
  bool take_prev;    // the step goes back to the previous vertex whatever was proposed
};

// draw: gives block 0 of the trial's acceptance stream
template <typename Draw>
__device__ __forceinline__ N2vTest n2v_test(const fw_kargs& a, int32_t post, int32_t prev, uint32_t trial, float T, float w_ret,
                                            Draw draw) {
  N2vTest t;
  t.uF = 0.0f;
  t.decided = true;
  t.accept = true;
  t.take_prev = false;
  if (prev == -1 || trial == kMaxTrials - 1u) return t;
  const uint4 bits = draw();
  t.uF = u24(bits.x) * a.n2v_fmax;
  if (a.n2v_extra > 0.0f) {
    const float gx = a.n2v_extra * w_ret;
    const float gb = a.n2v_fmax * T;
    const float lhs0 = u24(bits.y) * (gb + gx);
    t.take_prev = lhs0 < gx;
    if (t.take_prev || post == prev) return t;
  } else if (post == prev) {
    t.accept = t.uF < a.inv_p;
    return t;
  }
  const float f_lo = a.inv_q < 1.0f ? a.inv_q : 1.0f;
  const float f_hi = a.inv_q < 1.0f ? 1.0f : a.inv_q;
  if (t.uF < f_lo) return t;            // accepted as a common neighbour and as any other
  t.accept = false;
  if (!(t.uF < f_hi)) return t;         // rejected as either
  t.decided = false;
  return t;
}

template <bool kLanes>
__device__ __forceinline__ N2vTest n2v_test(const fw_kargs& a, int32_t post, int32_t prev, uint32_t walker, uint32_t step,
                                            uint32_t trial, float T, float w_ret) {
  return n2v_test(a, post, prev, trial, T, w_ret,
                  [&] { return philox4x32_10<kLanes>(walker, step, kStreamAccept | (trial << 8), 0u, a.seed_lo, a.seed_hi); });
}

// the other half: `common` = the proposal is a neighbour of prev
__device__ __forceinline__ bool n2v_finish(const fw_kargs& a, const N2vTest& t, bool common) {
  return t.decided ? t.accept : t.uF < (common ? 1.0f : a.inv_q);
}

// per-lane Philox word queue (same addressing as DrawQueue, different walker in every lane)
struct LaneDraw {
  uint32_t q0 = 0, q1 = 0, q2 = 0, q3 = 0;
  uint32_t avail = 0;
  uint32_t blk = 0;
};

__device__ __forceinline__ float next_uniform_lane(LaneDraw& d, const fw_kargs& a, uint32_t walker, uint32_t step,
                                                   uint32_t stream) {
  if (d.avail == 0u) {
    const uint4 b = philox4x32_10<true>(walker, step, stream, d.blk, a.seed_lo, a.seed_hi);
    d.q0 = b.x; d.q1 = b.y; d.q2 = b.z; d.q3 = b.w;
    d.avail = 4u;
    ++d.blk;
  }
  const float u = u24(d.q0);
  d.q0 = d.q1; d.q1 = d.q2; d.q2 = d.q3;
  --d.avail;
  return u;
}

// ---- draws of a wave that works on one walker -------------------------------------------------------------

__device__ __forceinline__ uint32_t uniform_u32(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ uint32_t readlane_u32(uint32_t x, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)x, (int)l); }

// The draws of a trial, lane by lane: lanes 0 .. 47 hold blocks 0, 1, 2 of the sequences' streams (lane = block * 16 + sequence), the
// next three one block each of the streams below.
constexpr uint32_t kWaveLane = 48u, kStopLane = 49u, kAcceptLane = 50u;

__device__ __forceinline__ uint4 wave_draws(const fw_kargs& a, uint32_t walker, uint32_t step, uint32_t trial, uint32_t lane) {
  const uint32_t sbase = trial << 8;
  uint32_t stream = sbase | (lane & 15u);
  stream = lane == kWaveLane ? kStreamWave | sbase : stream;
  stream = lane == kStopLane ? kStreamStop : stream;
  stream = lane == kAcceptLane ? kStreamAccept | sbase : stream;
  return philox4x32_10<true>(walker, step, stream, lane < kWaveLane ? lane >> 4 : 0u, a.seed_lo, a.seed_hi);
}

// The uniforms of a sequence's reservoir, two per accepted group: the words of its stream in order.
struct WavePairs {
  uint4 e;       // wave_draws, later blocks of the sequence's own stream
  uint32_t seq;
  uint32_t i;    // pairs taken
};

__device__ __forceinline__ void next_pair(WavePairs& p, const fw_kargs& a, uint32_t walker, uint32_t step, uint32_t sbase,
                                          uint32_t lane, float& first, float& second) {
  uint32_t from = p.seq + 16u * (p.i >> 1);
  if (p.i >= 6u) {  // past the blocks made beforehand
    if (p.i == 6u || (p.i & 127u) == 0u) p.e = philox4x32_10<true>(walker, step, p.seq | sbase, 64u * (p.i >> 7) + lane, a.seed_lo, a.seed_hi);
    from = (p.i >> 1) & 63u;
  }
  first = u24(readlane_u32((p.i & 1u) ? p.e.z : p.e.x, from));
  second = u24(readlane_u32((p.i & 1u) ? p.e.w : p.e.y, from));
  ++p.i;
}

}  // namespace
