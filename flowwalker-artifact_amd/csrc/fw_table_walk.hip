// List tables and the walk over them.
//
// A sampling step of fw_walk_kernel.hip reads a whole neighbour list, and everything it computes from it -- the scan of a
// group of 1024 biases, the group totals, their running sums -- is the same for every walker that ever stands there; a
// walker contributes two uniforms per accepted group.  When the walkers of a call would read the lists many times over,
// the walker-independent part is made once (one pass over the edges: 8 bytes read and 8 written per edge) and a step
// becomes a few look-ups, so one lane walks one walker from its start to its end: no task table, no parking, no sorting
// (fw_table_walk; calls of few walkers, but for MetaPath, take a wave for each: fw_table_walk_wave).
// The sampler's definition (fw_walk_kernel.hip) is untouched: the tables hold the very sums, prefixes and totals the streaming
// kernels compute, in their order of additions, and the walk takes the same draws, so every walker gets the same vertex.
//
// Reference behaviour: as fw_walk_kernel.hip (include/walker.cuh:1307-1580, include/sampler.cuh:46-200).
//
// Layout.  vrec[v] = {region, degree, total, CSR offset}: `region` in blocks of 128 bytes (the memory's request size) into
// `data`, `total` = the list's total as the step's sampler adds it up.  A region, in units of 32 bytes:
//   list of one group (at most 256 aligned quartets):  the entries, then, but for lists of at most 16 quartets, row M
//   longer list:  header (sums), then per group {entries, row M (8 units)}
//   row M: for every lane of the group (a lane holds up to four quartets) the running maximum of the positive lanes' prefixes;
//     from the last positive lane on +inf.  The sampler picks the first lane whose prefix exceeds the target, or else the last positive lane:
//     the first entry above the target.
//   entries: lane after lane, for each of its elements a pair {key, neighbour}, 16 pairs a block.  Inside its lane the sampler picks the first element whose
//     running sum exceeds the target, or else the last positive one; key = that running sum, for an element without bias the one before it, from the
//     lane's last positive element on +inf, and all of it not below row M's entry of the lane before nor above the lane's own.  So the keys of
//     a whole group never decrease, and the element is the first one whose key is above the target.
//   Where the weights are close to evenly spread over a group the walk looks for that element from the proportional guess on and row M is not read: the
//   block of the guess holds it for 65 % (1024 weights from 1 to 100) to 95 % of the targets, one next to it nearly always.  So a step reads some 1.4 blocks of
//   a group, with row M it read 2.2 (DeepWalk R-MAT 24, symmetrised: 2.50e9 -> 1.72e9 blocks in all, 47.4 -> 32.8 ms, of which
//   1.84e9 and 35.5 while its blocks were kept in the L2).  A group whose weights are not (uneven_group)
//   has the sign of its total set, or in a list of one group the top bit of `region`, and is entered through row M.  Of a full group that is one or two of row M's
//   blocks and one of pairs; otherwise row M, which begins where the entries end, may lie in three blocks and a lane's pairs in two.
//   sums: blocks of 16 running sums of a sequence's groups and their 16 totals, every sequence from a block of its own, filled up
//     with the last sum; with more than one sequence (workgroup granularity) a block in front: the inclusive scan of the
//     sequences' totals, as keys like the above (16 floats).
// All keys of a row or a group never decrease, so any search finds the same entry.

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fw_internal.h"
#include "fw_step_device.h"

namespace {

constexpr uint32_t kGq = 64u * kGroupQuartets;  // quartets of a full group
constexpr uint32_t kGroupUnits = kGq + 8u;      // units of a group in a list of several: the entries of 64 lanes and row M
constexpr uint32_t kNoRow = 16u;                // quartets of a list without row M: its entries are at most four blocks
constexpr uint32_t kUneven = 0x80000000u;       // in vrec's region: row M first
constexpr float kInf = __builtin_inff();
// Waves per SIMD of the walk: 4, 5, 6 and 8 were measured while a step read row M (DeepWalk R-MAT 24 47.9 / 49.1 / 50.0 / 72.1 ms, the last
// one with spilled registers; R-MAT 22 6.8 / 6.8 / 7.0 / 11.3): more walkers in flight only compete for the caches.
constexpr int kWaves = 4;

typedef float f4_at4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint32_t list_quartets(uint32_t off, uint32_t deg) { return ((off & 3u) + deg + 3u) >> 2; }

// blocks of sums of one sequence of a list of `ngroups` groups (the longest sequence has ceil(ngroups / sequences))
__device__ __forceinline__ uint32_t seq_blocks(uint32_t ngroups, bool wg, uint32_t nw_shift) {
  const uint32_t most = wg ? (ngroups + (1u << nw_shift) - 1u) >> nw_shift : ngroups;
  return (most + 15u) >> 4;
}

// units of a long list's header
__device__ __forceinline__ uint32_t header_units(uint32_t ngroups, bool wg, uint32_t nw_shift) {
  const uint32_t nb = seq_blocks(ngroups, wg, nw_shift);
  return 4u * (wg ? 1u + (nb << nw_shift) : nb);
}

__device__ __forceinline__ uint32_t region_blocks(uint32_t off, uint32_t deg, bool wg, uint32_t nw_shift) {
  if (deg == 0u) return 0u;
  const uint32_t nq = list_quartets(off, deg);
  uint32_t units;
  if (nq <= kGq) {
    units = nq + (nq <= kNoRow ? 0u : (nq < 64u ? (nq + 7u) >> 3 : 8u));
  } else {
    const uint32_t ngroups = (nq + kGq - 1u) / kGq;
    units = header_units(ngroups, wg, nw_shift) + nq + 8u * ngroups;
  }
  return (units + 3u) >> 2;
}

// blocks of a long list's region in MetaPath's tables: its totals, per label its sums, per group the ends of its labels
__device__ __forceinline__ uint32_t label_region_blocks(uint32_t off, uint32_t deg, bool wg, uint32_t nw_shift, uint32_t n_labels) {
  const uint32_t nq = list_quartets(off, deg);
  if (nq <= kGq) return 0u;
  const uint32_t ngroups = (nq + kGq - 1u) / kGq;
  return 1u + n_labels * (header_units(ngroups, wg, nw_shift) >> 2) + ((ngroups + 7u) >> 3);
}

// ---- making the tables --------------------------------------------------------------------------------

// Region sizes (scanned into positions afterwards) and the work lists of the lists longer than a group: `longs` their
// vertices, `items` {vertex, group} for every group of them.  ctrs: [0] long lists, [1] items.  Every workgroup counts its
// range of vertices first, so that it takes its places in the work lists with one update each.
__global__ __launch_bounds__(1024) void fw_table_plan_kernel(const uint32_t* __restrict__ xadj, int32_t V, int32_t hub_threshold,
                                                             uint32_t nw_shift, uint32_t n_labels, uint32_t* __restrict__ blocks,
                                                             uint32_t* longs, uint2* items, uint32_t* ctrs) {
  __shared__ uint32_t s_n[2], s_at[2];
  if (threadIdx.x < 2u) s_n[threadIdx.x] = 0u;
  __syncthreads();
  const uint32_t per = ((uint32_t)V + gridDim.x - 1u) / gridDim.x;
  const uint32_t v0 = blockIdx.x * per;
  const uint32_t v1 = v0 + per < (uint32_t)V ? v0 + per : (uint32_t)V;
  uint32_t n_long = 0u, n_items = 0u;
  for (uint32_t v = v0 + threadIdx.x; v < v1; v += blockDim.x) {
    const uint32_t off = xadj[v], deg = xadj[v + 1] - off;
    const bool wg = (int32_t)deg > hub_threshold;
    blocks[v] = n_labels != 0u ? label_region_blocks(off, deg, wg, nw_shift, n_labels) : region_blocks(off, deg, wg, nw_shift);
    const uint32_t nq = list_quartets(off, deg);
    if (nq > kGq) {
      ++n_long;
      n_items += (nq + kGq - 1u) / kGq;
    }
  }
  if (n_long != 0u) {
    atomicAdd(&s_n[0], n_long);
    atomicAdd(&s_n[1], n_items);
  }
  __syncthreads();
  if (threadIdx.x < 2u) s_at[threadIdx.x] = s_n[threadIdx.x] != 0u ? atomicAdd(&ctrs[threadIdx.x], s_n[threadIdx.x]) : 0u;
  if (blockIdx.x == 0u && threadIdx.x == 0u) blocks[V] = 0u;
  __syncthreads();
  if (s_n[0] == 0u) return;
  for (uint32_t v = v0 + threadIdx.x; v < v1; v += blockDim.x) {
    const uint32_t off = xadj[v], deg = xadj[v + 1] - off;
    const uint32_t nq = list_quartets(off, deg);
    if (nq > kGq) {
      const uint32_t ngroups = (nq + kGq - 1u) / kGq;
      longs[atomicAdd(&s_at[0], 1u)] = v;
      const uint32_t at = atomicAdd(&s_at[1], ngroups);
      for (uint32_t g = 0; g < ngroups; ++g) items[at + g] = make_uint2(v, g);
    }
  }
}

// The 4 kJ biases and neighbours of lane `lane` in the group of `nqg` quartets that starts at quartet kb of a list (an entry outside the
// list has no bias).  Sets `bad` when a bias is negative or not a number.
template <int kJ>
__device__ __forceinline__ void load_lane(const float* __restrict__ weight, const int32_t* __restrict__ adjncy, uint32_t off,
                                          uint32_t deg, uint32_t kb, uint32_t nqg, uint32_t lane, float (&x)[4 * kJ],
                                          int32_t (&nb)[4 * kJ], bool& bad) {
  const uint32_t a0 = off & ~3u;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const uint32_t k = lane + 64u * (uint32_t)j;
    float4 w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int4 n = make_int4(-1, -1, -1, -1);
    const uint32_t base = a0 + 4u * (kb + k);
    if (k < nqg) {
      w = *reinterpret_cast<const float4*>(weight + base);
      n = *reinterpret_cast<const int4*>(adjncy + base);
    }
    const uint32_t li = base - off;  // wraps below 0 for the head quartet
    const uint32_t lim = k < nqg ? deg : 0u;
    x[4 * j + 0] = li < lim ? w.x : 0.0f;
    x[4 * j + 1] = li + 1u < lim ? w.y : 0.0f;
    x[4 * j + 2] = li + 2u < lim ? w.z : 0.0f;
    x[4 * j + 3] = li + 3u < lim ? w.w : 0.0f;
    nb[4 * j + 0] = li < lim ? n.x : -1;
    nb[4 * j + 1] = li + 1u < lim ? n.y : -1;
    nb[4 * j + 2] = li + 2u < lim ? n.z : -1;
    nb[4 * j + 3] = li + 3u < lim ? n.w : -1;
  }
#pragma unroll
  for (int i = 0; i < 4 * kJ; ++i) bad = bad || !(x[i] >= 0.0f);
}

// The first quartet of lane `lane` among the entries of a group of nqg quartets: the quartets lane, lane + 64, ... of the group, for lane after lane.
__device__ __forceinline__ uint32_t lane_start(const uint32_t lane, const uint32_t nqg) {
  const uint32_t J = (nqg + 63u) >> 6, full = nqg - 64u * (J - 1u);  // lanes with J quartets, the others have one less
  return J * lane - (lane > full ? lane - full : 0u);
}

// The lane's pairs: e0 = its prefix before its own elements, below and above = row M's entries of the lane before and of its own.  The first n of its
// kJ quartets are stored.
template <int kJ>
__device__ __forceinline__ void store_lane(uint2* out, uint32_t n, float e0, float below, float above, const float (&x)[4 * kJ],
                                           const int32_t (&nb)[4 * kJ]) {
  uint32_t pm = 0u;
#pragma unroll
  for (int i = 0; i < 4 * kJ; ++i) pm |= (x[i] > 0.0f ? 1u : 0u) << i;
  const int last = 31 - __builtin_clz(pm | 1u);
  float e = e0, key = 0.0f;
  uint4* o = reinterpret_cast<uint4*>(out);
#pragma unroll
  for (int i = 0; i < 4 * kJ; i += 2) {
    uint32_t k[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      e = e + x[i + b];
      key = x[i + b] > 0.0f ? e : key;
      float g = pm != 0u && i + b >= last ? kInf : key;
      g = g < below ? below : g;
      k[b] = __float_as_uint(g > above ? above : g);
    }
    if ((uint32_t)i < 4u * n) o[i >> 1] = make_uint4(k[0], (uint32_t)nb[i], k[1], (uint32_t)nb[i + 1]);
  }
}

// Whether a group is entered through row M: a quarter of its lanes end more than 20 pairs from where even weights would have them, or one in 32 more than
// three blocks.  M: the running maximum of the positive lanes' prefixes; lanes: the nl lanes of the group's segment.
// A wave's walkers wait for the one that looks most often, and row M is two reads more for all of them.  16 / 20 / 24 pairs, us: 50,000 DeepWalk walkers, weights log-normal
// with sigma 1 on R-MAT 12 204 / 186 / 183, sigma 2 on R-MAT 20 414 / 424 / 440, Pareto 1.5 on R-MAT 16 360 / 370 / 381, even (1 to 100) on R-MAT 20 379 / 369 / 365.
// Without / with the second condition, 100,000 walkers on lists of 1000 of whose 64 lanes twelve have next to nothing and the one among them the share of all: 688 / 470; the
// others as before.  (Even weights: 278.)
__device__ __forceinline__ bool uneven_group(const float M, const float T, const uint32_t c, const uint32_t nqg, const uint64_t lanes, const uint32_t nl) {
  const float d = M * (float)(4u * nqg) - T * (float)(4u * lane_start(c + 1u, nqg));
  const uint32_t off = (uint32_t)__builtin_popcountll(__ballot(!(__builtin_fabsf(d) <= 20.0f * T)) & lanes);
  const uint32_t far = (uint32_t)__builtin_popcountll(__ballot(!(__builtin_fabsf(d) <= 48.0f * T)) & lanes);
  return 4u * off > nl || 32u * far > nl;
}

// One list of at most kSeg quartets per segment of kSeg lanes (one or two DPP rows, or the wave); off, deg, region are the
// segment's.  Returns the list's total in every lane of the segment, with its sign set for an uneven list.  The scan network is the packed step's.
template <int kSeg>
__device__ __forceinline__ float table_segment(const float* __restrict__ weight, const int32_t* __restrict__ adjncy, uint32_t off,
                                               uint32_t deg, unsigned char* region, int lane, bool& bad) {
  const uint32_t c = (uint32_t)lane & (uint32_t)(kSeg - 1);
  const uint32_t nq = deg != 0u ? list_quartets(off, deg) : 0u;
  float x[4];
  int32_t nb[4];
  load_lane<1>(weight, adjncy, off, deg, 0u, nq, c, x, nb, bad);
  float q = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) q = q + x[i];
  float I = row_scan(q);
  if (kSeg >= 32) I = dpp_add_bcast15(I);
  if (kSeg == 64) I = dpp_add_bcast31(I);
  const bool pos = q > 0.0f;
  float M = pos ? I : 0.0f;
  M = dpp_max<0x111, 0xF>(M);
  M = dpp_max<0x112, 0xF>(M);
  M = dpp_max<0x114, 0xF>(M);
  M = dpp_max<0x118, 0xF>(M);
  if (kSeg >= 32) M = dpp_max<0x142, 0xA>(M);
  if (kSeg == 64) M = dpp_max<0x143, 0xC>(M);
  const float T = bperm_f((lane | (kSeg - 1)) << 2, I);
  const uint64_t mpos = __ballot(pos) >> (lane & ~(kSeg - 1));
  const uint64_t mine = kSeg == 64 ? mpos : (mpos & ((1ull << (kSeg & 63)) - 1ull));
  const uint32_t lastpos = 63u - (uint32_t)__builtin_clzll(mine | 1ull);
  const int seg = lane & ~(kSeg - 1);
  bool uneven = false;
  if (kSeg > 16) uneven = uneven_group(M, T, c, nq, (nq < 64u ? (1ull << nq) - 1ull : ~0ull) << seg, nq);
  M = c >= lastpos ? kInf : M;
  const float prev = bperm_f((lane - 1) << 2, M);
  if (nq > kNoRow && c < ((nq + 7u) & ~7u)) reinterpret_cast<float*>(region + 32u * nq)[c] = M;
  if (c < nq) store_lane<1>(reinterpret_cast<uint2*>(region + 32u * c), 1u, I - q, c != 0u ? prev : 0.0f, M, x, nb);
  return uneven ? -T : T;
}

// One group of more than 64 quartets or of a long list, by a whole wave.  Returns its total, with its sign set for an uneven group.
__device__ __forceinline__ float table_group(const float* __restrict__ weight, const int32_t* __restrict__ adjncy, uint32_t off,
                                             uint32_t deg, uint32_t kb, uint32_t nqg, unsigned char* entries, int lane,
                                             bool& bad) {
  constexpr int kEl = 4 * kGroupQuartets;
  float x[kEl];
  int32_t nb[kEl];
  load_lane<kGroupQuartets>(weight, adjncy, off, deg, kb, nqg, (uint32_t)lane, x, nb, bad);
  float q = 0.0f;
#pragma unroll
  for (int i = 0; i < kEl; ++i) q = q + x[i];
  const float I = wave_scan(q);
  const bool pos = q > 0.0f;
  float M = wave_prefix_max(pos ? I : 0.0f);
  const uint32_t lastpos = 63u - (uint32_t)__builtin_clzll(__ballot(pos) | 1ull);
  const uint32_t nl = nqg < 64u ? nqg : 64u;
  const float T = readlane_f(I, 63);
  const bool uneven = uneven_group(M, T, (uint32_t)lane, nqg, nl < 64u ? (1ull << nl) - 1ull : ~0ull, nl);
  M = (uint32_t)lane >= lastpos ? kInf : M;
  const float prev = bperm_f((lane - 1) << 2, M);
  reinterpret_cast<float*>(entries + 32u * nqg)[lane] = M;
  if ((uint32_t)lane < nl) {
    const uint32_t at = lane_start((uint32_t)lane, nqg);
    store_lane<kGroupQuartets>(reinterpret_cast<uint2*>(entries + 32u * at), lane_start((uint32_t)lane + 1u, nqg) - at, I - q,
                               lane != 0 ? prev : 0.0f, M, x, nb);
  }
  return uneven ? -T : T;
}

// Lists of one group: a wave takes 64 consecutive vertices; lists of at most 16 (32) quartets four (two) at a time, the others
// one after the other.  vrec of the wave's vertices is stored together at the end (long lists get their total from
// fw_table_sums_kernel).  base: region positions.
// Bound: memory (8 bytes read and about 9 written per edge; one pass).
__global__ __launch_bounds__(256) void fw_table_lists_kernel(const uint32_t* __restrict__ xadj, const int32_t* __restrict__ adjncy,
                                                             const float* __restrict__ weight, int32_t V,
                                                             const uint32_t* __restrict__ base, uint4* vrec, unsigned char* data,
                                                             uint32_t* flag) {
  __shared__ float s_total[4][64];
  const int lane = lane_id();
  const int wave = (int)(threadIdx.x >> 6);
  const uint64_t chunks = ((uint64_t)(uint32_t)V + 63u) >> 6;
  bool bad = false;
  for (uint64_t ch = (uint64_t)blockIdx.x * 4u + (uint64_t)wave; ch < chunks; ch += (uint64_t)gridDim.x * 4u) {
    const uint32_t v = (uint32_t)(ch * 64u) + (uint32_t)lane;
    const bool have = v < (uint32_t)V;
    uint32_t off = 0u, deg = 0u, reg = 0u;
    if (have) {
      off = xadj[v];
      deg = xadj[v + 1] - off;
      reg = base[v];
    }
    const uint32_t nq = deg != 0u ? list_quartets(off, deg) : 0u;
    s_total[wave][lane] = 0.0f;
    uint64_t m = __ballot(nq != 0u && nq <= 16u);
    while (m != 0ull) {
      int src = -1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int l = m != 0ull ? __builtin_ctzll(m) : -1;
        m &= m - 1ull;
        src = (lane >> 4) == r ? l : src;
      }
      const int from = src < 0 ? 0 : src;
      const uint32_t o = __shfl(off, from), df = __shfl(deg, from), g = __shfl(reg, from);  // every lane takes part
      const uint32_t d = src < 0 ? 0u : df;
      const float T = table_segment<16>(weight, adjncy, o, d, data + (uint64_t)g * 128u, lane, bad);
      if (src >= 0 && (lane & 15) == 0) s_total[wave][src] = T;
    }
    m = __ballot(nq > 16u && nq <= 32u);
    while (m != 0ull) {
      int src = -1;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int l = m != 0ull ? __builtin_ctzll(m) : -1;
        m &= m - 1ull;
        src = (lane >> 5) == r ? l : src;
      }
      const int from = src < 0 ? 0 : src;
      const uint32_t o = __shfl(off, from), df = __shfl(deg, from), g = __shfl(reg, from);  // every lane takes part
      const uint32_t d = src < 0 ? 0u : df;
      const float T = table_segment<32>(weight, adjncy, o, d, data + (uint64_t)g * 128u, lane, bad);
      if (src >= 0 && (lane & 31) == 0) s_total[wave][src] = T;
    }
    for (m = __ballot(nq > 32u && nq <= 64u); m != 0ull; m &= m - 1ull) {
      const int l = __builtin_ctzll(m);
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, l), d = (uint32_t)__builtin_amdgcn_readlane((int)deg, l);
      const uint32_t g = (uint32_t)__builtin_amdgcn_readlane((int)reg, l);
      const float T = table_segment<64>(weight, adjncy, o, d, data + (uint64_t)g * 128u, lane, bad);
      if (lane == 0) s_total[wave][l] = T;
    }
    for (m = __ballot(nq > 64u && nq <= kGq); m != 0ull; m &= m - 1ull) {
      const int l = __builtin_ctzll(m);
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, l), d = (uint32_t)__builtin_amdgcn_readlane((int)deg, l);
      const uint32_t g = (uint32_t)__builtin_amdgcn_readlane((int)reg, l);
      const float T = table_group(weight, adjncy, o, d, 0u, list_quartets(o, d), data + (uint64_t)g * 128u, lane, bad);
      if (lane == 0) s_total[wave][l] = T;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float total = s_total[wave][lane];
    bad = bad || !(__builtin_fabsf(total) < kInf);
    if (have) vrec[v] = make_uint4(reg | (total < 0.0f ? kUneven : 0u), deg, __float_as_uint(__builtin_fabsf(total)), off);
    __builtin_amdgcn_wave_barrier();
  }
  if (__ballot(bad) != 0ull && lane == 0) *flag = 1u;
}

// The groups of the long lists, one wave per group.  Group totals go to the list's sums.
__global__ __launch_bounds__(256) void fw_table_groups_kernel(const uint4* __restrict__ vrec, const int32_t* __restrict__ adjncy,
                                                              const float* __restrict__ weight, const uint2* __restrict__ items,
                                                              uint32_t n_items, int32_t hub_threshold, uint32_t nw_shift,
                                                              unsigned char* data, uint32_t* flag) {
  const int lane = lane_id();
  bool bad = false;
  for (uint32_t it = blockIdx.x * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); it < n_items;
       it += gridDim.x * 4u) {
    const uint2 item = items[it];
    const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)item.x), g = (uint32_t)__builtin_amdgcn_readfirstlane((int)item.y);
    const uint4 rec = vrec[v];
    const uint32_t off = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec.w), deg = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec.y);
    unsigned char* const region = data + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)rec.x) * 128u;
    const uint32_t nq = list_quartets(off, deg);
    const uint32_t ngroups = (nq + kGq - 1u) / kGq;
    const bool wg = (int32_t)deg > hub_threshold;
    const uint32_t left = nq - g * kGq;
    unsigned char* const entries = region + (uint64_t)32u * (header_units(ngroups, wg, nw_shift) + kGroupUnits * g);
    const float T = table_group(weight, adjncy, off, deg, g * kGq, left < kGq ? left : kGq, entries, lane, bad);
    const uint32_t k = wg ? g >> nw_shift : g;
    const uint32_t block = wg ? 1u + (g & ((1u << nw_shift) - 1u)) * seq_blocks(ngroups, wg, nw_shift) + (k >> 4) : k >> 4;
    if (lane == 0) reinterpret_cast<float*>(region)[32u * block + 16u + (k & 15u)] = T;
  }
  if (__ballot(bad) != 0ull && lane == 0) *flag = 1u;
}

// The running sums of a list, from its groups' totals: at wave granularity one sequence (64 totals at a time, added up
// in order), at workgroup granularity one sequence per lane and the scan of their totals.  Returns the list's total.
__device__ __forceinline__ float list_sums(float* region, uint32_t ngroups, bool wg, uint32_t nw_shift, int lane) {
  const uint32_t nb = seq_blocks(ngroups, wg, nw_shift);
  float total;
  if (wg) {
    const uint32_t nw = 1u << nw_shift;
    float S = 0.0f;
    if ((uint32_t)lane < nw) {
      float* const sums = region + 32u + 32u * nb * (uint32_t)lane;
      const uint32_t L = (ngroups >> nw_shift) + ((uint32_t)lane < (ngroups & (nw - 1u)) ? 1u : 0u);
      for (uint32_t k = 0; k < 16u * nb; ++k) {
        float* const at = sums + 32u * (k >> 4) + (k & 15u);
        if (k < L) S = S + __builtin_fabsf(at[16]);  // (the sign: see the layout)
        at[0] = S;
      }
    }
    const float J = row_scan(S);
    total = readlane_f(J, (int)nw - 1);
    const uint64_t mpos = __ballot(S > 0.0f);
    const uint32_t lastpos = 63u - (uint32_t)__builtin_clzll(mpos | 1ull);
    const float key = wave_prefix_max(S > 0.0f ? J : 0.0f);
    if (lane < 16) region[lane] = (uint32_t)lane >= lastpos ? kInf : key;
  } else {
    float S = 0.0f;
    for (uint32_t g0 = 0; g0 < 16u * nb; g0 += 64u) {
      const uint32_t g = g0 + (uint32_t)lane;
      float* const at = region + 32u * (g >> 4) + (g & 15u);
      const float T = g < ngroups ? __builtin_fabsf(at[16]) : 0.0f;
      float mine = 0.0f;
#pragma unroll 8
      for (int l = 0; l < 64; ++l) {
        S = S + readlane_f(T, l);  // + 0 past the end changes nothing
        mine = lane == l ? S : mine;
      }
      if (g < 16u * nb) at[0] = mine;
    }
    total = S;
  }
  return total;
}

// The long lists, one wave per list.
__global__ __launch_bounds__(256) void fw_table_sums_kernel(uint4* __restrict__ vrec, const uint32_t* __restrict__ longs, uint32_t n_longs,
                                                            int32_t hub_threshold, uint32_t nw_shift, unsigned char* data, uint32_t* flag) {
  const int lane = lane_id();
  bool bad = false;
  for (uint32_t it = blockIdx.x * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); it < n_longs;
       it += gridDim.x * 4u) {
    const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)longs[it]);
    const uint4 rec = vrec[v];
    const uint32_t ngroups = (list_quartets(rec.w, rec.y) + kGq - 1u) / kGq;
    float* const region = reinterpret_cast<float*>(data + (uint64_t)rec.x * 128u);
    const bool wg = (int32_t)rec.y > hub_threshold;
    const float total = list_sums(region, ngroups, wg, nw_shift, lane);
    bad = bad || !(total < kInf);
    if (lane == 0) vrec[v].z = __float_as_uint(total);
  }
  if (__ballot(bad) != 0ull && lane == 0) *flag = 1u;
}

// ---- hash sets (node2vec) -----------------------------------------------------------------------------
//
// node2vec asks whether the proposal is a neighbour of the previous vertex, and for a large 1/p what the entries that lead
// back weigh.  A binary search answers with a chain of some ten dependent reads that scatter over the list (most of what a step
// cost: R-MAT 24 spent 41 of 89 ms on it); a hash set answers with one read of 64 bytes.  Every list has a set of its own, half full on
// average: one entry per distinct neighbour, in the bucket its hash names, -1 in free places.  A bucket more than 16
// neighbours fall into (one in some hundred) says so, and its walkers search the list as before.

constexpr int32_t kSetOverflow = (int32_t)0x80000000;  // in the last place of a bucket
constexpr uint32_t kSetPart = 1040u;    // buckets a workgroup makes at a time, for every eight groups of a long list: the parts
                                        // of a list of d > 1020 entries, ceil(groups / 8) of them, cover its d / 8 + 1 buckets
constexpr uint32_t kSetSmall = 1024u / 8u + 1u;  // buckets of a list of one group

__device__ __forceinline__ uint32_t set_bucket(int32_t neighbour, uint32_t buckets) {
  // xxHash32's first two primes (Y. Collet) with the first fold of its finish between them: R-MAT ids differ in few bits, and the
  // high bits, which pick the bucket, take all of them in
  uint32_t h = (uint32_t)neighbour * 0x9E3779B1u;
  h = (h ^ (h >> 15)) * 0x85EBCA77u;
  return __umulhi(h, buckets);
}

// Entry i of a list into its bucket, if that is one of the `part` buckets from b0 on.  out_w: the weights' places of those buckets.
__device__ __forceinline__ void set_insert(const int32_t* __restrict__ adj, const float* __restrict__ w, uint32_t deg, uint32_t i,
                                           uint32_t buckets, uint32_t b0, uint32_t part, int32_t* s_slots, uint32_t* s_count,
                                           float* out_w) {
  const int32_t x = adj[i];
  if (i != 0u && adj[i - 1u] == x) return;  // the lists ascend: equal neighbours lie together, the first stands for all
  const uint32_t b = set_bucket(x, buckets) - b0;
  if (b >= part) return;
  const uint32_t at = atomicAdd(&s_count[b], 1u);
  if (at >= 16u) return;
  s_slots[16u * b + at] = x;
  if (out_w != nullptr) {
    float sum = 0.0f;
    for (uint32_t j = i; j < deg && adj[j] == x; ++j) sum = sum + w[j];
    out_w[16u * b + at] = sum;
  }
}

// Lists of one group, one wave per list.  Bound: memory (4 bytes read and about 10 written per edge).
__global__ __launch_bounds__(256) void fw_sets_small_kernel(const uint4* __restrict__ vrec, const int32_t* __restrict__ adjncy,
                                                            const float* __restrict__ weight, int32_t V, int32_t* sets, float* set_weights) {
  __shared__ __align__(16) int32_t s_slots[4][16u * kSetSmall];
  __shared__ uint32_t s_count[4][kSetSmall];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint64_t chunks = ((uint64_t)(uint32_t)V + 63u) >> 6;
  for (uint64_t ch = (uint64_t)blockIdx.x * 4u + (uint64_t)wave; ch < chunks; ch += (uint64_t)gridDim.x * 4u) {
    const uint32_t v0 = (uint32_t)(ch * 64u);
    uint32_t off = 0u, deg = 0u;
    if (v0 + (uint32_t)lane < (uint32_t)V) {
      const uint4 rec = vrec[v0 + (uint32_t)lane];
      off = rec.w;
      deg = rec.y;
    }
    for (uint64_t m = __ballot(deg != 0u && list_quartets(off, deg) <= kGq); m != 0ull; m &= m - 1ull) {
      const int l = __builtin_ctzll(m);
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, l), d = (uint32_t)__builtin_amdgcn_readlane((int)deg, l);
      const uint32_t nb = fw_set_buckets(d);
      const uint64_t first = 16u * fw_set_first(o, v0 + (uint32_t)l);
      int4* const slots = reinterpret_cast<int4*>(s_slots[wave]);
      for (uint32_t i = (uint32_t)lane; i < 4u * nb; i += 64u) slots[i] = make_int4(-1, -1, -1, -1);
      for (uint32_t i = (uint32_t)lane; i < nb; i += 64u) s_count[wave][i] = 0u;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (uint32_t i = (uint32_t)lane; i < d; i += 64u)
        set_insert(adjncy + o, weight + o, d, i, nb, 0u, nb, s_slots[wave], s_count[wave], set_weights ? set_weights + first : nullptr);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (uint32_t i = (uint32_t)lane; i < 4u * nb; i += 64u) {
        int4 x = slots[i];
        if ((i & 3u) == 3u && s_count[wave][i >> 2] > 16u) x.w = kSetOverflow;
        reinterpret_cast<int4*>(sets + first)[i] = x;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// Long lists: one workgroup per eight groups of a list makes kSetPart buckets and reads the whole list for them: a list of 100,000
// entries is read 13 times, from the cache, and the reads grow with the square of the length, which the rule that decides on sets prices.
__global__ __launch_bounds__(512) void fw_sets_long_kernel(const uint4* __restrict__ vrec, const int32_t* __restrict__ adjncy,
                                                           const float* __restrict__ weight, const uint2* __restrict__ items,
                                                           uint32_t n_items, int32_t* sets, float* set_weights) {
  __shared__ __align__(16) int32_t s_slots[16u * kSetPart];
  __shared__ uint32_t s_count[kSetPart];
  for (uint32_t it = blockIdx.x; it < n_items; it += gridDim.x) {
    const uint2 item = items[it];
    if ((item.y & 7u) != 0u) continue;
    const uint4 rec = vrec[item.x];
    const uint32_t nb = fw_set_buckets(rec.y);
    const uint32_t b0 = (item.y >> 3) * kSetPart;
    if (b0 >= nb) continue;
    const uint32_t part = nb - b0 < kSetPart ? nb - b0 : kSetPart;
    const uint64_t first = 16u * (fw_set_first(rec.w, item.x) + b0);
    int4* const slots = reinterpret_cast<int4*>(s_slots);
    for (uint32_t i = threadIdx.x; i < 4u * part; i += blockDim.x) slots[i] = make_int4(-1, -1, -1, -1);
    for (uint32_t i = threadIdx.x; i < part; i += blockDim.x) s_count[i] = 0u;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < rec.y; i += blockDim.x)
      set_insert(adjncy + rec.w, weight + rec.w, rec.y, i, nb, b0, part, s_slots, s_count, set_weights ? set_weights + first : nullptr);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 4u * part; i += blockDim.x) {
      int4 x = slots[i];
      if ((i & 3u) == 3u && s_count[i >> 2] > 16u) x.w = kSetOverflow;
      reinterpret_cast<int4*>(sets + first)[i] = x;
    }
    __syncthreads();
  }
}

// The place of `target` in the set of vertex v's list: its index in the sets, -1 (not there) or -2 (its bucket overflowed).
__device__ __forceinline__ int64_t set_find(const int32_t* __restrict__ sets, uint32_t v, uint32_t off, uint32_t deg, int32_t target) {
  const uint64_t first = 16u * (fw_set_first(off, v) + set_bucket(target, fw_set_buckets(deg)));
  int32_t at = -1;
  int4 x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = reinterpret_cast<const int4*>(sets + first)[i];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    at = x[i].x == target ? 4 * i : at;
    at = x[i].y == target ? 4 * i + 1 : at;
    at = x[i].z == target ? 4 * i + 2 : at;
    at = x[i].w == target ? 4 * i + 3 : at;
  }
  if (at >= 0) return (int64_t)first + at;
  return x[3].w == kSetOverflow ? -2 : -1;
}

// ---- MetaPath: lists by label -----------------------------------------------------------------------------
//
// A bias is 1 where the edge has the step's label and 0 elsewhere, so every sum the sampler makes is a count, exact in
// whichever order it is added up, and "the first element whose running sum is above t" is the element of rank floor(t)
// among those of the label (the last one if t reaches the count).  So the neighbours of a group are stored sorted by label, in the order
// the sampler's lanes hold them, at the group's own places of the edge array (4 bytes written per edge), and a step reads
// its vertex's record and one neighbour: 10^7 walks of 5 steps on R-MAT 26 take 1.36 ms, 6.85 through parking.
// vrec[2v] = {region, degree, 0, CSR offset}, vrec[2v + 1] = where each label's neighbours end in a list of one group (8 x 16 bits).
// A longer list has a region, in blocks of 128 bytes: the labels' totals (floats), per label the sums of its groups as
// above, per group the ends of its labels.

// The ends of up to 8 labels in a group of at most 1024 elements, two in a word.
struct LabelCounts {
  uint32_t w[FW_MAX_TABLE_LABELS / 2];
};

constexpr int kLabelWords = FW_MAX_TABLE_LABELS / 2;

template <int kW = kLabelWords>
__device__ __forceinline__ uint32_t label_field(const LabelCounts& c, uint32_t s) {
  uint32_t x = c.w[0];
#pragma unroll
  for (uint32_t i = 1; i < (uint32_t)kW; ++i) x = (s >> 1) == i ? c.w[i] : x;
  return (s & 1u) ? x >> 16 : x & 0xFFFFu;
}

template <int kW>
__device__ __forceinline__ void label_count(LabelCounts& c, uint32_t s) {
  const uint32_t add = 1u << ((s & 1u) * 16u);
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kW; ++i) c.w[i] += (s >> 1) == i ? add : 0u;
}

// The value of the lane the DPP control names, 0 where there is none or the row is not in the mask.
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t dpp_or_0(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kCtrl, kRows, 0xF, false);
}

// One group per segment of kSeg lanes (a quad, a DPP row or the wave), lane c holding the quartets c + 64 j as in load_lane: its neighbours by label into
// by_label.  Returns the ends of the labels in every lane; totals: their counts.
template <int kSeg, int kJ, int kW>
__device__ __forceinline__ LabelCounts label_group(const int32_t* __restrict__ label, const int32_t* __restrict__ adjncy,
                                                   const fw_label_set& set, uint32_t off, uint32_t deg, uint32_t kb, uint32_t nqg,
                                                   int lane, int32_t* by_label, LabelCounts& totals) {
  const uint32_t c = (uint32_t)lane & (uint32_t)(kSeg - 1);
  const uint32_t a0 = off & ~3u;
  uint64_t slots = 0u;  // four bits each
  int32_t nb[4 * kJ];
  LabelCounts mine = {}, at;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const uint32_t k = c + 64u * (uint32_t)j;
    int4 l = make_int4(0, 0, 0, 0), n = make_int4(-1, -1, -1, -1);
    const uint32_t base = a0 + 4u * (kb + k);
    if (k < nqg) {
      l = *reinterpret_cast<const int4*>(label + base);
      n = *reinterpret_cast<const int4*>(adjncy + base);
    }
    const uint32_t lim = k < nqg ? deg : 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int32_t x = i == 0 ? l.x : i == 1 ? l.y : i == 2 ? l.z : l.w;
      nb[4 * j + i] = i == 0 ? n.x : i == 1 ? n.y : i == 2 ? n.z : n.w;
      uint32_t s = FW_MAX_TABLE_LABELS;  // none of the schema's, or not in the list (an index before it wraps)
#pragma unroll
      for (int m = 2 * kW - 1; m >= 0; --m) s = m < set.n && x == set.label[m] ? (uint32_t)m : s;
      s = base + (uint32_t)i - off < lim ? s : (uint32_t)FW_MAX_TABLE_LABELS;
      slots |= (uint64_t)s << (4 * (4 * j + i));
      label_count<kW>(mine, s);  // (the slot of no label is in no word)
    }
  }
  uint32_t before = 0u;
  LabelCounts ends = {};
  totals = LabelCounts{};
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    uint32_t x = mine.w[w], t;
    if (kSeg == 4) {
      const uint32_t y = dpp_or_0<0x111, 0xF>(x);
      x += c >= 1u ? y : 0u;
      const uint32_t z = dpp_or_0<0x112, 0xF>(x);
      x += c >= 2u ? z : 0u;
      t = dpp_or_0<0xFF, 0xF>(x);  // of the quad's last lane
    } else {
      x += dpp_or_0<0x111, 0xF>(x);
      x += dpp_or_0<0x112, 0xF>(x);
      x += dpp_or_0<0x114, 0xF>(x);
      x += dpp_or_0<0x118, 0xF>(x);
      if (kSeg == 64) x += dpp_or_0<0x142, 0xA>(x);
      if (kSeg == 64) x += dpp_or_0<0x143, 0xC>(x);
      t = kSeg == 64 ? (uint32_t)__builtin_amdgcn_readlane((int)x, 63) : (uint32_t)__shfl((int)x, kSeg - 1, kSeg);
    }
    totals.w[w] = t;
    const uint32_t e0 = before + (t & 0xFFFFu), e1 = e0 + (t >> 16);
    at.w[w] = (before | (e0 << 16)) + (x - mine.w[w]);
    ends.w[w] = e0 | (e1 << 16);
    before = e1;
  }
  const uint32_t first = kb == 0u ? off : a0 + 4u * kb;
#pragma unroll
  for (int i = 0; i < 4 * kJ; ++i) {
    const uint32_t s = (uint32_t)(slots >> (4 * i)) & 15u;
    if (s < (uint32_t)FW_MAX_TABLE_LABELS) by_label[first + label_field<kW>(at, s)] = nb[i];
    label_count<kW>(at, s);
  }
  return ends;
}

__device__ __forceinline__ uint4 label_words(const LabelCounts& c) { return make_uint4(c.w[0], c.w[1], c.w[2], c.w[3]); }

// The lists of the lanes with `mine`, 64 / kSeg at a time.
template <int kSeg, int kW>
__device__ __forceinline__ void label_segments(const int32_t* __restrict__ label, const int32_t* __restrict__ adjncy,
                                               const fw_label_set& set, uint32_t off, uint32_t deg, bool mine, uint32_t v0, int lane,
                                               uint4* vrec, int32_t* by_label) {
  const uint64_t m = __ballot(mine);
  const int n = __builtin_popcountll(m);
  const uint64_t below = (1ull << lane) - 1ull;
  // lane i: the i-th lane with a list (the others' numbers go behind them)
  const int at = mine ? __builtin_popcountll(m & below) : n + __builtin_popcountll(~m & below);
  const int order = __builtin_amdgcn_ds_permute(at << 2, lane);
  for (int i0 = 0; i0 < n; i0 += 64 / kSeg) {
    const int i = i0 + lane / kSeg;  // below 64: n is at most 64 and i0 a multiple of 64 / kSeg
    const int src = __shfl(order, i);
    const uint32_t o = __shfl(off, src), df = __shfl(deg, src);  // every lane takes part
    const uint32_t d = i < n ? df : 0u;
    LabelCounts totals;
    const LabelCounts e = label_group<kSeg, 1, kW>(label, adjncy, set, o, d, 0u, d != 0u ? list_quartets(o, d) : 0u, lane, by_label, totals);
    if (i < n && (lane & (kSeg - 1)) == 0) vrec[2u * (uint64_t)(v0 + (uint32_t)src) + 1u] = label_words(e);
  }
}

// Lists of one group: a wave takes 64 consecutive vertices; lists of at most 4 (16) quartets sixteen (four) at a time, the others one
// after the other.  kW: words of the labels' counts (two labels each).
// Bound: instructions (12 bytes of traffic per edge and 32 per vertex would take 3 ms on R-MAT 26, 1.07 G edges, 67 M vertices;
// measured 13.6 ms, 27.6 with sixteen lanes for the shortest lists, scans through LDS and 148 registers).
template <int kW>
__global__ __launch_bounds__(256, 7) void fw_label_lists_kernel(const uint32_t* __restrict__ xadj, const int32_t* __restrict__ adjncy,
                                                             const int32_t* __restrict__ label, int32_t V, const fw_label_set set,
                                                             const uint32_t* __restrict__ base, uint4* vrec, int32_t* by_label) {
  const int lane = lane_id();
  const uint64_t chunks = ((uint64_t)(uint32_t)V + 63u) >> 6;
  for (uint64_t ch = (uint64_t)blockIdx.x * 4u + (uint64_t)(threadIdx.x >> 6); ch < chunks; ch += (uint64_t)gridDim.x * 4u) {
    const uint32_t v0 = (uint32_t)(ch * 64u), v = v0 + (uint32_t)lane;
    uint32_t off = 0u, deg = 0u;
    if (v < (uint32_t)V) {
      off = xadj[v];
      deg = xadj[v + 1] - off;
      vrec[2u * (uint64_t)v] = make_uint4(base[v], deg, 0u, off);
    }
    const uint32_t nq = deg != 0u ? list_quartets(off, deg) : 0u;
    if (v < (uint32_t)V && (nq == 0u || nq > kGq)) vrec[2u * (uint64_t)v + 1u] = make_uint4(0u, 0u, 0u, 0u);
    LabelCounts totals;
    label_segments<4, kW>(label, adjncy, set, off, deg, nq != 0u && nq <= 4u, v0, lane, vrec, by_label);
    label_segments<16, kW>(label, adjncy, set, off, deg, nq > 4u && nq <= 16u, v0, lane, vrec, by_label);
    uint64_t m;
    for (m = __ballot(nq > 16u && nq <= kGq); m != 0ull; m &= m - 1ull) {
      const int l = __builtin_ctzll(m);
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, l), d = (uint32_t)__builtin_amdgcn_readlane((int)deg, l);
      const uint32_t n = list_quartets(o, d);
      const LabelCounts e = n <= 64u ? label_group<64, 1, kW>(label, adjncy, set, o, d, 0u, n, lane, by_label, totals)
                                     : label_group<64, kGroupQuartets, kW>(label, adjncy, set, o, d, 0u, n, lane, by_label, totals);
      if (lane == 0) vrec[2u * (uint64_t)(v0 + (uint32_t)l) + 1u] = label_words(e);
    }
  }
}

// The groups of the long lists, one wave per group: their neighbours by label, ends and totals (1.8 ms on R-MAT 26).
template <int kW>
__global__ __launch_bounds__(256, 7) void fw_label_groups_kernel(const uint4* __restrict__ vrec, const int32_t* __restrict__ adjncy,
                                                              const int32_t* __restrict__ label, const uint2* __restrict__ items,
                                                              uint32_t n_items, const fw_label_set set, int32_t hub_threshold,
                                                              uint32_t nw_shift, unsigned char* data, int32_t* by_label) {
  const int lane = lane_id();
  for (uint32_t it = blockIdx.x * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); it < n_items;
       it += gridDim.x * 4u) {
    const uint2 item = items[it];
    const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)item.x), g = (uint32_t)__builtin_amdgcn_readfirstlane((int)item.y);
    const uint4 rec = vrec[2u * (uint64_t)v];
    const uint32_t off = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec.w), deg = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec.y);
    unsigned char* const region = data + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)rec.x) * 128u;
    const uint32_t nq = list_quartets(off, deg);
    const uint32_t ngroups = (nq + kGq - 1u) / kGq;
    const bool wg = (int32_t)deg > hub_threshold;
    const uint32_t left = nq - g * kGq;
    LabelCounts totals;
    const LabelCounts e = label_group<64, kGroupQuartets, kW>(label, adjncy, set, off, deg, g * kGq, left < kGq ? left : kGq, lane, by_label, totals);
    const uint32_t k = wg ? g >> nw_shift : g;
    const uint32_t block = wg ? 1u + (g & ((1u << nw_shift) - 1u)) * seq_blocks(ngroups, wg, nw_shift) + (k >> 4) : k >> 4;
    const uint32_t hb = header_units(ngroups, wg, nw_shift) >> 2;  // blocks of one label's sums
    if (lane < set.n)
      reinterpret_cast<float*>(region)[32u * (1u + (uint32_t)lane * hb + block) + 16u + (k & 15u)] = (float)label_field(totals, (uint32_t)lane);
    if (lane == 0) reinterpret_cast<uint4*>(region + (uint64_t)128u * (1u + (uint32_t)set.n * hb))[g] = label_words(e);
  }
}

// The running sums of the long lists, one wave per list and label.
__global__ __launch_bounds__(256) void fw_label_sums_kernel(const uint4* __restrict__ vrec, const uint32_t* __restrict__ longs, uint32_t n_longs,
                                                            const uint32_t n_labels, int32_t hub_threshold, uint32_t nw_shift,
                                                            unsigned char* data) {
  const int lane = lane_id();
  const uint64_t n = (uint64_t)n_longs * n_labels;
  for (uint64_t it = (uint64_t)blockIdx.x * 4u + (uint64_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); it < n;
       it += (uint64_t)gridDim.x * 4u) {
    const uint32_t s = (uint32_t)(it % n_labels);
    const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)longs[it / n_labels]);
    const uint4 rec = vrec[2u * (uint64_t)v];
    const uint32_t ngroups = (list_quartets(rec.w, rec.y) + kGq - 1u) / kGq;
    const bool wg = (int32_t)rec.y > hub_threshold;
    float* const region = reinterpret_cast<float*>(data + (uint64_t)rec.x * 128u);
    const float total = list_sums(region + 32u * (1u + s * (header_units(ngroups, wg, nw_shift) >> 2)), ngroups, wg, nw_shift, lane);
    if (lane == 0) region[s] = total;
  }
}

// ---- the walk -----------------------------------------------------------------------------------------

// First entry above t of the n entries of a row (they never decrease, the last one is above t; rows are padded to 8
// entries with +inf), from a guess.  Eight entries per look, so that nearly every walker of a wave finds its entry with the first; when
// the guess was off twice the rest is halved.
__device__ __forceinline__ uint32_t row_search(const float* row, uint32_t n, uint32_t guess, float t) {
  const uint32_t wmax = ((n + 7u) & ~7u) - 8u;
  uint32_t lo = 0u, hi = n - 1u;
  uint32_t w = guess > 3u ? guess - 3u : 0u;
  for (int looks = 0;; ++looks) {
    w = w < wmax ? w : wmax;
    const f4_at4 m0 = *reinterpret_cast<const f4_at4*>(row + w);
    const f4_at4 m1 = *reinterpret_cast<const f4_at4*>(row + w + 4u);
    uint32_t cnt = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float m = i < 4 ? m0[i & 3] : m1[i & 3];
      cnt += m <= t ? 1u : 0u;
    }
    if (cnt == 0u) {
      if (w <= lo) return w;
      hi = w;
      w = looks == 0 || hi - lo <= 16u ? (hi > lo + 7u ? hi - 7u : lo) : (lo + hi) >> 1;
    } else {
      if (cnt < 8u) return w + cnt;
      lo = w + 8u;
      if (lo >= hi) return hi;
      w = looks == 0 || hi - lo <= 16u ? lo : (lo + hi) >> 1;
    }
  }
}

// The same in two looks: every eighth entry, then the eight that one of them ends.
// Where row M is in the caches, or a wave has few walkers and waits for memory anyway, row_search's looks cost more than the other block of a row; elsewhere less.
// row_search / this one, us: 1,000,000 DeepWalk walkers, log-normal weights with sigma 2, R-MAT 12 (1 MB of regions) 1201 / 1007, Pareto R-MAT 16 (25 MB) 2107 / 1952, R-MAT 20
// (270 MB) 2654 / 2992, R-MAT 22 6337 / 7343; 50,000 walkers, R-MAT 20, 509 / 444.
__device__ __forceinline__ uint32_t row_eighths(const float* row, uint32_t n, float t) {
  const uint32_t e = (n + 7u) >> 3;
  uint32_t k = 0u;
#pragma unroll
  for (uint32_t i = 0; i < 7u; ++i) k += row[8u * (i < e ? i : e - 1u) + 7u] <= t ? 1u : 0u;  // (the row's last entry is +inf)
  const f4_at4 m0 = *reinterpret_cast<const f4_at4*>(row + 8u * k);
  const f4_at4 m1 = *reinterpret_cast<const f4_at4*>(row + 8u * k + 4u);
  uint32_t l = 8u * k;
#pragma unroll
  for (int i = 0; i < 8; ++i) l += (i < 4 ? m0[i & 3] : m1[i & 3]) <= t ? 1u : 0u;
  return l;
}

// A look at one block of pairs for every lane with `need` (the lanes of m): first = the neighbour of its first key above t, at_start = that is the
// block's first, none = there is none.  All lanes take part.  Four or eight lanes read a walker's block together, 16 bytes a load each: a lane that loads its block alone makes eight requests to the first-level cache, each of which may wait for the address's translation.
// A lane for each block / eight lanes: DeepWalk R-MAT 24 (5 GB of regions) 4.9e9 / 0.95e9 translation misses, 66.4 / 35.5 ms; R-MAT 22 5.92 / 4.92 ms, node2vec
// R-MAT 20 with q = 4 5.99 / 5.35; with row M and the pairs by each lane these were 47.4, 6.65 and 6.26.
// Four lanes take half the instructions of eight, which counts where the blocks are near: eight / four, 20,108 DeepWalk walkers on R-MAT 12 0.184 / 0.160 ms, 50,021
// node2vec walkers on R-MAT 20 0.461 / 0.433, 805,111 DeepWalk walkers on a uniform graph of 40,000 vertices 0.345 / 0.320, DeepWalk R-MAT 22 4.94 / 4.86; but a block that is not
// kept is asked for in halves then: R-MAT 24 33.2 / 35.5.
// A block comes once, and among gigabytes of them nobody wants it again before it is gone: there (kStream) it is not kept in the L2, which holds more
// of the records and sums instead.
typedef uint32_t u4_vec __attribute__((ext_vector_type(4)));

struct BlockLook {
  uint32_t first;
  bool at_start, none;
};

template <bool kStream>
__device__ __forceinline__ BlockLook look_at_blocks(const unsigned char* data, const uint64_t m, const bool need, const uint32_t block, const float t,
                                                    const uint32_t lane) {
  const uint32_t n = (uint32_t)__builtin_popcountll(m);
  const uint32_t rank = (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull));
  const int to = (int)(need ? rank : n + lane - rank) << 2;  // the lanes that look first, in order, then the others
  const int blocks = __builtin_amdgcn_ds_permute(to, (int)(need ? block : 0u));
  const int targets = __builtin_amdgcn_ds_permute(to, (int)__float_as_uint(t));
  constexpr uint32_t kLanes = kStream ? 8u : 4u, kParts = 8u / kLanes, kLoads = kLanes, kAt = 64u / kLanes;  // lanes a block, pieces a lane, blocks a load
  const uint32_t of = lane / kLanes, piece = lane & (kLanes - 1u);
  uint4 x[kLoads][kParts];
#pragma unroll
  for (uint32_t i = 0; i < kLoads; ++i) {
    if (kAt * i < n) {
      const uint32_t b = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(kAt * i + of) << 2, blocks);
      const u4_vec* const at = reinterpret_cast<const u4_vec*>(data + (uint64_t)b * 128u + 16u * piece);
#pragma unroll
      for (uint32_t j = 0; j < kParts; ++j) {
        const u4_vec y = kStream ? __builtin_nontemporal_load(at + 4u * j) : at[4u * j];
        x[i][j] = make_uint4(y[0], y[1], y[2], y[3]);
      }
    }
  }
  BlockLook r = {0u, false, true};
#pragma unroll
  for (uint32_t i = 0; i < kLoads; ++i) {
    if (kAt * i < n) {
      const float ti = __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute((int)(kAt * i + of) << 2, targets));
      const uint32_t at = kLanes * (rank & (kAt - 1u));
      uint64_t m0 = 0ull;
      uint32_t above = 0u, mine = x[i][kParts - 1u].w;
#pragma unroll
      for (uint32_t j = kParts; j-- > 0u;) {  // (where no lane has a key above t in the front half, all of them offer one of the back half)
        const bool c0 = !(__uint_as_float(x[i][j].x) <= ti), c1 = !(__uint_as_float(x[i][j].z) <= ti);
        m0 = __ballot(c0);
        above |= ((uint32_t)((m0 | __ballot(c1)) >> at) & ((1u << kLanes) - 1u)) << (kLanes * j);
        mine = c0 ? x[i][j].y : c1 ? x[i][j].w : mine;
      }
      const uint32_t f = at + ((uint32_t)__builtin_ctz(above | 0x80u) & (kLanes - 1u));
      const uint32_t nb = (uint32_t)__builtin_amdgcn_ds_bpermute((int)f << 2, (int)mine);
      if (need && rank / kAt == i) r = {nb, ((m0 >> at) & 1ull) != 0ull, above == 0u};
    }
  }
  return r;
}

// Where a step's neighbour is looked for: the first of the n pairs of a group, from block `pairs` of the tables on, whose key is above t.  It does
// not lie before block `lo` of them and is guessed to lie in block b.
struct PairPlace {
  uint32_t pairs, n, b, lo;
  float t;
};

// That neighbour, for the lanes with `need`; all lanes take part.  From the guess on block after block; after four looks what is left is halved
// (which few meet: but for one lane in 32 the pairs of a group that is not marked lie within five blocks of their guess, and a shorter list has five at most).
template <bool kStream>
__device__ __forceinline__ uint32_t pair_search(const unsigned char* data, bool need, PairPlace p, const uint32_t lane) {
  const uint32_t top = (p.n - 1u) >> 4;
  uint32_t end = top + 1u;  // where the blocks end that may hold it; behind the last one it is `found`
  uint32_t found = 0u;
  p.b = p.b < top ? p.b : top;
  for (uint32_t looks = 0u;; ++looks) {
    const uint64_t m = __ballot(need);
    if (m == 0ull) return found;
    const BlockLook k = look_at_blocks<kStream>(data, m, need, p.pairs + p.b, p.t, lane);
    if (need) {
      if (k.none && p.b < top) {  // (what follows the pairs in the last block comes after a key that is above t)
        p.lo = p.b + 1u;
        need = p.lo != end;
        p.b = looks >= 3u ? (p.lo + end) >> 1 : p.lo;
      } else {
        found = k.first;
        need = k.at_start && p.b > p.lo;
        end = p.b;
        p.b = looks >= 3u ? (p.lo + end) >> 1 : p.b - 1u;
      }
    }
  }
}

__device__ __forceinline__ void load16(const float* p, float (&s)[16]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 x = reinterpret_cast<const float4*>(p)[i];
    s[4 * i] = x.x; s[4 * i + 1] = x.y; s[4 * i + 2] = x.z; s[4 * i + 3] = x.w;
  }
}

// The reservoir over the groups of one sequence (nb blocks of sums): the group it ends with, its uniform and where its total is.  The
// test of the streaming kernels, S_k u > S_j, is monotone in k, so the next accepted group is the first of the 16 sums in
// registers that passes it; only when none does is another block looked for, from where the sums would reach S_j / u if
// they grew evenly.  (One look at memory per accepted group made every wave wait for the longest such chain of its 64 walkers.)
__device__ __forceinline__ const float* sums_reservoir(const fw_kargs& a, const float* sums, const uint32_t nb, LaneDraw& dq,
                                                       const uint32_t walker, const uint32_t step, const uint32_t stream,
                                                       uint32_t& k_out, float& tu_out) {
  float s[16];
  load16(sums, s);
  float S_last = s[15];
  if (nb > 1u) S_last = sums[32u * (nb - 1u) + 15u];
  float Sj = 0.0f, u = 1.0f, tu = 0.0f;  // the first group that has a total is always accepted
  uint32_t b = 0u, k = 0u;
  while (S_last * u > Sj) {
    if (!(s[15] * u > Sj)) {
      uint32_t lo = b, hi = nb - 1u;  // block lo has none, block hi has one
      const float per = (float)nb * __builtin_amdgcn_rcpf(S_last);
      const float want = Sj * __builtin_amdgcn_rcpf(u) * per;
      uint32_t i = want < (float)nb ? (uint32_t)want : hi;
      for (int tries = 0;; ++tries) {
        i = i < hi ? (i > lo ? i : lo + 1u) : hi;
        load16(sums + 32u * i, s);
        const float before = sums[32u * i - 17u];  // the last sum of the block before
        if (before * u > Sj && i - 1u > lo) {
          hi = i - 1u;
        } else if (s[15] * u > Sj || i == hi) {
          break;
        } else {
          lo = i;
        }
        i = tries < 2 ? (hi == i - 1u ? hi : i + 1u) : lo + ((hi - lo + 1u) >> 1);
      }
      b = i;
    }
    // The first of the 16 that passes, by halves (one of them does): 28 instructions where 16 comparisons took 64, and the wave runs as
    // many rounds as the walker with the most accepted groups (50,021 node2vec walkers on R-MAT 20 552 -> 490 us, 100 DeepWalk walkers 145 -> 127,
    // DeepWalk R-MAT 22 6.77 -> 6.64 ms).
    float h8[8], h4[4], h2[2];
    const bool c8 = !(s[7] * u > Sj);
#pragma unroll
    for (int i = 0; i < 8; ++i) h8[i] = c8 ? s[8 + i] : s[i];
    const bool c4 = !(h8[3] * u > Sj);
#pragma unroll
    for (int i = 0; i < 4; ++i) h4[i] = c4 ? h8[4 + i] : h8[i];
    const bool c2 = !(h4[1] * u > Sj);
    h2[0] = c2 ? h4[2] : h4[0];
    h2[1] = c2 ? h4[3] : h4[1];
    const bool c1 = !(h2[0] * u > Sj);
    k = 16u * b + (c8 ? 8u : 0u) + (c4 ? 4u : 0u) + (c2 ? 2u : 0u) + (c1 ? 1u : 0u);
    Sj = c1 ? h2[1] : h2[0];
    tu = next_uniform_lane(dq, a, walker, step, stream);
    u = next_uniform_lane(dq, a, walker, step, stream);
  }
  k_out = k;
  tu_out = tu;
  return sums + 32u * (k >> 4) + 16u + (k & 15u);
}

// The sequence of groups a step at workgroup granularity goes to, by the scan of the sequences' totals.
__device__ __forceinline__ uint32_t which_sequence(const fw_kargs& a, const float* scan, const float total, const uint32_t walker,
                                                   const uint32_t step, const uint32_t sbase) {
  const float target = u24(philox4x32_10<true>(walker, step, kStreamWave | sbase, 0u, a.seed_lo, a.seed_hi).x) * total;
  float keys[16];
  load16(scan, keys);
  uint32_t seq = 0u;
#pragma unroll
  for (int i = 0; i < 16; ++i) seq += keys[i] <= target ? 1u : 0u;
  return seq;
}

// MetaPath's step: the selected neighbour, or -1 when no edge has the label.  ends: vrec[2v + 1].
__device__ __forceinline__ int32_t label_pick(const fw_kargs& a, const fw_table_args& tb, const uint4 rec, uint4 ends, const uint32_t s,
                                              const uint4 d, const uint32_t walker, const uint32_t step) {
  const uint32_t nq = list_quartets(rec.w, rec.y);
  float tu = u24(d.x);
  uint32_t first = rec.w;
  if (nq > kGq) {
    const unsigned char* region = tb.data + (uint64_t)rec.x * 128u;
    const float total = reinterpret_cast<const float*>(region)[s];
    if (!(total > 0.0f)) return -1;
    const uint32_t ngroups = (nq + kGq - 1u) / kGq;
    const bool wg = (int32_t)rec.y > a.hub_threshold;
    const uint32_t nb = seq_blocks(ngroups, wg, tb.nw_shift);
    const uint32_t hb = header_units(ngroups, wg, tb.nw_shift) >> 2;
    const float* sums = reinterpret_cast<const float*>(region) + 32u * (1u + s * hb);
    uint32_t seq = 0u;
    LaneDraw dq;
    dq.q0 = d.x; dq.q1 = d.y; dq.q2 = d.z; dq.q3 = d.w;
    dq.avail = 4u;
    dq.blk = 1u;
    if (wg) {
      seq = which_sequence(a, sums, total, walker, step, 0u);
      sums += 32u + 32u * nb * seq;
      dq = LaneDraw();
    }
    uint32_t k;
    (void)sums_reservoir(a, sums, nb, dq, walker, step, seq, k, tu);
    const uint32_t g = wg ? seq + (k << tb.nw_shift) : k;
    if (g != 0u) first = (rec.w & ~3u) + 4u * kGq * g;
    ends = reinterpret_cast<const uint4*>(region + (uint64_t)128u * (1u + (uint32_t)tb.labels.n * hb))[g];
  }
  const LabelCounts e = {{ends.x, ends.y, ends.z, ends.w}};
  const uint32_t start = s != 0u ? label_field(e, s - 1u) : 0u, n = label_field(e, s) - start;
  if (n == 0u) return -1;
  const uint32_t r = (uint32_t)(tu * (float)n);
  return tb.by_label[first + start + (r < n ? r : n - 1u)];
}

// One proposal of the step's sampler for a list with a positive total: where the selected neighbour is looked for.  d: block 0 of the step's stream 0.
__device__ __forceinline__ PairPlace table_pick(const fw_kargs& a, const fw_table_args& tb, const uint4 rec, const uint4 d,
                                              const uint32_t walker, const uint32_t step, const uint32_t sbase) {
  const float total = __uint_as_float(rec.z);
  const uint32_t nq = list_quartets(rec.w, rec.y);
  uint32_t entries = rec.x & ~kUneven;  // the block they begin with
  uint32_t nqg = nq;
  float T = total, tu = u24(d.x);
  bool uneven = (rec.x & kUneven) != 0u;
  if (nq > kGq) {
    const uint32_t ngroups = (nq + kGq - 1u) / kGq;
    const bool wg = (int32_t)rec.y > a.hub_threshold;
    const uint32_t nb = seq_blocks(ngroups, wg, tb.nw_shift);
    const float* sums = reinterpret_cast<const float*>(tb.data + (uint64_t)entries * 128u);
    uint32_t seq = 0u;
    LaneDraw dq;
    if (wg) {  // which sequence, then the reservoir over it with draws of its own stream
      seq = which_sequence(a, sums, total, walker, step, sbase);
      sums += 32u + 32u * nb * seq;
    } else {
      dq.q0 = d.x; dq.q1 = d.y; dq.q2 = d.z; dq.q3 = d.w;
      dq.avail = 4u;
      dq.blk = 1u;
    }
    uint32_t k;
    T = *sums_reservoir(a, sums, nb, dq, walker, step, seq | sbase, k, tu);
    const uint32_t g = wg ? seq + (k << tb.nw_shift) : k;
    entries += (header_units(ngroups, wg, tb.nw_shift) + kGroupUnits * g) >> 2;
    nqg = nq - g * kGq < kGq ? nq - g * kGq : kGq;
    uneven = T < 0.0f;
    T = __builtin_fabsf(T);
  }
  PairPlace p = {entries, 4u * nqg, (uint32_t)(tu * (float)(4u * nqg)) >> 4, 0u, tu * T};
  if (uneven) {
    const uint32_t nl = nqg < 64u ? nqg : 64u;
    const float* const row = reinterpret_cast<const float*>(tb.data + (uint64_t)entries * 128u + 32u * nqg);
    const uint32_t l = tb.rows_near != 0u ? row_eighths(row, nl, p.t) : row_search(row, nl, (uint32_t)(tu * (float)nl), p.t);
    p.lo = p.b = lane_start(l, nqg) >> 2;
  }
  return p;
}

// One lane, one walker, from its start to its end; a lane whose walk is over takes the next query of its wave's range.
// Path entries are collected in LDS (16 per walker, by their place in the path matrix modulo 16) and leave as whole 64-byte
// lines; the entries of a row before its first and after its last whole line, and the -1 behind the walk, are stored by the
// wave together, one row at a time.
// kStream: the blocks of pairs are not kept in the L2.
template <int kApp, bool kStream>
__global__ __launch_bounds__(256, kWaves) void fw_table_walk(const fw_kargs a, const fw_table_args tb) {
  __shared__ __align__(16) int32_t s_buf[4][64 * 16];
  __shared__ unsigned long long s_acc[4];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  __shared__ uint8_t s_slot[kApp == FW_APP_METAPATH ? FW_MAX_SCHEMA : 1];  // of every label of the schema, in the tables
  if (threadIdx.x < 4u) s_acc[threadIdx.x] = 0ull;
  if (kApp == FW_APP_METAPATH && threadIdx.x < (uint32_t)a.schema_len) {
    int slot = 0;
    while (slot + 1 < tb.labels.n && tb.labels.label[slot] != a.schema[threadIdx.x]) ++slot;
    s_slot[threadIdx.x] = (uint8_t)slot;
  }
  __syncthreads();
  int32_t* const buf = s_buf[wave];
  const uint32_t my_buf = (uint32_t)lane * 16u;
  const uint32_t swz = ((uint32_t)lane >> 2) & 3u;  // spreads the lanes' 16-byte pieces over the banks
  auto slot_at = [&](uint32_t slot) { return my_buf + ((((slot >> 2) ^ swz) << 2) | (slot & 3u)); };
  const uint32_t md = (uint32_t)a.max_depth;
  const bool short_rows = md <= 16u;  // in at most two lines: every lane stores what is left of its own row by itself
  const uint32_t align0 = (uint32_t)(reinterpret_cast<uintptr_t>(a.paths) >> 2) & 15u;

  const uint32_t n = (uint32_t)a.n;
  const uint64_t first = ((uint64_t)blockIdx.x * 4u + (uint64_t)wave) * tb.lanes;  // the next ranges come from the dispenser
  uint32_t cursor = first < n ? (uint32_t)first : n;
  uint32_t last = n - cursor > tb.lanes ? cursor + tb.lanes : n;
  bool more = (uint64_t)gridDim.x * 4u * tb.lanes < n;

  bool active = false, fresh = false;
  uint32_t q = 0u, len = 0u, s0 = 0u, fpos = 0u;
  int32_t v = 0, prev = -1;
  uint32_t prev_off = 0u, prev_deg = 0u, trial = 0u;
  float w_ret = 0.0f;
  uint4 rec = make_uint4(0u, 0u, 0u, 0u);
  uint32_t n_steps = 0u, n_hub = 0u;
  unsigned long long n_edges = 0ull, hub_edges = 0ull;

  for (;;) {
    bool ended = false;
    bool partial = false;  // the row's first entries fill up a line that is not all its own
    {
      const bool want = !active && (uint32_t)lane < tb.lanes;
      const uint64_t m = __ballot(want);
      if (m != 0ull && cursor == last && more) {
        uint32_t at = 0u;
        // Walks of few steps use up a wave's queries so fast that the updates of the dispenser's one word bound them
        // (MetaPath, 10^7 walks of 5 steps: 2.01 -> 1.36 ms with this and the rule for short rows below, of which that one alone
        // gives 0.03): they take four times as many at once while all waves together can.  Longer rows gain nothing (PPR
        // R-MAT 22 1.15 -> 1.17, DeepWalk there 6.8 -> 6.8).
        const uint32_t take = short_rows && tb.lanes == 64u && n - last > gridDim.x * 4u * 1024u ? 256u : tb.lanes;
        if (lane == 0) at = atomicAdd(a.dispenser, take);
        at = gridDim.x * 4u * tb.lanes + (uint32_t)__builtin_amdgcn_readfirstlane((int)at);  // (below 2^32: n is below 2^31)
        more = at < n;
        if (more) {
          cursor = at;
          last = n - at > take ? at + take : n;
        }
      }
      if (m != 0ull && cursor < last) {
        const uint32_t qn = cursor + (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull));
        if (want && qn < last) {
          q = qn;
          v = a.starts[qn];
          len = 1u;
          fpos = 0u;
          s0 = (align0 + q * md) & 15u;
          if (s0 == 15u) {
            a.paths[(uint64_t)q * md] = v;
            fpos = 1u;
          } else {
            buf[slot_at(s0)] = v;
          }
          prev = -1;
          trial = 0u;
          active = true;
          fresh = true;
          ended = !((uint32_t)v < (uint32_t)a.V && md > 1u);
        }
        const uint32_t took = (uint32_t)__builtin_popcountll(m);
        cursor = last - cursor > took ? cursor + took : last;
      }
      if (__ballot(active) == 0ull) break;
    }
    const uint32_t walker = a.walker_base + q;
    const uint32_t step = len - 1u;
    const uint32_t sbase = kApp == FW_APP_NODE2VEC ? trial << 8 : 0u;
    uint4 ends = make_uint4(0u, 0u, 0u, 0u);
    if (active && !ended && fresh) {
      if (kApp == FW_APP_METAPATH) {
        rec = tb.vrec[2u * (uint64_t)(uint32_t)v];
        ends = tb.vrec[2u * (uint64_t)(uint32_t)v + 1u];
      } else {
        rec = tb.vrec[v];
      }
    }
    const uint4 d = philox4x32_10<true>(walker, step, sbase, 0u, a.seed_lo, a.seed_hi);
    int32_t nv = -1;
    bool go = active && !ended;  // to a neighbour with a positive bias, if there is one (include/walker.cuh:1373-1374)
    if constexpr (kApp != FW_APP_METAPATH) {
      go = go && __uint_as_float(rec.z) > 0.0f;
      PairPlace place = {0u, 1u, 0u, 0u, 0.0f};
      if (go) place = table_pick(a, tb, rec, d, walker, step, sbase);
      nv = (int32_t)pair_search<kStream>(tb.data, go, place, (uint32_t)lane);
    }
    if (active && !ended) {
      if constexpr (kApp == FW_APP_METAPATH) {  // (in front of this block it costs four more spilled scalar registers: R-MAT 26 1.37 -> 1.38 ms)
        nv = label_pick(a, tb, rec, ends, s_slot[step % (uint32_t)a.schema_len], d, walker, step);
        go = nv >= 0;
      }
      if (!go) {
        ended = true;
      } else {
        bool moved = true;
        if (kApp == FW_APP_NODE2VEC && prev >= 0) {
          if (a.n2v_extra > 0.0f && fresh) {
            const int64_t at = tb.set_weights != nullptr ? set_find(tb.sets, (uint32_t)v, rec.w, rec.y, prev) : -2;
            w_ret = at >= 0 ? tb.set_weights[at] : 0.0f;
            if (at == -2) w_ret = return_weight(a.adjncy + rec.w, a.weight + rec.w, rec.y, prev);
          }
          const N2vTest t = n2v_test<true>(a, nv, prev, walker, step, trial, __uint_as_float(rec.z), w_ret);
          if (t.take_prev) {
            nv = prev;
          } else {
            bool common = false;
            if (!t.decided) {
              const int64_t at = tb.sets != nullptr ? set_find(tb.sets, (uint32_t)prev, prev_off, prev_deg, nv) : -2;
              common = at >= 0;
              if (at == -2) common = sorted_contains(a.adjncy + prev_off, (int32_t)prev_deg, nv);
            }
            moved = n2v_finish(a, t, common);
          }
        }
        fresh = moved;
        if (moved) {
          if ((int32_t)rec.y > a.park_threshold) {
            n_hub += 1u;
            hub_edges += rec.y;
          } else {
            n_steps += 1u;
            n_edges += rec.y;
          }
          const uint32_t slot = (s0 + len) & 15u;
          buf[slot_at(slot)] = nv;
          if (kApp == FW_APP_NODE2VEC) {
            prev = v;
            prev_off = rec.w;
            prev_deg = rec.y;
            trial = 0u;
          }
          v = nv;
          len += 1u;
          ended = len >= md;
          if (kApp == FW_APP_PPR && !ended) {  // include/app.cuh:88-94
            const uint32_t bits = philox4x32_10<true>(walker, step, kStreamStop, 0u, a.seed_lo, a.seed_hi).x;
            ended = u24(bits) < a.tp;
          }
          if (slot == 15u) {
            if (len >= 16u) {
              const uint4* src = reinterpret_cast<const uint4*>(buf + my_buf);
              uint4* dst = reinterpret_cast<uint4*>(a.paths + ((uint64_t)q * md + (uint64_t)(len - 16u)));
#pragma unroll
              for (uint32_t j = 0; j < 4u; ++j) dst[j] = src[j ^ swz];
              fpos = len;
            } else {
              partial = true;
            }
          }
        } else {
          trial += 1u;
        }
      }
    }
    uint64_t ev = __ballot(active && (ended || partial));
    if (ev != 0ull) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const uint32_t end = ended ? md : len;
      if (short_rows) {
        if (active && (ended || partial)) {
          int32_t* const row = a.paths + (uint64_t)q * md;
          for (uint32_t p = fpos; p < end; ++p) row[p] = p < len ? buf[slot_at((s0 + p) & 15u)] : -1;
        }
        ev = 0ull;
      }
      if constexpr (kApp == FW_APP_NODE2VEC) {
        // One row at a time, 64 entries a store.  Four at a time, as below, are the slower way here but for the shortest walks (one row / four, medians of five
        // processes, all vertices of R-MAT 24, symmetrised, 80 steps 58.2 / 59.0 ms, half of them 33.7 / 34.1, 41 steps 17.14 / 17.29, 20 steps 8.37 / 8.38; R-MAT 22 80
        // steps 7.99 / 8.01, 20 steps 2.61 / 2.60; R-MAT 20, symmetrised, p = 0.25, q = 4, 40 steps 6.28 / 6.31).
        for (; ev != 0ull; ev &= ev - 1ull) {
          const uint32_t l = (uint32_t)__builtin_ctzll(ev);
          const uint32_t lq = readlane_u32(q, l), from = readlane_u32(fpos, l), to = readlane_u32(end, l);
          const uint32_t have = readlane_u32(len, l), ls0 = readlane_u32(s0, l);
          int32_t* const row = a.paths + (uint64_t)lq * md;
          for (uint32_t p = from + (uint32_t)lane; p < to; p += 64u) {
            const uint32_t slot = (ls0 + p) & 15u;
            row[p] = p < have ? buf[l * 16u + ((((slot >> 2) ^ ((l >> 2) & 3u)) << 2) | (slot & 3u))] : -1;
          }
        }
      } else {
        // Four rows at a time, 16 lanes each: one line from LDS, then pieces of 16 bytes.  (Rows one after the other, 64 entries a store, waited for LDS
        // twice a row: 1,000,003 PPR walkers from the hub of R-MAT 21 636 -> 623 us, PPR R-MAT 22 1115 -> 1108, of 20 steps 1015 -> 983, DeepWalk of 20 steps
        // there 2175 -> 2160, of 80 unchanged.)
        while (ev != 0ull) {
          int row_lane[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            row_lane[i] = ev != 0ull ? __builtin_ctzll(ev) : -1;
            ev &= ev - 1ull;  // (0 stays 0)
          }
          const uint32_t part = (uint32_t)lane >> 4, sub = (uint32_t)lane & 15u;
          const int l = part < 2u ? (part == 0u ? row_lane[0] : row_lane[1]) : (part == 2u ? row_lane[2] : row_lane[3]);
          const int src = l >= 0 ? l : 0;
          const uint32_t lq = (uint32_t)__shfl((int)q, src), have = (uint32_t)__shfl((int)len, src);
          const uint32_t from = (uint32_t)__shfl((int)fpos, src), ls0 = (uint32_t)__shfl((int)s0, src);
          const uint32_t row_end = (uint32_t)__shfl((int)end, src);
          const uint32_t to = l >= 0 ? row_end : 0u;
          int32_t* const row = a.paths + (uint64_t)lq * md;
          // what is not stored of the walk lies in one line: that line, then -1 in pieces of 16 bytes
          const uint32_t line = from - ((ls0 + from) & 15u);  // (wraps where the row begins inside the line; to is below 2^31)
          const uint32_t p = line + sub;
          if (p >= from && p < to) row[p] = p < have ? buf[(uint32_t)src * 16u + ((((sub >> 2) ^ (((uint32_t)src >> 2) & 3u)) << 2) | (sub & 3u))] : -1;
          uint32_t piece = line + 16u + 4u * sub;
          for (; piece + 4u <= to; piece += 64u) *reinterpret_cast<int4*>(row + piece) = make_int4(-1, -1, -1, -1);
          for (; piece < to; ++piece) row[piece] = -1;  // up to three, of one lane
        }
      }
      __builtin_amdgcn_wave_barrier();
      if (partial) fpos = len;
      if (ended) active = false;
    }
  }
  // workload counters: summed inside the workgroup, then one of 64 lines of counters (one line would be contended)
  if (n_steps != 0u) {
    atomicAdd(&s_acc[0], (unsigned long long)n_steps);
    atomicAdd(&s_acc[1], n_edges);
  }
  if (n_hub != 0u) {
    atomicAdd(&s_acc[2], (unsigned long long)n_hub);
    atomicAdd(&s_acc[3], hub_edges);
  }
  __syncthreads();
  if (threadIdx.x < 4u && s_acc[threadIdx.x] != 0ull)
    atomicAdd(&tb.counters[(blockIdx.x & (FW_TABLE_STRIPES - 1u)) * 8u + threadIdx.x], s_acc[threadIdx.x]);
}

// ---- the walk of few walkers ------------------------------------------------------------------------------
//
// A call of few walkers is a chain of dependent reads per step, and nothing else fills the time: the chip has lanes and memory to
// spare.  So a whole wave walks one walker.  A step takes its record and the group's pairs around the proportional
// guess (1 KB of them, an eighth of a full group, so the guess is nearly always good enough); for a long list
// the sums of 64 groups before that.  Every search is a comparison in all lanes and a ballot, and the draws a step may take are
// made by the lanes side by side while the record is on its way.
// Results are fw_table_walk's: the same sums, the same draws, the same comparisons.

constexpr int kWalkerWaves = 8;  // waves per SIMD

// sums_reservoir by a wave.  S_last: the sequence's last sum.  total: of the group it ends with.
__device__ __forceinline__ uint32_t wave_reservoir(const fw_kargs& a, const float* sums, const uint32_t nb, const float S_last,
                                                   const uint4 d, const uint32_t walker, const uint32_t step, const uint32_t seq,
                                                   const uint32_t sbase, const uint32_t lane, float& tu_out, float& total) {
  const uint32_t at = 32u * (lane >> 4) + (lane & 15u);  // of the lane's sum in four blocks of sums
  uint32_t c0 = 0u;  // first of the four blocks in registers
  float s = 0.0f, T = 0.0f;
  if ((lane >> 4) < nb) {
    s = sums[at];
    T = sums[at + 16u];
  }
  WavePairs pairs{d, seq, 0u};
  float Sj = 0.0f, u = 1.0f, tu = 0.0f;
  uint32_t k = 0u;
  float Tk = 0.0f;
  while (S_last * u > Sj) {
    uint64_t m = __ballot(s * u > Sj);
    if (m == 0ull) {  // behind the blocks in registers: 64 blocks' last sums at a time, then the four blocks from the first that passes
      uint32_t lo = c0 + 4u, hi = nb - 1u;
      while (hi - lo >= 4u) {
        const uint32_t stride = (hi - lo + 64u) >> 6;
        uint32_t b = lo + (lane + 1u) * stride - 1u;
        b = b < hi ? b : hi;
        const uint32_t f = (uint32_t)__builtin_ctzll(__ballot(sums[32u * b + 15u] * u > Sj || b == hi));
        hi = readlane_u32(b, f);
        lo = f != 0u ? readlane_u32(b, f - 1u) + 1u : lo;
      }
      c0 = lo;
      s = T = 0.0f;
      if (c0 + (lane >> 4) < nb) {
        s = sums[32u * c0 + at];
        T = sums[32u * c0 + at + 16u];
      }
      m = __ballot(s * u > Sj);
    }
    const uint32_t l = (uint32_t)__builtin_ctzll(m | (1ull << 63));
    k = 16u * c0 + l;
    Sj = readlane_f(s, (int)l);
    Tk = readlane_f(T, (int)l);
    next_pair(pairs, a, walker, step, sbase, lane, tu, u);
  }
  tu_out = tu;
  total = Tk;
  return k;
}

// table_pick by a wave: everything but the lanes' own pieces is the same in all lanes.
__device__ __forceinline__ int32_t wave_pick(const fw_kargs& a, const fw_table_args& tb, const uint4 rec, const uint4 d,
                                             const uint32_t walker, const uint32_t step, const uint32_t sbase, const uint32_t lane) {
  const uint32_t nq = list_quartets(rec.w, rec.y);
  const unsigned char* entries = tb.data + (uint64_t)(rec.x & ~kUneven) * 128u;
  uint32_t nqg = nq;
  float T = __uint_as_float(rec.z), tu;
  bool uneven = (rec.x & kUneven) != 0u;
  if (nq <= kGq) {
    tu = u24(readlane_u32(d.x, 0u));
  } else {
    const uint32_t ngroups = (nq + kGq - 1u) / kGq;
    const bool wg = (int32_t)rec.y > a.hub_threshold;
    const uint32_t nb = seq_blocks(ngroups, wg, tb.nw_shift);
    const float* sums = reinterpret_cast<const float*>(entries);
    uint32_t seq = 0u;
    float S_last = T;
    if (wg) {  // which sequence, then the reservoir over it with draws of its own stream
      const float target = u24(readlane_u32(d.x, kWaveLane)) * T;
      seq = (uint32_t)__builtin_popcountll(__ballot(lane < 16u && sums[lane & 15u] <= target));
      sums += 32u + 32u * nb * seq;
      S_last = sums[32u * (nb - 1u) + 15u];
    }
    const uint32_t k = wave_reservoir(a, sums, nb, S_last, d, walker, step, seq, sbase, lane, tu, T);
    const uint32_t g = wg ? seq + (k << tb.nw_shift) : k;
    entries += (uint64_t)32u * (header_units(ngroups, wg, tb.nw_shift) + kGroupUnits * g);
    nqg = nq - g * kGq < kGq ? nq - g * kGq : kGq;
    uneven = T < 0.0f;
    T = __builtin_fabsf(T);
  }
  const float t = tu * T;
  // Two pairs a lane, from some before the guess on, which mostly hold the one; what else may be needed stands out of the way, since the first look is all that
  // a step mostly pays for (walks of 80 steps, look and repeats in one loop / so: 100 walkers on a small graph 67.6 / 64.9 us, 1,000 on R-MAT 20 113.8 / 109.3).  Of an uneven
  // group row M comes at the same time (after it, as the pairs' place was found: log-normal weights with sigma 2, 1,000 walkers on R-MAT 20 129 us, now 121).
  const uint4* pairs = reinterpret_cast<const uint4*>(entries);
  const uint32_t n2 = 2u * nqg;
  const uint32_t guess = (uint32_t)(tu * (float)n2);
  const uint32_t wmax = n2 > 64u ? n2 - 64u : 0u;
  uint32_t w = guess > 32u ? guess - 32u : 0u;
  w = w < wmax ? w : wmax;
  uint4 p = make_uint4(0x7F800000u, 0u, 0x7F800000u, 0u);
  if (w + lane < n2) p = pairs[w + lane];
  float m = kInf;
  if (lane < (uneven ? nqg : 0u)) m = reinterpret_cast<const float*>(entries + 32u * nqg)[lane];
  uint64_t m0 = __ballot(!(__uint_as_float(p.x) <= t)), above = m0 | __ballot(!(__uint_as_float(p.z) <= t));
  if (__builtin_expect(uneven || above == 0ull || ((m0 & 1ull) != 0ull && w != 0u), 0)) {
    if (uneven) {  // it names the lane whose pairs they are
      const uint32_t l = (uint32_t)__builtin_ctzll(__ballot(!(m <= t)) | (1ull << 63));
      const uint32_t first = 2u * lane_start(l, nqg);
      if (first < w || 2u * lane_start(l + 1u, nqg) > w + 64u) {
        w = first < wmax ? first : wmax;
        if (w + lane < n2) p = pairs[w + lane];
        m0 = __ballot(!(__uint_as_float(p.x) <= t));
        above = m0 | __ballot(!(__uint_as_float(p.z) <= t));
      }
    } else {  // the pieces next to these (those of a group that is not marked are at most 48 from the guess: one look more)
      for (uint32_t lo = 0u;;) {
        if (above == 0ull) {  // (the last pair's key is above: there are more)
          lo = w = w + 64u;
        } else if ((m0 & 1ull) != 0ull && w > lo) {
          w = w > lo + 63u ? w - 63u : lo;
        } else {
          break;
        }
        p = make_uint4(0x7F800000u, 0u, 0x7F800000u, 0u);
        if (w + lane < n2) p = pairs[w + lane];
        m0 = __ballot(!(__uint_as_float(p.x) <= t));
        above = m0 | __ballot(!(__uint_as_float(p.z) <= t));
      }
    }
  }
  const uint32_t f = (uint32_t)__builtin_ctzll(above);
  return (int32_t)(((m0 >> f) & 1ull) != 0ull ? readlane_u32(p.y, f) : readlane_u32(p.w, f));
}

// set_find by a wave, from the lane's place of the bucket (lanes 0 .. 15)
__device__ __forceinline__ int64_t wave_set_find(const int32_t* __restrict__ sets, uint32_t v, uint32_t off, uint32_t deg, int32_t target,
                                                 uint32_t lane) {
  const uint64_t first = 16u * (fw_set_first(off, v) + set_bucket(target, fw_set_buckets(deg)));
  const int32_t x = sets[first + (lane & 15u)];
  const uint32_t hit = (uint32_t)__ballot(x == target) & 0xFFFFu;
  if (hit != 0u) return (int64_t)first + __builtin_ctz(hit);
  return __builtin_amdgcn_readlane(x, 15) == kSetOverflow ? -2 : -1;
}

// One wave, one walker.  Bound: latency, two dependent reads a step (three and four on long lists; node2vec one more a trial): 1.25 us a step of
// 1,000 walkers on R-MAT 20, where a lane walked each 2.0 (100 walkers on a small graph 70.1 -> 64.6 us a call, 1,000 from hubs 124.2 -> 113.7, since only marked groups read row M).
template <int kApp>
__global__ __launch_bounds__(256, kWalkerWaves) void fw_table_walk_wave(const fw_kargs a, const fw_table_args tb) {
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t md = (uint32_t)a.max_depth;
  const uint32_t q = blockIdx.x * 4u + uniform_u32(threadIdx.x >> 6);
  if (q >= (uint32_t)a.n) return;
  uint32_t n_steps = 0u, n_hub = 0u;
  unsigned long long n_edges = 0ull, hub_edges = 0ull;
  const uint32_t walker = a.walker_base + q;
  int32_t* const path = a.paths + (uint64_t)q * md;
  uint32_t v = uniform_u32((uint32_t)a.starts[q]);
  int32_t mine = lane == 0u ? (int32_t)v : -1;  // the path's entry of the lane's place among the 64 that are not stored yet
  uint32_t len = 1u, kept = 0u;  // entries, and those that are stored
  if (v < (uint32_t)a.V && md > 1u) {
    uint32_t prev_off = 0u, prev_deg = 0u;
    int32_t prev = -1;
    uint4 r = tb.vrec[v];
    for (bool ended = false; !ended;) {
      const uint32_t step = len - 1u;
      uint4 d = wave_draws(a, walker, step, 0u, lane);
      const uint4 rec = make_uint4(uniform_u32(r.x), uniform_u32(r.y), uniform_u32(r.z), uniform_u32(r.w));
      if (!(__uint_as_float(rec.z) > 0.0f)) break;  // no neighbour with a positive bias (include/walker.cuh:1373-1374)
      int32_t nv = wave_pick(a, tb, rec, d, walker, step, 0u, lane);
      if (kApp == FW_APP_NODE2VEC && prev >= 0) {
        float w_ret = 0.0f;
        if (a.n2v_extra > 0.0f) {
          const int64_t at = tb.set_weights != nullptr ? wave_set_find(tb.sets, v, rec.w, rec.y, prev, lane) : -2;
          if (at >= 0) w_ret = tb.set_weights[at];
          if (at == -2) w_ret = return_weight(a.adjncy + rec.w, a.weight + rec.w, rec.y, prev);
        }
        for (uint32_t trial = 0u;;) {
          r = tb.vrec[(uint32_t)nv < (uint32_t)a.V ? (uint32_t)nv : v];  // mostly the next vertex: on its way during the test
          const uint4 bits = make_uint4(readlane_u32(d.x, kAcceptLane), readlane_u32(d.y, kAcceptLane), 0u, 0u);
          const N2vTest t = n2v_test(a, nv, prev, trial, __uint_as_float(rec.z), w_ret, [&] { return bits; });
          if (t.take_prev) {
            nv = prev;
            r = tb.vrec[(uint32_t)prev];
            break;
          }
          bool common = false;
          if (!t.decided) {
            const int64_t at = tb.sets != nullptr ? wave_set_find(tb.sets, (uint32_t)prev, prev_off, prev_deg, nv, lane) : -2;
            common = at >= 0;
            if (at == -2) common = sorted_contains(a.adjncy + prev_off, (int32_t)prev_deg, nv);
          }
          if (n2v_finish(a, t, common)) break;
          trial += 1u;
          d = wave_draws(a, walker, step, trial, lane);
          nv = wave_pick(a, tb, rec, d, walker, step, trial << 8, lane);
        }
      }
      if ((int32_t)rec.y > a.park_threshold) {
        n_hub += 1u;
        hub_edges += rec.y;
      } else {
        n_steps += 1u;
        n_edges += rec.y;
      }
      const bool loaded = kApp == FW_APP_NODE2VEC && prev >= 0;  // r is the new vertex's already
      if (kApp == FW_APP_NODE2VEC) {
        prev = (int32_t)v;
        prev_off = rec.w;
        prev_deg = rec.y;
      }
      v = (uint32_t)nv;
      len += 1u;
      ended = len >= md;
      if (kApp == FW_APP_PPR && !ended) ended = u24(readlane_u32(d.x, kStopLane)) < a.tp;  // include/app.cuh:88-94
      if (!ended && !loaded) r = tb.vrec[v];
      mine = lane == len - 1u - kept ? nv : mine;
      if (len - kept == 64u) {
        path[kept + lane] = mine;
        mine = -1;
        kept = len;
      }
    }
  }
  for (uint32_t p = kept + lane; p < md; p += 64u) {
    path[p] = mine;
    mine = -1;
  }
  if (lane == 0u) {
    unsigned long long* const c = &tb.counters[(blockIdx.x & (FW_TABLE_STRIPES - 1u)) * 8u];
    if (n_steps != 0u) {
      atomicAdd(&c[0], (unsigned long long)n_steps);
      atomicAdd(&c[1], n_edges);
    }
    if (n_hub != 0u) {
      atomicAdd(&c[2], (unsigned long long)n_hub);
      atomicAdd(&c[3], hub_edges);
    }
  }
}

// Around the walk: the counters start at zero, and their sums go to the host (pinned memory: the call waits for the stream
// anyway, and a copy of its own would cost a small call as much as its launch).
__global__ void fw_table_begin_kernel(unsigned long long* counters, uint32_t* scratch, uint32_t words) {
  for (uint32_t i = threadIdx.x; i < FW_TABLE_STRIPES * 8u; i += blockDim.x) counters[i] = 0ull;
  for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) scratch[i] = 0u;
}
__global__ __launch_bounds__(64) void fw_table_end_kernel(const unsigned long long* __restrict__ counters, unsigned long long* out) {
  unsigned long long c[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    c[k] = counters[threadIdx.x * 8u + (uint32_t)k];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) c[k] += __shfl_xor(c[k], d);
  }
  if (threadIdx.x == 0u) {
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = c[k];
  }
}

template <int kApp>
int launch_table_walk(const fw_kargs& a, fw_table_args tb, int grid, hipStream_t stream, int* grid_used) {
  int dev = 0, cus = 0;
  FW_HIP(hipGetDevice(&dev));
  FW_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const uint32_t n = (uint32_t)a.n;
  uint64_t waves;
  if constexpr (kApp != FW_APP_METAPATH) {  // (whose step is two reads, and no search)
    // As many walkers as there are waves resident: a wave each.  Measured, wave per walker / lane per walker, us of a call of 40 steps on R-MAT 20,
    // symmetrised: 1,000 walkers DeepWalk 62 / 89, PPR 53 / 81, node2vec 109 / 172; 8,000: 100 / 145, 61 / 88, 174 / 280 (q = 4: 457 / 704); twice as many walkers as
    // waves fit (16,000): 146 / 162, 67 / 94, 269 / 328, where the line does not lie yet; a uniform graph of mean degree 4: 1,000 47 / 68, 39 / 54, 74 / 91; 8,192 DeepWalk 78 / 85, PPR 50 / 71.
    // Lists of one group leave a wave little to search, and node2vec's tests are made for one walker at a time, so where few proposals are turned down fewer waves
    // per SIMD already cost more than lanes do.  Uniform graphs of mean degree 4 and 40, q = 0.5: 6,144 walkers 124 / 120 and 125 / 131, 7,000 135 / 120 and 136 / 132, 8,192 142 / 122 and 147 / 135;
    // without adjacency tests, p = 1, q = 1: 4,096 91 / 91 and 94 / 98, 5,500 113 / 94 and 115 / 102.  Before waves and lanes searched from the guess, some lists of two groups, p = q = 1: mean list
    // 144 (R-MAT 14) 5,500 105 / 94, 6,144 111 / 96; mean list 192 (R-MAT 12) 6,144 119 / 109, but with p = 2 123 / 128.  With q = 2 on these, on lists of 300 on average, and for
    // DeepWalk waves win throughout.
    uint32_t per_simd = kWalkerWaves;
    if (kApp == FW_APP_NODE2VEC && a.inv_q >= 1.0f && tb.mean_list > 0.0f && tb.mean_list <= 256.0f)
      per_simd = a.inv_q == 1.0f ? (tb.long_lists == 0u ? 4u : 5u) : (tb.long_lists == 0u ? 6u : kWalkerWaves);
    if (grid <= 0 && n <= (uint32_t)cus * 4u * per_simd) {
      const unsigned blocks = (n + 3u) / 4u;
      hipLaunchKernelGGL((fw_table_walk_wave<kApp>), dim3(blocks), dim3(256), 0, stream, a, tb);
      FW_HIP(hipGetLastError());
      if (grid_used) *grid_used = (int)blocks;
      return FW_OK;
    }
  }
  if (grid > 0) {
    waves = (uint64_t)grid * 4u;
    tb.lanes = 64u;
  } else {
    // few queries are spread over the chip, down to one lane per wave for MetaPath and a few for the others: their walks are chains of dependent
    // look-ups, and a wave waits for the slowest of its lanes (16 waves per CU instead of 8: 16,000 to 200,000 walkers within 5 % either way)
    const uint32_t spread = (uint32_t)cus * 8u;
    tb.lanes = n / spread < 64u ? n / spread + 1u : 64u;
    if (tb.lanes > 64u) tb.lanes = 64u;
    waves = ((uint64_t)n + tb.lanes - 1u) / tb.lanes;
    // many: as many waves as fit, and a wave takes as many queries as it has lanes from the dispenser whenever its own are
    // used up, so that lanes are idle only at the very end (waves with a fixed share of the queries each idled for 30 % of
    // their lanes' time, when the last of a share walked: DeepWalk R-MAT 24 76.6 -> 47.9 ms, R-MAT 22 9.86 -> 6.79, PPR
    // there 1.62 -> 1.16)
    const uint64_t most = (uint64_t)cus * 4u * kWaves;
    if (waves > most) waves = most;
  }
  if (tb.lanes < 64u) tb.rows_near = 1u;  // (see row_eighths)
  const unsigned blocks = (unsigned)((waves + 3u) / 4u);
  // Blocks of pairs from gigabytes of regions are not kept in the L2 where many walkers ask for them.  Kept / not kept, us, walks of 80 steps, 40 for node2vec: R-MAT 24
  // (2.7 GB) DeepWalk 20,000 walkers 306 / 341, 50,000 383 / 399, 200,000 561 / 572, 400,000 769 / 797, 1,000,000 1682 / 1608, from 2,048 hubs 3166 / 2964; symmetrised (5.2 GB) 200,000
  // 672 / 688, 400,000 1409 / 1365, 1,000,000 2683 / 2524, from hubs 4214 / 3865; node2vec there 200,000 968 / 991, 400,000 1064 / 1066, 1,000,000 of 20 steps from hubs 1426 / 1404;
  // R-MAT 23 symmetrised (2.7 GB) DeepWalk 200,000 640 / 657, 400,000 1368 / 1345, 1,000,000 2511 / 2379, node2vec 400,000 1047 / 1063.  PPR gains nowhere, its walks are short:
  // 200,000 walkers on R-MAT 24 179 / 195, 1,000,003 from the longest list 539 / 548, 4,000,000 1067 / 1069, all 16,777,216 3632 / 3672; symmetrised 224 / 243, 614 / 621, 1172 / 1178.
  // node2vec that has no hash sets yet searches lists for its tests, which the L2 then holds more of: R-MAT 24 50,021 walkers of 41 steps 502 / 470, 129,000 635 / 625, log-normal weights
  // with sigma 1 50,021 550 / 519, R-MAT 23 symmetrised 744 / 740, 892 / 902, R-MAT 24 symmetrised 769 / 778, 912 / 930; with sets 50,021 on R-MAT 24 285 / 293.
  constexpr uint32_t kStreamWalkers = 1u << 19;
  if constexpr (kApp == FW_APP_DEEPWALK || kApp == FW_APP_NODE2VEC) {
    if (tb.stream_pairs != 0u && (n >= kStreamWalkers || (kApp == FW_APP_NODE2VEC && tb.sets == nullptr))) {
      hipLaunchKernelGGL((fw_table_walk<kApp, true>), dim3(blocks), dim3(256), 0, stream, a, tb);
      FW_HIP(hipGetLastError());
      if (grid_used) *grid_used = (int)blocks;
      return FW_OK;
    }
  }
  hipLaunchKernelGGL((fw_table_walk<kApp, false>), dim3(blocks), dim3(256), 0, stream, a, tb);
  FW_HIP(hipGetLastError());
  if (grid_used) *grid_used = (int)blocks;
  return FW_OK;
}

}  // namespace

int fw_launch_table_walk(const fw_kargs& a, const fw_table_args& tb, int app, int grid, hipStream_t stream, int* grid_used) {
  switch (app) {
    case FW_APP_DEEPWALK: return launch_table_walk<FW_APP_DEEPWALK>(a, tb, grid, stream, grid_used);
    case FW_APP_PPR: return launch_table_walk<FW_APP_PPR>(a, tb, grid, stream, grid_used);
    case FW_APP_NODE2VEC: return launch_table_walk<FW_APP_NODE2VEC>(a, tb, grid, stream, grid_used);
    case FW_APP_METAPATH: return launch_table_walk<FW_APP_METAPATH>(a, tb, grid, stream, grid_used);
    default:
      fw_set_error("no list tables for app %d", app);
      return FW_ERR_INVALID;
  }
}

int fw_table_begin(unsigned long long* d_counters, uint32_t* d_scratch, uint32_t words, hipStream_t stream) {
  hipLaunchKernelGGL(fw_table_begin_kernel, dim3(1), dim3(512), 0, stream, d_counters, d_scratch, words);
  FW_HIP(hipGetLastError());
  return FW_OK;
}

int fw_table_end(const unsigned long long* d_counters, unsigned long long* h_out, hipStream_t stream) {
  static_assert(FW_TABLE_STRIPES == 64u, "one lane per line of counters");
  hipLaunchKernelGGL(fw_table_end_kernel, dim3(1), dim3(64), 0, stream, d_counters, h_out);
  FW_HIP(hipGetLastError());
  return FW_OK;
}

int fw_table_plan(const fw_graph* g, int32_t hub_threshold, uint32_t nw_shift, int n_labels, uint32_t* d_blocks, uint32_t* d_longs, uint2* d_items, uint32_t* d_ctrs,
                  hipStream_t stream) {
  hipLaunchKernelGGL(fw_table_plan_kernel, dim3(1024), dim3(1024), 0, stream, g->xadj, g->V, hub_threshold, nw_shift, (uint32_t)n_labels, d_blocks,
                     d_longs, d_items, d_ctrs);
  FW_HIP(hipGetLastError());
  return FW_OK;
}

int fw_table_make(const fw_graph* g, fw_tables* t, hipStream_t stream, int* launches) {
  int cus = 0;
  FW_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device));
  auto grid_for = [&](uint64_t waves) {
    const uint64_t blocks = (waves + 3u) / 4u, most = (uint64_t)cus * 64u;
    return (unsigned)(blocks < most ? (blocks ? blocks : 1u) : most);
  };
  hipLaunchKernelGGL(fw_table_lists_kernel, dim3(grid_for(((uint64_t)g->V + 63u) / 64u)), dim3(256), 0, stream, g->xadj, g->adjncy,
                     g->weight, g->V, t->blocks, t->vrec, t->data, t->flag);
  FW_HIP(hipGetLastError());
  *launches += 1;
  if (t->n_longs != 0u) {
    hipLaunchKernelGGL(fw_table_groups_kernel, dim3(grid_for(t->n_items)), dim3(256), 0, stream, t->vrec, g->adjncy, g->weight,
                       t->items, t->n_items, t->hub_threshold, t->nw_shift, t->data, t->flag);
    FW_HIP(hipGetLastError());
    hipLaunchKernelGGL(fw_table_sums_kernel, dim3(grid_for(t->n_longs)), dim3(256), 0, stream, t->vrec, t->longs, t->n_longs,
                       t->hub_threshold, t->nw_shift, t->data, t->flag);
    FW_HIP(hipGetLastError());
    *launches += 2;
  }
  return FW_OK;
}

int fw_label_tables_make(const fw_graph* g, fw_tables* t, hipStream_t stream, int* launches) {
  int cus = 0;
  FW_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device));
  auto grid_for = [&](uint64_t waves) {
    const uint64_t blocks = (waves + 3u) / 4u, most = (uint64_t)cus * 64u;
    return (unsigned)(blocks < most ? (blocks ? blocks : 1u) : most);
  };
  auto make = [&](auto words) -> int {
    constexpr int kW = decltype(words)::value;
    hipLaunchKernelGGL((fw_label_lists_kernel<kW>), dim3(grid_for(((uint64_t)g->V + 63u) / 64u)), dim3(256), 0, stream, g->xadj,
                       g->adjncy, g->label, g->V, t->labels, t->blocks, t->vrec, t->by_label);
    FW_HIP(hipGetLastError());
    if (t->n_longs != 0u)
      hipLaunchKernelGGL((fw_label_groups_kernel<kW>), dim3(grid_for(t->n_items)), dim3(256), 0, stream, t->vrec, g->adjncy,
                         g->label, t->items, t->n_items, t->labels, t->hub_threshold, t->nw_shift, t->data, t->by_label);
    FW_HIP(hipGetLastError());
    return FW_OK;
  };
  const int n = t->labels.n;
  const int rc = n <= 2 ? make(std::integral_constant<int, 1>()) : n <= 4 ? make(std::integral_constant<int, 2>())
                 : n <= 6 ? make(std::integral_constant<int, 3>()) : make(std::integral_constant<int, 4>());
  if (rc != FW_OK) return rc;
  *launches += 1;
  if (t->n_longs != 0u) {
    hipLaunchKernelGGL(fw_label_sums_kernel, dim3(grid_for((uint64_t)t->n_longs * (uint64_t)t->labels.n)), dim3(256), 0, stream,
                       t->vrec, t->longs, t->n_longs, (uint32_t)t->labels.n, t->hub_threshold, t->nw_shift, t->data);
    FW_HIP(hipGetLastError());
    *launches += 2;
  }
  return FW_OK;
}

int fw_sets_make(const fw_graph* g, const fw_tables* t, hipStream_t stream, int* launches) {
  int cus = 0;
  FW_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device));
  const uint64_t blocks = (((uint64_t)g->V + 63u) / 64u + 3u) / 4u, most = (uint64_t)cus * 64u;
  hipLaunchKernelGGL(fw_sets_small_kernel, dim3((unsigned)(blocks < most ? blocks : most)), dim3(256), 0, stream, t->vrec, g->adjncy,
                     g->weight, g->V, t->sets, t->set_weights);
  FW_HIP(hipGetLastError());
  *launches += 1;
  if (t->n_items != 0u) {
    hipLaunchKernelGGL(fw_sets_long_kernel, dim3(t->n_items < most ? t->n_items : (unsigned)most), dim3(512), 0, stream, t->vrec,
                       g->adjncy, g->weight, t->items, t->n_items, t->sets, t->set_weights);
    FW_HIP(hipGetLastError());
    *launches += 1;
  }
  return FW_OK;
}
