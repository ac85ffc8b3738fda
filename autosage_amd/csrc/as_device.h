// Device-side helpers for gfx950 (wave64) kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace as {

__device__ __forceinline__ int lane_id() { return static_cast<int>(threadIdx.x & 63u); }
__device__ __forceinline__ int wave_in_block() { return static_cast<int>(threadIdx.x >> 6); }

// Broadcast lane `src` (wave-uniform) of v to the whole wave through an SGPR.
__device__ __forceinline__ int bcast_i32(int v, int src) {
  return __builtin_amdgcn_readlane(v, src);
}
__device__ __forceinline__ float bcast_f32(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
__device__ __forceinline__ int uniform_i32(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}
// A 64-bit value every lane holds identically, moved to SGPRs so that
// control flow and address arithmetic on it stay scalar.
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
  const uint64_t u = static_cast<uint64_t>(v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(u));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(u >> 32));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}
// Element offset of row c in a row-major [*, F] matrix, for c < 2^31 and
// F < 2^31 (one 32x32->64 multiply).
__device__ __forceinline__ int64_t row_offset(int c, int64_t F) {
  return static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(c)) *
                              static_cast<uint64_t>(static_cast<uint32_t>(F)));
}

// V consecutive floats owned by one lane.  Component-wise arithmetic is
// written out so that no packed-fp32 instruction is needed.
template <int V>
struct alignas(4 * V) FVec {
  float v[V];
};

template <int V>
__device__ __forceinline__ FVec<V> load_vec(const float* p) {
  return *reinterpret_cast<const FVec<V>*>(p);
}
// Load from a wave-uniform base plus a per-lane byte offset below 2^32, the
// shape of the SGPR-base global load.
template <int V>
__device__ __forceinline__ FVec<V> load_vec_off(const float* base, uint32_t byte_offset) {
  return *reinterpret_cast<const FVec<V>*>(reinterpret_cast<const char*>(base) + byte_offset);
}
template <int V>
__device__ __forceinline__ void store_vec(float* p, const FVec<V>& a) {
  *reinterpret_cast<FVec<V>*>(p) = a;
}

// Butterfly reductions over the 64 lanes: every lane ends with the same bits
// (each step adds a pair in both lanes, and fp32 addition is commutative).
__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max_f32(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ int wave_sum_i32(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// Inclusive prefix sum over the wave (Hillis-Steele with shfl_up).
__device__ __forceinline__ int wave_incl_scan_i32(int v) {
  const int lane = lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// ---- rows of edges ------------------------------------------------------------
// Lane i: the row of edge b + min(i, cnt - 1), given r, the row of edge b.
// Every lane of the wave must be active.  The rounds end at the last row
// whatever crow holds, and the result is clamped to [0, n).
__device__ __forceinline__ int block_edge_rows(const int64_t* __restrict__ crow, int64_t n, int64_t b, int cnt,
                                               int64_t r) {
  const int lane = lane_id();
  const int i = lane < cnt ? lane : cnt - 1;
  int row = -1;
  for (int64_t rr = r;; rr += 64) {
    // rel: where row rr + lane ends (row n - 1 for lanes past it), relative
    // to b, clamped to [0, 64]
    const int64_t left = n - 1 - rr;  // >= 0
    const int lim = left < 64 ? static_cast<int>(left) : 64;
    const int64_t d = crow[rr + 1 + (lane < lim ? lane : lim)] - b;
    const int rel = d < 0 ? 0 : (d > 64 ? 64 : static_cast<int>(d));
    // pos = #{l : rel_l <= i}, the ends being non-decreasing in l
    int pos = 0;
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) {
      const int v = __builtin_amdgcn_ds_bpermute((pos + s - 1) * 4, rel);
      pos = v <= i ? pos + s : pos;
    }
    const int rel_last = __builtin_amdgcn_readlane(rel, 63);
    if (pos == 63 && rel_last <= i) pos = 64;
    if (row < 0 && pos < 64) row = static_cast<int>(rr + pos);
    if (rel_last >= cnt || rr + 64 >= n) break;
  }
  const int last = static_cast<int>(n - 1);
  return row < 0 || row > last ? last : row;
}

// The row holding edge e: the last r < n with crow[r] <= e (0 if none), by
// the whole wave, 64 probes a step; ends after log64(n) steps whatever crow
// holds.
__device__ __forceinline__ int64_t wave_row_of_edge(const int64_t* __restrict__ crow, int64_t n, int64_t e) {
  int64_t lo = 0;
  int64_t hi = n;
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + 63) / 64;
    const int64_t probe = lo + lane_id() * step;
    const uint64_t below = __ballot(probe < hi && crow[probe] <= e);
    if (below != 0) lo += static_cast<int64_t>(63 - __builtin_clzll(below)) * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

}  // namespace as
