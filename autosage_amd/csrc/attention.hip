// CSR row softmax and the SDDMM -> row softmax -> SpMM attention.
//
// Reference behaviour: _csr_row_softmax (autosage/_auto.py:744-759) and
// csr_attention_forward (autosage/_auto.py:762-780), which run as separate
// torch / native stages there.
//
// Row softmax (defines this library's denominator order):
//   m = max_e s_e                      (exact, order-free)
//   d = sum_e exp(s_e - m): chain l adds e = rs+l, rs+l+64, ... in order
//       (l < 64), then a 32/16/8/4/2/1 butterfly (identical bits in every lane)
//   p_e = exp(s_e - m) / d             (IEEE division)
//
// The exact attention runs the three stages in one call: the SDDMM (reference
// dot order) times `scale` into the workspace, the row softmax in place, the
// SpMM with the probabilities as weights (CSR order).  One kernel that did all
// three per row read the same rows of K and V, but a wave waited for its row's
// three passes in turn and a long row's chain for its gathers.  us, that kernel
// -> the stages (F_qk / F_v):
//   40k rows, 400k edges                     32/32 58 -> 43, 100/100 113 -> 69
//   170k rows, 2.4M edges, longest 10,000    64/64 651 -> 215, 40/47 1406 -> 213
//   1M rows, 16M edges, even                 64/64 1695 -> 1355, 64/128 2220 -> 1956
#include <type_traits>

#include "as_device.h"
#include "as_internal.h"
#include "elem16.h"

namespace as {

namespace {

// Rows of the fp32 softmax and of the softmax backward: a workgroup takes
// kSmRows consecutive rows.  Rows of at most kSmShort edges take 16 lanes each
// (8 a wave in 2 sets, one read of the row, an edge a lane and slot); rows up
// to kSmWaveRow edges a wave each, longer ones the whole workgroup.  All give the
// bits of one wave striding over the row: edge rs + l + 64k belongs to chain l,
// and the butterfly's first two steps (32, 16) are, for a short row, the sums
// of the slots of one lane.
//
// What bounds it: the chain row pointers -> edges -> butterfly -> store of the
// short rows, hidden by the rows in flight (1, 2, 3 sets of rows a wave: 1M
// rows, 16M edges, power law with hubs of 10,000 edges, 109 / 98 / 95 us
// forward, 88 / 73 / 68 backward; 233k rows of 200 edges 179 / 197 / 195), and
// the hubs' chains.  A wave per row with a pass per statistic took 367 and 269
// us there: most lanes idle, one load in flight, the scores read three times;
// with hubs of 200,000 edges (1M rows, 50M edges) 3353 and 2727 us against 388 and
// 324.
constexpr int kSmBatch = 2;                                   // sets of rows a wave has in flight
constexpr int kSmLanes = 16;
constexpr int kSmWaveRows = kSmBatch * kWave / kSmLanes;      // rows of one wave
constexpr int kSmRows = kWavesPerBlock * kSmWaveRows;
static_assert(kSmRows < kWave, "a wave reads the workgroup's row pointers with one load");
constexpr int kSmSlots = 4;
constexpr int kSmShort = kSmLanes * kSmSlots;
constexpr int kSmUnroll = 8;                       // loads in flight per lane on longer rows
constexpr int kSmChunk = kWave * kSmUnroll;        // edges per wave and step there
constexpr int64_t kSmWaveRow = 4096;

// The rows of one workgroup, as every wave of it sees them.
struct SoftmaxRows {
  int64_t start;   // lane i < kSmRows: where row i starts
  int64_t rs[kSmBatch];  // this lane group's rows: batch k, row 4k + group of the wave
  int len[kSmBatch];     // their edges if short rows, else 0
  uint64_t wave;   // bit i: row i is a wave's row and this wave's
  uint64_t block;  // bit i: row i is the workgroup's
};

__device__ __forceinline__ int64_t shfl_i64(int64_t v, int src) {
  return static_cast<int64_t>(__shfl(static_cast<long long>(v), src, kWave));
}

__device__ __forceinline__ SoftmaxRows softmax_rows(const int64_t* __restrict__ crow, int64_t n, int64_t row0) {
  const int lane = lane_id();
  const int wave = wave_in_block();
  const int64_t left = n - row0;
  SoftmaxRows s;
  s.start = crow[row0 + (lane < left ? lane : left)];
  const int64_t len = shfl_i64(s.start, lane < kWave - 1 ? lane + 1 : lane) - s.start;
  const int first = wave * kSmWaveRows;
  const bool mine = lane >= first && lane < first + kSmWaveRows;
  s.wave = __ballot(mine && len > kSmShort && len <= kSmWaveRow);
  s.block = __ballot(lane < kSmRows && len > kSmWaveRow);
#pragma unroll
  for (int k = 0; k < kSmBatch; ++k) {
    const int src = first + k * (kWave / kSmLanes) + lane / kSmLanes;
    s.rs[k] = shfl_i64(s.start, src);
    const int64_t l = shfl_i64(len, src);
    s.len[k] = l > 0 && l <= kSmShort ? static_cast<int>(l) : 0;
  }
  return s;
}

// Bounds of row i of the workgroup, wave-uniform.
__device__ __forceinline__ void softmax_row_bounds(const SoftmaxRows& s, int i, int64_t& rs, int64_t& re) {
  rs = uniform_i64(shfl_i64(s.start, i));
  re = uniform_i64(shfl_i64(s.start, i + 1));
}

// Butterfly over 16 lanes.  Rotations by 8, 4, 2, 1 pair the values that xor
// would: after a step of o the lanes a and a ^ o hold the same bits.
template <int CTRL>
__device__ __forceinline__ float row_ror(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float group_sum16(float v) {
  v += row_ror<0x128>(v);
  v += row_ror<0x124>(v);
  v += row_ror<0x122>(v);
  return v + row_ror<0x121>(v);
}
__device__ __forceinline__ float group_max16(float v) {
  v = fmaxf(v, row_ror<0x128>(v));
  v = fmaxf(v, row_ror<0x124>(v));
  v = fmaxf(v, row_ror<0x122>(v));
  return fmaxf(v, row_ror<0x121>(v));
}

// kSmUnroll values per lane from e on (fill past re).
__device__ __forceinline__ void softmax_load(const float* p, int64_t e, int64_t re, float fill,
                                             float (&v)[kSmUnroll]) {
#pragma unroll
  for (int i = 0; i < kSmUnroll; ++i) v[i] = e + i * kWave < re ? p[e + i * kWave] : fill;
}

__global__ __launch_bounds__(kBlock) void csr_row_softmax_kernel(const int64_t* __restrict__ crow,
                                                                 const float* scores, float* probs, int64_t n,
                                                                 int64_t block_base) {
  // probs may be scores: a thread writes an edge after its last look at it
  __shared__ float tile[kWavesPerBlock][kSmUnroll][kWave];
  __shared__ float wave_max[kWavesPerBlock];
  const int lane = lane_id();
  const int wave = wave_in_block();
  const SoftmaxRows rows = softmax_rows(crow, n, (block_base + blockIdx.x) * kSmRows);
  {
    const int gl = lane % kSmLanes;
    float v[kSmBatch][kSmSlots];
    bool any[kSmBatch][kSmSlots];  // wave-uniform: some row has an edge in slot i
#pragma unroll
    for (int k = 0; k < kSmBatch; ++k) {
#pragma unroll
      for (int i = 0; i < kSmSlots; ++i) {
        any[k][i] = __ballot(rows.len[k] > i * kSmLanes) != 0;
        v[k][i] = -INFINITY;
        if (any[k][i] && gl + i * kSmLanes < rows.len[k]) v[k][i] = scores[rows.rs[k] + gl + i * kSmLanes];
      }
    }
#pragma unroll
    for (int k = 0; k < kSmBatch; ++k) {
      const float m = group_max16(fmaxf(fmaxf(v[k][0], v[k][1]), fmaxf(v[k][2], v[k][3])));
#pragma unroll
      for (int i = 0; i < kSmSlots; ++i) {
        if (any[k][i]) v[k][i] = gl + i * kSmLanes < rows.len[k] ? expf(v[k][i] - m) : 0.f;
        else v[k][i] = 0.f;
      }
      const float d = group_sum16((v[k][0] + v[k][2]) + (v[k][1] + v[k][3]));
#pragma unroll
      for (int i = 0; i < kSmSlots; ++i) {
        if (any[k][i] && gl + i * kSmLanes < rows.len[k]) probs[rows.rs[k] + gl + i * kSmLanes] = v[k][i] / d;
      }
    }
  }
  float v[kSmUnroll];
  for (uint64_t left = rows.wave; left != 0; left &= left - 1) {
    int64_t rs, re;
    softmax_row_bounds(rows, __builtin_ctzll(left), rs, re);
    const bool once = re - rs <= kSmChunk;  // the row stays in registers
    float m = -INFINITY;
    for (int64_t e = rs + lane; e < re; e += kSmChunk) {
      softmax_load(scores, e, re, -INFINITY, v);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) m = fmaxf(m, v[i]);
    }
    m = wave_max_f32(m);
    float d = 0.f;
    for (int64_t e = rs + lane; e < re; e += kSmChunk) {
      if (!once) softmax_load(scores, e, re, -INFINITY, v);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        v[i] = e + i * kWave < re ? expf(v[i] - m) : 0.f;
        d += v[i];
      }
    }
    d = wave_sum_f32(d);
    for (int64_t e = rs + lane; e < re; e += kSmChunk) {
      if (!once) softmax_load(scores, e, re, -INFINITY, v);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        if (e + i * kWave < re) probs[e + i * kWave] = (once ? v[i] : expf(v[i] - m)) / d;
      }
    }
  }
  for (uint64_t left = rows.block; left != 0; left &= left - 1) {  // the same rows in every wave
    int64_t rs, re;
    softmax_row_bounds(rows, __builtin_ctzll(left), rs, re);
    constexpr int64_t kStep = kWavesPerBlock * kSmChunk;
    const int64_t e0 = rs + wave * kSmChunk + lane;
    float m = -INFINITY;
    for (int64_t e = e0; e < re; e += kStep) {
      softmax_load(scores, e, re, -INFINITY, v);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) m = fmaxf(m, v[i]);
    }
    m = wave_max_f32(m);
    if (lane == 0) wave_max[wave] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; ++w) m = fmaxf(m, wave_max[w]);
    // the waves share the exponentials (left in probs), every wave adds them
    // in the chains' order
    float d = 0.f;
    softmax_load(scores, e0, re, -INFINITY, v);
    for (int64_t t = rs; t < re; t += kStep) {
      const int64_t e = e0 + (t - rs);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        const bool in = e + i * kWave < re;
        const float x = in ? expf(v[i] - m) : 0.f;
        if (in) probs[e + i * kWave] = x;
        tile[wave][i][lane] = x;
      }
      softmax_load(scores, e + kStep, re, -INFINITY, v);
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; ++w) {
#pragma unroll
        for (int i = 0; i < kSmUnroll; ++i) d += tile[w][i][lane];
      }
      __syncthreads();
    }
    d = wave_sum_f32(d);
    for (int64_t e = e0; e < re; e += kStep) {
      softmax_load(probs, e, re, 0.f, v);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        if (e + i * kWave < re) probs[e + i * kWave] = v[i] / d;
      }
    }
  }
}

// The same row softmax on bf16 / fp16 scores: each score converts exactly to
// fp32, m, d and p_e are computed in fp32 and p_e is rounded to the 16-bit
// type (round to nearest even) once.  Rows of at most kSm16GroupDegree edges
// take a group of 16 lanes (4 rows per wave, csr_row_softmax16_grouped_kernel),
// longer rows a wave each with a running max and sum (csr_row_softmax16_kernel);
// the sums of d differ in order from the fp32 kernel's, which can move a
// result by one 16-bit unit near a tie.
constexpr int64_t kSm16GroupDegree = 64;
constexpr int kSm16Group = 16;

template <typename T>
__global__ __launch_bounds__(kBlock) void csr_row_softmax16_grouped_kernel(const int64_t* __restrict__ crow,
                                                                           const T* __restrict__ scores,
                                                                           uint16_t* __restrict__ probs, int64_t n,
                                                                           int64_t idx_base) {
  constexpr int kRowsPerWave = kWave / kSm16Group;
  const int lane = lane_id();
  const int g = lane / kSm16Group;
  const int gl = lane % kSm16Group;
  const int64_t row =
      (idx_base + static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave_in_block()) * kRowsPerWave + g;
  int64_t rs = 0, re = 0;
  if (row < n) {
    rs = crow[row];
    re = crow[row + 1];
    if (re - rs > kSm16GroupDegree) re = rs;  // a whole wave takes it
  }
  // a lane holds its <= 4 scores: one read of the row, one exp per score
  constexpr int kPer = static_cast<int>(kSm16GroupDegree / kSm16Group);
  float v[kPer];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int64_t e = rs + gl + i * kSm16Group;
    v[i] = e < re ? Elem<T>::at(scores, e) : -INFINITY;
    m = fmaxf(m, v[i]);
  }
#pragma unroll
  for (int o = 1; o < kSm16Group; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
  float d = 0.f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int64_t e = rs + gl + i * kSm16Group;
    v[i] = e < re ? expf(v[i] - m) : 0.f;
    d += v[i];
  }
#pragma unroll
  for (int o = 1; o < kSm16Group; o <<= 1) d += __shfl_xor(d, o, kWave);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int64_t e = rs + gl + i * kSm16Group;
    if (e < re) probs[e] = Elem<T>::bits(static_cast<double>(v[i] / d));
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void csr_row_softmax16_kernel(const int64_t* __restrict__ crow,
                                                                   const T* __restrict__ scores,
                                                                   uint16_t* __restrict__ probs, int64_t n,
                                                                   int64_t idx_base) {
  const int lane = lane_id();
  const int64_t row = idx_base + static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave_in_block();
  if (row >= n) return;
  const int64_t rs = uniform_i64(crow[row]);
  const int64_t re = uniform_i64(crow[row + 1]);
  if (re - rs <= kSm16GroupDegree) return;  // the grouped kernel takes it
  // one read for m and d: each lane keeps a running max and the sum of
  // exp(s - max), rescaled when the max grows; the lanes then merge
  float m = -INFINITY;
  float d = 0.f;
  for (int64_t e = rs + lane; e < re; e += kWave) {
    const float v = Elem<T>::at(scores, e);
    if (v > m) {
      d = d * expf(m - v) + 1.f;
      m = v;
    } else if (v != -INFINITY) {  // -inf adds nothing (and -inf - -inf is NaN)
      d += expf(v - m);
    }
  }
  const float mw = wave_max_f32(m);
  d = m == -INFINITY ? 0.f : d * expf(m - mw);
  d = wave_sum_f32(d);
  for (int64_t e = rs + lane; e < re; e += kWave)
    probs[e] = Elem<T>::bits(static_cast<double>(expf(Elem<T>::at(scores, e) - mw) / d));
}

// Backward of the row softmax: given p = softmax(s) and dp = dL/dp,
//   t = sum_e dp_e · p_e   (lane l: e = rs+l, rs+l+64, ... with fmaf, in
//                           order; then the 32/16/8/4/2/1 butterfly)
//   ds_e = p_e · (dp_e - t)
// in fp32 (16-bit inputs convert exactly; each ds_e is rounded once).
template <typename T>
__device__ __forceinline__ float sm_load(const T* __restrict__ p, int64_t e) {
  if constexpr (std::is_same<T, float>::value) return p[e];
  else return Elem<T>::at(p, e);
}
template <typename T>
__device__ __forceinline__ void sm_store(T* __restrict__ p, int64_t e, float v) {
  if constexpr (std::is_same<T, float>::value) p[e] = v;
  else p[e].bits = Elem<T>::bits(static_cast<double>(v));
}

template <typename T>
__device__ __forceinline__ void softmax_load2(const T* __restrict__ probs, const T* __restrict__ grad, int64_t e,
                                              int64_t re, float (&p)[kSmUnroll], float (&g)[kSmUnroll]) {
#pragma unroll
  for (int i = 0; i < kSmUnroll; ++i) {
    const bool in = e + i * kWave < re;
    p[i] = in ? sm_load(probs, e + i * kWave) : 0.f;
    g[i] = in ? sm_load(grad, e + i * kWave) : 0.f;
  }
}

// The rows of csr_row_softmax_kernel.
template <typename T>
__global__ __launch_bounds__(kBlock) void csr_row_softmax_backward_kernel(const int64_t* __restrict__ crow,
                                                                          const T* __restrict__ probs,
                                                                          const T* __restrict__ grad,
                                                                          T* __restrict__ grad_scores, int64_t n,
                                                                          int64_t block_base) {
  __shared__ float tile_p[kWavesPerBlock][kSmUnroll][kWave];
  __shared__ float tile_g[kWavesPerBlock][kSmUnroll][kWave];
  const int lane = lane_id();
  const int wave = wave_in_block();
  const SoftmaxRows rows = softmax_rows(crow, n, (block_base + blockIdx.x) * kSmRows);
  {
    const int gl = lane % kSmLanes;
    float p[kSmBatch][kSmSlots], g[kSmBatch][kSmSlots];
    bool any[kSmBatch][kSmSlots];
#pragma unroll
    for (int k = 0; k < kSmBatch; ++k) {
#pragma unroll
      for (int i = 0; i < kSmSlots; ++i) {
        any[k][i] = __ballot(rows.len[k] > i * kSmLanes) != 0;
        p[k][i] = g[k][i] = 0.f;
        if (any[k][i] && gl + i * kSmLanes < rows.len[k]) {
          p[k][i] = sm_load(probs, rows.rs[k] + gl + i * kSmLanes);
          g[k][i] = sm_load(grad, rows.rs[k] + gl + i * kSmLanes);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kSmBatch; ++k) {
      float x[kSmSlots];
#pragma unroll
      for (int i = 0; i < kSmSlots; ++i)
        x[i] = gl + i * kSmLanes < rows.len[k] ? __builtin_fmaf(g[k][i], p[k][i], 0.f) : 0.f;
      const float t = group_sum16((x[0] + x[2]) + (x[1] + x[3]));
#pragma unroll
      for (int i = 0; i < kSmSlots; ++i) {
        if (any[k][i] && gl + i * kSmLanes < rows.len[k])
          sm_store(grad_scores, rows.rs[k] + gl + i * kSmLanes, p[k][i] * (g[k][i] - t));
      }
    }
  }
  float p[kSmUnroll], g[kSmUnroll];
  for (uint64_t left = rows.wave; left != 0; left &= left - 1) {
    int64_t rs, re;
    softmax_row_bounds(rows, __builtin_ctzll(left), rs, re);
    const bool once = re - rs <= kSmChunk;
    float t = 0.f;
    for (int64_t e = rs + lane; e < re; e += kSmChunk) {
      softmax_load2(probs, grad, e, re, p, g);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) t = e + i * kWave < re ? __builtin_fmaf(g[i], p[i], t) : t;
    }
    t = wave_sum_f32(t);
    for (int64_t e = rs + lane; e < re; e += kSmChunk) {
      if (!once) softmax_load2(probs, grad, e, re, p, g);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        if (e + i * kWave < re) sm_store(grad_scores, e + i * kWave, p[i] * (g[i] - t));
      }
    }
  }
  for (uint64_t left = rows.block; left != 0; left &= left - 1) {  // the same rows in every wave
    int64_t rs, re;
    softmax_row_bounds(rows, __builtin_ctzll(left), rs, re);
    constexpr int64_t kStep = kWavesPerBlock * kSmChunk;
    const int64_t e0 = rs + wave * kSmChunk + lane;
    float t = 0.f;
    softmax_load2(probs, grad, e0, re, p, g);
    for (int64_t b = rs; b < re; b += kStep) {
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        tile_p[wave][i][lane] = p[i];
        tile_g[wave][i][lane] = g[i];
      }
      softmax_load2(probs, grad, e0 + (b - rs) + kStep, re, p, g);
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; ++w) {
#pragma unroll
        for (int i = 0; i < kSmUnroll; ++i) {
          const float u = __builtin_fmaf(tile_g[w][i][lane], tile_p[w][i][lane], t);
          t = b + w * kSmChunk + i * kWave + lane < re ? u : t;
        }
      }
      __syncthreads();
    }
    t = wave_sum_f32(t);
    for (int64_t e = e0; e < re; e += kStep) {
      softmax_load2(probs, grad, e, re, p, g);
#pragma unroll
      for (int i = 0; i < kSmUnroll; ++i) {
        if (e + i * kWave < re) sm_store(grad_scores, e + i * kWave, p[i] * (g[i] - t));
      }
    }
  }
}

template <typename T>
int launch_softmax_backward(const int64_t* crow, const void* probs, const void* grad, void* grad_scores, int64_t n,
                            hipStream_t s) {
  const int64_t blocks = (n + kSmRows - 1) / kSmRows;
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
    hipLaunchKernelGGL(csr_row_softmax_backward_kernel<T>, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, s, crow,
                       static_cast<const T*>(probs), static_cast<const T*>(grad), static_cast<T*>(grad_scores), n, b0);
  }
  return check_launch("csr_row_softmax_backward");
}

void launch_softmax_f32(const int64_t* crow, const float* scores, float* probs, int64_t n, hipStream_t s) {
  const int64_t blocks = (n + kSmRows - 1) / kSmRows;
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
    hipLaunchKernelGGL(csr_row_softmax_kernel, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, s, crow, scores,
                       probs, n, b0);
  }
}

// The scores, overwritten by the probabilities.
size_t attention_workspace(int64_t nnz) { return static_cast<size_t>(nnz > 0 ? nnz : 1) * sizeof(float); }

}  // namespace

}  // namespace as

extern "C" {

int as_csr_row_softmax_f32(const int64_t* crow, const float* scores, float* probs, int64_t n, int64_t nnz,
                           void* stream) {
  as::clear_error();
  if (n < 0 || n > INT32_MAX || nnz < 0) return as::fail(AS_ERR_INVALID_ARGUMENT, "softmax sizes out of range");
  if (n == 0 || nnz == 0) return AS_OK;
  if (crow == nullptr || scores == nullptr || probs == nullptr)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "null pointer argument");
  as::launch_softmax_f32(crow, scores, probs, n, static_cast<hipStream_t>(stream));
  return as::check_launch("csr_row_softmax");
}

int as_csr_row_softmax_backward(const int64_t* crow, const void* probs, const void* grad, void* grad_scores,
                                int64_t n, int64_t nnz, int dtype, void* stream) {
  as::clear_error();
  if (dtype != AS_DTYPE_F32 && dtype != AS_DTYPE_BF16 && dtype != AS_DTYPE_F16)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "dtype must be AS_DTYPE_F32, AS_DTYPE_BF16 or AS_DTYPE_F16");
  if (n < 0 || n > INT32_MAX || nnz < 0) return as::fail(AS_ERR_INVALID_ARGUMENT, "softmax sizes out of range");
  const size_t align = dtype == AS_DTYPE_F32 ? 4 : 2;
  if (!as::aligned(probs, align) || !as::aligned(grad, align) || !as::aligned(grad_scores, align))
    return as::fail(AS_ERR_INVALID_ARGUMENT, "probs, grad and grad_scores must be aligned to their element size");
  if (n == 0 || nnz == 0) return AS_OK;
  if (crow == nullptr || probs == nullptr || grad == nullptr || grad_scores == nullptr)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "null pointer argument");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == AS_DTYPE_F32) return as::launch_softmax_backward<float>(crow, probs, grad, grad_scores, n, s);
  if (dtype == AS_DTYPE_BF16) return as::launch_softmax_backward<as::Bf16>(crow, probs, grad, grad_scores, n, s);
  return as::launch_softmax_backward<as::Fp16>(crow, probs, grad, grad_scores, n, s);
}

int as_csr_row_softmax_16(const int64_t* crow, const void* scores, void* probs, int64_t n, int64_t nnz, int dtype,
                          void* stream) {
  as::clear_error();
  if (dtype != AS_DTYPE_BF16 && dtype != AS_DTYPE_F16)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "dtype must be AS_DTYPE_BF16 or AS_DTYPE_F16");
  if (n < 0 || n > INT32_MAX || nnz < 0) return as::fail(AS_ERR_INVALID_ARGUMENT, "softmax sizes out of range");
  if (!as::aligned(scores, 2) || !as::aligned(probs, 2))
    return as::fail(AS_ERR_INVALID_ARGUMENT, "scores and probs must be 2-byte aligned");
  if (n == 0 || nnz == 0) return AS_OK;
  if (crow == nullptr || scores == nullptr || probs == nullptr)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "null pointer argument");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // short rows: 4 per wave
  const int64_t group_waves = (n + 3) / 4;
  const int64_t gblocks = (group_waves + as::kWavesPerBlock - 1) / as::kWavesPerBlock;
  for (int64_t b0 = 0; b0 < gblocks; b0 += as::kMaxBlocksPerLaunch) {
    const int64_t nb = gblocks - b0 < as::kMaxBlocksPerLaunch ? gblocks - b0 : as::kMaxBlocksPerLaunch;
    const dim3 grid(static_cast<unsigned>(nb));
    if (dtype == AS_DTYPE_BF16)
      hipLaunchKernelGGL(as::csr_row_softmax16_grouped_kernel<as::Bf16>, grid, dim3(as::kBlock), 0, s, crow,
                         static_cast<const as::Bf16*>(scores), static_cast<uint16_t*>(probs), n,
                         b0 * as::kWavesPerBlock);
    else
      hipLaunchKernelGGL(as::csr_row_softmax16_grouped_kernel<as::Fp16>, grid, dim3(as::kBlock), 0, s, crow,
                         static_cast<const as::Fp16*>(scores), static_cast<uint16_t*>(probs), n,
                         b0 * as::kWavesPerBlock);
  }
  // long rows: a wave each
  const int64_t blocks = (n + as::kWavesPerBlock - 1) / as::kWavesPerBlock;
  for (int64_t b0 = 0; b0 < blocks; b0 += as::kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < as::kMaxBlocksPerLaunch ? blocks - b0 : as::kMaxBlocksPerLaunch;
    const dim3 grid(static_cast<unsigned>(nb));
    if (dtype == AS_DTYPE_BF16)
      hipLaunchKernelGGL(as::csr_row_softmax16_kernel<as::Bf16>, grid, dim3(as::kBlock), 0, s, crow,
                         static_cast<const as::Bf16*>(scores), static_cast<uint16_t*>(probs), n,
                         b0 * as::kWavesPerBlock);
    else
      hipLaunchKernelGGL(as::csr_row_softmax16_kernel<as::Fp16>, grid, dim3(as::kBlock), 0, s, crow,
                         static_cast<const as::Fp16*>(scores), static_cast<uint16_t*>(probs), n,
                         b0 * as::kWavesPerBlock);
  }
  return as::check_launch("csr_row_softmax_16");
}

size_t as_csr_attention_workspace_bytes(int64_t n, int64_t nnz) {
  (void)n;
  return as::attention_workspace(nnz < 0 ? 0 : nnz);
}

int as_csr_attention_f32(const int64_t* crow, const int64_t* col, const float* query, const float* key,
                         const float* value, float* out, int64_t n, int64_t nnz, int64_t f_qk, int64_t f_v,
                         float scale, void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  if (n < 0 || n > INT32_MAX || nnz < 0 || f_qk < 0 || f_v < 0)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "attention sizes out of range");
  if (f_qk >= as::kMaxFeatures || f_v >= as::kMaxFeatures)
    return as::fail(AS_ERR_UNSUPPORTED, "F_qk and F_v must be below 2^28 (32-bit lane offsets)");
  if (n == 0 || f_v == 0) return AS_OK;
  if (crow == nullptr || value == nullptr || out == nullptr || (nnz > 0 && (col == nullptr || query == nullptr ||
                                                                           key == nullptr)))
    return as::fail(AS_ERR_INVALID_ARGUMENT, "null pointer argument");
  if (f_qk == 0 && nnz > 0)
    return as::fail(AS_ERR_UNSUPPORTED, "attention with zero query/key features is handled by the caller");
  if (workspace == nullptr || workspace_bytes < as::attention_workspace(nnz))
    return as::fail(AS_ERR_WORKSPACE, "attention needs %zu workspace bytes, got %zu", as::attention_workspace(nnz),
                    workspace_bytes);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  float* scores = static_cast<float*>(workspace);
  if (nnz > 0) {
    as::launch_sddmm_scaled(crow, col, query, key, scores, n, nnz, f_qk, scale, s);
    as::launch_softmax_f32(crow, scores, scores, n, s);
  }
  if (f_v >= 4 && nnz > 0) as::launch_spmm_groups(crow, col, scores, value, out, n, n, nnz, f_v, s);
  else as::launch_spmm_wave_rows(crow, col, scores, value, out, n, nnz, f_v, true, s);
  return as::check_launch("csr_attention");
}

}  // extern "C"
