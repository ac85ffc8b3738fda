// CSR SDDMM: out[e] = <query[row(e)], key[col[e]]> for every nonzero e.
//
// Reference behaviour: csrc/sddmm_csr_op.cu:19-50 (row kernel),
// :52-83 (hub kernel), :108-187 (launchers).
//
// Summation order (both reference kernels, :12-17 and :39-49): the 32 lanes
// of a warp each keep one fp32 partial, lane l adding features l, l+32,
// l+64, ... with fma; the 32 partials are then combined by the 16/8/4/2/1
// shfl_down tree.  The fp32 kernel reproduces exactly that order, so all
// fp32 SDDMM entry points give identical bits; the 16-bit kernels follow
// their own rule (below).
#include "as_device.h"
#include "as_internal.h"
#include "elem16.h"

namespace as {

size_t spmm_split_workspace_bytes(int64_t n);

namespace {

constexpr int kChunkEdges = 2048;  // edges per hub work item

// Work items of the 16-bit split schedule and of the fp32 product by rows: hub h
// (order[h], h < counts[0]) is cut into ceil(deg / kChunkEdges) chunks; chunk_off[h]
// is the exclusive prefix and counts[2] the total.  One workgroup of 1024 threads.
__global__ __launch_bounds__(1024) void hub_chunk_scan_kernel(const int64_t* __restrict__ crow,
                                                              const int32_t* __restrict__ order,
                                                              int32_t* __restrict__ counts,
                                                              int32_t* __restrict__ chunk_off) {
  __shared__ int lds[1024 / kWave];
  const int64_t hubs = counts[0];
  const int64_t per = (hubs + 1023) / 1024;
  const int64_t begin = static_cast<int64_t>(threadIdx.x) * per;
  const int64_t end = begin + per < hubs ? begin + per : hubs;
  int local = 0;
  for (int64_t h = begin; h < end; ++h) {
    const int64_t r = order[h];
    local += static_cast<int>((crow[r + 1] - crow[r] + kChunkEdges - 1) / kChunkEdges);
  }
  // block exclusive scan
  const int lane = lane_id();
  const int wave = wave_in_block();
  const int incl = wave_incl_scan_i32(local);
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  int before = 0;
  int total = 0;
  for (int w = 0; w < 1024 / kWave; ++w) {
    before += (w < wave) ? lds[w] : 0;
    total += lds[w];
  }
  int running = before + incl - local;
  for (int64_t h = begin; h < end; ++h) {
    chunk_off[h] = running;
    const int64_t r = order[h];
    running += static_cast<int>((crow[r + 1] - crow[r] + kChunkEdges - 1) / kChunkEdges);
  }
  if (threadIdx.x == 0) counts[2] = total;
}

// ---- fp32 SDDMM by blocks of edges ------------------------------------------
// The edges in CSR order, 64 a block, whatever the rows; every output keeps
// the reference's order (file comment).  8 lanes per edge and 8 edges per
// lane group: lane j of group g holds partials 4j .. 4j+3 of edges 8g .. 8g+7,
// one 16-byte key load (and query load) per 32 features and edge, so every
// gather instruction carries 8 edges however short the rows are.  Loads are
// aligned to 4 bytes only, so any F >= 4 takes vector lanes: the last partial
// block reads at F - 4 and shifts.
// The tree's three lane steps halve the edges a lane keeps (8, 4, 2, 1): the
// lane with the step's bit set keeps the upper half and receives its partner's
// part of it, 28 lane exchanges for 64 edges where a butterfly per edge takes
// 96, and lane i ends with edge i (one coalesced store).
//
// What bounds it: the gathers, at the memory's rate where K is beyond the
// caches (1M rows, 16.8M edges, F = 64: 0.655 ms, 6.6 TB/s of gathered bytes),
// at the L2's where it is not.  Against one wave per row and the split
// schedule (us): 100k rows, 1.2M edges, F = 47 446 -> 34, F = 64 125 -> 30, F = 100
// 690 -> 52 (F % 32 != 0 used to take 4-byte lanes and 2 edges an instruction);
// 1M rows, 50M edges, hubs of 200k edges, F = 64 1508 -> 809, F = 100 7370 -> 1535.
//
// How a row's 32-feature blocks are taken.  F % 32 == 0: one block of all 8
// edges at a time (each a whole 128-byte line of X).  Otherwise rows start
// inside lines and neighbouring blocks share one, so an edge's blocks (up to 4)
// are read together before the next edge's; taken one at a time the shared
// lines were fetched twice (F = 100, 1M rows: 1.63 ms, 2 blocks of 2 edges at a
// time 1.44, 4 blocks of 2 edges 1.46, 4 blocks of 1 edge 1.24).
typedef float Float4U __attribute__((ext_vector_type(4), aligned(4)));

template <bool OFF32>
struct RowOff;
template <>
struct RowOff<true> {
  uint32_t v;
};
template <>
struct RowOff<false> {
  int64_t v;
};
template <bool OFF32>
__device__ __forceinline__ RowOff<OFF32> row_off(int row, uint32_t row_bytes, uint32_t lane_off) {
  if constexpr (OFF32) return {static_cast<uint32_t>(row) * row_bytes + lane_off};
  else return {static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(row)) * row_bytes + lane_off)};
}
template <bool OFF32>
__device__ __forceinline__ Float4U load4(const char* __restrict__ base, RowOff<OFF32> off, int delta) {
  if constexpr (OFF32) return *reinterpret_cast<const Float4U*>(base + (off.v + static_cast<uint32_t>(delta)));
  else return *reinterpret_cast<const Float4U*>(base + (off.v + delta));
}

__device__ __forceinline__ Float4U shifted(Float4U v, int shift) {
  if (shift & 1) v = Float4U{v.y, v.z, v.w, v.w};
  if (shift & 2) v = Float4U{v.z, v.w, v.w, v.w};
  return v;
}

__device__ __forceinline__ float lane_xor4(float v) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (4 << 10) | 0x1f));
}
__device__ __forceinline__ float lane_xor2(float v) {  // quad_perm [2,3,0,1]
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_xor1(float v) {  // quad_perm [1,0,3,2]
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));
}

// Adds 32-feature blocks [m0, m0 + MB) of the 8 edges to p, UE edges at a
// time.  Block m of lane j holds features 32m + 4j ..; the row's last block
// (MASK) reads at F - 4 where that passes F.  TAIL: 0 F % 32 == 0, 1 whole
// vectors (4 | F), 2 shifted vectors (F >= 4), 3 elements (F < 4).
template <int MB, int TAIL, bool MASK, bool OFF32, bool ONE>
__device__ __forceinline__ void edge_blocks_dots(const char* __restrict__ kb, const char* __restrict__ qb, int F,
                                                 int m0, const RowOff<OFF32> (&ko)[8],
                                                 const RowOff<OFF32> (&qo)[ONE ? 1 : 8], float (&p)[8][4]) {
  constexpr int UE = MB == 1 ? 8 : (MB == 2 ? 2 : 1);
  const int j4 = 4 * (lane_id() & 7);
  int delta[MB], shift[MB], left[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int start = 32 * (m0 + m) + j4;
    delta[m] = (m0 + m) * 128;
    left[m] = F - start;
    shift[m] = 0;
    if (TAIL == 1 || TAIL == 2) {
      if (MASK && m == MB - 1) {
        const int from = start < F - 4 ? start : F - 4;
        delta[m] = (from - j4) * 4;
        shift[m] = start - from;  // used where left > 0, then <= 3
      }
    }
  }
#pragma unroll
  for (int h = 0; h < 8; h += UE) {
    Float4U k[UE][MB];
    Float4U q[ONE ? 1 : UE][MB];
#pragma unroll
    for (int u = 0; u < UE; ++u) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        if constexpr (TAIL == 3) {
          k[u][m] = Float4U{0.f, 0.f, 0.f, 0.f};
          if (!ONE || u == 0) q[ONE ? 0 : u][m] = Float4U{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 3; ++s) {
            if (s < left[m]) {
              k[u][m][s] = *reinterpret_cast<const float*>(kb + ko[h + u].v + 4 * s);
              if (!ONE || u == 0)
                q[ONE ? 0 : u][m][s] = *reinterpret_cast<const float*>(qb + qo[ONE ? 0 : h + u].v + 4 * s);
            }
          }
        } else {
          k[u][m] = load4<OFF32>(kb, ko[h + u], delta[m]);
          if (!ONE || u == 0) q[ONE ? 0 : u][m] = load4<OFF32>(qb, qo[ONE ? 0 : h + u], delta[m]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UE; ++u) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const bool masked = TAIL != 0 && MASK && m == MB - 1;
        Float4U kk = k[u][m];
        Float4U qq = q[ONE ? 0 : u][m];
        if (TAIL == 2 && masked) {
          kk = shifted(kk, shift[m]);
          qq = shifted(qq, shift[m]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const float t = __builtin_fmaf(qq[s], kk[s], p[h + u][s]);
          // a skipped feature leaves the sum as it is (0 * k would not, for
          // an infinite k or a sum of -0)
          p[h + u][s] = !masked || (TAIL == 1 ? 0 : s) < left[m] ? t : p[h + u][s];
        }
      }
    }
    if constexpr (UE < 8) __builtin_amdgcn_sched_barrier(0);
  }
}

// One block of 64 edges: the dot product of edge `lane`.  my_c / my_row: lane
// i holds the column / row of edge i.  ONE: every edge is in row my_row.
// F's 32-feature blocks are taken CB at a time, the last LAST together.
template <int CB, int LAST, int TAIL, bool OFF32, bool ONE>
__device__ __forceinline__ float edge_block_dots(const char* __restrict__ kb, const char* __restrict__ qb, int F,
                                                 int my_c, int my_row) {
  const int lane = lane_id();
  const uint32_t row_bytes = static_cast<uint32_t>(F) * 4u;
  const uint32_t lane_off = static_cast<uint32_t>((lane & 7) * 16);
  RowOff<OFF32> ko[8];
  RowOff<OFF32> qo[ONE ? 1 : 8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int addr = ((lane & 56) + u) * 4;
    ko[u] = row_off<OFF32>(__builtin_amdgcn_ds_bpermute(addr, my_c), row_bytes, lane_off);
    if constexpr (!ONE) qo[u] = row_off<OFF32>(__builtin_amdgcn_ds_bpermute(addr, my_row), row_bytes, lane_off);
  }
  if constexpr (ONE) qo[0] = row_off<OFF32>(my_row, row_bytes, lane_off);
  float p[8][4];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
#pragma unroll
    for (int s = 0; s < 4; ++s) p[u][s] = 0.f;
  }
  const int last = (F + 31) / 32 - LAST;
  if constexpr (CB > 0) {
    for (int m = 0; m < last; m += CB) edge_blocks_dots<CB, TAIL, false, OFF32, ONE>(kb, qb, F, m, ko, qo, p);
  }
  edge_blocks_dots<LAST, TAIL, TAIL != 0, OFF32, ONE>(kb, qb, F, CB > 0 ? last : 0, ko, qo, p);
  const bool b4 = (lane & 4) != 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float keep = b4 ? p[u + 4][s] : p[u][s];
      const float send = b4 ? p[u][s] : p[u + 4][s];
      p[u][s] = keep + lane_xor4(send);
    }
  }
  const bool b2 = (lane & 2) != 0;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float keep = b2 ? p[u + 2][s] : p[u][s];
      const float send = b2 ? p[u][s] : p[u + 2][s];
      p[u][s] = keep + lane_xor2(send);
    }
  }
  const bool b1 = (lane & 1) != 0;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const float keep = b1 ? p[1][s] : p[0][s];
    const float send = b1 ? p[0][s] : p[1][s];
    p[0][s] = keep + lane_xor1(send);
  }
  return (p[0][0] + p[0][2]) + (p[0][1] + p[0][3]);
}

constexpr int kEdgeWaves = 4;  // waves per workgroup

template <int CB, int LAST, int TAIL, bool OFF32>
__global__ __launch_bounds__(kEdgeWaves * kWave) __attribute__((amdgpu_waves_per_eu(4))) void sddmm_edges_kernel(
    const int64_t* __restrict__ crow, const int64_t* __restrict__ col, const float* __restrict__ query,
    const float* __restrict__ key, float* __restrict__ out, int64_t n, int64_t nnz, int F, float scale,
    int64_t per_wave, int64_t wave_base) {
  const int64_t w = wave_base + static_cast<int64_t>(blockIdx.x) * kEdgeWaves + wave_in_block();
  const int64_t b0 = uniform_i64(w * per_wave);
  if (b0 >= nnz) return;  // wave-uniform
  const int lane = lane_id();
  const int64_t b1 = uniform_i64(b0 + per_wave < nnz ? b0 + per_wave : nnz);
  const char* __restrict__ kb = reinterpret_cast<const char*>(key);
  const char* __restrict__ qb = reinterpret_cast<const char*>(query);
  int next_c = b0 + lane < b1 ? static_cast<int>(col[b0 + lane]) : 0;
  int64_t r = uniform_i64(wave_row_of_edge(crow, n, b0));
  for (int64_t b = b0; b < b1; b += kWave) {
    const int cnt = b1 - b < kWave ? static_cast<int>(b1 - b) : kWave;
    const int my_c = next_c;
    if (b + kWave < b1) next_c = b + kWave + lane < b1 ? static_cast<int>(col[b + kWave + lane]) : 0;
    float d;
    if (uniform_i64(crow[r + 1]) >= b + cnt) {  // every edge of the block is in row r
      d = edge_block_dots<CB, LAST, TAIL, OFF32, true>(kb, qb, F, my_c, static_cast<int>(r));
    } else {
      const int my_row = block_edge_rows(crow, n, b, cnt, r);
      r = __builtin_amdgcn_readlane(my_row, cnt - 1);
      d = edge_block_dots<CB, LAST, TAIL, OFF32, false>(kb, qb, F, my_c, my_row);
    }
    if (lane < cnt) out[b + lane] = d * scale;  // scale 1: the dot product's bits
  }
}

struct SddmmArgs {
  const int64_t* crow;
  const int64_t* col;
  const float* q;
  const float* k;
  float* out;
  int64_t n;
  int64_t f;
};

// Blocks of 64 edges a wave: 4 spread the row search and the start of the
// chain over 256 edges (1M rows, 50M edges, F = 64 us at 1 / 2 / 4 / 8 blocks:
// 1106 / 909 / 811 / 764), except that wide rows of a few edges, whose gathers run
// at the memory's rate anyway, are better off in launch order (1M rows, 16.8M
// edges: F = 96 924 / 951 / 963, F = 128 1229 / 1246 / 1259 at 1 / 2 / 4).
// Fewer than 4 where that would leave fewer than 16,384 waves.
constexpr int64_t kMaxEdgeBlocks = 4;
constexpr int64_t kFillWaves = 16384;
constexpr int64_t kShortRowDegree = 32;
constexpr int64_t kWideRow = 96;

// n_keys: rows of the key, or -1 where the caller does not know them (64-bit
// offsets then).
void launch_sddmm_edges(const SddmmArgs& a, int64_t nnz, int64_t n_keys, float scale, hipStream_t s) {
  int64_t per = nnz / (kFillWaves * kWave);
  const bool in_order = a.f >= kWideRow && nnz < kShortRowDegree * a.n;
  per = per < 1 || in_order ? 1 : (per > kMaxEdgeBlocks ? kMaxEdgeBlocks : per);
  const int64_t per_wave = per * kWave;
  const int64_t waves = (nnz + per_wave - 1) / per_wave;
  const int64_t blocks = (waves + kEdgeWaves - 1) / kEdgeWaves;
  const int64_t rows = a.n > n_keys ? a.n : n_keys;
  const bool off32 = n_keys > 0 && rows * a.f * 4 <= (int64_t(1) << 32);
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
#define AS_E32(CB, LAST, TAIL)                                                                                     \
  do {                                                                                                           \
    if (off32)                                                                                                   \
      hipLaunchKernelGGL((sddmm_edges_kernel<CB, LAST, TAIL, true>), grid, dim3(kEdgeWaves * kWave), 0, s, a.crow, \
                         a.col, a.q, a.k, a.out, a.n, nnz, static_cast<int>(a.f), scale, per_wave,               \
                         b0 * kEdgeWaves);                                                                       \
    else                                                                                                         \
      hipLaunchKernelGGL((sddmm_edges_kernel<CB, LAST, TAIL, false>), grid, dim3(kEdgeWaves * kWave), 0, s,      \
                         a.crow, a.col, a.q, a.k, a.out, a.n, nnz, static_cast<int>(a.f), scale, per_wave,       \
                         b0 * kEdgeWaves);                                                                       \
  } while (0)
    const dim3 grid(static_cast<unsigned>(nb));
    const int nbl = static_cast<int>((a.f + 31) / 32);
    const bool vec = a.f % 4 == 0;
    if (a.f < 4) AS_E32(0, 1, 3);
    else if (a.f == 32) AS_E32(0, 1, 0);
    else if (a.f % 32 == 0) AS_E32(1, 1, 0);
    else if (a.f < 32 && vec) AS_E32(0, 1, 1);
    else if (a.f < 32) AS_E32(0, 1, 2);
    else if (a.f < 64 && vec) AS_E32(0, 2, 1);
    else if (a.f < 64) AS_E32(0, 2, 2);
    else {
      switch (nbl % 4) {
        case 0: if (vec) AS_E32(4, 4, 1); else AS_E32(4, 4, 2); break;
        case 1: if (vec) AS_E32(4, 1, 1); else AS_E32(4, 1, 2); break;
        case 2: if (vec) AS_E32(4, 2, 1); else AS_E32(4, 2, 2); break;
        default: if (vec) AS_E32(4, 3, 1); else AS_E32(4, 3, 2); break;
      }
    }
#undef AS_E32
  }
}

// Workgroups given to the hub chunks of the scheduled kernel: one per chunk
// up to this cap (the host knows only an upper bound on the chunk count;
// workgroups past the real count exit at once).  A small fixed pool was a
// bottleneck when a low threshold makes tens of thousands of rows hub rows
// (cfg4, threshold 197: 2.96 ms with 4,096 pool waves against 1.82 ms at
// threshold 256), and a pool much smaller than the chunk count leaves the
// hub pass as a tail behind the light rows.
constexpr int64_t kHubBlocksMax = 65536;

// ---- fp32 SDDMM by rows --------------------------------------------------------
// One wave per row, rows of at least kRowsHub edges in chunks of kChunkEdges over
// workgroups of their own (the first of the launch); the reference's order again.
// A lane holds its part of the query row (4 features of every 32) and 2 or 4 edges
// of a lane group are in flight with whole rows of the key.
//
// What bounds it: where the key is beyond the caches, the rate of its rows, read
// whole by one instruction sequence: a few percent ahead of the blocks of edges,
// which read a row's 128-byte lines one 32-feature block after the other.  us,
// blocks / rows: 500k rows of 40 edges F = 64 771 / 739, F = 128 1534 / 1481, F =
// 256 3012 / 2819; 1M rows of 50 F = 64 1949 / 1844; 300k rows of 100 F = 256 4503 /
// 4232.  Where hubs' columns are cached it falls far behind (1M rows, 50M edges
// with hubs in the columns too, F = 64 819 / 1494), and with short rows as well (1M
// rows of 6, F = 64 274 / 542), so the scheduler times it on graphs that may suit it
// and nothing runs it unasked.
constexpr int64_t kRowsHub = 1024;
constexpr int kRowsLanes = 8;  // per edge: lane j holds partials 4j .. 4j + 3

__device__ __forceinline__ float row_dot_tree(float (&p)[4]) {
#pragma unroll
  for (int o = 4; o >= 1; o >>= 1) {
#pragma unroll
    for (int s = 0; s < 4; ++s) p[s] += __shfl_xor(p[s], o, kWave);
  }
  return (p[0] + p[2]) + (p[1] + p[3]);
}

// The dot products of edges first + 8u + lane group (u < UE) below end.
template <int MF, int UE>
__device__ __forceinline__ void row_dots(const int64_t* __restrict__ col, const float* __restrict__ key,
                                         float* __restrict__ out, int64_t F, const FVec<4> (&qv)[MF], int64_t first,
                                         int64_t end, int g, int j) {
  constexpr int NG = kWave / kRowsLanes;
  FVec<4> kv[UE][MF];
#pragma unroll
  for (int u = 0; u < UE; ++u) {
    const int64_t e = first + u * NG + g;
    const int c = static_cast<int>(col[e < end ? e : end - 1]);
    const float* kr = key + row_offset(c, F) + 4 * j;
#pragma unroll
    for (int m = 0; m < MF; ++m) kv[u][m] = load_vec<4>(kr + 32 * m);
  }
#pragma unroll
  for (int u = 0; u < UE; ++u) {
    float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < MF; ++m) {
#pragma unroll
      for (int s = 0; s < 4; ++s) p[s] = __builtin_fmaf(qv[m].v[s], kv[u][m].v[s], p[s]);
    }
    const float d = row_dot_tree(p);
    const int64_t e = first + u * NG + g;
    if (e < end && j == 0) out[e] = d;
  }
}

template <int MF>
__global__ __launch_bounds__(kBlock) void sddmm_rows_kernel(
    const int64_t* __restrict__ crow, const int64_t* __restrict__ col, const float* __restrict__ query,
    const float* __restrict__ key, float* __restrict__ out, int64_t n, int64_t F, const int32_t* __restrict__ order,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ chunk_off, int64_t hub_blocks,
    int64_t block_base) {
  constexpr int NG = kWave / kRowsLanes;
  const int lane = lane_id();
  const int g = lane / kRowsLanes;
  const int j = lane % kRowsLanes;
  const int wave = wave_in_block();
  const int64_t block = block_base + blockIdx.x;
  FVec<4> qv[MF];
  auto load_query = [&](int64_t row) {
#pragma unroll
    for (int m = 0; m < MF; ++m) qv[m] = load_vec<4>(query + row * F + 32 * m + 4 * j);
  };
  if (block < hub_blocks) {
    const int64_t hubs = counts[0];
    const int64_t items = counts[2];
    for (int64_t item = block; item < items; item += hub_blocks) {
      int64_t lo = 0;
      int64_t hi = hubs - 1;
      while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (chunk_off[mid] <= item) lo = mid;
        else hi = mid - 1;
      }
      const int64_t row = uniform_i64(order[lo]);
      const int64_t cs = uniform_i64(crow[row]) + (item - uniform_i64(chunk_off[lo])) * kChunkEdges;
      const int64_t re = uniform_i64(crow[row + 1]);
      const int64_t ce = cs + kChunkEdges < re ? cs + kChunkEdges : re;
      load_query(row);
      for (int64_t b = cs + wave * NG; b < ce; b += kWavesPerBlock * NG)
        row_dots<MF, 1>(col, key, out, F, qv, b, ce, g, j);
    }
    return;
  }
  const int64_t row = (block - hub_blocks) * kWavesPerBlock + wave;
  if (row >= n) return;
  const int64_t rs = uniform_i64(crow[row]);
  const int64_t re = uniform_i64(crow[row + 1]);
  if (re - rs >= kRowsHub || re <= rs) return;
  constexpr int UE = MF <= 2 ? 4 : 2;
  load_query(row);
  for (int64_t b = rs; b < re; b += NG * UE) row_dots<MF, UE>(col, key, out, F, qv, b, re, g, j);
}

bool sddmm_rows_fit(const SddmmArgs& a) {
  return a.f % 32 == 0 && a.f >= 32 && a.f <= 256 && aligned(a.q, 16) && aligned(a.k, 16);
}

// hub_blocks workgroups for the chunks of hub rows (an upper bound of them; 0: no
// row can have kRowsHub edges, order, counts and chunk_off are not read).
void launch_sddmm_rows(const SddmmArgs& a, int64_t hub_blocks, const int32_t* order, const int32_t* counts,
                       const int32_t* chunk_off, hipStream_t s) {
  const int64_t blocks = hub_blocks + (a.n + kWavesPerBlock - 1) / kWavesPerBlock;
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
    const dim3 grid(static_cast<unsigned>(nb));
#define AS_ROWS(MF)                                                                                              \
  hipLaunchKernelGGL(sddmm_rows_kernel<MF>, grid, dim3(kBlock), 0, s, a.crow, a.col, a.q, a.k, a.out, a.n, a.f, order, \
                     counts, chunk_off, hub_blocks, b0)
    switch (static_cast<int>(a.f / 32)) {
      case 1: AS_ROWS(1); break;
      case 2: AS_ROWS(2); break;
      case 3: AS_ROWS(3); break;
      case 4: AS_ROWS(4); break;
      case 5: AS_ROWS(5); break;
      case 6: AS_ROWS(6); break;
      case 7: AS_ROWS(7); break;
      default: AS_ROWS(8); break;
    }
#undef AS_ROWS
  }
}

// ---- bf16 / fp16 SDDMM -------------------------------------------------------
// out[e] = the fp64 sum of the exact products q[row(e), f]·k[col(e), f],
// rounded to fp32 and then to the element type (round to nearest even both
// times).  Products of two 16-bit values are exact in fp64, so an exact fp64
// sum does not depend on the order of the additions, and every schedule here
// gives the same bits.  There is no reference kernel for these types (its op
// takes float32 only, csrc/sddmm_csr_op.cu:94; its scheduler runs the
// gather-dot baseline, autosage/_auto.py:575-581).
//
// Vector lanes (F a multiple of 8 up to 512, 16-byte aligned rows; by blocks
// of edges any F from 8 to 512): a lane
// holds 8 consecutive features, chunk j + G·m of the row for m < MB; G lanes
// per edge (the power of two covering F/8, at most 32), 64/G edges per
// gather instruction.  The query row is converted to fp64 once per row and
// kept in registers.  Other shapes take element lanes: 64 lanes per edge,
// lane l adding features l, l + 64, ...
// Edges are taken in blocks of 64: one coalesced load brings the block's
// column indices (one block ahead), and ds_bpermute hands each lane group its
// edge's column, so a pass waits for one round of key gathers only; UE
// gathers per lane are in flight (all 64 edges of a block at once for G <= 8,
// else 32, 16 or 8 at a time).
template <typename T, int G, int MB, bool OFF32>
__device__ __forceinline__ void dots16_vec(const int64_t* __restrict__ col, const T* __restrict__ key,
                                           uint16_t* __restrict__ out, int64_t F, const double (&qd)[MB][8],
                                           int64_t first, int64_t end, int64_t step, int g, int j) {
  constexpr int NG = kWave / G;
  constexpr int UE = NG >= 8 ? kWave / NG : (MB == 1 ? 8 : 4);  // gathers in flight per lane
  constexpr int kSub = NG * UE;                                    // edges per sub-pass, <= 64
  static_assert(kSub <= kWave, "a sub-pass stays inside its block of 64 edges");
  const int lane = lane_id();
  const int64_t chunks = F / 8;
  const char* __restrict__ kb = reinterpret_cast<const char*>(key);
  const uint32_t row_bytes = static_cast<uint32_t>(F * sizeof(T));
  uint32_t lane_off[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) lane_off[m] = static_cast<uint32_t>((j + G * m < chunks ? j + G * m : 0) * 16);
  int next_c = first + lane < end ? static_cast<int>(col[first + lane]) : 0;
  for (int64_t base = first; base < end; base += step) {
    const int my_c = next_c;
    const int64_t nb = base + step;
    if (nb < end) next_c = nb + lane < end ? static_cast<int>(col[nb + lane]) : 0;
    const int cnt = end - base < kWave ? static_cast<int>(end - base) : kWave;
    for (int u0 = 0; u0 < cnt; u0 += kSub) {
      // edge u0 + u·NG + g; steps u with u0 + u·NG >= cnt hold no edge of
      // any group and are skipped (wave-uniform)
      RawVec<16> kv[UE][MB];
#pragma unroll
      for (int u = 0; u < UE; ++u) {
        if (u0 + u * NG < cnt) {
          const int idx = u0 + u * NG + g;  // < 64
          const int c = __builtin_amdgcn_ds_bpermute(idx * 4, my_c);
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            if constexpr (OFF32) {
              kv[u][m] = load_raw<16>(kb + (__umul24(static_cast<uint32_t>(c), row_bytes) + lane_off[m]));
            } else {
              kv[u][m] = load_raw<16>(kb + static_cast<int64_t>(c) * row_bytes + lane_off[m]);
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UE; ++u) {
        if (u0 + u * NG < cnt) {
          double acc = 0.0;
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            if (j + G * m < chunks) {
#pragma unroll
              for (int p = 0; p < 8; ++p)
                acc = __builtin_fma(qd[m][p], static_cast<double>(Elem<T>::get(kv[u][m].w, p)), acc);
            }
          }
#pragma unroll
          for (int o = 1; o < G; o <<= 1) acc += __shfl_xor(acc, o, kWave);
          const int idx = u0 + u * NG + g;
          if (j == 0 && idx < cnt) out[base + idx] = Elem<T>::bits(acc);
        }
      }
    }
  }
}

template <typename T, int G, int MB>
__device__ __forceinline__ void load_query16(const T* __restrict__ qrow, int64_t F, int j, double (&qd)[MB][8]) {
  const int64_t chunks = F / 8;
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int64_t chunk = j + G * m;
    const RawVec<16> v = load_raw<16>(reinterpret_cast<const char*>(qrow + (chunk < chunks ? chunk : 0) * 8));
#pragma unroll
    for (int p = 0; p < 8; ++p) qd[m][p] = chunk < chunks ? static_cast<double>(Elem<T>::get(v.w, p)) : 0.0;
  }
}

template <typename T>
__device__ __forceinline__ void dots16_scalar(const int64_t* __restrict__ col, const T* __restrict__ qrow,
                                              const T* __restrict__ key, uint16_t* __restrict__ out, int64_t F,
                                              int64_t first, int64_t end, int64_t step) {
  const int lane = lane_id();
  for (int64_t e = first; e < end; e += step) {
    const int64_t c = uniform_i64(col[e]);
    const T* __restrict__ kr = key + c * F;
    double acc = 0.0;
    for (int64_t f = lane; f < F; f += kWave)
      acc = __builtin_fma(static_cast<double>(Elem<T>::at(qrow, f)), static_cast<double>(Elem<T>::at(kr, f)), acc);
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) acc += __shfl_xor(acc, o, kWave);
    if (lane == 0) out[e] = Elem<T>::bits(acc);
  }
}

// Edges [cs, ce) of `row`, taken by `waves` waves (this one is `wave`).
template <typename T, int G, int MB, bool VEC, bool OFF32>
__device__ __forceinline__ void sddmm16_edges(const int64_t* __restrict__ col, const T* __restrict__ query,
                                              const T* __restrict__ key, uint16_t* __restrict__ out, int64_t F,
                                              int64_t row, int64_t cs, int64_t ce, int wave, int waves) {
  if constexpr (VEC) {
    const int lane = lane_id();
    const int g = lane / G;
    const int j = lane % G;
    double qd[MB][8];
    load_query16<T, G, MB>(query + row * F, F, j, qd);
    dots16_vec<T, G, MB, OFF32>(col, key, out, F, qd, cs + static_cast<int64_t>(wave) * kWave, ce,
                         static_cast<int64_t>(waves) * kWave, g, j);
  } else {
    dots16_scalar<T>(col, query + row * F, key, out, F, cs + wave, ce, waves);
  }
}

// The split schedule for 16-bit elements:
// workgroups [0, hub_blocks) stride over the 2048-edge chunks of the rows of
// degree >= hub_threshold, the rest take the other rows one per wave.
template <typename T, int G, int MB, bool VEC, bool OFF32>
__device__ __forceinline__ void sddmm16_scheduled_body(
    const int64_t* __restrict__ crow, const int64_t* __restrict__ col, const T* __restrict__ query,
    const T* __restrict__ key, uint16_t* __restrict__ out, int64_t n, int64_t F, int64_t hub_threshold,
    const int32_t* __restrict__ order, const int32_t* __restrict__ counts, const int32_t* __restrict__ chunk_off,
    int64_t hub_blocks, int64_t block_base) {
  const int wave = wave_in_block();
  const int waves = static_cast<int>(blockDim.x >> 6);
  const int64_t block = block_base + blockIdx.x;
  if (block < hub_blocks) {
    const int64_t hubs = counts[0];
    const int64_t items = counts[2];
    for (int64_t item = block; item < items; item += hub_blocks) {
      int64_t lo = 0;
      int64_t hi = hubs - 1;
      while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (chunk_off[mid] <= item) lo = mid;
        else hi = mid - 1;
      }
      const int64_t row = uniform_i64(order[lo]);
      const int64_t rs = uniform_i64(crow[row]);
      const int64_t re = uniform_i64(crow[row + 1]);
      const int64_t cs = rs + (item - uniform_i64(chunk_off[lo])) * kChunkEdges;
      const int64_t ce = cs + kChunkEdges < re ? cs + kChunkEdges : re;
      sddmm16_edges<T, G, MB, VEC, OFF32>(col, query, key, out, F, row, cs, ce, wave, waves);
    }
    return;
  }
  const int64_t row = (block - hub_blocks) * waves + wave;
  if (row >= n) return;
  const int64_t rs = uniform_i64(crow[row]);
  const int64_t re = uniform_i64(crow[row + 1]);
  if (re - rs >= hub_threshold || re == rs) return;
  sddmm16_edges<T, G, MB, VEC, OFF32>(col, query, key, out, F, row, rs, re, 0, 1);
}

// The kernel, and the same with at most 80 VGPRs (6 waves per SIMD, a few
// bytes spilled) for 16 lanes per edge: F = 128 in bf16 on cfg4 takes 1.97 ms
// with it against 2.21 at 89 VGPRs (5 waves), while F = 64 (8 lanes) gains
// nothing (1.163 against 1.155).
#define AS_SDDMM16_PARAMS                                                                                    \
  const int64_t *__restrict__ crow, const int64_t *__restrict__ col, const T *__restrict__ query,          \
      const T *__restrict__ key, uint16_t *__restrict__ out, int64_t n, int64_t F, int64_t hub_threshold, \
      const int32_t *__restrict__ order, const int32_t *__restrict__ counts,                              \
      const int32_t *__restrict__ chunk_off, int64_t hub_blocks, int64_t block_base
#define AS_SDDMM16_ARGS crow, col, query, key, out, n, F, hub_threshold, order, counts, chunk_off, hub_blocks, block_base
template <typename T, int G, int MB, bool VEC, bool OFF32>
__global__ __launch_bounds__(512) void sddmm16_scheduled_kernel(AS_SDDMM16_PARAMS) {
  sddmm16_scheduled_body<T, G, MB, VEC, OFF32>(AS_SDDMM16_ARGS);
}
template <typename T, int G, int MB, bool VEC, bool OFF32>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(6))) void sddmm16_scheduled_kernel_w6(
    AS_SDDMM16_PARAMS) {
  sddmm16_scheduled_body<T, G, MB, VEC, OFF32>(AS_SDDMM16_ARGS);
}
#undef AS_SDDMM16_PARAMS
#undef AS_SDDMM16_ARGS

struct Sddmm16Args {
  const int64_t* crow;
  const int64_t* col;
  const void* q;
  const void* k;
  void* out;
  int64_t n;       // rows of the graph and of the query
  int64_t f;
  int64_t n_keys;  // rows of the key (n for a square graph)
};

// Every query and key byte offset fits 32 bits, and every row index 24 bits.
inline bool sddmm16_off32(const Sddmm16Args& a) {
  const int64_t rows = a.n > a.n_keys ? a.n : a.n_keys;
  return rows <= (int64_t(1) << 24) && rows * a.f * 2 <= (int64_t(1) << 32);
}

template <typename T, int G, int MB, bool VEC, bool OFF32>
void launch_sddmm16_v(const Sddmm16Args& a, dim3 grid, dim3 block, int64_t hub_threshold, const int32_t* order,
                      const int32_t* counts, const int32_t* chunk_off, int64_t hub_blocks, int64_t b0,
                      hipStream_t s) {
  if constexpr (VEC && G == 16) {
    hipLaunchKernelGGL((sddmm16_scheduled_kernel_w6<T, G, MB, VEC, OFF32>), grid, block, 0, s, a.crow, a.col,
                       static_cast<const T*>(a.q), static_cast<const T*>(a.k), static_cast<uint16_t*>(a.out), a.n,
                       a.f, hub_threshold, order, counts, chunk_off, hub_blocks, b0);
  } else {
    hipLaunchKernelGGL((sddmm16_scheduled_kernel<T, G, MB, VEC, OFF32>), grid, block, 0, s, a.crow, a.col,
                       static_cast<const T*>(a.q), static_cast<const T*>(a.k), static_cast<uint16_t*>(a.out), a.n,
                       a.f, hub_threshold, order, counts, chunk_off, hub_blocks, b0);
  }
}

// Lanes per edge G and chunks per lane MB for F features (vector lanes), or
// G = 0 for element lanes.
inline void sddmm16_lanes(int64_t f, int& g, int& mb) {
  g = 0;
  mb = 1;
  if (f < 8 || f > 512) return;
  const int64_t chunks = (f + 7) / 8;
  g = 1;
  while (g < chunks && g < 32) g <<= 1;
  mb = chunks > 32 ? 2 : 1;
}
// The split schedule's: element lanes for ragged rows.
inline void sddmm16_shape(const Sddmm16Args& a, int& g, int& mb) {
  sddmm16_lanes(a.f % 8 == 0 && aligned(a.q, 16) && aligned(a.k, 16) ? a.f : 0, g, mb);
}

template <typename T>
void launch_sddmm16(const Sddmm16Args& a, int waves, int64_t hub_threshold, int64_t item_upper,
                    const int32_t* order, const int32_t* counts, const int32_t* chunk_off, hipStream_t s) {
  const int64_t hub_blocks = item_upper < kHubBlocksMax ? item_upper : kHubBlocksMax;
  const int64_t blocks = hub_blocks + (a.n + waves - 1) / waves;
  const dim3 block(static_cast<unsigned>(waves * kWave));
  int g, mb;
  sddmm16_shape(a, g, mb);
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
    const dim3 grid(static_cast<unsigned>(nb));
  const bool off32 = sddmm16_off32(a);
#define AS_S16(G, MB, VEC)                                                                                      \
  do {                                                                                                         \
    if (off32)                                                                                                 \
      launch_sddmm16_v<T, G, MB, VEC, true>(a, grid, block, hub_threshold, order, counts, chunk_off, hub_blocks, \
                                            b0, s);                                                            \
    else                                                                                                       \
      launch_sddmm16_v<T, G, MB, VEC, false>(a, grid, block, hub_threshold, order, counts, chunk_off,          \
                                             hub_blocks, b0, s);                                               \
  } while (0)
    if (mb == 2) {
      AS_S16(32, 2, true);
    } else {
      switch (g) {
        case 1: AS_S16(1, 1, true); break;
        case 2: AS_S16(2, 1, true); break;
        case 4: AS_S16(4, 1, true); break;
        case 8: AS_S16(8, 1, true); break;
        case 16: AS_S16(16, 1, true); break;
        case 32: AS_S16(32, 1, true); break;
        default:
          launch_sddmm16_v<T, 64, 1, false, false>(a, grid, block, hub_threshold, order, counts, chunk_off,
                                                   hub_blocks, b0, s);
          break;
      }
    }
#undef AS_S16
  }
}

// ---- 16-bit SDDMM by blocks of edges ---------------------------------------
// The same dot products as above (the same lane layout, fp64 sums and
// butterfly: the same bits) over the edges in CSR order, 64 at a time, with
// no regard to rows: wave w takes blocks [w·B, w·B + B) of 64 edges.  Every
// gather instruction then carries 64/G edges however short the rows are (a
// wave per row issues one partly filled gather for a row of a few edges and
// waits for it), and long rows need no schedule of their own.  The query row
// is gathered per edge (consecutive edges share it, so those gathers hit
// the caches).
//
// Rows of the edges: the wave loads the ends of the 64 rows from r, the row
// of the block's first edge, and lane i finds the row of edge b + i by a
// binary search over them (ds_bpermute).  A block spanning more than 64 rows
// (empty rows) takes further rounds of 64.  r comes from a table for the
// wave's first block (edge_wave_rows_kernel, one binary search over crow per
// wave) and is the row of the previous block's last edge after that.
// 2 blocks a wave: cfg4 (50M edges, median degree 8) bf16 F = 64 takes
// 0.975 ms against 0.986 at 4 and 1.000 at 8 (the split schedule: 1.133);
// the 2.4M-row, 124M-edge attention graph at F = 64 1.988 against 2.000 and
// 2.032 (split: 2.756); the skewed 115M-edge graph at F = 128 2.890 against
// 2.930 and 3.011 (split: 3.257).
#ifndef AS_SDDMM16_EDGE_BLOCKS
#define AS_SDDMM16_EDGE_BLOCKS 2
#endif
constexpr int64_t kEdgeBlocksPerWave = AS_SDDMM16_EDGE_BLOCKS;
constexpr int64_t kEdgesPerWave = kWave * kEdgeBlocksPerWave;
int64_t edge_waves(int64_t nnz) { return (nnz + kEdgesPerWave - 1) / kEdgesPerWave; }

size_t sddmm_edges_ws(int64_t nnz) {
  return align_up(static_cast<size_t>(edge_waves(nnz) > 0 ? edge_waves(nnz) : 1) * sizeof(int32_t), 256);
}

// rows[w] = the row holding edge w·kEdgesPerWave: the last r < n with
// crow[r] <= e (rows before it that are empty end at or before e).
__global__ __launch_bounds__(256) void edge_wave_rows_kernel(const int64_t* __restrict__ crow, int64_t n,
                                                             int64_t waves, int32_t* __restrict__ rows) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (w >= waves) return;
  const int64_t e = w * kEdgesPerWave;
  int64_t lo = 0;
  int64_t hi = n - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (crow[mid] <= e) lo = mid;
    else hi = mid - 1;
  }
  rows[w] = static_cast<int32_t>(lo);
}

// Byte offset of 16-byte chunk lane_off of row `row` of a [*, F] matrix.
template <bool OFF32>
__device__ __forceinline__ const char* chunk_at(const char* base, int row, uint32_t row_bytes, uint32_t lane_off) {
  if constexpr (OFF32) {
    return base + (__umul24(static_cast<uint32_t>(row), row_bytes) + lane_off);
  } else {
    return base + static_cast<int64_t>(row) * row_bytes + lane_off;
  }
}

// Ragged rows (RAG: F % 8 != 0, or rows that are not 16-byte aligned; F >= 8):
// the same lanes with loads aligned to an element, the row's last chunk read
// at F - 8.  The features it shares with the chunk before are cleared on both
// sides (0 * 0 adds nothing to a sum, which starts at +0).  One wave per edge
// with a 2-byte lane a feature, us before -> after: 200k rows, 3.2M edges bf16
// F = 47 434 -> 88, F = 100 491 -> 113; 1M rows, 16M edges F = 47 1985 -> 536,
// F = 100 2302 -> 783 (F = 48 457, F = 104 760).
// A lane's chunks j + G·m of rows of F features.
template <int G, int MB, bool RAG>
struct Chunks16 {
  int chunks;
  uint32_t off[MB];
  uint32_t mask[RAG ? MB : 1][4];
  __device__ __forceinline__ Chunks16(int64_t F, int j) {
    chunks = static_cast<int>(RAG ? (F + 7) / 8 : F / 8);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int c = j + G * m;
      off[m] = static_cast<uint32_t>((c < chunks ? c : 0) * 16);
      if constexpr (RAG) {
        const int dup = c == chunks - 1 ? static_cast<int>(chunks * 8 - F) : 0;
        off[m] -= static_cast<uint32_t>(dup * 2);
#pragma unroll
        for (int i = 0; i < 4; ++i) mask[m][i] = 2 * i + 1 < dup ? 0u : (2 * i < dup ? 0xffff0000u : ~0u);
      }
    }
  }
  template <typename T>
  __device__ __forceinline__ double get(const RawVec<16>& v, int m, int p) const {
    if constexpr (RAG) {
      const uint32_t w = v.w[p >> 1] & mask[m][p >> 1];
      return static_cast<double>(Elem<T>::get(&w, p & 1));
    } else {
      return static_cast<double>(Elem<T>::get(v.w, p));
    }
  }
};

// The dot products of one block of cnt <= 64 edges starting at edge b,
// vector lanes: lane j of lane group g holds chunks j + G·m of the edge's
// query and key rows.  my_c / my_row: lane i holds the column / row of edge
// b + i.
template <typename T, int G, int MB, bool OFF32, bool RAG>
__device__ __forceinline__ void edge_block16_vec(const char* __restrict__ kb, const char* __restrict__ qb,
                                                 uint16_t* __restrict__ out, int64_t F, int64_t b, int cnt, int my_c,
                                                 int my_row) {
  constexpr int NG = kWave / G;  // edges per gather instruction
  // key (and query) gathers in flight per lane and chunk; fewer at 32 lanes
  // an edge, which would spill at 4
  constexpr int UE = MB == 1 ? (G >= 32 ? 2 : (4 < G ? 4 : G)) : 1;
  constexpr int kSub = NG * UE;  // edges per sub-pass, divides 64
  static_assert(kWave % kSub == 0, "a sub-pass stays inside its block of 64 edges");
  const int lane = lane_id();
  const int g = lane / G;
  const int j = lane % G;
  const Chunks16<G, MB, RAG> lanes(F, j);
  const uint32_t row_bytes = static_cast<uint32_t>(F * sizeof(T));
  for (int u0 = 0; u0 < cnt; u0 += kSub) {
    RawVec<16> kv[UE][MB];
    RawVec<16> qv[UE][MB];
#pragma unroll
    for (int u = 0; u < UE; ++u) {
      if (u0 + u * NG < cnt) {
        const int addr = (u0 + u * NG + g) * 4;  // an edge of this block (< 64)
        const int c = __builtin_amdgcn_ds_bpermute(addr, my_c);
        const int rw = __builtin_amdgcn_ds_bpermute(addr, my_row);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          kv[u][m] = load_raw16<RAG>(chunk_at<OFF32>(kb, c, row_bytes, lanes.off[m]));
          qv[u][m] = load_raw16<RAG>(chunk_at<OFF32>(qb, rw, row_bytes, lanes.off[m]));
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UE; ++u) {
      if (u0 + u * NG < cnt) {
        double acc = 0.0;
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          if (j + G * m < lanes.chunks) {
#pragma unroll
            for (int p = 0; p < 8; ++p)
              acc = __builtin_fma(lanes.template get<T>(qv[u][m], m, p), lanes.template get<T>(kv[u][m], m, p), acc);
          }
        }
#pragma unroll
        for (int o = 1; o < G; o <<= 1) acc += __shfl_xor(acc, o, kWave);
        const int idx = u0 + u * NG + g;
        if (j == 0 && idx < cnt) out[b + idx] = Elem<T>::bits(acc);
      }
    }
  }
}

// A wave whose edges [b0, b1) all lie in row `row` (long rows): the lane's
// query chunks are loaded once and the blocks need no row lookup.  The same
// products, sums and butterfly.
template <typename T, int G, int MB, bool OFF32, bool RAG>
__device__ __forceinline__ void one_row_edges16_vec(const int64_t* __restrict__ col, const char* __restrict__ kb,
                                                    const char* __restrict__ qb, uint16_t* __restrict__ out,
                                                    int64_t F, int64_t b0, int64_t b1, int row) {
  constexpr int NG = kWave / G;
  constexpr int UE = MB == 1 ? (4 < G ? 4 : G) : 1;
  constexpr int kSub = NG * UE;
  static_assert(kWave % kSub == 0, "a sub-pass stays inside its block of 64 edges");
  const int lane = lane_id();
  const int g = lane / G;
  const int j = lane % G;
  const Chunks16<G, MB, RAG> lanes(F, j);
  const uint32_t row_bytes = static_cast<uint32_t>(F * sizeof(T));
  RawVec<16> q[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) q[m] = load_raw16<RAG>(chunk_at<OFF32>(qb, row, row_bytes, lanes.off[m]));
  int next_c = b0 + lane < b1 ? static_cast<int>(col[b0 + lane]) : 0;
  for (int64_t b = b0; b < b1; b += kWave) {
    const int cnt = b1 - b < kWave ? static_cast<int>(b1 - b) : kWave;
    const int my_c = next_c;
    if (b + kWave < b1) next_c = b + kWave + lane < b1 ? static_cast<int>(col[b + kWave + lane]) : 0;
    for (int u0 = 0; u0 < cnt; u0 += kSub) {
      RawVec<16> kv[UE][MB];
#pragma unroll
      for (int u = 0; u < UE; ++u) {
        if (u0 + u * NG < cnt) {
          const int c = __builtin_amdgcn_ds_bpermute((u0 + u * NG + g) * 4, my_c);
#pragma unroll
          for (int m = 0; m < MB; ++m) kv[u][m] = load_raw16<RAG>(chunk_at<OFF32>(kb, c, row_bytes, lanes.off[m]));
        }
      }
#pragma unroll
      for (int u = 0; u < UE; ++u) {
        if (u0 + u * NG < cnt) {
          double acc = 0.0;
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            if (j + G * m < lanes.chunks) {
#pragma unroll
              for (int p = 0; p < 8; ++p)
                acc = __builtin_fma(lanes.template get<T>(q[m], m, p), lanes.template get<T>(kv[u][m], m, p), acc);
            }
          }
#pragma unroll
          for (int o = 1; o < G; o <<= 1) acc += __shfl_xor(acc, o, kWave);
          const int idx = u0 + u * NG + g;
          if (j == 0 && idx < cnt) out[b + idx] = Elem<T>::bits(acc);
        }
      }
    }
  }
}

template <typename T, int G, int MB, bool VEC, bool OFF32, bool RAG>
__global__ __launch_bounds__(kEdgeWaves * kWave) __attribute__((amdgpu_waves_per_eu(8))) void sddmm16_edges_kernel(
    const int64_t* __restrict__ crow, const int64_t* __restrict__ col, const T* __restrict__ query,
    const T* __restrict__ key, uint16_t* __restrict__ out, int64_t n, int64_t nnz, int64_t F,
    const int32_t* __restrict__ wave_rows, int64_t waves, int64_t wave_base) {
  const int64_t w = wave_base + static_cast<int64_t>(blockIdx.x) * kEdgeWaves + wave_in_block();
  if (w >= waves) return;  // wave-uniform
  const int lane = lane_id();
  const int64_t b0 = uniform_i64(w * kEdgesPerWave);
  const int64_t b1 = uniform_i64(b0 + kEdgesPerWave < nnz ? b0 + kEdgesPerWave : nnz);
  int64_t r = uniform_i64(wave_rows[w]);
  const char* __restrict__ kb = reinterpret_cast<const char*>(key);
  const char* __restrict__ qb = reinterpret_cast<const char*>(query);
  if constexpr (VEC) {
    if (uniform_i64(crow[r + 1]) >= b1) {  // every edge of the wave is in row r
      one_row_edges16_vec<T, G, MB, OFF32, RAG>(col, kb, qb, out, F, b0, b1, static_cast<int>(r));
      return;
    }
  }
  int next_c = b0 + lane < b1 ? static_cast<int>(col[b0 + lane]) : 0;
  for (int64_t b = b0; b < b1; b += kWave) {
    const int cnt = b1 - b < kWave ? static_cast<int>(b1 - b) : kWave;
    const int my_c = next_c;
    if (b + kWave < b1) next_c = b + kWave + lane < b1 ? static_cast<int>(col[b + kWave + lane]) : 0;
    const int my_row = block_edge_rows(crow, n, b, cnt, r);
    r = __builtin_amdgcn_readlane(my_row, cnt - 1);
    if constexpr (VEC) {
      edge_block16_vec<T, G, MB, OFF32, RAG>(kb, qb, out, F, b, cnt, my_c, my_row);
    } else {
      // element lanes: lane l adds features l, l + 64, ... of each edge in
      // turn (the order of dots16_scalar)
      for (int idx = 0; idx < cnt; ++idx) {
        const int64_t c = __builtin_amdgcn_readlane(my_c, idx);
        const int64_t rw = __builtin_amdgcn_readlane(my_row, idx);
        const T* __restrict__ kr = key + c * F;
        const T* __restrict__ qr = query + rw * F;
        double acc = 0.0;
        for (int64_t f = lane; f < F; f += kWave)
          acc = __builtin_fma(static_cast<double>(Elem<T>::at(qr, f)), static_cast<double>(Elem<T>::at(kr, f)), acc);
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) acc += __shfl_xor(acc, o, kWave);
        if (lane == 0) out[b + idx] = Elem<T>::bits(acc);
      }
    }
  }
}

template <typename T>
void launch_sddmm16_edges(const Sddmm16Args& a, int64_t nnz, int32_t* wave_rows, hipStream_t s) {
  const int64_t waves = edge_waves(nnz);
  hipLaunchKernelGGL(edge_wave_rows_kernel, dim3(static_cast<unsigned>((waves + 255) / 256)), dim3(256), 0, s,
                     a.crow, a.n, waves, wave_rows);
  int g, mb;
  const bool ragged = a.f % 8 != 0 || !aligned(a.q, 16) || !aligned(a.k, 16);
  sddmm16_lanes(a.f, g, mb);
  const bool off32 = sddmm16_off32(a);
  const int64_t blocks = (waves + kEdgeWaves - 1) / kEdgeWaves;
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
    const dim3 grid(static_cast<unsigned>(nb));
    const dim3 block(kEdgeWaves * kWave);
#define AS_E16(G, MB, VEC, OFF, RAG)                                                                         \
  hipLaunchKernelGGL((sddmm16_edges_kernel<T, G, MB, VEC, OFF, RAG>), grid, block, 0, s, a.crow, a.col,           \
                     static_cast<const T*>(a.q), static_cast<const T*>(a.k), static_cast<uint16_t*>(a.out), a.n, \
                     nnz, a.f, wave_rows, waves, b0 * kEdgeWaves)
#define AS_E16_V(G, MB)                                    \
  do {                                                     \
    if (ragged && off32) AS_E16(G, MB, true, true, true);   \
    else if (ragged) AS_E16(G, MB, true, false, true);      \
    else if (off32) AS_E16(G, MB, true, true, false);       \
    else AS_E16(G, MB, true, false, false);                 \
  } while (0)
    if (mb == 2) {
      AS_E16_V(32, 2);
    } else {
      switch (g) {
        case 1: AS_E16_V(1, 1); break;
        case 2: AS_E16_V(2, 1); break;
        case 4: AS_E16_V(4, 1); break;
        case 8: AS_E16_V(8, 1); break;
        case 16: AS_E16_V(16, 1); break;
        case 32: AS_E16_V(32, 1); break;
        default: AS_E16(64, 1, false, false, false); break;
      }
    }
#undef AS_E16_V
#undef AS_E16
  }
}

int validate_sddmm(const SddmmArgs& a, int64_t nnz) {
  if (a.n < 0 || a.n > INT32_MAX || a.f < 0)
    return fail(AS_ERR_INVALID_ARGUMENT, "SDDMM dimensions exceed the kernel index range");
  if (a.f >= as::kMaxFeatures) return fail(AS_ERR_UNSUPPORTED, "F must be below 2^28 (32-bit lane offsets)");
  if (nnz < 0) return fail(AS_ERR_INVALID_ARGUMENT, "nnz must be non-negative");
  if (a.n > 0 && a.crow == nullptr) return fail(AS_ERR_INVALID_ARGUMENT, "null crow pointer");
  if (nnz > 0 && (a.col == nullptr || a.q == nullptr || a.k == nullptr || a.out == nullptr))
    return fail(AS_ERR_INVALID_ARGUMENT, "null pointer argument");
  return AS_OK;
}

size_t sddmm_split_ws(int64_t n) {
  return spmm_split_workspace_bytes(n) + align_up(static_cast<size_t>(n > 0 ? n : 1) * sizeof(int32_t), 256);
}

}  // namespace

void launch_sddmm_scaled(const int64_t* crow, const int64_t* col, const float* query, const float* key, float* out,
                         int64_t n, int64_t nnz, int64_t f, float scale, hipStream_t s) {
  launch_sddmm_edges(SddmmArgs{crow, col, query, key, out, n, f}, nnz, n, scale, s);
}

}  // namespace as

extern "C" {

int as_sddmm_csr_edges_f32(const int64_t* crow, const int64_t* col, const float* query, const float* key, float* out,
                           int64_t n, int64_t n_keys, int64_t nnz, int64_t f, void* stream) {
  as::clear_error();
  if (n_keys > INT32_MAX) return as::fail(AS_ERR_INVALID_ARGUMENT, "n_keys exceeds kernel index range");
  as::SddmmArgs a{crow, col, query, key, out, n, f};
  int st = as::validate_sddmm(a, nnz);
  if (st != AS_OK) return st;
  if (n == 0 || nnz == 0) return AS_OK;
  if (f == 0) return as::fail(AS_ERR_UNSUPPORTED, "SDDMM with zero features is handled by the caller");
  as::launch_sddmm_edges(a, nnz, n_keys, 1.f, static_cast<hipStream_t>(stream));
  return as::check_launch("sddmm_csr");
}

int as_sddmm_csr_rows_f32(const int64_t* crow, const int64_t* col, const float* query, const float* key, float* out,
                          int64_t n, int64_t nnz, int64_t f, void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  as::SddmmArgs a{crow, col, query, key, out, n, f};
  int st = as::validate_sddmm(a, nnz);
  if (st != AS_OK) return st;
  if (n == 0 || nnz == 0) return AS_OK;
  if (!as::sddmm_rows_fit(a))
    return as::fail(AS_ERR_UNSUPPORTED, "SDDMM by rows takes multiples of 32 features up to 256, 16-byte aligned");
  if (workspace == nullptr || workspace_bytes < as::sddmm_split_ws(n))
    return as::fail(AS_ERR_WORKSPACE, "SDDMM by rows needs %zu workspace bytes, got %zu", as::sddmm_split_ws(n),
                    workspace_bytes);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  int32_t* order = reinterpret_cast<int32_t*>(ws);
  const size_t order_bytes = as::align_up(static_cast<size_t>(n) * sizeof(int32_t), 256);
  int32_t* counts = reinterpret_cast<int32_t*>(ws + order_bytes);
  int32_t* chunk_off = reinterpret_cast<int32_t*>(ws + as::spmm_split_workspace_bytes(n));
  int64_t hubs = nnz / as::kRowsHub;
  if (hubs > n) hubs = n;
  int64_t hub_blocks = 0;
  if (hubs > 0) {
    st = as::launch_bin_rows(crow, n, as::kRowsHub, 1, 1, order, counts, ws + order_bytes + 256, s);
    if (st != AS_OK) return st;
    hipLaunchKernelGGL(as::hub_chunk_scan_kernel, dim3(1), dim3(1024), 0, s, crow, order, counts, chunk_off);
    hub_blocks = nnz / as::kChunkEdges + hubs;
    if (hub_blocks > as::kHubBlocksMax) hub_blocks = as::kHubBlocksMax;
  }
  as::launch_sddmm_rows(a, hub_blocks, order, counts, chunk_off, s);
  return as::check_launch("sddmm_csr_rows");
}

int as_sddmm_csr_f32(const int64_t* crow, const int64_t* col, const float* query, const float* key, float* out,
                     int64_t n, int64_t nnz, int64_t f, void* stream) {
  return as_sddmm_csr_edges_f32(crow, col, query, key, out, n, -1, nnz, f, stream);
}

size_t as_sddmm_split_workspace_bytes(int64_t n) { return as::sddmm_split_ws(n < 0 ? 0 : n); }

int as_sddmm_csr_split_f32(const int64_t* crow, const int64_t* col, const float* query, const float* key,
                           float* out, int64_t n, int64_t nnz, int64_t f, int waves_per_block,
                           int64_t hub_threshold, void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  as::SddmmArgs a{crow, col, query, key, out, n, f};
  if (waves_per_block != 2 && waves_per_block != 4 && waves_per_block != 8)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "warps_per_block must be 2, 4, or 8");
  if (hub_threshold <= 0 || hub_threshold > INT32_MAX)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "hub_threshold must be a positive 32-bit integer");
  int st = as::validate_sddmm(a, nnz);
  if (st != AS_OK) return st;
  if (n == 0 || nnz == 0) return AS_OK;
  if (f == 0) return as::fail(AS_ERR_UNSUPPORTED, "SDDMM with zero features is handled by the caller");
  if (workspace == nullptr || workspace_bytes < as::sddmm_split_ws(n))
    return as::fail(AS_ERR_WORKSPACE, "split SDDMM needs %zu workspace bytes, got %zu", as::sddmm_split_ws(n),
                    workspace_bytes);
  // every schedule gives the same bits, and the blocks of edges need none
  as::launch_sddmm_edges(a, nnz, -1, 1.f, static_cast<hipStream_t>(stream));
  return as::check_launch("sddmm_csr_split");
}

int as_sddmm_csr_rounded_16(const int64_t* crow, const int64_t* col, const void* query, const void* key, void* out,
                            int64_t n, int64_t nnz, int64_t f, int dtype, int waves_per_block, int64_t hub_threshold,
                            void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  if (dtype != AS_DTYPE_BF16 && dtype != AS_DTYPE_F16)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "dtype must be AS_DTYPE_BF16 or AS_DTYPE_F16");
  if (waves_per_block != 2 && waves_per_block != 4 && waves_per_block != 8)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "warps_per_block must be 2, 4, or 8");
  if (hub_threshold <= 0 || hub_threshold > INT32_MAX)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "hub_threshold must be a positive 32-bit integer");
  if (!as::aligned(query, 2) || !as::aligned(key, 2) || !as::aligned(out, 2))
    return as::fail(AS_ERR_INVALID_ARGUMENT, "query, key and out must be 2-byte aligned");
  // the fp32 argument check covers the shapes and null pointers
  const as::SddmmArgs shape{crow, col, static_cast<const float*>(query), static_cast<const float*>(key),
                            static_cast<float*>(out), n, f};
  int st = as::validate_sddmm(shape, nnz);
  if (st != AS_OK) return st;
  if (n == 0 || nnz == 0) return AS_OK;
  if (f == 0) return as::fail(AS_ERR_UNSUPPORTED, "SDDMM with zero features is handled by the caller");
  if (workspace == nullptr || workspace_bytes < as::sddmm_split_ws(n))
    return as::fail(AS_ERR_WORKSPACE, "16-bit SDDMM needs %zu workspace bytes, got %zu", as::sddmm_split_ws(n),
                    workspace_bytes);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const as::Sddmm16Args a{crow, col, query, key, out, n, f, n};
  char* ws = static_cast<char*>(workspace);
  int32_t* order = reinterpret_cast<int32_t*>(ws);
  const size_t order_bytes = as::align_up(static_cast<size_t>(n) * sizeof(int32_t), 256);
  int32_t* counts = reinterpret_cast<int32_t*>(ws + order_bytes);
  void* bin_ws = ws + order_bytes + 256;
  int32_t* chunk_off = reinterpret_cast<int32_t*>(ws + as::spmm_split_workspace_bytes(n));
  int64_t heavy_upper = nnz / hub_threshold;
  if (heavy_upper > n) heavy_upper = n;
  int64_t item_upper = 0;
  if (heavy_upper > 0) {
    st = as::launch_bin_rows(crow, n, hub_threshold, 1, 1, order, counts, bin_ws, s);
    if (st != AS_OK) return st;
    hipLaunchKernelGGL(as::hub_chunk_scan_kernel, dim3(1), dim3(1024), 0, s, crow, order, counts, chunk_off);
    item_upper = nnz / as::kChunkEdges + heavy_upper;
  }
  // with item_upper == 0 there are no hub workgroups and no row reaches the
  // threshold, so the kernel reads neither the order nor the counts
  if (dtype == AS_DTYPE_BF16)
    as::launch_sddmm16<as::Bf16>(a, waves_per_block, hub_threshold, item_upper, order, counts, chunk_off, s);
  else
    as::launch_sddmm16<as::Fp16>(a, waves_per_block, hub_threshold, item_upper, order, counts, chunk_off, s);
  return as::check_launch("sddmm_csr_rounded_16");
}

size_t as_sddmm_edges_16_workspace_bytes(int64_t nnz) { return as::sddmm_edges_ws(nnz < 0 ? 0 : nnz); }

int as_sddmm_csr_edges_16_rect(const int64_t* crow, const int64_t* col, const void* query, const void* key,
                               void* out, int64_t n, int64_t n_keys, int64_t nnz, int64_t f, int dtype,
                               void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  if (n_keys < 0 || n_keys > INT32_MAX) return as::fail(AS_ERR_INVALID_ARGUMENT, "n_keys exceeds kernel index range");
  if (dtype != AS_DTYPE_BF16 && dtype != AS_DTYPE_F16)
    return as::fail(AS_ERR_INVALID_ARGUMENT, "dtype must be AS_DTYPE_BF16 or AS_DTYPE_F16");
  if (!as::aligned(query, 2) || !as::aligned(key, 2) || !as::aligned(out, 2))
    return as::fail(AS_ERR_INVALID_ARGUMENT, "query, key and out must be 2-byte aligned");
  const as::SddmmArgs shape{crow, col, static_cast<const float*>(query), static_cast<const float*>(key),
                            static_cast<float*>(out), n, f};
  int st = as::validate_sddmm(shape, nnz);
  if (st != AS_OK) return st;
  if (n == 0 || nnz == 0) return AS_OK;
  if (f == 0) return as::fail(AS_ERR_UNSUPPORTED, "SDDMM with zero features is handled by the caller");
  if (workspace == nullptr || workspace_bytes < as::sddmm_edges_ws(nnz))
    return as::fail(AS_ERR_WORKSPACE, "16-bit SDDMM by edge blocks needs %zu workspace bytes, got %zu",
                    as::sddmm_edges_ws(nnz), workspace_bytes);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const as::Sddmm16Args a{crow, col, query, key, out, n, f, n_keys};
  int32_t* wave_rows = static_cast<int32_t*>(workspace);
  if (dtype == AS_DTYPE_BF16)
    as::launch_sddmm16_edges<as::Bf16>(a, nnz, wave_rows, s);
  else
    as::launch_sddmm16_edges<as::Fp16>(a, nnz, wave_rows, s);
  return as::check_launch("sddmm_csr_edges_16");
}

int as_sddmm_csr_edges_16(const int64_t* crow, const int64_t* col, const void* query, const void* key, void* out,
                          int64_t n, int64_t nnz, int64_t f, int dtype, void* workspace, size_t workspace_bytes,
                          void* stream) {
  return as_sddmm_csr_edges_16_rect(crow, col, query, key, out, n, n < 0 ? 0 : n, nnz, f, dtype, workspace,
                                    workspace_bytes, stream);
}

}  // extern "C"
