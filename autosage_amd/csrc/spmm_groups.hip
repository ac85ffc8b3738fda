// CSR SpMM Y = A·X for fp32 features: short rows in lane groups, long rows by
// workgroups, in one launch without a binning.
//
// Every output element is one fp32 accumulator updated in CSR edge order
// (fmaf with a weight, acc + x without), as in spmm.hip: the bits of the
// sequential CPU product (csrc/spmm_csr_vec4.cu:42-50, autosage/ops.py:124-143).
//
// Short rows (light_groups): ceil(F/4) lanes per row, 4 features a lane, so a
// gather instruction carries 64·4/F rows' edges; loads of 16 bytes aligned to 4,
// the last lane of a row reading its last 4 features (the overlap is computed
// twice and stored twice, the same bits), so any F >= 4 has vector lanes.  A
// wave owns up to 60 consecutive rows and hands the next one to each lane group
// that finishes; a batch of 8 edges' column indices is loaded one batch ahead.
//
// Long rows (at least kSpmmLongRow edges; half of that in small graphs): one chain per feature is a chain of
// dependent additions, but its gathers need not wait for it.  The first
// workgroups of the launch each scan a strided share of crow for long rows and
// take them one after another (per slice of at most 64 features): 3 waves gather
// tiles of 48 to 192 edges into LDS, 3 tiles in flight and their indices 3 more
// ahead; the 4th wave adds the tiles in edge order, one feature a lane.
// Workgroups are dispatched in index order, so the long rows start first.
//
// What bounds it: short rows, the gathers; long rows, a tile's gathers in
// flight and the adding wave (about 10 ns an edge: a row of 10,000 edges takes 0.1
// ms, where one wave that gathers and adds took 0.35 ms).  The adding wave reads
// the next 8 values from LDS before it adds 8 (13 ns an edge without).  us, one
// wave per row -> this kernel:
//   200k rows, 3.2M edges, longest 1,000: F = 16 142 -> 80, F = 64 138 -> 96, F = 128 196 -> 147
//   170k rows, 2.4M edges, longest 10,000: F = 32 350 -> 98, F = 47 395 -> 138, F = 128 425 -> 162
//   40k rows, 400k edges, even: F = 16 12 -> 7, F = 64 18 -> 15, F = 100 28 -> 27
//   1M rows, 16.8M edges, even: F = 16 506 -> 376, F = 128 1217 -> 1298 (as_spmm_csr_f32
//   keeps one wave per row for wide, even rows where the caller knows them)
#include "as_device.h"
#include "as_internal.h"

namespace as {
namespace {

typedef float Float4U __attribute__((ext_vector_type(4), aligned(4)));

struct GroupArgs {
  const int64_t* crow;
  const int64_t* col;
  const float* val;
  const float* x;
  float* y;
  int64_t n;
  int64_t nnz;
  int64_t F;
  int lpr;             // lanes per row
  int rpw;             // rows in flight per wave
  int pool;            // consecutive rows of a wave, <= 60
  int tile;            // features per tile (a multiple of 4, <= 256)
  int tiles;
  int64_t hub_stride;  // hub workgroups per feature slice (0: no long rows)
  int hub_slices;
  int hub_width;       // features per slice (a multiple of 4, <= 64)
  int64_t long_row;  // edges from which a workgroup takes a row
};

// ---- long rows ---------------------------------------------------------------
constexpr int kHubSets = 3;       // tiles of gathers in flight
constexpr int kHubU = 4;          // gathers per lane and tile
constexpr int kHubProducers = kWavesPerBlock - 1;
constexpr int kHubChunk = 256;    // rows scanned at a time
constexpr int kHubLine = 8;       // rows of one 64-byte line of crow
constexpr int kHubTileFloats = kHubProducers * kHubU * 64 * 4;

struct HubShared {
  alignas(16) float tile[2][kHubTileFloats];
  alignas(16) float w[2][kHubProducers * kWave];
  int64_t first[kHubChunk];
  int64_t len[kHubChunk];
  int32_t row[kHubChunk];
  int32_t count;
};

// Where the stream of tiles of a chunk's long rows stands, the same in every
// wave; len and first are those of list entry `row` (the last one past the end).
struct HubCursor {
  int row;
  int64_t k;  // edges of the row taken so far
  int64_t len;
  int64_t first;
};
__device__ __forceinline__ void hub_enter(HubCursor& c, const HubShared& sh, int row, int rows) {
  const int r = row < rows ? row : rows - 1;
  c.row = row;
  c.k = 0;
  c.len = uniform_i64(sh.len[r]);
  c.first = uniform_i64(sh.first[r]);
}

// STRIDE: floats per edge of a tile (16, 32 or 64 >= the slice's width).
template <int STRIDE>
struct HubShape {
  static constexpr int kEpl = 256 / STRIDE;              // edges per gather instruction
  static constexpr int kWaveEdges = kHubU * kEpl;        // edges per producer wave and tile, <= 64
  static constexpr int kTileEdges = kHubProducers * kWaveEdges;
  static_assert(kWaveEdges <= kWave && kTileEdges * STRIDE <= kHubTileFloats, "a tile fits its buffer");
};

template <int STRIDE, bool HAS_VAL, bool OFF32>
__device__ __forceinline__ void hub_produce(const GroupArgs& a, HubShared& sh, int rows, int64_t tiles, int f0,
                                            int width) {
  using S = HubShape<STRIDE>;
  constexpr int LP = STRIDE / 4;  // lanes per edge
  const int lane = lane_id();
  const int wave = wave_in_block();
  const int L = (width + 3) / 4;
  const int g = lane / LP;
  const int j = lane % LP < L ? lane % LP : L - 1;  // lanes past the slice repeat its last vector
  const int start = 4 * j < width - 4 ? 4 * j : width - 4;
  const uint32_t lane_bytes = static_cast<uint32_t>((f0 + start) * 4);
  const uint32_t row_bytes = static_cast<uint32_t>(a.F * 4);
  const char* __restrict__ xb = reinterpret_cast<const char*>(a.x);
  // this lane's column: edge `mine` of its tile
  const int mine = wave * S::kWaveEdges + (lane < S::kWaveEdges ? lane : S::kWaveEdges - 1);
  // this lane's gathers: edges u·kEpl + g of the wave's
  float* out = &sh.tile[0][(wave * S::kWaveEdges + g) * STRIDE + 4 * j];
  HubCursor at;
  hub_enter(at, sh, 0, rows);
  int ic[kHubSets];
  float iw[kHubSets], gw[kHubSets];
  Float4U xs[kHubSets][kHubU];
  // every load is issued whatever the tile holds (absent edges read the row's
  // last edge again), so that the waits count the loads in flight
  auto index_stage = [&](int s) {
    int64_t e = at.k + mine;
    e = at.first + (e < at.len ? e : at.len - 1);
    ic[s] = reinterpret_cast<const int*>(a.col)[2 * e];  // the low word
    iw[s] = 0.f;
    if constexpr (HAS_VAL) iw[s] = a.val[e];
    at.k += S::kTileEdges;
    if (at.k >= at.len) hub_enter(at, sh, at.row + 1, rows);
  };
  auto gather_stage = [&](int s) {
    gw[s] = iw[s];
#pragma unroll
    for (int u = 0; u < kHubU; ++u) {
      const int c = __builtin_amdgcn_ds_bpermute((u * S::kEpl + g) * 4, ic[s]);
      if constexpr (OFF32)
        xs[s][u] = *reinterpret_cast<const Float4U*>(xb + (static_cast<uint32_t>(c) * row_bytes + lane_bytes));
      else
        xs[s][u] = *reinterpret_cast<const Float4U*>(
            xb + (static_cast<uint64_t>(static_cast<uint32_t>(c)) * row_bytes + lane_bytes));
    }
  };
#pragma unroll
  for (int s = 0; s < kHubSets; ++s) index_stage(s);
#pragma unroll
  for (int s = 0; s < kHubSets; ++s) {
    gather_stage(s);
    index_stage(s);
  }
  int buffer = 0;
  for (int64_t t = 0; t < tiles; t += kHubSets) {
#pragma unroll
    for (int s = 0; s < kHubSets; ++s) {
#pragma unroll
      for (int u = 0; u < kHubU; ++u) {
        *reinterpret_cast<float4*>(out + buffer * kHubTileFloats + u * S::kEpl * STRIDE) =
            float4{xs[s][u].x, xs[s][u].y, xs[s][u].z, xs[s][u].w};
      }
      if constexpr (HAS_VAL) sh.w[buffer][mine] = gw[s];
      __syncthreads();
      gather_stage(s);
      index_stage(s);
      buffer ^= 1;
    }
  }
}

template <int STRIDE, bool HAS_VAL>
__device__ __forceinline__ void hub_consume(const GroupArgs& a, HubShared& sh, int rows, int64_t tiles, int f0,
                                            int width) {
  using S = HubShape<STRIDE>;
  constexpr int B = 8;
  static_assert(S::kTileEdges % B == 0, "whole batches");
  const int lane = lane_id();
  const int L = (width + 3) / 4;
  // the slice's last vector starts at feature width - 4
  int pos = lane < 4 * (L - 1) ? lane : 4 * (L - 1) + lane - (width - 4);
  if (lane >= width) pos = 0;
  HubCursor at;
  hub_enter(at, sh, 0, rows);
  float acc = 0.f;
  int buffer = 0;
  const int64_t steps = (tiles + kHubSets - 1) / kHubSets * kHubSets;
  for (int64_t t = 0; t < steps; ++t) {
    __syncthreads();
    if (at.row < rows) {
      const int64_t left = at.len - at.k;
      const int cnt = left < S::kTileEdges ? static_cast<int>(left) : S::kTileEdges;
      const float* v = &sh.tile[buffer][pos];
      const float4* w = reinterpret_cast<const float4*>(&sh.w[buffer][0]);
      float x[2][B];
      float4 y[2][B / 4];
      auto load = [&](int p, int b) {
#pragma unroll
        for (int i = 0; i < B; ++i) x[p][i] = v[(b * B + i) * STRIDE];
        if constexpr (HAS_VAL) {
#pragma unroll
          for (int i = 0; i < B / 4; ++i) y[p][i] = w[b * (B / 4) + i];
        }
      };
      auto next = [&](int p, int i) {
        if constexpr (HAS_VAL) {
          const float4 q = y[p][i / 4];
          return __builtin_fmaf(i % 4 == 0 ? q.x : i % 4 == 1 ? q.y : i % 4 == 2 ? q.z : q.w, x[p][i], acc);
        } else {
          return acc + x[p][i];
        }
      };
      constexpr int kBatches = S::kTileEdges / B;
      load(0, 0);
      if (cnt == S::kTileEdges) {
#pragma unroll
        for (int b = 0; b < kBatches; ++b) {
          if (b + 1 < kBatches) load((b + 1) & 1, b + 1);
          __builtin_amdgcn_sched_barrier(0);  // the reads first
#pragma unroll
          for (int i = 0; i < B; ++i) acc = next(b & 1, i);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        for (int e = 0; e < cnt; e += B) {
#pragma unroll
          for (int i = 0; i < B; ++i) {
            const float z = next(0, i);
            acc = e + i < cnt ? z : acc;
          }
          v += B * STRIDE;
          w += B / 4;
          if (e + B < cnt) load(0, 0);
        }
      }
      at.k += S::kTileEdges;
      if (at.k >= at.len) {
        if (lane < width) a.y[static_cast<int64_t>(sh.row[at.row]) * a.F + f0 + lane] = acc;
        acc = 0.f;
        hub_enter(at, sh, at.row + 1, rows);
      }
    }
    buffer ^= 1;
  }
}

template <int STRIDE, bool HAS_VAL, bool OFF32>
__device__ __forceinline__ void hub_rows(const GroupArgs& a, HubShared& sh, int rows, int f0, int width) {
  using S = HubShape<STRIDE>;
  int64_t tiles = 0;
  for (int r = 0; r < rows; ++r) tiles += (uniform_i64(sh.len[r]) + S::kTileEdges - 1) / S::kTileEdges;
  if (wave_in_block() < kHubProducers) hub_produce<STRIDE, HAS_VAL, OFF32>(a, sh, rows, tiles, f0, width);
  else hub_consume<STRIDE, HAS_VAL>(a, sh, rows, tiles, f0, width);
}

template <bool HAS_VAL, bool OFF32>
__device__ __forceinline__ void hub_block(const GroupArgs& a, int64_t block, HubShared& sh) {
  const int slice = static_cast<int>(block % a.hub_slices);
  const int64_t first_line = block / a.hub_slices;
  const int f0 = slice * a.hub_width;
  const int width = static_cast<int>(a.F - f0 < a.hub_width ? a.F - f0 : a.hub_width);
  const int64_t lines = (a.n + kHubLine - 1) / kHubLine;
  constexpr int kChunkLines = kHubChunk / kHubLine;
  for (int64_t line0 = first_line; line0 < lines; line0 += a.hub_stride * kChunkLines) {
    // the chunk's long rows
    __syncthreads();
    if (threadIdx.x == 0) sh.count = 0;
    __syncthreads();
    const int t = static_cast<int>(threadIdx.x);  // kHubChunk == kBlock
    const int64_t line = line0 + static_cast<int64_t>(t / kHubLine) * a.hub_stride;
    const int64_t row = line * kHubLine + t % kHubLine;
    if (line < lines && row < a.n) {
      const int64_t rs = a.crow[row];
      const int64_t len = a.crow[row + 1] - rs;
      if (len >= a.long_row) {
        const int at = atomicAdd(&sh.count, 1);
        sh.first[at] = rs;
        sh.len[at] = len;
        sh.row[at] = static_cast<int>(row);
      }
    }
    __syncthreads();
    const int rows = __builtin_amdgcn_readfirstlane(sh.count);
    if (rows == 0) continue;
    if (a.hub_width <= 16) hub_rows<16, HAS_VAL, OFF32>(a, sh, rows, f0, width);
    else if (a.hub_width <= 32) hub_rows<32, HAS_VAL, OFF32>(a, sh, rows, f0, width);
    else hub_rows<64, HAS_VAL, OFF32>(a, sh, rows, f0, width);
  }
}

// ---- short rows ----------------------------------------------------------------
constexpr int kGroupUnroll = 8;  // edges of a batch

// A lane group's next batch.
struct Batch {
  int64_t row;  // -1: the group has no row left
  int cnt;
  bool last;    // of its row
  bool hub;     // a long row (no edges here, not stored)
};

// IPB: index loads per lane and batch (kGroupUnroll / lanes per row where a row
// has fewer than kGroupUnroll lanes, a power of two then).
template <int IPB, bool HAS_VAL, bool OFF32>
__device__ __forceinline__ void light_groups(const GroupArgs& a, int64_t light) {
  constexpr int U = kGroupUnroll;
  const int lane = lane_id();
  const int64_t w = light / a.tiles * kWavesPerBlock + wave_in_block();
  const int64_t row0 = uniform_i64(w * a.pool);
  if (row0 >= a.n) return;
  const int pool = static_cast<int>(a.n - row0 < a.pool ? a.n - row0 : a.pool);
  const int64_t ends = a.crow[row0 + (lane < pool ? lane : pool)];
  const int lpr = a.lpr;
  const int group = lane / lpr;
  const int sl = lane - group * lpr;
  const int gbase = lane - sl;
  const bool live = group < a.rpw;
  const int f0 = static_cast<int>(light % a.tiles) * a.tile;
  const int width = static_cast<int>(a.F - f0 < a.tile ? a.F - f0 : a.tile);
  const bool active = live && 4 * sl < width;
  // the last lane reads the tile's last 4 features (some twice; a tile of
  // fewer reaches into the one before it)
  const int fl = f0 + (4 * sl < width - 4 ? 4 * sl : width - 4);
  const uint32_t lane_bytes = static_cast<uint32_t>(fl * 4);
  const uint32_t row_bytes = static_cast<uint32_t>(a.F * 4);
  const char* __restrict__ xb = reinterpret_cast<const char*>(a.x);
  const uint64_t below = live ? (uint64_t(1) << gbase) - 1 : 0;

  int handed = 0;  // rows of the pool given to groups (wave-uniform)
  int64_t k = 0, end = 0;
  Batch next{-1, 0, false, false};
  int ic[IPB];
  float iw[IPB];
  auto fetch = [&]() {
    const bool need = live && k >= end;
    const uint64_t asks = __ballot(need && sl == 0);
    if (asks != 0) {
      const int idx = handed + __builtin_popcountll(asks & below);
      handed += __builtin_popcountll(asks);
      const int i0 = idx < pool ? idx : pool;
      const int i1 = idx < pool ? idx + 1 : pool;
      const int64_t rs = static_cast<int64_t>(__shfl(static_cast<long long>(ends), i0, kWave));
      const int64_t re = static_cast<int64_t>(__shfl(static_cast<long long>(ends), i1, kWave));
      if (need) {
        next.row = idx < pool ? row0 + idx : -1;
        next.hub = a.hub_stride > 0 && re - rs >= a.long_row;
        k = rs;
        end = next.hub ? rs : re;
      }
    }
    const int64_t left = end - k;
    next.cnt = left < U ? static_cast<int>(left) : U;
    next.last = left <= U;
#pragma unroll
    for (int i = 0; i < IPB; ++i) {
      // past the batch's edges its last one again (of an empty batch, some
      // edge), so that every load is issued and the waits can count them
      const int e = sl + i * lpr;
      int64_t at = k + (e < next.cnt ? e : (next.cnt > 0 ? next.cnt - 1 : 0));
      if (at >= a.nnz) at = a.nnz - 1;
      ic[i] = reinterpret_cast<const int*>(a.col)[2 * at];  // the low word
      iw[i] = 1.f;
      if constexpr (HAS_VAL) iw[i] = a.val[at];
    }
    k += next.cnt;
  };
  fetch();
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  while (__ballot(next.row >= 0) != 0) {
    const Batch cur = next;
    Float4U xv[U];
    float ws[U];
    auto gather = [&](int u) {
      const int src = (IPB == 1 ? gbase + u : gbase + u % (U / IPB)) * 4;
      const int reg = IPB == 1 ? 0 : u / (U / IPB);
      const int c = __builtin_amdgcn_ds_bpermute(src, ic[reg]);
      if constexpr (HAS_VAL) ws[u] = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(iw[reg])));
      if constexpr (OFF32)
        xv[u] = *reinterpret_cast<const Float4U*>(xb + (static_cast<uint32_t>(c) * row_bytes + lane_bytes));
      else
        xv[u] = *reinterpret_cast<const Float4U*>(
            xb + (static_cast<uint64_t>(static_cast<uint32_t>(c)) * row_bytes + lane_bytes));
    };
    auto add = [&](int u) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float t = HAS_VAL ? __builtin_fmaf(ws[u], xv[u][v], acc[v]) : acc[v] + xv[u][v];
        acc[v] = u < cur.cnt ? t : acc[v];
      }
    };
#pragma unroll
    for (int u = 0; u < U / 2; ++u) gather(u);
    const bool more = __ballot(cur.cnt > U / 2) != 0;
    if (more) {
#pragma unroll
      for (int u = U / 2; u < U; ++u) gather(u);
    }
    fetch();
#pragma unroll
    for (int u = 0; u < U / 2; ++u) add(u);
    if (more) {
#pragma unroll
      for (int u = U / 2; u < U; ++u) add(u);
    }
    if (cur.last) {
      if (active && cur.row >= 0 && !cur.hub)
        *reinterpret_cast<Float4U*>(a.y + cur.row * a.F + fl) = Float4U{acc[0], acc[1], acc[2], acc[3]};
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[v] = 0.f;
    }
  }
}

// Workgroups [0, hub_stride · hub_slices) take the long rows, the rest the
// short ones.
template <int IPB, bool HAS_VAL, bool OFF32>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void spmm_groups_kernel(
    GroupArgs a, int64_t block_base) {
  __shared__ HubShared sh;
  const int64_t hub_blocks = a.hub_stride * a.hub_slices;
  const int64_t block = block_base + blockIdx.x;
  if (block < hub_blocks) hub_block<HAS_VAL, OFF32>(a, block, sh);
  else light_groups<IPB, HAS_VAL, OFF32>(a, block - hub_blocks);
}

// Workgroups on the long rows, over all feature slices (at least 128 a slice;
// 512 / 1024 / 2048 with 3.2M edges at F = 128: 262 / 167 / 149 us).
constexpr int64_t kHubBlocks = 2048;
// Edges (times 64-feature slices) up to which a slice holds 32 features: the
// longest row's chain decides there, and tiles of 96 edges instead of 48 shorten
// it (720k edges, longest row 8,000, F = 64 119 -> 100 us, F = 128 133 -> 96); beyond, the
// indices read per slice cost more (3.2M edges, longest 1,000, F = 64 96 -> 104, F = 128
// 148 -> 162; 10M edges F = 64 202 -> 233).
constexpr int64_t kNarrowSliceEdges = 3000000;

template <int IPB>
void launch_groups(const GroupArgs& a, int64_t light, bool off32, hipStream_t s) {
  const int64_t blocks = light + a.hub_stride * a.hub_slices;
  for (int64_t b0 = 0; b0 < blocks; b0 += kMaxBlocksPerLaunch) {
    const int64_t nb = blocks - b0 < kMaxBlocksPerLaunch ? blocks - b0 : kMaxBlocksPerLaunch;
    const dim3 grid(static_cast<unsigned>(nb));
    if (a.val != nullptr) {
      if (off32) hipLaunchKernelGGL((spmm_groups_kernel<IPB, true, true>), grid, dim3(kBlock), 0, s, a, b0);
      else hipLaunchKernelGGL((spmm_groups_kernel<IPB, true, false>), grid, dim3(kBlock), 0, s, a, b0);
    } else {
      if (off32) hipLaunchKernelGGL((spmm_groups_kernel<IPB, false, true>), grid, dim3(kBlock), 0, s, a, b0);
      else hipLaunchKernelGGL((spmm_groups_kernel<IPB, false, false>), grid, dim3(kBlock), 0, s, a, b0);
    }
  }
}

}  // namespace

void launch_spmm_groups(const int64_t* crow, const int64_t* col, const float* val, const float* x, float* y, int64_t n,
                        int64_t n_cols, int64_t nnz, int64_t f, hipStream_t s) {
  GroupArgs a{crow, col, val, x, y, n, nnz, f, 0, 0, 0, 0, 0, 0, 1, 64, kSpmmLongRow};
  a.tiles = static_cast<int>((f + 255) / 256);
  a.tile = static_cast<int>(((f + a.tiles - 1) / a.tiles + 3) / 4 * 4);
  a.lpr = a.tile / 4;
  if (a.lpr < kGroupUnroll) {
    int p = 1;
    while (p < a.lpr) p <<= 1;
    a.lpr = p;
  }
  a.rpw = kWave / a.lpr;
  // rows per lane group: more smooth out rows of different lengths and hide the
  // start of a row, which matters less where rows are a few edges; fewer where
  // that would leave fewer than 16,384 waves (200k rows, 3.2M edges, power law,
  // F = 64, us at 1 / 2 / 4: 122 / 104 / 96; 200k rows of 4 edges, F = 128: 75 / 75 / 78)
  const int64_t most = nnz < 12 * n ? 2 : 4;
  int64_t m = n / (static_cast<int64_t>(a.rpw) * 16384);
  m = m < 1 ? 1 : (m > most ? most : m);
  a.pool = static_cast<int>(a.rpw * m < 60 ? a.rpw * m : 60);
  // graphs of few rows leave the chip idle, so rows that are short elsewhere go to
  // workgroups too (1000 rows of 30 edges, longest 200, F = 64: 17.4 -> 12.0 us; 2,600
  // rows of 59, longest 640, F = 16: 22.9 -> 19.1; level at 10,000 rows)
  a.long_row = n < 8192 ? kSpmmLongRow / 2 : kSpmmLongRow;
  if (nnz >= a.long_row) {
    const int64_t wide = (f + 63) / 64;
    a.hub_slices = static_cast<int>(nnz * wide <= kNarrowSliceEdges ? (f + 31) / 32 : wide);
    a.hub_width = static_cast<int>(((f + a.hub_slices - 1) / a.hub_slices + 3) / 4 * 4);
    const int64_t want = kHubBlocks / a.hub_slices > 128 ? kHubBlocks / a.hub_slices : 128;
    // at least 16 rows to scan; with 64 a workgroup took the long rows of a small
    // graph one after the other (5,000 rows of 64 edges, longest 1,200, F = 16:
    // 43.8 -> 24.4 us; 10,000 of 40, longest 2,000: 41.9 -> 28.5)
    const int64_t share = (n + 15) / 16;
    a.hub_stride = want < share ? want : share;
  }
  const int64_t waves = (n + a.pool - 1) / a.pool;
  const int64_t light = (waves + kWavesPerBlock - 1) / kWavesPerBlock * a.tiles;
  const bool off32 = n_cols >= 0 && n_cols * f * 4 <= (int64_t(1) << 32);
  switch (a.lpr) {
    case 1: launch_groups<8>(a, light, off32, s); break;
    case 2: launch_groups<4>(a, light, off32, s); break;
    case 4: launch_groups<2>(a, light, off32, s); break;
    default: launch_groups<1>(a, light, off32, s); break;
  }
}

}  // namespace as
