// CSR of an edge list, and the transpose of a CSR, on the device.
//
// Reference behaviour: edge_index_to_csr (autosage/utils/csr.py:6-26): a stable
// sort of the row ids (torch argsort), the other ends in that order, and the
// cumulative counts.  The transposed CSR of the backward lists, per column,
// the source rows in ascending order: a stable sort of the edges by column.
//
// Both are one stable sort of 32-bit ids with the edge numbers, over the bits
// that ids below n have (rocPRIM's radix sort; torch sorts 64-bit keys, below a
// million of them by merging), then one pass that writes the sorted edges' other
// ends and finds every row's start by a lower bound over the sorted ids.  No
// count of the ids.
//
// The input is checked ahead of the sort, so that the host, which has to know
// the answer before it hands the CSR out, waits for one short kernel while the
// sort is already queued behind it, and not for the sort.
//
// What bounds it: the sort's passes (8 bits each).  us, torch composition (with its
// host syncs) -> here: 40k nodes, 400k edges CSR 204 -> 60, transpose 322 -> 64 (without
// the check 53 and 59); without it 1M nodes, 16M edges 2514 -> 812 and 2766 -> 873; 114M
// edges 17.0 -> 5.3 and 17.7 -> 5.6 ms.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include "as_device.h"
#include "as_internal.h"

namespace as {

namespace {

// An id as a sort key; ids outside [0, n) become n and sort behind every row.
struct IdKey {
  int64_t n;
  __host__ __device__ uint32_t operator()(int64_t id) const {
    return static_cast<uint32_t>(id >= 0 && id < n ? id : n);
  }
};

using KeyIterator = rocprim::transform_iterator<const int64_t*, IdKey, uint32_t>;
// Radix passes from 64k edges on (rocPRIM merges up to a million by default: 400k
// edges 133 against 79 us).  A pass waits on its blocks' chain of prefix sums, which
// wide blocks of few edges shorten where there are few: 1,024 threads of 4 edges
// against the default's 400k edges 79 -> 50 us, 1M 133 -> 102, but 16M 805 -> 866.
constexpr int64_t kShortSort = 4000000;
using ShortSort = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<256, 12>, rocprim::kernel_config<1024, 4>, 8,
                                        rocprim::block_radix_rank_algorithm::match>,
    65536>;
using LongSort =
    rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config, rocprim::default_config, 65536>;

int id_bits(int64_t n) {
  int bits = 1;
  while ((n >> bits) != 0) ++bits;
  return bits;
}

template <typename Config>
hipError_t sort_ids_with(void* temp, size_t& bytes, const int64_t* ids, int64_t n, int64_t edges, uint32_t* keys,
                    uint32_t* order, hipStream_t s) {
  return rocprim::radix_sort_pairs<Config>(temp, bytes, KeyIterator(ids, IdKey{n}), keys,
                                               rocprim::counting_iterator<uint32_t>(0), order,
                                               static_cast<unsigned>(edges), 0u, static_cast<unsigned>(id_bits(n)), s);
}

hipError_t sort_ids(void* temp, size_t& bytes, const int64_t* ids, int64_t n, int64_t edges, uint32_t* keys,
                    uint32_t* order, hipStream_t s) {
  return edges < kShortSort ? sort_ids_with<ShortSort>(temp, bytes, ids, n, edges, keys, order, s)
                            : sort_ids_with<LongSort>(temp, bytes, ids, n, edges, keys, order, s);
}

size_t sort_temp_bytes(int64_t n, int64_t edges) {
  size_t bytes = 0;
  (void)sort_ids(nullptr, bytes, nullptr, n, edges, nullptr, nullptr, nullptr);
  return bytes;
}

size_t ids_bytes(int64_t edges) { return align_up(static_cast<size_t>(edges > 0 ? edges : 1) * sizeof(uint32_t), 256); }

// keys, order, the edges' rows (transpose only), the sort's own
size_t build_bytes(int64_t n, int64_t edges) { return 3 * ids_bytes(edges) + align_up(sort_temp_bytes(n, edges), 256); }

// Sets *bad, host memory: one store by the first lane of a wave that found
// something wrong, written back at once.
__device__ __forceinline__ void report_bad(bool wrong, int32_t* bad) {
  if (__ballot(wrong) != 0 && lane_id() == 0) {
    *static_cast<volatile int32_t*>(bad) = 1;
    __threadfence_system();
  }
}

// Does an id lie outside [0, n)?
__global__ __launch_bounds__(kBlock) void check_ids_kernel(const int64_t* __restrict__ ids, int64_t n, int64_t edges,
                                                           int32_t* bad) {
  const int64_t step = static_cast<int64_t>(gridDim.x) * kBlock;
  bool wrong = false;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < edges; i += step)
    wrong |= ids[i] < 0 || ids[i] >= n;
  report_bad(wrong, bad);
}

// When the check's answer is in *bad (pinned host memory; null: no check):
// after wait(), which every way out of the call passes.
class CheckDone {
 public:
  CheckDone() = default;
  CheckDone(const CheckDone&) = delete;
  CheckDone& operator=(const CheckDone&) = delete;
  ~CheckDone() {
    wait();
    if (event_ != nullptr) (void)hipEventDestroy(event_);
  }
  // Behind the launch of the check.
  bool record(hipStream_t s) {
    recorded_ = hipEventCreateWithFlags(&event_, hipEventDisableTiming) == hipSuccess &&
                hipEventRecord(event_, s) == hipSuccess;
    if (!recorded_) (void)hipStreamSynchronize(s);
    return recorded_;
  }
  bool wait() {
    if (!recorded_) return true;
    recorded_ = false;
    return hipEventSynchronize(event_) == hipSuccess;
  }

 private:
  hipEvent_t event_ = nullptr;
  bool recorded_ = false;
};

// rows[e] = the row of edge e: a wave per kExpand edges.  With bad, also: does
// a column lie outside [0, n), do the row pointers descend or hold fewer than
// `edges` edges?  (The rows are checked by all threads in turn.)
constexpr int64_t kExpand = 4 * kWave;
__global__ __launch_bounds__(kBlock) void edge_rows_kernel(const int64_t* __restrict__ crow,
                                                           const int64_t* __restrict__ col, int64_t n, int64_t edges,
                                                           int32_t* __restrict__ rows, int32_t* bad) {
  const int64_t w = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + wave_in_block();
  if (bad != nullptr) {
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    bool wrong = first == 0 && crow[n] - crow[0] < edges;
    for (int64_t r = first; r < n; r += static_cast<int64_t>(gridDim.x) * kBlock) wrong |= crow[r + 1] < crow[r];
    for (int64_t e = w * kExpand + lane_id(); e < edges && e < (w + 1) * kExpand; e += kWave)
      wrong |= col[e] < 0 || col[e] >= n;
    report_bad(wrong, bad);
  }
  const int64_t b0 = uniform_i64(w * kExpand);
  if (b0 >= edges) return;
  const int64_t b1 = uniform_i64(b0 + kExpand < edges ? b0 + kExpand : edges);
  int64_t r = uniform_i64(wave_row_of_edge(crow, n, b0));
  for (int64_t b = b0; b < b1; b += kWave) {
    const int cnt = b1 - b < kWave ? static_cast<int>(b1 - b) : kWave;
    const int row = block_edge_rows(crow, n, b, cnt, r);
    r = __builtin_amdgcn_readlane(row, cnt - 1);
    if (lane_id() < cnt) rows[b + lane_id()] = row;
  }
}

// Workgroups [0, edge_blocks): sorted edge i's number and other end; the rest:
// crow[r] = ids below r.
template <typename T>
__global__ __launch_bounds__(kBlock) void sorted_edges_kernel(const uint32_t* __restrict__ keys,
                                                              const uint32_t* __restrict__ order,
                                                              const T* __restrict__ other, int64_t n, int64_t edges,
                                                              int64_t edge_blocks, int64_t* __restrict__ crow,
                                                              int64_t* __restrict__ col, int64_t* __restrict__ perm) {
  if (blockIdx.x < edge_blocks) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= edges) return;
    const uint32_t e = order[i];
    col[i] = static_cast<int64_t>(other[e]);
    if (perm != nullptr) perm[i] = static_cast<int64_t>(e);
    return;
  }
  const int64_t r = (static_cast<int64_t>(blockIdx.x) - edge_blocks) * kBlock + threadIdx.x;
  if (r > n) return;
  int64_t lo = 0, hi = edges;
  while (lo < hi) {
    const int64_t mid = lo + (hi - lo) / 2;
    if (static_cast<int64_t>(keys[mid]) < r) lo = mid + 1;
    else hi = mid;
  }
  crow[r] = lo;
}

template <typename T>
int launch_sorted_edges(const uint32_t* keys, const uint32_t* order, const T* other, int64_t n, int64_t edges,
                        int64_t* crow, int64_t* col, int64_t* perm, hipStream_t s) {
  const int64_t edge_blocks = (edges + kBlock - 1) / kBlock;
  const int64_t blocks = edge_blocks + (n + 1 + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(sorted_edges_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s, keys, order,
                     other, n, edges, edge_blocks, crow, col, perm);
  return check_launch("csr_build");
}

// One thread per edge and per row in one launch, 32-bit ids.
bool sizes_fit(int64_t n, int64_t edges) {
  return n > 0 && edges > 0 && n < INT32_MAX && edges < INT32_MAX && n + edges < INT32_MAX - 4096;
}

int validate_build(const void* ids, const void* other, int64_t n, int64_t edges, const void* crow, const void* col,
                   const void* workspace, size_t workspace_bytes) {
  if (!sizes_fit(n, edges))
    return fail(AS_ERR_INVALID_ARGUMENT, "the CSR build takes 1 or more rows and edges, together fewer than 2^31 - 4096");
  if (ids == nullptr || other == nullptr || crow == nullptr || col == nullptr)
    return fail(AS_ERR_INVALID_ARGUMENT, "null pointer argument");
  if (workspace == nullptr || workspace_bytes < build_bytes(n, edges))
    return fail(AS_ERR_WORKSPACE, "the CSR build needs %zu workspace bytes, got %zu", build_bytes(n, edges),
                workspace_bytes);
  return AS_OK;
}

}  // namespace

}  // namespace as

extern "C" {

size_t as_csr_build_workspace_bytes(int64_t n, int64_t edges) {
  if (!as::sizes_fit(n, edges)) return 0;
  return as::build_bytes(n, edges);
}

int as_csr_from_edges(const int64_t* rows, const int64_t* cols, int64_t n, int64_t edges, int64_t* crow, int64_t* col,
                      int64_t* perm, int32_t* bad, void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  int st = as::validate_build(rows, cols, n, edges, crow, col, workspace, workspace_bytes);
  if (st != AS_OK) return st;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  as::CheckDone check;
  if (bad != nullptr) {
    *bad = 0;
    const int64_t blocks = (edges + 4 * as::kBlock - 1) / (4 * as::kBlock);
    hipLaunchKernelGGL(as::check_ids_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)),
                       dim3(as::kBlock), 0, s, rows, n, edges, bad);
    if (!check.record(s)) return as::fail(AS_ERR_LAUNCH, "checking the edges failed");
  }
  char* ws = static_cast<char*>(workspace);
  uint32_t* keys = reinterpret_cast<uint32_t*>(ws);
  uint32_t* order = reinterpret_cast<uint32_t*>(ws + as::ids_bytes(edges));
  size_t temp = workspace_bytes - 3 * as::ids_bytes(edges);
  if (as::sort_ids(ws + 3 * as::ids_bytes(edges), temp, rows, n, edges, keys, order, s) != hipSuccess)
    return as::fail(AS_ERR_LAUNCH, "sorting the edges failed");
  st = as::launch_sorted_edges<int64_t>(keys, order, cols, n, edges, crow, col, perm, s);
  if (!check.wait()) return as::fail(AS_ERR_LAUNCH, "checking the edges failed");
  return st;
}

int as_csr_transpose(const int64_t* crow, const int64_t* col, int64_t n, int64_t nnz, int64_t* crow_t, int64_t* col_t,
                     int64_t* perm, int32_t* bad, void* workspace, size_t workspace_bytes, void* stream) {
  as::clear_error();
  int st = as::validate_build(crow, col, n, nnz, crow_t, col_t, workspace, workspace_bytes);
  if (st != AS_OK) return st;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  as::CheckDone check;
  char* ws = static_cast<char*>(workspace);
  uint32_t* keys = reinterpret_cast<uint32_t*>(ws);
  uint32_t* order = reinterpret_cast<uint32_t*>(ws + as::ids_bytes(nnz));
  int32_t* rows = reinterpret_cast<int32_t*>(ws + 2 * as::ids_bytes(nnz));
  if (bad != nullptr) *bad = 0;
  const int64_t waves = (nnz + as::kExpand - 1) / as::kExpand;
  hipLaunchKernelGGL(as::edge_rows_kernel,
                     dim3(static_cast<unsigned>((waves + as::kWavesPerBlock - 1) / as::kWavesPerBlock)),
                     dim3(as::kBlock), 0, s, crow, col, n, nnz, rows, bad);
  if (bad != nullptr && !check.record(s)) return as::fail(AS_ERR_LAUNCH, "checking the graph failed");
  size_t temp = workspace_bytes - 3 * as::ids_bytes(nnz);
  if (as::sort_ids(ws + 3 * as::ids_bytes(nnz), temp, col, n, nnz, keys, order, s) != hipSuccess)
    return as::fail(AS_ERR_LAUNCH, "sorting the edges failed");
  st = as::launch_sorted_edges<int32_t>(keys, order, rows, n, nnz, crow_t, col_t, perm, s);
  if (!check.wait()) return as::fail(AS_ERR_LAUNCH, "checking the graph failed");
  return st;
}

}  // extern "C"
