// Temporal CSR build on the device (the GPU counterpart of the reference's
// get_neighbors, vendor/bts_sampler/sampler/include/neighbors.h:209-284).
//
// The reference appends every event to vector<>s of its dst node in event
// order. Here the same lists are laid out contiguously in HBM:
//   1. key[i] = col[i] (range-checked), val[i] = i, record[i] = (ts, row, eid)
//   2. stable LSD radix sort of (key, val) over ceil(log2(N+1)) bits -- a
//      stable sort keyed by dst keeps event order inside each node's list
//      (val as a counting iterator: the sort writes it out itself, 9 us more
//      for 7 saved in step 1)
//   3. gather the records through the sorted event index (int32 / int64 SoA):
//      the event order inside a list is random to the memory system, so an
//      event costs one 128-byte line as a record and one per array otherwise
//      (7.8 M events, 1.1 M nodes: 293 -> 162 us; writing the records adds 20)
//   4. indptr from the boundaries of the sorted keys (no atomics), by the
//      gather's threads: its lines bound that kernel, and the keys' few more
//      bytes mostly hide behind them (163.3 + 23.8 us apart, 168.6 together)
#include <rocprim/device/device_radix_sort.hpp>

#include <climits>

#include "common.h"

namespace {

constexpr int kBlock = 256;

unsigned key_bits(int64_t num_nodes) {
  unsigned b = 1;
  while (b < 32 && (int64_t(1) << b) <= num_nodes) ++b;  // keys lie in [0, N]
  return b;
}

size_t sort_temp_bytes(int64_t num_edges, unsigned bits) {
  size_t temp = 0;
  if (num_edges <= 0) return 0;
  hipError_t e = rocprim::radix_sort_pairs(
      nullptr, temp, static_cast<uint32_t *>(nullptr),
      static_cast<uint32_t *>(nullptr), static_cast<int32_t *>(nullptr),
      static_cast<int32_t *>(nullptr), static_cast<size_t>(num_edges), 0u,
      bits, hipStream_t(0));
  return e == hipSuccess ? temp : 0;
}

// One event as the gather reads it.
struct __attribute__((aligned(16))) EventRecord {
  int64_t ts;
  int32_t row, eid;
};

__global__ __launch_bounds__(kBlock) void k_tcsr_keys(
    int64_t num_edges, int64_t num_nodes, const int64_t *__restrict__ row,
    const int64_t *__restrict__ col, const int64_t *__restrict__ eid,
    const int64_t *__restrict__ ts, uint32_t *__restrict__ keys, int32_t *__restrict__ vals,
    EventRecord *__restrict__ rec, int32_t *__restrict__ err) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= num_edges) return;
  const int64_t d = col[i];
  const int64_t s = row[i];
  int bad = 0;
  int64_t id = i;
  if (d < 0 || d >= num_nodes || s < 0 || s >= num_nodes) bad |= SGL_DERR_NODE_RANGE;
  if (eid != nullptr) {
    id = eid[i];
    if (id < 0 || id > INT_MAX) bad |= SGL_DERR_EID_RANGE;
  }
  if (bad && err != nullptr) atomicOr(err, bad);
  // Invalid dst ids sort past every valid node and never reach indptr.
  keys[i] = (d >= 0 && d < num_nodes) ? uint32_t(d) : uint32_t(num_nodes);
  vals[i] = int32_t(i);
  rec[i] = EventRecord{ts[i], int32_t(s), int32_t(id)};
}

// Thread j in [0, E] writes indptr[n] = j for every node n in (key[j-1],
// key[j]]; a run of more than kLongGap nodes without events by the whole wave
// (5 M nodes, 1,000 events: 1,392 us a thread each, 199 so).
constexpr int64_t kLongGap = 32;
__device__ __forceinline__ void write_indptr(int64_t j, int64_t num_edges, int64_t num_nodes,
                                             const uint32_t *__restrict__ skeys, int64_t *__restrict__ indptr) {
  int64_t first = 0, last = -1;  // (no nodes past thread E)
  if (j <= num_edges) {
    first = j == 0 ? 0 : int64_t(skeys[j - 1]) + 1;
    last = j == num_edges ? num_nodes : min(int64_t(skeys[j]), num_nodes);
  }
  const bool wide = last - first >= kLongGap;
  const int lane = threadIdx.x & (sgl::kWave - 1);
  for (uint64_t m = __ballot(wide); m != 0; m &= m - 1) {
    const int l = __ffsll(static_cast<unsigned long long>(m)) - 1;
    const long long f = __shfl(static_cast<long long>(first), l, sgl::kWave);
    const long long e = __shfl(static_cast<long long>(last), l, sgl::kWave);
    const int64_t at = j - lane + l;
    for (int64_t n = f + lane; n <= e; n += sgl::kWave) indptr[n] = at;
  }
  if (!wide)
    for (int64_t n = first; n <= last; ++n) indptr[n] = j;
}

__global__ __launch_bounds__(kBlock) void k_tcsr_gather(
    int64_t num_edges, int64_t num_nodes, const int32_t *__restrict__ order, const uint32_t *__restrict__ skeys,
    const EventRecord *__restrict__ rec, int32_t *__restrict__ nbr, int32_t *__restrict__ eid_out,
    int64_t *__restrict__ ts_out, int64_t *__restrict__ indptr) {
  const int64_t j = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (j < num_edges) {
    const EventRecord r = rec[order[j]];  // order: a permutation of [0, num_edges)
    nbr[j] = r.row;
    eid_out[j] = r.eid;
    ts_out[j] = r.ts;
  }
  write_indptr(j, num_edges, num_nodes, skeys, indptr);  // (every lane: a wave writes long runs together)
}

__global__ __launch_bounds__(kBlock) void k_tcsr_indptr(int64_t num_nodes, int64_t *__restrict__ indptr) {  // no edges
  const int64_t n = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (n <= num_nodes) indptr[n] = 0;
}

// The sampler's packed copy of a CSR: int32 times, (nbr, eid) pairs and every
// 32nd time, plus what decides whether a caller may use them. flags[0] counts
// the places where a time is smaller than the one before it, less those at a
// list's first entry (0: every list is sorted); flags[1] is set when a time
// does not fit in int32. One pass over the edges and one over the list starts;
// bound by the bytes (28 per edge). Tensor operations for the same (two
// reductions, a stack, and a sort-based lookup of the decreasing places among
// the list starts) took about 900 us at 7.8 M edges and 1.1 M nodes, this 61
// (219 MB: 3.6 TB/s). A thread that meets a time outside int32 stops: a graph
// of such times is told in 61 us at 20 M edges (103 by two reductions, 192
// with its copy written).
constexpr int64_t kFenceSpan = 32;
__global__ __launch_bounds__(kBlock) void k_recent_pack(
    int64_t num_edges, int64_t num_nodes, const int64_t *__restrict__ indptr, const int32_t *__restrict__ nbr,
    const int32_t *__restrict__ eid, const int64_t *__restrict__ ts, int2 *__restrict__ nbr_eid,
    int32_t *__restrict__ ts32, int32_t *__restrict__ fence, int64_t *__restrict__ flags) {
  const int64_t step = int64_t(gridDim.x) * kBlock, first = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  int64_t down = 0;
  bool wide = false;
  for (int64_t i = first; i < num_edges; i += step) {
    const int64_t t = ts[i];
    const int64_t before = i > 0 ? ts[i - 1] : t;  // (the neighbouring lane's line)
    const int2 ids = make_int2(nbr[i], eid[i]);
    wide = t != int64_t(int32_t(t));
    if (wide) break;  // nothing of the copy is used
    nbr_eid[i] = ids;
    ts32[i] = int32_t(t);
    if (i % kFenceSpan == 0) fence[i / kFenceSpan] = int32_t(t);
    down += t < before;
  }
  // list starts (the entries past the last list, if any, form one more)
  for (int64_t n = first; n <= num_nodes && !wide; n += step) {
    const int64_t s = indptr[n], e = n < num_nodes ? indptr[n + 1] : num_edges;
    if (s > 0 && s < e) down -= ts[s] < ts[s - 1];
  }
  __shared__ int64_t s_down[kBlock / sgl::kWave];
  const int wave = threadIdx.x / sgl::kWave;
  const int64_t d = sgl::wave_reduce_sum(down);
  if (threadIdx.x % sgl::kWave == 0) s_down[wave] = d;
  const int any = __syncthreads_or(wide);
  if (threadIdx.x == 0) {
    int64_t tot = 0;
#pragma unroll
    for (int w = 0; w < kBlock / sgl::kWave; ++w) tot += s_down[w];
    if (tot != 0) atomicAdd(reinterpret_cast<unsigned long long *>(flags), static_cast<unsigned long long>(tot));
    if (any) atomicOr(reinterpret_cast<unsigned long long *>(flags + 1), 1ull);
  }
}

}  // namespace

extern "C" int sgl_recent_pack(int64_t num_nodes, int64_t num_edges, const int64_t *indptr, const int32_t *nbr,
                               const int32_t *eid, const int64_t *ts, int32_t *nbr_eid, int32_t *ts32,
                               int32_t *fence, int64_t *flags, hipStream_t stream) {
  SGL_REQUIRE(num_nodes >= 0 && num_nodes < INT_MAX, "recent_pack: num_nodes %lld out of range [0, 2^31-1)", (long long)num_nodes);
  SGL_REQUIRE(num_edges >= 0 && num_edges < INT_MAX, "recent_pack: num_edges %lld out of range [0, 2^31-1)", (long long)num_edges);
  SGL_REQUIRE(indptr && flags, "recent_pack: NULL indptr or flags");
  if (num_edges == 0) return SGL_OK;
  SGL_REQUIRE(nbr && eid && ts && nbr_eid && ts32 && fence, "recent_pack: NULL array");
  SGL_REQUIRE((reinterpret_cast<uintptr_t>(nbr_eid) & 7u) == 0, "recent_pack: nbr_eid not 8-byte aligned");
  const int64_t most = std::max(num_edges, num_nodes + 1);
  const unsigned grid = unsigned(std::min<int64_t>((most + kBlock - 1) / kBlock, sgl::kMaxGrid));
  k_recent_pack<<<grid, kBlock, 0, stream>>>(num_edges, num_nodes, indptr, nbr, eid, ts,
                                             reinterpret_cast<int2 *>(nbr_eid), ts32, fence, flags);
  SGL_CHECK_LAUNCH();
  return SGL_OK;
}

extern "C" size_t sgl_tcsr_workspace_bytes(int64_t num_nodes, int64_t num_edges) {
  if (num_nodes < 0 || num_edges < 0) return 0;
  const size_t e = size_t(num_edges);
  return 4 * sgl::align_up(e * 4) + sgl::align_up(e * sizeof(EventRecord)) +
         sgl::align_up(sort_temp_bytes(num_edges, key_bits(num_nodes))) + 256;
}

extern "C" int sgl_tcsr_build(int64_t num_nodes, int64_t num_edges,
                              const int64_t *row, const int64_t *col,
                              const int64_t *eid, const int64_t *ts,
                              int64_t *indptr, int32_t *nbr, int32_t *eid_out,
                              int64_t *ts_out, void *workspace,
                              size_t workspace_bytes, int32_t *err_flag,
                              hipStream_t stream) {
  SGL_REQUIRE(num_nodes >= 0 && num_nodes < INT_MAX, "tcsr: num_nodes %lld out of range [0, 2^31-1)", (long long)num_nodes);
  SGL_REQUIRE(num_edges >= 0 && num_edges < INT_MAX, "tcsr: num_edges %lld out of range [0, 2^31-1)", (long long)num_edges);
  SGL_REQUIRE(indptr != nullptr, "tcsr: indptr is NULL");
  SGL_REQUIRE(num_edges == 0 || (row && col && ts && nbr && eid_out && ts_out), "tcsr: NULL input/output array");
  const size_t need = sgl_tcsr_workspace_bytes(num_nodes, num_edges);
  if (workspace_bytes < need || (num_edges > 0 && workspace == nullptr)) {
    sgl::set_error("tcsr: workspace %zu bytes < required %zu", workspace_bytes, need);
    return SGL_ERR_WORKSPACE;
  }
  const unsigned bits = key_bits(num_nodes);
  if (num_edges > 0) {
    const size_t e = size_t(num_edges);
    sgl::Carver c(workspace);
    uint32_t *keys_in = c.take<uint32_t>(e);
    uint32_t *keys_out = c.take<uint32_t>(e);
    int32_t *vals_in = c.take<int32_t>(e);
    int32_t *vals_out = c.take<int32_t>(e);
    EventRecord *rec = c.take<EventRecord>(e);
    size_t temp = sort_temp_bytes(num_edges, bits);
    void *temp_ptr = c.take<char>(temp);
    const unsigned grid = unsigned((e + kBlock - 1) / kBlock);
    k_tcsr_keys<<<grid, kBlock, 0, stream>>>(num_edges, num_nodes, row, col, eid, ts, keys_in, vals_in, rec,
                                             err_flag);
    SGL_CHECK_LAUNCH();
    SGL_CHECK_HIP(rocprim::radix_sort_pairs(temp_ptr, temp, keys_in, keys_out, vals_in, vals_out, e, 0u, bits, stream));
    const unsigned grid1 = unsigned((e + 1 + kBlock - 1) / kBlock);
    k_tcsr_gather<<<grid1, kBlock, 0, stream>>>(num_edges, num_nodes, vals_out, keys_out, rec, nbr, eid_out, ts_out,
                                                indptr);
    SGL_CHECK_LAUNCH();
  } else {
    k_tcsr_indptr<<<unsigned((num_nodes + 1 + kBlock - 1) / kBlock), kBlock, 0, stream>>>(num_nodes, indptr);
    SGL_CHECK_LAUNCH();
  }
  return SGL_OK;
}
