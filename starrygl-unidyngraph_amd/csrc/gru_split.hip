// The fp32 memory update (GRU over the mailbox, GRUCell, mailbox write) and the
// memory commit for batches that leave most of the GPU idle, as two launches.
//
// Reference: CTDGMemoryUpdater.forward  backends/ctdg/runtime/models.py:244-254,
//            CTDGMemoryBank.write_mailbox / _write_slots  memory.py:183-248,
//            CTDGMemoryBank._apply_memory_update  memory.py:254-269.
//
// k_gru_mailbox (state.hip) gives 16 roots to a workgroup, which streams all
// four weight matrices through one chain of products: at 400 roots 25 CUs work
// and 231 wait, and the chain's length (a 372-deep product of 300 columns,
// then two 100-deep ones, on 16 waves) sets the time. Most of that work does
// not depend on the hidden state: W_ih x_k of every slot and the cell's
// W_hh m. k_gru_inputs computes those for every (16 roots, slot, 64 columns)
// in parallel into a workspace, and stages the mailbox messages, which hold
// memory rows as they are before the update. k_gru_cells then needs only the
// recurrent products (none in the first slot, where h = 0) and the cell's
// W_ih h; nothing in it reads another root's memory or mailbox row, so it also
// writes the memory table (the commit's launch is saved) and, by its other
// workgroups, the staged messages. Per value the same products in the same
// order as k_gru_mailbox: the same bits.
//   D = 100, S = 372, K = 1: 31.4 (+ 4.7 the commit) -> 9.6 + 11.6 us at 320
//   roots; rows without messages (the updater module, 333): 30.1 ->
//   8.1 + 11.0 us, and 85 -> 21 us with the host's part (8 fills fewer).
#include <algorithm>
#include <climits>

#include "common.h"
#include "gru.h"
#include "mfma.h"

namespace {

constexpr int kRows = 16;       // roots per tile
constexpr int kInBlock = 256;   // k_gru_inputs: a 16-column block a wave
constexpr int kInWaves = kInBlock / sgl::kWave;
constexpr int kMsgParts = 2;    // workgroups of a tile's messages
constexpr int kMaxWidth = 512;  // S = 2D + F (so D <= 256: at most 16 column chunks)

// Narrow hidden rows need few waves for their products; the messages (a root a
// wave, a chain of loads each) then set the time. With messages at least this
// many workgroups of a tile stage them and this many waves a workgroup write
// them (split / one launch and the commit, us, 1,000 events: D 4, F 1, K 1
// 21.5 -> 11.3 / 12.8; D 16, F 16, K 4 23.3 -> 17.3 / 20.0; D 32, F 172, K 1
// 18.1 -> 15.7 / 18.6; from D 64 on the products have as many).
constexpr unsigned kMsgGroups = 4, kMsgWaves = 4;
constexpr unsigned kXcds = 8;

// Above these capacities the one-launch kernel has a tile for most CUs and the
// workspace's traffic is no longer free (split / one launch, us: D 100, S 372,
// K 1: 2,048 rows 29 / 34, 4,096 35 / 32; D 172, S 360, K 4: 116 / 137 and 176 /
// 139; D 64, S 144, K 2: 18 / 22 and 24 / 23). Rows that are not whole 16 bytes
// load word by word, which wide products pay for earlier (D 172, S 345, K 1:
// 1,024 rows 43 / 53, 1,280 53 / 53, 2,048 61 / 54), as do a partial column
// block and more than 12 waves (D 200, S 400, K 2: 1,024 rows 86 / 93, 2,048
// 103 / 95; D 192 94 / 112, D 240 133 / 155).
int64_t split_max_rows(int D, int F) {
  const bool words = D % 4 != 0 || F % 4 != 0;
  return (D > 128 && words) || (D > 192 && D % 16 != 0) ? 1024 : 2048;
}

struct Events {  // one batch's messages (all NULL: none are written)
  const int64_t *src, *dst;
  const float *efeat, *ts;
  const int64_t *batch_start;
  const unsigned long long *win_src, *win_dst;
  const int32_t *cnt_src, *cnt_dst;
};

// The commit's arrays (memory.py:254-269; memory_ts NULL: no commit).
struct Commit {
  float *memory_ts;
  const float *ts_max;
  uint32_t *bits;
  const int32_t *sample_cnt;
  int32_t *any_edges;
  float *root_dt;
};

// A root's messages (memory.py:218-248): the src-role message of node u is
// [mem(u) | mem(other) | f_e] of its last src event e and goes to slot p =
// next_mail_pos[u], the dst-role one, of its last dst event, to (p + #src
// events) % K, so with one slot the dst role wins; the pointer advances by
// both counts.
struct Message {
  int64_t u, e[2];
  int p, slot[2], next;
  bool on[2];
  __device__ __forceinline__ Message(const Events &ev, const int64_t *roots, const int32_t *next_mail_pos, int r, int K) {
    const int64_t off = ev.batch_start != nullptr ? *ev.batch_start : 0;
    u = roots[r];
    const int cs = ev.cnt_src[r], cd = ev.cnt_dst[r];
    e[0] = off + int64_t(ev.win_src[r] & 0xffffffffull);
    e[1] = off + int64_t(ev.win_dst[r] & 0xffffffffull);
    p = next_mail_pos[u];
    slot[0] = p;
    slot[1] = (p + cs) % K;
    on[0] = cs > 0 && !(cd > 0 && slot[1] == p);
    on[1] = cd > 0;
    next = int((int64_t(p) + cs + cd) % K);
  }
};

// ws: ceil(rows / 16) * 16 rows of (K + 1) * 3D gate inputs, then as many rows
// of two staged messages of S. Gate inputs [slot][3D]: W_ih x + b_ih of root
// r's mailbox row `slot`, or (slot K) the cell's W_hh m + b_hh. Grid: (tiles,
// K + 1 and with messages one more, groups of kInWaves column blocks; of the
// messages' workgroups each wave takes a root).
__global__ __launch_bounds__(kInBlock) void k_gru_inputs(
    int D, int K, int F, const int32_t *__restrict__ num_roots, int rows, const int64_t *__restrict__ roots,
    const float *__restrict__ memory, const float *__restrict__ mailbox, const float *__restrict__ w_ih,
    const float *__restrict__ b_ih, const float *__restrict__ wc_hh, const float *__restrict__ bc_hh, Events ev,
    const int32_t *__restrict__ next_mail_pos, float *__restrict__ ws, float *__restrict__ staged) {
  extern __shared__ __align__(16) float xs[];
  const int U = num_roots != nullptr ? *num_roots : rows;
  const int r0 = blockIdx.x * kRows, slot = blockIdx.y;
  if (r0 >= U) return;
  const int nrows = min(kRows, U - r0);
  const int S = 2 * D + F, G = 3 * D;
  const bool mem = slot == K;
  const int kd = mem ? D : S, ld = sgl::lds_ld(kd);
  const float *table = mem ? memory : mailbox;
  const int tid = threadIdx.x, wave = tid / sgl::kWave, lane = tid % sgl::kWave;
  if (slot > K) {
    // (an event index of a role without events is 0: its reads are in bounds)
    for (int i = blockIdx.z * kInWaves + wave; i < nrows; i += gridDim.z * kInWaves) {
      const Message msg(ev, roots, next_mail_pos, r0 + i, K);
      const int64_t other[2] = {ev.dst[msg.e[0]], ev.src[msg.e[1]]};
      constexpr int kSlots = kMaxWidth / sgl::kWave;
      float part[2][kSlots];
#pragma unroll
      for (int role = 0; role < 2; ++role)
#pragma unroll
        for (int jj = 0; jj < kSlots; ++jj) {
          const int c = lane + sgl::kWave * jj;
          const float *src = c < D ? memory + msg.u * D + c : c < 2 * D ? memory + other[role] * D + (c - D)
                                                                       : ev.efeat + msg.e[role] * F + (c - 2 * D);
          part[role][jj] = msg.on[role] && c < S ? *src : 0.f;
        }
#pragma unroll
      for (int role = 0; role < 2; ++role)
#pragma unroll
        for (int jj = 0; jj < kSlots; ++jj)
          if (msg.on[role] && lane + sgl::kWave * jj < S)
            staged[(size_t(r0 + i) * 2 + role) * S + lane + sgl::kWave * jj] = part[role][jj];
    }
    return;
  }
  if (16 * int(blockIdx.z) * kInWaves >= G) return;  // launched for the messages only
  // the tile's rows (a row's id is read by its own lanes: one barrier fewer)
  auto row_of = [&](int i) {
    const int64_t root = roots != nullptr ? roots[r0 + i] : int64_t(r0 + i);
    return mem ? root * D : (root * K + slot) * S;
  };
  if ((kd & 3) == 0 && sgl::aligned16(table)) {
    const int n4 = kd >> 2;
    for (int idx = tid; idx < kRows * n4; idx += kInBlock) {
      const int i = idx / n4, j = idx - i * n4;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (i < nrows) v = reinterpret_cast<const float4 *>(table + row_of(i))[j];
      *reinterpret_cast<float4 *>(xs + i * ld + 4 * j) = v;
    }
  } else {
    for (int idx = tid; idx < kRows * kd; idx += kInBlock) {
      const int i = idx / kd, j = idx - i * kd;
      xs[i * ld + j] = i < nrows ? table[row_of(i) + j] : 0.f;
    }
  }
  __syncthreads();
  const int n0 = 16 * (blockIdx.z * kInWaves + wave);
  if (n0 >= G) return;
  const int col = n0 + (lane & 15);
  const float *bias = mem ? bc_hh : b_ih;
  const float bv = col < G ? bias[col] : 0.f;
  const sgl::f32x4 acc = sgl::mfma_block16<sgl::kNT>(xs, ld, mem ? wc_hh : w_ih, kd, n0, kd, G);
  if (col < G) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 4 * (lane >> 4) + v;
      if (i < nrows) ws[(size_t(r0 + i) * (K + 1) + slot) * G + col] = acc[v] + bv;
    }
  }
}

// The three gates' products of one 16-column chunk: acc[t] = A[16][0..D) .
// W[t*D + n0 + j][0..D). b0 holds the first 64 k of the weights on entry (the
// caller loads them before it waits for what A is made of); per gate the order
// of the sums is mfma_block16's. (A second register set, to load the next 64 k
// before a chunk's products, spills: 11.3 -> 16.8 us.)
using Chunk3 = float[3][sgl::kChunkGroups][4];
struct GateWeights {
  __amdgpu_buffer_rsrc_t rsrc;
  int D, n, q;
  bool vec;
  __device__ GateWeights(const float *W, int D_, int n0, int lane)
      : rsrc(sgl::weight_rsrc(W, uint32_t(3 * D_) * uint32_t(D_))), D(D_), n(n0 + (lane & 15)), q(lane >> 4),
        vec((D_ & 3) == 0 && sgl::aligned16(W)) {}
  __device__ __forceinline__ void load(Chunk3 &b, int kb) const {
#pragma unroll
    for (int t = 0; t < 3; ++t) sgl::load_w_chunk<sgl::kNT>(b[t], rsrc, D, t * D + n, kb, q, vec);
  }
};
__device__ __forceinline__ void gates3(const float *hs, int ldh, const GateWeights &W, Chunk3 &b0, sgl::f32x4 (&acc)[3]) {
  const float *arow = hs + (threadIdx.x & 15) * ldh;
  constexpr int kc = 16 * sgl::kChunkGroups;
  sgl::f32x4 p[3], r[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) p[t] = r[t] = sgl::f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < W.D; kb += kc) {
    if (kb > 0) W.load(b0, kb);
#pragma unroll
    for (int t = 0; t < 3; ++t) sgl::mfma_chunk_any(p[t], r[t], b0[t], arow, kb, W.D, W.q, true);
  }
#pragma unroll
  for (int t = 0; t < 3; ++t) acc[t] = p[t] + r[t];
}

// Grid: (tiles, 1 + message parts), one wave per 16 hidden columns and with
// messages at least kMsgWaves (TH: their most threads; fewer leave a lane more
// registers). A lane's loads
// take clamped rows and columns instead of branches, so that all of them are
// in flight together.
template <int TH>
__global__ __launch_bounds__(TH) void k_gru_cells(
    int D, int K, int F, const int32_t *__restrict__ num_roots, int rows, const int64_t *__restrict__ roots,
    float *__restrict__ memory, float *__restrict__ mailbox, float *__restrict__ mailbox_ts,
    int32_t *__restrict__ next_mail_pos, const float *__restrict__ w_hh, const float *__restrict__ b_hh,
    const float *__restrict__ wc_ih, const float *__restrict__ bc_ih, Events ev, Commit cm,
    const float *__restrict__ ws, const float *__restrict__ staged, float *__restrict__ new_mem) {
  extern __shared__ __align__(16) float hs[];  // [16][lds_ld(D)]
  const int U = num_roots != nullptr ? *num_roots : rows;
  const int r0 = blockIdx.x * kRows;
  if (r0 >= U) return;
  const int nrows = min(kRows, U - r0);
  const int tid = threadIdx.x, wave = tid / sgl::kWave, lane = tid % sgl::kWave, nwaves = blockDim.x / sgl::kWave;
  const int S = 2 * D + F, G = 3 * D;

  if (blockIdx.y > 0) {
    // the staged messages, a root a wave (every mailbox row has been read by
    // the first launch)
    constexpr int per = kRows / kMsgParts;
    const int part = int(blockIdx.y) - 1;
    if (cm.memory_ts != nullptr && part == 0 && tid < nrows) {  // the commit's per-root words
      const int64_t u = roots[r0 + tid];
      const float tmax = *cm.ts_max;
      if (cm.root_dt != nullptr) cm.root_dt[r0 + tid] = tmax - cm.memory_ts[u];  // time since the root's last update
      cm.memory_ts[u] = tmax;
      cm.bits[u >> 5] = 0u;  // leave the bitmap clear for the next step
      if (cm.sample_cnt != nullptr && cm.sample_cnt[r0 + tid] > 0) *cm.any_edges = 1;
    }
    for (int i = part * per + wave; i < min(nrows, (part + 1) * per); i += nwaves) {
      const Message msg(ev, roots, next_mail_pos, r0 + i, K);
      constexpr int kSlots = kMaxWidth / sgl::kWave;
      float v[2][kSlots];
#pragma unroll
      for (int role = 0; role < 2; ++role)
#pragma unroll
        for (int jj = 0; jj < kSlots; ++jj) {
          const int c = lane + sgl::kWave * jj;
          v[role][jj] = msg.on[role] && c < S ? staged[(size_t(r0 + i) * 2 + role) * S + c] : 0.f;
        }
#pragma unroll
      for (int role = 0; role < 2; ++role) {
        if (!msg.on[role]) continue;  // uniform in the wave
        float *out = mailbox + (msg.u * K + msg.slot[role]) * S;
#pragma unroll
        for (int jj = 0; jj < kSlots; ++jj)
          if (lane + sgl::kWave * jj < S) out[lane + sgl::kWave * jj] = v[role][jj];
        if (lane == 0) mailbox_ts[msg.u * K + msg.slot[role]] = ev.ts[msg.e[role]];
      }
      if (lane == 0) next_mail_pos[msg.u] = msg.next;
    }
    return;
  }

  // this lane's column and its four rows of the tile
  const int n0 = 16 * wave, col = n0 + (lane & 15), i0 = 4 * (lane >> 4);
  if (n0 >= D) {  // a wave launched for the messages only: this workgroup's barriers
    for (int k = 1; k < K; ++k) {
      __syncthreads();
      __syncthreads();
    }
    __syncthreads();
    return;
  }
  const bool cok = col < D;
  const int cc = min(col, D - 1);
  const int ldh = sgl::lds_ld(D);
  float m[4], h[4], gi[4][3], gm[4][3];
  size_t row[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) row[v] = size_t(r0 + min(i0 + v, nrows - 1));
  auto load_gates = [&](float (&g)[4][3], int slot) {
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int t = 0; t < 3; ++t) g[v][t] = ws[(row[v] * (K + 1) + slot) * G + t * D + cc];
  };
  const GateWeights wc(wc_ih, D, n0, lane), wh(w_hh, D, n0, lane);
  Chunk3 b0;
  (K > 1 ? wh : wc).load(b0, 0);
  load_gates(gi, 0);
  load_gates(gm, K);
  float bh[3], bc[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    bh[t] = b_hh[t * D + cc];
    bc[t] = bc_ih[t * D + cc];
  }
  int64_t id[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) id[v] = roots != nullptr ? roots[row[v]] : int64_t(row[v]);
#pragma unroll
  for (int v = 0; v < 4; ++v) m[v] = memory[id[v] * D + cc];
  // slot 0: h = 0, so the recurrent product is the bias
#pragma unroll
  for (int v = 0; v < 4; ++v) h[v] = sgl::gru_combine(gi[v][0], gi[v][1], gi[v][2], bh[0], bh[1], bh[2], 0.f);
  auto publish = [&]() {
    if (cok) {
#pragma unroll
      for (int v = 0; v < 4; ++v) hs[(i0 + v) * ldh + col] = h[v];
    }
    __syncthreads();
  };
  sgl::f32x4 a[3];
  for (int k = 1; k < K; ++k) {
    load_gates(gi, k);
    publish();
    gates3(hs, ldh, wh, b0, a);
    if (k + 1 < K) wh.load(b0, 0);
    else wc.load(b0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      h[v] = sgl::gru_combine(gi[v][0], gi[v][1], gi[v][2], a[0][v] + bh[0], a[1][v] + bh[1], a[2][v] + bh[2], h[v]);
    __syncthreads();  // every wave has read hs
  }
  publish();
  gates3(hs, ldh, wc, b0, a);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    if (cok && i0 + v < nrows) {
      const float o = sgl::gru_combine(a[0][v] + bc[0], a[1][v] + bc[1], a[2][v] + bc[2], gm[v][0], gm[v][1], gm[v][2],
                                       m[v]);
      new_mem[row[v] * D + col] = o;
      // (this lane read the element above, nobody else does)
      if (cm.memory_ts != nullptr) memory[id[v] * D + col] = o;
    }
  }
}

size_t padded_rows(int64_t rows) { return size_t((rows + kRows - 1) / kRows * kRows); }
size_t ws_bytes(int D, int K, int F, int64_t rows) {
  return padded_rows(rows) * (size_t(K + 1) * size_t(3 * D) + 2 * size_t(2 * D + F)) * sizeof(float);
}

int launch_split(int D, int K, int F, int64_t capacity, const int32_t *num_roots, int rows, const int64_t *roots,
                 const float *memory, float *mailbox, float *mailbox_ts, int32_t *next_mail_pos, const float *w_ih,
                 const float *w_hh, const float *b_ih, const float *b_hh, const float *wc_ih, const float *wc_hh,
                 const float *bc_ih, const float *bc_hh, const Events &ev, const Commit &cm, float *new_mem, float *ws,
                 hipStream_t stream) {
  // (a multiple of the XCDs, to which workgroups are dealt in turn: a tile's
  // workgroups of both launches share an L2, where the first leaves what the
  // second reads)
  const unsigned tiles = unsigned((capacity + kRows * kXcds - 1) / (kRows * kXcds) * kXcds);
  const bool msgs = ev.win_src != nullptr;
  const unsigned groups = std::max(unsigned(((3 * D + 15) / 16 + kInWaves - 1) / kInWaves), msgs ? kMsgGroups : 1u);
  float *staged = ws + padded_rows(capacity) * size_t(K + 1) * size_t(3 * D);
  // an op timed by the caller: from the first launch's start to the second's end
  const sgl::LaunchTimer timed = sgl::pending_timer();
  sgl::pending_timer() = sgl::LaunchTimer{timed.start, nullptr};
  const size_t lds_in = sizeof(float) * kRows * size_t(sgl::lds_ld(2 * D + F));
  sgl::launch(&k_gru_inputs, dim3(tiles, unsigned(K + 1 + (msgs ? 1 : 0)), groups), dim3(kInBlock), lds_in, stream, D,
              K, F, num_roots, rows, roots, memory, static_cast<const float *>(mailbox), w_ih, b_ih, wc_hh, bc_hh, ev,
              static_cast<const int32_t *>(next_mail_pos), ws, staged);
  SGL_CHECK_LAUNCH();
  sgl::pending_timer() = sgl::LaunchTimer{nullptr, timed.stop};
  const unsigned waves = std::max(unsigned((D + 15) / 16), msgs ? kMsgWaves : 1u);
  const size_t lds_h = sizeof(float) * kRows * size_t(sgl::lds_ld(D));
  const auto cells = waves <= 8 ? &k_gru_cells<512> : waves <= 12 ? &k_gru_cells<768> : &k_gru_cells<1024>;
  sgl::launch(cells, dim3(tiles, msgs ? 1 + kMsgParts : 1), dim3(waves * sgl::kWave), lds_h, stream, D, K, F, num_roots,
              rows, roots, const_cast<float *>(memory), mailbox, mailbox_ts, next_mail_pos, w_hh, b_hh, wc_ih, bc_ih, ev,
              cm,
              static_cast<const float *>(ws), static_cast<const float *>(staged), new_mem);
  SGL_CHECK_LAUNCH();
  return SGL_OK;
}

}  // namespace

extern "C" size_t sgl_memory_update_workspace_bytes(int32_t D, int32_t K, int32_t F, int64_t capacity) {
  if (D <= 0 || K <= 0 || F < 0 || capacity <= 0 || 2 * D + F > kMaxWidth || capacity > split_max_rows(D, F)) return 0;
  if (sgl_memory_update_lds_bytes(D, F) > 160 * 1024) return 0;  // shapes that sgl_memory_update refuses stay refused
  return ws_bytes(D, K, F, capacity);
}

extern "C" int sgl_memory_update_commit(int32_t D, int32_t K, int32_t F, int64_t capacity, const int32_t *num_roots,
                                        const int64_t *roots, float *memory, float *mailbox, float *mailbox_ts,
                                        int32_t *next_mail_pos, const float *w_ih, const float *w_hh,
                                        const float *b_ih, const float *b_hh, const float *wc_ih, const float *wc_hh,
                                        const float *bc_ih, const float *bc_hh, const int64_t *src, const int64_t *dst,
                                        const float *efeat, const float *ts, const int64_t *batch_start,
                                        const uint64_t *win_src, const uint64_t *win_dst, const int32_t *cnt_src,
                                        const int32_t *cnt_dst, float *new_mem, float *memory_ts, const float *ts_max,
                                        uint32_t *node_bits, const int32_t *sample_cnt, int32_t *any_edges,
                                        float *root_dt, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  SGL_REQUIRE(D > 0 && K > 0 && F >= 0 && 2 * D + F <= kMaxWidth, "memory_update_commit: bad dims D=%d K=%d F=%d", D, K, F);
  SGL_REQUIRE(capacity >= 0 && capacity <= INT_MAX / 2, "memory_update_commit: capacity out of range");
  if (capacity == 0) return SGL_OK;
  SGL_REQUIRE(num_roots && roots && memory && mailbox && mailbox_ts && next_mail_pos && w_ih && w_hh && b_ih && b_hh &&
                  wc_ih && wc_hh && bc_ih && bc_hh && src && dst && ts && win_src && win_dst && cnt_src && cnt_dst &&
                  new_mem && (F == 0 || efeat) && memory_ts && ts_max && node_bits && any_edges,
              "memory_update_commit: NULL array");
  if (workspace == nullptr || workspace_bytes < ws_bytes(D, K, F, capacity)) {
    sgl::set_error("memory_update_commit: workspace %zu bytes < required %zu", workspace_bytes,
                   ws_bytes(D, K, F, capacity));
    return SGL_ERR_WORKSPACE;
  }
  const Events ev{src, dst, efeat, ts, batch_start, reinterpret_cast<const unsigned long long *>(win_src),
                  reinterpret_cast<const unsigned long long *>(win_dst), cnt_src, cnt_dst};
  return launch_split(D, K, F, capacity, num_roots, 0, roots, memory, mailbox, mailbox_ts, next_mail_pos, w_ih, w_hh,
                      b_ih, b_hh, wc_ih, wc_hh, bc_ih, bc_hh, ev,
                      Commit{memory_ts, ts_max, node_bits, sample_cnt, any_edges, root_dt}, new_mem,
                      static_cast<float *>(workspace), stream);
}

extern "C" int sgl_memory_rows(int32_t D, int32_t K, int32_t F, int64_t rows, const float *memory,
                               const float *mailbox, const float *w_ih, const float *w_hh, const float *b_ih,
                               const float *b_hh, const float *wc_ih, const float *wc_hh, const float *bc_ih,
                               const float *bc_hh, float *new_mem, void *workspace, size_t workspace_bytes,
                               hipStream_t stream) {
  SGL_REQUIRE(D > 0 && K > 0 && F >= 0 && 2 * D + F <= kMaxWidth, "memory_rows: bad dims D=%d K=%d F=%d", D, K, F);
  SGL_REQUIRE(rows >= 0 && rows <= INT_MAX / 2, "memory_rows: row count out of range");
  if (rows == 0) return SGL_OK;
  SGL_REQUIRE(memory && mailbox && w_ih && w_hh && b_ih && b_hh && wc_ih && wc_hh && bc_ih && bc_hh && new_mem,
              "memory_rows: NULL array");
  if (workspace == nullptr || workspace_bytes < ws_bytes(D, K, F, rows)) {
    sgl::set_error("memory_rows: workspace %zu bytes < required %zu", workspace_bytes, ws_bytes(D, K, F, rows));
    return SGL_ERR_WORKSPACE;
  }
  return launch_split(D, K, F, rows, nullptr, int(rows), nullptr, memory, const_cast<float *>(mailbox), nullptr, nullptr,
                      w_ih, w_hh, b_ih, b_hh, wc_ih, wc_hh, bc_ih, bc_hh, Events{}, Commit{}, new_mem,
                      static_cast<float *>(workspace), stream);
}
