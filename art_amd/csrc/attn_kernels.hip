// Packed-row attention for gfx950 (MI355X, CDNA4).
//
// The reference materialises a dense [1,S,S] additive bias from the packed
// row's ids (src/art/local/train.py:177-215):
//     visible(i, j) = j <= i && (group[i] == group[j] || parent[i] == group[j])
// and passes it to the model as `causal_mask` (train.py:239-241).  Here the
// matrix is never built.  A plan (once per packed row, shared by every layer
// and head) turns the 64-bit ids into int32 equality codes and classifies each
// (query block, key block) pair as invisible / partly visible / fully visible;
// the attention kernels walk only the visible blocks and evaluate the rule per
// element only in the partly visible ones.
//
// Forward work-group: 128 queries x one head, 4 wavefronts of 32 queries, three
// work-groups per CU.  Scores
// are computed transposed (S^T = K Q^T, MFMA 32x32x16), so that a lane owns one
// query: the row maximum and sum are in-lane reductions plus one exchange between
// the two half-waves, the accumulator of S^T is already in the B-operand layout of
// the second product O^T = V^T P^T, and the running rescale of O^T is a per-lane
// scalar.  K and V tiles are brought into a 2-stage LDS ring by buffer_load ... lds.
// Bound: on long lists power (the clock falls to 1.7 GHz) with the MFMAs, the softmax's vector work and the LDS reads each
// busy for more than half of the time; on packed rows (lists of a few tiles, a sixth of a work-group's time before its first
// tile) latency.  Hence several independent work-groups of 4 waves per CU, one hiding the other's set-up and store, and
// lists made for 128 queries.  Against one work-group of 8 waves per CU with three stages, two of 4 waves with tiles of 64
// keys took 16384 positions of 8 prompts of 137 + 4 x 461, 28 / 4 heads of 128, from 205 to 154 us (dQ 279 -> 244, dK/dV
// 433 -> 297); at up to 3 % more on dense rows of 16384 (16 / 2 heads of 128: 2772 -> 2895 us forward and backward at 12288).
// Steps of 32 keys (AttnKeySteps) since, us before (tiles of 64, one stage of query tiles in dK/dV) / now, heads of 128:
//   forward, three work-groups per CU: the packed row 150 / 129, the same with 16 / 2 heads 88 / 76, 8192 positions of it 83 / 71;
//     dense 16384 1766 / 1771, 4096 130 / 132, 8192 with 16 / 2 heads 274 / 273
//   dQ: the packed row 248 / 214, 16 / 2 heads 142 / 119; dense 16384 2521 / 2447, 8192 660 / 643
//   dK/dV: the packed row 303 / 262, 16 / 2 heads 219 / 154; dense 3832 / 3471, 945 / 896; heads of 64, 14 / 2: 8192 dense 296 / 270
// A head dimension of 64 has too few MFMAs per key for steps of 32 in the forward (8192 dense: 138 -> 160 us).
#include <stdlib.h>

#include "common.hpp"
#include "gemm_nt.hpp"

namespace artk {

constexpr int ATT_ROW = 256;   // row lengths are multiples of this
constexpr int ATT_BM = 128;    // queries per work-group
constexpr int ATT_BN = 64;     // keys per tile
constexpr int ATT_STAGES = 2;
constexpr int ATT_MAX_KB = 1024;  // key blocks per row the list in LDS can hold
constexpr int ATT_BQ2 = 64;    // dK/dV kernel: queries per tile
constexpr int ATT_BK2 = 64;    // dK/dV kernel: keys per work-group (2 key groups x 32)

// ----------------------------------------------------------------------------
// Plan
// ----------------------------------------------------------------------------

// Every kernel of the plan takes a batch of rows: blockIdx.y (attn_heads_kernel: blockIdx.x) is the row, whose
// plan lies `stride` bytes behind the one before.  Positions S .. Sp - 1 fill up the last block: they get codes
// nothing else carries, so they see, and are seen by, themselves only.
template <class T>
__device__ __forceinline__ T* attn_row(T* p, int64_t stride, int row) {
  return (T*)((char*)p + stride * row);
}

// heads = the positions whose group id differs from the one before, ascending: the first position of a group
// is always one of them, so the equality codes need S x (runs) comparisons instead of S^2 (a packed row has a
// run per prompt and completion).  One work-group per row, each thread a contiguous piece.
__global__ __launch_bounds__(1024) void attn_heads_kernel(const int64_t* __restrict__ group_ids, int S,
                                                          int64_t stride, int* __restrict__ heads,
                                                          int* __restrict__ n_heads) {
  __shared__ int wtot[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t* g = group_ids + (int64_t)blockIdx.x * S;
  heads = attn_row(heads, stride, blockIdx.x);
  const int per = (S + 1023) / 1024;
  const int t0 = (int)threadIdx.x * per, t1 = t0 + per < S ? t0 + per : S;
  int n = 0;
  int64_t prev = t0 > 0 && t0 < S ? g[t0 - 1] : 0;
  for (int t = t0; t < t1; ++t) {
    const int64_t id = g[t];
    n += t == 0 || id != prev;
    prev = id;
  }
  int run = n;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(run, d, 64);
    if (lane >= d) run += v;
  }
  if (lane == 63) wtot[wave] = run;
  __syncthreads();
  int off = run - n;
  for (int w = 0; w < wave; ++w) off += wtot[w];
  prev = t0 > 0 && t0 < S ? g[t0 - 1] : 0;
  for (int t = t0; t < t1; ++t) {
    const int64_t id = g[t];
    if (t == 0 || id != prev) heads[off++] = t;
    prev = id;
  }
  if (threadIdx.x == 1023) *attn_row(n_heads, stride, blockIdx.x) = off;
}

// gc[t] = first position whose group id equals group_ids[t];
// pc[t] = first position whose group id equals parent_ids[t], or -2 if none.
// Then group[i] == group[j] <=> gc[i] == gc[j] and parent[i] == group[j] <=>
// pc[i] == gc[j].  uni[c] = {gc, pc} of positions 32 c .. 32 c + 31 where they all agree,
// else ATT_MIXED in that component.
constexpr int ATT_MIXED = (int)0x80000000;
__global__ __launch_bounds__(256) void attn_codes_kernel(const int64_t* __restrict__ group_ids,
                                                         const int64_t* __restrict__ parent_ids,
                                                         int S, int64_t stride, const int* __restrict__ heads,
                                                         const int* __restrict__ n_heads, int* __restrict__ gc,
                                                         int* __restrict__ pc, int2* __restrict__ uni) {
  __shared__ int64_t hid[256];
  __shared__ int hpos[256];
  const int row = blockIdx.y;
  group_ids += (int64_t)row * S;
  parent_ids += (int64_t)row * S;
  heads = attn_row(heads, stride, row);
  const int nh = *attn_row(n_heads, stride, row);
  const int t = blockIdx.x * 256 + threadIdx.x;
  const bool in = t < S;
  const int64_t g = in ? group_ids[t] : 0;
  const int64_t pa = in ? parent_ids[t] : 0;
  int first_g = -1, first_p = -2;
  for (int h0 = 0; h0 < nh; h0 += 256) {
    const int lim = nh - h0 < 256 ? nh - h0 : 256;
    __syncthreads();
    if ((int)threadIdx.x < lim) {
      const int pos = heads[h0 + threadIdx.x];
      hpos[threadIdx.x] = pos;
      hid[threadIdx.x] = group_ids[pos];
    }
    __syncthreads();
    for (int j = lim - 1; j >= 0; --j) {   // descending, so the first match wins within this piece
      const int64_t id = hid[j];
      const int pos = hpos[j];
      if (id == g && (first_g < 0 || first_g >= hpos[0])) first_g = pos;
      if (id == pa && (first_p < 0 || first_p >= hpos[0])) first_p = pos;
    }
  }
  const int gcv = in ? first_g : -3 - t, pcv = in ? first_p : -2;
  attn_row(gc, stride, row)[t] = gcv;
  attn_row(pc, stride, row)[t] = pcv;
  const int lane = threadIdx.x & 63, base = lane & 32;
  const unsigned long long mine = 0xffffffffull << base;
  const bool ug = (__ballot(gcv == __shfl(gcv, base, 64)) & mine) == mine;
  const bool up = (__ballot(pcv == __shfl(pcv, base, 64)) & mine) == mine;
  if ((lane & 31) == 0) attn_row(uni, stride, row)[t / 32] = make_int2(ug ? gcv : ATT_MIXED, up ? pcv : ATT_MIXED);
}

__device__ __forceinline__ bool attn_visible(int i, int j, int gi, int pi, int gj) {
  return j <= i && (gj == gi || gj == pi);
}

// Visibility of one (owner block, tile) pair, by cells of 32 queries x 32 keys:
//   bits 14-15  1 = some pairs visible, 2 = all
//   bits 16-23  cell c has at least one visible pair
//   bits 24-31  every pair of cell c is visible (no per-element test needed)
// 0 when nothing is visible.
//   info  (forward, dQ): owner = 128 queries, tile = 64 keys; wave w (of 4) = queries 32w..32w+31, its cells are
//                        c = 2w (keys 0..31) and 2w + 1 (keys 32..63).
//   info2 (dK/dV):       owner = 64 keys, tile = 64 queries; wave w (of 4) = cell w = keys 32(w&1).. x
//                        queries 32(w>>1)..
// One wavefront takes 128 queries x 64 keys = 8 cells of 32 x 32 and writes the entry of info and both
// entries of info2.  A cell whose queries share their codes and whose keys share theirs is decided from
// uni; only the others are evaluated pair by pair (64 lanes = 32 keys x 2 halves of the queries).
__device__ __forceinline__ uint32_t attn_entry(uint32_t any, uint32_t all, uint32_t cells) {
  return any ? ((all == cells ? 2u : 1u) << 14) | (any << 16) | (all << 24) : 0u;
}
// info_row: the query block's row of info.
__device__ __forceinline__ void attn_classify_pair(const int* gc, const int* pc, const int2* uni, int nQb2, int owner, int kb, uint32_t* info_row, uint32_t* info2) {
  const int lane = threadIdx.x & 63;
  uint32_t any = 0, all = 0;   // bit 2 w + kg: cell of queries 32 w.., keys 32 kg..
  if (kb * ATT_BN <= owner * ATT_BM + ATT_BM - 1) {
    const int qc = owner * (ATT_BM / 32) + ((lane & 7) >> 1), kc = kb * 2 + (lane & 1);  // lanes 0..7: one cell each
    const int2 uq = uni[qc];
    const int gk = uni[kc].x;
    const bool live = kc <= qc;
    const bool known = !live || (uq.x != ATT_MIXED && uq.y != ATT_MIXED && gk != ATT_MIXED);
    const bool eq = live && known && (gk == uq.x || gk == uq.y);
    any = (uint32_t)__ballot(eq) & 0xffu;
    all = (uint32_t)__ballot(eq && kc < qc) & 0xffu;
    for (uint32_t left = (uint32_t)__ballot(!known) & 0xffu; left; left &= left - 1) {
      const int cell = __builtin_ctz(left);
      const int q0 = (owner * (ATT_BM / 32) + (cell >> 1)) * 32 + 16 * (lane >> 5);
      const int j = (kb * 2 + (cell & 1)) * 32 + (lane & 31);
      const int gj = gc[j];
      int cnt = 0;
#pragma unroll
      for (int ii = 0; ii < 16; ++ii) cnt += attn_visible(q0 + ii, j, gc[q0 + ii], pc[q0 + ii], gj) ? 1 : 0;
      any |= (uint32_t)(__ballot(cnt > 0) != 0ull) << cell;
      all |= (uint32_t)(__ballot(cnt == 16) == ~0ull) << cell;
    }
  }
  if (lane == 0) {
    info_row[kb] = attn_entry(any, all, 0xffu);
    info2[(int64_t)kb * nQb2 + 2 * owner] = attn_entry(any & 0xfu, all & 0xfu, 0xfu);
    info2[(int64_t)kb * nQb2 + 2 * owner + 1] = attn_entry(any >> 4, all >> 4, 0xfu);
  }
}
__global__ __launch_bounds__(256) void attn_classify_kernel(const int* __restrict__ gc, const int* __restrict__ pc,
                                                            const int2* __restrict__ uni, int64_t stride, int nKb,
                                                            int nQb2, uint32_t* __restrict__ info,
                                                            uint32_t* __restrict__ info2) {
  const int row = blockIdx.z, owner = blockIdx.y, kb = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (kb >= nKb) return;
  attn_classify_pair(attn_row(gc, stride, row), attn_row(pc, stride, row), attn_row(uni, stride, row), nQb2, owner, kb,
                     attn_row(info, stride, row) + (int64_t)owner * nKb, attn_row(info2, stride, row));
}

// list[row][0..cnt[row]) = tile index | info for the tiles of info[row][*] that
// are not 0, ascending.  One work-group per row of either table (the key blocks after the query blocks).
struct AttnTable {
  const uint32_t* info;
  uint32_t* list;
  int* cnt;
  int nrow, ncol;
};
__global__ __launch_bounds__(256) void attn_compact_kernel(AttnTable a, AttnTable b, int64_t stride) {
  __shared__ int wtot[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool second = (int)blockIdx.x >= a.nrow;
  const int row = second ? (int)blockIdx.x - a.nrow : (int)blockIdx.x;
  const int ncol = second ? b.ncol : a.ncol;
  const uint32_t* info = attn_row(second ? b.info : a.info, stride, blockIdx.y) + (int64_t)row * ncol;
  uint32_t* list = attn_row(second ? b.list : a.list, stride, blockIdx.y) + (int64_t)row * ncol;
  int base = 0;
  for (int c0 = 0; c0 < ncol; c0 += 256) {
    const int c = c0 + threadIdx.x;
    const uint32_t v = c < ncol ? info[c] : 0u;
    const unsigned long long m = __ballot(v != 0);
    const int rank = __popcll(m & ((1ull << lane) - 1ull));
    __syncthreads();
    if (lane == 0) wtot[wave] = __popcll(m);
    __syncthreads();
    int off = base;
    for (int w = 0; w < wave; ++w) off += wtot[w];
    if (v) list[off + rank] = (uint32_t)c | v;
    base += wtot[0] + wtot[1] + wtot[2] + wtot[3];
  }
  if (threadIdx.x == 0) attn_row(second ? b.cnt : a.cnt, stride, blockIdx.y)[row] = base;
}

// order[r] = the block with the r-th largest count (ties: the later block first): work-groups are dispatched
// in this order, so the long ones do not end up alone at the end of a launch.  Work-group x = 0 sorts the
// query blocks, 1 the key blocks (and adds up their counts); at most 1024 counts each, by rank.
__global__ __launch_bounds__(1024) void attn_order_kernel(const int* __restrict__ cnt, int n, int* __restrict__ order,
                                                          const int* __restrict__ cnt2, int n2,
                                                          int* __restrict__ order2, int* __restrict__ total2,
                                                          int64_t stride) {
  __shared__ int c[ATT_MAX_KB];
  const bool second = blockIdx.x == 1;
  const int m = second ? n2 : n;
  const int t = threadIdx.x;
  if (t < m) c[t] = attn_row(second ? cnt2 : cnt, stride, blockIdx.y)[t];
  __syncthreads();
  if (t >= m) return;
  int rank = 0, sum = 0;
  for (int i = 0; i < m; ++i) {
    sum += c[i];
    rank += (c[i] > c[t] || (c[i] == c[t] && i > t)) ? 1 : 0;
  }
  if (second && t == 0) *attn_row(total2, stride, blockIdx.y) = sum;
  attn_row(second ? order2 : order, stride, blockIdx.y)[rank] = t;
}

// Device-memory layout of the plan of one row of S positions (a multiple of 256).
struct AttnPlan {
  int* gc;
  int* pc;
  int nQb, nKb;        // forward / dQ: query blocks of 128, key tiles of 64
  uint32_t* info;      // [nQb][nKb]
  uint32_t* list;      // [nQb][nKb]
  int* cnt;            // [nQb]
  int* order;          // [nQb] query blocks by falling number of visible tiles
  int nQb2, nKb2;      // dK/dV: key blocks of 64, query tiles of 64
  uint32_t* info2;     // [nKb2][nQb2]
  uint32_t* list2;     // [nKb2][nQb2]
  int* cnt2;           // [nKb2]
  int* order2;         // [nKb2]
  int* total2;         // sum of cnt2
  int2* uni;           // [S / 32]
  int* heads;          // [S]
  int* n_heads;
  int64_t stride;      // bytes from one row's plan to the next
};

static size_t attn_plan_layout(void* base, size_t bytes, int64_t S, AttnPlan& pl) {
  Workspace ws(base, bytes);
  pl.nQb = (int)(S / ATT_BM);
  pl.nKb = (int)(S / ATT_BN);
  pl.nQb2 = (int)(S / ATT_BQ2);
  pl.nKb2 = (int)(S / ATT_BK2);
  pl.gc = ws.take<int>((size_t)S);
  pl.pc = ws.take<int>((size_t)S);
  pl.info = ws.take<uint32_t>((size_t)pl.nQb * pl.nKb);
  pl.list = ws.take<uint32_t>((size_t)pl.nQb * pl.nKb);
  pl.cnt = ws.take<int>((size_t)pl.nQb);
  pl.order = ws.take<int>((size_t)pl.nQb);
  pl.info2 = ws.take<uint32_t>((size_t)pl.nQb2 * pl.nKb2);
  pl.list2 = ws.take<uint32_t>((size_t)pl.nQb2 * pl.nKb2);
  pl.cnt2 = ws.take<int>((size_t)pl.nKb2);
  pl.order2 = ws.take<int>((size_t)pl.nKb2);
  pl.total2 = ws.take<int>(1);
  pl.uni = ws.take<int2>((size_t)S / 32);
  pl.heads = ws.take<int>((size_t)S);
  pl.n_heads = ws.take<int>(1);
  pl.stride = (int64_t)align_up(ws.used, 256);
  return ws.ok() || base == nullptr ? ws.used : (size_t)-1;
}

// The plan of a short row in two launches instead of the chain of five above (18 us and the gaps between them in front of
// a layer of 60 us at 1009 positions).  In the first, a work-group per query block finds the codes of the whole row for
// itself, in LDS, and classifies and lists its own tiles, a wave per 64 keys; the second lists the tiles of the key blocks
// and sorts.  Every array of the plan gets the values that the chain writes.  (In one launch with one work-group per row
// the mixed cells of the whole row take 30 us on their one CU.)
// Positions, padded: one per thread of a work-group.  The two kernels take 14.1 us at 1009 positions; the chain, for longer rows,
// 18.7 at 1100 and 17.7 at 2048.
constexpr int ATT_SHORT = 1024;
__global__ __launch_bounds__(1024) void attn_plan_short_kernel(const int64_t* __restrict__ group_ids,
                                                               const int64_t* __restrict__ parent_ids, int S, AttnPlan pl) {
  static_assert(ATT_SHORT <= 1024 && ATT_SHORT / ATT_BN <= 16, "one position per thread, a key tile per wave");
  __shared__ int64_t hid[ATT_SHORT];
  __shared__ int hpos[ATT_SHORT], gc[ATT_SHORT], pc[ATT_SHORT];
  __shared__ int2 uni[ATT_SHORT / 32];
  __shared__ uint32_t info[16];
  __shared__ int wtot[16];
  const int row = blockIdx.y, owner = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int padded = pl.nKb * ATT_BN;
  const bool in = t < S;
  const int64_t g = in ? group_ids[(int64_t)row * S + t] : 0, pa = in ? parent_ids[(int64_t)row * S + t] : 0;

  // positions where a run of equal group ids begins
  const int64_t prev = in && t > 0 ? group_ids[(int64_t)row * S + t - 1] : 0;
  const bool head = in && (t == 0 || g != prev);
  const unsigned long long hm = __ballot(head);
  if (lane == 0) wtot[wave] = __popcll(hm);
  __syncthreads();
  int at = __popcll(hm & ((1ull << lane) - 1ull)), nh = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    at += w < wave ? wtot[w] : 0;
    nh += wtot[w];
  }
  if (head) {
    hpos[at] = t;
    hid[at] = g;
    if (owner == 0) attn_row(pl.heads, pl.stride, row)[at] = t;
  }
  if (owner == 0 && t == 0) *attn_row(pl.n_heads, pl.stride, row) = nh;
  __syncthreads();

  // codes
  int first_g = -1, first_p = -2;
  for (int j = nh - 1; j >= 0; --j) {  // descending: the first match wins
    const int64_t id = hid[j];
    if (id == g) first_g = hpos[j];
    if (id == pa) first_p = hpos[j];
  }
  const int gcv = in ? first_g : -3 - t, pcv = in ? first_p : -2;
  gc[t] = gcv;
  pc[t] = pcv;
  const int base = lane & 32;
  const unsigned long long mine = 0xffffffffull << base;
  const bool ug = (__ballot(gcv == __shfl(gcv, base, 64)) & mine) == mine;
  const bool up = (__ballot(pcv == __shfl(pcv, base, 64)) & mine) == mine;
  if (owner == 0 && t < padded) {
    attn_row(pl.gc, pl.stride, row)[t] = gcv;
    attn_row(pl.pc, pl.stride, row)[t] = pcv;
  }
  if ((lane & 31) == 0) {
    const int2 u = make_int2(ug ? gcv : ATT_MIXED, up ? pcv : ATT_MIXED);
    uni[t / 32] = u;
    if (owner == 0 && t < padded) attn_row(pl.uni, pl.stride, row)[t / 32] = u;
  }
  __syncthreads();

  if (wave < pl.nKb)
    attn_classify_pair(gc, pc, uni, pl.nQb2, owner, wave, info, attn_row(pl.info2, pl.stride, row));
  __syncthreads();
  if (wave == 0) {
    const uint32_t v = lane < pl.nKb ? info[lane] : 0u;
    const unsigned long long m = __ballot(v != 0);
    if (v) attn_row(pl.list, pl.stride, row)[owner * pl.nKb + __popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)lane | v;
    if (lane < pl.nKb) attn_row(pl.info, pl.stride, row)[owner * pl.nKb + lane] = v;
    if (lane == 0) attn_row(pl.cnt, pl.stride, row)[owner] = __popcll(m);
  }
}

__global__ __launch_bounds__(1024) void attn_plan_short_order_kernel(AttnPlan pl) {
  __shared__ int cnt2[16];
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave < pl.nKb2) {
    const uint32_t v = lane < pl.nQb2 ? attn_row(pl.info2, pl.stride, row)[wave * pl.nQb2 + lane] : 0u;
    const unsigned long long m = __ballot(v != 0);
    if (v) attn_row(pl.list2, pl.stride, row)[wave * pl.nQb2 + __popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)lane | v;
    if (lane == 0) attn_row(pl.cnt2, pl.stride, row)[wave] = cnt2[wave] = __popcll(m);
  }
  __syncthreads();
  // order of dispatch, by rank: wave 0 the query blocks, wave 1 the key blocks
  if (wave < 2) {
    const bool second = wave == 1;
    const int m = second ? pl.nKb2 : pl.nQb;
    const int mine = lane < m ? (second ? cnt2[lane] : attn_row(pl.cnt, pl.stride, row)[lane]) : 0;
    int rank = 0, sum = 0;
    for (int i = 0; i < m; ++i) {
      const int c = __shfl(mine, i, 64);
      sum += c;
      rank += (c > mine || (c == mine && i > lane)) ? 1 : 0;
    }
    if (second && lane == 0) *attn_row(pl.total2, pl.stride, row) = sum;
    if (lane < m) attn_row(second ? pl.order2 : pl.order, pl.stride, row)[rank] = lane;
  }
}

// ----------------------------------------------------------------------------
// Tiles and fragments shared by the three kernels
// ----------------------------------------------------------------------------
// An operand tile in LDS is 64 or 32 rows (keys or queries) x D elements, row-major
// as in HBM, its 16-byte chunks XOR-swizzled by row.  Two ways to read it:
//   row fragments  (ds_read_b128): lane (m, h) gets 8 consecutive d of row m,
//                   the A operand of a product that contracts over d;
//   transposed fragments (ds_read_b64_tr_b16, a gfx950 instruction): lane (m, h)
//                   gets element d = m of 8 rows, the A operand of a product
//                   that contracts over the tile's rows.  No transposed copies
//                   of K, V, Q or dO exist anywhere.
template <int D>
struct AttnTile {
  static constexpr int CHK = D / 8;                    // 16-byte chunks of a row
  static constexpr int ROW = D * 2;                    // bytes
  static constexpr int BYTES = 64 * ROW;
  static constexpr int N4 = BYTES / 1024 / 4;          // DMA instructions per wave
  // XOR applied to the chunk index of a row.  Two access patterns must be free of
  // bank conflicts (256 bytes = 16 chunk slots per bank line; with D = 64 two rows
  // share a line): a row-fragment read takes one chunk of 16 consecutive rows, a
  // transposed read takes 4 consecutive chunks (aligned to 4) of 4 consecutive
  // rows (aligned to 4).  So rows that differ in their low bits must land in
  // different aligned groups of 4 chunks, and the 16 rows of a fragment read in 16
  // different slots: the low row bits go to the high chunk bits and vice versa.
  __device__ static __forceinline__ int swz(int row) {
    return CHK == 16 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
  }
  // per-lane byte offset (global side) of DMA instruction `instr` of a tile whose
  // rows are `stride` elements apart
  __device__ static __forceinline__ int voff(int instr, int lane, int64_t stride) {
    const int r = instr * (64 / CHK) + lane / CHK;
    const int c = (lane % CHK) ^ swz(r);
    return (int)(r * stride * 2) + c * 16;
  }
  // The same from three registers (row and chunk of instruction 0; the row's offset in the scalar offset of the
  // instruction) instead of one per instruction: instructions begin a multiple of 4 (D = 64: 8) rows apart, so their
  // swizzles differ by an XOR.
  __device__ static __forceinline__ int row_of(int instr) { return instr * (64 / CHK); }
  __device__ static __forceinline__ int lane_row(int lane, int64_t stride) { return lane / CHK * (int)(stride * 2); }
  __device__ static __forceinline__ int lane_chunk(int lane) { return ((lane % CHK) ^ swz(lane / CHK)) << 4; }
  __device__ static __forceinline__ int chunk_of(int chunk, int instr) { return chunk ^ (swz(row_of(instr)) << 4); }
  // row fragment: row `row`, d = 16 s + 8 h ..
  __device__ static __forceinline__ bf16x8 row_frag(const char* tile, int row, int s, int h) {
    return *(const bf16x8*)(tile + row * ROW + (((2 * s + h) ^ swz(row)) * 16));
  }
};

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short shortx4;
typedef __attribute__((address_space(3))) shortx4* lds_shortx4_ptr;

// The LDS transpose read works on groups of 16 lanes: lane 4e+g of a group
// supplies the address of 4 consecutive halfwords, and lane i receives, as
// element e, halfword i%4 of what lane 4e + i/4 addressed.  With lane 4e+g
// pointing at row (k0 + e), columns d0 + 4g .., lane i ends up with column
// d0 + i of rows k0 .. k0+3.
struct TrLane {
  int row_off;   // row this lane addresses, relative to the slab: 4h + e
  int dcol;      // first of its 4 columns, relative to the 32-column tile: 16 (b & 1) + 4 g
  __device__ __forceinline__ TrLane(int lane) {
    const int b = lane >> 4, i = lane & 15;
    row_off = 4 * (b >> 1) + (i >> 2);
    dcol = 16 * (b & 1) + 4 * (i & 3);
  }
};

// The reads of a tile, from byte offsets that the caller prepares once.  A row is a power of two of bytes long, so the chunk
// of step s (row fragments) or of the 32 columns dt (transposed ones) can be XORed into the offset of chunk 0, and
// rows 16 apart have the same swizzle.  One register per row instead of one per address: where those are short.
template <int D>
__device__ __forceinline__ int frag_base(int row, int h) {
  return row * AttnTile<D>::ROW + ((h ^ AttnTile<D>::swz(row)) << 4);
}
__device__ __forceinline__ bf16x8 frag_at(const char* tile, int base, int s) {
  return *(const bf16x8*)(tile + (base ^ (s << 5)));
}
// Transposed fragment of a 16-row slab and 32 columns: lane (m, h) gets column m of rows 4h + {0..3} and
// 8 + 4h + {0..3} -- the row order in which the accumulator of the score tile, used as the other operand, holds a slab.
struct TrBase {
  int lo, hi;  // rows k0 + 4h + {0..3} and 8 below
};
template <int D>
__device__ __forceinline__ TrBase tr_base(const TrLane& t, int k0) {
  using T = AttnTile<D>;
  const int r0 = k0 + t.row_off, r1 = r0 + 8, c = (t.dcol & 4) * 2;
  return {r0 * T::ROW + (((t.dcol >> 3) ^ T::swz(r0)) << 4) + c, r1 * T::ROW + (((t.dcol >> 3) ^ T::swz(r1)) << 4) + c};
}
// Slab u (16 rows each) below k0, columns 32 dt ..
template <int D>
__device__ __forceinline__ bf16x8 tr_at(const char* tile, const TrBase& b, int u, int dt) {
  const char* slab = tile + u * 16 * AttnTile<D>::ROW;
  const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_ptr)(slab + (b.lo ^ (dt << 6))));
  const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4_ptr)(slab + (b.hi ^ (dt << 6))));
  typedef __attribute__((__vector_size__(8 * sizeof(short)))) short shortx8;
  const shortx8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

// attn_smem_note: the kernels below track the completion of their LDS DMA by hand (wait_vmcnt
// before the barrier that publishes a stage).  Two things would make the compiler drain every
// outstanding DMA instead, serialising the ring: a second LDS variable in the kernel (it then
// puts s_waitcnt vmcnt(0) in front of LDS reads that follow a DMA issue), and __syncthreads(),
// whose fence waits for all memory operations; hence one LDS array per kernel, carved by
// hand, and barrier_lds_only() inside the loops.
// Makes the compiler finish the load of v here (it waits for a value where an instruction first
// uses it).  Left alone it would put the wait for a prologue load at the first use inside the main
// loop, where the same s_waitcnt vmcnt(..) then also waits for the DMA ring on every iteration.
template <class V>
__device__ __forceinline__ void pin_loaded(V& v) {
  asm volatile("" : "+v"(v));
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Descriptor of one head's rows 0 .. S-1 (`stride` elements apart): rows past the end, which fill up the last
// tile of a row whose length is no multiple of the tile's, arrive in LDS as zeros.
template <int D>
__device__ __forceinline__ dma_rsrc_t attn_head_rsrc(const uint16_t* head, int64_t stride, int S) {
  return dma_make_rsrc(head, (uint32_t)(((int64_t)(S - 1) * stride + D) * 2));
}
__device__ __forceinline__ dma_rsrc_t attn_rsrc(const void* p) { return dma_make_rsrc(p, 0x7fffffffu); }

// ----------------------------------------------------------------------------
// Forward
// ----------------------------------------------------------------------------
constexpr int ATT_THREADS = 2 * ATT_BM;  // forward and dQ: a wave per 32 queries

// (query head, query block) of a work-group of the forward and dQ kernels.  A unit is the work-groups of
// the heads that share one key/value head and query block: they read the same K and V tiles, so a unit
// runs on one XCD (block b is placed on XCD b % 8), its heads one after the other; long blocks first.
// With `even` (forward and dQ; the dK/dV kernel, whose work-groups are not ordered by their work alone, became slower):
// - There are 8 / Hkv XCDs to a key/value head.  They are dealt the blocks forwards and backwards by turns, or the first
//   of them would get the longest block of every turn (of 64 blocks of a dense causal row and 2 key/value heads: 5 %
//   more work than the average).
// - The first two work-groups of each of an XCD's 32 CUs start together, and share the CU's speed.  The second ones come
//   shortest first, so that a CU with the longest block of the row has the shortest beside it.  Longest first throughout,
//   one CU had 128 + 96 tiles of work to begin with and another 98 + 66, which was then free for the longest of the rest,
//   twice (clock stamps at 8192 positions, 16 heads: CUs ended between 232 and 306 us).
// Dense causal row of 8192 positions, heads of 128, forward / dQ in us: 16 / 2 heads 289 / 404 -> 271 / 390 (half of it
// by either), 16 / 16 heads 287 / 403 -> 274 / 392.
constexpr int ATT_XCD_CUS = 32;
__device__ __forceinline__ bool attn_block(int Hq, int Hkv, int nQb, const int* order, bool even, int& hq, int& qb) {
  const int rep = Hq / Hkv;
  int loc = blockIdx.x >> 3;
  int x = blockIdx.x & 7;
  if (even) {
    const int n = (int)(gridDim.x >> 3), end = n < 2 * ATT_XCD_CUS ? n : 2 * ATT_XCD_CUS;
    if (blockIdx.y == 0 && loc >= ATT_XCD_CUS && loc < end) loc = ATT_XCD_CUS + end - 1 - loc;
    if (8 % Hkv == 0 && (loc / rep & 1)) x = (8 / Hkv - 1 - x / Hkv) * Hkv + x % Hkv;
  }
  const int unit = (loc / rep) * 8 + x;
  const int hkv = unit % Hkv;
  hq = hkv * rep + loc % rep;
  if (unit / Hkv >= nQb) return false;
  qb = order[unit / Hkv];
  return true;
}
static unsigned attn_grid(int Hq, int Hkv, int nQb) {
  return (unsigned)((nQb * Hkv + 7) / 8 * 8 * (Hq / Hkv));
}

struct AttnFwdParams {
  const uint16_t* Q;   // element (s, h, d) at s * q_ss + h * q_hs + d
  const uint16_t* K;
  const uint16_t* V;
  uint16_t* O;
  float* lse;          // [Hq][S], natural log
  int64_t q_ss, q_hs, k_ss, k_hs, v_ss, v_hs, o_ss, o_hs;
  const int* gc;
  const int* pc;
  const uint32_t* list;
  const int* cnt;
  const int* order;
  int64_t plan_stride, q_bs, k_bs, v_bs, o_bs;   // per row of the batch (blockIdx.y)
  int S, Hq, Hkv, nQb, nKb;
  float scale_log2e;
};

// The keys of a query block, KEYS at a time, in the forward and dQ kernels.  Step i is part i % STEPS of tile i / STEPS of
// the list; steps that no wave sees are left out.  LDS stage of a step: its rows of K, of V and their codes.
// KEYS = 32 takes half the LDS and a third fewer registers (so three work-groups of the forward fit a CU where two did), and
// a wave computes 32 x 32 cells that it sees instead of 32 x 64: 13 % less on the packed row of the header, where 43 %
// fewer elements are tested too.  It costs two barriers and two reductions of the maximum per 64 keys, so everything per
// step is kept short: the offsets into LDS move with the stage, those of the DMA are precomputed, the next entry of the list
// is read while the step is computed (without that: 1900 us instead of 1840 on the dense row).
template <int D, int KT>
struct AttnKeySteps {
  using T = AttnTile<D>;
  static constexpr int KEYS = 32 * KT;
  static constexpr int STEPS = ATT_BN / KEYS;           // of a tile of the list
  static constexpr int V_OFF = KEYS * T::ROW;
  static constexpr int CODE_OFF = 2 * V_OFF;
  static constexpr int STAGE = CODE_OFF + 1024;
  static constexpr int DMAS = V_OFF / 4096;             // per operand and wave
  static constexpr int LIST_OFF = ATT_STAGES * STAGE;
  static constexpr int LDS = LIST_OFF + ATT_MAX_KB * 4 + 8;
  dma_rsrc_t rsrc_k, rsrc_v, rsrc_c;
  int voff_k[DMAS], voff_v[DMAS];
  int64_t k_ss, v_ss;
  int cur, nxt, n;           // this step, the next, their number
  uint32_t entry, e_nxt;     // and their tiles' entries

  __device__ static __forceinline__ bool seen(uint32_t e, int half) { return STEPS == 1 || (e >> (16 + half) & 0x55u) != 0; }
  __device__ static __forceinline__ int key(uint32_t e, int i) {
    return (int)(e & 0x3fff) * ATT_BN + (STEPS == 2 ? 32 * (i & 1) : 0);
  }
  __device__ __forceinline__ int key() const { return key(entry, cur); }
  // Cells of `wave` in this step: bit kt of any: its 32 queries see part of keys 32 kt ..; of mixed: but not all of them.
  __device__ __forceinline__ int any(int wave) const { return entry >> (16 + 2 * wave + (STEPS == 2 ? cur & 1 : 0)) & (2 * KT - 1); }
  __device__ __forceinline__ int mixed(int wave) const { return ~entry >> (24 + 2 * wave + (STEPS == 2 ? cur & 1 : 0)) & (2 * KT - 1); }
  // From the next step on; e1: the entry behind its tile's.
  __device__ __forceinline__ void advance(uint32_t e1) {
    if (STEPS == 2) {
      const bool same = !(nxt & 1) && seen(e_nxt, 1);
      nxt = same ? nxt + 1 : (nxt | 1) + (seen(e1, 0) ? 1 : 2);
      e_nxt = same ? e_nxt : e1;
    } else {
      ++nxt;
      e_nxt = e1;
    }
  }
  // DMA of the keys from k0 on into the stage at st: this wave's share of the rows, and the codes (every wave writes the
  // same bytes).
  __device__ __forceinline__ void issue(char* st, int k0, int wave, int lane) const {
    const int so_k = (int)(k0 * k_ss * 2), so_v = (int)(k0 * v_ss * 2);
#pragma unroll
    for (int i = 0; i < DMAS; ++i) {
      dma_load16(rsrc_k, voff_k[i], so_k, lds_addr_of(st + (wave * DMAS + i) * 1024));
      dma_load16(rsrc_v, voff_v[i], so_v, lds_addr_of(st + V_OFF + (wave * DMAS + i) * 1024));
    }
    dma_load4(rsrc_c, (lane & (KEYS - 1)) * 4, k0 * 4, lds_addr_of(st + CODE_OFF));
  }
  // The first two steps are on their way before anything else is read.  (A row of the plan has four entries or more.)
  __device__ __forceinline__ void begin(char* smem, const uint16_t* k_head, int64_t k_stride, const uint16_t* v_head,
                                        int64_t v_stride, int S, const int* codes, const uint32_t* list, int tiles, int wave,
                                        int lane) {
    rsrc_k = attn_head_rsrc<D>(k_head, k_stride, S);
    rsrc_v = attn_head_rsrc<D>(v_head, v_stride, S);
    rsrc_c = attn_rsrc(codes);
    k_ss = k_stride;
    v_ss = v_stride;
#pragma unroll
    for (int i = 0; i < DMAS; ++i) {
      voff_k[i] = T::voff(wave * DMAS + i, lane, k_ss);
      voff_v[i] = T::voff(wave * DMAS + i, lane, v_ss);
    }
    n = STEPS * tiles;
    cur = nxt = 0;
    entry = e_nxt = 0;
    if (tiles > 0) {
      entry = e_nxt = __builtin_amdgcn_readfirstlane(list[0]);
      const uint32_t e1 = __builtin_amdgcn_readfirstlane(list[1]);
      cur = nxt = seen(entry, 0) ? 0 : 1;
      issue(smem, key(), wave, lane);
      advance(e1);
      if (nxt < n) issue(smem + STAGE, key(e_nxt, nxt), wave, lane);
    }
    for (int i = threadIdx.x; i < tiles; i += ATT_THREADS) ((uint32_t*)(smem + LIST_OFF))[i] = list[i];
  }
  // The entry that end() needs, read while the step is computed (past the end of the list: not used).
  __device__ __forceinline__ uint32_t ahead(const char* smem) const { return ((const uint32_t*)(smem + LIST_OFF))[nxt / STEPS + 1]; }
  // End of the step in `stage`.
  __device__ __forceinline__ void end(char* smem, int stage, uint32_t e1, int wave, int lane) {
    cur = nxt;
    entry = e_nxt;
    // After the last step nothing is on its way and nobody reads LDS again.  (A barrier here held back the waves whose last
    // step was an earlier one: forward of 2 x 1300 positions, 28 / 4 heads, 28.5 us, now 26.7; 8192 packed 75.8, now 72.3.)
    if (cur >= n) return;
    advance(__builtin_amdgcn_readfirstlane(e1));
    wait_vmcnt<0>();
    barrier_lds_only();  // the next step is there, and every wave is done with this one
    if (nxt < n) issue(smem + stage * STAGE, key(e_nxt, nxt), wave, lane);
  }
};

template <int D>
__global__ __launch_bounds__(ATT_THREADS, 3) void attn_fwd_kernel(AttnFwdParams p) {
  using T = AttnTile<D>;
  // 32 keys of a step.  (The same for every launch of a head dimension: a row's bits do not depend on its batch.  Steps of 64, two
  // work-groups per CU, in launches of up to two per CU at D = 128, us, 64 / 32: 1 x 4096 of 300 + 2 x 1800, 16 / 2 heads 73 / 69;
  // 1 x 2048, 28 / 4 heads 26.5 / 25.2; 1 x 1009 13.9 / 13.9; 1 x 500 13.2 / 13.7; batches 2 x 1999 33 / 30, 8 x 1300, 16 / 2 48 / 39.)
  constexpr int KT = D == 128 ? 1 : 2;
  using G = AttnKeySteps<D, KT>;
  constexpr float LAZY = KT == 1 ? 4.f : 8.f;
  __shared__ __attribute__((aligned(1024))) char smem[G::LDS];  // one LDS object (see attn_smem_note)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const TrLane tr(lane);
  const int row = blockIdx.y;
  int hq, qb;
  if (!attn_block(p.Hq, p.Hkv, p.nQb, attn_row(p.order, p.plan_stride, row), true, hq, qb)) return;
  const int hkv = hq / (p.Hq / p.Hkv);
  const int q = qb * ATT_BM + wave * 32 + n;
  const int qc = q < p.S ? q : p.S - 1;  // queries past the end compute something that is not stored
  const int* const gc = attn_row(p.gc, p.plan_stride, row);
  const uint32_t* const list = attn_row(p.list, p.plan_stride, row) + (int64_t)qb * p.nKb;
  G ks;
  ks.begin(smem, p.K + row * p.k_bs + (int64_t)hkv * p.k_hs, p.k_ss, p.V + row * p.v_bs + (int64_t)hkv * p.v_hs, p.v_ss, p.S,
           gc, list, attn_row(p.cnt, p.plan_stride, row)[qb], wave, lane);

  // this lane's query as B-operand fragments of S^T = K Q^T
  bf16x8 qf[D / 16];
  {
    const uint16_t* qp = p.Q + row * p.q_bs + (int64_t)qc * p.q_ss + (int64_t)hq * p.q_hs + 8 * h;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qf[s] = *(const bf16x8*)(qp + 16 * s);
  }
  int gi = gc[q], pi = attn_row(p.pc, p.plan_stride, row)[q];

  floatx16 o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[dt][j] = 0.f;
  float m_run = -1e30f, l_run = 0.f;

#pragma unroll
  for (int s = 0; s < D / 16; ++s) pin_loaded(qf[s]);
  pin_loaded(gi);
  pin_loaded(pi);
  int bk = frag_base<D>(n, h);     // of the stage at hand
  TrBase bt = tr_base<D>(tr, 0);
  bt.lo += G::V_OFF;
  bt.hi += G::V_OFF;
  int stage = 0;
  wait_vmcnt<0>();
  barrier_lds_only();
  int fresh = 64;  // keys until the reference of the exponentials follows lazily
  while (ks.cur < ks.n) {
    const uint32_t ahead = ks.ahead(smem);
    const int key0 = ks.key(), active = ks.any(wave), partial = ks.mixed(wave);
    pin_loaded(bk);  // (or what follows from them is kept in registers of its own)
    pin_loaded(bt.lo);
    pin_loaded(bt.hi);
    if (active) {
      const int* const codes = (const int*)(smem + stage * G::STAGE + G::CODE_OFF);
      // S^T tiles: 32 keys each x this wave's 32 queries
      floatx16 sc[KT];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 16; ++j) sc[kt][j] = 0.f;
      {
        // K fragments PF steps ahead of the MFMAs that use them (LDS latency)
        constexpr int NS = D / 16, PF = KT == 1 ? 4 : 3;
        bf16x8 kf[NS][KT];
#pragma unroll
        for (int s = 0; s < PF; ++s)
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) kf[s][kt] = frag_at(smem + 32 * kt * T::ROW, bk, s);
        __builtin_amdgcn_sched_group_barrier(0x100, KT * PF, 0);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (s + PF < NS)
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) kf[s + PF][kt] = frag_at(smem + 32 * kt * T::ROW, bk, s + PF);
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
            sc[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s][kt], qf[s], sc[kt], 0, 0, 0);
          if (s + PF < NS) __builtin_amdgcn_sched_group_barrier(0x100, KT, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, KT, 0);
        }
      }

      // mask, running max (of the raw scores: the scale is positive and rides in the exponent's
      // multiply-add below)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        if (partial >> kt & 1) {
          // Mostly it is the queries that differ: the wave with the end of a completion in it goes through all its tiles
          // like this, and where its list is the longest the launch waits for it.  So where the 32 keys share their code and
          // come before the queries, one test per lane is enough, and otherwise the codes are read together.  Forward in us,
          // steps of 64 keys / of 32 with a test per element and read / this: 8192 positions of one conversation that does not
          // end with the row, 16 / 2 heads, 299 / 347 / 293; 5284 of 5 x (109 + 5 x 157) 35.6 / 39.7 / 35.1; 2314 of 246 +
          // 2 x 851, 28 / 4 heads, 43.1 / 47.4 / 41.1; the header's row 150 / 129 / 129.  (In steps of 64 it costs short lists 2 %.)
          if (KT == 1) {
            const int code = codes[n];
            const int c = __builtin_amdgcn_readfirstlane(code);
            if (__all(code == c) && key0 + 32 <= qb * ATT_BM + wave * 32) {
              const bool seen = gi == c || pi == c;
#pragma unroll
              for (int j = 0; j < 16; ++j) sc[kt][j] = seen ? sc[kt][j] : -INFINITY;
              continue;
            }
          }
          int4 kc[4];
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) kc[g4] = *(const int4*)(codes + 32 * kt + 8 * g4 + 4 * h);
          if (KT == 1)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {  // (or they are read one after the other)
              pin_loaded(kc[g4].x);
              pin_loaded(kc[g4].y);
              pin_loaded(kc[g4].z);
              pin_loaded(kc[g4].w);
            }
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) {
            const int key = key0 + 32 * kt + 8 * g4 + 4 * h;
            const int kcv[4] = {kc[g4].x, kc[g4].y, kc[g4].z, kc[g4].w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (!attn_visible(q, key + e, gi, pi, kcv[e])) sc[kt][4 * g4 + e] = -INFINITY;
          }
        }
      float mloc = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 16; ++j) mloc = fmaxf(mloc, sc[kt][j]);
      {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
        mloc = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * p.scale_log2e;  // both halves of a query
      }
      // The reference of the exponentials follows the running maximum lazily: it moves only when
      // some query of the wave has a score more than LAZY (in units of log2) above it, so the
      // 64 output accumulators are rescaled on few tiles instead of on most early ones.  Until
      // then exponentials are at most 2^LAZY, which fp32 sums and bf16 operands hold without
      // loss; the final division by the sum is the same.
      // It follows at once over a wave's first 64 keys: the term at the reference is 1 and has no rounding error (out
      // against 64 bits on dense rows 2.122e-3, and 2.137e-3 if it follows over the first 32 alone).
      // For the same reason steps of 32 keys follow from 2^4 on: a move that the first half of 64 keys causes does not see the
      // maximum of the second.  out against 64 bits in steps of 64 / of 32 with 2^8 / of 32 with 2^4, 16384 packed positions, 28 / 4
      // heads: normal q and k 2.191e-3 / 2.141e-3 / 2.140e-3 (145 us / 145 us in steps of 32), q four times as large 2.028e-3 /
      // 2.063e-3 / 1.837e-3 (144 / 146).
      const bool move = __any(mloc > m_run + (fresh > 0 ? 0.f : LAZY));
      fresh -= 32 * KT;
      if (move) {
        const float m_new = fmaxf(m_run, mloc);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
          for (int j = 0; j < 16; ++j) o[dt][j] *= alpha;
      }
      float lsum = 0.f;
      bf16x8 pf[2 * KT];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kt][j], p.scale_log2e, -m_run));
          lsum += e;
          pf[2 * kt + j / 8][j % 8] = (__bf16)e;
        }
      l_run += lsum;

      // O^T += V^T P^T, V^T fragments by transposing reads of the V tile
#pragma unroll
      for (int s2 = 0; s2 < 2 * KT; ++s2) {
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_at<D>(smem, bt, s2, dt), pf[s2], o[dt], 0, 0, 0);
      }
    }
    const int step = stage ? -G::STAGE : G::STAGE;
    bk += step;
    bt.lo += step;
    bt.hi += step;
    ks.end(smem, stage, ahead, wave, lane);
    stage ^= 1;
  }

  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (q >= p.S) return;  // (both lanes of a query)
  uint16_t* op = p.O + row * p.o_bs + (int64_t)q * p.o_ss + (int64_t)hq * p.o_hs;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
#pragma unroll
    for (int j = 0; j < 16; ++j) o[dt][j] *= inv;
    store_block_bf16(op + 32 * dt, o[dt], h);
  }
  if (h == 0) p.lse[((int64_t)row * p.Hq + hq) * p.S + q] = (m_run + __builtin_amdgcn_logf(l_tot)) * LN2;
}

// ----------------------------------------------------------------------------
// Backward
//   P = exp(scale * S + bias - lse),  dV = P^T dO,  dP = dO V^T,
//   dS = P o (dP - delta),  delta_i = sum_d dO[i,d] O[i,d],
//   dQ = scale * dS K,  dK = scale * dS^T Q.
// Two kernels, both free of atomics (bit-reproducible): one owns a block of
// keys and accumulates dK, dV over the query tiles that see it, the other owns
// a block of queries and accumulates dQ over its visible key tiles.  Each
// recomputes P from lse.
// ----------------------------------------------------------------------------
// How many heads of a group one dK/dV work-group takes for a key block with cnt query tiles.
// A step is one (query tile, head); a work-group that takes all heads of a group writes dK and dV directly,
// shares write fp32 partial sums.  So shares are as large as still lets the launch fill the GPU evenly: 5/4 of the
// steps that a resident work-group gets on average, two thirds where the key blocks alone are at least two rounds of
// work-groups.  Forward and backward in us by the divisor of that average (tenths), one round, work-groups numbered share
// by share (attn_kv_item):
//   16384 positions, 8 prompts of 137 + 4 x 461, 16 / 2 heads of 128:  40: 419, 30: 414, 15: 402, 8: 376, 6: 410
//   8192 positions, 28 / 4 heads:                                      40: 374, 30: 361, 15: 345, 8: 322, 6: 354
//   12000 positions, 28 / 4 heads                                      40: 520, 12: 463, 8: 473, 6: 523
//   16384 positions, 14 / 2 heads of 64:                               40: 217, 15: 207, 8: 202, 6: 205
// A launch that fits the GPU at once (not numbered) hardly depends on it: 2 rows of 1009 positions, 16 / 2 heads, 40: 88, 15: 88, 8: 87,
// 4: 86; 2700, 14 / 2 heads of 64, 118, 118, 117, 116.
// two rounds, 16384 positions, 28 / 4 heads (numbered by head):  6: 629, 15: 595, 40: 623, 100: 707 (backward).
// A share also costs evenness: its steps come in pieces that the dispatch order (longest list first) does not rank.
// Where the lists are long on average the set-up is small against one head's steps, and every work-group takes one
// head: from 24 tiles on where the key blocks are one round (16 where they are less), from 100 on where they are two (there
// the partial sums of all heads weigh more).  us, shares / one head each, by the average list:
//   less than a round: 19: 423 / 407 (4096 positions, 28 / 4 heads), 20: 313 / 303 (4096, 16 / 2), 24: 540 / 529 (16384, 14 / 2
//     of 64), 39: 1375 / 1342 (8192, 28 / 4), 64: 1326 / 1267 (8192, 16 / 2)
//   a round: 20: 1079 / 1175 (12000, 28 / 4), 29: 1180 / 1201 (16384, 16 / 2), 32: 719 / 591 (4096, 28 / 4, backward and forward)
//   two rounds (16384, 28 / 4): 19: 1416 / 1590, 30: 2055 / 2230, 72: 4700 / 4820, 128: 8207 / 8139
struct AttnKvSplit {
  const int* total;  // steps of one head, from the plan
  int long_total;    // total from which lists are long
  int heads_all;     // query heads
  int div;           // steps of a share = total * heads_all / div
  int light_max;     // >= 0 (artk_attn_bwd_tuning): all heads where they make at most this many steps, else one
  bool packed;       // work-groups are numbered share by share (attn_kv_item)
  __device__ __forceinline__ bool one_head(int64_t stride, int row) const {  // every work-group of the row takes one head
    return light_max < 0 && *attn_row(total, stride, row) >= long_total;
  }
  __device__ __forceinline__ int heads(int cnt, int rep, int64_t stride, int row) const {
    if (light_max >= 0) return cnt * rep <= light_max ? rep : 1;
    const int all = *attn_row(total, stride, row);
    if (all >= long_total) return 1;
    const int steps = (int)((int64_t)all * heads_all / div);
    int g = cnt > 0 ? steps / cnt : rep;
    g = g < 1 ? 1 : (g > rep ? rep : g);
    const int groups = (rep + g - 1) / g;
    return (rep + groups - 1) / groups;   // even shares
  }
};

// (first query head, key block) of a work-group of the dK/dV kernel whose number on its XCD is `item`: the shares of its XCD's
// units (as in attn_block) in their order, none left out.  A grid has room for a work-group per head; numbered by head,
// those without a share lie between the others, and each holds its place on a CU for about 3 us (16384 positions of 8
// prompts of 137 + 4 x 461, 28 / 4 heads: 5832 of 7168).  Numbered like this they come last.  The search costs a work-group
// a microsecond, so it is for grids that do not fit the GPU at once.  It takes one unit per thread; fewer than two rounds of key
// blocks are at most 192 units per XCD.  `scratch`: 8 words of LDS.  False: no share left.
constexpr int ATT_KV_UNITS = 256;
__device__ __forceinline__ bool attn_kv_item(int Hq, int Hkv, int nKb, const int* order, const int* cnt, const AttnKvSplit& split,
                                             int64_t stride, int row, int item, uint32_t* scratch, int& hq, int& kb) {
  const int rep = Hq / Hkv, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int unit = (int)threadIdx.x * 8 + (blockIdx.x & 7), rank = unit / Hkv;
  int b = 0, per = 1, shares = 0;
  if (rank < nKb) {
    b = order[rank];
    per = split.heads(cnt[b], rep, stride, row);
    shares = (rep + per - 1) / per;
  }
  int end = shares;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(end, d, 64);
    if (lane >= d) end += v;
  }
  if (lane == 63) scratch[wave] = (uint32_t)end;
  __syncthreads();
  const int total = (int)(scratch[0] + scratch[1] + scratch[2] + scratch[3]);
  if (item >= total) return false;
  for (int w = 0; w < wave; ++w) end += (int)scratch[w];
  const int at = item - (end - shares);
  if (at >= 0 && at < shares) {
    scratch[4] = (uint32_t)((unit % Hkv) * rep + at * per);
    scratch[5] = (uint32_t)b;
  }
  __syncthreads();
  hq = __builtin_amdgcn_readfirstlane((int)scratch[4]);
  kb = __builtin_amdgcn_readfirstlane((int)scratch[5]);
  __syncthreads();
  return true;
}

// 32 rows of a head as the operand fragments of one wave (lane (n, h): row n, 8 columns from 16 s + 8 h on).  Loaded row by
// row, so that an instruction reads whole cache lines, and handed round through LDS of the wave's own: in fragment order an
// instruction touches 32 rows for 32 bytes each, and the three operands of dQ take 9 us of a work-group's 40.  Backward in us,
// fragment order / this: 16384 packed positions, 28 / 4 heads 497 / 489, 16 / 2 heads 288 / 283; 4096, 28 / 4 159 / 157.
template <int D>
struct AttnWaveRows {
  using T = AttnTile<D>;
  static constexpr int BYTES = 32 * T::ROW, N = BYTES / 1024;
  bf16x8 v[N];
  __device__ __forceinline__ void load(const uint16_t* head, int64_t stride, int row0, int S, int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = row0 + T::row_of(i) + lane / T::CHK;
      v[i] = *(const bf16x8*)(head + (int64_t)(r < S ? r : S - 1) * stride + lane % T::CHK * 8);
    }
  }
  __device__ __forceinline__ void fragments(char* lds, int lane, bf16x8 (&f)[D / 16]) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = T::row_of(i) + lane / T::CHK;
      *(bf16x8*)(lds + r * T::ROW + ((lane % T::CHK) ^ T::swz(r)) * 16) = v[i];
    }
    __builtin_amdgcn_wave_barrier();  // (LDS operations of a wave complete in order)
#pragma unroll
    for (int s = 0; s < D / 16; ++s) f[s] = T::row_frag(lds, lane & 31, s, lane >> 5);
    __builtin_amdgcn_wave_barrier();
  }
};

struct AttnBwdParams {
  const uint16_t *Q, *K, *V, *dO;
  const uint16_t* O;
  const float* lse;                 // [Hq][S]
  float* lse2;                      // [Hq][Sp]  lse * log2(e), Sp = S rounded up to a multiple of 256
  float* delta;                     // [Hq][Sp]
  uint16_t *dQ, *dK, *dV;
  float *pK, *pV;                   // [rows of the launch][Hq/Hkv][Sp][Hkv][D] partial sums per share (grouped-query
                                    // heads only)
  int row0;                         // dK/dV kernel and its reduction: first row of the launch
  int64_t plan_stride, q_bs, k_bs, v_bs, o_bs, do_bs, dq_bs, dk_bs, dv_bs;  // per row of the batch (blockIdx.y)
  int64_t o_ss, o_hs;
  int64_t q_ss, q_hs, k_ss, k_hs, v_ss, v_hs, do_ss, do_hs, dq_ss, dq_hs, dk_ss, dk_hs, dv_ss, dv_hs;
  const int* gc;
  const int* pc;
  const uint32_t* list;    // per query block of 128: key tiles of 64
  const int* cnt;
  const int* order;
  const uint32_t* listT;   // per key block of 64: query tiles of 64
  const int* cntT;
  const int* orderT;
  int S, Sp, Hq, Hkv, nQb, nKb, nQb2, nKb2;
  AttnKvSplit split;
  float scale, scale_log2e;
};

// ---- dQ: 128 queries x one head per work-group, lane = query ----------------
// Runs first and leaves delta and lse2 of its queries for the dK/dV kernel: it holds their dO anyway, so a
// pass of its own over O and dO (47 us for 16384 positions, 28 heads of 128) became a read of O.
template <int D>
__global__ __launch_bounds__(ATT_THREADS, D == 64 ? 3 : 2) void attn_bwd_dq_kernel(AttnBwdParams p) {
  using T = AttnTile<D>;
  using G = AttnKeySteps<D, 1>;
  using R = AttnWaveRows<D>;
  constexpr int ROWS_OFF = (G::LDS + 1023) / 1024 * 1024;
  __shared__ __attribute__((aligned(1024))) char smem[ROWS_OFF + 4 * R::BYTES];  // one LDS object (see attn_smem_note)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const TrLane tr(lane);
  const int row = blockIdx.y;
  int hq, qb;
  if (!attn_block(p.Hq, p.Hkv, p.nQb, attn_row(p.order, p.plan_stride, row), true, hq, qb)) return;
  const int hkv = hq / (p.Hq / p.Hkv);
  const int q = qb * ATT_BM + wave * 32 + n;
  const int qc = q < p.S ? q : p.S - 1;  // queries past the end compute something that is not stored
  const int* const gc = attn_row(p.gc, p.plan_stride, row);
  const uint32_t* const list = attn_row(p.list, p.plan_stride, row) + (int64_t)qb * p.nKb;
  G ks;
  ks.begin(smem, p.K + row * p.k_bs + (int64_t)hkv * p.k_hs, p.k_ss, p.V + row * p.v_bs + (int64_t)hkv * p.v_hs, p.v_ss, p.S,
           gc, list, attn_row(p.cnt, p.plan_stride, row)[qb], wave, lane);

  // Q, dO and O of this wave's queries as B-operand fragments
  bf16x8 qf[D / 16], dof[D / 16];
  float delta = 0.f;
  {
    const int q0 = qb * ATT_BM + wave * 32;
    R rq, rg, ro;
    rg.load(p.dO + row * p.do_bs + (int64_t)hq * p.do_hs, p.do_ss, q0, p.S, lane);
    ro.load(p.O + row * p.o_bs + (int64_t)hq * p.o_hs, p.o_ss, q0, p.S, lane);
    rq.load(p.Q + row * p.q_bs + (int64_t)hq * p.q_hs, p.q_ss, q0, p.S, lane);
    char* const own = smem + ROWS_OFF + wave * R::BYTES;
    bf16x8 of[D / 16];
    rg.fragments(own, lane, dof);
    ro.fragments(own, lane, of);
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) delta += (float)of[s][e] * (float)dof[s][e];
    rq.fragments(own, lane, qf);
  }
  delta += __shfl_xor(delta, 32, 64);
  int gi = gc[q], pi = attn_row(p.pc, p.plan_stride, row)[q];
  float nlse2 = -LOG2E * p.lse[((int64_t)row * p.Hq + hq) * p.S + qc];
  if (h == 0) {
    const int64_t o = ((int64_t)row * p.Hq + hq) * p.Sp + q;
    p.lse2[o] = -nlse2;
    p.delta[o] = q < p.S ? delta : 0.f;
  }

  floatx16 dq[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) dq[dt][j] = 0.f;

#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    pin_loaded(qf[s]);
    pin_loaded(dof[s]);
  }
  pin_loaded(gi);
  pin_loaded(pi);
  pin_loaded(nlse2);
  pin_loaded(delta);
  int bk = frag_base<D>(n, h);     // of the stage at hand
  TrBase bt = tr_base<D>(tr, 0);
  int stage = 0;
  wait_vmcnt<0>();
  barrier_lds_only();
  while (ks.cur < ks.n) {
    const uint32_t ahead = ks.ahead(smem);
    const int key0 = ks.key(), active = ks.any(wave), partial = ks.mixed(wave);
    const int* codes = (const int*)(smem + stage * G::STAGE + G::CODE_OFF);
    pin_loaded(bk);  // (or what follows from them is kept in registers of its own)
    pin_loaded(bt.lo);
    pin_loaded(bt.hi);
    if (active) {
      floatx16 sc, dp;
#pragma unroll
      for (int j = 0; j < 16; ++j) sc[j] = dp[j] = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; ++s) {
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_at(smem, bk, s), qf[s], sc, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_at(smem + G::V_OFF, bk, s), dof[s], dp, 0, 0, 0);
      }
      // the mask comes behind the multiply-add: whatever a query's lse and the scale are, P is 0 where it sees nothing
#pragma unroll
      for (int j = 0; j < 16; ++j) sc[j] = __builtin_fmaf(sc[j], p.scale_log2e, nlse2);
      if (partial) {  // one branch for all elements: tested inside the loop below it becomes one per element
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const int kk = 8 * g4 + 4 * h;
          const int4 kc = *(const int4*)(codes + kk);
          const int kcv[4] = {kc.x, kc.y, kc.z, kc.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (!attn_visible(q, key0 + kk + e, gi, pi, kcv[e])) sc[4 * g4 + e] = -INFINITY;
        }
      }
      bf16x8 dsf[2];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float pr = __builtin_amdgcn_exp2f(sc[j]);
        dsf[j / 8][j % 8] = (__bf16)(pr * (dp[j] - delta));
      }
      // dQ^T += K^T dS^T, K^T fragments by transposing reads of the K tile
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          dq[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_at<D>(smem, bt, s2, dt), dsf[s2], dq[dt], 0, 0, 0);
      }
    }
    const int step = stage ? -G::STAGE : G::STAGE;
    bk += step;
    bt.lo += step;
    bt.hi += step;
    ks.end(smem, stage, ahead, wave, lane);
    stage ^= 1;
  }
  if (q >= p.S) return;
  uint16_t* op = p.dQ + row * p.dq_bs + (int64_t)q * p.dq_ss + (int64_t)hq * p.dq_hs;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
#pragma unroll
    for (int j = 0; j < 16; ++j) dq[dt][j] *= p.scale;
    store_block_bf16(op + 32 * dt, dq[dt], h);
  }
}

// ---- dK, dV: 64 keys x some query heads of a group per work-group, lane = key ------------
// 4 wavefronts = 2 key groups of 32 x 2 halves of each 64-query tile; two work-groups per CU (D = 64:
// three), so that the exp2 / convert work, the DMA latency and the set-up of one overlap the MFMAs of the
// other.  The two waves of a key group keep separate accumulators, added through LDS at the end.
// Bound: LDS reads, exp2 and the MFMAs, which two waves of a SIMD overlap in part.  The wave's K rows and the upper half of
// its V rows (D = 128) stay in registers for the whole kernel: 36 KiB of fragments per step of 32 MFMAs instead of 48, and
// room in LDS for a second stage, so that a query tile comes in during the step before instead of between two barriers of
// its own.  The registers for that come from one per fragment row instead of one per address, and from P before dP (half
// the fragments in flight).  One stage, V rows all in LDS / now, backward in us: dense causal rows of 16384 positions,
// 28 / 4 heads of 128: 6640 / 6280; 8192, 16 / 2: 1000 / 976; 8192, 14 / 2 heads of 64: 518 / 465; the row of the header's
// figures 570 / 525 (dQ and both masks as one branch per step instead of one per element included).  Offsets that move with
// the stage instead of a sum per read: 6400 -> 6330 on the dense row.
// A work-group that does not take all heads of its group writes fp32 partial sums, which
// attn_kv_reduce_kernel adds in a fixed order.
// LDS: two stages of a Q tile, a dO tile (64 queries) and lse2 / delta / group / parent codes of those queries; then
// columns 0 .. 63 of the block's V rows.  The K rows and what is left of the V rows pass through the second stage on
// their way to registers.
template <int D>
struct AttnQStage {
  using T = AttnTile<D>;
  using TV = AttnTile<64>;
  static constexpr int DO_OFF = T::BYTES;
  static constexpr int ROW_OFF = 2 * T::BYTES;
  static constexpr int STAGE = ROW_OFF + 1024;
  static constexpr int V_OFF = 2 * STAGE;
  static constexpr int LDS = V_OFF + TV::BYTES;
  static constexpr int VR = D / 16 - 4;                  // 16-column steps of V in registers
};

// DMA of one query tile into a stage: this wave's share of the Q and dO tiles and
// one of the four per-query arrays (wave 0: lse2, 1: delta, 2: group codes, 3: parent codes).
// row_q, row_do, chunk: this lane's row and chunk in instruction 0, in bytes (AttnTile::row_of).
template <int D>
__device__ __forceinline__ void attn_issue_q(char* st, int hq, int q0, const uint16_t* q_row, const uint16_t* do_row,
                                             dma_rsrc_t rsrc_row, int row_q, int row_do, int chunk, const AttnBwdParams& p, int wave,
                                             int lane) {
  using T = AttnTile<D>;
  using G = AttnQStage<D>;
  const dma_rsrc_t rsrc_q = attn_head_rsrc<D>(q_row + hq * p.q_hs, p.q_ss, p.S);
  const dma_rsrc_t rsrc_do = attn_head_rsrc<D>(do_row + hq * p.do_hs, p.do_ss, p.S);
#pragma unroll
  for (int i = 0; i < T::N4; ++i) {
    const int r = T::row_of(wave * T::N4 + i), c = T::chunk_of(chunk, wave * T::N4 + i);
    dma_load16(rsrc_q, row_q + c, (int)((q0 + r) * p.q_ss * 2), lds_addr_of(st + (wave * T::N4 + i) * 1024));
    dma_load16(rsrc_do, row_do + c, (int)((q0 + r) * p.do_ss * 2), lds_addr_of(st + G::DO_OFF + (wave * T::N4 + i) * 1024));
  }
  const int arr = wave;
  dma_load4(rsrc_row, lane * 4, (int)(((arr < 2 ? (int64_t)hq * p.Sp : 0) + q0) * 4), lds_addr_of(st + G::ROW_OFF + arr * 256));
}

// DMA of 64 rows from row0 on of one head into an LDS tile of D columns.
template <int D>
__device__ __forceinline__ void attn_issue_block(char* dst, int row0, dma_rsrc_t rsrc, int64_t stride, int wave, int lane) {
  using T = AttnTile<D>;
#pragma unroll
  for (int i = 0; i < T::N4; ++i)
    dma_load16(rsrc, T::voff(wave * T::N4 + i, lane, stride), (int)(row0 * stride * 2),
               lds_addr_of(dst + (wave * T::N4 + i) * 1024));
}

template <int D>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void attn_bwd_kv_kernel(AttnBwdParams p) {
  using T = AttnTile<D>;
  using G = AttnQStage<D>;
  // one LDS object for the stages and the tile list (see attn_smem_note)
  __shared__ __attribute__((aligned(1024))) char smem[G::LDS + ATT_MAX_KB * 4];
  uint32_t* const s_list = (uint32_t*)(smem + G::LDS);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int kg = wave & 1, qh = wave >> 1;
  const TrLane tr(lane);
  const int brow = p.row0 + blockIdx.y;
  const int rep = p.Hq / p.Hkv;
  const int* const order = attn_row(p.orderT, p.plan_stride, brow);
  const int* const counts = attn_row(p.cntT, p.plan_stride, brow);
  const bool packed = p.split.packed && !p.split.one_head(p.plan_stride, brow);
  int hq, kb;
  if (packed ? !attn_kv_item(p.Hq, p.Hkv, p.nKb2, order, counts, p.split, p.plan_stride, brow, blockIdx.x >> 3, s_list, hq, kb)
             : !attn_block(p.Hq, p.Hkv, p.nKb2, order, false, hq, kb))
    return;
  const int hkv = hq / rep;
  const int key = kb * ATT_BK2 + kg * 32 + n;
  const int cnt = counts[kb];
  const int per = p.split.heads(cnt, rep, p.plan_stride, brow);
  int share = hq - hkv * rep;
  if (packed) share /= per;
  if (share * per >= rep) return;
  hq = hkv * rep + share * per;  // first head of this work-group's share
  const int nheads = rep - share * per < per ? rep - share * per : per;
  const int* const gc = attn_row(p.gc, p.plan_stride, brow);
  const uint32_t* const list = attn_row(p.listT, p.plan_stride, brow) + (int64_t)kb * p.nQb2;
  for (int i = threadIdx.x; i < cnt; i += 256) s_list[i] = list[i];
  int gk = gc[key];

  const uint16_t* const q_row = p.Q + brow * p.q_bs;
  const uint16_t* const do_row = p.dO + brow * p.do_bs;
  const int arr = wave;
  const int64_t stat_row = (int64_t)brow * p.Hq * p.Sp;
  const void* row_src = arr == 0 ? (const void*)(p.lse2 + stat_row) : arr == 1 ? (const void*)(p.delta + stat_row)
                        : arr == 2 ? (const void*)gc : (const void*)attn_row(p.pc, p.plan_stride, brow);
  const dma_rsrc_t rsrc_row = attn_rsrc(row_src);
  int row_q = T::lane_row(lane, p.q_ss), row_do = T::lane_row(lane, p.do_ss), chunk = T::lane_chunk(lane);
  {
    const uint16_t* const k_head = p.K + brow * p.k_bs + (int64_t)hkv * p.k_hs;
    const uint16_t* const v_head = p.V + brow * p.v_bs + (int64_t)hkv * p.v_hs;
    attn_issue_block<D>(smem + G::STAGE, kb * ATT_BK2, attn_head_rsrc<D>(k_head, p.k_ss, p.S), p.k_ss, wave, lane);
    attn_issue_block<64>(smem + G::V_OFF, kb * ATT_BK2, attn_head_rsrc<64>(v_head, p.v_ss, p.S), p.v_ss, wave, lane);
    if constexpr (D > 64)
      attn_issue_block<D - 64>(smem + G::STAGE + T::BYTES, kb * ATT_BK2, attn_head_rsrc<D - 64>(v_head + 64, p.v_ss, p.S),
                               p.v_ss, wave, lane);
  }
  const int total = cnt * nheads;
  if (total > 0)  // the first tile of the flattened (head, visible query tile) sequence
    attn_issue_q<D>(smem, hq, __builtin_amdgcn_readfirstlane(list[0] & 0x3fff) * ATT_BQ2, q_row, do_row, rsrc_row,
                    row_q, row_do, chunk, p, wave, lane);

  floatx16 dk[D / 32], dv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) dk[dt][j] = dv[dt][j] = 0.f;

  pin_loaded(gk);
  wait_vmcnt<0>();
  barrier_lds_only();  // the list, the block's K and V rows and the first tile are there
  const char* const vblk = smem + G::V_OFF;
  const int krow = 32 * kg + n;  // this wave's keys inside the block
  bf16x8 kf[D / 16], vr[G::VR > 0 ? G::VR : 1];
#pragma unroll
  for (int s = 0; s < D / 16; ++s) kf[s] = T::row_frag(smem + G::STAGE, krow, s, h);
#pragma unroll
  for (int s = 0; s < G::VR; ++s) vr[s] = G::TV::row_frag(smem + G::STAGE + T::BYTES, krow, s, h);
#pragma unroll
  for (int s = 0; s < D / 16; ++s) pin_loaded(kf[s]);
#pragma unroll
  for (int s = 0; s < G::VR; ++s) pin_loaded(vr[s]);
  int bq = frag_base<D>(32 * qh + n, h), bv = frag_base<64>(krow, h);
  TrBase bt = tr_base<D>(tr, 32 * qh);
  bq += G::STAGE;
  bt.lo += G::STAGE;
  bt.hi += G::STAGE;
  int ti = 0, head = hq;
  for (int it = 0; it < total; ++it) {
    const int step = it & 1 ? G::STAGE : -G::STAGE;
    bq += step;
    bt.lo += step;
    bt.hi += step;
    wait_vmcnt<0>();
    barrier_lds_only();  // this tile is there, and every wave is done with the one before (it = 0: with the K and V rows)
    const int entry = __builtin_amdgcn_readfirstlane(s_list[ti]);
    if (++ti == cnt) {
      ti = 0;
      ++head;
    }
    pin_loaded(row_q);  // (or what follows from them is kept in registers of its own; so below)
    pin_loaded(row_do);
    pin_loaded(chunk);
    if (it + 1 < total)
      attn_issue_q<D>(smem + ((it + 1) & 1) * G::STAGE, head, __builtin_amdgcn_readfirstlane(s_list[ti] & 0x3fff) * ATT_BQ2,
                      q_row, do_row, rsrc_row, row_q, row_do, chunk, p, wave, lane);
    const char* const st = smem + (it & 1) * G::STAGE;
    const int q0 = (entry & 0x3fff) * ATT_BQ2;
    const bool active = (entry >> (16 + wave)) & 1;        // this wave's keys x query half
    const bool partial = !((entry >> (24 + wave)) & 1);
    const char* dot = smem + G::DO_OFF;  // (bq and bt move with the stage)
    const float* r_lse2 = (const float*)(st + G::ROW_OFF);
    const float* r_delta = r_lse2 + 64;
    const int* r_gc = (const int*)(r_lse2 + 128);
    const int* r_pc = r_gc + 64;
    if (!active) continue;
    pin_loaded(bq);
    pin_loaded(bv);
    pin_loaded(bt.lo);
    pin_loaded(bt.hi);

    constexpr int NS = D / 16;
    floatx16 sc, dp;
#pragma unroll
    for (int j = 0; j < 16; ++j) sc[j] = dp[j] = 0.f;
    {
      // fragments PF steps ahead of the MFMAs that use them (LDS latency; more would not fit the registers)
      constexpr int PF = 3;
      bf16x8 qf[NS];
#pragma unroll
      for (int s = 0; s < PF; ++s) qf[s] = frag_at(smem, bq, s);
      __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if (s + PF < NS) qf[s + PF] = frag_at(smem, bq, s + PF);
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[s], kf[s], sc, 0, 0, 0);
        if (s + PF < NS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    }
    // the mask comes behind the multiply-add: whatever a query's lse and the scale are, P is 0 where it sees nothing
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const floatx4 l4 = *(const floatx4*)(r_lse2 + 32 * qh + 8 * g4 + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[4 * g4 + e] = __builtin_fmaf(sc[4 * g4 + e], p.scale_log2e, -l4[e]);
    }
    if (partial) {  // one branch for all elements: tested inside the loop below it becomes one per element
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int qi = 32 * qh + 8 * g4 + 4 * h;
        const int4 a4 = *(const int4*)(r_gc + qi);
        const int4 b4 = *(const int4*)(r_pc + qi);
        const int gq[4] = {a4.x, a4.y, a4.z, a4.w}, pq[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (!attn_visible(q0 + qi + e, key, gq[e], pq[e], gk)) sc[4 * g4 + e] = -INFINITY;
      }
    }
    {
      constexpr int PF = 2;
      bf16x8 of[NS], vf[NS];
#pragma unroll
      for (int s = 0; s < PF; ++s) {
        of[s] = frag_at(dot, bq, s);
        vf[s] = frag_at(vblk, bv, s);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * PF, 1);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if (s + PF < NS) {
          of[s + PF] = frag_at(dot, bq, s + PF);
          vf[s + PF] = s + PF < 4 ? frag_at(vblk, bv, s + PF) : vr[s + PF < 4 ? 0 : s + PF - 4];
        }
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(of[s], vf[s], dp, 0, 0, 0);
        if (s + PF < 4) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        else if (s + PF < NS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      }
    }
    bf16x8 pf[2], dsf[2];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int qi = 32 * qh + 8 * g4 + 4 * h;
      const floatx4 d4 = *(const floatx4*)(r_delta + qi);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 4 * g4 + e;
        const float pr = __builtin_amdgcn_exp2f(sc[j]);
        pf[j / 8][j % 8] = (__bf16)pr;
        dsf[j / 8][j % 8] = (__bf16)(pr * (dp[j] - d4[e]));
      }
    }
    // dV^T += dO^T P, dK^T += Q^T dS: transposing reads of the dO and Q tiles
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) {
        dv[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_at<D>(dot, bt, u, dt), pf[u], dv[dt], 0, 0, 0);
        dk[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_at<D>(smem, bt, u, dt), dsf[u], dk[dt], 0, 0, 0);
      }
    }
  }

  // add the accumulators of the two query halves: the upper waves park theirs in
  // LDS ([key group][register][lane], conflict-free), the lower waves add and store
  float* red = (float*)smem;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    __syncthreads();
    if (qh == 1) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          red[((kg * (D / 2) + dt * 16 + j) << 6) + lane] = pass == 0 ? dk[dt][j] : dv[dt][j];
    }
    __syncthreads();
    if (qh == 0) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float v = red[((kg * (D / 2) + dt * 16 + j) << 6) + lane];
          if (pass == 0) dk[dt][j] += v; else dv[dt][j] += v;
        }
    }
  }
  if (qh == 1 || key >= p.S) return;

  if (per < rep) {
    const int64_t o = (((((int64_t)blockIdx.y * rep + share) * p.Sp + key) * p.Hkv + hkv) * D) + 4 * h;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        floatx4 a, b;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[e] = dk[dt][4 * g4 + e];
          b[e] = dv[dt][4 * g4 + e];
        }
        *(floatx4*)(p.pK + o + 32 * dt + 8 * g4) = a;
        *(floatx4*)(p.pV + o + 32 * dt + 8 * g4) = b;
      }
    return;
  }
  uint16_t* kp = p.dK + brow * p.dk_bs + (int64_t)key * p.dk_ss + (int64_t)hkv * p.dk_hs + 4 * h;
  uint16_t* vp = p.dV + brow * p.dv_bs + (int64_t)key * p.dv_ss + (int64_t)hkv * p.dv_hs + 4 * h;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      bf16x4 a, b;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = (__bf16)(dk[dt][4 * g4 + e] * p.scale);
        b[e] = (__bf16)dv[dt][4 * g4 + e];
      }
      *(bf16x4*)(kp + 32 * dt + 8 * g4) = a;
      *(bf16x4*)(vp + 32 * dt + 8 * g4) = b;
    }
}

// dK = scale * sum_r pK[r], dV = sum_r pV[r] over the shares r of a group's heads, in
// index order; 4 elements per thread.
__global__ __launch_bounds__(256) void attn_kv_reduce_kernel(AttnBwdParams p, int D) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int d4 = D / 4, brow = p.row0 + blockIdx.y, rep = p.Hq / p.Hkv;
  const int64_t n = (int64_t)p.Sp * p.Hkv * d4;
  const int c = (int)(i % d4);
  const int hh = (int)((i / d4) % p.Hkv);
  const int64_t s = i / ((int64_t)d4 * p.Hkv);
  if (s >= p.S) return;
  const int per = p.split.heads(attn_row(p.cntT, p.plan_stride, brow)[s / ATT_BK2], rep, p.plan_stride, brow);
  if (per == rep) return;  // written directly by the dK/dV kernel
  const floatx4* pk = (const floatx4*)p.pK + (int64_t)blockIdx.y * rep * n + i;
  const floatx4* pv = (const floatx4*)p.pV + (int64_t)blockIdx.y * rep * n + i;
  floatx4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
  for (int r = 0; r * per < rep; ++r) {
    a += pk[(int64_t)r * n];
    b += pv[(int64_t)r * n];
  }
  bf16x4 oa, ob;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    oa[e] = (__bf16)(a[e] * p.scale);
    ob[e] = (__bf16)b[e];
  }
  *(bf16x4*)(p.dK + brow * p.dk_bs + s * p.dk_ss + (int64_t)hh * p.dk_hs + 4 * c) = oa;
  *(bf16x4*)(p.dV + brow * p.dv_bs + s * p.dv_ss + (int64_t)hh * p.dv_hs + 4 * c) = ob;
}

}  // namespace artk

// Threshold override of artk_attn_bwd_tuning for calls made on this thread (-1: automatic).
static thread_local int g_light_max_override = -1;

using namespace artk;

extern "C" {

static int64_t attn_padded(int64_t S) { return (S + ATT_ROW - 1) / ATT_ROW * ATT_ROW; }

size_t artk_attn_plan_rows_bytes(int64_t B, int64_t S) {
  AttnPlan pl;
  attn_plan_layout(nullptr, 0, attn_padded(S), pl);
  return (size_t)(B * pl.stride) + 256;
}
size_t artk_attn_plan_row_stride(int64_t S) {
  AttnPlan pl;
  attn_plan_layout(nullptr, 0, attn_padded(S), pl);
  return (size_t)pl.stride;
}
size_t artk_attn_plan_bytes(int64_t S) { return artk_attn_plan_rows_bytes(1, S); }

static int32_t attn_check_len(int64_t B, int64_t S) {
  ARTK_CHECK_ARG(B > 0 && S > 0, "B and S must be positive");
  if (attn_padded(S) / ATT_BN > ATT_MAX_KB || B > 65535) {
    set_error("row length %lld must be at most %d (and the batch at most 65535 rows)", (long long)S, ATT_MAX_KB * ATT_BN);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  return ARTK_OK;
}
static int32_t attn_check_multiple(int64_t S) {
  if (S % ATT_ROW != 0 || S / ATT_BN > ATT_MAX_KB) {
    set_error("row length %lld must be a multiple of %d and at most %d", (long long)S, ATT_ROW,
              ATT_MAX_KB * ATT_BN);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  return ARTK_OK;
}

int32_t artk_attn_plan_rows(const int64_t* group_ids, const int64_t* parent_ids, int64_t B, int64_t S, void* plan,
                            size_t plan_bytes, artk_stream_t stream) {
  ARTK_CHECK_ARG(group_ids && parent_ids && plan, "null pointer argument");
  int32_t rc = attn_check_len(B, S);
  if (rc) return rc;
  AttnPlan pl;
  if (plan_bytes < artk_attn_plan_rows_bytes(B, S) ||
      attn_plan_layout(plan, plan_bytes, attn_padded(S), pl) == (size_t)-1) {
    set_error("plan buffer too small: need %zu bytes, got %zu", artk_attn_plan_rows_bytes(B, S), plan_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  const unsigned b = (unsigned)B;
  if (attn_padded(S) <= ATT_SHORT) {
    attn_plan_short_kernel<<<dim3((unsigned)pl.nQb, b), 1024, 0, st>>>(group_ids, parent_ids, (int)S, pl);
    ARTK_CHECK_LAUNCH();
    attn_plan_short_order_kernel<<<b, 1024, 0, st>>>(pl);
    ARTK_CHECK_LAUNCH();
    return ARTK_OK;
  }
  attn_heads_kernel<<<b, 1024, 0, st>>>(group_ids, (int)S, pl.stride, pl.heads, pl.n_heads);
  ARTK_CHECK_LAUNCH();
  attn_codes_kernel<<<dim3((unsigned)(attn_padded(S) / 256), b), 256, 0, st>>>(group_ids, parent_ids, (int)S, pl.stride,
                                                                              pl.heads, pl.n_heads, pl.gc, pl.pc,
                                                                              pl.uni);
  ARTK_CHECK_LAUNCH();
  attn_classify_kernel<<<dim3((unsigned)((pl.nKb + 3) / 4), (unsigned)pl.nQb, b), 256, 0, st>>>(
      pl.gc, pl.pc, pl.uni, pl.stride, pl.nKb, pl.nQb2, pl.info, pl.info2);
  ARTK_CHECK_LAUNCH();
  const AttnTable t1{pl.info, pl.list, pl.cnt, pl.nQb, pl.nKb}, t2{pl.info2, pl.list2, pl.cnt2, pl.nKb2, pl.nQb2};
  attn_compact_kernel<<<dim3((unsigned)(pl.nQb + pl.nKb2), b), 256, 0, st>>>(t1, t2, pl.stride);
  ARTK_CHECK_LAUNCH();
  attn_order_kernel<<<dim3(2, b), 1024, 0, st>>>(pl.cnt, pl.nQb, pl.order, pl.cnt2, pl.nKb2, pl.order2, pl.total2,
                                                 pl.stride);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

int32_t artk_attn_plan(const int64_t* group_ids, const int64_t* parent_ids, int64_t S, void* plan,
                       size_t plan_bytes, artk_stream_t stream) {
  ARTK_CHECK_ARG(group_ids && parent_ids && plan, "null pointer argument");
  ARTK_CHECK_ARG(S > 0, "S must be positive");
  int32_t rc = attn_check_multiple(S);
  if (rc) return rc;
  return artk_attn_plan_rows(group_ids, parent_ids, 1, S, plan, plan_bytes, stream);
}

// strides: (batch, position, head) of nt tensors, in elements.
static int32_t attn_check(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int32_t D, const int64_t* strides, int nt) {
  ARTK_CHECK_ARG(Hq > 0 && Hkv > 0, "S, Hq, Hkv must be positive");
  int32_t rc = attn_check_len(B, S);
  if (rc) return rc;
  if (D != 64 && D != 128) {
    set_error("head dimension %d is not supported (64 or 128)", D);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  if (Hq % Hkv != 0) {
    set_error("query heads (%d) must be a multiple of key/value heads (%d)", Hq, Hkv);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  for (int i = 0; i < nt; ++i) {
    const int64_t *s = strides + 3 * i;
    ARTK_CHECK_ARG(s[1] > 0 && s[1] % 8 == 0 && s[2] > 0 && s[2] % 8 == 0 && s[0] >= 0 && s[0] % 8 == 0,
                   "strides must be positive multiples of 8 elements");
    ARTK_CHECK_ARG(attn_padded(S) * s[1] * 2 < (1ll << 31), "operand spans 2 GiB or more");
  }
  return ARTK_OK;
}

size_t artk_attn_fwd_workspace_bytes(int64_t S, int32_t Hkv, int32_t D) {
  (void)S; (void)Hkv; (void)D;
  return 256;  // the forward needs no scratch; kept so that every op has the same calling pattern
}

int32_t artk_attn_fwd_rows(const void* q, const void* k, const void* v, const void* plan, int64_t B, int64_t S,
                           int32_t Hq, int32_t Hkv, int32_t D, const int64_t* strides, float scale, void* out,
                           float* lse, artk_stream_t stream) {
  ARTK_CHECK_ARG(q && k && v && plan && out && lse && strides, "null pointer argument");
  ARTK_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out),
                 "q, k, v, out must be 16-byte aligned");
  int32_t rc = attn_check(B, S, Hq, Hkv, D, strides, 4);
  if (rc) return rc;
  ARTK_CHECK_ARG(scale > 0.f && scale < INFINITY, "scale must be positive and finite");
  AttnPlan pl;
  attn_plan_layout(const_cast<void*>(plan), (size_t)1 << 40, attn_padded(S), pl);
  hipStream_t st = (hipStream_t)stream;
  AttnFwdParams p;
  p.Q = (const uint16_t*)q;
  p.K = (const uint16_t*)k;
  p.V = (const uint16_t*)v;
  p.O = (uint16_t*)out;
  p.lse = lse;
  p.q_bs = strides[0];  p.q_ss = strides[1];   p.q_hs = strides[2];
  p.k_bs = strides[3];  p.k_ss = strides[4];   p.k_hs = strides[5];
  p.v_bs = strides[6];  p.v_ss = strides[7];   p.v_hs = strides[8];
  p.o_bs = strides[9];  p.o_ss = strides[10];  p.o_hs = strides[11];
  p.gc = pl.gc;
  p.pc = pl.pc;
  p.list = pl.list;
  p.cnt = pl.cnt;
  p.order = pl.order;
  p.plan_stride = pl.stride;
  p.S = (int)S;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.nQb = pl.nQb;
  p.nKb = pl.nKb;
  p.scale_log2e = scale * LOG2E;
  const dim3 grid(attn_grid(Hq, Hkv, pl.nQb), (unsigned)B);
  prof_begin(PROF_ATTN_FWD, st);
  if (D == 128)
    attn_fwd_kernel<128><<<grid, ATT_THREADS, 0, st>>>(p);
  else
    attn_fwd_kernel<64><<<grid, ATT_THREADS, 0, st>>>(p);
  prof_end(PROF_ATTN_FWD, st);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

int32_t artk_attn_fwd(const void* q, const void* k, const void* v, const void* plan, int64_t S,
                      int32_t Hq, int32_t Hkv, int32_t D, int64_t q_stride_s, int64_t q_stride_h,
                      int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_s, int64_t v_stride_h,
                      int64_t o_stride_s, int64_t o_stride_h, float scale, void* out, float* lse,
                      void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  (void)workspace; (void)workspace_bytes;
  ARTK_CHECK_ARG(S > 0, "S, Hq, Hkv must be positive");
  int32_t rc = attn_check_multiple(S);
  if (rc) return rc;
  const int64_t strides[12] = {0, q_stride_s, q_stride_h, 0, k_stride_s, k_stride_h,
                               0, v_stride_s, v_stride_h, 0, o_stride_s, o_stride_h};
  return artk_attn_fwd_rows(q, k, v, plan, 1, S, Hq, Hkv, D, strides, scale, out, lse, stream);
}

struct AttnBwdScratch {
  float *delta, *lse2, *pk, *pv;
  int64_t kv_rows;
};
// Rows of a batch whose dK and dV are computed by one launch.  The partial sums of grouped-query heads are two fp32 arrays
// of q's shape, so the rows of a batch share 448 MiB of them (what 16384 positions of 28 heads of 128 need), or what one
// row needs.  Half of that costs 5 % of the backward of 8 rows of 2048 (663 -> 695 us), whose launches no longer fill
// the GPU.
static int64_t attn_kv_rows(int64_t B, int64_t S, int Hq, int Hkv, int D) {
  if (Hq == Hkv || B <= 0 || S <= 0 || Hq <= 0 || D <= 0) return B;
  const int64_t most = (448ll << 20) / (attn_padded(S) * Hq * D * 8);
  const int64_t launches = most > 0 ? (B + most - 1) / most : B;
  return (B + launches - 1) / launches;
}
static void carve_attn_bwd(Workspace& ws, int64_t B, int64_t S, int Hq, int Hkv, int D, AttnBwdScratch& c) {
  const size_t row = (size_t)(attn_padded(S) * Hq);
  c.delta = ws.take<float>(B * row);
  c.lse2 = ws.take<float>(B * row);
  c.kv_rows = attn_kv_rows(B, S, Hq, Hkv, D);
  c.pk = Hq != Hkv ? ws.take<float>(c.kv_rows * row * D) : nullptr;
  c.pv = Hq != Hkv ? ws.take<float>(c.kv_rows * row * D) : nullptr;
}
size_t artk_attn_bwd_rows_workspace_bytes(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int32_t D) {
  Workspace ws(nullptr, 0);
  AttnBwdScratch c;
  carve_attn_bwd(ws, B, S, Hq, Hkv, D, c);
  return ws.used + 256;
}
size_t artk_attn_bwd_workspace_bytes(int64_t S, int32_t Hq, int32_t Hkv, int32_t D) {
  return artk_attn_bwd_rows_workspace_bytes(1, S, Hq, Hkv, D);
}

int32_t artk_attn_bwd_rows(const void* q, const void* k, const void* v, const void* out, const float* lse,
                           const void* d_out, const void* plan, int64_t B, int64_t S, int32_t Hq, int32_t Hkv,
                           int32_t D, const int64_t* strides, float scale, void* dq, void* dk, void* dv,
                           void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  ARTK_CHECK_ARG(q && k && v && out && lse && d_out && plan && strides && dq && dk && dv,
                 "null pointer argument");
  ARTK_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out) && aligned16(d_out) &&
                     aligned16(dq) && aligned16(dk) && aligned16(dv),
                 "tensors must be 16-byte aligned");
  int32_t rc = attn_check(B, S, Hq, Hkv, D, strides, 8);
  if (rc) return rc;
  // the dK/dV kernel addresses lse2 and delta by head through 31-bit offsets
  ARTK_CHECK_ARG(attn_padded(S) * Hq * 4 < (1ll << 31), "S * Hq is too large");
  Workspace ws(workspace, workspace_bytes);
  AttnBwdScratch c;
  carve_attn_bwd(ws, B, S, Hq, Hkv, D, c);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  AttnPlan pl;
  attn_plan_layout(const_cast<void*>(plan), (size_t)1 << 40, attn_padded(S), pl);
  hipStream_t st = (hipStream_t)stream;
  AttnBwdParams p;
  p.Q = (const uint16_t*)q;
  p.K = (const uint16_t*)k;
  p.V = (const uint16_t*)v;
  p.O = (const uint16_t*)out;
  p.dO = (const uint16_t*)d_out;
  p.lse = lse;
  p.lse2 = c.lse2;
  p.delta = c.delta;
  p.dQ = (uint16_t*)dq;
  p.dK = (uint16_t*)dk;
  p.dV = (uint16_t*)dv;
  p.pK = c.pk;
  p.pV = c.pv;
  p.q_bs = strides[0];   p.q_ss = strides[1];   p.q_hs = strides[2];
  p.k_bs = strides[3];   p.k_ss = strides[4];   p.k_hs = strides[5];
  p.v_bs = strides[6];   p.v_ss = strides[7];   p.v_hs = strides[8];
  p.o_bs = strides[9];   p.o_ss = strides[10];  p.o_hs = strides[11];
  p.do_bs = strides[12]; p.do_ss = strides[13]; p.do_hs = strides[14];
  p.dq_bs = strides[15]; p.dq_ss = strides[16]; p.dq_hs = strides[17];
  p.dk_bs = strides[18]; p.dk_ss = strides[19]; p.dk_hs = strides[20];
  p.dv_bs = strides[21]; p.dv_ss = strides[22]; p.dv_hs = strides[23];
  p.gc = pl.gc;
  p.pc = pl.pc;
  p.list = pl.list;
  p.cnt = pl.cnt;
  p.order = pl.order;
  p.listT = pl.list2;
  p.cntT = pl.cnt2;
  p.orderT = pl.order2;
  p.plan_stride = pl.stride;
  p.S = (int)S;
  p.Sp = (int)attn_padded(S);
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.nQb = pl.nQb;
  p.nKb = pl.nKb;
  p.nQb2 = pl.nQb2;
  p.nKb2 = pl.nKb2;
  p.scale = scale;
  p.scale_log2e = scale * LOG2E;
  const dim3 grid_q(attn_grid(Hq, Hkv, pl.nQb), (unsigned)B);
  prof_begin(PROF_ATTN_BWD_Q, st);
  if (D == 128)
    attn_bwd_dq_kernel<128><<<grid_q, ATT_THREADS, 0, st>>>(p);
  else
    attn_bwd_dq_kernel<64><<<grid_q, ATT_THREADS, 0, st>>>(p);
  prof_end(PROF_ATTN_BWD_Q, st);
  ARTK_CHECK_LAUNCH();
  for (int64_t row0 = 0; row0 < B; row0 += c.kv_rows) {
    const int64_t rows = B - row0 < c.kv_rows ? B - row0 : c.kv_rows;
    const int slots = num_cus() * (D == 64 ? 3 : 2);  // resident work-groups
    const int64_t units = rows * pl.nKb2 * Hkv;
    const bool two_rounds = units >= 2 * slots;
    p.row0 = (int)row0;
    p.split.total = pl.total2;
    p.split.long_total = (two_rounds ? 100 : units >= slots ? 24 : 16) * pl.nKb2;
    p.split.heads_all = (int)(rows * Hq);   // (rows of a batch are taken to be alike)
    p.split.div = two_rounds ? slots * 3 / 2 : slots * 4 / 5;
    p.split.light_max = g_light_max_override;  // artk_attn_bwd_tuning
    const dim3 grid_kv(attn_grid(Hq, Hkv, pl.nKb2), (unsigned)rows);
    p.split.packed = Hq != Hkv && !two_rounds && (int64_t)grid_kv.x * grid_kv.y > slots &&
                     pl.nKb2 * (int64_t)Hkv <= 8 * ATT_KV_UNITS;
    prof_begin(PROF_ATTN_BWD_KV, st);
    if (D == 128)
      attn_bwd_kv_kernel<128><<<grid_kv, 256, 0, st>>>(p);
    else
      attn_bwd_kv_kernel<64><<<grid_kv, 256, 0, st>>>(p);
    prof_end(PROF_ATTN_BWD_KV, st);
    ARTK_CHECK_LAUNCH();
    if (Hq != Hkv) {
      const int64_t n4 = (int64_t)p.Sp * Hkv * (D / 4);
      attn_kv_reduce_kernel<<<dim3((unsigned)((n4 + 255) / 256), (unsigned)rows), 256, 0, st>>>(p, D);
      ARTK_CHECK_LAUNCH();
    }
  }
  return ARTK_OK;
}

int32_t artk_attn_bwd(const void* q, const void* k, const void* v, const void* out, const float* lse,
                      const void* d_out, const void* plan, int64_t S, int32_t Hq, int32_t Hkv,
                      int32_t D, const int64_t* strides, float scale, void* dq, void* dk, void* dv,
                      void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  ARTK_CHECK_ARG(S > 0 && strides, "S, Hq, Hkv must be positive");
  int32_t rc = attn_check_multiple(S);
  if (rc) return rc;
  int64_t s3[24];
  for (int i = 0; i < 8; ++i) {
    s3[3 * i] = 0;
    s3[3 * i + 1] = strides[2 * i];
    s3[3 * i + 2] = strides[2 * i + 1];
  }
  return artk_attn_bwd_rows(q, k, v, out, lse, d_out, plan, 1, S, Hq, Hkv, D, s3, scale, dq, dk, dv, workspace,
                            workspace_bytes, stream);
}

int32_t artk_attn_bwd_tuning(int32_t light_max) {
  g_light_max_override = light_max < 0 ? -1 : light_max;
  return ARTK_OK;
}

}  // extern "C"
