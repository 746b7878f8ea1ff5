// MoE expert path for gfx950: router top-k, stable expert-contiguous
// permutation, and per-expert LoRA linears as grouped GEMMs
//   y[i,:] = x[row(i),:] W_e^T + s (x[row(i),:] A_e^T) B_e^T      e = expert of row i
// over the permuted (token, expert) rows, with their backward.
//
// The reference has no MoE code at this commit; the contract comes from the
// benchmark configuration (128 experts, top-8, Qwen3-30B-A3B-style expert
// shapes, rank-8 LoRA per expert).  Routing follows the usual definition
// (softmax over router logits in fp32, top-k, renormalise); the selection is
// made on the logits, which order like the softmax, ties to the lower expert
// index, and the permutation is the stable sort of the token-major (token, slot)
// list by expert id, so both integer outputs are reproducible bit for bit.
#include "common.hpp"
#include "gemm_nt.hpp"
#include "lora_common.hpp"
#include "skinny_stats.hpp"

#include <math.h>

namespace artk {

// ----------------------------------------------------------------------------
// Routing: one wavefront per token.  (The launch is moe_topk_pack_kernel.)
// ----------------------------------------------------------------------------
constexpr int MOE_NI = 2;  // 8 waves, 2 per SIMD (see gemm_nt.hpp)
constexpr int MOE_MAX_E = 256;
constexpr int MOE_MAX_K = 16;

// Largest value of the wave, in every lane, by DPP (a shuffle goes through LDS and has its latency).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_max(float v) {
  const int x = __float_as_int(v);  // (lanes without a source keep their own value)
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, ROWS, 0xf, false)));
}
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = dpp_max<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8: lane 15 of a row of 16 has the row's
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_max<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Token t of the routing, by one wave.  A round is a maximum over the experts that are left and a ballot for each 64 of them
// (top-8 of 128 with an arg-max of shuffles: 8192 tokens 21 us, 203 tokens 9; now 12 and 5).
__device__ __forceinline__ void moe_topk_token(const float* __restrict__ logits, int64_t t, int E, int k,
                                               int* __restrict__ topk_idx, float* __restrict__ topk_w) {
  const int lane = threadIdx.x & 63;
  // NaN counts as -inf, so the order below is total: decreasing value, ties (also
  // among -inf) to the lower expert index; every round picks an index in [0, E).
  float x[4];
  unsigned taken = 0;  // bit i: element i of this lane is selected or past E
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = lane + 64 * i;
    float v = e < E ? logits[t * E + e] : -INFINITY;
    x[i] = v == v ? v : -INFINITY;
    if (e >= E) taken |= 1u << i;
  }
  float m = 0.f;
  float myp = 0.f;  // lane j keeps the probability mass of slot j
  int mye = 0;      // ... and its expert
  float psum = 0.f;
  for (int j = 0; j < k; ++j) {
    float bv = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) bv = fmaxf(bv, taken >> i & 1 ? -INFINITY : x[i]);
    bv = wave_max_dpp(bv);
    if (j == 0) m = bv;
    int bi = -1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned long long at = __ballot(!(taken >> i & 1) && x[i] == bv);
      if (bi < 0 && at != 0) bi = 64 * i + __builtin_ctzll(at);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (lane + 64 * i == bi) taken |= 1u << i;
    // exp(-inf - m) = 0; a row without any finite logit (m = -inf) has no mass at all
    const float pj = bv == -INFINITY ? 0.f : expf(bv - m);
    psum += pj;
    if (lane == j) {
      myp = pj;
      mye = bi;
    }
  }
  if (lane < k) {
    topk_idx[t * k + lane] = mye;
    topk_w[t * k + lane] = psum > 0.f ? myp / psum : 0.f;
  }
}

// ----------------------------------------------------------------------------
// Stable counting sort of the n = T*k keys (expert ids) in chunks of 1024.
// ----------------------------------------------------------------------------
constexpr int PERM_CHUNK = 1024;

__global__ __launch_bounds__(PERM_CHUNK) void moe_hist_kernel(const int* __restrict__ keys, int n,
                                                              int E, int* __restrict__ cnt) {
  __shared__ int hist[MOE_MAX_E];
  for (int i = threadIdx.x; i < E; i += PERM_CHUNK) hist[i] = 0;
  __syncthreads();
  const int f = blockIdx.x * PERM_CHUNK + threadIdx.x;
  // keys come from the top-k and lie in [0, E); anything else is ignored
  if (f < n && (unsigned)keys[f] < (unsigned)E) atomicAdd(&hist[keys[f]], 1);
  __syncthreads();
  for (int i = threadIdx.x; i < E; i += PERM_CHUNK) cnt[blockIdx.x * E + i] = hist[i];
}

// offsets[e]: first sorted position of expert e; base[b][e]: first sorted
// position of chunk b's entries of expert e; tile_prefix / blk_prefix: prefix
// sums of ceil(rows_e / 256) and ceil(rows_e / 16) (work lists of the grouped
// kernels).  One block of 1024 threads: thread (part, e) walks a quarter of the
// chunks of expert e, eight independent loads at a time.  order [E+1] (or nullptr): the
// experts by falling number of rows, ties by index, then moe_split_rows.
constexpr int SCAN_PARTS = 4;
constexpr int SG_COLS = 128;  // rows of an expert in one pass of the streaming product over its weights

// The streaming product deals whole experts to the XCDs, back and forth in falling order of their rows.
__device__ __forceinline__ int moe_dealt_to(int rank) { return rank & 8 ? 7 - (rank & 7) : rank & 7; }
// Experts with more rows than this are split between the XCDs instead: none if no XCD gets more than 5 / 4 of its share of
// the passes (share[x]) that way, else those with more than 1 / 32 of all rows (there are fewer than 32).
__device__ __forceinline__ int moe_split_rows(const int* share, int n_rows) {
  int all = 0, most = 0;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    all += share[x];
    most = most > share[x] ? most : share[x];
  }
  return 4 * 8 * most > 5 * all ? n_rows / 32 : 0x7fffffff;
}
struct MoeScanLds {
  int part[SCAN_PARTS][MOE_MAX_E];  // rows of an expert in a quarter of the chunks
  int wsum[3][MOE_MAX_E / 64];
  int off[MOE_MAX_E], rows[MOE_MAX_E], rank[MOE_MAX_E], share[8];
};
struct MoeScanOut {
  int *offsets, *tile_prefix, *blk_prefix, *order;
};
// The prefix sums over the experts, from l.part on (a barrier lies behind its last write); l.off and l.rows are there
// when it returns.
__device__ __forceinline__ void moe_scan_experts(MoeScanLds& l, int E, const MoeScanOut& o) {
  const int e = threadIdx.x % MOE_MAX_E, pt = threadIdx.x / MOE_MAX_E;
  // exclusive prefix sums over the experts (threads of part 0: one expert each)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int tot = 0, run = 0, tp = 0, bp = 0;
  if (pt == 0) {
    if (e < E)
#pragma unroll
      for (int q = 0; q < SCAN_PARTS; ++q) tot += l.part[q][e];
    run = tot;
    tp = (tot + TILE - 1) / TILE;
    bp = (tot + 15) / 16;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int a = __shfl_up(run, d, 64), t = __shfl_up(tp, d, 64), c = __shfl_up(bp, d, 64);
      if (lane >= d) {
        run += a;
        tp += t;
        bp += c;
      }
    }
    if (lane == 63) {
      l.wsum[0][wave] = run;
      l.wsum[1][wave] = tp;
      l.wsum[2][wave] = bp;
    }
  }
  __syncthreads();
  if (pt == 0) {
    for (int w = 0; w < wave; ++w) {
      run += l.wsum[0][w];
      tp += l.wsum[1][w];
      bp += l.wsum[2][w];
    }
    // inclusive sums -> entry e + 1; entry 0 is zero
    if (e < E) {
      o.offsets[e + 1] = run;
      o.tile_prefix[e + 1] = tp;
      o.blk_prefix[e + 1] = bp;
      l.off[e] = run - tot;
      l.rows[e] = tot;
      l.rank[e] = 0;
    }
    if (e == 0) {
      o.offsets[0] = 0;
      o.tile_prefix[0] = 0;
      o.blk_prefix[0] = 0;
    }
    if (e < 8) l.share[e] = 0;
  }
  __syncthreads();
}
__device__ __forceinline__ void moe_scan_order(MoeScanLds& l, int E, int* order) {
  const int e = threadIdx.x % MOE_MAX_E, pt = threadIdx.x / MOE_MAX_E;
  if (order == nullptr) return;
  const int j0 = pt * (MOE_MAX_E / SCAN_PARTS), j1 = j0 + MOE_MAX_E / SCAN_PARTS;
  if (e < E) {
    const int c = l.rows[e];
    int before = 0;
#pragma unroll 8
    for (int j = j0; j < (j1 < E ? j1 : E); ++j) before += (l.rows[j] > c || (l.rows[j] == c && j < e)) ? 1 : 0;
    atomicAdd(&l.rank[e], before);
  }
  __syncthreads();
  if (pt == 0 && e < E) {
    order[l.rank[e]] = e;
    atomicAdd(&l.share[moe_dealt_to(l.rank[e])], (l.rows[e] + SG_COLS - 1) / SG_COLS);
  }
  __syncthreads();
  if (threadIdx.x == 0) order[E] = moe_split_rows(l.share, l.off[E - 1] + l.rows[E - 1]);
}

__global__ __launch_bounds__(SCAN_PARTS * MOE_MAX_E) void moe_scan_kernel(const int* __restrict__ cnt, int nb, int E,
                                                                          int* __restrict__ base, MoeScanOut o) {
  __shared__ MoeScanLds l;
  const int e = threadIdx.x % MOE_MAX_E, pt = threadIdx.x / MOE_MAX_E;
  const int per = (nb + SCAN_PARTS - 1) / SCAN_PARTS;
  const int b0 = pt * per, b1 = b0 + per < nb ? b0 + per : nb;
  int s = 0;
  if (e < E) {
    for (int b = b0; b < b1; b += 8) {
      int v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = b + u < b1 ? cnt[(b + u) * E + e] : 0;
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
  }
  l.part[pt][e] = s;
  __syncthreads();
  moe_scan_experts(l, E, o);
  if (e < E) {
    int pos = l.off[e];
    for (int q = 0; q < pt; ++q) pos += l.part[q][e];
    for (int b = b0; b < b1; b += 8) {
      int v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = b + u < b1 ? cnt[(b + u) * E + e] : 0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (b + u < b1) base[(b + u) * E + e] = pos;
        pos += v[u];
      }
    }
  }
  moe_scan_order(l, E, o.order);
}

// Lanes of the wave whose key (0 .. 255) is this lane's; lanes with key < 0 match nobody.
__device__ __forceinline__ unsigned long long moe_same_key(int key) {
  unsigned long long same = __ballot(key >= 0);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const bool bit = key >> b & 1;
    const unsigned long long with = __ballot(bit);
    same &= bit ? with : ~with;
  }
  return key >= 0 ? same : 0ull;
}
struct MoePerm {
  int *perm, *inv_perm, *row_token;
  __device__ __forceinline__ void place(int f, int pos, int k) const {
    perm[pos] = f;
    inv_perm[f] = pos;
    row_token[pos] = f / k;
  }
};

// The whole sort of a few chunks by one work-group: for 1624 keys histogram, scan and placement are 3 + 5 + 6 us as three
// launches, and the gaps between them, and 7 as one.  (A launch per step is what many chunks need: their placement is spread.)
// Routing of 128 experts in us, one launch / three: 1624 keys 11.3 / 12.4, 3072 12.6 / 12.7, 3584 13.1 / 13.0, 4096 13.6 / 12.8 in
// the replay of a graph; a block's forward at 4096 keys, gaps included, 284.0 / 284.6.
constexpr int SORT_CHUNKS = 4;
__global__ __launch_bounds__(PERM_CHUNK) void moe_sort_kernel(const int* __restrict__ keys, int n, int E, int k, MoeScanOut o,
                                                              MoePerm out) {
  static_assert(SORT_CHUNKS == SCAN_PARTS && PERM_CHUNK == SCAN_PARTS * MOE_MAX_E, "a part of the scan per chunk");
  constexpr int NW = PERM_CHUNK / 64;
  __shared__ MoeScanLds l;
  __shared__ int hist[SORT_CHUNKS * NW][MOE_MAX_E];  // by chunk and wave: counts, then counts of the waves before in the chunk
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int key[SORT_CHUNKS], rank[SORT_CHUNKS];
#pragma unroll
  for (int c = 0; c < SORT_CHUNKS; ++c) {
    const int f = c * PERM_CHUNK + threadIdx.x;
    key[c] = f < n ? keys[f] : -1;
    if ((unsigned)key[c] >= (unsigned)E) key[c] = -1;  // never produced by the top-k
  }
  for (int i = threadIdx.x; i < SORT_CHUNKS * NW * MOE_MAX_E; i += PERM_CHUNK) (&hist[0][0])[i] = 0;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < SORT_CHUNKS; ++c) {
    const unsigned long long same = moe_same_key(key[c]);
    rank[c] = __popcll(same & ((1ull << lane) - 1ull));
    if (key[c] >= 0 && rank[c] == 0) hist[c * NW + wave][key[c]] = __popcll(same);
  }
  __syncthreads();
  {
    const int e = threadIdx.x % MOE_MAX_E, c = threadIdx.x / MOE_MAX_E;
    int s = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const int v = hist[c * NW + w][e];
      hist[c * NW + w][e] = s;
      s += v;
    }
    l.part[c][e] = s;
  }
  __syncthreads();
  moe_scan_experts(l, E, o);
#pragma unroll
  for (int c = 0; c < SORT_CHUNKS; ++c) {
    if (key[c] < 0) continue;
    int pos = l.off[key[c]] + hist[c * NW + wave][key[c]] + rank[c];
#pragma unroll
    for (int q = 0; q < c; ++q) pos += l.part[q][key[c]];
    out.place(c * PERM_CHUNK + threadIdx.x, pos, k);
  }
  moe_scan_order(l, E, o.order);
}

// Stable placement of one chunk: position = base[chunk][key] + number of earlier
// entries of the chunk with the same key.  That rank is the count in the earlier
// waves (per-wave histograms in LDS) plus the count among the earlier lanes of the
// own wave.
__global__ __launch_bounds__(PERM_CHUNK) void moe_scatter_kernel(const int* __restrict__ keys, int n, int E, int k,
                                                                 const int* __restrict__ base, MoePerm out) {
  constexpr int NW = PERM_CHUNK / 64;
  __shared__ int hist[NW][256];  // E <= 256
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < NW * 256; i += PERM_CHUNK) (&hist[0][0])[i] = 0;
  __syncthreads();
  const int f = blockIdx.x * PERM_CHUNK + threadIdx.x;
  int key = f < n ? keys[f] : -1;
  if ((unsigned)key >= (unsigned)E) key = -1;  // never produced by the top-k
  const unsigned long long same = moe_same_key(key);
  int rank = __popcll(same & ((1ull << lane) - 1ull));
  if (key >= 0 && rank == 0) hist[wave][key] = __popcll(same);
  __syncthreads();
  if (key >= 0) {
    for (int w = 0; w < wave; ++w) rank += hist[w][key];
    out.place(f, base[blockIdx.x * E + key] + rank, k);
  }
}

// Largest g with prefix[g] <= x, for a non-decreasing prefix[0..G] with prefix[G] > x.
__device__ __forceinline__ int find_group(const int* __restrict__ prefix, int G, int x) {
  int lo = 0, hi = G;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= x) lo = mid; else hi = mid;
  }
  return lo;
}

// ----------------------------------------------------------------------------
// Grouped GEMM: 256-row tiles never straddle experts.
// ----------------------------------------------------------------------------
struct MoeGemmParams {
  const void* W;           // [E,M,K] bf16
  const void* X;           // activations, [*,K] bf16
  const int* gather;       // permuted row i reads X row gather[i]; nullptr: row i
  const uint16_t* Pe;      // [E,M,r] low-rank factor of the weights
  const uint16_t* Qe;      // [n_rows,RP] zero-padded, scaled low-rank activations
  uint16_t* out;           // [n_rows,M]
  const int* offsets;      // [E+1]
  const int* tile_prefix;  // [E+1]
  int64_t M, K;
  int E, r, RP, MT;
  const int* order;        // [E+1] experts by falling number of rows, then moe_split_rows
};

// One tile of the grouped product: expert, rows and weight tile.
struct MoeTile {
  int e, mt, nvalid;
  int64_t row0, row_end;
};

__device__ __forceinline__ MoeTile moe_tile(const MoeGemmParams& p, int t, int n_work) {
  // Ids run expert by expert and, inside an expert, weight tile by weight tile over its row
  // tiles: the two or three work-groups that need the same weight tile have neighbouring ids,
  // start together and read it from HBM once (the L2 of their XCD serves the others); the MT
  // work-groups that share a row tile are only a few ids apart and still run side by side.
  const int id = xcd_remap(t, n_work);
  MoeTile m;
  m.e = find_group(p.tile_prefix, p.E, id / p.MT);
  const int first = p.tile_prefix[m.e], n_e = p.tile_prefix[m.e + 1] - first;
  const int local = id - first * p.MT;
  m.mt = local / n_e;
  m.row0 = p.offsets[m.e] + (int64_t)(local - m.mt * n_e) * TILE;
  m.row_end = p.offsets[m.e + 1];
  m.nvalid = (int)(m.row_end - m.row0 < TILE ? m.row_end - m.row0 : TILE);
  return m;
}

__device__ __forceinline__ void moe_tile_loaders(TileLoaders<MOE_NI>& L, const MoeGemmParams& p,
                                                 const MoeTile& m) {
  // rows past the expert's end are not fetched (their output columns are never stored)
  L.init((const char*)p.W + (int64_t)m.e * p.M * p.K * 2, p.K, (int64_t)m.mt * TILE, p.M, p.X, p.K, m.row0,
         m.row_end, 0, (int)p.K, p.gather, true);
}

// Persistent work-groups: tiles t, t + grid, ... of the device-side work list; the
// next tile's first DMA stage starts before the rank-r steps and the store of the
// current one (short K loops: 12 or 32 steps per tile).
__global__ __launch_bounds__(nthreads<MOE_NI>()) void moe_gemm_kernel(MoeGemmParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[GEMM_LDS_BYTES];
  const int n_work = p.tile_prefix[p.E] * p.MT;
  int t = blockIdx.x;
  if (t >= n_work) return;
  MoeTile cur = moe_tile(p, t, n_work);
  {
    TileLoaders<MOE_NI> first;
    moe_tile_loaders(first, p, cur);
    first.issue_first(smem);
  }
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave_m<MOE_NI>(wave), wn = wave_n<MOE_NI>(wave);
  const int half = lane >> 5;
  for (;;) {
    const int t2 = t + gridDim.x;
    const bool more = t2 < n_work;
    MoeTile nxt = cur;
    if (more) nxt = moe_tile(p, t2, n_work);

    TileAcc<MOE_NI> acc;
    acc.zero();
    {
      TileLoaders<MOE_NI> L;  // its first stage is already on the way
      moe_tile_loaders(L, p, cur);
      gemm_tile_run_cols(acc, smem, L, cur.nvalid);  // a tail tile computes only its live 32-row blocks
    }
    if (more) {
      TileLoaders<MOE_NI> L;
      moe_tile_loaders(L, p, nxt);
      L.issue_first(smem);
    }

    const int e = cur.e, mt = cur.mt, nvalid = cur.nvalid;
    const int64_t row0 = cur.row0;
    if (p.Pe != nullptr) {
      int64_t prow[4], qrow[MOE_NI];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int64_t r = (int64_t)mt * TILE + wm * 128 + i * 32 + (lane & 31);
        prow[i] = r < p.M ? r : p.M - 1;
      }
#pragma unroll
      for (int i = 0; i < MOE_NI; ++i) {
        int c = acc_col<MOE_NI>(wn, i, lane);
        qrow[i] = row0 + (c < nvalid ? c : nvalid - 1);
      }
      lowrank_steps(acc, p.Pe + (int64_t)e * p.M * p.r, p.r, p.r, prow, p.Qe, p.RP, p.RP, qrow, p.RP);
    }

#pragma unroll
    for (int ni = 0; ni < MOE_NI; ++ni) {
      // lanes l and l + 32 share the column, so they take these branches together
      // (store_block_bf16 exchanges data between them)
      const int c = acc_col<MOE_NI>(wn, ni, lane);
      const bool col_ok = c < nvalid;
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        const int64_t m0 = (int64_t)mt * TILE + wm * 128 + mi * 32;
        if (m0 >= p.M) continue;  // wave-uniform
        if (m0 + 32 <= p.M) {
          if (col_ok) store_block_bf16(p.out + (row0 + c) * p.M + m0, acc.c[mi][ni], half);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int64_t m = m0 + q * 8 + half * 4;
            if (m >= p.M || !col_ok) continue;
            bf16x4 o;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = (__bf16)acc.c[mi][ni][q * 4 + k];
            *(bf16x4*)(p.out + (row0 + c) * p.M + m) = o;
          }
        }
      }
    }
    if (!more) break;
    t = t2;
    cur = nxt;
  }
}

// ----------------------------------------------------------------------------
// The same grouped product where an expert has few rows: the launch reads every weight once for a handful of columns
// and is as long as those reads.  A work-group streams 128 weight rows of one expert past up to 128 of its rows at a
// time (4 waves, 32 weight rows each), two work-groups per CU.  The weights come from HBM and have a ring of three or
// four stages of 64 K elements, the activations from L2 and have two; waves 0 and 1 issue the weights' DMA, waves 2 and
// 3 the activations', because a wave's DMA completes in order and a wait for the younger activations would wait for
// the weights behind them.  So up to 96 KiB of weights are on their way per CU where the 256 x 256 tile above has 32.
// ----------------------------------------------------------------------------
constexpr int SG_ROWS = 128;                      // weight rows of a work-group
constexpr int SG_P_BYTES = SG_ROWS * BK * 2;      // 16 KiB
constexpr int SG_LDS_BYTES = 80 * 1024;           // two work-groups per CU
template <int NQ> constexpr int sg_stages() { return NQ <= 2 ? 4 : 3; }

// acc[i] += 32 weight rows of this wave x columns 32 i .. 32 i + 31 over nk K steps.  Every wave calls it together; LDS
// may be reused when it returns.  ONCE: nobody reads the weights again, they pass the caches by (0.8 GB in 135 us instead of
// 150).  Whatever their size: a model's other layers come before they are read again.  Four products of a block, through / past
// the caches, after 1 GiB of other writes: 8 experts (75 MB) 124 / 102 us, 16 151 / 101, 32 210 / 146; the same block again and
// again, with nothing in between: 80 / 101, 107 / 101, 160 / 146.
template <int NQ, bool ONCE>
__device__ __forceinline__ void moe_stream_run(floatx16 (&acc)[NQ], char* smem, dma_rsrc_t prsrc, const int (&pv)[2],
                                               int pstep, dma_rsrc_t qrsrc, const int (&qv)[2 * NQ], int nk) {
  constexpr int NST = sg_stages<NQ>(), Q_BYTES = NQ * 4096, Q_OFF = NST * SG_P_BYTES;
  static_assert(Q_OFF + 2 * Q_BYTES <= SG_LDS_BYTES, "rings");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds = lds_addr_of(smem);
  auto issue_p = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int g = wave * 8 + i;
      dma_load16<ONCE>(prsrc, pv[i & 1], g * pstep + kt * (BK * 2), lds + buf * SG_P_BYTES + g * 1024);
    }
  };
  auto issue_q = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 2 * NQ; ++i)
      dma_load16(qrsrc, qv[i], kt * (BK * 2), lds + Q_OFF + (kt & 1) * Q_BYTES + ((wave - 2) * 2 * NQ + i) * 1024);
  };
  int off[4];
  {
    const int rl = lane & 31, f = swz(rl);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) off[kk] = rl * 128 + (((kk * 2 + (lane >> 5)) ^ f) << 4);
  }
  if (wave < 2) {
#pragma unroll
    for (int i = 0; i < NST - 1; ++i)
      if (i < nk) issue_p(i, i);
  } else {
    issue_q(0);
  }
  int buf = 0, fill = NST - 1;  // weight stage of K step kt, and the one that is free after its barrier
  for (int kt = 0; kt < nk; ++kt) {
    // stage kt has landed: of the weights, only the stages after it may be on their way
    if (wave >= 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (kt + NST - 1 <= nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * 8) : "memory");
    else if (NST == 4 && kt + 2 == nk) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    barrier_lds_only();  // ... for every wave, and every wave is done with stage kt - 1
    if (wave < 2) {
      if (kt + NST - 1 < nk) issue_p(kt + NST - 1, fill);
    } else {
      if (kt + 1 < nk) issue_q(kt + 1);
    }
    const char* sp = smem + buf * SG_P_BYTES + wave * 4096;
    const char* sq = smem + Q_OFF + (kt & 1) * Q_BYTES;
    bf16x8 p[4], q[4][NQ];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      p[kk] = *(const bf16x8*)(sp + off[kk]);
#pragma unroll
      for (int i = 0; i < NQ; ++i) q[kk][i] = *(const bf16x8*)(sq + off[kk] + i * 4096);
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < NQ; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p[kk], q[kk][i], acc[i], 0, 0, 0);
    buf = buf + 1 == NST ? 0 : buf + 1;
    fill = fill + 1 == NST ? 0 : fill + 1;
  }
  barrier_lds_only();
}

// n <= 32 NQ rows of expert e, from sorted row row0 on, against its weight rows m0 ..
template <int NQ, bool ONCE>
__device__ __forceinline__ void moe_stream_cols(const MoeGemmParams& p, char* smem, int e, int64_t m0, int64_t row0,
                                                int n) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5;
  const int r = lane >> 3, pc = lane & 7;
  const int64_t wrows = p.M - m0 < SG_ROWS ? p.M - m0 : SG_ROWS;  // rows past the end arrive as zeros
  const dma_rsrc_t prsrc =
      dma_make_rsrc((const char*)p.W + ((int64_t)e * p.M + m0) * p.K * 2, (uint32_t)(wrows * p.K * 2));
  const int pv[2] = {(int)(r * p.K * 2) + ((pc ^ r) << 4), (int)(r * p.K * 2) + ((pc ^ r ^ 1) << 4)};  // as PanelLoader
  const dma_rsrc_t qrsrc = dma_make_rsrc((const char*)p.X + (p.gather ? 0 : row0 * p.K * 2), 0x7fffffffu);
  int qv[2 * NQ];
#pragma unroll
  for (int i = 0; i < 2 * NQ; ++i) {
    const int row = ((wave & 1) * 2 * NQ + i) * 8 + r;
    int64_t src = row < n ? row : n - 1;
    if (p.gather) src = p.gather[row0 + src];
    qv[i] = (int)(src * p.K * 2) + ((pc ^ swz(row)) << 4);
  }
  floatx16 acc[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
  moe_stream_run<NQ, ONCE>(acc, smem, prsrc, pv, (int)(8 * p.K * 2), qrsrc, qv, (int)(p.K / BK));

  const int64_t mw = m0 + wave * 32;  // first weight row of this wave
  if (mw >= p.M) return;              // (M is a multiple of 64: a wave's rows are all there or none)
  if (p.Pe != nullptr) {
    const uint16_t* Pe = p.Pe + ((int64_t)e * p.M + mw + (lane & 31)) * p.r;
    for (int e0 = 0; e0 < p.RP; e0 += 16) {
      const int c = e0 + half * 8;
      const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
      bf16x8 pf = *(const bf16x8*)(Pe + (c < p.r ? c : 0));
      bf16x8 qf[NQ];
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int col = i * 32 + (lane & 31);
        qf[i] = *(const bf16x8*)(p.Qe + (row0 + (col < n ? col : n - 1)) * p.RP + c);
      }
      pf = c < p.r ? pf : z;
#pragma unroll
      for (int i = 0; i < NQ; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pf, qf[i], acc[i], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int col = i * 32 + (lane & 31);
    if (col < n) store_block_bf16(p.out + (row0 + col) * p.M + mw, acc[i], half);
  }
}

template <bool ONCE>
__device__ __forceinline__ void moe_stream_pass(const MoeGemmParams& p, char* smem, int e, int64_t m0, int64_t row0,
                                                int n) {
  if (n > 96) moe_stream_cols<4, ONCE>(p, smem, e, m0, row0, n < SG_COLS ? n : SG_COLS);
  else if (n > 64) moe_stream_cols<3, ONCE>(p, smem, e, m0, row0, n);
  else if (n > 32) moe_stream_cols<2, ONCE>(p, smem, e, m0, row0, n);
  else moe_stream_cols<1, ONCE>(p, smem, e, m0, row0, n);
}

// An XCD has the experts that it is dealt (lanes 32 .. 63), whose rows are then in one L2, and an eighth of the units of every
// expert that is split (lanes 0 .. 31; they come first in the order).  Without the split, XCDs have nothing to do where there are
// fewer than eight experts, and one of them works alone where an expert has most of the rows: forward of a block (hidden
// 2048, intermediate 768), us, 256 x 256 tiles / dealt only / with the split: 8000 rows on one of 128 experts
// 160 / 688 / 198, 4000 rows on each of two 154 / 399 / 181, 4 experts of 125 rows and intermediate 5632 236 / 220 / 186.
// An XCD's units are numbered expert by expert, weight tile by weight tile, and the passes of an expert with more than SG_COLS
// rows (even shares of them, in whole 32) are neighbours, so they read a weight tile together.
__global__ __launch_bounds__(256, 2) void moe_stream_gemm_kernel(MoeGemmParams p) {
  static_assert(MOE_MAX_E <= 8 * 32, "a lane per expert of an XCD");
  __shared__ __attribute__((aligned(1024))) char smem[SG_LDS_BYTES];
  const int lane = threadIdx.x & 63, l32 = lane & 31;
  const int x = blockIdx.x & 7;
  const bool parts = lane < 32;
  const int pos = parts ? l32 : 8 * l32 + ((l32 & 1) ? 7 - x : x);  // of this lane's expert in the order (moe_dealt_to)
  const int split_rows = p.order[p.E];
  int ex = 0, first = 0, n_e = 0;
  if (pos < p.E) {
    ex = p.order[pos];
    first = p.offsets[ex];
    n_e = p.offsets[ex + 1] - first;
  }
  const int passes = (n_e + SG_COLS - 1) / SG_COLS;
  int from = 0, units = passes * p.MT;  // this XCD's units of the expert
  if (parts) {
    const int y = (x + l32) & 7;
    from = units * y / 8;
    units = units * (y + 1) / 8 - from;
  }
  if ((n_e > split_rows) != parts) units = 0;
  int end = units;  // units of the experts up to this one
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(end, d, 64);
    if (lane >= d) end += v;
  }
  const int shift = end - units - from;
  const int total = __builtin_amdgcn_readlane(end, 63);
  for (int loc = blockIdx.x >> 3; loc < total; loc += gridDim.x >> 3) {
    const int l = __popcll(__ballot(end <= loc));
    const int e = __builtin_amdgcn_readlane(ex, l), n = __builtin_amdgcn_readlane(n_e, l);
    const int np = __builtin_amdgcn_readlane(passes, l), row0 = __builtin_amdgcn_readlane(first, l);
    const int unit = loc - __builtin_amdgcn_readlane(shift, l);
    const int per = ((n + np - 1) / np + 31) & ~31, c0 = (unit % np) * per;
    const int64_t m0 = (int64_t)(unit / np) * SG_ROWS;
    const int left = n - c0 < per ? n - c0 : per;
    if (np == 1) moe_stream_pass<true>(p, smem, e, m0, row0, left);
    else if (left > 0) moe_stream_pass<false>(p, smem, e, m0, row0 + c0, left);
  }
}

// order [E+1] as moe_scan_kernel leaves it.
__global__ __launch_bounds__(MOE_MAX_E) void moe_order_kernel(const int* __restrict__ offsets, int E, int* __restrict__ order) {
  __shared__ int rows[MOE_MAX_E], share[8];
  const int e = threadIdx.x, c = e < E ? offsets[e + 1] - offsets[e] : 0;
  rows[e] = c;
  if (e < 8) share[e] = 0;
  __syncthreads();
  if (e < E) {
    int rank = 0;
    for (int j = 0; j < E; ++j) rank += (rows[j] > c || (rows[j] == c && j < e)) ? 1 : 0;
    order[rank] = e;
    atomicAdd(&share[moe_dealt_to(rank)], (c + SG_COLS - 1) / SG_COLS);
  }
  __syncthreads();
  if (e == 0) order[E] = moe_split_rows(share, offsets[E] - offsets[0]);
}

// Grouped row products: 16-row blocks never straddle experts.
//   out[i, j] = sum_k X[row(i), k] Mt_e[j, k],  Mt [E,R,K]
// (the f32 output also times row_w[row_idx[i]], when given)
__global__ __launch_bounds__(256) void moe_rowdot16_kernel(
    const uint16_t* __restrict__ X, const int* __restrict__ gather, const uint16_t* __restrict__ Mt,
    const int* __restrict__ offsets, const int* __restrict__ blk_prefix, int E, int64_t K, int R,
    int RP, float scale, const float* __restrict__ row_w, const int* __restrict__ row_idx,
    float* __restrict__ out_f32, uint16_t* __restrict__ out_bf16) {
  __shared__ floatx4 red[3][64];
  const int b = blockIdx.x;
  if (b >= blk_prefix[E]) return;
  const int e = find_group(blk_prefix, E, b);
  const int64_t row0 = offsets[e] + (int64_t)(b - blk_prefix[e]) * 16;
  const int64_t row_end = offsets[e + 1];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int jm = blockIdx.y * 16 + (lane & 15);
  int64_t row = row0 + (lane & 15);
  if (row >= row_end) row = row_end - 1;
  const int64_t src = gather ? gather[row] : row;
  const uint16_t* xp = X + src * K + (lane >> 4) * 8;
  const uint16_t* mp = Mt + ((int64_t)e * R + (jm < R ? jm : 0)) * K + (lane >> 4) * 8;
  floatx4 acc = rowdot_accumulate(xp, mp, jm < R, K, wave);
  acc = rowdot_block_sum(acc, red);
  if (wave == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t i = row0 + (lane >> 4) * 4 + q;
      if (i < row_end) {
        if (jm < R) out_f32[i * R + jm] = row_w ? acc[q] * row_w[row_idx[i]] : acc[q];
        out_bf16[i * RP + jm] = f32_to_bf16(acc[q] * scale);
      }
    }
  }
}

// ----------------------------------------------------------------------------
// The expert block around its grouped products (artk_moe_experts_fwd / _bwd).  As torch element-wise and
// gather calls these steps were 2.9 of the 4.8 ms of a block of 8192 tokens (top-8 of 128 experts, hidden
// 2048, intermediate 768): the routing weights in fp32 copies of [T, k, H], the gating through four fp32
// arrays, an index backward with a sort.  Here each is one pass with 16-byte accesses, and the routing
// weight of a row never meets a [rows, H] array: the backward of the down projection reads the rows of the
// token gradient through the gather, and the weight multiplies the rank-r products and the gated gradient.
// ----------------------------------------------------------------------------

// bf16 adapters of one block from its six parameters (f32 or bf16), each as the forward reads it and transposed as the
// backward does: gate and up share their input, so their A are stacked ([E, 2r, H]) and their B form a block-diagonal
// [E, 2I, 2r]; down's are copied.  HBM-bound: 76 MB for 128 experts, hidden 2048, intermediate 768 and rank 8 take 17 us.  (A
// copy alone took 11, and the transposes as a launch of the backward, which read the copies once more, 12 to 15.)  A forward
// that no backward follows leaves the transposes out (203 tokens 260 -> 257 us, rank 16 277 -> 264).
struct MoePack {
  const void *gate_A, *gate_B, *up_A, *up_B, *down_A, *down_B;
  uint16_t *A_gu, *B_gu, *A_d, *B_d;
  uint16_t *At_gu, *Bt_gu, *At_d, *Bt_d;  // [E,H,2r], [E,2r,2I], [E,I,r], [E,r,H]; all null: no backward follows
  int64_t H, I;
  int E, r, bf16;
};

__device__ __forceinline__ uint4 load8_bf16(const void* src, int64_t i, int is_bf16) {
  if (is_bf16) return *(const uint4*)((const uint16_t*)src + i);
  const float4 a = *(const float4*)((const float*)src + i), b = *(const float4*)((const float*)src + i + 4);
  return make_uint4(pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(b.x, b.y), pack_bf16x2(b.z, b.w));
}

// Block `blk` of 256 threads.  Every dimension is a multiple of 8: a thread takes an 8 x 8 block of one matrix, of gate's and
// of up's A, whose transposed rows lie side by side.
__device__ __forceinline__ void moe_pack_block(const MoePack& p, int64_t blk) {
  int64_t i = blk * 256 + threadIdx.x;
  const int64_t nH = (int64_t)p.E * p.r * p.H / 64, nI = (int64_t)p.E * p.r * p.I / 64;
  // 0: gate_A and up_A [E,r,H]; 1: gate_B, 2: up_B [E,I,r]; 3: down_A [E,r,I]; 4: down_B [E,H,r]
  int m = 0;
  for (; m < 5; ++m) {
    const int64_t size = m == 0 || m == 4 ? nH : nI;
    if (i < size) break;
    i -= size;
  }
  if (m == 5) return;
  const int64_t R = m == 0 || m == 3 ? p.r : m == 4 ? p.H : p.I, C = m == 0 ? p.H : m == 3 ? p.I : p.r;
  const int64_t CB = C / 8, per = R / 8 * CB, e = i / per;
  const int64_t r0 = (i - e * per) / CB * 8, c0 = (i - e * per) % CB * 8;
  const int64_t src = (e * R + r0) * C + c0;
  auto load = [&](const void* from, uint4 (&v)[8]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = load8_bf16(from, src + q * C, p.bf16);
  };
  auto store = [&](uint16_t* to, int64_t ld, const uint4 (&v)[8]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) *(uint4*)(to + q * ld) = v[q];
  };
  const bool transposed = p.At_gu != nullptr;
  uint4 v[8], t[8];
  if (m == 0) {
    uint4 u[8], ut[8];
    load(p.gate_A, v);
    load(p.up_A, u);
    uint16_t* to = p.A_gu + (e * 2 * p.r + r0) * p.H + c0;
    store(to, p.H, v);
    store(to + p.r * p.H, p.H, u);
    if (!transposed) return;
    transpose8x8(v, t);
    transpose8x8(u, ut);
    to = p.At_gu + (e * p.H + c0) * 2 * p.r + r0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      *(uint4*)(to + q * 2 * p.r) = t[q];
      *(uint4*)(to + q * 2 * p.r + p.r) = ut[q];
    }
    return;
  }
  load(m == 1 ? p.gate_B : m == 2 ? p.up_B : m == 3 ? p.down_A : p.down_B, v);
  if (m > 2) {
    store((m == 3 ? p.A_d : p.B_d) + src, C, v);
    if (!transposed) return;
    transpose8x8(v, t);
    store((m == 3 ? p.At_d : p.Bt_d) + (e * C + c0) * R + r0, R, t);
    return;
  }
  // gate | up of B, and zeros beside them
  const int up = m - 1;
  uint16_t* to = p.B_gu + ((e * 2 + up) * p.I + r0) * 2 * p.r + c0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    *(uint4*)(to + q * 2 * p.r + up * p.r) = v[q];
    *(uint4*)(to + q * 2 * p.r + (1 - up) * p.r) = make_uint4(0, 0, 0, 0);
  }
  if (!transposed) return;
  transpose8x8(v, t);
  to = p.Bt_gu + (e * 2 * p.r + c0) * 2 * p.I + r0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    *(uint4*)(to + (up * p.r + q) * 2 * p.I + up * p.I) = t[q];
    *(uint4*)(to + (up * p.r + q) * 2 * p.I + (1 - up) * p.I) = make_uint4(0, 0, 0, 0);
  }
}

// Routing of T tokens by the first blocks, the block's adapters by the rest (they have nothing to do with each other).
__global__ __launch_bounds__(256) void moe_topk_pack_kernel(const float* __restrict__ logits, int64_t T, int E, int k,
                                                            int* __restrict__ topk_idx, float* __restrict__ topk_w,
                                                            MoePack p) {
  const int64_t first = (T + 3) / 4;
  if (blockIdx.x >= first) {
    moe_pack_block(p, blockIdx.x - first);
    return;
  }
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t < T) moe_topk_token(logits, t, E, k, topk_idx, topk_w);
}

__device__ __forceinline__ void unpack8(const uint4& v, float (&f)[8]) {
  unpack2(v.x, f[0], f[1]);
  unpack2(v.y, f[2], f[3]);
  unpack2(v.z, f[4], f[5]);
  unpack2(v.w, f[6], f[7]);
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
}

// h[i, c] = silu(gu[i, c]) gu[i, I + c]; 6 B per element of h, HBM-bound.
__global__ __launch_bounds__(256) void moe_silu_mul_kernel(const uint16_t* __restrict__ gu, int64_t n8, int I8,
                                                           uint16_t* __restrict__ h) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int64_t row = i / I8;
  const int c = (int)(i - row * I8);
  const uint4* src = (const uint4*)gu + row * 2 * I8 + c;
  float g[8], u[8];
  unpack8(src[0], g);
  unpack8(src[I8], u);
#pragma unroll
  for (int j = 0; j < 8; ++j) g[j] = g[j] / (1.f + expf(-g[j])) * u[j];
  ((uint4*)h)[i] = pack8(g);
}

// Gradient of the gating for dh = w_i * dhr[i, :] (w_i: routing weight of sorted row i), written over gu's
// layout: g_gu[i, c] = dh u silu'(g), g_gu[i, I + c] = dh silu(g).
__global__ __launch_bounds__(256) void moe_silu_bwd_kernel(const uint16_t* __restrict__ gu,
                                                           const uint16_t* __restrict__ dhr,
                                                           const float* __restrict__ topk_w,
                                                           const int* __restrict__ perm, int64_t n8, int I8,
                                                           uint16_t* __restrict__ g_gu) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int64_t row = i / I8;
  const int c = (int)(i - row * I8);
  const uint4* src = (const uint4*)gu + row * 2 * I8 + c;
  uint4* dst = (uint4*)g_gu + row * 2 * I8 + c;
  float g[8], u[8], d[8];
  unpack8(src[0], g);
  unpack8(src[I8], u);
  unpack8(((const uint4*)dhr)[i], d);
  const float w = topk_w[perm[row]];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float s = 1.f / (1.f + expf(-g[j])), dh = d[j] * w;
    d[j] = dh * u[j] * (s * (1.f + g[j] * (1.f - s)));
    u[j] = dh * (g[j] * s);
  }
  dst[0] = pack8(d);
  dst[I8] = pack8(u);
}

// out[t, :] = sum_j w[t, j] rows[inv_perm[t k + j], :] in slot order (w == nullptr: plain sum); the k
// sorted rows of a token are read once, 8 columns per thread, eight loads in flight.  Nobody reads
// them again: non-temporal loads, 57 -> 51 us for 65536 rows of 2048, level up to 16384 rows.
__global__ __launch_bounds__(256) void moe_combine_kernel(const uint16_t* __restrict__ rows,
                                                          const int* __restrict__ inv_perm,
                                                          const float* __restrict__ w, int64_t n8, int H8, int k,
                                                          uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int64_t t = i / H8;
  const int c = (int)(i - t * H8);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < k; j0 += 8) {
    uint4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
      u32x4 x = {0, 0, 0, 0};
      if (j0 + j < k) {
        const u32x4* src = (const u32x4*)rows + (int64_t)inv_perm[t * k + j0 + j] * H8 + c;
        x = __builtin_nontemporal_load(src);
      }
      v[j] = make_uint4(x[0], x[1], x[2], x[3]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float wj = j0 + j >= k ? 0.f : (w ? w[t * k + j0 + j] : 1.f);
      float f[8];
      unpack8(v[j], f);
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] += wj * f[q];
    }
  }
  ((uint4*)out)[i] = pack8(acc);
}

__global__ __launch_bounds__(256) void transpose_bf16_batched_kernel(const uint16_t* __restrict__ in,
                                                                     uint16_t* __restrict__ out,
                                                                     int64_t R, int64_t C) {
  __shared__ uint16_t tile[64][66];
  in += (int64_t)blockIdx.z * R * C;
  out += (int64_t)blockIdx.z * R * C;
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    int64_t r = r0 + i, c = c0 + tx;
    tile[i][tx] = (r < R && c < C) ? in[r * C + c] : (uint16_t)0;
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    int64_t c = c0 + i, r = r0 + tx;
    if (c < C && r < R) out[c * R + r] = tile[tx][i];
  }
}

static int32_t check_moe(int64_t n_rows, int64_t in, int64_t out, int E, int r) {
  ARTK_CHECK_ARG(n_rows > 0 && in > 0 && out > 0 && E > 0 && r > 0, "sizes must be positive");
  if (in % BK != 0 || out % BK != 0) {
    set_error("in (%lld) and out (%lld) must be multiples of %d", (long long)in, (long long)out, BK);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  if (r % 8 != 0 || r > 64 || E > MOE_MAX_E) {
    set_error("LoRA rank must be a multiple of 8 and <= 64, experts <= %d", MOE_MAX_E);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  if (n_rows >= (1ll << 31) / 8) {
    set_error("too many rows");
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  return ARTK_OK;
}

// Up to SG_COLS rows per expert the streaming kernel is the faster one.  Four products of a block, us, 256 x 256 tiles
// / streamed (hidden 2048, intermediate 768): 128 experts, 203 tokens (13 rows each) 517 / 423, 512 (32) 569 / 498,
// 1024 (64) 681 / 579, 2048 (128) 728 / 705, 3000 (188) 888 / 868; 64 experts, 400 tokens (50) 333 / 279,
// 1024 (128) 405 / 389, 1300 (163) 418 / 432.
static bool moe_streams(int64_t n_rows, int E) { return n_rows <= (int64_t)E * SG_COLS; }

// For a product whose routing did not leave the order (2 us).
static int32_t launch_moe_order(const int* offsets, int64_t n_rows, int E, int* order, hipStream_t st) {
  if (!moe_streams(n_rows, E)) return ARTK_OK;
  moe_order_kernel<<<1, MOE_MAX_E, 0, st>>>(offsets, E, order);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

// order: read by the streaming kernel only.
static int32_t launch_moe_gemm(const void* W, const void* X, const int* gather, const uint16_t* Pe,
                               const uint16_t* Qe, void* out, const int* offsets,
                               const int* tile_prefix, int64_t n_rows, int64_t M, int64_t K, int E,
                               int r, int RP, const int* order, hipStream_t st) {
  MoeGemmParams p;
  p.W = W;
  p.X = X;
  p.gather = gather;
  p.Pe = Pe;
  p.Qe = Qe;
  p.out = (uint16_t*)out;
  p.offsets = offsets;
  p.tile_prefix = tile_prefix;
  p.M = M;
  p.K = K;
  p.E = E;
  p.r = r;
  p.RP = RP;
  p.MT = (int)((M + TILE - 1) / TILE);
  const int64_t max_row_tiles = (n_rows + TILE - 1) / TILE + E;
  prof_begin(PROF_MOE_GEMM, st);
  if (moe_streams(n_rows, E)) {
    p.MT = (int)((M + SG_ROWS - 1) / SG_ROWS);
    p.order = order;
    // (as many as there are units if the XCDs' shares are even; the rest comes in a second turn)
    const int64_t per_xcd = (E + 7) / 8 + (n_rows + 8 * SG_COLS - 1) / (8 * SG_COLS);
    moe_stream_gemm_kernel<<<(unsigned)(8 * per_xcd * p.MT), 256, 0, st>>>(p);
  } else {
    // persistent: one work-group per CU walks the device-side work list
    const int cus = num_cus();
    const int64_t upper = (int64_t)max_row_tiles * p.MT;
    moe_gemm_kernel<<<(unsigned)(upper < cus ? upper : cus), nthreads<MOE_NI>(), 0, st>>>(p);
  }
  prof_end(PROF_MOE_GEMM, st);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

static int32_t launch_moe_rowdot(const void* X, const int* gather, const uint16_t* Mt,
                                 const int* offsets, const int* blk_prefix, int64_t n_rows, int E,
                                 int64_t K, int R, int RP, float scale, float* out_f32,
                                 uint16_t* out_bf16, hipStream_t st, const float* row_w = nullptr,
                                 const int* row_idx = nullptr) {
  dim3 grid((unsigned)((n_rows + 15) / 16 + E), (unsigned)(RP / 16));
  moe_rowdot16_kernel<<<grid, 256, 0, st>>>((const uint16_t*)X, gather, Mt, offsets, blk_prefix, E, K,
                                            R, RP, scale, row_w, row_idx, out_f32, out_bf16);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

}  // namespace artk

using namespace artk;

extern "C" {

static unsigned blocks256(int64_t n) { return (unsigned)((n + 255) / 256); }

size_t artk_moe_route_workspace_bytes(int64_t T, int32_t E, int32_t k) {
  Workspace ws(nullptr, 0);
  const int64_t n = T * k;
  const int64_t nb = (n + PERM_CHUNK - 1) / PERM_CHUNK;
  ws.take<int>((size_t)(nb * E));
  ws.take<int>((size_t)(nb * E));
  return ws.used + 256;
}

static int32_t moe_route(const float* router_logits, int64_t T, int32_t E, int32_t k, int32_t* topk_idx,
                         float* topk_w, int32_t* perm, int32_t* inv_perm, int32_t* row_token,
                         int32_t* expert_offsets, int32_t* tile_prefix, int32_t* blk_prefix, int32_t* order,
                         const MoePack* pack, void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  ARTK_CHECK_ARG(router_logits && topk_idx && topk_w && perm && inv_perm && row_token &&
                     expert_offsets && tile_prefix && blk_prefix,
                 "null pointer argument");
  ARTK_CHECK_ARG(T > 0 && E > 0 && k > 0 && k <= E, "T, E, k must be positive and k <= E");
  if (E > MOE_MAX_E || k > MOE_MAX_K || T * k >= (1ll << 30)) {
    set_error("supported: experts <= %d, top-k <= %d", MOE_MAX_E, MOE_MAX_K);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  const int n = (int)(T * k);
  const int nb = (n + PERM_CHUNK - 1) / PERM_CHUNK;
  Workspace ws(workspace, workspace_bytes);
  int* cnt = ws.take<int>((size_t)nb * E);
  int* base = ws.take<int>((size_t)nb * E);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t pack_blocks = pack ? blocks256((int64_t)pack->E * pack->r * (2 * pack->H + 3 * pack->I) / 64) : 0;
  moe_topk_pack_kernel<<<(unsigned)((T + 3) / 4 + pack_blocks), 256, 0, st>>>(router_logits, T, E, k, topk_idx, topk_w,
                                                                              pack ? *pack : MoePack{});
  ARTK_CHECK_LAUNCH();
  const MoeScanOut scan{expert_offsets, tile_prefix, blk_prefix, order};
  const MoePerm out{perm, inv_perm, row_token};
  if (nb <= SORT_CHUNKS) {
    moe_sort_kernel<<<1, PERM_CHUNK, 0, st>>>(topk_idx, n, E, k, scan, out);
    ARTK_CHECK_LAUNCH();
    return ARTK_OK;
  }
  moe_hist_kernel<<<nb, PERM_CHUNK, 0, st>>>(topk_idx, n, E, cnt);
  ARTK_CHECK_LAUNCH();
  moe_scan_kernel<<<1, SCAN_PARTS * MOE_MAX_E, 0, st>>>(cnt, nb, E, base, scan);
  ARTK_CHECK_LAUNCH();
  moe_scatter_kernel<<<nb, PERM_CHUNK, 0, st>>>(topk_idx, n, E, k, base, out);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

int32_t artk_moe_route(const float* router_logits, int64_t T, int32_t E, int32_t k, int32_t* topk_idx,
                       float* topk_w, int32_t* perm, int32_t* inv_perm, int32_t* row_token,
                       int32_t* expert_offsets, int32_t* tile_prefix, int32_t* blk_prefix,
                       void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  return moe_route(router_logits, T, E, k, topk_idx, topk_w, perm, inv_perm, row_token, expert_offsets, tile_prefix,
                   blk_prefix, nullptr, nullptr, workspace, workspace_bytes, stream);
}

size_t artk_moe_lora_grouped_fwd_workspace_bytes(int64_t n_rows, int64_t in, int64_t out, int32_t E,
                                                 int32_t r) {
  (void)in;
  (void)out;
  Workspace ws(nullptr, 0);
  ws.take<uint16_t>((size_t)n_rows * round16(r));
  ws.take<int>((size_t)E + 1);
  return ws.used + 256;
}

int32_t artk_moe_lora_grouped_fwd(const void* x, const int32_t* gather, const void* W, const void* A,
                                  const void* B, float scale, const int32_t* expert_offsets,
                                  const int32_t* tile_prefix, const int32_t* blk_prefix,
                                  int64_t n_rows, int64_t in, int64_t out, int32_t E, int32_t r,
                                  void* y, float* xa, void* workspace, size_t workspace_bytes,
                                  artk_stream_t stream) {
  int32_t rc = check_moe(n_rows, in, out, E, r);
  if (rc) return rc;
  ARTK_CHECK_ARG(x && W && A && B && expert_offsets && tile_prefix && blk_prefix && y && xa,
                 "null pointer argument");
  ARTK_CHECK_ARG(aligned16(x) && aligned16(W) && aligned16(A) && aligned16(B) && aligned16(y),
                 "pointers must be 16-byte aligned");
  // gathered rows are addressed with 31-bit byte offsets from x; gather[i] < n_rows
  if (gather != nullptr && n_rows * in * 2 >= (1ll << 31)) {
    set_error("with a row gather, n_rows * in * 2 bytes (%lld) must stay below 2 GiB",
              (long long)(n_rows * in * 2));
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  const int RP = round16(r);
  Workspace ws(workspace, workspace_bytes);
  uint16_t* xa16 = ws.take<uint16_t>((size_t)n_rows * RP);
  int* order = ws.take<int>((size_t)E + 1);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  if ((rc = launch_moe_rowdot(x, gather, (const uint16_t*)A, expert_offsets, blk_prefix, n_rows, E, in,
                              r, RP, scale, xa, xa16, st)))
    return rc;
  if ((rc = launch_moe_order(expert_offsets, n_rows, E, order, st))) return rc;
  return launch_moe_gemm(W, x, gather, (const uint16_t*)B, xa16, y, expert_offsets, tile_prefix, n_rows,
                         out, in, E, r, RP, order, st);
}

// Scratch of the grouped backward, carved in the same order by the size query and the call.
struct MoeBwdScratch {
  uint16_t *Bt, *At, *gb16;
  float *gb, *rowp, *dummy;
  int* order;
};
static void carve_moe_bwd(Workspace& ws, int64_t n_rows, int64_t in, int64_t out, int E, int r, MoeBwdScratch& c) {
  const int RP = round16(r);
  c.Bt = ws.take<uint16_t>((size_t)E * r * out);  // [E,r,out]
  c.At = ws.take<uint16_t>((size_t)E * in * r);   // [E,in,r]
  c.gb = ws.take<float>((size_t)n_rows * r);
  c.gb16 = ws.take<uint16_t>((size_t)n_rows * RP);
  c.rowp = ws.take<float>((size_t)stats_grouped_chunks(n_rows, out, r, E, false) * n_rows * r);
  c.dummy = ws.take<float>(1024);
  c.order = ws.take<int>((size_t)E + 1);
}

size_t artk_moe_lora_grouped_bwd_workspace_bytes(int64_t n_rows, int64_t in, int64_t out, int32_t E,
                                                 int32_t r) {
  Workspace ws(nullptr, 0);
  MoeBwdScratch c;
  carve_moe_bwd(ws, n_rows, in, out, E, r, c);
  return ws.used + 256;
}

int32_t artk_moe_lora_grouped_bwd(const void* g, const void* x, const int32_t* gather, const void* W_t,
                                  const void* A, const void* B, const float* xa, float scale,
                                  const int32_t* expert_offsets, const int32_t* tile_prefix,
                                  const int32_t* blk_prefix, int64_t n_rows, int64_t in, int64_t out,
                                  int32_t E, int32_t r, void* dx, float* dA, float* dB,
                                  void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  int32_t rc = check_moe(n_rows, in, out, E, r);
  if (rc) return rc;
  ARTK_CHECK_ARG(g && x && W_t && A && B && xa && expert_offsets && tile_prefix && blk_prefix && dx &&
                     dA && dB,
                 "null pointer argument");
  ARTK_CHECK_ARG(aligned16(g) && aligned16(x) && aligned16(W_t) && aligned16(A) && aligned16(B) && aligned16(dx) && aligned16(xa) &&
                     aligned16(dA) && aligned16(dB),
                 "pointers must be 16-byte aligned");
  if (n_rows * (in > out ? in : out) * 2 >= (1ll << 31)) {
    set_error("n_rows * max(in, out) * 2 bytes (%lld) must stay below 2 GiB (31-bit row offsets)",
              (long long)(n_rows * (in > out ? in : out) * 2));
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  const int RP = round16(r);
  Workspace ws(workspace, workspace_bytes);
  MoeBwdScratch c;
  carve_moe_bwd(ws, n_rows, in, out, E, r, c);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  if ((rc = launch_small_transpose2(B, c.Bt, E, out, r, A, c.At, E, r, in, st))) return rc;
  // one pass over g: g B_e per row (partials over column chunks) and dB_e = s g^T (x A_e^T) per expert
  if ((rc = launch_stats_grouped(g, n_rows, nullptr, n_rows, out, c.Bt, xa, r, E, expert_offsets, c.rowp, dB,
                                 scale, 0, c.dummy, st)))
    return rc;
  {
    StatsReduceJob ja{c.rowp, stats_grouped_chunks(n_rows, out, r, E, false), n_rows, 1.f, c.gb, 0, c.gb16, RP, scale};
    StatsReduceJob jb{nullptr, 0, 0, 0.f, nullptr, 0, nullptr, 0, 0.f};
    if ((rc = launch_stats_reduce(ja, jb, r, st))) return rc;
  }
  if ((rc = launch_moe_order(expert_offsets, n_rows, E, c.order, st))) return rc;
  if ((rc = launch_moe_gemm(W_t, g, nullptr, c.At, c.gb16, dx, expert_offsets, tile_prefix, n_rows, in, out,
                            E, r, RP, c.order, st)))
    return rc;
  // one pass over x (through the row gather when there is one): dA_e [r,in] = s (g B_e)^T x
  return launch_stats_grouped(x, gather ? (int64_t)0x3fffffff / in : n_rows, gather, n_rows, in, nullptr, c.gb, r,
                              E, expert_offsets, nullptr, dA, scale, 1, c.dummy, st);
}

// ---- the whole expert block ---------------------------------------------------------------------------
// What the forward leaves for the backward, carved in the same order by the size query and both calls.
struct MoeSaved {
  uint16_t *Bt_gu, *At_gu, *Bt_d, *At_d;  // bf16 adapters, transposed: [E,2r,2I], [E,H,2r], [E,r,H], [E,I,r]
  float *xa_gu, *xaw_d;               // x A^T [n,2r]; routing weight times h A_d^T [n,r]
  uint16_t *gu, *h;                   // gate|up [n,2I], silu(gate) up [n,I]
  int* order;                         // [E+1] experts by falling number of rows, then moe_split_rows
};
static void carve_moe_saved(Workspace& ws, const artk_moe_experts_t& a, MoeSaved& c, bool backward = true) {
  const size_t n = (size_t)(a.T * a.k), E = (size_t)a.E, r = (size_t)a.r, H = (size_t)a.H, I = (size_t)a.I;
  c.Bt_gu = c.At_gu = c.Bt_d = c.At_d = nullptr;
  if (backward) {
    c.Bt_gu = ws.take<uint16_t>(E * 2 * r * 2 * I);
    c.At_gu = ws.take<uint16_t>(E * H * 2 * r);
    c.Bt_d = ws.take<uint16_t>(E * r * H);
    c.At_d = ws.take<uint16_t>(E * I * r);
  }
  c.xa_gu = ws.take<float>(n * 2 * r);
  c.xaw_d = ws.take<float>(n * r);
  c.gu = ws.take<uint16_t>(n * 2 * I);
  c.h = ws.take<uint16_t>(n * I);
  c.order = ws.take<int>(E + 1);
}
struct MoeFwdScratch {
  char* route;
  size_t route_bytes;
  uint16_t *A_gu, *B_gu, *A_d, *B_d;  // bf16 adapters [E,2r,H], [E,2I,2r], [E,r,I], [E,H,r]
  uint16_t *xa16_gu, *xa16_d, *down;
};
static void carve_moe_fwd(Workspace& ws, const artk_moe_experts_t& a, MoeFwdScratch& c) {
  const size_t n = (size_t)(a.T * a.k), E = (size_t)a.E, r = (size_t)a.r, H = (size_t)a.H, I = (size_t)a.I;
  c.A_gu = ws.take<uint16_t>(E * 2 * r * H);
  c.B_gu = ws.take<uint16_t>(E * 2 * I * 2 * r);
  c.A_d = ws.take<uint16_t>(E * r * I);
  c.B_d = ws.take<uint16_t>(E * H * r);
  c.route_bytes = artk_moe_route_workspace_bytes(a.T, a.E, a.k);
  c.route = ws.take<char>(c.route_bytes);
  c.xa16_gu = ws.take<uint16_t>(n * round16(2 * a.r));
  c.xa16_d = ws.take<uint16_t>(n * round16(a.r));
  c.down = ws.take<uint16_t>(n * a.H);
}
struct MoeBlockBwdScratch {
  float *gb, *rowp, *dummy;
  uint16_t *gb16, *dhr, *g_gu, *dx_rows;
};
static void carve_moe_block_bwd(Workspace& ws, const artk_moe_experts_t& a, MoeBlockBwdScratch& c) {
  const size_t n = (size_t)(a.T * a.k), r = (size_t)a.r, H = (size_t)a.H, I = (size_t)a.I;
  const size_t p_d = (size_t)stats_grouped_chunks(a.T * a.k, a.H, a.r, a.E, true) * r;
  const size_t p_gu = (size_t)stats_grouped_chunks(a.T * a.k, 2 * a.I, 2 * a.r, a.E, true) * 2 * r;
  c.rowp = ws.take<float>((p_d > p_gu ? p_d : p_gu) * n);
  c.gb = ws.take<float>(n * 2 * r);
  c.gb16 = ws.take<uint16_t>(n * round16(2 * a.r));
  c.dummy = ws.take<float>(1024);
  c.dhr = ws.take<uint16_t>(n * I);
  c.g_gu = ws.take<uint16_t>(n * 2 * I);
  c.dx_rows = ws.take<uint16_t>(n * H);
}

static int32_t check_moe_experts(const artk_moe_experts_t* a, bool backward, bool saved = true) {
  ARTK_CHECK_ARG(a != nullptr, "null argument");
  ARTK_CHECK_ARG(a->T > 0 && a->k > 0 && a->E > 0 && a->k <= a->E, "T, E, k must be positive and k <= E");
  if (a->E > MOE_MAX_E || a->k > MOE_MAX_K || a->T * a->k >= (1ll << 30)) {
    set_error("supported: experts <= %d, top-k <= %d", MOE_MAX_E, MOE_MAX_K);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  const int64_t n = a->T * a->k;
  int32_t rc = check_moe(n, a->H, 2 * a->I, a->E, 2 * a->r);
  if (rc == 0) rc = check_moe(n, a->I, a->H, a->E, a->r);
  if (rc) return rc;
  const int64_t widest = backward && 2 * a->I > a->H ? 2 * a->I : a->H;
  if (n * widest * 2 >= (1ll << 31)) {
    set_error("T * k * %lld * 2 bytes (%lld) must stay below 2 GiB (31-bit row offsets)", (long long)widest,
              (long long)(n * widest * 2));
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  ARTK_CHECK_ARG(a->x && a->topk_idx && a->topk_w && a->perm && a->inv_perm && a->row_token && a->offsets &&
                     a->tile_prefix && a->blk_prefix && (a->saved || !saved),
                 "null pointer argument");
  ARTK_CHECK_ARG(aligned16(a->x) && (aligned16(a->saved) || !saved), "pointers must be 16-byte aligned");
  return ARTK_OK;
}

size_t artk_moe_experts_saved_bytes(const artk_moe_experts_t* a) {
  Workspace ws(nullptr, 0);
  MoeSaved c;
  carve_moe_saved(ws, *a, c);
  return ws.used + 256;
}
size_t artk_moe_experts_fwd_workspace_bytes(const artk_moe_experts_t* a) {
  Workspace ws(nullptr, 0);
  MoeFwdScratch c;
  carve_moe_fwd(ws, *a, c);
  return ws.used + 256;
}
size_t artk_moe_experts_eval_workspace_bytes(const artk_moe_experts_t* a) {
  Workspace ws(nullptr, 0);
  MoeSaved s;
  MoeFwdScratch c;
  carve_moe_saved(ws, *a, s, false);
  carve_moe_fwd(ws, *a, c);
  return ws.used + 256;
}
size_t artk_moe_experts_bwd_workspace_bytes(const artk_moe_experts_t* a) {
  Workspace ws(nullptr, 0);
  MoeBlockBwdScratch c;
  carve_moe_block_bwd(ws, *a, c);
  return ws.used + 256;
}


static int32_t launch_moe_combine(const uint16_t* rows, const artk_moe_experts_t* a, const float* w, void* out, hipStream_t st) {
  const int64_t n8 = a->T * a->H / 8;
  moe_combine_kernel<<<blocks256(n8), 256, 0, st>>>(rows, a->inv_perm, w, n8, (int)(a->H / 8), a->k, (uint16_t*)out);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

// The forward pass; with `backward` the buffer a->saved keeps what one needs, else everything lies in the workspace.
static int32_t moe_experts_forward(const artk_moe_experts_t* a, bool backward, void* workspace, size_t workspace_bytes,
                                   artk_stream_t stream) {
  int32_t rc = check_moe_experts(a, false, backward);
  if (rc) return rc;
  ARTK_CHECK_ARG(a->router_logits && a->W_gu && a->W_d && a->gate_A && a->gate_B && a->up_A && a->up_B && a->down_A &&
                     a->down_B && a->y,
                 "null pointer argument");
  ARTK_CHECK_ARG(aligned16(a->W_gu) && aligned16(a->W_d) && aligned16(a->gate_A) && aligned16(a->gate_B) &&
                     aligned16(a->up_A) && aligned16(a->up_B) && aligned16(a->down_A) && aligned16(a->down_B) &&
                     aligned16(a->y),
                 "pointers must be 16-byte aligned");
  Workspace ws(workspace, workspace_bytes), sv(a->saved, a->saved_bytes);
  MoeFwdScratch c;
  MoeSaved s;
  carve_moe_saved(backward ? sv : ws, *a, s, backward);
  carve_moe_fwd(ws, *a, c);
  if (!ws.ok() || (backward && !sv.ok())) {
    set_error("workspace too small: need %zu and %zu bytes, got %zu and %zu", ws.used, sv.used, workspace_bytes,
              a->saved_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t n = a->T * a->k, H = a->H, I = a->I;
  const int E = a->E, r = a->r;
  const MoePack pack{a->gate_A, a->gate_B, a->up_A, a->up_B, a->down_A, a->down_B,
                     c.A_gu, c.B_gu, c.A_d, c.B_d, s.At_gu, s.Bt_gu, s.At_d, s.Bt_d, H, I, E, r, a->adapters_bf16};
  if ((rc = moe_route(a->router_logits, a->T, E, a->k, a->topk_idx, a->topk_w, a->perm, a->inv_perm, a->row_token,
                      a->offsets, a->tile_prefix, a->blk_prefix, s.order, &pack, c.route, c.route_bytes, stream)))
    return rc;
  if ((rc = launch_moe_rowdot(a->x, a->row_token, c.A_gu, a->offsets, a->blk_prefix, n, E, H, 2 * r, round16(2 * r),
                              a->scale, s.xa_gu, c.xa16_gu, st)))
    return rc;
  if ((rc = launch_moe_gemm(a->W_gu, a->x, a->row_token, c.B_gu, c.xa16_gu, s.gu, a->offsets, a->tile_prefix, n, 2 * I,
                            H, E, 2 * r, round16(2 * r), s.order, st)))
    return rc;
  moe_silu_mul_kernel<<<blocks256(n * I / 8), 256, 0, st>>>(s.gu, n * I / 8, (int)(I / 8), s.h);
  ARTK_CHECK_LAUNCH();
  if ((rc = launch_moe_rowdot(s.h, nullptr, c.A_d, a->offsets, a->blk_prefix, n, E, I, r, round16(r), a->scale,
                              s.xaw_d, c.xa16_d, st, a->topk_w, a->perm)))
    return rc;
  if ((rc = launch_moe_gemm(a->W_d, s.h, nullptr, c.B_d, c.xa16_d, c.down, a->offsets, a->tile_prefix, n, H, I, E, r,
                            round16(r), s.order, st)))
    return rc;
  return launch_moe_combine(c.down, a, a->topk_w, a->y, st);
}

int32_t artk_moe_experts_fwd(const artk_moe_experts_t* a, void* workspace, size_t workspace_bytes,
                             artk_stream_t stream) {
  return moe_experts_forward(a, true, workspace, workspace_bytes, stream);
}
int32_t artk_moe_experts_eval(const artk_moe_experts_t* a, void* workspace, size_t workspace_bytes,
                              artk_stream_t stream) {
  return moe_experts_forward(a, false, workspace, workspace_bytes, stream);
}

int32_t artk_moe_experts_bwd(const artk_moe_experts_t* a, void* workspace, size_t workspace_bytes,
                             artk_stream_t stream) {
  int32_t rc = check_moe_experts(a, true);
  if (rc) return rc;
  ARTK_CHECK_ARG(a->g && a->Wt_gu && a->Wt_d && a->dx && a->dgate_A && a->dgate_B && a->dup_A && a->dup_B &&
                     a->ddown_A && a->ddown_B,
                 "null pointer argument");
  ARTK_CHECK_ARG(aligned16(a->g) && aligned16(a->Wt_gu) && aligned16(a->Wt_d) && aligned16(a->dx) &&
                     aligned16(a->dgate_A) && aligned16(a->dgate_B) && aligned16(a->dup_A) && aligned16(a->dup_B) &&
                     aligned16(a->ddown_A) && aligned16(a->ddown_B),
                 "pointers must be 16-byte aligned");
  Workspace ws(workspace, workspace_bytes), sv(a->saved, a->saved_bytes);
  MoeBlockBwdScratch c;
  MoeSaved s;
  carve_moe_block_bwd(ws, *a, c);
  carve_moe_saved(sv, *a, s);
  if (!ws.ok() || !sv.ok()) {
    set_error("workspace too small: need %zu and %zu bytes, got %zu and %zu", ws.used, sv.used, workspace_bytes,
              a->saved_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t n = a->T * a->k, H = a->H, I = a->I;
  const int E = a->E, r = a->r;
  const StatsBlock down{s.order}, gate_up_B{s.order, a->dup_B, r, I}, gate_up_A{s.order, a->dup_A, r, 0};
  const StatsReduceJob none{nullptr, 0, 0, 0.f, nullptr, 0, nullptr, 0, 0.f};
  // down, on the unweighted rows g[token]: g B_d per row and dB_d = s g^T (w h A_d^T) in one pass
  if ((rc = launch_stats_grouped(a->g, a->T, a->row_token, n, H, s.Bt_d, s.xaw_d, r, E, a->offsets, c.rowp, a->ddown_B,
                                 a->scale, 0, c.dummy, st, &down)))
    return rc;
  {
    StatsReduceJob ja{c.rowp, stats_grouped_chunks(n, H, r, E, true), n, 1.f, c.gb, 0, c.gb16, round16(r), a->scale};
    ja.row_w = a->topk_w;
    ja.row_idx = a->perm;
    if ((rc = launch_stats_reduce(ja, none, r, st))) return rc;
  }
  if ((rc = launch_moe_gemm(a->Wt_d, a->g, a->row_token, s.At_d, c.gb16, c.dhr, a->offsets, a->tile_prefix, n, I, H, E,
                            r, round16(r), s.order, st)))
    return rc;
  if ((rc = launch_stats_grouped(s.h, n, nullptr, n, I, nullptr, c.gb, r, E, a->offsets, nullptr, a->ddown_A, a->scale,
                                 1, c.dummy, st, &down)))
    return rc;
  moe_silu_bwd_kernel<<<blocks256(n * I / 8), 256, 0, st>>>(s.gu, c.dhr, a->topk_w, a->perm, n * I / 8, (int)(I / 8),
                                                            c.g_gu);
  ARTK_CHECK_LAUNCH();
  // gate|up
  if ((rc = launch_stats_grouped(c.g_gu, n, nullptr, n, 2 * I, s.Bt_gu, s.xa_gu, 2 * r, E, a->offsets, c.rowp,
                                 a->dgate_B, a->scale, 0, c.dummy, st, &gate_up_B)))
    return rc;
  {
    StatsReduceJob ja{c.rowp, stats_grouped_chunks(n, 2 * I, 2 * r, E, true), n, 1.f, c.gb, 0, c.gb16, round16(2 * r),
                      a->scale};
    if ((rc = launch_stats_reduce(ja, none, 2 * r, st))) return rc;
  }
  if ((rc = launch_moe_gemm(a->Wt_gu, c.g_gu, nullptr, s.At_gu, c.gb16, c.dx_rows, a->offsets, a->tile_prefix, n, H,
                            2 * I, E, 2 * r, round16(2 * r), s.order, st)))
    return rc;
  if ((rc = launch_stats_grouped(a->x, a->T, a->row_token, n, H, nullptr, c.gb, 2 * r, E, a->offsets, nullptr,
                                 a->dgate_A, a->scale, 1, c.dummy, st, &gate_up_A)))
    return rc;
  return launch_moe_combine(c.dx_rows, a, nullptr, a->dx, st);
}

int32_t artk_transpose_bf16_batched(const void* in, void* out, int64_t n, int64_t R, int64_t C,
                                    artk_stream_t stream) {
  ARTK_CHECK_ARG(in && out, "null pointer argument");
  ARTK_CHECK_ARG(n > 0 && n < 65536 && R > 0 && C > 0, "n, R, C must be positive (n < 65536)");
  dim3 grid((unsigned)((C + 63) / 64), (unsigned)((R + 63) / 64), (unsigned)n);
  transpose_bf16_batched_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)in,
                                                                       (uint16_t*)out, R, C);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

}  // extern "C"
