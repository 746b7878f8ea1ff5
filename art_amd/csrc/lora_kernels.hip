// LoRA linear forward / backward for gfx950:
//   y  = x W^T + s (x A^T) B^T
//   dx = g W   + s (g B) A        dA = s (g B)^T x        dB = s g^T (x A^T)
// W [out,in] frozen bf16, A [r,in], B [out,r], s = alpha / r.
//
// The reference configures this layer (src/art/local/state.py:86-92,
// src/art/dev/model.py:52-67: r = 8, alpha = 16, seven target modules) and
// leaves the arithmetic to peft 0.15.2 / unsloth 2025.5.1; the formulas above
// are those packages' documented LoRA linear.
//
// The dense products run on the shared 256x256 MFMA main loop.  The rank-r
// products ride along as extra K = 16 MFMA steps whose operands (the low-rank
// factors) are read straight from global memory, so y and dx are each one GEMM
// launch.  The skinny products are bandwidth-bound: x A^T in the forward is a row
// product (rowdot_multi_kernel); in the backward g B and dB come from one pass over g
// and dA from one pass over x (lora_stats_kernel, skinny_stats.hpp).
#include "common.hpp"
#include "gemm_nt.hpp"
#include "gemm_plain8.hpp"
#include "gemm_small.hpp"
#include "lora_common.hpp"
#include "skinny_stats.hpp"

namespace artk {

constexpr int LORA_NI = 2;  // 8 waves, 2 per SIMD (see gemm_nt.hpp)

// ----------------------------------------------------------------------------
// out[n, m] = sum_k Q[n,k] P[m,k] + sum_e Qe[n,e] Pe[m,e]     (bf16 out)
// ----------------------------------------------------------------------------
struct LoraGemmParams {
  const void* P;       // [M,K] row operand (weight)
  const void* Q;       // [N,K] column operand (activations)
  const uint16_t* Pe;  // [M,r] low-rank factor of the row operand, or nullptr
  const uint16_t* Qe;  // [N,RP] low-rank factor of the column operand (scale folded in, zero padded)
  const uint16_t* bias;  // [M] added to every output row, or nullptr
  uint16_t* out;       // [N,M]
  int64_t M, N, K;
  int r, RP, MT, NT;
};

// Rank-r steps of one tile: acc += sum_e Qe[col, e] Pe[row, e].
__device__ __forceinline__ void lora_tile_lowrank(TileAcc<LORA_NI>& acc, const uint16_t* Pe, int r,
                                                  const uint16_t* Qe, int RP, int64_t M, int64_t N, int mt,
                                                  int nt) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave_m<LORA_NI>(wave), wn = wave_n<LORA_NI>(wave);
  int64_t prow[4], qrow[LORA_NI];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int64_t rr = (int64_t)mt * TILE + wm * 128 + i * 32 + (lane & 31);
    prow[i] = rr < M ? rr : M - 1;
  }
#pragma unroll
  for (int i = 0; i < LORA_NI; ++i) {
    int64_t c = (int64_t)nt * TILE + acc_col<LORA_NI>(wn, i, lane);
    qrow[i] = c < N ? c : N - 1;
  }
  lowrank_steps(acc, Pe, r, r, prow, Qe, RP, RP, qrow, RP);
}

// Optional bias and the bf16 store of one finished tile: out[col, m] (out is [N, M]).
__device__ __forceinline__ void lora_tile_store(TileAcc<LORA_NI>& acc, const uint16_t* bias, uint16_t* out,
                                                int64_t M, int64_t N, int mt, int nt) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave_m<LORA_NI>(wave), wn = wave_n<LORA_NI>(wave);
  const int half = lane >> 5;
  if (bias != nullptr) {
    // element j of tile mi is output feature m0 + (j / 4) 8 + 4 half + j % 4
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
      const int64_t m0 = (int64_t)mt * TILE + wm * 128 + mi * 32;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int64_t mq = m0 + q * 8 + half * 4;
        mq = mq + 4 <= M ? mq : 0;  // rows past the end are never stored
        const bf16x4 bv = *(const bf16x4*)(bias + mq);
#pragma unroll
        for (int ni = 0; ni < LORA_NI; ++ni)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc.c[mi][ni][q * 4 + e] += (float)bv[e];
      }
    }
  }

#pragma unroll
  for (int ni = 0; ni < LORA_NI; ++ni) {
    // lanes l and l + 32 share the column, so they take these branches together
    // (store_block_bf16 exchanges data between them)
    const int64_t col = (int64_t)nt * TILE + acc_col<LORA_NI>(wn, ni, lane);
    const bool col_ok = col < N;
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
      const int64_t m0 = (int64_t)mt * TILE + wm * 128 + mi * 32;
      if (m0 >= M) continue;  // wave-uniform
      if (m0 + 32 <= M) {
        if (col_ok) store_block_bf16(out + col * M + m0, acc.c[mi][ni], half);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int64_t m = m0 + q * 8 + half * 4;
          if (m >= M || !col_ok) continue;
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (__bf16)acc.c[mi][ni][q * 4 + e];
          *(bf16x4*)(out + col * M + m) = o;
        }
      }
    }
  }
}

// Rank-r steps and bf16 store of one finished tile.
__device__ __forceinline__ void lora_gemm_epilogue(TileAcc<LORA_NI>& acc, const LoraGemmParams& p, int mt,
                                                   int nt) {
  if (p.Pe != nullptr) lora_tile_lowrank(acc, p.Pe, p.r, p.Qe, p.RP, p.M, p.N, mt, nt);
  lora_tile_store(acc, p.bias, p.out, p.M, p.N, mt, nt);
}

// Persistent work-groups: tiles t, t + grid, ...; the first DMA stage of the next
// tile is started before the rank-r steps and the store of the current one.
__global__ __launch_bounds__(nthreads<LORA_NI>()) void lora_gemm_kernel(LoraGemmParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[GEMM_LDS_BYTES];
  const int n_tiles = p.MT * p.NT;
  int t = blockIdx.x;
  int mt, nt;
  tile_coords(xcd_remap(t, n_tiles), p.MT, p.NT, mt, nt);
  {
    PlainTileLoaders first;
    first.init(p.P, p.K, (int64_t)mt * TILE, p.M, p.Q, p.K, (int64_t)nt * TILE, p.N, 0, (int)p.K);
    first.issue_first(smem);
  }
  for (;;) {
    const int t2 = t + gridDim.x;
    const bool more = t2 < n_tiles;
    int mt2 = 0, nt2 = 0;
    if (more) tile_coords(xcd_remap(t2, n_tiles), p.MT, p.NT, mt2, nt2);
    TileAcc<LORA_NI> acc;
    acc.zero();
    {
      PlainTileLoaders cur;  // its first stage is already on the way
      cur.init(p.P, p.K, (int64_t)mt * TILE, p.M, p.Q, p.K, (int64_t)nt * TILE, p.N, 0, (int)p.K);
      gemm_tile_run_plain8<false>(acc, smem, cur);
    }
    if (more) {
      PlainTileLoaders nxt;
      nxt.init(p.P, p.K, (int64_t)mt2 * TILE, p.M, p.Q, p.K, (int64_t)nt2 * TILE, p.N, 0, (int)p.K);
      nxt.issue_first(smem);
    }
    lora_gemm_epilogue(acc, p, mt, nt);
    if (!more) break;
    t = t2;
    mt = mt2;
    nt = nt2;
  }
}

// ----------------------------------------------------------------------------
// Several products over one column operand in ONE persistent launch.
// A job is one output matrix out[n, m] (bf16 [N, M]); it sums one or more K segments,
//   out[n, m] = sum_s ( sum_k Q_s[n,k] P_s[m,k] + sum_e Qe_s[n,e] Pe_s[m,e] )  (+ bias[m]).
// Forward of projections that read the same x: one job per projection (P = W_i, Q = x), one
// segment each.  Input gradient of the same projections: one job (dx) whose segments are the
// projections (P = W_i^T [in, out_i], Q = g_i [T, out_i], K = out_i), so the upstream gradients
// are never concatenated and dx is written once.  A segment switch inside a tile costs one
// exposed first-stage fetch (the two LDS stages are busy until the segment's last K step).
// ----------------------------------------------------------------------------
constexpr int LORA_MAX_SEG = ARTK_LORA_MULTI_MAX;
struct LoraSeg {
  const void* P;       // [M,K] row operand
  const void* Q;       // [N,K] column operand
  const uint16_t* Pe;  // [M,r]
  const uint16_t* Qe;  // [N,RP]
  int64_t K;
  int r, RP;
};
struct LoraJob {
  uint16_t* out;         // [N,M]
  const uint16_t* bias;  // [M] or nullptr
  int64_t M;
  int MT, tile0, seg0, nseg;
};
struct LoraMultiParams {
  LoraSeg seg[LORA_MAX_SEG];
  LoraJob job[LORA_MAX_SEG];
  int64_t N;
  int NT, n_jobs, n_tiles;
};

__device__ __forceinline__ void lora_multi_locate(const LoraMultiParams& p, int t, int& j, int& mt, int& nt) {
  const int id = xcd_remap(t, p.n_tiles);
  j = 0;
  while (j + 1 < p.n_jobs && id >= p.job[j + 1].tile0) ++j;
  tile_coords(id - p.job[j].tile0, p.job[j].MT, p.NT, mt, nt);
}

__global__ __launch_bounds__(nthreads<LORA_NI>()) void lora_multi_gemm_kernel(LoraMultiParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[GEMM_LDS_BYTES];
  int t = blockIdx.x;
  int j, mt, nt;
  lora_multi_locate(p, t, j, mt, nt);
  {
    const LoraSeg& sg = p.seg[p.job[j].seg0];
    PlainTileLoaders first;
    first.init(sg.P, sg.K, (int64_t)mt * TILE, p.job[j].M, sg.Q, sg.K, (int64_t)nt * TILE, p.N, 0, (int)sg.K);
    first.issue_first(smem);
  }
  for (;;) {
    const int t2 = t + gridDim.x;
    const bool more = t2 < p.n_tiles;
    int j2 = 0, mt2 = 0, nt2 = 0;
    if (more) lora_multi_locate(p, t2, j2, mt2, nt2);
    const int64_t M = p.job[j].M;
    const int seg0 = p.job[j].seg0, nseg = p.job[j].nseg;
    TileAcc<LORA_NI> acc;
    acc.zero();
    // (one branch around all segments, not one per segment: see gemm_plain8.hpp)
    if (plain8_leader()) {
      for (int s = 0; s < nseg; ++s) {
        const LoraSeg& sg = p.seg[seg0 + s];
        PlainTileLoaders cur;  // the first segment's first stage is already on the way
        cur.init(sg.P, sg.K, (int64_t)mt * TILE, M, sg.Q, sg.K, (int64_t)nt * TILE, p.N, 0, (int)sg.K);
        if (s > 0) cur.issue_first_leader(smem);
        gemm_tile_run<2, 2, false>(acc, smem, cur);
      }
    } else {
      for (int s = 0; s < nseg; ++s) {
        const NoLoaders none{0, (int)p.seg[seg0 + s].K};
        gemm_tile_run<2, 2, false>(acc, smem, none);
      }
    }
    if (more) {
      const LoraSeg& sg = p.seg[p.job[j2].seg0];
      PlainTileLoaders nxt;
      nxt.init(sg.P, sg.K, (int64_t)mt2 * TILE, p.job[j2].M, sg.Q, sg.K, (int64_t)nt2 * TILE, p.N, 0, (int)sg.K);
      nxt.issue_first(smem);
    }
    for (int s = 0; s < nseg; ++s) {
      const LoraSeg& sg = p.seg[seg0 + s];
      if (sg.Pe != nullptr) lora_tile_lowrank(acc, sg.Pe, sg.r, sg.Qe, sg.RP, M, p.N, mt, nt);
    }
    lora_tile_store(acc, p.job[j].bias, p.job[j].out, M, p.N, mt, nt);
    if (!more) break;
    t = t2;
    j = j2;
    mt = mt2;
    nt = nt2;
  }
}

// ----------------------------------------------------------------------------
// The same jobs on 128 x 128 tiles with the K range split over `split` work-groups (gemm_small.hpp), for products
// whose 256 x 256 tiles do not fill the GPU.  Tiles are numbered through the jobs (job[].tile0 and MT count 128-row
// tiles here), unit = tile * split + part.  The parts of a tile are equal shares of the K steps of all segments
// together; with split > 1 each leaves its fp32 accumulators in `part` as [unit][wave][block][4][lane][4] and
// lora_small_reduce_kernel adds them in order.
// ----------------------------------------------------------------------------
struct LoraSmallParams {
  LoraMultiParams m;
  float* part;
  int split, ksteps[LORA_MAX_SEG];   // K steps of all segments of a job
};

__device__ __forceinline__ void lora_small_locate(const LoraSmallParams& p, int tile, int& j, int& mt, int& nt) {
  j = 0;
  while (j + 1 < p.m.n_jobs && tile >= p.m.job[j + 1].tile0) ++j;
  tile_coords(tile - p.m.job[j].tile0, p.m.job[j].MT, p.m.NT, mt, nt);
}

// Bias and bf16 store of the 32 x 32 block whose first output feature is m0 and whose lane's column is col.
__device__ __forceinline__ void lora_block_store(floatx16& c, const uint16_t* bias, uint16_t* out, int64_t M,
                                                 int64_t N, int64_t m0, int64_t col, int half) {
  if (m0 >= M) return;  // wave-uniform; M is a multiple of 64, so blocks are whole
  if (bias != nullptr) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bf16x4 bv = *(const bf16x4*)(bias + m0 + q * 8 + half * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) c[q * 4 + e] += (float)bv[e];
    }
  }
  if (col < N) store_block_bf16(out + col * M + m0, c, half);
}

__global__ __launch_bounds__(ST2_THREADS, 2) void lora_small_gemm_kernel(LoraSmallParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[ST2_LDS_BYTES];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int unit = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = unit / p.split, part = unit - tile * p.split;
  int j, mt, nt;
  lora_small_locate(p, tile, j, mt, nt);
  const LoraJob& job = p.m.job[j];
  const int total = p.ksteps[j];
  int b = (int)((int64_t)total * part / p.split), e = (int)((int64_t)total * (part + 1) / p.split);
  SmallAcc acc;
  acc.zero();
  const int wm = wave >> 1, wn = wave & 1, half = lane >> 5;
  for (int s = 0; s < job.nseg; ++s) {
    const LoraSeg& sg = p.m.seg[job.seg0 + s];
    const int ks = (int)(sg.K / BK);
    const int lo = b < 0 ? 0 : b, hi = e < ks ? e : ks;
    if (lo < hi) {
      SmallPanel lp, lq;
      lp.init(sg.P, sg.K, (int64_t)mt * ST2, job.M, lane);
      lq.init(sg.Q, sg.K, (int64_t)nt * ST2, p.m.N, lane);
      small_tile_run(acc, smem, lp, lq, lo * BK, hi - lo);
    }
    b -= ks;
    e -= ks;
    if (part == 0 && sg.Pe != nullptr) {
      // rank-r steps (see lowrank_steps), by the first part
      for (int e0 = 0; e0 < sg.RP; e0 += 16) {
        const int c = e0 + half * 8;
        const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
        bf16x8 pf[2], qf[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          int64_t pr = (int64_t)mt * ST2 + wm * 64 + i * 32 + (lane & 31), qr = (int64_t)nt * ST2 + wn * 64 + i * 32 + (lane & 31);
          pr = pr < job.M ? pr : job.M - 1;
          qr = qr < p.m.N ? qr : p.m.N - 1;
          pf[i] = *(const bf16x8*)(sg.Pe + pr * sg.r + (c < sg.r ? c : 0));
          qf[i] = *(const bf16x8*)(sg.Qe + qr * sg.RP + c);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) pf[i] = c < sg.r ? pf[i] : z;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc.c[i >> 1][i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pf[i >> 1], qf[i & 1], acc.c[i >> 1][i & 1], 0, 0, 0);
      }
    }
  }
  if (p.split > 1) {
    float* dst = p.part + (((int64_t)unit * 4 + wave) * 4) * 1024 + lane * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(floatx4*)(dst + i * 1024 + 256 * q) = floatx4{acc.c[i >> 1][i & 1][4 * q], acc.c[i >> 1][i & 1][4 * q + 1],
                                                     acc.c[i >> 1][i & 1][4 * q + 2], acc.c[i >> 1][i & 1][4 * q + 3]};
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    lora_block_store(acc.c[i >> 1][i & 1], job.bias, job.out, job.M, p.m.N, (int64_t)mt * ST2 + wm * 64 + (i >> 1) * 32,
                     (int64_t)nt * ST2 + wn * 64 + (i & 1) * 32 + (lane & 31), half);
}

// One work-group per tile and wave of the product kernel, one wave per 32 x 32 block.
__global__ __launch_bounds__(256) void lora_small_reduce_kernel(LoraSmallParams p) {
  const int lane = threadIdx.x & 63, i = threadIdx.x >> 6;
  const int tile = blockIdx.x >> 2, wave = blockIdx.x & 3;
  int j, mt, nt;
  lora_small_locate(p, tile, j, mt, nt);
  const LoraJob& job = p.m.job[j];
  floatx16 c;
#pragma unroll
  for (int k = 0; k < 16; ++k) c[k] = 0.f;
  const float* src = p.part + (((int64_t)tile * p.split * 4 + wave) * 4 + i) * 1024 + lane * 4;
#pragma unroll 4
  for (int s = 0; s < p.split; ++s)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 v = *(const floatx4*)(src + (int64_t)s * 16384 + 256 * q);
#pragma unroll
      for (int k = 0; k < 4; ++k) c[4 * q + k] += v[k];
    }
  lora_block_store(c, job.bias, job.out, job.M, p.m.N, (int64_t)mt * ST2 + (wave >> 1) * 64 + (i >> 1) * 32,
                   (int64_t)nt * ST2 + (wave & 1) * 64 + (i & 1) * 32 + (lane & 31), lane >> 5);
}

// ----------------------------------------------------------------------------
// The same jobs on 256 x 256 tiles with the K range of a tile in `split` parts, for long products of a few tiles: unit =
// tile * split + part, one work-group each; every part leaves its fp32 accumulators in `part` as
// [unit][wave][mi][ni][4][lane][4] and lora_split_reduce_kernel adds them in order.  Tiles are numbered as for the
// persistent kernels (job[].tile0 and MT count 256-row tiles).  Bound by the main loop: half the bytes into LDS per product
// of a 128 x 128 tile, for 0.25 MiB of partials a unit.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(nthreads<LORA_NI>()) void lora_split_gemm_kernel(LoraSmallParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[GEMM_LDS_BYTES];
  // ids run through the tiles of a part first: the 32 work-groups of an XCD share panels of one K range
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int part = id / p.m.n_tiles, tile = id - part * p.m.n_tiles, unit = tile * p.split + part;
  int j, mt, nt;
  lora_small_locate(p, tile, j, mt, nt);
  const LoraJob& job = p.m.job[j];
  const int total = p.ksteps[j];
  const int b = (int)((int64_t)total * part / p.split), e = (int)((int64_t)total * (part + 1) / p.split);
  // the segments that the part's K steps b .. e - 1 fall into (no part is empty); off: first step of segment s0
  int s0 = 0, off = 0;
  while (b >= off + (int)(p.m.seg[job.seg0 + s0].K / BK)) off += (int)(p.m.seg[job.seg0 + s0++].K / BK);
  TileAcc<LORA_NI> acc;
  acc.zero();
  // (one branch around all segments, and no segment skipped inside: see gemm_plain8.hpp)
  if (plain8_leader()) {
    int at = off, s = s0;
    do {
      const LoraSeg& sg = p.m.seg[job.seg0 + s];
      const int ks = (int)(sg.K / BK), lo = b > at ? b - at : 0, hi = e - at < ks ? e - at : ks;
      PlainTileLoaders cur;
      cur.init(sg.P, sg.K, (int64_t)mt * TILE, job.M, sg.Q, sg.K, (int64_t)nt * TILE, p.m.N, lo * BK, hi * BK);
      cur.issue_first_leader(smem);
      gemm_tile_run<2, 2, false>(acc, smem, cur);
      at += ks;
      ++s;
    } while (at < e);
  } else {
    int at = off, s = s0;
    do {
      const int ks = (int)(p.m.seg[job.seg0 + s].K / BK), lo = b > at ? b - at : 0, hi = e - at < ks ? e - at : ks;
      const NoLoaders none{lo * BK, hi * BK};
      gemm_tile_run<2, 2, false>(acc, smem, none);
      at += ks;
      ++s;
    } while (at < e);
  }
  // rank-r steps, by the first part
  for (int s = 0; s < (part == 0 ? job.nseg : 0); ++s) {
    const LoraSeg& sg = p.m.seg[job.seg0 + s];
    if (sg.Pe != nullptr) lora_tile_lowrank(acc, sg.Pe, sg.r, sg.Qe, sg.RP, job.M, p.m.N, mt, nt);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float* dst = p.part + ((int64_t)unit * 8 + wave) * 8192 + lane * 4;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < LORA_NI; ++ni)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(floatx4*)(dst + (mi * LORA_NI + ni) * 1024 + 256 * q) =
            floatx4{acc.c[mi][ni][4 * q], acc.c[mi][ni][4 * q + 1], acc.c[mi][ni][4 * q + 2], acc.c[mi][ni][4 * q + 3]};
}

// One wave per 32 x 32 block: 16 work-groups per tile.
__global__ __launch_bounds__(256) void lora_split_reduce_kernel(LoraSmallParams p) {
  const int lane = threadIdx.x & 63;
  const int tile = blockIdx.x >> 4, blk = (blockIdx.x & 15) * 4 + (threadIdx.x >> 6);  // blk = wave * 8 + mi * 2 + ni
  const int wave = blk >> 3, mi = (blk >> 1) & 3, ni = blk & 1;
  int j, mt, nt;
  lora_small_locate(p, tile, j, mt, nt);
  const LoraJob& job = p.m.job[j];
  const int64_t m0 = (int64_t)mt * TILE + wave_m<LORA_NI>(wave) * 128 + mi * 32;
  const int64_t col = (int64_t)nt * TILE + acc_col<LORA_NI>(wave_n<LORA_NI>(wave), ni, lane);
  if (m0 >= job.M || (int64_t)nt * TILE + wave_n<LORA_NI>(wave) * 64 + ni * 32 >= p.m.N) return;  // wave-uniform
  floatx16 c;
#pragma unroll
  for (int k = 0; k < 16; ++k) c[k] = 0.f;
  const float* src = p.part + ((int64_t)tile * p.split * 64 + blk) * 1024 + lane * 4;
#pragma unroll 4
  for (int s = 0; s < p.split; ++s)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 v = *(const floatx4*)(src + (int64_t)s * 65536 + 256 * q);
#pragma unroll
      for (int k = 0; k < 4; ++k) c[4 * q + k] += v[k];
    }
  lora_block_store(c, job.bias, job.out, job.M, p.m.N, m0, col, lane >> 5);
}

// ----------------------------------------------------------------------------
// Row products of one X with several factors: out_i[t, j] = sum_k X[t,k] Mt_i[j,k], Mt_i [R_i,K], on MFMA 16x16x32.
// The factor rows of all i are numbered through (e0[i] ..); a work-group takes 16 NJ of them (blockIdx.y) and 16 rows of
// X.  K is dealt to its four waves in pieces of 64 (two MFMA steps; a lane takes 32 contiguous bytes of its row, so a wave
// reads whole cache lines), two of them in flight at a time.  Writes f32 [T,R] (unscaled) and bf16 [T,RP] (scaled, zero
// padded to RP).
// Where there are rows enough the factors are packed (e0 by R: two ranks of 8 are one block) and X is read once for
// ranks that add up to 64; else every 16 factor rows are a work-group's, every factor starts a block of its own (e0 by RP) and
// there are more work-groups.  us, a work-group per 16 rows and factor / packed: [8192, 2048] and 2 ranks of 8 21 / 14,
// [4096, 2048] and 3 of 8 14 / 9, [8192, 896] and 2 of 8 9 / 7, [1000, 3584] and 2 of 8 11 / 13; one factor: [8192, 2048] of 64
// 37 / 23, [8192, 896] of 40 15 / 12, [4100, 3584] of 24 18 / 17.
// (Eight waves and twice the pieces in flight: one factor of rank 8 over 8192 rows, K = 896 6.1 / 10.4, 1536 7.9 / 10.3,
// 2048 11.8 / 9.4, 2560 10.5 / 14.8, 4096 15.3 / 15.5, 8192 31.7 / 30.3; two factors at 2048 11.6 / 12.4.  Not kept for one
// width.)
// ----------------------------------------------------------------------------
struct RowdotMulti {
  const uint16_t* Mt[LORA_MAX_SEG];
  float* out_f32[LORA_MAX_SEG];
  uint16_t* out_bf16[LORA_MAX_SEG];
  int R[LORA_MAX_SEG], RP[LORA_MAX_SEG], e0[LORA_MAX_SEG + 1];
  int n;
};
template <int NJ>
__global__ __launch_bounds__(256) void rowdot_multi_kernel(const uint16_t* __restrict__ X, RowdotMulti m, int64_t T,
                                                           int64_t K, float scale) {
  constexpr int NW = 4, STEP = NW * 64, U = 2;
  __shared__ floatx4 red[NJ][NW][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t0 = (int64_t)blockIdx.x * 16;
  const int64_t trow = t0 + (lane & 15) < T ? t0 + (lane & 15) : T - 1;
  const uint16_t *xp = X + trow * K + (lane >> 4) * 16, *mp[NJ];
  bool ok[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int e = (blockIdx.y * NJ + j) * 16 + (lane & 15);
    const uint16_t* f = m.Mt[0];
    int el = e, R = m.R[0];
#pragma unroll
    for (int i = 1; i < LORA_MAX_SEG; ++i)
      if (i < m.n && e >= m.e0[i]) {
        f = m.Mt[i];
        el = e - m.e0[i];
        R = m.R[i];
      }
    ok[j] = el < R;
    mp[j] = f + (int64_t)(ok[j] ? el : 0) * K + (lane >> 4) * 16;
  }
  const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
  floatx4 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = wave * 64; k0 < K; k0 += U * STEP) {
    bf16x8 f[U][2][NJ], x[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * STEP < K ? k0 + u * STEP : k0;  // (wave-uniform)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[u][h] = *(const bf16x8*)(xp + k + 8 * h);
#pragma unroll
        for (int j = 0; j < NJ; ++j) f[u][h][j] = *(const bf16x8*)(mp[j] + k + 8 * h);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // (or the scheduler sinks the loads to their MFMAs to save registers)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // (past the end both operands are zero: the re-read row may hold infinities; a branch would take the loads with it)
      const bool in = k0 + u * STEP < K;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[u][h] = in ? x[u][h] : z;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[u][h], in && ok[j] ? f[u][h][j] : z, acc[j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) red[j][wave][lane] = acc[j];
  __syncthreads();
  // wave j adds up block j, in a fixed order; a lane holds factor row lane % 16 of rows (lane / 16) * 4 + q
  for (int j = wave; j < NJ; j += NW) {
    floatx4 s = red[j][0][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[j][w][lane];
    const int e = (blockIdx.y * NJ + j) * 16 + (lane & 15);
    float* of = m.out_f32[0];
    uint16_t* ob = m.out_bf16[0];
    int el = e, R = m.R[0], RP = m.RP[0];
    bool packed = m.e0[1] == m.R[0];
#pragma unroll
    for (int i = 1; i < LORA_MAX_SEG; ++i)
      if (i < m.n && e >= m.e0[i]) {
        of = m.out_f32[i];
        ob = m.out_bf16[i];
        el = e - m.e0[i];
        R = m.R[i];
        RP = m.RP[i];
        packed = m.e0[i + 1] - m.e0[i] == R;
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t t = t0 + (lane >> 4) * 4 + q;
      if (t >= T || el >= RP) continue;
      if (el < R) of[t * R + el] = s[q];
      ob[t * RP + el] = el < R ? f32_to_bf16(s[q] * scale) : (uint16_t)0;
      if (packed && el < R && el + 8 >= R && RP > R) ob[t * RP + el + 8] = 0;  // (R is a multiple of 8, RP the next of 16)
    }
  }
}

static int32_t check_lora(int64_t T, int64_t in, int64_t out, int r) {
  ARTK_CHECK_ARG(T > 0 && in > 0 && out > 0 && r > 0, "T, in, out, r must be positive");
  if (in % BK != 0 || out % BK != 0) {
    set_error("in (%lld) and out (%lld) must be multiples of %d", (long long)in, (long long)out, BK);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  if (r % 8 != 0 || r > 64) {
    set_error("LoRA rank %d must be a multiple of 8 and at most 64", r);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  return ARTK_OK;
}

// How the products of one call run: 256 x 256 tiles (split == 0), 128 x 128 tiles with the K range in `split` parts, or
// 256 x 256 tiles in `split` parts (wide).
struct LoraTiling {
  int split;
  int tiles;  // 128 x 128 tiles of all jobs; wide: 256 x 256
  bool wide = false;
  size_t part_floats() const {
    return wide ? (size_t)tiles * split * TILE * TILE : split > 1 ? (size_t)tiles * split * ST2 * ST2 : 0;
  }
};
// M and K steps of the n jobs over N columns.
// The estimate, in us, was fitted to both paths over 200 to 8192 rows and in / out sizes of 896 to 44032 (168
// products; the choice is within 2 % of the best measured one on average):
//   256 x 256: 1 us per K step and round of work-groups while few CUs run, 1.45 at the power limit of a full chip;
//   128 x 128: 0.58 us per K step alone on a CU, 1.0 for two side by side;
//   a split adds the reduction's launch and a write and a read of 64 KiB per unit.
// Both sides at some of them (us, 256 x 256 / best 128 x 128): 333 rows, 896 -> 896: 22 / 14 (no split); 333 rows,
// 22016 -> 2048: 331 / 66 (split 8); 2531 rows, 11008 -> 2048: 182 / 132; 8192 rows, 2048 -> 2048: 61 / 72;
// 2531 rows, 2048 -> 22016: 209 / 235.
static LoraTiling lora_tiling(const int64_t* M, const int64_t* ksteps, int n, int64_t N) {
  const int64_t cus = num_cus();
  const int64_t nt2 = (N + TILE - 1) / TILE, nt1 = (N + ST2 - 1) / ST2;
  int64_t tiles2 = 0, tiles1 = 0, k = 0;
  for (int i = 0; i < n; ++i) {
    tiles2 += (M[i] + TILE - 1) / TILE * nt2;
    tiles1 += (M[i] + ST2 - 1) / ST2 * nt1;
    k = ksteps[i] > k ? ksteps[i] : k;
  }
  LoraTiling best{0, (int)tiles1};
  const double fill = tiles2 < cus ? (double)tiles2 / (double)cus : 1.0;
  double cost = 0.93 * (8.0 + (double)((tiles2 + cus - 1) / cus * k) * (1.0 + 0.45 * fill));
  if (tiles1 > (1 << 24)) return best;
  for (int split = 1; split <= 16 && split <= k; ++split) {
    const double per_cu = (double)(tiles1 * split) / (double)cus;
    const double full = (double)(tiles1 * split / (2 * cus)), rest = per_cu - 2.0 * full;
    const double conc = full + (rest <= 0.0 ? 0.0 : rest <= 1.0 ? 0.58 : 0.58 + 0.42 * (rest - 1.0));
    const double c = 8.0 + (double)((k + split - 1) / split) * conc +
                     (split > 1 ? 5.0 + 0.3 * split + 0.02 * (double)(tiles1 * split) : 0.0);
    if (c < cost) {
      cost = c;
      best.split = split;
    }
  }
  // 256 x 256 tiles in parts: a round of work-groups at the rate of its fill, then the partials' write and read.  Both
  // sides, us with the reduction (best of the other two / in parts): rows x K -> M 2531 x 11008 -> 2048 139 / 114,
  // 1500 x 11008 -> 2048 85 / 74, 4090 x 11008 -> 2048 182 / 169, 1200 x 18944 -> 3584 264 / 190, 2500 x 18944 -> 3584
  // 449 / 399, 1300 x 22016 -> 2048 170 / 125, 2000 x 22016 -> 2048 200 / 172, 1300 x 37888 -> 3584 481 / 363.
  for (int split = 2; split <= 8 && split * 16 <= k; ++split) {
    const int64_t units = tiles2 * split;
    if (units > 2 * cus) break;
    const double f = units < cus ? (double)units / (double)cus : 1.0;
    const double c = 0.93 * (8.0 + (double)((units + cus - 1) / cus * ((k + split - 1) / split)) * (1.0 + 0.45 * f)) + 7.0 +
                     0.11 * (double)units;
    if (c < cost) {
      cost = c;
      best.split = split;
      best.tiles = (int)tiles2;
      best.wide = true;
    }
  }
  return best;
}
// The tiling of a call with one job per projection (forward) or one job over all of them (input gradient).
static LoraTiling lora_tiling_fwd(const artk_lora_proj_t* proj, int n, int64_t T, int64_t in) {
  int64_t M[LORA_MAX_SEG], ks[LORA_MAX_SEG];
  for (int i = 0; i < n; ++i) {
    M[i] = proj[i].out;
    ks[i] = in / BK;
  }
  return lora_tiling(M, ks, n, T);
}
static LoraTiling lora_tiling_bwd(const artk_lora_proj_t* proj, int n, int64_t T, int64_t in) {
  int64_t ks = 0;
  for (int i = 0; i < n; ++i) ks += proj[i].out / BK;
  return lora_tiling(&in, &ks, 1, T);
}

// Runs the jobs of m (256-row tile numbering) as `t` says; part: t.part_floats() floats.
static int32_t launch_lora_jobs(const LoraMultiParams& m, const LoraTiling& t, float* part, hipStream_t st) {
  const int cus = num_cus();
  prof_begin(PROF_LORA_GEMM, st);
  if (t.split == 0) {
    if (m.n_jobs == 1 && m.job[0].nseg == 1) {
      const LoraJob& j = m.job[0];
      const LoraSeg& g = m.seg[j.seg0];
      LoraGemmParams p;
      p.P = g.P;
      p.Q = g.Q;
      p.Pe = g.Pe;
      p.Qe = g.Qe;
      p.bias = j.bias;
      p.out = j.out;
      p.M = j.M;
      p.N = m.N;
      p.K = g.K;
      p.r = g.r;
      p.RP = g.RP;
      p.MT = j.MT;
      p.NT = m.NT;
      lora_gemm_kernel<<<(unsigned)(m.n_tiles < cus ? m.n_tiles : cus), nthreads<LORA_NI>(), 0, st>>>(p);
    } else {
      lora_multi_gemm_kernel<<<(unsigned)(m.n_tiles < cus ? m.n_tiles : cus), nthreads<LORA_NI>(), 0, st>>>(m);
    }
  } else if (t.wide) {
    LoraSmallParams p;
    p.m = m;
    p.part = part;
    p.split = t.split;
    for (int i = 0; i < m.n_jobs; ++i) {
      p.ksteps[i] = 0;
      for (int g = 0; g < m.job[i].nseg; ++g) p.ksteps[i] += (int)(m.seg[m.job[i].seg0 + g].K / BK);
    }
    lora_split_gemm_kernel<<<(unsigned)(m.n_tiles * t.split), nthreads<LORA_NI>(), 0, st>>>(p);
    ARTK_CHECK_LAUNCH();
    lora_split_reduce_kernel<<<(unsigned)(m.n_tiles * 16), 256, 0, st>>>(p);
  } else {
    LoraSmallParams p;
    p.m = m;
    p.part = part;
    p.split = t.split;
    p.m.NT = (int)((m.N + ST2 - 1) / ST2);
    int tile = 0;
    for (int i = 0; i < m.n_jobs; ++i) {
      LoraJob& j = p.m.job[i];
      j.MT = (int)((j.M + ST2 - 1) / ST2);
      j.tile0 = tile;
      tile += j.MT * p.m.NT;
      p.ksteps[i] = 0;
      for (int g = 0; g < j.nseg; ++g) p.ksteps[i] += (int)(m.seg[j.seg0 + g].K / BK);
    }
    lora_small_gemm_kernel<<<(unsigned)(tile * t.split), ST2_THREADS, 0, st>>>(p);
    if (t.split > 1) {
      ARTK_CHECK_LAUNCH();
      lora_small_reduce_kernel<<<(unsigned)(tile * 4), 256, 0, st>>>(p);
    }
  }
  prof_end(PROF_LORA_GEMM, st);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

static int32_t launch_lora_gemm(const void* P, const void* Q, const uint16_t* Pe, const uint16_t* Qe,
                                const uint16_t* bias, void* out, int64_t M, int64_t N, int64_t K, int r,
                                int RP, const LoraTiling& t, float* part, hipStream_t st) {
  LoraMultiParams m;
  m.N = N;
  m.NT = (int)((N + TILE - 1) / TILE);
  m.n_jobs = 1;
  m.seg[0] = LoraSeg{P, Q, Pe, Qe, K, r, RP};
  m.job[0] = LoraJob{(uint16_t*)out, bias, M, (int)((M + TILE - 1) / TILE), 0, 0, 1};
  m.n_tiles = m.job[0].MT * m.NT;
  return launch_lora_jobs(m, t, part, st);
}

// Row products of a long K over few rows: one work-group per 16 rows leaves most CUs idle (2531 rows of 11008: 159
// work-groups, 23 us, however many waves they have), so they run as the ROW half of the one-pass kernel, a work-group
// per chunk of columns and slab of rows, and a reduction.
// (us, product / split: rows x K 333 x 4864 11 / 10, 333 x 11008 19 / 11, 1200 x 18944 31 / 16, 2531 x 11008 20 / 17, 4090 x 11008 22 / 22;
// the split is one launch more.  The only case where a projection has other sums alone than among others.)
static bool rowdot_split(int64_t T, int64_t K, int n, int r) { return n == 1 && r <= 16 && K >= 8192 && T < 12 * num_cus(); }
static size_t rowdot_split_floats(int64_t T, int64_t K, int n, int r) {
  return rowdot_split(T, K, n, r) ? (size_t)stats_geom(T, K, r, K).n_chunks * T * r + 1024 : 0;
}
// (part: rowdot_split_floats(T, K, 1, r) floats)
static int32_t launch_rowdot_split(const void* X, const void* Mt, int64_t T, int64_t K, int r, int RP, float scale,
                                   float* out_f32, uint16_t* out_bf16, float* part, hipStream_t st) {
  const StatsGeom g = stats_geom(T, K, r, K);
  int32_t rc = launch_stats(X, T, K, (const uint16_t*)Mt, nullptr, r, g, part + 1024, nullptr, part, st);
  if (rc) return rc;
  return launch_stats_reduce(StatsReduceJob{part + 1024, g.n_chunks, T, 1.f, out_f32, 0, out_bf16, RP, scale},
                             StatsReduceJob{nullptr, 0, 0, 0.f, nullptr, 0, nullptr, 0, 0.f}, r, st);
}

// Fills m.e0 and launches.
static int32_t launch_rowdot(const void* X, RowdotMulti& m, int64_t T, int64_t K, float scale, hipStream_t st) {
  const bool pack = T >= 16 * num_cus();
  int e = 0;
  for (int i = 0; i < m.n; ++i) {
    m.e0[i] = e;
    e += pack ? m.R[i] : m.RP[i];
  }
  for (int i = m.n; i <= LORA_MAX_SEG; ++i) m.e0[i] = e;
  const int nj = (e + 15) / 16;
  auto launch = [&](auto nj_tag) {
    constexpr int NJ = decltype(nj_tag)::value;
    rowdot_multi_kernel<NJ><<<dim3((unsigned)((T + 15) / 16), (unsigned)((nj + NJ - 1) / NJ)), 256, 0, st>>>(
        (const uint16_t*)X, m, T, K, scale);
  };
  if (!pack || nj == 1) launch(std::integral_constant<int, 1>{});
  else if (nj == 2) launch(std::integral_constant<int, 2>{});
  else launch(std::integral_constant<int, 4>{});
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

}  // namespace artk

using namespace artk;

extern "C" {

static LoraTiling lora_tiling_one(int64_t T, int64_t K, int64_t M) {
  const int64_t ks = K / BK;
  return lora_tiling(&M, &ks, 1, T);
}

size_t artk_lora_linear_fwd_workspace_bytes(int64_t T, int64_t in, int64_t out, int32_t r) {
  Workspace ws(nullptr, 0);
  ws.take<uint16_t>((size_t)T * round16(r));  // s * x A^T, bf16 [T,RP]
  ws.take<float>(lora_tiling_one(T, in, out).part_floats());
  ws.take<float>(rowdot_split_floats(T, in, 1, r));
  return ws.used + 256;
}

int32_t artk_lora_linear_fwd(const void* x, const void* W, const void* A, const void* B, const void* bias,
                             float scale, int64_t T, int64_t in, int64_t out, int32_t r, void* y, float* xa,
                             void* workspace, size_t workspace_bytes, artk_stream_t stream) {
  int32_t rc = check_lora(T, in, out, r);
  if (rc) return rc;
  ARTK_CHECK_ARG(x && W && A && B && y && xa, "null pointer argument");
  ARTK_CHECK_ARG(aligned16(x) && aligned16(W) && aligned16(A) && aligned16(B) && aligned16(y) &&
                     (bias == nullptr || aligned16(bias)),
                 "pointers must be 16-byte aligned");
  const int RP = round16(r);
  Workspace ws(workspace, workspace_bytes);
  uint16_t* xa16 = ws.take<uint16_t>((size_t)T * RP);
  const LoraTiling tiling = lora_tiling_one(T, in, out);
  float* part = ws.take<float>(tiling.part_floats());
  float* rpart = ws.take<float>(rowdot_split_floats(T, in, 1, r));
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  RowdotMulti m;
  m.n = 1;
  m.Mt[0] = (const uint16_t*)A;
  m.out_f32[0] = xa;
  m.out_bf16[0] = xa16;
  m.R[0] = r;
  m.RP[0] = RP;
  if (rowdot_split(T, in, 1, r)) rc = launch_rowdot_split(x, A, T, in, r, RP, scale, xa, xa16, rpart, st);
  else rc = launch_rowdot(x, m, T, in, scale, st);
  if (rc) return rc;
  return launch_lora_gemm(W, x, (const uint16_t*)B, xa16, (const uint16_t*)bias, y, out, T, in, r, RP, tiling, part, st);
}

// Scratch of the backward, carved in the same order by the size query and the call.
struct LoraBwdScratch {
  uint16_t *Bt, *At, *gb16;
  float *gb, *rowp_g, *colp_g, *colp_x, *dummy, *part;
  StatsGeom gg, gx;
  LoraTiling tiling;  // of the input gradient
};
static void carve_lora_bwd(Workspace& ws, int64_t T, int64_t in, int64_t out, int r, LoraBwdScratch& c) {
  const int RP = round16(r);
  c.gg = stats_geom(T, out, r, out);
  c.gx = stats_geom(T, in, r, in);
  c.Bt = ws.take<uint16_t>((size_t)r * out);   // B^T [r,out]: factor of the g B product
  c.At = ws.take<uint16_t>((size_t)in * r);    // A^T [in,r]: low-rank factor of dx
  c.gb = ws.take<float>((size_t)T * r);        // g B, f32 [T,r]
  c.gb16 = ws.take<uint16_t>((size_t)T * RP);  // s * g B, bf16 [T,RP]
  c.rowp_g = ws.take<float>((size_t)c.gg.n_chunks * T * r);
  c.colp_g = ws.take<float>((size_t)c.gg.n_slabs * out * r);
  c.colp_x = ws.take<float>((size_t)c.gx.n_slabs * in * r);
  c.dummy = ws.take<float>(1024);
  c.tiling = lora_tiling_one(T, out, in);
  c.part = ws.take<float>(c.tiling.part_floats());
}

size_t artk_lora_linear_bwd_workspace_bytes(int64_t T, int64_t in, int64_t out, int32_t r) {
  Workspace ws(nullptr, 0);
  LoraBwdScratch c;
  carve_lora_bwd(ws, T, in, out, r, c);
  return ws.used + 256;
}

int32_t artk_lora_linear_bwd(const void* g, const void* x, const void* W_t, const void* A,
                             const void* B, const float* xa, float scale, int64_t T, int64_t in,
                             int64_t out, int32_t r, void* dx, float* dA, float* dB, void* workspace,
                             size_t workspace_bytes, artk_stream_t stream) {
  int32_t rc = check_lora(T, in, out, r);
  if (rc) return rc;
  ARTK_CHECK_ARG(g && x && W_t && A && B && xa && dx && dA && dB, "null pointer argument");
  ARTK_CHECK_ARG(aligned16(g) && aligned16(x) && aligned16(W_t) && aligned16(A) && aligned16(B) && aligned16(dx) && aligned16(xa) &&
                     aligned16(dA) && aligned16(dB),
                 "pointers must be 16-byte aligned");
  const int RP = round16(r);
  Workspace ws(workspace, workspace_bytes);
  LoraBwdScratch c;
  carve_lora_bwd(ws, T, in, out, r, c);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  if ((rc = launch_small_transpose2(B, c.Bt, 1, out, r, A, c.At, 1, r, in, st))) return rc;
  // one pass over g: partials of g B (over column chunks) and of g^T (x A^T) (over row slabs)
  if ((rc = launch_stats(g, T, out, c.Bt, xa, r, c.gg, c.rowp_g, c.colp_g, c.dummy, st))) return rc;
  {
    StatsReduceJob ja{c.rowp_g, c.gg.n_chunks, T, 1.f, c.gb, 0, c.gb16, RP, scale};
    StatsReduceJob jb{c.colp_g, c.gg.n_slabs, out, scale, dB, 0, nullptr, 0, 0.f};
    if ((rc = launch_stats_reduce(ja, jb, r, st))) return rc;
  }
  // dx = g W + (s g B) A
  if ((rc = launch_lora_gemm(W_t, g, c.At, c.gb16, nullptr, dx, in, T, out, r, RP, c.tiling, c.part, st))) return rc;
  // one pass over x: dA [r,in] = s (g B)^T x
  if ((rc = launch_stats(x, T, in, nullptr, c.gb, r, c.gx, nullptr, c.colp_x, c.dummy, st))) return rc;
  {
    StatsReduceJob ja{c.colp_x, c.gx.n_slabs, in, scale, dA, 1, nullptr, 0, 0.f};
    StatsReduceJob jb{nullptr, 0, 0, 0.f, nullptr, 0, nullptr, 0, 0.f};
    if ((rc = launch_stats_reduce(ja, jb, r, st))) return rc;
  }
  return ARTK_OK;
}

// ---- several projections of the same input -------------------------------------------------
static int32_t check_multi(const artk_lora_proj_t* proj, int32_t n, int64_t T, int64_t in, bool bwd) {
  ARTK_CHECK_ARG(proj != nullptr && n >= 1 && n <= ARTK_LORA_MULTI_MAX, "1 to %d projections", ARTK_LORA_MULTI_MAX);
  int r_total = 0;
  for (int i = 0; i < n; ++i) {
    const artk_lora_proj_t& q = proj[i];
    int32_t rc = check_lora(T, in, q.out, q.r);
    if (rc) return rc;
    r_total += q.r;
    if (bwd) {
      ARTK_CHECK_ARG(q.W_t && q.A && q.B && q.g && q.xa && q.dA && q.dB, "projection %d: null pointer argument", i);
      ARTK_CHECK_ARG(aligned16(q.W_t) && aligned16(q.A) && aligned16(q.B) && aligned16(q.g) && aligned16(q.xa) &&
                         aligned16(q.dA) && aligned16(q.dB),
                     "projection %d: pointers must be 16-byte aligned", i);
    } else {
      ARTK_CHECK_ARG(q.W && q.A && q.B && q.y && q.xa, "projection %d: null pointer argument", i);
      ARTK_CHECK_ARG(aligned16(q.W) && aligned16(q.A) && aligned16(q.B) && aligned16(q.y) && aligned16(q.xa) &&
                         (q.bias == nullptr || aligned16(q.bias)),
                     "projection %d: pointers must be 16-byte aligned", i);
    }
  }
  if (bwd && r_total > 64) {
    set_error("the ranks of the projections add up to %d; at most 64 in one call", r_total);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  return ARTK_OK;
}

size_t artk_lora_linear_multi_fwd_workspace_bytes(int64_t T, int64_t in, const artk_lora_proj_t* proj,
                                                  int32_t n) {
  if (proj == nullptr || n < 1 || n > ARTK_LORA_MULTI_MAX) return 256;
  Workspace ws(nullptr, 0);
  for (int i = 0; i < n; ++i) ws.take<uint16_t>((size_t)T * round16(proj[i].r));
  ws.take<float>(lora_tiling_fwd(proj, n, T, in).part_floats());
  ws.take<float>(rowdot_split_floats(T, in, n, proj[0].r));
  return ws.used + 256;
}

int32_t artk_lora_linear_multi_fwd(const void* x, const artk_lora_proj_t* proj, int32_t n, float scale,
                                   int64_t T, int64_t in, void* workspace, size_t workspace_bytes,
                                   artk_stream_t stream) {
  int32_t rc = check_multi(proj, n, T, in, false);
  if (rc) return rc;
  ARTK_CHECK_ARG(x != nullptr && aligned16(x), "x must be a 16-byte aligned pointer");
  Workspace ws(workspace, workspace_bytes);
  uint16_t* xa16[ARTK_LORA_MULTI_MAX];
  for (int i = 0; i < n; ++i) xa16[i] = ws.take<uint16_t>((size_t)T * round16(proj[i].r));
  const LoraTiling tiling = lora_tiling_fwd(proj, n, T, in);
  float* part = ws.take<float>(tiling.part_floats());
  float* rpart = ws.take<float>(rowdot_split_floats(T, in, n, proj[0].r));
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  RowdotMulti m;
  LoraMultiParams p;
  m.n = n;
  int tile = 0;
  p.N = T;
  p.NT = (int)((T + TILE - 1) / TILE);
  p.n_jobs = n;
  for (int i = 0; i < n; ++i) {
    const artk_lora_proj_t& q = proj[i];
    const int RP = round16(q.r);
    m.Mt[i] = (const uint16_t*)q.A;
    m.out_f32[i] = q.xa;
    m.out_bf16[i] = xa16[i];
    m.R[i] = q.r;
    m.RP[i] = RP;
    p.seg[i] = LoraSeg{q.W, x, (const uint16_t*)q.B, xa16[i], in, q.r, RP};
    const int MT = (int)((q.out + TILE - 1) / TILE);
    p.job[i] = LoraJob{(uint16_t*)q.y, (const uint16_t*)q.bias, q.out, MT, tile, i, 1};
    tile += MT * p.NT;
  }
  p.n_tiles = tile;
  if (rowdot_split(T, in, n, proj[0].r))
    rc = launch_rowdot_split(x, proj[0].A, T, in, proj[0].r, round16(proj[0].r), scale, proj[0].xa, xa16[0], rpart, st);
  else
    rc = launch_rowdot(x, m, T, in, scale, st);
  if (rc) return rc;
  return launch_lora_jobs(p, tiling, part, st);
}

struct LoraMultiBwdScratch {
  LoraBwdScratch one[ARTK_LORA_MULTI_MAX];  // per projection: Bt, At, gb16, rowp_g, colp_g (gb, colp_x unused)
  float* gb_cat;   // [T, r_total]: g_i B_i side by side, the Y of the pass over x
  float* colp_x;   // [n_slabs][in][r_total]
  float* dummy;
  float* part;
  StatsGeom gx;
  LoraTiling tiling;
  int r_total;
};
static void carve_lora_multi_bwd(Workspace& ws, int64_t T, int64_t in, const artk_lora_proj_t* proj, int n,
                                 LoraMultiBwdScratch& c) {
  c.r_total = 0;
  int64_t out_all = 0;
  for (int i = 0; i < n; ++i) {
    c.r_total += proj[i].r;
    out_all += proj[i].out;
  }
  for (int i = 0; i < n; ++i) {
    const int64_t out = proj[i].out;
    const int r = proj[i].r, RP = round16(r);
    LoraBwdScratch& o = c.one[i];
    o.gg = stats_geom(T, out, r, out_all);
    o.Bt = ws.take<uint16_t>((size_t)r * out);
    o.At = ws.take<uint16_t>((size_t)in * r);
    o.gb16 = ws.take<uint16_t>((size_t)T * RP);
    o.rowp_g = ws.take<float>((size_t)o.gg.n_chunks * T * r);
    o.colp_g = ws.take<float>((size_t)o.gg.n_slabs * out * r);
  }
  c.gx = stats_geom(T, in, c.r_total, in);
  c.gb_cat = ws.take<float>((size_t)T * c.r_total);
  c.colp_x = ws.take<float>((size_t)c.gx.n_slabs * in * c.r_total);
  c.dummy = ws.take<float>(1024);
  c.tiling = lora_tiling_bwd(proj, n, T, in);
  c.part = ws.take<float>(c.tiling.part_floats());
}

size_t artk_lora_linear_multi_bwd_workspace_bytes(int64_t T, int64_t in, const artk_lora_proj_t* proj,
                                                  int32_t n) {
  if (proj == nullptr || n < 1 || n > ARTK_LORA_MULTI_MAX) return 0;
  Workspace ws(nullptr, 0);
  LoraMultiBwdScratch c;
  carve_lora_multi_bwd(ws, T, in, proj, n, c);
  return ws.used + 256;
}

int32_t artk_lora_linear_multi_bwd(const void* x, const artk_lora_proj_t* proj, int32_t n, float scale,
                                   int64_t T, int64_t in, void* dx, void* workspace, size_t workspace_bytes,
                                   artk_stream_t stream) {
  return artk_lora_linear_multi_bwd_typed(x, proj, n, scale, T, in, 0, dx, workspace, workspace_bytes, stream);
}

int32_t artk_lora_linear_multi_bwd_typed(const void* x, const artk_lora_proj_t* proj, int32_t n, float scale,
                                         int64_t T, int64_t in, int32_t grad_bf16, void* dx, void* workspace,
                                         size_t workspace_bytes, artk_stream_t stream) {
  int32_t rc = check_multi(proj, n, T, in, true);
  if (rc) return rc;
  ARTK_CHECK_ARG(x != nullptr && dx != nullptr && aligned16(x) && aligned16(dx),
                 "x and dx must be 16-byte aligned pointers");
  Workspace ws(workspace, workspace_bytes);
  LoraMultiBwdScratch c;
  carve_lora_multi_bwd(ws, T, in, proj, n, c);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  LoraMultiParams p;
  p.N = T;
  p.NT = (int)((T + TILE - 1) / TILE);
  p.n_jobs = 1;
  const int MT = (int)((in + TILE - 1) / TILE);
  p.job[0] = LoraJob{(uint16_t*)dx, nullptr, in, MT, 0, 0, n};
  p.n_tiles = MT * p.NT;
  StatsReduceJob jx{c.colp_x, c.gx.n_slabs, in, scale, nullptr, 1, nullptr, 0, 0.f};
  jx.n_split = n;
  jx.to_bf16 = grad_bf16 != 0;
  SmallTransposeMulti tr;
  StatsMulti sm;
  StatsReduceMulti rm;
  tr.n = 2 * n;
  sm.n = n;
  rm.n = 2 * n;
  bool one_shape = true;
  int r0 = 0;
  for (int i = 0; i < n; ++i) {
    const artk_lora_proj_t& q = proj[i];
    LoraBwdScratch& o = c.one[i];
    const int RP = round16(q.r);
    one_shape = one_shape && stats_shape(q.r) == stats_shape(proj[0].r);
    tr.t[2 * i] = SmallTranspose{(const uint16_t*)q.B, o.Bt, 1, q.out, q.r};
    tr.t[2 * i + 1] = SmallTranspose{(const uint16_t*)q.A, o.At, 1, q.r, in};
    // one pass over g_i: partials of g_i B_i (over column chunks) and of g_i^T (x A_i^T) (over row slabs)
    sm.p[i] = stats_params(q.g, T, q.out, o.Bt, q.xa, q.r, o.gg, o.rowp_g, o.colp_g, c.dummy);
    StatsReduceJob ja{o.rowp_g, o.gg.n_chunks, T, 1.f, c.gb_cat, 0, o.gb16, RP, scale};
    ja.out_ld = c.r_total;
    ja.out_off = r0;
    rm.job[2 * i] = ja;
    rm.job[2 * i + 1] = StatsReduceJob{o.colp_g, o.gg.n_slabs, q.out, scale, q.dB, 0, nullptr, 0, 0.f};
    rm.job[2 * i + 1].to_bf16 = grad_bf16 != 0;
    rm.R[2 * i] = rm.R[2 * i + 1] = q.r;
    p.seg[i] = LoraSeg{q.W_t, q.g, o.At, o.gb16, q.out, q.r, RP};
    jx.outs[i] = q.dA;
    jx.e_start[i] = r0;
    r0 += q.r;
  }
  jx.e_start[n] = r0;
  if ((rc = launch_small_transpose_multi(tr, st))) return rc;
  if (!one_shape) {  // one launch per projection
    for (int i = 0; i < n; ++i)
      if ((rc = launch_stats_params(sm.p[i], st))) return rc;
  } else if ((rc = launch_stats_multi(sm, stats_shape(proj[0].r), st))) {
    return rc;
  }
  if ((rc = launch_stats_reduce_multi(rm, st))) return rc;
  // dx = sum_i ( g_i W_i + (s g_i B_i) A_i ): one launch, the projections as K segments
  if ((rc = launch_lora_jobs(p, c.tiling, c.part, st))) return rc;
  // one pass over x: [dA_0; dA_1; ...] = s [g_0 B_0 | g_1 B_1 | ...]^T x
  if ((rc = launch_stats(x, T, in, nullptr, c.gb_cat, c.r_total, c.gx, nullptr, c.colp_x, c.dummy, st))) return rc;
  StatsReduceJob none{nullptr, 0, 0, 0.f, nullptr, 0, nullptr, 0, 0.f};
  return launch_stats_reduce(jx, none, c.r_total, st);
}

// ---- the same linear with the frozen weight kept as NF4 codes -------------------------------
// The bf16 weight exists only inside the call: it is dequantised into the workspace (forward:
// [out,in]; backward: [in,out], written transposed straight from the codes), consumed by the
// GEMM and forgotten, so neither a bf16 copy nor a transposed copy of W stays resident.
static int32_t check_nf4_weight(const artk_nf4_t* W, int64_t in) {
  ARTK_CHECK_ARG(W != nullptr && W->packed != nullptr, "null NF4 weight");
  ARTK_CHECK_ARG(W->blocksize >= 32 && in % W->blocksize == 0,
                 "the input size must be a multiple of the quantisation block size");
  return ARTK_OK;
}

size_t artk_lora_linear_fwd_nf4_workspace_bytes(int64_t T, int64_t in, int64_t out, int32_t r) {
  Workspace ws(nullptr, 0);
  ws.take<uint16_t>((size_t)out * in);
  ws.take<char>(artk_lora_linear_fwd_workspace_bytes(T, in, out, r));
  return ws.used + 256;
}

int32_t artk_lora_linear_fwd_nf4(const void* x, const artk_nf4_t* W, const void* A, const void* B,
                                 const void* bias, float scale, int64_t T, int64_t in, int64_t out, int32_t r,
                                 void* y, float* xa, void* workspace, size_t workspace_bytes,
                                 artk_stream_t stream) {
  int32_t rc = check_lora(T, in, out, r);
  if (rc) return rc;
  if ((rc = check_nf4_weight(W, in))) return rc;
  Workspace ws(workspace, workspace_bytes);
  uint16_t* Wd = ws.take<uint16_t>((size_t)out * in);
  const size_t inner = artk_lora_linear_fwd_workspace_bytes(T, in, out, r);
  char* rest = ws.take<char>(inner);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  if ((rc = artk_nf4_dequant(W->packed, W->absmax, W->absmax_q, W->code2, W->absmax2, W->offset, out * in,
                             W->blocksize, Wd, stream)))
    return rc;
  return artk_lora_linear_fwd(x, Wd, A, B, bias, scale, T, in, out, r, y, xa, rest, inner, stream);
}

size_t artk_lora_linear_bwd_nf4_workspace_bytes(int64_t T, int64_t in, int64_t out, int32_t r) {
  Workspace ws(nullptr, 0);
  ws.take<uint16_t>((size_t)out * in);
  ws.take<char>(artk_lora_linear_bwd_workspace_bytes(T, in, out, r));
  return ws.used + 256;
}

int32_t artk_lora_linear_bwd_nf4(const void* g, const void* x, const artk_nf4_t* W, const void* A,
                                 const void* B, const float* xa, float scale, int64_t T, int64_t in,
                                 int64_t out, int32_t r, void* dx, float* dA, float* dB, void* workspace,
                                 size_t workspace_bytes, artk_stream_t stream) {
  int32_t rc = check_lora(T, in, out, r);
  if (rc) return rc;
  if ((rc = check_nf4_weight(W, in))) return rc;
  Workspace ws(workspace, workspace_bytes);
  uint16_t* Wt = ws.take<uint16_t>((size_t)out * in);
  const size_t inner = artk_lora_linear_bwd_workspace_bytes(T, in, out, r);
  char* rest = ws.take<char>(inner);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  if ((rc = artk_nf4_dequant_t(W->packed, W->absmax, W->absmax_q, W->code2, W->absmax2, W->offset, out, in,
                               W->blocksize, Wt, stream)))
    return rc;
  return artk_lora_linear_bwd(g, x, Wt, A, B, xa, scale, T, in, out, r, dx, dA, dB, rest, inner, stream);
}

}  // extern "C"
