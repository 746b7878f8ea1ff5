// 128 x 128 NT bf16 tiles for products that are too small to fill the GPU with 256 x 256 tiles (gemm_nt.hpp):
// 256 threads = 4 wavefronts in a 2 x 2 grid, wave tile 64 x 64 = 2 x 2 MFMA 32x32x16 tiles, K steps of 64, two
// LDS stages of 2 x 16 KiB.  A work-group needs 64 KiB of LDS, so two run per CU: one computes while the other
// waits for its DMA, and a product has four times as many units of work.  Per flop it moves twice the bytes of a
// 256 x 256 tile into LDS, so it loses where that one fills the chip.  The LDS row layout, the swizzle and the
// buffer-bounded DMA are those of gemm_plain8.hpp.
#pragma once
#include "common.hpp"
#include "gemm_nt.hpp"

namespace artk {

constexpr int ST2 = 128;                           // tile rows of either operand
constexpr int ST2_OPER_BYTES = ST2 * BK * 2;       // 16 KiB
constexpr int ST2_STAGE_BYTES = 2 * ST2_OPER_BYTES;
constexpr int ST2_LDS_BYTES = 2 * ST2_STAGE_BYTES;  // 64 KiB
constexpr int ST2_THREADS = 256;

struct SmallAcc {
  floatx16 c[2][2];  // [mi][ni]: rows wm * 64 + mi * 32 .., columns wn * 64 + ni * 32 + lane % 32
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) c[i >> 1][i & 1][j] = 0.f;
  }
};

// One operand's 128-row panel starting at row0 of a [nrows, ld] matrix; rows past the end read as zero.
struct SmallPanel {
  dma_rsrc_t rsrc;
  int voff[2], step;
  __device__ __forceinline__ void init(const void* base, int64_t ld, int64_t row0, int64_t nrows, int lane) {
    const int64_t left = nrows - row0;
    const int64_t nvalid = left >= ST2 ? ST2 : (left > 0 ? left : 0);
    const int64_t bytes = nvalid * ld * 2;
    rsrc = dma_make_rsrc((const char*)base + row0 * ld * 2, (uint32_t)(bytes < 0x7fffffff ? bytes : 0x7fffffff));
    const int r = lane >> 3, pc = lane & 7;
    voff[0] = (int)(r * ld * 2) + ((pc ^ r) << 4);  // swz(8g + r) = r ^ (g & 1)
    voff[1] = (int)(r * ld * 2) + ((pc ^ r ^ 1) << 4);
    step = (int)(8 * ld * 2);
  }
  // This wave's quarter of the panel at K offset k0 into the operand stage at LDS address `lds`.
  __device__ __forceinline__ void issue(uint32_t lds, int wave, int k0) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = wave * 4 + i;
      dma_load16(rsrc, voff[i & 1], g * step + k0 * 2, lds + g * 1024);
    }
  }
};

// acc += P[prow0.., k0 : k0 + 64 n] Q[qrow0.., same]^T.  Every wave of the work-group calls it together; LDS may be
// reused when it returns.
__device__ __forceinline__ void small_tile_run(SmallAcc& acc, char* smem, const SmallPanel& lp, const SmallPanel& lq,
                                               int k0, int n) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds = lds_addr_of(smem);
  int off[4];
  {
    const int rl = lane & 31, f = swz(rl);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) off[kk] = rl * 128 + (((kk * 2 + (lane >> 5)) ^ f) << 4);
  }
  const int p_off = (wave >> 1) * 64 * 128, q_off = ST2_OPER_BYTES + (wave & 1) * 64 * 128;
  lp.issue(lds, wave, k0);
  lq.issue(lds + ST2_OPER_BYTES, wave, k0);
  for (int kt = 0; kt < n; ++kt) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    barrier_lds_only();  // stage kt has landed for every wave, and every wave is done with the other stage
    if (kt + 1 < n) {
      const uint32_t nxt = lds + ((kt + 1) & 1) * ST2_STAGE_BYTES;
      lp.issue(nxt, wave, k0 + (kt + 1) * BK);
      lq.issue(nxt + ST2_OPER_BYTES, wave, k0 + (kt + 1) * BK);
    }
    const char* st = smem + (kt & 1) * ST2_STAGE_BYTES;
    bf16x8 p[4][2], q[4][2];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        p[kk][i] = *(const bf16x8*)(st + p_off + off[kk] + i * 4096);
        q[kk][i] = *(const bf16x8*)(st + q_off + off[kk] + i * 4096);
      }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc.c[i >> 1][i & 1] =
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(p[kk][i >> 1], q[kk][i & 1], acc.c[i >> 1][i & 1], 0, 0, 0);
  }
  barrier_lds_only();
}

}  // namespace artk
