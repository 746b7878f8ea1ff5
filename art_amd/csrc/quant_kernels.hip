// 4-bit NormalFloat (NF4) base weights -> bf16, gfx950.
//
// The reference loads the base model with `load_in_4bit=True`
// (src/art/dev/model.py:29): bitsandbytes keeps each frozen linear weight as
// 4-bit NF4 codes, two per byte (first element in the high nibble), with one
// absolute maximum per block of 64 elements, optionally itself quantised to
// 8 bits ("double quantisation": a 256-entry code book, one fp32 scale per 256
// blocks, and a scalar offset).  The LoRA GEMMs of this library take bf16
// weights; this kernel produces them from the packed form.  HBM-bound:
// 0.5 B (+ 0.06 B of scales) read and 2 B written per element, a few per cent
// of the time of the GEMM that follows.
#include "common.hpp"

namespace artk {

// The 16 NF4 levels (Dettmers et al., "QLoRA", 2023, appendix E; the
// bitsandbytes code book for quant_type="nf4").
__constant__ float NF4_LEVELS[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f, 0.33791524171829224f,
    0.44070982933044434f, 0.5626170039176941f, 0.7229568362236023f, 1.0f};

struct Nf4Params {
  const uint8_t* packed;     // n / 2 bytes
  const float* absmax;       // [n / blocksize] or nullptr
  const uint8_t* absmax_q;   // [n / blocksize] (nested form)
  const float* code2;        // [256]
  const float* absmax2;      // [ceil(n / blocksize / 256)]
  float offset;
  int64_t n;
  int blocksize;             // power of two, >= 32
  uint16_t* out;             // [n] bf16
};

// Scales of N quantisation blocks, all loads of a level on their way together (one branch around them, not one each).
template <int N>
__device__ __forceinline__ void nf4_scales(const Nf4Params& p, const int64_t (&blk)[N], float (&scale)[N]) {
  if (p.absmax != nullptr) {
#pragma unroll
    for (int i = 0; i < N; ++i) scale[i] = p.absmax[blk[i]];
    return;
  }
  int code[N];
  float second[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    code[i] = p.absmax_q[blk[i]];
    second[i] = p.absmax2[blk[i] >> 8];
  }
  // separate multiply and add: the CPU restatement does not contract them
#pragma unroll
  for (int i = 0; i < N; ++i) scale[i] = __fadd_rn(__fmul_rn(p.code2[code[i]], second[i]), p.offset);
}
// 8 elements from their 4 packed bytes.
__device__ __forceinline__ uint4 nf4_expand(const float* lut, uint32_t w, float scale) {
  uint32_t o[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const uint32_t byte = (w >> (8 * b)) & 0xff;
    o[b] = (uint32_t)f32_to_bf16(lut[byte >> 4] * scale) | ((uint32_t)f32_to_bf16(lut[byte & 15] * scale) << 16);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// A thread turns 4 packed bytes into 8 elements, so a wave reads 256 contiguous bytes and writes 1 KiB contiguous, NF4_UNROLL
// times with all reads on their way first: 2048 x 11008 elements in 10.6 us (one at a time 11.8, 12.8 with a division per
// element group; with quantised maxima 11.2 / 12.5 / 14.7).  Below NF4_FULL work-groups per CU of one read each there is
// nothing left to fill the GPU with four: 896 x 896 3.3 us with one, 3.5 with four; 896 x 4864 4.5 / 4.6, 2048 x 2048 4.4 / 4.4,
// 2048 x 3072 5.4 / 5.3.
constexpr int NF4_FULL = 8;
template <int NF4_UNROLL>
__global__ __launch_bounds__(256) void nf4_dequant_kernel(Nf4Params p) {
  __shared__ float lut[16];
  if (threadIdx.x < 16) lut[threadIdx.x] = NF4_LEVELS[threadIdx.x];
  __syncthreads();
  const int shift = __builtin_ctz(p.blocksize);
  const int64_t i0 = ((int64_t)blockIdx.x * NF4_UNROLL * 256 + threadIdx.x) * 8;
  uint32_t w[NF4_UNROLL];
  int64_t blk[NF4_UNROLL];
  float scale[NF4_UNROLL];
#pragma unroll
  for (int u = 0; u < NF4_UNROLL; ++u) {
    const int64_t i = i0 + u * 2048 < p.n ? i0 + u * 2048 : 0;
    w[u] = *(const uint32_t*)(p.packed + i / 2);
    blk[u] = i >> shift;
  }
  nf4_scales(p, blk, scale);
#pragma unroll
  for (int u = 0; u < NF4_UNROLL; ++u)
    if (i0 + u * 2048 < p.n) *(uint4*)(p.out + i0 + u * 2048) = nf4_expand(lut, w[u], scale[u]);
}

// Same values written transposed: the weight is [R, C] (C elements per row, quantisation blocks
// run along a row), the output is bf16 [C, R].  A work-group takes 64 rows x 256 columns: a thread expands an 8 x 8 block and
// transposes it in registers, and LDS gathers the 64 rows of a column, which are stored as one cache line.  (Two bytes at a
// time through LDS: 2048 x 11008 elements 18.2 us, now 14.1; 3584 x 18944 46.6, now 33.6.)
__global__ __launch_bounds__(256) void nf4_dequant_t_kernel(Nf4Params p, int64_t R, int64_t C) {
  __shared__ float lut[16];
  __shared__ uint4 tile[256][8];  // [column][8 rows], chunk XORed by the column's group of 8
  if (threadIdx.x < 16) lut[threadIdx.x] = NF4_LEVELS[threadIdx.x];
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 256;
  const int cb = threadIdx.x & 31, rb = threadIdx.x >> 5;
  const int64_t c = c0 + cb * 8, r = r0 + rb * 8;
  if (r < R && c < C) {  // (R and C are multiples of 8: a block is inside or outside as a whole)
    const int shift = __builtin_ctz(p.blocksize);
    uint32_t w[8];
    int64_t blk[8];
    float scale[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int64_t e = (r + q) * C + c;
      w[q] = *(const uint32_t*)(p.packed + e / 2);
      blk[q] = e >> shift;
    }
    nf4_scales(p, blk, scale);
    uint4 v[8], t[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = nf4_expand(lut, w[q], scale[q]);
    transpose8x8(v, t);
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[cb * 8 + j][rb ^ (cb & 7)] = t[j];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int cc = i * 32 + (threadIdx.x >> 3), k = threadIdx.x & 7;
    if (c0 + cc < C && r0 + k * 8 < R) *(uint4*)(p.out + (c0 + cc) * R + r0 + k * 8) = tile[cc][k ^ ((cc >> 3) & 7)];
  }
}

// The same for matrices of fewer than NF4_T_FULL such tiles per CU: 64 rows x 64 columns per work-group, a thread expands 8
// columns of two rows and puts the pairs into LDS.  us, this / tiles of 64 x 256: 896 x 896 3.4 / 4.5, 896 x 4864 4.9 / 5.9,
// 2048 x 2048 4.8 / 5.4, 2048 x 3072 6.2 / 6.5, 3584 x 3584 11.4 / 9.2.
constexpr int NF4_T_FULL = 2;
__global__ __launch_bounds__(256) void nf4_dequant_t_small_kernel(Nf4Params p, int64_t R, int64_t C) {
  __shared__ float lut[16];
  __shared__ uint4 tile[64][8];  // [column][8 rows], chunk XORed by the column's group of 8
  if (threadIdx.x < 16) lut[threadIdx.x] = NF4_LEVELS[threadIdx.x];
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const int cb = threadIdx.x & 7, rp = threadIdx.x >> 3;
  const int64_t c = c0 + cb * 8, r = r0 + rp * 2;
  if (r < R && c < C) {  // (R and C are multiples of 8)
    const int shift = __builtin_ctz(p.blocksize);
    const int64_t blk[2] = {(r * C + c) >> shift, (r * C + C + c) >> shift};
    const uint32_t w0 = *(const uint32_t*)(p.packed + (r * C + c) / 2), w1 = *(const uint32_t*)(p.packed + (r * C + C + c) / 2);
    float scale[2];
    nf4_scales(p, blk, scale);
    const uint4 a = nf4_expand(lut, w0, scale[0]), b = nf4_expand(lut, w1, scale[1]);
    const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t lo = av[j / 2] >> (16 * (j & 1)) & 0xffffu, hi = bv[j / 2] >> (16 * (j & 1)) & 0xffffu;
      ((uint32_t*)&tile[cb * 8 + j][(rp >> 2) ^ cb])[rp & 3] = lo | hi << 16;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int cc = i * 32 + (threadIdx.x >> 3), k = threadIdx.x & 7;
    if (c0 + cc < C && r0 + k * 8 < R) *(uint4*)(p.out + (c0 + cc) * R + r0 + k * 8) = tile[cc][k ^ (cc >> 3)];
  }
}

static int32_t check_nf4(const void* packed, const float* absmax, const void* absmax_q, const float* code2,
                         const float* absmax2, int64_t n, int32_t blocksize, const void* out) {
  ARTK_CHECK_ARG(packed && out, "null pointer argument");
  ARTK_CHECK_ARG(absmax != nullptr || (absmax_q && code2 && absmax2),
                 "give absmax, or absmax_q + code2 + absmax2");
  ARTK_CHECK_ARG(aligned16(packed) && aligned16(out), "packed and out must be 16-byte aligned");
  if (n <= 0 || n % 32 != 0 || blocksize < 32 || (blocksize & (blocksize - 1)) != 0 || n % blocksize != 0) {
    set_error("n (%lld) must be a positive multiple of the block size (%d), a power of two >= 32",
              (long long)n, blocksize);
    return ARTK_ERR_UNSUPPORTED_SHAPE;
  }
  return ARTK_OK;
}

static Nf4Params nf4_params(const void* packed, const float* absmax, const void* absmax_q, const float* code2,
                            const float* absmax2, float offset, int64_t n, int32_t blocksize, void* out) {
  Nf4Params p;
  p.packed = (const uint8_t*)packed;
  p.absmax = absmax;
  p.absmax_q = (const uint8_t*)absmax_q;
  p.code2 = code2;
  p.absmax2 = absmax2;
  p.offset = offset;
  p.n = n;
  p.blocksize = blocksize;
  p.out = (uint16_t*)out;
  return p;
}

}  // namespace artk

using namespace artk;

extern "C" {

int32_t artk_nf4_dequant(const void* packed, const float* absmax, const void* absmax_q,
                         const float* code2, const float* absmax2, float offset, int64_t n,
                         int32_t blocksize, void* out_bf16, artk_stream_t stream) {
  int32_t rc = check_nf4(packed, absmax, absmax_q, code2, absmax2, n, blocksize, out_bf16);
  if (rc) return rc;
  Nf4Params p = nf4_params(packed, absmax, absmax_q, code2, absmax2, offset, n, blocksize, out_bf16);
  const int64_t reads = (n / 8 + 255) / 256;  // work-groups with a read per thread
  ARTK_CHECK_ARG(reads < (1ll << 33), "too many elements");
  if (reads >= NF4_FULL * num_cus())
    nf4_dequant_kernel<4><<<(unsigned)((reads + 3) / 4), 256, 0, (hipStream_t)stream>>>(p);
  else
    nf4_dequant_kernel<1><<<(unsigned)reads, 256, 0, (hipStream_t)stream>>>(p);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

int32_t artk_nf4_dequant_t(const void* packed, const float* absmax, const void* absmax_q,
                           const float* code2, const float* absmax2, float offset, int64_t rows,
                           int64_t cols, int32_t blocksize, void* out_bf16, artk_stream_t stream) {
  ARTK_CHECK_ARG(rows > 0 && cols > 0 && rows % 8 == 0 && cols % 8 == 0, "rows and cols must be positive multiples of 8");
  ARTK_CHECK_ARG(rows < 65536 * 64, "too many rows");
  int32_t rc = check_nf4(packed, absmax, absmax_q, code2, absmax2, rows * cols, blocksize, out_bf16);
  if (rc) return rc;
  Nf4Params p = nf4_params(packed, absmax, absmax_q, code2, absmax2, offset, rows * cols, blocksize, out_bf16);
  const unsigned row_tiles = (unsigned)((rows + 63) / 64);
  if ((cols + 255) / 256 * row_tiles >= NF4_T_FULL * num_cus())
    nf4_dequant_t_kernel<<<dim3((unsigned)((cols + 255) / 256), row_tiles), 256, 0, (hipStream_t)stream>>>(p, rows, cols);
  else
    nf4_dequant_t_small_kernel<<<dim3((unsigned)((cols + 63) / 64), row_tiles), 256, 0, (hipStream_t)stream>>>(p, rows, cols);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

}  // extern "C"
