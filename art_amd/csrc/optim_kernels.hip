// Optimizer step for the LoRA parameters, gfx950.
//
// The reference trains the adapters with HF Trainer's `paged_adamw_8bit`
// (bitsandbytes) and `max_grad_norm = 0.1`, `weight_decay = 0.1`, betas
// (0.9, 0.99), constant learning rate (src/art/dev/model.py:69-85).  Here all
// adapter parameters of the model live in ONE flat fp32 buffer (likewise their
// gradients and the two moments), so a step is two launches over contiguous
// memory instead of several small kernels per tensor: a fixed-order sum of
// squares for the global gradient norm, and a fused update that applies the
// clip coefficient, the decoupled weight decay and the Adam update, and also
// writes the bf16 copy of the parameters that the GEMM kernels read.  Moments
// are fp32 (the reference quantises them to 8 bits block-wise; that is a memory
// optimisation of bitsandbytes, not part of the update rule).
// Both kernels are HBM-bound: 4 B/param and 16 B read + 14 B written per param.
#include "common.hpp"

namespace artk {

constexpr int SUMSQ_BLOCKS = 1024;

// Loads and stores of what a step touches once.  A step over more than the 256 MiB Infinity Cache holds finds nothing
// of it there the next time, and reading and writing it past the cache leaves the gradients, which the norm has just
// read, in it: 20.2 M elements with 8-bit moments 103 -> 94 us a step (loads or stores alone: no gain; the gradients
// too: 110).
// With fp32 moments a step of 449 MB still finds enough there (78 us, 80 past the cache); 605 MB: 117 -> 104 us.
// The kernels of a step in a trace, through the caches / past them, step after step; and each after 1 GiB of other writes,
// as behind a backward pass: 8-bit moments 11.6 M elements 62 / 62; 76 / 73, 15.0 M 73 / 75; 93 / 92, 20.2 M 95 / 92;
// 115 / 110, 40.4 M 192 / 171; 211 / 203; fp32 11.6 M 63 / 65; 83 / 79, 15.0 M 80 / 80; 103 / 98, 20.2 M 120 / 106;
// 140 / 130, 40.4 M 269 / 218; 280 / 267.
static inline bool step_once8(int64_t n) { return 18 * n > (256ll << 20); }
static inline bool step_once32(int64_t n) { return 30 * n > (512ll << 20); }
template <bool ONCE, class T>
__device__ __forceinline__ T once_load(const T* p) {
  if constexpr (ONCE) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool ONCE, class T>
__device__ __forceinline__ void once_store(T v, T* p) {
  if constexpr (ONCE) __builtin_nontemporal_store(v, p);
  else *p = v;
}
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// part[b] = sum of x[i]^2 over the slice of block b, accumulated in double in a
// fixed order; sumsq_final_kernel adds the partials in index order.
__global__ __launch_bounds__(256) void sumsq_partial_kernel(const float* __restrict__ x, int64_t n,
                                                            double* __restrict__ part) {
  __shared__ double red[4];
  const int64_t per = ((n + SUMSQ_BLOCKS - 1) / SUMSQ_BLOCKS + 3) & ~(int64_t)3;
  const int64_t b0 = (int64_t)blockIdx.x * per;
  const int64_t b1 = b0 + per < n ? b0 + per : n;
  double acc = 0.0;
  for (int64_t i = b0 + threadIdx.x * 4; i < b1; i += 1024) {
    if (i + 4 <= b1 && ((uintptr_t)(x + i) & 15) == 0) {
      const float4 v = *(const float4*)(x + i);
      acc += (double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z + (double)v.w * v.w;
    } else {
      for (int64_t j = i; j < i + 4 && j < b1; ++j) acc += (double)x[j] * x[j];
    }
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(64) void sumsq_final_kernel(const double* __restrict__ part,
                                                         float* __restrict__ out) {
  // lane l adds its 16 consecutive partials in index order, then a fixed butterfly over the wave
  double s = 0.0;
  for (int i = 0; i < SUMSQ_BLOCKS / 64; ++i) s += part[threadIdx.x * (SUMSQ_BLOCKS / 64) + i];
  s = wave_sum(s);
  if (threadIdx.x == 0) out[0] = (float)s;
}

struct AdamWParams {
  float* p;
  const float* g;
  float* m;
  float* v;
  uint16_t* p_bf16;         // or nullptr
  const float* grad_sumsq;  // or nullptr: no clipping
  int64_t n;
  float lr, beta1, beta2, eps, weight_decay, max_grad_norm;
  float step_size;          // lr / (1 - beta1^t)
  float inv_bc2_sqrt;       // 1 / sqrt(1 - beta2^t)
};

__device__ __forceinline__ float adamw_one(float& p, float g, float& m, float& v, const AdamWParams& a,
                                           float clip) {
  g *= clip;
  p *= 1.f - a.lr * a.weight_decay;
  m = m + (g - m) * (1.f - a.beta1);
  v = v * a.beta2 + (1.f - a.beta2) * g * g;
  const float denom = sqrtf(v) * a.inv_bc2_sqrt + a.eps;
  p -= a.step_size * (m / denom);
  return p;
}

template <bool ONCE>
__global__ __launch_bounds__(256) void adamw_kernel(AdamWParams a) {
  float clip = 1.f;
  if (a.grad_sumsq != nullptr) {
    // torch.nn.utils.clip_grad_norm_: coef = max_norm / (norm + 1e-6), clamped to 1
    const float c = a.max_grad_norm / (sqrtf(a.grad_sumsq[0]) + 1e-6f);
    clip = c < 1.f ? c : 1.f;
  }
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= a.n) return;
  if (i + 4 <= a.n) {
    const f32x4 p4 = once_load<ONCE>((const f32x4*)(a.p + i)), m4 = once_load<ONCE>((const f32x4*)(a.m + i));
    const f32x4 v4 = once_load<ONCE>((const f32x4*)(a.v + i)), g4 = *(const f32x4*)(a.g + i);
    float p[4], m[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p[j] = p4[j];
      m[j] = m4[j];
      v[j] = v4[j];
      adamw_one(p[j], g4[j], m[j], v[j], a, clip);
    }
    once_store<ONCE>(f32x4{p[0], p[1], p[2], p[3]}, (f32x4*)(a.p + i));
    once_store<ONCE>(f32x4{m[0], m[1], m[2], m[3]}, (f32x4*)(a.m + i));
    once_store<ONCE>(f32x4{v[0], v[1], v[2], v[3]}, (f32x4*)(a.v + i));
    if (a.p_bf16) {
      const uint32_t lo = (uint32_t)f32_to_bf16(p[0]) | ((uint32_t)f32_to_bf16(p[1]) << 16);
      const uint32_t hi = (uint32_t)f32_to_bf16(p[2]) | ((uint32_t)f32_to_bf16(p[3]) << 16);
      *(uint2*)(a.p_bf16 + i) = make_uint2(lo, hi);
    }
  } else {
    for (int64_t j = i; j < a.n; ++j) {
      float p = a.p[j], m = a.m[j], v = a.v[j];
      adamw_one(p, a.g[j], m, v, a, clip);
      a.p[j] = p;
      a.m[j] = m;
      a.v[j] = v;
      if (a.p_bf16) a.p_bf16[j] = f32_to_bf16(p);
    }
  }
}

// ----------------------------------------------------------------------------
// AdamW with 8-bit block-wise moments (the storage form of `paged_adamw_8bit`).
// Each moment is one byte per element: an index into a 256-entry code book of
// values in [-1, 1] (exp_avg) or [0, 1] (exp_avg_sq), times one fp32 absolute
// maximum per block of 256 elements.  Dequantise, update in fp32, new block maxima, requantise to the
// nearest code.
// ----------------------------------------------------------------------------
struct AdamW8Params {
  float* p;
  const float* g;
  uint8_t* c1;
  uint8_t* c2;
  float* absmax1;
  float* absmax2;
  const float* qmap1;
  const float* qmap2;
  uint16_t* p_bf16;
  const float* grad_sumsq;
  int64_t n;
  float lr, beta1, beta2, eps, weight_decay, max_grad_norm;
  float step_size;   // -lr * sqrt(1 - beta2^t) / (1 - beta1^t)
  float eps_scaled;  // sqrt(1 - beta2^t) * eps
};

// Nearest entry of an ascending 256-entry code book (ties to the lower index): entry k up to thr[k], the largest value
// that is not nearer to entry k + 1.  The leading 16 bits of the fp32 value (sign, exponent, 7 mantissa bits) select a
// byte: the first entry whose threshold is not below everything in that bin.  In the books in use no bin holds two
// thresholds (the finest octave, [0.5, 1), has 71 entries in 128 bins), so the code is that byte, or one more where the
// value is above its threshold: two LDS gathers and no loop.  A book with a fuller bin, or without all its thresholds, walks
// from there, over the entries themselves.  (A bisection, eight dependent gathers per value, took 182 us for 20.2 M elements; a start byte and
// a walk that compares with two neighbours 84 us, 137 vector instructions per element.)
constexpr int LUT_E0 = 104;                      // exponents 104 .. 127: [2^-23, 1]; smaller values share bin 0
constexpr int LUT_HALF = (128 - LUT_E0) * 128;   // bins of one sign
constexpr int LUT_BINS = 2 * LUT_HALF;           // ascending: negative bins first
// (in LDS by sign bit, then magnitude, so that an index is one multiply-add)

// Lower end of bin j (ascending order), -inf for the first one, inf past the last.
__device__ __forceinline__ float lut_edge(int j) {
  if (j == LUT_HALF) return 0.f;
  if (j >= LUT_BINS) return INFINITY;
  if (j > LUT_HALF) return __uint_as_float((uint32_t)(j - LUT_HALF + LUT_E0 * 128) << 16);
  return j == 0 ? -INFINITY : -__uint_as_float((uint32_t)(LUT_HALF - j + LUT_E0 * 128) << 16);
}

// The largest float that the rule gives to entry `cur` rather than to the next one, and whether it was found within 32 floats
// of the middle.  It is in the books in use; not between -a and a for instance, where everything near 0 is a tie once
// the differences are rounded.  A book with such a gap takes the walk below.
__device__ bool code_threshold(float cur, float next, float& thr) {
  auto lower = [&](float x) { return x < next && x - cur <= next - x; };
  auto key = [](float x) {  // floats in the order of integers, and back
    const int i = (int)__float_as_uint(x);
    return i < 0 ? (int)0x80000000 - i : i;
  };
  auto val = [](int k) { return __uint_as_float((uint32_t)(k < 0 ? (int)0x80000000 - k : k)); };
  int k = key(0.5f * cur + 0.5f * next);
  bool found = false;
  for (int step = 0; step < 32 && !found; ++step) {
    const bool here = lower(val(k)), above = lower(val(k + 1));
    found = here && !above;
    if (!found) k += here ? 1 : -1;
  }
  thr = val(k);
  return found;
}

// Start bytes and whether two gathers do (thr[255] is infinite).
__device__ bool build_lut(uint8_t* lut, const float* thr, int tid, int nthreads) {
  const int per = LUT_BINS / nthreads;
  int lo = -1, hi = 255;  // thr[lo] < first <= thr[hi]
  const float first = lut_edge(tid * per);
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (thr[mid] < first) lo = mid; else hi = mid;
  }
  bool one = true;
  for (int j = tid * per; j < (tid + 1) * per; ++j) {
    const float e = lut_edge(j), end = lut_edge(j + 1);
    while (hi < 255 && thr[hi] < e) ++hi;
    lut[j < LUT_HALF ? LUT_BINS - 1 - j : j - LUT_HALF] = (uint8_t)hi;
    one = one && (hi >= 254 || thr[hi + 1] >= end);
  }
  return one;
}

template <bool ONE>
__device__ __forceinline__ int nearest_code(const float* map, const float* thr, const uint8_t* lut, float x) {
  const uint32_t u = __float_as_uint(x);
  int k = (int)(u >> 16 & 0x7fff) - LUT_E0 * 128;
  k = k < 0 ? 0 : (k > LUT_HALF - 1 ? LUT_HALF - 1 : k);
  int lo = lut[k + (int)(u >> 31) * LUT_HALF];
  if constexpr (ONE) {
    lo += x > thr[lo] ? 1 : 0;
    return x != x ? 1 : lo;
  }
  // (entries at or before the start byte's may be the nearest one of a book without thresholds)
  lo = lo > 254 ? 254 : lo;
  while (lo > 0 && map[lo] > x) --lo;
  float cur = map[lo], next = map[lo + 1];
  while (lo < 254 && next <= x) {
    ++lo;
    cur = next;
    next = map[lo + 1];
  }
  if (x != x) return 1;
  return (x - cur <= next - x) ? lo : lo + 1;
}

// x / max for the elements of a block (|x| <= max).  With max scaled to [0.5, 1) and x by the same power of two, one
// correction of x times the correctly rounded reciprocal gives the correctly rounded quotient (Markstein): 4
// instructions per element for the 10 of a division and no branch (one on the range of max cost 25 spilled registers
// and twice the time).  An element that the scaling takes below the normal range is nearest to the smallest code
// either way.  Infinite max: finite elements give 0, infinite ones NaN.  Zero or NaN: see the kernel.
struct BlockMax {
  float d, y;
  int e;
  __device__ __forceinline__ explicit BlockMax(float max) {
    const bool plain = max > 0.f && max < INFINITY;
    e = plain ? -__builtin_amdgcn_frexp_expf(max) : 0;
    d = plain ? __builtin_amdgcn_frexp_mantf(max) : 1.f;
    y = plain ? 1.f / d : 0.f;
  }
  __device__ __forceinline__ float quotient(float x) const {
    x = __builtin_amdgcn_ldexpf(x, e);
    const float q = x * y;
    return fmaf(fmaf(-q, d, x), y, q);
  }
};

// One wave = one block of 256 elements, 4 consecutive elements per lane: 16-byte loads of parameters and
// gradients, 4-byte loads of the codes, block maxima by wave reduction without a barrier.  18 B per
// element, of which the gradient's second read after the norm comes from the Infinity Cache.  The grid
// is two work-groups of 16 waves per CU that walk the blocks, so the tables are built once per
// work-group and not once per 256 elements.  20.2 M elements, this kernel alone: 182 us as one work-group per block with a
// bisection, 104 us with a start table, 84 us with quotients without divisions (137 vector instructions per
// element), 75 us with thresholds in place of neighbours (119, which still are all of its time).
constexpr int ADAM8_THREADS = 1024;

template <bool ONCE>
__global__ __launch_bounds__(ADAM8_THREADS, 8) void adamw8bit_kernel(AdamW8Params a, int64_t n_blocks, int vec) {
  __shared__ float map1[256], map2[256], thr1[256], thr2[256];
  __shared__ uint8_t lut1[LUT_BINS], lut2[LUT_BINS];
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < 256) map1[tid] = a.qmap1[tid];
  else if (tid < 512) map2[tid - 256] = a.qmap2[tid - 256];
  float clip = 1.f;
  if (a.grad_sumsq != nullptr) {
    const float c = a.max_grad_norm / (sqrtf(a.grad_sumsq[0]) + 1e-6f);
    clip = c < 1.f ? c : 1.f;
  }
  __syncthreads();
  bool ok = true;
  if (tid < 512) {
    const float* map = tid < 256 ? map1 : map2;
    float* thr = tid < 256 ? thr1 : thr2;
    const int k = tid & 255;
    float t = INFINITY;
    if (k < 255) ok = code_threshold(map[k], map[k + 1], t);
    thr[k] = t;
  }
  ok = __syncthreads_and(ok);
  ok = build_lut(lut1, thr1, tid, ADAM8_THREADS) && ok;
  ok = build_lut(lut2, thr2, tid, ADAM8_THREADS) && ok;
  const bool one = __syncthreads_and(ok);  // (the same for the whole work-group)
  const int64_t stride = (int64_t)gridDim.x * (ADAM8_THREADS / 64);
  for (int64_t b = (int64_t)blockIdx.x * (ADAM8_THREADS / 64) + (tid >> 6); b < n_blocks; b += stride) {
    const int64_t i = b * 256 + lane * 4;
    const bool full = vec && b * 256 + 256 <= a.n;   // wave-uniform
    float g[4] = {0.f, 0.f, 0.f, 0.f}, pv[4] = {0.f, 0.f, 0.f, 0.f};
    uint32_t c1 = 0, c2 = 0;
    if (full) {
      *(float4*)g = *(const float4*)(a.g + i);
      *(f32x4*)pv = once_load<ONCE>((const f32x4*)(a.p + i));
      c1 = once_load<ONCE>((const uint32_t*)(a.c1 + i));
      c2 = once_load<ONCE>((const uint32_t*)(a.c2 + i));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < a.n) {
          g[j] = a.g[i + j];
          pv[j] = a.p[i + j];
          c1 |= (uint32_t)a.c1[i + j] << (8 * j);
          c2 |= (uint32_t)a.c2[i + j] << (8 * j);
        }
    }
    const float s1 = a.absmax1[b], s2 = a.absmax2[b];
    float m[4], v[4], mx1, mx2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      m[j] = v[j] = 0.f;
      if (full || i + j < a.n) {
        const float gc = g[j] * clip;
        m[j] = map1[c1 >> (8 * j) & 255] * s1;
        v[j] = map2[c2 >> (8 * j) & 255] * s2;
        m[j] = m[j] * a.beta1 + (1.f - a.beta1) * gc;
        v[j] = v[j] * a.beta2 + (1.f - a.beta2) * gc * gc;
      }
      // (fmaxf passes over NaN: the maximum is NaN only where the whole block is)
      mx1 = j == 0 ? fabsf(m[j]) : fmaxf(mx1, fabsf(m[j]));
      mx2 = j == 0 ? fabsf(v[j]) : fmaxf(mx2, fabsf(v[j]));
    }
    mx1 = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wave_max(mx1))));
    mx2 = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wave_max(mx2))));
    const BlockMax q1(mx1), q2(mx2);
    if (lane == 0) {
      a.absmax1[b] = mx1;
      a.absmax2[b] = mx2;
    }
    // parameters leave before the codes are searched: their registers are needed there
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pv[j] = pv[j] + a.step_size * (m[j] / (sqrtf(v[j]) + a.eps_scaled));
      if (a.weight_decay > 0.f) pv[j] = pv[j] * (1.f - a.lr * a.weight_decay);
    }
    if (full) {
      once_store<ONCE>(*(f32x4*)pv, (f32x4*)(a.p + i));
      if (a.p_bf16)
        *(uint2*)(a.p_bf16 + i) = make_uint2((uint32_t)f32_to_bf16(pv[0]) | ((uint32_t)f32_to_bf16(pv[1]) << 16),
                                             (uint32_t)f32_to_bf16(pv[2]) | ((uint32_t)f32_to_bf16(pv[3]) << 16));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < a.n) {
          a.p[i + j] = pv[j];
          if (a.p_bf16) a.p_bf16[i + j] = f32_to_bf16(pv[j]);
        }
    }
    // a block without a positive maximum holds the code of 0, also for NaN
    if (!(mx1 > 0.f)) m[0] = m[1] = m[2] = m[3] = 0.f;
    if (!(mx2 > 0.f)) v[0] = v[1] = v[2] = v[3] = 0.f;
    c1 = c2 = 0;
    if (one) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        c1 |= (uint32_t)nearest_code<true>(map1, thr1, lut1, q1.quotient(m[j])) << (8 * j);
        c2 |= (uint32_t)nearest_code<true>(map2, thr2, lut2, q2.quotient(v[j])) << (8 * j);
      }
    } else {
      for (int j = 0; j < 4; ++j) {
        c1 |= (uint32_t)nearest_code<false>(map1, thr1, lut1, q1.quotient(m[j])) << (8 * j);
        c2 |= (uint32_t)nearest_code<false>(map2, thr2, lut2, q2.quotient(v[j])) << (8 * j);
      }
    }
    if (full) {
      once_store<ONCE>(c1, (uint32_t*)(a.c1 + i));
      once_store<ONCE>(c2, (uint32_t*)(a.c2 + i));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < a.n) {
          a.c1[i + j] = (uint8_t)(c1 >> (8 * j));
          a.c2[i + j] = (uint8_t)(c2 >> (8 * j));
        }
    }
  }
}

}  // namespace artk

using namespace artk;

extern "C" {

size_t artk_sumsq_f32_workspace_bytes(void) { return SUMSQ_BLOCKS * sizeof(double) + 256; }

int32_t artk_sumsq_f32(const float* x, int64_t n, float* out, void* workspace, size_t workspace_bytes,
                       artk_stream_t stream) {
  ARTK_CHECK_ARG(x && out && n > 0, "null pointer or empty input");
  Workspace ws(workspace, workspace_bytes);
  double* part = ws.take<double>(SUMSQ_BLOCKS);
  if (!ws.ok()) {
    set_error("workspace too small: need %zu bytes, got %zu", ws.used, workspace_bytes);
    return ARTK_ERR_WORKSPACE_TOO_SMALL;
  }
  hipStream_t st = (hipStream_t)stream;
  sumsq_partial_kernel<<<SUMSQ_BLOCKS, 256, 0, st>>>(x, n, part);
  ARTK_CHECK_LAUNCH();
  sumsq_final_kernel<<<1, 64, 0, st>>>(part, out);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

int32_t artk_adamw_step(float* params, const float* grads, float* exp_avg, float* exp_avg_sq,
                        void* params_bf16, int64_t n, float lr, float beta1, float beta2, float eps,
                        float weight_decay, int32_t step, const float* grad_sumsq, float max_grad_norm,
                        artk_stream_t stream) {
  ARTK_CHECK_ARG(params && grads && exp_avg && exp_avg_sq, "null pointer argument");
  ARTK_CHECK_ARG(n > 0 && step >= 1, "n must be positive and step >= 1");
  ARTK_CHECK_ARG(aligned16(params) && aligned16(grads) && aligned16(exp_avg) && aligned16(exp_avg_sq) &&
                     (params_bf16 == nullptr || (((uintptr_t)params_bf16) & 7) == 0),
                 "buffers must be 16-byte aligned (bf16 copy: 8-byte)");
  ARTK_CHECK_ARG(beta1 >= 0.f && beta1 < 1.f && beta2 >= 0.f && beta2 < 1.f, "betas must be in [0, 1)");
  AdamWParams a;
  a.p = params;
  a.g = grads;
  a.m = exp_avg;
  a.v = exp_avg_sq;
  a.p_bf16 = (uint16_t*)params_bf16;
  a.grad_sumsq = grad_sumsq;
  a.n = n;
  a.lr = lr;
  a.beta1 = beta1;
  a.beta2 = beta2;
  a.eps = eps;
  a.weight_decay = weight_decay;
  a.max_grad_norm = max_grad_norm;
  // bias corrections in double on the host, as torch computes them with Python floats
  const double bc1 = 1.0 - pow((double)beta1, (double)step);
  const double bc2 = 1.0 - pow((double)beta2, (double)step);
  a.step_size = (float)((double)lr / bc1);
  a.inv_bc2_sqrt = (float)(1.0 / sqrt(bc2));
  const int64_t n4 = (n + 3) / 4;
  if (step_once32(n)) adamw_kernel<true><<<(unsigned)((n4 + 255) / 256), 256, 0, (hipStream_t)stream>>>(a);
  else adamw_kernel<false><<<(unsigned)((n4 + 255) / 256), 256, 0, (hipStream_t)stream>>>(a);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

int32_t artk_adamw8bit_step(float* params, const float* grads, void* state1, void* state2, float* absmax1,
                            float* absmax2, const float* qmap1, const float* qmap2, void* params_bf16,
                            int64_t n, float lr, float beta1, float beta2, float eps, float weight_decay,
                            int32_t step, const float* grad_sumsq, float max_grad_norm,
                            artk_stream_t stream) {
  ARTK_CHECK_ARG(params && grads && state1 && state2 && absmax1 && absmax2 && qmap1 && qmap2,
                 "null pointer argument");
  ARTK_CHECK_ARG(n > 0 && step >= 1, "n must be positive and step >= 1");
  ARTK_CHECK_ARG(beta1 >= 0.f && beta1 < 1.f && beta2 >= 0.f && beta2 < 1.f, "betas must be in [0, 1)");
  AdamW8Params a;
  a.p = params;
  a.g = grads;
  a.c1 = (uint8_t*)state1;
  a.c2 = (uint8_t*)state2;
  a.absmax1 = absmax1;
  a.absmax2 = absmax2;
  a.qmap1 = qmap1;
  a.qmap2 = qmap2;
  a.p_bf16 = (uint16_t*)params_bf16;
  a.grad_sumsq = grad_sumsq;
  a.n = n;
  a.lr = lr;
  a.beta1 = beta1;
  a.beta2 = beta2;
  a.eps = eps;
  a.weight_decay = weight_decay;
  a.max_grad_norm = max_grad_norm;
  const double c1 = 1.0 - pow((double)beta1, (double)step);
  const double c2 = sqrt(1.0 - pow((double)beta2, (double)step));
  a.step_size = (float)(-(double)lr * c2 / c1);
  a.eps_scaled = (float)(c2 * (double)eps);
  const int64_t n_blocks = (n + 255) / 256, per_group = ADAM8_THREADS / 64;
  int64_t grid = (n_blocks + per_group - 1) / per_group;
  if (grid > 2 * num_cus()) grid = 2 * num_cus();
  // 16-byte accesses where every buffer allows them (buffers of FlatParams do)
  const int vec = aligned16(params) && aligned16(grads) && (((uintptr_t)state1 | (uintptr_t)state2) & 3) == 0 &&
                  ((uintptr_t)params_bf16 & 7) == 0;
  if (step_once8(n)) adamw8bit_kernel<true><<<(unsigned)grid, ADAM8_THREADS, 0, (hipStream_t)stream>>>(a, n_blocks, vec);
  else adamw8bit_kernel<false><<<(unsigned)grid, ADAM8_THREADS, 0, (hipStream_t)stream>>>(a, n_blocks, vec);
  ARTK_CHECK_LAUNCH();
  return ARTK_OK;
}

}  // extern "C"
