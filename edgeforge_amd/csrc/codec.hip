// Block codec on the device: the reference quantizer (Q4_0 scale search, Q8_0), 16-bit float
// packing, and row lookup (dequantization / widening) for embeddings.
//
// The quantizer is the reference's per-block algorithm (src/quant.cpp:26-99, 151-175), one thread
// per 32-weight block, written so that every rounding is the reference's, in its order (correctly
// rounded divides, no contraction but where the product is exact), so the packed bytes are identical.
#include <cmath>

#include "codec.h"

#pragma clang fp contract(off)

namespace efh {
namespace {

// binary32 -> binary16, round to nearest even (include/ef/fp16.h:69-91).
__device__ uint16_t f32_to_fp16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  const uint16_t sign = static_cast<uint16_t>((u >> 16) & 0x8000u);
  const uint32_t a = u & 0x7FFFFFFFu;
  if (a > 0x7F800000u) return static_cast<uint16_t>(sign | 0x7E00u | ((a >> 13) & 0x3FFu));
  if (a >= 0x477FF000u) return static_cast<uint16_t>(sign | 0x7C00u);
  if (a < 0x38800000u) {
    if (a <= 0x33000000u) return sign;
    const uint32_t m = (a & 0x7FFFFFu) | 0x800000u;
    const uint32_t sh = 126u - (a >> 23);
    uint32_t r = m >> sh;
    const uint32_t rest = m & ((1u << sh) - 1u), half = 1u << (sh - 1u);
    if (rest > half || (rest == half && (r & 1u))) ++r;
    return static_cast<uint16_t>(sign | r);
  }
  const uint32_t x = a - 0x38000000u;
  return static_cast<uint16_t>(sign | ((x + 0xFFFu + ((x >> 13) & 1u)) >> 13));
}

// binary32 -> bfloat16, round to nearest even, NaN kept quiet (include/ef/fp16.h:32-40).
__device__ uint16_t f32_to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

__device__ float fp16_round(float d) { return half_bits_to_float(f32_to_fp16_bits(d)); }

// clamp(static_cast<int>(v), lo, hi) of a rounded v, as a float, as the reference's x86-64 build
// executes the cast (cvttss2si): NaN and out-of-range values give INT_MIN, so lo.  CLEAN: the caller
// knows that |v| < 2^31.
template <bool CLEAN>
__device__ __forceinline__ float clamp_code(float v, float lo, float hi) {
  const float c = __builtin_amdgcn_fmed3f(v, lo, hi);
  return CLEAN || fabsf(v) < 2147483648.0f ? c : lo;
}

// Squared error of the block's codes at scale d: each error and square and the running sum round as the
// reference's (code times scale is exact: 4 by 11 bits, so the subtraction may be a fused one).
template <bool CLEAN>
__device__ __forceinline__ double q4_sse(const float (&x)[32], float d) {
  const float inv = __fdiv_rn(1.0f, d);
  const double dd = static_cast<double>(d);
  double sse = 0.0;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    const double e = __builtin_fma(-static_cast<double>(clamp_code<CLEAN>(rintf(x[j] * inv), -8.0f, 7.0f)), dd,
                                   static_cast<double>(x[j]));
    sse += e * e;
  }
  return sse;
}

// q4_group's scale for one 32-weight block (src/quant.cpp:26-99); 0 means every code 8.  Only the scale is
// kept from try to try: the codes follow from it.  A wave
// without NaN whose codes all fit an int takes the short clamp.
__device__ float q4_scale(const float (&x)[32], bool search) {
  float amax = 0.0f, smax = 0.0f;
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    const float a = fabsf(x[j]);
    nan = nan || a != a;
    if (a > amax) {
      amax = a;
      smax = x[j];
    }
  }
  if (!(amax > 0.0f) || !isfinite(amax)) return 0.0f;
  if (!search) {  // one candidate: its error decides nothing
    const float d = fp16_round(fminf(fmaxf(__fdiv_rn(smax, -8.0f), -65504.0f), 65504.0f));
    return d != 0.0f ? d : 0.0f;
  }
  // at |d| >= 2^-24, the least fp16 scale, |x / d| <= amax 2^24
  const bool clean = __all(!nan && amax < 64.0f);
  auto sse_of = [&](float d) { return clean ? q4_sse<true>(x, d) : q4_sse<false>(x, d); };
  float best = 0.0f;
  double best_sse = -1.0;
  for (int c = 0; c < 6; ++c) {
    const float num = c == 0 ? smax : amax;
    const float den = c == 0 ? -8.0f : (c == 5 ? 8.0f : 6.75f + 0.25f * static_cast<float>(c));  // 7, 7.25, 7.5, 7.75, 8
    const float d = fp16_round(fminf(fmaxf(__fdiv_rn(num, den), -65504.0f), 65504.0f));
    if (d == 0.0f) continue;
    const double sse = sse_of(d);
    if (best_sse < 0.0 || sse < best_sse) {
      best_sse = sse;
      best = d;
    }
  }
  if (best_sse < 0.0) return 0.0f;
  for (int round = 0; round < 2; ++round) {
    // least squares over the codes of the best scale: integer products and their sum are exact
    const float inv = __fdiv_rn(1.0f, best);
    double num = 0.0;
    float den = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const float c = clean ? clamp_code<true>(rintf(x[j] * inv), -8.0f, 7.0f)
                            : clamp_code<false>(rintf(x[j] * inv), -8.0f, 7.0f);
      num = __builtin_fma(static_cast<double>(x[j]), static_cast<double>(c), num);
      den += c * c;
    }
    if (den == 0.0f) break;
    double ls = num / static_cast<double>(den);
    ls = ls < -65504.0 ? -65504.0 : (ls > 65504.0 ? 65504.0 : ls);
    const float d = fp16_round(static_cast<float>(ls));
    if (d == 0.0f || d == best) break;
    const double sse = sse_of(d);
    if (!(sse < best_sse)) break;
    best_sse = sse;
    best = d;
  }
  return best;
}

// A workgroup packs kQuantBlocks consecutive blocks: their weights come in coalesced through LDS (rows of
// 33 floats, so that the threads' reads fall in distinct banks) and their bytes leave through it the
// same way.  Bound by vector issue: eight tries of 32 weights at seven instructions, four of them on
// doubles (the reference's sequential double sums).  Q4_0 with the search, 5632x2048: 54.5 us per call
// with strided loads, codes kept per try and twice the instructions, 39.8 us so (1.3 TB/s; 500x512
// 14.5 -> 10.5), without it 15.9 -> 12.8; Q8_0 11.7 -> 10.9 (5.4 TB/s).  256 blocks per workgroup cost small
// matrices 0.7 to 2 us.
constexpr int kQuantBlocks = 64;  // one wave: small matrices reach more CUs, and the tail is short

template <bool Q4>
__global__ __launch_bounds__(kQuantBlocks) void quantize_blocks_kernel(const float* __restrict__ w, long blocks,
                                                                       int search, uint8_t* __restrict__ out) {
  constexpr int kBytes = Q4 ? 18 : 34, kLd = 33;
  __shared__ __attribute__((aligned(16))) float xs[kQuantBlocks * kLd];
  const long g0 = static_cast<long>(blockIdx.x) * kQuantBlocks;
  const int n = static_cast<int>(min(static_cast<long>(kQuantBlocks), blocks - g0)), t = threadIdx.x;
  const float* src = w + g0 * 32;
  const bool aligned = reinterpret_cast<uintptr_t>(src) % 16 == 0;
  auto put4 = [&](int q, float4 v) {  // the workgroup's weights 4 q .. 4 q + 3
    float* p = xs + (q >> 3) * kLd + 4 * (q & 7);
    p[0] = v.x;
    p[1] = v.y;
    p[2] = v.z;
    p[3] = v.w;
  };
  if (n == kQuantBlocks && aligned) {
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = reinterpret_cast<const float4*>(src)[t + kQuantBlocks * i];
#pragma unroll
    for (int i = 0; i < 8; ++i) put4(t + kQuantBlocks * i, v[i]);
  } else if (aligned) {  // the last blocks
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = t + kQuantBlocks * i < n * 8 ? reinterpret_cast<const float4*>(src)[t + kQuantBlocks * i]
                                          : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int i = 0; i < 8; ++i) put4(t + kQuantBlocks * i, v[i]);
  } else {  // weights off a 16-byte boundary
    float v[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i] = t + kQuantBlocks * i < n * 32 ? src[t + kQuantBlocks * i] : 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int e = t + kQuantBlocks * i;
      xs[(e >> 5) * kLd + (e & 31)] = v[i];
    }
  }
  __syncthreads();
  float x[32];
#pragma unroll
  for (int j = 0; j < 32; ++j) x[j] = t < n ? xs[t * kLd + j] : 0.0f;
  __syncthreads();
  uint32_t words[Q4 ? 4 : 8];
  uint16_t h;
  if constexpr (Q4) {
    const float d = q4_scale(x, search != 0);
    h = f32_to_fp16_bits(d);
    const float inv = d != 0.0f ? __fdiv_rn(1.0f, d) : 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) words[k] = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const float c = d != 0.0f ? clamp_code<false>(rintf(x[j] * inv), -8.0f, 7.0f) : 0.0f;
      const uint32_t code = static_cast<uint32_t>(static_cast<int>(c) + 8);
      words[(j & 15) >> 2] |= code << (8 * (j & 3) + (j < 16 ? 0 : 4));
    }
  } else {  // Q8_0 (src/quant.cpp:166-175)
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j) amax = fmaxf(amax, fabsf(x[j]));
    float d = 0.0f;
    if (amax > 0.0f && isfinite(amax)) d = fp16_round(fminf(__fdiv_rn(amax, 127.0f), 65504.0f));
    h = f32_to_fp16_bits(d);
    const float inv = d != 0.0f ? __fdiv_rn(1.0f, d) : 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) words[k] = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int c = static_cast<int>(clamp_code<false>(rintf(x[j] * inv), -127.0f, 127.0f));
      words[j >> 2] |= (static_cast<uint32_t>(c) & 0xFFu) << (8 * (j & 3));
    }
  }
  // the block's bytes: 16-bit pieces at an even offset
  uint16_t* o16 = reinterpret_cast<uint16_t*>(xs) + t * (kBytes / 2);
  if (t < n) {
    o16[0] = h;
#pragma unroll
    for (int k = 0; k < (Q4 ? 4 : 8); ++k) {
      o16[1 + 2 * k] = static_cast<uint16_t>(words[k] & 0xFFFFu);
      o16[2 + 2 * k] = static_cast<uint16_t>(words[k] >> 16);
    }
  }
  __syncthreads();
  uint8_t* dst = out + g0 * kBytes;
  const int bytes = n * kBytes, whole = reinterpret_cast<uintptr_t>(dst) % 16 == 0 ? bytes / 16 : 0;
  for (int i = t; i < whole; i += kQuantBlocks)
    reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(xs)[i];
  for (int i = 16 * whole + t; i < bytes; i += kQuantBlocks) dst[i] = reinterpret_cast<const uint8_t*>(xs)[i];
}

__global__ void pack16_kernel(int qtype, const float* __restrict__ w, size_t n, uint16_t* __restrict__ out) {
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    out[i] = qtype == EF_QTYPE_BF16 ? f32_to_bf16_bits(w[i]) : f32_to_fp16_bits(w[i]);
  }
}

// Row lookup: out[b][:] = row ids[b] of W as FP32 (kern::row_f32, src/qkernels.cpp:299-305).
__global__ void rows_f32_kernel(const uint8_t* __restrict__ W, int qtype, long rows, long cols, long rb,
                                const int32_t* __restrict__ ids, float* __restrict__ out, long ldo) {
  const int b = blockIdx.y;
  const int32_t id = ids[b];
  float* o = out + b * ldo;
  const bool ok = id >= 0 && id < rows;
  const uint8_t* row = W + (ok ? id : 0) * rb;
  for (long c = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; c < cols;
       c += static_cast<long>(gridDim.x) * blockDim.x) {
    float v = 0.0f;
    if (!ok) {
      v = __int_as_float(0x7FC00000);  // an out-of-range id yields NaN rows (callers validate ids first)
    } else if (qtype == EF_QTYPE_F32) {
      v = reinterpret_cast<const float*>(row)[c];
    } else if (qtype == EF_QTYPE_BF16) {
      v = __uint_as_float(static_cast<uint32_t>(reinterpret_cast<const uint16_t*>(row)[c]) << 16);
    } else if (qtype == EF_QTYPE_F16) {
      v = half_bits_to_float(reinterpret_cast<const uint16_t*>(row)[c]);
    } else {
      const long blk = c >> 5, j = c & 31;
      if (qtype == EF_QTYPE_Q4_0) {
        const uint8_t* p = row + blk * 18;
        const float d = half_bits_to_float(static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 8));
        const int code = j < 16 ? (p[2 + j] & 15) : (p[2 + j - 16] >> 4);
        v = static_cast<float>(code - 8) * d;
      } else {
        const uint8_t* p = row + blk * 34;
        const float d = half_bits_to_float(static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 8));
        v = static_cast<float>(static_cast<int8_t>(p[2 + j])) * d;
      }
    }
    o[c] = v;
  }
}

}  // namespace

int launch_quantize(int qtype, const float* w, size_t rows, size_t cols, int search, void* out, hipStream_t s) {
  if (qtype == EF_QTYPE_Q4_0 || qtype == EF_QTYPE_Q8_0) {
    const size_t blocks = rows * (cols / 32);
    const unsigned grid = static_cast<unsigned>((blocks + kQuantBlocks - 1) / kQuantBlocks);
    if (qtype == EF_QTYPE_Q4_0) {
      hipLaunchKernelGGL(quantize_blocks_kernel<true>, dim3(grid), dim3(kQuantBlocks), 0, s, w,
                         static_cast<long>(blocks), search, static_cast<uint8_t*>(out));
    } else {
      hipLaunchKernelGGL(quantize_blocks_kernel<false>, dim3(grid), dim3(kQuantBlocks), 0, s, w,
                         static_cast<long>(blocks), search, static_cast<uint8_t*>(out));
    }
  } else if (qtype == EF_QTYPE_BF16 || qtype == EF_QTYPE_F16) {
    const size_t n = rows * cols;
    const unsigned grid = static_cast<unsigned>(std::min<size_t>((n + 255) / 256, 65536));
    hipLaunchKernelGGL(pack16_kernel, dim3(grid), dim3(256), 0, s, qtype, w, n, static_cast<uint16_t*>(out));
  } else {
    EFH_HIP(hipMemcpyAsync(out, w, rows * cols * 4, hipMemcpyDeviceToDevice, s));
  }
  EFH_HIP(hipGetLastError());
  return EF_HIP_OK;
}

int launch_rows_f32(const ef_hip_weight_s* W, const int32_t* ids, int batch, float* out, size_t ldo, hipStream_t s) {
  const unsigned gx = static_cast<unsigned>(std::min<size_t>((W->cols + 255) / 256, 64));
  hipLaunchKernelGGL(rows_f32_kernel, dim3(gx, batch), dim3(256), 0, s, W->dev, W->qtype, static_cast<long>(W->rows),
                     static_cast<long>(W->cols), static_cast<long>(W->row_bytes), ids, out, static_cast<long>(ldo));
  EFH_HIP(hipGetLastError());
  return EF_HIP_OK;
}

}  // namespace efh

// ---- synthetic inputs -----------------------------------------------------------------------------------
// N(mean, scale^2) floats from Philox4x32-10 (Salmon et al., "Parallel random numbers: as easy as
// 1, 2, 3", SC'11) and the Box-Muller transform: element i uses counter (i / 4, offset), key seed.
// Deterministic for (seed, offset, i) on every run; used to build synthetic weights and inputs.
namespace efh {
namespace {

__device__ __forceinline__ void philox_round(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
  const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c[0];
  const uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * c[2];
  const uint32_t n0 = static_cast<uint32_t>(p1 >> 32) ^ c[1] ^ k0;
  const uint32_t n2 = static_cast<uint32_t>(p0 >> 32) ^ c[3] ^ k1;
  c[1] = static_cast<uint32_t>(p1);
  c[3] = static_cast<uint32_t>(p0);
  c[0] = n0;
  c[2] = n2;
}

__global__ void fill_normal_kernel(float* __restrict__ out, size_t n, uint64_t seed, uint64_t offset, float mean,
                                   float scale) {
  const size_t q = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q * 4 >= n) return;
  uint32_t c[4] = {static_cast<uint32_t>(q), static_cast<uint32_t>(q >> 32), static_cast<uint32_t>(offset),
                   static_cast<uint32_t>(offset >> 32)};
  uint32_t k0 = static_cast<uint32_t>(seed), k1 = static_cast<uint32_t>(seed >> 32);
  for (int r = 0; r < 10; ++r) {
    philox_round(c, k0, k1);
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  float z[4];
  for (int h = 0; h < 2; ++h) {
    const float u1 = (static_cast<float>(c[2 * h] >> 8) + 0.5f) * 0x1p-24f;  // (0, 1)
    const float u2 = static_cast<float>(c[2 * h + 1] >> 8) * 0x1p-24f;       // [0, 1)
    const float r = sqrtf(-2.0f * logf(u1));
    z[2 * h] = r * cosf(6.28318530717958647692f * u2);
    z[2 * h + 1] = r * sinf(6.28318530717958647692f * u2);
  }
  for (int j = 0; j < 4; ++j)
    if (q * 4 + j < n) out[q * 4 + j] = mean + scale * z[j];
}

}  // namespace

int launch_fill_normal(float* out, size_t n, uint64_t seed, uint64_t offset, float mean, float scale,
                       hipStream_t s) {
  const size_t quads = (n + 3) / 4;
  hipLaunchKernelGGL(fill_normal_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, s, out, n,
                     seed, offset, mean, scale);
  EFH_HIP(hipGetLastError());
  return EF_HIP_OK;
}

}  // namespace efh
