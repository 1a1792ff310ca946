// pack.hip -- weight quantisation on the GPU, bit-exact with the reference's
// torch arithmetic (IEEE fp32 division, round-half-to-even).
//
//   INT4 (moe_int4_kernel.py:37-93): per (row, group) scale = max|w| / 7 in
//   fp32 floored at fp32 eps; q = rint(w / scale) clamped to [-8, 7]; nibble
//   q + 8, even k in the low nibble; scale stored as fp16.
//   INT8 (quant_shim.py:84-96 rule): per row scale = max|w| / 127 (floored at
//   fp32 eps); q = rint(w / scale) clamped to [-128, 127]; scale stored fp16.
#include "exq_internal.h"

namespace exq {
namespace {

constexpr float kFp32Eps = 1.1920928955078125e-07f;  // 2^-23

// 8 consecutive weights as loaded (16 bytes, two of them for f32), nontemporal
// (each is read once), and as fp32.
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
template <int DT>
struct Raw8 {
  u32x4_t q[DT == EXQ_DTYPE_F32 ? 2 : 1];
};
template <int DT>
__device__ __forceinline__ Raw8<DT> load_raw8(const void* w, int64_t i) {
  Raw8<DT> r;
  const char* p = reinterpret_cast<const char*>(w) + i * (DT == EXQ_DTYPE_F32 ? 4 : 2);
  r.q[0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  if constexpr (DT == EXQ_DTYPE_F32)
    r.q[1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p + 16));
  return r;
}
template <int DT>
__device__ __forceinline__ void unpack8(const Raw8<DT>& r, float (&v)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (DT == EXQ_DTYPE_F32) {
      v[j] = __uint_as_float(r.q[0][j]);
      v[4 + j] = __uint_as_float(r.q[1][j]);
    } else if constexpr (DT == EXQ_DTYPE_BF16) {
      v[2 * j] = __uint_as_float(r.q[0][j] << 16);
      v[2 * j + 1] = __uint_as_float(r.q[0][j] & 0xffff0000u);
    } else {
      v[2 * j] = f16_bits_to_f32(r.q[0][j] & 0xffffu);
      v[2 * j + 1] = f16_bits_to_f32(r.q[0][j] >> 16);
    }
  }
}

// rint(v / scale) of 8 weights, clamped to [lo, hi], with the quotient rounded
// as IEEE division rounds it.  v * (1 / scale) is within 3 ulp of the quotient,
// so both round to the same integer unless the product lies within TIE of a
// half-way point (|v / scale| <= hi + 1, so 3 ulp are 1.5e-6 for INT4 and 2.4e-5
// for INT8); only then the divisions are done.  That is 2 TIE of all weights, 2e-5
// (INT4) and 2e-4 (INT8); a wave takes the branch when any of its 512 weights does,
// 1 % and 10 % of them.  (A NaN product takes the first form; it is NaN in both.)
template <int HI>
__device__ __forceinline__ void quantize8(const float (&v)[8], float scale, int (&q)[8]) {
  constexpr float TIE = HI == 7 ? 1e-5f : 1e-4f;
  const float inv = 1.0f / scale;
  float t[8], worst = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float x = v[j] * inv;
    t[j] = rintf(x);
    worst = fmaxf(worst, fabsf(x - t[j]));
  }
  if (worst > 0.5f - TIE) {
#pragma unroll
    for (int j = 0; j < 8; ++j) t[j] = rintf(v[j] / scale);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) q[j] = (int)fminf(fmaxf(t[j], (float)(-HI - 1)), (float)HI);
}

__device__ __forceinline__ float load1(const void* w, int dtype, int64_t i) {
  return load_as_f32(w, dtype, i);
}

// Eight consecutive k per thread and step; the tpg = 2^shift threads of a group
// (g / 8, at most 64) reduce max|w| with lane shuffles.  K is a multiple of g,
// so weights, packed words and groups are all linear in the chunk index (no row
// arithmetic), and a work-group's PACK_U steps are PACK_U loads in flight per
// thread.  Bound: HBM.  OLMoE bank in f16 (805 MB in, 214 MB out): 346 -> 214
// us (4.8 TB/s) against one chunk per thread with a 64-bit division for its
// row and eight IEEE divisions.
constexpr int PACK_U = 4;

template <int DT>
__global__ void __launch_bounds__(256) pack_int4_kernel(const void* __restrict__ w,
                                                        int64_t chunks, int shift,
                                                        uint32_t* __restrict__ packed,
                                                        uint16_t* __restrict__ scales) {
  const int tpg = 1 << shift;
  const int64_t c0 = (int64_t)blockIdx.x * (256 * PACK_U) + threadIdx.x;
  Raw8<DT> r[PACK_U];
#pragma unroll
  for (int u = 0; u < PACK_U; ++u) {
    const int64_t c = c0 + u * 256;
    if (c < chunks) {
      r[u] = load_raw8<DT>(w, c * 8);
    } else {
      r[u] = Raw8<DT>{};
    }
  }
#pragma unroll
  for (int u = 0; u < PACK_U; ++u) {
    const int64_t c = c0 + u * 256;
    float v[8];
    unpack8<DT>(r[u], v);
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(v[j]));
    for (int d = 1; d < tpg; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    const float scale = fmaxf(m / 7.0f, kFp32Eps);
    if (c >= chunks) continue;
    int q[8];
    quantize8<7>(v, scale, q);
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) word |= (uint32_t)(q[j] + 8) << (4 * j);
    __builtin_nontemporal_store(word, packed + c);
    if ((c & (tpg - 1)) == 0) scales[c >> shift] = (uint16_t)f32_to_f16_bits(scale);
  }
}

// Fallback for group sizes whose chunk count is not a power of two (e.g. the
// K < 128 collapse to g = K): one thread per (row, group), serial over g.
__global__ void __launch_bounds__(256) pack_int4_serial_kernel(
    const void* __restrict__ w, int dtype, int64_t rows, int K, int g,
    uint8_t* __restrict__ packed, uint16_t* __restrict__ scales) {
  const int ng = K / g;
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= rows * ng) return;
  const int64_t row = tid / ng;
  const int grp = (int)(tid - row * ng);
  const int64_t base = row * K + (int64_t)grp * g;
  float m = 0.f;
  for (int k = 0; k < g; ++k) m = fmaxf(m, fabsf(load1(w, dtype, base + k)));
  const float scale = fmaxf(m / 7.0f, kFp32Eps);
  for (int k = 0; k < g; k += 2) {
    float q0 = fminf(fmaxf(rintf(load1(w, dtype, base + k) / scale), -8.f), 7.f);
    float q1 = fminf(fmaxf(rintf(load1(w, dtype, base + k + 1) / scale), -8.f), 7.f);
    packed[(base + k) / 2] = (uint8_t)(((int)q0 + 8) | (((int)q1 + 8) << 4));
  }
  scales[row * ng + grp] = (uint16_t)f32_to_f16_bits(scale);
}

// INT8 rows with K % 8 == 0: WPR waves per row (1 up to 4096 weights, else the
// four of a work-group), each lane R chunks of 8 weights, all loaded at once and
// kept in registers between the row's maximum and the quantisation.  Bound:
// HBM; 13 OLMoE w13 experts in f16 (109 MB in, 55 MB out) 110 -> 31 us against
// one work-group per row that read every weight twice, one at a time.
template <int DT, int WPR, int R>
__global__ void __launch_bounds__(256) quant_int8_rows_kernel(const void* __restrict__ w,
                                                              int64_t rows, int K,
                                                              int8_t* __restrict__ q,
                                                              uint16_t* __restrict__ scales) {
  __shared__ float red[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * (4 / WPR) + (WPR == 1 ? wave : 0);
  if (row >= rows) return;  // wave-uniform; work-group-uniform for WPR 4
  const int first = (WPR == 1 ? 0 : wave) * 64 + lane, cpr = K / 8;
  Raw8<DT> r[R];
  float m = 0.f;
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int c = first + u * (64 * WPR);
    r[u] = c < cpr ? load_raw8<DT>(w, row * K + (int64_t)c * 8) : Raw8<DT>{};
  }
#pragma unroll
  for (int u = 0; u < R; ++u) {
    float v[8];
    unpack8<DT>(r[u], v);
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(v[j]));
  }
  for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if constexpr (WPR == 4) {
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  }
  const float scale = fmaxf(m / 127.0f, kFp32Eps);
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int c = first + u * (64 * WPR);
    if (c >= cpr) continue;
    float v[8];
    unpack8<DT>(r[u], v);
    int qv[8];
    quantize8<127>(v, scale, qv);
    u32x2_t o;
    o.x = (uint32_t)(qv[0] & 255) | (uint32_t)(qv[1] & 255) << 8 | (uint32_t)(qv[2] & 255) << 16 |
          (uint32_t)qv[3] << 24;
    o.y = (uint32_t)(qv[4] & 255) | (uint32_t)(qv[5] & 255) << 8 | (uint32_t)(qv[6] & 255) << 16 |
          (uint32_t)qv[7] << 24;
    __builtin_nontemporal_store(o, reinterpret_cast<u32x2_t*>(q + row * K + (int64_t)c * 8));
  }
  if (first == 0) scales[row] = (uint16_t)f32_to_f16_bits(scale);
}

// Other rows: one work-group per row, max|w| over K, then quantise.
__global__ void __launch_bounds__(256) quant_int8_kernel(const void* __restrict__ w, int dtype,
                                                         int K, int8_t* __restrict__ q,
                                                         uint16_t* __restrict__ scales) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const int64_t base = row * K;
  float m = 0.f;
  for (int k = threadIdx.x; k < K; k += blockDim.x) m = fmaxf(m, fabsf(load1(w, dtype, base + k)));
  for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float scale = fmaxf(m / 127.0f, kFp32Eps);
  for (int k = threadIdx.x; k < K; k += blockDim.x) {
    const float v = rintf(load1(w, dtype, base + k) / scale);
    q[base + k] = (int8_t)(int)fminf(fmaxf(v, -128.f), 127.f);
  }
  if (threadIdx.x == 0) scales[row] = (uint16_t)f32_to_f16_bits(scale);
}

// Store v (fp32) in the weights' dtype, rounded to nearest even.
__device__ __forceinline__ void store1(void* out, int dtype, int64_t i, float v) {
  if (dtype == EXQ_DTYPE_F32)
    reinterpret_cast<float*>(out)[i] = v;
  else if (dtype == EXQ_DTYPE_BF16)
    reinterpret_cast<uint16_t*>(out)[i] = (uint16_t)f32_to_bf16_bits(v);
  else
    reinterpret_cast<uint16_t*>(out)[i] = (uint16_t)f32_to_f16_bits(v);
}

// Maximum and clamp that keep NaN, as torch's amax and clamp do (quant_shim.py:
// 92-95): a NaN or infinite weight makes its whole row (INT8) or group (INT4)
// NaN.  fmaxf / fminf alone would return the other operand.
__device__ __forceinline__ float max_keep_nan(float a, float b) {
  return __builtin_isnan(a) ? a : (__builtin_isnan(b) ? b : fmaxf(a, b));
}
__device__ __forceinline__ float clamp_keep_nan(float v, float lo, float hi) {
  return __builtin_isnan(v) ? v : fminf(fmaxf(v, lo), hi);
}

// Fake quantisation (quantise then dequantise in place of the weights):
// INT4 per group of g along the row (a short last group counts as padded with
// zeros), INT8 per row; out = q * scale with the fp32 scale, in the weights'
// dtype.  One wave per (row, group) for INT4 (g <= 512, lanes stride the
// group), one work-group per row for INT8.
// (`out` may alias `w`: each element is read, then written, by one lane.)
__global__ void __launch_bounds__(256) fake_int4_kernel(const void* w, int dtype, int64_t rows,
                                                        int K, int g, void* out) {
  const int ng = (K + g - 1) / g;
  const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= rows * ng) return;  // wave-uniform
  const int lane = threadIdx.x & 63;
  const int64_t row = unit / ng;
  const int k0 = (int)(unit - row * ng) * g;
  const int k1 = k0 + g < K ? k0 + g : K;
  const int64_t base = row * K;
  float m = 0.f;
  for (int k = k0 + lane; k < k1; k += 64) m = max_keep_nan(m, fabsf(load1(w, dtype, base + k)));
  for (int d = 1; d < 64; d <<= 1) m = max_keep_nan(m, __shfl_xor(m, d, 64));
  const float scale = max_keep_nan(m / 7.0f, kFp32Eps);
  for (int k = k0 + lane; k < k1; k += 64) {
    const float q = clamp_keep_nan(rintf(load1(w, dtype, base + k) / scale), -8.f, 7.f);
    store1(out, dtype, base + k, q * scale);
  }
}

__global__ void __launch_bounds__(256) fake_int8_kernel(const void* w, int dtype, int K,
                                                        void* out) {
  __shared__ float red[4];
  const int64_t base = (int64_t)blockIdx.x * K;
  float m = 0.f;
  for (int k = threadIdx.x; k < K; k += blockDim.x)
    m = max_keep_nan(m, fabsf(load1(w, dtype, base + k)));
  for (int d = 1; d < 64; d <<= 1) m = max_keep_nan(m, __shfl_xor(m, d, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = max_keep_nan(max_keep_nan(red[0], red[1]), max_keep_nan(red[2], red[3]));
  const float scale = max_keep_nan(m / 127.0f, kFp32Eps);
  for (int k = threadIdx.x; k < K; k += blockDim.x) {
    const float q = clamp_keep_nan(rintf(load1(w, dtype, base + k) / scale), -128.f, 127.f);
    store1(out, dtype, base + k, q * scale);
  }
}

}  // namespace
}  // namespace exq

using namespace exq;

extern "C" int exq_fake_quant(const void* weights, int dtype, int64_t rows, int64_t K, int bits,
                              int64_t group_size, void* out, exq_stream stream) {
  const char* fn = "exq_fake_quant";
  EXQ_REQUIRE(is_float_dtype(dtype), "%s: dtype must be f32, f16 or bf16", fn);
  EXQ_REQUIRE(bits == 4 || bits == 8, "%s: bits must be 4 or 8 (got %d)", fn, bits);
  EXQ_REQUIRE(rows >= 0 && rows <= INT32_MAX && K >= 1 && K <= INT32_MAX, "%s: bad sizes", fn);
  EXQ_REQUIRE(bits == 8 || (group_size >= 1 && group_size <= 512),
              "%s: group_size=%lld must be in [1, 512]", fn, (long long)group_size);
  if (rows == 0) return EXQ_SUCCESS;
  EXQ_REQUIRE(weights && out, "%s: null pointer", fn);
  hipStream_t s = as_stream(stream);
  if (bits == 4) {
    const int64_t units = rows * cdiv(K, group_size);
    EXQ_REQUIRE(cdiv(units, 4) <= INT32_MAX, "%s: too many groups", fn);
    hipLaunchKernelGGL(fake_int4_kernel, dim3((unsigned)cdiv(units, 4)), dim3(256), 0, s, weights,
                       dtype, rows, (int)K, (int)group_size, out);
  } else {
    hipLaunchKernelGGL(fake_int8_kernel, dim3((unsigned)rows), dim3(256), 0, s, weights, dtype,
                       (int)K, out);
  }
  return check_launch(fn);
}

extern "C" int exq_pack_int4(const void* weights, int dtype, int64_t rows, int64_t K,
                             int64_t group_size, uint8_t* packed, uint16_t* scales,
                             exq_stream stream) {
  const char* fn = "exq_pack_int4";
  EXQ_REQUIRE(is_float_dtype(dtype), "%s: dtype must be f32, f16 or bf16", fn);
  EXQ_REQUIRE(rows >= 0 && K >= 2 && K % 2 == 0 && K <= INT32_MAX,
              "%s: K=%lld must be even and positive", fn, (long long)K);
  EXQ_REQUIRE(group_size >= 2, "%s: group_size=%lld", fn, (long long)group_size);
  const int64_t g = K < group_size ? K : group_size;  // K < g collapses to one group
  EXQ_REQUIRE(K % g == 0 && g % 2 == 0, "%s: K=%lld must be divisible by group_size=%lld", fn,
              (long long)K, (long long)g);
  if (rows == 0) return EXQ_SUCCESS;
  EXQ_REQUIRE(weights && packed && scales, "%s: null pointer", fn);
  EXQ_REQUIRE(cdiv(rows * (K / 2), 256) <= INT32_MAX, "%s: %lld x %lld weights is too large", fn,
              (long long)rows, (long long)K);
  const int tpg = (int)(g / 8);
  const bool fast = g % 8 == 0 && tpg <= 64 && (tpg & (tpg - 1)) == 0 &&
                    ((uintptr_t)weights % 16 == 0) && ((uintptr_t)packed % 4 == 0);
  hipStream_t s = as_stream(stream);
  if (fast) {
    const int64_t chunks = rows * (K / 8);
    const int shift = __builtin_ctz((unsigned)tpg);
    with_dtype(dtype, [&](auto dt) {
      constexpr int DT = decltype(dt)::value;
      hipLaunchKernelGGL(pack_int4_kernel<DT>, dim3((unsigned)cdiv(chunks, 256 * PACK_U)),
                         dim3(256), 0, s, weights, chunks, shift,
                         reinterpret_cast<uint32_t*>(packed), scales);
    });
  } else {
    const int64_t threads = rows * (K / g);
    hipLaunchKernelGGL(pack_int4_serial_kernel, dim3((unsigned)cdiv(threads, 256)), dim3(256), 0,
                       s, weights, dtype, rows, (int)K, (int)g, packed, scales);
  }
  return check_launch(fn);
}

extern "C" int exq_quantize_int8(const void* weights, int dtype, int64_t rows, int64_t K,
                                 int8_t* q, uint16_t* scales, exq_stream stream) {
  const char* fn = "exq_quantize_int8";
  EXQ_REQUIRE(is_float_dtype(dtype), "%s: dtype must be f32, f16 or bf16", fn);
  EXQ_REQUIRE(rows >= 0 && rows <= INT32_MAX && K >= 1 && K <= INT32_MAX, "%s: bad sizes", fn);
  if (rows == 0) return EXQ_SUCCESS;
  EXQ_REQUIRE(weights && q && scales, "%s: null pointer", fn);
  hipStream_t s = as_stream(stream);
  if (K % 8 == 0 && K <= 16384 && (uintptr_t)weights % 16 == 0 && (uintptr_t)q % 8 == 0) {
    with_dtype(dtype, [&](auto dt) {
      constexpr int DT = decltype(dt)::value;
      const dim3 per4((unsigned)cdiv(rows, 4)), per1((unsigned)rows), b(256);
      if (K <= 1024)
        hipLaunchKernelGGL((quant_int8_rows_kernel<DT, 1, 2>), per4, b, 0, s, weights, rows,
                           (int)K, q, scales);
      else if (K <= 2048)
        hipLaunchKernelGGL((quant_int8_rows_kernel<DT, 1, 4>), per4, b, 0, s, weights, rows,
                           (int)K, q, scales);
      else if (K <= 4096)
        hipLaunchKernelGGL((quant_int8_rows_kernel<DT, 1, 8>), per4, b, 0, s, weights, rows,
                           (int)K, q, scales);
      else
        hipLaunchKernelGGL((quant_int8_rows_kernel<DT, 4, 8>), per1, b, 0, s, weights, rows,
                           (int)K, q, scales);
    });
  } else {
    hipLaunchKernelGGL(quant_int8_kernel, dim3((unsigned)rows), dim3(256), 0, s, weights, dtype,
                       (int)K, q, scales);
  }
  return check_launch(fn);
}
