// elementwise.hip -- row gather, deterministic combine, SiLU-and-mul, and the
// library's status plumbing.
#include <stdarg.h>
#include <stdio.h>

#include "exq_internal.h"

namespace exq {

namespace {
thread_local char g_last_error[512] = "";
}

int set_error(int status, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return status;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return set_error(EXQ_ERROR_HIP, "%s: launch failed: %s", what, hipGetErrorString(e));
  return EXQ_SUCCESS;
}

namespace {

// ---- gather ------------------------------------------------------------------
// One work-group per sorted row; 16-byte vector copies (row bytes % 16 == 0).
__global__ void __launch_bounds__(256) gather_rows_kernel(const uint4* __restrict__ hidden,
                                                          const int64_t* __restrict__ order,
                                                          uint4* __restrict__ out, int top_k,
                                                          int vec_per_row, int n_tokens) {
  const int i = blockIdx.x;
  const int64_t tok = order[i] / top_k;
  if (tok < 0 || tok >= n_tokens) return;
  const uint4* src = hidden + tok * vec_per_row;
  uint4* dst = out + (int64_t)i * vec_per_row;
  for (int v = threadIdx.x; v < vec_per_row; v += blockDim.x) dst[v] = src[v];
}

// ---- combine -----------------------------------------------------------------
__global__ void inverse_perm_kernel(const int64_t* __restrict__ order, int n,
                                    int32_t* __restrict__ inv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const int64_t s = order[i];
    if (s >= 0 && s < n) inv[s] = i;
  }
}

// VEC consecutive values of a float-typed array as fp32 (VEC = 8: one or two
// 16-byte accesses, element i a multiple of 8 from a 16-byte aligned base).
template <int DT, int VEC>
__device__ __forceinline__ void load_vec(const void* p, int64_t i, float (&v)[VEC]) {
  if constexpr (VEC == 1) {
    v[0] = load_as_f32(p, DT, i);
  } else if constexpr (DT == EXQ_DTYPE_F32) {
    const float4* q = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p) + i);
    const float4 a = q[0], b = q[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const uint4 q = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p) + i);
    const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[2 * j] = DT == EXQ_DTYPE_BF16 ? bf16_bits_to_f32(d[j] & 0xffffu)
                                      : f16_bits_to_f32(d[j] & 0xffffu);
      v[2 * j + 1] = DT == EXQ_DTYPE_BF16 ? __uint_as_float(d[j] & 0xffff0000u)
                                          : f16_bits_to_f32(d[j] >> 16);
    }
  }
}
template <int DT, int VEC>
__device__ __forceinline__ void store_vec(void* p, int64_t i, const float (&v)[VEC]) {
  if constexpr (VEC == 1) {
    store_from_f32(p, DT, i, v[0]);
  } else if constexpr (DT == EXQ_DTYPE_F32) {
    float4* q = reinterpret_cast<float4*>(reinterpret_cast<float*>(p) + i);
    q[0] = float4{v[0], v[1], v[2], v[3]};
    q[1] = float4{v[4], v[5], v[6], v[7]};
  } else {
    uint32_t d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      d[j] = DT == EXQ_DTYPE_BF16
                 ? f32_to_bf16_bits(v[2 * j]) | (f32_to_bf16_bits(v[2 * j + 1]) << 16)
                 : f32_to_f16_bits(v[2 * j]) | (f32_to_f16_bits(v[2 * j + 1]) << 16);
    *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p) + i) = uint4{d[0], d[1], d[2], d[3]};
  }
}

// result[t, h] = sum_j w[t, j] * down[inv[t*k + j], h], j ascending, fp32.
// Grid: tokens x column blocks; one thread per VEC consecutive columns (8 with
// H % 8 == 0 and 16-byte aligned rows, otherwise 1).  A token's positions and
// weights are scalar loads, and its rows go out SLOTS at a time.  Bound: bytes.
// unsort_output of 24,576 bf16 rows in 4,096 tokens, against one column and one row
// at a time: 2048 columns 82.3 -> 42.0 us, 2047 columns 82.6 -> 69.1 (93 with the
// threads laid out over all outputs, whose 64-bit division found the token).
template <int DT, int VEC, int SLOTS>
__global__ void __launch_bounds__(256) combine_kernel(const void* __restrict__ down,
                                                      const int32_t* __restrict__ inv,
                                                      const void* __restrict__ w, int wdtype,
                                                      int top_k, int H, int n_rows,
                                                      void* __restrict__ out) {
  const int64_t t = blockIdx.x;
  const int64_t h = ((int64_t)blockIdx.y * blockDim.x + threadIdx.x) * VEC;
  if (h >= H) return;
  const int64_t slot0 = t * top_k;
  float acc[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) acc[c] = 0.f;
  for (int j0 = 0; j0 < top_k; j0 += SLOTS) {
    int pos[SLOTS];
    float wt[SLOTS], v[SLOTS][VEC];
#pragma unroll
    for (int j = 0; j < SLOTS; ++j)  // slots past the last repeat it, with weight 0
      pos[j] = inv[slot0 + (j0 + j < top_k ? j0 + j : top_k - 1)];
    if (wdtype == EXQ_DTYPE_F32) {
      const float* wp = reinterpret_cast<const float*>(w) + slot0;
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) wt[j] = wp[j0 + j < top_k ? j0 + j : top_k - 1];
    } else {
      const uint16_t* wp = reinterpret_cast<const uint16_t*>(w) + slot0;
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        const uint32_t b = wp[j0 + j < top_k ? j0 + j : top_k - 1];
        wt[j] = wdtype == EXQ_DTYPE_BF16 ? bf16_bits_to_f32(b) : f16_bits_to_f32(b);
      }
    }
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      // (a position outside the rows: sort_order was not a permutation)
      const int row = (uint32_t)pos[j] < (uint32_t)n_rows ? pos[j] : 0;
      load_vec<DT, VEC>(down, (int64_t)row * H + h, v[j]);
    }
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      const bool use = j0 + j < top_k && (uint32_t)pos[j] < (uint32_t)n_rows;
      const float wj = use ? wt[j] : 0.f;
#pragma unroll
      for (int c = 0; c < VEC; ++c) acc[c] = fmaf(wj, use ? v[j][c] : 0.f, acc[c]);
    }
  }
  store_vec<DT, VEC>(out, t * H + h, acc);
}

// ---- SiLU-and-mul ------------------------------------------------------------
// One thread per VEC consecutive outputs of a row (8 with I % 8 == 0 and 16-byte
// aligned tensors, otherwise 1).  Bound: bytes; 2,648 x 1024 f16 outputs 9.8 ->
// 5.5 us against one output per thread.
template <int DT, int VEC>
__global__ void __launch_bounds__(256) silu_mul_kernel(const void* __restrict__ x, int64_t rows,
                                                       int64_t I, void* __restrict__ out) {
  const int64_t per = I / VEC, n = rows * per;
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < n; u += (int64_t)gridDim.x * 256) {
    const int64_t m = u / per, j = (u - m * per) * VEC;
    float g[VEC], up[VEC];
    load_vec<DT, VEC>(x, m * 2 * I + j, g);
    load_vec<DT, VEC>(x, m * 2 * I + I + j, up);
#pragma unroll
    for (int c = 0; c < VEC; ++c) g[c] = silu_f32(g[c]) * up[c];
    store_vec<DT, VEC>(out, m * I + j, g);
  }
}

}  // namespace
}  // namespace exq

using namespace exq;

namespace exq {
namespace {

// Streaming-read ceiling: every thread reads 16-byte pieces grid-strided, 8 in
// flight per iteration, and folds them into one word per work-group (so no
// load is dead).  The loads are nontemporal (`nt`): read once, the lines are
// not kept, which streams from HBM faster than the default policy (measured
// over 2 GiB: 6.3 against 5.7 TB/s).
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t fold_nt(const uint4* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return v.x ^ v.y ^ v.z ^ v.w;
}

__global__ void __launch_bounds__(256) stream_read_kernel(const uint4* __restrict__ buf,
                                                          int64_t n16,
                                                          uint32_t* __restrict__ sink) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  uint32_t acc = 0;
  for (; i + 7 * stride < n16; i += 8 * stride) {
    u32x4_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(buf + i + j * stride));
#pragma unroll
    for (int j = 0; j < 8; ++j) acc ^= v[j].x ^ v[j].y ^ v[j].z ^ v[j].w;
  }
  for (; i < n16; i += stride) acc ^= fold_nt(buf + i);
  for (int d = 1; d < 64; d <<= 1) acc ^= __shfl_xor(acc, d, 64);
  if ((threadIdx.x & 63) == 0) atomicXor(&sink[blockIdx.x], acc);
}

}  // namespace
}  // namespace exq

extern "C" int exq_stream_read(const void* buf, int64_t bytes, uint32_t* sink, int64_t sink_words,
                               exq_stream stream) {
  const char* fn = "exq_stream_read";
  EXQ_REQUIRE(bytes >= 0 && bytes % 16 == 0, "%s: bytes=%lld must be a multiple of 16", fn,
              (long long)bytes);
  EXQ_REQUIRE(sink_words >= 1, "%s: need a sink word per work-group", fn);
  if (bytes == 0) return EXQ_SUCCESS;
  EXQ_REQUIRE(buf && sink && (uintptr_t)buf % 16 == 0, "%s: null or misaligned pointer", fn);
  const int64_t grid = sink_words < 8192 ? sink_words : 8192;
  hipLaunchKernelGGL(exq::stream_read_kernel, dim3((unsigned)grid), dim3(256), 0,
                     exq::as_stream(stream), reinterpret_cast<const uint4*>(buf), bytes / 16,
                     sink);
  return exq::check_launch(fn);
}

extern "C" int exq_abi_version(void) { return EXQ_ABI_VERSION; }

extern "C" const char* exq_last_error(void) { return g_last_error; }

extern "C" const char* exq_status_name(int status) {
  switch (status) {
    case EXQ_SUCCESS: return "EXQ_SUCCESS";
    case EXQ_ERROR_INVALID_ARGUMENT: return "EXQ_ERROR_INVALID_ARGUMENT";
    case EXQ_ERROR_UNSUPPORTED: return "EXQ_ERROR_UNSUPPORTED";
    case EXQ_ERROR_WORKSPACE_TOO_SMALL: return "EXQ_ERROR_WORKSPACE_TOO_SMALL";
    case EXQ_ERROR_HIP: return "EXQ_ERROR_HIP";
    default: return "EXQ_ERROR_UNKNOWN";
  }
}

extern "C" int exq_gather_hidden(const void* hidden, int dtype, int64_t n_tokens,
                                 int64_t hidden_size, const int64_t* sort_order,
                                 int64_t n_active, int64_t top_k, void* out,
                                 exq_stream stream) {
  EXQ_REQUIRE(is_float_dtype(dtype), "exq_gather_hidden: dtype must be f32, f16 or bf16");
  EXQ_REQUIRE(top_k >= 1 && n_active >= 0 && n_active <= INT32_MAX && n_tokens >= 0,
              "exq_gather_hidden: bad sizes");
  const int64_t row_bytes = hidden_size * dtype_bytes(dtype);
  EXQ_REQUIRE(hidden_size > 0 && row_bytes % 16 == 0,
              "exq_gather_hidden: row bytes (%lld) must be a multiple of 16",
              (long long)row_bytes);
  if (n_active == 0) return EXQ_SUCCESS;
  EXQ_REQUIRE(hidden && sort_order && out, "exq_gather_hidden: null pointer");
  EXQ_REQUIRE(((uintptr_t)hidden | (uintptr_t)out) % 16 == 0,
              "exq_gather_hidden: hidden/out must be 16-byte aligned");
  const int vec = (int)(row_bytes / 16);
  hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)n_active), dim3(vec < 256 ? vec : 256),
                     0, as_stream(stream), reinterpret_cast<const uint4*>(hidden), sort_order,
                     reinterpret_cast<uint4*>(out), (int)top_k, vec, (int)n_tokens);
  return check_launch("gather_rows_kernel");
}

namespace exq {

// result[t] = sum_j w[t, j] * down[inv[t * k + j]] (combine_kernel).
static int launch_combine(const void* down_out, int dtype, const int32_t* inv, int64_t n_active,
                          const void* router_weights, int weights_dtype, int64_t n_tokens,
                          int64_t top_k, int64_t hidden_size, void* result, hipStream_t s) {
  const bool vec = hidden_size % 8 == 0 && ((uintptr_t)down_out | (uintptr_t)result) % 16 == 0;
  const int64_t cols = hidden_size / (vec ? 8 : 1), nby = cdiv(cols, 256);
  const dim3 grid((unsigned)n_tokens, (unsigned)nby), block((unsigned)(64 * cdiv(cols, 64 * nby)));
  auto launch = [&](auto dt, auto vc, auto slots) {
    hipLaunchKernelGGL(
        (combine_kernel<decltype(dt)::value, decltype(vc)::value, decltype(slots)::value>), grid,
        block, 0, s, down_out, inv, router_weights, weights_dtype, (int)top_k, (int)hidden_size,
        (int)n_active, result);
  };
  with_dtype(dtype, [&](auto dt) {
    auto with_slots = [&](auto vc) {  // rows in flight: few spare loads in the last batch
      if (top_k <= 2)
        launch(dt, vc, std::integral_constant<int, 2>{});
      else if (top_k <= 4 || cdiv(top_k, 4) % 2 == 1)
        launch(dt, vc, std::integral_constant<int, 4>{});
      else
        launch(dt, vc, std::integral_constant<int, 8>{});
    };
    if (vec)
      with_slots(std::integral_constant<int, 8>{});
    else
      with_slots(std::integral_constant<int, 1>{});
  });
  return check_launch("combine_kernel");
}

}  // namespace exq

extern "C" size_t exq_combine_workspace_size(int64_t n_active) {
  return align_up((size_t)(n_active > 0 ? n_active : 0) * sizeof(int32_t), 256);
}

extern "C" int exq_combine(const void* down_out, int dtype, const int64_t* sort_order,
                           int64_t n_active, const void* router_weights, int weights_dtype,
                           int64_t n_tokens, int64_t top_k, int64_t hidden_size, void* result,
                           void* workspace, size_t workspace_bytes, exq_stream stream) {
  EXQ_REQUIRE(is_float_dtype(dtype) && is_float_dtype(weights_dtype),
              "exq_combine: dtypes must be f32, f16 or bf16");
  EXQ_REQUIRE(top_k >= 1 && n_tokens >= 0 && n_active == n_tokens * top_k &&
                  n_active <= INT32_MAX && hidden_size > 0,
              "exq_combine: n_active (%lld) must equal n_tokens*top_k (%lld)",
              (long long)n_active, (long long)(n_tokens * top_k));
  EXQ_REQUIRE(cdiv(hidden_size, 256) <= 65535, "exq_combine: hidden_size=%lld too large",
              (long long)hidden_size);
  if (n_tokens == 0) return EXQ_SUCCESS;
  if (workspace_bytes < exq_combine_workspace_size(n_active))
    return set_error(EXQ_ERROR_WORKSPACE_TOO_SMALL, "exq_combine: workspace %zu < %zu bytes",
                     workspace_bytes, exq_combine_workspace_size(n_active));
  EXQ_REQUIRE(down_out && sort_order && router_weights && result && workspace,
              "exq_combine: null pointer");
  int32_t* inv = reinterpret_cast<int32_t*>(workspace);
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(inverse_perm_kernel, dim3((unsigned)cdiv(n_active, 256)), dim3(256), 0, s,
                     sort_order, (int)n_active, inv);
  int st = check_launch("inverse_perm_kernel");
  if (st) return st;
  return launch_combine(down_out, dtype, inv, n_active, router_weights, weights_dtype, n_tokens,
                        top_k, hidden_size, result, s);
}

namespace {
// Workspace of exq_unsort_combine: inverse positions, then (only when the sort
// does not fit one work-group) sort order, sorted ids and boundaries.
struct UnsortLayout {
  size_t order, ids, ends, total;
};
UnsortLayout unsort_layout(int64_t n, int64_t n_experts) {
  UnsortLayout L;
  const bool one = inverse_sort_fits(n, n_experts + 1);
  size_t off = align_up((size_t)(n > 0 ? n : 0) * 4, 256);
  L.order = off;  off += one ? 0 : align_up((size_t)n * 8, 256);
  L.ids = off;    off += one ? 0 : align_up((size_t)n * 8, 256);
  L.ends = off;   off += one ? 0 : align_up((size_t)(n_experts + 1) * 4, 256);
  L.total = off;
  return L;
}
}  // namespace

extern "C" size_t exq_unsort_combine_workspace_size(int64_t n_tokens, int64_t top_k,
                                                    int64_t n_experts) {
  return unsort_layout(n_tokens * top_k, n_experts).total;
}

extern "C" int exq_unsort_combine(const void* sorted_rows, int dtype, const void* router_indices,
                                  int ids_dtype, const void* router_weights, int weights_dtype,
                                  int64_t n_tokens, int64_t top_k, int64_t n_experts,
                                  int64_t hidden_size, void* result, void* workspace,
                                  size_t workspace_bytes, exq_stream stream) {
  const char* fn = "exq_unsort_combine";
  EXQ_REQUIRE(is_float_dtype(dtype) && is_float_dtype(weights_dtype),
              "%s: dtypes must be f32, f16 or bf16", fn);
  EXQ_REQUIRE(is_index_dtype(ids_dtype), "%s: ids must be i32 or i64", fn);
  EXQ_REQUIRE(top_k >= 1 && n_tokens >= 0 && n_tokens * top_k <= INT32_MAX && hidden_size > 0 &&
                  n_experts >= 1 && n_experts < 4096,
              "%s: bad sizes", fn);
  EXQ_REQUIRE(cdiv(hidden_size, 256) <= 65535, "%s: hidden_size=%lld too large", fn,
              (long long)hidden_size);
  if (n_tokens == 0) return EXQ_SUCCESS;
  const int64_t n = n_tokens * top_k;
  const UnsortLayout L = unsort_layout(n, n_experts);
  if (workspace_bytes < L.total)
    return set_error(EXQ_ERROR_WORKSPACE_TOO_SMALL, "%s: workspace %zu < %zu bytes", fn,
                     workspace_bytes, L.total);
  EXQ_REQUIRE(sorted_rows && router_indices && router_weights && result && workspace,
              "%s: null pointer", fn);
  hipStream_t s = as_stream(stream);
  unsigned char* ws = reinterpret_cast<unsigned char*>(workspace);
  int32_t* inv = reinterpret_cast<int32_t*>(ws);
  int st;
  if (inverse_sort_fits(n, n_experts + 1)) {
    st = launch_inverse_sort(router_indices, ids_dtype, (int)n, (int)n_experts, inv, s);
  } else {
    int64_t* order = reinterpret_cast<int64_t*>(ws + L.order);
    st = exq_dispatch(router_indices, ids_dtype, n, n_experts, order,
                      reinterpret_cast<int64_t*>(ws + L.ids),
                      reinterpret_cast<int32_t*>(ws + L.ends), stream);
    if (st) return st;
    hipLaunchKernelGGL(inverse_perm_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, s, order,
                       (int)n, inv);
    st = check_launch("inverse_perm_kernel");
  }
  if (st) return st;
  return launch_combine(sorted_rows, dtype, inv, n, router_weights, weights_dtype, n_tokens,
                        top_k, hidden_size, result, s);
}

extern "C" int exq_silu_and_mul(const void* input, int dtype, int64_t rows, int64_t inter,
                                void* out, exq_stream stream) {
  EXQ_REQUIRE(is_float_dtype(dtype), "exq_silu_and_mul: dtype must be f32, f16 or bf16");
  EXQ_REQUIRE(rows >= 0 && inter >= 1, "exq_silu_and_mul: bad sizes");
  if (rows == 0) return EXQ_SUCCESS;
  EXQ_REQUIRE(input && out, "exq_silu_and_mul: null pointer");
  const bool vec = inter % 8 == 0 && ((uintptr_t)input | (uintptr_t)out) % 16 == 0;
  int64_t blocks = cdiv(rows * (inter / (vec ? 8 : 1)), 256);
  if (blocks > 65536) blocks = 65536;
  with_dtype(dtype, [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    if (vec)
      hipLaunchKernelGGL((silu_mul_kernel<DT, 8>), dim3((unsigned)blocks), dim3(256), 0,
                         as_stream(stream), input, rows, inter, out);
    else
      hipLaunchKernelGGL((silu_mul_kernel<DT, 1>), dim3((unsigned)blocks), dim3(256), 0,
                         as_stream(stream), input, rows, inter, out);
  });
  return check_launch("silu_mul_kernel");
}
