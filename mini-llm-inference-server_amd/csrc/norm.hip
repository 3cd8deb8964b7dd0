// The decoder layer's row-wise kernels around its matrix products (reference src/minillm/model/llama.py:37-55,
// 117-127: RMSNorm, the residual sums and SwiGLU), 16-bit activations with fp32 arithmetic.
//
// Bound by memory: each element is read once and written once, 16 bytes per thread and access.  As elementwise
// launches a norm took eight (cast, square, mean, + eps, rsqrt, scale, cast, weight; the mean alone 8.2 us), the
// residual sum one, SwiGLU two.  One kernel each: a Llama-3.1-8B layer on 8 decode rows 298 -> 244 us, on three
// prompts (768 tokens) 502.5 -> 412.0 us.
#include "common.h"

namespace mllm {
namespace {

template <typename T>
__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]);
template <>
__device__ __forceinline__ void unpack8<BF16>(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(v[i] << 16);
    f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
  }
}
template <>
__device__ __forceinline__ void unpack8<F16>(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = f16_bits_to_f32((uint16_t)v[i]);
    f[2 * i + 1] = f16_bits_to_f32((uint16_t)(v[i] >> 16));
  }
}
template <typename T>
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
  return u32x4{pack2<T>(f[0], f[1]), pack2<T>(f[2], f[3]), pack2<T>(f[4], f[5]), pack2<T>(f[6], f[7])};
}

// One workgroup per row: out = w * T(x * rsqrt(mean(x^2) + eps)), the cast before the weight as the module states
// it.  With ADD, x is first replaced by T(x + y), which is also written to `sum`.  A row of up to kKeep x 2,048
// elements stays in registers between the two passes, a longer one is read again (with ADD, from `sum`: each thread
// reads what it wrote).  With SPLIT, y is the fp32 sum of the row's `ksplit` partial sums (mllm_linear_partial).
constexpr int kNormThreads = 256;
constexpr int kKeep = 4;  // 16-byte pieces per thread kept in registers

// Adds piece i (8 columns) of the parts to f, in their order.
__device__ __forceinline__ void add_parts(const float* part, int ksplit, int64_t stride, int64_t at, float (&f)[8]) {
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll 8
  for (int k = 0; k < ksplit; ++k) {
    lo += *reinterpret_cast<const f32x4*>(part + k * stride + at);
    hi += *reinterpret_cast<const f32x4*>(part + k * stride + at + 4);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[e] += lo[e];
    f[4 + e] += hi[e];
  }
}

template <typename T, bool ADD, bool SPLIT = false>
__global__ __launch_bounds__(kNormThreads) void rms_norm_kernel(const uint16_t* __restrict__ x,
                                                                const uint16_t* __restrict__ y,
                                                                const uint16_t* __restrict__ w, uint16_t* sum,
                                                                uint16_t* __restrict__ out, int64_t dim, float eps,
                                                                const float* __restrict__ part = nullptr,
                                                                int ksplit = 0, int64_t part_stride = 0) {
  __shared__ float red[kNormThreads / 64];
  const int64_t row = (int64_t)blockIdx.x * dim;
  const int pieces = (int)(dim / 8);
  u32x4 keep[kKeep];
  float ss = 0.f;
  auto first_pass = [&](int i) {
    u32x4 v = ld16(x + row + 8 * (int64_t)i);
    float f[8];
    unpack8<T>(v, f);
    if constexpr (ADD) {
      if constexpr (SPLIT) {
        add_parts(part, ksplit, part_stride, row + 8 * (int64_t)i, f);
      } else {
        float g[8];
        unpack8<T>(ld16(y + row + 8 * (int64_t)i), g);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] += g[e];
      }
      v = pack8<T>(f);
      st16(sum + row + 8 * (int64_t)i, v);
      unpack8<T>(v, f);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
    return v;
  };
#pragma unroll
  for (int u = 0; u < kKeep; ++u) {
    const int i = u * kNormThreads + (int)threadIdx.x;
    if (i < pieces) keep[u] = first_pass(i);
  }
  for (int i = kKeep * kNormThreads + (int)threadIdx.x; i < pieces; i += kNormThreads) first_pass(i);
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float r = rsqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)dim + eps);
  auto second_pass = [&](int i, u32x4 v) {
    float f[8], g[8];
    unpack8<T>(v, f);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] *= r;
    unpack8<T>(pack8<T>(f), f);
    unpack8<T>(ld16(w + 8 * (int64_t)i), g);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] *= g[e];
    st16(out + row + 8 * (int64_t)i, pack8<T>(f));
  };
#pragma unroll
  for (int u = 0; u < kKeep; ++u) {
    const int i = u * kNormThreads + (int)threadIdx.x;
    if (i < pieces) second_pass(i, keep[u]);
  }
  for (int i = kKeep * kNormThreads + (int)threadIdx.x; i < pieces; i += kNormThreads)
    second_pass(i, ld16((ADD ? sum : x) + row + 8 * (int64_t)i));
}

// out = T(silu(gate) * up) over n elements (a multiple of 8), silu(g) = g / (1 + exp(-g)) in fp32.
template <typename T>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gate,
                                                       const uint16_t* __restrict__ up, uint16_t* __restrict__ out,
                                                       int64_t pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  float g[8], u[8];
  unpack8<T>(ld16(gate + 8 * i), g);
  unpack8<T>(ld16(up + 8 * i), u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = g[e] / (1.f + expf(-g[e])) * u[e];
  st16(out + 8 * i, pack8<T>(g));
}

// out = T(residual + the sum of the parts) over n elements (a multiple of 8); no residual: the sum alone.
template <typename T>
__global__ __launch_bounds__(256) void sum_partials_kernel(const float* __restrict__ part, int ksplit, int64_t n,
                                                           const uint16_t* __restrict__ residual,
                                                           uint16_t* __restrict__ out) {
  const int64_t i = 8 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (residual) unpack8<T>(ld16(residual + i), f);
  add_parts(part, ksplit, n, i, f);
  st16(out + i, pack8<T>(f));
}

// cos and sin rows of the rotary embedding: out[t][d] = T(cos(float(pos[t]) * inv_freq[d % half])), one thread per
// frequency and both of its places.  Bound by the launch: as seven elementwise launches a step's rows took 25 us.
template <typename T>
__global__ __launch_bounds__(256) void rope_table_kernel(const int64_t* __restrict__ pos, int64_t n,
                                                         const float* __restrict__ inv_freq, int half,
                                                         uint16_t* __restrict__ cos_out,
                                                         uint16_t* __restrict__ sin_out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n * half) return;
  const int64_t t = i / half;
  const int d = (int)(i - t * half);
  const float ang = (float)pos[t] * inv_freq[d];
  const uint16_t c = cvt1<T>(cosf(ang)), s = cvt1<T>(sinf(ang));
  const int64_t o = 2 * t * half + d;
  cos_out[o] = cos_out[o + half] = c;
  sin_out[o] = sin_out[o + half] = s;
}

}  // namespace
}  // namespace mllm

extern "C" int mllm_rms_norm(const void* x, const void* residual, const void* weight, int64_t rows, int64_t dim,
                             float eps, int32_t dtype, void* sum, void* out, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(dtype == MLLM_DTYPE_BF16 || dtype == MLLM_DTYPE_F16, MLLM_ERR_UNSUPPORTED,
               "mllm_rms_norm: dtype must be bfloat16 or float16");
  MLLM_REQUIRE(rows >= 0 && dim > 0 && dim % 8 == 0 && dim < (1ll << 31), MLLM_ERR_INVALID,
               "mllm_rms_norm: need rows >= 0 and a positive dim, a multiple of 8");
  MLLM_REQUIRE(rows <= kMaxGroups256, MLLM_ERR_UNSUPPORTED, "mllm_rms_norm: fewer than 2^24 rows");
  MLLM_REQUIRE(!residual == !sum, MLLM_ERR_INVALID, "mllm_rms_norm: residual and sum go together");
  if (rows == 0) return MLLM_OK;
  MLLM_REQUIRE(x && weight && out, MLLM_ERR_INVALID, "mllm_rms_norm: null pointer");
  MLLM_REQUIRE(((uintptr_t)x | (uintptr_t)residual | (uintptr_t)weight | (uintptr_t)sum | (uintptr_t)out) % 16 == 0,
               MLLM_ERR_UNSUPPORTED, "mllm_rms_norm: rows must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto tag) {
    using T = decltype(tag);
    const auto xp = (const uint16_t*)x, yp = (const uint16_t*)residual, wp = (const uint16_t*)weight;
    if (residual)
      rms_norm_kernel<T, true><<<(unsigned)rows, kNormThreads, 0, st>>>(xp, yp, wp, (uint16_t*)sum, (uint16_t*)out, dim, eps);
    else
      rms_norm_kernel<T, false><<<(unsigned)rows, kNormThreads, 0, st>>>(xp, yp, wp, nullptr, (uint16_t*)out, dim, eps);
  };
  if (dtype == MLLM_DTYPE_BF16)
    launch(BF16{});
  else
    launch(F16{});
  return check_launch("mllm_rms_norm");
}

extern "C" int mllm_silu_mul(const void* gate, const void* up, int64_t n, int32_t dtype, void* out, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(dtype == MLLM_DTYPE_BF16 || dtype == MLLM_DTYPE_F16, MLLM_ERR_UNSUPPORTED,
               "mllm_silu_mul: dtype must be bfloat16 or float16");
  MLLM_REQUIRE(n >= 0 && n % 8 == 0, MLLM_ERR_INVALID, "mllm_silu_mul: n must be a multiple of 8");
  MLLM_REQUIRE(n <= kMaxGroups256 * 2048, MLLM_ERR_UNSUPPORTED, "mllm_silu_mul: too many elements");
  if (n == 0) return MLLM_OK;
  MLLM_REQUIRE(gate && up && out, MLLM_ERR_INVALID, "mllm_silu_mul: null pointer");
  MLLM_REQUIRE(((uintptr_t)gate | (uintptr_t)up | (uintptr_t)out) % 16 == 0, MLLM_ERR_UNSUPPORTED,
               "mllm_silu_mul: operands must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)((n / 8 + 255) / 256);
  if (dtype == MLLM_DTYPE_BF16)
    silu_mul_kernel<BF16><<<grid, 256, 0, st>>>((const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)out, n / 8);
  else
    silu_mul_kernel<F16><<<grid, 256, 0, st>>>((const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)out, n / 8);
  return check_launch("mllm_silu_mul");
}

extern "C" int mllm_sum_partials(const float* part, int32_t ksplit, int64_t rows, int64_t dim, const void* residual,
                                 int32_t dtype, void* out, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(dtype == MLLM_DTYPE_BF16 || dtype == MLLM_DTYPE_F16, MLLM_ERR_UNSUPPORTED,
               "mllm_sum_partials: dtype must be bfloat16 or float16");
  MLLM_REQUIRE(ksplit >= 1 && rows >= 0 && dim > 0 && dim % 8 == 0 && rows < (1ll << 31) && dim < (1ll << 31),
               MLLM_ERR_INVALID, "mllm_sum_partials: bad sizes");
  if (rows == 0) return MLLM_OK;
  MLLM_REQUIRE(part && out, MLLM_ERR_INVALID, "mllm_sum_partials: null pointer");
  MLLM_REQUIRE(((uintptr_t)part | (uintptr_t)residual | (uintptr_t)out) % 16 == 0, MLLM_ERR_UNSUPPORTED,
               "mllm_sum_partials: operands must be 16-byte aligned");
  const int64_t n = rows * dim, groups = (n / 8 + 255) / 256;
  MLLM_REQUIRE(groups <= kMaxGroups256, MLLM_ERR_UNSUPPORTED, "mllm_sum_partials: too many elements");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == MLLM_DTYPE_BF16)
    sum_partials_kernel<BF16><<<(unsigned)groups, 256, 0, st>>>(part, ksplit, n, (const uint16_t*)residual, (uint16_t*)out);
  else
    sum_partials_kernel<F16><<<(unsigned)groups, 256, 0, st>>>(part, ksplit, n, (const uint16_t*)residual, (uint16_t*)out);
  return check_launch("mllm_sum_partials");
}

extern "C" int mllm_sum_partials_norm(const float* part, int32_t ksplit, const void* residual, const void* weight,
                                      int64_t rows, int64_t dim, float eps, int32_t dtype, void* sum, void* out,
                                      void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(dtype == MLLM_DTYPE_BF16 || dtype == MLLM_DTYPE_F16, MLLM_ERR_UNSUPPORTED,
               "mllm_sum_partials_norm: dtype must be bfloat16 or float16");
  MLLM_REQUIRE(ksplit >= 1 && rows >= 0 && dim > 0 && dim % 8 == 0 && dim < (1ll << 31), MLLM_ERR_INVALID,
               "mllm_sum_partials_norm: bad sizes");
  MLLM_REQUIRE(rows <= kMaxGroups256, MLLM_ERR_UNSUPPORTED, "mllm_sum_partials_norm: fewer than 2^24 rows");
  if (rows == 0) return MLLM_OK;
  MLLM_REQUIRE(part && residual && weight && sum && out, MLLM_ERR_INVALID, "mllm_sum_partials_norm: null pointer");
  MLLM_REQUIRE(((uintptr_t)part | (uintptr_t)residual | (uintptr_t)weight | (uintptr_t)sum | (uintptr_t)out) % 16 == 0,
               MLLM_ERR_UNSUPPORTED, "mllm_sum_partials_norm: rows must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto tag) {
    rms_norm_kernel<decltype(tag), true, true><<<(unsigned)rows, kNormThreads, 0, st>>>(
        (const uint16_t*)residual, nullptr, (const uint16_t*)weight, (uint16_t*)sum, (uint16_t*)out, dim, eps, part,
        ksplit, rows * dim);
  };
  if (dtype == MLLM_DTYPE_BF16)
    launch(BF16{});
  else
    launch(F16{});
  return check_launch("mllm_sum_partials_norm");
}

extern "C" int mllm_rope_table(const int64_t* positions, int64_t n, const float* inv_freq, int32_t half, int32_t dtype,
                               void* cos, void* sin, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(dtype == MLLM_DTYPE_BF16 || dtype == MLLM_DTYPE_F16, MLLM_ERR_UNSUPPORTED,
               "mllm_rope_table: dtype must be bfloat16 or float16");
  MLLM_REQUIRE(n >= 0 && half > 0 && n < (1ll << 31), MLLM_ERR_INVALID, "mllm_rope_table: bad sizes");
  if (n == 0) return MLLM_OK;
  MLLM_REQUIRE(positions && inv_freq && cos && sin, MLLM_ERR_INVALID, "mllm_rope_table: null pointer");
  const int64_t groups = (n * half + 255) / 256;
  MLLM_REQUIRE(groups <= kMaxGroups256, MLLM_ERR_UNSUPPORTED, "mllm_rope_table: too many positions");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == MLLM_DTYPE_BF16)
    rope_table_kernel<BF16><<<(unsigned)groups, 256, 0, st>>>(positions, n, inv_freq, half, (uint16_t*)cos, (uint16_t*)sin);
  else
    rope_table_kernel<F16><<<(unsigned)groups, 256, 0, st>>>(positions, n, inv_freq, half, (uint16_t*)cos, (uint16_t*)sin);
  return check_launch("mllm_rope_table");
}
