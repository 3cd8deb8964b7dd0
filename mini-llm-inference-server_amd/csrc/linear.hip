// Linear layers of few rows (a decode step's tokens): y[M, N] = x[M, K] . w[N, K]^T, 16-bit operands, fp32 sums,
// M <= 64 (reference src/minillm/model/llama.py:75-120: the q, k, v, o, gate, up and down projections).
//
// Bound by the weights, 2 N K bytes read once.  A workgroup of eight wavefronts takes 128 weight rows, 16 per
// wavefront, over a range of K, in chunks of 256: each wavefront loads its rows' part of the next chunk from HBM into
// registers (8 KB in flight) while it multiplies the one at hand with v_mfma_f32_16x16x32 (lane (n, g) holds weight
// row n at k = 32 u + 8 g .. +7).  x goes through LDS, shared by the wavefronts, two chunks ahead: loaded into
// registers by each wavefront instead, its lines passed through the same in-order load queue as the weights' and the
// time grew with M (o projection of Llama-3.1-8B, 8 / 32 / 64 rows: 10.1 / 14.3 / 21.7 us against 9.4 / 10.5 / 12.2).
// mllm_linear_partial gives each output tile to several workgroups, one per part of K, so that few output rows
// still fill the chip (o: 32 tiles x 8 parts; without parts 32.6 us); their fp32 sums are added, in order, by the
// kernel that reads them (mllm_sum_partials, or the norm behind the o projection).  mllm_linear_swiglu has the
// output rows to do without: 64 gate and 64 up rows per workgroup, T(silu(gate) * up) written at once.
// Measured (Llama-3.1-8B, bf16, 8 / 32 / 64 rows, us; in brackets the library product, for q, k, v three of them):
//   q k v  13.7 / 14.9 / 17.0 (44.6 / 36.5 / 44.1)    gate, up  43.4 / 44.3 / 48.4 (55.7 / 50.2 / 53.5)
//   o       9.4 / 10.5 / 12.2 (15.8 / 13.2 / 15.2)    down      23.7 / 24.7 / 27.4 (25.0 / 29.5 / 38.8)
// gate and up stream 5.4 TB/s.  Tiles of 64 rows with two wavefronts along K measured 13.1, 9.2, 49.0 and 23.6 us at
// 8 rows.  A row's result depends neither on the other rows nor on M.
#include <initializer_list>

#include "common.h"

namespace mllm {
namespace {

constexpr int kWaves = 8;
constexpr int kSteps = 8;             // k-steps of 32 per chunk
constexpr int kChunk = 32 * kSteps;   // K per chunk
constexpr int kTileRows = 16 * kWaves;
constexpr int kMaxRows = 64;          // of x

struct LinearArgs {
  const uint16_t* x;
  int M, K;
  const uint16_t* w[3];  // up to three weights share x; SwiGLU: gate, up
  int n[3];              // their rows
  int tile0[3];          // first tile of each
  int ksplit, ncols;     // partial sums: parts of K, columns (all weights' rows)
  float* part;           // [ksplit][M][ncols]
  uint16_t* y;           // SwiGLU: [M][n[0]]
};

template <typename T, int MT, bool SWIGLU>
__global__ __launch_bounds__(64 * kWaves) void linear_kernel(const LinearArgs a) {
  constexpr int kRow = 2 * kChunk, kBuf = 16 * MT * kRow, kPart = kWaves * MT * 64 * 16;
  __shared__ __attribute__((aligned(1024))) char lds[3 * kBuf > kPart ? 3 * kBuf : kPart];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ks = blockIdx.x % a.ksplit, tile = blockIdx.x / a.ksplit;  // the parts of one tile side by side
  const int p = SWIGLU ? 0 : (tile >= a.tile0[2] ? 2 : (tile >= a.tile0[1] ? 1 : 0));
  constexpr int kCols = SWIGLU ? kTileRows / 2 : kTileRows;  // output columns of the workgroup
  const int n0 = kCols * (tile - a.tile0[p]), rows = a.n[p];
  const int blk = SWIGLU ? wave % (kWaves / 2) : wave;  // SwiGLU: wavefronts 0 .. 3 gate, 4 .. 7 up
  // a row past the end loads the last one and is not stored
  const uint16_t* wp = a.w[SWIGLU ? wave / (kWaves / 2) : p] + (int64_t)min(n0 + 16 * blk + n, rows - 1) * a.K + 8 * g;

  // this workgroup's chunks of K, begun at another place by each tile so that the launch does not walk the memory
  // channels in step
  const int all = a.K / kChunk, first = all * ks / a.ksplit, chunks = all * (ks + 1) / a.ksplit - first;
  const int skew = tile % chunks;
  auto chunk = [&](int i) { return first + (i + skew < chunks ? i + skew : i + skew - chunks); };

  // x chunk in LDS: rows of 512 bytes, 16-byte piece j of row m at j ^ (m % 16).  Rows past M are not loaded: what
  // they hold reaches only outputs that are not stored.
  const int dmas = (a.M * kRow + 1023) / 1024;
  const char* xb = reinterpret_cast<const char*>(a.x);
  auto load_x = [&](int c) {
    const unsigned dst = lds_offset(lds + c % 3 * kBuf);
    const char* base = xb + (int64_t)chunk(c) * kRow;
    for (int i = wave; i < dmas; i += kWaves) {
      const int byte = 1024 * i + 16 * lane, m = byte / kRow, j = byte % kRow / 16;
      dma16(base, (unsigned)min(m, a.M - 1) * (unsigned)(2 * a.K) + 16u * (j ^ (m & 15)), dst + 1024 * i);
    }
  };
  u32x4 wa[kSteps], wb[kSteps];
  auto load_w = [&](u32x4 (&w)[kSteps], int c) {
#pragma unroll
    for (int u = 0; u < kSteps; ++u) w[u] = ld16(wp + (int64_t)chunk(c) * kChunk + 32 * u);
  };
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const u32x4 (&w)[kSteps], int c) {
    const char* b = lds + c % 3 * kBuf + n * kRow;
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = Mfma<T>::m16x16x32(w[u], ld16(b + 16 * m * kRow + 16 * ((4 * u + g) ^ n)), acc[m]);
  };
  // step c: x(c + 2), into the slot of x(c - 1), and w(c + 1) go out, chunk c is multiplied; the barrier that ends
  // the step leaves at most w(c + 1) in flight, so every wavefront's part of x(c + 1) has landed
  auto step = [&](const u32x4 (&w)[kSteps], u32x4 (&next)[kSteps], int c) {
    if (c + 2 < chunks) load_x(c + 2);
    load_w(next, c + 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(w, c);
    barrier_vm<kSteps>();
  };

  load_x(0);
  load_w(wa, 0);
  if (chunks > 1) load_x(1);
  barrier_vm<0>();
  int c = 0;
  for (; c + 2 < chunks; c += 2) {
    step(wa, wb, c);
    step(wb, wa, c + 1);
  }
  if (chunks - c == 2) {
    step(wa, wb, c);
    multiply(wb, c + 1);
  } else {
    multiply(wa, c);
  }

  if constexpr (!SWIGLU) {  // lane (n, g): row 16 m + n of x, columns n0 + 16 wave + 4 g .. + 3
    int col = n0 + 16 * wave + 4 * g;
    if (col >= rows) return;
    for (int i = 0; i < p; ++i) col += a.n[i];
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (16 * m + n < a.M)
        *reinterpret_cast<f32x4*>(a.part + ((int64_t)ks * a.M + 16 * m + n) * a.ncols + col) = acc[m];
  } else {
    barrier_vm<0>();  // every wavefront has read its last x
    f32x4* up = reinterpret_cast<f32x4*>(lds);  // [block][MT][64], from the wavefronts of up
    if (wave >= kWaves / 2) {
#pragma unroll
      for (int m = 0; m < MT; ++m) up[(blk * MT + m) * 64 + lane] = acc[m];
    }
    __syncthreads();
    const int col = n0 + 16 * blk + 4 * g;
    if (wave >= kWaves / 2 || col >= rows) return;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (16 * m + n >= a.M) continue;
      const f32x4 u = up[(blk * MT + m) * 64 + lane];
      float s[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = acc[m][e] / (1.f + expf(-acc[m][e])) * u[e];
      st8(a.y + (int64_t)(16 * m + n) * rows + col, u32x2{pack2<T>(s[0], s[1]), pack2<T>(s[2], s[3])});
    }
  }
}

template <typename T, bool SWIGLU>
int launch(const LinearArgs& a, int tiles, hipStream_t st) {
  const unsigned grid = (unsigned)tiles * (unsigned)a.ksplit;
  if (a.M <= 16)
    linear_kernel<T, 1, SWIGLU><<<grid, 64 * kWaves, 0, st>>>(a);
  else if (a.M <= 32)
    linear_kernel<T, 2, SWIGLU><<<grid, 64 * kWaves, 0, st>>>(a);
  else if (a.M <= 48)
    linear_kernel<T, 3, SWIGLU><<<grid, 64 * kWaves, 0, st>>>(a);
  else
    linear_kernel<T, 4, SWIGLU><<<grid, 64 * kWaves, 0, st>>>(a);
  return check_launch(SWIGLU ? "mllm_linear_swiglu" : "mllm_linear_partial");
}

int check_operands(const char* fn, const void* x, int64_t m, int64_t k, int32_t dtype) {
  MLLM_REQUIRE(dtype == MLLM_DTYPE_BF16 || dtype == MLLM_DTYPE_F16, MLLM_ERR_UNSUPPORTED,
               std::string(fn) + ": dtype must be bfloat16 or float16");
  MLLM_REQUIRE(m >= 0 && m <= kMaxRows, MLLM_ERR_UNSUPPORTED, std::string(fn) + ": at most 64 rows");
  MLLM_REQUIRE(k > 0 && k % kChunk == 0 && k < (1 << 24), MLLM_ERR_UNSUPPORTED,
               std::string(fn) + ": k must be a multiple of 256");
  MLLM_REQUIRE(m == 0 || x, MLLM_ERR_INVALID, std::string(fn) + ": null pointer");
  return MLLM_OK;
}

}  // namespace
}  // namespace mllm

// Parts of K per output tile: as many as give every CU about one workgroup, so that the launch is one round (256 CUs: o of
// Llama-3.1-8B 9.4 us at 8 parts against 12.5 at 4; q, k and v 13.7 at 5 against 14.3 at 4), at most 8 (each part's sums
// are written and read again) and none shorter than two chunks.
extern "C" int mllm_linear_ksplit(int64_t k, int64_t n0, int64_t n1, int64_t n2, int32_t num_cus) {
  using namespace mllm;
  int64_t tiles = 0;
  for (const int64_t n : {n0, n1, n2}) tiles += (n + kTileRows - 1) / kTileRows;
  int64_t ks = tiles > 0 ? (num_cus > 0 ? num_cus : device_cus()) / tiles : 1;
  if (ks > 8) ks = 8;
  if (ks > k / kChunk / 2) ks = k / kChunk / 2;
  return ks < 1 ? 1 : (int)ks;
}

extern "C" int mllm_linear_partial(const void* x, int64_t m, int64_t k, const void* w0, int64_t n0, const void* w1,
                                   int64_t n1, const void* w2, int64_t n2, int32_t ksplit, float* part, int32_t dtype,
                                   void* stream) {
  using namespace mllm;
  const int rc = check_operands("mllm_linear_partial", x, m, k, dtype);
  if (rc != MLLM_OK) return rc;
  MLLM_REQUIRE(ksplit >= 1 && ksplit <= k / kChunk, MLLM_ERR_INVALID,
               "mllm_linear_partial: ksplit must be in [1, k / 256]");
  const void* w[3] = {w0, w1, w2};
  const int64_t n[3] = {n0, n1, n2};
  LinearArgs a{};
  uintptr_t ptrs = (uintptr_t)x | (uintptr_t)part;
  int64_t tiles = 0, cols = 0;
  for (int i = 0; i < 3; ++i) {
    MLLM_REQUIRE(n[i] >= 0 && n[i] % 16 == 0 && n[i] < (1 << 28) && (i > 0 || n[i] > 0), MLLM_ERR_UNSUPPORTED,
                 "mllm_linear_partial: the weights' rows must be multiples of 16");
    MLLM_REQUIRE(n[i] == 0 || w[i], MLLM_ERR_INVALID, "mllm_linear_partial: null pointer");
    a.w[i] = (const uint16_t*)w[i];
    a.n[i] = (int)n[i];
    a.tile0[i] = n[i] ? (int)tiles : 0x7fffffff;
    ptrs |= (uintptr_t)w[i];
    tiles += (n[i] + kTileRows - 1) / kTileRows;
    cols += n[i];
  }
  MLLM_REQUIRE(n1 > 0 || n2 == 0, MLLM_ERR_INVALID, "mllm_linear_partial: weights are given from the first on");
  MLLM_REQUIRE(tiles * ksplit <= kMaxGroups256 / 2 && cols < (1ll << 31), MLLM_ERR_UNSUPPORTED,
               "mllm_linear_partial: too many tiles");
  if (m == 0) return MLLM_OK;
  MLLM_REQUIRE(part, MLLM_ERR_INVALID, "mllm_linear_partial: null pointer");
  MLLM_REQUIRE(ptrs % 16 == 0, MLLM_ERR_UNSUPPORTED, "mllm_linear_partial: operands must be 16-byte aligned");
  a.x = (const uint16_t*)x;
  a.M = (int)m;
  a.K = (int)k;
  a.ksplit = ksplit;
  a.ncols = (int)cols;
  a.part = part;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return dtype == MLLM_DTYPE_BF16 ? launch<BF16, false>(a, (int)tiles, st) : launch<F16, false>(a, (int)tiles, st);
}

extern "C" int mllm_linear_swiglu(const void* x, int64_t m, int64_t k, const void* gate, const void* up, int64_t n,
                                  int32_t dtype, void* out, void* stream) {
  using namespace mllm;
  const int rc = check_operands("mllm_linear_swiglu", x, m, k, dtype);
  if (rc != MLLM_OK) return rc;
  MLLM_REQUIRE(n > 0 && n % 16 == 0 && n < (1 << 28), MLLM_ERR_UNSUPPORTED,
               "mllm_linear_swiglu: the weights' rows must be a multiple of 16");
  if (m == 0) return MLLM_OK;
  MLLM_REQUIRE(gate && up && out, MLLM_ERR_INVALID, "mllm_linear_swiglu: null pointer");
  MLLM_REQUIRE(((uintptr_t)x | (uintptr_t)gate | (uintptr_t)up | (uintptr_t)out) % 16 == 0, MLLM_ERR_UNSUPPORTED,
               "mllm_linear_swiglu: operands must be 16-byte aligned");
  LinearArgs a{};
  a.x = (const uint16_t*)x;
  a.M = (int)m;
  a.K = (int)k;
  a.w[0] = (const uint16_t*)gate;
  a.w[1] = (const uint16_t*)up;
  a.n[0] = (int)n;
  a.tile0[1] = a.tile0[2] = 0x7fffffff;
  a.ksplit = 1;
  a.y = (uint16_t*)out;
  const int tiles = (int)((n + kTileRows / 2 - 1) / (kTileRows / 2));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return dtype == MLLM_DTYPE_BF16 ? launch<BF16, true>(a, tiles, st) : launch<F16, true>(a, tiles, st);
}
