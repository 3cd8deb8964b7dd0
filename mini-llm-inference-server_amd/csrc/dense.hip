// Contiguous (non-paged) causal attention: the backend's `prefill` method
// (reference src/minillm/attention/torch_ref.py:20-44, base.py:19-33).
//
// q [B, H, Tq, Dh], k/v [B, Hkv, Tk, Dh] with arbitrary element strides; query i sits at position
// Tk - Tq + i and sees keys 0 .. Tk - Tq + i; with key_valid [B, Tk] it sees only real keys among them,
// and a query that has none sees its own position.  Four kernels:
//   dense_mfma_kernel   bf16 / fp16, Dh 64 or 128, 16-byte aligned rows: workgroups of 128 query rows whose
//                       four wavefronts share each 64-key K/V tile through LDS (many rows);
//   dense_split_kernel  the same operands: workgroups of 32 query rows whose four wavefronts share the keys
//                       out among them and merge their partial results in LDS (few rows);
//   dense_f32_kernel    fp32, Dh 64 or 128, 16-byte aligned rows, on the fp32 MFMA instructions;
//   dense_kernel        everything else (any Dh up to 256, any strides), one workgroup per query row, fp32 scalar
//                       arithmetic.
// Scores and the running max and sum are fp32 everywhere.  The 16-bit MFMA kernels give the PV product the fp32
// probabilities as a sum of 16-bit operands, each the rounding error of those before it: three in bf16 (8 bits each:
// the fp32 value), two in fp16 (22 bits: the fp32 value to one unit of its last place).
#include <math.h>

#include "common.h"

namespace mllm {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxDh = 256;

struct DenseArgs {
  const char* q;
  const char* k;
  const char* v;
  const uint8_t* key_valid;
  char* out;
  int64_t q_sb, q_sh, q_st;
  int64_t k_sb, k_sh, k_st;
  int64_t v_sb, v_sh, v_st;
  int64_t o_sb, o_sh, o_st;
  int64_t kv_sb, kv_st;
  int B, H, Hkv, Tq, Tk, Dh;
  int G;  // query heads of one KV head that share a workgroup (MFMA kernels)
  float scale;
};

template <int DT>
__device__ __forceinline__ float ld_elem(const char* base, int64_t idx) {
  if constexpr (DT == MLLM_DTYPE_F32)
    return reinterpret_cast<const float*>(base)[idx];
  else if constexpr (DT == MLLM_DTYPE_BF16)
    return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(base)[idx]);
  else
    return f16_bits_to_f32(reinterpret_cast<const uint16_t*>(base)[idx]);
}

template <int DT>
__device__ __forceinline__ void st_elem(char* base, int64_t idx, float f) {
  if constexpr (DT == MLLM_DTYPE_F32)
    reinterpret_cast<float*>(base)[idx] = f;
  else if constexpr (DT == MLLM_DTYPE_BF16)
    reinterpret_cast<uint16_t*>(base)[idx] = f32_to_bf16_bits(f);
  else
    reinterpret_cast<uint16_t*>(base)[idx] = f32_to_f16_bits(f);
}

__device__ __forceinline__ float block_max(float v, float* red) {
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  float r = red[0];
  for (int i = 1; i < kThreads / 64; ++i) r = fmaxf(r, red[i]);
  return r;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < kThreads / 64; ++i) r += red[i];
  return r;
}

template <int DT>
__global__ __launch_bounds__(kThreads) void dense_kernel(const DenseArgs a) {
  __shared__ float qs[kMaxDh];
  __shared__ float ps[kThreads];
  __shared__ float red[kThreads / 64];
  const int i = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x;
  const int kvh = h / (a.H / a.Hkv);
  const int qpos = a.Tk - a.Tq + i;
  const char* kb = a.k;
  const int64_t k_row0 = (int64_t)b * a.k_sb + (int64_t)kvh * a.k_sh;
  const int64_t v_row0 = (int64_t)b * a.v_sb + (int64_t)kvh * a.v_sh;
  const int64_t q_row = (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)i * a.q_st;
  for (int d = tid; d < a.Dh; d += kThreads) qs[d] = ld_elem<DT>(a.q, q_row + d);

  // a query with no real key among 0 .. qpos sees only its own position
  bool own_only = false;
  if (a.key_valid) {
    int any = 0;
    for (int j = tid; j <= qpos; j += kThreads) any |= a.key_valid[(int64_t)b * a.kv_sb + (int64_t)j * a.kv_st] != 0;
    own_only = block_sum((float)any, red) == 0.f;
  }
  __syncthreads();

  float m_run = -INFINITY, l_run = 0.f, acc = 0.f;
  for (int j0 = 0; j0 <= qpos; j0 += kThreads) {
    const int j = j0 + tid;
    float s = -INFINITY;
    bool allowed = j <= qpos;
    if (allowed && a.key_valid)
      allowed = own_only ? (j == qpos) : (a.key_valid[(int64_t)b * a.kv_sb + (int64_t)j * a.kv_st] != 0);
    if (allowed) {
      float dot = 0.f;
      const int64_t kr = k_row0 + (int64_t)j * a.k_st;
      for (int d = 0; d < a.Dh; ++d) dot += qs[d] * ld_elem<DT>(kb, kr + d);
      s = dot * a.scale;
    }
    const float cm = block_max(s, red);
    const float m_new = fmaxf(m_run, cm);
    const float p = (s == -INFINITY) ? 0.f : expf(s - m_new);
    ps[tid] = p;
    const float cs = block_sum(p, red);
    const float alpha = (m_run == -INFINITY) ? 0.f : expf(m_run - m_new);
    l_run = l_run * alpha + cs;
    m_run = m_new;
    if (tid < a.Dh) {
      float part = 0.f;
      const int jn = min(kThreads, qpos + 1 - j0);
      for (int jj = 0; jj < jn; ++jj) {
        const float pj = ps[jj];
        if (pj != 0.f) part += pj * ld_elem<DT>(a.v, v_row0 + (int64_t)(j0 + jj) * a.v_st + tid);
      }
      acc = acc * alpha + part;
    }
    __syncthreads();
  }
  if (tid < a.Dh)
    st_elem<DT>(a.out, (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)i * a.o_st + tid, acc / l_run);
}


// ---------------------------------------------------------------- bf16 / fp16 on the matrix cores
// Per wavefront: 32 query rows (row = token * G + head of the G query heads that share the KV head), keys in
// tiles of 32 NB:
//   S^T[keys x 32 rows] = K . Q^T     v_mfma_f32_32x32x16 (K rows by ds_read_b128; Q^T in VGPRs)
//   O^T[Dh x 32 rows]  += V^T . P^T   v_mfma_f32_32x32x16, once with each part of P
//                                     (V^T by ds_read_b64_tr_b16, the LDS transpose read)
// S^T and P^T share a lane layout (lane l: row l % 32), so P never leaves its lanes.  Tiles reach LDS by direct
// global->LDS loads, one 2 Dh-byte key row after the other, the 16-byte chunks of row r XOR-swizzled so that
// the operand reads hit distinct banks: Dh 128: K chunk ^ (r % 16), V chunk ^ 4 (r % 4); Dh 64 (two rows per
// 256 bytes of banks): K chunk ^ (r / 2 % 8), V chunk ^ 4 (r / 2 % 2).  Keys past a workgroup's last visible key
// are loaded as copies of that key's row and masked.
// Bound by the MFMA streams (with P in three parts four products' worth per tile, in two three) and, for few rows, by a
// tile's latency chain.  Against one workgroup per row on the vector ALU, bf16, 32 query and 8 KV heads, Dh 128: one
// sequence of 512 tokens 637.6 -> 11.5 us a call, four left-padded of 777 3,776 -> 49.0 us, the same distance from
// float64 (1.6e-3 and 4.8e-4 relative: the output's rounding).  P as two bf16 parts took 11.3 and 44.1 us, but left the
// weights 16 bits: sums that cancel were off by 6e-7 of the values where fp32 weights leave 1e-7.  Kernel alone, two
// parts / three: four of 777 without padding 40.8 / 48.0 us, four of 1,100 69.3 / 82.5 us; fp16, where only the scale of P
// and the earlier rescaling are new, 44.4 / 46.2 us.
// A masked key has P = 0, and 0 x V is 0 only while V is finite; the sums of values near the largest may overflow where
// a weight of at most 1 would not (P is larger by up to 2^kSlack).  Rows whose result is not finite are therefore computed
// again key by key (row_by_key), which skips the keys of zero weight and has no weight above 1.

template <int DH>
struct Geo {
  static constexpr int kRow = 2 * DH;           // bytes of one key row in LDS
  static constexpr int kChunks = DH / 8;        // 16-byte chunks per row
  static constexpr int kRowsPerDma = 64 / kChunks;
  static constexpr int kSteps = DH / 16;        // 16-dim steps of the score product
  static constexpr int kDt = DH / 32;           // 32-dim output tiles
  static __device__ __forceinline__ int k_swz(int r) { return DH == 128 ? (r & 15) : ((r >> 1) & 7); }
  static __device__ __forceinline__ int v_swz(int r) { return DH == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); }
  // byte offset of this lane's first K operand in a tile (row lane % 32, dims step 0); step kk flips bits 5-7
  // (^ 32 kk) and 32 rows further adds 32 kRow
  static __device__ __forceinline__ unsigned k_read(int lane) {
    const int n = lane & 31, h = lane >> 5, s = k_swz(n);
    return (unsigned)(n * kRow + 16 * (h ^ (s & 1)) + 16 * (s & 14));
  }
  // byte offset of its first V^T read (keys 4h .. 4h + 3, dims tile 0); tile dt flips bits 6-7 (^ 64 dt), the
  // keys 8 further add 8 kRow and 16-key group u adds 16 u kRow
  static __device__ __forceinline__ unsigned v_read(int lane) {
    const int h = lane >> 5, r = 4 * h + ((lane >> 2) & 3);
    return (unsigned)(r * kRow + 16 * v_swz(r) + 32 * ((lane >> 4) & 1) + 8 * (lane & 3));
  }
};

// Which keys of batch row b are real, as the wavefront holds it: bit j of lane i's word is key
// 64 (base + i) + j.  `first` is the first real key (kNoKey if there is none in the windows up to the limit).
constexpr int kNoKey = 0x7fffffff;
struct KeyMask {
  uint32_t lo = ~0u, hi = ~0u;
  int base = 0, first = 0;
};
// Bit i: byte i of w is not 0.
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t w) {
  const uint32_t t = ((((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) >> 7) & 0x01010101u;
  return (t * 0x01020408u) >> 24;
}
// Words base .. base + 63 (keys past the row are not real).  Contiguous masks: a lane reads the 64 bytes of its
// word at once (16-byte loads at any address), the row's last, partial word is read a byte per lane.
__device__ __forceinline__ void load_window(const DenseArgs& a, int b, int base, int lane, KeyMask& km) {
  const uint8_t* kv = a.key_valid + (int64_t)b * a.kv_sb;
  km.base = base;
  km.lo = km.hi = 0;
  if (a.kv_st == 1) {
    const int full = a.Tk / 64, word = base + lane;
    if (word < full) {
      u32x4 x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) __builtin_memcpy(&x[i], kv + (int64_t)64 * word + 16 * i, 16);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t m = nonzero_bytes(x[i][e]) << (16 * (i & 1) + 4 * e);
          if (i < 2)
            km.lo |= m;
          else
            km.hi |= m;
        }
    }
    if (full >= base && full < base + 64 && 64 * full < a.Tk) {
      const int j = 64 * full + lane;
      const uint64_t m = __ballot(j < a.Tk && kv[min(j, a.Tk - 1)] != 0);
      if (word == full) {
        km.lo = (uint32_t)m;
        km.hi = (uint32_t)(m >> 32);
      }
    }
    return;
  }
  for (int i = 0; i < 64 && 64 * (base + i) < a.Tk; ++i) {
    const int j = 64 * (base + i) + lane;
    const uint64_t m = __ballot(j < a.Tk && kv[(int64_t)min(j, a.Tk - 1) * a.kv_st] != 0);
    if (lane == i) {
      km.lo = (uint32_t)m;
      km.hi = (uint32_t)(m >> 32);
    }
  }
}
__device__ __forceinline__ uint64_t mask_word(const KeyMask& km, int tile64) {
  const int i = tile64 - km.base;
  return (uint64_t)(uint32_t)__builtin_amdgcn_readlane(km.lo, i) |
         ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(km.hi, i) << 32);
}
// The first real key below `limit`, and the mask window that holds it (window 0 if there is none).
__device__ __forceinline__ void find_first(const DenseArgs& a, int b, int limit, int lane, KeyMask& km) {
  km.first = kNoKey;
  for (int base = 0; 64 * base < limit; base += 64) {
    load_window(a, b, base, lane, km);
    const uint64_t any = __ballot((km.lo | km.hi) != 0);
    if (any) {
      const int i = __builtin_ctzll(any);
      km.first = 64 * (base + i) + __builtin_ctzll(mask_word(km, base + i));
      return;
    }
  }
}

// One query row by one wavefront, key by key in fp32: dense_kernel's arithmetic (keys of zero weight skipped).
template <int DT>
__device__ __forceinline__ void row_by_key(const DenseArgs& a, int b, int h, int i, int first, int lane) {
  const int kvh = h / (a.H / a.Hkv);
  const int qpos = a.Tk - a.Tq + i;
  const bool own_only = a.key_valid && first > qpos;
  const int64_t k_row0 = (int64_t)b * a.k_sb + (int64_t)kvh * a.k_sh;
  const int64_t v_row0 = (int64_t)b * a.v_sb + (int64_t)kvh * a.v_sh;
  const int64_t q_row = (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)i * a.q_st;
  float m_run = -INFINITY, l_run = 0.f, acc[kMaxDh / 64] = {};
  for (int j0 = 0; j0 <= qpos; j0 += 64) {
    const int j = j0 + lane;
    bool allowed = j <= qpos;
    if (allowed && a.key_valid)
      allowed = own_only ? (j == qpos) : (a.key_valid[(int64_t)b * a.kv_sb + (int64_t)j * a.kv_st] != 0);
    float s = -INFINITY;
    if (allowed) {
      float dot = 0.f;
      const int64_t kr = k_row0 + (int64_t)j * a.k_st;
      for (int d = 0; d < a.Dh; ++d) dot += ld_elem<DT>(a.q, q_row + d) * ld_elem<DT>(a.k, kr + d);
      s = dot * a.scale;
    }
    float cm = s;
    for (int off = 32; off > 0; off >>= 1) cm = fmaxf(cm, __shfl_xor(cm, off, 64));
    const float m_new = fmaxf(m_run, cm);
    const float p = (s == -INFINITY) ? 0.f : expf(s - m_new);
    float cs = p;
    for (int off = 32; off > 0; off >>= 1) cs += __shfl_xor(cs, off, 64);
    const float alpha = (m_run == -INFINITY) ? 0.f : expf(m_run - m_new);
    l_run = l_run * alpha + cs;
    m_run = m_new;
#pragma unroll
    for (int e = 0; e < kMaxDh / 64; ++e) acc[e] *= alpha;
    for (int jj = 0; jj < min(64, qpos + 1 - j0); ++jj) {
      const float pj = __shfl(p, jj, 64);
      if (pj == 0.f) continue;
#pragma unroll
      for (int e = 0; e < kMaxDh / 64; ++e)
        if (64 * e + lane < a.Dh) acc[e] += pj * ld_elem<DT>(a.v, v_row0 + (int64_t)(j0 + jj) * a.v_st + 64 * e + lane);
    }
  }
  const int64_t o = (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)i * a.o_st;
#pragma unroll
  for (int e = 0; e < kMaxDh / 64; ++e)
    if (64 * e + lane < a.Dh) st_elem<DT>(a.out, o + 64 * e + lane, acc[e] / l_run);
}

// The float value of the low / high half of a packed pair; P's 16-bit parts, the power of 2 it is kept larger by, and by
// how many powers a row's max may grow before its sums are rescaled.
template <typename T>
struct Half;
template <>
struct Half<BF16> {
  static constexpr int kDt = MLLM_DTYPE_BF16;
  static constexpr int kParts = 3;
  static constexpr float kBias = 0.f, kSlack = 8.f;
  static __device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};
template <>
struct Half<F16> {
  static constexpr int kDt = MLLM_DTYPE_F16;
  static constexpr int kParts = 2;
  // The parts end at fp16's smallest step, 2^-24, so P fills the range up to 65,504 (at most 2^15.9): the step is then
  // 2^-39 of the row's largest weight or less, and a weight 2^-24 of it still has 15 bits.  2^6 larger with a slack of
  // 8 left that weight 6 bits.
  static constexpr float kBias = 15.f, kSlack = 0.9f;
  static __device__ __forceinline__ float lo(uint32_t w) { return f16_bits_to_f32((uint16_t)w); }
  static __device__ __forceinline__ float hi(uint32_t w) { return f16_bits_to_f32((uint16_t)(w >> 16)); }
};

// A wavefront's state over its 32 rows.
template <int DH>
struct RowState {
  f32x16 o[Geo<DH>::kDt];
  float m = -INFINITY, l = 0.f;
};

// S^T of one tile at LDS byte `kb` (this lane's k_read offset within it).
template <typename T, int DH, int NB>
__device__ __forceinline__ void score_tile(const char* lds, unsigned kb, const u32x4 (&qf)[Geo<DH>::kSteps],
                                           f32x16 (&s)[NB]) {
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
#pragma unroll
  for (int kk = 0; kk < Geo<DH>::kSteps; ++kk) {
    const char* p = lds + (kb ^ (32u * kk));
#pragma unroll
    for (int b = 0; b < NB; ++b) s[b] = Mfma<T>::m32x32x16(ld16(p + b * 32 * Geo<DH>::kRow), qf[kk], s[b]);
  }
}

// Online softmax (exp2 domain) of one tile's scores (keys kv0 .. kv0 + 32 NB - 1): masks, moves the running max
// when some row's grew by more than 2^kSlack, and leaves P's 16-bit parts in pp.  vm: the tile's real keys
// (all ones without a mask); rows without a real key (qp < first) keep only their own position.  A row may meet
// whole masked tiles before its first key (m = -inf): its P and sum then stay 0.
template <typename T, int DH, int NB, bool MASKED>
__device__ __forceinline__ void softmax_tile(f32x16 (&s)[NB], u32x4 (&pp)[Half<T>::kParts][NB][2], RowState<DH>& st,
                                             int kv0, int qp, int wave_qp_lo, int first, uint64_t vm, int h, float c) {
  constexpr uint64_t kAll = NB == 2 ? ~0ull : 0xffffffffull;
  if (MASKED && vm != kAll) {
    const uint64_t vh = vm >> (4 * h);
    const bool own = qp < first;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t w = (uint32_t)(vh >> (32 * b));
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k0 = 8 * (r >> 2) + (r & 3);
        const int key = kv0 + 32 * b + k0 + 4 * h;
        const bool see = own ? key == qp : (((w >> k0) & 1u) != 0 && key <= qp);
        s[b][r] = see ? s[b][r] : -INFINITY;
      }
    }
  } else if (kv0 + 32 * NB - 1 > wave_qp_lo) {  // some key of the tile lies past the wavefront's first row
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kv0 + 32 * b + 8 * (r >> 2) + 4 * h + (r & 3);
        s[b][r] = key > qp ? -INFINITY : s[b][r];
      }
  }
  float m4[4] = {s[0][0], s[0][1], s[0][2], s[0][3]};
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (b > 0 || r >= 4) m4[r & 3] = __builtin_fmaxf(m4[r & 3], s[b][r]);
  const float mx = max_xor32(__builtin_fmaxf(__builtin_fmaxf(m4[0], m4[1]), __builtin_fmaxf(m4[2], m4[3])));
  if (__any((mx - st.m) * c > Half<T>::kSlack)) {
    const float m_new = fmaxf(st.m, mx);
    const float alpha = m_new == st.m ? 1.f : fast_exp2((st.m - m_new) * c);  // -inf - -inf is no rescale
    st.l *= alpha;
#pragma unroll
    for (int dt = 0; dt < Geo<DH>::kDt; ++dt) st.o[dt] *= alpha;
    st.m = m_new;
  }
  const float mc = st.m == -INFINITY ? 0.f : st.m * c - Half<T>::kBias;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[b][r] = fast_exp2(__builtin_fmaf(s[b][r], c, -mc));
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float p0 = s[b][8 * u + 2 * e], p1 = s[b][8 * u + 2 * e + 1];
#pragma unroll
        for (int i = 0; i < Half<T>::kParts; ++i) {
          const uint32_t w = pack2<T>(p0, p1);
          pp[i][b][u][e] = w;
          p0 -= Half<T>::lo(w);
          p1 -= Half<T>::hi(w);
        }
      }
  float s4[4] = {s[0][0], s[0][1], s[0][2], s[0][3]};
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (b > 0 || r >= 4) s4[r & 3] += s[b][r];
  st.l += sum_xor32((s4[0] + s4[1]) + (s4[2] + s4[3]));
}

// O^T += V^T P^T for one tile at LDS byte `vb` (this lane's v_read offset within it).
template <typename T, int DH, int NB>
__device__ __forceinline__ void pv_tile(const char* lds, unsigned vb, const u32x4 (&pp)[Half<T>::kParts][NB][2],
                                        RowState<DH>& st) {
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int dt = 0; dt < Geo<DH>::kDt; ++dt) {
        const char* p = lds + (vb ^ (64u * dt)) + 16 * (2 * b + u) * Geo<DH>::kRow;
        const u32x2 lo = ld_tr(p), hi = ld_tr(p + 8 * Geo<DH>::kRow);
        const u32x4 vt = u32x4{lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int i = 0; i < Half<T>::kParts; ++i) st.o[dt] = Mfma<T>::m32x32x16(vt, pp[i][b][u], st.o[dt]);
      }
    }
}

// Q^T operand: this lane's row at dims 16 kk + 8 h .. +7.
template <int DH>
__device__ __forceinline__ void load_q(const DenseArgs& a, int b, int head, int tok, bool valid, int h,
                                       u32x4 (&qf)[Geo<DH>::kSteps]) {
  const uint16_t* q = reinterpret_cast<const uint16_t*>(a.q) + (int64_t)b * a.q_sb + (int64_t)head * a.q_sh +
                      (int64_t)(valid ? tok : 0) * a.q_st;
#pragma unroll
  for (int kk = 0; kk < Geo<DH>::kSteps; ++kk) {
    const u32x4 v = ld16(q + 16 * kk + 8 * h);
    qf[kk] = valid ? v : u32x4{0, 0, 0, 0};
  }
}

__device__ __forceinline__ bool not_finite(float x) { return !(__builtin_fabsf(x) < INFINITY); }
// Bit n: row n (of the wavefront's 32) has a value that is not finite among this lane pair's.
template <int N>
__device__ __forceinline__ uint32_t bad_rows_of(const f32x16 (&o)[N]) {
  bool bad = false;
#pragma unroll
  for (int dt = 0; dt < N; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) bad |= not_finite(o[dt][r]);
  const uint64_t m = __ballot(bad);
  return (uint32_t)m | (uint32_t)(m >> 32);
}

// The workgroup's (query tile, batch, KV head): the KV head varies fastest (with 8 of them, each XCD serves one
// and keeps its K and V in its L2), the last query tiles (the longest contexts) come first.
struct Item {
  int t0, b, kvh;
};
__device__ __forceinline__ Item item_of(const DenseArgs& a, int tokens) {
  int x = blockIdx.x;
  const int nkv = a.H / a.G;
  Item it;
  it.kvh = x % nkv;
  x /= nkv;
  it.b = x % a.B;
  it.t0 = ((a.Tq + tokens - 1) / tokens - 1 - x / a.B) * tokens;
  return it;
}

// 128 query rows per workgroup, 32 per wavefront; 64-key tiles through a K ring of three and a V ring of two
// (Dh 128: 80 KB, two workgroups per CU: one's softmax and prologue run beside the other's MFMAs).  Step j: S(j)
// is at hand; V(j+1) and K(j+3) are issued into the slots of V(j-1) and K(j), both last read in step j-1; PV(j)
// and S(j+1) run at raised priority, then the softmax of tile j+1; the barrier ending the step waits for every load
// but K(j+3).
template <typename T, int DH, bool MASKED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void dense_mfma_kernel(const DenseArgs a) {
  using G = Geo<DH>;
  constexpr int kBN = 64, kTile = kBN * G::kRow, kVBase = 3 * kTile, kDma = 16 / G::kRowsPerDma;
  __shared__ __attribute__((aligned(1024))) char lds[5 * kTile];
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tokens = 128 / a.G, tpw = 32 / a.G;
  const Item it = item_of(a, tokens);
  const int off = a.Tk - a.Tq;  // position of query 0
  const int tok = it.t0 + wave * tpw + n / a.G;
  const bool row_valid = tok < a.Tq;
  const int head = it.kvh * a.G + n % a.G;
  const int qp = row_valid ? off + tok : a.Tk - 1;
  const int wave_t0 = it.t0 + wave * tpw;
  const int wave_qp_lo = off + wave_t0;
  const int wave_qp_hi = wave_t0 < a.Tq ? off + min(wave_t0 + tpw, a.Tq) - 1 : -1;
  const int kv_end = off + min(it.t0 + tokens, a.Tq), last = kv_end - 1;
  const int ntiles = (kv_end + kBN - 1) / kBN;
  const float c = a.scale * kLog2e;

  KeyMask km;
  int ts = 0;  // the first tile with a key some row sees
  if constexpr (MASKED) {
    find_first(a, it.b, kv_end, lane, km);
    ts = min(km.first, off + it.t0) / kBN;
    if (ts / 64 * 64 != km.base) load_window(a, it.b, ts / 64 * 64, lane, km);
  }
  auto key_word = [&](int t) -> uint64_t {
    if constexpr (!MASKED) return ~0ull;
    if (t - km.base >= 64) load_window(a, it.b, t, lane, km);
    return mask_word(km, t);
  };

  const int kvh = it.kvh * a.G / (a.H / a.Hkv);
  const char* kc = a.k + 2 * ((int64_t)it.b * a.k_sb + (int64_t)kvh * a.k_sh);
  const char* vc = a.v + 2 * ((int64_t)it.b * a.v_sb + (int64_t)kvh * a.v_sh);
  const unsigned k_stb = (unsigned)(2 * a.k_st), v_stb = (unsigned)(2 * a.v_st);
  const int lr = lane / G::kChunks, lc = lane % G::kChunks;
  unsigned koff[kDma], voff[kDma];  // this lane's offsets from a full tile's first row
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = 16 * wave + G::kRowsPerDma * i + lr;
    koff[i] = (unsigned)r * k_stb + 16u * (lc ^ G::k_swz(r));
    voff[i] = (unsigned)r * v_stb + 16u * (lc ^ G::v_swz(r));
  }
  // this wavefront's share (rows 16 wave .. + 15) of tile t, kDma loads of kRowsPerDma rows
  auto dma = [&](const char* p, unsigned stb, const unsigned (&offs)[kDma], int t, char* slot) {
    const int kv0 = t * kBN;
    const unsigned dst = lds_offset(slot) + 16 * wave * G::kRow;
    const char* base = p + (int64_t)kv0 * stb;
    if (kv0 + kBN <= kv_end) {
#pragma unroll
      for (int i = 0; i < kDma; ++i) dma16(base, offs[i], dst + 1024 * i);
    } else {  // the last tile: keys past `last` load the row of `last` (masked)
#pragma unroll
      for (int i = 0; i < kDma; ++i) {
        const int r = 16 * wave + G::kRowsPerDma * i + lr;
        dma16(base, offs[i] - (unsigned)max(kv0 + r - last, 0) * stb, dst + 1024 * i);
      }
    }
  };
  auto k_slot = [&](int t) { return lds + (t - ts) % 3 * kTile; };
  auto v_slot = [&](int t) { return lds + kVBase + (t - ts) % 2 * kTile; };
  const unsigned kread = G::k_read(lane), vread = kVBase + G::v_read(lane);

  RowState<DH> st;
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.o[dt][r] = 0.f;

  dma(kc, k_stb, koff, ts, k_slot(ts));
  dma(vc, v_stb, voff, ts, v_slot(ts));
  if (ts + 1 < ntiles) dma(kc, k_stb, koff, ts + 1, k_slot(ts + 1));
  if (ts + 2 < ntiles) dma(kc, k_stb, koff, ts + 2, k_slot(ts + 2));
  u32x4 qf[G::kSteps];
  load_q<DH>(a, it.b, head, tok, row_valid, h, qf);
#pragma unroll
  for (int kk = 0; kk < G::kSteps; ++kk) asm volatile("" ::"v"(qf[kk]) : "memory");
  barrier_vm<0>();

  f32x16 s[2];
  u32x4 pp[Half<T>::kParts][2][2];
  if (ts * kBN <= wave_qp_hi) {
    score_tile<T, DH, 2>(lds, kread, qf, s);
    softmax_tile<T, DH, 2, MASKED>(s, pp, st, ts * kBN, qp, wave_qp_lo, km.first, key_word(ts), h, c);
  }
  barrier_lds();  // K(ts) has been read

  for (int j = ts; j < ntiles; ++j) {
    const bool k_ahead = j + 3 < ntiles;
    if (j + 1 < ntiles) dma(vc, v_stb, voff, j + 1, v_slot(j + 1));
    if (k_ahead) dma(kc, k_stb, koff, j + 3, k_slot(j + 3));
    const bool do_pv = j * kBN <= wave_qp_hi, do_s = j + 1 < ntiles && (j + 1) * kBN <= wave_qp_hi;
    const unsigned vb = vread + (j - ts) % 2 * kTile, kb = kread + (j + 1 - ts) % 3 * kTile;
    __builtin_amdgcn_s_setprio(1);
    if (do_pv) pv_tile<T, DH, 2>(lds, vb, pp, st);
    if (do_s) score_tile<T, DH, 2>(lds, kb, qf, s);
    __builtin_amdgcn_s_setprio(0);
    if (do_s)
      softmax_tile<T, DH, 2, MASKED>(s, pp, st, (j + 1) * kBN, qp, wave_qp_lo, km.first, key_word(j + 1), h, c);
    if (k_ahead)
      barrier_vm<kDma>();
    else
      barrier_vm<0>();
  }

  // each wavefront's 32 x Dh block transposed through its own part of the K ring, then whole 16-byte chunks
  const float inv = 1.f / st.l;
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt) st.o[dt] *= inv;
  uint32_t bad = bad_rows_of<G::kDt>(st.o);
  char* ost = lds + wave * (32 * G::kRow);
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int r = 4 * g4;
      const u32x2 pk = u32x2{pack2<T>(st.o[dt][r], st.o[dt][r + 1]), pack2<T>(st.o[dt][r + 2], st.o[dt][r + 3])};
      *reinterpret_cast<u32x2*>(ost + n * G::kRow + 16 * ((4 * dt + g4) ^ (n & (G::kChunks - 1))) + 8 * h) = pk;
    }
#pragma unroll
  for (int i = 0; i < 32 / G::kRowsPerDma; ++i) {
    const int row = G::kRowsPerDma * i + lr;
    const u32x4 v = *reinterpret_cast<const u32x4*>(ost + row * G::kRow + 16 * (lc ^ (row & (G::kChunks - 1))));
    const int rtok = wave_t0 + row / a.G;
    if (rtok < a.Tq && !((bad >> row) & 1u)) {
      uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + (int64_t)it.b * a.o_sb +
                    (int64_t)(it.kvh * a.G + row % a.G) * a.o_sh + (int64_t)rtok * a.o_st;
      st16(o + 8 * lc, v);
    }
  }
  while (bad) {
    const int row = __builtin_ctz(bad);
    bad &= bad - 1;
    const int rtok = wave_t0 + row / a.G;
    if (rtok < a.Tq) row_by_key<Half<T>::kDt>(a, it.b, it.kvh * a.G + row % a.G, rtok, km.first, lane);
  }
}

// 32 query rows per workgroup; wavefront w takes the 32-key tiles w, w + 4, .. through 32 KV rows of LDS of its own
// (Dh 128: 64 KB, two workgroups per CU), so the loop has no workgroup barrier: K(t+4) is issued when S(t) has
// read K(t), V(t+4) when PV(t) has read V(t).  At the end the four partial (m, l, O) of each row are merged in LDS,
// wavefront w for the 32-dim output tile w.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <typename T, int DH, bool MASKED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void dense_split_kernel(const DenseArgs a) {
  using G = Geo<DH>;
  constexpr int kBN = 32, kTile = kBN * G::kRow, kDma = kBN / G::kRowsPerDma;
  __shared__ __attribute__((aligned(1024))) char lds[8 * kTile];
  __shared__ float2 ml[4][32];
  __shared__ uint32_t bad_rows;
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tokens = 32 / a.G;
  const Item it = item_of(a, tokens);
  const int off = a.Tk - a.Tq;
  const int tok = it.t0 + n / a.G;
  const bool row_valid = tok < a.Tq;
  const int head = it.kvh * a.G + n % a.G;
  const int qp = row_valid ? off + tok : a.Tk - 1;
  const int qp_lo = off + it.t0;
  const int kv_end = off + min(it.t0 + tokens, a.Tq), last = kv_end - 1;
  const int ntiles = (kv_end + kBN - 1) / kBN;
  const float c = a.scale * kLog2e;
  if (threadIdx.x == 0) bad_rows = 0;

  KeyMask km;
  int ts = 0;
  if constexpr (MASKED) {
    find_first(a, it.b, kv_end, lane, km);
    ts = min(km.first, qp_lo) / kBN;
    if (ts / 2 / 64 * 64 != km.base) load_window(a, it.b, ts / 2 / 64 * 64, lane, km);
  }
  auto key_word = [&](int t) -> uint64_t {
    if constexpr (!MASKED) return 0xffffffffull;
    if (t / 2 - km.base >= 64) load_window(a, it.b, t / 2, lane, km);
    return (mask_word(km, t / 2) >> (32 * (t & 1))) & 0xffffffffull;
  };

  const int kvh = it.kvh * a.G / (a.H / a.Hkv);
  const char* kc = a.k + 2 * ((int64_t)it.b * a.k_sb + (int64_t)kvh * a.k_sh);
  const char* vc = a.v + 2 * ((int64_t)it.b * a.v_sb + (int64_t)kvh * a.v_sh);
  const unsigned k_stb = (unsigned)(2 * a.k_st), v_stb = (unsigned)(2 * a.v_st);
  const int lr = lane / G::kChunks, lc = lane % G::kChunks;
  char* kbuf = lds + 2 * wave * kTile;
  char* vbuf = kbuf + kTile;
  unsigned koff[kDma], voff[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = G::kRowsPerDma * i + lr;
    koff[i] = (unsigned)r * k_stb + 16u * (lc ^ G::k_swz(r));
    voff[i] = (unsigned)r * v_stb + 16u * (lc ^ G::v_swz(r));
  }
  auto dma = [&](const char* p, unsigned stb, const unsigned (&offs)[kDma], int t, char* slot) {
    const int kv0 = t * kBN;
    const unsigned dst = lds_offset(slot);
    const char* base = p + (int64_t)kv0 * stb;
    if (kv0 + kBN <= kv_end) {
#pragma unroll
      for (int i = 0; i < kDma; ++i) dma16(base, offs[i], dst + 1024 * i);
    } else {
#pragma unroll
      for (int i = 0; i < kDma; ++i)
        dma16(base, offs[i] - (unsigned)max(kv0 + G::kRowsPerDma * i + lr - last, 0) * stb, dst + 1024 * i);
    }
  };

  RowState<DH> st;
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.o[dt][r] = 0.f;

  u32x4 qf[G::kSteps];
  load_q<DH>(a, it.b, head, tok, row_valid, h, qf);
  int t = ts + wave;
  if (t < ntiles) {
    dma(kc, k_stb, koff, t, kbuf);
    dma(vc, v_stb, voff, t, vbuf);
  }
  const unsigned kread = (unsigned)(2 * wave * kTile) + G::k_read(lane);
  const unsigned vread = (unsigned)((2 * wave + 1) * kTile) + G::v_read(lane);
  for (; t < ntiles; t += 4) {
    const bool more = t + 4 < ntiles;
    f32x16 s[1];
    u32x4 pp[Half<T>::kParts][1][2];
    wait_vm<kDma>();  // K(t) has landed (V(t) is younger)
    score_tile<T, DH, 1>(lds, kread, qf, s);
    wait_lds();  // K(t) has been read
    if (more) dma(kc, k_stb, koff, t + 4, kbuf);
    softmax_tile<T, DH, 1, MASKED>(s, pp, st, t * kBN, qp, qp_lo, km.first, key_word(t), h, c);
    if (more)
      wait_vm<kDma>();
    else
      wait_vm<0>();
    pv_tile<T, DH, 1>(lds, vread, pp, st);
    wait_lds();
    if (more) dma(vc, v_stb, voff, t + 4, vbuf);
  }

  // partials of this wavefront into its own buffers: [dims tile][register][lane]
  float* part = reinterpret_cast<float*>(lds);
  constexpr int kPart = 2 * kTile / 4;  // floats per wavefront: 16 kDt x 64
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave * kPart + (16 * dt + r) * 64 + lane] = st.o[dt][r];
  if (h == 0) ml[wave][n] = make_float2(st.m, st.l);
  __syncthreads();
  f32x16 o[1] = {};
  if (wave < G::kDt) {
    float m = -INFINITY, l = 0.f, wgt[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) m = fmaxf(m, ml[w][n].x);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float2 x = ml[w][n];
      wgt[w] = x.x == m ? 1.f : fast_exp2((x.x - m) * c);  // a wavefront without a key of this row: 2^-inf
      l += wgt[w] * x.y;
    }
    const float inv = 1.f / l;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) v += wgt[w] * part[w * kPart + (16 * wave + r) * 64 + lane];
      o[0][r] = v * inv;
    }
    const uint32_t bad = bad_rows_of<1>(o);
    if (bad && lane == 0) atomicOr(&bad_rows, bad);
  }
  __syncthreads();
  if (wave < G::kDt && row_valid && !((bad_rows >> n) & 1u)) {
    uint16_t* op = reinterpret_cast<uint16_t*>(a.out) + (int64_t)it.b * a.o_sb + (int64_t)head * a.o_sh +
                   (int64_t)tok * a.o_st + 32 * wave + 4 * h;
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      st8(op + 8 * g4, u32x2{pack2<T>(o[0][4 * g4], o[0][4 * g4 + 1]), pack2<T>(o[0][4 * g4 + 2], o[0][4 * g4 + 3])});
  }
  for (uint32_t bad = bad_rows; bad; bad &= bad - 1) {
    const int row = __builtin_ctz(bad);
    const int rtok = it.t0 + row / a.G;
    if (row % 4 == wave && rtok < a.Tq)
      row_by_key<Half<T>::kDt>(a, it.b, it.kvh * a.G + row % a.G, rtok, km.first, lane);
  }
}

// ---------------------------------------------------------------- fp32 on the matrix cores
// 16 query rows (row = token * G + head) per workgroup of four wavefronts; wavefront w takes the 16-key tiles w, w + 4,
// .. straight from global memory into registers, and the four partial (m, l, O) of each row are merged in LDS.
//   S^T[16 keys x 16 rows] = K . Q^T     DH / 4 x v_mfma_f32_16x16x4_f32: lane (n, g) holds K row n and Q row n at
//                                        dims 16 j + 4 g .. +3 (16-byte loads), product (j, e) takes element e, so the
//                                        dims run through k in that order on both sides
//   O^T[Dh x 16 rows]     += V^T . P^T   DH / 4 products: key step i takes the keys 4 g + i, whose P is register i of
//                                        S^T's lane; lane (n, g) holds V row 4 g + i at dims 64 x + 4 n .. +3, so
//                                        product (x, e)'s row r is dim 64 x + 4 r + e
// Bound by the fp32 MFMA stream (64 x 32 cycles a tile) and the softmax between its halves.  One workgroup per
// query row on the vector ALU took 316.4 us for 300 queries on 700 keys (8 query, 2 KV heads, Dh 128), this kernel
// 21.2 us with four wavefronts (eight: 22.9, two: 37.3 us; four sequences of 550 tokens with 32 and 8 heads: 138 us
// with four, 210 with eight, 128 with two), at 3.2e-7 from float64 against 4.7e-7.  Loading the next tile into a
// second register set measured no faster.
// Everything stays fp32 (the products of v_mfma_f32 are fp32 fused multiply-adds) with expf, and the running max moves
// on every tile.
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

constexpr int kWavesF32 = 4;
template <int DH, bool MASKED>
__global__ __launch_bounds__(64 * kWavesF32) void dense_f32_kernel(const DenseArgs a) {
  constexpr int W = kWavesF32, kBN = 16, kJ = DH / 16, kX = DH / 64;
  constexpr int kPad = DH + 4;  // floats per row of the merge buffer: rows 16 bytes apart in the banks
  __shared__ __attribute__((aligned(16))) float part[W][16][kPad];
  __shared__ float2 ml[W][16];
  __shared__ uint32_t bad_rows;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tokens = 16 / a.G;
  const Item it = item_of(a, tokens);
  const int off = a.Tk - a.Tq;
  const int tok = it.t0 + n / a.G;
  const bool row_valid = tok < a.Tq;
  const int head = it.kvh * a.G + n % a.G;
  const int qp = row_valid ? off + tok : a.Tk - 1;
  const int qp_lo = off + it.t0;
  const int kv_end = off + min(it.t0 + tokens, a.Tq), last = kv_end - 1;
  const int ntiles = (kv_end + kBN - 1) / kBN;
  if (threadIdx.x == 0) bad_rows = 0;

  KeyMask km;
  int ts = 0;
  if constexpr (MASKED) {
    find_first(a, it.b, kv_end, lane, km);
    ts = min(km.first, qp_lo) / kBN;
    if (ts / 4 / 64 * 64 != km.base) load_window(a, it.b, ts / 4 / 64 * 64, lane, km);
  }

  const int kvh = it.kvh * a.G / (a.H / a.Hkv);
  const float* kc = reinterpret_cast<const float*>(a.k) + (int64_t)it.b * a.k_sb + (int64_t)kvh * a.k_sh;
  const float* vc = reinterpret_cast<const float*>(a.v) + (int64_t)it.b * a.v_sb + (int64_t)kvh * a.v_sh;
  f32x4 kf[kJ], vf[4][kX], qf[kJ];
  auto load_k = [&](int t) {
    const float* p = kc + (int64_t)min(t * kBN + n, last) * a.k_st + 4 * g;
#pragma unroll
    for (int j = 0; j < kJ; ++j) kf[j] = *reinterpret_cast<const f32x4*>(p + 16 * j);
  };
  auto load_v = [&](int t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* p = vc + (int64_t)min(t * kBN + 4 * g + i, last) * a.v_st + 4 * n;
#pragma unroll
      for (int x = 0; x < kX; ++x) vf[i][x] = *reinterpret_cast<const f32x4*>(p + 64 * x);
    }
  };
  int t = ts + wave;
  load_k(t);
  load_v(t);
  {
    const float* q = reinterpret_cast<const float*>(a.q) + (int64_t)it.b * a.q_sb + (int64_t)head * a.q_sh +
                     (int64_t)(row_valid ? tok : 0) * a.q_st + 4 * g;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      qf[j] = *reinterpret_cast<const f32x4*>(q + 16 * j);
      if (!row_valid) qf[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  f32x4 o[kX][4];
#pragma unroll
  for (int x = 0; x < kX; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[x][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  for (; t < ntiles; t += W) {
    f32x4 s2[2] = {};  // two chains
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) s2[e & 1] = mfma_f32(kf[j][e], qf[j][e], s2[e & 1]);
    load_k(t + W);  // past the last tile: copies of the last row, unused
    f32x4 s = (s2[0] + s2[1]) * a.scale;
    const int key0 = t * kBN + 4 * g;
    uint32_t vm = 0xffffu;
    if constexpr (MASKED) {
      if (t / 4 - km.base >= 64) load_window(a, it.b, t / 4, lane, km);
      vm = (uint32_t)(mask_word(km, t / 4) >> (16 * (t & 3))) & 0xffffu;
    }
    if (MASKED && vm != 0xffffu) {
      const bool own = qp < km.first;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool see = own ? key0 + i == qp : (((vm >> (4 * g + i)) & 1u) != 0 && key0 + i <= qp);
        s[i] = see ? s[i] : -INFINITY;
      }
    } else if (t * kBN + kBN - 1 > qp_lo) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = key0 + i > qp ? -INFINITY : s[i];
    }
    const float mx = max_xor32(max_xor16(__builtin_fmaxf(__builtin_fmaxf(s[0], s[1]), __builtin_fmaxf(s[2], s[3]))));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = m_new == m_run ? 1.f : expf(m_run - m_new);
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = s[i] == -INFINITY ? 0.f : expf(s[i] - m_new);
    l_run = l_run * alpha + sum_xor32(sum_xor16((p[0] + p[1]) + (p[2] + p[3])));
    m_run = m_new;
#pragma unroll
    for (int x = 0; x < kX; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[x][e] *= alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int x = 0; x < kX; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[x][e] = mfma_f32(vf[i][x][e], p[i], o[x][e]);
    load_v(t + W);
  }

  // o[x][e][r] is dim 64 x + 16 g + 4 r + e of row n
#pragma unroll
  for (int x = 0; x < kX; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<f32x4*>(&part[wave][n][64 * x + 16 * g + 4 * r]) =
          f32x4{o[x][0][r], o[x][1][r], o[x][2][r], o[x][3][r]};
  if (g == 0) ml[wave][n] = make_float2(m_run, l_run);
  __syncthreads();
  constexpr int kVecs = 16 * DH / 4, kPer = (kVecs + 64 * W - 1) / (64 * W);  // 16-byte pieces of the output, per thread
  f32x4 res[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int idx = u * 64 * W + (int)threadIdx.x, row = idx / (DH / 4), d = 4 * (idx % (DH / 4));
    if (idx < kVecs) {
      float m = -INFINITY, l = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) m = fmaxf(m, ml[w][row].x);
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float2 y = ml[w][row];
        const float wgt = y.x == m ? 1.f : expf(y.x - m);  // a wavefront without a key of this row: 0
        l += wgt * y.y;
        v += wgt * *reinterpret_cast<const f32x4*>(&part[w][row][d]);
      }
      res[u] = v / l;
      const f32x4 z = res[u];
      if (not_finite(z[0]) || not_finite(z[1]) || not_finite(z[2]) || not_finite(z[3])) atomicOr(&bad_rows, 1u << row);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int idx = u * 64 * W + (int)threadIdx.x, row = idx / (DH / 4), d = 4 * (idx % (DH / 4));
    const int rtok = it.t0 + row / a.G;
    if (idx < kVecs && rtok < a.Tq && !((bad_rows >> row) & 1u))
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + (int64_t)it.b * a.o_sb +
                                (int64_t)(it.kvh * a.G + row % a.G) * a.o_sh + (int64_t)rtok * a.o_st + d) = res[u];
  }
  for (uint32_t bad = bad_rows; bad; bad &= bad - 1) {
    const int row = __builtin_ctz(bad);
    const int rtok = it.t0 + row / a.G;
    if (row % W == wave && rtok < a.Tq)
      row_by_key<MLLM_DTYPE_F32>(a, it.b, it.kvh * a.G + row % a.G, rtok, km.first, lane);
  }
}

// What the MFMA kernels take besides the head size: 16-byte aligned rows (per16 elements in 16 bytes), key rows at
// most 32 MB apart (32-bit offsets within a tile), a positive scale (the running max is kept in unscaled scores).
bool mfma_operands(const DenseArgs& a, int per16) {
  const uintptr_t ptrs = (uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.out;
  const int64_t strides = a.q_sb | a.q_sh | a.q_st | a.k_sb | a.k_sh | a.k_st | a.v_sb | a.v_sh | a.v_st | a.o_sb |
                          a.o_sh | a.o_st;
  return ptrs % 16 == 0 && strides % per16 == 0 && a.k_st >= 0 && a.v_st >= 0 && a.k_st < (1 << 24) &&
         a.v_st < (1 << 24) && a.scale > 0.f && a.scale < INFINITY && a.Tk < (1 << 30);
}

// Workgroups of `rows` query rows.
int64_t items(const DenseArgs& a, int rows) {
  const int tokens = rows / a.G;
  return (int64_t)((a.Tq + tokens - 1) / tokens) * a.B * (a.H / a.G);
}

// Rows per workgroup of the 16-bit kernels: 128 from 1.5 workgroups per CU on, if they are fewer than those of 32, else 32.
// Measured (256 CUs, bf16, 32 query and 8 KV heads, Dh 128; 128 rows against 32, us): 128 workgroups of 128 rows (one sequence of
// 512 tokens) 23.4 / 12.5, 256 (one of 1,024) 41.0 / 29.8, 400 (two of 777) 39.0 / 38.4, 384 (four of 384) 21.7 / 26.3,
// 512 (four of 512) 28.2 / 38.6, 800 (four of 777) 49.4 / 68.8: a workgroup of 32 rows reads four times the K and V per
// row.  Where one workgroup of either size holds all of a head's queries, the 128-row one leaves wavefronts without a row,
// and one that has some walks all the keys: 1 or 8 queries on 1,024 keys, 64 sequences 47.4 / 43.0 and 48.2 / 43.8, 12 queries
// (two workgroups of 32 rows) 56.2 / 82.9.
int mfma_rows(const DenseArgs& a, int cus) {
  const int64_t large = items(a, 128);
  return 2 * large >= 3 * (int64_t)cus && large < items(a, 32) ? 128 : 32;
}

// Query heads of one KV head that share a row of the 16-bit kernels' workgroups.
int mfma_pack(int group) { return 32 % group == 0 ? group : 1; }

template <typename T, int DH>
int launch_mfma(const DenseArgs& a, hipStream_t st) {
  const int rows = mfma_rows(a, device_cus());
  const unsigned groups = (unsigned)items(a, rows);
  if (rows == 128) {
    if (a.key_valid)
      dense_mfma_kernel<T, DH, true><<<groups, 256, 0, st>>>(a);
    else
      dense_mfma_kernel<T, DH, false><<<groups, 256, 0, st>>>(a);
  } else {
    if (a.key_valid)
      dense_split_kernel<T, DH, true><<<groups, 256, 0, st>>>(a);
    else
      dense_split_kernel<T, DH, false><<<groups, 256, 0, st>>>(a);
  }
  return check_launch("mllm_dense_attention");
}

int launch_f32(const DenseArgs& a, hipStream_t st) {
  const unsigned groups = (unsigned)items(a, 16);
  if (a.Dh == 128) {
    if (a.key_valid)
      dense_f32_kernel<128, true><<<groups, 64 * kWavesF32, 0, st>>>(a);
    else
      dense_f32_kernel<128, false><<<groups, 64 * kWavesF32, 0, st>>>(a);
  } else if (a.key_valid) {
    dense_f32_kernel<64, true><<<groups, 64 * kWavesF32, 0, st>>>(a);
  } else {
    dense_f32_kernel<64, false><<<groups, 64 * kWavesF32, 0, st>>>(a);
  }
  return check_launch("mllm_dense_attention");
}

}  // namespace
}  // namespace mllm

extern "C" int mllm_dense_rows(int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t q_len,
                               int32_t num_cus) {
  using namespace mllm;
  if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || q_len <= 0) return 0;
  DenseArgs a{};
  a.B = batch;
  a.H = num_heads;
  a.Hkv = num_kv_heads;
  a.Tq = q_len;
  a.G = mfma_pack(num_heads / num_kv_heads);
  return mfma_rows(a, num_cus > 0 ? num_cus : device_cus());
}

extern "C" int mllm_dense_attention(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_st, const void* k, int64_t k_sb,
                                    int64_t k_sh, int64_t k_st, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_st,
                                    const uint8_t* key_valid, int64_t kv_sb, int64_t kv_st, int32_t batch,
                                    int32_t num_heads, int32_t num_kv_heads, int32_t q_len, int32_t kv_len,
                                    int32_t head_dim, float softmax_scale, int32_t dtype, void* out, int64_t o_sb,
                                    int64_t o_sh, int64_t o_st, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(dtype >= 0 && dtype <= 2, MLLM_ERR_UNSUPPORTED, "mllm_dense_attention: unsupported dtype");
  MLLM_REQUIRE(batch >= 0 && q_len >= 0 && kv_len >= q_len, MLLM_ERR_INVALID,
               "mllm_dense_attention: need kv_len >= q_len >= 0");
  MLLM_REQUIRE(head_dim > 0 && head_dim <= kMaxDh, MLLM_ERR_UNSUPPORTED, "mllm_dense_attention: head_dim must be in [1, 256]");
  MLLM_REQUIRE(num_kv_heads > 0 && num_heads % num_kv_heads == 0, MLLM_ERR_INVALID,
               "mllm_dense_attention: num_heads must be a multiple of num_kv_heads");
  MLLM_REQUIRE(num_heads <= 65535 && batch <= 65535, MLLM_ERR_UNSUPPORTED, "mllm_dense_attention: grid too large");
  if (batch == 0 || q_len == 0 || num_heads == 0) return MLLM_OK;
  MLLM_REQUIRE(q && k && v && out, MLLM_ERR_INVALID, "mllm_dense_attention: null pointer");
  const int group = num_heads / num_kv_heads;
  DenseArgs a{(const char*)q, (const char*)k, (const char*)v, key_valid, (char*)out, q_sb, q_sh, q_st, k_sb, k_sh,
              k_st, v_sb, v_sh, v_st, o_sb, o_sh, o_st, kv_sb, kv_st, batch, num_heads, num_kv_heads, q_len,
              kv_len, head_dim, mfma_pack(group), softmax_scale};
  dim3 grid(q_len, num_heads, batch);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // (more workgroups than a launch takes: dense_kernel, whose grid has the heads and the batch along y and z)
  if (dtype == MLLM_DTYPE_F32 && (head_dim == 128 || head_dim == 64) && mfma_operands(a, 4)) {
    a.G = 16 % group == 0 ? group : 1;
    if (items(a, 16) <= kMaxGroups256) return launch_f32(a, st);
  }
  if (dtype != MLLM_DTYPE_F32 && mfma_operands(a, 8) && items(a, 32) <= kMaxGroups256) {
    const bool bf16 = dtype == MLLM_DTYPE_BF16;
    if (head_dim == 128)
      return bf16 ? launch_mfma<BF16, 128>(a, st) : launch_mfma<F16, 128>(a, st);
    if (head_dim == 64) return bf16 ? launch_mfma<BF16, 64>(a, st) : launch_mfma<F16, 64>(a, st);
  }
  if (dtype == MLLM_DTYPE_F32)
    dense_kernel<MLLM_DTYPE_F32><<<grid, kThreads, 0, st>>>(a);
  else if (dtype == MLLM_DTYPE_F16)
    dense_kernel<MLLM_DTYPE_F16><<<grid, kThreads, 0, st>>>(a);
  else
    dense_kernel<MLLM_DTYPE_BF16><<<grid, kThreads, 0, st>>>(a);
  return check_launch("mllm_dense_attention");
}
