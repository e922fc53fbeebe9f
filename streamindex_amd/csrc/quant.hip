// FP8 / FP4 activation quantisation and the token compressor for gfx950.
//
// Reference behaviour being replaced:
//   * flash_sparse/utils/quantization.py:19-37  (act_quant_simulate: per-block
//     fp8 e4m3 quantise-dequantise, scale = amax / 448)
//   * flash_sparse/utils/quantization.py:40-65  (fp4_act_quant_simulate: per-block
//     e2m1 grid snap, scale = amax / 6)
//   * flash_sparse/reference.py:176-272          (reference_token_compressor,
//     eq. 11-12 with overlap, eq. 22-23 without)
//   * flash_sparse/utils/compression.py:13-24    (softmax_gated_pool)
//
// The simulate kernels reproduce the reference's torch arithmetic step by
// step, including the rounding to the input dtype after every elementwise op
// (bf16 / fp16 results are rounded to nearest even, as torch's CPU and GPU
// kernels do), so their outputs are bit-identical to the reference formulas.
// The packing kernels write the production formats the quantised indexer
// reads: fp8 e4m3 values with one fp32 scale per block, and fp4 e2m1 values
// packed two per byte (element 2i in the low nibble) with power-of-two
// (UE8M0) scales.  All are bandwidth-bound: one thread handles 8 elements, a
// block of `bs` elements is reduced across bs/8 adjacent lanes.  (With 8
// two-byte loads a thread and a 64-bit division to find its block, packing
// 134M bf16 values to fp4 took 125 us; 64 us, the rate
// of a copy, with 16-byte loads, shifts and the conversion instruction.)
#include <hip/hip_fp16.h>

#include <string>

#include "si_common.h"
#include "si_status.h"

namespace si {

// ---- rounding helpers --------------------------------------------------------
// dtype codes: 0 = fp32, 1 = bf16, 2 = fp16
template <int DT>
struct Elt;
template <>
struct Elt<0> {
  using T = float;
  static __device__ __forceinline__ float load(const void* p, int64_t i) { return static_cast<const float*>(p)[i]; }
  static __device__ __forceinline__ float round(float x) { return x; }
  static __device__ __forceinline__ void store(void* p, int64_t i, float x) { static_cast<float*>(p)[i] = x; }
};
__device__ __forceinline__ float bf16_round(float x) {
  // round to nearest even (NaN kept quiet)
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return __uint_as_float(u | 0x00400000u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return __uint_as_float(u & 0xffff0000u);
}
template <>
struct Elt<1> {
  static __device__ __forceinline__ float load(const void* p, int64_t i) {
    return __uint_as_float(static_cast<uint32_t>(static_cast<const uint16_t*>(p)[i]) << 16);
  }
  static __device__ __forceinline__ float round(float x) { return bf16_round(x); }
  static __device__ __forceinline__ void store(void* p, int64_t i, float x) {
    static_cast<uint16_t*>(p)[i] = static_cast<uint16_t>(__float_as_uint(bf16_round(x)) >> 16);
  }
};
template <>
struct Elt<2> {
  static __device__ __forceinline__ float load(const void* p, int64_t i) {
    return __half2float(static_cast<const __half*>(p)[i]);
  }
  static __device__ __forceinline__ float round(float x) { return __half2float(__float2half_rn(x)); }
  static __device__ __forceinline__ void store(void* p, int64_t i, float x) {
    static_cast<__half*>(p)[i] = __float2half_rn(x);
  }
};

// N consecutive elements as fp32 (N = 1, or a 16-byte vector).
template <int DT, int N>
__device__ __forceinline__ void load_vec(const void* p, int64_t i, float (&v)[N]) {
  if constexpr (N == 1) {
    v[0] = Elt<DT>::load(p, i);
  } else if constexpr (DT == 0) {
    static_assert(N == 4, "16 bytes");
    const f32x4 w = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = w[e];
  } else {
    static_assert(N == 8, "16 bytes");
    const u32x4 w = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p) + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint16_t h = static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
      if constexpr (DT == 1) v[e] = __uint_as_float(static_cast<uint32_t>(h) << 16);
      else v[e] = __half2float(__ushort_as_half(h));
    }
  }
}
template <int DT, int N>
__device__ __forceinline__ void store_vec(void* p, int64_t i, const float (&v)[N]) {
  if constexpr (N == 1) {
    Elt<DT>::store(p, i, v[0]);
  } else if constexpr (DT == 0) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(p) + i) = f32x4{v[0], v[1], v[2], v[3]};
  } else {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (DT == 1)
        w[e] = (__float_as_uint(bf16_round(v[2 * e])) >> 16) | (__float_as_uint(bf16_round(v[2 * e + 1])) & 0xffff0000u);
      else
        w[e] = static_cast<uint32_t>(__half_as_ushort(__float2half_rn(v[2 * e]))) |
               (static_cast<uint32_t>(__half_as_ushort(__float2half_rn(v[2 * e + 1]))) << 16);
    }
    *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p) + i) = w;
  }
}

// Nearest fp8 e4m3 (OCP "fn": bias 7, no infinities, max 448) value to x,
// ties to even; |x| <= 448 here (callers clamp).  Returns the value as float.
__device__ __forceinline__ float e4m3_round(float x) {
  const float a = __builtin_fabsf(x);
  if (!(a > 0.f)) return x;  // +-0 (and NaN) unchanged
  int e;
  __builtin_frexpf(a, &e);        // a = f 2^e, f in [0.5, 1)
  int ex = e - 1;                 // a = g 2^ex, g in [1, 2)
  if (ex < -6) ex = -6;           // subnormals share the 2^-6 binade's quantum
  const float q = __builtin_ldexpf(1.0f, ex - 3);  // spacing: 3 mantissa bits
  const float r = __builtin_rintf(a / q) * q;      // a / q exact (power of two); rint = ties to even
  return __builtin_copysignf(r > 448.f ? 448.f : r, x);
}
// Byte encoding of an e4m3 value produced by e4m3_round.
__device__ __forceinline__ uint8_t e4m3_bits(float v) {
  const uint32_t sign = __float_as_uint(v) >> 31;
  const float a = __builtin_fabsf(v);
  uint32_t code;
  if (a < 0.015625f) {  // subnormal: m 2^-9
    code = static_cast<uint32_t>(a * 512.f);
  } else {
    int e;
    const float f = __builtin_frexpf(a, &e);  // a = f 2^e
    const uint32_t m = static_cast<uint32_t>((f * 2.f - 1.f) * 8.f);
    code = (static_cast<uint32_t>(e - 1 + 7) << 3) | m;
  }
  return static_cast<uint8_t>((sign << 7) | code);
}

// e2m1 grid as the reference lists it (ascending), used by the simulation's
// argmin; and the encoding of |value| for the packed format.
__constant__ float kFp4Grid[15] = {-6.f, -4.f, -3.f, -2.f, -1.5f, -1.f, -0.5f, 0.f, 0.5f, 1.f, 1.5f, 2.f, 3.f, 4.f, 6.f};

// Nearest e2m1 value, ties to the even code (0, 1, 2, 4 have even codes).
__device__ __forceinline__ uint32_t e2m1_code(float x) {
  const float a = __builtin_fabsf(x);
  uint32_t c;
  if (a <= 0.25f) c = 0;            // 0.25: tie between 0 (code 0) and 0.5 (code 1) -> 0
  else if (a < 0.75f) c = 1;        // 0.5
  else if (a <= 1.25f) c = 2;       // 1.0 (0.75 -> 1.0, 1.25 -> 1.0)
  else if (a < 1.75f) c = 3;        // 1.5
  else if (a <= 2.5f) c = 4;        // 2.0 (1.75 -> 2.0, 2.5 -> 2.0)
  else if (a < 3.5f) c = 5;         // 3.0
  else if (a <= 5.f) c = 6;         // 4.0 (3.5 -> 4.0, 5 -> 4.0)
  else c = 7;                       // 6.0
  return (c != 0 && __builtin_signbitf(x)) ? (c | 8u) : c;
}

// ---- simulate kernels (bit-identical to the reference formulas) --------------
struct QuantArgs {
  const void* x;
  void* y;          // simulate: dequantised values (same dtype); pack: values
  float* scale;     // pack: one scale per block
  int64_t nblocks;
  int bs;           // block size (multiple of 8, bs / 8 a power of two <= 64)
  int lg;           // log2(bs / 8): the lanes that share a block
  int vec;          // x is 16-byte aligned
  int mode;         // pack: 0 = fp32 scale (amax / max), 1 = power-of-two (UE8M0) scale
};

template <int DT>
__device__ __forceinline__ float block_amax(const QuantArgs& q, int64_t base, int g, float (&v)[8]) {
  float m = 0.f;
  if (q.vec) {
    if constexpr (DT == 0) {
      float a[4], b[4];
      load_vec<0, 4>(q.x, base, a);
      load_vec<0, 4>(q.x, base + 4, b);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = a[e];
        v[4 + e] = b[e];
      }
    } else {
      load_vec<DT, 8>(q.x, base, v);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = Elt<DT>::load(q.x, base + e);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) m = __builtin_fmaxf(m, __builtin_fabsf(v[e]));
  for (int w = 1; w < g; w <<= 1) m = __builtin_fmaxf(m, __shfl_xor(m, w, 64));
  return m;
}

// act_quant_simulate: amax -> clamp_min(1e-4) -> scale = amax / 448 ->
// clamp(x / scale, +-448) -> e4m3 -> float * scale -> dtype (each op rounded to
// the dtype as torch does).
template <int DT>
__global__ __launch_bounds__(256) void fp8_simulate_kernel(QuantArgs q) {
  const int g = 1 << q.lg;  // lanes per block
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t blk = t >> q.lg;
  if (blk >= q.nblocks) return;  // whole lane groups leave together (g divides 64)
  float v[8];
  float amax = block_amax<DT>(q, t * 8, g, v);
  amax = Elt<DT>::round(__builtin_fmaxf(amax, 1e-4f));
  const float scale = Elt<DT>::round(amax / 448.f);
  const int64_t base = t * 8;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float y = Elt<DT>::round(v[e] / scale);
    y = __builtin_fminf(__builtin_fmaxf(y, -448.f), 448.f);
    Elt<DT>::store(q.y, base + e, e4m3_round(y) * scale);
  }
}

// fp4_act_quant_simulate: amax -> clamp_min(6 * 2^-126) -> scale = amax / 6 ->
// clamp(x / scale, +-6) -> argmin |scaled - grid| (first minimum, diffs in the
// dtype) -> grid value * scale.
template <int DT>
__global__ __launch_bounds__(256) void fp4_simulate_kernel(QuantArgs q) {
  const int g = 1 << q.lg;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t blk = t >> q.lg;
  if (blk >= q.nblocks) return;
  float v[8];
  float amax = block_amax<DT>(q, t * 8, g, v);
  amax = Elt<DT>::round(__builtin_fmaxf(amax, 6.f * 0x1p-126f));
  const float scale = Elt<DT>::round(amax / 6.f);
  const int64_t base = t * 8;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float y = Elt<DT>::round(v[e] / scale);
    y = __builtin_fminf(__builtin_fmaxf(y, -6.f), 6.f);
    float best = __builtin_fabsf(Elt<DT>::round(y - kFp4Grid[0]));
    int bi = 0;
#pragma unroll
    for (int i = 1; i < 15; ++i) {
      const float d = __builtin_fabsf(Elt<DT>::round(y - kFp4Grid[i]));
      if (d < best) {
        best = d;
        bi = i;
      }
    }
    Elt<DT>::store(q.y, base + e, kFp4Grid[bi] * scale);
  }
}

// ---- packing kernels (production formats) ------------------------------------
__device__ __forceinline__ float pow2_ceil(float x) {  // smallest 2^k >= x (x > 0, normal)
  int e;
  const float f = __builtin_frexpf(x, &e);  // x = f 2^e, f in [0.5, 1)
  return f == 0.5f ? x : __builtin_ldexpf(1.0f, e);
}

// fp8 e4m3 + one fp32 scale per block: scale = max(amax, 1e-4) / 448 (mode 0)
// or its power-of-two ceiling (mode 1); value = e4m3(clamp(x / scale, +-448)).
template <int DT>
__global__ __launch_bounds__(256) void fp8_pack_kernel(QuantArgs q) {
  const int g = 1 << q.lg;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t blk = t >> q.lg;
  if (blk >= q.nblocks) return;
  float v[8];
  const float amax = __builtin_fmaxf(block_amax<DT>(q, t * 8, g, v), 1e-4f);
  float scale = amax / 448.f;
  if (q.mode == 1) scale = pow2_ceil(scale);
  if ((t & (g - 1)) == 0) q.scale[blk] = scale;
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float y = v[e] / scale;
    y = __builtin_fminf(__builtin_fmaxf(y, -448.f), 448.f);
    w[e >> 2] |= static_cast<uint32_t>(e4m3_bits(e4m3_round(y))) << (8 * (e & 3));
  }
  *reinterpret_cast<uint2*>(static_cast<uint8_t*>(q.y) + t * 8) = uint2{w[0], w[1]};
}

// fp4 e2m1 packed two per byte (element 2i low nibble) + power-of-two scale
// per block: scale = 2^ceil(log2(max(amax, 6 * 2^-126) / 6)), so |x / scale| <= 6.
template <int DT>
__global__ __launch_bounds__(256) void fp4_pack_kernel(QuantArgs q) {
  const int g = 1 << q.lg;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t blk = t >> q.lg;
  if (blk >= q.nblocks) return;
  float v[8];
  const float amax = __builtin_fmaxf(block_amax<DT>(q, t * 8, g, v), 6.f * 0x1p-126f);
  const float scale = pow2_ceil(amax / 6.f);
  if ((t & (g - 1)) == 0) q.scale[blk] = scale;
  uint32_t w = 0u;
  const float inv = 1.f / scale;  // exact, as is the product: scale is a normal power of two up to 2^126
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] *= inv;
  bool nan = false;
#pragma unroll
  for (int e = 0; e < 8; e += 2) nan |= __builtin_isunordered(v[e], v[e + 1]);
  if (__builtin_amdgcn_ballot_w64(nan || !(amax < __builtin_inff())) == 0) {
    // The conversion instruction rounds as e2m1_code does but keeps the sign of
    // a value that rounds to zero (e2m1_code: 130 instructions for the 8).
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[0], v[1], 1.0f, 0);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[2], v[3], 1.0f, 1);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[4], v[5], 1.0f, 2);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[6], v[7], 1.0f, 3);
    const uint32_t nonzero = (w | (w >> 1) | (w >> 2)) & 0x11111111u;
    w &= 0x77777777u | (nonzero << 3);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) w |= e2m1_code(v[e]) << (4 * e);
  }
  *reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(q.y) + t * 4) = w;
}

// ---- token compressor / softmax-gated pool ----------------------------------
struct PoolArgs {
  const void* ca;  // [B, S, C] content, stream a
  const void* za;  // [B, S, C] scores, stream a
  const void* cb;  // stream b (overlap) or null
  const void* zb;
  const float* ba;  // [m, C] bias of stream a (fp32)
  const float* bb;  // [m, C] bias of stream b or null
  void* out;        // [B, S / m, C]
  int64_t B, S, C, m, nblk;
  int overlap;
};

// Overlap (CSA, eq. 11-12): softmax over the 2m scores [z_a + b_a of block i ;
// z_b + b_b of block i-1] (block 0: the b half is -inf / 0); no overlap (HCA,
// eq. 22-23): softmax over the m scores of block i.  fp32 arithmetic, output
// rounded to the dtype.
//
// One item per (batch, compressed entry, N channels); R threads of a workgroup
// share an item, each taking every R-th chunk of U rows, and meet in LDS.
// Bound: HBM.  Every score and content row is read once, 16 bytes a lane
// (N = 8, fp32: 4), U scores and U contents in flight per thread, with the
// running maximum moved once a chunk (an entry of up to U rows never rescales).
// N = 1 serves the channel counts and addresses that are not whole 16-byte
// vectors.  R and U: launch_compress.
template <int DT, int N, int R, int U>
__global__ __launch_bounds__(256) void token_compress_kernel(PoolArgs p) {
  constexpr int ITEMS = 256 / R;
  const int local = static_cast<int>(threadIdx.x) % ITEMS;
  const int part = static_cast<int>(threadIdx.x) / ITEMS;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * ITEMS + local;
  const int64_t cv = p.C / N;
  const bool live = item < p.B * p.nblk * cv;
  if (R == 1 && !live) return;
  const int64_t at = live ? item : 0;
  int64_t c, i, b;
  if (p.B * p.nblk * cv <= 0x7fffffff) {  // (32-bit divisions where they do)
    const uint32_t x = static_cast<uint32_t>(at), y = x / static_cast<uint32_t>(cv);
    c = static_cast<int64_t>(x % static_cast<uint32_t>(cv)) * N;
    i = y % static_cast<uint32_t>(p.nblk);
    b = y / static_cast<uint32_t>(p.nblk);
  } else {
    c = at % cv * N;
    i = (at / cv) % p.nblk;
    b = at / (cv * p.nblk);
  }
  const int64_t rowa = (b * p.S + i * p.m) * p.C + c;
  const int64_t rowb = rowa - p.m * p.C;  // block i-1
  const int64_t rows = p.overlap && i > 0 ? 2 * p.m : p.m;
  float mx[N], den[N], num[N];
#pragma unroll
  for (int e = 0; e < N; ++e) {
    mx[e] = -__builtin_inff();
    den[e] = 0.f;
    num[e] = 0.f;
  }
  for (int64_t j0 = part * U; j0 < rows; j0 += R * U) {
    float z[U][N], v[U][N];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t j = j0 + u;
      if (j < rows) {
        const bool second = j >= p.m;
        const int64_t off = second ? rowb + (j - p.m) * p.C : rowa + j * p.C;
        float bias[N];
        load_vec<DT, N>(second ? p.zb : p.za, off, z[u]);
        load_vec<DT, N>(second ? p.cb : p.ca, off, v[u]);
        const float* bp = second ? p.bb + (j - p.m) * p.C + c : p.ba + j * p.C + c;
#pragma unroll
        for (int e = 0; e < N; e += N < 4 ? N : 4) {
          if constexpr (N == 1) {
            bias[0] = bp[0];
          } else {
            const f32x4 w = *reinterpret_cast<const f32x4*>(bp + e);
#pragma unroll
            for (int q = 0; q < 4; ++q) bias[e + q] = w[q];
          }
        }
#pragma unroll
        for (int e = 0; e < N; ++e) z[u][e] += bias[e];
      } else {
#pragma unroll
        for (int e = 0; e < N; ++e) {
          z[u][e] = -__builtin_inff();
          v[u][e] = 0.f;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < N; ++e) {
      float m = mx[e];
#pragma unroll
      for (int u = 0; u < U; ++u) m = __builtin_fmaxf(m, z[u][e]);
      const float ref = m == -__builtin_inff() ? 0.f : m;  // (every score so far -inf: all weights 0)
      const float s = __expf(mx[e] - ref);
      den[e] *= s;
      num[e] *= s;
      mx[e] = m;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float w = __expf(z[u][e] - ref);
        den[e] += w;
        num[e] += w * v[u][e];
      }
    }
  }
  if constexpr (R > 1) {
    __shared__ float part_lds[R][3 * N][ITEMS];
#pragma unroll
    for (int e = 0; e < N; ++e) {
      part_lds[part][e][local] = mx[e];
      part_lds[part][N + e][local] = den[e];
      part_lds[part][2 * N + e][local] = num[e];
    }
    __syncthreads();
    if (part != 0 || !live) return;
#pragma unroll
    for (int e = 0; e < N; ++e) {
      float m = mx[e];
      for (int q = 1; q < R; ++q) m = __builtin_fmaxf(m, part_lds[q][e][local]);
      const float ref = m == -__builtin_inff() ? 0.f : m;
      float d = 0.f, a = 0.f;
      for (int q = 0; q < R; ++q) {
        const float s = __expf(part_lds[q][e][local] - ref);
        d += part_lds[q][N + e][local] * s;
        a += part_lds[q][2 * N + e][local] * s;
      }
      den[e] = d;
      num[e] = a;
    }
  }
#pragma unroll
  for (int e = 0; e < N; ++e) num[e] = num[e] / den[e];
  store_vec<DT, N>(p.out, at * N, num);
}

// softmax_gated_pool over the middle axis of [outer, L, inner] tensors.
template <int DT>
__global__ __launch_bounds__(256) void gated_pool_kernel(const void* kv, const void* score, void* out, int64_t outer,
                                                          int64_t L, int64_t inner) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= outer * inner) return;
  const int64_t o = t / inner, in = t % inner;
  const int64_t base = o * L * inner + in;
  float mx = -__builtin_inff();
  for (int64_t l = 0; l < L; ++l) mx = __builtin_fmaxf(mx, Elt<DT>::load(score, base + l * inner));
  float den = 0.f, num = 0.f;
  for (int64_t l = 0; l < L; ++l) {
    const float w = __expf(Elt<DT>::load(score, base + l * inner) - mx);
    den += w;
    num += w * Elt<DT>::load(kv, base + l * inner);
  }
  Elt<DT>::store(out, t, num / den);
}

template <template <int> class K, typename A>
static int launch_dt(int dt, int64_t threads, const A& args, const char* name, hipStream_t st) {
  const int64_t blocks = (threads + 255) / 256;
  if (blocks > 0x7fffffffLL) return set_error(SI_ERR_UNSUPPORTED, "tensor too large");
  if (blocks == 0) return SI_OK;
  switch (dt) {
    case 0: hipLaunchKernelGGL(K<0>::fn, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, args); break;
    case 1: hipLaunchKernelGGL(K<1>::fn, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, args); break;
    case 2: hipLaunchKernelGGL(K<2>::fn, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, args); break;
    default: return set_error(SI_ERR_UNSUPPORTED, "dtype must be fp32, bf16 or fp16");
  }
  return check_launch(name);
}
template <int DT> struct Fp8Sim { static constexpr auto fn = fp8_simulate_kernel<DT>; };
template <int DT> struct Fp4Sim { static constexpr auto fn = fp4_simulate_kernel<DT>; };
template <int DT> struct Fp8Pack { static constexpr auto fn = fp8_pack_kernel<DT>; };
template <int DT> struct Fp4Pack { static constexpr auto fn = fp4_pack_kernel<DT>; };

template <int DT, int N, int R, int U>
static int launch_compress_r(const PoolArgs& p, hipStream_t st) {
  const int64_t items = p.B * p.nblk * (p.C / N);
  const int64_t blocks = (items + 256 / R - 1) / (256 / R);
  if (blocks > 0x7fffffffLL) return set_error(SI_ERR_UNSUPPORTED, "tensor too large");
  if (blocks == 0) return SI_OK;
  hipLaunchKernelGGL((token_compress_kernel<DT, N, R, U>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, p);
  return check_launch("token_compress_kernel");
}
// Threads per item (R) and rows per chunk (U).  Loads in flight hide the memory
// latency: an entry of more than U rows is split over several threads where the
// items alone do not fill the GPU, and not where they do (each added thread costs a
// share of an LDS exchange).  us, one thread against R (bf16, 16-byte vectors):
//   S = 512, C = 64:  m = 2 x 24  19 -> 6 (R = 8), m = 12  6.8 -> 5.8 (2)
//   S = 64K, C = 576:  m = 24  34 (1), 41 with R = 4;  m = 64  83 (before) -> 37 (8)
//   S = 64K, C = 64:  m = 16  11 -> 6 (4)
// Many single channels (N = 1) of few rows need no chunk at all, each chunk's unused
// rows cost more than the rescales: S = 64K, C = 100, m = 1  33 -> 24, m = 16  16 -> 13.
template <int DT, int N>
static int launch_compress_n(const PoolArgs& p, hipStream_t st) {
  const int64_t items = p.B * p.nblk * (p.C / N);
  const int64_t rows = p.overlap ? 2 * p.m : p.m;
  if (N == 1 && rows <= 32 && items >= (3 << 16)) return launch_compress_r<DT, N, 1, 1>(p, st);
  int R = 1;
  if (N > 1 && p.m >= 32) R = 8;
  while (R < 8 && R * 8 < rows && items * R < (N == 1 ? 1 << 19 : 1 << 17)) R *= 2;
  switch (R) {
    case 1: return launch_compress_r<DT, N, 1, 8>(p, st);
    case 2: return launch_compress_r<DT, N, 2, 8>(p, st);
    case 4: return launch_compress_r<DT, N, 4, 8>(p, st);
    default: return launch_compress_r<DT, N, 8, 8>(p, st);
  }
}
template <int DT>
static int launch_compress(const PoolArgs& p, hipStream_t st) {
  constexpr int N = DT == 0 ? 4 : 8;
  const uintptr_t ptrs = reinterpret_cast<uintptr_t>(p.ca) | reinterpret_cast<uintptr_t>(p.za) |
                         reinterpret_cast<uintptr_t>(p.cb) | reinterpret_cast<uintptr_t>(p.zb) |
                         reinterpret_cast<uintptr_t>(p.ba) | reinterpret_cast<uintptr_t>(p.bb) |
                         reinterpret_cast<uintptr_t>(p.out);
  return p.C % N || (ptrs & 15) ? launch_compress_n<DT, 1>(p, st) : launch_compress_n<DT, N>(p, st);
}

static int log2_lanes(int64_t bs) {
  int lg = 0;
  while ((8ll << lg) < bs) ++lg;
  return lg;
}
static int aligned16(const void* x) {
  return (reinterpret_cast<uintptr_t>(x) & 15) == 0;
}

static int check_block(int64_t n, int64_t bs) {
  if (bs < 8 || bs > 512 || bs % 8 || ((bs / 8) & (bs / 8 - 1)))
    return set_error(SI_ERR_UNSUPPORTED, "block_size must be 8 * 2^j <= 512, got " + std::to_string(bs));
  if (n < 0 || n % bs) return set_error(SI_ERR_INVALID, "element count must be a multiple of block_size");
  return SI_OK;
}

}  // namespace si

using namespace si;

extern "C" int si_quant_simulate(const void* x, void* y, int dtype, int64_t n, int64_t block_size, int fp4,
                                 void* stream) {
  int rc = check_block(n, block_size);
  if (rc) return rc;
  if (n > 0 && (!x || !y)) return set_error(SI_ERR_INVALID, "null pointer argument");
  QuantArgs q{x, y, nullptr, n / block_size, static_cast<int>(block_size), log2_lanes(block_size), aligned16(x), 0};
  const int64_t threads = n / 8;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return fp4 ? launch_dt<Fp4Sim>(dtype, threads, q, "fp4_simulate_kernel", st)
             : launch_dt<Fp8Sim>(dtype, threads, q, "fp8_simulate_kernel", st);
}

extern "C" int si_quant_pack(const void* x, void* y, float* scale, int dtype, int64_t n, int64_t block_size, int fp4,
                             int pow2_scale, void* stream) {
  int rc = check_block(n, block_size);
  if (rc) return rc;
  if (n > 0 && (!x || !y || !scale)) return set_error(SI_ERR_INVALID, "null pointer argument");
  if ((reinterpret_cast<uintptr_t>(y) & 7) || (fp4 && (reinterpret_cast<uintptr_t>(y) & 3)))
    return set_error(SI_ERR_INVALID, "output must be 8-byte aligned");
  QuantArgs q{x, y, scale, n / block_size, static_cast<int>(block_size), log2_lanes(block_size), aligned16(x),
              pow2_scale ? 1 : 0};
  const int64_t threads = n / 8;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return fp4 ? launch_dt<Fp4Pack>(dtype, threads, q, "fp4_pack_kernel", st)
             : launch_dt<Fp8Pack>(dtype, threads, q, "fp8_pack_kernel", st);
}

extern "C" int si_token_compress(const void* c_a, const void* z_a, const float* b_a, const void* c_b, const void* z_b,
                                 const float* b_b, int dtype, int64_t B, int64_t S, int64_t C, int64_t m, int overlap,
                                 void* out, void* stream) {
  if (B < 0 || S < 0 || C <= 0 || m <= 0) return set_error(SI_ERR_INVALID, "bad dimension");
  const int64_t nblk = S / m;
  if (B * nblk > 0 && (!c_a || !z_a || !b_a || !out || (overlap && (!c_b || !z_b || !b_b))))
    return set_error(SI_ERR_INVALID, "null pointer argument");
  PoolArgs p{c_a, z_a, c_b, z_b, b_a, b_b, out, B, S, C, m, nblk, overlap ? 1 : 0};
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case 0: return launch_compress<0>(p, st);
    case 1: return launch_compress<1>(p, st);
    case 2: return launch_compress<2>(p, st);
    default: return set_error(SI_ERR_UNSUPPORTED, "dtype must be fp32, bf16 or fp16");
  }
}

extern "C" int si_gated_pool(const void* kv, const void* score, void* out, int dtype, int64_t outer, int64_t L,
                             int64_t inner, void* stream) {
  if (outer < 0 || L <= 0 || inner < 0) return set_error(SI_ERR_INVALID, "bad dimension");
  if (outer * inner > 0 && (!kv || !score || !out)) return set_error(SI_ERR_INVALID, "null pointer argument");
  const int64_t threads = outer * inner;
  const int64_t blocks = (threads + 255) / 256;
  if (blocks == 0) return SI_OK;
  if (blocks > 0x7fffffffLL) return set_error(SI_ERR_UNSUPPORTED, "tensor too large");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(blocks));
  switch (dtype) {
    case 0: hipLaunchKernelGGL(gated_pool_kernel<0>, grid, dim3(256), 0, st, kv, score, out, outer, L, inner); break;
    case 1: hipLaunchKernelGGL(gated_pool_kernel<1>, grid, dim3(256), 0, st, kv, score, out, outer, L, inner); break;
    case 2: hipLaunchKernelGGL(gated_pool_kernel<2>, grid, dim3(256), 0, st, kv, score, out, outer, L, inner); break;
    default: return set_error(SI_ERR_UNSUPPORTED, "dtype must be fp32, bf16 or fp16");
  }
  return check_launch("gated_pool_kernel");
}
