// wide.hip -- linears over many rows at once (a prompt's tokens, an encoder
// output's frames, op-layer batches): a rows kernel that applies the norm /
// residual prologue and writes the activations as split 16-bit planes, and an
// MFMA GEMM over those planes.
//
// What bounds it: in the K loop the matrix cores, two thirds of its cycles; a
// launch of one round spends as long again on its start and its outputs (29 %
// of the matrix cores' cycles at 13824 x 1152 x 512).  An fp32 activation needs
// more than one 16-bit part, so every weight x row product costs one MFMA a
// part; the parts are made once per row here instead of once per weight tile
// in the GEMM (gemm.hip splits the fp32 rows again in every workgroup, which is
// right for the few rows of a decode step and costs more than the MFMAs from
// about a hundred rows on).
//   int8 / int4 weights are whole numbers below 2^11, exact in fp16, so two
//   fp16 parts do: x 2^s = hi + lo 2^-12 + e, round to nearest each, with s
//   per row putting the largest |x| in [2^14, 2^15).  The second part is kept
//   2^12 larger and meets weights 2^12 smaller (exact as well), so |e| <=
//   2^-23 |x 2^s| down to 2^-14, 2^-28 of the row's largest value: the last
//   of 24 bits.  The error against 64 bits is that of the fp32 sums (2.1e-7 at
//   13824 x 1152 x 512 rows with either split).  A block of 64 elements with a
//   smaller one (zeros aside) is stored as its fp32 bits instead, and a GEMM
//   tile takes the steps of its blocks like that last, all their rows split
//   into three bf16 parts, exactly, like the kernels of gemm.hip.
//   bf16 / bfp16 weights have an 8-bit exponent, which fp16 does not hold:
//   three bf16 parts, x = hi + mid + lo exactly, as in gemm.hip.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_dev.h"
#include "wide.h"

namespace xe {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;
constexpr int kBK = 64;             // k per step
constexpr int kNoRec = 0x7ffffff0;  // past every buffer: loads return zeros
constexpr int kMaxK = 16384;        // rows kernel: 8 float4 a thread of 512
constexpr int kMaxKs = 8;           // K splits
constexpr int kRowPad = 128;        // rexp is readable up to a multiple of it
constexpr int kLds = 160 * 1024;    // LDS of a CU
constexpr int kLoExp = 12;          // fp16 parts: the second one is kept 2^kLoExp larger
constexpr int kMaxSteps = kMaxK / kBK;

// rexp of a row: its s, and above it whether blocks of the row are stored as
// fp32: upper halves in plane 0, lower halves in plane 1
__host__ __device__ __forceinline__ int rexp_word(int s, bool raw) { return (s & 0xffff) | (raw ? 1 << 16 : 0); }
__device__ __forceinline__ int rexp_s(int w) { return static_cast<int16_t>(w); }
__device__ __forceinline__ bool rexp_raw(int w) { return (w >> 16) & 1; }
// byte of (row, step) in the flags behind rexp, written for rows with rexp_raw
__device__ __forceinline__ size_t raw_at(int row, int step, int steps) {
  return (static_cast<size_t>(row / kRowPad) * steps + step) * kRowPad + row % kRowPad;
}

template <int WT>
constexpr int planes_of() {
  return WT == XE_I8 || WT == XE_I4 ? 2 : 3;
}

// ---------------------------------------------------------------------------
// rows kernel
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ uint32_t pack_lo16(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x05040100u);
}
__device__ __forceinline__ float trunc_bf16(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

// One workgroup a row: t = x (+ post(sub)) -> res_out, h = norm(t) -> planes.
// A thread holds float4 chunks threadIdx.x + T j, j < NV, from the first load
// to the plane stores (K <= 4 T NV), so the row is read once.  Bound by
// its chain of block reductions (one per norm statistic, one for the row's
// largest and smallest |h|), which the other rows' workgroups of the CU
// overlap.
template <int NV, int P, int T>
__global__ __launch_bounds__(T) void wide_rows_kernel(gdev::GemvParams p, uint16_t *planes, int *rexp, uint8_t *raw_flags) {
  __shared__ float red[2 * 4 * gdev::kMaxWaves];
  __shared__ float mx[T / 64];
  __shared__ float mn[T / 64];
  const int b = blockIdx.x, K = p.k, K4 = K / 4;
  const float fk = static_cast<float>(K);
  float t[NV][4], g[NV][4], be[NV][4];
  int slot = 0;
  const float *xr = static_cast<const float *>(p.x) + static_cast<size_t>(b) * p.ldx;
  const uint16_t *xh = static_cast<const uint16_t *>(p.x) + static_cast<size_t>(b) * p.ldx;
  const bool ln = p.norm == XE_NORM_LN;
  const bool has_sub = p.sub || p.sub_part;
  float su[NV][4], pw[NV][4];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int i = 4 * (static_cast<int>(threadIdx.x) + j * T);
    const bool on = i < K;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f), s4 = v, w4 = v, g4 = v, b4 = v;
    if (on) {
      if (p.x_bf16) {
        const u32x2 h = *reinterpret_cast<const u32x2 *>(xh + i);
        v = make_float4(__uint_as_float(h.x << 16), __uint_as_float(h.x & 0xffff0000u), __uint_as_float(h.y << 16),
                        __uint_as_float(h.y & 0xffff0000u));
      } else {
        v = ld4(xr + i);
      }
      if (p.norm != XE_NORM_NONE) g4 = ld4(p.gamma + i);
      if (ln) b4 = ld4(p.beta + i);
      if (p.post_w) w4 = ld4(p.post_w + i);
      if (p.sub) s4 = ld4(p.sub + static_cast<size_t>(b) * K + i);
      if (p.sub_part) {  // the producer's K splits in split order, then its epilogue
        float4 q[kMaxKs];
#pragma unroll
        for (int z = 0; z < kMaxKs; z++)
          if (z < p.sub_ks) q[z] = ld4(p.sub_part + (static_cast<size_t>(z) * p.batch + b) * K + i);
#pragma unroll
        for (int z = 0; z < kMaxKs; z++)
          if (z < p.sub_ks) {
            s4.x += q[z].x;
            s4.y += q[z].y;
            s4.z += q[z].z;
            s4.w += q[z].w;
          }
        if (p.sub_scale) {
          const float4 c = ld4(p.sub_scale + i);
          s4 = make_float4(s4.x * c.x, s4.y * c.y, s4.z * c.z, s4.w * c.w);
        }
        if (p.sub_bias) {
          const float4 c = ld4(p.sub_bias + i);
          s4 = make_float4(s4.x + c.x, s4.y + c.y, s4.z + c.z, s4.w + c.w);
        }
      }
    }
    t[j][0] = v.x, t[j][1] = v.y, t[j][2] = v.z, t[j][3] = v.w;
    su[j][0] = s4.x, su[j][1] = s4.y, su[j][2] = s4.z, su[j][3] = s4.w;
    pw[j][0] = w4.x, pw[j][1] = w4.y, pw[j][2] = w4.z, pw[j][3] = w4.w;
    g[j][0] = g4.x, g[j][1] = g4.y, g[j][2] = g4.z, g[j][3] = g4.w;
    be[j][0] = b4.x, be[j][1] = b4.y, be[j][2] = b4.z, be[j][3] = b4.w;
  }
  if (p.post_w) {  // Gemma's (1 + w) RMSNorm of the sublayer output
    float s2[1] = {0.f};
#pragma unroll
    for (int j = 0; j < NV; j++)
#pragma unroll
      for (int c = 0; c < 4; c++) s2[0] = __builtin_fmaf(su[j][c], su[j][c], s2[0]);
    gdev::block_sums<T / 64, 1>(s2, red, slot);
    const float inv = 1.0f / sqrtf(s2[0] / fk + p.eps);
#pragma unroll
    for (int j = 0; j < NV; j++)
#pragma unroll
      for (int c = 0; c < 4; c++) su[j][c] = su[j][c] * inv * (1.0f + pw[j][c]);
  }
  if (has_sub) {
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int i = static_cast<int>(threadIdx.x) + j * T;
#pragma unroll
      for (int c = 0; c < 4; c++) t[j][c] += su[j][c];
      if (p.res_out && i < K4)
        reinterpret_cast<float4 *>(p.res_out + static_cast<size_t>(b) * K)[i] =
            make_float4(t[j][0], t[j][1], t[j][2], t[j][3]);
    }
  }
  if (p.norm != XE_NORM_NONE) {
    float mean = 0.f;
    if (ln) {
      float s[1] = {0.f};
#pragma unroll
      for (int j = 0; j < NV; j++) s[0] += (t[j][0] + t[j][1]) + (t[j][2] + t[j][3]);
      gdev::block_sums<T / 64, 1>(s, red, slot);
      mean = s[0] / fk;
    }
    float s2[1] = {0.f};
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const bool on = static_cast<int>(threadIdx.x) + j * T < K4;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        t[j][c] -= mean;
        if (on) s2[0] = __builtin_fmaf(t[j][c], t[j][c], s2[0]);
      }
    }
    gdev::block_sums<T / 64, 1>(s2, red, slot);
    const float inv = 1.0f / sqrtf(s2[0] / fk + p.eps);
    const float one = p.norm == XE_NORM_RMS1P ? 1.0f : 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++)
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float h = t[j][c] * inv * (one + g[j][c]);
        t[j][c] = ln ? h + be[j][c] : h;
      }
  }
  if constexpr (P == 2) {
    // the largest |h|, and the smallest that is not zero (bits of 2 |h| less
    // one: zero comes last)
    float a = 0.f;
    uint32_t low = ~0u;
#pragma unroll
    for (int j = 0; j < NV; j++)
      if (static_cast<int>(threadIdx.x) + j * T < K4)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          a = fmaxf(a, fabsf(t[j][c]));
          low = min(low, 2u * __float_as_uint(t[j][c]) - 1u);
        }
    a = gdev::wave_max(a);
    float least = -gdev::wave_max(low != ~0u ? -__uint_as_float((low >> 1) + 1u) : -INFINITY);
    if ((threadIdx.x & 63) == 0) {
      mx[threadIdx.x >> 6] = a;
      mn[threadIdx.x >> 6] = least;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < T / 64; w++) {
      a = fmaxf(a, mx[w]);
      least = fminf(least, mn[w]);
    }
    int e = 0;
    if (a > 0.f && a < INFINITY) (void)frexpf(a, &e);  // a in [2^(e-1), 2^e)
    int s = 15 - e;
    least = __builtin_ldexpf(least, s);
    const bool raw = least < 0x1p-14f;
    const bool all = least < 0x1p-85f;  // more than x 2^s holds as well: every block as x itself
    if (all) s = 0;
    if (threadIdx.x == 0) rexp[b] = rexp_word(s, raw);
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int i = static_cast<int>(threadIdx.x) + j * T;
      if (i >= K4) continue;
      union {
        _Float16 h[4];
        u32x2 u;
      } hi, lo;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float v = __builtin_ldexpf(t[j][c], s);
        hi.h[c] = static_cast<_Float16>(v);
        lo.h[c] = static_cast<_Float16>((v - static_cast<float>(hi.h[c])) * static_cast<float>(1 << kLoExp));
      }
      if (raw) {  // a block is 16 lanes
        bool low4 = all;
#pragma unroll
        for (int c = 0; c < 4; c++) low4 |= t[j][c] != 0.f && fabsf(__builtin_ldexpf(t[j][c], s)) < 0x1p-14f;
        const bool blk = ((__ballot(low4) >> (threadIdx.x & 48)) & 0xffffu) != 0;
        if ((threadIdx.x & 15) == 0) raw_flags[raw_at(b, i / (kBK / 4), (K + kBK - 1) / kBK)] = blk;
        if (blk) {
          hi.u = u32x2{pack_hi16(t[j][0], t[j][1]), pack_hi16(t[j][2], t[j][3])};
          lo.u = u32x2{pack_lo16(t[j][0], t[j][1]), pack_lo16(t[j][2], t[j][3])};
        }
      }
      const size_t o = static_cast<size_t>(b) * K + 4 * i;
      *reinterpret_cast<u32x2 *>(planes + o) = hi.u;
      *reinterpret_cast<u32x2 *>(planes + static_cast<size_t>(p.batch) * K + o) = lo.u;
    }
  } else {
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int i = static_cast<int>(threadIdx.x) + j * T;
      if (i >= K4) continue;
      float r[4], l[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        r[c] = t[j][c] - trunc_bf16(t[j][c]);
        l[c] = r[c] - trunc_bf16(r[c]);
      }
      const size_t o = static_cast<size_t>(b) * K + 4 * i, pl = static_cast<size_t>(p.batch) * K;
      *reinterpret_cast<u32x2 *>(planes + o) = u32x2{pack_hi16(t[j][0], t[j][1]), pack_hi16(t[j][2], t[j][3])};
      *reinterpret_cast<u32x2 *>(planes + pl + o) = u32x2{pack_hi16(r[0], r[1]), pack_hi16(r[2], r[3])};
      *reinterpret_cast<u32x2 *>(planes + 2 * pl + o) = u32x2{pack_hi16(l[0], l[1]), pack_hi16(l[2], l[3])};
    }
  }
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------
struct WideParams {
  const void *w;
  const float *scale;
  const uint8_t *exps;
  const float *bias;
  int m, k, n;
  const uint16_t *planes;
  const int *rexp;
  const uint8_t *raw;
  int act;
  float *y;
  int ldy;
  uint16_t *pack;
  int pack_hd, pack_t;
  float *part;
  int spk;       // steps a split
  int vec;       // the output rows take 16-byte stores
  int tx, tw;    // row tiles, weight tiles
};

// gelu_tanh(x) = x / 2 (1 + tanh u) = x / (1 + exp(-2 u)): the same function
// without the cancellation of 1 + tanh u, and a tenth of tanhf's instructions
// (a big tile's 64 outputs a thread: 6 us of its epilogue).
__device__ __forceinline__ float gelu_tanh_wide(float x) {
  const float u2 = 2.0f * 0.79788456f * (x + 0.044715f * x * x * x);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * u2));
}

// LDS offset of the epilogue's tables (and of what says which steps run on
// fp32 rows): behind the operand buffers and the waves' output areas (which
// overlap).
constexpr int epi_offset(int buffers, int out) { return ((buffers > out ? buffers : out) + 15) / 16 * 16; }
constexpr int epi_tables(int bx, int bw) { return 4 * (bx + 2 * bw) + 48 + 2 * kMaxSteps; }

template <int WT>
struct WTraits {
  static constexpr int kRowB = WT == XE_BF16 ? 128 : WT == XE_I4 ? 32 : 64;  // LDS bytes of a row's 64 k
};

// LDS byte offset of 16-byte chunk c of row r: chunks XOR-permuted by the row
// so that the 8 rows read together by 8 lanes cover all banks (rows of 128,
// 64 and 32 bytes repeat their banks every 2, 4 and 8 rows).  The permutation
// has period 16 rows at most, so rows 16 apart differ by a constant, and
// chunk c ^ d of a row is at this offset ^ (d << 4): a lane needs one offset
// register and constants.
template <int ROWB>
__device__ __forceinline__ int lds_chunk(int r, int c) {
  if constexpr (ROWB == 128) return r * 128 + ((c ^ (r & 7)) << 4);
  else if constexpr (ROWB == 64) return r * 64 + ((c ^ ((r >> 2) & 3)) << 4);
  else return r * 32 + ((c ^ ((r >> 3) & 1)) << 4);
}

__device__ __forceinline__ uint32_t add_f16x2(uint32_t a, _Float16 c) {
  const f16x2 v = __builtin_bit_cast(f16x2, a) + f16x2{c, c};
  return __builtin_bit_cast(uint32_t, v);
}

// 8 int8 -> 8 fp16: q + 128 in the low byte of 0x6400 is 1024 + q + 128 in fp16
__device__ __forceinline__ f16x8 i8_to_f16(uint32_t q0, uint32_t q1) {
  q0 ^= 0x80808080u;
  q1 ^= 0x80808080u;
  const u32x4 o = {add_f16x2(__builtin_amdgcn_perm(0x64646464u, q0, 0x04010400u), static_cast<_Float16>(-1152.0f)),
                   add_f16x2(__builtin_amdgcn_perm(0x64646464u, q0, 0x04030402u), static_cast<_Float16>(-1152.0f)),
                   add_f16x2(__builtin_amdgcn_perm(0x64646464u, q1, 0x04010400u), static_cast<_Float16>(-1152.0f)),
                   add_f16x2(__builtin_amdgcn_perm(0x64646464u, q1, 0x04030402u), static_cast<_Float16>(-1152.0f))};
  return __builtin_bit_cast(f16x8, o);
}

// 8 int4 (k order, low nibble first) -> 8 fp16: n ^ 8 = n + 8 in 0..15
__device__ __forceinline__ f16x8 i4_to_f16(uint32_t q) {
  q ^= 0x88888888u;
  const uint32_t ev = q & 0x0f0f0f0fu, od = (q >> 4) & 0x0f0f0f0fu;
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) {  // byte i of ev, 0x64, byte i of od, 0x64
    const uint32_t sel = 0x0c000c00u | static_cast<uint32_t>(i) | (static_cast<uint32_t>(4 + i) << 16);
    o[i] = add_f16x2(__builtin_amdgcn_perm(od, ev, sel) | 0x64006400u, static_cast<_Float16>(-1032.0f));
  }
  return __builtin_bit_cast(f16x8, o);
}

// 8 bfp16 mantissas of one block with its exponent byte -> 8 bf16 (exact:
// at most 8 significant bits)
__device__ __forceinline__ bf16x8 bfp_to_bf16(uint32_t q0, uint32_t q1, uint32_t e) {
  const float s = __builtin_ldexpf(1.0f, static_cast<int>(e) - 133);
  float f[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    f[i] = static_cast<float>(static_cast<int>(__builtin_amdgcn_sbfe(static_cast<int>(q0), 8 * i, 8))) * s;
    f[4 + i] = static_cast<float>(static_cast<int>(__builtin_amdgcn_sbfe(static_cast<int>(q1), 8 * i, 8))) * s;
  }
  const u32x4 o = {pack_hi16(f[0], f[1]), pack_hi16(f[2], f[3]), pack_hi16(f[4], f[5]), pack_hi16(f[6], f[7])};
  return __builtin_bit_cast(bf16x8, o);
}

// The same numbers as bf16: 8 int8, 8 int4
__device__ __forceinline__ bf16x8 i8_to_bf16(uint32_t q0, uint32_t q1) {
  float f[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    f[i] = static_cast<float>(static_cast<int>(__builtin_amdgcn_sbfe(static_cast<int>(q0), 8 * i, 8)));
    f[4 + i] = static_cast<float>(static_cast<int>(__builtin_amdgcn_sbfe(static_cast<int>(q1), 8 * i, 8)));
  }
  const u32x4 o = {pack_hi16(f[0], f[1]), pack_hi16(f[2], f[3]), pack_hi16(f[4], f[5]), pack_hi16(f[6], f[7])};
  return __builtin_bit_cast(bf16x8, o);
}
__device__ __forceinline__ bf16x8 i4_to_bf16(uint32_t q) {
  float f[8];
#pragma unroll
  for (int i = 0; i < 8; i++) f[i] = static_cast<float>(static_cast<int>(__builtin_amdgcn_sbfe(static_cast<int>(q), 4 * i, 4)));
  const u32x4 o = {pack_hi16(f[0], f[1]), pack_hi16(f[2], f[3]), pack_hi16(f[4], f[5]), pack_hi16(f[6], f[7])};
  return __builtin_bit_cast(bf16x8, o);
}

// fp16 weights for the second part of the rows
__device__ __forceinline__ u32x4 lo_weights(u32x4 w) {
  const f16x8 v = __builtin_bit_cast(f16x8, w) * static_cast<_Float16>(1.0f / (1 << kLoExp));
  return __builtin_bit_cast(u32x4, v);
}

template <int WT>
__device__ __forceinline__ f32x16 mfma(u32x4 w, u32x4 x, f32x16 c) {
  if constexpr (WT == XE_I8 || WT == XE_I4)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
}

// Tile: 32 RX WXN rows x 32 RW WWN weight rows a workgroup of WXN x WWN waves
// (32 RX x 32 RW each), K in steps of 64.  Per step the row planes and the
// weights as stored go global -> registers -> LDS (two buffers, one barrier a
// step; the loads of NS steps are in flight), and come back as
// v_mfma_f32_32x32x16 operands: lane half h takes k 32 h .. + 31 of the step,
// 8 of them a MFMA, the same for rows and weights; weights convert to 16 bits
// after the LDS read.  The weight operand is A, so a lane's results are
// quads of neighbouring outputs of one row; the wave turns them through LDS
// and stores whole row segments, 16 bytes a lane (4-byte stores straight from
// the accumulators took 7 to 10 us of a 48 us launch at 13824 x 1152 x 512).
// Workgroups are numbered so that the row tiles of one weight tile run on one
// XCD, one after the other: its weights are read from HBM once.
template <int WT, int WXN, int WWN, int RX, int RW, int NS, int NB>
__global__ __launch_bounds__(64 * WXN * WWN) __attribute__((amdgpu_waves_per_eu(2))) void wide_gemm_kernel(WideParams p) {
  constexpr int T = 64 * WXN * WWN;
  constexpr int P = planes_of<WT>();
  constexpr int BX = 32 * RX * WXN, BW = 32 * RW * WWN;
  constexpr int ROWB = WTraits<WT>::kRowB;
  constexpr int XB = P * BX * 128, WB = BW * ROWB, EB = WT == XE_BFP16 ? BW * 8 : 0;
  constexpr int BUF = XB + WB + EB;
  constexpr int OS = 32 * RW + 4;                             // row stride (floats) of a wave's output area
  constexpr int OB = 32 * RX * OS * 4;                        // its bytes, over the operand buffers after the K loop
  constexpr int kTab = epi_tables(BX, BW);
  // the tables go in before the K loop where they fit behind its buffers
  constexpr bool kEarly = epi_offset(NB * BUF, WXN * WWN * OB) + kTab <= kLds;
  constexpr int kEpi = epi_offset(kEarly ? NB * BUF : 0, WXN * WWN * OB);
  constexpr int NX = P * BX * 8 / T;                          // 16-byte row chunks a thread
  constexpr int NW = (WT == XE_BF16 ? BW * 8 : BW * 4) / T;   // weight chunks a thread
  constexpr int PA = RX * RW == 1 ? P : 1;                    // accumulators a block (independent MFMA chains)
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  // XCD-aware order: blocks go to the XCDs round-robin
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int wt = (seq / p.tx) * 8 + xcd, xt = seq % p.tx;
  if (wt >= p.tw) return;
  const int n0 = xt * BX, m0 = wt * BW;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wx = wave % WXN, ww = wave / WXN;
  const int K = p.k;
  const int z = blockIdx.y;
  const int step0 = z * p.spk;
  const int nsteps = min((K + kBK - 1) / kBK, step0 + p.spk) - step0;
  const int kend = min(K, (step0 + nsteps) * kBK);
  const __amdgpu_buffer_rsrc_t rx = gdev::coherent_rsrc(p.planes);
  const __amdgpu_buffer_rsrc_t rw = gdev::coherent_rsrc(p.w);
  const __amdgpu_buffer_rsrc_t re = gdev::coherent_rsrc(WT == XE_BFP16 ? static_cast<const void *>(p.exps) : p.w);

  // row chunks: thread t takes chunk t % 8 of plane rows t / 8 + T / 8 j
  const int xc = threadIdx.x & 7, xr = threadIdx.x >> 3;
  int xoff[NX];  // rows past the end: out of range, loads return zeros
#pragma unroll
  for (int j = 0; j < NX; j++) {
    const int pr = xr + T / 8 * j, pl = pr / BX, r = pr % BX;
    xoff[j] = n0 + r < p.n ? ((pl * p.n + n0 + r) * K + 8 * xc) * 2 : kNoRec;
  }
  constexpr int CPR = WT == XE_BF16 ? 8 : 4;        // weight chunks a row
  constexpr int KPC = kBK / CPR;                    // k of a chunk
  constexpr int BPC = WT == XE_I4 ? 8 : 16;         // bytes of a chunk
  const int wc = threadIdx.x % CPR, wr = threadIdx.x / CPR;
  int woff[NW], eoff[NW];
#pragma unroll
  for (int j = 0; j < NW; j++) {
    const int r = m0 + wr + (T / CPR) * j;
    woff[j] = r < p.m ? r * (K / KPC) * BPC + wc * BPC : kNoRec;
    eoff[j] = r < p.m ? r * (K / 8) + 2 * wc : kNoRec;
  }
  struct Stage {
    u32x4 x[NX];
    u32x4 w[NW];
    uint32_t e[NW];
  };
  // tables behind the operand buffers: the rows' exponents, the weight rows'
  // scales and biases; a word a wave (fp32 blocks among its rows), the number
  // of steps without any, the steps in the order they are taken, their flags
  int *const rs = reinterpret_cast<int *>(lds + kEpi);
  float *const wsc = reinterpret_cast<float *>(rs + BX), *const wbi = wsc + BW;
  int *const seen = reinterpret_cast<int *>(wbi + BW);
  uint8_t *const order = reinterpret_cast<uint8_t *>(seen + 12), *const hit = order + kMaxSteps;
  int nfast = nsteps;  // steps without fp32 blocks: all in their order, or the first nfast of `order`
  auto issue_at = [&](int step, Stage &st) {  // past the last step: zeros
    const int k0 = (step0 + step) * kBK;
    const bool xok = k0 + 8 * xc < kend, wok = k0 + KPC * wc < kend;
#pragma unroll
    for (int j = 0; j < NX; j++)
      st.x[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, xok ? xoff[j] : kNoRec, 2 * k0, 0));
#pragma unroll
    for (int j = 0; j < NW; j++) {
      const int off = wok ? woff[j] : kNoRec;
      if constexpr (WT == XE_I4) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw, off, k0 / KPC * BPC, 0));
        st.w[j] = u32x4{v.x, v.y, 0u, 0u};
      } else {
        st.w[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, off, k0 / KPC * BPC, 0));
      }
      if constexpr (WT == XE_BFP16)
        st.e[j] = __builtin_amdgcn_raw_buffer_load_b16(re, wok ? eoff[j] : kNoRec, k0 / 8, 0);
    }
  };
  auto issue = [&](int step, Stage &st, auto sorted) {
    if constexpr (decltype(sorted)::value) step = step < nfast ? __builtin_amdgcn_readfirstlane(order[step]) : nsteps;
    issue_at(step, st);
  };
  const int xput = lds_chunk<128>(xr, xc);
  const int wput = WT == XE_I4 ? lds_chunk<32>(wr, wc >> 1) + 8 * (wc & 1) : lds_chunk<ROWB>(wr, wc);
  auto put_w = [&](uint8_t *ws, const Stage &st) {
    uint8_t *es = ws + WB;
#pragma unroll
    for (int j = 0; j < NW; j++) {
      uint8_t *d = ws + wput + (T / CPR) * j * ROWB;
      if constexpr (WT == XE_I4) *reinterpret_cast<u32x2 *>(d) = u32x2{st.w[j].x, st.w[j].y};
      else *reinterpret_cast<u32x4 *>(d) = st.w[j];
      if constexpr (WT == XE_BFP16)
        *reinterpret_cast<uint16_t *>(es + (wr + (T / CPR) * j) * 8 + 2 * wc) = static_cast<uint16_t>(st.e[j]);
    }
  };
  auto put = [&](int buf, const Stage &st) {
    uint8_t *xs = lds + buf;
#pragma unroll
    for (int j = 0; j < NX; j++) *reinterpret_cast<u32x4 *>(xs + xput + T / 8 * j * 128) = st.x[j];
    put_w(xs + XB, st);
  };

  f32x16 acc[RX][RW][PA];
#pragma unroll
  for (int a = 0; a < RX; a++)
#pragma unroll
    for (int b = 0; b < RW; b++)
#pragma unroll
      for (int q = 0; q < PA; q++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[a][b][q][i] = 0.f;

  const int lr = lane & 31, lh = lane >> 5;
  const int xget = lds_chunk<128>(wx * 32 * RX + lr, 4 * lh);
  const int wget = lds_chunk<ROWB>(ww * 32 * RW + lr, WT == XE_I4 ? lh : WT == XE_BF16 ? 4 * lh : 2 * lh);
  // this lane's 32 weights of a step, a block each (bf16: read with the rows)
  constexpr int QW = WT == XE_BF16 ? 1 : WT == XE_I4 ? 4 : 8;
  constexpr int QN = NB == 3 ? 2 : 1;
  uint32_t q[QN][RW][QW], ex[QN][RW];
  u32x4 wf[2][RW], xf[2][RX][P];
  auto rdq_at = [&](const uint8_t *ws, uint32_t(&qv)[RW][QW], uint32_t(&ev)[RW]) {
    const uint8_t *es = ws + WB;
    if constexpr (WT != XE_BF16)
#pragma unroll
      for (int b = 0; b < RW; b++) {
#pragma unroll
        for (int c = 0; c < QW / 4; c++) {
          const u32x4 v = *reinterpret_cast<const u32x4 *>(ws + (wget ^ (c << 4)) + 32 * b * ROWB);
          qv[b][4 * c] = v.x, qv[b][4 * c + 1] = v.y, qv[b][4 * c + 2] = v.z, qv[b][4 * c + 3] = v.w;
        }
        if constexpr (WT == XE_BFP16) ev[b] = *reinterpret_cast<const uint32_t *>(es + (ww * 32 * RW + 32 * b + lr) * 8 + 4 * lh);
      }
  };
  auto rdq = [&](int buf, uint32_t(&qv)[RW][QW], uint32_t(&ev)[RW]) { rdq_at(lds + buf + XB, qv, ev); };
  auto rdx = [&](int buf, int s, int d) {
    const uint8_t *xs = lds + buf, *ws = xs + XB;
#pragma unroll
    for (int a = 0; a < RX; a++)
#pragma unroll
      for (int pl = 0; pl < P; pl++)
        xf[d][a][pl] = *reinterpret_cast<const u32x4 *>(xs + (xget ^ (s << 4)) + (pl * BX + 32 * a) * 128);
    if constexpr (WT == XE_BF16)
#pragma unroll
      for (int b = 0; b < RW; b++) wf[d][b] = *reinterpret_cast<const u32x4 *>(ws + (wget ^ (s << 4)) + 32 * b * ROWB);
  };

  // The steps in which a row of the tile has an fp32 block: every row as x 2^s
  // in fp32 (which holds two parts exactly) and into three bf16 parts on its
  // way to LDS (one buffer, two barriers a step), three MFMAs a product.
  // Rare, so short code before speed: 13824 x 1152 x 512 rows, one call in a
  // row of calls, 75 us with every step here, 50 with none.
  auto raw_steps = [&](Stage &sj) {
    constexpr int XR = 3 * BX * 128;
    static_assert(P != 2 || XR + WB <= NB * BUF, "three row planes fit the operand buffers");
    uint8_t *const ws = lds + XR;
    const int steps = (K + kBK - 1) / kBK;
    auto at = [&](int i) { return i < nsteps ? __builtin_amdgcn_readfirstlane(order[i]) : nsteps; };
    int s1 = at(nfast);
    issue_at(s1, sj);
    for (int i1 = nfast; i1 < nsteps; i1++) {
#pragma unroll
      for (int j = 0; j < NX / 2; j++) {
        const int r = xr + T / 8 * j, rw = rs[r];
        const bool raw = n0 + r < p.n && rexp_raw(rw) && p.raw[raw_at(n0 + r, step0 + s1, steps)];
        const f16x8 hi = __builtin_bit_cast(f16x8, sj.x[j]), lo = __builtin_bit_cast(f16x8, sj.x[j + NX / 2]);
        float v[8], m[8], l[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const uint32_t h = sj.x[j][i / 2], g = sj.x[j + NX / 2][i / 2];
          const uint32_t w = i & 1 ? (h & 0xffff0000u) | g >> 16 : h << 16 | (g & 0xffffu);
          v[i] = raw ? __builtin_ldexpf(__uint_as_float(w), rexp_s(rw))
                     : static_cast<float>(hi[i]) + static_cast<float>(lo[i]) * (1.0f / (1 << kLoExp));
          m[i] = v[i] - trunc_bf16(v[i]);
          l[i] = m[i] - trunc_bf16(m[i]);
        }
        uint8_t *d = lds + xput + T / 8 * j * 128;
        *reinterpret_cast<u32x4 *>(d) = u32x4{pack_hi16(v[0], v[1]), pack_hi16(v[2], v[3]), pack_hi16(v[4], v[5]), pack_hi16(v[6], v[7])};
        *reinterpret_cast<u32x4 *>(d + BX * 128) = u32x4{pack_hi16(m[0], m[1]), pack_hi16(m[2], m[3]), pack_hi16(m[4], m[5]), pack_hi16(m[6], m[7])};
        *reinterpret_cast<u32x4 *>(d + 2 * BX * 128) = u32x4{pack_hi16(l[0], l[1]), pack_hi16(l[2], l[3]), pack_hi16(l[4], l[5]), pack_hi16(l[6], l[7])};
      }
      put_w(ws, sj);
      __syncthreads();
      s1 = at(i1 + 1);
      issue_at(s1, sj);
      rdq_at(ws, q[0], ex[0]);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        u32x4 w[RW];
#pragma unroll
        for (int b = 0; b < RW; b++)
          w[b] = __builtin_bit_cast(u32x4, WT == XE_I8 ? i8_to_bf16(q[0][b][(2 * s) % QW], q[0][b][(2 * s + 1) % QW]) : i4_to_bf16(q[0][b][s % QW]));
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
#pragma unroll
          for (int a = 0; a < RX; a++) {
            const u32x4 xv = *reinterpret_cast<const u32x4 *>(lds + (xget ^ (s << 4)) + (pl * BX + 32 * a) * 128);
#pragma unroll
            for (int b = 0; b < RW; b++) acc[a][b][0] = mfma<XE_BF16>(w[b], xv, acc[a][b][0]);
          }
      }
      __syncthreads();
    }
  };
  // Which steps those are: order, nfast.
  auto sort_steps = [&]() {
    const int steps = (K + kBK - 1) / kBK;
    for (int i = threadIdx.x; i < nsteps; i += T) hit[i] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < nsteps * BX; i += T) {
      const int r = i % BX, st = i / BX;
      if (n0 + r < p.n && rexp_raw(rs[r]) && p.raw[raw_at(n0 + r, step0 + st, steps)]) hit[st] = 1;
    }
    __syncthreads();
    if (wave == 0) {
      int fast = 0;
      for (int i0 = 0; i0 < nsteps; i0 += 64) {
        const bool on = i0 + lane < nsteps, raw = on && hit[i0 + lane];
        const uint64_t fm = __ballot(on && !raw), below = (uint64_t(1) << lane) - 1;
        const int before = fast + __popcll(fm & below);  // steps without fp32 blocks before this one
        if (on) order[raw ? nsteps - 1 - (i0 + lane - before) : before] = static_cast<uint8_t>(i0 + lane);
        fast += __popcll(fm);
      }
      if (lane == 0) seen[8] = fast;
    }
    __syncthreads();
    nfast = __builtin_amdgcn_readfirstlane(seen[8]);
  };

  // Step s.  The loads of step s + D (D = NB - 1) go from their registers to
  // the LDS buffer that step s - 1 freed, and those of step s + D + NS go out,
  // behind the first MFMAs.  The operands of the next k chunk are read before
  // a chunk's MFMAs; with three buffers the first chunk of step s + 1 too is
  // read before the barrier that ends step s (its buffer was complete a
  // barrier ago), so no MFMA waits behind a barrier and an LDS round trip
  // (1152 x 6912 x 512 rows, one split: 1.44 us a step with two buffers).
  constexpr int D = NB - 1;
  Stage st[NS];
  int bc = 0, bp = D * BUF;  // LDS offset of the buffer of this step and of the one being filled
  auto nxt = [&](int b) { return b + BUF == NB * BUF ? 0 : b + BUF; };
  auto step = [&](int j, int next_issue, auto more, auto sorted) {
    Stage &sj = st[(j + D) % NS];
    const int bn = nxt(bc);
    if constexpr (NB == 2) {
      rdq(bc, q[0], ex[0]);
      rdx(bc, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < 4; s++) {
      uint32_t(&qv)[RW][QW] = q[j % QN];
      if (s < 3) {
        rdx(bc, s + 1, (s + 1) & 1);
      } else if constexpr (NB == 3) {
        rdx(bn, 0, 0);
        rdq(bn, q[(j + 1) % QN], ex[(j + 1) % QN]);
      }
#pragma unroll
      for (int b = 0; b < RW; b++) {
        if constexpr (WT == XE_I8) wf[s & 1][b] = __builtin_bit_cast(u32x4, i8_to_f16(qv[b][2 * s], qv[b][2 * s + 1]));
        else if constexpr (WT == XE_I4) wf[s & 1][b] = __builtin_bit_cast(u32x4, i4_to_f16(qv[b][s]));
        else if constexpr (WT == XE_BFP16)
          wf[s & 1][b] = __builtin_bit_cast(u32x4, bfp_to_bf16(qv[b][2 * s], qv[b][2 * s + 1], (ex[j % QN][b] >> (8 * s)) & 0xffu));
      }
#pragma unroll
      for (int pl = 0; pl < P; pl++) {
        if constexpr (P == 2 && PA == 1)  // else the second part's sums are scaled at the end
          if (pl == 1)
#pragma unroll
            for (int b = 0; b < RW; b++) wf[s & 1][b] = lo_weights(wf[s & 1][b]);
#pragma unroll
        for (int a = 0; a < RX; a++)
#pragma unroll
          for (int b = 0; b < RW; b++)
            acc[a][b][pl % PA] = mfma<WT>(wf[s & 1][b], xf[s & 1][a][pl], acc[a][b][pl % PA]);
      }
      if (s == 0) {
        put(bp, sj);
        if constexpr (decltype(more)::value) issue(next_issue, sj, sorted);
      }
    }
    __syncthreads();
    bc = bn;
    bp = nxt(bp);
  };
#pragma unroll
  for (int j = 0; j < NS; j++) issue_at(j, st[j]);
  // what the epilogue needs, loaded behind the first operands
  int t_rs = 0;
  float t_sc = 1.0f, t_bi = 0.0f;
  if constexpr (P == 2) t_rs = p.rexp[n0 + threadIdx.x % BX];
  {
    const int m = min(m0 + static_cast<int>(threadIdx.x) % BW, p.m - 1);
    if constexpr (WT == XE_I8 || WT == XE_I4) t_sc = p.scale[m];
    if (p.bias) t_bi = p.bias[m];
  }
  auto put_tables = [&]() {
    if constexpr (P == 2) {
      static_assert(kEarly && T / 64 <= 8, "the row exponents are in LDS before the K loop");
      const bool mine = rexp_raw(t_rs) && n0 + static_cast<int>(threadIdx.x) % BX < p.n;
      const bool any = __any(mine);
      if (lane == 0) seen[wave] = any;
    }
    if (threadIdx.x < BX) rs[threadIdx.x] = t_rs;
    if (threadIdx.x < BW) {
      wsc[threadIdx.x] = t_sc;
      wbi[threadIdx.x] = t_bi;
    }
  };
  if constexpr (kEarly) put_tables();
  auto fill = [&](auto sorted) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      put(d * BUF, st[d % NS]);
      issue(d + NS, st[d % NS], sorted);
    }
    __syncthreads();
    if constexpr (NB == 3) {
      rdx(0, 0, 0);
      rdq(0, q[0], ex[0]);
    }
  };
  // whole groups of NS steps, so that every stage is a fixed set of
  // registers; the remainder's loads are in flight by then
  auto fast_steps = [&](auto sorted) {
    int s0 = 0;
    for (; s0 + NS <= nfast; s0 += NS) {
#pragma unroll
      for (int j = 0; j < NS; j++) step(j, s0 + j + D + NS, std::true_type{}, sorted);
    }
#pragma unroll
    for (int j = 0; j < NS - 1; j++)
      if (s0 + j < nfast) step(j, 0, std::false_type{}, sorted);
  };
  fill(std::false_type{});
  bool fp32 = false;
  if constexpr (P == 2) {
    int any = 0;
#pragma unroll
    for (int i = 0; i < T / 64; i++) any |= seen[i];
    fp32 = __builtin_amdgcn_readfirstlane(any) != 0;
  }
  if (!fp32) {
    fast_steps(std::false_type{});
  } else if constexpr (P == 2) {
    sort_steps();
#pragma unroll
    for (int j = 0; j < NS; j++) issue(j, st[j], std::true_type{});
    fill(std::true_type{});
    fast_steps(std::true_type{});
    raw_steps(st[0]);
  }

  // A lane's results: weight rows 8 (i / 4) + 4 (lane / 32) + i % 4 of row
  // lane % 32 of each block.  The epilogue in registers, then through the
  // wave's own LDS area (the operand buffers are free since the last barrier)
  // into stores along the rows.
  if constexpr (!kEarly) {
    put_tables();
    __syncthreads();
  }
  float *const out = reinterpret_cast<float *>(lds + wave * OB);
  const bool geglu = p.act == ACT_GEGLU_TANH && !p.part;
#pragma unroll
  for (int a = 0; a < RX; a++) {
    int sx = 0;
    if constexpr (P == 2) sx = -rexp_s(rs[wx * 32 * RX + 32 * a + lr]);
    float *const orow = out + (32 * a + lr) * OS;
#pragma unroll
    for (int b = 0; b < RW; b++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++) {
        const int ml = 32 * b + 8 * i4 + 4 * lh;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float t = acc[a][b][0][4 * i4 + i];
#pragma unroll
          for (int q = 1; q < PA; q++) t += P == 2 ? acc[a][b][q][4 * i4 + i] * (1.0f / (1 << kLoExp)) : acc[a][b][q][4 * i4 + i];
          if constexpr (P == 2) t = __builtin_ldexpf(t, sx);
          v[i] = t;
        }
        if (!p.part) {
          const f32x4 sc = *reinterpret_cast<const f32x4 *>(wsc + ww * 32 * RW + ml);
          const f32x4 bi = *reinterpret_cast<const f32x4 *>(wbi + ww * 32 * RW + ml);
#pragma unroll
          for (int i = 0; i < 4; i++) v[i] = v[i] * sc[i] + bi[i];
          if (p.act == ACT_RELU) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = v[i] > 0.f ? v[i] : 0.f;
          } else if (p.act == ACT_GELU_ERF) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = gdev::gelu_erf(v[i]);
          }
        }
        if (geglu)  // weight rows 2 r (gate) and 2 r + 1 (up)
          *reinterpret_cast<f32x2 *>(orow + ml / 2) = f32x2{gelu_tanh_wide(v[0]) * v[1], gelu_tanh_wide(v[2]) * v[3]};
        else
          *reinterpret_cast<f32x4 *>(orow + ml) = f32x4{v[0], v[1], v[2], v[3]};
      }
  }
  // the wave's rows: CQ quads each
  const int cq = geglu ? 4 * RW : 8 * RW, cols = geglu ? p.m / 2 : p.m;
  const int c0 = (m0 + ww * 32 * RW) / (geglu ? 2 : 1);
  const int ld = p.part ? p.m : p.ldy;
  float *const y = p.part ? p.part + static_cast<size_t>(z) * p.n * p.m : p.y;
  for (int id = lane; id < 32 * RX * cq; id += 64) {
    const int r = id / cq, c = 4 * (id % cq);
    const int n = n0 + wx * 32 * RX + r, m = c0 + c;
    if (n >= p.n || m >= cols) continue;
    const f32x4 v = *reinterpret_cast<const f32x4 *>(out + r * OS + c);
    if (p.pack && !p.part) {
      const uint32_t lo = adev::f32_to_bf16_rne(v.x) | static_cast<uint32_t>(adev::f32_to_bf16_rne(v.y)) << 16;
      const uint32_t hi = adev::f32_to_bf16_rne(v.z) | static_cast<uint32_t>(adev::f32_to_bf16_rne(v.w)) << 16;
      *reinterpret_cast<u32x2 *>(p.pack + (static_cast<size_t>(m / p.pack_hd) * p.pack_t + n) * p.pack_hd + m % p.pack_hd) = u32x2{lo, hi};
    } else if (p.vec) {
      *reinterpret_cast<f32x4 *>(y + static_cast<size_t>(n) * ld + m) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (m + i < cols) y[static_cast<size_t>(n) * ld + m + i] = v[i];
    }
  }
}

// The K splits' sums, in split order, through the epilogue.  Thread: four
// neighbouring outputs of a row (a weight count that is no multiple of four:
// one at a time).
template <int V>
__global__ __launch_bounds__(kT) void wide_finish_kernel(WideParams p, int ks, int scaled) {
  const int per = (p.m + V - 1) / V;
  const size_t total = static_cast<size_t>(p.n) * per;
  const size_t id = static_cast<size_t>(blockIdx.x) * kT + threadIdx.x;
  if (id >= total) return;
  const int n = static_cast<int>(id / per), m = static_cast<int>(id % per) * V;
  float q[kMaxKs][V], v[V] = {};
#pragma unroll
  for (int z = 0; z < kMaxKs; z++)
    if (z < ks) {
      const float *src = p.part + (static_cast<size_t>(z) * p.n + n) * p.m + m;
      if constexpr (V == 4) {
        const float4 t = ld4(src);
        q[z][0] = t.x, q[z][1] = t.y, q[z][2] = t.z, q[z][3] = t.w;
      } else {
        q[z][0] = src[0];
      }
    }
#pragma unroll
  for (int z = 0; z < kMaxKs; z++)
    if (z < ks)
#pragma unroll
      for (int i = 0; i < V; i++) v[i] += q[z][i];
#pragma unroll
  for (int i = 0; i < V; i++) {
    v[i] = v[i] * (scaled ? p.scale[m + i] : 1.0f) + (p.bias ? p.bias[m + i] : 0.0f);
    if (p.pack) {
      const int mm = m + i;
      p.pack[(static_cast<size_t>(mm / p.pack_hd) * p.pack_t + n) * p.pack_hd + mm % p.pack_hd] = adev::f32_to_bf16_rne(v[i]);
      continue;
    }
    if (p.act == ACT_GEGLU_TANH) continue;
    if (p.act == ACT_RELU) v[i] = v[i] > 0.f ? v[i] : 0.f;
    else if (p.act == ACT_GELU_ERF) v[i] = gdev::gelu_erf(v[i]);
    p.y[static_cast<size_t>(n) * p.ldy + m + i] = v[i];
  }
  if constexpr (V == 4)
    if (p.act == ACT_GEGLU_TANH) {
      p.y[static_cast<size_t>(n) * p.ldy + m / 2] = gelu_tanh_wide(v[0]) * v[1];
      p.y[static_cast<size_t>(n) * p.ldy + m / 2 + 1] = gelu_tanh_wide(v[2]) * v[3];
    }
}

// Tile and K split of a shape.
//   big    128 rows x 256 weight rows, 8 waves: half the operand bytes a MFMA
//          of the small tile; one workgroup a CU
//   small  64 x 64, 4 waves, loads of four steps in flight: shapes whose big
//          tiles leave CUs idle
// Cost in microseconds, fitted to launches over one dimension at a time (512
// rows, int8 / bf16 weights): a big tile's step takes 1.27 / 1.83 us (the
// matrix cores busy for two thirds of it) and its launch 6 us of latency; a
// small tile's 0.44 / 0.58 us, alone on its CU or 1.25 times that for each
// workgroup of it (three planes: measured with loads that spill); a K split
// writes and reads its partials at about 4 TB/s.
struct Shape {
  bool big;
  int ks, spk;
};
// us of a step: small tile (two planes, three), big tile
constexpr double kStepUs[2][2] = {{0.44, 0.58}, {1.27, 1.83}};
constexpr int kTileX[2] = {64, 128}, kTileW[2] = {64, 256};

Shape choose_shape(int m, int k, int n, int wdtype, size_t ws_floats, double *cost_us = nullptr) {
  const int steps = (k + kBK - 1) / kBK;
  const bool p2 = wide_planes(wdtype) == 2;
  Shape best{false, 1, steps};
  double best_cost = -1;
  for (int big = 0; big < 2; big++) {
    const long tiles = static_cast<long>((m + kTileW[big] - 1) / kTileW[big]) * ((n + kTileX[big] - 1) / kTileX[big]);
    const double step = kStepUs[big][p2 ? 0 : 1];
    for (int ks = 1; ks <= kMaxKs; ks++) {
      const int spk = (steps + ks - 1) / ks;
      if ((steps + spk - 1) / spk != ks) continue;
      if (ks > 1 && (spk < 4 || static_cast<size_t>(ks) * n * m > ws_floats)) continue;
      const double wgs = static_cast<double>(tiles) * ks / 256.0;
      double cost = big ? 6.0 + spk * step * std::ceil(wgs) : 3.0 + spk * step * std::max(1.0, 1.25 * wgs);
      if (ks > 1) cost += 3.0 + static_cast<double>(ks) * n * m * 2e-6;
      if (best_cost < 0 || cost < best_cost) {
        best_cost = cost;
        best = {big != 0, ks, spk};
      }
    }
  }
  if (cost_us) *cost_us = best_cost;
  return best;
}

// LDS buffers: three where they leave room (160 KB a CU; the small tile for
// two workgroups), so with two planes
constexpr int buffers(int wdtype) { return wdtype == XE_BF16 || wdtype == XE_BFP16 ? 2 : 3; }

using WideFn = void (*)(WideParams);
template <int WT>
WideFn pick(bool big) {
  return big ? wide_gemm_kernel<WT, 2, 4, 2, 2, 2, buffers(WT)> : wide_gemm_kernel<WT, 2, 2, 1, 1, 4, buffers(WT)>;
}

int lds_bytes(int wdtype, bool big) {
  const int bx = kTileX[big], bw = kTileW[big], rowb = wdtype == XE_BF16 ? 128 : wdtype == XE_I4 ? 32 : 64;
  const int bufs = buffers(wdtype) * (wide_planes(wdtype) * bx * 128 + bw * rowb + (wdtype == XE_BFP16 ? bw * 8 : 0));
  const int out = big ? 8 * 64 * 68 * 4 : 4 * 32 * 36 * 4;  // the waves' output areas
  const int early = epi_offset(bufs, out) + epi_tables(bx, bw);
  return early <= kLds ? early : std::max(bufs, epi_offset(0, out) + epi_tables(bx, bw));
}

template <int P>
void rows_launch(const gdev::GemvParams &p, const WideRows &rows, hipStream_t s) {
  // beyond 8 chunks a thread (200 registers) twice the threads
  const int nv = (p.k / 4 + kT - 1) / kT, threads = nv <= 8 ? kT : 2 * kT;
  auto fn = nv <= 1 ? wide_rows_kernel<1, P, kT> : nv <= 2 ? wide_rows_kernel<2, P, kT> : nv <= 4 ? wide_rows_kernel<4, P, kT>
            : nv <= 8 ? wide_rows_kernel<8, P, kT> : wide_rows_kernel<8, P, 2 * kT>;
  hipLaunchKernelGGL(fn, dim3(p.batch), dim3(threads), 0, s, p, rows.planes, rows.rexp, rows.raw);
  XE_HIP(hipGetLastError());
}

bool al16(const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }

}  // namespace

int wide_planes(int wdtype) { return wdtype == XE_I8 || wdtype == XE_I4 ? 2 : 3; }
size_t wide_plane_elems(int wdtype, int n, int k) { return static_cast<size_t>(wide_planes(wdtype)) * n * k; }
size_t wide_rexp_ints(int n) { return (static_cast<size_t>(n) + kRowPad - 1) / kRowPad * kRowPad; }
size_t wide_raw_ints(int n, int k) { return wide_rexp_ints(n) / 4 * ((k + kBK - 1) / kBK); }

bool wide_takes(int m, int k, int n, int wdtype, const void *x, int ldx) {
  if (wdtype != XE_I8 && wdtype != XE_I4 && wdtype != XE_BF16 && wdtype != XE_BFP16) return false;
  // 32-bit buffer offsets; the rows kernel's registers; 16-byte row loads
  return m > 0 && n > 0 && k > 0 && k % 16 == 0 && k <= kMaxK && ldx % 4 == 0 && al16(x) &&
         static_cast<size_t>(m) * k * (wdtype == XE_BF16 ? 2 : 1) < (size_t(1) << 31) - 4096 &&
         wide_plane_elems(wdtype, n + kRowPad, k) * 2 < (size_t(1) << 31);
}

// The rows kernel and its launch take about 6 us; the kernels of gemm.hip,
// which need no planes but split the rows in every weight tile, 8 us and 11.5
// us for every 1e9 multiply-adds (int8 and bf16 alike), after a prologue of 5
// us for a norm.  Measured here / there, us: int8 1152 x 1152 at 512 rows 18.5
// / 16.6, 3072 x 768 at 512 20.6 / 24.4, 4096 x 4096 at 200 37 / 40, 1152 x
// 6912 at 512 51 / 64, 13824 x 1152 at 512 49 / 107, 14336 x 4096 at 512 121 /
// 342; bf16 3072 x 768 at 512 28 / 23.5 (where the estimates are within 5 %
// the other kernels stay).
// Near that line both launches are looked at again, by their rounds: there
// gemm_est_us, here what the cost above leaves out.  Weight tiles run on XCD
// (tile) mod 8, 32 CUs each (bf16 2560 x 5120 at 384 rows, ten weight tiles, 8
// splits: 78 / 61), and a big tile's further round adds 8 us; a small tile's workgroups beyond one a CU come in whole
// ones (int8 5281 x 1152 at 192 after a norm 27.8 / 25.3); partials of a
// weight count that is no multiple of four are stored one by one (int8 3961 x
// 5952 at 128 48.8 / 45.0, 3960 of it 44.9 / 45.3); three planes on the small
// tile spill registers, at a cost that no such count tells (a fifth better by
// the estimate, or the other kernels stay: bf16 after a norm 3072 x 768 at 300
// 25.1 / 21.3).
// Products below 2^28 multiply-adds or of K < 512 stay too: both sides are
// launches, latency and outputs to store (bf16 after a norm: 8243 x 48 at 200
// rows 21.8 / 17.0, 3799 x 256 at 450 22.5 / 20.8).
// Of 826 measured products that the first line alone gives to these kernels 79
// were more than 4 % slower here; four are left (4566 x 9536, 8 to 15 %), and
// 30 others would gain 6 to 20 %.
bool wide_preferred(int m, int k, int n, int wdtype, bool prologue) {
  const double mac = static_cast<double>(m) * k * n;
  if (n <= 64 || k < 512 || mac < (1 << 28)) return false;  // one stream tile of gemm.hip, small products
  double us = 0;
  const Shape sh = choose_shape(m, k, n, wdtype, gemm_op_ws_floats(), &us);
  const double rows = 6.0 + 2e-6 * n * k;
  if (us + rows >= 0.95 * (8.0 + 11.5e-9 * mac + (prologue ? 5.0 : 0.0))) return false;
  const bool p2 = wide_planes(wdtype) == 2;
  const int tw = (m + kTileW[sh.big] - 1) / kTileW[sh.big], tx = (n + kTileX[sh.big] - 1) / kTileX[sh.big];
  const double rounds = std::ceil((tw + 7) / 8 * tx * sh.ks / 32.0), step = kStepUs[sh.big][p2 ? 0 : 1];
  double here = sh.big ? 6.0 + sh.spk * step * rounds + 8.0 * (rounds - 1)
                       : 3.0 + sh.spk * (rounds > 1 ? 1.25 * step * rounds : p2 ? step : step + 0.14);
  if (sh.ks > 1) here += 3.0 + static_cast<double>(sh.ks) * n * m * (m % 4 ? 3e-6 : 2e-6);
  here += rows;
  const double there = gemm_est_us(m, k, n) + (!prologue ? 0.0 : k > 4096 ? 2e-3 * k : 5.0);
  return here < (p2 || sh.big ? 1.0 : 0.8) * there;
}

int wide_splits(int m, int k, int n, int wdtype, size_t ws_floats) {
  return choose_shape(m, k, n, wdtype, ws_floats).ks;
}

bool wide_big_tile(int m, int k, int n, int wdtype, size_t ws_floats) {
  return choose_shape(m, k, n, wdtype, ws_floats).big;
}

void launch_wide_rows(const gdev::GemvParams &p, int wdtype, const WideRows &rows, hipStream_t s) {
  XE_REQUIRE(p.k % 16 == 0 && p.k <= kMaxK && p.batch > 0, "wide rows: unsupported shape");
  XE_REQUIRE(al16(p.x) && p.ldx % 4 == 0 && al16(p.sub) && al16(p.sub_part) && al16(p.post_w) && al16(p.res_out) &&
                 al16(p.gamma) && al16(p.beta) && al16(p.sub_scale) && al16(p.sub_bias) && al16(rows.planes),
             "wide rows: operands must be 16-byte aligned");
  XE_REQUIRE(!p.sub_part || (p.sub_ks >= 1 && p.sub_ks <= kMaxKs && p.sub_out_scale == 1.0f),
             "wide rows: too many split partials");
  if (wide_planes(wdtype) == 2) {
    XE_REQUIRE(rows.rexp && rows.raw, "wide rows: row exponents missing");
    rows_launch<2>(p, rows, s);
  } else {
    rows_launch<3>(p, rows, s);
  }
}

void launch_wide_gemm(const WideGemm &g, hipStream_t s) {
  XE_REQUIRE(wide_takes(g.m, g.k, g.n, g.wdtype, g.rows.planes, 0), "wide gemm: unsupported shape");
  XE_REQUIRE((g.wdtype != XE_I8 && g.wdtype != XE_I4) || (g.scale && g.rows.rexp && g.rows.raw), "wide gemm: int8/int4 weight without scales");
  XE_REQUIRE(g.wdtype != XE_BFP16 || g.exps, "wide gemm: bfp16 weight without exponents");
  XE_REQUIRE(g.act != ACT_GEGLU_TANH || (g.m % 4 == 0 && !g.pack), "wide gemm: GeGLU rows must pair within 4-row groups");
  XE_REQUIRE(!g.pack || (g.m % g.pack_hd == 0 && g.pack_hd % 4 == 0), "wide gemm: packed heads must hold whole quads");
  const size_t ws = g.part || g.ws ? g.ws_floats : 0;
  const Shape sh = choose_shape(g.m, g.k, g.n, g.wdtype, ws);
  XE_REQUIRE(!g.part || sh.ks > 1, "wide gemm: partials of an unsplit product");
  WideParams p{};
  p.w = g.w;
  p.scale = g.scale;
  p.exps = g.exps;
  p.bias = g.bias;
  p.m = g.m;
  p.k = g.k;
  p.n = g.n;
  p.planes = g.rows.planes;
  p.rexp = g.rows.rexp;
  p.raw = g.rows.raw;
  p.act = g.act;
  p.y = g.y;
  p.ldy = g.ldy;
  p.pack = g.pack;
  p.pack_hd = g.pack_hd;
  p.pack_t = g.pack_t;
  p.part = sh.ks > 1 ? (g.part ? g.part : g.ws) : nullptr;
  p.spk = sh.spk;
  const int cols = g.act == ACT_GEGLU_TANH && !p.part ? g.m / 2 : g.m;
  p.vec = cols % 4 == 0 && (p.part ? al16(p.part) : al16(g.y) && g.ldy % 4 == 0);
  p.tx = (g.n + kTileX[sh.big] - 1) / kTileX[sh.big];
  p.tw = (g.m + kTileW[sh.big] - 1) / kTileW[sh.big];
  WideFn fn = nullptr;
  switch (g.wdtype) {
    case XE_I8: fn = pick<XE_I8>(sh.big); break;
    case XE_I4: fn = pick<XE_I4>(sh.big); break;
    case XE_BF16: fn = pick<XE_BF16>(sh.big); break;
    default: fn = pick<XE_BFP16>(sh.big); break;
  }
  const int lds = lds_bytes(g.wdtype, sh.big);
  if (lds > 64 * 1024)
    XE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL(fn, dim3((p.tw + 7) / 8 * 8 * p.tx, sh.ks), dim3(sh.big ? 512 : 256), lds, s, p);
  XE_HIP(hipGetLastError());
  if (sh.ks > 1 && !g.part) {
    const int scaled = g.wdtype == XE_I8 || g.wdtype == XE_I4 ? 1 : 0;
    const bool v4 = g.m % 4 == 0;
    const size_t items = static_cast<size_t>(g.n) * (v4 ? g.m / 4 : g.m);
    const unsigned blocks = static_cast<unsigned>((items + kT - 1) / kT);
    if (v4) hipLaunchKernelGGL(wide_finish_kernel<4>, dim3(blocks), dim3(kT), 0, s, p, sh.ks, scaled);
    else hipLaunchKernelGGL(wide_finish_kernel<1>, dim3(blocks), dim3(kT), 0, s, p, sh.ks, scaled);
    XE_HIP(hipGetLastError());
  }
}

}  // namespace xe
