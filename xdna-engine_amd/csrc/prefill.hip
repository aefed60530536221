// prefill.hip -- attention of a prompt: many query rows over the bf16 KV
// cache at once, instead of one query per step (attn_dev.h).
//
// The reference feeds a prompt token by token (opt125m_decode.rs:296-315,
// whisper.rs:344-389); the results are the same with every token of the
// prompt in one pass, since a token's keys and values depend on earlier
// tokens alone.
//
// Arithmetic as in the single-query kernel: fp32 queries, bf16 keys and
// values, fp32 scores, online softmax in the log2 domain, fp32 sums.  On the
// matrix cores fp32 operands are three bf16 parts, exactly (q, and the
// probabilities), against the bf16 cache rows as stored.
#include "prefill.h"

namespace xe {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;
constexpr int kTile = 64;  // keys a tile

__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ float trunc_bf16(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }

// v = sum of three bf16 parts, exactly (truncation: 8 significant bits each).
__device__ __forceinline__ void split3(const float (&v)[8], bf16x8 (&o)[3]) {
  float r[8], l[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    r[i] = v[i] - trunc_bf16(v[i]);
    l[i] = r[i] - trunc_bf16(r[i]);
  }
  o[0] = __builtin_bit_cast(bf16x8, u32x4{pack_hi16(v[0], v[1]), pack_hi16(v[2], v[3]), pack_hi16(v[4], v[5]), pack_hi16(v[6], v[7])});
  o[1] = __builtin_bit_cast(bf16x8, u32x4{pack_hi16(r[0], r[1]), pack_hi16(r[2], r[3]), pack_hi16(r[4], r[5]), pack_hi16(r[6], r[7])});
  o[2] = __builtin_bit_cast(bf16x8, u32x4{pack_hi16(l[0], l[1]), pack_hi16(l[2], l[3]), pack_hi16(l[4], l[5]), pack_hi16(l[6], l[7])});
}

// One wave a (row, head): q heads first, then k, then v heads.
template <int HD>
__global__ __launch_bounds__(kT) void prompt_append_kernel(PromptAttn a, adev::AttnParams tp, int heads, int first) {
  __shared__ float kt[kT / 64][HD];  // a wave's transformed key
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int id = blockIdx.x * (kT / 64) + wave;
  const int n = id / heads, h = first + id % heads;
  if (n >= a.batch * a.t_n) return;
  const int b = n / a.t_n, posi = a.t0 + n % a.t_n;
  float *row = a.qkv + static_cast<size_t>(n) * a.ldq;
  if (h < a.hq) {
    float *q = row + h * HD;
    adev::head_transform<HD, false>(tp, q, q, a.q_norm_w, posi);
    return;
  }
  const bool is_k = h < a.hq + a.hkv;
  const int kvh = is_k ? h - a.hq : h - a.hq - a.hkv;
  const float *src = row + (is_k ? a.k_off : a.v_off) + kvh * HD;
  float v[HD / 64];
  if (is_k && (a.k_norm_w || a.rope_cos)) {
    adev::head_transform<HD, false>(tp, src, kt[wave], a.k_norm_w, posi);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < HD / 64; i++) v[i] = kt[wave][lane + 64 * i];
  } else {
#pragma unroll
    for (int i = 0; i < HD / 64; i++) v[i] = src[lane + 64 * i];
  }
  uint16_t *dst = (is_k ? a.kc : a.vc) + a.kv_bstride * b + (static_cast<size_t>(kvh) * a.max_ctx + posi) * HD;
#pragma unroll
  for (int i = 0; i < HD / 64; i++) dst[lane + 64 * i] = adev::f32_to_bf16_rne(v[i]);
}

// 16-byte chunk c of row r in a tile of NC chunks a row, permuted so that 8
// rows read together cover all banks (K: rows are keys; V: rows are dims,
// written eight apart by neighbouring lanes, so the row's eights take part).
template <int NC>
__device__ __forceinline__ int k_chunk(int r, int c) { return (r * NC + (c ^ (r & 7))) * 16; }
__device__ __forceinline__ int v_chunk(int r, int c) { return r * 128 + ((c ^ (r & 7) ^ ((r >> 3) & 7)) << 4); }

// A workgroup takes 16 QW query rows of one (stream, kv head) -- the G heads
// of a GQA group are rows of the same tile, token by token -- and walks the
// keys in tiles of 64; KW waves share a tile's keys (KW = 1: each wave its
// own 16 rows and all 64 keys; KW = 2: half the rows a workgroup, so twice
// the workgroups when the rows are few, merged at the end).
// Scores come out transposed (S^T = K Q^T, v_mfma_f32_16x16x32_bf16, K rows
// as A), so a lane holds keys 4 g + i of its query row n = lane % 16, g =
// lane / 16: exactly the B operand of O^T = V^T P^T with the k slots of lane
// group g read as keys 4 g .. + 3 of two 16-key blocks, and the
// probabilities never leave their lane.  V is transposed while it is staged,
// its keys in that slot order.  The next tile's rows are loaded to registers
// while a tile computes.
template <int HD, int KW>
__global__ __launch_bounds__(kT) void prompt_attn_kernel(PromptAttn a, int G) {
  constexpr int QW = 4 / KW;
  constexpr int NC = HD / 8;               // 16-byte chunks of a key row
  constexpr int KL = kTile * NC / kT;      // K chunks a thread
  constexpr int VI = (kTile / 4) * NC;     // V items: 4 keys x 8 dims
  constexpr int VL = (VI + kT - 1) / kT;   // V items a thread (HD 64: half the threads)
  constexpr int NBK = 4 / KW;              // 16-key blocks a wave
  constexpr int HB = HD / 16, HC = HD / 32;
  __shared__ __attribute__((aligned(16))) uint8_t ks[kTile * HD * 2];
  __shared__ __attribute__((aligned(16))) uint8_t vs[kTile * HD * 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int qw = wave % QW, kw = wave / QW;
  const int ln = lane & 15, lg = lane >> 4;
  const int rows = a.t_n * G;
  const int kvh = blockIdx.y, b = blockIdx.z;
  const int r0 = blockIdx.x * 16 * QW;
  const int r = r0 + 16 * qw + ln;         // this lane's query row of the (stream, kv head)
  const int rc = min(r, rows - 1);
  const int t = rc / G, g = rc % G;
  const int lim = a.fixed_len > 0 ? a.fixed_len - 1 : a.t0 + t;  // last key it attends
  const int kmax = a.fixed_len > 0 ? a.fixed_len - 1 : a.t0 + min(r0 + 16 * QW - 1, rows - 1) / G;
  const uint16_t *kb = a.kc + a.kv_bstride * b + static_cast<size_t>(kvh) * a.max_ctx * HD;
  const uint16_t *vb = a.vc + a.kv_bstride * b + static_cast<size_t>(kvh) * a.max_ctx * HD;

  u32x4 kr[KL], vr[VL][4];
  auto load = [&](int tile) {  // rows past the last key: that key's (masked or never used)
#pragma unroll
    for (int i = 0; i < KL; i++) {
      const int id = threadIdx.x + i * kT, key = min(tile * kTile + id / NC, kmax);
      kr[i] = *reinterpret_cast<const u32x4 *>(kb + static_cast<size_t>(key) * HD + (id % NC) * 8);
    }
#pragma unroll
    for (int i = 0; i < VL; i++) {
      const int id = threadIdx.x + i * kT;
      if (VI % kT != 0 && id >= VI) continue;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int key = min(tile * kTile + 4 * (id / NC) + j, kmax);
        vr[i][j] = *reinterpret_cast<const u32x4 *>(vb + static_cast<size_t>(key) * HD + (id % NC) * 8);
      }
    }
  };
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < KL; i++) {
      const int id = threadIdx.x + i * kT;
      *reinterpret_cast<u32x4 *>(ks + k_chunk<NC>(id / NC, id % NC)) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VL; i++) {
      const int id = threadIdx.x + i * kT;
      if (VI % kT != 0 && id >= VI) continue;
      // keys 4 kq .. + 3: 32-key half kq / 8, block (kq / 4) % 2, lane group kq % 4
      const int kq = id / NC, hc = id % NC;
      const int c = (kq >> 3) * 4 + (kq & 3), half = (kq >> 2) & 1;
#pragma unroll
      for (int e = 0; e < 8; e++) {  // dim 8 hc + e of the four keys
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
        const u32x2 o = {__builtin_amdgcn_perm(vr[i][1][e >> 1], vr[i][0][e >> 1], sel),
                         __builtin_amdgcn_perm(vr[i][3][e >> 1], vr[i][2][e >> 1], sel)};
        *reinterpret_cast<u32x2 *>(vs + v_chunk(8 * hc + e, c) + 8 * half) = o;
      }
    }
  };
  load(0);

  // the query row's parts: dims 32 c + 8 lg .. + 7
  bf16x8 qf[HC][3];
  const float *q = a.qkv + static_cast<size_t>(b * a.t_n + t) * a.ldq + (kvh * G + g) * HD;
#pragma unroll
  for (int c = 0; c < HC; c++) {
    const f32x4 x0 = *reinterpret_cast<const f32x4 *>(q + 32 * c + 8 * lg);
    const f32x4 x1 = *reinterpret_cast<const f32x4 *>(q + 32 * c + 8 * lg + 4);
    const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    split3(v, qf[c]);
  }
  f32x4 o[HB];
#pragma unroll
  for (int i = 0; i < HB; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float sc2 = a.scale * adev::kLog2e;
  const int tiles = kmax / kTile + 1;
  for (int tile = 0; tile < tiles; tile++) {
    put();
    __syncthreads();
    if (tile + 1 < tiles) load(tile + 1);
    // scores of this wave's key blocks
    f32x4 s[NBK];
#pragma unroll
    for (int k = 0; k < NBK; k++) s[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < HC; c++) {
      bf16x8 kf[NBK];
#pragma unroll
      for (int k = 0; k < NBK; k++)
        kf[k] = *reinterpret_cast<const bf16x8 *>(ks + k_chunk<NC>(16 * (kw * NBK + k) + ln, 4 * c + lg));
#pragma unroll
      for (int p = 0; p < 3; p++)
#pragma unroll
        for (int k = 0; k < NBK; k++) s[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[k], qf[c][p], s[k], 0, 0, 0);
    }
    float mb = m;
#pragma unroll
    for (int k = 0; k < NBK; k++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int key = tile * kTile + 16 * (kw * NBK + k) + 4 * lg + i;
        s[k][i] = key <= lim ? s[k][i] * sc2 : -INFINITY;
        mb = fmaxf(mb, s[k][i]);
      }
    mb = fmaxf(mb, __shfl_xor(mb, 16, 64));
    mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
    const float mu = mb == -INFINITY ? 0.f : mb;  // no key yet: every weight below is exp2(-inf) = 0
    const float corr = __builtin_amdgcn_exp2f(m - mu);
    m = mb;
    l *= corr;
#pragma unroll
    for (int i = 0; i < HB; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) o[i][j] *= corr;
#pragma unroll
    for (int c = 0; c < NBK / 2; c++) {
      float pv[8];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        pv[i] = __builtin_amdgcn_exp2f(s[2 * c][i] - mu);
        pv[4 + i] = __builtin_amdgcn_exp2f(s[2 * c + 1][i] - mu);
      }
#pragma unroll
      for (int i = 0; i < 8; i++) l += pv[i];
      bf16x8 pf[3];
      split3(pv, pf);
      const int vc = (kw * NBK / 2 + c) * 4 + lg;
#pragma unroll
      for (int i0 = 0; i0 < HB; i0 += 4) {
        bf16x8 vf[4];
#pragma unroll
        for (int i = 0; i < 4; i++) vf[i] = *reinterpret_cast<const bf16x8 *>(vs + v_chunk(16 * (i0 + i) + ln, vc));
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            o[i0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[i], pf[p], o[i0 + i], 0, 0, 0);
      }
    }
    __syncthreads();  // the tile is read before the next one is put
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  if constexpr (KW == 2) {  // the upper key half's wave hands (m, l, O) to the lower's
    static_assert(2 * 64 * 2 * HB * 4 + 2 * 2 * 64 * 4 <= kTile * HD * 2, "the merge area fits the staged tiles");
    float *ob = reinterpret_cast<float *>(ks) + qw * 64 * (2 * HB);  // half of O at a time in each tile's area
    float *ob2 = reinterpret_cast<float *>(vs) + qw * 64 * (2 * HB);
    float(*ml)[2][64] = reinterpret_cast<float(*)[2][64]>(ks + 2 * 64 * 2 * HB * 4);
    if (kw == 1) {
      ml[qw][0][lane] = m;
      ml[qw][1][lane] = l;
#pragma unroll
      for (int i = 0; i < HB; i++)
        *reinterpret_cast<f32x4 *>((i < HB / 2 ? ob : ob2) + ((i % (HB / 2)) * 64 + lane) * 4) = o[i];
    }
    __syncthreads();
    if (kw == 1) return;
    const float m1 = ml[qw][0][lane], l1 = ml[qw][1][lane];
    const float mx = fmaxf(m, m1);  // key 0 is every row's: m is finite
    const float f0 = __builtin_amdgcn_exp2f(m - mx), f1 = __builtin_amdgcn_exp2f(m1 - mx);
    l = l * f0 + l1 * f1;
#pragma unroll
    for (int i = 0; i < HB; i++) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>((i < HB / 2 ? ob : ob2) + ((i % (HB / 2)) * 64 + lane) * 4);
#pragma unroll
      for (int j = 0; j < 4; j++) o[i][j] = o[i][j] * f0 + v[j] * f1;
    }
  }
  if (r >= rows) return;
  const float inv = 1.0f / l;
  float *dst = a.out + static_cast<size_t>(b * a.t_n + t) * a.ld_out + (kvh * G + g) * HD + 4 * lg;
#pragma unroll
  for (int i = 0; i < HB; i++) {
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = a.div_norm ? o[i][j] / l : o[i][j] * inv;
    *reinterpret_cast<f32x4 *>(dst + 16 * i) = v;
  }
}

__global__ __launch_bounds__(kT) void last_rows_kernel(const float *src, float *dst, int t_n, int n) {
  const int b = blockIdx.y, i = blockIdx.x * kT + threadIdx.x;
  if (i < n) dst[static_cast<size_t>(b) * n + i] = src[(static_cast<size_t>(b) * t_n + t_n - 1) * n + i];
}

}  // namespace

bool prompt_attn_takes(int hd, int group) {
  return (hd == 64 || hd == 128 || hd == 256) && group >= 1 && group <= 8;
}

void launch_prompt_append(const PromptAttn &a, hipStream_t s) {
  XE_REQUIRE(prompt_attn_takes(a.hd, a.hq / a.hkv), "prompt attention: unsupported head size");
  XE_REQUIRE(a.t0 >= 0 && a.t_n >= 1 && a.t0 + a.t_n <= a.max_ctx, "prompt attention: positions past the cache");
  adev::AttnParams tp{};
  tp.norm_eps = a.norm_eps;
  tp.rope_cos = a.rope_cos;
  tp.rope_sin = a.rope_sin;
  const int first = a.q_norm_w || a.rope_cos ? 0 : a.hq;  // q heads need no transform: k and v only
  const int heads = a.hq + 2 * a.hkv - first;
  const unsigned blocks = (static_cast<unsigned>(a.batch) * a.t_n * heads + kT / 64 - 1) / (kT / 64);
  auto fn = a.hd == 64 ? prompt_append_kernel<64> : a.hd == 128 ? prompt_append_kernel<128> : prompt_append_kernel<256>;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(kT), 0, s, a, tp, heads, first);
  XE_HIP(hipGetLastError());
}

void launch_prompt_attn(const PromptAttn &a, hipStream_t s) {
  const int G = a.hq / a.hkv;
  XE_REQUIRE(prompt_attn_takes(a.hd, G) && a.hq == G * a.hkv, "prompt attention: unsupported head size");
  XE_REQUIRE(a.fixed_len <= a.max_ctx && (a.fixed_len > 0 || a.t0 + a.t_n <= a.max_ctx), "prompt attention: keys past the cache");
  const int rows = a.t_n * G;
  // 64 rows a workgroup once those cover the chip, else 32
  const bool wide = static_cast<long>((rows + 63) / 64) * a.hkv * a.batch >= 256;
  const int br = wide ? 64 : 32;
  const dim3 grid((rows + br - 1) / br, a.hkv, a.batch);
  auto fn = a.hd == 64    ? (wide ? prompt_attn_kernel<64, 1> : prompt_attn_kernel<64, 2>)
            : a.hd == 128 ? (wide ? prompt_attn_kernel<128, 1> : prompt_attn_kernel<128, 2>)
                          : (wide ? prompt_attn_kernel<256, 1> : prompt_attn_kernel<256, 2>);
  hipLaunchKernelGGL(fn, grid, dim3(kT), 0, s, a, G);
  XE_HIP(hipGetLastError());
}

void launch_last_rows(const float *src, float *dst, int batch, int t_n, int n, hipStream_t s) {
  hipLaunchKernelGGL(last_rows_kernel, dim3((n + kT - 1) / kT, batch), dim3(kT), 0, s, src, dst, t_n, n);
  XE_HIP(hipGetLastError());
}

}  // namespace xe
