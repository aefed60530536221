// w8a8.hip -- W8A8 dynamic linear, every step on the GPU.
//
// The reference's int8 CtxAOp path (forward_view_int8,
// rust/npu-asr/src/ctx2.rs:771-830) quantises the activations on the host
// (quant_scale / quant_i8, :1352-1377), runs int8 x int8 -> i32 on the NPU
// and dequantises on the host (dequant_epi, :1386-1435); the host dequant is
// the cost it names (":145-149, int8 lost to bf16 on host dequant").  Here
// the four steps are kernels on one stream:
//
//   1. amax_partial_kernel   max|a| of grid-stride slices (exact: max is
//                            associative and NaN-ignoring like f32::max)
//   2. quant_kernel          every workgroup folds the partial maxima into
//                            scale_a = amax / 127 (1.0 for an all-zero
//                            tensor), then a_i8 = round-half-away(a /
//                            scale_a) clamped to +-127 (NaN -> 0, Rust's
//                            saturating cast)
//   3. the i32 product       <= 8 rows: the sdot4 GEMV (gemv.hip); more rows
//                            (the reference's batched tiles, Mp <= 512): an
//                            int8 MFMA GEMM over 64 x 64 tiles in LDS
//                            (v_mfma_i32_32x32x32_i8) or, for a few rows of a
//                            short K, one that loads its operands straight
//                            (v_mfma_i32_16x16x64_i8), exact integer
//                            accumulation
//   4. the epilogue          fused into the product: v = (acc * scale_a) *
//                            ws[c] (+ bias[c], or SiLU(v + bias[c]) with the
//                            reference's fast_sigmoid), in the reference's
//                            operation order; the build has no FMA
//                            contraction, so the result is the reference's
//                            bit for bit.
#include "gemv_dev.h"

namespace xe {
namespace {

constexpr int kT = 256;
constexpr int kAmaxBlocks = 256;    // one a CU; a quantising workgroup folds them one a thread
constexpr int kNoRec = 0x7ffffff0;  // past every buffer: loads return zeros

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float block_max(float v) {
  __shared__ float red[kT / 64];
  v = gdev::wave_max(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float m = red[0];
#pragma unroll
  for (int w = 1; w < kT / 64; w++) m = fmaxf(m, red[w]);
  return m;
}

// VEC: the activations are 16-byte aligned (their count is a multiple of
// four).  Four loads of a thread are in flight: both passes are bound by
// latency (512 x 768: 5.6 + 4.3 us with one 4-byte load at a time).
template <bool VEC>
__global__ __launch_bounds__(kT) void amax_partial_kernel(const float *__restrict__ a, size_t n,
                                                          float *__restrict__ partial) {
  constexpr int U = 4;
  float m = 0.f;
  const size_t stride = static_cast<size_t>(gridDim.x) * kT, n4 = VEC ? n / 4 : n;
  for (size_t i = static_cast<size_t>(blockIdx.x) * kT + threadIdx.x; i < n4; i += U * stride) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t j = i + u * stride;
      v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (j < n4) {
        if constexpr (VEC) v[u] = reinterpret_cast<const f32x4 *>(a)[j];
        else v[u].x = a[j];
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      m = fmaxf(m, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
  }
  m = block_max(m);
  if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

__device__ __forceinline__ int quant_one(float a, float sa) {
  float v = roundf(a / sa);
  if (v != v) v = 0.0f;
  v = v < -127.0f ? -127.0f : (v > 127.0f ? 127.0f : v);
  return static_cast<int>(v);
}

template <bool VEC>
__global__ __launch_bounds__(kT) void quant_kernel(const float *__restrict__ a, size_t n,
                                                   const float *__restrict__ partial,
                                                   int8_t *__restrict__ aq, float *__restrict__ scale_out) {
  static_assert(kAmaxBlocks == kT, "one partial maximum a thread");
  const size_t stride = static_cast<size_t>(gridDim.x) * kT, n4 = VEC ? n / 4 : n;
  const size_t i0 = static_cast<size_t>(blockIdx.x) * kT + threadIdx.x;
  f32x4 first = {0.f, 0.f, 0.f, 0.f};  // in flight beside the partial maxima
  if constexpr (VEC) {
    if (i0 < n4) first = reinterpret_cast<const f32x4 *>(a)[i0];
  } else {
    if (i0 < n4) first.x = a[i0];
  }
  const float amax = block_max(partial[threadIdx.x]);
  const float sa = amax > 0.0f ? amax / 127.0f : 1.0f;
  if (blockIdx.x == 0 && threadIdx.x == 0) scale_out[0] = sa;
  for (size_t i = i0; i < n4; i += stride) {
    f32x4 v = first;
    if constexpr (VEC) {
      if (i != i0) v = reinterpret_cast<const f32x4 *>(a)[i];
      const uint32_t q = (quant_one(v.x, sa) & 0xff) | (quant_one(v.y, sa) & 0xff) << 8 | (quant_one(v.z, sa) & 0xff) << 16 |
                         static_cast<uint32_t>(quant_one(v.w, sa)) << 24;
      reinterpret_cast<uint32_t *>(aq)[i] = q;
    } else {
      aq[i] = static_cast<int8_t>(quant_one(i == i0 ? v.x : a[i], sa));
    }
  }
}

// int8 tile GEMM: 64 activation rows x 64 weight rows a workgroup, four waves
// of 32 x 32 (v_mfma_i32_32x32x32_i8), K in steps of 128.  Operands as stored
// go global -> registers -> LDS by rows (16-byte chunks XOR-permuted by the
// row, two buffers, one barrier a step, loads of two steps in flight); a lane
// half takes the same 64 k of both operands, so the integer sums are exact
// whatever their order.  The weight operand is A: a lane's results are quads
// of neighbouring outputs of one row, dequantised in registers and turned
// through the wave's LDS area into 16-byte row stores (4-byte stores to 16
// rows at a time bound the kernel below: 25 us at 3072 x 768 x 512).
constexpr int kTB = 64, kTK = 128;

// us with the 16-row kernel / the tile kernel, quantisation included: 3072 x
// 768 at 16 rows 11.0 / 12.5, at 32 14.1 / 12.7, at 64 23 / 12.8, at 512 33 /
// 15.8; 300 x 256 at 32 11.0 / 11.4; 4096 x 1024 at 16 12.2 / 12.8; 2048 x
// 2048 at 16 16.4 / 15.0; 8192 x 4096 at 16 28 / 20, at 512 207 / 50.
bool tile_preferred(int k, int batch) { return batch > 32 || k >= (batch > 16 ? 512 : 1536); }
constexpr int kTS = 36;  // row stride (floats) of a wave's output area

__device__ __forceinline__ int tile_chunk(int r, int c) { return r * kTK + ((c ^ (r & 7)) << 4); }

__global__ __launch_bounds__(kT) void w8a8_tile_kernel(const int8_t *__restrict__ wq, const int8_t *__restrict__ aq,
                                                       int m, int k, int batch, int vec, W8a8Epi e) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][2][kTB * kTK];  // [buffer][activations, weights]
  static_assert(4 * 32 * kTS * 4 <= sizeof(lds), "the output areas fit the operand buffers");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wx = wave & 1, ww = wave >> 1, lr = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.x * kTB, b0 = blockIdx.y * kTB;
  const __amdgpu_buffer_rsrc_t rw = gdev::coherent_rsrc(wq);
  const __amdgpu_buffer_rsrc_t ra = gdev::coherent_rsrc(aq);
  // loads: thread t takes chunk t % 8 of rows t / 8 and t / 8 + 32
  const int xc = threadIdx.x & 7, xr = threadIdx.x >> 3;
  int xoff[2], woff[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int r = xr + 32 * j;
    xoff[j] = b0 + r < batch ? (b0 + r) * k + 16 * xc : kNoRec;
    woff[j] = m0 + r < m ? (m0 + r) * k + 16 * xc : kNoRec;
  }
  const int nsteps = (k + kTK - 1) / kTK;
  struct Stage {
    i32x4 x[2], w[2];
  } st[2];
  auto issue = [&](int step, Stage &s) {  // past the last step: zeros
    const int k0 = step * kTK;
    const bool ok = k0 + 16 * xc < k;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      s.x[j] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, ok ? xoff[j] : kNoRec, k0, 0));
      s.w[j] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, ok ? woff[j] : kNoRec, k0, 0));
    }
  };
  const int at = tile_chunk(xr, xc);
  auto put = [&](int buf, const Stage &s) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
      *reinterpret_cast<i32x4 *>(lds[buf][0] + at + 32 * j * kTK) = s.x[j];
      *reinterpret_cast<i32x4 *>(lds[buf][1] + at + 32 * j * kTK) = s.w[j];
    }
  };
  const int xget = tile_chunk(wx * 32 + lr, 4 * lh), wget = tile_chunk(ww * 32 + lr, 4 * lh);
  i32x16 acc[2];  // even and odd chunks: independent MFMA chains
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[q][i] = 0;
  // the epilogue's scales, in flight during the K loop
  float sc[4][4], bi[4][4];
  const float sa = e.acc ? 1.0f : e.scale_a[0];
#pragma unroll
  for (int i4 = 0; i4 < 4; i4++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = min(m0 + ww * 32 + 8 * i4 + 4 * lh + i, m - 1);
      sc[i4][i] = e.acc ? 1.0f : e.ws[r];
      bi[i4][i] = !e.acc && e.epi != EPI_NONE ? e.bias[r] : 0.0f;
    }
  auto step = [&](int j, int next) {
    put((j + 1) & 1, st[(j + 1) & 1]);
    issue(next, st[(j + 1) & 1]);
    i32x4 xv[4], wv[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      xv[s] = *reinterpret_cast<const i32x4 *>(lds[j & 1][0] + (xget ^ (s << 4)));
      wv[s] = *reinterpret_cast<const i32x4 *>(lds[j & 1][1] + (wget ^ (s << 4)));
    }
#pragma unroll
    for (int s = 0; s < 4; s++) acc[s & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wv[s], xv[s], acc[s & 1], 0, 0, 0);
    __syncthreads();
  };
  issue(0, st[0]);
  issue(1, st[1]);
  put(0, st[0]);
  issue(2, st[0]);
  __syncthreads();
  int s0 = 0;
  for (; s0 + 2 <= nsteps; s0 += 2) {
    step(0, s0 + 3);
    step(1, s0 + 4);
  }
  if (s0 < nsteps) step(0, s0 + 3);

  // a lane's results: weight rows 8 (i / 4) + 4 (lane / 32) + i % 4 of
  // activation row lane % 32
  uint32_t *const out = reinterpret_cast<uint32_t *>(&lds[0][0][0]) + wave * 32 * kTS;
#pragma unroll
  for (int i4 = 0; i4 < 4; i4++) {
    i32x4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int32_t a = acc[0][4 * i4 + i] + acc[1][4 * i4 + i];
      v[i] = e.acc ? a : __float_as_int(w8a8_value(e.epi, a, sa, sc[i4][i], bi[i4][i]));
    }
    *reinterpret_cast<i32x4 *>(out + lr * kTS + 8 * i4 + 4 * lh) = v;
  }
  uint32_t *const y = e.acc ? reinterpret_cast<uint32_t *>(e.acc) : reinterpret_cast<uint32_t *>(e.y);
#pragma unroll
  for (int id = lane; id < 32 * 8; id += 64) {
    const int r = id >> 3, c = 4 * (id & 7);
    const int b = b0 + wx * 32 + r, row = m0 + ww * 32 + c;
    if (b >= batch || row >= m) continue;
    const i32x4 v = *reinterpret_cast<const i32x4 *>(out + r * kTS + c);
    uint32_t *d = y + static_cast<size_t>(b) * m + row;
    if (vec) {
      *reinterpret_cast<i32x4 *>(d) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (row + i < m) d[i] = static_cast<uint32_t>(v[i]);
    }
  }
}

// int8 MFMA GEMM of a few rows: acc[b, r] = sum_k aq[b, k] * wq[r, k].  Workgroup: 4 waves
// x 16 weight rows, NJ blocks of 16 activation rows; K in steps of 64 (one
// v_mfma_i32_16x16x64_i8 per column block).  A lane loads 16 consecutive k of
// its weight row and of its activation row at the same k offset (both
// operands use the same k assignment, so the integer dot products are exact
// whatever order the instruction sums them in).  Rows past m / batch and k
// past K read zeros (buffer loads with an out-of-range offset).
template <int NJ>
__global__ __launch_bounds__(kT) void w8a8_mfma_kernel(const int8_t *__restrict__ wq, const int8_t *__restrict__ aq,
                                                       int m, int k, int batch, W8a8Epi e) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = blockIdx.x * 64 + wave * 16;
  const int b0 = blockIdx.y * 16 * NJ;
  const __amdgpu_buffer_rsrc_t rw = gdev::coherent_rsrc(wq);
  const __amdgpu_buffer_rsrc_t ra = gdev::coherent_rsrc(aq);
  const int row = r0 + (lane & 15);
  const int kl = 16 * (lane >> 4);
  const bool row_ok = row < m;
  int brow[NJ];
  bool b_ok[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    brow[j] = b0 + 16 * j + (lane & 15);
    b_ok[j] = brow[j] < batch;
  }
  i32x4 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) acc[j] = i32x4{0, 0, 0, 0};
  constexpr int U = 4;  // K steps whose loads are in flight together
  const int nsteps = (k + 63) / 64;
  for (int s0 = 0; s0 < nsteps; s0 += U) {
    i32x4 wa[U], xb[U][NJ];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kk = (s0 + u) * 64 + kl;
      const bool k_ok = kk < k;
      wa[u] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                            rw, (row_ok && k_ok) ? row * k + kk : kNoRec, 0, 2));
#pragma unroll
      for (int j = 0; j < NJ; j++)
        xb[u][j] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 ra, (b_ok[j] && k_ok) ? brow[j] * k + kk : kNoRec, 0, 0));
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
        acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[u], xb[u][j], acc[j], 0, 0, 0);
  }
  // lane holds weight rows r0 + 4 * (lane / 16) + i of activation row
  // b0 + 16 j + lane % 16
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int b = brow[j];
    if (b >= batch) continue;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = r0 + 4 * (lane >> 4) + i;
      if (r < m) w8a8_store(e, b, r, m, acc[j][i]);
    }
  }
}

}  // namespace

void launch_w8a8_quant(const float *a, size_t n, float *partial, int8_t *aq, float *scale_out,
                       hipStream_t s) {
  XE_REQUIRE(n > 0, "w8a8: empty activation tensor");
  const bool vec = n % 4 == 0 && (reinterpret_cast<uintptr_t>(a) & 15) == 0;
  hipLaunchKernelGGL(vec ? amax_partial_kernel<true> : amax_partial_kernel<false>, dim3(kAmaxBlocks), dim3(kT), 0, s, a, n,
                     partial);
  XE_HIP(hipGetLastError());
  const size_t blocks = std::min<size_t>(((vec ? n / 4 : n) + kT - 1) / kT, 8 * gdev::cu_count());
  hipLaunchKernelGGL(vec ? quant_kernel<true> : quant_kernel<false>, dim3(static_cast<unsigned>(blocks)), dim3(kT), 0, s, a,
                     n, partial, aq, scale_out);
  XE_HIP(hipGetLastError());
}

size_t w8a8_partial_floats() { return kAmaxBlocks; }

void launch_w8a8_mfma(const int8_t *wq, const int8_t *aq, int m, int k, int batch, const W8a8Epi &e,
                      hipStream_t s) {
  XE_REQUIRE(m > 0 && k > 0 && batch > 0, "w8a8 gemm: empty shape");
  XE_REQUIRE(k % 16 == 0, "w8a8 gemm: K must be a multiple of 16");
  XE_REQUIRE(static_cast<size_t>(m) * k < (size_t(1) << 31) && static_cast<size_t>(batch) * k < (size_t(1) << 31),
             "w8a8 gemm: operand above 2 GB");
  if (tile_preferred(k, batch)) {
    const void *y = e.acc ? static_cast<const void *>(e.acc) : e.y;
    const int vec = m % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    hipLaunchKernelGGL(w8a8_tile_kernel, dim3((m + kTB - 1) / kTB, (batch + kTB - 1) / kTB), dim3(kT), 0, s, wq, aq, m, k,
                       batch, vec, e);
    XE_HIP(hipGetLastError());
    return;
  }
  const int nj = batch <= 16 ? 1 : 2;
  const dim3 grid((m + 63) / 64, (batch + 16 * nj - 1) / (16 * nj));
  if (nj == 1) hipLaunchKernelGGL(w8a8_mfma_kernel<1>, grid, dim3(kT), 0, s, wq, aq, m, k, batch, e);
  else hipLaunchKernelGGL(w8a8_mfma_kernel<2>, grid, dim3(kT), 0, s, wq, aq, m, k, batch, e);
  XE_HIP(hipGetLastError());
}

}  // namespace xe
