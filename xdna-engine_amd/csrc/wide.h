// wide.h -- launch surface of the many-row linears (wide.hip): the norm /
// residual prologue that writes split 16-bit planes of the activation rows,
// and the MFMA GEMM that reads them.
#pragma once

#include "gemv_dev.h"

namespace xe {

// Rows as planes: x = sum of 16-bit parts, plane q of row r at
// planes[(q * n + r) * k + i].
//   int8 / int4 weights   2 fp16 parts of x * 2^s (s in rexp[r]: the power of
//                         two that puts the row's largest |x| in [2^14,
//                         2^15)), the second one times 2^12.  Blocks of 64
//                         elements, one of them not zero and below 2^-28 of
//                         that: the fp32 bits, upper and lower halves (raw
//                         says which blocks)
//   bf16 / bfp16 weights  3 bf16 parts of x, exactly
struct WideRows {
  uint16_t *planes = nullptr;
  int *rexp = nullptr;     // wide_rexp_ints(n) ints (int8 / int4 weights)
  uint8_t *raw = nullptr;  // wide_raw_ints(n, k) ints (int8 / int4 weights)
};
int wide_planes(int wdtype);
size_t wide_plane_elems(int wdtype, int n, int k);
size_t wide_rexp_ints(int n);
size_t wide_raw_ints(int n, int k);
// One buffer for all three: floats it takes, and its parts.
inline size_t wide_rows_floats(int wdtype, int n, int k) {
  return wide_rexp_ints(n) + wide_raw_ints(n, k) + (wide_plane_elems(wdtype, n, k) + 1) / 2;
}
inline WideRows wide_rows_in(float *buf, int n, int k) {
  WideRows r;
  r.rexp = reinterpret_cast<int *>(buf);
  r.raw = reinterpret_cast<uint8_t *>(buf + wide_rexp_ints(n));
  r.planes = reinterpret_cast<uint16_t *>(buf + wide_rexp_ints(n) + wide_raw_ints(n, k));
  return r;
}

// One linear over n rows whose planes are in `rows`.
struct WideGemm {
  int wdtype = XE_I8;
  const void *w = nullptr;
  const float *scale = nullptr;
  const uint8_t *exps = nullptr;
  const float *bias = nullptr;
  int m = 0, k = 0, n = 0;
  WideRows rows;
  int act = ACT_NONE;
  float *y = nullptr;
  int ldy = 0;
  // bf16 head-major output instead of y: [m / pack_hd][pack_t][pack_hd], row n
  // being position n (the Whisper cross K / V caches)
  uint16_t *pack = nullptr;
  int pack_hd = 0, pack_t = 0;
  // K split (wide_splits): raw sums of split z to part[(z * n + row) * m + r];
  // nothing else is written.  null: wide_gemm finishes them itself in ws.
  float *part = nullptr;
  // workspace of a K split the GEMM finishes itself, ws_floats floats
  float *ws = nullptr;
  size_t ws_floats = 0;
};

// Whether the shapes, sizes and alignments suit these kernels.
bool wide_takes(int m, int k, int n, int wdtype, const void *x, int ldx);
// Whether a linear of n rows over an m x k weight is faster here than on the
// kernels of gemm.hip (prologue: those need one too).
bool wide_preferred(int m, int k, int n, int wdtype, bool prologue);
// Microseconds of a product on the kernels of gemm.hip (their own shapes).
double gemm_est_us(int m, int k, int n);
// K splits wide_gemm takes for a shape, with at most ws_floats floats of partials.
int wide_splits(int m, int k, int n, int wdtype, size_t ws_floats);
// Whether its tiles are the 128 x 256 ones (else 64 x 64).
bool wide_big_tile(int m, int k, int n, int wdtype, size_t ws_floats);
// x (+ sub, post norm, norm) of n rows -> planes; the fields x, x_bf16, ldx,
// batch, k, sub, sub_part .., post_w, res_out, norm, gamma, beta, eps of p.
void launch_wide_rows(const gdev::GemvParams &p, int wdtype, const WideRows &rows, hipStream_t s);
void launch_wide_gemm(const WideGemm &g, hipStream_t s);

}  // namespace xe
