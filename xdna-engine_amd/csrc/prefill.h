// prefill.h -- launch surface of the prompt kernels (prefill.hip): the
// per-head transforms and KV-cache append of many tokens, and causal (or
// cross) attention of many query rows over a bf16 KV cache.
#pragma once

#include "attn_dev.h"

namespace xe {

// Rows: row n = b * t_n + t is token t0 + t of stream b (t_n tokens a stream).
struct PromptAttn {
  float *qkv = nullptr;   // [rows][ldq]: q heads at 0 (transformed in place), k at k_off, v at v_off
  int ldq = 0, k_off = 0, v_off = 0;
  uint16_t *kc = nullptr, *vc = nullptr;  // bf16 [stream][hkv][max_ctx][hd]
  size_t kv_bstride = 0;
  int max_ctx = 0;
  int batch = 1, t_n = 1, t0 = 0;
  int hq = 1, hkv = 1, hd = 64;
  float scale = 1.0f;
  const float *q_norm_w = nullptr, *k_norm_w = nullptr;  // Gemma per-head RMSNorm (1 + w)
  float norm_eps = 1e-6f;
  const float *rope_cos = nullptr, *rope_sin = nullptr;
  int div_norm = 0;       // p = e / sum (OPT) instead of e * (1 / sum)
  int fixed_len = 0;      // > 0: every row attends keys [0, fixed_len) (cross attention), else keys [0, t0 + t]
  float *out = nullptr;   // [rows][ld_out]
  int ld_out = 0;
};

bool prompt_attn_takes(int hd, int group);
// q heads: norm + RoPE in place (Gemma); k, v rows into the cache as bf16.
void launch_prompt_append(const PromptAttn &a, hipStream_t s);
void launch_prompt_attn(const PromptAttn &a, hipStream_t s);
// dst[b] = src[b * t_n + t_n - 1] (rows of n floats): the last token's row of each stream.
void launch_last_rows(const float *src, float *dst, int batch, int t_n, int n, hipStream_t s);

}  // namespace xe
