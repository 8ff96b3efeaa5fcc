// Entry point that only the native host path (gdn_host.cpp) binds; it is not
// part of the public C ABI.
#pragma once
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif
// b = x w_b^T and a = x w_a^T, the layer's two gate projections, in one pass
// over x (transformers modeling_qwen3_5_moe.py:426-427, called at :449-450):
//   x   [M, K] bf16, rows contiguous; K 1024 or 2048
//   w_b, w_a  [n, K] bf16 nn.Linear weights, rows contiguous; n 16 or 32
//   b, a      [M, n] bf16, rows contiguous
// All 16-byte aligned.
int gdn_gate_proj(const void *x, const void *w_b, const void *w_a, int32_t M, int32_t K, int32_t n, void *b, void *a,
                  void *stream);
#ifdef __cplusplus
}
#endif
