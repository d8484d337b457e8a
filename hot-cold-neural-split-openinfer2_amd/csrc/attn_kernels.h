// Argument blocks shared by the attention sources: the single-token kernels
// (attention.hip) and the prompt kernels (attn_prompt.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace oi2 {

constexpr int kHeadDim = 128;                 // head_dim (engine.py:72: hidden / n_q)

// RoPE of the pair (x1, x2) at angle table entries (c, s), all fp16
// (engine.py:150-157: cat(x1 cos - x2 sin, x1 sin + x2 cos) as fp16 ops).  Each
// sum takes its sine product rounded to fp16 and its cosine product exact, and
// is rounded once.  Every projection kernel uses this one form, so that a token
// gets the same q and k whichever of them a call's row count picks; written
// out with fma, because left to contraction the kernels could differ.
struct RopePair {
  _Float16 a, b;
};
__device__ __forceinline__ RopePair rope_f16(_Float16 x1, _Float16 x2, _Float16 c, _Float16 s) {
  return {__builtin_elementwise_fma(x1, c, -(x2 * s)), __builtin_elementwise_fma(x2, c, x1 * s)};
}

// Rows of x times weight blocks of 128 rows (one head each): q / k / v with
// RoPE, q to a buffer and k, v into the cache (mode 0), or o_proj (mode 1).
struct ProjArgs {
  const uint16_t* x;          // this launch's input rows (rows, H) fp16
  int rows, row0;             // their number, at most kProjMaxRows, and the first one's index in the call
  const uint8_t* w0;          // weight blocks of 128 rows (.., H), fp8 e4m3fn
  const uint8_t* w1;
  const uint8_t* w2;
  int blocks0, blocks1;       // 128-row blocks in w0 and w1; the rest are w2's
  int mode;
  // mode 0: what follows is the whole call's
  uint16_t* q;                // (rows, n_q * 128)
  int q_width;                // n_q * 128
  uint16_t* k_cache;
  uint16_t* v_cache;
  int n_kv, cap, past, seq;
  const float* cos;           // (seq, 64)
  const float* sin;
  uint32_t* counters;         // n_counters words that the launch clears
  int n_counters;
  // mode 1
  uint16_t* out;              // (rows, H)
  const uint16_t* residual;   // (rows, H) or null
  uint16_t* x_out;
};

constexpr int kProjMaxRows = 0x7FFFFFFF / (2 * 4096) / 128 * 128;   // 32-bit byte offsets into the rows, whole tiles
void launch_proj(const ProjArgs& a, int n_heads, hipStream_t st);

// Attention of (batch, seq) query rows over cache positions [0, past + seq).
struct FlashArgs {
  const uint16_t* q;          // (batch * seq, H)
  const uint16_t* k_cache;    // (batch, n_kv, cap, 128)
  const uint16_t* v_cache;
  int n_kv, cap, past, seq, batch, causal;
  float scale;
  uint16_t* out;              // (batch * seq, H)
};

void launch_flash(const FlashArgs& a, hipStream_t st);

}  // namespace oi2
