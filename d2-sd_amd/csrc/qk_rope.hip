// gfx950 kernel: per-head RMSNorm of the new queries and keys followed by
// rotary position embedding, in place, in one launch.
//
// Replaces generation/verification.py:113-123 (Qwen3: attn.q_norm / k_norm,
// then the transposes and _apply_rotary_pos_emb_qwen3; GPT-OSS: RoPE only,
// _apply_rotary_pos_emb_gpt_oss) — about ten elementwise kernels and two
// layout copies per layer — for the node-major [tokens, heads, head_dim]
// layout the verify attention reads, so no transpose is needed at all.
//
// Numerics follow the reference's bf16 tensor ops step for step
// (transformers Qwen3RMSNorm and rotate_half RoPE):
//   h   = float(x) * (1 / sqrt(mean(float(x)^2) + eps))      fp32
//   y   = bf16(w * bf16(h))                                   (norm on)
//   out = bf16(bf16(y * cos) + bf16(rotate_half(y) * sin))
// with rotate_half(y)[i] = -y[i + D/2] (i < D/2), y[i - D/2] (i >= D/2) and
// cos/sin of D columns (Qwen3, halves equal) or D/2 columns (GPT-OSS).
//
// Two kernels, chosen per call by alignment: with every row (q, k, norm weights,
// cos, sin) on a 16-byte boundary a head takes D / 8 lanes of 8 dims each (one
// 16-byte load per operand and lane, 512 / D heads per wave; the rotation
// partner is lane l ^ D/16); otherwise one wave per head, lane l holding dims
// l + 64 j (2-byte loads).  The work is one short round trip per wave, so the
// launch is bound by latency and by the number of waves and load instructions
// it issues: 150 tokens x 40 heads of 128, 36 launches in a graph, 143 us with
// one wave per head, 120 us with four heads per wave (3.97 -> 3.33 us each).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "d2sd_internal.h"
#include "plan.h"

namespace d2sd {

__device__ __forceinline__ float bf(uint16_t v) { return __uint_as_float((unsigned)v << 16); }

// round-to-nearest-even float -> bf16 (finite inputs)
__device__ __forceinline__ uint16_t to_bf(float f) {
  const unsigned u = __float_as_uint(f);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

template <int D>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(const QkRopeParams p) {
  constexpr int E = D / 64;  // dims per lane
  const int wave = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int heads = p.num_qo_heads + p.num_kv_heads;
  if (wave >= p.num_tokens * heads) return;
  const int t = wave / heads, h = wave - t * heads;
  const bool is_k = h >= p.num_qo_heads;
  uint16_t* x = (uint16_t*)(is_k ? p.k : p.q) + (long long)t * (is_k ? p.k_stride_n : p.q_stride_n) +
                (long long)(is_k ? h - p.num_qo_heads : h) * (is_k ? p.k_stride_h : p.q_stride_h);
  const uint16_t* w = (const uint16_t*)(is_k ? p.k_norm : p.q_norm);

  // every load up front, in one round (absent weights / tables read x as a
  // stand-in, never used)
  const uint16_t* cs = p.cos ? (const uint16_t*)p.cos + (long long)t * p.cs_stride : x;
  const uint16_t* sn = p.cos ? (const uint16_t*)p.sin + (long long)t * p.cs_stride : x;
  const uint16_t* wp = w ? w : x;
  float y[E], wv[E], cv[E], sv[E];
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const int d = lane + 64 * j;
    const int dc = p.cos && p.half_cos ? (d & (D / 2 - 1)) : d;
    y[j] = bf(x[d]);
    wv[j] = bf(wp[d]);
    cv[j] = bf(cs[dc]);
    sv[j] = bf(sn[dc]);
  }
  if (w) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < E; ++j) ss += y[j] * y[j];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
    const float r = 1.0f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
    for (int j = 0; j < E; ++j) y[j] = bf(to_bf(wv[j] * bf(to_bf(y[j] * r))));
  }
  if (p.cos) {
    float rot[E];
    if constexpr (D == 64) {
      const float other = __shfl_xor(y[0], 32);
      rot[0] = lane < 32 ? -other : other;
    } else {
#pragma unroll
      for (int j = 0; j < E; ++j) rot[j] = j < E / 2 ? -y[j + E / 2] : y[j - E / 2];
    }
    float out[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const float a = bf(to_bf(y[j] * cv[j]));
      const float b = bf(to_bf(rot[j] * sv[j]));
      out[j] = a + b;
    }
#pragma unroll
    for (int j = 0; j < E; ++j) y[j] = out[j];
  }
#pragma unroll
  for (int j = 0; j < E; ++j) x[lane + 64 * j] = to_bf(y[j]);
}

template <int D>
__global__ __launch_bounds__(256) void qk_norm_rope_vec_kernel(const QkRopeParams p) {
  constexpr int LPH = D / 8;  // lanes per head
  const int heads = p.num_qo_heads + p.num_kv_heads;
  const int idx = (int)((blockIdx.x * blockDim.x + threadIdx.x) / LPH);
  const int l = (int)(threadIdx.x % LPH);
  // lanes past the last head work on it again and store nothing, so that
  // every lane of a wave takes part in the exchanges
  const bool on = idx < p.num_tokens * heads;
  const int at = on ? idx : p.num_tokens * heads - 1;
  const int t = at / heads, h = at - t * heads;
  const bool is_k = h >= p.num_qo_heads;
  uint16_t* x = (uint16_t*)(is_k ? p.k : p.q) + (long long)t * (is_k ? p.k_stride_n : p.q_stride_n) +
                (long long)(is_k ? h - p.num_qo_heads : h) * (is_k ? p.k_stride_h : p.q_stride_h) + 8 * l;
  const uint16_t* w = (const uint16_t*)(is_k ? p.k_norm : p.q_norm);
  // every load up front, in one round (absent weights / tables read x as a
  // stand-in, never used)
  const int dc = p.half_cos ? (8 * l) & (D / 2 - 1) : 8 * l;
  const uint16_t* cs = p.cos ? (const uint16_t*)p.cos + (long long)t * p.cs_stride + dc : x;
  const uint16_t* sn = p.cos ? (const uint16_t*)p.sin + (long long)t * p.cs_stride + dc : x;
  const uint4 xv = *(const uint4*)x, wq = *(const uint4*)(w ? w + 8 * l : x);
  const uint4 cq = *(const uint4*)cs, sq = *(const uint4*)sn;
  float y[8], wv[8], cv[8], sv[8];
  auto expand = [](const uint4& u, float (&f)[8]) {
    const unsigned a[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[2 * j] = __uint_as_float(a[j] << 16);
      f[2 * j + 1] = __uint_as_float(a[j] & 0xFFFF0000u);
    }
  };
  expand(xv, y);
  expand(wq, wv);
  expand(cq, cv);
  expand(sq, sv);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) ss += y[j] * y[j];
#pragma unroll
  for (int off = LPH / 2; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
  if (w) {
    const float r = 1.0f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = bf(to_bf(wv[j] * bf(to_bf(y[j] * r))));
  }
  if (p.cos) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float other = __shfl_xor(y[j], LPH / 2);
      const float rot = l < LPH / 2 ? -other : other;
      cv[j] = bf(to_bf(y[j] * cv[j])) + bf(to_bf(rot * sv[j]));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = cv[j];
  }
  unsigned o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = (unsigned)to_bf(y[2 * j]) | (unsigned)to_bf(y[2 * j + 1]) << 16;
  if (on) *(uint4*)x = uint4{o[0], o[1], o[2], o[3]};
}

// every operand row on a 16-byte boundary (strides in elements of 2 bytes)
static bool rows_aligned(const QkRopeParams& p) {
  const uintptr_t a = (uintptr_t)p.q | (uintptr_t)p.k | (uintptr_t)p.q_norm | (uintptr_t)p.k_norm |
                      (uintptr_t)p.cos | (uintptr_t)p.sin;
  const long long st = (long long)p.q_stride_n | p.q_stride_h | p.k_stride_n | p.k_stride_h | (p.cos ? p.cs_stride : 0);
  return (a & 15) == 0 && (st & 7) == 0;
}

hipError_t launch_qk_norm_rope(const QkRopeParams& p, hipStream_t s) {
  const long long waves = (long long)p.num_tokens * (p.num_qo_heads + p.num_kv_heads);
  if (waves <= 0) return hipSuccess;
  if (rows_aligned(p)) {
    const dim3 grid((unsigned)((waves * (p.head_dim / 8) + 255) / 256)), block(256);
    switch (p.head_dim) {
      case 64: hipLaunchKernelGGL(qk_norm_rope_vec_kernel<64>, grid, block, 0, s, p); break;
      case 128: hipLaunchKernelGGL(qk_norm_rope_vec_kernel<128>, grid, block, 0, s, p); break;
      case 256: hipLaunchKernelGGL(qk_norm_rope_vec_kernel<256>, grid, block, 0, s, p); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
  switch (p.head_dim) {
    case 64: hipLaunchKernelGGL(qk_norm_rope_kernel<64>, grid, block, 0, s, p); break;
    case 128: hipLaunchKernelGGL(qk_norm_rope_kernel<128>, grid, block, 0, s, p); break;
    case 256: hipLaunchKernelGGL(qk_norm_rope_kernel<256>, grid, block, 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace d2sd
