// Per-token asymmetric int8 fake quantisation of one value, shared by the stand-alone kernels (fake_quant.hip) and the
// converted linear that quantises its activation on the way (int4_linear.hip), so that both produce the same bits.
#pragma once
#include "common.h"
#include "nf4_math.h"

namespace ttamd {

constexpr float kF32Eps = 1.1920928955078125e-07f;  // torch.finfo(torch.float32).eps

struct TokenQParams {
  float scale, inv_scale, zp;
};

// asymmetric int8 qparams from the row extrema (already widened to include 0)
// (the zero point is chosen with the fp32 scale; a bf16 qparam precision rounds the scale afterwards, and the rounded
// scale is what quantises and dequantises)
__device__ __forceinline__ TokenQParams token_qparams(float mn, float mx, bool qp_bf16, float eps) {
  TokenQParams p;
  float scale = (mx - mn) / 255.0f;
  scale = scale > eps ? scale : eps;
  const float dmin = mn / scale, dmax = mx / scale;
  float zp = ((-128.0f + dmin) + (127.0f + dmax) > 0.0f) ? (-128.0f - dmin) : (127.0f - dmax);
  zp = zp < -128.0f ? -128.0f : (zp > 127.0f ? 127.0f : zp);
  p.zp = __builtin_rintf(zp);
  if (qp_bf16) scale = round_to_bf16(scale);
  p.scale = scale;
  p.inv_scale = 1.0f / scale;
  return p;
}

template <bool BF16>
__device__ __forceinline__ float token_fq(float x, const TokenQParams& p) {
  float q = __builtin_rintf(x * p.inv_scale) + p.zp;
  q = q < -128.0f ? -128.0f : (q > 127.0f ? 127.0f : q);
  return Arith<BF16>::rnd((q - p.zp) * p.scale);
}

__device__ __forceinline__ void wave_minmax(float& mn, float& mx) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, off, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
  }
}

}  // namespace ttamd
