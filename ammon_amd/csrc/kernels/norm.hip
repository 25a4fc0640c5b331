// norm.hip -- RMSNorm, one workgroup per row (reference src/kernels.rs:75-128).
//
// ss = sum x_j^2 (lanes stride the row in 16-byte chunks; wave64 butterfly,
// then the four wave totals in order), s = 1 / sqrt(ss / dim + eps), and
// o_j = w_j * (s * x_j) in the reference's multiplication order.  out may
// alias x (the reference's rmsnorm_inplace): each lane rewrites only the
// elements it read, after the barrier inside block_sum.
//
// All latency at a few rows, and a read of x at many.  Aligned rows of up to
// 8192 elements are held in registers: every load of the row and the weight is
// requested at once and x is read once (two passes of a loop: 16 rows of 4096
// took 4.8 us, 2048 rows 15.0; so 4.8 and 12.9, and the 16-token SwiGLU block
// that begins with it 88 -> 83).
// The sum is the loops', operation for operation (square_sum).
#include "device_common.h"

// ss + the four squares, each with one rounding, in this order.  Written as
// sums of products the unrolled form below took the first pair as
// fma(x0, x0, x1 x1), and a row's result depended on its width and on its
// weights' alignment.
AMMON_DEV float square_sum(const float4 &v, float ss) {
  return fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, fmaf(v.x, v.x, ss))));
}

// Rows of up to 4 R AMMON_WG elements.
template <int R>
AMMON_DEV void rmsnorm_registers(const ammon_k_rmsnorm &p, const float *x, float *out, float *red) {
  const uint32_t quads = p.dim / 4;
  float4 v[R], w[R];
  uint2 wb[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t c = threadIdx.x + r * AMMON_WG;
    v[r] = c < quads ? ((const float4 *)x)[c] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t c = min(threadIdx.x + r * AMMON_WG, quads - 1);
    if (p.w_dtype == AMMON_K_BF16)
      wb[r] = ((const uint2 *)p.w)[c];
    else
      w[r] = ((const float4 *)p.w)[c];
  }
  float ss = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    ss = square_sum(v[r], ss);
  }
  ss = block_sum(ss, red);
  ss = ss / (float)p.dim;
  ss = ss + p.eps;
  const float s = 1.0f / sqrtf(ss);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t c = threadIdx.x + r * AMMON_WG;
    if (c >= quads) continue;
    if (p.w_dtype == AMMON_K_BF16)
      w[r] = make_float4(bf16_lo(wb[r].x), bf16_hi(wb[r].x), bf16_lo(wb[r].y), bf16_hi(wb[r].y));
    ((float4 *)out)[c] = make_float4(w[r].x * (s * v[r].x), w[r].y * (s * v[r].y),
                                     w[r].z * (s * v[r].z), w[r].w * (s * v[r].w));
  }
}

extern "C" __global__ __launch_bounds__(AMMON_WG) void ammon_rmsnorm(ammon_k_rmsnorm p) {
  __shared__ float red[AMMON_WAVES];
  const uint32_t row = blockIdx.x;
  const float *x = p.x + (size_t)row * p.dim;
  float *out = p.out + (size_t)row * p.dim;
  const uintptr_t wbits = p.w_dtype == AMMON_K_F32 ? (uintptr_t)p.w : 0;
  const bool vec = (p.dim & 3u) == 0 &&
                   ((((uintptr_t)x) | ((uintptr_t)out) | wbits) & 15u) == 0;
  if (vec && ((uintptr_t)p.w & 7u) == 0) {  // uniform
    if (p.dim <= 4 * AMMON_WG) return rmsnorm_registers<1>(p, x, out, red);
    if (p.dim <= 8 * AMMON_WG) return rmsnorm_registers<2>(p, x, out, red);
    if (p.dim <= 16 * AMMON_WG) return rmsnorm_registers<4>(p, x, out, red);
    if (p.dim <= 32 * AMMON_WG) return rmsnorm_registers<8>(p, x, out, red);
  }
  float ss = 0.f;
  if (vec) {
    for (uint32_t c = threadIdx.x; c < p.dim / 4; c += AMMON_WG) {
      ss = square_sum(((const float4 *)x)[c], ss);
    }
  } else {
    for (uint32_t j = threadIdx.x; j < p.dim; j += AMMON_WG) ss += x[j] * x[j];
  }
  ss = block_sum(ss, red);
  ss = ss / (float)p.dim;
  ss = ss + p.eps;
  const float s = 1.0f / sqrtf(ss);
  if (vec) {
    for (uint32_t c = threadIdx.x; c < p.dim / 4; c += AMMON_WG) {
      float4 v = ((const float4 *)x)[c];
      float w[4];
      if (p.w_dtype == AMMON_K_BF16) {
        const uint16_t *wb = (const uint16_t *)p.w + (size_t)c * 4;
        w[0] = bf16_to_f32(wb[0]); w[1] = bf16_to_f32(wb[1]);
        w[2] = bf16_to_f32(wb[2]); w[3] = bf16_to_f32(wb[3]);
      } else {
        float4 wv = ((const float4 *)p.w)[c];
        w[0] = wv.x; w[1] = wv.y; w[2] = wv.z; w[3] = wv.w;
      }
      ((float4 *)out)[c] = make_float4(w[0] * (s * v.x), w[1] * (s * v.y),
                                       w[2] * (s * v.z), w[3] * (s * v.w));
    }
  } else {
    for (uint32_t j = threadIdx.x; j < p.dim; j += AMMON_WG)
      out[j] = load_elem(p.w, p.w_dtype, j) * (s * x[j]);
  }
}
