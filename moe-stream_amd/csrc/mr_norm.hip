// mr_norm.hip -- RMSNorm of the MoE input and the residual add of its output, as
// separate kernels for the multi-kernel decode path of mr_moe_forward_residual
// (the fused decode kernels do both inside their own launch).
//
// rms_norm(h) = (h * inv) * w, inv = 1 / sqrt(mean(h^2) + eps)   (norm.rs:16-37)
// hidden' = h + moe(rms_norm(h))                                  (layer.rs:462-473)
//
// inv is computed by one wave in the same order as the fused kernels' rms_inv
// (lane l sums the squares of elements 4*(l + 64*j) .. +3 for j = 0, 1, ... in order,
// then a butterfly), so both paths see the same bits of the normalised input.
#include "mr_device.h"
#include "mr_internal.h"

namespace mr {

__global__ __launch_bounds__(256) void k_rms_norm(const float* __restrict__ h, const float* __restrict__ w,
                                                  float eps, int H, float* __restrict__ out) {
#pragma clang fp contract(off)
  const float* hr = h + (size_t)blockIdx.x * H;
  float* orow = out + (size_t)blockIdx.x * H;
  __shared__ float inv_s;
  // Latency bounds it at few rows: the wave's loads go out eight at a time (one at a time: 8.5 us
  // for 4 rows of 2880), in the order of the sum.
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    float s = 0.f;
    for (int c0 = lane * 4; c0 < H; c0 += 8 * 256) {
      f32x4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const f32x4*>(hr + min(c0 + 256 * j, H - 4));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (c0 + 256 * j < H) {
          s = s + v[j].x * v[j].x;
          s = s + v[j].y * v[j].y;
          s = s + v[j].z * v[j].z;
          s = s + v[j].w * v[j].w;
        }
    }
    s = wave_sum_fast(s);
    if (lane == 0) inv_s = 1.f / sqrtf(s / (float)H + eps);
  }
  __syncthreads();
  const float inv = inv_s;
  for (int i = threadIdx.x * 4; i < H; i += 1024) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(hr + i), g = *reinterpret_cast<const f32x4*>(w + i);
    *reinterpret_cast<f32x4*>(orow + i) =
        f32x4{(v.x * inv) * g.x, (v.y * inv) * g.y, (v.z * inv) * g.z, (v.w * inv) * g.w};
  }
}

__global__ __launch_bounds__(256) void k_residual_add(const float* __restrict__ h, const float* __restrict__ m,
                                                      uint64_t n, float* out) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = h[i] + m[i];  // residual + moe_out
}

hipError_t launch_rms_norm(const Launch& K, const float* h, const float* w, float eps, uint32_t T, uint32_t H,
                           float* out) {
  ProfScope ps(K, "rms_norm");
  hipLaunchKernelGGL(k_rms_norm, dim3(T), dim3(256), 0, K.s, h, w, eps, (int)H, out);
  return hipGetLastError();
}

hipError_t launch_residual_add(const Launch& K, const float* h, const float* m, uint64_t n, float* out) {
  ProfScope ps(K, "residual_add");
  hipLaunchKernelGGL(k_residual_add, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, K.s, h, m, n, out);
  return hipGetLastError();
}

}  // namespace mr
