// mr_valu.hip -- router, top-k and vector-ALU expert kernels for gfx950.
//
// These kernels are the straightforward decode path: one launch per step
// (router GEMV, top-k, gate+up+SwiGLU, down+combine), one wave per output
// row, activations staged in LDS. They are the correctness baseline the fused
// decode kernels (mr_fused.hip, mr_fused_q4k.hip) are checked and timed against,
// and they run every layout the ABI accepts (MXFP4 and Q4_K, any H, I multiple of
// the block).
#include "mr_device.h"
#include "mr_fused_common.h"
#include "mr_internal.h"

namespace mr {

// ---------------------------------------------------------------------------
// zero fill (graph-capture safe replacement for hipMemsetAsync)
__global__ void k_zero(uint32_t* __restrict__ p, uint64_t n_words) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (; i < n_words; i += stride) p[i] = 0u;
}

hipError_t launch_zero(const Launch& K, void* dst, uint64_t nbytes) {
  uint64_t words = nbytes / 4;
  if (words == 0) return hipSuccess;
  uint32_t blocks = (uint32_t)((words + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  ProfScope ps(K, "zero");
  hipLaunchKernelGGL(k_zero, dim3(blocks), dim3(256), 0, K.s, (uint32_t*)dst, words);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Router GEMV: logits[t][e] = x[t] . Wr[e] + b[e] + mask[e]  (layer.rs:806-837, 1016-1026)
// One wave per expert row; float4 loads; grid (ceil(E/4), T).
__global__ __launch_bounds__(256) void k_router_logits(const float* __restrict__ x,
                                                       const float* __restrict__ wr,
                                                       const float* __restrict__ br,
                                                       const float* __restrict__ mask,
                                                       float* __restrict__ logits, int H, int E) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = blockIdx.x * 4 + wave;
  const int t = blockIdx.y;
  if (e >= E) return;
  const float* xr = x + (size_t)t * H;
  const float* w = wr + (size_t)e * H;
  float acc = 0.f;
  // six steps' loads at once: latency bounds it (one step at a time: 7.3 us at H = 2880)
  for (int c0 = lane * 4; c0 < H; c0 += 6 * 256) {
    f32x4 a[6], b[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      const int c = min(c0 + 256 * j, H - 4);
      a[j] = *reinterpret_cast<const f32x4*>(xr + c);
      b[j] = *reinterpret_cast<const f32x4*>(w + c);
    }
#pragma unroll
    for (int j = 0; j < 6; ++j)
      if (c0 + 256 * j < H) {
        acc = __builtin_fmaf(a[j].x, b[j].x, acc);
        acc = __builtin_fmaf(a[j].y, b[j].y, acc);
        acc = __builtin_fmaf(a[j].z, b[j].z, acc);
        acc = __builtin_fmaf(a[j].w, b[j].w, acc);
      }
  }
  acc = wave_sum_fast(acc);
  if (lane == 0) {
    if (br) acc = acc + br[e];
    if (mask) acc = acc + mask[e];
    logits[(size_t)t * E + e] = acc;
  }
}

// Router GEMM for many tokens on the fp32 MFMA (v_mfma_f32_16x16x4f32): a 1024-thread
// workgroup takes 16 tokens x 16 experts x one of nks ranges of H's 16-element blocks; its
// 16 waves take the range's blocks in turn (wave w: blocks w, w+16, ...), each issuing all of
// its loads before its first MFMA, and the 16 partial tiles are summed in LDS in wave order.
// A CU reaches only a fraction of HBM bandwidth with its own loads, so H is split over
// workgroups until the grid spans the CUs (k_router_topk_finish adds the nks partials in
// order: the same bits on every run). MFMA operands: lane (i, g) = lane % 16, lane / 16 holds
// x[t0+i][k..k+3] and Wr[e0+i][k..k+3] for k = 16b + 4g, and MFMA j of the block multiplies
// their element j, so the four MFMAs cover the block's 16 elements; D[4g + r][i] is token
// t0+4g+r, expert e0+i. Tokens past T and experts past E repeat the last row (not stored).
// part: [nks][T][E]. H % 4 == 0 and ceil(H/16) <= nks * 16 * kRouterBlocks.
// A workgroup takes TT x TE such tiles (TT token tiles, TE expert tiles) so that each loaded row
// serves several: the loads, 16 rows to every 16 lanes, bound it (4,096 tokens x 128 experts x 2048:
// 80 us with one tile each, 51 us with 2 x 2). A tile's sums are the same bits whatever TT and TE.
constexpr int kRouterWaves = 16, kRouterBlocks = 6, kRouterMaxSplit = 4;
template <int TT, int TE>
__global__ __launch_bounds__(1024) void k_router_logits_mfma(const float* __restrict__ x,
                                                             const float* __restrict__ wr,
                                                             float* __restrict__ part, int T, int H, int E,
                                                             int nks) {
  __shared__ f32x4 red[TT * TE][kRouterWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.y * (16 * TT), e0 = blockIdx.x * (16 * TE);
  const int nb = (H + 15) >> 4, per = (nb + nks - 1) / nks;
  const int kb0 = (int)blockIdx.z * per, kb1 = min(nb, kb0 + per);
  const float* xr[TT];
  const float* wrow[TE];
#pragma unroll
  for (int t = 0; t < TT; ++t) xr[t] = x + (size_t)min(t0 + 16 * t + i, T - 1) * H + 4 * g;
#pragma unroll
  for (int e = 0; e < TE; ++e) wrow[e] = wr + (size_t)min(e0 + 16 * e + i, E - 1) * H + 4 * g;
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[TT][TE];
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int e = 0; e < TE; ++e) acc[t][e] = z;
  constexpr int kAhead = TT * TE == 1 ? kRouterBlocks : kRouterBlocks / 2;  // blocks whose loads go out together
#pragma unroll
  for (int j0 = 0; j0 < kRouterBlocks; j0 += kAhead) {
    f32x4 a[kAhead][TT], w[kAhead][TE];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int b = kb0 + wave + kRouterWaves * (j0 + j);
      const bool in = b < kb1 && 16 * b + 4 * g < H;
#pragma unroll
      for (int t = 0; t < TT; ++t) a[j][t] = in ? *reinterpret_cast<const f32x4*>(xr[t] + 16 * b) : z;
#pragma unroll
      for (int e = 0; e < TE; ++e) w[j][e] = in ? *reinterpret_cast<const f32x4*>(wrow[e] + 16 * b) : z;
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      if (kb0 + wave + kRouterWaves * (j0 + j) < kb1) {  // wave-uniform
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int e = 0; e < TE; ++e)
              acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][t][c], w[j][e][c], acc[t][e], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int e = 0; e < TE; ++e) red[t * TE + e][wave][lane] = acc[t][e];
  __syncthreads();
  if (wave < TT * TE) {
    const f32x4(*r)[64] = red[wave];
    f32x4 s = r[0][lane];
#pragma unroll
    for (int q = 1; q < kRouterWaves; ++q) {
      const f32x4 p = r[q][lane];
      s = f32x4{s[0] + p[0], s[1] + p[1], s[2] + p[2], s[3] + p[3]};
    }
    const int e = e0 + 16 * (wave % TE) + i;
    float* out = part + (size_t)blockIdx.z * T * E;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int t = t0 + 16 * (wave / TE) + 4 * g + q;
      if (t < T && e < E) out[(size_t)t * E + e] = s[q];
    }
  }
}

hipError_t launch_router_logits(const Launch& K, const mr_layer& L, const float* x, uint32_t T,
                                float* logits) {
  ProfScope ps(K, "router_logits");
  dim3 grid((L.E + 3) / 4, T);
  hipLaunchKernelGGL(k_router_logits, grid, dim3(256), 0, K.s, x, L.d.router_w, L.d.router_b,
                     L.d.dummy_mask, logits, (int)L.H, (int)L.E);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Top-k (top_k_routing, layer.rs:2346-2403; softmax_topk_kernel,
// fused_ops.metal:131-316). One wave per token; each lane holds up to 8 of the
// E <= 512 values. Selection = first k of a stable descending sort: the
// largest value wins, ties go to the lower expert index.
// Top-k of the logits v[j] of experts lane + 64 j (live[j]: e < E): by logit, and in the
// standard mode, where two logits at the selection boundary could round to one probability,
// again by the probabilities as the reference computes them (prob_exact_needed, prob_keys);
// rows whose probabilities are NaN then take experts 0..k-1, as the reference's stable sort does.
__device__ void topk_vals(float (&v)[8], bool (&live)[8], int k, uint32_t flags, int32_t* out_idx,
                          float* out_w, float* sel_v /* LDS [16] */, int* sel_i /* LDS [16] */) {
  static_assert(kRouteVals == 8, "one key column per lane value");
  const int lane = threadIdx.x & 63;
  const bool softmax_after = (flags & MR_ROUTE_SOFTMAX_AFTER_TOPK) != 0u;
  int E = 0;  // live[j] is e < E
#pragma unroll
  for (int j = 0; j < 8; ++j) E += __popcll(__ballot(live[j]));
  // keys: + 0.f makes -0.0 and +0.0 share a key; a NaN takes key 1, below every number
  // (-inf is 0x007FFFFF), as in the fused routing
  uint32_t hk[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) hk[j] = live[j] ? (v[j] == v[j] ? order_key(v[j] + 0.f) : 1u) : 0u;
  // k rounds of a wave argmax on 64-bit keys: the value's order key above the complemented
  // expert index, so the larger value wins and, between equal values, the lower index. DPP
  // steps inside 16-lane rows, then the four rows by readlane. Returns the k-th key.
  auto select = [&]() {
    bool lv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) lv[j] = live[j];
    uint32_t kth = 0u;
    for (int r = 0; r < k; ++r) {
      uint64_t best = 0ull;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t e = (uint32_t)(lane + 64 * j);
        const uint64_t key = ((uint64_t)hk[j] << 32) | (0xFFFFFFFFu - e);
        if (lv[j]) best = key > best ? key : best;
      }
      best = wave_max_u64(best);
      const int bi = (int)(0xFFFFFFFFu - (uint32_t)best);
      if ((bi & 63) == lane) lv[bi >> 6] = false;
      if (lane == 0) sel_i[r] = bi;
      kth = (uint32_t)(best >> 32);
    }
    __builtin_amdgcn_wave_barrier();
    return kth;
  };
  const uint32_t kth = select();
  if (!softmax_after && prob_exact_needed(hk, kth)) {
    prob_keys(v, E, hk);
    select();
  }
  // the selected logits
#pragma unroll 1
  for (int r = 0; r < k; ++r) {
    const float lr = entry_value(v, sel_i[r]);
    if (lane == 0) sel_v[r] = lr;
  }
  __builtin_amdgcn_wave_barrier();
  float mx_all = 0.f, sum_all = 1.f;
  if (!softmax_after) {  // standard mode: probabilities over all experts
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (live[j]) m = fmaxf(m, v[j]);
    mx_all = wave_max(m);
    float sm = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (live[j]) sm += __expf(v[j] - mx_all);
    sum_all = wave_sum(sm);
  }
  if (lane == 0) {
    if (softmax_after) {
      float m = -INFINITY;
      for (int r = 0; r < k; ++r) m = fmaxf(m, sel_v[r]);
      float ex[16], sx = 0.f;
      for (int r = 0; r < k; ++r) {
        ex[r] = __expf(sel_v[r] - m);
        sx = sx + ex[r];
      }
      for (int r = 0; r < k; ++r) out_w[r] = ex[r] / sx;
    } else {
      float pr[16];
      for (int r = 0; r < k; ++r) pr[r] = __expf(sel_v[r] - mx_all) / sum_all;
      if (flags & MR_ROUTE_NORM_TOPK) {
        float sx = 0.f;
        for (int r = 0; r < k; ++r) sx = sx + pr[r];
        for (int r = 0; r < k; ++r) out_w[r] = pr[r] / sx;
      } else {
        for (int r = 0; r < k; ++r) out_w[r] = pr[r];
      }
    }
    for (int r = 0; r < k; ++r) out_idx[r] = sel_i[r];
  }
}

__device__ void topk_wave(const float* row, int E, int k, uint32_t flags, int32_t* out_idx,
                          float* out_w, float* sel_v /* LDS [16] */, int* sel_i /* LDS [16] */) {
  const int lane = threadIdx.x & 63;
  float v[8];
  bool live[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    int e = lane + 64 * j;
    live[j] = e < E;
    v[j] = live[j] ? row[e] : 0.f;
  }
  topk_vals(v, live, k, flags, out_idx, out_w, sel_v, sel_i);
}

// Router logits from the H-split partials of k_router_logits_mfma (summed in split order,
// then + bias + mask, the order of k_router_logits), written to logits, then the top-k.
__global__ __launch_bounds__(64) void k_router_topk_finish(const float* __restrict__ part, int nks, int T,
                                                           const float* __restrict__ br,
                                                           const float* __restrict__ mask,
                                                           float* __restrict__ logits, int E, int k,
                                                           uint32_t flags, int32_t* __restrict__ idx,
                                                           float* __restrict__ w) {
  __shared__ float sv[16];
  __shared__ int si[16];
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  float v[8];
  bool live[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int e = lane + 64 * j;
    live[j] = e < E;
    float s = 0.f;
    if (live[j]) {
      s = part[(size_t)t * E + e];
      for (int q = 1; q < nks; ++q) s = s + part[((size_t)q * T + t) * E + e];
      if (br) s = s + br[e];
      if (mask) s = s + mask[e];
      logits[(size_t)t * E + e] = s;
    }
    v[j] = s;
  }
  topk_vals(v, live, k, flags, idx + (size_t)t * k, w + (size_t)t * k, sv, si);
}

hipError_t launch_router_topk(const Launch& K, const mr_layer& L, const float* x, uint32_t T, float* logits,
                              float* part, int32_t* idx, float* w) {
  const uint32_t nb = (L.H + 15) / 16, tiles = ((L.E + 15) / 16) * ((T + 15) / 16);
  uint32_t nks = std::max<uint32_t>((nb + 16 * kRouterBlocks - 1) / (16 * kRouterBlocks), (256 + tiles - 1) / tiles);
  nks = std::min<uint32_t>(nks, kRouterMaxSplit);
  if (T < 16 || L.H % 4 != 0 || nb > nks * 16u * kRouterBlocks) {
    hipError_t e = launch_router_logits(K, L, x, T, logits);
    return e == hipSuccess ? launch_topk(K, logits, T, L.E, L.d.top_k, L.d.route_flags, idx, w) : e;
  }
  {
    ProfScope ps(K, "router_logits");
    // 2 x 2 tiles once the grid still spans the CUs with a quarter of the workgroups
    if (tiles * nks >= 4 * 256)
      hipLaunchKernelGGL((k_router_logits_mfma<2, 2>), dim3((L.E + 31) / 32, (T + 31) / 32, nks), dim3(64 * kRouterWaves),
                         0, K.s, x, L.d.router_w, part, (int)T, (int)L.H, (int)L.E, (int)nks);
    else
      hipLaunchKernelGGL((k_router_logits_mfma<1, 1>), dim3((L.E + 15) / 16, (T + 15) / 16, nks), dim3(64 * kRouterWaves),
                         0, K.s, x, L.d.router_w, part, (int)T, (int)L.H, (int)L.E, (int)nks);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ProfScope ps(K, "topk");
  hipLaunchKernelGGL(k_router_topk_finish, dim3(T), dim3(64), 0, K.s, part, (int)nks, (int)T, L.d.router_b,
                     L.d.dummy_mask, logits, (int)L.E, (int)L.d.top_k, L.d.route_flags, idx, w);
  return hipGetLastError();
}

__global__ __launch_bounds__(64) void k_topk(const float* __restrict__ logits, int E, int k,
                                             uint32_t flags, int32_t* __restrict__ idx,
                                             float* __restrict__ w) {
  __shared__ float sv[16];
  __shared__ int si[16];
  const int t = blockIdx.x;
  topk_wave(logits + (size_t)t * E, E, k, flags, idx + (size_t)t * k, w + (size_t)t * k, sv, si);
}

hipError_t launch_topk(const Launch& K, const float* logits, uint32_t T, uint32_t E, uint32_t k,
                       uint32_t flags, int32_t* idx, float* w) {
  ProfScope ps(K, "topk");
  hipLaunchKernelGGL(k_topk, dim3(T), dim3(64), 0, K.s, logits, (int)E, (int)k, flags, idx, w);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Dot products of R quantized weight rows with an LDS-resident vector whose 32-element blocks lie
// xst floats apart. Each lane adds up its units (every 64th block of 32 elements) in order; the
// lanes' partial sums are acc. Units and the order of every sum are the same for any R, so a row's
// result does not depend on the rows beside it.
// A unit reads 128 bytes of the vector for 17 or 18 bytes of weights, so R rows share a read, and with
// xst = 36 the lanes' blocks start in different banks (at 32 all in one): one row at a time the vector's reads
// bounded it (experts of 8 tokens, 32 of 2880 x 2880, gate/up 148 us and down 105 us; now 104 and 68 us).
// What bounds it now: the latency of the weight loads, one 17-byte window per lane and row, 90 units on 64
// lanes in two rounds. Of the waves' time 67% (gate/up) and 72% (down) is waiting, 0.1% of it for LDS; VALU
// issue takes 17 and 12% of the SIMDs' cycles.
constexpr int kXStride = 36;

// MXFP4: unit = one 17-byte block; sum_b d_b * sum_j kvalue_j x_j.
template <int R>
__device__ __forceinline__ void rows_dot_mxfp4(const uint8_t* const (&row)[R], const float* xs, int xst, int in_features,
                                               int lane, float (&acc)[R]) {
  const int nb = in_features >> 5;
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.f;
  for (int b = lane; b < nb; b += 64) {
    uint32_t sc[R], q[R][4];
#pragma unroll
    for (int r = 0; r < R; ++r) mx_load_block(row[r] + (size_t)b * 17, sc[r], q[r]);
    f32x4 xb[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) xb[c] = *reinterpret_cast<const f32x4*>(xs + xst * b + 4 * c);
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = __builtin_fmaf(mx_block_kdot(q[r], xb), e8m0_half(sc[r]), acc[r]);
  }
}

// Q4_K: unit = one 32-element sub-block s of a 144-byte super-block:
// (d*sc) * sum q x - (dmin*m) * sum x  (dequant.rs:218-262 regrouped).
template <int R>
__device__ __forceinline__ void rows_dot_q4k(const uint8_t* const (&row)[R], const float* xs, int xst, int in_features,
                                             int lane, float (&acc)[R]) {
  const int nu = in_features >> 5;  // 8 sub-blocks per 256
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.f;
  for (int u = lane; u < nu; u += 64) {
    const int b = u >> 3, s = u & 7;
    f32x4 xb[8];
    float sx = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      xb[i] = *reinterpret_cast<const f32x4*>(xs + xst * u + 4 * i);
      sx += (xb[i].x + xb[i].y) + (xb[i].z + xb[i].w);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t* bw = reinterpret_cast<const uint32_t*>(row[r] + (size_t)b * 144);
      uint32_t dd = bw[0];
      uint32_t scw[3] = {bw[1], bw[2], bw[3]};
      uint32_t sc, m;
      q4k_scale_min((uint32_t)s, scw, sc, m);
      float d = h2f(dd & 0xFFFFu), dmin = h2f(dd >> 16);
      const uint32_t* qw = bw + 4 + 8 * (s >> 1);
      const int shift = (s & 1) * 4;
      float sq = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint32_t word = (qw[i] >> shift) & 0x0F0F0F0Fu;
        sq = __builtin_fmaf((float)((word >> 0) & 0xFFu), xb[i].x, sq);
        sq = __builtin_fmaf((float)((word >> 8) & 0xFFu), xb[i].y, sq);
        sq = __builtin_fmaf((float)((word >> 16) & 0xFFu), xb[i].z, sq);
        sq = __builtin_fmaf((float)((word >> 24) & 0xFFu), xb[i].w, sq);
      }
      acc[r] += (d * (float)sc) * sq - (dmin * (float)m) * sx;
    }
  }
}

template <int TYPE, int R>
__device__ __forceinline__ void rows_dot(const uint8_t* const (&row)[R], const float* xs, int xst, int n, int lane,
                                         float (&acc)[R]) {
  if constexpr (TYPE == MR_GGML_MXFP4)
    rows_dot_mxfp4<R>(row, xs, xst, n, lane, acc);
  else
    rows_dot_q4k<R>(row, xs, xst, n, lane, acc);
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = wave_sum_fast(acc[r]);
}

__host__ __device__ constexpr uint64_t row_bytes_of(int type, uint64_t cols) {
  return type == MR_GGML_MXFP4 ? (cols / 32) * 17 : (cols / 256) * 144;
}

// ---------------------------------------------------------------------------
// Kernel (2): gate+up dequant-matvec + bias + SwiGLU for each (token, slot).
// grid (ceil(I / 16), slots, T), 256 threads: 4 waves x 4 rows each.
struct GateUpArgs {
  const uint8_t* gate;
  const uint8_t* up;
  const uint64_t* gate_off;  // [E] byte offsets
  const uint64_t* up_off;
  const float* gate_b;       // [E, I] or null
  const float* up_b;
  const float* x;            // [T, H]
  const int32_t* idx;        // [T, k] or null (shared expert: expert 0)
  float* act;                // [T, k, I]
  const float* sh_gate_inp;  // shared expert only: [H] or null
  float* sh_sig;             // shared expert only: [T] sigmoid(x . gate_inp)
  int H, I, E, k, act_kind;
  float alpha, limit;
  int xst;  // floats between x's 32-element blocks in LDS
};

template <int TYPE>
__global__ __launch_bounds__(256) void k_gateup_valu(GateUpArgs a) {
  extern __shared__ float xs[];  // [H / 32][xst]
  const int t = blockIdx.z, slot = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* xt = a.x + (size_t)t * a.H;
  for (int c = threadIdx.x * 4; c < a.H; c += 1024)
    *reinterpret_cast<f32x4*>(xs + (c >> 5) * a.xst + (c & 31)) = *reinterpret_cast<const f32x4*>(xt + c);
  __syncthreads();
  const int e = a.idx ? a.idx[(size_t)t * a.k + slot] : 0;
  if (e < 0 || e >= a.E) return;  // invalid routing entry contributes nothing
  if (a.sh_sig && blockIdx.x == 0 && wave == 0) {
    float z = 0.f;
    if (a.sh_gate_inp)
      for (int c = lane; c < a.H; c += 64) z = __builtin_fmaf(xs[(c >> 5) * a.xst + (c & 31)], a.sh_gate_inp[c], z);
    z = wave_sum(z);
    if (lane == 0) a.sh_sig[t] = a.sh_gate_inp ? sigmoidf_(z) : 1.0f;
  }
  const uint8_t* G = a.gate + a.gate_off[e];
  const uint8_t* U = a.up + a.up_off[e];
  const uint64_t rb = row_bytes_of(TYPE, (uint64_t)a.H);
  const int row0 = blockIdx.x * 16 + wave * 4;
  if (row0 >= a.I) return;
  // R gate rows and the same up rows at a time. Q4_K with 4: 177 VGPRs, two waves per SIMD, which costs more
  // than the shared reads give once there are many workgroups (experts of 256 tokens, us, R = 4 / 2 / rows one
  // by one: 128 of 768 x 2048, 8 per token, 3064 / 2514 / 3207; 24 of 256 x 512, 3 per token, 272 / 235 / 234; 1 token
  // of the former 38 / 38 / 57). MXFP4 with 4: 122 VGPRs.
  constexpr int R = TYPE == MR_GGML_Q4_K ? 2 : 4;
#pragma unroll
  for (int i0 = 0; i0 < 4; i0 += R) {
    if (i0) __builtin_amdgcn_sched_barrier(0);  // one after the other
    const uint8_t* rows[2 * R];  // past I the last row again, not stored
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint64_t off = (uint64_t)min(row0 + i0 + i, a.I - 1) * rb;
      rows[i] = G + off, rows[R + i] = U + off;
    }
    float d[2 * R];
    rows_dot<TYPE, 2 * R>(rows, xs, a.xst, a.H, lane, d);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = row0 + i0 + i;
      if (lane == 0 && r < a.I) {
        float g = d[i], u = d[R + i];
        if (a.gate_b) g = g + a.gate_b[(size_t)e * a.I + r];
        if (a.up_b) u = u + a.up_b[(size_t)e * a.I + r];
        float h = a.act_kind == MR_ACT_SWIGLU_OAI ? swiglu_oai(g, u, a.alpha, a.limit) : silu_mul(g, u);
        a.act[((size_t)t * a.k + slot) * a.I + r] = h;
      }
    }
  }
}

// Kernel (3): down dequant-matvec + bias + weighted combine over the k routed
// experts in ascending expert index (layer.rs:1092-1106, 1446-1448), then the
// shared expert scaled by its sigmoid gate (layer.rs:1935-1951).
// grid (ceil(H / 16), T), 256 threads; LDS holds the token's k activations.
struct DownArgs {
  const uint8_t* down;
  const uint64_t* down_off;
  const float* down_b;   // [E, H] or null
  const float* act;      // [T, k, I]
  const int32_t* idx;    // [T, k]
  const float* w;        // [T, k]
  float* y;              // [T, H]
  int H, I, E, k;
  // shared expert (optional)
  const uint8_t* sh_down;  // [H, Ish] (type sh_type)
  const float* act_sh;     // [T, Ish]
  const float* sh_sig;     // [T]
  int Ish;
  int xst;  // floats between the activations' 32-element blocks in LDS
};

template <int TYPE, int SH_TYPE>
__global__ __launch_bounds__(256) void k_down_valu(DownArgs a) {
  extern __shared__ float lds[];  // ([k * I] + [Ish]) / 32 blocks of xst
  __shared__ int order[16];
  const int t = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* at = a.act + (size_t)t * a.k * a.I;
  const int n_act = a.k * a.I;
  for (int c = threadIdx.x * 4; c < n_act; c += 1024)
    *reinterpret_cast<f32x4*>(lds + (c >> 5) * a.xst + (c & 31)) = *reinterpret_cast<const f32x4*>(at + c);
  float* lds_sh = lds + (n_act >> 5) * a.xst;
  if (a.sh_down)
    for (int c = threadIdx.x * 4; c < a.Ish; c += 1024)
      *reinterpret_cast<f32x4*>(lds_sh + (c >> 5) * a.xst + (c & 31)) =
          *reinterpret_cast<const f32x4*>(a.act_sh + (size_t)t * a.Ish + c);
  if (threadIdx.x == 0) {
    // slots sorted by expert index, ascending (insertion sort, k <= 16)
    const int32_t* it = a.idx + (size_t)t * a.k;
    for (int s = 0; s < a.k; ++s) {
      int j = s;
      while (j > 0 && it[order[j - 1]] > it[s]) {
        order[j] = order[j - 1];
        --j;
      }
      order[j] = s;
    }
  }
  __syncthreads();
  const uint64_t rb = row_bytes_of(TYPE, (uint64_t)a.I);
  const uint64_t rb_sh = row_bytes_of(SH_TYPE, (uint64_t)a.Ish);
  const int row0 = blockIdx.x * 16 + wave * 4;
  if (row0 >= a.H) return;
  int rr[4];  // past H the last row again, not stored
#pragma unroll
  for (int i = 0; i < 4; ++i) rr[i] = min(row0 + i, a.H - 1);
  float yv[4] = {0.f, 0.f, 0.f, 0.f}, o[4];
  const uint8_t* rows[4];
  for (int j = 0; j < a.k; ++j) {
    const int slot = order[j];
    const int e = a.idx[(size_t)t * a.k + slot];
    if (e < 0 || e >= a.E) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[i] = a.down + a.down_off[e] + (uint64_t)rr[i] * rb;
    rows_dot<TYPE, 4>(rows, lds + slot * (a.I >> 5) * a.xst, a.xst, a.I, lane, o);
    const float w = a.w[(size_t)t * a.k + slot];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (a.down_b) o[i] = o[i] + a.down_b[(size_t)e * a.H + rr[i]];
      yv[i] = yv[i] + o[i] * w;
    }
  }
  if (a.sh_down) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[i] = a.sh_down + (uint64_t)rr[i] * rb_sh;
    rows_dot<SH_TYPE, 4>(rows, lds_sh, a.xst, a.Ish, lane, o);
#pragma unroll
    for (int i = 0; i < 4; ++i) yv[i] = yv[i] + o[i] * a.sh_sig[t];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (lane == 0 && row0 + i < a.H) a.y[(size_t)t * a.H + row0 + i] = yv[i];
}

// LDS stride of 32-element blocks for n floats: padded where that stays within 64 KiB.
static int x_stride(uint64_t n) { return n / 32 * kXStride * sizeof(float) <= 65536 ? kXStride : 32; }

template <int TYPE>
static hipError_t gateup_dispatch(const Launch& K, const char* name, const GateUpArgs& a,
                                  uint32_t slots, uint32_t T) {
  dim3 grid((a.I + 15) / 16, slots, T);
  size_t lds = (size_t)a.H / 32 * a.xst * sizeof(float);
  ProfScope ps(K, name);
  hipLaunchKernelGGL(k_gateup_valu<TYPE>, grid, dim3(256), lds, K.s, a);
  return hipGetLastError();
}

template <int TYPE, int SH>
static hipError_t down_dispatch2(const Launch& K, const DownArgs& a, uint32_t T) {
  dim3 grid((a.H + 15) / 16, T);
  size_t lds = ((size_t)a.k * a.I + (a.sh_down ? a.Ish : 0)) / 32 * a.xst * sizeof(float);
  ProfScope ps(K, "down");
  hipLaunchKernelGGL((k_down_valu<TYPE, SH>), grid, dim3(256), lds, K.s, a);
  return hipGetLastError();
}

template <int TYPE>
static hipError_t down_dispatch(const Launch& K, const DownArgs& a, int sh_type, uint32_t T) {
  if (sh_type == MR_GGML_MXFP4) return down_dispatch2<TYPE, MR_GGML_MXFP4>(K, a, T);
  return down_dispatch2<TYPE, MR_GGML_Q4_K>(K, a, T);
}

hipError_t launch_experts_valu(const Launch& s, const mr_layer& L, const float* x, uint32_t T,
                               const int32_t* idx, const float* w, float* act, float* act_sh,
                               float* y) {
  const mr_pack& G = *L.d.gate;
  const mr_pack& U = *L.d.up;
  const mr_pack& D = *L.d.down;
  const bool has_sh = L.d.sh_gate != nullptr;
  float* sh_sig = has_sh ? act_sh + (size_t)T * L.Ish : nullptr;
  hipError_t err;
  if (has_sh) {
    const mr_pack& SG = *L.d.sh_gate;
    GateUpArgs sa{SG.base, L.d.sh_up->base, SG.d_offsets, L.d.sh_up->d_offsets, nullptr, nullptr,
                  x, nullptr, act_sh, L.d.sh_gate_inp, sh_sig, (int)L.H, (int)L.Ish, 1, 1,
                  MR_ACT_SILU, 0.f, 0.f, x_stride(L.H)};
    err = SG.type == MR_GGML_MXFP4 ? gateup_dispatch<MR_GGML_MXFP4>(s, "shared_gateup", sa, 1, T)
                                   : gateup_dispatch<MR_GGML_Q4_K>(s, "shared_gateup", sa, 1, T);
    if (err != hipSuccess) return err;
  }
  GateUpArgs ga{G.base, U.base, G.d_offsets, U.d_offsets, L.d.gate_bias, L.d.up_bias, x, idx, act,
                nullptr, nullptr, (int)L.H, (int)L.I, (int)L.E, (int)L.d.top_k, (int)L.d.act,
                L.d.alpha, L.d.limit, x_stride(L.H)};
  err = L.type == MR_GGML_MXFP4 ? gateup_dispatch<MR_GGML_MXFP4>(s, "gateup", ga, L.d.top_k, T)
                                : gateup_dispatch<MR_GGML_Q4_K>(s, "gateup", ga, L.d.top_k, T);
  if (err != hipSuccess) return err;
  DownArgs da{D.base, D.d_offsets, L.d.down_bias, act, idx, w, y, (int)L.H, (int)L.I, (int)L.E,
              (int)L.d.top_k, has_sh ? L.d.sh_down->base : nullptr, act_sh, sh_sig, (int)L.Ish,
              x_stride((uint64_t)L.d.top_k * L.I + L.Ish)};
  const int sh_type = has_sh ? L.d.sh_down->type : MR_GGML_Q4_K;
  return L.type == MR_GGML_MXFP4 ? down_dispatch<MR_GGML_MXFP4>(s, da, sh_type, T)
                                 : down_dispatch<MR_GGML_Q4_K>(s, da, sh_type, T);
}

// ---------------------------------------------------------------------------
// Dequantization (dequantize_mxfp4 dequant.rs:605-628; dequantize_q4k 218-262),
// bit-exact: single multiplies, no contraction.
__global__ void k_dequant_mxfp4(const uint8_t* __restrict__ src, float* __restrict__ out,
                                uint64_t n_blocks) {
  uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_blocks) return;
  uint32_t sc, q[4];
  mx_load_block(src + b * 17, sc, q);
  const float d = e8m0_half(sc);
  float* y = out + b * 32;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 v0 = MR_KV2(q[i], 0), v1 = MR_KV2(q[i], 1), v2 = MR_KV2(q[i], 2),
                v3 = MR_KV2(q[i], 3);
    y[4 * i + 0] = v0.x * d, y[16 + 4 * i + 0] = v0.y * d;
    y[4 * i + 1] = v1.x * d, y[16 + 4 * i + 1] = v1.y * d;
    y[4 * i + 2] = v2.x * d, y[16 + 4 * i + 2] = v2.y * d;
    y[4 * i + 3] = v3.x * d, y[16 + 4 * i + 3] = v3.y * d;
  }
}

__global__ void k_dequant_q4k(const uint8_t* __restrict__ src, float* __restrict__ out,
                              uint64_t n_units) {
#pragma clang fp contract(off)
  uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n_units) return;
  const uint64_t b = u >> 3;
  const uint32_t s = (uint32_t)(u & 7);
  const uint32_t* bw = reinterpret_cast<const uint32_t*>(src + b * 144);
  uint32_t dd = bw[0];
  uint32_t scw[3] = {bw[1], bw[2], bw[3]};
  uint32_t sc, m;
  q4k_scale_min(s, scw, sc, m);
  const float d1 = h2f(dd & 0xFFFFu) * (float)sc;
  const float m1 = h2f(dd >> 16) * (float)m;
  const uint32_t* qw = bw + 4 + 8 * (s >> 1);
  const int shift = (s & 1) * 4;
  float* y = out + u * 32;
  for (int i = 0; i < 8; ++i) {
    uint32_t word = (qw[i] >> shift) & 0x0F0F0F0Fu;
    for (int j = 0; j < 4; ++j) {
      float p = d1 * (float)((word >> (8 * j)) & 0xFFu);
      y[4 * i + j] = p - m1;
    }
  }
}

hipError_t launch_dequant(const Launch& K, const mr_pack& p, uint32_t expert, float* out) {
  ProfScope ps(K, "dequant");
  hipStream_t s = K.s;
  const uint8_t* src = p.base + p.h_offsets[expert];
  const uint64_t n_el = (uint64_t)p.out_features * p.in_features;
  if (p.type == MR_GGML_MXFP4) {
    uint64_t nb = n_el / 32;
    hipLaunchKernelGGL(k_dequant_mxfp4, dim3((uint32_t)((nb + 255) / 256)), dim3(256), 0, s, src,
                       out, nb);
  } else {
    uint64_t nu = n_el / 32;
    hipLaunchKernelGGL(k_dequant_q4k, dim3((uint32_t)((nu + 255) / 256)), dim3(256), 0, s, src,
                       out, nu);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Synthetic blocks (same arithmetic as moe_rocm/synth.py).
__global__ void k_synth_mxfp4(uint8_t* __restrict__ dst, uint64_t n_blocks, uint64_t first,
                              uint64_t seed) {
  uint64_t l = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n_blocks) return;
  const uint64_t b = first + l;
  uint64_t d0 = draw(seed, 3 * b), d1 = draw(seed, 3 * b + 1), d2 = draw(seed, 3 * b + 2);
  uint8_t* p = dst + l * 17;
  p[0] = (uint8_t)(119u + (uint32_t)(((d0 >> 32) * 9ull) >> 32));
  for (int i = 0; i < 8; ++i) p[1 + i] = (uint8_t)(d1 >> (8 * i));
  for (int i = 0; i < 8; ++i) p[9 + i] = (uint8_t)(d2 >> (8 * i));
}

__device__ __forceinline__ float irwin_hall12(uint64_t a, uint64_t b, uint64_t c) {
  uint32_t s = 0;
  for (int i = 0; i < 4; ++i) s += (uint32_t)((a >> (16 * i)) & 0xFFFFu);
  for (int i = 0; i < 4; ++i) s += (uint32_t)((b >> (16 * i)) & 0xFFFFu);
  for (int i = 0; i < 4; ++i) s += (uint32_t)((c >> (16 * i)) & 0xFFFFu);
  return ((float)s - 393216.0f) * (1.0f / 65536.0f);
}

__global__ void k_synth_q4k(uint8_t* __restrict__ dst, uint64_t n_blocks, uint64_t first,
                            uint64_t seed) {
#pragma clang fp contract(off)
  uint64_t l = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n_blocks) return;
  const uint64_t b = first + l;
  uint64_t d[24];
  for (int i = 0; i < 24; ++i) d[i] = draw(seed, 24 * b + i);
  float zd = irwin_hall12(d[0], d[1], d[2]);
  float zm = irwin_hall12(d[3], d[4], d[5]);
  uint32_t hd = f2h_rne(fabsf(zd) * 0.01f);
  uint32_t hm = f2h_rne(fabsf(zm) * 0.005f);
  uint8_t* p = dst + l * 144;
  p[0] = (uint8_t)hd, p[1] = (uint8_t)(hd >> 8), p[2] = (uint8_t)hm, p[3] = (uint8_t)(hm >> 8);
  for (int i = 0; i < 140; ++i) p[4 + i] = (uint8_t)(d[6 + i / 8] >> (8 * (i % 8)));
}

hipError_t launch_synth(const Launch& K, int type, void* dst, uint64_t n_blocks, uint64_t seed) {
  hipStream_t s = K.s;
  const uint64_t per = 65535ull * 256ull;
  for (uint64_t off = 0; off < n_blocks; off += per) {
    uint64_t n = n_blocks - off < per ? n_blocks - off : per;
    dim3 grid((uint32_t)((n + 255) / 256));
    if (type == MR_GGML_MXFP4)
      hipLaunchKernelGGL(k_synth_mxfp4, grid, dim3(256), 0, s, (uint8_t*)dst + off * 17, n, off,
                         seed);
    else
      hipLaunchKernelGGL(k_synth_q4k, grid, dim3(256), 0, s, (uint8_t*)dst + off * 144, n, off,
                         seed);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace mr
