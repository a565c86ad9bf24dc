// mr_grouped_q4k.hip -- multi-token (prefill / batched) Q4_K MoE experts as grouped GEMMs on
// the gfx950 f16 MFMA (v_mfma_f32_16x16x32_f16).
//
// The reference runs each expert once over all of its tokens (index_select, gate/up/act/down,
// index_add: layer.rs:2148-2183; on the GPU one projection per expert, metal/mod.rs:911-962).
// Here, after the grouping of mr_grouped.hip (k_group: (token, slot) pairs by expert):
//   k_split_f16        activation rows -> two f16 terms per element (the f16 nearest to x * p and
//                      the f16 nearest to the rest, p a power of two per row: 22 significant
//                      bits) plus the f32 sum of every 32-element sub-block as three f16 terms;
//                      with a shared expert also its sigmoid gate of the row.
//   k_grouped_q4k<1>   gate and up for one (expert, 64, 128 or 256 rows, pair tile); epilogue bias +
//                      activation x routing weight -> h, in f32 in the down input images' place or,
//                      where the item's 256 rows are one super-block of the down input, split into
//                      its image, with its own p.
//   k_split_h          h in f32 -> the down input images, in place.
//   k_grouped_q4k<0>   down for one (expert, 128 or 256 rows, pair tile) -> o [pair][H].
//   k_combine          (mr_grouped.hip) the pairs of a token in ascending expert order, then the
//                      shared expert scaled by its sigmoid gate (layer.rs:1092-1106, 1935-1951).
// The shared expert is one more group (every token, weight 1, SiLU) of the same two launches.
//
// Arithmetic per 256-element super-block (dequant.rs:218-262 regrouped):
//   sum_k w_k x_k = d * sum_k (sc_j q_k) x_k - dmin * sum_j m_j X_j,
// with sc_j q_k <= 63 * 15 = 945 an exact f16, so the first sum is one f16 MFMA chain per term
// over all eight sub-blocks (products of 10 by 11 bits, f32 accumulation) and needs no work on
// its accumulators per sub-block; the second is one MFMA (m_j exact, X_j in three f16 terms).
#include "mr_device.h"
#include "mr_fused_common.h"
#include "mr_internal.h"

#include <algorithm>
#include <type_traits>

namespace mr {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kQXcds = 8;      // workgroups are dispatched round robin over the 8 XCDs
// Image of one (row, super-block): 8 K steps n = 4h + 2u + hl, each [term][lane group g][8 halves],
// then the sub-block sums [term 0..2, zero][8 halves]. Half j of (n, g) is element
// 128 h + 64 (g / 2) + 32 hl + 16 (g % 2) + 8 u + kQPerm[j]: a weight lane of group g holds 16 of
// the 64 quant bytes of half h (low nibbles of one sub-block, hl = 0, high nibbles of the next),
// takes 8 of them per u, and unpacks bytes 0, 2 and 1, 3 of a dword into two pairs of halves.
constexpr int kQImgSb = 8 * 128 + 64;
// Offset past every buffer of the GEMM (images: at most this many bytes, weight matrices: far
// fewer): a load there fetches nothing and reads zero.
constexpr int kPast = 0x7F000000;
__device__ constexpr int kQPerm[8] = {0, 2, 1, 3, 4, 6, 5, 7};  // its own inverse

__device__ __forceinline__ uint32_t f16_bits(float v) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v); }
// v = hi + lo, the two terms of the split (each rounded to nearest)
__device__ __forceinline__ void split2(float v, uint32_t& hi, uint32_t& lo) {
  const _Float16 h = (_Float16)v;
  hi = (uint32_t)__builtin_bit_cast(uint16_t, h);
  lo = f16_bits(v - (float)h);
}
// The power of two p that brings a largest magnitude mx to [2^14, 2^15) (mx = 0: 1), and 1/p.
__device__ __forceinline__ void pow2_scale(float mx, float& p, float& pinv) {
  const int ex = (int)((__float_as_uint(mx) >> 23) & 0xFFu);  // biased; 0: zero or denormal
  const int pe = mx > 0.f ? min(max(127 + 14 + 127 - ex, 2), 252) : 127;
  p = __uint_as_float((uint32_t)pe << 23);
  pinv = __uint_as_float((uint32_t)(254 - pe) << 23);
}
// Sub-block sum X (already scaled by p) -> its three f16 terms of 2^-5 X (32 elements below
// 2^15 sum to less than 2^20, past f16).
__device__ __forceinline__ uint32_t sum_term(float X, int t) {
  float r = X * 0.03125f;
  uint32_t b = 0u;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const _Float16 h = (_Float16)r;
    if (q == t) b = (uint32_t)__builtin_bit_cast(uint16_t, h);
    r = r - (float)h;
  }
  return b;
}

// Bounds-checked buffer of nbytes (raw, 32-bit offsets).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const uint8_t* p, uint32_t nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0, (int)nbytes, 0x00027000);
}

// ---- activation rows -> images ----------------------------------------------------------------
// Image of a super-block: lane l holds elements 4l .. 4l+3, v. Element 4l + c: h = l >> 5, g / 2 =
// l >> 4 & 1, hl = l >> 3 & 1, g % 2 = l >> 2 & 1, u = l >> 1 & 1, bytes 4 (l & 1) + c, i.e. halves
// 4 (l & 1) + {0, 2, 1, 3}.
__device__ __forceinline__ void split_sb(f32x4 v, float p, int lane, uint8_t* dst) {
  const int at = (4 * (lane >> 5) + (lane & 2) + ((lane >> 3) & 1)) * 128 +
                 (2 * ((lane >> 4) & 1) + ((lane >> 2) & 1)) * 16 + (lane & 1) * 8;
  uint32_t h[4], l[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) split2(v[c] * p, h[c], l[c]);
  *reinterpret_cast<uint2*>(dst + at) = make_uint2(h[0] | h[2] << 16, h[1] | h[3] << 16);
  *reinterpret_cast<uint2*>(dst + at + 64) = make_uint2(l[0] | l[2] << 16, l[1] | l[3] << 16);
  float ps = (v.x + v.y) + (v.z + v.w);  // sub-block sum over the 8 lanes 8j .. 8j+7
  ps += dpp_f<kDppXor1>(ps);
  ps += dpp_f<kDppXor2>(ps);
  ps = add_xor4(ps);
  const int t = lane & 7, j = lane >> 3;
  if (t < 4) *reinterpret_cast<uint16_t*>(dst + 1024 + t * 16 + kQPerm[j] * 2) = (uint16_t)sum_term(ps * p, t);
}

// One workgroup per row, its waves over the row's super-blocks in turn (lane l: elements 4l ..
// 4l+3), twice: the row's largest magnitude, then the split (the second read hits L1). sig: the
// shared expert's gate sigmoid(x . gate_inp) of the row, 1 without gate_inp (layer.rs:1935-1951).
__global__ __launch_bounds__(256) void k_split_f16(const float* __restrict__ src, int D, uint8_t* __restrict__ img,
                                                   float* __restrict__ pinv_out, const float* __restrict__ gi,
                                                   float* __restrict__ sig) {
  __shared__ float red[8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nsb = D >> 8;
  const int64_t r = blockIdx.x;
  const float* row = src + (size_t)r * D;
  float mx = 0.f, z = 0.f;
  for (int sb = wave; sb < nsb; sb += 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(row + sb * 256 + 4 * lane);
    mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    if (gi) {
      const f32x4 gv = *reinterpret_cast<const f32x4*>(gi + sb * 256 + 4 * lane);
#pragma unroll
      for (int c = 0; c < 4; ++c) z = __builtin_fmaf(v[c], gv[c], z);
    }
  }
  mx = wave_max(mx);
  if (gi) z = wave_sum_fast(z);
  if (lane == 0) red[wave] = mx, red[4 + wave] = z;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float p, pinv;
  pow2_scale(mx, p, pinv);
  if (threadIdx.x == 0) {
    pinv_out[r] = pinv;
    if (sig) sig[r] = gi ? sigmoidf_((red[4] + red[5]) + (red[6] + red[7])) : 1.0f;
  }
  for (int sb = wave; sb < nsb; sb += 4)
    split_sb(*reinterpret_cast<const f32x4*>(row + sb * 256 + 4 * lane), p, lane, img + ((size_t)r * nsb + sb) * kQImgSb);
}

// h, one super-block in f32 at the start of each image's place -> the images: a wave per super-block,
// which it holds in registers before it writes. The routed pairs' n0 super-blocks, then the shared
// expert's n1 (a launch of their own: 4.7 us).
__global__ __launch_bounds__(256) void k_split_h(uint8_t* img0, float* pinv0, int64_t n0, uint8_t* img1, float* pinv1,
                                                 int64_t n1) {
  const int lane = threadIdx.x & 63;
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= n0 + n1) return;
  uint8_t* dst = b < n0 ? img0 + (size_t)b * kQImgSb : img1 + (size_t)(b - n0) * kQImgSb;
  const f32x4 v = *reinterpret_cast<const f32x4*>(dst + 16 * lane);
  float p, pinv;
  pow2_scale(wave_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)))), p, pinv);
  if (lane == 0) *(b < n0 ? pinv0 + b : pinv1 + (b - n0)) = pinv;
  split_sb(v, p, lane, dst);
}

// ---- shared-expert gate: sigmoid(x . gate_inp) per token (layer.rs:1935-1951) -------------------
// The order of the per-token path (k_gateup_valu): lane-strided fma, then a wave sum.
__global__ __launch_bounds__(64) void k_sh_gate(const float* __restrict__ x, int H, const float* __restrict__ gi,
                                                float* __restrict__ sig) {
  const int t = blockIdx.x, lane = threadIdx.x;
  float z = 0.f;
  if (gi)
#pragma unroll 8
    for (int c = lane; c < H; c += 64) z = __builtin_fmaf(x[(size_t)t * H + c], gi[c], z);  // loads issued ahead
  z = wave_sum(z);
  if (lane == 0) sig[t] = gi ? sigmoidf_(z) : 1.0f;
}

// ---- grouped GEMM ---------------------------------------------------------------------------
struct GQ4Group {
  ExpertLoc w0;        // gate (GATEUP) or down
  ExpertLoc w1;        // up (GATEUP)
  const float* b0;     // gate bias [E][M] or null (GATEUP)
  const float* b1;     // up bias
  const uint8_t* img;  // images [rows][K/256]
  const float* pinv;   // their 1/p: [rows] (GATEUP), [rows][K/256] (down)
  uint8_t* himg;       // GATEUP: the down input images [pairs][M/256], or h in f32 (256 floats) at each one's start
  float* hpinv;        // and their 1/p
  float* out;          // down: [pairs][M]
  int M, K, act;
};
struct GQ4Args {
  GQ4Group r, s;             // routed experts; the shared expert over tokens 0 .. sh_T - 1
  const int32_t* pair_tok;   // GATEUP: image row of pair p (down: row = p)
  const float* pair_w;       // GATEUP: routing weight of pair p
  const int32_t* exp_off;    // [E+1] pair offsets
  const int32_t* tile_off;   // [E+1] pair tile offsets
  const int32_t* tile_exp;   // expert of each pair tile
  int E, sh_T;               // sh_T = 0: no shared expert
  float alpha, limit;
};

// Work item: (expert e, rows of each matrix, tile of 16 PG pairs), NW waves. Gate/up: wave w rows
// 16 w .. 16 w + 15 of the gate and of the up matrix, so that a lane holds both values of a
// (row, pair). NW = 16, 256 rows: a down input super-block forms inside one item, which splits it;
// NW = 8 or 4: h goes through memory, for k_split_h. (Two tiles of each matrix in eight waves, so that a
// fragment read serves four MFMAs, PG = 4: the whole call 941 -> 926 us at the size below, but 161 -> 171 us
// for 1,024 tokens of 16 experts of 1024 x 3072, and 3% slower at 512 to 1,024 tokens of the size below.)
// Down: 4 waves of 32 rows (PG = 1) or of 64 (PG = 4: 323 us at the size below, with 8 of 32 rows 348, as
// its accumulators fit there). Which of them runs: see q4_items. The activations are the MFMA's A operand (rows:
// pairs), the weights its B operand (columns: weight rows): lane (i, g) = lane % 16, lane / 16
// holds weight row i of every tile, and of D weight row i for pairs 4g .. 4g+3 of each pair group.
//   A wave's weights come in halves of a super-block, 64 bytes per row, one or two halves ahead in
//   registers; four lanes load a row's 64 bytes (16 rows per load), and an LDS slice of the wave
//   turns them into operand order. Lane (i, g) unpacks a nibble pair of row i with one and (two
//   f16 denormals q 2^-24 or 16 q 2^-24) and one packed multiply by sc 2^10 or sc 2^6, which is
//   exact: sc q 2^-14.
//   Images are staged in LDS in operand order (1 KB per (K step, term, pair group)), kKS K steps
//   per stage, double buffered, one stage ahead in registers, loaded like the weights, four
//   lanes per row. In both the 16-byte pieces of a row are spread over the banks (xor).
//   Nothing in the loop may spill: a reload's wait would drain the prefetched loads (measured:
//   PG = 1 gate/up in 256-row items 90 us with 36 registers spilled, 50 us with none).
// What bounds it: MFMA and VALU issue, which this chip hardly overlaps (measured on two waves of a
// SIMD: an MFMA of 16.7 cycles plus four VALU of 2.7 take 26.3), at a clock that falls to 1.7 GHz
// on long batches: 128 experts of 768 x 2048, 32,768 pairs: gate/up 1.00 -> 0.54 ms and down
// 0.49 -> 0.30 ms against the int8 MFMA with its scale products on the accumulators per sub-block.
// Few pairs: the same unpacking against the weight stream (512 experts of 512 x 2048, 3,840
// pairs: gate/up 300 -> 191 us, 3.1 TB/s; 128 pairs of 128 experts of 768 x 2048: 78 -> 37 us).
// 16-row tiles per wave (see the kernel), and the rows of a matrix per work item
constexpr int q4_tiles(bool gateup, int pg) { return gateup || pg == 1 ? 2 : 4; }
constexpr int q4_rows(bool gateup, int pg, int waves) { return 16 * q4_tiles(gateup, pg) / (gateup ? 2 : 1) * waves; }

template <bool GATEUP, int PG, int NW>
__global__ __launch_bounds__(64 * NW, q4_tiles(GATEUP, PG) == 4 ? 2 : NW == 4 ? 3 : 4) void k_grouped_q4k(GQ4Args a) {
  constexpr int NT = q4_tiles(GATEUP, PG), kRows = q4_rows(GATEUP, PG, NW);
  static_assert(256 % kRows == 0, "row counts are multiples of 256");
  constexpr bool kSplit = GATEUP && kRows == 256;  // the epilogue writes images
  constexpr int kTM = GATEUP ? NT / 2 : NT;  // tiles of one matrix per wave
  static_assert(!kSplit || kTM == 1, "the split takes 16 rows of a matrix per wave: half a sub-block");
  constexpr int kPF = PG == 1 ? 2 : 1;       // half super-blocks of weights in flight
  constexpr int kKS = PG == 1 ? 8 : 2;       // K steps per stage
  constexpr int kNS = 8 / kKS;               // stages per super-block
  constexpr int kPW = kKS * 2 * PG / NW;     // stage pieces (K step, term, pair group) per wave
  constexpr int kStage = kKS * 2 * PG * 1024;
  constexpr int kPairs = 16 * PG;
  constexpr int kEpRow = kQImgSb + 16;  // epilogue: bytes between the images of two pairs
  constexpr int kEp = kSplit ? kPairs * kEpRow : 0;
  __shared__ __align__(16) uint8_t lds[kEp > 2 * kStage ? kEp : 2 * kStage];
  __shared__ __align__(16) uint8_t xst[2][PG == 1 ? 16 : PG * 1024];  // sub-block sums, operand order (PG = 1: in registers)
  __shared__ __align__(16) uint8_t ast[NW][NT * 1024];  // half a super-block of the wave's rows: [tile][row][64 bytes]
  __shared__ __align__(16) uint8_t hst[NW][NT * 256];   // and their headers: [tile][row][16 bytes]
  __shared__ __align__(16) float pst[2][kPairs];       // down: 1/p of (pair, super-block); gate/up: [0] of the pair
  __shared__ __align__(16) float pw[kPairs];           // GATEUP: routing weights
  __shared__ __align__(16) float wred[kSplit ? NW : 1][kPairs], wsum[kSplit ? NW : 1][kPairs];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int n_sh_t = (a.sh_T + kPairs - 1) / kPairs;
  const int n_rt_s = a.s.M / kRows, n_rt_r = a.r.M / kRows;
  const int n_sh = a.sh_T ? n_rt_s * n_sh_t : 0;
  const int n_work = n_sh + n_rt_r * a.tile_off[a.E];
  const int per_xcd = (n_work + kQXcds - 1) / kQXcds;
  const int loc = blockIdx.x / kQXcds;
  int w = (blockIdx.x % kQXcds) * per_xcd + loc;
  if (loc >= per_xcd || w >= n_work) return;  // uniform
  const bool sh = w < n_sh;
  const GQ4Group& q = sh ? a.s : a.r;
  int e = 0, rt, p0, np;
  if (sh) {
    rt = w / n_sh_t;
    p0 = (w - rt * n_sh_t) * kPairs;
    np = min(kPairs, a.sh_T - p0);
  } else {
    w -= n_sh;
    e = a.tile_exp[w / n_rt_r];  // items n_rt tile_off[e] .. n_rt tile_off[e+1] - 1 are expert e's
    const int t_beg = a.tile_off[e], nt_e = a.tile_off[e + 1] - t_beg, wl = w - n_rt_r * t_beg;
    rt = wl / nt_e;
    p0 = a.exp_off[e] + (wl - rt * nt_e) * kPairs;
    np = min(kPairs, a.exp_off[e + 1] - p0);
  }
  const int M = q.M, nsb = q.K >> 8;
  const uint32_t rb = (uint32_t)nsb * 144u;
  // tile t of this wave: GATEUP: gate (t < kTM) or up rows wrow0 + 16 (t % kTM) .. ; down: rows wrow0
  // + 16 t .. . M % 256 == 0.
  const int wrow0 = rt * kRows + wave * (16 * kTM);
  // Buffer loads: one lane offset for all tiles, the tile and super-block in the scalar offset.
  const __amdgpu_buffer_rsrc_t wb0 = buffer_of(expert_at(q.w0, e), (uint32_t)M * rb);
  const __amdgpu_buffer_rsrc_t wb1 = GATEUP ? buffer_of(expert_at(q.w1, e), (uint32_t)M * rb) : wb0;
  uint32_t wt[NT];  // uniform
#pragma unroll
  for (int t = 0; t < NT; ++t) wt[t] = (uint32_t)(wrow0 + 16 * (t % kTM)) * rb;
  // loads take 4 lanes per row: row lr, 16-byte piece lp; headers one lane per row
  const int lr = lane >> 2, lp = lane & 3;
  const int aoff = lr * (int)rb + 16 + 16 * lp;
  // header of tile g % NT, row i
  const uint8_t* hsrc = expert_at(GATEUP && g % NT >= kTM ? q.w1 : q.w0, e) + (uint32_t)(wrow0 + 16 * (g % kTM) + i) * (uint64_t)rb;
  const int awr = (lr * 4 + (lp ^ (lr >> 2))) * 16, ard = (i * 4 + (g ^ (i >> 2))) * 16;  // in a tile of ast
  const int bwr = (lp * 16 + (lr ^ (4 * lp))) * 16, brd = (g * 16 + (i ^ (4 * g))) * 16;  // in a stage piece
  const int32_t* tok = GATEUP && !sh ? a.pair_tok : nullptr;

  auto run = [&](auto npg_c) {
    constexpr int NPG = decltype(npg_c)::value;  // pair groups of this item that hold pairs
    // Stage pieces of this thread: pieces wave kPW .. + kPW - 1, piece (K step, term, pair group) in
    // that order; 4 lanes bring the 64 bytes of pair 16 pg + lr. Buffer loads
    // from the images of this call's rows (GATEUP; at most kPast bytes) or of the item's pairs.
    const uint32_t ib = (uint32_t)nsb * kQImgSb;
    const __amdgpu_buffer_rsrc_t xb = buffer_of(GATEUP ? q.img : q.img + (size_t)p0 * ib, kPast);
    auto row_of = [&](int pl) {  // image row of pair pl of the item
      const int pc = min(pl, np - 1);
      return GATEUP ? (tok ? tok[p0 + pc] : p0 + pc) : pc;
    };
    uint32_t brow[kPW];
#pragma unroll
    for (int c = 0; c < kPW; ++c) {
      const int pg = (wave * kPW + c) % PG;
      brow[c] = pg < NPG ? (uint32_t)row_of(16 * pg + lr) * ib + 16 * lp : (uint32_t)kPast;
    }
    // (K step, term) of the pieces: those of one share it
    auto bkt = [&](int c) { return (uint32_t)((wave * kPW + c) / PG) * 64u; };
    // the sub-block sums: PG = 1: the lane's own operand; else waves 0 .. NPG-1 bring those of
    // pair group `wave`
    const uint32_t xrow = PG == 1 ? (uint32_t)row_of(i) * ib + 1024 + 16 * g
                          : wave < NPG ? (uint32_t)row_of(16 * wave + lr) * ib + 1024 + 16 * lp : (uint32_t)kPast;
    const uint32_t prow = GATEUP ? (uint32_t)row_of(tid & (kPairs - 1)) : (uint32_t)((row_of(tid & (kPairs - 1))) * nsb);
    const float* pbase = GATEUP ? q.pinv : q.pinv + (size_t)p0 * nsb;
    if (tid < kPairs) {
      if (GATEUP) {
        pst[0][tid] = pbase[prow];
        pw[tid] = sh ? 1.f : a.pair_w[p0 + min(tid, np - 1)];
      }
    }
    i32x4 bR[kPW], xR = {0, 0, 0, 0};
    float pR = 0.f;
    auto load_x = [&](int sb) {
      xR = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, (int)xrow, sb * kQImgSb, 0));
    };
    auto load_b = [&](int sb, int s) {
#pragma unroll
      for (int c = 0; c < kPW; ++c)
        bR[c] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               xb, (int)brow[c], (int)(bkt(c) + (uint32_t)(sb * kQImgSb + s * (kKS * 128))), 0));
      if (s == 0) {
        if (PG > 1) load_x(sb);
        if (!GATEUP) pR = pbase[prow + (uint32_t)sb];
      }
    };
    auto store_b = [&](int sb, int s, int buf) {
#pragma unroll
      for (int c = 0; c < kPW; ++c)
        *reinterpret_cast<i32x4*>(&lds[buf * kStage + (wave * kPW + c) * 1024 + bwr]) = bR[c];
      if (s == 0) {
        if (PG > 1 && wave < NPG) *reinterpret_cast<i32x4*>(&xst[sb & 1][wave * 1024 + bwr]) = xR;
        if (!GATEUP) pst[sb & 1][tid & (kPairs - 1)] = pR;
      }
    };
    // Weight loads are issued for every half super-block and one past the last, where nothing is
    // fetched.
    i32x4 aR[kPF][NT], hR;
    auto load_hdr = [&](int sb) {
      hR = *(const __attribute__((address_space(1))) i32x4*)(hsrc + (uint32_t)(min(sb, nsb - 1) * 144));
    };
    auto load_a = [&](int sb, int half) {
      const int off = aoff + 64 * half + (sb < nsb ? 0 : kPast);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        aR[half % kPF][t] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                          GATEUP && t >= kTM ? wb1 : wb0, off, (int)wt[t] + sb * 144, 0));
    };
    load_b(0, 0);
    load_hdr(0);
    load_a(0, 0);
    if (kPF == 2) load_a(0, 1);

    const uint32_t psel = 0x07000700u | (uint32_t)(g & 2) | (uint32_t)((g & 2) + 1) << 16;  // v_perm: bytes {s, 0x64} twice
    f32x4 acc[NT][NPG];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int pg = 0; pg < NPG; ++pg) acc[t][pg] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int sb = 0; sb < nsb; ++sb) {
      const f16x2 k1024 = {(_Float16)-1024.f, (_Float16)-1024.f};
      auto as2 = [](uint32_t u) { return __builtin_bit_cast(f16x2, u); };
      f32x4 S[NT][NPG];
      i32x4 raw[NT];
      f16x2 sc_lo[NT], sc_hi[NT];
      // half a super-block: its weights, and the scales of the lane's two sub-blocks
      auto begin_half = [&](int half) {
        // (the wave's own LDS accesses stay in order)
#pragma unroll
        for (int t = 0; t < NT; ++t) *reinterpret_cast<i32x4*>(&ast[wave][t * 1024 + awr]) = aR[half % kPF][t];
        if (half == 0) *reinterpret_cast<i32x4*>(&hst[wave][(lane % (16 * NT)) * 16]) = hR;
        if (PG == 1 && half) load_x(sb);
        if (kPF == 2)
          load_a(sb + 1, half);
        else
          load_a(half ? sb + 1 : sb, half ^ 1);
        if (half == 0) load_hdr(sb + 1);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          raw[t] = *reinterpret_cast<const i32x4*>(&ast[wave][t * 1024 + ard]);
          const i32x4 hw = *reinterpret_cast<const i32x4*>(&hst[wave][t * 256 + i * 16]);
          const uint32_t w0 = (uint32_t)hw[1], w2 = (uint32_t)hw[3];
          const uint32_t sw = half ? (w2 & 0x0F0F0F0Fu) | ((w0 >> 2) & 0x30303030u) : w0 & 0x3F3F3F3Fu;
          // bytes 2 (g / 2), + 1: the scales of sub-blocks 4 half + these, as f16 1024 + sc, then
          // 2^10 sc and, for nibbles left in place (16 q), 2^6 sc
          const f16x2 s2 = (as2(__builtin_amdgcn_perm(0x64646464u, sw, psel)) + k1024) * f16x2{(_Float16)1024.f, (_Float16)64.f};
          sc_lo[t] = __builtin_shufflevector(s2, s2, 0, 0);
          sc_hi[t] = __builtin_shufflevector(s2, s2, 1, 1);
        }
      };
#pragma unroll
      for (int s = 0; s < kNS; ++s) {
        const int buf = (sb * kNS + s) & 1;
        if (s * kKS % 4 == 0) begin_half(s * kKS / 4);
        store_b(sb, s, buf);  // last read two stages ago, before the previous barrier
        __syncthreads();
        if (s + 1 < kNS)
          load_b(sb, s + 1);
        else
          load_b(min(sb + 1, nsb - 1), 0);
        // The stage's K steps. Each fragment is read from LDS two fragments ahead; with two waves
        // per SIMD (NT = 4), step ks + 1's weights are unpacked among step ks's MFMAs.
        constexpr int kWB = NT == 4 ? 2 : 1;  // unpacked K steps in registers
        f16x8 wf[kWB][NT], xf[3];
        auto unpack = [&](int n, f16x8 (&o)[NT]) {
          const int u = (n >> 1) & 1, hl = n & 1;
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const uint32_t x0 = (uint32_t)raw[t][2 * u], x1 = (uint32_t)raw[t][2 * u + 1];
            const uint32_t msk = hl ? 0x00F000F0u : 0x000F000Fu;
            const f16x2 sc = hl ? sc_hi[t] : sc_lo[t];
            const f16x2 a0 = as2(x0 & msk) * sc, a1 = as2((x0 >> 8) & msk) * sc;
            const f16x2 a2 = as2(x1 & msk) * sc, a3 = as2((x1 >> 8) & msk) * sc;
            o[t] = f16x8{a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
          }
        };
        constexpr int kF = 2 * NPG;  // fragments (term, pair group) per K step
        auto frag = [&](int f) {     // f: fragment of the stage
          return *reinterpret_cast<const f16x8*>(
              &lds[buf * kStage + ((f / kF * 2 + f % kF / NPG) * PG + f % NPG) * 1024 + brd]);
        };
        xf[0] = frag(0);
        xf[1] = frag(1);
        if constexpr (kWB == 2) unpack(s * kKS, wf[0]);
#pragma unroll
        for (int f = 0; f < kKS * kF; ++f) {
          const int ks = f / kF, pg = f % NPG;
          if (f + 2 < kKS * kF) xf[(f + 2) % 3] = frag(f + 2);
          if constexpr (kWB == 2) {
            if (f % kF == 0 && ks + 1 < kKS) unpack(s * kKS + ks + 1, wf[(ks + 1) & 1]);
          } else {
            if (kKS == 8 && f == 4 * kF) begin_half(1);
            if (f % kF == 0) unpack(s * kKS + ks, wf[0]);
          }
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const f32x4 z = {0.f, 0.f, 0.f, 0.f};
            S[t][pg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[f % 3], wf[ks & (kWB - 1)][t],
                                                              s == 0 && f < NPG ? z : S[t][pg], 0, 0, 0);
          }
          if constexpr (kWB == 2) {
            if (f + 2 < kKS * kF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
            if (ks + 1 < kKS) __builtin_amdgcn_sched_group_barrier(0x002, (72 + kF - 1) / kF, 0);
          } else {
            if (f % kF == kF - 1) __builtin_amdgcn_sched_barrier(0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // acc += (d S - dmin M) (down: / p): M is the min term's MFMA, the eight mins of row i as
      // f16 in image order in every lane group against the sums' terms
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const i32x4 hw = *reinterpret_cast<const i32x4*>(&hst[wave][t * 256 + i * 16]);
        const uint32_t dd = (uint32_t)hw[0], w1 = (uint32_t)hw[2], w2 = (uint32_t)hw[3];
        const float dv = 16384.f * (float)__builtin_bit_cast(_Float16, (uint16_t)dd);  // the weights are 2^-14 sc q
        const float dm = -32.f * (float)__builtin_bit_cast(_Float16, (uint16_t)(dd >> 16));  // the sums are 2^-5 X
        const uint32_t m03 = w1 & 0x3F3F3F3Fu, m47 = ((w2 >> 4) & 0x0F0F0F0Fu) | ((w1 >> 2) & 0x30303030u);
        auto m2 = [&](uint32_t m, uint32_t sel) { return as2(__builtin_amdgcn_perm(0x64646464u, m, sel)) + k1024; };
        const f16x2 ma = m2(m03, 0x07020700u), mb = m2(m03, 0x07030701u), mc = m2(m47, 0x07020700u), md = m2(m47, 0x07030701u);
        const f16x8 mf = {ma.x, ma.y, mb.x, mb.y, mc.x, mc.y, md.x, md.y};
#pragma unroll
        for (int pg = 0; pg < NPG; ++pg) {
          const f16x8 xf = PG == 1 ? __builtin_bit_cast(f16x8, xR)
                                   : *reinterpret_cast<const f16x8*>(&xst[sb & 1][pg * 1024 + brd]);
          const f32x4 z = {0.f, 0.f, 0.f, 0.f};
          const f32x4 m = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf, mf, z, 0, 0, 0);
          f32x4 pv = {1.f, 1.f, 1.f, 1.f};
          if (!GATEUP) pv = *reinterpret_cast<const f32x4*>(&pst[sb & 1][16 * pg + 4 * g]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (GATEUP)
              acc[t][pg][r] = __builtin_fmaf(dm, m[r], __builtin_fmaf(dv, S[t][pg][r], acc[t][pg][r]));
            else
              acc[t][pg][r] = __builtin_fmaf(__builtin_fmaf(dm, m[r], dv * S[t][pg][r]), pv[r], acc[t][pg][r]);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }

    if constexpr (!GATEUP) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int row = wrow0 + 16 * t + i;
#pragma unroll
        for (int pg = 0; pg < NPG; ++pg)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int pl = 16 * pg + 4 * g + r;
            if (pl < np) q.out[(size_t)(p0 + pl) * M + row] = acc[t][pg][r];
          }
      }
    } else {
      // h = act(gate + b_g, up + b_u) x routing weight in registers (this lane: rows 16 t + i of
      // the wave's, pairs 4g + r of each group).
      float hv[kTM][NPG][4];
#pragma unroll
      for (int t = 0; t < kTM; ++t) {
        const int row = wrow0 + 16 * t + i;
        const float bg = !sh && q.b0 ? q.b0[(size_t)e * M + row] : 0.f, bu = !sh && q.b1 ? q.b1[(size_t)e * M + row] : 0.f;
#pragma unroll
        for (int pg = 0; pg < NPG; ++pg) {
          const f32x4 pv = *reinterpret_cast<const f32x4*>(&pst[0][16 * pg + 4 * g]);
          const f32x4 rw = *reinterpret_cast<const f32x4*>(&pw[16 * pg + 4 * g]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float gv = __builtin_fmaf(acc[t][pg][r], pv[r], bg), uv = __builtin_fmaf(acc[kTM + t][pg][r], pv[r], bu);
            hv[t][pg][r] = (q.act == MR_ACT_SWIGLU_OAI ? swiglu_oai(gv, uv, a.alpha, a.limit) : silu_mul(gv, uv)) * rw[r];
          }
        }
      }
      if constexpr (!kSplit) {
#pragma unroll
        for (int t = 0; t < kTM; ++t) {
          const int row = wrow0 + 16 * t + i;
#pragma unroll
          for (int pg = 0; pg < NPG; ++pg)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int pl = 16 * pg + 4 * g + r;
              if (pl < np)
                reinterpret_cast<float*>(q.himg + ((size_t)(p0 + pl) * (M >> 8) + (row >> 8)) * kQImgSb)[row & 255] =
                    hv[t][pg][r];
            }
        }
      } else {
        // The item's 256 rows of a pair, one super-block, are split. Largest magnitudes and sums go
        // over the 16 lanes of a row group, the magnitudes over the waves through LDS; the halves
        // are put in place in LDS and leave as whole 16-byte pieces.
#pragma unroll
        for (int pg = 0; pg < NPG; ++pg)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float m = fabsf(hv[0][pg][r]), s = hv[0][pg][r];
            m = fmaxf(m, dpp_f<kDppXor1>(m)), s += dpp_f<kDppXor1>(s);
            m = fmaxf(m, dpp_f<kDppXor2>(m)), s += dpp_f<kDppXor2>(s);
            m = fmaxf(m, dpp_f<kDppHMirror>(m)), s += dpp_f<kDppHMirror>(s);
            m = fmaxf(m, dpp_f<kDppMirror>(m)), s += dpp_f<kDppMirror>(s);
            if (i == 0) {
              wred[wave][16 * pg + 4 * g + r] = m;
              wsum[wave][16 * pg + 4 * g + r] = s;  // half a sub-block
            }
          }
        __syncthreads();  // the magnitudes are in place and every wave is done with the stages
        // element 16 el + i of the super-block, el = wave: sub-block el / 2, i.e. h = el / 8,
        // g = 2 (el / 4 % 2) + el % 2, hl = el / 2 % 2, u = i / 8
        auto at = [&](int el) {
          return (4 * (el >> 3) + 2 * (i >> 3) + ((el >> 1) & 1)) * 128 + ((el >> 1) & 2) * 16 + (el & 1) * 16 + kQPerm[i & 7] * 2;
        };
#pragma unroll
        for (int pg = 0; pg < NPG; ++pg) {
          f32x4 m4 = *reinterpret_cast<const f32x4*>(&wred[0][16 * pg + 4 * g]);
#pragma unroll
          for (int v = 1; v < NW; ++v) {
            const f32x4 o4 = *reinterpret_cast<const f32x4*>(&wred[v][16 * pg + 4 * g]);
#pragma unroll
            for (int r = 0; r < 4; ++r) m4[r] = fmaxf(m4[r], o4[r]);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int pl = 16 * pg + 4 * g + r;
            float p, pinv;
            pow2_scale(m4[r], p, pinv);
            uint8_t* im = &lds[pl * kEpRow];
            uint32_t h, l;
            split2(hv[0][pg][r] * p, h, l);
            uint8_t* d = im + at(wave);
            *reinterpret_cast<uint16_t*>(d) = (uint16_t)h;
            *reinterpret_cast<uint16_t*>(d + 64) = (uint16_t)l;
            const int sub = wave / 2;
            // its sum, of this wave's half and the next one's. Four lanes write the terms of one value: both
            // halves come from LDS, since the lanes' own sums may differ in the last bit (the compiler fuses
            // the routing weight's product into the first addition), and a sum whose f16 rounding parts two
            // lanes would be off by 2^-11.
            if (i < 4 && wave % 2 == 0) {
              const float X = wsum[wave][pl] + wsum[(wave + 1) % NW][pl];
              *reinterpret_cast<uint16_t*>(im + 1024 + i * 16 + kQPerm[sub] * 2) = (uint16_t)sum_term(X * p, i);
            }
            if (wave == 0 && i == 0 && pl < np) q.hpinv[(size_t)(p0 + pl) * (M >> 8) + rt] = pinv;
          }
        }
        __syncthreads();
        constexpr int kPieces = kQImgSb / 16;
        for (int c = tid; c < np * kPieces; c += NW * 64) {
          const int pl = c / kPieces, o = (c - pl * kPieces) * 16;
          *reinterpret_cast<i32x4*>(q.himg + ((size_t)(p0 + pl) * (M >> 8) + rt) * kQImgSb + o) =
              *reinterpret_cast<const i32x4*>(&lds[pl * kEpRow + o]);
        }
      }
    }
  };
  if constexpr (PG == 1) {
    run(std::integral_constant<int, 1>{});
  } else {
    static_assert(PG == 4, "pair tiles of 16 or 64");
    const int npg = (np + 15) >> 4;
    if (npg == 4) run(std::integral_constant<int, 4>{});
    else if (npg == 3) run(std::integral_constant<int, 3>{});
    else if (npg == 2) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
  }
}

// ---- host side -------------------------------------------------------------------------------
namespace {
constexpr uint64_t kQAlign = 256;
uint64_t qup(uint64_t v) { return (v + kQAlign - 1) / kQAlign * kQAlign; }
uint64_t img_bytes(uint64_t rows, uint64_t D) { return rows * (D / 256) * kQImgSb; }
struct Q4Plan {
  uint64_t pair_tok, pair_w, pair_of, exp_off, tile_off, tile_exp, hist;
  uint64_t xp, himg, hp, hsimg, hsp, xo, osh, sig, total;
};
// The x images are last read by the gate/up launch and o is first written by the down launch:
// they share xo.
Q4Plan q4_plan(uint64_t T, uint64_t k, uint64_t E, uint64_t I, uint64_t H, uint64_t Ish) {
  Q4Plan p{};
  const uint64_t P = T * k;
  uint64_t o = 0;
  p.pair_tok = o, o += qup(P * 4);
  p.pair_w = o, o += qup(P * 4);
  p.pair_of = o, o += qup(P * 4);
  p.exp_off = o, o += qup((E + 1) * 4);
  p.tile_off = o, o += qup((E + 1) * 4);
  p.tile_exp = o, o += qup(group_tiles_max(P, E, kGroupTileMin) * 4);
  p.hist = o, o += qup(group_hist_bytes(P, E));
  p.xp = o, o += qup(T * 4);
  p.himg = o, o += qup(img_bytes(P, I));
  p.hp = o, o += qup(P * (I / 256) * 4);
  p.xo = o, o += qup(std::max(img_bytes(T, H), P * H * 4));
  if (Ish) {
    p.hsimg = o, o += qup(img_bytes(T, Ish));
    p.hsp = o, o += qup(T * (Ish / 256) * 4);
    p.osh = o, o += qup(T * H * 4);
    p.sig = o, o += qup(T * 4);
  }
  p.total = o;
  return p;
}
}  // namespace

uint64_t grouped_q4k_scratch_bytes(uint64_t T, uint64_t k, uint64_t E, uint64_t I, uint64_t H, uint64_t Ish) {
  return q4_plan(T, k, E, I, H, Ish).total;
}

hipError_t launch_sh_gate(const Launch& K, const float* x, uint32_t T, int H, const float* gate_inp, float* sig) {
  ProfScope ps(K, "shared_gate");
  hipLaunchKernelGGL(k_sh_gate, dim3(T), dim3(64), 0, K.s, x, H, gate_inp, sig);
  return hipGetLastError();
}

// Q4_K routed experts (and a Q4_K shared expert) with K dimensions in whole super-blocks.
bool grouped_q4k_supported(const mr_layer& L) {
  if (L.type != MR_GGML_Q4_K || L.d.top_k > 16 || L.E > 1024) return false;
  if (L.H % 256 != 0 || L.I % 256 != 0 || L.H % 4 != 0) return false;
  if (L.d.sh_gate && (L.d.sh_gate->type != MR_GGML_Q4_K || L.d.sh_down->type != MR_GGML_Q4_K || L.Ish % 256 != 0))
    return false;
  return true;
}

// One grouped GEMM launch over at most `tiles` routed and `sh_tiles` shared pair tiles.
template <bool GATEUP, int PG, int NW>
static void launch_q4(const Launch& K, const GQ4Args& a, uint64_t tiles, uint64_t sh_tiles) {
  constexpr int rows = q4_rows(GATEUP, PG, NW);
  const dim3 grid(grouped_grid((uint64_t)(a.r.M / rows) * tiles + (uint64_t)(a.s.M / rows) * sh_tiles));
  hipLaunchKernelGGL((k_grouped_q4k<GATEUP, PG, NW>), grid, dim3(64 * NW), 0, K.s, a);
}

// Pairs per tile and waves (of 16 rows) per gate/up item of a call.
struct Q4Items {
  int tile, gu_waves;
};
// With items(tile, rows) the expected number of gate/up work items (about half the experts hold a
// part-filled tile more than their pairs fill). Measured (the whole call, us), 16-pair tiles / 64-pair
// tiles unless said otherwise:
// - 64 pairs read and unpack an expert's weights once for up to four 16-pair groups; they pay from a mean of
//   16 to 30 pairs per expert on: 128 experts of 768 x 2048, top 8, mean 16 181 / 195, 24 212 / 218, 32
//   253 / 234, 64 397 / 373; 512 experts of 512 x 2048, top 10, mean 20 534 / 538 and, with popularity
//   ~ rank^-1.1, 418 / 384. So the line is 16, where a skewed batch gains what an even one loses.
// - But an item of 64 pairs x 256 rows takes 35 us and more, and alone on its CU gains nothing: below half an
//   item per CU the 16-pair tiles win at any mean (16 experts of 512 x 2048, top 4: 48 items 71 / 110, 80
//   96 / 119, 112 119 / 123, 144 144 / 139, 208 197 / 157; 16 of 256 x 2048, top 2, 96 tokens: 44 / 69).
// - 16-pair gate/up items of 8 waves or of 4 (128 or 64 rows): the latter while 128 rows would be less than an
//   item per CU (102 items of 128 rows: 4 waves 48, 8 waves 51; 236: 72 / 78; 432: 92 / 88; 360: 83 / 81). Items of
//   256 rows that split h themselves save k_split_h but leave CUs idle and are slower or equal everywhere:
//   2 tokens of the first layer 62 us, with 64 rows 48; 8 tokens of 16 experts of 256 x 2048 51 / 39; 64 tokens
//   of the first layer 146, with 128 rows 129; at best (32 tokens of 60 experts of 1024 x 2048 with a shared
//   one) 77 / 77.
static Q4Items q4_items(uint64_t T, uint64_t k, uint64_t E, uint64_t I, uint64_t Ish) {
  const uint64_t P = T * k;
  auto items = [&](uint64_t tile, uint64_t rows) {
    return I / rows * (P / tile + std::min(P, E / 2)) + Ish / rows * ((T + tile - 1) / tile);
  };
  if (P > 16 * E && items(64, 256) >= 128) return {64, 16};
  return {16, items(16, 128) >= 256 ? 8 : 4};
}

hipError_t launch_grouped_q4k(const Launch& K, const mr_layer& L, const float* x, uint32_t T, const int32_t* idx,
                              const float* w, float* y, void* scratch, const float* resid) {
  const int k = (int)L.d.top_k, E = (int)L.E, H = (int)L.H, I = (int)L.I, Ish = L.d.sh_gate ? (int)L.Ish : 0;
  // The kernels address the images of a call's rows within kPast bytes: more tokens than that
  // holds run in parts (a token's result depends on that token alone).
  const uint32_t T_max = (uint32_t)((uint64_t)kPast / img_bytes(1, (uint64_t)H));
  if (T > T_max) {
    for (uint32_t t0 = 0; t0 < T; t0 += T_max) {
      const hipError_t e = launch_grouped_q4k(K, L, x + (size_t)t0 * H, std::min(T_max, T - t0), idx + (size_t)t0 * k,
                                              w + (size_t)t0 * k, y + (size_t)t0 * H, scratch,
                                              resid ? resid + (size_t)t0 * H : nullptr);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  const int P = (int)T * k;
  const Q4Plan p = q4_plan(T, k, E, I, H, Ish);
  char* b = static_cast<char*>(scratch);
  auto f32_at = [&](uint64_t o) { return reinterpret_cast<float*>(b + o); };
  auto i32_at = [&](uint64_t o) { return reinterpret_cast<int32_t*>(b + o); };
  auto u8_at = [&](uint64_t o) { return reinterpret_cast<uint8_t*>(b + o); };
  const Q4Items c = q4_items((uint64_t)T, (uint64_t)k, (uint64_t)E, (uint64_t)I, (uint64_t)Ish);
  const int tile = c.tile;
  const GroupOut go{i32_at(p.pair_tok), f32_at(p.pair_w),   i32_at(p.pair_of), i32_at(p.exp_off),
                    i32_at(p.tile_off), i32_at(p.tile_exp), i32_at(p.hist)};
  hipError_t e;
  if ((e = launch_group(K, idx, w, P, k, E, tile, go)) != hipSuccess) return e;
  float* sig = Ish ? f32_at(p.sig) : nullptr;
  {
    ProfScope ps(K, "split_q4k");
    hipLaunchKernelGGL(k_split_f16, dim3(T), dim3(256), 0, K.s, x, H, u8_at(p.xo), f32_at(p.xp),
                       Ish ? L.d.sh_gate_inp : nullptr, sig);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  const uint64_t tiles = group_tiles_max(P, E, tile), sh_tiles = Ish ? (T + tile - 1) / tile : 0;
  GQ4Args a{};
  a.r.w0 = expert_loc(L.d.gate), a.r.w1 = expert_loc(L.d.up), a.r.b0 = L.d.gate_bias, a.r.b1 = L.d.up_bias;
  a.r.img = u8_at(p.xo), a.r.pinv = f32_at(p.xp), a.r.himg = u8_at(p.himg), a.r.hpinv = f32_at(p.hp);
  a.r.M = I, a.r.K = H, a.r.act = (int)L.d.act;
  if (Ish) {
    a.s.w0 = expert_loc(L.d.sh_gate), a.s.w1 = expert_loc(L.d.sh_up);
    a.s.img = a.r.img, a.s.pinv = a.r.pinv, a.s.himg = u8_at(p.hsimg), a.s.hpinv = f32_at(p.hsp);
    a.s.M = Ish, a.s.K = H, a.s.act = MR_ACT_SILU;
    a.sh_T = (int)T;
  }
  a.pair_tok = go.pair_tok, a.pair_w = go.pair_w, a.exp_off = go.exp_off, a.tile_off = go.tile_off, a.tile_exp = go.tile_exp;
  a.E = E, a.alpha = L.d.alpha, a.limit = L.d.limit;
  {
    ProfScope ps(K, "grouped_q4k_gateup");
    if (tile == 64)
      launch_q4<true, 4, 16>(K, a, tiles, sh_tiles);
    else if (c.gu_waves == 8)
      launch_q4<true, 1, 8>(K, a, tiles, sh_tiles);
    else
      launch_q4<true, 1, 4>(K, a, tiles, sh_tiles);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (tile != 64) {
    ProfScope ps(K, "split_h");
    const int64_t n0 = (int64_t)P * (I / 256), n1 = (int64_t)T * (Ish / 256);
    hipLaunchKernelGGL(k_split_h, dim3((unsigned)((n0 + n1 + 3) / 4)), dim3(256), 0, K.s, u8_at(p.himg), f32_at(p.hp), n0,
                       Ish ? u8_at(p.hsimg) : nullptr, Ish ? f32_at(p.hsp) : nullptr, n1);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  GQ4Args d{};
  d.r.w0 = expert_loc(L.d.down);
  d.r.img = u8_at(p.himg), d.r.pinv = f32_at(p.hp), d.r.out = f32_at(p.xo), d.r.M = H, d.r.K = I;
  if (Ish) {
    d.s.w0 = expert_loc(L.d.sh_down);
    d.s.img = u8_at(p.hsimg), d.s.pinv = f32_at(p.hsp), d.s.out = f32_at(p.osh), d.s.M = H, d.s.K = Ish;
    d.sh_T = (int)T;
  }
  d.exp_off = go.exp_off, d.tile_off = go.tile_off, d.tile_exp = go.tile_exp, d.E = E;
  {
    ProfScope ps(K, "grouped_q4k_down");
    if (tile == 64)
      launch_q4<false, 4, 4>(K, d, tiles, sh_tiles);
    else
      launch_q4<false, 1, 4>(K, d, tiles, sh_tiles);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return launch_combine(K, f32_at(p.xo), go.pair_of, idx, w, L.d.down_bias, T, k, H, Ish ? f32_at(p.osh) : nullptr, sig,
                        resid, y);
}

}  // namespace mr
