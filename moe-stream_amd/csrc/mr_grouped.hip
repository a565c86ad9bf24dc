// mr_grouped.hip -- multi-token (prefill / batched) MXFP4 MoE experts as grouped
// GEMMs on the gfx950 scaled MX-fp4 MFMA.
//
// The reference runs each expert once over all of its tokens: index_select of
// the expert's tokens, gate/up/act/down, x routing weight, index_add back
// (layer.rs:2148-2183; CPU: mxfp4_matmul per expert, layer.rs:1449-1514). Here:
//   k_group       (token, slot) pairs grouped by expert; per-expert pair offsets and
//                 pair tile offsets (tiles of 16, 32 or 64 pairs) and each tile's expert; pair
//                 index of every (token, slot).
//   k_split_rows  x rows -> e4m3 B images (terms 0-2 of the split of each 32-element block).
//   k_grouped_gemm<true>   gate and up for one (expert, 128-row tile, pair tile):
//                 A = native MXFP4 weight rows, B = the pairs' x images; epilogue
//                 bias + activation x routing weight, split into the h images
//                 [pair][I/32] (the split of k_split_rows).
//   k_grouped_gemm<false>  down for one (expert, 256-row tile, pair tile) on the
//                 h images -> o [pair][H].
//   k_combine     y[t] = sum over t's pairs in ascending expert order of
//                 (o + w*b_down) (the order of layer.rs:1092-1106).
// Every weight byte of an expert is read by the pair tiles of its
// row tiles; work items are laid out so those repeats, and the repeats of the
// pairs' activation images over row tiles, hit the same XCD's L2.
#include "mr_device.h"
#include "mr_fused_common.h"
#include "mr_internal.h"
#include "mr_mx_mfma.h"

#include <algorithm>
#include <cmath>
#include <climits>
#include <type_traits>

namespace mr {

// Terms of the activation split that the grouped GEMMs read, and all that their splits
// compute and write (the images keep the 4-term layout; term 3 is left unwritten).
constexpr int kGemmTerms = 3;

constexpr int kXcds = 8;        // MI355X accelerator complex dies (one L2 each)
constexpr int kMaxSteps = 32;   // K steps (4 blocks) per row: K <= 4096

// ---- grouping ---------------------------------------------------------------------------
// Count the (token, slot) entries of every expert, lay the experts out in order (exp_off; in
// tiles of `tile` pairs: tile_off, and each tile's expert) and give every entry a position inside
// its expert's range by an LDS counter. The order of the entries inside an expert depends on
// timing, but nothing computed from them does: each pair's GEMM column and epilogue depend on
// that pair alone, and a token's pairs are combined in ascending expert order, which the ranges
// fix.
// A workgroup takes kGroupEntries entries, held in registers between the count and the placement.
// More entries take several workgroups: k_group_count writes each one's counts, and in k_group
// every workgroup adds up the counts of those before it (32,768 entries of 128 experts: 103 us
// in one workgroup of 256 threads that read them twice, 11 us for the two launches).
constexpr int kGroupJ = 8;  // entries per thread, loaded together
constexpr int kGroupThreads = 1024;
constexpr int kGroupEntries = kGroupThreads * kGroupJ;

__device__ __forceinline__ void group_load(const int32_t* __restrict__ idx, int P, int E, int q0, int (&ev)[kGroupJ]) {
#pragma unroll
  for (int j = 0; j < kGroupJ; ++j) {
    const int q = q0 + kGroupThreads * j;
    ev[j] = q < P ? min(max(idx[q], 0), E - 1) : -1;
  }
}

__global__ __launch_bounds__(kGroupThreads) void k_group_count(const int32_t* __restrict__ idx, int P, int E,
                                                               int32_t* __restrict__ hist) {
  __shared__ int cnt[1024];
  const int tid = threadIdx.x;
  cnt[tid] = 0;
  int ev[kGroupJ];
  group_load(idx, P, E, blockIdx.x * kGroupEntries + tid, ev);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kGroupJ; ++j)
    if (ev[j] >= 0) atomicAdd(&cnt[ev[j]], 1);
  __syncthreads();
  if (tid < E) hist[blockIdx.x * E + tid] = cnt[tid];
}

__global__ __launch_bounds__(kGroupThreads) void k_group(const int32_t* __restrict__ idx, const float* __restrict__ w,
                                                         int P, int k, int E, int tile, GroupOut o) {
  __shared__ int cnt[1024], toff[1025], wsum[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q0 = blockIdx.x * kGroupEntries + tid;
  cnt[tid] = 0;
  int ev[kGroupJ];
  float wv[kGroupJ];
  group_load(idx, P, E, q0, ev);
#pragma unroll
  for (int j = 0; j < kGroupJ; ++j) wv[j] = ev[j] >= 0 ? w[q0 + kGroupThreads * j] : 0.f;
  __syncthreads();
  int c = 0, before = 0;  // this thread's expert (tid): entries in all, and in earlier workgroups
  if (gridDim.x == 1) {
#pragma unroll
    for (int j = 0; j < kGroupJ; ++j)
      if (ev[j] >= 0) atomicAdd(&cnt[ev[j]], 1);
    __syncthreads();
    c = cnt[tid];
  } else if (tid < E) {
    for (int b = 0; b < (int)gridDim.x; ++b) {
      const int v = o.hist[b * E + tid];
      c += v;
      before += b < (int)blockIdx.x ? v : 0;
    }
  }
  const int tc = (c + tile - 1) / tile;
  int po = c, to = tc;  // inclusive prefix over the wave, then over the workgroup, then exclusive
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int a = __shfl_up(po, d, 64), b = __shfl_up(to, d, 64);
    if (lane >= d) po += a, to += b;
  }
  if (lane == 63) wsum[0][wave] = po, wsum[1][wave] = to;
  __syncthreads();
  po -= c, to -= tc;
  for (int v = 0; v < wave; ++v) po += wsum[0][v], to += wsum[1][v];
  if (tid < E) {
    cnt[tid] = po + before;  // becomes the next free position
    toff[tid] = to;
    if (blockIdx.x == 0) o.exp_off[tid] = po, o.tile_off[tid] = to;
    if (tid == E - 1) {
      toff[E] = to + tc;
      if (blockIdx.x == 0) o.exp_off[E] = po + c, o.tile_off[E] = to + tc;
    }
  }
  __syncthreads();
  const int n_tiles = toff[E];
  for (int t = blockIdx.x * kGroupThreads + tid; t < n_tiles; t += gridDim.x * kGroupThreads) {
    int lo = 0, hi = E;  // toff[lo] <= t < toff[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (toff[mid] <= t) lo = mid; else hi = mid;
    }
    o.tile_exp[t] = lo;
  }
#pragma unroll
  for (int j = 0; j < kGroupJ; ++j) {
    if (ev[j] >= 0) {
      const int q = q0 + kGroupThreads * j;
      const int pos = atomicAdd(&cnt[ev[j]], 1);
      o.pair_tok[pos] = q / k, o.pair_w[pos] = wv[j], o.pair_of[q] = pos;
    }
  }
}

// ---- activation rows -> B images ------------------------------------------------------------
// Row r of `src` (D floats) -> img[r][D/32][kImgBytes] + sc[r][D/32]; 8 lanes per block, on a
// (block groups of 32, rows) grid (rows past gridDim.y loop).
__global__ __launch_bounds__(256) void k_split_rows(const float* __restrict__ src, int n_rows, int D,
                                                    uint8_t* __restrict__ img, uint32_t* __restrict__ sc) {
  const int nb = D >> 5;
  const int b = blockIdx.x * 32 + (threadIdx.x >> 3);
  const int m = threadIdx.x & 7;
  const bool in = b < nb;  // the same for the block's 8 lanes (the split's DPP stays in them)
  for (int r = blockIdx.y; r < n_rows; r += gridDim.y) {
    const float* p = src + (size_t)r * D + min(b, nb - 1) * 32 + 2 * m;
    const f32x2 lo = *reinterpret_cast<const f32x2*>(p);       // elements 2m, 2m+1
    const f32x2 hi = *reinterpret_cast<const f32x2*>(p + 16);  // elements 2m+16, 2m+17
    uint32_t codes[kTerms], scales;
    split_block8<kGemmTerms>(lo.x, hi.x, lo.y, hi.y, codes, scales);
    if (in) {
      const size_t bb = (size_t)r * nb + b;
      uint32_t* dst = reinterpret_cast<uint32_t*>(img + bb * kImgBytes);
#pragma unroll
      for (int t = 0; t < kGemmTerms; ++t) dst[t * 8 + m] = codes[t];
      if (m == 0) sc[bb] = scales;
    }
  }
}

// ---- grouped GEMM -------------------------------------------------------------------------
struct GroupedArgs {
  ExpertLoc w0;  // gate (GATEUP) or down
  ExpertLoc w1;  // up (GATEUP)
  const float* b0;  // gate bias [E][M] (GATEUP) or null
  const float* b1;  // up bias
  const uint8_t* img;    // B images [rows][K/32][kImgBytes]
  const uint32_t* isc;   // [rows][K/32]
  const int32_t* pair_tok;  // B row of pair p (GATEUP: its token) or null (row = p)
  const float* pair_w;      // GATEUP: routing weight of pair p, or null (weight 1)
  const int32_t* exp_off;
  const int32_t* tile_off;
  const int32_t* tile_exp;
  int single_p;  // > 0: one expert (e = 0) over pairs 0 .. single_p - 1 (the shared expert over
                 // every token); exp_off, tile_off and tile_exp are not read
  float* out;        // [P][M] (down)
  uint8_t* himg;     // GATEUP: the down input images [P][M/32][kImgBytes]
  uint32_t* hsc;     // GATEUP: their scale words [P][M/32]
  int M, K, E;
  int act;
  float alpha, limit;
};

// Grouped GEMM work item: (expert e, row tile, tile of 16 kPG pairs); 4 waves. A wave owns kGT
// 16-row A tiles (gate/up: 32 gate rows and the same 32 up rows, so that the activation and the
// split of the down input image run in registers, 128 rows per item; down: 4 x 64 = 256 rows)
// and the tile's pairs as kPG groups of 16.
// The MFMAs take the first kGemmTerms = 3 e4m3 terms of the pairs' activation split (the
// residual after three terms is below 2^-12 of each 32-element block's max, bf16 operands
// hold 8 significant bits). A K step holds 4 weight blocks; MFMA m of the step takes term m of
// all four: K block j of MFMA m is weight block j (its A operand: native MXFP4 codes and the
// block's scale byte, read per lane) against term m of block j of the 16 pairs (with that
// term's scale byte). A lane's A operand is then the same in the step's 3 MFMAs, so each A
// window is read from LDS and aligned once per step, and D accumulates the term-summed dot
// product of row x pair: no term columns to add afterwards, 16 pairs per MFMA, and a wave
// keeps kGT x kPG accumulator tiles.
// K advances 4 blocks per step:
//   A: each row's 68 bytes of a step as 6 aligned 16-byte pieces, lane-contiguous (a wave
//      load covers ~11 rows' contiguous bytes; 20-byte windows loaded per lane straight
//      from global cost 3x the L1 accesses), kAhead steps ahead in registers, then written to
//      the wave's LDS slice, from which the 4 lanes of a row read the same block window;
//   B: the step's pairs x 4 blocks x the 96 bytes of terms 0-2 of their images (6 KB per pair
//      group) and their scale words, one step ahead in registers (the images are L2 hits), then
//      written to a double-buffered LDS stage shared by the 4 waves. (Direct global->LDS loads
//      would save the registers, but the compiler then waits for all of them before any LDS
//      read, which serialises the prefetch.)
// What bounds it: the per-step chain (stage written, barrier, LDS reads, alignment, MFMAs) at two
// or three waves per SIMD; a step on 64 pairs issues 48 MFMAs per wave for one such chain, on 32
// pairs 24. 64 pairs fit the registers since the A loads take a scalar base and 32-bit offsets
// (64-bit addresses with 64-bit limits: 239 VGPRs at 32 pairs, now 194) and the B operands are
// read per pair group. 2,039 tokens of 4 in 32 experts of 2880 x 2880: 610 + 308 us for the two
// launches in 32-pair tiles with the expert searched in the tile offsets, now 524 + 269 us (512
// TFLOP/s of layer arithmetic, 3 times that issued). 4 tokens: 46 + 28 us, now 40 + 25 us in
// 16-pair tiles.
constexpr int kGW = 4;               // waves per work item
#ifndef MR_GROUPED_GT_GU
#define MR_GROUPED_GT_GU 4
#endif
#ifndef MR_GROUPED_GT_DN
#define MR_GROUPED_GT_DN 4
#endif
// 16-row A tiles per wave (gate/up, down) and the rows of a matrix per work item
template <bool GATEUP> constexpr int kGTof = GATEUP ? MR_GROUPED_GT_GU : MR_GROUPED_GT_DN;
template <bool GATEUP> constexpr int kRowsOf = (GATEUP ? kGW / 2 : kGW) * kGTof<GATEUP> * 16;
constexpr int kAPR = 6;                            // A pieces per row and step: 68 bytes at any offset
#ifndef MR_GROUPED_AROW
#define MR_GROUPED_AROW 104
#endif
constexpr int kARow = MR_GROUPED_AROW;  // LDS bytes per A row: 26 dwords, so 16 rows fall in 16 different banks
static_assert(kARow % 4 == 0 && kARow >= 6 * 16, "an A row holds a step's 6 pieces, dword-aligned");
constexpr int kBBuf = 2;                           // B stages in LDS
static_assert(kTerms == 4, "images of 4 terms (8 parts of 16 bytes per block); the GEMMs read terms 0-2");
constexpr int kBParts = 4 * 6;  // 16-byte parts of a pair per K step: 4 blocks x terms 0-2

template <bool GATEUP, int kPG>
__global__ __launch_bounds__(256, kPG == 1 ? 3 : 2) void k_grouped_gemm(GroupedArgs a) {
  constexpr int kPairTile = 16 * kPG;
  // LDS slot (16 bytes) of part q (0 .. 5) of (pair pr, block b) in a B stage: (6 b + q) kBRow + pr
  constexpr int kBRow = kPairTile + 1;
  constexpr int kBStep = kBParts * kBRow * 16;  // bytes of a stage
  constexpr int kBPieces = (kPairTile * kBParts + 255) / 256;  // 16-byte pieces loaded per thread and step
  __shared__ __align__(16) uint8_t bst[kBBuf][kBStep];
  __shared__ __align__(16) uint32_t bsc[kBBuf][kPairTile * 4];
  constexpr int kGT = kGTof<GATEUP>;               // 16-row A tiles per wave
  constexpr int kASlots = kGT * 16 * kAPR;         // A pieces per wave and step
  constexpr int kAK = (kASlots + 63) / 64;         // A piece loads per lane and step
  __shared__ __align__(16) uint8_t ast[kGW][kGT * 16 * kARow];
  __shared__ float bias_s[GATEUP ? 2 * (kGW / 2) * kGT * 16 + kPairTile : 1];  // GATEUP: the tile's gate,
                                                                               // up biases, pair weights
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: wave-level branches stay scalar
  const int i = lane & 15, g = lane >> 4;
  constexpr int kRows = kRowsOf<GATEUP>;  // rows of a matrix per item
  // Work items are ordered (expert, row tile, pair tile of the expert), and each XCD
  // (workgroups are dispatched round-robin over kXcds) takes one contiguous range of them:
  // the items that share an expert's row tile (A) or its pairs' images (B) run on the same
  // XCD and meet in its L2.
  const int n_rt = (a.M + kRows - 1) / kRows;
  const bool single = a.single_p > 0;
  const int n_tiles = single ? (a.single_p + kPairTile - 1) / kPairTile : a.tile_off[a.E];
  const int n_work = n_rt * n_tiles;
  const int per_xcd = (n_work + kXcds - 1) / kXcds;
  const int loc = blockIdx.x / kXcds;
  const int w = (blockIdx.x % kXcds) * per_xcd + loc;
  if (loc >= per_xcd || w >= n_work) return;  // uniform: no work item for this workgroup
  // expert: n_rt * tile_off[e] <= w < n_rt * tile_off[e+1], so pair tile w / n_rt is one of its own
  const int e = single ? 0 : a.tile_exp[w / n_rt];
  const int e_beg = single ? 0 : a.exp_off[e], e_end = single ? a.single_p : a.exp_off[e + 1];
  const int nt_e = single ? n_tiles : a.tile_off[e + 1] - a.tile_off[e];
  const int wl = w - (single ? 0 : n_rt * a.tile_off[e]);
  const int rt = wl / nt_e, tl = wl - rt * nt_e;
  const int p0 = e_beg + tl * kPairTile;
  const int np = min(kPairTile, e_end - p0);
  const int npg = (np + 15) >> 4;  // pair groups holding pairs (uniform)

  const int nbK = a.K >> 5, S = (nbK + 3) >> 2;
  const uint64_t rb = (uint64_t)nbK * 17;
  // Rows of this wave: gate/up: tiles 0 .. kTR-1 are the gate rows wrow0 .. wrow0 + 16 kTR - 1
  // and tiles kTR .. 2kTR-1 the same up rows, so that a lane holds the gate and up values of
  // the same (row, pair) for the activation; down: kGT tiles of consecutive rows.
  constexpr int kTR = GATEUP ? kGT / 2 : kGT;  // 16-row tiles per matrix of a wave
  static_assert(!GATEUP || kGT == 4, "gate/up: two gate and two up tiles, one 32-row split block per wave");
  const int wrow0 = rt * kRows + wave * (kTR * 16);
  if (GATEUP) {  // read by the epilogue (after the K loop's barriers)
    for (int q = tid; q < 2 * kRows + kPairTile; q += kGW * 64) {
      if (q < 2 * kRows) {
        const int mat = q >= kRows, orow = rt * kRows + q - mat * kRows;
        const float* bsrc = mat ? a.b1 : a.b0;
        bias_s[q] = (bsrc && orow < a.M) ? bsrc[(size_t)e * a.M + orow] : 0.f;
      } else {
        bias_s[q] = a.pair_w ? a.pair_w[p0 + min(q - 2 * kRows, np - 1)] : 1.f;
      }
    }
  }
  const uint8_t* Wm[2] = {expert_at(a.w0, e), GATEUP ? expert_at(a.w1, e) : expert_at(a.w0, e)};
  // This lane's row i: its rows in every tile of one matrix are 16 rows (a multiple of 16
  // bytes) apart, so the byte position of a block in its 16-byte piece is the same for all of
  // them (lead0[matrix]; the gate and up matrices may start at different offsets).
  uint32_t lead0[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
    lead0[mt] = (uint32_t)(reinterpret_cast<uintptr_t>(Wm[mt]) + (uintptr_t)min(wrow0 + i, a.M - 1) * rb) & 15u;
  // A piece slots of this lane: slot k*64 + lane = (tile, row, piece) of the wave's rows
  // A load's matrix is the same in all lanes: its 16-byte aligned base stays in scalar registers
  // and a lane keeps 32-bit offsets (a matrix holds at most 4,096 rows of 2,176 bytes): that of
  // its piece at step 0, unaligned, and that of the row's last piece.
  static_assert((16 * kAPR * kTR) % 64 == 0, "a load's slots lie in one matrix");
  const uint8_t* abase[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
    abase[mt] = reinterpret_cast<const uint8_t*>(reinterpret_cast<uintptr_t>(Wm[mt]) & ~(uintptr_t)15);
  uint32_t aoff[kAK], alast[kAK];
  int aslot[kAK];
#pragma unroll
  for (int k = 0; k < kAK; ++k) {
    const int sl = min(k * 64 + lane, kASlots - 1);
    const int tt = sl / (16 * kAPR), rr = (sl / kAPR) % 16;
    const uint32_t row = ((uint32_t)reinterpret_cast<uintptr_t>(Wm[k * 64 / (16 * kAPR * kTR)]) & 15u) +
                         (uint32_t)min(wrow0 + 16 * (tt % kTR) + rr, a.M - 1) * (uint32_t)rb;
    aoff[k] = row + 16u * (uint32_t)(sl % kAPR);
    alast[k] = (row + (uint32_t)rb - 1u) & ~15u;
    aslot[k] = (tt * 16 + rr) * kARow + (sl % kAPR) * 16;
  }

  // B pieces of this thread: piece j*256 + tid = (pair, block, part) in that order, so
  // consecutive lanes read consecutive parts of a block (threads past the last piece repeat it)
  const uint8_t* bsrc[kBPieces];
  int bslot[kBPieces], bblk[kBPieces];
#pragma unroll
  for (int j = 0; j < kBPieces; ++j) {
    const int q = min(j * 256 + tid, kPairTile * kBParts - 1), part = q % 6, blk = (q / 6) & 3, pr = q / 24;
    bslot[j] = (blk * 6 + part) * kBRow + pr;
    bblk[j] = blk;
    const int p = p0 + min(pr, np - 1);
    const int r = a.pair_tok ? a.pair_tok[p] : p;
    bsrc[j] = a.img + (size_t)r * nbK * kImgBytes + part * 16;
  }
  const uint32_t* ssrc;  // scale word tid (the first 4 kPairTile threads): pair tid/4, block tid%4
  {
    const int p = p0 + min(tid >> 2, np - 1);
    const int r = a.pair_tok ? a.pair_tok[p] : p;
    ssrc = a.isc + (size_t)r * nbK;
  }
  struct BRegs {
    i32x4 v[kBPieces];
    uint32_t sc;
  };
  auto load_b = [&](int st, BRegs& br) {
#pragma unroll
    for (int j = 0; j < kBPieces; ++j) {
      const size_t boff = (size_t)min(4 * st + bblk[j], nbK - 1) * kImgBytes;
      br.v[j] = *(const __attribute__((address_space(1))) i32x4*)(bsrc[j] + boff);
    }
    br.sc = *(const __attribute__((address_space(1))) uint32_t*)(ssrc + min(4 * st + (tid & 3), nbK - 1));
  };
  auto store_b = [&](const BRegs& br, int buf) {
#pragma unroll
    for (int j = 0; j < kBPieces; ++j) *reinterpret_cast<i32x4*>(&bst[buf][bslot[j] * 16]) = br.v[j];
    if (wave < kPG) bsc[buf][tid] = br.sc;  // 4 kPairTile words: kPG waves
  };
  auto load_a = [&](int st, i32x4 (&apv)[kAK]) {  // pieces past the row end read its last piece
#pragma unroll
    for (int k = 0; k < kAK; ++k) {
      const uint32_t src = min((aoff[k] + 68u * (uint32_t)st) & ~15u, alast[k]);
      apv[k] = *(const __attribute__((address_space(1))) i32x4*)(abase[k * 64 / (16 * kAPR * kTR)] + src);
    }
  };
  auto store_a = [&](const i32x4 (&apv)[kAK]) {  // slots past kASlots are not stored
#pragma unroll
    for (int k = 0; k < kAK; ++k)
      if (k * 64 + 64 <= kASlots || k * 64 + lane < kASlots)
        {
          if constexpr (kARow % 8 == 0) {  // 8-byte aligned: rows are kARow bytes apart
            uint64_t* d = reinterpret_cast<uint64_t*>(&ast[wave][aslot[k]]);
            d[0] = ((uint64_t)(uint32_t)apv[k][1] << 32) | (uint32_t)apv[k][0];
            d[1] = ((uint64_t)(uint32_t)apv[k][3] << 32) | (uint32_t)apv[k][2];
          } else {
            uint32_t* d = reinterpret_cast<uint32_t*>(&ast[wave][aslot[k]]);
            d[0] = (uint32_t)apv[k][0], d[1] = (uint32_t)apv[k][1], d[2] = (uint32_t)apv[k][2], d[3] = (uint32_t)apv[k][3];
          }
        }
  };
  // MFMA m of a step takes term m of the activation split for all 4 blocks of the step. Lane
  // (pair i of the group, K group g): its A operand is weight block g of the step in all three
  // MFMAs; its B bytes 0-15 are K [16g, 16g+16), half g%2 of K block g/2, and bytes 16-31 half
  // g%2 of K block 2 + g/2, i.e. part 2m + g%2 of (pair i, block g/2) and of (pair i, block
  // 2 + g/2), 12 kBRow slots further; its B scale byte is (pair i, block g, term m) at 16i + 4g + m.
  // A stage's slots are part-major: the 16 lanes of a read take 16 neighbouring slots, and the
  // odd row length spreads the consecutive parts that a wave writes over the banks.
  const int brd0 = (((g >> 1) * 6 + (g & 1)) * kBRow + i) * 16;
  const int sc_lane = i * 16 + 4 * g;

  // A loads run kAhead steps ahead: two (a register set for each parity) where a step is short;
  // one step of 4 pair groups covers them, and the second set would spill. Measured (the whole
  // call, us, 32 experts of 2880 x 2880, 4 per token), two against one: 128 tokens on 2 groups
  // 192 / 197, 32 tokens on 1 group 156 / 160, 2039 tokens on 4 groups 787 / 780.
  constexpr int kAhead = kPG == 4 ? 1 : 2;
  i32x4 apv[kAhead][kAK];
  BRegs bR;
  load_b(0, bR);
#pragma unroll
  for (int d = 0; d < kAhead; ++d) load_a(min(d, S - 1), apv[d]);

  f32x4 acc[kGT][kPG];
#pragma unroll
  for (int tt = 0; tt < kGT; ++tt)
#pragma unroll
    for (int pg = 0; pg < kPG; ++pg) acc[tt][pg] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Step st: A pieces in register set st % 2 (loaded two steps ahead), B pieces in one
  // register set (one step ahead: the images are L2 hits), B in LDS buffer st % 2. Every step
  // issues the same loads, B first (past the last step: the last step's data again), so the
  // compiler's waits before the LDS writes count exactly the loads issued after them.
  // `part` (a std::bool_constant): the step may hold blocks past the row end. Only such steps
  // test every A window for it; full steps compile without those selects.
  auto step = [&](int st, i32x4 (&cur)[kAK], auto part) {
    constexpr bool kPart = decltype(part)::value;
    const int buf = st % kBBuf;
    store_a(cur);      // this wave's A slice (its reads of step st-1 are done: LDS ops stay in order)
    store_b(bR, buf);  // buffer st % 2 was last read in step st-2, before the previous barrier
    __syncthreads();   // step st's B stage is complete
    load_b(min(st + 1, S - 1), bR);
    load_a(min(st + kAhead, S - 1), cur);
    const uint8_t* bb_base = &bst[buf][0];
    const uint8_t* sc_base = reinterpret_cast<const uint8_t*>(&bsc[buf][0]);
    uint32_t wo[2];  // per matrix: block g's scale byte in the row's LDS slice (68 st = 4 st mod 16)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) wo[mt] = ((lead0[mt] + 4u * (uint32_t)st) & 15u) + 17u * (uint32_t)g;
    // B operands of (term mm, pair group pg), read two ahead of their MFMAs; the A operands (this
    // lane's block g of each tile's row i) once per step for all MFMAs. A block past the row end
    // (read inside the LDS stage) gets zero codes, so it adds nothing.
    struct BOps {
      i32x4 b[2];
      int sb;
    };
    auto read_b = [&](int n, BOps& o) {
      const int mm = n / kPG, pg = n % kPG;
      const uint8_t* bp = bb_base + brd0 + (2 * mm * kBRow + 16 * pg) * 16;
      o.b[0] = *reinterpret_cast<const i32x4*>(bp);
      o.b[1] = *reinterpret_cast<const i32x4*>(bp + 12 * kBRow * 16);
      o.sb = (int)sc_base[sc_lane + mm + pg * 256];
    };
    RawBlk r[kGT];
#pragma unroll
    for (int tt = 0; tt < kGT; ++tt) {
      const uint32_t* wp = reinterpret_cast<const uint32_t*>(&ast[wave][(tt * 16 + i) * kARow + (wo[tt / kTR] & ~3u)]);
      r[tt].d[0] = wp[0], r[tt].d[1] = wp[1], r[tt].d[2] = wp[2], r[tt].d[3] = wp[3], r[tt].d[4] = wp[4];
    }
    BOps o[3];
    read_b(0, o[0]);
    read_b(1, o[1]);
    const bool valid = !kPart || 4 * st + g < nbK;
    AOp ao[kGT];
    int sa[kGT];
#pragma unroll
    for (int tt = 0; tt < kGT; ++tt) {
      // byte alignment by v_alignbyte (a shift of 4 bytes selects the upper dword): the same
      // as shifting the dword pair right by t bytes, which the compiler would otherwise do
      // through a stack copy of the window
      const uint32_t w3 = wo[tt / kTR] & 3u, t = w3 + 1u;  // the codes start t bytes into the window (1..4)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t v = t == 4u ? r[tt].d[q + 1] : __builtin_amdgcn_alignbyte(r[tt].d[q + 1], r[tt].d[q], t);
        ao[tt].q[q] = valid ? v : 0u;
      }
      sa[tt] = valid ? (int)((r[tt].d[0] >> (8u * w3)) & 0xFFu) : 127;
    }
#pragma unroll
    for (int n = 0; n < kGemmTerms * kPG; ++n) {
      if (n + 2 < kGemmTerms * kPG) read_b(n + 2, o[(n + 2) % 3]);
      const int pg = n % kPG;
      if (pg < npg) {
        const BOps& c = o[n % 3];
        const i32x8 B = {c.b[0][0], c.b[0][1], c.b[0][2], c.b[0][3], c.b[1][0], c.b[1][1], c.b[1][2], c.b[1][3]};
#pragma unroll
        for (int tt = 0; tt < kGT; ++tt)  // tiles past M repeat row M-1; their rows are not stored
          acc[tt][pg] = mfma_op(ao[tt], sa[tt], B, c.sb, acc[tt][pg]);
      }
    }
  };
  // Steps 0 .. nbK/4 - 1 hold only blocks inside the row; the one or two steps after the loop
  // (the last one possibly partial) run the checked variant.
  const int s_full = nbK >> 2;
  int st = 0;
  for (; st + 1 < s_full; st += 2) {
    step(st, apv[0], std::false_type{});
    step(st + 1, apv[kAhead - 1], std::false_type{});
  }
  if (st < S) {
    step(st, apv[0], std::true_type{});
    if (st + 1 < S) step(st + 1, apv[kAhead - 1], std::true_type{});
  }

  // Epilogue: acc[tt][pg][r] of lane (i, g) is row wrow0 + 16 tt + 4g + r x pair 16 pg + i.
  if constexpr (!GATEUP) {  // down: the lane's 4 consecutive rows of a pair as one 16-byte store
#pragma unroll
    for (int tt = 0; tt < kGT; ++tt)
#pragma unroll
      for (int pg = 0; pg < kPG; ++pg) {
        const int pl = pg * 16 + i, row = wrow0 + 16 * tt + 4 * g;  // M % 32 == 0: row < M -> row + 3 < M
        if (pl < np && row < a.M) *reinterpret_cast<f32x4*>(a.out + (size_t)(p0 + pl) * a.M + row) = acc[tt][pg];
      }
    return;
  }
  // Gate/up: lane (i, g) holds gate rows 4g .. 4g+3 and 16+4g .. 16+4g+3 of the wave's 32
  // rows (tiles 0, 1) and the same up rows (tiles 2, 3) for pairs i and 16 + i. h = act(gate +
  // b_g, up + b_u) x routing weight is formed in registers and the wave's 32 rows of each pair,
  // one block of the down input image, are split there: the lane holds split lanes 2g and 2g+1
  // (elements 4g, 4g+16, 4g+1, 4g+17 and 4g+2, 4g+18, 4g+3, 4g+19; the split of k_split_rows),
  // the block's other elements are in lanes xor 16 and xor 32.
  const int lr0 = wave * (kTR * 16);  // the wave's first row within the item (bias_s index)
  const int nbM = a.M >> 5;
#pragma unroll
  for (int pg = 0; pg < kPG; ++pg) {
    if (pg >= npg) break;  // uniform
    const int pl = pg * 16 + i;
    const float pw = bias_s[2 * kRows + min(pl, kPairTile - 1)];
    float hv[2][4];  // [tile][r]: row 16 tile + 4g + r
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int lr = lr0 + 16 * t2 + 4 * g + r;
        float gv = acc[t2][pg][r], uv = acc[2 + t2][pg][r];
        if (a.b0) gv = gv + bias_s[lr];
        if (a.b1) uv = uv + bias_s[kRows + lr];
        hv[t2][r] = (a.act == MR_ACT_SWIGLU_OAI ? swiglu_oai(gv, uv, a.alpha, a.limit) : silu_mul(gv, uv)) * pw;
      }
    uint32_t ca[kTerms], cb[kTerms], scales;
    split_block_x2<kGemmTerms>(hv[0][0], hv[1][0], hv[0][1], hv[1][1], hv[0][2], hv[1][2], hv[0][3], hv[1][3], ca, cb,
                               scales);
    if (pl < np && wrow0 < a.M) {  // M % 32 == 0: the wave's 32 rows are all inside
      const size_t bi = (size_t)(p0 + pl) * nbM + (wrow0 >> 5);
      uint32_t* dst = reinterpret_cast<uint32_t*>(a.himg + bi * kImgBytes);
#pragma unroll
      for (int t = 0; t < kGemmTerms; ++t)
        *reinterpret_cast<uint2*>(dst + t * 8 + 2 * g) = make_uint2(ca[t], cb[t]);
      if (g == 0) a.hsc[bi] = scales;
    }
  }
}

// ---- combine -----------------------------------------------------------------------------
// y[t][row] = sum over t's pairs in ascending pair index (= ascending expert) of
// o[pair][row] + w * b_down[e][row], then + sig[t] * o_sh[t][row] when a shared expert ran
// (layer.rs:1935-1951); with a residual input, y = resid + that (layer.rs:462-473; resid may be y:
// a thread reads what it overwrites). Added here it costs one read of h; as a launch of its own it
// read the sum back and wrote it again (2,039 tokens of 2880: 16 us after this kernel's 20; 4: 4.7).
// One thread per (token, 4 rows) on a (row groups, tokens) grid (tokens past gridDim.y loop); the
// token's (at most KM) pair indices stay in registers and are taken smallest first, and all of a
// thread's loads issue before the sums. H % 4 == 0.
template <int KM>
__global__ __launch_bounds__(256) void k_combine(const float* __restrict__ o, const int32_t* __restrict__ pair_of,
                                                 const int32_t* __restrict__ idx, const float* __restrict__ w,
                                                 const float* __restrict__ down_b, int T, int k, int H,
                                                 const float* __restrict__ o_sh, const float* __restrict__ sh_sig,
                                                 const float* resid, float* y) {
  const int row = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (row >= H) return;
  for (int t = blockIdx.y; t < T; t += gridDim.y) {
    int ps[KM];
#pragma unroll
    for (int s = 0; s < KM; ++s) ps[s] = s < k ? pair_of[t * k + s] : INT_MAX;
    f32x4 v[KM], bv[KM];
    float wv[KM];
#pragma unroll
    for (int r = 0; r < KM; ++r) {
      if (r < k) {
        int best = INT_MAX, bs = 0;
#pragma unroll
        for (int s = 0; s < KM; ++s)
          if (ps[s] < best) best = ps[s], bs = s;
#pragma unroll
        for (int s = 0; s < KM; ++s)
          if (s == bs) ps[s] = INT_MAX;
        v[r] = *reinterpret_cast<const f32x4*>(o + (size_t)best * H + row);
        if (down_b) {
          wv[r] = w[t * k + bs];
          bv[r] = *reinterpret_cast<const f32x4*>(down_b + (size_t)idx[t * k + bs] * H + row);
        }
      }
    }
    f32x4 hv = {0.f, 0.f, 0.f, 0.f};
    if (resid) hv = *reinterpret_cast<const f32x4*>(resid + (size_t)t * H + row);
    f32x4 sv = {0.f, 0.f, 0.f, 0.f};
    float sg = 0.f;
    if (o_sh) {
      sv = *reinterpret_cast<const f32x4*>(o_sh + (size_t)t * H + row);
      sg = sh_sig[t];
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < KM; ++r) {
      if (r < k) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float x = v[r][c];
          if (down_b) x = x + wv[r] * bv[r][c];
          acc[c] = acc[c] + x;
        }
      }
    }
    if (o_sh)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = acc[c] + sg * sv[c];
    if (resid)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = hv[c] + acc[c];
    *reinterpret_cast<f32x4*>(y + (size_t)t * H + row) = acc;
  }
}

// ---- host side -------------------------------------------------------------------------------
namespace {
constexpr uint64_t kAlign = 256;
uint64_t up(uint64_t v) { return (v + kAlign - 1) / kAlign * kAlign; }
struct GroupedPlan {
  uint64_t pair_tok, pair_w, pair_of, exp_off, tile_off, tile_exp, hist, sc_x, img_h, sc_h, xo;
  uint64_t img_hsh, sc_hsh, osh, sig, total;
};
GroupedPlan grouped_plan(uint64_t T, uint64_t k, uint64_t E, uint64_t I, uint64_t H, uint64_t Ish) {
  GroupedPlan p{};
  const uint64_t P = T * k;
  uint64_t o = 0;
  p.pair_tok = o, o += up(P * 4);
  p.pair_w = o, o += up(P * 4);
  p.pair_of = o, o += up(P * 4);
  p.exp_off = o, o += up((E + 1) * 4);
  p.tile_off = o, o += up((E + 1) * 4);
  p.tile_exp = o, o += up(group_tiles_max(P, E, kGroupTileMin) * 4);
  p.hist = o, o += up(group_hist_bytes(P, E));
  p.sc_x = o, o += up(T * (H / 32) * 4);
  p.img_h = o, o += up(P * (I / 32) * kImgBytes);
  p.sc_h = o, o += up(P * (I / 32) * 4);
  // the x images are last read by the gate/up launches and the down outputs first written by
  // the down launches: they share xo
  p.xo = o, o += up(std::max(T * (H / 32) * kImgBytes, P * H * 4));
  p.img_hsh = o, o += up(T * (Ish / 32) * kImgBytes);  // the shared expert (Ish = 0: none)
  p.sc_hsh = o, o += up(T * (Ish / 32) * 4);
  p.osh = o, o += up(Ish ? T * H * 4 : 0);
  p.sig = o, o += up(Ish ? T * 4 : 0);
  p.total = o;
  return p;
}
}  // namespace

uint64_t grouped_scratch_bytes(uint64_t T, uint64_t k, uint64_t E, uint64_t I, uint64_t H, uint64_t Ish) {
  return grouped_plan(T, k, E, I, H, Ish).total;
}

GroupedScratch grouped_scratch(const Scratch& s, uint64_t T, uint64_t k, uint64_t E, uint64_t I, uint64_t H,
                               uint64_t Ish) {
  const GroupedPlan p = grouped_plan(T, k, E, I, H, Ish);
  char* b = static_cast<char*>(s.grouped);
  GroupedScratch g{};
  g.pair_tok = reinterpret_cast<int32_t*>(b + p.pair_tok);
  g.pair_w = reinterpret_cast<float*>(b + p.pair_w);
  g.pair_of = reinterpret_cast<int32_t*>(b + p.pair_of);
  g.exp_off = reinterpret_cast<int32_t*>(b + p.exp_off);
  g.tile_off = reinterpret_cast<int32_t*>(b + p.tile_off);
  g.tile_exp = reinterpret_cast<int32_t*>(b + p.tile_exp);
  g.hist = reinterpret_cast<int32_t*>(b + p.hist);
  g.img_x = reinterpret_cast<uint8_t*>(b + p.xo);
  g.sc_x = reinterpret_cast<uint32_t*>(b + p.sc_x);
  g.img_h = reinterpret_cast<uint8_t*>(b + p.img_h);
  g.sc_h = reinterpret_cast<uint32_t*>(b + p.sc_h);
  g.obuf = reinterpret_cast<float*>(b + p.xo);
  g.img_hsh = reinterpret_cast<uint8_t*>(b + p.img_hsh);
  g.sc_hsh = reinterpret_cast<uint32_t*>(b + p.sc_hsh);
  g.osh = reinterpret_cast<float*>(b + p.osh);
  g.sig = reinterpret_cast<float*>(b + p.sig);
  return g;
}
// MXFP4 routed experts, and an MXFP4 shared expert of any width (a multiple of 32), which runs
// as one more group: every token, weight 1, SiLU, then its sigmoid gate in the combine.
bool grouped_supported(const mr_layer& L) {
  if (L.type != MR_GGML_MXFP4 || L.d.top_k > 16 || L.H % 32 != 0 || L.I % 32 != 0 || L.E > 1024 ||
      L.H > 4u * 32 * kMaxSteps || L.I > 4u * 32 * kMaxSteps)
    return false;
  if (L.d.sh_gate && (L.d.sh_gate->type != MR_GGML_MXFP4 || L.d.sh_up->type != MR_GGML_MXFP4 ||
                      L.d.sh_down->type != MR_GGML_MXFP4 || L.Ish == 0 || L.Ish % 32 != 0 ||
                      L.Ish > 4u * 32 * kMaxSteps))
    return false;
  return true;
}

uint64_t group_hist_bytes(uint64_t P, uint64_t E) {
  return P > (uint64_t)kGroupEntries ? (P + kGroupEntries - 1) / kGroupEntries * E * 4 : 0;
}

hipError_t launch_group(const Launch& K, const int32_t* idx, const float* w, int P, int k, int E, int tile,
                        const GroupOut& o) {
  ProfScope ps(K, "group");
  const dim3 grid((unsigned)((P + kGroupEntries - 1) / kGroupEntries));
  if (grid.x > 1) {
    hipLaunchKernelGGL(k_group_count, grid, dim3(kGroupThreads), 0, K.s, idx, P, E, o.hist);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_group, grid, dim3(kGroupThreads), 0, K.s, idx, w, P, k, E, tile, o);
  return hipGetLastError();
}

hipError_t launch_combine(const Launch& K, const float* o, const int32_t* pair_of, const int32_t* idx, const float* w,
                          const float* down_b, uint32_t T, int k, int H, const float* o_sh, const float* sh_sig,
                          const float* resid, float* y) {
  ProfScope ps(K, "combine");
  const dim3 grid((unsigned)((H / 4 + 255) / 256), std::min<uint32_t>(T, 65535u));
  if (k <= 4)
    hipLaunchKernelGGL(k_combine<4>, grid, dim3(256), 0, K.s, o, pair_of, idx, w, down_b, (int)T, k, H, o_sh, sh_sig,
                       resid, y);
  else if (k <= 8)
    hipLaunchKernelGGL(k_combine<8>, grid, dim3(256), 0, K.s, o, pair_of, idx, w, down_b, (int)T, k, H, o_sh, sh_sig,
                       resid, y);
  else
    hipLaunchKernelGGL(k_combine<16>, grid, dim3(256), 0, K.s, o, pair_of, idx, w, down_b, (int)T, k, H, o_sh,
                       sh_sig, resid, y);
  return hipGetLastError();
}

// Workgroups for a grouped GEMM of at most `items` work items: a multiple of the XCD count, so
// that every XCD's contiguous range of ceil(n_work / 8) items has a workgroup for each item
// (workgroup b takes item (b mod 8) * ceil(n_work / 8) + b / 8).
unsigned grouped_grid(uint64_t items) { return (unsigned)((items + kXcds - 1) / kXcds * kXcds); }

// One grouped GEMM launch over at most `tiles` pair tiles of 16 kPG pairs.
template <bool GATEUP>
static hipError_t launch_gemm(const Launch& K, const GroupedArgs& a, int pg, uint64_t tiles) {
  constexpr int rows = kRowsOf<GATEUP>;
  const dim3 grid(grouped_grid((uint64_t)((a.M + rows - 1) / rows) * tiles)), block(kGW * 64);
  if (pg == 4)
    hipLaunchKernelGGL((k_grouped_gemm<GATEUP, 4>), grid, block, 0, K.s, a);
  else if (pg == 2)
    hipLaunchKernelGGL((k_grouped_gemm<GATEUP, 2>), grid, block, 0, K.s, a);
  else
    hipLaunchKernelGGL((k_grouped_gemm<GATEUP, 1>), grid, block, 0, K.s, a);
  return hipGetLastError();
}

// 16-pair groups per work item, for `pairs` pairs over `experts` experts of `rows` gate rows and `hidden`
// down rows. More groups reuse a step's weight windows and their alignment for more MFMAs; fewer waste less
// on part-filled tiles and leave room for three workgroups per CU. The lines lie at a mean of 12 and 64
// pairs per expert. Whole call, us, 32 experts of 2880 x 2880, 1 / 2 / 4 groups, even routing and
// popularity ~ rank^-1.1:
//   mean     even                  skewed
//   8        162 / 176 / 192       151 / 169 / 176
//   12       183 / 184 / 200
//   16       204 / 194 / 206       218 / 195 / 225
//   32       261 / 248 / 227       283 / 247 / 249
//   64       374 / 309 / 300       408 / 332 / 333
//   128      626 / 500 / 452       669 / 530 / 480
//   255     1173 / 913 / 778
// From 32 to 64 an even batch gains up to 8% by 4 groups, but a skewed one nothing, and its down launch
// (fewer, longer items) loses: 110 -> 122 us at 64. Few work items take fewer groups, so that the CUs are
// not left idle: below two items per CU 4 groups lose to 2 (16 experts of 1600 x 1504, 500 tokens of 4,
// 372 items: 113 / 109 us), below seven for eight CUs 2 lose to 1 (24 experts of 1024 x 2048, 256 tokens of 3,
// 192 items: 121 / 100 us; but 28 of 1152 x 2304, 128 tokens of 3, 252 items: 68 / 74).
// Past that the rounds decide between 4 and 2 (512 workgroups are on the CUs at once; a part-filled
// last round half counts, as rounds overlap). An item of 4 groups takes about 1.6 times as long as one of
// 2; 1.4 leaves the choice at 4 where the estimate of the tiles is too coarse. 2 / 4 groups: 8 experts of
// 2944 x 1152, 384 tokens of 4 111 / 129 us; 18 of 1920 x 1440, 1,200 tokens of 2 134 / 158; 12 of 2720 x
// 1216, 2,048 tokens of 2 238 / 229 (but 1,536 tokens, a few items past two rounds, 182 / 203).
static int pair_groups(uint64_t pairs, uint64_t experts, int rows, int hidden) {
  int pg = pairs > 64 * experts ? 4 : pairs > 12 * experts ? 2 : 1;
  const uint64_t n_rt = (uint64_t)((rows + kRowsOf<true> - 1) / kRowsOf<true>);
  while (pg > 1 && std::max(pairs / (16 * pg), std::min(pairs, experts)) * n_rt < (pg == 4 ? 512u : 224u)) pg >>= 1;
  if (pg < 4) return pg;
  auto cost = [&](int g) {  // about half the experts hold a part-filled tile more than their pairs fill
    const double tiles = (double)pairs / (16 * g) + 0.5 * (double)std::min(pairs, experts);
    auto rounds = [&](uint64_t n) {
      const double r = tiles * (double)n / 512;
      return 0.5 * (std::max(r, 1.0) + std::ceil(r));
    };
    return rounds(n_rt) * hidden + rounds((uint64_t)((hidden + kRowsOf<false> - 1) / kRowsOf<false>)) * rows;
  };
  return 1.4 * cost(4) < cost(2) ? 4 : 2;
}

hipError_t launch_grouped(const Launch& K, const mr_layer& L, const float* x, uint32_t T, const int32_t* idx,
                          const float* w, float* y, const GroupedScratch& gs, const float* resid) {
  const int k = (int)L.d.top_k, E = (int)L.E, H = (int)L.H, I = (int)L.I;
  const int P = (int)T * k;
  const int pg = pair_groups((uint64_t)P, (uint64_t)E, I, H), tile = 16 * pg;
  const uint64_t max_tiles = group_tiles_max((uint64_t)P, (uint64_t)E, (uint64_t)tile);
  hipError_t e;
  const GroupOut go{gs.pair_tok, gs.pair_w, gs.pair_of, gs.exp_off, gs.tile_off, gs.tile_exp, gs.hist};
  if ((e = launch_group(K, idx, w, P, k, E, tile, go)) != hipSuccess) return e;
  {
    ProfScope ps(K, "split_x");
    hipLaunchKernelGGL(k_split_rows, dim3((unsigned)((H / 32 + 31) / 32), std::min<uint32_t>(T, 65535u)), dim3(256), 0,
                       K.s, x, (int)T, H, gs.img_x, gs.sc_x);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  GroupedArgs a{};
  a.w0 = expert_loc(L.d.gate), a.w1 = expert_loc(L.d.up);
  a.b0 = L.d.gate_bias, a.b1 = L.d.up_bias;
  a.img = gs.img_x, a.isc = gs.sc_x, a.pair_tok = gs.pair_tok, a.pair_w = gs.pair_w;
  a.exp_off = gs.exp_off, a.tile_off = gs.tile_off, a.tile_exp = gs.tile_exp, a.himg = gs.img_h, a.hsc = gs.sc_h;
  a.M = I, a.K = H, a.E = E;
  a.act = (int)L.d.act, a.alpha = L.d.alpha, a.limit = L.d.limit;
  {
    ProfScope ps(K, "grouped_gateup");
    if ((e = launch_gemm<true>(K, a, pg, max_tiles)) != hipSuccess) return e;
  }
  // The shared expert (layer.rs:1898-1953): one group of every token on the same x images,
  // weight 1 and SiLU (the routed experts' activation does not apply), its down outputs
  // [T][H], then sigmoid(x . gate_inp) per token, which the combine applies after the routed
  // sum.
  const int Ish = L.d.sh_gate ? (int)L.Ish : 0, pgs = pair_groups(T, 1, Ish, H), tiles = ((int)T + 16 * pgs - 1) / (16 * pgs);
  if (Ish) {
    GroupedArgs sg{};
    sg.w0 = expert_loc(L.d.sh_gate), sg.w1 = expert_loc(L.d.sh_up);
    sg.img = gs.img_x, sg.isc = gs.sc_x, sg.single_p = (int)T;
    sg.himg = gs.img_hsh, sg.hsc = gs.sc_hsh;
    sg.M = Ish, sg.K = H, sg.E = 1, sg.act = MR_ACT_SILU;
    {
      ProfScope ps(K, "grouped_shared_gateup");
      if ((e = launch_gemm<true>(K, sg, pgs, tiles)) != hipSuccess) return e;
    }
  }
  GroupedArgs d{};
  d.w0 = expert_loc(L.d.down);
  d.img = gs.img_h, d.isc = gs.sc_h, d.pair_tok = nullptr, d.pair_w = gs.pair_w;
  d.exp_off = gs.exp_off, d.tile_off = gs.tile_off, d.tile_exp = gs.tile_exp, d.out = gs.obuf;
  d.M = H, d.K = I, d.E = E;
  {
    ProfScope ps(K, "grouped_down");
    if ((e = launch_gemm<false>(K, d, pg, max_tiles)) != hipSuccess) return e;
  }
  if (!Ish) return launch_combine(K, gs.obuf, gs.pair_of, idx, w, L.d.down_bias, T, k, H, nullptr, nullptr, resid, y);
  GroupedArgs sd{};
  sd.w0 = expert_loc(L.d.sh_down);
  sd.img = gs.img_hsh, sd.isc = gs.sc_hsh, sd.single_p = (int)T, sd.out = gs.osh;
  sd.M = H, sd.K = Ish, sd.E = 1;
  {
    ProfScope ps(K, "grouped_shared_down");
    if ((e = launch_gemm<false>(K, sd, pgs, tiles)) != hipSuccess) return e;
  }
  if ((e = launch_sh_gate(K, x, T, H, L.d.sh_gate_inp, gs.sig)) != hipSuccess) return e;
  return launch_combine(K, gs.obuf, gs.pair_of, idx, w, L.d.down_bias, T, k, H, gs.osh, gs.sig, resid, y);
}

}  // namespace mr
