// gemm_sb.hpp -- prefill GEMM Y = X W^T for the K-quants (Q4_K, Q6_K) on gfx950.
//
// What sets it apart from gemm_tiled.hip: a K-quant weight is an integer times
// one scale per 256-element super-block,
//   Q4_K  w = d (s_j q) + dmin        s_j 6 bits, q 4 bits: s_j q <= 945
//   Q6_K  w = (d / 64) (s_j (q - 32)) s_j 8 bits, q 6 bits: |..| <= 8160
// so the sub-block scale s_j goes into the fp16 weight operand (Q4_K: the
// product is an fp16 exactly; Q6_K: hi = fp16(s_j (q - 32)) and the exact rest
// lo) and the matrix cores accumulate 64 or 128 elements (sb_chain) before one
// f32 FMA per output applies d.  With 32-element blocks and a scale per block
// that FMA comes once per step and the scale's product with it, which made the
// vector ALU the bound (3.4 VALU operations per MFMA), and Q6_K's
// 16-element groups had to be padded with zeros to 32 (four products per
// 32 elements; here three: x_lo w_hi, x_hi w_lo, x_hi w_hi; the x_lo w_lo left
// out is at most 2^-22 of x w, where |s (q - 32)| > 2048, and x itself carries 22
// bits.  Products that all have one sign show it: 2.4e-7 in sums of four
// super-blocks and 3.4e-7 in sums of four with K = 14336, where the 16-element
// blocks had 3.8e-7 and 1.4e-6 from their longer f32 sums.  In shorter sums it
// is formed: sb_lo_first).
// Activations are fp16 hi + lo of the row scaled by a power of two, as in
// gemm_tiled.hip (its pack_a_kernel writes them).
//
// Weights come as stage records (kquant.hip): for each stage of 64 elements
// and each row, contiguous over the rows,
//   kGemmQ4S 40 B: 32 quant bytes, f16 s 2^10 of the two scale groups, f32 d 2^14
//   kGemmQ6S 80 B: 64 quant bytes (0..63), f16 s of the four groups, f32 d / 64
// K-slots: step t (0, 1) of stage s, k-group g holds elements 64 s + 16 g +
// 8 t .. + 7, so a lane's quants of a stage are contiguous and share one scale.
// Q4_K's quants become weights in two operations per pair: the nibbles masked
// in place are fp16 subnormals (q 2^-24, or 16 q 2^-24) and one packed
// multiply by s 2^10 (s 2^6) gives s q 2^-14 exactly; d carries the 2^14.
//
// Schedule (128-token tiles: 8 waves, each 64 tokens x 64 rows).  A ring of
// stages is filled by global -> LDS copies.  A step is a phase of 16 MFMAs per
// product; the operands of a phase are read from LDS during the phase before,
// into registers whose last reader has just passed, and a row group's next
// weights are formed right after its last MFMA, so no phase starts with a
// burst of LDS reads (the bound of gemm_tiled.hip's schedule after the VALU).
// The barrier of a stage stands behind the last LDS read of its slot, in the
// middle of its second step.  LF (sb_lo_first): the same with the two steps'
// products in another order, both steps' operands in registers.
#pragma once

#include "gemm_dev.hpp"
#include "gemm_sb_api.hpp"

#include <algorithm>

namespace {

template <int BM>
struct SbCfg {
  static constexpr int WGM = BM == 128 ? 2 : 1;
  static constexpr int WGN = TWAVES / WGM;
  static constexpr int IT = BM / WGM / 16, NT = TBN / WGN / 16;
};

template <int TYPE>
constexpr int sb_rec() { return TYPE == wh::kGemmQ4S ? 40 : 80; }  // bytes per row and stage

// Stages after the first that the matrix cores accumulate before d is applied
// (0: 64 elements, 1: 128), for the sb super-blocks that a workgroup sums per
// tile.  An MFMA rounds its products at the size of its C operand, so a long
// chain loses more than the f32 FMAs of a short one; in a long sum the FMAs do,
// since the sum outgrows the chain.  Against 64 bits, Q4_K 14336 x 4096: chains
// of 256 elements 2.8e-7 at M=32, 3.0e-7 at M=512; of 64 2.0e-7 and 2.7e-7; of 128
// 2.6e-7 at M=512 (14 super-blocks); of 32 2.2e-7 at M=32.  From 8 super-blocks on,
// in 12 shapes of 8 to 28 and both types, 128 elements took 0.94 to 0.97 of the time
// of 64 (M=512 14336 x 4096 Q4_K 127.3 -> 121.5 us, Q6_K 169.2 -> 162.4) and are
// nearer for Q4_K (14336 x 4096 2.66e-7 -> 2.57e-7, 4096 x 14336 3.02e-7 -> 2.71e-7)
// and for Q6_K from 14 on (4096 x 14336 1.85e-7 -> 1.69e-7); Q6_K loses up to 3% at 8
// to 12 (8192 x 2048 1.40e-7 -> 1.44e-7; 2.08e-7 with 16-element blocks).
inline int sb_chain(int bm, int sb) { return bm == 128 && sb >= 8 ? 1 : 0; }

// Q6_K where a workgroup sums one or two super-blocks, and the 64-token tiles of
// longer prompts (gemm_tiled.hip's tile_bm; up to four): the products with an
// x_lo or w_lo of both steps of a stage, x_lo w_lo among them, come before the
// x_hi w_hi of either.  An MFMA rounds four times at the size of C, and the two
// products of lo limbs between the x_hi w_hi of the two steps are most of a short
// sum's error.  Against 64 bits (without; with one scale per 16 elements, whose
// quants are exact), 1e-7: 2048 x 1024 at 20 and 64 tokens 0.85 (1.07; 0.98), 1024 x
// 2048 at 50 0.89 (1.18; 1.08), 4096 x 4096 at 20 0.94 (1.34; 1.32).  Time 2048 x 1024
// at 20 tokens 14.4 us (13.9), 14336 x 1024 at 64 27.3 us (25.8); the longer sums of
// 14336 x 4096 do not need it (1.29; 1.59) and would take 30.6 us instead of 28.2.
// Q4_K, whose products are exact fp16s, has two products per step; it takes this
// order in the FFN's gate and up of up to seven super-blocks in 128-token tiles,
// where one pass sums twice as far as two passes in split-K did (FFN 1536 x 4096
// at 804 tokens 4.87e-7 -> 4.78e-7, in the same time; its stream-K kernel has no
// registers left for it).
inline bool sb_lo_first(int type, int bm, int n_tokens, int sb, bool ffn) {
  if (type == wh::kGemmQ4S) return ffn && bm == 128 && sb < 8;
  return bm <= 64 && !ffn && (n_tokens > 64 || sb <= 2);
}

template <int TYPE, int BM, bool LO>
struct SbStage {
  static constexpr int FR = BM / 16 * (LO ? 2 : 1);              // fragments per step
  static constexpr int A_FR = 2 * FR;                            // per stage
  static constexpr int A_DMA = (A_FR + TWAVES - 1) / TWAVES;     // copies per wave (wrapping)
  static constexpr int W_BYTES = TBN * sb_rec<TYPE>();
  static constexpr int W_X4 = W_BYTES / (TWAVES * 1024);         // 16-byte copies per wave
  static constexpr int W_X1 = (W_BYTES - W_X4 * TWAVES * 1024) / (TWAVES * 256);  // 4-byte copies of the rest
  static_assert(W_X4 * TWAVES * 1024 + W_X1 * TWAVES * 256 == W_BYTES, "whole copy instructions");
  static constexpr int BYTES = A_FR * FRAG + W_BYTES;
  static constexpr int COPIES = A_DMA + W_X4 + W_X1;             // vmcnt per stage
  // Ring depth: two stages in flight behind the one computed.  More only
  // lengthens the fill before the first product (M=32 14336 x 4096, Q4_K: 24.2
  // us with 8 stages, 23.1 with 5, 22.6 with 3).
  static constexpr int N = 3;
  static_assert(N * BYTES <= 160 * 1024 && (N - 1) * COPIES < 64, "ring size, vmcnt range");
};

// Four 4-bit quants masked out of u (bits 0..3 and 16..19, or 4..7 and 20..23)
// as fp16 subnormals, times the scale.
__device__ __forceinline__ half2v sb_nib(uint32_t u, uint32_t mask, half2v s) {
  return __builtin_bit_cast(half2v, u & mask) * s;
}

// Weight rows r0.. of one tile, K stages [st_a, st_b): the GEMM over it.  Grid
// and stream-K (SK) as gemm_tiled_kernel; units are super-blocks.
template <int TYPE, int BM, bool FFNP, bool SK, bool LO, bool LF>
__global__ __launch_bounds__(TWAVES * 64, 1) void gemm_sb_kernel(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ W2, const _Float16* __restrict__ frag,
    const float* __restrict__ rscale, const float* __restrict__ bsum, float* __restrict__ y, int n_tokens, int n_rows,
    int nsb, int sb_per_split, int tiles_n, int n_tiles, uint32_t* __restrict__ sk_flags, float* __restrict__ sk_part,
    int sk_upw, int sk_sub, uint32_t sk_wait,
    int chain) {
  using C = SbCfg<BM>;
  using S = SbStage<TYPE, BM, LO>;
  constexpr int IT = C::IT, NT = C::NT, REC = sb_rec<TYPE>(), N = S::N;
  constexpr bool Q4 = TYPE == wh::kGemmQ4S;
  constexpr int HALF = TBN / 2;  // FFNP: rows of each matrix per tile
  extern __shared__ __align__(16) uint8_t smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave / C::WGN) * (16 * IT);  // token offset of the wave tile
  const int wn = (wave % C::WGN) * (16 * NT);  // row offset
  const int g = lane >> 4, ln = lane & 15;     // k-group; token (A) / weight row (B) within a 16-tile
  const int bid = blockIdx.x;
  const size_t stage_stride = static_cast<size_t>(n_rows) * REC;

  // The workgroup's work is a sequence of segments, each the super-blocks
  // [sb_a, sb_b) of a tile L; without SK one.
  int u = 0, u_end = 1, v = 0;
  if constexpr (SK) {
    v = (bid % 8) * static_cast<int>(gridDim.x / 8) + bid / 8;
    u = v * sk_upw;
    u_end = min(n_tiles * nsb, u + sk_upw);
  }
  __shared__ int sk_ok;
  for (bool first = true; u < u_end; first = false) {
  int L, sb_a, sb_b;
  if constexpr (SK) {
    L = u / nsb;
    sb_a = u % nsb;
    sb_b = min(nsb, sb_a + (u_end - u));
    u += sb_b - sb_a;
  } else {
    const int q = n_tiles / 8, rem = n_tiles % 8;
    const int xcd = bid % 8, local = bid / 8;
    L = xcd * q + min(xcd, rem) + local;
    sb_a = blockIdx.y * sb_per_split;
    sb_b = max(sb_a, min(nsb, sb_a + sb_per_split));
    u = u_end;
  }
  const int T = L / tiles_n, R = L % tiles_n;
  const int t0 = T * BM, r0 = R * (FFNP ? HALF : TBN);
  if (!first) __syncthreads();  // every wave is done with the ring of the previous segment

  // Source offsets of this lane's weight copies: the tile's rows of a stage
  // are one contiguous range; past the last row the last 16 bytes are read
  // again (rows whose products are not stored).  FFNP: the upper half of the
  // range is the same rows of W2; copies do not straddle the halves.
  static_assert(!FFNP || (HALF * REC) % 1024 == 0, "gate / up halves in whole copy instructions");
  const uint32_t w_end = (static_cast<uint32_t>(n_rows) * REC + 15u) / 16u * 16u;
  auto w_pos = [&](int c) { return c < S::W_X4 ? c * TWAVES * 1024 + 1024 * wave
                                               : S::W_X4 * TWAVES * 1024 + (c - S::W_X4) * TWAVES * 256 + 256 * wave; };
  auto w_up = [&](int c) { return FFNP && w_pos(c) >= HALF * REC; };
  const uint32_t smem_base = lds_addr(smem);
  const uint32_t frag_lane_off = 16u * (4u * (lane & 15) + (lane >> 4));  // stored token-major

  uint32_t w_off[S::W_X4 + S::W_X1];
#pragma unroll
  for (int c = 0; c < S::W_X4 + S::W_X1; c++) {
    const uint32_t by = c < S::W_X4 ? 16u : 4u;
    const uint32_t p = static_cast<uint32_t>(r0) * REC + static_cast<uint32_t>(w_pos(c) - (w_up(c) ? HALF * REC : 0)) + by * lane;
    w_off[c] = min(p, w_end - by);
  }

  // the copies, stage after stage: running source addresses (wave-uniform),
  // stages left, slot
  const uint8_t *pa, *pw, *pu = nullptr;
  uint32_t islot;
  int to_issue;
  auto issue = [&]() {
    if (to_issue <= 0) return;
    to_issue--;
#pragma unroll
    for (int f = 0; f < S::A_DMA; f++) {
      const int fi = (wave * S::A_DMA + f) % S::A_FR;  // copied twice where a stage has fewer than the waves copy
      const int src = LO ? fi : (fi / S::FR) * (BM / 8) + 2 * (fi % S::FR);
      copy16_to_lds(pa + src * FRAG, frag_lane_off, islot + fi * FRAG);
    }
#pragma unroll
    for (int c = 0; c < S::W_X4 + S::W_X1; c++) {
      const uint8_t* wb = w_up(c) ? pu : pw;
      if (c < S::W_X4) copy16_to_lds(wb, w_off[c], islot + S::A_FR * FRAG + w_pos(c));
      else copy4_to_lds(wb, w_off[c], islot + S::A_FR * FRAG + w_pos(c));
    }
    pa += 2 * (BM / 8) * FRAG;
    pw += stage_stride;
    if constexpr (FFNP) pu += stage_stride;
    islot += S::BYTES;
    if (islot == smem_base + N * S::BYTES) islot = smem_base;
  };

  float4v acc[IT][NT], cc[IT][NT];

  // LDS offsets of this lane's operands within a slot
  const uint32_t a_lds = static_cast<uint32_t>((wm >> 4) * (LO ? 2 : 1) * FRAG + 16 * lane);
  const uint32_t w_lds = static_cast<uint32_t>(S::A_FR * FRAG + ((FFNP ? wn / 2 : wn) + ln) * REC + (Q4 ? 8 : 16) * g);
  // row group n: FFNP: groups 2m and 2m + 1 are the same rows of gate and up
  auto w_grp = [](int n) { return (FFNP ? ((n & 1) ? HALF : 0) + 16 * (n >> 1) : 16 * n) * REC; };
  const uint32_t s_lds = w_lds + (Q4 ? 32 + 2 * (g >> 1) - 8 * g : 64 + 2 * g - 16 * g);
  const uint32_t d_lds = w_lds + (Q4 ? 36 - 8 * g : 72 - 16 * g);

  half8 ah[IT], al[IT], bw[NT], bl[NT];
  half8 ah1[IT], al1[IT], bw1[NT];  // LF: the stage's second step
  uint2 rq[NT];          // quants: Q4_K both steps of the stage, Q6_K one step
  half2v sc[NT];         // the lane's scale of the stage in both halves
  float dn[NT];          // d of the chain whose products are pending
  auto read_a = [&](const uint8_t* slot, int t, int limb, half8 (&dst)[IT]) {
#pragma unroll
    for (int i = 0; i < IT; i++)
      dst[i] = *reinterpret_cast<const half8*>(slot + a_lds + (t * S::FR + (LO ? 2 * i + limb : i)) * FRAG);
  };
  // quants (and scales) of a row group: Q4_K once per stage, Q6_K per step
  auto read_q = [&](const uint8_t* slot, int t) {
#pragma unroll
    for (int n = 0; n < NT; n++)
      rq[n] = *reinterpret_cast<const uint2*>(slot + w_lds + w_grp(n) + (Q4 ? 0 : 8 * t));
  };
  auto read_d = [&](const uint8_t* slot) {
#pragma unroll
    for (int n = 0; n < NT; n++) dn[n] = *reinterpret_cast<const float*>(slot + d_lds + w_grp(n));
  };
  auto read_s = [&](const uint8_t* slot) {
#pragma unroll
    for (int n = 0; n < NT; n++) {
      const _Float16 sv = *reinterpret_cast<const _Float16*>(slot + s_lds + w_grp(n));
      sc[n] = half2v{sv, sv};
    }
  };
  // Q6_K: pair c of q - 32: bytes under 0x64 are fp16 1024 + q; minus 1056
  auto q6_pair = [](uint2 q, int c) {
    const half2v off = {static_cast<_Float16>(-1056.f), static_cast<_Float16>(-1056.f)};
    const uint32_t w = __builtin_amdgcn_perm(0x64646464u, c < 2 ? q.x : q.y, (c & 1) ? 0x04030402u : 0x04010400u);
    return __builtin_bit_cast(half2v, w) + off;
  };
  // weights of row group n for step t from rq / sc
  auto form = [&](int n, int t) {
    half2v p[4];
    if constexpr (Q4) {
      const uint32_t q = t ? rq[n].y : rq[n].x;
      const half2v s16 = sc[n] * half2v{static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
      p[0] = sb_nib(q, 0x000F000Fu, sc[n]);
      p[1] = sb_nib(q, 0x00F000F0u, s16);
      p[2] = sb_nib(q >> 8, 0x000F000Fu, sc[n]);
      p[3] = sb_nib(q >> 8, 0x00F000F0u, s16);
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) p[c] = q6_pair(rq[n], c) * sc[n];  // rounded
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
      bw[n][2 * c] = p[c][0];
      bw[n][2 * c + 1] = p[c][1];
    }
  };
  // Q6_K: the rest s (q - 32) - hi of row group n
  auto form_lo = [&](int n) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const half2v hi = {bw[n][2 * c], bw[n][2 * c + 1]};
      const half2v r = __builtin_elementwise_fma(q6_pair(rq[n], c), sc[n], -hi);
      bl[n][2 * c] = r[0];
      bl[n][2 * c + 1] = r[1];
    }
  };
  // acc += d cc of row group n, whose next chain starts from zero
  auto apply = [&](int n, float d) {
#pragma unroll
    for (int i = 0; i < IT; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        acc[i][n][r] = __builtin_fmaf(d, cc[i][n][r], acc[i][n][r]);
        cc[i][n][r] = 0.f;
      }
  };
  auto mma = [&](int i, int n, half8 a, half8 b) {
    cc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, cc[i][n], 0, 0, 0);
  };

#pragma unroll
  for (int i = 0; i < IT; i++)
#pragma unroll
    for (int n = 0; n < NT; n++) acc[i][n] = float4v{0.f, 0.f, 0.f, 0.f};
  // dmin: acc += dmin[row][sb] S[token][sb] over super-blocks [sb_lo, sb_hi), as
  // matrix-core products over windows of 32: lane group g holds super-blocks
  // 8g .. 8g + 7 of the window in both operands (B: the fp16 table behind the
  // records, those outside masked to zero; A: the packing's sums as hi + lo fp16
  // limbs of S 2^-10).
  auto add_dmin = [&](int sb_lo, int sb_hi) {
    const int nsbp = (nsb + 7) & ~7;
    const size_t table = static_cast<size_t>(nsb) * 4 * stage_stride;
    const uint16_t* dm1 = reinterpret_cast<const uint16_t*>(W + table);
    const uint16_t* dm2 = FFNP ? reinterpret_cast<const uint16_t*>(W2 + table) : dm1;
    const uint16_t* s16 = reinterpret_cast<const uint16_t*>(bsum);
    // opaque, so that the loads' offsets are formed here and not held in
    // registers through the stage loop
    int lnv = ln;
    asm volatile("" : "+v"(lnv));
    for (int w0 = sb_lo & ~31; w0 < sb_hi; w0 += 32) {
      const int s0 = w0 + 8 * g;
      const bool in = s0 < nsbp;
      uint32_t mk[4];
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const int a = s0 + 2 * d;
        mk[d] = (a >= sb_lo && a < sb_hi ? 0x0000FFFFu : 0u) | (a + 1 >= sb_lo && a + 1 < sb_hi ? 0xFFFF0000u : 0u);
      }
      u32x4 bd[NT];
#pragma unroll
      for (int n = 0; n < NT; n++) {
        const int row = r0 + (FFNP ? wn / 2 + 16 * (n >> 1) : wn + 16 * n) + lnv;
        const uint32_t off = static_cast<uint32_t>(min(row, n_rows - 1) * nsbp + s0);
        bd[n] = in ? *reinterpret_cast<const u32x4*>(((n & 1) ? dm2 : dm1) + off) : u32x4{0u, 0u, 0u, 0u};
      }
      u32x4 sh[IT], sl[IT];
#pragma unroll
      for (int i = 0; i < IT; i++) {
        const uint32_t off = static_cast<uint32_t>((t0 + wm + 16 * i + lnv) * 2 * nsbp + s0);
        sh[i] = in ? *reinterpret_cast<const u32x4*>(s16 + off) : u32x4{0u, 0u, 0u, 0u};
        sl[i] = in ? *reinterpret_cast<const u32x4*>(s16 + off + nsbp) : u32x4{0u, 0u, 0u, 0u};
      }
      __builtin_amdgcn_sched_barrier(0);  // every load issued before the first use
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int d = 0; d < 4; d++) bd[n][d] &= mk[d];
#pragma unroll
      for (int i = 0; i < IT; i++) {
#pragma unroll
        for (int n = 0; n < NT; n++) {
          float4v t = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, sh[i]), __builtin_bit_cast(half8, bd[n]),
                                                             float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          t = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, sl[i]), __builtin_bit_cast(half8, bd[n]), t, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; r++) acc[i][n][r] = __builtin_fmaf(1024.f, t[r], acc[i][n][r]);
        }
        __builtin_amdgcn_sched_barrier(0);  // one token group's products at a time
      }
    }
  };
  // Stream-K: 128-token tiles add it over all of the tile, in the workgroup that
  // finishes it; in parts of up to three super-blocks, of which a tile has five or
  // more, and in 64-token tiles, each part its own (own_dmin), so that what is
  // handed over has the result's size and not the quants' mean's (1536 x 4096 at 804
  // tokens, error 2.27e-7 -> 2.15e-7, 53.6 us either way; it costs a pass of the
  // table per part: 10240 x 5632 at 100 tokens, four super-blocks each, 56.1 -> 57.2
  // us).  64-token tiles add it before they wait for the other parts, for which the
  // 128-token kernel has no registers.
  constexpr bool EARLY = SK && BM < 128;
  const bool own_dmin = !SK || EARLY || sk_upw <= 3;
  // A head part (SK) that does not get every other owner's slot in time runs
  // a second pass over the rest of the tile, into the same accumulators.
  int done = sb_b;  // end of the super-blocks summed here
#pragma unroll 1
  for (int pass = 0; pass < 2; pass++) {
  const int sb0 = pass ? sb_b : sb_a;
  if (pass > 0) done = nsb;
  const int n_stages = 4 * ((pass ? nsb : sb_b) - sb0);
  if (pass > 0) __syncthreads();  // the ring of the first pass is no longer read
  to_issue = n_stages;
  islot = smem_base;
  pa = reinterpret_cast<const uint8_t*>(frag) + (static_cast<size_t>(T) * nsb + sb0) * 8 * (BM / 8) * FRAG;
  pw = W + static_cast<size_t>(4 * sb0) * stage_stride;
  if constexpr (FFNP) pu = W2 + static_cast<size_t>(4 * sb0) * stage_stride;
#pragma unroll
  for (int i = 0; i < IT; i++)
#pragma unroll
    for (int n = 0; n < NT; n++) cc[i][n] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < NT; n++) dn[n] = 0.f;
#pragma unroll
  for (int st = 0; st < N; st++) issue();
  wait_stages<S::COPIES, N - 1>(n_stages - 1);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // operands of the first step
  read_q(smem, 0);
  read_s(smem);
  if constexpr (Q4) {
    read_a(smem, 0, 1, al);
    form(0, 0);
    if constexpr (NT > 2) form(1, 0);
  } else {
    if constexpr (LO) read_a(smem, 0, 1, al);
#pragma unroll
    for (int n = 0; n < (LF ? NT : NT / 2); n++) form(n, 0);
  }
  int cur = 0;  // slot of the stage computed
  // One stage per trip: unrolled over the four of a super-block the body
  // needs 20 to 60 more registers and spills (Q6_K 14336 x 4096, M=512: 182 us).
#pragma unroll 1
  for (int st = 0; st < n_stages; st++) {
      const uint8_t* slot = smem + cur * S::BYTES;
      const int nxt = cur + 1 == N ? 0 : cur + 1;
      const uint8_t* nslot = smem + nxt * S::BYTES;
      // first / last stage of a chain; the branch stays: straight through, the
      // 128-token body spills
      const bool head = (st & chain) == 0, tail = (st & chain) == chain;
      // behind the last read of the stage's slot: the next stage landed
      // (every wave's copies), then the slot is refilled
      auto turn = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_stages<S::COPIES, N - 2>(n_stages - 2 - st);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue();
      };
      if constexpr (LF && Q4) {
        // x_lo of both steps, then x_hi of both: one operand set read while the
        // other is multiplied, the second step's weights in bw1
        auto form1 = [&](int n) {
          const uint32_t q = rq[n].y;
          const half2v s16 = sc[n] * half2v{static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
          const half2v p[4] = {sb_nib(q, 0x000F000Fu, sc[n]), sb_nib(q, 0x00F000F0u, s16),
                               sb_nib(q >> 8, 0x000F000Fu, sc[n]), sb_nib(q >> 8, 0x00F000F0u, s16)};
#pragma unroll
          for (int c = 0; c < 4; c++) {
            bw1[n][2 * c] = p[c][0];
            bw1[n][2 * c + 1] = p[c][1];
          }
        };
        auto phase = [&](half8 (&a)[IT], half8 (&b)[NT], auto then) {
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++) mma(i, n, a[i], b[n]);
            then(n);
            __builtin_amdgcn_sched_barrier(0);
          }
        };
        read_a(slot, 1, 1, ah);
        phase(al, bw, [&](int n) {
          if (head && n == 0) apply(NT - 1, dn[NT - 1]);
          if (n < NT / 2) form(n + NT / 2, 0);
          else form1(n - NT / 2);
        });
        read_a(slot, 0, 0, al);
        phase(ah, bw1, [&](int n) {
          if (n < NT / 2) form1(n + NT / 2);
        });
        read_a(slot, 1, 0, ah);
        if (tail) read_d(slot);
        phase(al, bw, [](int) {});
        turn();
        read_q(nslot, 0);
        read_s(nslot);
        read_a(nslot, 0, 1, al);
        phase(ah, bw1, [&](int n) {
          if (tail && n > 0) apply(n - 1, dn[n - 1]);
          if (n >= NT / 2) form(n - NT / 2, 0);
        });
        cur = nxt;
        continue;
      }
      if constexpr (LF && !Q4) {
        auto step = [&](half8 (&a)[IT], half8 (&b)[NT], auto then) {
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++) mma(i, n, a[i], b[n]);
            then(n);
            __builtin_amdgcn_sched_barrier(0);
          }
        };
        uint2 rq1[NT];
        // the first step's x_lo w_hi; its x_hi and the second's x_lo and quants read
        read_a(slot, 0, 0, ah);
        if constexpr (LO) read_a(slot, 1, 1, al1);
#pragma unroll
        for (int n = 0; n < NT; n++) rq1[n] = *reinterpret_cast<const uint2*>(slot + w_lds + w_grp(n) + 8);
#pragma unroll
        for (int n = 0; n < NT; n++) {
#pragma unroll
          for (int i = 0; i < IT; i++)
            if constexpr (LO) mma(i, n, al[i], bw[n]);
          if (head && n == 0) apply(NT - 1, dn[NT - 1]);
          form_lo(n);
          __builtin_amdgcn_sched_barrier(0);
        }
        // its x_lo w_lo and x_hi w_lo; the second step's weights formed and its x_hi read
        read_a(slot, 1, 0, ah1);
        if (tail) read_d(slot);
        if constexpr (LO) step(al, bl, [](int) {});
        step(ah, bl, [&](int n) {
          rq[n] = rq1[n];
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const half2v p = q6_pair(rq1[n], c) * sc[n];
            bw1[n][2 * c] = p[0];
            bw1[n][2 * c + 1] = p[1];
          }
        });
        // the second step's x_lo w_hi
#pragma unroll
        for (int n = 0; n < NT; n++) {
#pragma unroll
          for (int i = 0; i < IT; i++)
            if constexpr (LO) mma(i, n, al1[i], bw1[n]);
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const half2v hi = {bw1[n][2 * c], bw1[n][2 * c + 1]};
            const half2v r = __builtin_elementwise_fma(q6_pair(rq[n], c), sc[n], -hi);
            bl[n][2 * c] = r[0];
            bl[n][2 * c + 1] = r[1];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        turn();
        read_q(nslot, 0);
        read_s(nslot);
        if constexpr (LO) step(al1, bl, [](int) {});
        step(ah1, bl, [](int) {});
        // x_hi w_hi of both; the next stage's x_lo read and weights formed
        if constexpr (LO) read_a(nslot, 0, 1, al);
        step(ah, bw, [](int) {});
        step(ah1, bw1, [&](int n) {
          if (tail && n > 0) apply(n - 1, dn[n - 1]);
          form(n, 0);
        });
        cur = nxt;
        continue;
      }
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const bool zero = head && t == 0, last = tail && t == 1;
        if constexpr (Q4) {
          // phase x_lo (x_hi without LO): x_hi read; the weights of the step's later row groups
          if constexpr (LO) read_a(slot, t, 0, ah);
          if (last) read_d(slot);
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++) mma(i, n, al[i], bw[n]);
            if (zero && n == 0) apply(NT - 1, dn[NT - 1]);
            if (NT > 2 && n < 2) form(n + 2, t);
            if (NT == 2 && n == 0) form(1, t);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (t == 1) turn();
          if (t == 1) {
            read_q(nslot, 0);
            read_s(nslot);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++)
              if constexpr (LO) mma(i, n, ah[i], bw[n]);
            if (n == 0) read_a(t ? nslot : slot, t ^ 1, 1, al);
            if (last && n > 0) apply(n - 1, dn[n - 1]);
            if (NT > 2 && n >= 2) form(n - 2, t ^ 1);
            if (NT == 2 && n == 1) form(0, t ^ 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
          // phase x_lo w_hi: x_hi read; the later w_hi and first w_lo formed
          read_a(slot, t, 0, ah);
          if (last) read_d(slot);
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++)
              if constexpr (LO) mma(i, n, al[i], bw[n]);
            if (zero && n == 0) apply(NT - 1, dn[NT - 1]);
            if (n < NT / 2) form(n + NT / 2, t);
            else form_lo(n - NT / 2);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (t == 1) turn();
          // phase x_hi w_lo: the later w_lo formed, the next quants read
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++) mma(i, n, ah[i], bl[n]);
            if (n < NT / 2) form_lo(n + NT / 2);
            if (n == NT / 2) {
              read_q(t ? nslot : slot, t ^ 1);
              if (t == 1) read_s(nslot);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          // phase x_hi w_hi: the next x_lo read, the next step's first w_hi formed
#pragma unroll
          for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int i = 0; i < IT; i++) mma(i, n, ah[i], bw[n]);
            if (LO && n == 0) read_a(t ? nslot : slot, t ^ 1, 1, al);
            if (last && n > 0) apply(n - 1, dn[n - 1]);
            if (n >= NT / 2) form(n - NT / 2, t ^ 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      cur = nxt;
  }
  apply(NT - 1, dn[NT - 1]);
  if constexpr (Q4 && EARLY) add_dmin(sb0, done);
  if constexpr (!SK) break;
  if (pass > 0 || sb_a > 0 || sb_b == nsb) break;  // a tail part, the whole tile, or done here
  // head part: wait for the owners of the rest of the tile, then add their slots in order
  const int w_last = min(static_cast<int>(gridDim.x) - 1, ((L + 1) * nsb - 1) / sk_upw);
  if (threadIdx.x == 0) {
    int ok = 1;
    const uint64_t t_start = __builtin_amdgcn_s_memrealtime();
    for (int w = v + 1; w <= w_last && ok; w++) {
      while (__hip_atomic_load(sk_flags + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
             static_cast<uint32_t>(sk_sub + 1)) {
        if (__builtin_amdgcn_s_memrealtime() - t_start > sk_wait) {  // ticks of the 100 MHz clock
          ok = 0;
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
    sk_ok = ok;
  }
  __syncthreads();
  if (sk_ok) {
    for (int w = v + 1; w <= w_last; w++) {
      const i32x4 rs = sk_rsrc(sk_part + static_cast<size_t>(w) * BM * TBN);
#pragma unroll
      for (int i = 0; i < IT; i++)
#pragma unroll
        for (int n = 0; n < NT; n++)
          acc[i][n] += gt_buffer_load_x4(rs, 16 * ((i * NT + n) * (TWAVES * 64) + static_cast<int>(threadIdx.x)), 0,
                                         kSkCoherent);
    }
    break;
  }
  // otherwise: the rest of the tile, here
  }  // pass
  if constexpr (Q4 && !EARLY)
    if (own_dmin || sb_a == 0) add_dmin(sb_a, own_dmin ? done : nsb);

  if constexpr (SK) {
    if (sb_a > 0) {
      // a tail part: the raw accumulators to this workgroup's slot, then its flag
      const i32x4 rs = sk_rsrc(sk_part + static_cast<size_t>(v) * BM * TBN);
#pragma unroll
      for (int i = 0; i < IT; i++)
#pragma unroll
        for (int n = 0; n < NT; n++)
          gt_buffer_store_x4(acc[i][n], rs, 16 * ((i * NT + n) * (TWAVES * 64) + static_cast<int>(threadIdx.x)), 0,
                             kSkCoherent);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every store complete before the flag
      __syncthreads();
      if (threadIdx.x == 0)
        __hip_atomic_store(sk_flags + v, static_cast<uint32_t>(sk_sub + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      continue;
    }
  }

  // the lane's place recomputed here, not held through the stage loop
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int eg = (tid & 63) >> 4, el = tid & 15;
  if constexpr (FFNP) {
    // h = silu(g) * u for the gate / up pairs, as (g * (1 / (1 + e^-g))) * u
#pragma unroll
    for (int i = 0; i < IT; i++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int t = t0 + wm + 16 * i + 4 * eg + r;
        if (t >= n_tokens) continue;
        const float s = rscale[t];
#pragma unroll
        for (int m = 0; m < NT / 2; m++) {
          const int col = r0 + wn / 2 + 16 * m + el;
          if (col >= n_rows) continue;
          const float gv = acc[i][2 * m][r] * s, uv = acc[i][2 * m + 1][r] * s;
          y[static_cast<size_t>(t) * n_rows + col] = (gv * (1.0f / (1.0f + expf(-gv)))) * uv;
        }
      }
    }
  } else {
    float* out = y + static_cast<size_t>(blockIdx.y) * n_tokens * n_rows;  // split-K: plane blockIdx.y
#pragma unroll
    for (int i = 0; i < IT; i++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int t = t0 + wm + 16 * i + 4 * eg + r;
        if (t >= n_tokens) continue;
        const float s = rscale[t];
#pragma unroll
        for (int n = 0; n < NT; n++) {
          const int row = r0 + wn + 16 * n + el;
          if (row < n_rows) out[static_cast<size_t>(t) * n_rows + row] = acc[i][n][r] * s;
        }
      }
    }
  }
  }  // segment
}

template <int TYPE, int BM, bool FFNP, bool SK, bool LO, bool LF = false>
int sb_launch(const wh::SbGemm& a, hipStream_t s) {
  const int tiles_n = (a.n_rows + (FFNP ? TBN / 2 : TBN) - 1) / (FFNP ? TBN / 2 : TBN);
  const int n_tiles = (a.n_tokens + BM - 1) / BM * tiles_n;
  const int nsb = a.k / 256;
  const size_t lds = static_cast<size_t>(SbStage<TYPE, BM, LO>::N) * SbStage<TYPE, BM, LO>::BYTES;
  auto* kernel = &gemm_sb_kernel<TYPE, BM, FFNP, SK, LO, LF>;
  WH_ENSURE_LDS(lds, kernel);
  const dim3 grid(static_cast<unsigned>(SK ? a.sk_g : n_tiles), static_cast<unsigned>(SK ? 1 : a.splits));
  const int upw = SK ? (n_tiles * nsb + a.sk_g - 1) / a.sk_g : 0;
  const int sbps = (nsb + a.splits - 1) / a.splits;
  kernel<<<grid, TWAVES * 64, lds, s>>>(
      a.w, a.w2, a.frag, a.rs, a.bs, a.y, a.n_tokens, a.n_rows, nsb, sbps, tiles_n, n_tiles,
      a.sk_flags, a.sk_part, upw, a.sk_sub, a.sk_wait, sb_chain(BM, SK ? std::min(nsb, upw) : sbps));
  WH_LAUNCH_CHECK("k-quant gemm kernel launch");
  return WH_OK;
}

template <int TYPE, int BM>
int sb_launch_bm(const wh::SbGemm& a, hipStream_t s) {
  if constexpr (BM >= 64) {
    if (a.sk_g) {
      if (a.ffn) return sb_launch<TYPE, BM, true, true, true>(a, s);
      return a.lo ? sb_launch<TYPE, BM, false, true, true>(a, s) : sb_launch<TYPE, BM, false, true, false>(a, s);
    }
  }
  if (sb_lo_first(TYPE, BM, a.n_tokens, (a.k / 256 + a.splits - 1) / a.splits, a.ffn)) {
    if constexpr (TYPE == wh::kGemmQ4S) {
      if constexpr (BM == 128) return sb_launch<TYPE, BM, true, false, true, true>(a, s);
    } else if constexpr (BM <= 64) {
      return a.lo ? sb_launch<TYPE, BM, false, false, true, true>(a, s) : sb_launch<TYPE, BM, false, false, false, true>(a, s);
    }
  }
  if (a.ffn) return sb_launch<TYPE, BM, true, false, true>(a, s);
  return a.lo ? sb_launch<TYPE, BM, false, false, true>(a, s) : sb_launch<TYPE, BM, false, false, false>(a, s);
}

template <int TYPE>
int sb_launch_type(const wh::SbGemm& a, hipStream_t s) {
  switch (a.bm) {
    case 32: return sb_launch_bm<TYPE, 32>(a, s);
    case 64: return sb_launch_bm<TYPE, 64>(a, s);
    default: return sb_launch_bm<TYPE, 128>(a, s);
  }
}

}  // namespace
