// kquant.hip -- the 256-element K-quant blocks (Q4_K, Q6_K) as woolly-gguf
// decodes them, on gfx950: bit-exact dequantization and a GEMV defined as that
// dequantization followed by the f32 dot product.
//
// Reference: woolly_gguf::dequantize (crates/woolly-gguf/src/dequantize.rs:189-205)
// with dequantize_q4_k_scalar (:404-458, the x86 path) and dequantize_q6_k
// (:460-536).  woolly reads these blocks its own way (not ggml's layout):
//   Q4_K (144 B): bytes 0..11 pack eight 6-bit scales, scale i from byte
//     src = 3i/2: even i -> b[src] & 63, odd i -> ((b[src] >> 6) |
//     ((b[src+1] & 15) << 2)) & 63; f16 d at 12..13, f16 dmin at 14..15,
//     quants at 16..143: element i is the low nibble of qs[i/2] for even i, the
//     high nibble for odd i; value d * scale[i/32] * q + dmin.
//   Q6_K (210 B): ql = 0..127, qh = 128..191, u8 scales = 192..207, f16 d at
//     208..209; element i takes 4 bits from ql[64(i/128) + 32((i%128)/64) +
//     16((i%64)/32) + i%16] (low nibble below 128, high nibble from 128 on) and
//     2 bits from qh[32(i/128) + 16((i%128)/64) + 8((i%64)/32) + (i%32)/4]
//     at shift 2((i%32)%4) (+2 for the upper half; at shift 6 that pair is the
//     low bits of the next qh byte, 0 past the last one); value
//     ((d * scale[i/16]) * (q - 32)) / 64.
// Every product and sum is rounded in the reference's order with unfused
// operations, so the results are bit-identical to the CPU.
#include "wh_blocks.hpp"

namespace {

using whd::b16;
using whd::kq_quad;
using whd::q4k_scale;

template <int TYPE>
constexpr int kq_bytes() { return TYPE == WH_TYPE_Q4_K ? 144 : 210; }

// Four consecutive outputs per thread and quad (64 quads, one KiB, per block
// and wavefront).  Bound by the f32 output written (1 KiB against 144 or 210 B
// read per block), as long as the loads are few and wide: the byte-wise decode
// of kq_quad took 105 us (Q4_K) and 100 us (Q6_K) for 14336 x 4096; with one
// 16-byte header load and two quant bytes per quad (Q4_K), or one dword of ql,
// two bytes of qh, the scale and d (Q6_K), 57 us and 60 us (4.7 TB/s; a fill of
// that size writes 6.9 TB/s).  Blocks per wavefront and pass: Q4_K two (one: 67 us, four
// 66 us), Q6_K one (two: 67 us); 8 workgroups per CU (Q4_K with 16: 69 us).
template <int TYPE>
constexpr int kq_run() { return TYPE == WH_TYPE_Q4_K ? 2 : 1; }

// Quad c of a block as kq_quad decodes it (same operations in the same order).
// Q4_K: b 16-byte aligned.
template <int TYPE>
__device__ __forceinline__ void kq_quad_wide(const uint8_t* b, int c, float v[4]) {
  if constexpr (TYPE == WH_TYPE_Q4_K) {
    const uint4 h = *reinterpret_cast<const uint4*>(b);
    const uint32_t q = *reinterpret_cast<const uint16_t*>(b + 16 + 2 * c);
    const float d = whd::f16_bits_to_f32(h.w & 0xFFFFu), dmin = whd::f16_bits_to_f32(h.w >> 16);
    // scales 2p and 2p + 1 are bits 0..5 and 14..19 of the 24 bits at bit 24p
    const int p = c >> 4;
    const uint32_t lo = p == 0 ? h.x : (p == 1 ? (h.x >> 24) | (h.y << 8) : (p == 2 ? (h.y >> 16) | (h.z << 16) : h.z >> 8));
    const uint32_t s = (lo >> ((c & 8) ? 14 : 0)) & 63u;
    const float ds = __fmul_rn(d, static_cast<float>(s));
#pragma unroll
    for (int t = 0; t < 4; t++) v[t] = __fadd_rn(__fmul_rn(ds, static_cast<float>((q >> (4 * t)) & 15u)), dmin);
  } else {
    uint32_t ql;
    uint16_t qh;
    __builtin_memcpy(&ql, b + 16 * (c >> 3) + 4 * (c & 3), 4);  // blocks are 2-byte aligned
    __builtin_memcpy(&qh, b + 128 + c, 2);
    const float d = whd::f16_bits_to_f32(b16(b + 208)), s = static_cast<float>(b[192 + (c >> 2)]);
    const float ds = __fmul_rn(d, s);
    // the two bytes of qh; past the last one (byte 64 is a scale) the bits are 0
    uint32_t hi = c == 63 ? qh & 0xFFu : qh;
    if (c >= 32) {
      ql >>= 4;
      hi >>= 2;
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const uint32_t q = ((ql >> (8 * t)) & 15u) | (((hi >> (2 * t)) & 3u) << 4);
      v[t] = __fmul_rn(__fmul_rn(ds, static_cast<float>(static_cast<int>(q) - 32)), 0.015625f);
    }
  }
}

// OUT16: output 16-byte aligned (16-byte stores); WIDE: and, for Q4_K, the data
// too (the loads of kq_quad_wide).  Q4_K 14336 x 4096 of repeated random bytes:
// 42.9 us with both aligned, 54.1 with the output alone (82.3 with 4-byte stores).
template <int TYPE, bool WIDE, bool OUT16>
__global__ __launch_bounds__(256) void kq_dequant_kernel(const uint8_t* __restrict__ data, float* __restrict__ out,
                                                         size_t n) {
  constexpr int kRun = kq_run<TYPE>();
  const size_t nblk = (n + 255) / 256;
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const size_t waves = static_cast<size_t>(gridDim.x) * (blockDim.x >> 6);
  const size_t wave = static_cast<size_t>(blockIdx.x) * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // a zero the compiler cannot see through: the block address counts as the
  // lane's own, so the header comes by vector loads (a scalar load per block
  // misses the small scalar cache every time)
  uint32_t lane0 = 0;
  asm("" : "+v"(lane0));
  data += lane0;
  for (size_t b0 = wave; b0 < nblk; b0 += waves * kRun) {
    if (WIDE && (b0 + (kRun - 1) * waves + 1) * 256 <= n) {
      float v[kRun][4];
#pragma unroll
      for (int u = 0; u < kRun; u++) kq_quad_wide<TYPE>(data + (b0 + u * waves) * kq_bytes<TYPE>(), lane, v[u]);
#pragma unroll
      for (int u = 0; u < kRun; u++)
        *reinterpret_cast<float4*>(out + (b0 + u * waves) * 256 + 4 * lane) =
            make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
      continue;
    }
    for (size_t b = b0; b < nblk && b < b0 + kRun * waves; b += waves) {
      const size_t e = b * 256 + 4 * lane;
      float v[4];
      if (WIDE && (b + 1) * 256 <= n) {
        kq_quad_wide<TYPE>(data + b * kq_bytes<TYPE>(), lane, v);
        *reinterpret_cast<float4*>(out + e) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
        kq_quad<TYPE>(data + b * kq_bytes<TYPE>(), lane, v);
        if (OUT16 && !WIDE && e + 4 <= n) {  // (WIDE: the matrix's last block only)
          *reinterpret_cast<float4*>(out + e) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
          for (int t = 0; t < 4 && e + t < n; t++) out[e + t] = v[t];
        }
      }
    }
  }
}

// y[row] = sum_k dequant(W)[row, k] * x[k] (+ residual[row]): one wave per row
// (grid-stride), lane l takes quad l (elements 4l..4l+3) of every block of the
// row.  y may be the residual itself (each row is read, then written, by one lane).
template <int TYPE>
__global__ __launch_bounds__(256) void kq_gemv_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                      const float* residual, float* y, size_t n_rows, size_t nb) {
  const int lane = threadIdx.x & 63;
  const size_t waves = static_cast<size_t>(gridDim.x) * (blockDim.x >> 6);
  for (size_t row = static_cast<size_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6); row < n_rows;
       row += waves) {
    const uint8_t* rp = w + row * nb * kq_bytes<TYPE>();
    float acc = 0.f;
    for (size_t b = 0; b < nb; b++) {
      float v[4];
      kq_quad<TYPE>(rp + b * kq_bytes<TYPE>(), lane, v);
      const float* xb = x + 256 * b + 4 * lane;
#pragma unroll
      for (int t = 0; t < 4; t++) acc = __builtin_fmaf(v[t], xb[t], acc);
    }
    acc = whd::wave_sum(acc);
    if (lane == 0) y[row] = residual ? residual[row] + acc : acc;
  }
}

// ------------------------------------------------------ prefill repacking
// A K-quant matrix is rewritten once per handle or call into the stage records
// of the prefill GEMM (kGemmQ4S, kGemmQ6S in wh_common.hpp): the integer
// quants and sub-block scales as they are, the scales and d as floats.  d is
// exact (times a power of two).  An infinite d makes d * s * q infinite, or NaN
// where s or q is 0; the GEMM multiplies d with sums of s * q * x, in which that
// zero is lost, so the record's d is NaN then.  zero() tells whether any s or q
// of the super-block is 0, and is asked for an infinite d only.
template <typename Zero>
__device__ __forceinline__ float record_d(uint32_t bits16, float p, Zero zero) {
  float d = whd::f16_bits_to_f32(bits16) * p;
  if ((bits16 & 0x7FFFu) == 0x7C00u && zero()) d = __builtin_nanf("");
  return d;
}

// Workgroup -> (row group, super-block), super-blocks fastest.  Consecutive
// workgroups run on different XCDs, and a row's super-blocks share cache lines
// (144 or 210 bytes each), so each XCD takes a contiguous part of the order
// (Q4_K 14336 x 4096: 19.7 -> 16.9 us, 28672 x 8192: 65.6 -> 53.6 us).
__device__ __forceinline__ unsigned kq_group() {
  const unsigned q = gridDim.x / 8, rem = gridDim.x % 8, xcd = blockIdx.x % 8;
  return xcd * q + min(xcd, rem) + blockIdx.x / 8;
}

// Q4_K: a workgroup stages one super-block of 64 rows in LDS (144-byte runs),
// wave s forms their records of the super-block's stage s, and the records go
// out through LDS as contiguous runs.  16-byte aligned input.
constexpr int kQ4Rows = 64;
__global__ __launch_bounds__(256) void kq_repack_q4k_kernel(const uint8_t* __restrict__ w, int n_rows, unsigned nsb,
                                                            uint8_t* __restrict__ out, uint16_t* __restrict__ dmin_t,
                                                            int dmin_stride) {
  __shared__ uint4 stage[kQ4Rows * 9];
  __shared__ uint2 rec2[4][kQ4Rows * 5];
  const unsigned at = kq_group();
  const int sb = static_cast<int>(at % nsb), r0 = static_cast<int>(at / nsb) * kQ4Rows;
  const int rows = min(kQ4Rows, n_rows - r0);
  const int s = static_cast<int>(threadIdx.x) >> 6, row = static_cast<int>(threadIdx.x) & 63;
  for (int i = threadIdx.x; i < 9 * rows; i += 256)
    stage[i] = *reinterpret_cast<const uint4*>(w + (static_cast<size_t>(r0 + i / 9) * nsb + sb) * 144 + 16 * (i % 9));
  __syncthreads();
  // even quants of a dword into its low half, odd ones into the high half
  auto split = [](uint32_t u) {
    auto gather = [](uint32_t x) {
      x = (x | (x >> 4)) & 0x00FF00FFu;
      return (x | (x >> 8)) & 0xFFFFu;
    };
    return gather(u & 0x0F0F0F0Fu) | (gather((u >> 4) & 0x0F0F0F0Fu) << 16);
  };
  auto scale = [](uint32_t v) {
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(static_cast<float>(v << 10))));
  };
  if (row < rows) {
    const uint4 h = stage[9 * row], qa = stage[9 * row + 1 + 2 * s], qb = stage[9 * row + 2 + 2 * s];
    // scales 2s, 2s + 1: bits 0..5 and 14..19 of the 24 bits at bit 24s
    const uint32_t pr = s == 0 ? h.x : (s == 1 ? (h.x >> 24) | (h.y << 8) : (s == 2 ? (h.y >> 16) | (h.z << 16) : h.z >> 8));
    uint2* rec = rec2[s] + 5 * row;
    rec[0] = make_uint2(split(qa.x), split(qa.y));
    rec[1] = make_uint2(split(qa.z), split(qa.w));
    rec[2] = make_uint2(split(qb.x), split(qb.y));
    rec[3] = make_uint2(split(qb.z), split(qb.w));
    auto zero = [&]() {
      const uint32_t* b = reinterpret_cast<const uint32_t*>(stage + 9 * row);
      uint32_t z = 0;
#pragma unroll 1
      for (int i = 4; i < 36; i++) z |= (b[i] - 0x11111111u) & ~b[i] & 0x88888888u;  // a zero nibble
#pragma unroll 1
      for (int j = 0; j < 8; j++) z |= q4k_scale(reinterpret_cast<const uint8_t*>(b), j) == 0;
      return z != 0;
    };
    rec[4] = make_uint2(scale(pr & 63u) | (scale((pr >> 14) & 63u) << 16),
                        __float_as_uint(record_d(h.w & 0xFFFFu, 16384.f, zero)));
    if (s == 0) {
      uint16_t* tr = dmin_t + static_cast<size_t>(r0 + row) * dmin_stride;
      tr[sb] = static_cast<uint16_t>(h.w >> 16);
      if (sb + 1 == static_cast<int>(nsb))  // the row's last super-block clears the padding
        for (int z = static_cast<int>(nsb); z < dmin_stride; z++) tr[z] = 0;
    }
  }
  __syncthreads();
  uint2* dst = reinterpret_cast<uint2*>(out + (static_cast<size_t>(4 * sb + s) * n_rows + r0) * 40);
  for (int i = row; i < 5 * rows; i += 64) dst[i] = rec2[s][i];
}

// Q6_K: a workgroup stages one super-block of 32 rows in LDS (13 loads of 16
// bytes and one of 2 per row, only 2-byte aligned in memory: 14336 x 4096 takes
// 24.1 us with them, 35.3 with a dword per lane), each thread forms half a record: 32 elements share 16 bytes of ql
// (element i and i + 16 the same byte) and 8 bytes of qh (9 for the upper half
// of the block, whose bits start 2 higher and run into the next byte).  The
// records go through LDS too, so that the stores are contiguous.
constexpr int kQ6Rows = 32, kQ6Stride = 53;  // dwords per staged block
__global__ __launch_bounds__(256) void kq_repack_q6k_kernel(const uint8_t* __restrict__ w, int n_rows, unsigned nsb,
                                                            uint8_t* __restrict__ out) {
  __shared__ uint32_t stage[kQ6Rows * kQ6Stride];
  __shared__ uint4 rec4[4][kQ6Rows * 5];
  const unsigned at = kq_group();
  const int sb = static_cast<int>(at % nsb), r0 = static_cast<int>(at / nsb) * kQ6Rows;
  const int rows = min(kQ6Rows, n_rows - r0);
  const int wave = static_cast<int>(threadIdx.x) >> 6, lane = static_cast<int>(threadIdx.x) & 63;
#pragma unroll
  for (int i = 0; i < kQ6Rows * 14 / 256 + 1; i++) {
    const int p = 256 * i + static_cast<int>(threadIdx.x), r = p / 14, c = p % 14;
    if (r >= rows) break;
    const uint8_t* b = w + (static_cast<size_t>(r0 + r) * nsb + sb) * 210 + 16 * c;
    uint32_t* d = stage + r * kQ6Stride + 4 * c;
    if (c < 13) {
      uint4 v;
      __builtin_memcpy(&v, b, 16);
      d[0] = v.x;
      d[1] = v.y;
      d[2] = v.z;
      d[3] = v.w;
    } else {
      d[0] = *reinterpret_cast<const uint16_t*>(b);  // the block's last two bytes: d
    }
  }
  __syncthreads();
  const int s = wave, r = lane >> 1, half = lane & 1;
  const uint32_t* b = stage + r * kQ6Stride;
  // the quants of elements 32 grp .. 32 grp + 31, a byte each
  auto quants = [&](int grp, uint32_t (&q)[8]) {
    const bool upper = grp >= 4;
    const uint32_t h[3] = {b[32 + 2 * grp], b[33 + 2 * grp], grp == 7 ? 0u : b[34 + 2 * grp]};
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const uint32_t nib = (b[4 * grp + (c & 3)] >> (upper ? 4 : 0)) & 0x0F0F0F0Fu;
      // byte c of h with the byte behind it, the pairs of bits from bit 0 (2)
      const uint32_t two = __builtin_amdgcn_alignbit(h[c / 4 + 1], h[c / 4], 8 * (c & 3)) >> (upper ? 2 : 0);
      q[c] = nib | (two & 3u) << 4 | (two & 0xCu) << 10 | (two & 0x30u) << 16 | (two & 0xC0u) << 22;
    }
  };
  uint32_t q[8];
  quants(2 * s + half, q);
  uint4* rec = rec4[s] + 5 * r;
  rec[2 * half] = make_uint4(q[0], q[1], q[2], q[3]);
  rec[2 * half + 1] = make_uint4(q[4], q[5], q[6], q[7]);
  const uint32_t sc = b[48 + s] >> (16 * half);  // scales 4s + 2 half, + 1
  auto scale = [](uint32_t v) {
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(static_cast<float>(v & 0xFFu))));
  };
  auto zero = [&]() {
    auto zero_byte = [](uint32_t v) { return (v - 0x01010101u) & ~v & 0x80808080u; };
    uint32_t z = zero_byte(b[48]) | zero_byte(b[49]) | zero_byte(b[50]) | zero_byte(b[51]);
#pragma unroll 1
    for (int grp = 0; grp < 8; grp++) {
      uint32_t v[8];
      quants(grp, v);
#pragma unroll
      for (int c = 0; c < 8; c++) z |= zero_byte(v[c] ^ 0x20202020u);  // q - 32
    }
    return z != 0;
  };
  uint32_t* meta = reinterpret_cast<uint32_t*>(rec + 4);
  meta[half] = scale(sc) | (scale(sc >> 8) << 16);
  meta[2 + half] = half ? 0u : __float_as_uint(record_d(b[52] & 0xFFFFu, 0.015625f, zero));
  __syncthreads();
  uint4* dst = reinterpret_cast<uint4*>(out + (static_cast<size_t>(4 * sb + s) * n_rows + r0) * 80);
  for (int i = lane; i < 5 * rows; i += 64) dst[i] = rec4[s][i];
}

unsigned kq_grid(size_t work, unsigned per_block) {
  size_t g = (work + per_block - 1) / per_block;
  const size_t cap = static_cast<size_t>(wh::cu_count()) * 16;
  if (g > cap) g = cap;
  return static_cast<unsigned>(g < 1 ? 1 : g);
}

}  // namespace

namespace wh {

int launch_dequantize_kquant(int type, const void* data, size_t n, float* out, hipStream_t s) {
  if (n == 0) return WH_OK;
  const uint8_t* p = static_cast<const uint8_t*>(data);
  const size_t wgs = (n + 1023) / 1024, cap = static_cast<size_t>(wh::cu_count()) * 8;  // a block per wavefront
  const unsigned grid = static_cast<unsigned>(wgs < cap ? wgs : cap);
  const bool o16 = wh::aligned(out, 16);
  auto go = [&](auto kernel) { kernel<<<grid, 256, 0, s>>>(p, out, n); };
  if (type == WH_TYPE_Q4_K) {
    if (o16) go(wh::aligned(data, 16) ? kq_dequant_kernel<WH_TYPE_Q4_K, true, true> : kq_dequant_kernel<WH_TYPE_Q4_K, false, true>);
    else go(kq_dequant_kernel<WH_TYPE_Q4_K, false, false>);
  } else {
    go(o16 ? kq_dequant_kernel<WH_TYPE_Q6_K, true, true> : kq_dequant_kernel<WH_TYPE_Q6_K, false, false>);
  }
  WH_LAUNCH_CHECK("dequantize (k-quant) kernel launch");
  return WH_OK;
}

int launch_gemv_kquant(int type, const void* w, const float* x, float* y, size_t n_rows, size_t k, hipStream_t s,
                       const float* residual) {
  if (n_rows == 0) return WH_OK;
  const uint8_t* p = static_cast<const uint8_t*>(w);
  const unsigned grid = kq_grid(n_rows, 4);
  if (type == WH_TYPE_Q4_K) kq_gemv_kernel<WH_TYPE_Q4_K><<<grid, 256, 0, s>>>(p, x, residual, y, n_rows, k / 256);
  else kq_gemv_kernel<WH_TYPE_Q6_K><<<grid, 256, 0, s>>>(p, x, residual, y, n_rows, k / 256);
  WH_LAUNCH_CHECK("gemv (k-quant) kernel launch");
  return WH_OK;
}

int launch_repack_kquant(int type, const void* w, size_t n_rows, size_t k, void* out, hipStream_t s) {
  if (n_rows == 0 || k == 0) return WH_OK;
  const uint8_t* p = static_cast<const uint8_t*>(w);
  uint8_t* o = static_cast<uint8_t*>(out);
  const int rows = static_cast<int>(n_rows);
  // super-blocks and row groups in x, the one grid dimension beyond 65535
  const unsigned nsb = static_cast<unsigned>(k / 256);
  auto grid = [&](int group) { return static_cast<unsigned>(nsb * ((n_rows + group - 1) / group)); };
  if (type == WH_TYPE_Q4_K) {
    uint16_t* dmin_t = reinterpret_cast<uint16_t*>(o + n_rows * (k / 64) * 40);
    kq_repack_q4k_kernel<<<grid(kQ4Rows), 256, 0, s>>>(p, rows, nsb, o, dmin_t, static_cast<int>(q4s_dmin_stride(k)));
  } else {
    kq_repack_q6k_kernel<<<grid(kQ6Rows), 256, 0, s>>>(p, rows, nsb, o);
  }
  WH_LAUNCH_CHECK("k-quant repack kernel launch");
  return WH_OK;
}

}  // namespace wh
