// gemm_dev.hpp -- device helpers shared by the prefill GEMMs (gemm_tiled.hip,
// gemm_sb.hpp): MFMA operand types, global -> LDS copies, the waits on them and
// the stream-K partial tiles.
#pragma once

#include "wh_blocks.hpp"

// raw buffer load / store of 16 bytes (llvm.amdgcn.raw.buffer.{load,store}.v4f32)
__device__ float __attribute__((ext_vector_type(4))) gt_buffer_load_x4(int __attribute__((ext_vector_type(4))) rsrc,
                                                                       int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.buffer.load.v4f32");
__device__ void gt_buffer_store_x4(float __attribute__((ext_vector_type(4))) v, int __attribute__((ext_vector_type(4))) rsrc,
                                   int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.store.v4f32");

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int TBN = 256;              // weight rows per tile
constexpr int TWAVES = 8;             // 2 per SIMD
constexpr int FRAG = 1024;            // bytes per activation fragment (16 tokens x 32 k, one limb)

// Global -> LDS copies (global_load_lds): lane l's 16 (or 4) bytes at
// base + voff land at LDS address lds + 16 l (4 l).  Issued through inline asm
// so that the compiler does not treat them as pending LDS writes (it would
// otherwise wait for every copy in flight before each LDS read); completion
// is tracked explicitly with wait_vmcnt.  The copy reads its LDS address from
// M0, a register the compiler reserves: the statement saves M0 in an SGPR of
// its own, sets it (one wait state before the copy reads it, as GFX9-family
// parts require after an SALU write of M0) and restores it, so M0 holds the
// compiler's value again after every copy.
__device__ __forceinline__ void copy16_to_lds(const void* base, uint32_t voff, uint32_t lds) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);  // wave-uniform by construction
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(voff), "s"(base), "s"(m0)
      : "memory");
}
__device__ __forceinline__ void copy4_to_lds(const void* base, uint32_t voff, uint32_t lds) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(voff), "s"(base), "s"(m0)
      : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  // generic -> LDS address space (an address-space cast), then its 32-bit address
  return static_cast<uint32_t>((uintptr_t)((const __attribute__((address_space(3))) uint8_t*)p));
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Stream-K partial tiles: a buffer resource over one slot (128 KB or less)
// and the cache policy of the slot's loads and stores, sc1 (bit 4 of the
// buffer instructions' cache-policy operand on gfx950): the policy the memory
// model gives agent-scope atomic loads and stores, coherent across the XCDs'
// L2s without a cache-wide writeback or invalidate.
constexpr int kSkCoherent = 16;
__device__ __forceinline__ int __attribute__((ext_vector_type(4))) sk_rsrc(const float* base) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  int __attribute__((ext_vector_type(4))) r;
  r[0] = static_cast<int>(static_cast<uint32_t>(a));
  r[1] = static_cast<int>(static_cast<uint32_t>(a >> 32) & 0xFFFFu);
  r[2] = 1 << 20;  // 1 MB of records: every slot offset is in range
  r[3] = 0x00020000;
  return r;
}

// Waits until at most min(n, J) stages of N copies each are in flight.
template <int N, int J>
__device__ __forceinline__ void wait_stages(int n) {
  if constexpr (J == 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= J) wait_vmcnt<J * N>();
    else wait_stages<N, J - 1>(n);
  }
}
