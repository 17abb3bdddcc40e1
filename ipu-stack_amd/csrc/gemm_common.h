// Device helpers shared by the GEMM kernels: LDS DMA, and the arithmetic of the
// fp16 kernels' epilogues.
#pragma once

#include "device_common.h"

#define LDS_AS __attribute__((address_space(3)))

namespace ipus {

constexpr int kBufferFlags = 0x00020000;  // raw buffer, dword 3 of the descriptor

typedef short short4_t __attribute__((vector_size(8)));

inline int hip_status(hipError_t e) { return e == hipSuccess ? 0 : IPUS_ERROR_HIP_BASE - (int)e; }

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, uint8_t* lds, uint32_t voffset,
                                      uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (LDS_AS void*)lds, 16, voffset, soffset, 0, 0);
}

// Offset of a chunk outside the operand (past M or N along an MN-contiguous
// row, or past K on the last K step of a K-contiguous row): beyond every
// buffer range (< 2^31) plus any K offset (< 2^31) without wrapping, so the
// load returns 0.
constexpr uint32_t kPadOffset = 0x80000000u;

// Epilogues: the plain fp16 product; GELU of it; or the sum of it and an
// addend element (C += A . B, the reference's accumulate mode).
enum Epilogue : int { kEpiPlain = 0, kEpiGelu = 1, kEpiAdd = 2 };

// fp16 result of one accumulator; with GELU, GELU of that fp16 value (the
// same number the separate GELU kernel would produce from the stored GEMM
// output).  The add epilogue applies add_f16 to this value afterwards.
template <int Epi>
__device__ __forceinline__ half_t epilogue(float acc) {
  const half_t h = (half_t)acc;
  if constexpr (Epi == kEpiGelu) return (half_t)gelu_tanh((float)h);
  return h;
}

// The fp16 Add kernel's arithmetic (k_memory.hip add_kernel): both operands
// widened to fp32, summed, rounded once to fp16, so a fused accumulate is
// bit-identical to a GEMM followed by an Add.
__device__ __forceinline__ half_t add_f16(half_t product, half_t addend) {
  return (half_t)((float)addend + (float)product);
}
__device__ __forceinline__ u32x4 add_f16x8(u32x4 product, u32x4 addend) {
  const half8_t p = __builtin_bit_cast(half8_t, product), a = __builtin_bit_cast(half8_t, addend);
  half8_t r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = add_f16(p[e], a[e]);
  return __builtin_bit_cast(u32x4, r);
}

// Operand edges of the LDS-DMA kernels.  kWhole: K a multiple of the K step,
// every row pitch a multiple of 8 elements, 16-byte aligned addresses.  kKTail:
// the same with a partial last step.  kDwords: operand pitches and addresses that
// are only multiples of 4 bytes (any K, and any C): the DMA fetches the same 16-byte
// chunks, dword-aligned; a chunk that runs past M or N along a row holds
// elements of the next row, which reach only rows or columns of C that are not
// stored, and a chunk that runs past K along a row is cleared past K in LDS
// (clear_past_k) before the last step reads it.
// kElements (k_gemm_f16_tile.hip only): any pitch, address and extent; the
// chunks go through registers instead, read at element alignment.
enum Edge : int { kWhole = 0, kKTail = 1, kDwords = 2, kElements = 3 };

// 16-byte access at element (2-byte) alignment: one global_load/store_dwordx4
// (the device runs in unaligned access mode).
typedef u32x4 __attribute__((aligned(2))) u32x4_elements;
// Elements at .. at + 7 of an operand of `total` elements, zero past its end.
__device__ __forceinline__ u32x4 load_chunk(const uint16_t* x, uint64_t at, uint64_t total) {
  if (at + 8 <= total) return *reinterpret_cast<const u32x4_elements*>(x + at);
  u32x4 v = {0, 0, 0, 0};
#pragma unroll
  for (uint32_t e = 0; e < 8; ++e)
    if (at + e < total) v[e / 2] |= (uint32_t)x[at + e] << (16 * (e % 2));
  return v;
}
// 16 bytes of C (8 columns of one row), `valid` columns of them inside the row.
__device__ __forceinline__ void store_elements(uint16_t* p, u32x4 v, uint32_t valid) {
  if (valid >= 8) {
    *reinterpret_cast<u32x4_elements*>(p) = v;
  } else {
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e)
      if (e < valid) p[e] = (uint16_t)(v[e / 2] >> (16 * (e % 2)));
  }
}

// Eight elements of an addend row of any alignment, `valid` of them inside it.
__device__ __forceinline__ u32x4 load_elements(const uint16_t* p, uint32_t valid) {
  u32x4 v = {0, 0, 0, 0};
#pragma unroll
  for (uint32_t e = 0; e < 8; ++e)
    if (e < valid) v[e / 2] |= (uint32_t)p[e] << (16 * (e % 2));
  return v;
}
// The first `valid` elements of a chunk, zero past them.
__device__ __forceinline__ u32x4 keep_elements(u32x4 v, uint32_t valid) {
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w)
    v[w] &= (2 * w < valid ? 0xffffu : 0u) | (2 * w + 1 < valid ? 0xffff0000u : 0u);
  return v;
}
// The same on a chunk in LDS.
__device__ __forceinline__ void clear_chunk_past(uint8_t* chunk, uint32_t valid) {
  u32x4* p = reinterpret_cast<u32x4*>(chunk);
  *p = keep_elements(*p, valid);
}

}  // namespace ipus
