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

}  // namespace ipus
