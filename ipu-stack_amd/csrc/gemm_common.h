// Device helpers shared by the GEMM kernels: LDS DMA, and the arithmetic of the
// fp16 kernels' epilogues.
#pragma once

#include "device_common.h"
#include "kernels.h"

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
// The first `valid` elements of a chunk, zero past them.
__device__ __forceinline__ u32x4 keep_elements(u32x4 v, uint32_t valid) {
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w)
    v[w] &= (2 * w < valid ? 0xffffu : 0u) | (2 * w + 1 < valid ? 0xffff0000u : 0u);
  return v;
}
// Elements at .. at + 7 (at < total) of an operand of `total` elements, any past
// its end the last one.  That chunk's elements are eight independent loads,
// clamped to the operand, not eight tests and loads in turn.
__device__ __forceinline__ u32x4 load_chunk(const uint16_t* x, uint64_t at, uint64_t total) {
  if (at + 8 <= total) return *reinterpret_cast<const u32x4_elements*>(x + at);
  uint32_t e[8];
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i) e[i] = x[at + i < total ? at + i : total - 1];
  return u32x4{e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16};
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
// The same on a chunk in LDS.
__device__ __forceinline__ void clear_chunk_past(uint8_t* chunk, uint32_t valid) {
  u32x4* p = reinterpret_cast<u32x4*>(chunk);
  *p = keep_elements(*p, valid);
}

// Split launches of the 32 x 32 tile kernels: workgroup (x, y, z) takes k in
// [z * chunk, (z + 1) * chunk) of its tile; every split holds at least one k.
struct SplitK {
  float* parts = nullptr;        // [batches * tiles][splits][fragments][threads][4]
  uint32_t* counters = nullptr;  // one per tile, all 0 between launches
  uint32_t splits = 1, chunk = 0;  // chunk: a multiple of the K step
};

// Every split leaves its sums (one 16-byte slot per thread and fragment, rows
// past C none); the last one, where this is true, adds all of them into acc, in
// the order of K.
template <int Threads, int MT, int NT, class Stored>
__device__ __forceinline__ bool add_splits(const SplitK& split, uint64_t tile, float4_t (&acc)[MT][NT], Stored stored) {
  constexpr uint64_t kSlots = (uint64_t)Threads * MT * NT;
  float* part = split.parts + (tile * split.splits * kSlots + threadIdx.x) * 4;
  auto slot = [&](uint32_t z, int i, int j) { return part + (z * kSlots + (uint64_t)(i * NT + j) * Threads) * 4; };
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (stored(i)) store_device4(slot(blockIdx.z, i, j), acc[i][j]);
  __shared__ uint32_t arrived;
  if (!arrive(split.counters + tile, split.splits, &arrived)) return false;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
      if (!stored(i)) continue;
      // Eight loads in flight (past the last split: the last one again, not added).
      for (uint32_t z0 = 0; z0 < split.splits; z0 += 8) {
        float4_t x[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
          x[u] = load_device4(slot(z0 + u < split.splits ? z0 + u : split.splits - 1, i, j));
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
          if (z0 + u < split.splits) acc[i][j] += x[u];
      }
    }
  }
  return true;
}

// K splits for at most 128 tiles of 32 x 32 (decode projections, small products
// with a long K), where the walk over K of few workgroups leaves CUs and memory
// idle: at most one workgroup per CU and 8 splits.  Modelled time, us: step_us
// per K step of `step` (fp16, 128 k: 0.25; 0.2 from L2, 0.28-0.49 from HBM; fp32,
// 64 k: 0.30), and for a split launch 2 for the partial sums, the count and the
// merge, 0.1 per split and 1.1 per MB of partial sums.  Measured, fp16, unsplit
// and at this choice, weights in HBM: 8 x 4096 x
// 4096 18.0 -> 13.4 (4 splits 13.9; transposed weights 10.6 -> 10.1), 8 x 2048 x 8192
// 31.6 -> 13.1 (8 splits 13.4), 16 x 1024 x 4096 11.5 -> 6.8, 8 x 512 x 8192 19.9 ->
// 7.1, 64 x 64 x 8192 15.5 -> 6.3, 256 x 256 x 4096 10.2 -> 7.4, 8 x 1024 x 2048 6.9 -> 5.8.
// Not worth it: 320 x 320 x 2000 5.5 -> 6.6, 64 x 2048 x 2048 6.8 -> 7.0, 8 x 4096 x
// 1024 4.7 -> 6.0.
// fp32: 8 x 4096 x 4096 21.6 -> 16.6, 16 x 1024 x 4096 21.2 -> 8.6, 8 x 2048 x 2048 12.0 ->
// 8.3, 8 x 512 x 8192 39.0 -> 10.2, 64 x 64 x 8192 38.3 -> 8.9, 64 x 2048 x 2048 13.5 -> 11.0, 64 x
// 1024 x 1024 7.1 -> 6.9; 320 x 320 x 1000 stays unsplit (7.3).
// The plan is made for plan_tiles, the tiles of the folded product where the
// batches could be folded (launch_gemm_f16), so that it does not depend on the
// epilogue; `launched` tiles (at most 32 per folded one) use the workspace.
inline bool split_plan(const GemmArgs& a, uint64_t plan_tiles, uint64_t launched, uint32_t step, double step_us,
                       SplitK* s) {
  if (!a.workspace.data || plan_tiles > 128 || launched > a.workspace.counter_count) return false;
  const uint32_t steps = (a.inner + step - 1) / step;
  constexpr uint64_t kTileBytes = 32 * 32 * sizeof(float);
  const uint64_t rows = (uint64_t)a.rows * a.batches;
  const double stored = (double)plan_tiles * (rows < 32 ? rows : 32) * 32 * sizeof(float);
  double best_us = steps * step_us;
  uint32_t best = 1;
  for (uint32_t want = 2; want <= 8 && want * plan_tiles <= 256 && want * 2 <= steps; ++want) {
    const uint32_t per = (steps + want - 1) / want, splits = (steps + per - 1) / per;
    if (launched * splits * kTileBytes > a.workspace.bytes) break;
    const double us = per * step_us + 2.0 + 0.1 * splits + 1.1e-6 * stored * splits;
    if (us < best_us) {
      best_us = us;
      best = splits;
      s->chunk = per * step;
    }
  }
  if (best < 2) return false;
  s->splits = best;
  s->parts = (float*)a.workspace.data;
  s->counters = a.workspace.counters;
  return true;
}

}  // namespace ipus
