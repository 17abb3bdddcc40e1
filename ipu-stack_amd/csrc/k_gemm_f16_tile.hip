// fp16 GEMM on gfx950 MFMA for the products that the 256 x 256 kernel
// (k_gemm_f16.hip) leaves part of the chip idle on: 128 x 128, 64 x 64 or 32 x
// 32 tiles of C, fp32 accumulation, fp16 output, the same operand conditions
// (fast_ok), layouts, epilogues and edges.  Replaces gemm_f16_amp
// (device/gemm_f16_amp.S:186-440) for those shapes.
//
// What bounds it: with few tiles per CU the K loop is a stream of operand
// tiles from L2 and the Infinity Cache, not of MFMAs (128 x 128 tiles on
// 2048^3, ns per 64-k step: the DMA alone 345-434, 215 where the operands fit
// L2 = 64 B/clk/CU; the MFMAs alone 230-330; both 425-550).  So:
//   * operand tiles go global -> LDS by DMA (buffer_load ... lds), four stages
//     deep: three steps are in flight while one is read, with counted waits
//     (vmcnt) so that a step waits only for its own stage;
//   * the fragments of step k + 1 are read into the second register buffer
//     between the MFMAs of step k, so one barrier per step both publishes
//     stage k + 1 and frees stage k for the DMA of step k + 4;
//   * 128 x 128 and 64 x 64 tiles run two K groups of four waves: group g
//     takes the 32-k substep g of every step, so that two waves per SIMD
//     cover each other's waits with the same LDS reads as four waves (128 x
//     128, 2048^3: 21.6 -> 21.1 us, 1024^3 11.1 -> 9.4, 729 x 4304 x 1152 13.0
//     -> 11.8); the groups' fp32 sums are added through LDS at the end;
//   * few 32 x 32 tiles with a long K split K over workgroups, and the last one
//     adds the partial sums in the order of K (split_plan, gemm_common.h);
//   * C leaves through LDS in whole row runs, as in the 256 x 256 kernel.
// Measured, us per launch, before (256 x 256 kernel or the register-staged
// small-tile kernel) and now: 2048^3 38.0 -> 21.1 (128 x 128), 729 x 4304 x
// 1152 26.0 -> 11.8 (128 x 128), 1024^3 9.5 -> 5.3 (64 x 64), 729 x 1152 x 1152
// 10.4 -> 5.6, 729 x 1152 x 4304 31 -> 17.6 (64 x 64), 512 x 512 x 4096 28 -> 8.4
// (32 x 32).  Not kept: prefetching lines into L2 8 to 16 steps ahead with one
// load per wave (2048^3 21.1 -> 22.1, 729 x 1152 x 4304 on 64 x 64 17.7 ->
// 20.9), two stages and two workgroups per CU (2048^3 24.9), 128-k steps on 64
// x 64 tiles (2048^3 33.0 against 27.7).
//
// Operands the DMA cannot fetch (odd row pitches or addresses, kElements) take
// the same kernel with the tiles going through registers: chunks are read at
// element alignment two steps before they are stored to LDS.
#include "../../include/ipus.h"

#include "device_common.h"
#include "gemm_common.h"
#include "kernels.h"
#include "tile_choice.h"
#include "tile_grid.h"

namespace ipus {
namespace {

// Tile of C (TM x TN), part of one wave (WM x WN), K groups, k per step.
template <int BM, int BN, int WM_, int WN_, int KG_, int BK_>
struct TileShape {
  static constexpr int TM = BM, TN = BN, WM = WM_, WN = WN_, KG = KG_, BK = BK_;
  static constexpr int S = 4;  // LDS stages
  static constexpr int kWavesM = TM / WM, kWavesN = TN / WN;
  static constexpr int kWaves = kWavesM * kWavesN * KG;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kABytes = TM * BK * 2, kBBytes = TN * BK * 2;
  static constexpr int kStageBytes = kABytes + kBBytes;
  static constexpr int kDmaA = kABytes / 1024 / kWaves, kDmaB = kBBytes / 1024 / kWaves;
  static constexpr int kDma = kDmaA + kDmaB;
  static constexpr int kMT = WM / 16, kNT = WN / 16;
  static constexpr int kSub = BK / 32 / KG;  // 32-k substeps per step and K group
  static_assert(kABytes % (1024 * kWaves) == 0 && kBBytes % (1024 * kWaves) == 0, "whole DMA instructions per wave");
  static_assert(KG == 1 || KG == 2, "the exchange of partial sums is between two groups");
};

typedef TileShape<128, 128, 64, 64, 2, 64> Tile128;
typedef TileShape<64, 64, 32, 32, 2, 64> Tile64;
typedef TileShape<32, 32, 16, 16, 1, 128> Tile32;

// LDS tiles.  K-contiguous operand: subtiles of 64 k, each [rows][64 k] with
// the 16-byte chunk XORed by row & 7.  MN-contiguous: [k][mn], the chunk XORed
// by mn_swz(k).  A fragment read (ds_read_b64_tr_b16) takes 32 bytes of the 16
// rows 8 g + {0..3} (g = 0..3, + 4 for its second half): the XOR spreads them
// evenly over the 8 bank groups of 32 bytes, for rows of 256 bytes by row
// bits 0, 1 and 3; 128-byte rows alternate halves of the banks by row bit 0 by
// themselves, 64-byte rows quarters by bits 0 and 1.
template <int RowBytes>
__device__ __forceinline__ uint32_t mn_swz(uint32_t k) {
  if constexpr (RowBytes >= 256)
    return ((k & 3u) | (((k >> 3) & 1u) << 2)) << 1;
  else if constexpr (RowBytes == 128)
    return (((k >> 1) & 1u) | (((k >> 3) & 1u) << 1)) << 1;
  else
    return ((k >> 3) & 1u) << 1;
}

// Two workgroups share a CU except with 128 x 128 tiles (LDS); the registers of 64
// x 64 tiles' kElements form have to be held to that (4 waves per SIMD).
template <class T, bool TransposeLeft, bool TransposeRight, int Epi, int E, bool Split>
__global__ __launch_bounds__(T::kThreads, E == kElements && T::TM == 64 ? 4 : 1) void gemm_f16_tile_kernel(
    uint16_t* out, const uint16_t* __restrict__ left, const uint16_t* __restrict__ right,
    uint32_t M, uint32_t N, uint32_t K, uint64_t left_batch_stride, uint64_t right_batch_stride,
    const uint16_t* addend, uint64_t addend_batch_stride, uint32_t addend_row_stride,
    SplitK split) {
  static_assert(!Split || (T::KG == 1 && E != kElements), "splits: one K group, operands by DMA");
  constexpr int TM = T::TM, TN = T::TN, BK = T::BK, S = T::S, KG = T::KG;
  constexpr int kMT = T::kMT, kNT = T::kNT, kSub = T::kSub;
  constexpr int kDmaA = T::kDmaA, kDmaB = T::kDmaB;
  constexpr bool KTail = E == kKTail || E == kDwords;
  constexpr bool kRegs = E == kElements;  // operands through registers, not by DMA
  // Four stages, each a distinct LDS object: the compiler can then see that
  // a DMA into one never aliases the fragment reads of another.
  __shared__ __attribute__((aligned(1024))) uint8_t lds0[T::kStageBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t lds1[T::kStageBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t lds2[T::kStageBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t lds3[T::kStageBytes];
  constexpr bool kAK = !TransposeLeft;   // A rows (m) K-contiguous
  constexpr bool kBK_ = TransposeRight;  // B^T rows (n) K-contiguous

  const uint32_t nbm = (M + TM - 1) / TM, nbn = (N + TN - 1) / TN;
  const uint32_t tiles = nbm * nbn;
  const uint32_t block = Split ? blockIdx.x : grid_tile(blockIdx.x, blockIdx.z);
  if (!Split && block >= tiles) return;
  // XCD-contiguous tiles: workgroup ids are dealt round-robin to 8 XCDs.
  const uint32_t xcd = block % 8, per = tiles / 8, rest = tiles % 8;
  const uint32_t pid = xcd * per + (xcd < rest ? xcd : rest) + block / 8;
  constexpr uint32_t kGroup = 8;
  const uint32_t group = pid / (kGroup * nbn);
  const uint32_t first_m = group * kGroup;
  const uint32_t group_rows = (nbm - first_m) < kGroup ? (nbm - first_m) : kGroup;
  const uint32_t in_group = pid % (kGroup * nbn);
  const uint32_t bm = first_m + in_group % group_rows;
  const uint32_t bn = in_group / group_rows;
  const uint32_t m0 = bm * TM, n0 = bn * TN;

  const uint64_t batch = blockIdx.y;
  const uint16_t* A = left + batch * left_batch_stride;
  const uint16_t* B = right + batch * right_batch_stride;
  uint16_t* C = out + batch * (uint64_t)M * N;
  // This workgroup's K range (the whole of K unless Split).
  const uint32_t k_begin = Split ? blockIdx.z * split.chunk : 0;
  const uint32_t k_len = Split ? (K - k_begin < split.chunk ? K - k_begin : split.chunk) : K;
  const uint16_t* a_base = kAK ? A + (uint64_t)m0 * K + k_begin : A + m0 + (uint64_t)k_begin * M;
  const uint16_t* b_base = kBK_ ? B + (uint64_t)n0 * K + k_begin : B + n0 + (uint64_t)k_begin * N;
  const uint64_t a_bytes = (uint64_t)M * K * 2 - (uint64_t)(a_base - A) * 2;
  const uint64_t b_bytes = (uint64_t)N * K * 2 - (uint64_t)(b_base - B) * 2;
  const int a_range = (int)(a_bytes > 0x7fffffffull ? 0x7fffffff : a_bytes);
  const int b_range = (int)(b_bytes > 0x7fffffffull ? 0x7fffffff : b_bytes);

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t kg = wave % KG, wmn = wave / KG;  // K group; position in the M x N grid
  const uint32_t wm = (wmn / T::kWavesN) * T::WM, wn = (wmn % T::kWavesN) * T::WN;
  const uint32_t r16 = lane % 16, g4 = lane / 16;

  // Chunk (row or k row, logical k or mn offset in elements) that the lane
  // fetches for DMA instruction `inst` of a tile.
  auto chunk_of = [&]<bool KContig, int TMN>(uint32_t inst, uint32_t* row, uint32_t* col) __attribute__((always_inline)) {
    if constexpr (KContig) {
      const uint32_t sub = inst / (TMN / 8), r = (inst % (TMN / 8)) * 8 + lane / 8;
      *row = r;
      *col = sub * 64 + ((lane % 8) ^ (r & 7u)) * 8;
    } else {
      const uint32_t k = inst * (1024 / (2 * TMN)) + lane / (TMN / 8);
      *row = k;
      *col = ((lane % (TMN / 8)) ^ mn_swz<2 * TMN>(k)) * 8;
    }
  };
  uint32_t a_voff[kDmaA], b_voff[kDmaB];
  auto offsets = [&]<bool KContig, int TMN, int N_>(uint32_t ld, uint32_t mn_limit, uint32_t (&voff)[N_]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < N_; ++j) {
      uint32_t row, col;
      chunk_of.template operator()<KContig, TMN>(wave * N_ + j, &row, &col);
      voff[j] = KContig || col < mn_limit ? (row * ld + col) * 2 : kPadOffset;
    }
  };
  offsets.template operator()<kAK, TM>(kAK ? K : M, M - m0, a_voff);
  offsets.template operator()<kBK_, TN>(kBK_ ? K : N, N - n0, b_voff);
  const uint32_t a_kstep = kAK ? BK * 2 : BK * M * 2;
  const uint32_t b_kstep = kBK_ ? BK * 2 : BK * N * 2;

  const uint32_t ksteps = (k_len + BK - 1) / BK;
  const uint32_t k_tail = k_len % BK;
  // The DMA of step k into a stage.  Past the last step the descriptors are
  // empty: no memory is read (the stage is never read either), but the
  // instructions are issued, so the wait counts stay exact.
  // KTail: on the last step, K-contiguous chunks and MN-contiguous rows past
  // K get an offset past the range and read 0 (the step's K offset travels in
  // the scalar offset, which the range check does not cover).
  auto dma = [&](uint8_t* stage, uint32_t k) __attribute__((always_inline)) {
    const uint32_t limit = KTail && k == ksteps - 1 ? k_tail : 0u;
    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, k < ksteps ? a_range : 0, kBufferFlags);
    const __amdgpu_buffer_rsrc_t b_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)b_base, 0, k < ksteps ? b_range : 0, kBufferFlags);
    auto one = [&]<bool KContig, int TMN>(__amdgpu_buffer_rsrc_t rsrc, uint8_t* tile, uint32_t inst, uint32_t voff, uint32_t soff) __attribute__((always_inline)) {
      if (KTail && limit != 0) {
        uint32_t row, col;
        chunk_of.template operator()<KContig, TMN>(inst, &row, &col);
        voff = (KContig ? col : row) < limit ? voff : kPadOffset;
      }
      // kDwords: on the last step a chunk can run past the operand's end, so the
      // step's offset moves into the vector offset, which the range check covers.
      const uint32_t v = E == kDwords && k == ksteps - 1 ? soff : 0u;
      dma16(rsrc, tile + inst * 1024, voff + v, soff - v);
    };
#pragma unroll
    for (int j = 0; j < kDmaA; ++j)
      one.template operator()<kAK, TM>(a_rsrc, stage, wave * kDmaA + j, a_voff[j], k * a_kstep);
#pragma unroll
    for (int j = 0; j < kDmaB; ++j)
      one.template operator()<kBK_, TN>(b_rsrc, stage + T::kABytes, wave * kDmaB + j, b_voff[j], k * b_kstep);
  };

  // kElements: this thread's chunks of step k, read at element alignment.  Chunks
  // run on into the next row (which reaches only elements of C that are not
  // stored); rows past M or N and chunks past K are zero.
  auto load_regs = [&](uint32_t k, u32x4 (&v)[kDmaA + kDmaB]) __attribute__((always_inline)) {
    auto one = [&]<bool KContig, int TMN>(const uint16_t* X, uint32_t inst, uint32_t mn0, uint32_t MN) __attribute__((always_inline)) {
      uint32_t row, col;
      chunk_of.template operator()<KContig, TMN>(inst, &row, &col);
      const uint64_t total = (uint64_t)MN * K, k0 = (uint64_t)k * BK;
      const u32x4 zero = {0, 0, 0, 0};
      if constexpr (KContig) {
        const uint64_t at_k = k0 + col;
        const uint32_t mn = mn0 + row;
        return at_k < K && mn < MN ? load_chunk(X, (uint64_t)mn * K + at_k, total) : zero;
      } else {
        const uint64_t at_k = k0 + row;
        return at_k < K && mn0 + col < MN ? load_chunk(X, at_k * MN + mn0 + col, total) : zero;
      }
    };
#pragma unroll
    for (int j = 0; j < kDmaA; ++j) v[j] = one.template operator()<kAK, TM>(A, wave * kDmaA + j, m0, M);
#pragma unroll
    for (int j = 0; j < kDmaB; ++j) v[kDmaA + j] = one.template operator()<kBK_, TN>(B, wave * kDmaB + j, n0, N);
  };
  // Into step k's stage; the chunk that K ends in is cleared past K only here, so
  // that no load of the last step waits for the one before.
  auto store_regs = [&](uint8_t* stage, uint32_t k, u32x4 (&v)[kDmaA + kDmaB]) __attribute__((always_inline)) {
    auto clear = [&]<bool KContig, int TMN>(u32x4& x, uint32_t inst) __attribute__((always_inline)) {
      if constexpr (KContig) {
        uint32_t row, col;
        chunk_of.template operator()<KContig, TMN>(inst, &row, &col);
        if (k_tail > col && k_tail - col < 8) x = keep_elements(x, k_tail - col);
      }
    };
    if (k + 1 == ksteps && k_tail % 8 != 0) {
#pragma unroll
      for (int j = 0; j < kDmaA; ++j) clear.template operator()<kAK, TM>(v[j], wave * kDmaA + j);
#pragma unroll
      for (int j = 0; j < kDmaB; ++j) clear.template operator()<kBK_, TN>(v[kDmaA + j], wave * kDmaB + j);
    }
#pragma unroll
    for (int j = 0; j < kDmaA; ++j)
      *reinterpret_cast<u32x4*>(stage + (wave * kDmaA + j) * 1024 + lane * 16) = v[j];
#pragma unroll
    for (int j = 0; j < kDmaB; ++j)
      *reinterpret_cast<u32x4*>(stage + T::kABytes + (wave * kDmaB + j) * 1024 + lane * 16) = v[kDmaA + j];
  };
  u32x4 regs[2][kRegs ? kDmaA + kDmaB : 1];
  if constexpr (kRegs) {
    load_regs(0, regs[0]);
    load_regs(1, regs[1]);
    store_regs(lds0, 0, regs[0]);
    store_regs(lds1, 1, regs[1]);
    load_regs(2, regs[0]);
    load_regs(3, regs[1]);
  }

  auto k_base = [&](uint32_t w0) { return (w0 + r16) * 128 + ((g4 ^ (r16 & 7)) << 4); };
  auto m_base = [&]<int RB>(uint32_t w0) {
    const uint32_t r4 = r16 / 4, c1 = (r16 % 4) / 2;
    return (8 * g4 + r4) * RB + (((w0 / 8 + c1) ^ mn_swz<RB>(8 * g4 + r4)) << 4) + 8 * (r16 % 2);
  };
  const uint32_t a_base_l = kAK ? k_base(wm) : m_base.template operator()<2 * TM>(wm);
  const uint32_t b_base_l = kBK_ ? k_base(wn) : m_base.template operator()<2 * TN>(wn);
  // Fragment of tile t (16 rows), substep ss of the step.
  auto frag = [&]<bool KContig, int TMN>(const uint8_t* tile, uint32_t base, uint32_t t, uint32_t ss) __attribute__((always_inline)) {
    if constexpr (KContig) {
      const uint8_t* p = tile + (base ^ ((ss % 2) * 64)) + 2048 * t + (ss / 2) * (TMN * 128);
      return __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4*>(p));
    } else {
      constexpr uint32_t RB = 2 * TMN;
      const uint8_t* p = tile + (base ^ (t << 5)) + ss * (32 * RB);
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS short4_t*)p);
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS short4_t*)(p + 4 * RB));
      return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  constexpr int kItems = kMT + kNT;
  half8_t fa[2][kSub][kMT], fb[2][kSub][kNT];
  // Fragment item r of a step (kSub * kItems of them): substep r / kItems of
  // this wave's K group; B tiles first.
  auto read_item = [&](const uint8_t* stage, int buf, int r) __attribute__((always_inline)) {
    const int u = r / kItems, x = r % kItems;
    const uint32_t ss = kg * kSub + u;
    if (x < kNT) fb[buf][u][x] = frag.template operator()<kBK_, TN>(stage + T::kABytes, b_base_l, x, ss);
    else fa[buf][u][x - kNT] = frag.template operator()<kAK, TM>(stage, a_base_l, x - kNT, ss);
  };

  float4_t acc[kMT][kNT];
#pragma unroll
  for (int i = 0; i < kMT; ++i)
#pragma unroll
    for (int j = 0; j < kNT; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // kDwords: K-contiguous rows of the last step's stage hold elements past K
  // in the chunk that K ends in; cleared once every wave's DMA has landed.
  auto clear_past_k = [&](uint8_t* stage) __attribute__((always_inline)) {
    const uint32_t chunk = k_tail / 8, valid = k_tail % 8;
    if (valid == 0) return;
    auto rows = [&](uint8_t* tile, uint32_t count) {
      for (uint32_t r = threadIdx.x; r < count; r += T::kThreads)
        clear_chunk_past(tile + chunk / 8 * (count * 128) + r * 128 + (((chunk % 8) ^ (r & 7u)) << 4), valid);
    };
    if constexpr (kAK) rows(stage, TM);
    if constexpr (kBK_) rows(stage + T::kABytes, TN);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  constexpr int kDma = T::kDma;
  constexpr int kMfma = kSub * kMT * kNT, kReads = kSub * kItems;
  // The first step's fragments, with the DMA of `Behind` stages still in flight.
  auto start = [&]<int Behind>() __attribute__((always_inline)) {
    if constexpr (kRegs) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(Behind * kDma) : "memory");
    if (E == kDwords && ksteps == 1) clear_past_k(lds0);
#pragma unroll
    for (int r = 0; r < kReads; ++r) read_item(lds0, 0, r);
  };
  // Step kt: its fragments are in register buffer buf.  After the barrier
  // every wave's DMA of stage kt + 1 (`next`) has landed and every wave's
  // reads of stage kt (`cur`) have returned, so cur takes the DMA of step
  // kt + 4 and next is read between the MFMAs.
  // kElements: the step stores the chunks of step kt + 2, loaded two steps ago,
  // into their stage (`ahead`, last read in step kt - 2) and loads those of
  // step kt + 4; the barrier publishes the stores of the step before.
  // Tail t (1, 2, 3): the t-th of the at most three steps after the last group of
  // four, which have nothing left to fetch.
  auto step = [&]<int Tail>(uint8_t* cur, uint8_t* next, uint8_t* ahead, int buf, uint32_t kt) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kRegs) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (Tail <= 1) store_regs(ahead, kt + 2, regs[buf]);
      if constexpr (Tail == 0) load_regs(kt + S, regs[buf]);
    } else {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((Tail ? S - 1 - Tail : S - 2) * kDma) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (Tail == 0) dma(cur, kt + S);
    }
    if (E == kDwords && kt + 2 == ksteps) clear_past_k(next);
    __builtin_amdgcn_sched_barrier(0);
    int r = 0;
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      const int u = m / (kMT * kNT), i = m / kNT % kMT, j = m % kNT;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[buf][u][j], fa[buf][u][i], acc[i][j], 0, 0, 0);
      // Reads spread over the first three quarters of the MFMAs.
      while (r < kReads && r * kMfma * 3 / 4 <= m * kReads) {
        read_item(next, 1 - buf, r);
        ++r;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (!kRegs && ksteps <= 2) {
    // Nothing to issue past the second stage: 256^3 replayed 3.01 -> 2.91 us.
    dma(lds0, 0);
    dma(lds1, 1);
    start.template operator()<1>();
    step.template operator()<3>(lds0, lds1, lds2, 0, 0);
    if (ksteps == 2) step.template operator()<3>(lds1, lds2, lds3, 1, 1);
  } else {
    if constexpr (!kRegs) {
      dma(lds0, 0);
      dma(lds1, 1);
      dma(lds2, 2);
      dma(lds3, 3);
    }
    start.template operator()<S - 1>();
    uint32_t kt = 0;
    for (; kt + 3 < ksteps; kt += 4) {
      step.template operator()<0>(lds0, lds1, lds2, 0, kt);
      step.template operator()<0>(lds1, lds2, lds3, 1, kt + 1);
      step.template operator()<0>(lds2, lds3, lds0, 0, kt + 2);
      step.template operator()<0>(lds3, lds0, lds1, 1, kt + 3);
    }
    if (kt < ksteps) step.template operator()<1>(lds0, lds1, lds2, 0, kt);
    if (kt + 1 < ksteps) step.template operator()<2>(lds1, lds2, lds3, 1, kt + 1);
    if (kt + 2 < ksteps) step.template operator()<3>(lds2, lds3, lds0, 0, kt + 2);
  }
  // Every DMA has landed (those past the last step too) and every wave is done
  // with the stages.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // acc[i][j][e] = C[m0 + wm + 16 i + lane % 16][n0 + wn + 16 j + 4 (lane / 16) + e]
  constexpr int kRowsT = kMT / KG;  // 16-row tiles of C that each K group finishes
  if constexpr (KG == 2) {
    // Each group hands the other half of its rows over through LDS.
    constexpr uint32_t kSlot = kRowsT * kNT * 1024;
    uint8_t* mine = (kg == 0 ? lds0 : lds1) + wmn * kSlot;
    const uint8_t* theirs = (kg == 0 ? lds1 : lds0) + wmn * kSlot;
    static_assert(T::kWavesM * T::kWavesN * kSlot <= T::kStageBytes, "exchange fits a stage");
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      if ((uint32_t)i / kRowsT == kg) continue;
#pragma unroll
      for (int j = 0; j < kNT; ++j)
        *reinterpret_cast<float4_t*>(mine + ((i % kRowsT) * kNT + j) * 1024 + lane * 16) = acc[i][j];
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      if ((uint32_t)i / kRowsT != kg) continue;
#pragma unroll
      for (int j = 0; j < kNT; ++j)
        acc[i][j] += *reinterpret_cast<const float4_t*>(theirs + ((i % kRowsT) * kNT + j) * 1024 + lane * 16);
    }
  }
  if constexpr (Split) {
    auto stored = [&](int i) { return m0 + wm + 16 * i + r16 < M; };
    if (!add_splits<T::kThreads>(split, batch * tiles + pid, acc, stored)) return;
  }
  // The wave's rows go out through its own slot of LDS as whole runs of
  // 2 * WN bytes: row r, 16-byte chunk c at chunk c ^ (r & (chunks - 1)).
  constexpr uint32_t kRB = 2 * T::WN, kRC = kRB / 16;
  constexpr uint32_t kOutSlot = 16 * kRowsT * kRB;
  static_assert(T::kWaves * kOutSlot <= T::kStageBytes, "staged output fits a stage");
  uint8_t* cst = lds2 + wave * kOutSlot;
#pragma unroll
  for (int i = 0; i < kMT; ++i) {
    if (KG > 1 && (uint32_t)i / kRowsT != kg) continue;
    const uint32_t r = 16 * (i % kRowsT) + r16;
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
      half4_t h;
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = epilogue<Epi>(acc[i][j][e]);
      const uint32_t c = 2 * j + g4 / 2;
      *reinterpret_cast<half4_t*>(cst + r * kRB + ((c ^ (r & (kRC - 1))) << 4) + (g4 % 2) * 8) = h;
    }
  }
  const uint32_t row0 = m0 + wm + (KG > 1 ? kg * 16 * kRowsT : 0), col0 = n0 + wn;
#pragma unroll
  for (uint32_t k = 0; k < (16 * kRowsT * kRC + kWave - 1) / kWave; ++k) {
    const uint32_t v = k * kWave + lane, r = v / kRC, c = v % kRC;
    if (v >= 16 * kRowsT * kRC) break;  // 32 x 32 tiles: half a wave's lanes store
    u32x4 x = *reinterpret_cast<const u32x4*>(cst + r * kRB + ((c ^ (r & (kRC - 1))) << 4));
    // Rows past M and columns past N are not stored (N % 8 == 0 except with
    // kDwords and kElements).  out may be the addend: the same lane reads each chunk and then
    // writes it.
    if (row0 + r < M && col0 + c * 8 < N) {
      const uint64_t at = (uint64_t)(row0 + r) * N + col0 + c * 8;
      const uint32_t valid = N - (col0 + c * 8);
      if constexpr (Epi == kEpiAdd) {
        const uint16_t* d = addend + batch * addend_batch_stride + (uint64_t)(row0 + r) * addend_row_stride + col0 + c * 8;
        x = add_f16x8(x, E >= kDwords ? load_elements(d, valid) : *reinterpret_cast<const u32x4*>(d));
      }
      if constexpr (E >= kDwords) store_elements(C + at, x, valid);
      else *reinterpret_cast<u32x4*>(C + at) = x;
    }
  }
}

template <class T, int Epi>
int launch_tile(hipStream_t stream, const GemmArgs& a, GemmAccess access, uint64_t plan_tiles) {
  const uint64_t tiles = (uint64_t)((a.rows + T::TM - 1) / T::TM) * ((a.columns + T::TN - 1) / T::TN);
  if (tiles > 0x7fffffffu) return IPUS_ERROR_INVALID_ARGUMENT;
  static_assert((uint64_t)kTileGridX * T::kThreads < (1ull << 32), "a grid dimension holds fewer than 2^32 work-items");
  const TileGrid grid = tile_grid(tiles);
  SplitK split;
  auto go = [&](auto kernel) {
    // A split launch has at most 128 tiles a batch (split_plan), so the third
    // dimension is free for its splits.
    hipLaunchKernelGGL(kernel, dim3(grid.x, a.batches, split.splits > 1 ? split.splits : grid.z), dim3(T::kThreads), 0, stream,
                       (uint16_t*)a.out, (const uint16_t*)a.left, (const uint16_t*)a.right, a.rows,
                       a.columns, a.inner, a.left_batch_stride, a.right_batch_stride,
                       (const uint16_t*)a.addend, a.addend_batch_stride, a.addend_row_stride, split);
  };
  const bool tl = a.transpose_left, tr = a.transpose_right;
  auto layouts = [&]<int E, bool Split = false>() {
    if (!tl && !tr) go(gemm_f16_tile_kernel<T, false, false, Epi, E, Split>);
    else if (!tl) go(gemm_f16_tile_kernel<T, false, true, Epi, E, Split>);
    else if (!tr) go(gemm_f16_tile_kernel<T, true, false, Epi, E, Split>);
    else go(gemm_f16_tile_kernel<T, true, true, Epi, E, Split>);
  };
  if constexpr (T::TM == 32) {
    if (access != GemmAccess::kElement && split_plan(a, plan_tiles, tiles * a.batches, T::BK, 0.25, &split)) {
      if (access == GemmAccess::kDword) layouts.template operator()<kDwords, true>();
      else if (a.inner % T::BK == 0) layouts.template operator()<kWhole, true>();
      else layouts.template operator()<kKTail, true>();
      return hip_status(hipGetLastError());
    }
  }
  if (access == GemmAccess::kElement) layouts.template operator()<kElements>();
  else if (access == GemmAccess::kDword) layouts.template operator()<kDwords>();
  else if (a.inner % T::BK == 0) layouts.template operator()<kWhole>();
  else layouts.template operator()<kKTail>();
  return hip_status(hipGetLastError());
}

template <class T>
int launch_epilogue(hipStream_t stream, const GemmArgs& a, GemmAccess access, uint64_t plan_tiles) {
  if (a.addend) return launch_tile<T, kEpiAdd>(stream, a, access, plan_tiles);
  if (a.gelu) return launch_tile<T, kEpiGelu>(stream, a, access, plan_tiles);
  return launch_tile<T, kEpiPlain>(stream, a, access, plan_tiles);
}

}  // namespace

int launch_gemm_f16_tile(hipStream_t stream, const GemmArgs& a, uint32_t tile, GemmAccess access,
                         uint32_t plan_rows, uint32_t plan_batches) {
  const uint64_t plan_tiles = ((uint64_t)plan_rows + tile - 1) / tile * (((uint64_t)a.columns + tile - 1) / tile) * plan_batches;
  if (tile == 128) return launch_epilogue<Tile128>(stream, a, access, plan_tiles);
  if (tile == 64) return launch_epilogue<Tile64>(stream, a, access, plan_tiles);
  return launch_epilogue<Tile32>(stream, a, access, plan_tiles);
}

}  // namespace ipus
