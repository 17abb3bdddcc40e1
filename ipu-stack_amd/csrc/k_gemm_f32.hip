// fp32 GEMM on gfx950 MFMA, fp32 accumulation and output: replaces
// gemm_f32_64_amp (device/gemm_f32_64_amp.S:125-385), whose init mode clears the
// output and accumulates in fp32 (gemm_f32_64_amp.S:40-56).
//
// Every shape runs the tile kernel (v_mfma_f32_16x16x4_f32, at the end of this
// file) except many tiles of a short sum (tile_f32), K = 0 and operands past
// its 31-bit buffer ranges.  Those run the 128 x 128 kernel
// (v_mfma_f32_32x32x2_f32): 16-byte aligned operands whose
// contiguous axes, and N, are multiples of 4 with 16-byte loads (the kEdge
// mode, off the 128 x 128 x 32 grid, zero-fills loads past M, N or K and stores
// only rows < M and 4-column chunks < N), others in its kScalar mode with
// bounds-checked element loads and stores:
//   * block tile 128 x 128 x 32, 4 waves in a 2 x 2 grid, each wave 64 x 64
//     as 2 x 2 MFMA tiles;
//   * each operand is staged in LDS in the layout it has in memory, so no
//     tile is transposed on the way: an operand whose x axis (m or n) is
//     contiguous k-major ([k][x], 16-byte chunks XOR-swizzled by (k >> 2) &
//     7), one whose k axis is contiguous x-major ([x][k], rows of 32 k,
//     chunks XOR-swizzled by (x >> 1) & 7);
//   * the k pair of MFMA substep p is (p, 16 + p) for lanes 0-31 and 32-63, a
//     permutation of the step's 32 k that both operands share, so a lane reads
//     four substeps' values of an x-major tile as one 16-byte chunk (k-major
//     tiles: one element per substep);
//   * one LDS stage (32 KiB, so three workgroups share a CU): the next K
//     step's tiles load into registers during the MFMAs and are stored
//     between two barriers (4096^3: 121 -> 126 TFLOP/s against two stages
//     and two workgroups per CU);
//   * the MFMA computes C^T tiles so each lane holds 4 consecutive columns
//     of C (one 16-byte store).
#include "../../include/ipus.h"

#include "gemm_common.h"
#include "kernels.h"
#include "tile_choice.h"
#include "tile_grid.h"

namespace ipus {
namespace {

constexpr int kBM = 128, kBN = 128, kBK = 32;
constexpr int kThreads = 256;
constexpr int kTileBytes = kBK * kBM * 4;  // 16 KiB per operand tile

// Byte offset of element (k, x) in a [32 k][128 x] fp32 tile (k-major,
// the layout of an operand whose x axis is contiguous in memory).
__device__ __forceinline__ uint32_t swz32(uint32_t k, uint32_t x) {
  return k * 512u + ((((x >> 2) ^ ((k >> 2) & 7u)) << 4) | ((x & 3u) << 2));
}
// Byte offset of 16-byte chunk c (k = 4 c .. 4 c + 3) of row x in a
// [128 x][32 k] fp32 tile (x-major, the layout of an operand whose k axis is
// contiguous in memory).
__device__ __forceinline__ uint32_t xk_off(uint32_t x, uint32_t c) {
  return x * 128u + ((c ^ ((x >> 1) & 7u)) << 4);
}

// Tile modes: kGrid (every tile whole), kEdge (chunks of 4 floats past the
// extents read as 0 and are not stored; the contiguous axes and N are
// multiples of 4, so a chunk is wholly inside or outside), kScalar (any
// shape and alignment: element loads and stores, each bounds-checked).
enum TileMode : int { kGrid = 0, kEdge = 1, kScalar = 2 };

// Loads a 128 (x) by 32 (k) operand tile.
// XContig: element (x, k) at base[(k0 + k) * ld + x0 + x]  (stored [K][X])
// else:    element (x, k) at base[(x0 + x) * ld + k0 + k]  (stored [X][K])
template <bool XContig, int Mode>
__device__ __forceinline__ void load_tile32(const float* __restrict__ base, uint64_t ld,
                                            uint32_t x0, uint32_t k0, u32x4 v[4], uint32_t X,
                                            uint32_t K) {
  const uint32_t t = threadIdx.x;
  const u32x4 zero = {0, 0, 0, 0};
  if constexpr (XContig) {
    const uint32_t k = k0 + t / 32, x = x0 + (t % 32) * 4;
    const float* p = base + (uint64_t)k * ld + x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (Mode == kScalar) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[i][e] = k + 8 * i < K && x + e < X ? __float_as_uint(p[(uint64_t)(8 * i) * ld + e]) : 0u;
      } else {
        v[i] = Mode == kGrid || (k + 8 * i < K && x < X) ? load16(p + (uint64_t)(8 * i) * ld) : zero;
      }
    }
  } else {
    const uint32_t x = x0 + (t / 8) * 4, k = k0 + (t % 8) * 4;
    const float* p = base + (uint64_t)x * ld + k;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (Mode == kScalar) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[j][e] = x + j < X && k + e < K ? __float_as_uint(p[(uint64_t)j * ld + e]) : 0u;
      } else {
        v[j] = Mode == kGrid || (x + j < X && k < K) ? load16(p + (uint64_t)j * ld) : zero;
      }
    }
  }
}

template <bool XContig>
__device__ __forceinline__ void store_tile32(uint8_t* lds, const u32x4 v[4]) {
  const uint32_t t = threadIdx.x;
  if constexpr (XContig) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x4*>(lds + swz32(t / 32 + 8 * i, (t % 32) * 4)) = v[i];
  } else {
    // v[j] = x row (t/8)*4 + j, k chunk t%8: stored as loaded.
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<u32x4*>(lds + xk_off((t / 8) * 4 + j, t % 8)) = v[j];
  }
}

__device__ __forceinline__ float read32(const uint8_t* lds, uint32_t k, uint32_t x) {
  return *reinterpret_cast<const float*>(lds + swz32(k, x));
}

template <bool TransposeLeft, bool TransposeRight, int Mode>
__global__ __launch_bounds__(kThreads, 3) void gemm_f32_128_kernel(
    float* __restrict__ out, const float* __restrict__ left, const float* __restrict__ right,
    uint32_t M, uint32_t N, uint32_t K, uint64_t left_batch_stride, uint64_t right_batch_stride) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[2 * kTileBytes];

  const uint32_t nbm = (M + kBM - 1) / kBM, nbn = (N + kBN - 1) / kBN;
  const uint32_t tiles = nbm * nbn;
  uint32_t pid = blockIdx.x;
  if (tiles % 8 == 0) pid = (pid % 8) * (tiles / 8) + pid / 8;
  constexpr uint32_t kGroup = 8;
  const uint32_t group = pid / (kGroup * nbn);
  const uint32_t first_m = group * kGroup;
  const uint32_t group_rows = (nbm - first_m) < kGroup ? (nbm - first_m) : kGroup;
  const uint32_t in_group = pid % (kGroup * nbn);
  const uint32_t bm = first_m + in_group % group_rows;
  const uint32_t bn = in_group / group_rows;

  const uint64_t batch = blockIdx.y;
  const float* A = left + batch * left_batch_stride;
  const float* B = right + batch * right_batch_stride;
  float* C = out + batch * (uint64_t)M * N;
  const uint64_t lda = TransposeLeft ? M : K;
  const uint64_t ldb = TransposeRight ? K : N;
  constexpr bool kAX = TransposeLeft;    // A stored [K][M]: m contiguous
  constexpr bool kBX = !TransposeRight;  // B stored [K][N]: n contiguous

  const uint32_t m0 = bm * kBM, n0 = bn * kBN;
  const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const uint32_t wm = (wave / 2) * 64, wn = (wave % 2) * 64;

  float16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  u32x4 ra[4], rb[4];
  load_tile32<kAX, Mode>(A, lda, m0, 0, ra, M, K);
  load_tile32<kBX, Mode>(B, ldb, n0, 0, rb, N, K);
  store_tile32<kAX>(smem, ra);
  store_tile32<kBX>(smem + kTileBytes, rb);
  __syncthreads();

  const uint32_t ksteps = (K + kBK - 1) / kBK;
  for (uint32_t kt = 0; kt < ksteps; ++kt) {
    const bool more = kt + 1 < ksteps;
    if (more) {
      load_tile32<kAX, Mode>(A, lda, m0, (kt + 1) * kBK, ra, M, K);
      load_tile32<kBX, Mode>(B, ldb, n0, (kt + 1) * kBK, rb, N, K);
    }
    const uint8_t* la = smem;
    const uint8_t* lb = smem + kTileBytes;
    // The k pair of substep p is (p, 16 + p) for lanes 0-31 and 32-63 (a
    // permutation of the step's 32 k that A and B share): in an x-major
    // tile a lane's values for 4 consecutive substeps are one 16-byte chunk
    // of its row; a k-major tile is read one element per substep.
    const uint32_t g = lane / 32;
    auto frag4 = [&]<bool XContig>(const uint8_t* l, uint32_t x, uint32_t q) __attribute__((always_inline)) {
      if constexpr (XContig) {
        u32x4 v;
#pragma unroll
        for (int w = 0; w < 4; ++w) v[w] = __float_as_uint(read32(l, 16 * g + 4 * q + w, x));
        return v;
      } else {
        return *reinterpret_cast<const u32x4*>(l + xk_off(x, 4 * g + q));
      }
    };
#pragma unroll
    for (uint32_t q = 0; q < kBK / 8; ++q) {
      u32x4 fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = frag4.template operator()<kAX>(la, wm + 32 * i + lane % 32, q);
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = frag4.template operator()<kBX>(lb, wn + 32 * j + lane % 32, q);
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(fb[j][w]),
                                                            __uint_as_float(fa[i][w]), acc[i][j], 0, 0, 0);
    }
    if (more) {
      __syncthreads();  // every wave is done reading this tile
      store_tile32<kAX>(smem, ra);
      store_tile32<kBX>(smem + kTileBytes, rb);
    }
    __syncthreads();
  }

  const uint32_t row = m0 + wm + lane % 32;
  const uint32_t col = n0 + wn + 4 * (lane / 32);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (Mode != kGrid && row + 32 * i >= M) continue;
    float* crow = C + (uint64_t)(row + 32 * i) * N + col;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t c = col + 32 * j + 8 * g;
        if (Mode != kGrid && c >= N) continue;
        if constexpr (Mode == kScalar) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < N) crow[32 * j + 8 * g + e] = acc[i][j][4 * g + e];
        } else {
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e];
          *reinterpret_cast<float4_t*>(crow + 32 * j + 8 * g) = v;
        }
      }
  }
}

template <bool TL, bool TR>
int launch_fast(hipStream_t stream, const GemmArgs& a, bool chunked) {
  const uint32_t tiles = ((a.rows + kBM - 1) / kBM) * ((a.columns + kBN - 1) / kBN);
  const bool grid = a.rows % kBM == 0 && a.columns % kBN == 0 && a.inner % kBK == 0;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(tiles, a.batches), dim3(kThreads), 0, stream, (float*)a.out,
                       (const float*)a.left, (const float*)a.right, a.rows, a.columns, a.inner,
                       a.left_batch_stride, a.right_batch_stride);
  };
  if (!chunked) go(gemm_f32_128_kernel<TL, TR, kScalar>);
  else if (grid) go(gemm_f32_128_kernel<TL, TR, kGrid>);
  else go(gemm_f32_128_kernel<TL, TR, kEdge>);
  return hip_status(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Tile kernel: 64 x 64 or 32 x 32 tiles of C.
// Bound by the matrix pipes: a 64 x 64 x 32 step is 16 KiB of operands for
// 1,024 cycles of MFMA, so what counts is that no wave waits.  Operand tiles go
// global -> LDS by DMA, four stages deep, and the fragments of step k + 1 are
// read between the MFMAs of step k, as in k_gemm_f16_tile.hip; 64 x 64 tiles
// run two K groups of four waves (group h takes substeps 4 h .. 4 h + 3 of
// the eight k that each lane holds) and two workgroups per CU, four waves per
// SIMD in all.  Small tiles cost nothing here and fill the chip: 4096^3 1,066
// -> 918 us (129 -> 150 TFLOP/s, 95% of 157.3; 128 x 128 tiles 945), 1024^3 75
// -> 19.2 (64 tiles of 128 x 128 before), 64 x 1024 x 1024 75 -> 7.0 (32 x 32),
// 256^3 21 -> 3.6.  Errors against float64 are those of the kernel before (one
// fp32 sum over K per element: 5.7e-7 normwise at K = 1024) or, with two K
// groups, lower (4.1e-7).
// Few 32 x 32 tiles with a long K split K over workgroups (split_plan,
// gemm_common.h; shorter sums: 8 x 4096 x 4096 1.2e-6 -> 8.1e-7).
// ---------------------------------------------------------------------------
// Tile of C (TM x TN), part of one wave (WM x WN), K groups, k per step.
template <int BM, int BN, int WM_, int WN_, int KG_, int BK_>
struct TileShapeF32 {
  static constexpr int TM = BM, TN = BN, WM = WM_, WN = WN_, KG = KG_, BK = BK_;
  static constexpr int S = 4;  // LDS stages
  static constexpr int kWavesM = TM / WM, kWavesN = TN / WN;
  static constexpr int kWaves = kWavesM * kWavesN * KG;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kABytes = TM * BK * 4, kBBytes = TN * BK * 4;
  static constexpr int kStageBytes = kABytes + kBBytes;
  static constexpr int kDmaA = kABytes / 1024 / kWaves, kDmaB = kBBytes / 1024 / kWaves;
  static constexpr int kDma = kDmaA + kDmaB;
  static constexpr int kMT = WM / 16, kNT = WN / 16;
  static constexpr int kUnits = BK / 32;  // 32-k units per step
  static constexpr int kP = 8 / KG;       // MFMA substeps of a unit that a K group takes
  static_assert(kABytes % (1024 * kWaves) == 0 && kBBytes % (1024 * kWaves) == 0, "whole DMA instructions per wave");
  static_assert(KG == 1 || KG == 2, "the exchange of partial sums is between two groups");
};

typedef TileShapeF32<64, 64, 32, 32, 2, 32> TileF32x64;
typedef TileShapeF32<32, 32, 16, 16, 1, 64> TileF32x32;

// LDS tiles.  K-contiguous operand: units of 32 k, each [rows][32 k] (128-byte
// rows), 16-byte chunk XORed by row & 7.  MN-contiguous: [k][mn], the chunk
// XORed by mn_swz32(k): a fragment read takes 16 consecutive columns (64
// bytes) of the four rows 8 g + p (g = 0..3), which the XOR by row bits 3 and 4
// puts on different quarters of the banks (128-byte rows: on two halves).
template <int RowBytes>
__device__ __forceinline__ uint32_t mn_swz32(uint32_t k) {
  return RowBytes >= 256 ? ((k >> 3) & 3u) << 2 : ((k >> 3) & 1u) << 2;
}

template <class T, bool TransposeLeft, bool TransposeRight, int E, bool Split>
__global__ __launch_bounds__(T::kThreads, 1) void gemm_f32_tile_kernel(
    float* __restrict__ out, const float* __restrict__ left, const float* __restrict__ right,
    uint32_t M, uint32_t N, uint32_t K, uint64_t left_batch_stride, uint64_t right_batch_stride,
    SplitK split) {
  static_assert(!Split || T::KG == 1, "splits: one K group");
  constexpr int TM = T::TM, TN = T::TN, BK = T::BK, S = T::S, KG = T::KG;
  constexpr int kMT = T::kMT, kNT = T::kNT, kUnits = T::kUnits, kP = T::kP;
  constexpr int kDmaA = T::kDmaA, kDmaB = T::kDmaB;
  constexpr bool KTail = E != kWhole;
  // Distinct LDS objects: a DMA into one stage never aliases the reads of
  // another.
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
  // XCD-contiguous tiles, grouped 8 along M.
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
  const float* A = left + batch * left_batch_stride;
  const float* B = right + batch * right_batch_stride;
  float* C = out + batch * (uint64_t)M * N;
  // This workgroup's K range (the whole of K unless Split).
  const uint32_t k_begin = Split ? blockIdx.z * split.chunk : 0;
  const uint32_t k_len = Split ? (K - k_begin < split.chunk ? K - k_begin : split.chunk) : K;
  const float* a_base = kAK ? A + (uint64_t)m0 * K + k_begin : A + m0 + (uint64_t)k_begin * M;
  const float* b_base = kBK_ ? B + (uint64_t)n0 * K + k_begin : B + n0 + (uint64_t)k_begin * N;
  const uint64_t a_bytes = (uint64_t)M * K * 4 - (uint64_t)(a_base - A) * 4;
  const uint64_t b_bytes = (uint64_t)N * K * 4 - (uint64_t)(b_base - B) * 4;
  const int a_range = (int)(a_bytes > 0x7fffffffull ? 0x7fffffff : a_bytes);
  const int b_range = (int)(b_bytes > 0x7fffffffull ? 0x7fffffff : b_bytes);

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t kg = wave % KG, wmn = wave / KG;
  const uint32_t wm = (wmn / T::kWavesN) * T::WM, wn = (wmn % T::kWavesN) * T::WN;
  const uint32_t r16 = lane % 16, g4 = lane / 16;

  // MFMA substep p of a unit contracts k = 8 (l / 16) + p of both operands (a
  // permutation of the unit's 32 k), so a lane's eight k are contiguous.
  // Chunk (row or k row, logical k or mn offset in elements) that the lane
  // fetches for DMA instruction `inst` of a tile.
  auto chunk_of = [&]<bool KContig, int TMN>(uint32_t inst, uint32_t* row, uint32_t* col) __attribute__((always_inline)) {
    if constexpr (KContig) {
      const uint32_t sub = inst / (TMN / 8), r = (inst % (TMN / 8)) * 8 + lane / 8;
      *row = r;
      *col = sub * 32 + ((lane % 8) ^ (r & 7u)) * 4;
    } else {
      const uint32_t k = inst * (256 / TMN) + lane / (TMN / 4);
      *row = k;
      *col = ((lane % (TMN / 4)) ^ mn_swz32<4 * TMN>(k)) * 4;
    }
  };
  uint32_t a_voff[kDmaA], b_voff[kDmaB];
  auto offsets = [&]<bool KContig, int TMN, int N_>(uint32_t ld, uint32_t mn_limit, uint32_t (&voff)[N_]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < N_; ++j) {
      uint32_t row, col;
      chunk_of.template operator()<KContig, TMN>(wave * N_ + j, &row, &col);
      voff[j] = KContig || col < mn_limit ? (row * ld + col) * 4 : kPadOffset;
    }
  };
  offsets.template operator()<kAK, TM>(kAK ? K : M, M - m0, a_voff);
  offsets.template operator()<kBK_, TN>(kBK_ ? K : N, N - n0, b_voff);
  const uint32_t a_kstep = kAK ? BK * 4 : BK * M * 4;
  const uint32_t b_kstep = kBK_ ? BK * 4 : BK * N * 4;

  const uint32_t ksteps = (k_len + BK - 1) / BK;
  const uint32_t k_tail = k_len % BK;
  // The DMA of step k into a stage.  Past the last step the descriptors are
  // empty: no memory is read, but the instructions are issued, so the wait
  // counts stay exact.  KTail: chunks and rows past K on the last step get an
  // offset past the range and read 0.
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
  dma(lds0, 0);
  dma(lds1, 1);
  dma(lds2, 2);
  dma(lds3, 3);

  const uint32_t h0 = KG == 2 ? kg : 0;
  auto k_base = [&](uint32_t w0) { return (w0 + r16) * 128 + (((2 * g4 + h0) ^ (r16 & 7)) << 4); };
  auto m_base = [&]<int RB>(uint32_t w0) {
    return (8 * g4 + 4 * h0) * RB + (((w0 / 4 + r16 / 4) ^ mn_swz32<RB>(8 * g4)) << 4) + (r16 % 4) * 4;
  };
  const uint32_t a_base_l = kAK ? k_base(wm) : m_base.template operator()<4 * TM>(wm);
  const uint32_t b_base_l = kBK_ ? k_base(wn) : m_base.template operator()<4 * TN>(wn);
  // Four substeps (half h of the lane's 8 k of unit u) of tile t.
  auto frag = [&]<bool KContig, int TMN>(const uint8_t* tile, uint32_t base, uint32_t t, uint32_t u, uint32_t h) __attribute__((always_inline)) {
    if constexpr (KContig) {
      return *reinterpret_cast<const float4_t*>(tile + (base ^ (h << 4)) + 2048 * t + u * (TMN * 128));
    } else {
      constexpr uint32_t RB = 4 * TMN;
      const uint8_t* p = tile + (base ^ (t << 6)) + (u * 32 + 4 * h) * RB;
      float4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const float*>(p + e * RB);
      return v;
    }
  };
  constexpr int kH = kP / 4;  // halves a wave reads
  constexpr int kItems = (kMT + kNT) * kH * kUnits;
  float4_t fa[2][kUnits][kH][kMT], fb[2][kUnits][kH][kNT];
  auto read_item = [&](const uint8_t* stage, int buf, int r) __attribute__((always_inline)) {
    const int u = r / ((kMT + kNT) * kH), q = r % ((kMT + kNT) * kH), h = q / (kMT + kNT), x = q % (kMT + kNT);
    if (x < kNT) fb[buf][u][h][x] = frag.template operator()<kBK_, TN>(stage + T::kABytes, b_base_l, x, u, h);
    else fa[buf][u][h][x - kNT] = frag.template operator()<kAK, TM>(stage, a_base_l, x - kNT, u, h);
  };

  float4_t acc[kMT][kNT];
#pragma unroll
  for (int i = 0; i < kMT; ++i)
#pragma unroll
    for (int j = 0; j < kNT; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // kDwords (gemm_common.h): the chunk that K ends in, of K-contiguous rows of
  // the last step's stage, is cleared past K once every DMA has landed.
  auto clear_past_k = [&](uint8_t* stage) __attribute__((always_inline)) {
    const uint32_t chunk = k_tail / 4, valid = k_tail % 4;
    if (valid == 0) return;
    auto rows = [&](uint8_t* tile, uint32_t count) {
      for (uint32_t r = threadIdx.x; r < count; r += T::kThreads)
        clear_chunk_past(tile + chunk / 8 * (count * 128) + r * 128 + (((chunk % 8) ^ (r & 7u)) << 4), 2 * valid);
    };
    if constexpr (kAK) rows(stage, TM);
    if constexpr (kBK_) rows(stage + T::kABytes, TN);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  constexpr int kDma = T::kDma;
  constexpr int kMfma = kUnits * kP * kMT * kNT;
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 1) * kDma) : "memory");
  if (E == kDwords && ksteps == 1) clear_past_k(lds0);
#pragma unroll
  for (int r = 0; r < kItems; ++r) read_item(lds0, 0, r);
  // After the barrier every wave's DMA of stage kt + 1 has landed and every
  // wave's reads of stage kt have returned.
  // Tail t: as in k_gemm_f16_tile.hip, the steps after the last group of four.
  auto step = [&]<int Tail>(uint8_t* cur, uint8_t* next, int buf, uint32_t kt) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((Tail ? S - 1 - Tail : S - 2) * kDma) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (Tail == 0) dma(cur, kt + S);
    if (E == kDwords && kt + 2 == ksteps) clear_past_k(next);
    __builtin_amdgcn_sched_barrier(0);
    int r = 0;
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      const int u = m / (kP * kMT * kNT), p = m / (kMT * kNT) % kP, i = m / kNT % kMT, j = m % kNT;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[buf][u][p / 4][j][p % 4], fa[buf][u][p / 4][i][p % 4], acc[i][j], 0, 0, 0);
      while (r < kItems && r * kMfma * 3 / 4 <= m * kItems) {
        read_item(next, 1 - buf, r);
        ++r;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  uint32_t kt = 0;
  for (; kt + 3 < ksteps; kt += 4) {
    step.template operator()<0>(lds0, lds1, 0, kt);
    step.template operator()<0>(lds1, lds2, 1, kt + 1);
    step.template operator()<0>(lds2, lds3, 0, kt + 2);
    step.template operator()<0>(lds3, lds0, 1, kt + 3);
  }
  if (kt < ksteps) step.template operator()<1>(lds0, lds1, 0, kt);
  if (kt + 1 < ksteps) step.template operator()<2>(lds1, lds2, 1, kt + 1);
  if (kt + 2 < ksteps) step.template operator()<3>(lds2, lds3, 0, kt + 2);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // acc[i][j][e] = C[m0 + wm + 16 i + lane % 16][n0 + wn + 16 j + 4 (lane / 16) + e]
  constexpr int kRowsT = kMT / KG;
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
#pragma unroll
  for (int i = 0; i < kMT; ++i) {
    if (KG > 1 && (uint32_t)i / kRowsT != kg) continue;
    const uint32_t row = m0 + wm + 16 * i + r16;
    if (row >= M) continue;
    float* crow = C + (uint64_t)row * N;
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
      const uint32_t col = n0 + wn + 16 * j + 4 * g4;
      if (E != kDwords) {
        if (col < N) *reinterpret_cast<float4_t*>(crow + col) = acc[i][j];
      } else {
        // Rows start dword-aligned and N is any count.
        typedef float4_t __attribute__((aligned(4))) float4_dwords;
        if (col + 4 <= N) {
          *reinterpret_cast<float4_dwords*>(crow + col) = acc[i][j];
        } else {
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e)
            if (col + e < N) crow[col + e] = acc[i][j][e];
        }
      }
    }
  }
}

template <class T>
int launch_tile32(hipStream_t stream, const GemmArgs& a, bool chunked) {
  const uint64_t tiles = (uint64_t)((a.rows + T::TM - 1) / T::TM) * ((a.columns + T::TN - 1) / T::TN);
  if (tiles > 0x7fffffffu) return IPUS_ERROR_INVALID_ARGUMENT;
  static_assert((uint64_t)kTileGridX * T::kThreads < (1ull << 32), "a grid dimension holds fewer than 2^32 work-items");
  const TileGrid grid = tile_grid(tiles);
  SplitK split;
  auto go = [&](auto kernel) {
    // A split launch has at most 128 tiles a batch (split_plan), so the third
    // dimension is free for its splits.
    hipLaunchKernelGGL(kernel, dim3(grid.x, a.batches, split.splits > 1 ? split.splits : grid.z), dim3(T::kThreads), 0, stream,
                       (float*)a.out, (const float*)a.left, (const float*)a.right, a.rows,
                       a.columns, a.inner, a.left_batch_stride, a.right_batch_stride, split);
  };
  const bool tl = a.transpose_left, tr = a.transpose_right;
  auto layouts = [&]<int E, bool Split = false>() {
    if (!tl && !tr) go(gemm_f32_tile_kernel<T, false, false, E, Split>);
    else if (!tl) go(gemm_f32_tile_kernel<T, false, true, E, Split>);
    else if (!tr) go(gemm_f32_tile_kernel<T, true, false, E, Split>);
    else go(gemm_f32_tile_kernel<T, true, true, E, Split>);
  };
  if constexpr (T::TM == 32) {
    if (split_plan(a, tiles * a.batches, tiles * a.batches, T::BK, 0.30, &split)) {
      if (!chunked) layouts.template operator()<kDwords, true>();
      else if (a.inner % T::BK == 0) layouts.template operator()<kWhole, true>();
      else layouts.template operator()<kKTail, true>();
      return hip_status(hipGetLastError());
    }
  }
  if (!chunked) layouts.template operator()<kDwords>();
  else if (a.inner % T::BK == 0) layouts.template operator()<kWhole>();
  else layouts.template operator()<kKTail>();
  return hip_status(hipGetLastError());
}

}  // namespace

int launch_gemm_f32(hipStream_t stream, const GemmArgs& a) {
  if (a.batches == 0 || a.rows == 0 || a.columns == 0) return 0;
  if (a.batches > 65535) return IPUS_ERROR_INVALID_ARGUMENT;
  const bool aligned = ((uintptr_t)a.left % 16 == 0) && ((uintptr_t)a.right % 16 == 0) &&
                       ((uintptr_t)a.out % 16 == 0) && a.left_batch_stride % 4 == 0 &&
                       a.right_batch_stride % 4 == 0;
  // 4-float chunks run along the contiguous axis of each operand and of C:
  // N always, K for row-major A or transposed B, M for transposed A.
  const bool chunked = a.columns % 4 == 0 && (a.transpose_left ? a.rows % 4 == 0 : a.inner % 4 == 0) &&
                       (!a.transpose_right || a.inner % 4 == 0);
  // Other shapes and alignments, and K = 0 (every load masked, zeros
  // stored): the same kernel with element loads and stores.
  const bool vec = aligned && chunked && a.inner > 0;
  // The tile kernel addresses an operand tile through a buffer descriptor
  // with 31-bit offsets.  Any pitch of fp32 rows is dword-aligned, which its
  // kDwords form takes: 4096 x 4096 x 4097 1,490 -> 1,035 us, 1000 x 1001 x 1003 106
  // -> 22, 100 x 1001 x 1000 100 -> 8.4, against the 128 x 128 kernel's element
  // loads.
  const uint64_t a_span = (a.transpose_left ? (uint64_t)a.rows : 64ull) * a.inner * 4;
  const uint64_t b_span = (a.transpose_right ? 64ull : (uint64_t)a.columns) * a.inner * 4;
  const bool floats = (uintptr_t)a.left % 4 == 0 && (uintptr_t)a.right % 4 == 0 && (uintptr_t)a.out % 4 == 0;
  if (floats && a.inner > 0 && a_span < (1ull << 31) && b_span < (1ull << 31)) {
    const TileF32 tile = tile_f32(a.rows, a.columns, a.inner, a.batches, vec);
    if (tile == TileF32::k64) return launch_tile32<TileF32x64>(stream, a, vec);
    if (tile == TileF32::k32) return launch_tile32<TileF32x32>(stream, a, vec);
  }
  if (!a.transpose_left && !a.transpose_right) return launch_fast<false, false>(stream, a, vec);
  if (!a.transpose_left && a.transpose_right) return launch_fast<false, true>(stream, a, vec);
  if (a.transpose_left && !a.transpose_right) return launch_fast<true, false>(stream, a, vec);
  return launch_fast<true, true>(stream, a, vec);
}

}  // namespace ipus
