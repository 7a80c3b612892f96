// dc_gemm.hip — dense row-major GEMM C[m×n] = A[m×k]·B[k×n] on the gfx950 matrix cores.
//
// fp32: three bf16 pieces per value on v_mfma_f32_32x32x16_bf16, or v_mfma_f32_32x32x2_f32 (fp32
// accumulate in both).
// bf16: v_mfma_f32_32x32x16_bf16 (bf16 inputs, fp32 accumulate).
//
// Kernels, by the shapes that take them:
//   - gemm_f32_split_kernel<TM, TN, ...>: fp32, by eight bf16 products per fp32 product; 256×128,
//     128×128 or 64×64 macro tiles (the rule and its measurements: dc_gemm_route.hpp).
//   - gemm_f32_dma_kernel: fp32 full 64-tiles with a short k or few of them, on the fp32
//     instructions: direct-to-LDS loads, double-buffered LDS, 4 waves of 32×32.
//   - gemm_f32_kernel: the fp32 shapes left (fewer than 64 columns, at most 16 rows of B),
//     bounds-checked 64×64 tiles on the fp32 instructions.
//   - gemm_bf16_kernel<TM, TN, ...>: bf16, every shape. 256×256, 128×128 or 64×64 macro tiles by the
//     number of tiles; direct-to-LDS loads of row-major A and B where rows are 16-byte aligned,
//     else loads through registers; B fragments through transposing LDS reads.
//
// Operand layout. For a 32×32 MFMA lane l supplies row (A) / column (B) l % 32 and the k-group
// h = l / 32; the instruction pairs A and B values by (h, element index), so any assignment of
// actual k indices to (h, element) is valid as long as A and B agree. bf16: lane group h takes
// the 8 consecutive k's [8h, 8h+8) of each 16-wide k step; fp32 (one k per lane per MFMA): the
// kernels choose k orders that make each lane's LDS reads contiguous.
//
// Tile order: consecutive workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2). Block b is mapped to tile (b % 8) * (T / 8) + b / 8, so each XCD works on a contiguous
// range of tiles, and within it tiles are walked in groups of 8 tile-rows, column by column, so
// the blocks resident on one XCD share A row-panels and B column-panels in that XCD's L2.
#include <algorithm>

#include <cstddef>
#include <type_traits>
#include <utility>

#include "dc_device.hpp"
#include "dc_gemm_route.hpp"
#include "dc_internal.hpp"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kGroupM = 8;

struct TileCoord {
  int tm, tn;
};

__device__ inline TileCoord map_tile(int tiles_m, int tiles_n) {
  const int total = tiles_m * tiles_n;
  // (dc::gemm_grid's rows; workgroups past the last tile form that one too: an early exit here costs
  // every launch 0.1-0.2 us)
  const int b = min((int)(blockIdx.x + (blockIdx.y << dc::kGemmGridRowBits)), total - 1);
  const int t = (total % 8 == 0) ? (b % 8) * (total / 8) + b / 8 : b;
  const int group = kGroupM * tiles_n;
  const int g = t / group;
  const int first_m = g * kGroupM;
  const int gm = min(tiles_m - first_m, kGroupM);
  const int in_g = t - g * group;
  return TileCoord{first_m + in_g % gm, in_g / gm};
}

// ---------------------------------------------------------------------------------------------
// fp32, full 64×64 tiles (m, n multiples of 64, k of 32): direct-to-LDS loads, no staging registers and
// no transposing LDS stores. For a short k or few tiles (1024^3: 18.9 us; see dc_gemm_route.hpp).
//   A tile [64 rows][32 k] (128 B rows, unpadded): the 16-byte k-quad q of row R sits in slot
//   q ^ ((R >> 1) & 7), so a fragment read (16 lanes = rows R0..R0+15 at one quad) touches 16
//   distinct 16-byte bank groups.
//   B tile [32 k][64 n] in its natural row-major layout: the n-quad Q of k-row k sits at quad
//   Q ^ (8·((k >> 3) & 1)). Lane (r, h) of MFMA step kk reads B[ks + 8h + kk][n = r] with a 4-byte
//   LDS load: the h = 0 and h = 1 halves read rows 8 apart and land in opposite 128-byte halves of
//   the bank window.
// A wave's direct-to-LDS load writes 1 KiB (lane L -> bytes 16·L): the swizzles are applied on
// the global side (each lane fetches the quad that belongs in its slot).
// Pipeline as in the bf16 kernel: step 0 (k 0..15) runs its MFMAs with step 1's fragment reads
// between them; then the tile's one barrier (which also waits for tile kt+1's loads, issued a tile
// earlier); the loads of tile kt+2 go out into the buffer tile kt finished with, and step 1's
// MFMAs run with tile kt+1's step-0 fragment reads between them.
// ---------------------------------------------------------------------------------------------
constexpr int kT32 = 64;   // macro tile of the kernels on the fp32 instructions: 2×2 waves of 32×32
constexpr int kBK32 = 32;  // their k slice

// One LDS buffer per (operand, stage) as a separate __shared__ object, so the compiler can tell that
// loads into one stage's buffers do not alias reads of the other's (and need no wait before them).
struct F32DmaSmem {
  float* a[2];
  float* b[2];
};

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Waits until this wave's direct-to-LDS loads have landed (vmcnt(0); expcnt and lgkmcnt left
// alone), then the workgroup barrier: after it every wave's loads issued before are visible.
__device__ inline void dma_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // gfx9 encoding: vmcnt = 0, expcnt = 7, lgkmcnt = 15
  __syncthreads();
}

template <int BUF>
__device__ inline void f32_tile_to_lds(const F32DmaSmem& sm, __amdgpu_buffer_rsrc_t ra, const float* __restrict__ B, int N,
                                       int K, int n0, int k0, int wave, uint32_t avoff, const uint32_t (&bvoff)[2]) {
  // A: 8 blocks of 8 rows; wave w issues blocks w and w + 4
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row0 = 8 * (4 * i + wave);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(sm.a[BUF] + row0 * kBK32), 16, avoff,
                                             (row0 * K + k0) * (int)sizeof(float), 0, 0);
  }
  // B: 8 blocks of 4 k-rows (this k slice only, as its own buffer range)
  const auto rb = dc::range_rsrc(B + (size_t)k0 * N + n0, ((kBK32 - 1) * N + kT32) * (int)sizeof(float));
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int krow0 = 4 * (4 * i + wave);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(sm.b[BUF] + krow0 * kT32), 16, bvoff[i],
                                             krow0 * N * (int)sizeof(float), 0, 0);
  }
}

__global__ __launch_bounds__(kThreads, 2) void gemm_f32_dma_kernel(const float* __restrict__ A,
                                                                   const float* __restrict__ B, float* __restrict__ C,
                                                                   int N, int K, int tiles_m, int tiles_n) {
  constexpr int kQuads = kT32 / 4;  // n-quads per B row
  __shared__ __align__(16) float lds_a0[kT32 * kBK32], lds_a1[kT32 * kBK32], lds_b0[kBK32 * kT32], lds_b1[kBK32 * kT32];
  const F32DmaSmem sm{{lds_a0, lds_a1}, {lds_b0, lds_b1}};
  const TileCoord tc = map_tile(tiles_m, tiles_n);
  const int m0 = tc.tm * kT32, n0 = tc.tn * kT32;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r = lane & 31, h = lane >> 5;

  // load side: A panel as a buffer range (64 rows of K floats < 2 GiB, checked by the host)
  const auto ra = dc::range_rsrc(A + (size_t)m0 * K, kT32 * K * (int)sizeof(float));
  // A block 4i + w holds rows 8(4i + w) + L/8: (row >> 1) & 7 = (4·(w & 1) + L/16) & 7
  const uint32_t avoff =
      (uint32_t)(((lane >> 3) * K + 4 * ((lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7))) * (int)sizeof(float));
  uint32_t bvoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int kr = lane / kQuads;            // k-row within the block
    const int k = 4 * (4 * i + wave) + kr;   // k-row within the slice
    const int q = (lane % kQuads) ^ (8 * ((k >> 3) & 1));
    bvoff[i] = (uint32_t)((kr * N + 4 * q) * (int)sizeof(float));
  }

  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;

  const int kt_count = K / kBK32;
  f32_tile_to_lds<0>(sm, ra, B, N, K, n0, 0, wave, avoff, bvoff);
  dma_barrier();
  if (kt_count > 1) f32_tile_to_lds<1>(sm, ra, B, N, K, n0, kBK32, wave, avoff, bvoff);

  // Fragments of one 16-wide k step: two A quads, 8 B scalars.
  const int arow = wm * 32 + r, aswz = (r >> 1) & 7, n = wn * 32 + r;
  auto read_frags = [&](auto BUF, int ks, dc::f32x4 (&a)[2], float (&b)[8]) __attribute__((always_inline)) {
    constexpr int kB = decltype(BUF)::value;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      a[j] = *reinterpret_cast<const dc::f32x4*>(&(kB ? lds_a1 : lds_a0)[arow * kBK32 + 4 * ((ks / 4 + 2 * h + j) ^ aswz)]);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) b[kk] = (kB ? lds_b1 : lds_b0)[(ks + 8 * h + kk) * kT32 + 4 * ((n >> 2) ^ (8 * h)) + (n & 3)];
  };
  auto mfmas = [&](const dc::f32x4 (&a)[2], const float (&b)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[kk >> 2][kk & 3], b[kk], acc, 0, 0, 0);
  };
  auto interleave_reads = []() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 10; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // 1 LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
    }
  };
  dc::f32x4 fa0[2], fa1[2];
  float fb0[8], fb1[8];
  read_frags(std::integral_constant<int, 0>{}, 0, fa0, fb0);
  // Tile KT in LDS buffer BUF = KT % 2 (unrolled by two so buffer offsets are constants; a macro
  // keeps the fragment arrays plain registers). After the last tile the barrier and the reads of
  // the other buffer are harmless and unused.
#define DC_F32_TILE(BUF, KT)                                                                      \
  {                                                                                               \
    __builtin_amdgcn_sched_barrier(0);                                                            \
    read_frags(std::integral_constant<int, BUF>{}, 16, fa1, fb1);                                 \
    mfmas(fa0, fb0);                                                                              \
    interleave_reads();                                                                           \
    __builtin_amdgcn_sched_barrier(0);                                                            \
    dma_barrier(); /* tile KT+1 is in LDS; every wave is done reading buffer BUF */               \
    if ((KT) + 2 < kt_count) f32_tile_to_lds<BUF>(sm, ra, B, N, K, n0, ((KT) + 2) * kBK32, wave, avoff, bvoff); \
    __builtin_amdgcn_sched_barrier(0);                                                            \
    read_frags(std::integral_constant<int, 1 - (BUF)>{}, 0, fa0, fb0);                            \
    mfmas(fa1, fb1);                                                                              \
    interleave_reads();                                                                           \
    __builtin_amdgcn_sched_barrier(0);                                                            \
  }
  for (int kt = 0; kt < kt_count; kt += 2) {
    DC_F32_TILE(0, kt);
    if (kt + 1 < kt_count) DC_F32_TILE(1, kt + 1);
  }
#undef DC_F32_TILE

  // acc[v] holds C[row][col], row = 8*(v/4) + 4*h + v%4, col = r (within the wave's 32×32 tile).
  const int col = n0 + wn * 32 + r;
#pragma unroll
  for (int v = 0; v < 16; ++v) C[(size_t)(m0 + wm * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * N + col] = acc[v];
}

// ---------------------------------------------------------------------------------------------
// fp32, bounds-checked 64×64 tiles, 2×2 waves of 32×32. The next tile's global loads go to registers
// before the current tile's MFMAs and are stored to the other LDS buffer afterwards, with B
// transposed on the way in (b[n][k], row pitch 36 floats), so a lane's operands for 8 MFMAs are two
// contiguous, bank-conflict-free 16-byte LDS reads.
// ---------------------------------------------------------------------------------------------
struct F32Smem {
  static constexpr int kPitch = kBK32 + 4;  // floats per LDS row
  float a[2][kT32][kPitch];
  float b[2][kT32][kPitch];
};

// Global -> register prefetch for one slice of 32 k. A (64 rows × 32 k) as float4 slots, slot s -> row
// s / 8, kq = s % 8. B (32 × 64) as float4 slots, slot s -> nq = s / 32, k = s % 32 (a wave covers 32
// k-rows × 2 column quads, which spreads the transposed LDS writes over the banks).
struct F32Loader {
  static constexpr int kSlots = kT32 * kBK32 / 4 / kThreads;
  dc::f32x4 ra[kSlots];
  dc::f32x4 rb[kSlots];

  // p[0..4), those elements that are left; zeros where none is (valid false).
  static __device__ inline dc::f32x4 quad(const float* p, int left, bool valid) {
    dc::f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (valid) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < left) v[e] = p[e];
    }
    return v;
  }

  __device__ inline void load(const float* __restrict__ A, const float* __restrict__ B, int M, int N, int K,
                              int m0, int n0, int k0, int tid) {
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int s = tid + i * kThreads;
      const int gm = m0 + s / (kBK32 / 4), gk = k0 + 4 * (s % (kBK32 / 4));
      ra[i] = quad(A + (size_t)gm * K + gk, K - gk, gm < M);
    }
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int s = tid + i * kThreads;
      const int gk = k0 + s % kBK32, gn = n0 + 4 * (s / kBK32);
      rb[i] = quad(B + (size_t)gk * N + gn, N - gn, gk < K);
    }
  }

  __device__ inline void store(F32Smem& sm, int buf, int tid) {
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int s = tid + i * kThreads;
      *reinterpret_cast<dc::f32x4*>(&sm.a[buf][s / (kBK32 / 4)][4 * (s % (kBK32 / 4))]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int s = tid + i * kThreads;
#pragma unroll
      for (int e = 0; e < 4; ++e) sm.b[buf][4 * (s / kBK32) + e][s % kBK32] = rb[i][e];
    }
  }
};

__global__ __launch_bounds__(kThreads, 2) void gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                               float* __restrict__ C, int M, int N, int K, int tiles_m,
                                                               int tiles_n) {
  __shared__ F32Smem sm;
  const TileCoord tc = map_tile(tiles_m, tiles_n);
  const int m0 = tc.tm * kT32, n0 = tc.tn * kT32;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int r = lane & 31, h = lane >> 5;

  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;

  F32Loader ld;
  const int kt_count = (K + kBK32 - 1) / kBK32;
  ld.load(A, B, M, N, K, m0, n0, 0, tid);
  ld.store(sm, 0, tid);
  __syncthreads();

  for (int kt = 0; kt < kt_count; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < kt_count) ld.load(A, B, M, N, K, m0, n0, (kt + 1) * kBK32, tid);
#pragma unroll
    for (int ks = 0; ks < kBK32; ks += 16) {
      dc::f32x4 a[2], b[2];
      const float *pa = &sm.a[buf][wm * 32 + r][ks + 8 * h], *pb = &sm.b[buf][wn * 32 + r][ks + 8 * h];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        a[j] = *reinterpret_cast<const dc::f32x4*>(pa + 4 * j);
        b[j] = *reinterpret_cast<const dc::f32x4*>(pb + 4 * j);
      }
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[kk >> 2][kk & 3], b[kk >> 2][kk & 3], acc, 0, 0, 0);
    }
    if (kt + 1 < kt_count) ld.store(sm, buf ^ 1, tid);
    __syncthreads();
  }

  // acc[v] holds C[row][col], row = 8*(v/4) + 4*h + v%4, col = r (within the wave's 32×32 tile).
  const int col = n0 + wn * 32 + r;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = m0 + wm * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
    if (row < M && col < N) C[(size_t)row * N + col] = acc[v];
  }
}

// ---------------------------------------------------------------------------------------------
// bf16 inputs (raw bit patterns), fp32 accumulate: C = A·B straight from row-major A[M][K], B[K][N].
//
// Macro tile TM×TN, BK = 64, double-buffered LDS, WM×WN waves of 32·kMT × 32·kNT each (MFMA
// 32×32×16 tiles): 256×256 with 2×4 waves (128 KiB of LDS, one workgroup per CU, 128 accumulators
// per lane, two waves per SIMD so one's LDS and barrier waits overlap the other's MFMAs), 128×128
// and 64×64 with 2×2 waves (64 and 32 KiB, two and four workgroups per CU). KS > 1: KS such wave
// groups per workgroup, each with LDS buffers of its own, take the k tiles in turn (tile kt goes to
// group kt mod KS), and their sums are added in group order at the end: more loads in flight for a
// grid of few tiles. Measured (more beside the rule in dc_gemm_route.hpp): 2000×3000×1000 144 -> 21 us
// (560 TFLOP/s; the kernel it replaces loaded and transposed element by element), 1999×2999×999
// 31 us; 8192^3 0.84 ms (1300 TFLOP/s), as before. The big tile is bound by the matrix cores' power
// limit and its tile barriers, the small ones by the latency of one tile's loads per barrier.
//
// LDS image of a tile, in 1 KiB blocks of 64 16-byte chunks (chunk L of a block is lane L's):
// - A tile: TM rows (m) of 64 k, 128 B per row. The 16-byte k-octet q of row R sits in slot
//   q ^ ((R >> 1) & 7), so a fragment read (ds_read_b128: rows R0..R0+15 at one octet for each 16
//   lanes) touches 16 distinct 16-byte bank groups.
// - B tile: 64 rows (k) of TN n, 2·TN B per row, as B is stored. The 64-byte block b of row k
//   sits at block b ^ (k & 3) (TN = 64, two blocks per row: b ^ ((k >> 1) & 1)). The MFMA wants 8
//   consecutive k of one column n per lane; the transposing LDS read ds_read_b64_tr_b16 gives that:
//   within each 16 lanes, source lane s = 4j + p reads the 4 bf16 of row k0 + j at columns n0 +
//   4p..4p+3, and lane i receives B[k0 + j][n0 + i] for j = 0..3 (two such reads give k0..k0+7).
//   The 32 lanes of each half wave read 4 rows × 64 B at four different 64-byte offsets modulo
//   256 B: no bank conflicts.
// The swizzles are applied on the global side: each lane fetches the 16 bytes that belong in its
// LDS slot.
//
// Global -> LDS, two loaders:
// - kDma (16-byte aligned rows: k and n multiples of 8, aligned operands): direct-to-LDS loads
//   (buffer_load_dwordx4 ... lds: lane L writes LDS bytes 16·L of a block), so no registers stage
//   the tile and a tile's loads stay in flight for a whole tile of MFMAs. Rows past M and columns
//   past N re-read the last ones (their results are not stored); in a last tile of fewer than 64 k
//   the chunks past K are requested past the buffer range, which loads zeros.
// - registers (any other shape): 16-byte loads at the elements' own alignment, stored to the same
//   LDS slots a tile later. A tile past N is moved back to end there and rows past M re-read the last
//   one, so its loads need no checks (rows past M and columns that another tile owns are not stored);
//   the last tile of a ragged k, and matrices of fewer columns than a tile, take element-wise checked
//   loads.
//
// Pipeline of tile kt (buffer kt & 1): steps 0..2 run their MFMAs with the next step's fragment
// reads between them; then the tile's one barrier (which also waits for tile kt+1's loads, issued
// a tile earlier); right after it the loads of tile kt+2 go out into the buffer tile kt just
// finished with, and the last step's MFMAs run with tile kt+1's step-0 fragment reads between
// them, so no LDS latency is exposed after the barrier.
// ---------------------------------------------------------------------------------------------
constexpr int kBK2 = 64;
constexpr int kARow = kBK2 * 2;  // bytes per A row in LDS (64 k)

template <int TM, int TN>
struct Bf16Smem {
  unsigned short a[2][TM * kBK2];
  unsigned short b[2][kBK2 * TN];
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;
// 8 bf16 at the alignment of one (the unaligned 16-byte load)
typedef unsigned short u16x8_any __attribute__((ext_vector_type(8), aligned(2)));

// Buffer range of the kDma loader: the host keeps every byte offset below it (dc_gemm_route.hpp), so a
// lane that must load zeros asks for kPastRange, whatever the uniform offset added to it.
constexpr int32_t kDmaRange = dc::kBf16DmaRange;
constexpr uint32_t kPastRange = 0x80000000u;

// Issues the direct-to-LDS loads of the k tile at k0 (klim = k rows left from there) for the panels
// that start at A (row pitch K, in avoff) and B (row pitch N). Wave w's load i fills block i·WAVES + w
// of the A and of the B tile; avoff[i] / bvoff are the lane's byte offsets within the panel and the
// block's rows, the uniform part is the scalar offset.
template <int ABLOCKS, int BBLOCKS, int WAVES, int ROWS>
__device__ inline void bf16_tile_to_lds(unsigned short* la, unsigned short* lb, const unsigned short* __restrict__ A,
                                        const unsigned short* __restrict__ B, int N, int k0, int klim, int wave, int akq,
                                        const uint32_t* avoff, int brow, uint32_t bvoff) {
  const auto ra = dc::range_rsrc(A, kDmaRange), rb = dc::range_rsrc(B, kDmaRange);
#pragma unroll
  for (int i = 0; i < ABLOCKS; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(la + (i * WAVES + wave) * 512), 16,
                                             akq < klim ? avoff[i] : kPastRange, k0 * 2, 0, 0);
#pragma unroll
  for (int i = 0; i < BBLOCKS; ++i) {
    const int krow = ROWS * (i * WAVES + wave);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(lb + (i * WAVES + wave) * 512), 16,
                                             krow + brow < klim ? bvoff : kPastRange, (k0 + krow) * N * 2, 0, 0);
  }
}

template <int TM, int TN, int WM, int WN, int KS, bool kDma>
__global__ __launch_bounds__(64 * WM * WN * KS, (WM * WN == 8 ? 1 : 2)) void gemm_bf16_kernel(
    const unsigned short* __restrict__ A, const unsigned short* __restrict__ B, float* __restrict__ C, int M, int N,
    int K, int tiles_m, int tiles_n) {
  constexpr int kWaves = WM * WN;
  constexpr int kMT = TM / WM / 32, kNT = TN / WN / 32;  // MFMA tiles per wave
  constexpr int kABlocks = TM / 8 / kWaves, kBBlocks = TN / 8 / kWaves;  // 1 KiB blocks per wave and tile
  constexpr int kRows = 512 / TN;    // k-rows of B per block
  constexpr int kBRow = 2 * TN;      // bytes per B row in LDS
  using Smem = Bf16Smem<TM, TN>;
  __shared__ __align__(16) Smem sms[KS];
  const TileCoord tc = map_tile(tiles_m, tiles_n);
  const int m0 = tc.tm * TM;
  // (register loader: the last tile ends at N where N holds a whole tile)
  const int n0 = kDma || N < TN ? tc.tn * TN : min(tc.tn * TN, N - TN);
  // wave index in a scalar register: the loads' LDS bases and scalar offsets derive from it
  const int tid = threadIdx.x, lane = tid & 63, gwave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = gwave / kWaves, wave = gwave % kWaves;
  Smem& sm = sms[group];
  const int wm = wave / WN, wn = wave % WN;
  const int r = lane & 31, h = lane >> 5;
  const int kt_count = ((K + kBK2 - 1) / kBK2 + KS - 1) / KS;  // k tiles per group
  auto bswz = [](int k) __attribute__((always_inline)) { return TN == 64 ? (k >> 1) & 1 : k & 3; };

  // ---- load side. A: lane -> row L / 8 of a block, slot L % 8 = octet (L % 8) ^ ((row >> 1) % 8),
  // the same for each of the wave's blocks i·waves + w. B: lane -> row L / (TN / 8) of the block and
  // chunk L % (TN / 8), which holds the global chunk of the swizzle.
  const int arow = lane >> 3;
  const int akq = 8 * ((lane & 7) ^ ((4 * wave + (arow >> 1)) & 7));
  const int brow = lane / (TN / 8), bc = lane % (TN / 8);
  const int bchunk = 4 * ((bc >> 2) ^ bswz(kRows * wave + brow)) + (bc & 3);
  uint32_t avoff[kABlocks], bvoff = 0;
  u16x8 sa[kABlocks], sb[kBBlocks];
  if constexpr (kDma) {
#pragma unroll
    for (int i = 0; i < kABlocks; ++i)
      avoff[i] = (uint32_t)((min(8 * (i * kWaves + wave) + arow, M - 1 - m0) * K + akq) * 2);
    bvoff = (uint32_t)((brow * N + min(8 * bchunk, N - 8 - n0)) * 2);
  }
  // Loads the group's k tile KT (into LDS buffer BUF, or into registers).
  auto load_tile = [&](auto BUF, int KT) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(BUF)::value;
    const int k0 = (KT * KS + group) * kBK2;
    const int klim = K - k0;  // k rows of the tile that exist (64 or more: all; none: the tile is zero)
    if constexpr (kDma) {
      bf16_tile_to_lds<kABlocks, kBBlocks, kWaves, kRows>(sm.a[kBuf], sm.b[kBuf], A + (size_t)m0 * K, B + n0, N, k0, klim,
                                                          wave, akq, avoff, brow, bvoff);
    } else {
      const bool whole_k = klim >= kBK2;  // uniform, as is N >= TN
      if (whole_k) {
#pragma unroll
        for (int i = 0; i < kABlocks; ++i)
          sa[i] = *reinterpret_cast<const u16x8_any*>(A + (size_t)min(m0 + 8 * (i * kWaves + wave) + arow, M - 1) * K +
                                                      k0 + akq);
      } else {
#pragma unroll
        for (int i = 0; i < kABlocks; ++i) {
          const unsigned short* p = A + (size_t)min(m0 + 8 * (i * kWaves + wave) + arow, M - 1) * K + k0 + akq;
#pragma unroll
          for (int e = 0; e < 8; ++e) sa[i][e] = akq + e < klim ? p[e] : 0;
        }
      }
      if (whole_k && N >= TN) {
#pragma unroll
        for (int i = 0; i < kBBlocks; ++i)
          sb[i] = *reinterpret_cast<const u16x8_any*>(B + (size_t)(k0 + kRows * (i * kWaves + wave) + brow) * N + n0 +
                                                      8 * bchunk);
      } else {
#pragma unroll
        for (int i = 0; i < kBBlocks; ++i) {
          const int gk = kRows * (i * kWaves + wave) + brow, gn = n0 + 8 * bchunk;
          const unsigned short* p = B + (size_t)(k0 + gk) * N + gn;
#pragma unroll
          for (int e = 0; e < 8; ++e) sb[i][e] = gk < klim && gn + e < N ? p[e] : 0;
        }
      }
    }
  };
  // Register loader: stores the loaded tile into LDS buffer BUF.
  auto store_tile = [&](auto BUF) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(BUF)::value;
#pragma unroll
    for (int i = 0; i < kABlocks; ++i)
      *reinterpret_cast<u16x8*>(&sm.a[kBuf][(i * kWaves + wave) * 512 + lane * 8]) = sa[i];
#pragma unroll
    for (int i = 0; i < kBBlocks; ++i)
      *reinterpret_cast<u16x8*>(&sm.b[kBuf][(i * kWaves + wave) * 512 + lane * 8]) = sb[i];
  };

  // ---- read side, A: fragment rows R = 32·t + r (t: wave and tile offsets), so the swizzle is
  // (r >> 1) % 8; k-octet 2·step + h. Byte offsets of step s in buffer 0 (buffer and mt offsets are
  // immediates).
  const int rswz = (r >> 1) & 7;
  uint32_t aoff[4];
#pragma unroll
  for (int st = 0; st < 4; ++st)
    aoff[st] = (uint32_t)(wm * 32 * kMT + r) * kARow + 16u * (uint32_t)((2 * st + h) ^ rswz);
  // read side, B: source lane s = L % 16 = 4j + p reads row 8h + j (+16·step, +4 for the upper
  // four k: immediates) at columns wn·32·kNT + nt·32 + 16·((L / 16) & 1) + 4p; the row is ≡ j
  // (mod 4), so its 64-byte block kNT·wn + nt sits at block ^ bswz(j)
  uint32_t boff[kNT];
  {
    const int j = (lane & 15) >> 2, p4 = lane & 3, cg = (lane >> 4) & 1;
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      boff[nt] = (uint32_t)offsetof(Smem, b) + (uint32_t)((8 * h + j) * kBRow) +
                 64u * (uint32_t)((kNT * wn + nt) ^ bswz(j)) + (uint32_t)(32 * cg + 8 * p4);
  }

  f32x16 acc[kMT][kNT];
#pragma unroll
  for (int i = 0; i < kMT; ++i)
#pragma unroll
    for (int j = 0; j < kNT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  constexpr int kSteps = kBK2 / 16;
  static_assert(kSteps == 4, "four 16-wide k steps per tile");
  const unsigned char* lds = reinterpret_cast<const unsigned char*>(&sm);
  // B fragments of a whole tile (4 steps × kNT × 2 transposing reads) in one burst. The compiler
  // cannot tell these intrinsic reads apart from the LDS the direct-to-LDS loads write, so it
  // waits for every load in flight before each of them: the burst is issued while none is (right
  // after a barrier that waited for them all, before the next tile's loads go out).
  auto read_b_tile = [&](auto BUF, bf16x8 (*b)[kNT]) __attribute__((always_inline)) {
    constexpr uint32_t kBufB = (uint32_t)decltype(BUF)::value * kBK2 * kBRow;
#pragma unroll
    for (int st = 0; st < kSteps; ++st)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        const unsigned char* q = lds + boff[nt] + kBufB + st * 16 * kBRow;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(q));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(q + 4 * kBRow));
        b[st][nt] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
  };
  auto read_a = [&](auto BUF, int step, bf16x8* a) __attribute__((always_inline)) {
    constexpr uint32_t kBufA = (uint32_t)decltype(BUF)::value * TM * kARow;
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
      a[mt] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(lds + aoff[step] + kBufA + mt * 32 * kARow));
  };
  auto mfmas = [&](const bf16x8* a, const bf16x8* b) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[mt], b[nt], acc[mt][nt], 0, 0, 0);
  };
  // One A read after each of the first kMT MFMAs of the region (the rest run back to back).
  auto interleave_reads = []() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // 1 LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
    }
  };
  // The next tile is in LDS and every wave is done reading the other buffer.
  auto tile_barrier = [&](auto NEXT) __attribute__((always_inline)) {
    if constexpr (kDma) {
      dma_barrier();
    } else {
      store_tile(NEXT);
      __syncthreads();
    }
  };
  bf16x8 fa[2][kMT], fb[2][kSteps][kNT];
  constexpr std::integral_constant<int, 0> kBuf0{};
  constexpr std::integral_constant<int, 1> kBuf1{};
  load_tile(kBuf0, 0);
  tile_barrier(kBuf0);
  read_b_tile(kBuf0, fb[0]);
  read_a(kBuf0, 0, fa[0]);
  if (kt_count > 1) load_tile(kBuf1, 1);
  // Tile kt in LDS buffer BUF = kt % 2 (the loop is unrolled by two, so buffer offsets are
  // constants; a macro rather than a lambda keeps the fragment arrays plain registers).
#define DC_BF16_TILE(BUF, KT)                                                                      \
  {                                                                                                \
    _Pragma("unroll") for (int step = 0; step + 1 < kSteps; ++step) {                              \
      const int cur = step & 1;                                                                    \
      __builtin_amdgcn_sched_barrier(0);                                                           \
      read_a(kBuf##BUF, step + 1, fa[cur ^ 1]);                                                    \
      mfmas(fa[cur], fb[BUF][step]);                                                               \
      interleave_reads();                                                                          \
      __builtin_amdgcn_sched_barrier(0);                                                           \
    }                                                                                              \
    /* tile KT+1 is in LDS; every wave is done reading buffer BUF (after the last tile the */     \
    /* barrier and the reads of the other buffer are harmless and unused) */                      \
    tile_barrier(std::integral_constant<int, 1 - (BUF)>{});                                        \
    read_b_tile(std::integral_constant<int, 1 - (BUF)>{}, fb[1 - (BUF)]);                          \
    if ((KT) + 2 < kt_count) load_tile(kBuf##BUF, (KT) + 2);                                       \
    __builtin_amdgcn_sched_barrier(0);                                                             \
    read_a(std::integral_constant<int, 1 - (BUF)>{}, 0, fa[0]);                                    \
    mfmas(fa[1], fb[BUF][kSteps - 1]);                                                             \
    interleave_reads();                                                                            \
    __builtin_amdgcn_sched_barrier(0);                                                             \
  }
  // K > 0 (host check): at least one tile, and no zero-trip path that would keep the accumulators'
  // initial values live beside the loop
  __builtin_assume(kt_count > 0);
  int kt = 0;
  do {
    DC_BF16_TILE(0, kt);
    if (kt + 1 < kt_count) DC_BF16_TILE(1, kt + 1);
    kt += 2;
  } while (kt < kt_count);
#undef DC_BF16_TILE

  if constexpr (KS > 1) {  // the groups' sums, added in group order by group 0
    static_assert(sizeof(Smem) >= kWaves * 64 * kMT * kNT * 16 * sizeof(float), "a group's sums fit in its buffers");
    float* part = reinterpret_cast<float*>(&sm) + tid % (64 * kWaves);
    __syncthreads();
    if (group > 0)
#pragma unroll
      for (int i = 0; i < kMT * kNT * 16; ++i) part[i * 64 * kWaves] = acc[i / 16 / kNT][i / 16 % kNT][i % 16];
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KS; ++g) {
      const float* other = reinterpret_cast<const float*>(&sms[g]) + tid;
#pragma unroll
      for (int i = 0; i < kMT * kNT * 16; ++i) acc[i / 16 / kNT][i / 16 % kNT][i % 16] += other[i * 64 * kWaves];
    }
  }
  // acc[mt][nt][v] holds C[row][col], row = 8*(v/4) + 4*h + v%4, col = r (within the 32×32 tile).
  // Only the rows and columns of this tile's own place are stored.
  const bool whole = m0 + TM <= M && n0 + TN <= N && n0 == tc.tn * TN;
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      const int col = n0 + (wn * kNT + nt) * 32 + r;
      const bool cok = col < N && col >= tc.tn * TN;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = m0 + (wm * kMT + mt) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
        if (whole || (cok && row < M)) C[(size_t)row * N + col] = acc[mt][nt][v];
      }
    }
}

// ---------------------------------------------------------------------------------------------
// fp32 on the bf16 matrix cores: every fp32 value is the exact sum of three bf16 pieces,
// x = x0 + x1 + x2 (x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1, rounded to nearest, so |x1| <=
// 2^-8 |x| and |x2| <= 2^-17 |x|), and a·b is formed from eight of the nine products of pieces, each
// exact in fp32; the one left out, a2 b2, is at most 2^-34 |a b|. The sums of a0 b0 and those of the
// seven small products stand in accumulators of their own and are added once, at the end: an
// instruction's sum may be off by nearly an ulp (these matrix cores cut the addends at half an ulp of
// the largest before they round), which matters 2^-7 times less in the small sums, and the large ones
// are rounded once per 8 products (by the errors) where the fp32 instructions round each. So the result
// is closer to the float64 product than theirs: relative error with normal inputs 5.7e-7 against 1.62e-6
// at 8192^3, 1.3e-7 against 5.7e-7 at 1537×2049×1023; a sum of one term is within 0.62 ulp (0.50). (All
// in one accumulator, 256×256 tiles: 5.74 ms at 8192^3, 1.44e-6, one term up to an ulp off. Six products,
// without a1 b2 and a2 b1: 4.6 ms, each product off by up to 2^-24 of it, one term up to 1.5 ulp.)
// 8 bf16 products cost half of one fp32 product on this chip's matrix cores. Measured against the
// kernels on the fp32 instructions: 8192^3 7.30 -> 6.02 ms (183 TFLOP/s where those instructions peak
// at 157), 4096^3 925 -> 760 us, 1537×2049×1023 144 -> 53.5 us.
// Bound by the matrix cores at the clock that power allows (large grids) and by what a workgroup's
// barriers leave uncovered (small ones).
//
// Where the pieces do not hold the value: infinities and NaN (x - x0 is NaN, so the sum is), values
// that round up to infinity in bf16 (likewise), and nonzero magnitudes below kSplitMin, whose lowest
// pieces fall below bf16's subnormals (an error below 2^-134 each). A sum that is not finite, or that
// such small values in its row of A or column of B could have moved by more than 2^-32 of itself, is
// formed again with v_mfma_f32_32x32x2_f32 (f32_blocks_direct below), and only it is stored again: those
// inputs give what the fp32 instructions give, and every other sum has the same bits whatever the rest
// of its tile holds. Tiles in which nothing would stand are not formed by pieces at all: every row of
// A past kSplitMax in the first k tile, or that tile of A or of B nonzero and below kSplitMin throughout
// (the one case in which a sum's arithmetic depends on its tile). Measured at 8192^3 (fp32 instructions
// alone 7.3 ms; 6.1 without such values): an infinity in one row of every 256 8.3 ms, in every 16th row
// 19.4 (every block of 32×32 is formed twice); half of A at -3.4e38, or all of it NaN or near 2^-110, 13.2;
// a tenth of A's elements near 2^-110 6.2, with half the columns of B zero 6.6. At 1537×2049×1023 (144 us;
// 55.6): 123, 132, 82, 58 and 80 us. bf16 subnormals and products down to the fp32 subnormals are kept by
// the matrix cores (measured), so results near 2^-126 are as exact as before.
//
// Macro tile TM×TN, KS groups of WM×WN waves that take the k tiles (16 k each) in turn (as
// gemm_bf16_kernel). A tile's fp32 elements come through registers (16-byte loads at 4-byte alignment,
// D tiles ahead: so no shape or alignment needs another kernel), are split and stored to LDS as three
// bf16 planes, in the other of two buffers, while this tile's products run: about 7 VALU
// instructions per element beside 32 MFMAs (64-tiles: 8) per wave and tile. LDS images per plane:
// - A: rows of 16 k (32 B); the 16-byte half h of row R sits at h ^ ((R >> 3) & 1), so a
//   fragment read (16 rows at one half for each 16 lanes) touches 16 distinct 16-byte bank groups.
// - B: k rows of TN n with the 64-byte blocks swizzled, read through ds_read_b64_tr_b16
//   (as gemm_bf16_kernel).
// ---------------------------------------------------------------------------------------------
constexpr float kSplitMin = 0x1p-102f;
constexpr int kSplitMinExp = -101;             // its exponent as split_quad counts
constexpr float kSplitMax = 0x1.fefffep127f;  // the largest magnitude that does not round to infinity in bf16
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Calls f(std::integral_constant<int, I>) for I = 0, 1, ...: a compile-time unrolled loop.
template <typename F, int... I>
__device__ __attribute__((always_inline)) inline void for_each_index(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// The three bf16 pieces of four values, packed; *big and *tiny become the largest and smallest exponent
// seen (|x| in [2^(e-1), 2^e); 0 for zeros, infinities and NaN, which neither reads amiss: see below).
__device__ inline void split_quad(dc::f32x4 x, u32x2 (&piece)[3], int* big, int* tiny) {
  f32x2 v[2] = {{x.x, x.y}, {x.z, x.w}};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int e0 = __builtin_amdgcn_frexp_expf(v[i].x), e1 = __builtin_amdgcn_frexp_expf(v[i].y);
    *big = max(*big, max(e0, e1));
    *tiny = min(*tiny, min(e0, e1));
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(v[i], bf16x2));
      piece[p][i] = w;
      if (p < 2) {
        v[i].x -= __builtin_bit_cast(float, w << 16);
        v[i].y -= __builtin_bit_cast(float, w & 0xFFFF0000u);
      }
    }
  }
}

// A wave's 32×32 blocks (bits mt·kNT + nt of `need`, uniform) at row0, col0 of C with the fp32 matrix
// instructions, into acc. Fragments come straight from global memory, two steps of 32 k's in flight, so
// waves with nothing to do cost the others nothing: no LDS, no barrier. Lane group h takes the k's [16h,
// 16h + 16) of a step, so a step's loads of A use whole 128-byte lines at once. Rows past M re-read the
// last one; every column exists.
template <int kMT, int kNT>
__device__ __attribute__((always_inline)) inline void f32_blocks_direct(const float* __restrict__ A,
                                                                        const float* __restrict__ B, int M, int N, int K,
                                                                        int row0, int col0, int lane, uint32_t need,
                                                                        f32x16 (&acc)[kMT][kNT]) {
  constexpr int kDepth = 2, kStep = 32, kHalf = kStep / 2;
  const int r = lane & 31, h = lane >> 5;
  const float* pa[kMT];
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt) pa[mt] = A + (size_t)min(row0 + mt * 32 + r, M - 1) * K + kHalf * h;
  const float* pb = B + (size_t)(kHalf * h) * N + col0 + r;
  dc::f32x4 a[kDepth][kMT][kHalf / 4];
  float b[kDepth][kNT][kHalf];
  auto load = [&](int s, dc::f32x4 (&fa)[kMT][kHalf / 4], float (&fb)[kNT][kHalf]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kMT * kHalf / 4; ++i)
      fa[i / (kHalf / 4)][i % (kHalf / 4)] =
          *reinterpret_cast<const f32x4_any*>(pa[i / (kHalf / 4)] + kStep * s + 4 * (i % (kHalf / 4)));
#pragma unroll
    for (int i = 0; i < kHalf * kNT; ++i) fb[i % kNT][i / kNT] = pb[(size_t)(kStep * s + i / kNT) * N + 32 * (i % kNT)];
  };
  auto multiply = [&](const dc::f32x4 (&fa)[kMT][kHalf / 4], const float (&fb)[kNT][kHalf]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kMT * kNT; ++i)
      if (need >> i & 1u)
#pragma unroll
        for (int kk = 0; kk < kHalf; ++kk)
          acc[i / kNT][i % kNT] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i / kNT][kk >> 2][kk & 3], fb[i % kNT][kk],
                                                                       acc[i / kNT][i % kNT], 0, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < kMT * kNT * 16; ++i) acc[i / 16 / kNT][i / 16 % kNT][i % 16] = 0.0f;
  const int whole = K / kStep;  // steps
  int s = 0;
  if (whole >= kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) load(d, a[d], b[d]);
#pragma unroll 1
    for (; s + kDepth <= whole; s += kDepth)
#pragma unroll
      for (int d = 0; d < kDepth; ++d) {
        multiply(a[d], b[d]);
        load(min(s + kDepth + d, whole - 1), a[d], b[d]);
      }
  }
#pragma unroll 1
  for (; s < whole; ++s) {
    load(s, a[0], b[0]);
    multiply(a[0], b[0]);
  }
  if (K % kStep != 0) {
    const int left = K - kStep * whole - kHalf * h;  // of the lane group's k's
#pragma unroll
    for (int i = 0; i < kMT * kHalf; ++i)
      a[0][i / kHalf][i / 4 % (kHalf / 4)][i % 4] = i % kHalf < left ? pa[i / kHalf][kStep * whole + i % kHalf] : 0.0f;
#pragma unroll
    for (int i = 0; i < kNT * kHalf; ++i)
      b[0][i / kHalf][i % kHalf] = i % kHalf < left ? pb[(size_t)(kStep * whole + i % kHalf) * N + 32 * (i / kHalf)] : 0.0f;
    multiply(a[0], b[0]);
  }
}

// Whether a magnitude (as 2|x|'s bits - 1; zero: all ones) is nonzero and below kSplitMin.
constexpr uint32_t kTinyBits = 2u * __builtin_bit_cast(uint32_t, kSplitMin) - 1u;

// For each of `rows` rows of K at A and each of TN columns of the K rows at B: the bits of its largest
// magnitude into stat[row], stat[TM + column], and 1 into stat[TM + TN + ...] if it holds a nonzero
// one below kSplitMin. By the whole workgroup; stat is zero before.
template <int TM, int TN, int kThreadsPerBlock>
__device__ inline void panel_stats(const float* __restrict__ A, int rows, const float* __restrict__ B, int N, int K, int tid,
                                   uint32_t* stat) {
  constexpr int kIn = 8;  // 16-byte loads in flight; the last ones re-read the end (K >= 4)
  auto take = [&](const float* p) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4_any*>(p); };
  auto fold = [&](float x, uint32_t& big, uint32_t& tiny) __attribute__((always_inline)) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x) << 1;
    big = max(big, u);
    tiny = min(tiny, u - 1u);
  };
  auto put = [&](int i, uint32_t big, uint32_t tiny) __attribute__((always_inline)) {
    atomicMax(&stat[i], big >> 1);
    if (tiny < kTinyBits) stat[TM + TN + i] = 1u;
  };
#pragma unroll 1
  for (int row = tid >> 6; row < rows; row += kThreadsPerBlock / 64) {  // a wave per row
    const float* p = A + (size_t)row * K;
    uint32_t big = 0, tiny = 0xFFFFFFFFu;
#pragma unroll 1
    for (int k = 4 * (tid & 63); k < K; k += 256 * kIn) {
      dc::f32x4 x[kIn];
#pragma unroll
      for (int u = 0; u < kIn; ++u) x[u] = take(p + min(k + 256 * u, K - 4));
#pragma unroll
      for (int u = 0; u < 4 * kIn; ++u) fold(x[u / 4][u % 4], big, tiny);
    }
    put(row, big, tiny);
  }
  constexpr int kRows = 4 * kThreadsPerBlock / TN;
  const int col = 4 * (tid % (TN / 4));
  uint32_t big[4] = {}, tiny[4] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
#pragma unroll 1
  for (int k = tid / (TN / 4); k < K; k += kIn * kRows) {
    dc::f32x4 x[kIn];
#pragma unroll
    for (int u = 0; u < kIn; ++u) x[u] = take(B + col + (size_t)min(k + u * kRows, K - 1) * N);
#pragma unroll
    for (int u = 0; u < 4 * kIn; ++u) fold(x[u / 4][u % 4], big[u % 4], tiny[u % 4]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) put(TM + col + e, big[e], tiny[e]);
}

template <int TM, int TN>
struct SplitSmem {
  unsigned short a[2][3][TM * 16];
  unsigned short b[2][3][16][TN];
};

template <int TM, int TN, int WM, int WN, int KS, int D>
__global__ __launch_bounds__(64 * WM * WN * KS, (KS == 1 && WM * WN == 4 ? 2 : 1)) void gemm_f32_split_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N, int K, int tiles_m,
    int tiles_n) {
  constexpr int kWaves = WM * WN, kT = 64 * kWaves;
  constexpr int kMT = TM / WM / 32, kNT = TN / WN / 32;      // MFMA tiles per wave
  constexpr int kBK = 16;
  constexpr int kA = TM * 4 / kT, kB = TN * 4 / kT;  // quads per thread and k tile
  using Smem = SplitSmem<TM, TN>;
  __shared__ __align__(16) Smem sms[KS];
  __shared__ int s_redo, s_tiny, s_low, s_big;
  __shared__ uint32_t s_seen;
  const TileCoord tc = map_tile(tiles_m, tiles_n);
  const int m0 = tc.tm * TM;
  const int n0 = min(tc.tn * TN, N - TN);  // the last tile ends at N (N >= TN, by the host)
  const int tid = threadIdx.x, lane = tid & 63, gwave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = gwave / kWaves, wave = gwave % kWaves, t = tid % kT;
  Smem& sm = sms[group];
  const int wm = wave / WN, wn = wave % WN;
  const int r = lane & 31, h = lane >> 5;
  const int kt_count = ((K + kBK - 1) / kBK + KS - 1) / KS;  // k tiles per group
  auto bswz = [](int k) __attribute__((always_inline)) { return TN == 64 ? (k >> 1) & 1 : k & 3; };

  // ---- load side: the lane's element offsets from the tile's first (uniform) A and B element
  uint32_t ga[kA], gb[kB], wa[kA], wb[kB];  // wa, wb: LDS elements (buffer and plane 0)
#pragma unroll
  for (int i = 0; i < kA; ++i) {
    const int idx = i * kT + t, row = idx / 4, q = idx % 4;
    ga[i] = (uint32_t)(min(row, M - 1 - m0) * K + 4 * q);
    wa[i] = (uint32_t)(row * 16 + 8 * ((q >> 1) ^ ((row >> 3) & 1)) + 4 * (q & 1));
  }
#pragma unroll
  for (int i = 0; i < kB; ++i) {
    const int idx = i * kT + t, krow = idx / (TN / 4), nq = idx % (TN / 4);
    gb[i] = (uint32_t)(krow * N + 4 * nq);
    wb[i] = (uint32_t)(krow * TN + 32 * ((nq >> 3) ^ bswz(krow)) + 4 * (nq & 7));
  }
  dc::f32x4 sa[D][kA], sb[D][kB];  // D tiles of elements in flight
  int big = -200, tiny = 0;  // over the lane's elements: see split_quad
  // The group's k tile KT, every element of which exists.
  auto load_tile = [&](int KT, dc::f32x4 (&qa)[kA], dc::f32x4 (&qb)[kB]) __attribute__((always_inline)) {
    const int k0 = (KT * KS + group) * kBK;
    const float *at = A + (size_t)m0 * K + k0, *bt = B + (size_t)k0 * N + n0;
#pragma unroll
    for (int i = 0; i < kA; ++i) qa[i] = *reinterpret_cast<const f32x4_any*>(at + ga[i]);
#pragma unroll
    for (int i = 0; i < kB; ++i) qb[i] = *reinterpret_cast<const f32x4_any*>(bt + gb[i]);
  };
  // The group's k tile KT, zeros where it lies past K.
  auto load_checked = [&](int KT, dc::f32x4 (&qa)[kA], dc::f32x4 (&qb)[kB]) __attribute__((always_inline)) {
    const int k0 = (KT * KS + group) * kBK;
    const int klim = K - k0;  // k rows of the tile that exist (16 or more: all; none: the tile is zero)
    const float *at = A + (size_t)m0 * K + k0, *bt = B + (size_t)k0 * N + n0;
#pragma unroll
    for (int i = 0; i < kA; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) qa[i][e] = 4 * ((i * kT + t) % 4) + e < klim ? at[ga[i] + e] : 0.0f;
#pragma unroll
    for (int i = 0; i < kB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) qb[i][e] = (i * kT + t) / (TN / 4) < klim ? bt[gb[i] + e] : 0.0f;
  };
  auto split_tile = [&](auto BUF, const dc::f32x4 (&qa)[kA], const dc::f32x4 (&qb)[kB]) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(BUF)::value;
    u32x2 piece[3];
#pragma unroll
    for (int i = 0; i < kA; ++i) {
      split_quad(qa[i], piece, &big, &tiny);
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(&sm.a[kBuf][p][0] + wa[i]) = piece[p];
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) {
      split_quad(qb[i], piece, &big, &tiny);
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(&sm.b[kBuf][p][0][0] + wb[i]) = piece[p];
    }
  };

  // ---- read side
  const unsigned char* lds = reinterpret_cast<const unsigned char*>(&sm);
  const uint32_t aoff = (uint32_t)((wm * 32 * kMT + r) * 32 + 16 * (h ^ ((r >> 3) & 1)));
  uint32_t boff[kNT];
  {
    const int j = (lane & 15) >> 2, p4 = lane & 3, cg = (lane >> 4) & 1;
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      boff[nt] = (uint32_t)offsetof(Smem, b) + (uint32_t)((8 * h + j) * 2 * TN) +
                 64u * (uint32_t)((kNT * wn + nt) ^ bswz(j)) + (uint32_t)(32 * cg + 8 * p4);
  }
  f32x16 acc[kMT][kNT], low[kMT][kNT];  // a0 b0's sums; the other products'
#pragma unroll
  for (int i = 0; i < kMT; ++i)
#pragma unroll
    for (int j = 0; j < kNT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = low[i][j][v] = 0.0f;
  auto read_a = [&](int buf, int p, bf16x8 (&a)[kMT]) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
      a[mt] = __builtin_bit_cast(
          bf16x8, *reinterpret_cast<const u16x8*>(lds + aoff + ((buf * 3 + p) * TM + mt * 32) * 32));
  };
  auto read_b = [&](int buf, int p, bf16x8 (&b)[kNT]) __attribute__((always_inline)) {
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      const unsigned char* q = lds + boff[nt] + (buf * 3 + p) * 16 * 2 * TN;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(q));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(q + 4 * 2 * TN));
      b[nt] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  auto mfmas = [&](f32x16 (&sum)[kMT][kNT], const bf16x8 (&a)[kMT], const bf16x8 (&b)[kNT]) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt)
        sum[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[mt], b[nt], sum[mt][nt], 0, 0, 0);
  };
  // Fragments: plane 0 of B twice (the next tile's is read while this one's is still in use).
  bf16x8 a0[kMT], a1[kMT], a2[kMT], b0[2][kNT], b1[kNT], b2[kNT];
  constexpr int kMfmas = 5 * kMT * kNT, kSplits = kA + kB;  // of the first region
  // One k tile (buffer BUF) in two regions, of five products (those with a2 or a1) and of three (a0's;
  // a0 b0 is the last), the barrier between them. First region: the reads of the planes that come last,
  // and the split of the next tile (elements qa, qb) into the other buffer between the products. Second
  // region: the reads of the next tile's first fragments between the products, so none of the LDS time
  // is exposed.
  auto first = [&](auto BUF, const dc::f32x4 (&qa)[kA], const dc::f32x4 (&qb)[kB]) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(BUF)::value;
    __builtin_amdgcn_sched_barrier(0);
    read_a(kBuf, 0, a0);
    read_b(kBuf, 2, b2);
    split_tile(std::integral_constant<int, 1 - kBuf>{}, qa, qb);
    mfmas(low, a2, b0[kBuf]);
    mfmas(low, a2, b1);
    mfmas(low, a1, b1);
    mfmas(low, a1, b2);
    mfmas(low, a1, b0[kBuf]);
    __builtin_amdgcn_sched_group_barrier(0x100, kMT + 2 * kNT, 0);
#pragma unroll
    for (int i = 0; i < kMfmas; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, (28 * kSplits + kMfmas - 1) / kMfmas, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, (3 * kSplits + kMfmas - 1) / kMfmas, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto second = [&](auto BUF) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(BUF)::value, kNext = 1 - kBuf;
    __builtin_amdgcn_sched_barrier(0);
    read_a(kNext, 2, a2);
    read_b(kNext, 0, b0[kNext]);
    read_a(kNext, 1, a1);
    mfmas(low, a0, b2);
    mfmas(low, a0, b1);
    mfmas(acc, a0, b0[kBuf]);
    read_b(kNext, 1, b1);
#pragma unroll
    for (int i = 0; i < 2 * kMT * kNT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, (2 * kMT + 2 * kNT + 2 * kMT * kNT - 1) / (2 * kMT * kNT), 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (tid == 0) s_redo = s_tiny = s_low = s_seen = 0, s_big = -200;
  constexpr std::integral_constant<int, 0> kBuf0{};
  constexpr std::integral_constant<int, 1> kBuf1{};
  static_assert(D == 1 || D == 2, "the loop is unrolled by two");
  static_assert(TM <= 256, "the host checks 32-bit offsets in panels of 256 rows");
  // The group's last tile, the only one that can lie past K, comes first (checked loads); then tiles
  // 0, 1, ...: step p > 0 is tile p - 1. The host sees to kt_count >= 2 (k > 16 KS). Loads past the last step
  // re-read its tile (unused): no branch in the loop, so its waits for memory cover just the tile
  // that is split next.
  load_checked(kt_count - 1, sa[0], sb[0]);
  split_tile(kBuf0, sa[0], sb[0]);
  __syncthreads();  // the flags are set
  {  // bits: A's first tiles hold a nonzero value, one of at least kSplitMin; B's; a row of A's without a
     // value past kSplitMax
    float big_a = 0.0f, big_b = 0.0f;
    bool clean = false;
#pragma unroll
    for (int i = 0; i < kA; ++i) {
      bool past = false;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        big_a = __builtin_fmaxf(big_a, __builtin_fabsf(sa[0][i][e]));
        past |= !(__builtin_fabsf(sa[0][i][e]) <= kSplitMax);
      }
      uint64_t m = __ballot(past);  // four lanes hold a row
      m |= m >> 1;
      m |= m >> 2;
      clean |= (~m & 0x1111111111111111ull) != 0;
    }
#pragma unroll
    for (int i = 0; i < 4 * kB; ++i) big_b = __builtin_fmaxf(big_b, __builtin_fabsf(sb[0][i / 4][i % 4]));
    const uint32_t seen = (__any(big_a > 0.0f) ? 1u : 0u) | (__any(big_a >= kSplitMin) ? 2u : 0u) |
                          (__any(big_b > 0.0f) ? 4u : 0u) | (__any(big_b >= kSplitMin) ? 8u : 0u) | (clean ? 16u : 0u);
    if (lane == 0) atomicOr(&s_seen, seen);
  }
  for_each_index([&](auto I) __attribute__((always_inline)) {
    load_tile(min(I.value, kt_count - 2), sa[(1 + I.value) % D], sb[(1 + I.value) % D]);
  }, std::make_integer_sequence<int, D>{});
  __syncthreads();
  read_a(0, 2, a2);
  read_b(0, 0, b0[0]);
  read_a(0, 1, a1);
  read_b(0, 1, b1);
  // Step p in buffer I = p % 2: its products and the split of step p + 1, whose element set then
  // takes step p + 1 + D.
  auto one = [&](int p, auto I) __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value, set = (i + 1) % D;
    first(I, sa[set], sb[set]);
    __syncthreads();
    load_tile(min(p + D, kt_count - 2), sa[set], sb[set]);
    second(I);
  };
  // Nothing but small values in all of the first tiles (they are no exception here), or no sum that stands.
  const uint32_t seen = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_seen);
  const bool early = (seen & 3u) == 1u || (seen & 12u) == 4u || (seen & 16u) == 0u;
  __builtin_assume(kt_count > 1);
  if (!early) {
    int p = 0;
    do {  // (whole pairs: an exit between the two would cost copies of the accumulators)
      one(p, kBuf0);
      one(p + 1, kBuf1);
      p += 2;
    } while (p + 1 < kt_count);
    if (p < kt_count) one(p, kBuf0);
  }
  if (tiny < kSplitMinExp) s_tiny = 1;
#pragma unroll
  for (int i = 0; i < kMT * kNT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i / kNT][i % kNT][v] += low[i / kNT][i % kNT][v];

  if constexpr (KS > 1) {  // the groups' sums, added in group order by group 0
    constexpr int kSums = kT * kMT * kNT * 16;
    static_assert(sizeof(sms) >= (KS - 1) * kSums * sizeof(float), "the groups' sums fit in the buffers");
    float* part = reinterpret_cast<float*>(&sms[0]) + (group - 1) * kSums + t;
    __syncthreads();
    if (group > 0)
#pragma unroll
      for (int i = 0; i < kMT * kNT * 16; ++i) part[i * kT] = acc[i / 16 / kNT][i / 16 % kNT][i % 16];
    __syncthreads();
    if (group == 0)
#pragma unroll
      for (int g = 1; g < KS; ++g) {
        const float* other = reinterpret_cast<const float*>(&sms[0]) + (g - 1) * kSums + t;
#pragma unroll
        for (int i = 0; i < kMT * kNT * 16; ++i) acc[i / 16 / kNT][i / 16 % kNT][i % 16] += other[i * kT];
      }
  }
  __syncthreads();
  // Which sums stand: finite, and not moved by the pieces that small values lost, 2^-134 at most each, by
  // more than 2^-32 of themselves. By row and column, so that a sum's arithmetic depends on no other's.
  uint32_t* stat = reinterpret_cast<uint32_t*>(&sms[0]);
  static_assert(sizeof(Smem) >= 2 * (TM + TN) * sizeof(uint32_t), "the rows' and columns' figures fit in the buffers");
  constexpr float kLost = 0x1p-102f;
  bool scan = s_tiny != 0 && !early;  // uniform, as all of this
  if (scan) {  // unless every sum stands whatever its row and column hold (their infinities and NaN aside:
               // no sum that those reach is finite)
    atomicMax(&s_big, big);
    __syncthreads();
    const float least = __builtin_ldexpf(2.0f * (float)K * kLost, s_big);
    bool low = false;
#pragma unroll
    for (int i = 0; i < kMT * kNT * 16; ++i) low |= __builtin_fabsf(acc[i / 16 / kNT][i / 16 % kNT][i % 16]) < least;
    if (group == 0 && low) s_low = 1;
    __syncthreads();
    scan = s_low != 0;
  }
  if (scan) {
    for (int i = tid; i < 2 * (TM + TN); i += kT * KS) stat[i] = 0;
    __syncthreads();
    panel_stats<TM, TN, kT * KS>(A + (size_t)m0 * K, min(TM, M - m0), B + n0, N, K, tid, stat);
    __syncthreads();
  }
  auto stands = [&](int mt, int nt, int v) __attribute__((always_inline)) {
    const float x = __builtin_fabsf(acc[mt][nt][v]);
    float least = 0.0f;
    if (scan) {
      const int row = (wm * kMT + mt) * 32 + 8 * (v >> 2) + 4 * h + (v & 3), col = TM + (wn * kNT + nt) * 32 + r;
      if (stat[TM + TN + row]) least += __builtin_bit_cast(float, stat[col]);
      if (stat[TM + TN + col]) least += __builtin_bit_cast(float, stat[row]);
      least *= (float)K * kLost;
    }
    return x <= __FLT_MAX__ && !(x < least);
  };
  uint32_t bad[kMT][kNT] = {};  // per 32×32 block: the lane's sums that do not stand
  if (group == 0) {
    float z = 0.0f;  // stays zero where every sum is finite (x - x is not otherwise)
#pragma unroll
    for (int i = 0; i < kMT * kNT * 16; ++i) {
      const float x = acc[i / 16 / kNT][i / 16 % kNT][i % 16];
      z += x - x;
    }
    if (scan || early || !(z == 0.0f)) {
      uint32_t any = 0;
#pragma unroll
      for (int i = 0; i < kMT * kNT * 16; ++i) {
        const int mt = i / 16 / kNT, nt = i / 16 % kNT, v = i % 16;
        bad[mt][nt] |= (early || !stands(mt, nt, v) ? 1u : 0u) << v;
        any |= bad[mt][nt];
      }
      if (any != 0) s_redo = 1;
    }
  }
  __syncthreads();
  const bool redo = __builtin_amdgcn_readfirstlane(s_redo) != 0;
  // acc[mt][nt][v] holds C[row][col], row = 8*(v/4) + 4*h + v%4, col = r (within the 32×32 tile).
  // Only the columns of this tile's own place are stored; `again`: only the sums formed again.
  const bool whole = m0 + TM <= M && n0 + TN <= N && n0 == tc.tn * TN;
  auto store = [&](auto again) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        const int col = n0 + (wn * kNT + nt) * 32 + r;
        const bool cok = col < N && col >= tc.tn * TN;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = m0 + (wm * kMT + mt) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
          if ((whole || (cok && row < M)) && (!again || (bad[mt][nt] >> v & 1u))) C[(size_t)row * N + col] = acc[mt][nt][v];
        }
      }
  };
  if (group == 0 && !early) store(std::false_type{});
  if (!redo || group > 0) return;
  uint32_t need = 0;
#pragma unroll
  for (int i = 0; i < kMT * kNT; ++i) need |= __any(bad[i / kNT][i % kNT] != 0) ? 1u << i : 0u;
  need = (uint32_t)__builtin_amdgcn_readfirstlane((int)need);
  if (need == 0) return;
  f32_blocks_direct<kMT, kNT>(A, B, M, N, K, m0 + wm * kMT * 32, n0 + wn * kNT * 32, lane, need, acc);
  store(std::true_type{});
}

// Round-to-nearest-even fp32 -> bf16 (quiet NaN kept NaN).
__global__ __launch_bounds__(256) void f32_to_bf16_kernel(const float* __restrict__ x, unsigned short* __restrict__ y,
                                                          int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    uint32_t u = __builtin_bit_cast(uint32_t, x[i]);
    unsigned short h;
    if ((u & 0x7fffffffu) > 0x7f800000u) {
      h = (unsigned short)((u >> 16) | 0x0040u);
    } else {
      u += 0x7fffu + ((u >> 16) & 1u);
      h = (unsigned short)(u >> 16);
    }
    y[i] = h;
  }
}

dim3 tile_grid(int tiles_m, int tiles_n, int threads) {
  const dc::GemmGrid g = dc::gemm_grid((int64_t)tiles_m * tiles_n, threads);
  return dim3((unsigned)g.x, (unsigned)g.rows);
}

template <int TM, int TN, int WM, int WN, int KS, bool kDma>
void launch_bf16(dc_hip_ctx* ctx, const unsigned short* a, const unsigned short* b, float* c, int64_t m, int64_t n,
                 int64_t k) {
  constexpr int kThr = 64 * WM * WN * KS;
  const int tiles_m = (int)((m + TM - 1) / TM), tiles_n = (int)((n + TN - 1) / TN);
  gemm_bf16_kernel<TM, TN, WM, WN, KS, kDma><<<tile_grid(tiles_m, tiles_n, kThr), kThr, 0, ctx->stream>>>(
      a, b, c, (int)m, (int)n, (int)k, tiles_m, tiles_n);
}

template <int TM, int TN, int WM, int WN, int KS, int D>
void launch_split(dc_hip_ctx* ctx, const float* a, const float* b, float* c, int64_t m, int64_t n, int64_t k) {
  constexpr int kThr = 64 * WM * WN * KS;
  const int tiles_m = (int)((m + TM - 1) / TM), tiles_n = (int)((n + TN - 1) / TN);
  gemm_f32_split_kernel<TM, TN, WM, WN, KS, D><<<tile_grid(tiles_m, tiles_n, kThr), kThr, 0, ctx->stream>>>(
      a, b, c, (int)m, (int)n, (int)k, tiles_m, tiles_n);
}

int32_t check_dims(int64_t m, int64_t n, int64_t k) {
  if (m < 0 || n < 0 || k < 0) return DC_ERR_INVALID_ARGUMENT;
  if (m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2) return DC_ERR_INVALID_ARGUMENT;
  return DC_OK;
}

}  // namespace

extern "C" {

DC_HIP_API int32_t dc_hip_gemm_f32(dc_hip_ctx* ctx, const float* a, const float* b, float* c, int64_t m, int64_t n,
                                   int64_t k) {
  DC_RETURN_IF(check_dims(m, n, k));
  if (m == 0 || n == 0) return ctx ? DC_OK : DC_ERR_INVALID_ARGUMENT;
  if (!c || (k > 0 && (!a || !b))) return DC_ERR_INVALID_ARGUMENT;
  DC_CTX_ENTER(ctx);
  if (k == 0) return dc::zero_async(ctx, c, (size_t)(m * n) * sizeof(float));
  const int tiles_m = (int)((m + kT32 - 1) / kT32), tiles_n = (int)((n + kT32 - 1) / kT32);
  switch (dc::f32_gemm_kernel(m, n, k, dc::aligned16(a) && dc::aligned16(b), std::max(1, ctx->cu_count))) {
    case dc::F32Gemm::kDma64:
      gemm_f32_dma_kernel<<<tile_grid(tiles_m, tiles_n, kThreads), kThreads, 0, ctx->stream>>>(a, b, c, (int)n, (int)k,
                                                                                               tiles_m, tiles_n);
      break;
    case dc::F32Gemm::kChecked64:
      gemm_f32_kernel<<<tile_grid(tiles_m, tiles_n, kThreads), kThreads, 0, ctx->stream>>>(
          a, b, c, (int)m, (int)n, (int)k, tiles_m, tiles_n);
      break;
    case dc::F32Gemm::kSplit256x128: launch_split<256, 128, 4, 2, 1, 1>(ctx, a, b, c, m, n, k); break;
    case dc::F32Gemm::kSplit128: launch_split<128, 128, 2, 2, 1, 1>(ctx, a, b, c, m, n, k); break;
    case dc::F32Gemm::kSplit128x2: launch_split<128, 128, 2, 2, 2, 2>(ctx, a, b, c, m, n, k); break;
    case dc::F32Gemm::kSplit64: launch_split<64, 64, 2, 2, 1, 2>(ctx, a, b, c, m, n, k); break;
    case dc::F32Gemm::kSplit64x2: launch_split<64, 64, 2, 2, 2, 2>(ctx, a, b, c, m, n, k); break;
    case dc::F32Gemm::kSplit64x4: launch_split<64, 64, 2, 2, 4, 2>(ctx, a, b, c, m, n, k); break;
  }
  return dc::last_launch_status();
}

DC_HIP_API int32_t dc_hip_gemm_bf16(dc_hip_ctx* ctx, const uint16_t* a, const uint16_t* b, float* c, int64_t m,
                                    int64_t n, int64_t k) {
  DC_RETURN_IF(check_dims(m, n, k));
  if (m == 0 || n == 0) return ctx ? DC_OK : DC_ERR_INVALID_ARGUMENT;
  if (!c || (k > 0 && (!a || !b))) return DC_ERR_INVALID_ARGUMENT;
  DC_CTX_ENTER(ctx);
  if (k == 0) return dc::zero_async(ctx, c, (size_t)(m * n) * sizeof(float));
  const unsigned short* A = reinterpret_cast<const unsigned short*>(a);
  const unsigned short* B = reinterpret_cast<const unsigned short*>(b);
  using dc::Bf16Gemm;
  switch (dc::bf16_gemm_kernel(m, n, k, dc::aligned16(a) && dc::aligned16(b), std::max(1, ctx->cu_count))) {
    case Bf16Gemm::kDma256: launch_bf16<256, 256, 2, 4, 1, true>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kDma128: launch_bf16<128, 128, 2, 2, 1, true>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kDma128x2: launch_bf16<128, 128, 2, 2, 2, true>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kDma64: launch_bf16<64, 64, 2, 2, 1, true>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kDma64x2: launch_bf16<64, 64, 2, 2, 2, true>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kDma64x4: launch_bf16<64, 64, 2, 2, 4, true>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kReg128: launch_bf16<128, 128, 2, 2, 1, false>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kReg64: launch_bf16<64, 64, 2, 2, 1, false>(ctx, A, B, c, m, n, k); break;
    case Bf16Gemm::kReg64x4: launch_bf16<64, 64, 2, 2, 4, false>(ctx, A, B, c, m, n, k); break;
  }
  return dc::last_launch_status();
}

DC_HIP_API int32_t dc_hip_convert_f32_to_bf16(dc_hip_ctx* ctx, const float* input, uint16_t* output, int64_t n) {
  if (n < 0 || (n > 0 && (!input || !output))) return DC_ERR_INVALID_ARGUMENT;
  DC_CTX_ENTER(ctx);
  if (n == 0) return DC_OK;
  const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 16384));
  f32_to_bf16_kernel<<<grid, 256, 0, ctx->stream>>>(input, reinterpret_cast<unsigned short*>(output), n);
  return dc::last_launch_status();
}

}  // extern "C"
