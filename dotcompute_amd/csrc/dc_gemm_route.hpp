// dc_gemm_route.hpp — which GEMM kernel of dc_gemm.hip takes a shape: pure functions of the sizes, the
// alignment and the number of CUs, checked on the CPU by tests/cpp/host_tests.cpp.
#pragma once

#include <cstdint>

namespace dc {

// The grid of `tiles` workgroups: one row of them, or rows of kGemmGridRow where a single one would have
// more work items than a launch takes in a dimension (2^32 - 1); the last row may be partly empty. (A
// fixed row, so that the kernels need no launch dimensions: those cost 0.2 us a launch.)
constexpr int kGemmGridRowBits = 20;
constexpr int64_t kGemmGridRow = int64_t(1) << kGemmGridRowBits;
struct GemmGrid {
  int64_t x, rows;
};
inline GemmGrid gemm_grid(int64_t tiles, int64_t threads) {
  if (tiles * threads <= (int64_t)UINT32_MAX) return {tiles, 1};
  return {kGemmGridRow, (tiles + kGemmGridRow - 1) >> kGemmGridRowBits};
}

// fp32: "Split": the bf16 matrix cores, by tile (rows x columns) and k groups; the others the fp32
// instructions (Dma64: direct-to-LDS loads of full 64-tiles; Checked64: any shape).
enum class F32Gemm { kDma64, kChecked64, kSplit256x128, kSplit128, kSplit128x2, kSplit64, kSplit64x2, kSplit64x4 };

// Measured, us (256 CUs; the columns are 256x128, 128, 128x2, 64, 64x2, 64x4 split, fp32 Dma64, and the
// kernels on the fp32 instructions that the split ones replaced):
//    8192^3          6027                                            7304
//    4096x4096x1024   199  205  225  255  265  315  246   241     3500x3500x1000  168 185 199 200 209 253   -  486
//    3072x3072x1024   166  141  155  147  152  183  142   183     2560x2560x1024   86  92 100 110 113 139 108  108
//    2048x2048x1024    74   58   58   68   69   83   63    64     1537x2049x1023   73  58  53  65  66  84   -  144
//    1536x1536x1024    72   50   45   46   49   60   48    48     1280x1280x1024   70  50  44  33  33  39  33   33
//     512x8192x8192   547  441  399  514  514  531  503   500     64x8192x8192    519 345 285 141 111 102 137  137
//    1023^3            70   53   44  21.4 21.6 21.5   -    45     512x512x512      39  25  26 12.0 11.5 12.5 10.2 10.3
//    1280x1280x64    12.1  9.3 11.6  7.0  8.7  9.1  5.2   5.4     2048x2048x64   13.3 11.0 13.0 11.3 15.2 16.2 9.0 9.1
//    3072x3072x64    24.9 21.1 32.3 19.6 28.7 32.5 16.1  20.2     8192x8192x64    104 101 161 114 169 184  94    92
//    2048x2048x256   25.7 20.0 21.8 22.6 24.2 37.0 20.2  20.4     4096x4096x256    63  63  83  77  87 142  75    71
//    1799x1911x257   24.6 19.0 20.3 21.1 22.8 33.7   -   47.5     64x100000x256   102  53  75  35  41  68   -   117
inline F32Gemm f32_gemm_kernel(int64_t m, int64_t n, int64_t k, bool aligned16, int64_t cus) {
  auto tiles = [&](int64_t tm, int64_t tn) { return ((m + tm - 1) / tm) * ((n + tn - 1) / tn); };
  const int64_t t64 = tiles(64, 64);
  // The fp32 instructions do full tiles as fast as the split kernels' larger throughput allows where k is
  // too short for those to get going, or the tiles too few to fill the chip with either. (Their buffer
  // ranges, 64 rows of k floats or 32 rows of n, are checked: below 2 GiB.)
  if (m % 64 == 0 && n % 64 == 0 && k % 32 == 0 && aligned16 && 64 * k * 4 < INT32_MAX && 32 * n * 4 < INT32_MAX &&
      (k <= 64 || (k <= 256 && k * t64 <= 1152 * cus) || (k <= 1024 && t64 <= 2 * cus)))
    return F32Gemm::kDma64;
  // The split kernels take whole tiles of columns, two k tiles of 16 per group, and 32-bit element offsets
  // within a tile's panels.
  if (n < 64 || k <= 16 || 256 * k >= INT32_MAX || 16 * n >= INT32_MAX) return F32Gemm::kChecked64;
  if (m > 64 && n >= 128) {
    const int64_t t128 = tiles(128, 128);
    if (t128 > cus) {
      // By rounds of workgroups: one of 256x128 per CU, or two of 128x128, which together take 5 % longer
      // and alone 65 % as long.
      const int64_t rounds256 = (tiles(256, 128) + cus - 1) / cus, rest = t128 % (2 * cus);
      const int64_t cost128 = 105 * (t128 / (2 * cus)) + (rest == 0 ? 0 : rest <= cus ? 65 : 105);
      return k >= 512 && 100 * rounds256 <= cost128 ? F32Gemm::kSplit256x128 : F32Gemm::kSplit128;
    }
    if (2 * t128 > cus && k >= 768) return F32Gemm::kSplit128x2;
    if (4 * t128 > 3 * cus) return F32Gemm::kSplit128;
  }
  if (t64 > cus || k < 256) return F32Gemm::kSplit64;
  return k < 1536 ? F32Gemm::kSplit64x2 : F32Gemm::kSplit64x4;
}

// bf16: "Dma": direct-to-LDS loads, by tile (square) and k groups; "Reg": loads through registers.
enum class Bf16Gemm { kDma256, kDma128, kDma128x2, kDma64, kDma64x2, kDma64x4, kReg128, kReg64, kReg64x4 };

// Bytes that a direct-to-LDS load of the bf16 kernels can be away from its panel's first.
constexpr int32_t kBf16DmaRange = INT32_MAX;

// Measured, us (256 CUs; tiles 256 / 128 / 64, "x2", "x4": that many k groups):
//   3072x3072x1024 (144 tiles of 256): 27.5 / 32.6 / 33.8;  2048x8192x512 (256): 24.1 / 26.5 / 31.4
//   4352x4096x1024 (272): 57.4 / 52.0 / 60.9;  4608x4608x1024 (324): 60.4 / 56.8 / 73.7
//   5120x5120x1024 (400): 63.1 / 69.7 / 86.2;  6144x6144x1024 (576): 94.7 / 93.8 / 121.8
//   8192x8192x64: 54.4 / 46.3 / 46.1;  4096x4096x64: 14.0 / 14.5 / 15.5;  2048x2048x64: 9.6 / 6.8 / 6.0
//   8192x8192x128: 61.7 / 58.6 / 57.5;  4096x4096x128: 15.8 / 16.2 / 17.3;  4352x4096x64: 20.1 / 17.1 / 15.9
//   2000x3000x1000 (96 tiles of 256, 384 of 128): 29.0 / 21.2 / 28.8
//   2048^3 (256 of 128): 45.2 / 28.2 (x2 23.7) / 27.3;  1536^3 (144): 34.6 / 20.3 (x2 17.5) / 15.2
//   256x8192x8192 (512 of 64): 151 / 80 / 61, x2 51.8, x4 66;  1024^3 (256 of 64): 7.4, x2 6.6, x4 6.7
//   64x8192x8192 (128 of 64): 61, x2 43, x4 36;  512x512x4096 (64 of 64): 32, x2 24, x4 20
//   512^3: 4.6, x2 4.4, x4 4.9
// Register loader (128 / 64): 2047^3 42 / 52, 1535^3 33 / 29, 1023^3 21 / 12.4 (x4 11.0),
// 511x511x4095 61 / 48 (x4 32).
inline Bf16Gemm bf16_gemm_kernel(int64_t m, int64_t n, int64_t k, bool aligned16, int64_t cus) {
  auto tiles = [&](int64_t t) { return ((m + t - 1) / t) * ((n + t - 1) / t); };
  const int64_t t256 = tiles(256), t128 = tiles(128), t64 = tiles(64);
  if (n % 8 == 0 && k % 8 == 0 && aligned16) {
    // The widest tile that still gives the chip enough workgroups, but where a second round of the
    // 256-tiles would be mostly empty or k is too short for them; then, where even the small tiles leave
    // CUs idle, a k dimension split over the wave groups of a workgroup.
    struct Choice {
      Bf16Gemm kernel;
      int64_t tile, groups;
    } c;
    const bool brief = (k <= 64 && (t256 > cus || 4 * t256 <= 3 * cus)) || (k <= 128 && t256 > 2 * cus);
    if (2 * t256 > cus && (t256 <= cus || 10 * t256 > 13 * cus) && !brief) c = {Bf16Gemm::kDma256, 256, 1};
    else if (t128 > cus && !brief) c = {Bf16Gemm::kDma128, 128, 1};
    else if (4 * t128 > 3 * cus && k > 128) c = {Bf16Gemm::kDma128x2, 128, 2};
    else if (t64 > 2 * cus || k < 512) c = {Bf16Gemm::kDma64, 64, 1};
    else if (2 * t64 > cus || k < 2048) c = {Bf16Gemm::kDma64x2, 64, 2};
    else c = {Bf16Gemm::kDma64x4, 64, 4};
    // Every byte offset inside the buffer range: of the tile's rows of A, and of B's rows with those past
    // the last that the groups' k tiles ask for (zeros). Larger shapes go through registers.
    const int64_t rows = (k + 64 * c.groups - 1) / (64 * c.groups) * (64 * c.groups);
    if (c.tile * k * 2 < kBf16DmaRange && rows * n * 2 < kBf16DmaRange) return c.kernel;
  }
  if (n >= 128 && 4 * t128 > 3 * cus) return Bf16Gemm::kReg128;
  return t64 > cus || k < 1000 ? Bf16Gemm::kReg64 : Bf16Gemm::kReg64x4;
}

}  // namespace dc
