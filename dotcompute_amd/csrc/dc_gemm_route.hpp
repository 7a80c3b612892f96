// dc_gemm_route.hpp — which GEMM kernel of dc_gemm.hip takes a shape: pure functions of the sizes, the
// alignment and the number of CUs, checked on the CPU by tests/cpp/host_tests.cpp.
#pragma once

#include <cstdint>

namespace dc {

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

}  // namespace dc
