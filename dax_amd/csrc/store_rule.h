// Where the quantisers' bytes go, by how many there are.  Plain C++ on purpose: the host-side check in tests/host compiles this file
// without the HIP headers.
#pragma once

#include <stdint.h>

namespace daxq {

// past the caches (non-temporal), into them for the GEMM behind the quantiser, or into them and through the L2 to memory at once (a
// device-coherent store)
enum { kStorePast = 0, kStoreKeep = 1, kStoreThrough = 2 };

// Activations of at most this many quantised bytes are stored where the GEMM finds them again, in the caches (the Infinity Cache
// holds 256 MB), larger ones past them.  Forwards, us, past the caches -> kept: 512 x 5120 x 5120 25.5 -> 22.4, 4096 x 1536 x 1536
// 21.9 -> 19.8, 2900 x 1000 x 3080 fp16 20.4 -> 19.7, 4725 x 5120 x 5120 static e4m3 104.8 -> 102.6, 32760 x 4608, K = 1536 238.6 -> 229.9,
// 75600 x 5120 x 5120 e4m3 1498 -> 1505; converting a weight of 13824 x 5120 37.0 -> 38.3.  (The rows' own loads without the hint as
// well: 512 x 5120 22.2, 4096 x 1536 19.6, but 4725 x 5120 105.2 and 32760 x 1536 234.8.)
constexpr int64_t kKeepBytes = (int64_t)128 << 20;
// Kept bytes that only lie in the L2s are written back when the kernel has ended, and the GEMM waits for that: it starts 1.5 us
// behind the last acknowledged store with nothing to write back, 3.1 us with 2.6 MB (512 x 5120), 4.5 us with 6.3 MB (4096 x 1536).
// Stores through the L2 write while the kernel runs.  Quantiser + GEMM, us, kept / through (rows of one wavefront in ranges):
//   134 x 3472, K = 5120 (0.65 MB) 12.5 / 12.5    17 x 5120 x 5120 e4m3 (0.1) 9.05 / 9.22    64 x 5120 x 5120 (0.3) 12.1 / 12.4
//   512 x 5120 x 5120 (2.5) 22.3 / 22.0    2900 x 3080, K = 1000 (2.8) 19.7 / 19.4    313 x 4608, K = 13824 (4.1) 31.9 / 31.3
//   1024 x 5120 x 5120 e4m3 (5) 29.8 / 29.2    1230 x 2712, K = 5120 (6) 26.5 / 25.8    887 x 5120, K = 8960 e4m3 (7.6) 40.9 / 40.3
// ... in front of GEMMs against a hundred columns either way, by what the quantiser does not know (1 to 8 MB, bf16; fp32):
//   865 x 133, K = 2909 11.8 / 11.9; 12.6 / 12.3    1500 x 133, K = 5120 20.9 / 22.0; 23.7 / 22.8    2000 x 133, K = 1001 7.5 / 7.9; 7.7 / 8.0
//   2500 x 133, K = 2909 15.8 / 14.8; 18.2 / 16.7   600 x 133, K = 5120 13.1 / 12.9; 14.4 / 13.9     4000 x 100, K = 800 13.2 / 13.0; 14.8 / 14.4
// 8 to 32 MB, medians of eleven turns that differ by 0.5 to 3 %, INT8; e4m3: shapes go either way, and the losses are the larger ones
//   1500 x 5120, K = 13824 (21) 91.4 / 94.1; 89.0 / 92.2    1003 x 4608, K = 13824 (14) 62.0 / 63.2; 60.7 / 62.4    600 x 5120, K = 15360 (9) 58.2 / 58.7; 57.9 / 58.5
//   3200 x 1536, K = 8960 (29) 54.0 / 54.6; 53.0 / 55.1    8000 x 5120, K = 1536 (12) 71.1 / 72.4; 70.5 / 71.6    1800 x 5120 x 5120 (9) 47.4 / 47.9; 46.6 / 46.7
//   2225 x 5120, K = 4608 (10) 52.4 / 52.2; 51.5 / 50.9    16000 x 4608, K = 1536 (25) 117.8 / 116.6; 117.3 / 116.9    4725 x 5120 x 5120 (24) 107.6 / 107.2; 105.7 / 104.0
// from 32 MB on
//   4071 x 5120, K = 13824 (54) 216.7 / 216.2  13198 x 1536, K = 5120 (64) 111.8 / 109.2   16034 x 5120, K = 5160 e4m3 (80) 320 / 312
// and past the caches / through, beyond kKeepBytes, up to the Infinity Cache's 256 MB:
//   27000 x 512, K = 5120 (138) 122.0 / 113.6    30000 x 1536, K = 5120 (154) 246.7 / 236.8    20000 x 5120, K = 8960 e4m3 (179) 697 / 688
//   37800 x 13824, K = 5120 (194) 1951 / 1953    18000 x 5120, K = 13824 (249) 985 / 975    32760 x 1536, K = 8960 (294) 438.3 / 435.6
//   75600 x 5120 x 5120 e4m3 (387) 1540 / 1548   INT8 1565 / 1560    75600 x 5120, K = 13824 e4m3 (1045) 3965 / 3972
constexpr int64_t kThroughFrom = (int64_t)1 << 20, kThroughTo = (int64_t)8 << 20, kThroughAgain = (int64_t)32 << 20, kThroughMost = (int64_t)256 << 20;
// aligned: rows of bytes that start on multiples of 8
inline int store_of(int64_t bytes, bool aligned) {
    if (aligned && ((bytes >= kThroughFrom && bytes <= kThroughTo) || (bytes >= kThroughAgain && bytes <= kThroughMost))) return kStoreThrough;
    return bytes > kKeepBytes ? kStorePast : kStoreKeep;
}

// The kernels that fuse a producer and the quantiser: through the L2, where the GEMM behind finds what the caches hold and nothing is left
// to write back when the kernel ends, as long as the bytes are about what the Infinity Cache holds; past the caches beyond.
// A feed-forward (LayerNorm, up, GELU, down) on the GPU alone, us, past the caches / kept in the L2s / through them:
//   256 x 1536 x 8960 e4m3 46.3 / 38.9 / 38.5    512 x 5120 x 13824 INT8 104.3 / 89.0 / 88.6    1600 x 2560 x 4608 INT8 67.8 / 60.0 / 59.0
//   2048 x 1536 x 8960 e4m3 92.3 / 83.7 / 83.5   4095 x 1536 x 8960 INT8 151.8 / 141.6 / 141.3  5000 x 512 x 1024 e4m3 31.8 / 31.0 / 29.2
//   9450 x 5120 x 13824 e4m3 1012 / 1006 / 1004  16380 x 1536 x 8960 e4m3 493 / 486 / 481       32760 x 1536 x 8960 INT8 929 / 921 / 916
// (the smallest loses, 256 x 512 x 1024 14.9 / 14.8 / 15.2; the host takes 107 for such a block)
// The producer alone, two matrices in turn, us a launch, past / through (MB of bytes; INT8, which gains and loses more than e4m3):
//   LayerNorm x 5120  20000 rows (102) 58.1 / 54.2   37800 (194) 106.0 / 93.7   52000 (266) 146.0 / 127.6   60000 (307) 167.7 / 165.4   75600 (387) 213.1 / 222.4
//   GELU x 5000       40000 (205) 105.9 / 105.1   60000 (307) 151.7 / 159.3   75600 (387) 189.6 / 211.2        with the bf16 result, too: level up to 387 MB
//   GELU x 13824      9450 (131) 76.2 / 70.2   16380 (226) 123.9 / 109.6   20000 (276) 149.5 / 132.0   26000 (359) 191.9 / 195.5   37800 (523) 278.3 / 284.2   75600 (1045) 559.8 / 577.8
// In a feed-forward the two are within its own spread from 16380 rows x 5120 x 13824 on (24000 rows, 123 and 332 MB: 2584 / 2575).
constexpr int64_t kFusedThroughMost = (int64_t)280 << 20;
inline bool fused_store_through(int64_t bytes) { return bytes <= kFusedThroughMost; }

}  // namespace daxq
