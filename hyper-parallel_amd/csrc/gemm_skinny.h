// GEMMs with few rows of a (decode): host-side entry of gemm_skinny.hip, used by the dispatch in gemm.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hpfp8 {

// c[m, n] = sum_kb sa(m, kb) * sb(n / 128, kb) * (A_kb . B_kb^T) (+ bias); kSkinnyPow2: power-of-two scales, applied by the
// matrix instruction; kSkinnyTensor: one scale each (sa[0], sb[0]).
enum SkinnyMode { kSkinnyBlock, kSkinnyPow2, kSkinnyTensor };

struct SkinnyParams {
  const uint8_t* a;
  const uint8_t* b;
  const float* sa;
  const float* sb;
  int64_t lda, ldb;       // row strides of a and b in bytes
  int64_t sa_sm, sa_sk;   // element strides of sa over (row, k-block)
  int64_t sb_sn, sb_sk;   // element strides of sb over (128-row block, k-block)
  int sb_bytes;           // span of sb
  const uint16_t* bias;
  void* c;
  int64_t ldc;
  int M, N, K;
  int out_f32;
};

constexpr int kSkinnyMaxRows = 64;        // four fragments of 16 rows; one row more takes tiles (64 rows of [7168, 16384]: 27 us here,
                                          // 64 us with the 64 x 128 tiles that 65 rows take)
// Contractions from here on.  Measured, us with tiles / here: 8 rows of [1024, 1024] 6.2 / 3.4, of [4096, 1536] 9.0 / 4.5, 24 rows of
// [16384, 1920] 10.2 / 8.1; shorter ones: 16 rows of [4096, 256] 4.9 / 4.9.  Below kSkinnyAnyWidthK the wider b is the fewer rows: every
// run of columns reads all of a again, for few k-blocks, and one round of 64 x 128 or 128 x 256 tiles is nearly full from 24576 and from
// 49152 columns on.  Geometric means of this form's time over the tiles' for contractions from 512 to 1920, with one b for every call /
// several in turn, over widths up to 16384, up to 24576, up to 32768, up to 98304, beyond (up to 131072):
//    8 rows  0.78 / 0.71   0.88 / 0.80   0.92 / 0.84   0.82 / 0.80   0.88 / 0.82      16 rows  0.78 / 0.70 ... 0.87 / 0.81
//   32 rows  0.78 / 0.70   0.89 / 0.80   0.95 / 0.90   0.86 / 0.85   0.97 / 0.90      64 rows  0.81 / 0.71   0.98 / 0.87   1.15 / 1.07   1.09 / 1.04   1.23 / 1.09
// Of 64 rows [131072, 1024] 25.6 / 38.2 us.
constexpr int kSkinnyMinK = 512, kSkinnyAnyWidthK = 2048;
constexpr int64_t skinny_rows(int64_t N, int64_t K) {
  return K >= kSkinnyAnyWidthK || N <= 24576 ? kSkinnyMaxRows : (N <= 98304 ? 32 : 16);
}

int launch_skinny(const SkinnyParams& p, SkinnyMode mode, int cus, hipStream_t stream);

// a is bf16 (lda bytes between its rows), quantized 1x128 in the kernel; M <= kSkinnyMaxRowsBf16.  sa is not read.
constexpr int kSkinnyMaxRowsBf16 = 8;
int launch_skinny_rows_bf16(const SkinnyParams& p, bool pow2, int cus, hipStream_t stream);

}  // namespace hpfp8
