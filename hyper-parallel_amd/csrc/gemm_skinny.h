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
// [16384, 1920] 10.2 / 8.1, 64 rows of [36864, 512] 9.2 / 8.7; over 5 row counts up to 64, 6 widths from 1024 to 36864 and 4
// contractions from 512 to 1920 a third less on average and nowhere more.  Shorter ones: 16 rows of [4096, 256] 4.9 / 4.9.
constexpr int kSkinnyMinK = 512;

int launch_skinny(const SkinnyParams& p, SkinnyMode mode, int cus, hipStream_t stream);

// a is bf16 (lda bytes between its rows), quantized 1x128 in the kernel; M <= kSkinnyMaxRowsBf16.  sa is not read.
constexpr int kSkinnyMaxRowsBf16 = 8;
int launch_skinny_rows_bf16(const SkinnyParams& p, bool pow2, int cus, hipStream_t stream);

}  // namespace hpfp8
