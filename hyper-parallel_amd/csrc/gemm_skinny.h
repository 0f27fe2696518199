// GEMMs with few rows of a (decode): host-side entry of gemm_skinny.hip, used by the dispatch in gemm.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hpfp8 {

// c[m, n] = sum_kb sa(m, kb) * sb(n / 128, kb) * (A_kb . B_kb^T) (+ bias), or with `tensor` one scale each (sa[0], sb[0]).
struct SkinnyParams {
  const uint8_t* a;
  const uint8_t* b;
  const float* sa;
  const float* sb;
  int64_t lda, ldb;       // row strides of a and b in bytes
  int64_t sa_sm, sa_sk;   // element strides of sa over (row, k-block)
  int64_t sb_sn, sb_sk;   // element strides of sb over (128-row block, k-block)
  const uint16_t* bias;
  void* c;
  int64_t ldc;
  int M, N, K;
};

constexpr int kSkinnyMaxRows = 64;
constexpr int kSkinnyMaxCols = 1024;      // columns per compute unit (the bias of a workgroup's columns is kept in LDS)
constexpr int kSkinnyMinK = 2048;         // shorter contractions leave too few k-blocks per wave: the tile kernels
constexpr int kSkinnyWide = 128;          // from this many columns per compute unit on, units are 64 columns wide, which reads a half as often
                                          // (32 / 37 / 64 rows of [36864, 7168]: 55.1 / 59.1 / 74.4 us with 32 columns, 52.9 / 56.5 / 65.4)

int launch_skinny(const SkinnyParams& p, bool tensor, bool out_f32, int cus, hipStream_t stream);

}  // namespace hpfp8
