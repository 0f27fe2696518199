// Scaled FP8 GEMMs with few rows of a: c[m, n] = sum_kb sa(m, kb) * sb(n, kb) * (A_kb . B_kb^T), M <= 64 (decode).
//
// Bound by reading b once.  A tile kernel has one workgroup per 128 columns here: 56 of 256 compute units on
// N = 7168, each limited by what its vector-memory path delivers (about 25 bytes per clock).  Here
//   * a workgroup has F 16-column fragments at a time, as many as give every compute unit its columns in few runs
//     (skinny_fragments has the rule), and a's rows travel once per run.
//   * four waves fetch, four multiply.  Operands go global -> LDS -> registers through a ring of stages of KS k-blocks
//     that runs on across the runs of columns; one barrier per stage says that the stage has arrived and that the one
//     before has been read, whose slot is refilled.  (With four waves doing both in turn the issue of the transfers and
//     the multiplication add up: 8 rows of [36864, 7168] 59 us, 41 with them apart.)  The transfers are there for their
//     shape: one moves 8 rows x 128 bytes, whole cache lines, where loads straight into the matrix instruction's
//     register layout (16 rows x 64 bytes) reach half the rate per compute unit.
//   * the waves share the matrix work by fragments of the result, never by k-blocks: a sum runs over the k-blocks in
//     their order in one chain with the matrix instruction, scales and roundings of the tile kernels, so an element of c
//     has the same bits here and there -- whatever the number of rows, the column it stands in, the width of b (a column
//     shard) and the number of compute units.
//   * all workgroups walk through k in step, so with rows a power of two apart they ask few memory channels at a time.
//     Two things spread that: an XCD's workgroups have neighbouring columns (8 rows of [7168, 16384] 26.4 -> 21.7 us, of
//     [8192, 8192] 19.8 -> 13.6), and a stage is as many k-blocks as LDS has three of (8 rather than 4 k-blocks on
//     [7168, 16384]: 21.4 -> 20.4 us; 4 rather than 2 for 64 rows of it: 31.7 -> 26.8).
//   * a is moved in pieces of 8 rows, so that 37 rows cost 40 and not 48.
// Measured (weights rotating beyond the Infinity Cache): 8 rows of [7168, 16384] 20.6 us (5.7 TB/s), of [36864, 7168] 39.5
// us (6.7 TB/s); 37 rows of the latter 41.6, 64 rows 44.0.  64 rows of [7168, 16384] 26.8 us: a's rows are then two
// thirds of what passes a compute unit's vector-memory path.
// QUANT, up to 8 rows: a is the bf16 source.  Its quantizer would be a launch of 3.5 us that reads what fits in a corner of one XCD's
// L2; here every workgroup quantizes all of it, k-block by k-block as it arrives, in waves of their own (a k-block of a stage each, while
// the stage before is multiplied), for 1 KB more per k-block on the vector-memory path.  That leaves no room for wider forms than 3
// fragments; with the multiplying waves quantizing as well the two chains add up ([7168, 16384] 25.4 us).  us, 8 rows, quantizer and
// product / this: [7168, 16384] 23.3 / 21.5, [36864, 7168] 41.4 / 38.8, [7168, 7168] 12.4 / 11.3, [16384, 16384] 45.2 / 42.9,
// [10240, 5120] 13.2 / 11.1, [4096, 1536] 6.5 / 4.9, [1024, 1024] 5.4 / 3.8, 1 row alike; hpfp8_linear_few_rows has the exceptions.
// Transfers past the end go through an empty resource (with no scalar offset: out of range in any lane): they fetch
// nothing, write zeros and keep the number of operations in flight constant, which is what the waits count.
#include "gemm_skinny.h"
#include "gemm_tile.h"
#include "hpfp8_device.h"
#include "hpfp8_host.h"

namespace hpfp8 {

constexpr int kSkinnyWaves = 4;                         // so many fetch, so many multiply
// ME: 8-row pieces of a, one transfer each (M <= 8 ME); F: 16-column fragments of a workgroup.
// A stage: KS k-blocks, each b's rows, a's rows, the scales of a's rows (64) and of the fragments.
// QUANT: a comes as bf16, 8 rows of it in two transfers (ME = 2), and is quantized here.
constexpr int skinny_kstep(int me, int f, bool quant = false) { return quant ? (f == 1 ? 8 : 4) : (2 * f + me <= 6 ? 8 : (2 * f + me <= 12 ? 4 : 2)); }
// (QUANT: one wave more per k-block of a stage)
constexpr int skinny_threads(int f, bool quant) { return (2 * kSkinnyWaves + (quant ? skinny_kstep(2, f, true) : 0)) * 64; }
constexpr int skinny_block_bytes(int me, int f) { return (2 * f + me) * 1024 + 512; }
constexpr int skinny_stage_bytes(int me, int f, bool quant = false) { return skinny_kstep(me, f, quant) * skinny_block_bytes(me, f); }
constexpr int kSkinnySpare = 1024;       // behind the ring: where a transfer without a piece of its own goes
constexpr int skinny_stages(int me, int f, bool quant = false) {
  const int fit = (160 * 1024 - kSkinnySpare) / skinny_stage_bytes(me, f, quant);
  return fit > 8 ? 8 : fit;
}

// one wave's transfer global -> LDS: lane i's 16 bytes (at its own offset) go to dst + 16 i; NT: streamed, read once
template <bool NT>
__device__ __forceinline__ void transfer_1k(__amdgpu_buffer_rsrc_t rs, uint8_t* dst, uint32_t lane_off, int off);
template <>
__device__ __forceinline__ void transfer_1k<false>(__amdgpu_buffer_rsrc_t rs, uint8_t* dst, uint32_t lane_off, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, lane_off, off, 0, 0);
}
template <>
__device__ __forceinline__ void transfer_1k<true>(__amdgpu_buffer_rsrc_t rs, uint8_t* dst, uint32_t lane_off, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, lane_off, off, 0, 2);
}
// the same with 4 bytes per lane
__device__ __forceinline__ void transfer_256(__amdgpu_buffer_rsrc_t rs, uint8_t* dst, uint32_t lane_off, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 4, lane_off, off, 0, 0);
}

// One k-block of 8 rows, bf16 [8][128] in LDS -> its codes, in the image of an operand tile, over the first half of them, and its
// scales: quant_1x128_kmajor_kernel's arithmetic.  One wave does it, so every lane has read before one writes.  Lane 8 r + p has
// the values 8 p .. and 64 + 8 p .. of row r (odd rows the latter first, so that two rows read from different banks).
__device__ __forceinline__ void quantize_k_block(uint8_t* rows, float* scales, int lane, int pow2) {
  const int r = lane >> 3, p = lane & 7;
  const int part[2] = {p + (r & 1) * 8, p + 8 - (r & 1) * 8};
  uint4 v[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) v[i] = *reinterpret_cast<const uint4*>(rows + r * 256 + part[i] * 16);
  uint32_t m = umax(mag8(v[0]), mag8(v[1]));
  m = umax(m, dpp_u32<kDppQuadXor1>(m));
  m = umax(m, dpp_u32<kDppQuadXor2>(m));
  m = umax(m, dpp_u32<kDppRowHalfMirror>(m));
  float scale, scale_inv;
  scales_from_amax(__uint_as_float(m << 16), scale, scale_inv, pow2);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    *reinterpret_cast<uint2*>(rows + r * BK + ((part[i] >> 1) ^ row_swizzle(r)) * 16 + (part[i] & 1) * 8) = cvt8<false>(v[i], scale);
  if (p == 0) scales[r] = scale_inv;
}

// (Rows of a fragment past the last piece hold what lies behind it in the LDS: a row of the product depends on its own
// row of a alone, and rows past M are not stored.)
template <int MODE, int ME, int F, bool QUANT = false>
__global__ __launch_bounds__(skinny_threads(F, QUANT)) void gemm_skinny_kernel(const SkinnyParams p, int units) {
  static_assert(!QUANT || (ME == 2 && MODE != kSkinnyTensor), "eight rows of bf16, scales of their own");
  constexpr int MF = (ME + 1) / 2;                              // 16-row fragments of a
  constexpr int KS = skinny_kstep(ME, F, QUANT), U = skinny_stages(ME, F, QUANT);
  constexpr int kBlockBytes = skinny_block_bytes(ME, F), kStage = skinny_stage_bytes(ME, F, QUANT);
  constexpr int kA = 2 * F * 1024, kScales = (2 * F + ME) * 1024;     // a's rows and the scales inside a k-block's bytes
  constexpr int kCols = 16 * F;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[U * kStage + kSkinnySpare];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int kblocks = p.K >> 7;
  const int stages = (kblocks + KS - 1) / KS;                   // of one unit (a run of kCols columns)
  // this workgroup's units: first, first + step, ..; the workgroups of an XCD (ids congruent mod 8) have neighbouring ones
  const int step = gridDim.x, xcd = blockIdx.x % kXcds;
  const int first = xcd * (step / kXcds) + (xcd < step % kXcds ? xcd : step % kXcds) + blockIdx.x / kXcds;

  if (wave < kSkinnyWaves) {
    // ---- fetching.  A transfer moves 8 rows; lane i delivers to the i-th 16 bytes and fetches the chunk whose swizzled
    // home that is.  Offsets inside a resource: rows per lane, the k-block (less than a row) scalar.
    constexpr int KW = KS > kSkinnyWaves ? KS / kSkinnyWaves : 1;       // k-blocks a wave fetches per stage
    constexpr int W = KS < kSkinnyWaves ? kSkinnyWaves / KS : 1;        // waves that fetch one k-block together
    constexpr int NBP = (2 * F + W - 1) / W, NAP = (ME + W - 1) / W;    // a wave's transfers of b and of a per k-block
    constexpr int kScaleOps = MODE == kSkinnyTensor ? 0 : (W == 1 && !QUANT ? 2 : 1);
    constexpr int kStageOps = KW * (NBP + NAP + kScaleOps);
    constexpr int kLeft = (U - (QUANT ? 3 : 2)) * kStageOps;            // in flight behind the oldest stage that has to be there
    static_assert(U >= 3 && kLeft <= 63 && (U - 2) * kStageOps <= 63, "the wait counter holds 63");
    static_assert(!QUANT || (W == 1 && U >= 4), "a stage is quantized while the one before is multiplied");
    static_assert(W <= 2, "every wave of a k-block has scales to fetch");
    const int h = wave % W, kb0 = wave / W * KW;
    uint32_t b_off[NBP], a_off[NAP];
#pragma unroll
    for (int i = 0; i < NBP; ++i) {
      const int r = (i * W + h) * 8 + (lane >> 3);
      b_off[i] = (uint32_t)r * (uint32_t)p.ldb + ((lane & 7) ^ row_swizzle(r)) * 16;
    }
#pragma unroll
    for (int i = 0; i < NAP; ++i) {                             // (rows past M lie past the end of the resource)
      const int r = (i * W + h) * 8 + (lane >> 3);
      a_off[i] = QUANT ? (uint32_t)(i * 4 + (lane >> 4)) * (uint32_t)p.lda + (lane & 15) * 16       // 4 rows x 256 bytes
                       : (uint32_t)r * (uint32_t)p.lda + ((lane & 7) ^ row_swizzle(r)) * 16;
    }
    const uint32_t sa_off = (uint32_t)(lane < p.M ? lane : p.M - 1) * (uint32_t)p.sa_sm * 4u;
    const int a_bytes = (int)((p.M - 1) * p.lda + (QUANT ? 2 * p.K : p.K));
    const int sa_bytes = MODE == kSkinnyTensor || QUANT ? 0 : (int)(((p.M - 1) * p.sa_sm + (kblocks - 1) * p.sa_sk + 1) * 4);
    const int sa_step = (int)p.sa_sk * 4, sb_step = (int)p.sb_sk * 4;
    int unit = first, kb = kb0, slot = 0;                       // the next stage to fetch
    const uint8_t* b0;
    int b_bytes;
    uint32_t sb_off;
    auto enter = [&]() {                                        // the unit's part of b (past the last unit: nothing)
      const int n0 = unit < units ? unit * kCols : 0;
      const int rows = p.N - n0 < kCols ? p.N - n0 : kCols;
      b0 = p.b + (int64_t)n0 * p.ldb;
      b_bytes = unit < units ? (int)((rows - 1) * p.ldb + p.K) : 0;
      const int n = n0 + (lane < F ? lane : F - 1) * 16;        // lane i: the scale of fragment i (past the last: of the last)
      sb_off = (uint32_t)((n < p.N ? n : p.N - 1) >> 7) * (uint32_t)p.sb_sn * 4u;
    };
    enter();
    auto fetch = [&]() {
#pragma unroll
      for (int j = 0; j < KW; ++j) {
        const bool ok = kb + j < kblocks && b_bytes != 0;
        const int off = ok ? (kb + j) * BK : 0;
        uint8_t* const dst = lds + slot * kStage + (kb0 + j) * kBlockBytes;
#pragma unroll
        for (int i = 0; i < NBP; ++i) {                         // (2 F is a multiple of W: every wave has as many)
          const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)b0, 0, ok ? b_bytes : 0, 0x00020000);
          transfer_1k<true>(rb, dst + (i * W + h) * 1024, b_off[i], off);
        }
#pragma unroll
        for (int i = 0; i < NAP; ++i) {
          const bool in = ME % W == 0 || i * W + h < ME;
          const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.a, 0, ok && in ? a_bytes : 0, 0x00020000);
          transfer_1k<false>(ra, in ? dst + kA + (i * W + h) * 1024 : lds + U * kStage, a_off[i], in ? (QUANT ? 2 * off : off) : 0);
        }
        if (MODE != kSkinnyTensor) {
          const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc((void*)p.sa, 0, ok ? sa_bytes : 0, 0x00020000);
          const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc((void*)p.sb, 0, ok ? p.sb_bytes : 0, 0x00020000);
          if (h == 0 && !QUANT) transfer_256(rsa, dst + kScales, sa_off, ok ? (kb + j) * sa_step : 0);
          if (h == W - 1) transfer_256(rsb, dst + kScales + 256, sb_off, ok ? (kb + j) * sb_step : 0);
        }
      }
      slot = slot + 1 == U ? 0 : slot + 1;
      kb += KS;
      if (kb - kb0 >= kblocks) {
        kb = kb0;
        unit += step;
        enter();
      }
    };
    for (int u = 0; u < U - 1; ++u) fetch();
    if (QUANT) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((U - 2) * kStageOps) : "memory");     // the first stage has landed
    for (int u = first; u < units; u += step)
      for (int t = 0; t < stages; ++t) {
        // own transfers of this stage (QUANT: of the next one) have landed; then everyone's, and the stage before has been read
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kLeft) : "memory");
        fetch();
      }
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the empty transfers still write to this workgroup's LDS
    return;
  }

  auto sync = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the stage is there; the one before has been read
    __builtin_amdgcn_sched_barrier(0);
  };
  if (QUANT) {
    sync();
    if (wave >= 2 * kSkinnyWaves) {
      // ---- quantizing: a k-block of the next stage, while this one is multiplied.  (Past the last stage zeros: the empty transfers
      // have written them.)
      int slot = 0;
      auto quantize = [&]() {
        uint8_t* const src = lds + slot * kStage + (wave - 2 * kSkinnyWaves) * kBlockBytes;
        quantize_k_block(src + kA, reinterpret_cast<float*>(src + kScales), lane, MODE == kSkinnyPow2);
        slot = slot + 1 == U ? 0 : slot + 1;
      };
      quantize();
      for (int u = first; u < units; u += step)
        for (int t = 0; t < stages; ++t) {
          sync();
          quantize();
        }
      return;
    }
  }

  // ---- multiplying.  WF waves along the fragments of b, WJ along those of a; FW x JW results per wave (the last ones of
  // an uneven split are computed twice and stored once)
  constexpr int WF = F >= 3 ? 4 : F, WJ = kSkinnyWaves / WF;
  constexpr int FW = (F + WF - 1) / WF, JW = (MF + WJ - 1) / WJ;
  const int wf = (wave - kSkinnyWaves) % WF, wj = (wave - kSkinnyWaves) / WF;
  const bool active = wf < F && wj < MF;
  int frag[FW], rows16[JW];                                     // this wave's fragments of b and of a
#pragma unroll
  for (int q = 0; q < FW; ++q) frag[q] = wf + WF * q < F ? wf + WF * q : F - 1;
#pragma unroll
  for (int r = 0; r < JW; ++r) rows16[r] = wj + WJ * r < MF ? wj + WJ * r : MF - 1;
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  v4f acc[FW][JW];
#pragma unroll
  for (int q = 0; q < FW; ++q)
#pragma unroll
    for (int r = 0; r < JW; ++r) acc[q][r] = zero;
  const int pc0 = (2 * g) ^ row_swizzle(l16);
  float tensor_scale = 1.f;
  if (MODE == kSkinnyTensor) tensor_scale = p.sa[0] * p.sb[0];

  // one k-block of a stage: the arithmetic of gemm_kernel, operation for operation
  auto k_block = [&](const uint8_t* src) {
    v8i w[FW], x[JW];
    float sa[JW], sb[FW];
#pragma unroll
    for (int q = 0; q < FW; ++q) {
      w[q] = frag_read(src + frag[q] * 2048 + l16 * BK, pc0);
      if (MODE != kSkinnyTensor) sb[q] = *reinterpret_cast<const float*>(src + kScales + 256 + frag[q] * 4);
    }
#pragma unroll
    for (int r = 0; r < JW; ++r) {
      x[r] = frag_read(src + kA + rows16[r] * 2048 + l16 * BK, pc0);
      if (MODE != kSkinnyTensor) sa[r] = *reinterpret_cast<const float*>(src + kScales + (rows16[r] * 16 + l16) * 4);
    }
#pragma unroll
    for (int q = 0; q < FW; ++q)
#pragma unroll
      for (int r = 0; r < JW; ++r) {
        if (MODE == kSkinnyTensor) {
          acc[q][r] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[q], x[r], acc[q][r], 0, 0, 0, 0, 0, 0);
        } else if (MODE == kSkinnyPow2) {
          acc[q][r] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[q], x[r], acc[q][r], 0, 0, 0,
                                                                      (int)(__builtin_bit_cast(uint32_t, sb[q]) >> 23), 0,
                                                                      (int)(__builtin_bit_cast(uint32_t, sa[r]) >> 23));
        } else {
          const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[q], x[r], zero, 0, 0, 0, 0, 0, 0);
          const float s = sa[r] * sb[q];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[q][r][e] = __builtin_fmaf(part[e], s, acc[q][r][e]);
        }
      }
  };

  int slot = 0;
  for (int unit = first; unit < units; unit += step) {
    for (int t = 0; t < stages; ++t) {
      sync();
      if (active) {
        const uint8_t* const src = lds + slot * kStage;
        if ((t + 1) * KS <= kblocks) {
#pragma unroll
          for (int i = 0; i < KS; ++i) k_block(src + i * kBlockBytes);
        } else {
          for (int i = 0; t * KS + i < kblocks; ++i) k_block(src + i * kBlockBytes);
        }
      }
      slot = slot + 1 == U ? 0 : slot + 1;
    }
    // the unit's results: a lane holds four consecutive columns of one row
    if (!active) continue;
#pragma unroll
    for (int q = 0; q < FW; ++q) {
      const int col = unit * kCols + (wf + WF * q) * 16 + g * 4;
      const bool col_ok = wf + WF * q < F && col < p.N;
      uint2 braw = make_uint2(0, 0);
      if (p.bias && col_ok) braw = *reinterpret_cast<const uint2*>(p.bias + col);
#pragma unroll
      for (int r = 0; r < JW; ++r) {
        v4f s = acc[q][r];
        acc[q][r] = zero;
        const int row = (wj + WJ * r) * 16 + l16;
        if (MODE == kSkinnyTensor) s *= tensor_scale;
        if (p.bias) {
          s[0] += bf16lo(braw.x); s[1] += bf16hi(braw.x); s[2] += bf16lo(braw.y); s[3] += bf16hi(braw.y);
        }
        if (col_ok && row < p.M) {
          const int64_t o = (int64_t)row * p.ldc + col;
          if (p.out_f32) *reinterpret_cast<v4f*>(reinterpret_cast<float*>(p.c) + o) = s;
          else *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(p.c) + o) = u32x2{pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
        }
      }
    }
  }
}

// Fragments per workgroup.  A run costs what is larger, b's part of the memory bandwidth or what passes the compute unit's
// vector-memory path (1.4 : 1 per KB), and 1.4 times that where a stage is fewer than four k-blocks; taken is the form whose
// runs cost least, the narrowest of equals.  Over 10 widths from 4096 to 36864, 4 contractions from 4096 to 16384 and 5 row
// counts this is 0.7 % slower on average than the best of the six forms of each, 14 % at most (24 rows of [18432, 7168]).
// With a short contraction, and with rows quantized here, a run also costs about what three k-blocks of the narrowest form do, and a
// contraction that does not fill its last stage the whole of it.  Contractions from 512 to 1920, 1 to 64 rows and 1024 to 131072
// columns, 12610 sizes: 1.7 % slower than the best form of each on average, without these two terms 3.5 % and up to 78 % ([27008, 896],
// 8 rows: seven runs of one fragment 10.0 us, two of four 6.1); from 2048 on they gain 0.5 % on average and cost some sizes 5 %.
static int skinny_fragments(int64_t N, int64_t K, int me, int cus, bool quant = false) {
  const bool per_run = quant || K < kSkinnyAnyWidthK;
  const int forms[] = {1, 2, 3, 4, 6, 9};
  int best = 0;
  int64_t best_cost = 0;
  for (int f : forms) {
    if (quant && f > 3) break;
    const int64_t units = (N / 16 + f - 1) / f, runs = (units + cus - 1) / cus;
    const int64_t run = 14 * 2 * f > 10 * (2 * f + me) ? 14 * 2 * f : 10 * (2 * f + me);
    const int64_t step = skinny_kstep(me, f, quant), kblocks = per_run ? (K / BK + step - 1) / step * step : K / BK;
    const int64_t cost = runs * (kblocks * run * (step >= 4 ? 10 : 14) + (per_run ? 1000 : 0));
    if (!best || cost < best_cost) {
      best = f;
      best_cost = cost;
    }
  }
  return best;
}

template <int MODE, int ME, int F, bool QUANT = false>
static void launch_skinny_form(const SkinnyParams& p, int cus, hipStream_t stream) {
  const int units = (p.N / 16 + F - 1) / F;
  gemm_skinny_kernel<MODE, ME, F, QUANT><<<dim3((unsigned)(units < cus ? units : cus)), dim3(skinny_threads(F, QUANT)), 0, stream>>>(p, units);
}

template <int MODE, int ME>
static void launch_skinny_cols(const SkinnyParams& p, int cus, hipStream_t stream) {
  switch (skinny_fragments(p.N, p.K, ME, cus)) {
    case 1: launch_skinny_form<MODE, ME, 1>(p, cus, stream); break;
    case 2: launch_skinny_form<MODE, ME, 2>(p, cus, stream); break;
    case 3: launch_skinny_form<MODE, ME, 3>(p, cus, stream); break;
    case 4: launch_skinny_form<MODE, ME, 4>(p, cus, stream); break;
    case 6: launch_skinny_form<MODE, ME, 6>(p, cus, stream); break;
    default: launch_skinny_form<MODE, ME, 9>(p, cus, stream); break;
  }
}

template <int MODE>
static void launch_skinny_rows(const SkinnyParams& p, int cus, hipStream_t stream) {
  static_assert(kSkinnyMaxRows == 64, "one form per eight rows");
  switch ((p.M + 7) / 8) {
    case 1: launch_skinny_cols<MODE, 1>(p, cus, stream); break;
    case 2: launch_skinny_cols<MODE, 2>(p, cus, stream); break;
    case 3: launch_skinny_cols<MODE, 3>(p, cus, stream); break;
    case 4: launch_skinny_cols<MODE, 4>(p, cus, stream); break;
    case 5: launch_skinny_cols<MODE, 5>(p, cus, stream); break;
    case 6: launch_skinny_cols<MODE, 6>(p, cus, stream); break;
    case 7: launch_skinny_cols<MODE, 7>(p, cus, stream); break;
    default: launch_skinny_cols<MODE, 8>(p, cus, stream); break;
  }
}

int launch_skinny(const SkinnyParams& p, SkinnyMode mode, int cus, hipStream_t stream) {
  if (mode == kSkinnyTensor) launch_skinny_rows<kSkinnyTensor>(p, cus, stream);
  else if (mode == kSkinnyPow2) launch_skinny_rows<kSkinnyPow2>(p, cus, stream);
  else launch_skinny_rows<kSkinnyBlock>(p, cus, stream);
  return check_launch("gemm (few rows)");
}

template <int MODE>
static void launch_skinny_bf16(const SkinnyParams& p, int cus, hipStream_t stream) {
  switch (skinny_fragments(p.N, p.K, 2, cus, true)) {
    case 1: launch_skinny_form<MODE, 2, 1, true>(p, cus, stream); break;
    case 2: launch_skinny_form<MODE, 2, 2, true>(p, cus, stream); break;
    default: launch_skinny_form<MODE, 2, 3, true>(p, cus, stream); break;
  }
}

int launch_skinny_rows_bf16(const SkinnyParams& p, bool pow2, int cus, hipStream_t stream) {
  if (pow2) launch_skinny_bf16<kSkinnyPow2>(p, cus, stream);
  else launch_skinny_bf16<kSkinnyBlock>(p, cus, stream);
  return check_launch("linear (few rows)");
}

}  // namespace hpfp8
