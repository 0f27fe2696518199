// Scaled FP8 GEMMs with few rows of a: c[m, n] = sum_kb sa(m, kb) * sb(n, kb) * (A_kb . B_kb^T), M <= 64 (decode).
//
// Bound by reading b once.  A tile kernel has one workgroup per 128 columns here: 56 of 256 compute units on
// N = 7168, each limited by what its vector-memory path delivers (about 25 bytes per clock).  Here
//   * a unit of work is 32 columns (64 of a wide matrix); one workgroup per compute unit walks a contiguous run of units.
//   * operands go global -> LDS -> registers, each wave through a ring of its own of U k-blocks (no barriers: a wave
//     waits for its own transfers), and the ring runs on across units: while the sums of one are added up, the first
//     k-blocks of the next are under way.  The transfers are there for their shape: one moves 8 rows x 128 bytes, whole
//     cache lines, where loads straight into the matrix instruction's register layout (16 rows x 64 bytes) reach half
//     the rate per compute unit.
//   * each of a workgroup's four waves takes a contiguous quarter of the k-blocks (no wave waits for another before the
//     end) and the four sums meet in LDS, added in wave order: the result differs from a tile kernel's, which adds all
//     k-blocks in one chain, in the last bits of fp32.  (Kept in one chain -- the waves hand their partial products to
//     one another round by round -- 37 rows of [36864, 7168] take 85 us instead of 63.)
//   * a wave begins its quarter at a k-block that depends on the workgroup: begun at the same one, 256 workgroups whose
//     units start a multiple of 16 KB apart ask the same memory channels at the same time (8 rows of [7168, 16384]: 28
//     us, 22 us with it).
//   * a is moved in pieces of 8 rows, so that 37 rows cost 40 and not 48 (27.3 -> 26.4 us on [7168, 16384]).
// Measured (weights rotating beyond the Infinity Cache): 8 rows of [7168, 16384] 60 -> 20 us (5.8 TB/s), of [36864, 7168]
// 80 -> 47 us (5.6 TB/s); from about 24 rows on the vector-memory path of a compute unit, which carries a's rows once per
// unit, is the bound (64 rows of [7168, 16384]: 64 -> 31 us, of [36864, 7168] 65 us).
// Transfers past the end go through an empty resource: they fetch nothing, write zeros and keep the number of
// operations in flight constant, which is what the waits count.  (A result store in between adds to the count, which
// makes a wait stricter, never looser.)
#include "gemm_skinny.h"
#include "gemm_tile.h"
#include "hpfp8_device.h"
#include "hpfp8_host.h"

namespace hpfp8 {

constexpr int kSkinnyWaves = 4;
constexpr int kSkinnyThreads = kSkinnyWaves * 64;
// ME: 8-row pieces of a, one transfer each (M <= 8 ME); NF: 16-column fragments of a unit.
// LDS of one workgroup: the four rings, the partial sums of the fragments added up at a time, the bias of the workgroup's
// columns.  U k-blocks per ring: what 160 KB have room for, and at most 6 (more in flight gains nothing).
constexpr int kSkinnyBiasBytes = kSkinnyMaxCols * 2;
constexpr int skinny_frags(int me, int nf) { return nf * ((me + 1) / 2); }
constexpr int skinny_sum_frags(int me, int nf) {      // fragments summed between two barriers
  const int f = skinny_frags(me, nf);
  return f <= 8 ? f : (f == 12 ? 6 : 4);
}
constexpr int skinny_stage_bytes(int me, int nf) { return (2 * nf + me + me % 2) * 1024 + 256; }
constexpr int skinny_sum_bytes(int me, int nf) { return kSkinnyWaves * skinny_sum_frags(me, nf) * 1024; }
constexpr int skinny_stages(int me, int nf) {
  const int fit = (160 * 1024 - skinny_sum_bytes(me, nf) - kSkinnyBiasBytes) / (kSkinnyWaves * skinny_stage_bytes(me, nf));
  return fit > 6 ? 6 : fit;
}
constexpr int skinny_lds_bytes(int me, int nf) {
  return kSkinnyWaves * skinny_stages(me, nf) * skinny_stage_bytes(me, nf) + skinny_sum_bytes(me, nf) + kSkinnyBiasBytes;
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

// (Rows of a fragment past the last piece hold what the LDS held: a row of the product depends on its own row of a alone.)
template <bool TENSOR, bool OUT_F32, int ME, int NF>
__global__ __launch_bounds__(kSkinnyThreads) void gemm_skinny_kernel(const SkinnyParams p) {
  constexpr int MF = (ME + 1) / 2;                              // 16-row fragments of a
  constexpr int U = skinny_stages(ME, NF);
  constexpr int kCols = 16 * NF;
  constexpr int kStage = skinny_stage_bytes(ME, NF);            // one k-block: b's rows, a's rows, a's scales
  constexpr int kOps = 2 * NF + ME + (TENSOR ? 0 : 1);          // transfers of one k-block
  constexpr int kLeft = (U - 1) * kOps;                         // in flight behind the oldest k-block
  static_assert(U >= 2 && kLeft <= 63, "the wait counter holds 63");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[skinny_lds_bytes(ME, NF)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int kblocks = p.K >> 7;
  const int steps = (kblocks + kSkinnyWaves - 1) / kSkinnyWaves;
  uint8_t* const ring = lds + wave * (U * kStage);
  v4f* const red = reinterpret_cast<v4f*>(lds + kSkinnyWaves * U * kStage);      // [wave][fragment][lane]
  uint16_t* const bias_lds = reinterpret_cast<uint16_t*>(lds + kSkinnyWaves * U * kStage + skinny_sum_bytes(ME, NF));

  // this workgroup's units: a contiguous run
  const int units = p.N / kCols, base = units / (int)gridDim.x, more = units % (int)gridDim.x;
  const int wg = blockIdx.x;
  const int unit0 = wg * base + (wg < more ? wg : more), count = base + (wg < more ? 1 : 0);
  if (p.bias)
    for (int i = tid; i < count * kCols; i += kSkinnyThreads) bias_lds[i] = p.bias[unit0 * kCols + i];

  // a transfer moves 8 rows; lane i delivers to the i-th 16 bytes and fetches the chunk whose swizzled home that is
  uint32_t b_off[2 * NF], a_off[ME];
#pragma unroll
  for (int i = 0; i < 2 * NF; ++i) {
    const int r = i * 8 + (lane >> 3);
    b_off[i] = (uint32_t)r * (uint32_t)p.ldb + ((lane & 7) ^ row_swizzle(r)) * 16;
  }
#pragma unroll
  for (int i = 0; i < ME; ++i) {
    const int r = i * 8 + (lane >> 3);
    a_off[i] = (uint32_t)(r < p.M ? r : p.M - 1) * (uint32_t)p.lda + ((lane & 7) ^ row_swizzle(r)) * 16;
  }
  const uint32_t sa_off = (uint32_t)(lane < p.M ? lane : p.M - 1) * (uint32_t)p.sa_sm * 4u;
  const int a_bytes = (int)((p.M - 1) * p.lda + p.K), b_bytes = (int)((kCols - 1) * p.ldb + p.K);
  const int sa_bytes = TENSOR ? 0 : (int)(((p.M - 1) * p.sa_sm + (kblocks - 1) * p.sa_sk + 1) * 4);
  const int rot = (int)((blockIdx.x >> 3) * 5u % (unsigned)steps);

  // the k-block a wave touches in its t-th step on a unit (past the end of the contraction: kblocks)
  auto kb_of = [&](int t) {
    int r = t + rot;
    if (r >= steps) r -= steps;
    const int kb = wave * steps + r;
    return kb < kblocks ? kb : kblocks;
  };
  int l_t = 0, l_unit = 0, l_slot = 0;          // the next step to fetch: step of the unit, unit of the run, ring slot
  auto fetch = [&]() {
    const int kb = kb_of(l_t);
    const bool ok = l_unit < count && kb < kblocks;
    const uint8_t* const b0 = p.b + (int64_t)((unit0 + (ok ? l_unit : 0)) * kCols) * p.ldb;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)b0, 0, ok ? b_bytes : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.a, 0, ok ? a_bytes : 0, 0x00020000);
    const int off = ok ? kb * BK : 0;           // (an empty resource with no offset: out of range in any lane)
    uint8_t* const dst = ring + l_slot * kStage;
#pragma unroll
    for (int i = 0; i < 2 * NF; ++i) transfer_1k<true>(rb, dst + i * 1024, b_off[i], off);
#pragma unroll
    for (int i = 0; i < ME; ++i) transfer_1k<false>(ra, dst + NF * 2048 + i * 1024, a_off[i], off);
    if (!TENSOR) {
      const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc((void*)p.sa, 0, ok ? sa_bytes : 0, 0x00020000);
      transfer_256(rsa, dst + (NF + MF) * 2048, sa_off, ok ? (int)(kb * p.sa_sk * 4) : 0);
    }
    l_slot = l_slot + 1 == U ? 0 : l_slot + 1;
    if (++l_t == steps) {
      l_t = 0;
      ++l_unit;
    }
  };
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  constexpr int F = NF * MF;
  v4f acc[F];
#pragma unroll
  for (int i = 0; i < F; ++i) acc[i] = zero;
  const int pc0 = (2 * g) ^ row_swizzle(l16);
  float tensor_scale = 1.f;
  if (TENSOR) tensor_scale = p.sa[0] * p.sb[0];
  __syncthreads();                              // the bias is there (and no load but the transfers is in flight)
  for (int u = 0; u < U; ++u) fetch();

  int slot = 0;
  for (int unit = 0; unit < count; ++unit) {
    const int n0 = (unit0 + unit) * kCols;
    // (a scalar load: the scale of the unit's 128-row block of b)
    typedef const __attribute__((address_space(4))) float* const_f32_t;
    const const_f32_t sb_row = (const_f32_t)(uintptr_t)(p.sb + (TENSOR ? 0 : (int64_t)(n0 >> 7) * p.sb_sn));
    for (int t = 0; t < steps; ++t) {
      const int kb = kb_of(t);
      const float sb = TENSOR ? 1.f : sb_row[(int64_t)(kb < kblocks ? kb : 0) * p.sb_sk];
      __builtin_amdgcn_s_waitcnt((kLeft & 15) | ((kLeft >> 4) << 14) | 0x0F70);     // vmcnt(kLeft): this slot has arrived
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t* const src = ring + slot * kStage;
      v8i w[NF], x[MF];
      float sa[MF];
#pragma unroll
      for (int f = 0; f < NF; ++f) w[f] = frag_read(src + l16 * BK + f * 2048, pc0);
#pragma unroll
      for (int j = 0; j < MF; ++j) {
        x[j] = frag_read(src + l16 * BK + (NF + j) * 2048, pc0);
        if (!TENSOR) sa[j] = *reinterpret_cast<const float*>(src + (NF + MF) * 2048 + (j * 16 + l16) * 4);
      }
#pragma unroll
      for (int j = 0; j < MF; ++j) {
        const float s = TENSOR ? 1.f : sa[j] * sb;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const int i = f * MF + j;
          if (TENSOR) {
            acc[i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[f], x[j], acc[i], 0, 0, 0, 0, 0, 0);
          } else {
            const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[f], x[j], zero, 0, 0, 0, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][r] = __builtin_fmaf(part[r], s, acc[i][r]);
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // the slot has been read: it may be refilled
      __builtin_amdgcn_sched_barrier(0);
      fetch();
      slot = slot + 1 == U ? 0 : slot + 1;
    }
    // the unit's sums: every wave puts down its own, then each fragment is added up by one wave
    constexpr int G = skinny_sum_frags(ME, NF);
    static_assert(F % G == 0, "whole groups of fragments");
#pragma unroll
    for (int i0 = 0; i0 < F; i0 += G) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        red[(wave * G + i) * 64 + lane] = acc[i0 + i];
        acc[i0 + i] = zero;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");     // (not __syncthreads, which waits for the transfers)
      for (int i = wave; i < G; i += kSkinnyWaves) {
        v4f s = red[i * 64 + lane];
#pragma unroll
        for (int v = 1; v < kSkinnyWaves; ++v) s += red[(v * G + i) * 64 + lane];
        if (TENSOR) s *= tensor_scale;
        const int f = (i0 + i) / MF, j = (i0 + i) % MF, row = j * 16 + l16, col = f * 16 + g * 4;
        if (p.bias) {
          const uint2 braw = *reinterpret_cast<const uint2*>(bias_lds + unit * kCols + col);
          s[0] += bf16lo(braw.x); s[1] += bf16hi(braw.x); s[2] += bf16lo(braw.y); s[3] += bf16hi(braw.y);
        }
        if (row < p.M) {
          const int64_t o = (int64_t)row * p.ldc + n0 + col;
          if (OUT_F32) *reinterpret_cast<v4f*>(reinterpret_cast<float*>(p.c) + o) = s;
          else *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(p.c) + o) = u32x2{pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");     // the sums have been read
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // the empty transfers still write to this workgroup's LDS
}

template <bool TENSOR, bool OUT_F32, int ME>
static void launch_skinny_form(const SkinnyParams& p, int cus, hipStream_t stream) {
  if (p.N >= kSkinnyWide * cus) {
    const int units = p.N / 64;
    gemm_skinny_kernel<TENSOR, OUT_F32, ME, 4><<<dim3((unsigned)(units < cus ? units : cus)), dim3(kSkinnyThreads), 0, stream>>>(p);
  } else {
    const int units = p.N / 32;
    gemm_skinny_kernel<TENSOR, OUT_F32, ME, 2><<<dim3((unsigned)(units < cus ? units : cus)), dim3(kSkinnyThreads), 0, stream>>>(p);
  }
}

template <bool TENSOR, bool OUT_F32>
static void launch_skinny_rows(const SkinnyParams& p, int cus, hipStream_t stream) {
  static_assert(kSkinnyMaxRows == 64, "one form per eight rows");
  switch ((p.M + 7) / 8) {
    case 1: launch_skinny_form<TENSOR, OUT_F32, 1>(p, cus, stream); break;
    case 2: launch_skinny_form<TENSOR, OUT_F32, 2>(p, cus, stream); break;
    case 3: launch_skinny_form<TENSOR, OUT_F32, 3>(p, cus, stream); break;
    case 4: launch_skinny_form<TENSOR, OUT_F32, 4>(p, cus, stream); break;
    case 5: launch_skinny_form<TENSOR, OUT_F32, 5>(p, cus, stream); break;
    case 6: launch_skinny_form<TENSOR, OUT_F32, 6>(p, cus, stream); break;
    case 7: launch_skinny_form<TENSOR, OUT_F32, 7>(p, cus, stream); break;
    default: launch_skinny_form<TENSOR, OUT_F32, 8>(p, cus, stream); break;
  }
}

int launch_skinny(const SkinnyParams& p, bool tensor, bool out_f32, int cus, hipStream_t stream) {
  if (tensor) {
    if (out_f32) launch_skinny_rows<true, true>(p, cus, stream);
    else launch_skinny_rows<true, false>(p, cus, stream);
  } else {
    if (out_f32) launch_skinny_rows<false, true>(p, cus, stream);
    else launch_skinny_rows<false, false>(p, cus, stream);
  }
  return check_launch("gemm (few rows)");
}

}  // namespace hpfp8
