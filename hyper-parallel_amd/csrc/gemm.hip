// Scaled FP8 GEMMs for gfx950: c[m,n] = sum_kb sa(m,kb) * sb(n,kb) * (A_kb . B_kb^T).
//
// Layout of the work
//   * Both operands are K-contiguous E4M3 codes, so a 16-row x 128-byte slab of either is exactly
//     one operand of v_mfma_f32_16x16x128_f8f6f4: one matrix instruction consumes one whole
//     128-wide scaling block, and its fp32 result is promoted into the running accumulator with
//     one FMA per element (acc += partial * (sa * sb)).
//   * The weight-like operand b feeds the MFMA "A" port and the activation-like operand a the
//     "B" port: a lane then holds 4 consecutive n for one m, which makes the per-row scale
//     sa(m,kb) a per-lane constant.
//   * Workgroup tile 256(m) x 256(n) x 128(k), 8 waves as 4(m) x 2(n), wave tile 64 x 128
//     (128 fp32 accumulators per lane, 2 waves per SIMD so one wave's FMAs overlap the other's
//     MFMAs).  LDS holds two buffers for the a tile and three for the b tile (32 KB each); tiles
//     are DMA'd global -> LDS with 128-bit buffer loads (out-of-range rows read as zero), 16-byte
//     chunks XOR-swizzled by row so that both the DMA writes and the ds_read_b128 fragment reads
//     are bank-conflict free.
//   * Where a launch would leave compute units idle the tile is smaller: 128 x 256, 128 x 128 or 64 x 128 with four
//     multiplying waves (wave tiles 64 x 128, 64 x 64 and 64 x 32) or 64 x 64 with two, the same template (WM, NS, WN) and the same results bit
//     for bit; pick_shape has the rule and the figures.  There a SIMD has one wave that multiplies, which waits whenever a
//     transfer it issues finds the memory path occupied (78 clocks per transfer while the first k-blocks arrive, 21 later), so
//     four more waves do the transfers, 3, 4, 6 and 8 k-blocks at a time in LDS, the scales with them.  us, transfers by the
//     multiplying waves with two buffers of a / by waves of their own: 1000 x 7168 x 7168 62 / 54, 1531 x 2048 x 7168 41 / 33,
//     500 x 7168 x 16384 106 / 75, by rows 1024 x 1024 x 2048 16.7 / 11.0.  A k-block of one round of these tiles over 7168
//     columns takes 0.83, 0.60, 0.44 and 0.31 us with a weight from HBM (0.76, 0.47, 0.30, 0.22 with one that stays in the
//     caches), of 128 x 256, 128 x 128, 64 x 128 and 64 x 64; its transfers by themselves 0.54 and 0.39 in the first two.  With
//     power-of-two scales, without promotion, it takes as long from HBM (0.84, 0.59, 0.44, 0.31), so what multiplies is not what
//     is waited for there.  A launch's first microsecond or three are code and first tiles arriving through cold caches.
//   * The grid is persistent: one workgroup per CU walks a list of tiles, and the rounds of
//     consecutive tiles follow each other without a gap.  Each XCD (own L2) owns a contiguous run
//     of tile numbers.
//   * Results leave through the wave's own slice of a consumed LDS buffer, regrouped into whole rows of
//     256 bytes, as streaming stores through a buffer resource that ends with the tile's last valid row
//     (rows past the end of a ragged tile or of an expert are dropped by its range check); with
//     accumulate, c's old values are the accumulators' starting values, loaded before the tile's first round.
//   * One kernel template, by scale form: per tensor, 128x128 blocks of b (forward, dgrad), per-row
//     scales on both operands (wgrad), and the two blockwise forms again for scales that are powers of
//     two, which the matrix instruction applies itself (no promotion FMAs); dense, grouped by expert
//     along the rows (MoE forward and dgrad: an expert owns a range of rows of a and c and its own b), or
//     grouped along the contraction (MoE wgrad: an expert owns a range of k-blocks of both operands and
//     its own c); bf16 or fp32 output, optionally added onto what c holds.
#include <atomic>
#include <type_traits>

#include "gemm_skinny.h"
#include "gemm_tile.h"
#include "hpfp8_device.h"
#include "hpfp8_host.h"

namespace hpfp8 {

constexpr int BM = 256, BN = 256;
// LDS: two buffers for the a tile, then kBStages buffers for the b tile.  The b operand is the one
// that streams from HBM (each weight panel is used by one XCD only), so where LDS allows it gets a
// third buffer and its transfers run two k-blocks ahead; a's re-reads come from the Infinity Cache.
__host__ __device__ constexpr int b_stages(int mode) { return mode == 4 /* LDS also holds per-row b scales */ ? 2 : 3; }
constexpr int kRectTiles = 32;              // tiles of the rectangle one XCD (32 CUs) works on at a time

// kScalePow2: scales laid out as for kScaleBlock but every one a power of two; the matrix instruction
// applies them itself (its E8M0 block-scale operands) and accumulates across k-blocks, so there is no
// promotion arithmetic at all.
// kScalePow2Row: the same with the scales laid out as for kScaleRow.
enum ScaleMode { kScaleTensor = 0, kScaleBlock = 1, kScaleRow = 2, kScalePow2 = 3, kScalePow2Row = 4 };

enum Grouping { kDense = 0, kGroupedRows = 1, kGroupedK = 2 };

struct GemmParams {
  const uint8_t* a;
  const uint8_t* b;
  const float* sa;
  const float* sb;
  int64_t sa_sm, sa_sk;   // element strides of sa over (row, k-block)
  int64_t sb_sn, sb_sk;   // element strides of sb over (row or 128-row block, k-block)
  int64_t sb_se;          // grouped by rows: stride of sb between experts
  int64_t b_se;           // grouped by rows: bytes from one expert's b to the next
  int64_t c_se;           // grouped along the contraction: elements from one expert's c to the next
  int sb_bytes;           // size of the sb array in bytes (block form)
  void* c;
  int64_t ldc;
  const uint16_t* bias;
  const int32_t* offs;    // grouped by rows: inclusive prefix sums of rows per expert
  const int32_t* layout;  // grouped along the contraction: the table of grouped.hip
  int experts;
  int64_t lda, ldb;       // row strides of a and b in bytes (>= K)
  int M, N, K;            // M = total rows of a; grouped along the contraction: K = the padded token axis
  int tiles;              // dense: number of output tiles; grouped along the contraction: per expert
  int accumulate;
  // SwiGLU epilogue: b = W_gate_up codes [2 * inter, K] (gate rows first), N = 2 * inter; c = codes of the
  // activation [M, inter] (row stride ldc bytes), q_scale (may be null) / q_scale_inv its 1x128 scales, [inter / 128, M]
  int inter;
  int pow2_out;
  float* q_scale;
  float* q_scale_inv;
  int choose_cus;         // grouped by rows, tile chosen on the device: the compute units there are (test hook: minus the rows asked for)
};

// n / d for uniform values, without the compiler's division (some 30 dependent instructions; a tile lookup has four, and a
// workgroup does nothing else before its first transfers).  The reciprocal is not kept across a tile's products: hoisted out of
// the loop over tiles it took a vector register that 256 x 256 forms do not have, and came back from scratch memory behind a wait
// for every transfer under way.
__device__ __forceinline__ int quotient(int n, int d) {
  d = __builtin_amdgcn_readfirstlane(d);
  asm volatile("" : "+s"(d));
  if (n >= (1 << 22)) return n / d;
  int q = (int)((float)n * __builtin_amdgcn_rcpf((float)d));      // n and d exact in fp32, rcp within one ulp: off by one at most
  const int rest = n - q * d;
  q += rest >= d ? 1 : 0;
  q -= rest < 0 ? 1 : 0;
  return __builtin_amdgcn_readfirstlane(q);
}

// Tile number -> (m tile, n tile).  Consecutive numbers (one XCD's CUs at any moment) cover
// gm x gn rectangles of tiles (gm * gn = 32), n fastest inside a rectangle, so the L2 of that XCD
// serves each activation / weight panel to several CUs.  A panel of a is fetched once per column
// of rectangles (tiles_n / gn times in all) and a panel of b once per row of rectangles: the longer
// side of the rectangle goes along the shorter side of the tile grid, so that the larger operand,
// the one the Infinity Cache cannot hold, is the one fetched fewer times.  Rectangles at the right
// and bottom edges shrink.
__device__ __forceinline__ void rect_map(int t, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int gm = tiles_m > tiles_n ? 4 : 8, gn_full = kRectTiles / gm;
  const int per_ngroup = gn_full * tiles_m;
  const int ng = quotient(t, per_ngroup), rest = t - ng * per_ngroup;
  const int gn = (tiles_n - ng * gn_full) < gn_full ? (tiles_n - ng * gn_full) : gn_full;
  const int mg = quotient(rest, gm * gn);
  const int r3 = rest - mg * gm * gn;
  const int row = quotient(r3, gn);
  tm = mg * gm + row;
  tn = ng * gn_full + r3 - row * gn;
}

// One output tile of a workgroup's list.  A tile with no rows (row0 == row_end, n0 >= N) stands for
// "past the end of the list": transfers addressed to it fetch nothing.
struct TileInfo {
  int row0, row_end;   // rows [row0, row_end) of a and c that exist (row_end - row0 may be < BM)
  int n0;              // first row of b / column of c
  int expert;
  int kb0, kbn;        // grouped along the contraction: first k-block of the tile's expert and how many (>= 1)
  bool b_once;         // (grouped by rows, fetching waves) no other tile reads these rows of b, and they are not kept in the caches
};

// Position `d` k-blocks after k-block kb of the current tile (which has k0 k-blocks, the next one k1, every
// tile at least one): how many tiles further (0..2, d <= 2) and which k-block there.
__device__ __forceinline__ int tiles_ahead(int kb, int d, int k0, int k1, int& kb_out) {
  int pos = kb + d, q = 0;
  if (pos >= k0) {
    pos -= k0;
    q = 1;
    if (pos >= k1) { pos -= k1; q = 2; }
  }
  kb_out = pos;
  return q;
}

__device__ __forceinline__ TileInfo pick_tile(int q, TileInfo t0, TileInfo t1, TileInfo t2) {
  TileInfo r;
  r.row0 = q == 2 ? t2.row0 : (q == 1 ? t1.row0 : t0.row0);
  r.row_end = q == 2 ? t2.row_end : (q == 1 ? t1.row_end : t0.row_end);
  r.n0 = q == 2 ? t2.n0 : (q == 1 ? t1.n0 : t0.n0);
  r.expert = q == 2 ? t2.expert : (q == 1 ? t1.expert : t0.expert);
  r.kb0 = q == 2 ? t2.kb0 : (q == 1 ? t1.kb0 : t0.kb0);
  r.kbn = q == 2 ? t2.kbn : (q == 1 ? t1.kbn : t0.kbn);
  r.b_once = false;      // (the fetching waves look their tiles up)
  return r;
}

// Inclusive sum / maximum over the lanes of a wave, of values that are not negative (steps inside rows of 16 lanes, then
// across the rows).
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_or_zero(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false); }
template <class Op>
__device__ __forceinline__ int wave_scan(int x, Op op) {
  x = op(x, dpp_or_zero<0x111, 0xf>(x));   // row_shr:1
  x = op(x, dpp_or_zero<0x112, 0xf>(x));
  x = op(x, dpp_or_zero<0x114, 0xf>(x));
  x = op(x, dpp_or_zero<0x118, 0xf>(x));
  x = op(x, dpp_or_zero<0x142, 0xa>(x));   // row_bcast:15
  x = op(x, dpp_or_zero<0x143, 0xc>(x));   // row_bcast:31
  return x;
}

// Grouped by rows: 64 experts at a time, one per lane.  (One after the other, each behind the load of its offset, the experts
// took longer than a small problem's products: 64 experts [2048, 2048], 64 rows, all with one of them 24.6 us, 13.1 so.)
struct ExpertChunk {
  int first, row, tile;   // the chunk's first expert, the rows and the tiles before it
  int end, tile_end;      // this lane's expert: the row it ends with, the tiles up to its last one
};

// Offsets that decrease or run past the row count (a malformed table) are clamped, so that every address derived from them
// stays inside a.
__device__ __forceinline__ void expert_ends(ExpertChunk& c, const GemmParams& p, int lane) {
  int end = c.first + lane < p.experts ? p.offs[c.first + lane] : 0;
  end = wave_scan(end > c.row ? end : c.row, [](int a, int b) { return a > b ? a : b; });
  c.end = end < p.M ? end : p.M;
}
__device__ __forceinline__ int expert_rows(const ExpertChunk& c, int lane) {
  const int prev = __shfl_up(c.end, 1);
  return c.end - (lane == 0 ? c.row : prev);
}
__device__ __forceinline__ void count_tiles(ExpertChunk& c, int tile_rows, int tiles_n, int lane) {
  c.tile_end = c.tile + wave_scan((expert_rows(c, lane) + tile_rows - 1) / tile_rows, [](int a, int b) { return a + b; }) * tiles_n;
}
__device__ __forceinline__ bool next_experts(ExpertChunk& c, const GemmParams& p, int tile_rows, int tiles_n, int lane) {
  if (c.first + 64 >= p.experts) return false;
  c.first += 64;
  c.row = __builtin_amdgcn_readlane(c.end, 63);
  c.tile = __builtin_amdgcn_readlane(c.tile_end, 63);
  expert_ends(c, p, lane);
  count_tiles(c, tile_rows, tiles_n, lane);
  return true;
}

// Grouped by rows: the rows of the best tile for the rows that the experts have, 64 (x 128 columns), 128 or 256 (x 256).  What
// counts is the rounds of one tile per compute unit; rounds cost 26 : 50 : 83 (measured, us with 64 / 128 / 256 rows: 8192
// rows of one expert [4096, 7168], 16 / 4 / 2 rounds 313 / 201 / 178, bound by arithmetic; 2048 rows over 32 of them evenly, 4 / 2 / 2
// rounds 151 / 144 / 197, bound by reading b; 512 rows of one, one round each 23 / 42 / 64).  What this chooses was the fastest of the
// three or within 3 % of it in every line of the table at pick_grouped.  c: the first 64 experts.
__device__ __forceinline__ int grouped_tile_rows(const ExpertChunk& c, const GemmParams& p, int lane) {
  int low = 0, mid = 0, high = 0;
  for (ExpertChunk e = c;;) {
    const int rows = expert_rows(e, lane);
    const auto sum = [](int a, int b) { return a + b; };
    low += __builtin_amdgcn_readlane(wave_scan((rows + 63) / 64, sum), 63);
    mid += __builtin_amdgcn_readlane(wave_scan((rows + 127) / 128, sum), 63);
    high += __builtin_amdgcn_readlane(wave_scan((rows + 255) / 256, sum), 63);
    if (e.first + 64 >= p.experts) break;
    e.first += 64;
    e.row = __builtin_amdgcn_readlane(e.end, 63);
    expert_ends(e, p, lane);
  }
  const int cus = p.choose_cus, tiles_n = (p.N + 255) / 256;
  const int64_t low_cost = 26 * (int64_t)quotient(low * ((p.N + 127) / 128) + cus - 1, cus);
  const int64_t mid_cost = 50 * (int64_t)quotient(mid * tiles_n + cus - 1, cus);
  const int64_t high_cost = 83 * (int64_t)quotient(high * tiles_n + cus - 1, cus);
  return low_cost <= mid_cost && low_cost <= high_cost ? 64 : (mid_cost <= high_cost ? 128 : 256);
}

// Grouped by rows, rows of b that one tile alone reads are streamed past the caches where the experts with rows have more than the
// Infinity Cache (256 MiB) holds, so that little of them would be there when the next call comes; fewer may still be there, and
// streamed they never are.  us kept / streamed, with one b for every call (with two or more in turn), 16 rows each of experts [4096, 7168]:
//    6 (168 MiB)  28.7 / 30.9  (34.4 / 30.9)     9 (252)  43.7 / 52.7  (57.2 / 52.6)    10 (280)  55.4 / 54.3  (59.0 / 54.6)
//   16 (448)      83.2 / 72.0  (83.0 / 72.6)    24 (672)   121 / 106    (122 / 107)
// 512 rows of 32 (896) evenly 159 / 140, by Zipf's law 175 / 157; of 8 (224) evenly 36.7 / 39.4 (44.5 / 39.9), by Zipf's law 43.2 / 56.6.
// Over 1000 sizes from 180 to 460 MiB and from 1 to 100 rows per expert streaming takes 1.03 times as long on average (1.16 at most)
// from 260 to 280 MiB, 0.96 (1.06) to 300, and 0.91 (never more than 1) beyond.  (Dense products do not stream: their kernels are shorter by
// a quarter of a microsecond without it, which is 6 to 8 % of the smallest.)
constexpr int64_t kStreamFrom = (int64_t)300 << 20;

// one wave's transfer of 8 rows x 128 bytes to LDS, as data read once
__device__ __forceinline__ void stream_1k(__amdgpu_buffer_rsrc_t rs, uint8_t* dst, uint32_t lane_off, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, lane_off, off, 0, 2);
}

// WM, NS, WN: WM x WN waves multiply, each 64 rows x NS subtiles of 16 columns.  Tiles of 64 and of 128 rows have four more
// waves, which do the transfers.
__host__ __device__ constexpr bool fetchers(int wm) { return wm <= 2; }
__host__ __device__ constexpr int tile_threads(int wm, int wn) { return 64 * (wm * wn + (fetchers(wm) ? 4 : 0)); }

__host__ __device__ constexpr bool row_scales(int mode) { return mode == kScaleRow || mode == kScalePow2Row; }
__host__ __device__ constexpr int tile_stages(int mode, int wm, int tn) {         // k-blocks of b (and, with fetching waves, of a) in LDS
  return !fetchers(wm) ? b_stages(mode) : (tn == 256 ? 3 : (wm == 2 ? 4 : (tn == 128 ? 6 : 8)));
}
// With fetching waves the scales of a k-block travel with its tiles, into a slot of one part per fetching wave: 256 bytes of sb
// (the scale of the left or of the right half's block; with per-row scales 64 of the tile's rows) and the upper or the lower 64
// rows of sa.
constexpr int kScaleSlot = 2048;
// One LDS object for everything.  (With a second __shared__ array the compiler tells the two apart
// with alias scopes, and from then on makes every LDS read wait for all transfers into the array it
// reads, those to other buffers included: the transfers' latency would be paid in every round.)
__host__ __device__ constexpr int tile_lds(int mode, int wm, int tn) {
  const int stages = tile_stages(mode, wm, tn);
  const int scales = fetchers(wm) ? (mode == kScaleTensor ? 0 : (stages + 1) * kScaleSlot) : (mode == kScalePow2Row ? 3 * 256 * 4 : 0);
  return (fetchers(wm) ? stages : 2) * 64 * wm * BK + stages * tn * BK + scales;
}

// Per-row scales on both operands: the four products sb * sa that a lane needs for one 16 x 16 subtile, in the layout of the
// subtile's sums (rows of b 4 g + r, r = 0..3, and row of a l16, for lane 16 g + l16), as the outer products of one small matrix
// instruction: 16 blocks of 4 x 4, block l / 4 of lane l.  Its b rows are those of block `sub` of the four blocks that share
// g, so one register holds the b scales of four subtiles: lane l that of row 16 ((l / 4) % 4) + 4 (l / 16) + l % 4.
// A promotion is then one FMA per element as with a scale per block of b, where a multiplication by the b scale ahead of it made
// this form bound by instruction issue (a matrix instruction takes about 15 of a SIMD's issue cycles, a vector instruction 4: 47
// per group of one and eight against 32 of matrix pipe).  The four of a subtile are issued back to back: 43 cycles a group, where
// one in front of each large matrix instruction makes it 51.  us before / so: 7168 x 16384 x 4096 466 / 437 (one by one 469),
// 36864 x 7168 x 4096 1064 / 997, 2048 x 7168 x 1536 28.2 / 27.6, 1400 x 3072 x 4096 33.1 / 29.5, 1024 x 1024 x 4096 13.5 / 12.4.
// (The instruction keeps subnormal products, and the scales are multiplied first as in the block form: a pair whose product overflows
// gives NaN for a sum of 0, where multiplied one after the other it gave 0.)
__device__ __forceinline__ int scale_row(int lane) { return ((lane >> 2) & 3) * 16 + (lane >> 4) * 4 + (lane & 3); }
__device__ __forceinline__ v4f scale_products(float sb, float sa, int sub) {
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  switch (sub) {       // (a literal in the instruction; sub is known when the loops are unrolled)
    case 0: return __builtin_amdgcn_mfma_f32_4x4x1f32(sb, sa, zero, 2, 0, 0);
    case 1: return __builtin_amdgcn_mfma_f32_4x4x1f32(sb, sa, zero, 2, 1, 0);
    case 2: return __builtin_amdgcn_mfma_f32_4x4x1f32(sb, sa, zero, 2, 2, 0);
    default: return __builtin_amdgcn_mfma_f32_4x4x1f32(sb, sa, zero, 2, 3, 0);
  }
}

// group: grouped by rows, the first 64 experts with their ends; then those among which tiles are looked up (tile numbers are
// asked for in increasing order).
// pid, nwg: this workgroup among those that share the tile list.
// SA4: the activation scales have unit stride over rows (the k-block-major layout), so a lane's four
// of them are one 16-byte load.
// EPI: 0 = c is the GEMM's result; 1 / 2 = the gate/up projection of a SwiGLU MLP with the activation and its
// 1x128 quantization as the epilogue (1: exactly specified silu, 2: hardware exponential and reciprocal).  A tile's
// 256 columns are then the 128 gate columns and the 128 up columns of one scaling group of the activation: the b
// tile's upper 128 rows come from `inter` rows further down, the two waves that share 64 rows hold gate and up.
template <int MODE, int GROUPED, bool OUT_F32, bool ACC, bool SA4, int EPI, int WM, int NS, int WN>
__device__ __forceinline__ void gemm_tiles(const GemmParams& p, uint8_t* const lds, ExpertChunk group, const int pid, const int nwg) {
  constexpr int TM = 64 * WM, TN = 16 * NS * WN;       // the tile
  constexpr int WC = 16 * NS;                          // a wave's columns
  constexpr int kWaves = WM * WN;                      // that multiply
  constexpr bool kFetchers = fetchers(WM);             // four more do the transfers
  constexpr int kFetchWaves = kFetchers ? 4 : kWaves;
  constexpr int kATile = TM * BK, kBTile = TN * BK;    // one operand tile in LDS
  constexpr int NA = TM / 8 / kFetchWaves, NB = TN / 8 / kFetchWaves;     // transfers per wave and k-block
  constexpr int kSlice = kBTile / kWaves;              // a wave's part of a b buffer
  static_assert(EPI == 0 || TN == 256, "SwiGLU epilogue: 128 gate and 128 up columns per tile");
  static_assert(EPI == 0 || ((MODE == kScaleBlock || MODE == kScalePow2) && GROUPED == kDense && !OUT_F32 && !ACC),
                "SwiGLU epilogue: dense block-scaled forward");
  static_assert(!ACC || (OUT_F32 && MODE != kScaleTensor), "accumulating onto c: fp32 output, sums that start from c's values");
  static_assert(GROUPED != kGroupedK || (!ACC && (MODE == kScaleRow || MODE == kScalePow2Row)),
                "grouped along the contraction: the wgrad form");
  static_assert(!kFetchers || GROUPED != kGroupedK, "the fetching waves count k-blocks from 0");
  constexpr int kBStages = tile_stages(MODE, WM, TN);
  constexpr int kAStages = kFetchers ? kBStages : 2;
  constexpr bool kRowScales = row_scales(MODE);                             // per-row b scales
  constexpr bool kStagedScales = MODE == kScalePow2Row && !kFetchers;       // staged in LDS by the multiplying waves
  constexpr int kScaleRegs = (NS + 3) / 4;                                  // kScaleRow: registers of them, four subtiles each
  constexpr bool kPromote = MODE == kScaleBlock || MODE == kScaleRow;       // partial sums scaled by FMAs
  constexpr bool kHwScale = MODE == kScalePow2 || MODE == kScalePow2Row;    // scales applied by the MFMA
  constexpr int kBAhead = kBStages - 1;     // k-blocks between issuing a b transfer and using it
  constexpr int kScaleOps = MODE == kScaleTensor ? 0 : 2, kScaleSlots = kBStages + 1;
  // per-row scales of the b operand for one k-block (wgrad form, powers of two), three stages of 256 floats: the
  // stage of k-block kb+1 is filled while slower waves may still read that of kb-1
  uint8_t* const scale_lds = lds + kAStages * kATile + kBStages * kBTile;
  float* const sb_lds = reinterpret_cast<float*>(scale_lds);
  constexpr int kSbSlot = kFetchers ? kScaleSlot / 4 : 256;
  uint8_t* const b_lds = lds + kAStages * kATile;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool fetching = kFetchers && wave_id >= kWaves;
  const int wave = fetching ? wave_id - kWaves : wave_id;         // its part of a tile: of the transfers or of the products
  const int K = p.K, N = p.N;
  const int kblocks = K / BK;
  const int tiles_n = (N + TN - 1) / TN;

  // ---- the tile list of this workgroup.  The grid is persistent (one workgroup per CU); tiles are
  // numbered so that consecutive numbers cover rectangles of 32 tiles (rect_map), each XCD (workgroup ids
  // congruent mod 8, own L2) owns a contiguous run of numbers, and the workgroups of an XCD walk
  // through that run side by side, so at any moment they work on one rectangle.
  bool stream_b = false;               // grouped by rows: rows of b that one tile alone reads go past the caches
  int total_tiles = p.tiles;
  if (GROUPED == kGroupedK) total_tiles = p.experts * p.tiles;
  if (GROUPED == kGroupedRows) {
    // tiles are numbered expert by expert; an expert with no rows has none
    const ExpertChunk first = group;
    count_tiles(group, TM, tiles_n, lane);
    auto with_rows = [&]() { return __builtin_popcountll(__ballot(expert_rows(group, lane) != 0)); };
    int used = kFetchers ? with_rows() : 0;
    while (next_experts(group, p, TM, tiles_n, lane)) used += kFetchers ? with_rows() : 0;
    stream_b = kFetchers && (int64_t)used * N * K > kStreamFrom;
    total_tiles = __builtin_amdgcn_readlane(group.tile_end, 63);
    if (p.experts > 64) {
      group = first;
      count_tiles(group, TM, tiles_n, lane);
    }
  }
  int my_tiles, t_first, t_step;
  {
    // (the host launches a multiple of 8 workgroups, or fewer than 8)
    const bool few = nwg < kXcds;
    const int xcd = few ? pid : pid % kXcds, slot = few ? 0 : pid / kXcds;
    t_step = few ? 1 : nwg / kXcds;
    const int base = few ? quotient(total_tiles, nwg) : total_tiles / kXcds;
    const int big = total_tiles - base * (few ? nwg : kXcds);
    const int cnt = base + (xcd < big ? 1 : 0);
    t_first = xcd * base + (xcd < big ? xcd : big) + slot;
    my_tiles = slot < cnt ? quotient(cnt - slot + t_step - 1, t_step) : 0;
    if (GROUPED == kGroupedK) {
      // Tiles differ in length (an expert's contraction is its own token count) and are numbered longest expert
      // first.  They are dealt out in rounds of one tile per workgroup -- the XCD with index x takes positions
      // [x * t_step, (x + 1) * t_step) of every round, consecutive tiles as before -- so that every workgroup
      // gets the same mix of lengths and only the shortest tiles are left for the last, incomplete round.
      t_first = xcd * t_step + slot;
      t_step = nwg;
      my_tiles = t_first < total_tiles ? (total_tiles - t_first + nwg - 1) / nwg : 0;
    }
  }
  if (my_tiles == 0) return;
  const int n_pad = tiles_n * TN;
  auto lookup = [&](int k, TileInfo& ti) {
    int row0 = p.M, row_end = p.M, n0 = n_pad, expert = 0, kb0 = 0, kbn = GROUPED == kGroupedK ? 1 : kblocks, row_tiles = 0;
    if (k < my_tiles) {
      const int t = t_first + k * t_step;
      int tm, tn;
      if (GROUPED == kGroupedK) {
        const int i = quotient(t, p.tiles);
        expert = p.layout[4 * p.experts + i];
        kb0 = p.layout[4 * expert + 2];
        kbn = p.layout[4 * expert + 3];
        rect_map(t - i * p.tiles, (p.M + TM - 1) / TM, tiles_n, tm, tn);
        row0 = tm * TM;
        row_end = row0 + TM < p.M ? row0 + TM : p.M;
        n0 = tn * TN;
      } else if (GROUPED == kGroupedRows) {
        while (t >= __builtin_amdgcn_readlane(group.tile_end, 63) && next_experts(group, p, TM, tiles_n, lane)) {}
        const int l = __builtin_popcountll(__ballot(group.tile_end <= t));    // (experts without rows end where the one before ends)
        if (l < 64) {
          const int end = __builtin_amdgcn_readlane(group.end, l), prev = l ? __builtin_amdgcn_readlane(group.end, l - 1) : group.row;
          const int cnt = (end - prev + TM - 1) / TM;
          row_tiles = cnt;
          rect_map(t - (__builtin_amdgcn_readlane(group.tile_end, l) - cnt * tiles_n), cnt, tiles_n, tm, tn);
          expert = group.first + l;
          row0 = prev + tm * TM;
          row_end = end;
          if (row0 + TM < row_end) row_end = row0 + TM;
          n0 = tn * TN;
        }
      } else {
        rect_map(t, (p.M + TM - 1) / TM, tiles_n, tm, tn);
        row0 = tm * TM;
        row_end = row0 + TM < p.M ? row0 + TM : p.M;
        n0 = tn * TN;
      }
    }
    // (values found through the expert search sit in vector registers; as scalars they keep the
    // buffer resources built from them scalar too)
    ti.row0 = __builtin_amdgcn_readfirstlane(row0);
    ti.row_end = __builtin_amdgcn_readfirstlane(row_end);
    ti.n0 = __builtin_amdgcn_readfirstlane(n0);
    ti.expert = __builtin_amdgcn_readfirstlane(expert);
    ti.kb0 = __builtin_amdgcn_readfirstlane(kb0);
    ti.kbn = __builtin_amdgcn_readfirstlane(kbn);
    ti.b_once = stream_b && __builtin_amdgcn_readfirstlane(row_tiles) == 1;
  };
  // ---- global -> LDS tile DMA.  One wave instruction moves 8 rows x 128 B (lane i -> LDS slot
  // i); the lane picks the 16-byte global chunk whose swizzled home is its slot.  The buffer
  // resource of a transfer starts at the tile's first row and ends with the tensor, so lane
  // offsets do not depend on the tile and rows past the end of the tensor read as zero.
  // (The resource runs on to the end of the tensor rather than to the end of the tile: dense, transfers
  // through a resource that only just covers the rows they touch were measured markedly slower.  Grouped by rows, where most of a
  // tile may be rows of other experts that are not stored, it ends with the tile's own: us with resources that end with the tensor /
  // with the tile, 32 experts [4096, 7168] 512 rows evenly 148 / 141, by Zipf's law 193 / 176, 2048 rows 151 / 145 and 195 / 186, 8192
  // 258 / 258 and 309 / 301; tiles that are full take the same in both, with the tensor's end for those alone too: 16384 rows of 64 experts
  // [2048, 2048] evenly 82 / 82, 131072 of 8 3032 / 3033.)
  auto span_bytes = [&](int64_t rows, int64_t ld) {     // up to the end of the last row's K codes
    const int64_t bytes = rows > 0 ? (rows - 1) * ld + K : 0;
    return (int)(bytes < (int64_t)0x7FFFF000 ? bytes : (int64_t)0x7FFFF000);   // 256 rows always fit (host check)
  };
  auto rsrc_a_of = [&](const TileInfo& ti) {
    const int rows = ti.row_end > ti.row0 ? (GROUPED == kGroupedRows ? ti.row_end : p.M) - ti.row0 : 0;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(p.a + (int64_t)ti.row0 * p.lda), 0, span_bytes(rows, p.lda),
                                             0x00020000);
  };
  auto rsrc_b_of = [&](const TileInfo& ti) {
    // (SwiGLU epilogue: the tile's first b row is gate row n0 / 2; its up rows lie `inter` rows further down)
    const int brow0 = EPI ? ti.n0 >> 1 : ti.n0;
    const int rows = N - ti.n0 > 0 ? N - brow0 : 0;
    const uint8_t* base = p.b + (GROUPED == kGroupedRows ? (int64_t)ti.expert * p.b_se : 0) + (int64_t)(rows ? brow0 : 0) * p.ldb;
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, span_bytes(rows, p.ldb), 0x00020000);
  };
  uint32_t a_off[NA], b_off[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int q = wave * NA + i;                      // 8-row group inside the tile
    const int r = q * 8 + (lane >> 3);                // row inside the tile
    const int chunk = (lane & 7) ^ row_swizzle(r);    // logical 16-byte chunk of that row
    // The rows of the a tile are permuted on their way into LDS: LDS row 64 w + 16 j + l holds tile row
    // 64 w + 4 l + j.  The lane that owns LDS rows 16 j + l16 (j = 0..3) of its wave's 64 then owns four
    // consecutive rows of a, whose scales are one 16-byte load and whose results are four adjacent
    // rows of c.  (The b tile keeps its order.)
    const int ra = (r & ~63) + (r & 15) * 4 + ((r >> 4) & 3);
    a_off[i] = (uint32_t)ra * (uint32_t)p.lda + chunk * 16;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int r = (wave * NB + i) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ row_swizzle(r);
    b_off[i] = (uint32_t)(EPI && r >= 128 ? r - 128 + p.inter : r) * (uint32_t)p.ldb + chunk * 16;
  }
  // kStagedScales: the 256 per-row scales of the b tile for one k-block are one more 1 KB transfer
  // (wave 0), possible because that scale array is k-block-major (unit stride over rows).
  const __amdgpu_buffer_rsrc_t rsrc_sb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.sb, 0, kRowScales ? (int)((((int64_t)kblocks - 1) * p.sb_sk + N) * 4) : 0, 0x00020000);
  auto issue_sb_load = [&](const TileInfo& ti, int kb, int stage) {      // kb counted inside the tile's own contraction
    if (kStagedScales && wave == 0)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_sb, (lds_ptr_t)(sb_lds + stage * 256), 16,
                                               (uint32_t)(ti.n0 + lane * 4) * 4u,
                                               (int)(((GROUPED == kGroupedK ? ti.kb0 : 0) + kb) * p.sb_sk * 4), 0, 0);
  };
  // One transfer = 8 rows x 128 B per wave; `sub` selects which of the wave's 8-row groups of the tile.
  // Four transfers share one LDS base (M0) and differ in the instruction's immediate offset, which the
  // hardware adds to both the LDS and the memory address; the memory side is compensated in the lane offset.
  auto transfer = [&](const __amdgpu_buffer_rsrc_t& rs, uint32_t off, uint8_t* base, int kb, int sub) {
    uint8_t* sbase = base + (sub >> 2) * 4096;
    const uint32_t voff = off - (sub & 3) * 1024;
    switch (sub & 3) {   // the immediate must be a literal; sub is a compile-time constant after unrolling
      case 0: __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)sbase, 16, voff, kb * BK, 0, 0); break;
      case 1: __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)sbase, 16, voff, kb * BK, 1024, 0); break;
      case 2: __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)sbase, 16, voff, kb * BK, 2048, 0); break;
      default: __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)sbase, 16, voff, kb * BK, 3072, 0); break;
    }
  };
  auto issue_a = [&](const __amdgpu_buffer_rsrc_t& rs, int buf, int kb, int sub) {
    transfer(rs, a_off[sub], lds + buf * kATile + wave * (NA * 1024), kb, sub);
  };
  auto issue_b = [&](const __amdgpu_buffer_rsrc_t& rs, int buf, int kb, int sub) {
    transfer(rs, b_off[sub], b_lds + buf * kBTile + wave * (NB * 1024), kb, sub);
  };
  // Rows of b that one tile alone reads are streamed (b_once): they stay in no cache, which leaves those to a's rows.  Where several tiles
  // share them it would cost: 8192 rows of 32 experts [4096, 7168] 299 / 310 us.
  auto issue_stream_b = [&](const __amdgpu_buffer_rsrc_t& rs, int buf, int kb, int sub) {
    stream_1k(rs, b_lds + buf * kBTile + wave * (NB * 1024) + sub * 1024, b_off[sub], kb * BK);
  };

  // ---- fragment addressing
  const int wn = wave % WN, wm = wave / WN;
  const int l16 = lane & 15, g = lane >> 4;
  // A lane's two chunks of a fragment lie equally far behind the fragment's first row in both operands.  256 x 256 tiles keep these
  // two offsets (opaque: taken apart again, the parts would take two registers more) and the rest of an address is scalar.
  const int l16_row = l16 * BK;
  int frag_lo = (kFetchers ? 0 : l16_row) + ((2 * g) ^ row_swizzle(l16)) * 16, frag_hi = frag_lo ^ 16;
  if (!kFetchers) asm volatile("" : "+v"(frag_lo), "+v"(frag_hi));
  const int a_frag = wm * 64 * BK + (kFetchers ? l16_row : 0);                           // + j * 16 rows
  const int b_frag = wn * WC * BK + (kFetchers ? l16_row : 0);                           // + i * 16 rows, inside a b buffer

  // ---- scales.  Raw values for one k-block are loaded at the top of the round before it and only
  // combined (sa * sb) at its end, so nothing waits on global memory in between.
  // Both scale arrays are read through buffer resources with 32-bit byte offsets (the host checks
  // that they span less than 2 GiB): the row part of an offset is per tile, the k-block part a
  // scalar, so a round spends no vector arithmetic on addresses.
  const __amdgpu_buffer_rsrc_t rsrc_sa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.sa, 0, MODE == kScaleTensor ? 4 : (int)((((int64_t)p.M - 1) * p.sa_sm + ((int64_t)kblocks - 1) * p.sa_sk + 1) * 4),
      0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_sbb = __builtin_amdgcn_make_buffer_rsrc((void*)p.sb, 0, p.sb_bytes, 0x00020000);
  uint32_t sa_voff[4];         // byte offset of this lane's four rows in sa (SA4: [0] covers all four)
  int sb_soff = 0;             // block form: byte offset of the b tile's scale row
  uint32_t sb_voff = 0;        // kScaleRow: byte offset of this lane's column of the b tile in sb
  const int sa_kstep = (int)p.sa_sk * 4, sb_kstep = (int)p.sb_sk * 4;
  auto scale_target = [&](const TileInfo& ti) {
    int lane_s = lane;
    asm volatile("" : "+v"(lane_s));    // (keeps what the offsets are made of out of the registers held through the rounds)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = ti.row0 + wm * 64 + (lane_s & 15) * 4 + j;
      // (SA4 does not clamp: words past the end of the array read as zero, and rows past M are never stored)
      sa_voff[j] = SA4 ? (uint32_t)r * 4u : (uint32_t)(r < p.M ? r : p.M - 1) * (uint32_t)((int)p.sa_sm * 4);
    }
    if (MODE == kScaleRow) sb_voff = (uint32_t)(ti.n0 + wn * WC + scale_row(lane_s)) * 4u;      // (past N: columns that are not stored)
    int nblk_idx = EPI ? (ti.n0 >> 8) + wn * (p.inter >> 7) : (ti.n0 + wn * WC) >> 7;
    if (nblk_idx > (N >> 7) - 1) nblk_idx = (N >> 7) - 1;
    sb_soff = ((GROUPED == kGroupedRows ? ti.expert * (int)p.sb_se : 0) + nblk_idx * (int)p.sb_sn) * 4;
  };
  auto load_scales = [&](int kb, float raw[6]) {
    if (MODE == kScaleRow) {
#pragma unroll
      for (int h = 0; h < kScaleRegs; ++h)
        raw[4 + h] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_sb, sb_voff + h * 256, kb * sb_kstep, 0));
    }
    if (MODE == kScaleBlock || MODE == kScalePow2)
      raw[4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_sbb, 0, sb_soff + kb * sb_kstep, 0));
    if (MODE != kScaleTensor) {
      if (SA4) {
        const v4f four = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc_sa, sa_voff[0], kb * sa_kstep, 0));
#pragma unroll
        for (int j = 0; j < 4; ++j) raw[j] = four[j];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          raw[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_sa, sa_voff[j], kb * sa_kstep, 0));
      }
    }
  };
  if constexpr (kFetchers) {
    if (fetching) {
      // ---- the fetching waves: the k-blocks of the tile list one after the other, kBStages of them at a time in LDS.  After a
      // round's barrier the multiplying waves have left the buffers of its k-block, which are filled again at once; past
      // the end of the list nothing is fetched.
      constexpr int kOps = NA + NB + kScaleOps;          // a wave's transfers per k-block
      int f_tile = 0, f_kb = 0, buf = 0, slot = 0;
      __amdgpu_buffer_rsrc_t ra, rb;
      uint32_t sa_off, sb_off = 0;
      int sb_first = 0;
      bool b_once = false;
      auto enter = [&](const TileInfo& ti) {
        ra = rsrc_a_of(ti);
        rb = rsrc_b_of(ti);
        b_once = ti.b_once;
        const int row = ti.row0 + (wave >> 1) * 64 + lane;       // (rows past M repeat the last one's scale: they are not stored)
        sa_off = (uint32_t)(row < p.M ? row : p.M - 1) * (uint32_t)((int)p.sa_sm * 4);
        if (kRowScales) {
          sb_off = (uint32_t)(ti.n0 + wave * 64 + lane) * 4u;        // (past N: columns that are not stored)
        } else {
          int blk = EPI ? (ti.n0 >> 8) + (wave & 1) * (p.inter >> 7) : (ti.n0 + (wave & 1) * (TN / 2)) >> 7;
          if (blk > (N >> 7) - 1) blk = (N >> 7) - 1;
          sb_first = ((GROUPED == kGroupedRows ? ti.expert * (int)p.sb_se : 0) + blk * (int)p.sb_sn) * 4;
        }
      };
      auto fetch_a = [&]() {
#pragma unroll
        for (int sub = 0; sub < NA; ++sub) issue_a(ra, buf, f_kb, sub);
      };
      auto fetch_rest = [&]() {
        if (b_once) {
#pragma unroll
          for (int sub = 0; sub < NB; ++sub) issue_stream_b(rb, buf, f_kb, sub);
        } else {
#pragma unroll
          for (int sub = 0; sub < NB; ++sub) issue_b(rb, buf, f_kb, sub);
        }
        if (kScaleOps) {
          uint8_t* const dst = scale_lds + slot * kScaleSlot + wave * 256;
          __builtin_amdgcn_raw_ptr_buffer_load_lds(kRowScales ? rsrc_sb : rsrc_sbb, (lds_ptr_t)dst, 4, sb_off,
                                                   sb_first + f_kb * sb_kstep, 0, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_sa, (lds_ptr_t)(dst + 1024), 4, sa_off, f_kb * sa_kstep, 0, 0);
        }
        buf = buf + 1 == kBStages ? 0 : buf + 1;
        slot = slot + 1 == kScaleSlots ? 0 : slot + 1;
        if (++f_kb == kblocks) {
          f_kb = 0;
          TileInfo next;
          lookup(++f_tile, next);
          enter(next);
        }
      };
      {
        TileInfo first;
        lookup(0, first);
        enter(first);
      }
      // (two k-blocks ahead of the first wait and not all: the first has to land through cold caches and what is queued up
      // behind it keeps these waves from the barrier)
      for (int k = 0; k < kBStages; ++k) {
        fetch_a();
        fetch_rest();
        if (k == 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kOps) : "memory");
      }
      for (int tile = 0; tile < my_tiles; ++tile) {
        for (int kb = 0; kb < kblocks; ++kb) {
          // the next k-block has landed; everyone has left this one
          asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((kBStages - 2) * kOps) : "memory");
          fetch_a();
          // the last b buffer of a tile is what its results are staged in: it is filled again when they have been read
          if (kb == kblocks - 1) {
            if (EPI) {
              for (int i = 0; i < 8; ++i) asm volatile("s_barrier" ::: "memory");
            } else {
              asm volatile("s_barrier" ::: "memory");
            }
          }
          fetch_rest();
        }
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last transfers fetch nothing but write to this workgroup's LDS
      return;
    }
  }
  auto read_scales = [&](int slot, float raw[6]) {      // (kFetchers)
    if (MODE == kScaleTensor) return;
    const uint8_t* const src = scale_lds + slot * kScaleSlot + (wm * 2 + wn * 2 / WN) * 256;
    if (MODE == kScaleRow) {
#pragma unroll
      for (int h = 0; h < kScaleRegs; ++h)
        raw[4 + h] = *reinterpret_cast<const float*>(scale_lds + slot * kScaleSlot + (wn * WC + h * 64 + scale_row(lane)) * 4);
    }
    const v4f four = *reinterpret_cast<const v4f*>(src + 1024 + l16 * 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) raw[j] = four[j];
    if (!kRowScales) raw[4] = *reinterpret_cast<const float*>(src);
  };
  // kScalePow2: the exponent fields of the scales of the current k-block, which are their E8M0 codes:
  // e_a[j] for the activation rows j * 16 + l16 of this lane, e_b for the weight block
  int e_a[4] = {127, 127, 127, 127}, e_b = 127;
  float sb_cur[2] = {1.f, 1.f};       // kScaleRow
  auto combine_scales = [&](const float raw[6], float s[4]) {
    if (MODE == kScaleRow) {
#pragma unroll
      for (int h = 0; h < kScaleRegs; ++h) sb_cur[h] = raw[4 + h];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = MODE == kScaleBlock ? raw[j] * raw[4] : raw[j];
    if (kHwScale) {
#pragma unroll
      for (int j = 0; j < 4; ++j) e_a[j] = (int)(__builtin_bit_cast(uint32_t, raw[j]) >> 23);
      if (MODE == kScalePow2) e_b = (int)(__builtin_bit_cast(uint32_t, raw[4]) >> 23);
    }
  };

  // ---- accumulators.  When the result is added onto c (ACC), a tile's accumulators do not start from
  // zero but from the tile's old values, loaded right before its first round in the order in which
  // that round touches them: they cost no registers and only the first of them is waited for.  A
  // lane's four sums of one 16 x 16 subtile are four consecutive columns of one row: one 16-byte
  // load.  The resource ends with the tensor: rows past it (and the tiles past the end of the list)
  // read as zero.
  auto rsrc_c_of = [&](const TileInfo& ti) {
    const int ncol = ti.n0 + wn * WC;
    const bool ok = ti.row_end > ti.row0 && ncol < N;
    int64_t bytes = ok ? (((int64_t)p.M - ti.row0 - 1) * p.ldc + N - ncol) * 4 : 0;
    if (bytes > (int64_t)0x7FFFF000) bytes = 0x7FFFF000;       // 256 rows always fit (host check)
    const float* base = reinterpret_cast<const float*>(p.c) + (ok ? (int64_t)ti.row0 * p.ldc + ncol : 0);
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
  };
  const int c_jstep = (int)p.ldc * 4;                          // bytes between the rows of subtiles j and j + 1
  auto old_values = [&](const __amdgpu_buffer_rsrc_t& rs, uint32_t lane_off, int i, int j) {
    return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, lane_off + i * 64, j * c_jstep, 0));
  };
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  v4f acc[NS][4];
  auto load_old_values = [&](const TileInfo& ti) {
    int lane_c = lane;
    asm volatile("" : "+v"(lane_c));    // (keeps the lane offset out of the registers held through the rounds)
    const __amdgpu_buffer_rsrc_t rc = rsrc_c_of(ti);
    const uint32_t c_lane = ((uint32_t)(wm * 64 + (lane_c & 15) * 4) * (uint32_t)p.ldc + (lane_c >> 4) * 4) * 4u;
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = old_values(rc, c_lane, i, j);
  };
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero;

  // ---- prologue: k-block 0 of both operands, k-block 1 of b where it has three buffers, and the
  // first half of k-block 1 of a (and of b where it has two buffers)
  float s_cur[4] = {1.f, 1.f, 1.f, 1.f}, s_raw[6] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
  // (k-block numbers passed to transfers and scale loads are absolute: grouped along the contraction, a tile's
  // own k-blocks start at its expert's first block kb0; otherwise kb0 is 0)
  auto kfirst = [](const TileInfo& ti) { return GROUPED == kGroupedK ? ti.kb0 : 0; };
  auto kcount = [&](const TileInfo& ti) { return GROUPED == kGroupedK ? ti.kbn : kblocks; };
  // T0 is the tile being accumulated; transfers and scale loads run up to two k-blocks ahead and
  // so reach into T1 (and into T2 when K is a single k-block).
  TileInfo T0, T1, T2;
  lookup(0, T0);
  if constexpr (kFetchers) {
    asm volatile("s_barrier" ::: "memory");        // the first k-block is there
    read_scales(0, s_raw);
    combine_scales(s_raw, s_cur);
  } else {
    const __amdgpu_buffer_rsrc_t ra = rsrc_a_of(T0), rb = rsrc_b_of(T0);
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) issue_a(ra, 0, kfirst(T0), sub);
#pragma unroll
    for (int sub = 0; sub < NB; ++sub) issue_b(rb, 0, kfirst(T0), sub);
    scale_target(T0);
    load_scales(kfirst(T0), s_raw);
    lookup(1, T1);
    lookup(2, T2);
    int kb1;
    const TileInfo t1 = pick_tile(tiles_ahead(0, 1, kcount(T0), kcount(T1), kb1), T0, T1, T2);
    kb1 += kfirst(t1);
    if (kBAhead == 2) {
      const __amdgpu_buffer_rsrc_t rb1 = rsrc_b_of(t1);
#pragma unroll
      for (int sub = 0; sub < NB; ++sub) issue_b(rb1, 1, kb1, sub);
    }
    issue_sb_load(T0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    // k-block 0 has landed (with three b buffers the next one of b may be under way)
    __builtin_amdgcn_s_waitcnt(kBAhead == 2 ? 0x0F70 | NB : 0x0F70);
    __syncthreads();
    combine_scales(s_raw, s_cur);
    const __amdgpu_buffer_rsrc_t ra1 = rsrc_a_of(t1);
    issue_a(ra1, 1, kb1, 0);
    issue_a(ra1, 1, kb1, 1);
    if (kBAhead == 1) {
      const __amdgpu_buffer_rsrc_t rb1 = rsrc_b_of(t1);
      issue_b(rb1, 1, kb1, 0);
      issue_b(rb1, 1, kb1, 1);
    }
  }

  // The synchronisation point of a round sits before its last two n-subtiles, not at its end: what
  // follows the barrier (the weight fragments of the next round's first two subtiles, and the
  // activation fragments re-read one by one as the last subtile releases their registers) is then
  // covered by the matrix instructions still to be issued, and no round starts with every wave
  // waiting on LDS at once.  Fragments that cross the round boundary are carried in registers.
  // Rounds follow each other without a gap across tiles: the last rounds of a tile already fetch
  // the first k-blocks of the next one, and its stores drain while the next tile computes.
  // With few subtiles there are not enough of them behind the barrier to cover the activation fragments read one by one
  // (64 x 128 tiles: 770 clocks a round for 384 of work): they are read right behind it then, into a second set of registers (us,
  // before / so: block 400 x 1024 x 8192 21.7 / 19.8, 256 x 3072 x 3072 11.6 / 11.1, 1531 x 2048 x 7168 33 / 31).
  constexpr bool kTwoX = kFetchers && NS <= 4;
  v8i xf[4], xg[4], wf_n0, wf_n1;
  wf_n0 = frag_read(b_lds + b_frag, frag_lo, frag_hi);
#pragma unroll
  for (int j = 0; j < 4; ++j) xf[j] = frag_read(lds + a_frag + j * 16 * BK, frag_lo, frag_hi);
  wf_n1 = frag_read(b_lds + b_frag + 16 * BK, frag_lo, frag_hi);

  v4f part_c[4] = {zero, zero, zero, zero};
  float s_old[4] = {0.f, 0.f, 0.f, 0.f};
  v4f s_of[4] = {zero, zero, zero, zero};          // kScaleRow: products of scales for the subtile that is promoted
  int stage = 0;                       // a buffer holding the current k-block
  int bbuf = 0;                        // b buffer holding the current k-block
  int sbuf = 0;                        // scale stage (kStagedScales) or slot (kFetchers) holding the current k-block
  // transfer targets (ordinal in the tile list) and their buffer resources
  int ord_1 = 0, ord_2 = 0;
  TileInfo tile_1 = T0;
  int kofs_2 = kfirst(T0);             // first k-block of the tile the transfers two ahead go to
  __amdgpu_buffer_rsrc_t rs_a1 = rsrc_a_of(T0), rs_a2 = rs_a1, rs_b1 = rsrc_b_of(T0), rs_b2 = rs_b1;

  // per-tensor form: the one multiplier of the store phase, read once (inside the tile loop the loads
  // would be repeated for every tile and waited for)
  float tensor_scale = 1.f;
  if (MODE == kScaleTensor) tensor_scale = p.sa[0] * p.sb[0];

  for (int tile = 0; tile < my_tiles; ++tile) {
  if (ACC) load_old_values(T0);
  const int kbn0 = kcount(T0);         // k-blocks of this tile
  // one k-block: its activation fragments are xf; the next one's go to xn
  auto round = [&](int kb, v8i (&xf)[4], v8i (&xn)[4]) __attribute__((always_inline)) {
    // Where this round's transfers and scale loads go: one k-block ahead (scales, second half of
    // those tiles), two ahead (first half of those tiles, or the whole b tile when it has three
    // buffers).  Only in the last
    // two rounds of a tile does a target move on to the next tile of the list; its resource is
    // rebuilt then and stays valid when that tile becomes the current one.
    int kb1 = kb + 1, kb2 = kb + 2;
    if (!kFetchers && kb2 >= kbn0) {
      const int o1 = tile + tiles_ahead(kb, 1, kbn0, kcount(T1), kb1);
      const int o2 = tile + tiles_ahead(kb, 2, kbn0, kcount(T1), kb2);
      if (o1 != ord_1) {
        ord_1 = o1;
        tile_1 = pick_tile(o1 - tile, T0, T1, T2);
        rs_a1 = rsrc_a_of(tile_1);
        if (kBAhead == 1) rs_b1 = rsrc_b_of(tile_1);
        scale_target(tile_1);
      }
      if (o2 != ord_2) {
        ord_2 = o2;
        const TileInfo t2 = pick_tile(o2 - tile, T0, T1, T2);
        rs_a2 = rsrc_a_of(t2);
        rs_b2 = rsrc_b_of(t2);
        kofs_2 = kfirst(t2);
      }
    }
    const int kb1_rel = kb1;             // inside tile_1's own contraction (what issue_sb_load counts in)
    kb1 += kfirst(tile_1);
    kb2 += kofs_2;
    if (!kFetchers) load_scales(kb1, s_raw);
    const uint8_t* bcur = b_lds + bbuf * kBTile;
    int bnext = bbuf + 1 == kBStages ? 0 : bbuf + 1;           // holds the next k-block
    int bbuf_issue = bbuf + kBAhead;                           // receives the k-block kBAhead ahead
    if (bbuf_issue >= kBStages) bbuf_issue -= kBStages;
    const uint8_t* bnxt = b_lds + bnext * kBTile;
    const uint8_t* anxt = lds + (kFetchers ? bnext : stage ^ 1) * kATile;
    int snext = sbuf + 1 == (kFetchers ? kScaleSlots : 3) ? 0 : sbuf + 1;
    // Per round, with three b buffers: the rest of the next a tile at subtiles 0,1; the b tile two
    // rounds ahead at 2..5; after the barrier the first half of the a tile after next, into the
    // buffer whose fragments every wave has just left behind.  One transfer per subtile: a burst
    // would queue up in the texture path ahead of the LDS reads.
    // With two b buffers (kStagedScales) the b tile has to land within one round like the a tile, so
    // both go out in the four subtiles that follow the barrier, one transfer of each per subtile.
    auto issue_slot = [&](int i) {
      if (kFetchers) return;
      if (kBAhead == 2) {
        if (i < 2) {
          issue_a(rs_a1, stage ^ 1, kb1, i + 2);
        } else if (i < 6) {
          issue_b(rs_b2, bbuf_issue, kb2, i - 2);
        } else {
          issue_a(rs_a2, stage, kb2, i - 6);
        }
      } else if (i < 2) {
        issue_a(rs_a1, stage ^ 1, kb1, i + 2);
        issue_b(rs_b1, bnext, kb1, i + 2);
      } else if (i >= 6) {
        issue_a(rs_a2, stage, kb2, i - 6);
        issue_b(rs_b2, bbuf, kb2, i - 6);
      }
    };
    auto round_sync = [&]() {
      // Own transfers for the next round have landed and own LDS reads of this round's buffers are
      // done; then everyone's.  With three b buffers the NB b transfers of this round (the
      // youngest vector-memory operations) are for the round after next and may stay in flight.
      // (kFetchers: the fetching waves wait for them)
      if (kFetchers) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        return;
      }
      if (kBAhead == 2) __builtin_amdgcn_s_waitcnt(0x0070 | NB);  // vmcnt(NB) lgkmcnt(0)
      else __builtin_amdgcn_s_waitcnt(0x0070);               // vmcnt(0) lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
    };
    // weight fragment of subtile i + 2 (the first two of the next round once past the barrier)
    auto read_ahead = [&](int i) {
      return i + 2 < NS ? frag_read(bcur + b_frag + (i + 2) * 16 * BK, frag_lo, frag_hi)
                       : frag_read(bnxt + b_frag + (i + 2 - NS) * 16 * BK, frag_lo, frag_hi);
    };
    if (kPromote) {
      // Software pipeline over the 8 n-subtiles: the matrix instructions of subtile i are issued
      // interleaved with the promotion FMAs of subtile i-1, whose partial sums left the matrix
      // pipe four instructions earlier, so neither pipe waits for the other.
      v4f part[2][4];
      v8i wf[3];
      wf[0] = wf_n0;
      wf[1] = wf_n1;
#pragma unroll
      for (int j = 0; j < 4; ++j) part[1][j] = part_c[j];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        if (i == NS - 2) round_sync();
        wf[(i + 2) % 3] = read_ahead(i);
        if (kFetchers && i == NS - 2) read_scales(snext, s_raw);
        if (kTwoX && i == NS - 2) {
#pragma unroll
          for (int j = 0; j < 4; ++j) xn[j] = frag_read(anxt + a_frag + j * 16 * BK, frag_lo, frag_hi);
        }
        issue_slot(i);
        __builtin_amdgcn_sched_barrier(0);
        if (MODE == kScaleRow && i > 0) {
#pragma unroll
          for (int j = 0; j < 4; ++j) s_of[j] = scale_products(sb_cur[(i - 1) / 4], s_cur[j], (i - 1) % 4);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          part[i & 1][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[i % 3], xf[j], zero, 0, 0, 0, 0, 0, 0);
          if (MODE == kScaleRow) __builtin_amdgcn_sched_barrier(0);
          const int ip = (i + NS - 1) % NS;     // subtile being promoted; for i = 0 the last one of the previous round
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[ip][j][r] = __builtin_fmaf(part[(i - 1) & 1][j][r], MODE == kScaleRow ? s_of[j][r] : (i == 0 ? s_old[j] : s_cur[j]),
                                           acc[ip][j][r]);
          if (!kTwoX && i == NS - 1) xn[j] = frag_read(anxt + a_frag + j * 16 * BK, frag_lo, frag_hi);
          __builtin_amdgcn_sched_barrier(0);   // keep this (MFMA, FMAs) group together, in this order
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        part_c[j] = part[1][j];
        if (MODE == kScaleRow) s_of[j] = scale_products(sb_cur[kScaleRegs - 1], s_cur[j], (NS - 1) % 4);
      }
      wf_n0 = wf[NS % 3];
      wf_n1 = wf[(NS + 1) % 3];
    } else {
      v8i wf[3];
      wf[0] = wf_n0;
      wf[1] = wf_n1;
      // per-row b scales: this lane's row of subtile i is row i * 16 + l16 of the wave's 128
      const float* sb_own = sb_lds + sbuf * kSbSlot + wn * WC + l16;
      int e_bi[2] = {127, 127};
      if (MODE == kScalePow2Row) e_bi[0] = (int)(__builtin_bit_cast(uint32_t, sb_own[0]) >> 23);
      if (kStagedScales) issue_sb_load(tile_1, kb1_rel, snext);
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        if (i == NS - 2) round_sync();
        wf[(i + 2) % 3] = read_ahead(i);
        if (kFetchers && i == NS - 2) read_scales(snext, s_raw);
        if (kTwoX && i == NS - 2) {
#pragma unroll
          for (int j = 0; j < 4; ++j) xn[j] = frag_read(anxt + a_frag + j * 16 * BK, frag_lo, frag_hi);
        }
        if (MODE == kScalePow2Row && i < NS - 1) e_bi[(i + 1) & 1] = (int)(__builtin_bit_cast(uint32_t, sb_own[(i + 1) * 16]) >> 23);
        issue_slot(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // (weights on the A port, activations on the B port: a lane's own row is the one it supplies
          // the scale of)
          if (kHwScale)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[i % 3], xf[j], acc[i][j], 0, 0, 0,
                                                                        MODE == kScalePow2 ? e_b : e_bi[i & 1], 0, e_a[j]);
          else
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[i % 3], xf[j], acc[i][j], 0, 0, 0, 0, 0, 0);
          if (!kTwoX && i == NS - 1) xn[j] = frag_read(anxt + a_frag + j * 16 * BK, frag_lo, frag_hi);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      wf_n0 = wf[NS % 3];
      wf_n1 = wf[(NS + 1) % 3];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) s_old[j] = s_cur[j];
    combine_scales(s_raw, s_cur);
    stage ^= 1;
    bbuf = bnext;
    sbuf = snext;
  };
  if constexpr (kTwoX) {
    int kb = 0;
    for (; kb + 1 < kbn0; kb += 2) {
      round(kb, xf, xg);
      round(kb + 1, xg, xf);
    }
    if (kb < kbn0) {
      round(kb, xf, xg);
#pragma unroll
      for (int j = 0; j < 4; ++j) xf[j] = xg[j];
    }
  } else {
    for (int kb = 0; kb < kbn0; ++kb) round(kb, xf, xf);
  }
  // ---- the tile is complete: last promotion, then its stores
  if (kPromote) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v4f s = {s_old[j], s_old[j], s_old[j], s_old[j]};
      if (MODE == kScaleRow) s = s_of[j];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[NS - 1][j][r] = __builtin_fmaf(part_c[j][r], s[r], acc[NS - 1][j][r]);
    }
    // (the next tile's first round adds these zeros times the scales kept: also where those are not finite)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      part_c[j] = zero;
      s_old[j] = 0.f;
      s_of[j] = zero;
    }
  }
  // The wave's 64 x 128 results go out 16 rows at a time (pass j: rows 4 s + j, s = 0..15, of the wave's
  // 64, the a tile's rows being permuted in LDS) through its own 4 KB slice of the b buffer
  // whose k-block was consumed last (nothing is in flight to that buffer, and this wave alone
  // transfers into this slice later), so that a store instruction writes whole rows of 256 bytes
  // instead of 16 pieces of 8 bytes.  The slice holds 16 rows x 256 B, 16-byte chunks XOR-ed with
  // the row so that both the fragment-order writes and the row-order reads spread over all banks.
  const int row0 = T0.row0, row_end = T0.row_end, n0 = T0.n0;
  // Lane coordinates re-derived behind an opaque copy: store addresses built from them would
  // otherwise be hoisted out of the tile loop and held in registers through the main loop.
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));
  const int l16e = lane_e & 15, ge = lane_e >> 4;
  uint8_t* stg = b_lds + (bbuf == 0 ? kBStages - 1 : bbuf - 1) * kBTile + wave * kSlice;
  // With two b buffers the lower half of that slice already receives the next transfers: rows 0..7
  // then go to its upper half and rows 8..15 to the upper half of this wave's slice of the a buffer
  // that is being refilled (its upper half is filled after these stores).
  uint8_t* stg_hi = kBAhead == 1 ? lds + (stage ^ 1) * kATile + wave * 4096 + 2048 : stg + 2048;
  if (kBAhead == 1) stg += 2048;
  auto stg_row = [&](int row) { return (row < 8 ? stg : stg_hi) + (row & 7) * 256; };   // (row = l16e: the write side)
  const int ncol = n0 + wn * WC;                 // first column of the wave tile
  const bool cols_ok = ncol < N;
  constexpr int kHalves = OUT_F32 && NS == 8 ? 2 : 1;       // fp32 rows of 128 columns take two slices
  constexpr int kPerHalf = NS / kHalves;           // n-subtiles per slice
  const uint32_t stg_w = (uint32_t)(uintptr_t)(lds_ptr_t)stg_row(l16e);   // LDS byte address of this lane's row
  // Rows leave through a buffer resource that starts at the wave tile's first element and ends with the
  // tile's last valid row: the lane part of a store address is one offset computed once per tile, the
  // rest scalar, and rows past the end of a ragged tile (or of an expert) are dropped by the range check.
  constexpr int kEsize = OUT_F32 ? 4 : 2;
  const int rows_valid = row_end - row0 < TM ? row_end - row0 : TM;
  const __amdgpu_buffer_rsrc_t rsrc_st = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(reinterpret_cast<uint8_t*>(p.c) +
              ((int64_t)row0 * p.ldc + ncol + (GROUPED == kGroupedK ? (int64_t)T0.expert * p.c_se : 0)) * kEsize), 0,
      cols_ok && rows_valid > 0 ? (int)((((int64_t)rows_valid - 1) * p.ldc + WC) * kEsize) : 0, 0x00020000);
  const uint32_t st_lane = (uint32_t)(((wm * 64 + ge * 4) * (int)p.ldc) * kEsize + l16e * 16);
  const int st_row = (int)p.ldc * kEsize;        // bytes from one row of c to the next
  auto store_tile = [&](auto with_bias) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int h = 0; h < kHalves; ++h) {
#pragma unroll
        for (int ii = 0; ii < kPerHalf; ++ii) {
          const int i = h * kPerHalf + ii;
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = acc[i][j][r];
            if (MODE == kScaleTensor) v[r] *= tensor_scale;
          }
          if (decltype(with_bias)::value) {
            const uint2 braw = *reinterpret_cast<const uint2*>(p.bias + ncol + i * 16 + ge * 4);
            v[0] += bf16lo(braw.x); v[1] += bf16hi(braw.x); v[2] += bf16lo(braw.y); v[3] += bf16hi(braw.y);
          }
          // The staging writes are issued as bare instructions: the compiler would otherwise make
          // every LDS store wait for the tile transfers in flight (to other buffers) to land.
          if (OUT_F32) {
            const v4f o = {v[0], v[1], v[2], v[3]};
            asm volatile("ds_write_b128 %0, %1" ::"v"(stg_w + (((ii * 4 + ge) ^ l16e) * 16)), "v"(o) : "memory");
          } else {
            u32x2 o;
            o[0] = pack_bf16x2(v[0], v[1]);
            o[1] = pack_bf16x2(v[2], v[3]);
            asm volatile("ds_write_b64 %0, %1" ::"v"(stg_w + (((ii * 2 + (ge >> 1)) ^ l16e) * 16) + (ge & 1) * 8), "v"(o)
                         : "memory");
          }
          acc[i][j] = zero;
        }
#pragma unroll
        for (int k2 = 0; k2 < 4; k2 += 2) {      // two rows per lane at a time (registers are scarce here)
          v4i val[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            // staging row 4 (k2 + k) + ge; which half of the staging area it lies in does not depend on the lane
            const int row = 4 * (k2 + k) + ge;
            const uint8_t* half = (k2 + k) < 2 ? stg : stg_hi;
            val[k] = *reinterpret_cast<const v4i*>(half + (4 * ((k2 + k) & 1) + ge) * 256 + ((l16e ^ row) * 16));
          }
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            // staging row s of pass j is tile row 4 s + j (s = 4 (k2 + k) + ge: the ge part is in st_lane).
            // Streaming stores: the output is not read again here, and as ordinary stores a tile's
            // 128-256 KB would push operand panels out of the L2.
            // (rows of fewer than 256 bytes: the first lanes hold them)
            if (WC * kEsize >= 256 || l16e < WC * kEsize / 16)
              __builtin_amdgcn_raw_buffer_store_b128(val[k], rsrc_st, st_lane, (16 * (k2 + k) + j) * st_row + h * 256, 2);
          }
          // A 128-bit store reads its data registers over several cycles after it has issued, and a vector instruction
          // right behind it must not write them yet.  The compiler inserts the wait states for that only where the
          // store's scalar offset is a constant; this GPU needs them with an offset register too (a tile's stores
          // came out with the next LDS address in their first word, a few times per launch, when the memory pipe
          // was full).  The operands keep both values' registers until the wait states are over.
          asm volatile("s_nop 1" ::"v"(val[0]), "v"(val[1]) : "memory");
        }
      }
    }
  };
  if constexpr (EPI != 0) {
    // SwiGLU epilogue.  Per pass j (16 of the wave's 64 rows) the WN waves of a row write their bf16-rounded
    // results -- gate from the first half of them, up from the second -- into their staging slices as for a plain
    // store; after a barrier each of them takes its part of the 16 rows, reads gate and up of a row from the
    // slices (16 lanes x 8 columns: one scaling group of the activation), and computes, quantizes and stores
    // the activation exactly as the stand-alone kernel does on a bf16 gate/up tensor.  A second barrier keeps the
    // next pass's writes (and, after the last pass, the next tile's transfers) off slices still being read.
    static_assert(kBStages == 3, "staging rows 0..15 of a wave are contiguous");
    constexpr int kLanes = WC / 8;                   // lanes whose columns lie in one slice
    const uint8_t* gate_s = stg - wn * kSlice + l16e / kLanes * kSlice;
    const uint8_t* up_s = gate_s + WN / 2 * kSlice;
    const uint32_t stg_we = (uint32_t)(uintptr_t)(lds_ptr_t)(stg + l16e * 256);   // this lane's staging row
    const int gcol = n0 >> 1;                        // first activation column of the tile's scaling group
    const __amdgpu_buffer_rsrc_t rsrc_q = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<uint8_t*>(p.c) + (int64_t)row0 * p.ldc + gcol), 0,
        rows_valid > 0 ? (int)(((int64_t)rows_valid - 1) * p.ldc + 128) : 0, 0x00020000);
    const int64_t s_first = (int64_t)(n0 >> 8) * p.M + row0;
    const __amdgpu_buffer_rsrc_t rsrc_si = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.q_scale_inv + s_first), 0, rows_valid > 0 ? rows_valid * 4 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_sc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.q_scale ? p.q_scale + s_first : p.q_scale_inv), 0, p.q_scale && rows_valid > 0 ? rows_valid * 4 : 0,
        0x00020000);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int ii = 0; ii < NS; ++ii) {
        u32x2 o;
        o[0] = pack_bf16x2(acc[ii][j][0], acc[ii][j][1]);
        o[1] = pack_bf16x2(acc[ii][j][2], acc[ii][j][3]);
        asm volatile("ds_write_b64 %0, %1" ::"v"(stg_we + (((ii * 2 + (ge >> 1)) ^ l16e) * 16) + (ge & 1) * 8), "v"(o)
                     : "memory");
        acc[ii][j] = zero;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int it = 0; it < 4 / WN; ++it) {
        const int srow = 16 / WN * wn + 4 * it + ge;             // staging row: tile row wm * 64 + 4 * srow + j
        const int soff = srow * 256 + ((l16e % kLanes ^ srow) * 16);
        const v4i gv = *reinterpret_cast<const v4i*>(gate_s + soff);
        const v4i uv = *reinterpret_cast<const v4i*>(up_s + soff);
        uint4 a;
        a.x = swiglu2<EPI == 2>((uint32_t)gv[0], (uint32_t)uv[0]);
        a.y = swiglu2<EPI == 2>((uint32_t)gv[1], (uint32_t)uv[1]);
        a.z = swiglu2<EPI == 2>((uint32_t)gv[2], (uint32_t)uv[2]);
        a.w = swiglu2<EPI == 2>((uint32_t)gv[3], (uint32_t)uv[3]);
        const uint32_t m = row16_max_u32(mag8(a));
        float sc, sci;
        scales_from_amax(__uint_as_float(m << 16), sc, sci, p.pow2_out);
        const uint2 codes = cvt8<false>(a, sc);
        const int trow = wm * 64 + 4 * srow + j;
        u32x2 cw = {codes.x, codes.y};
        __builtin_amdgcn_raw_buffer_store_b64(cw, rsrc_q, (uint32_t)trow * (uint32_t)p.ldc + l16e * 8, 0, 2);
        if (l16e == 0) {
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sci), rsrc_si, trow * 4, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sc), rsrc_sc, trow * 4, 0, 0);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  } else if (cols_ok) {
    if (!p.bias) store_tile(std::false_type{});
    else store_tile(std::true_type{});
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NS; ++i) acc[i][j] = zero;
  }
  if constexpr (kFetchers) {
    // this tile's results have been read from the b buffer that the fetching waves fill next
    if (!EPI) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    lookup(tile + 1, T0);
  } else {
  T0 = T1;
  T1 = T2;
  lookup(tile + 3, T2);
  }
  }

  // Transfers issued past the end of the list (they fetch nothing) still target this workgroup's
  // LDS: drain them before the LDS can be handed to another workgroup.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
}

template <int MODE, int GROUPED, bool OUT_F32, bool ACC, bool SA4, int EPI = 0, int WM = 4, int NS = 8, int WN = 2>
__global__ __launch_bounds__(tile_threads(WM, WN)) void gemm_kernel(const GemmParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[tile_lds(MODE, WM, 16 * NS * WN)];
  ExpertChunk group{0, 0, 0, 0, 0};
  if (GROUPED == kGroupedRows) expert_ends(group, p, threadIdx.x & 63);
  gemm_tiles<MODE, GROUPED, OUT_F32, ACC, SA4, EPI, WM, NS, WN>(p, lds, group, blockIdx.x, gridDim.x);
}

// Grouped by rows, the tile chosen here, where the experts' rows are known.
template <int MODE, bool OUT_F32, bool SA4>
__global__ __launch_bounds__(512) void gemm_grouped_kernel(const GemmParams p) {
  constexpr int kMost = tile_lds(MODE, 4, 256) > tile_lds(MODE, 1, 128) ? tile_lds(MODE, 4, 256) : tile_lds(MODE, 1, 128);
  static_assert(tile_threads(4, 2) == 512 && tile_threads(2, 2) == 512 && tile_threads(1, 4) == 512 && kMost >= tile_lds(MODE, 2, 256), "");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kMost];
  ExpertChunk group{0, 0, 0, 0, 0};
  expert_ends(group, p, threadIdx.x & 63);
  const int rows = p.choose_cus < 0 ? -p.choose_cus : grouped_tile_rows(group, p, threadIdx.x & 63);
  if (rows == 64) gemm_tiles<MODE, kGroupedRows, OUT_F32, false, false, 0, 1, 2, 4>(p, lds, group, blockIdx.x, gridDim.x);
  else if (rows == 128) gemm_tiles<MODE, kGroupedRows, OUT_F32, false, false, 0, 2, 8, 2>(p, lds, group, blockIdx.x, gridDim.x);
  else gemm_tiles<MODE, kGroupedRows, OUT_F32, false, SA4, 0, 4, 8, 2>(p, lds, group, blockIdx.x, gridDim.x);
}

// Backward of a linear: both products, and the column sums that are its bias gradient, in one launch.
//   * One after the other each product ends in a round of tiles that fills some compute units, and with the few tiles of a small batch
//     that may be its only one; together the second product's tiles start wherever the first one's have ended.  One tile per workgroup,
//     longer tiles first, and the hardware deals them out as compute units come free (a tile's workgroup has the compute unit's LDS to
//     itself); pick_backward has the rule and the figures.
//   * Any of four tile shapes for either product, chosen by the host.
struct BackwardParams {
  GemmParams gemm[2];          // 0: grad_out . W, block scales; 1: grad_out^T . x, per-row scales
  int shape[2];                // TileShape
  int first[2], wgs[2];        // each product's workgroups (a multiple of 8 apart: the XCD is the workgroup's number modulo 8)
  int sums_first;              // from here on: column sums, 512 a workgroup
  const float* part;
  int blocks;
  uint16_t* sums;
};

enum TileShape { k256x256, k128x256, k128x128, k64x128, k64x64, k64x256 /* SwiGLU epilogue */ };

// ACC: added onto fp32
template <int MODE, bool ACC = false>
__device__ __forceinline__ void backward_tile(const GemmParams& p, int shape, int pid, int nwg, uint8_t* lds) {
  const ExpertChunk none{0, 0, 0, 0, 0};
  if (shape == k256x256) gemm_tiles<MODE, kDense, ACC, ACC, MODE != kScaleTensor, 0, 4, 8, 2>(p, lds, none, pid, nwg);
  else if (shape == k128x256) gemm_tiles<MODE, kDense, ACC, ACC, false, 0, 2, 8, 2>(p, lds, none, pid, nwg);
  else if (shape == k128x128) gemm_tiles<MODE, kDense, ACC, ACC, false, 0, 2, 4, 2>(p, lds, none, pid, nwg);
  else gemm_tiles<MODE, kDense, ACC, ACC, false, 0, 1, 2, 4>(p, lds, none, pid, nwg);
}
constexpr int backward_lds(int mode) {
  int most = 0;
  const int of[] = {tile_lds(mode, 4, 256), tile_lds(mode, 2, 256), tile_lds(mode, 2, 128), tile_lds(mode, 1, 128)};
  for (int v : of) most = v > most ? v : most;
  return most;
}

template <int MODE, int MODE_W, bool ACC = false>
__global__ __launch_bounds__(512) void gemm_backward_kernel(const BackwardParams q) {
  static_assert(tile_threads(4, 2) == 512 && tile_threads(2, 2) == 512 && tile_threads(1, 4) == 512, "");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[backward_lds(MODE) > backward_lds(MODE_W) ? backward_lds(MODE) : backward_lds(MODE_W)];
  const int wg = blockIdx.x;
  if (wg >= q.sums_first) {
    const int col = (wg - q.sums_first) * 512 + threadIdx.x;
    if (col < q.gemm[1].M) q.sums[col] = __builtin_bit_cast(uint16_t, (__bf16)column_sum_in_block_order(q.part, q.blocks, q.gemm[1].M, col));
    return;
  }
  const int one = wg >= q.first[1] && wg < q.first[1] + q.wgs[1];
  const int pid = wg - q.first[one];
  if (pid < 0 || pid >= q.wgs[one]) return;       // (behind a first product of fewer than 8 workgroups)
  if (one) backward_tile<MODE_W, ACC>(q.gemm[1], q.shape[1], pid, q.wgs[1], lds);
  else backward_tile<MODE>(q.gemm[0], q.shape[0], pid, q.wgs[0], lds);
}

// Test hook.  0: pick_shape and the rules below choose the form; 1: always 256 x 256 tiles; 2: the smallest tile a form has;
// 3: 128 x 256, 4: 128 x 128 and 5: 64 x 128 tiles where a form has them
static std::atomic<int> g_small_gemm_mode{0};   // (atomic: the test hook may be called from any thread)

// Workgroups to launch for `tiles` tiles: at most one per CU, a multiple of 8 (one share per XCD) unless there are fewer
// than 8 tiles.  Rounded up, so that a single round of tiles stays one (up to seven workgroups find no tile and leave):
// rounded down, 130 tiles on 128 workgroups took two rounds (block 256 x 8320 x 8448: 86 us, 47 so).
static int persistent_grid(int64_t tiles) {
  static const int cus = [] {           // (initialised once, also when the first calls come from several threads)
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  if (tiles < kXcds || cus < kXcds) return (int)(tiles < cus ? tiles : cus);
  const int64_t up = (tiles + kXcds - 1) / kXcds * kXcds, most = cus - cus % kXcds;
  return (int)(up < most ? up : most);
}

// The tile of a GEMM: 256 x 256 (8 waves), 128 x 256, 128 x 128 or 64 x 128 (4 waves that multiply, 4 that fetch) or 64 x 64 (2 and 4).
static int64_t shape_rows(TileShape shape) { return shape == k256x256 ? 256 : (shape == k128x256 || shape == k128x128 ? 128 : 64); }
static int64_t shape_cols(TileShape shape) { return shape == k64x64 ? 64 : (shape == k128x128 || shape == k64x128 ? 128 : 256); }

static int64_t tile_count(int64_t M, int64_t N, TileShape shape) {
  const int64_t tm = shape_rows(shape), tn = shape_cols(shape);
  return ((M + tm - 1) / tm) * ((N + tn - 1) / tn);
}

// Grouped by rows: the most tiles there can be (every expert with rows ends in a partial one).
static int64_t most_grouped_tiles(int64_t M, int64_t N, int64_t experts, TileShape shape) {
  const int64_t tm = shape_rows(shape), tn = shape_cols(shape), used = experts < M ? experts : M;
  return (M + used * (tm - 1)) / tm * ((N + tn - 1) / tn);
}

// The smallest tile with which the problem is still one round, one tile per compute unit; problems of several rounds
// take 256 x 256, which moves the fewest bytes through L2 and LDS per product, or 128 x 256 (better_low).  A workgroup's round trip per k-block
// is bound by what its compute unit's vector-memory path and LDS move, so with idle units a smaller tile is less work
// on the same critical path.  us with 256 x 256 / 128 x 256 / 128 x 128 / 64 x 128 tiles (tiles of the one taken):
//   block   256 x 7168 x 7168    80 / 53 / 39 / 30 (224)         512 x 7168 x 7168    79 / 52 / 39 / 51 (224)
//   block  1000 x 7168 x 7168    81 / 54 / 66 / 89 (224)        2048 x 7168 x 7168    91 / 103 / 124 / 152 (224)
//   block  1000 x 2048 x 4096    40 / 27 / 18 / 15 (256)        1400 x 2048 x 4096    40 / 27 / 18 / 25 (176)
//   block  1400 x 3072 x 3072    32 / 22 / 27 / 29 (132)
//   block  1531 x 7168 x 2048 (168 / 336 / 672 tiles)  26 / 31 / 30        4096 x 4096 x 4096  57 / 62 / 75
//   pow2   2048 x 4096 x 7168    76 / 51 / 65                   rows   2048 x 1024 x 4096    51 / 33 / 33 / 17
// and with 128 x 128 / 64 x 128 / 64 x 64 (up to 256 of the last)
//   block   128 x 7168 x 7168    39 / 31 / 23 (224)              400 x 1024 x 8192    29 / 22 / 20 (112)
//   rows, onto c  1024 x 1024 x 4096   23 / 18 / 16 (256)        tensor  512 x 1024 x 1024    7.3 / 6.7 / 6.0 (128)
// Between 128 x 256 and 256 x 256 tiles beyond one round: a round of the lower ones takes three fifths of one of the others, so they are
// better where they need three rounds and the others a second one for few tiles.  us with 256 x 256 / 128 x 256:
//   block  2300 x 8192 x 7168 (288 / 576 tiles) 164 / 141       3000 x 7168 x 7168 (336 / 672) 156 / 146
//   block  2000 x 14336 x 7168 (448 / 896)      172 / 193       8200 x 8192 x 2048 (1056 / 2080) 134 / 137
//   rows   4352 x 4096 x 2048 (272 / 544)        61 / 56        pow2  3000 x 7168 x 4096 85 / 78
static bool better_low(int64_t M, int64_t N, int64_t cus) {
  const int64_t low = (tile_count(M, N, k128x256) + cus - 1) / cus, high = (tile_count(M, N, k256x256) + cus - 1) / cus;
  return low == 1 || 3 * low < 5 * high;
}

static TileShape pick_shape(int64_t M, int64_t N) {
  const int mode = g_small_gemm_mode.load(std::memory_order_relaxed);
  const int64_t cus = persistent_grid((int64_t)1 << 40);
  if (mode != 0) return mode == 1 ? k256x256 : (mode == 2 ? k64x64 : (mode == 3 ? k128x256 : (mode == 4 ? k128x128 : k64x128)));
  if (tile_count(M, N, k64x64) <= cus) return k64x64;
  if (tile_count(M, N, k64x128) <= cus) return k64x128;
  if (tile_count(M, N, k128x128) <= cus) return k128x128;
  return better_low(M, N, cus) ? k128x256 : k256x256;
}

// SwiGLU epilogue: a tile's columns are the gate and the up half of one scaling group, 256 in all.  us with 256 / 128 / 64 rows:
//   500 x 8192 x 4096 (64 / 128 / 256 tiles)  46 / 31 / 22      1000 x 12288 x 4096 (192 / 384 / 768)  55 / 61 / 62
//   128 x 8192 x 7168 (32 / 32 / 64)          69 / 44 / 30       400 x 36864 x 7168 (288 / 576 / 1008) 154 / 142 / 136
static TileShape pick_shape_swiglu(int64_t M, int64_t N) {
  const int mode = g_small_gemm_mode.load(std::memory_order_relaxed);
  if (mode != 0) return mode == 1 ? k256x256 : (mode == 2 ? k64x256 : k128x256);
  const int64_t cus = persistent_grid((int64_t)1 << 40);
  if (tile_count(M, N, k64x256) <= cus) return k64x256;
  return better_low(M, N, cus) ? k128x256 : k256x256;
}

// Grouped by rows every expert ends in a partial tile, which costs as much as a whole one, so with few rows per expert low
// tiles are better, with many (or the rows of many with one expert) high ones; the rows of an expert are known on the device
// only.  Where even the most 64 x 64 or 64 x 128 tiles there can be are one round: those.  Of more than 256 rows per expert on average and
// two rounds of 256 x 256 tiles or more: those.  In between the kernel chooses (grouped_tile_rows).  us with 64 / 128 / 256 rows per
// tile, for rows spread evenly / by Zipf's law / half with one expert / all with one; one weight for every call, so that those of 8 and 16
// experts stay in the Infinity Cache (second lines: several in turn, so that none does):
//   32 experts [4096, 7168],   512 rows   141 / 140 / 189   158 / 177 / 180   156 / 174 / 245    23 /  42 /  64
//                             2048 rows   151 / 144 / 197   226 / 185 / 251   199 / 182 / 252    77 /  53 /  71
//                             8192 rows   441 / 249 / 226   484 / 296 / 301   496 / 346 / 295   314 / 201 / 179
//   8 experts  [4096, 7168],   512 rows    37 /  43 /  66    54 /  43 /  66    54 /  44 /  66    23 /  42 /  64
//                                          45 /  59 /  80    66 /  60 /  81    64 /  57 /  80    23 /  42 /  64
//   16 experts [1024, 4096],  2048 rows    16 /  26 /  40    29 /  27 /  40    27 /  27 /  40    15 /  26 /  40
//                                          22 /  33 /  47    35 /  33 /  47    32 /  32 /  47    16 /  27 /  40
//   64 experts [2048, 2048], 16384 rows   148 /  75 /  69   150 /  93 / 112   157 / 103 /  98   105 /  65 /  58
enum GroupedTiles { kSmallestTiles, kLowestTiles, kHighTiles, kChosenTiles, kLowTiles /* test hook: as chosen */ };

static GroupedTiles pick_grouped(int64_t M, int64_t N, int experts) {
  const int mode = g_small_gemm_mode.load(std::memory_order_relaxed);
  if (mode != 0) return mode == 1 ? kHighTiles : (mode == 2 ? kSmallestTiles : (mode == 5 ? kLowestTiles : kLowTiles));
  const int64_t cus = persistent_grid((int64_t)1 << 40);
  if (most_grouped_tiles(M, N, experts, k64x64) <= cus) return kSmallestTiles;
  if (most_grouped_tiles(M, N, experts, k64x128) <= cus) return kLowestTiles;
  return M > (int64_t)256 * experts && M / 256 * ((N + 255) / 256) >= 2 * cus ? kHighTiles : kChosenTiles;
}

static int64_t few_rows(int64_t N, int64_t K) {        // the most rows that count as few
  return K >= kSkinnyMinK && g_small_gemm_mode.load(std::memory_order_relaxed) == 0 ? skinny_rows(N, K) : 0;
}

// Both products of a linear's backward in one launch (gemm_backward_kernel) where that is shorter by more than a thirty-second: the time
// at which the last tile ends when the longer ones are dealt out first, for any of four shapes each, against the rounds of two launches
// and what lies between them.  A tile's time is that of its k-blocks in a full round and, for its first k-block and its stores, about
// what a launch of one such tile takes (ns).  us in three launches / in one, tokens x outputs x inputs:
//   block  1531 x 2048 x 7168     57 / 51       1400 x 4096 x 4096   61 / 53       2048 x 1024 x 1024  17.7 / 10.3
//   block   256 x 1024 x 1024   13.4 / 7.5       512 x 4096 x 4096   32 / 25       8192 x 1024 x 1024  39.3 / 31.5
//   block  4096 x 7168 x 7168    391 / 364      5000 x 5120 x 13824  659 / 633     3000 x 7168 x 2048   100 / 93
//   pow2    750 x 2432 x 3840   28.3 / 17.9     tensor  2048 x 1024 x 1024  15.5 / 9.4     1024 x 4096 x 2048  26.5 / 18.9
// Whole rounds, and many of them, are as fast one after the other: 4096 x 7168 x 16384 806 / 806 to 818.  Added onto fp32 a tile also waits for its
// old values, all tiles of a round at once where they are a launch of their own (two launches / one): block 4096 x 7168 x 7168 448 / 400,
// 2048 x 7168 x 4096 149 / 131, 1006 x 9472 x 3456 135 / 100, pow2 2048 x 7168 x 4096 137 / 124; without that time in the model pow2 2048 x
// 7168 x 4096 stayed with two launches, and block 300 x 1024 x 16384 took 49.9 in one where two take 42.6.
// Drawn over 1 to 8192 tokens and 128 to 16384 features, all recipes: where this chooses one launch (21272 sizes) it takes 0.69 of the two
// or three launches' time on average and in 1.1 % of them over 3 % more, most often for some hundred tokens, many outputs and few inputs
// (tensor 73 x 10752 x 1024 30.6 / 35.8), whose first product alone would take 64 x 64 tiles.
static int64_t tile_time(TileShape shape, int64_t kblocks) {
  switch (shape) {
    case k256x256: return 5000 + 1300 * kblocks;
    case k128x256: return 3500 + 900 * kblocks;
    case k128x128: return 2500 + 600 * kblocks;
    case k64x128: return 2000 + 440 * kblocks;
    default: return 2000 + 310 * kblocks;
  }
}
constexpr int64_t kLaunchTime = 3000;
static int64_t accumulate_time(TileShape shape) { return 10000 * shape_rows(shape) * shape_cols(shape) / (256 * 256); }      // fp32 read and written

// t1 tiles of d1 each, then t2 tiles of d2 <= d1, each to the compute unit that is free first
static int64_t dealt_out(int64_t t1, int64_t d1, int64_t t2, int64_t d2, int64_t cus) {
  const int64_t rounds = t1 / cus, rest = t1 % cus, low = rounds * d1, high = low + (rest ? d1 : 0);
  auto room = [&](int64_t t) { return (t >= high ? rest * ((t - high) / d2) : 0) + (cus - rest) * ((t - low) / d2); };
  int64_t j_low = high > low ? (high - low + d2 - 1) / d2 : 0, j_high = 0;
  for (int64_t t = high;;) {
    if (room(t) >= t2) return t;
    const int64_t a = low + j_low * d2, b = high + j_high * d2;
    t = a < b ? a : b;
    if (a <= t) ++j_low;
    if (b <= t) ++j_high;
  }
}

static bool pick_backward(int64_t M, int64_t N, int64_t K, int64_t padded, int launches, bool accumulate, TileShape shape[2]) {
  const int mode = g_small_gemm_mode.load(std::memory_order_relaxed);
  const TileShape shapes[] = {k256x256, k128x256, k128x128, k64x128};
  if (mode != 0) {                       // (test hook: that shape for both)
    if (mode == 2) return false;
    shape[0] = shape[1] = mode == 1 ? k256x256 : (mode == 3 ? k128x256 : (mode == 4 ? k128x128 : k64x128));
    return true;
  }
  if (M <= few_rows(K, N)) return false;
  const int64_t cus = persistent_grid((int64_t)1 << 40);
  const int64_t kb[2] = {N / BK, padded / BK}, rows[2] = {M, N};
  int64_t apart = (launches - 1) * kLaunchTime;
  for (int i = 0; i < 2; ++i) {
    const TileShape s = pick_shape(rows[i], K);
    const int64_t rounds = (tile_count(rows[i], K, s) + cus - 1) / cus;
    apart += tile_time(s, rounds * kb[i]) + (i && accumulate ? rounds * accumulate_time(s) : 0);      // (its tiles follow each other without a gap)
  }
  int64_t best = INT64_MAX, best_end = 0;
  for (TileShape s0 : shapes)
    for (TileShape s1 : shapes) {
      const int64_t t[2] = {tile_count(rows[0], K, s0), tile_count(rows[1], K, s1)};
      const int64_t d[2] = {tile_time(s0, kb[0]), tile_time(s1, kb[1]) + (accumulate ? accumulate_time(s1) : 0)};
      const int longer = d[1] > d[0] ? 1 : 0;
      const int64_t end = dealt_out(t[longer], d[longer], t[1 - longer], d[1 - longer], cus);
      const int64_t cost = end + (t[0] * d[0] + t[1] * d[1]) / (8 * cus);       // (of forms that end together the one with less to move)
      if (cost < best) {
        best = cost;
        best_end = end;
        shape[0] = s0;
        shape[1] = s1;
      }
    }
  return best_end < apart - apart / 32;
}

// Below this contraction a fused epilogue on tiles is still the better choice with few rows than the few-rows form and a launch
// behind it: what those save on the GPU (weight [8192, 1024], 8 rows 11.6 -> 9.0 us; [36864, 512], 64 rows 9.9 -> 13.5) the second
// call costs on the host (15 -> 25 us).
constexpr int64_t kEpilogueMaxK = 2048;
static_assert(kEpilogueMaxK >= kSkinnyAnyWidthK, "hpfp8_gemm_few_rows knows no width");

// Few rows of a (decode): bound by reading b once, which the tile kernels do not reach (gemm_skinny.hip; 8 rows of
// [7168, 16384]: 60 us with 64 x 128 tiles, 20.6 us; 64 rows: 64 and 26.8 us; 37 rows of [36864, 7168]: 81 us with 256 x 256
// tiles, 41.6 us), with the same bits.  try_skinny hands the problem over if it is one; otherwise false.
static bool try_skinny(const GemmParams& p, SkinnyMode mode, int out_type, hipStream_t stream, int& rc) {
  if (p.accumulate || p.M > few_rows(p.N, p.K)) return false;
  SkinnyParams q{};
  q.a = p.a; q.b = p.b; q.sa = p.sa; q.sb = p.sb; q.lda = p.lda; q.ldb = p.ldb;
  q.sa_sm = p.sa_sm; q.sa_sk = p.sa_sk; q.sb_sn = p.sb_sn; q.sb_sk = p.sb_sk; q.sb_bytes = p.sb_bytes;
  q.bias = p.bias; q.c = p.c; q.ldc = p.ldc; q.M = p.M; q.N = p.N; q.K = p.K; q.out_f32 = out_type == HPFP8_OUT_F32;
  rc = launch_skinny(q, mode, persistent_grid((int64_t)1 << 40), stream);
  return true;
}

template <int MODE, int GROUPED, bool SA4, int WM, int NS, int WN>
static int launch_sa(const GemmParams& p, int out_type, int64_t tiles, hipStream_t stream) {
  dim3 grid((unsigned)persistent_grid(tiles)), block(tile_threads(WM, WN));
  if (out_type == HPFP8_OUT_F32) {
    if constexpr (MODE != kScaleTensor && GROUPED == kDense) {   // (the per-tensor and grouped entry points have no accumulate)
      if (p.accumulate) {
        gemm_kernel<MODE, GROUPED, true, true, SA4, 0, WM, NS, WN><<<grid, block, 0, stream>>>(p);
        return check_launch("gemm");
      }
    }
    gemm_kernel<MODE, GROUPED, true, false, SA4, 0, WM, NS, WN><<<grid, block, 0, stream>>>(p);
  } else {
    gemm_kernel<MODE, GROUPED, false, false, SA4, 0, WM, NS, WN><<<grid, block, 0, stream>>>(p);
  }
  return check_launch("gemm");
}

template <int MODE, int GROUPED, int WM, int NS, int WN>
static int launch_shape(const GemmParams& p, int out_type, int64_t tiles, hipStream_t stream) {
  if constexpr (GROUPED == kGroupedK) return launch_sa<MODE, GROUPED, true, WM, NS, WN>(p, out_type, tiles, stream);   // (sa_sm = 1)
  if constexpr (MODE != kScaleTensor && !fetchers(WM)) {      // (fetched to LDS, sa may have any strides)
    if (p.sa_sm == 1) return launch_sa<MODE, GROUPED, true, WM, NS, WN>(p, out_type, tiles, stream);
  }
  if constexpr (GROUPED != kGroupedK) return launch_sa<MODE, GROUPED, false, WM, NS, WN>(p, out_type, tiles, stream);
}

template <int MODE, int GROUPED>
static int launch(GemmParams p, int out_type, TileShape shape, hipStream_t stream) {
  int64_t tiles = tile_count(p.M, p.N, shape);
  p.tiles = (int)tiles;                        // (grouped by rows: the kernel counts the experts' own tiles)
  if (GROUPED == kGroupedK) tiles *= p.experts;
  // upper bound on row tiles: every expert may add one partial tile
  if (GROUPED == kGroupedRows) tiles = most_grouped_tiles(p.M, p.N, p.experts, shape);
  if constexpr (GROUPED == kDense) {
    if (shape == k128x256) return launch_shape<MODE, GROUPED, 2, 8, 2>(p, out_type, tiles, stream);
    if (shape == k128x128) return launch_shape<MODE, GROUPED, 2, 4, 2>(p, out_type, tiles, stream);
  }
  if constexpr (GROUPED != kGroupedK) {
    if (shape == k64x128) return launch_shape<MODE, GROUPED, 1, 2, 4>(p, out_type, tiles, stream);
    if (shape == k64x64) return launch_shape<MODE, GROUPED, 1, 2, 2>(p, out_type, tiles, stream);
  }
  return launch_shape<MODE, GROUPED, 4, 8, 2>(p, out_type, tiles, stream);
}

template <int MODE>
static int launch_grouped(GemmParams p, int out_type, hipStream_t stream) {
  const GroupedTiles tiles = pick_grouped(p.M, p.N, p.experts);
  if (tiles == kSmallestTiles) return launch<MODE, kGroupedRows>(p, out_type, k64x64, stream);
  if (tiles == kLowestTiles) return launch<MODE, kGroupedRows>(p, out_type, k64x128, stream);
  if (tiles == kHighTiles) return launch<MODE, kGroupedRows>(p, out_type, k256x256, stream);
  p.choose_cus = tiles == kLowTiles ? -128 : persistent_grid((int64_t)1 << 40);
  dim3 grid((unsigned)persistent_grid(most_grouped_tiles(p.M, p.N, p.experts, k64x128))), block(512);
  const bool sa4 = p.sa_sm == 1;
  if (out_type == HPFP8_OUT_F32) {
    if (sa4) gemm_grouped_kernel<MODE, true, true><<<grid, block, 0, stream>>>(p);
    else gemm_grouped_kernel<MODE, true, false><<<grid, block, 0, stream>>>(p);
  } else {
    if (sa4) gemm_grouped_kernel<MODE, false, true><<<grid, block, 0, stream>>>(p);
    else gemm_grouped_kernel<MODE, false, false><<<grid, block, 0, stream>>>(p);
  }
  return check_launch("gemm (grouped)");
}

static int check_common(const char* what, const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                        const float* sb, int64_t M, int64_t N, int64_t K, const void* bias, const void* c,
                        int64_t ldc, int out_type, int accumulate) {
  HPFP8_REQUIRE(M >= 0 && N >= 0 && K >= 0, HPFP8_ERR_SHAPE, "%s: negative shape", what);
  HPFP8_REQUIRE(K > 0 && K % BK == 0 && N % kBlock == 0, HPFP8_ERR_SHAPE,
                "%s: K=%lld must be a positive multiple of 128 and N=%lld a multiple of 128", what, (long long)K,
                (long long)N);
  HPFP8_REQUIRE(out_type == HPFP8_OUT_BF16 || out_type == HPFP8_OUT_F32, HPFP8_ERR_ARG, "%s: bad out_type", what);
  HPFP8_REQUIRE(!accumulate || out_type == HPFP8_OUT_F32, HPFP8_ERR_ARG, "%s: accumulate needs fp32 output", what);
  HPFP8_REQUIRE(lda >= K && ldb >= K && lda % 16 == 0 && ldb % 16 == 0, HPFP8_ERR_SHAPE,
                "%s: lda=%lld and ldb=%lld must be multiples of 16 and at least K=%lld", what, (long long)lda,
                (long long)ldb, (long long)K);
  HPFP8_REQUIRE(ldc >= N, HPFP8_ERR_SHAPE, "%s: ldc=%lld smaller than N=%lld", what, (long long)ldc, (long long)N);
  // rows of c are written in 16-byte pieces
  HPFP8_REQUIRE(ldc % (out_type == HPFP8_OUT_F32 ? 4 : 8) == 0, HPFP8_ERR_ALIGN,
                "%s: ldc must be a multiple of %d", what, out_type == HPFP8_OUT_F32 ? 4 : 8);
  if (M == 0 || N == 0) return HPFP8_OK;
  HPFP8_REQUIRE(a && b && sa && sb && c, HPFP8_ERR_ARG, "%s: null buffer", what);
  HPFP8_REQUIRE(aligned16(a) && aligned16(b) && aligned16(c) && (!bias || aligned16(bias)), HPFP8_ERR_ALIGN,
                "%s: buffers must be 16-byte aligned", what);
  // 32-bit byte offsets inside one tile's buffer resource (256 rows); the operands themselves may be
  // of any size
  HPFP8_REQUIRE(BM * lda < (int64_t)0x7FFFFFFF && BN * ldb < (int64_t)0x7FFFFFFF, HPFP8_ERR_SHAPE,
                "%s: a row stride of 8 MiB or more is not supported", what);
  HPFP8_REQUIRE(M < (int64_t)0x7FFFFF00 && N < (int64_t)0x7FFFFF00, HPFP8_ERR_SHAPE, "%s: M or N too large", what);
  // a tile's 256 rows of c are stored (and its old values read) with 32-bit byte offsets
  HPFP8_REQUIRE(BM * ldc * 4 < (int64_t)0x7FFFF000, HPFP8_ERR_SHAPE, "%s: the row stride of c must stay below 8 MiB", what);
  return 1;
}

// Scale arrays are addressed with 32-bit byte offsets inside the kernels.
static int check_scale_span(const char* what, int64_t rows, int64_t kblocks, int64_t stride_r, int64_t stride_k,
                            const char* name) {
  HPFP8_REQUIRE(stride_r >= 0 && stride_k >= 0, HPFP8_ERR_SHAPE, "%s: negative %s stride", what, name);
  if (rows == 0) return 1;
  HPFP8_REQUIRE(((rows - 1) * stride_r + (kblocks - 1) * stride_k + 1) * 4 < (int64_t)0x7FFFFFFF, HPFP8_ERR_SHAPE,
                "%s: the %s array spans 2 GiB or more", what, name);
  return 1;
}

}  // namespace hpfp8

using namespace hpfp8;

extern "C" {

// checks and kernel arguments of a product with block scales or (sb_gran 1) per-row scales; 1: there is something to launch
static int blockwise_params(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                            const void* b, int64_t ldb, const float* sb, int64_t sb_stride_n, int64_t sb_stride_k,
                            int sb_gran, int64_t M, int64_t N, int64_t K, const void* bias, void* c,
                            int64_t ldc, int out_type, int accumulate, GemmParams& p) {
  HPFP8_REQUIRE(sb_gran == 1 || sb_gran == 128, HPFP8_ERR_ARG, "gemm_blockwise: sb_gran must be 1 or 128");
  int rc = check_common("gemm_blockwise", a, lda, b, ldb, sa, sb, M, N, K, bias, c, ldc, out_type, accumulate);
  if (rc <= 0) return rc;
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.sa = sa; p.sb = sb; p.lda = lda; p.ldb = ldb;
  p.sa_sm = sa_stride_m; p.sa_sk = sa_stride_k; p.sb_sn = sb_stride_n; p.sb_sk = sb_stride_k;
  rc = check_scale_span("gemm_blockwise", M, K / BK, sa_stride_m, sa_stride_k, "sa");
  if (rc <= 0) return rc;
  rc = check_scale_span("gemm_blockwise", sb_gran == 128 ? N / kBlock : N, K / BK, sb_stride_n, sb_stride_k, "sb");
  if (rc <= 0) return rc;
  p.sb_bytes = (int)(((N / kBlock - 1) * sb_stride_n + (K / BK - 1) * sb_stride_k + 1) * 4);
  p.c = c; p.ldc = ldc; p.bias = (const uint16_t*)bias;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.accumulate = accumulate;
  if (sb_gran == 128) return 1;
  // per-row b scales are read with unit stride: 1 KB per k-block to LDS (powers of two, 256 x 256 tiles), 256 bytes per fetching wave, or
  // into registers
  if (K == BK) sb_stride_k = N;     // a single k-block: the stride between k-blocks is never used
  p.sb_sk = sb_stride_k;
  HPFP8_REQUIRE(sb_stride_n == 1 && sb_stride_k >= N && sb_stride_k % 4 == 0 && aligned16(sb), HPFP8_ERR_SHAPE,
                "gemm_blockwise: with sb_gran=1 the b scales must be k-block-major (sb_stride_n = 1, sb_stride_k >= N, "
                "16-byte aligned rows)");
  HPFP8_REQUIRE(((K / BK - 1) * sb_stride_k + N) * 4 < (int64_t)0x7FFFFFFF, HPFP8_ERR_SHAPE,
                "gemm_blockwise: b scale array too large");
  return 1;
}

static int launch_blockwise(const GemmParams& p, int sb_gran, int out_type, bool pow2, hipStream_t stream) {
  const TileShape shape = pick_shape(p.M, p.N);
  int rc;
  if (sb_gran == 128) {
    if (try_skinny(p, pow2 ? kSkinnyPow2 : kSkinnyBlock, out_type, stream, rc)) return rc;
    if (pow2) return launch<kScalePow2, kDense>(p, out_type, shape, stream);
    return launch<kScaleBlock, kDense>(p, out_type, shape, stream);
  }
  if (pow2) return launch<kScalePow2Row, kDense>(p, out_type, shape, stream);
  return launch<kScaleRow, kDense>(p, out_type, shape, stream);
}

static int per_tensor_params(const void* a, int64_t lda, const float* sa_inv, const void* b, int64_t ldb, const float* sb_inv, int64_t M,
                             int64_t N, int64_t K, const void* bias, void* c, int64_t ldc, int out_type, GemmParams& p) {
  int rc = check_common("gemm_per_tensor", a, lda, b, ldb, sa_inv, sb_inv, M, N, K, bias, c, ldc, out_type, 0);
  if (rc <= 0) return rc;
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.sa = sa_inv; p.sb = sb_inv; p.lda = lda; p.ldb = ldb;
  p.c = c; p.ldc = ldc; p.bias = (const uint16_t*)bias;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  return 1;
}

static int launch_per_tensor(const GemmParams& p, int out_type, hipStream_t stream) {
  int rc;
  if (try_skinny(p, kSkinnyTensor, out_type, stream, rc)) return rc;
  return launch<kScaleTensor, kDense>(p, out_type, pick_shape(p.M, p.N), stream);
}

static int gemm_blockwise_impl(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                               const void* b, int64_t ldb, const float* sb, int64_t sb_stride_n, int64_t sb_stride_k,
                               int sb_gran, int64_t M, int64_t N, int64_t K, const void* bias, void* c,
                               int64_t ldc, int out_type, int accumulate, bool pow2, hpfp8_stream_t stream) {
  GemmParams p{};
  const int rc = blockwise_params(a, lda, sa, sa_stride_m, sa_stride_k, b, ldb, sb, sb_stride_n, sb_stride_k, sb_gran, M, N, K, bias, c, ldc,
                                  out_type, accumulate, p);
  return rc <= 0 ? rc : launch_blockwise(p, sb_gran, out_type, pow2, (hipStream_t)stream);
}

int hpfp8_gemm_blockwise(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                         const void* b, int64_t ldb, const float* sb, int64_t sb_stride_n, int64_t sb_stride_k,
                         int sb_gran, int64_t M, int64_t N, int64_t K, const void* bias, void* c,
                         int64_t ldc, int out_type, int accumulate, hpfp8_stream_t stream) {
  return gemm_blockwise_impl(a, lda, sa, sa_stride_m, sa_stride_k, b, ldb, sb, sb_stride_n, sb_stride_k, sb_gran, M, N, K,
                             bias, c, ldc, out_type, accumulate, false, stream);
}

int hpfp8_gemm_blockwise_pow2(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                              const void* b, int64_t ldb, const float* sb, int64_t sb_stride_n, int64_t sb_stride_k,
                              int sb_gran, int64_t M, int64_t N, int64_t K, const void* bias, void* c, int64_t ldc,
                              int out_type, int accumulate, hpfp8_stream_t stream) {
  return gemm_blockwise_impl(a, lda, sa, sa_stride_m, sa_stride_k, b, ldb, sb, sb_stride_n, sb_stride_k, sb_gran, M, N, K,
                             bias, c, ldc, out_type, accumulate, true, stream);
}

int hpfp8_gemm_blockwise_swiglu_quantize(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m,
                                         int64_t sa_stride_k, const void* b, int64_t ldb, const float* sb,
                                         int64_t sb_stride_n, int64_t sb_stride_k, int64_t M, int64_t inter, int64_t K,
                                         int fast, int pow2, int pow2_out, void* q, int64_t ldq, float* scale,
                                         float* scale_inv, hpfp8_stream_t stream) {
  const char* what = "gemm_blockwise_swiglu_quantize";
  HPFP8_REQUIRE((fast == 0 || fast == 1) && (pow2 == 0 || pow2 == 1) && (pow2_out == 0 || pow2_out == 1), HPFP8_ERR_ARG,
                "%s: fast, pow2 and pow2_out must be 0 or 1", what);
  HPFP8_REQUIRE(inter >= 0 && inter % kBlock == 0 && inter < (1 << 29), HPFP8_ERR_SHAPE,
                "%s: the activation's width %lld must be a multiple of 128", what, (long long)inter);
  HPFP8_REQUIRE(ldq >= inter && ldq % 16 == 0, HPFP8_ERR_SHAPE, "%s: ldq=%lld must be a multiple of 16 and at least the width",
                what, (long long)ldq);
  // (the common checks see the gate/up matrix this call does not write, [M, 2 * inter]; the code matrix it does
  // write is checked here: a tile's 256 rows are addressed with 32-bit byte offsets)
  HPFP8_REQUIRE(BM * ldq < (int64_t)0x7FFFF000, HPFP8_ERR_SHAPE, "%s: the row stride of q must stay below 8 MiB", what);
  int rc = check_common(what, a, lda, b, ldb, sa, sb, M, 2 * inter, K, nullptr, q, 2 * inter, HPFP8_OUT_F32, 0);
  if (rc <= 0) return rc;
  HPFP8_REQUIRE(scale_inv != nullptr, HPFP8_ERR_ARG, "%s: null scale_inv", what);
  // the up rows of a b tile are addressed `inter` rows past its gate rows, inside one buffer resource
  HPFP8_REQUIRE(2 * inter * ldb < (int64_t)0x7FFFF000, HPFP8_ERR_SHAPE, "%s: the weight's codes must span less than 2 GiB", what);
  GemmParams p{};
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.sa = sa; p.sb = sb; p.lda = lda; p.ldb = ldb;
  p.sa_sm = sa_stride_m; p.sa_sk = sa_stride_k; p.sb_sn = sb_stride_n; p.sb_sk = sb_stride_k;
  rc = check_scale_span(what, M, K / BK, sa_stride_m, sa_stride_k, "sa");
  if (rc <= 0) return rc;
  rc = check_scale_span(what, 2 * inter / kBlock, K / BK, sb_stride_n, sb_stride_k, "sb");
  if (rc <= 0) return rc;
  p.sb_bytes = (int)(((2 * inter / kBlock - 1) * sb_stride_n + (K / BK - 1) * sb_stride_k + 1) * 4);
  p.c = q; p.ldc = ldq;
  p.M = (int)M; p.N = (int)(2 * inter); p.K = (int)K;
  p.inter = (int)inter; p.pow2_out = pow2_out; p.q_scale = scale; p.q_scale_inv = scale_inv;
  const TileShape shape = pick_shape_swiglu(M, 2 * inter);
  const int64_t tiles = tile_count(M, 2 * inter, shape);
  p.tiles = (int)tiles;
  dim3 grid((unsigned)persistent_grid(tiles)), block(512);
  static_assert(tile_threads(4, 2) == 512 && tile_threads(2, 2) == 512 && tile_threads(1, 4) == 512, "");
  hipStream_t st = (hipStream_t)stream;
  const bool sa4 = sa_stride_m == 1;
#define HPFP8_LAUNCH_EPI(MODE, SA4, EPI) \
  do { \
    if (shape == k256x256) gemm_kernel<MODE, kDense, false, false, SA4, EPI, 4><<<grid, block, 0, st>>>(p); \
    else if (shape == k64x256) gemm_kernel<MODE, kDense, false, false, false, EPI, 1, 4, 4><<<grid, block, 0, st>>>(p); \
    else gemm_kernel<MODE, kDense, false, false, false, EPI, 2><<<grid, block, 0, st>>>(p); \
  } while (0)
  if (pow2) {
    if (sa4) { if (fast) HPFP8_LAUNCH_EPI(kScalePow2, true, 2); else HPFP8_LAUNCH_EPI(kScalePow2, true, 1); }
    else { if (fast) HPFP8_LAUNCH_EPI(kScalePow2, false, 2); else HPFP8_LAUNCH_EPI(kScalePow2, false, 1); }
  } else {
    if (sa4) { if (fast) HPFP8_LAUNCH_EPI(kScaleBlock, true, 2); else HPFP8_LAUNCH_EPI(kScaleBlock, true, 1); }
    else { if (fast) HPFP8_LAUNCH_EPI(kScaleBlock, false, 2); else HPFP8_LAUNCH_EPI(kScaleBlock, false, 1); }
  }
#undef HPFP8_LAUNCH_EPI
  return check_launch(what);
}

void hpfp8_debug_set_small_gemm(int mode) { g_small_gemm_mode.store(mode >= 1 && mode <= 5 ? mode : 0, std::memory_order_relaxed); }

int64_t hpfp8_gemm_few_rows(int64_t K) { return K >= kEpilogueMaxK ? few_rows(kBlock, K) : 0; }

// Up to 8 rows are quantized inside the product (gemm_skinny.hip has the figures).  With few runs of columns and a long contraction
// every compute unit's chain of k-blocks is longer than in two launches and what those cost more is less: us, 8 rows, two / one
// [1024, 10240] 11.0 / 10.1, [1024, 12288] 11.6 / 11.4 (1 row 10.4 / 10.9), [2048, 16384] 13.6 / 14.2, [4096, 16384] 16.2 / 14.4.
int64_t hpfp8_linear_few_rows(int64_t N, int64_t K) {
  if (K > 10240 && 4 * (N / 16) <= 3 * (int64_t)persistent_grid((int64_t)1 << 40)) return 0;
  return few_rows(kBlock, K) > kSkinnyMaxRowsBf16 ? kSkinnyMaxRowsBf16 : few_rows(kBlock, K);
}

int hpfp8_linear_few_rows_bf16(const void* x, const void* b, int64_t ldb, const float* sb, int64_t sb_stride_n, int64_t sb_stride_k,
                               int64_t M, int64_t N, int64_t K, int pow2, const void* bias, void* c, int64_t ldc, int out_type,
                               hpfp8_stream_t stream) {
  const char* what = "linear_few_rows";
  HPFP8_REQUIRE(pow2 == 0 || pow2 == 1, HPFP8_ERR_ARG, "%s: pow2 must be 0 or 1", what);
  HPFP8_REQUIRE(M <= kSkinnyMaxRowsBf16, HPFP8_ERR_SHAPE, "%s: more than %d rows", what, kSkinnyMaxRowsBf16);
  // (rows of x as long as those of the codes that the two launches would make: 8 rows of bf16 are addressed here, not 256)
  int rc = check_common(what, x, K, b, ldb, sb, sb, M, N, K, bias, c, ldc, out_type, 0);
  if (rc <= 0) return rc;
  rc = check_scale_span(what, N / kBlock, K / BK, sb_stride_n, sb_stride_k, "sb");
  if (rc <= 0) return rc;
  SkinnyParams p{};
  p.a = (const uint8_t*)x; p.lda = 2 * K; p.b = (const uint8_t*)b; p.ldb = ldb; p.sb = sb; p.sb_sn = sb_stride_n; p.sb_sk = sb_stride_k;
  p.sb_bytes = (int)(((N / kBlock - 1) * sb_stride_n + (K / BK - 1) * sb_stride_k + 1) * 4);
  p.bias = (const uint16_t*)bias; p.c = c; p.ldc = ldc; p.M = (int)M; p.N = (int)N; p.K = (int)K; p.out_f32 = out_type == HPFP8_OUT_F32;
  return launch_skinny_rows_bf16(p, pow2 != 0, persistent_grid((int64_t)1 << 40), (hipStream_t)stream);
}

int hpfp8_gemm_per_tensor(const void* a, int64_t lda, const float* sa_inv, const void* b, int64_t ldb,
                          const float* sb_inv, int64_t M, int64_t N, int64_t K, const void* bias, void* c,
                          int64_t ldc, int out_type, hpfp8_stream_t stream) {
  GemmParams p{};
  const int rc = per_tensor_params(a, lda, sa_inv, b, ldb, sb_inv, M, N, K, bias, c, ldc, out_type, p);
  return rc <= 0 ? rc : launch_per_tensor(p, out_type, (hipStream_t)stream);
}

int hpfp8_linear_backward(const hpfp8_operand* go, const hpfp8_operand* wt, const hpfp8_operand* go_t, const hpfp8_operand* xt, int64_t M,
                          int64_t N, int64_t K, void* dx, void* dw, int accumulate, const float* partial, void* db, int recipe,
                          hpfp8_stream_t stream) {
  const char* what = "linear_backward";
  HPFP8_REQUIRE(go && wt && go_t && xt && (db == nullptr || partial != nullptr), HPFP8_ERR_ARG, "%s: null argument", what);
  HPFP8_REQUIRE(recipe >= HPFP8_BLOCKWISE && recipe <= HPFP8_PER_TENSOR, HPFP8_ERR_ARG, "%s: bad recipe", what);
  HPFP8_REQUIRE(M > 0 && N > 0 && K > 0, HPFP8_ERR_SHAPE, "%s: bad shape", what);
  HPFP8_REQUIRE(!accumulate || recipe != HPFP8_PER_TENSOR, HPFP8_ERR_ARG, "%s: accumulate is of the blockwise recipes", what);
  const int out_w = accumulate ? HPFP8_OUT_F32 : HPFP8_OUT_BF16;
  const int64_t padded = (M + kBlock - 1) / kBlock * kBlock;
  hipStream_t st = (hipStream_t)stream;
  BackwardParams q{};
  int rc[2];
  if (recipe == HPFP8_PER_TENSOR) {
    rc[0] = per_tensor_params(go->codes, go->ld, go->scale_inv, wt->codes, wt->ld, wt->scale_inv, M, K, N, nullptr, dx, K, HPFP8_OUT_BF16, q.gemm[0]);
    if (rc[0] < 0) return rc[0];
    rc[1] = per_tensor_params(go_t->codes, go_t->ld, go_t->scale_inv, xt->codes, xt->ld, xt->scale_inv, N, K, padded, nullptr, dw, K, HPFP8_OUT_BF16,
                              q.gemm[1]);
  } else {
    rc[0] = blockwise_params(go->codes, go->ld, go->scale_inv, go->stride_r, go->stride_k, wt->codes, wt->ld, wt->scale_inv, wt->stride_r,
                             wt->stride_k, 128, M, K, N, nullptr, dx, K, HPFP8_OUT_BF16, 0, q.gemm[0]);
    if (rc[0] < 0) return rc[0];
    rc[1] = blockwise_params(go_t->codes, go_t->ld, go_t->scale_inv, go_t->stride_r, go_t->stride_k, xt->codes, xt->ld, xt->scale_inv, xt->stride_r,
                             xt->stride_k, 1, N, K, padded, nullptr, dw, K, out_w, accumulate ? 1 : 0, q.gemm[1]);
  }
  if (rc[1] < 0) return rc[1];
  TileShape shape[2];
  const bool k_major = recipe == HPFP8_PER_TENSOR || (go->stride_r == 1 && go_t->stride_r == 1);
  if (k_major && pick_backward(M, N, K, padded, db ? 3 : 2, accumulate != 0, shape)) {
    const int64_t tiles[2] = {tile_count(M, K, shape[0]), tile_count(N, K, shape[1])};
    const int64_t kblocks[2] = {N / BK, padded / BK};
    const int longer = tile_time(shape[1], kblocks[1]) + (accumulate ? accumulate_time(shape[1]) : 0) > tile_time(shape[0], kblocks[0]) ? 1 : 0;
    for (int i = 0; i < 2; ++i) {
      q.gemm[i].tiles = (int)tiles[i];
      q.shape[i] = shape[i];
      q.wgs[i] = (int)(tiles[i] < kXcds ? tiles[i] : (tiles[i] + kXcds - 1) / kXcds * kXcds);
    }
    const int second = (q.wgs[longer] + kXcds - 1) / kXcds * kXcds;
    q.first[longer] = 0;
    q.first[1 - longer] = second;
    q.sums_first = second + q.wgs[1 - longer];
    q.part = partial;
    q.blocks = (int)(padded / kBlock);
    q.sums = (uint16_t*)db;
    const dim3 grid((unsigned)(q.sums_first + (db ? (N + 511) / 512 : 0))), block(512);
    if (recipe == HPFP8_PER_TENSOR) gemm_backward_kernel<kScaleTensor, kScaleTensor><<<grid, block, 0, st>>>(q);
    else if (recipe == HPFP8_BLOCKWISE_POW2 && accumulate) gemm_backward_kernel<kScalePow2, kScalePow2Row, true><<<grid, block, 0, st>>>(q);
    else if (recipe == HPFP8_BLOCKWISE_POW2) gemm_backward_kernel<kScalePow2, kScalePow2Row><<<grid, block, 0, st>>>(q);
    else if (accumulate) gemm_backward_kernel<kScaleBlock, kScaleRow, true><<<grid, block, 0, st>>>(q);
    else gemm_backward_kernel<kScaleBlock, kScaleRow><<<grid, block, 0, st>>>(q);
    return check_launch(what);
  }
  int status = HPFP8_OK;
  if (db) status = hpfp8_column_sum_finish(partial, padded / kBlock, N, db, nullptr, stream);
  for (int i = 0; i < 2 && status == HPFP8_OK; ++i) {
    if (recipe == HPFP8_PER_TENSOR) status = launch_per_tensor(q.gemm[i], HPFP8_OUT_BF16, st);
    else status = launch_blockwise(q.gemm[i], i == 0 ? 128 : 1, i == 0 ? HPFP8_OUT_BF16 : out_w, recipe == HPFP8_BLOCKWISE_POW2, st);
  }
  return status;
}

static int gemm_grouped_impl(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                             const void* b, int64_t ldb, int64_t b_stride_e, const float* sb, int64_t sb_stride_e,
                             int64_t sb_stride_n, int64_t sb_stride_k, const int32_t* offs, int experts,
                             int64_t total_m, int64_t N, int64_t K, void* c, int64_t ldc, int out_type, bool pow2,
                             hpfp8_stream_t stream) {
  HPFP8_REQUIRE(experts >= 0 && experts <= 4096, HPFP8_ERR_SHAPE, "gemm_grouped: bad expert count %d", experts);
  int rc = check_common("gemm_grouped", a, lda, b, ldb, sa, sb, total_m, N, K, nullptr, c, ldc, out_type, 0);
  if (rc <= 0) return rc;
  if (experts == 0) return HPFP8_OK;
  HPFP8_REQUIRE(offs != nullptr, HPFP8_ERR_ARG, "gemm_grouped: null offs");
  HPFP8_REQUIRE(b_stride_e >= 0 && b_stride_e % 16 == 0, HPFP8_ERR_SHAPE,
                "gemm_grouped: the stride between experts' b matrices must be a non-negative multiple of 16 bytes");
  HPFP8_REQUIRE(sb_stride_e >= 0 && sb_stride_n >= 0 && sb_stride_k >= 0, HPFP8_ERR_SHAPE, "gemm_grouped: negative sb stride");
  GemmParams p{};
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.sa = sa; p.sb = sb; p.lda = lda; p.ldb = ldb; p.b_se = b_stride_e;
  p.sa_sm = sa_stride_m; p.sa_sk = sa_stride_k;
  p.sb_sn = sb_stride_n; p.sb_sk = sb_stride_k; p.sb_se = sb_stride_e;
  rc = check_scale_span("gemm_grouped", total_m, K / BK, sa_stride_m, sa_stride_k, "sa");
  if (rc <= 0) return rc;
  const int64_t sb_span = ((int64_t)(experts - 1) * sb_stride_e + (N / kBlock - 1) * sb_stride_n + (K / BK - 1) * sb_stride_k + 1) * 4;
  HPFP8_REQUIRE(sb_span < (int64_t)0x7FFFFFFF, HPFP8_ERR_SHAPE, "gemm_grouped: b scale array exceeds 2 GiB");
  p.sb_bytes = (int)sb_span;
  p.c = c; p.ldc = ldc; p.offs = offs; p.experts = experts;
  p.M = (int)total_m; p.N = (int)N; p.K = (int)K;
  if (pow2) return launch_grouped<kScalePow2>(p, out_type, (hipStream_t)stream);
  return launch_grouped<kScaleBlock>(p, out_type, (hipStream_t)stream);
}

int hpfp8_gemm_grouped_blockwise(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                                 const void* b, const float* sb, const int32_t* offs, int experts,
                                 int64_t total_m, int64_t N, int64_t K, void* c, int64_t ldc, int out_type,
                                 hpfp8_stream_t stream) {
  return gemm_grouped_impl(a, lda, sa, sa_stride_m, sa_stride_k, b, K, N * K, sb, (N / kBlock) * (K / BK), K / BK, 1, offs,
                           experts, total_m, N, K, c, ldc, out_type, false, stream);
}

int hpfp8_gemm_grouped_blockwise_pow2(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m,
                                      int64_t sa_stride_k, const void* b, const float* sb, const int32_t* offs,
                                      int experts, int64_t total_m, int64_t N, int64_t K, void* c, int64_t ldc,
                                      int out_type, hpfp8_stream_t stream) {
  return gemm_grouped_impl(a, lda, sa, sa_stride_m, sa_stride_k, b, K, N * K, sb, (N / kBlock) * (K / BK), K / BK, 1, offs,
                           experts, total_m, N, K, c, ldc, out_type, true, stream);
}

int hpfp8_gemm_grouped_blockwise_strided(const void* a, int64_t lda, const float* sa, int64_t sa_stride_m,
                                         int64_t sa_stride_k, const void* b, int64_t ldb, int64_t b_stride_e,
                                         const float* sb, int64_t sb_stride_e, int64_t sb_stride_n, int64_t sb_stride_k,
                                         const int32_t* offs, int experts, int64_t total_m, int64_t N, int64_t K,
                                         void* c, int64_t ldc, int out_type, int pow2, hpfp8_stream_t stream) {
  HPFP8_REQUIRE(pow2 == 0 || pow2 == 1, HPFP8_ERR_ARG, "gemm_grouped: pow2 must be 0 or 1");
  return gemm_grouped_impl(a, lda, sa, sa_stride_m, sa_stride_k, b, ldb, b_stride_e, sb, sb_stride_e, sb_stride_n,
                           sb_stride_k, offs, experts, total_m, N, K, c, ldc, out_type, pow2 != 0, stream);
}

int hpfp8_gemm_grouped_wgrad(const void* a, int64_t lda, const float* sa, const void* b, int64_t ldb, const float* sb,
                             const int32_t* layout, int experts, int64_t total_m, int64_t N, int64_t K, void* c,
                             int out_type, hpfp8_stream_t stream) {
  const char* what = "gemm_grouped_wgrad";
  HPFP8_REQUIRE(experts >= 0 && experts <= 4096, HPFP8_ERR_SHAPE, "%s: bad expert count %d", what, experts);
  HPFP8_REQUIRE(total_m >= 0 && total_m < (int64_t)0x7FFFFF00, HPFP8_ERR_SHAPE, "%s: bad row count", what);
  HPFP8_REQUIRE(N >= 0 && K >= 0 && N % kBlock == 0 && K % kBlock == 0, HPFP8_ERR_SHAPE,
                "%s: N=%lld and K=%lld must be multiples of 128", what, (long long)N, (long long)K);
  if (experts == 0 || N == 0 || K == 0) return HPFP8_OK;
  // the GEMM behind it: rows = N (rows of grad_out^T), columns = K (rows of x^T), contraction = the padded token axis
  const int64_t padded = (total_m / kBlock + experts) * kBlock;
  int rc = check_common(what, a, lda, b, ldb, sa, sb, N, K, padded, nullptr, c, K, out_type, 0);
  if (rc <= 0) return rc;
  HPFP8_REQUIRE(layout != nullptr, HPFP8_ERR_ARG, "%s: null layout", what);
  HPFP8_REQUIRE(aligned16(sa) && aligned16(sb), HPFP8_ERR_ALIGN, "%s: scale arrays must be 16-byte aligned", what);
  HPFP8_REQUIRE((padded / BK) * (N > K ? N : K) * 4 < (int64_t)0x7FFFFFFF, HPFP8_ERR_SHAPE, "%s: a scale array spans 2 GiB or more", what);
  HPFP8_REQUIRE((int64_t)experts * (((N + BM - 1) / BM) * ((K + BN - 1) / BN)) < (int64_t)0x7FFFFFFF, HPFP8_ERR_SHAPE, "%s: too many tiles", what);
  GemmParams p{};
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b; p.sa = sa; p.sb = sb; p.lda = lda; p.ldb = ldb;
  p.sa_sm = 1; p.sa_sk = N;          // [padded / 128, N]: block-major, as the grouped transposed quantizer writes them
  p.sb_sn = 1; p.sb_sk = K;          // [padded / 128, K]
  p.c = c; p.ldc = K; p.c_se = N * K; p.layout = layout; p.experts = experts;
  p.M = (int)N; p.N = (int)K; p.K = (int)padded;
  return launch<kScaleRow, kGroupedK>(p, out_type, k256x256, (hipStream_t)stream);
}

}  // extern "C"
