// bf16 MFMA GEMM for the Newton-Schulz iteration: C = bf16(alpha * P Q^T + beta * D) on gfx950.
//
// Both operands are K-contiguous (an "NT" product; a Q of K rows has a walk of its own), which is what every Newton-Schulz product
// reduces to once X and X^T are both kept: X X^T, A A^T (A symmetric) and B (X^T)^T.  A workgroup owns
// a BM x BN tile of C; its waves each own a (BM/WM) x (BN/WN) sub-tile built from 16x16x32 bf16 MFMAs
// with fp32 accumulators.  K is walked in slabs of BK = 64: the slab of P and Q is staged in LDS as
// rows of BK bf16 whose 16-byte chunks are XOR-swizzled with the row index: the LDS has 64 banks of 4
// bytes, 256 / (2 BK) rows span them once, so any 16 consecutive rows read at one logical chunk touch every
// bank exactly once and the 128-bit fragment reads are bank-conflict free.  STAGES slabs are resident: the
// next ones stream from HBM straight into LDS (buffer_load ... lds, no register round trip) while the
// current one feeds the MFMAs.
//
// Several problems in one launch.  A launch carries up to 32 products by value in its kernel arguments: small matrices
// fill the machine together and pay for one launch (24 matrices of 1536 x 1024: 1.24 ms for the whole Muon step against
// 6.15 ms with a launch per matrix, stage and fix-up on three streams; two of 512 x 256, with 64 x 64 tiles: 0.12 against 0.38).
//
// Tile order.  In every round of resident workgroups an XCD (block ids congruent mod 8) gets one contiguous eighth of the
// round's tiles and so reuses its L2, while the machine as a whole works on one nearly square block of tiles: the update
// products of 15360 x 5120 and 5120 x 13824 in one launch took 1209 us, against 1260 us when every XCD walks through its own
// contiguous eighth of a matrix's tiles and 1484 us when it walks through its eighth of both matrices' tiles; a plain
// 8192^3 product runs at 1.48 against 1.40 PFLOP/s.  One matrix at a time the orders are within 2 % of each other.
//
// K pieces.  When the tile count is not a multiple of the number of resident workgroups, tiles of the last, partial round
// may be split along K into pieces that fill the machine; each piece leaves an fp32 partial tile in a workspace and a
// small fix-up kernel sums the pieces in split order and runs the epilogue (the kernel boundary is the only
// synchronisation: no fences, no spinning).
#include "muon_gemm.h"

#include "mfsdp_common.h"

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <utility>

namespace mfsdp {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// 16 bytes of a parameter, aligned to one element (global memory takes any alignment at full vector width)
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));

constexpr int kXcds = 8;
constexpr int kSlabK = 64;  // K granularity of the schedule (operands are padded to it); a slab is BK <= 64 wide

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const __bf16 l = static_cast<__bf16>(lo);
  const __bf16 h = static_cast<__bf16>(hi);
  return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, l)) | (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, h)) << 16);
}

__device__ __forceinline__ float bf16_bits_to_float(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

// param[prow][pcol .. pcol + count - 1] <- round(param * decay) + neg_lr * o for the first `count` bf16 values o of `eight`
// (those inside the parameter).  Whole groups use 16-byte accesses aligned to an element only: rows of any length and
// parameters that start anywhere in a shard go the same way.
__device__ __forceinline__ void update_param8(const GemmProblem& a, int dtype, int prow, int pcol, const u32x4& eight, int count = 8) {
  const bool transposed = (a.flags & kGemmUpdateTransposed) != 0;
  const int update_rows = transposed ? a.N : a.M, update_cols = transposed ? a.M : a.N;
  if (prow >= update_rows || pcol >= update_cols) return;
  const int n = update_cols - pcol < count ? update_cols - pcol : count;
  const int64_t at = static_cast<int64_t>(prow) * update_cols + pcol;
  float o[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[2 * e] = __uint_as_float(eight[e] << 16);
    o[2 * e + 1] = __uint_as_float(eight[e] & 0xffff0000u);
  }
  const float decay = a.update_decay, neg_lr = a.update_neg_lr;
  if (dtype == MFSDP_F32) {
    float* p = static_cast<float*>(a.update_param) + at;
    if (n == 8) {
      f32x4 lo = reinterpret_cast<const f32x4_a4*>(p)[0], hi = reinterpret_cast<const f32x4_a4*>(p)[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = lo[e] * decay + neg_lr * o[e];
        hi[e] = hi[e] * decay + neg_lr * o[4 + e];
      }
      reinterpret_cast<f32x4_a4*>(p)[0] = lo;
      reinterpret_cast<f32x4_a4*>(p)[1] = hi;
    } else {
      for (int e = 0; e < n; ++e) p[e] = p[e] * decay + neg_lr * o[e];
    }
  } else {
    uint16_t* p = static_cast<uint16_t*>(a.update_param) + at;
    auto one = [&](uint16_t old, float ov) {
      const float scaled = bf16_bits_to_float(__builtin_bit_cast(uint16_t, static_cast<__bf16>(bf16_bits_to_float(old) * decay)));
      return __builtin_bit_cast(uint16_t, static_cast<__bf16>(scaled + neg_lr * ov));
    };
    if (n == 8) {
      u32x4 v = *reinterpret_cast<const u32x4_a2*>(p);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = static_cast<uint32_t>(one(static_cast<uint16_t>(v[e]), o[2 * e])) | (static_cast<uint32_t>(one(static_cast<uint16_t>(v[e] >> 16), o[2 * e + 1])) << 16);
      *reinterpret_cast<u32x4_a2*>(p) = v;
    } else {
      for (int e = 0; e < n; ++e) p[e] = one(p[e], o[e]);
    }
  }
}

// Kernel argument: the problems of a launch and which workgroup does what.  Block ids [0, tile_begin[n]) compute one
// whole tile each, problem after problem (longest K first); behind them come the K pieces of the split tiles.
// Three sizes.  One problem: nothing is searched and every field sits at a fixed place, so that a workgroup's first loads need
// no address from an earlier one (a product is 0.8 to 1.0 us shorter than with the table of eight; whole Muon step of one
// matrix: 2048x2048 413 -> 402 us, 4096x4096 1300 -> 1285, 1024x4096 256 -> 246).  Up to 8, the usual number of several: 0.8 us
// shorter with 1 KiB of arguments than with the 4 KiB that 32 problems take (empty kernels: 2.9 against 3.7 us), and fewer
// entries to search (whole Muon step: five ragged matrices 342 -> 330 us, two of 2048x5000 1101 -> 1077, a hidden2048 layer
// 2092 -> 2067).
template <int N>
struct LaunchArgs {
  int tile_begin[N + 1];   // first whole-tile block of a problem; entries past n repeat the end
  int piece_begin[N + 1];  // first piece block
  int split_begin[N + 1];  // first split tile (the fix-up kernel's order)
  int class_begin[N + 1];  // first whole-tile block of a class: neighbouring problems with the same K
  int n;
  int symmetric;
  int group_m;      // tile rows per block of the general products' tile order
  int round_tiles;  // resident workgroups, a multiple of 8
  int update_dtype;
  float alpha, beta;
  float* partials;  // fp32 BM x BN tiles, problem p's from partial_base on: [its split tiles][splits]
  GemmProblem problem[N];
};
static_assert(sizeof(LaunchArgs<kMaxGemmGroup>) <= 4096, "kernel arguments are limited to 4 KiB");

// The problem whose range of `begin` holds `block` (one scalar load of the whole table, then compares: a search by
// dependent loads would wait out the memory latency at every step).
template <int N>
__device__ __forceinline__ int problem_of(const int (&begin)[N], int n, int block) {
  if constexpr (N == 2) return 0;  // a launch for one problem
  if (n == 1) return 0;  // fewer classes than problems: their entries past the last repeat the end, too
  int p = 0;
#pragma unroll
  for (int i = 1; i < N - 1; ++i) p += block >= begin[i] ? 1 : 0;
  return p < n ? p : n - 1;
}

// logical tile index -> (tm, tn)
__device__ __forceinline__ void tile_coords(int group_m, int logical, int tiles_m, int tiles_n, bool symmetric, int* tm, int* tn) {
  if (symmetric) {
    // the lower triangle row by row: t = i(i+1)/2 + j, j <= i
    int i = static_cast<int>((__fsqrt_rn(8.0f * static_cast<float>(logical) + 1.0f) - 1.0f) * 0.5f);
    while ((i + 1) * (i + 2) / 2 <= logical) ++i;
    while (i * (i + 1) / 2 > logical) --i;
    *tm = i;
    *tn = logical - i * (i + 1) / 2;
    return;
  }
  // Super columns of up to kSuper tiles, all of nearly one width, walked down all rows in blocks of group_m x half a width:
  // what the whole machine works on at a time is then nearly square (16 x 16 tiles where a round has 256), and so is what
  // one XCD works on.  Widths as even as they come: a last super column of 4 of 20 tiles makes an XCD's share of it tall and
  // narrow, which reads more panels (256-tiles of 5120 x 5120 253 -> 241 us, of 5120 x 13824 603 -> 594 with 14, 14, 14, 12
  // instead of 16, 16, 16, 6).
  constexpr int kSuper = 16;
  int first_n = 0, cols = tiles_n, in = logical;
  if (tiles_n > kSuper) {
    const int supers = (tiles_n + kSuper - 1) / kSuper, width = (tiles_n + supers - 1) / supers;
    const int super = logical / (width * tiles_m);
    first_n = super * width;
    cols = min(width, tiles_n - first_n);
    in -= super * width * tiles_m;
  }
  const int band = in / (group_m * cols);  // group_m rows of this super column
  const int first_m = band * group_m, rows = min(group_m, tiles_m - first_m);
  in -= band * group_m * cols;
  const int half = (cols + 1) / 2;
  const int second = in >= rows * half ? 1 : 0;
  in -= second * rows * half;
  *tm = first_m + in % rows;
  *tn = first_n + second * half + in / rows;
}

// OCC workgroups are meant to share a CU: the register budget per wave is set for OCC * WM * WN / 4 waves per SIMD.
template <int BM, int BN, int WM, int WN, int BK, int STAGES, int OCC, int N>
__global__ void __launch_bounds__(WM * WN * 64, (OCC * WM * WN + 3) / 4)
gemm_nt_kernel(LaunchArgs<N> args) {
  constexpr int kThreads = WM * WN * 64;
  constexpr int kWaves = WM * WN;
  constexpr int kWaveM = BM / WM;     // rows of C per wave
  constexpr int kWaveN = BN / WN;
  constexpr int TM = kWaveM / 16;     // 16x16 MFMA tiles per wave
  constexpr int TN = kWaveN / 16;
  constexpr int TMH = TM / 2;         // tile rows one half step covers
  constexpr int kChunks = BK / 8;               // 16-byte chunks per slab row (row = BK bf16)
  constexpr int kRowsPerSweep = 128 / BK;       // slab rows that together span the 64 LDS banks once (256 bytes)
  constexpr int kRowsPerLoad = 512 / BK;        // slab rows one wave-level 1 KiB load fills
  constexpr int kSteps = BK / 32;               // k32 MFMA steps per slab, each run as two half steps of TMH tile rows
  constexpr int kLoadsP = BM / kRowsPerLoad / kWaves, kLoadsQ = BN / kRowsPerLoad / kWaves;
  constexpr int kLoadsPerSlab = kLoadsP + kLoadsQ;  // direct-to-LDS loads one wave issues per slab
  static_assert(BM % (kRowsPerLoad * kWaves) == 0 && BN % (kRowsPerLoad * kWaves) == 0, "slab must divide over the waves");
  static_assert(kSteps % 2 == 0 && TM % 2 == 0 && STAGES >= 2 && (STAGES - 1) * kLoadsPerSlab < 64, "pipeline shape");
  constexpr int kStageElems = (BM + BN) * BK;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  __bf16* smem = reinterpret_cast<__bf16*>(smem_raw);

  // ---- which problem, which tile, which K range
  const int block = blockIdx.x;
  const bool whole = block < args.tile_begin[N];
  int index = block;
  if (whole) {
    // Workgroup ids congruent mod 8 run on one XCD: in every round of resident workgroups an XCD gets one contiguous eighth
    // of the round's tiles (the first tiles % 8 XCDs one tile more), so that the workgroups sharing an L2 work on
    // neighbouring tiles -- of one matrix, or on a few whole matrices where a class holds many small ones -- while the
    // machine as a whole walks through one matrix after the other.  Classes one by one: every XCD gets its share of the
    // long and of the short tiles.
    const int c = problem_of(args.class_begin, args.n, block);
    const int round = (block - args.class_begin[c]) / args.round_tiles;
    const int first = args.class_begin[c] + round * args.round_tiles, tiles = min(args.round_tiles, args.class_begin[c + 1] - first);
    const int i = block - first, xcd = i % kXcds, each = tiles / kXcds, extra = tiles % kXcds;
    index = first + xcd * each + (xcd < extra ? xcd : extra) + i / kXcds;
  }
  const int problem = whole ? problem_of(args.tile_begin, args.n, index) : problem_of(args.piece_begin, args.n, index);
  const GemmProblem& a = args.problem[problem];
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  int logical, split = 0, piece_tile = 0;
  if (whole) {
    logical = index - args.tile_begin[problem];
  } else {
    const int piece = index - args.piece_begin[problem];
    piece_tile = piece / a.splits;
    split = piece - piece_tile * a.splits;
    logical = args.tile_begin[problem + 1] - args.tile_begin[problem] + piece_tile;
  }
  int tm, tn;
  tile_coords(args.group_m, logical, tiles_m, tiles_n, args.symmetric != 0, &tm, &tn);
  const int row0 = tm * BM;
  const int col0 = tn * BN;
  const int k_slabs_total = a.K / BK;
  const int ks_begin = whole ? 0 : static_cast<int>(static_cast<int64_t>(k_slabs_total) * split / a.splits);
  const int ks_end = whole ? k_slabs_total : static_cast<int>(static_cast<int64_t>(k_slabs_total) * (split + 1) / a.splits);

  // Every tile walks its K range from its first slab on: the tiles of an XCD that share a panel then share its slabs in
  // L2 (walks that start at different slabs were measured 3 to 37 % slower).
  const int n_slabs = ks_end - ks_begin;
  auto k0_of = [&](int i) { return (ks_begin + i) * BK; };

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform by construction: keeps LDS slab addresses scalar
  const int wave_m = wave / WN;
  const int wave_n = wave % WN;

  const __bf16* __restrict__ P = static_cast<const __bf16*>(a.P) + static_cast<int64_t>(row0) * a.ldp;
  const bool q_columns = BM == 256 && (a.flags & kGemmQColumns) != 0;
  const __bf16* __restrict__ Q = static_cast<const __bf16*>(a.Q) + (q_columns ? col0 : static_cast<int64_t>(col0) * a.ldq);

  // ---- slab loader.  A slab row holds BK bf16 = kChunks 16-byte chunks; chunk c of row r is stored at chunk
  // position c ^ ((r / kRowsPerSweep) % kChunks).  One wave-level direct-to-LDS load fills 1 KiB = kRowsPerLoad
  // rows: lane l lands at row l / kChunks, position l % kChunks, and therefore fetches the global chunk the
  // swizzle maps there.  Wave w takes the row groups w, w + kWaves, ...
  // The loads are buffer loads: the tile's first row is the descriptor's base, a lane's offset inside a row group (row
  // l / kChunks, the chunk the swizzle maps to position l % kChunks) is one loop-invariant register per operand --
  // the swizzle term does not depend on which of the wave's row groups it is -- and everything that changes from
  // load to load (row group, k) is a scalar offset: no vector address arithmetic in the loop.
  static_assert((kWaves * kRowsPerLoad / kRowsPerSweep) % kChunks == 0, "the swizzle must repeat from one row group of a wave to the next");
  const int dl_row = wave * kRowsPerLoad + lane / kChunks;
  const int dl_chunk = (lane % kChunks) ^ ((dl_row / kRowsPerSweep) % kChunks);
  const uint32_t lane_offset_p = static_cast<uint32_t>(dl_row * a.ldp + dl_chunk * 8) * 2u;
  auto operand_rsrc = [](const __bf16* base, int64_t rows, int ld) {
    const int64_t bytes = rows * ld * 2;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(base), 0, static_cast<int>(bytes < 0x7fffffff ? bytes : 0x7fffffff), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rsrc_p = operand_rsrc(P, a.M - row0, a.ldp);
  // a Q of K rows: its rows beyond M read as zero, as P's do (K runs over M)
  const __amdgpu_buffer_rsrc_t rsrc_q =
      q_columns ? __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(Q), 0, static_cast<int>((static_cast<int64_t>(a.M) * a.ldq - col0) * 2), 0x00020000)
                : operand_rsrc(Q, a.N - col0, a.ldq);
  typedef __attribute__((address_space(3))) void* LdsPtr;
  // One load at a time: a wave that issues several of these back to back stalls on the address queue, and its
  // MFMAs wait with it, so the main loop slips them in between MFMAs.
  auto load_p = [&](int k0, int stage, int i) {
    const int r0 = (i * kWaves + wave) * kRowsPerLoad;
    const int scalar_offset = (i * kWaves * kRowsPerLoad * a.ldp + k0) * 2;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_p, (LdsPtr)(smem + stage * kStageElems + r0 * BK), 16, lane_offset_p, scalar_offset, 0, 0);
  };
  auto stream_p = [&](int k0, int stage) {
#pragma unroll
    for (int i = 0; i < kLoadsP; ++i) load_p(k0, stage, i);
  };
  // Accumulator register r of lane l holds C[4*(l/16) + r][l%16] of its 16x16 tile.
  const int lcol = wave_n * kWaveN + (lane & 15);
  const int lrow = wave_m * kWaveM + (lane >> 4) * 4;
  // A whole tile takes its D operand on the way: D^T is the Q operand itself in both products that have one (X^T in
  // the update product, the symmetric A in A A), and K spans the rows of C there, so the Q slabs with k in
  // [row0, row0 + BM) hold D[k - row0][0 .. BN) of this tile as they pass through LDS.  The waves pick their values
  // out of those slabs (see the slab loop) and add (beta / alpha) D to the accumulators, so that alpha * acc is
  // alpha P Q^T + beta D with one rounding; nothing is fetched for D.  (Fetched behind the main loop the D tile
  // cost a 256 x 256 tile with K = 4096 11 of its 121 microseconds: every CU wants its 128 KiB from HBM at the same
  // moment, and the tile has to be staged through LDS because its rows do not match the accumulator layout.)
  const bool d_in_slabs = whole && a.D != nullptr;
  const float d_scale = d_in_slabs ? args.beta / args.alpha : 0.0f;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

  // The K walk, for a Q of N rows (K-contiguous, as P) and for one of K rows (kGemmQColumns: X itself in the update product, so
  // that no transpose of X is ever stored).  A slab of the latter is BK rows of BN bf16 in LDS, in chunks of 32 bytes: chunk c of
  // row r sits at c ^ f(r), f(r) the row's bits 0, 1 and 3, so that the eight rows that half a wave reads at a time (four
  // consecutive ones of two blocks of eight) cover all banks.  ds_read_b64_tr_b16 turns four rows by sixteen columns into four
  // consecutive k of a lane's column: two of them are a fragment, one is a lane's D values.
  auto walk = [&](auto q_columns_tag) __attribute__((always_inline)) {
  constexpr bool kQColumns = decltype(q_columns_tag)::value;
  constexpr int kQRowLanes = BN / 8, kQRowsPerLoad = 64 / kQRowLanes;
  static_assert(kWaves * kQRowsPerLoad == 16 && BK / kQRowsPerLoad / kWaves == kLoadsQ, "the swizzle must repeat from one row group of a wave to the next");
  const int q_row = wave * kQRowsPerLoad + lane / kQRowLanes;
  const int q_chunk = ((lane % kQRowLanes) >> 1) ^ ((q_row & 3) | ((q_row >> 1) & 4));
  const uint32_t lane_offset_q = kQColumns ? static_cast<uint32_t>(q_row * a.ldq + q_chunk * 16 + (lane & 1) * 8) * 2u
                                           : static_cast<uint32_t>(dl_row * a.ldq + dl_chunk * 8) * 2u;
  auto load_q = [&](int k0, int stage, int i) {
    const int r0 = kQColumns ? (i * kWaves + wave) * 512 : (i * kWaves + wave) * kRowsPerLoad * BK;  // first element in LDS
    const int scalar_offset = kQColumns ? (k0 + i * 16) * a.ldq * 2 : (i * kWaves * kRowsPerLoad * a.ldq + k0) * 2;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_q, (LdsPtr)(smem + stage * kStageElems + BM * BK + r0), 16, lane_offset_q, scalar_offset, 0, 0);
  };
  auto stream_q = [&](int k0, int stage) {
#pragma unroll
    for (int i = 0; i < kLoadsQ; ++i) load_q(k0, stage, i);
  };
  // lane 4 e + q of a group of sixteen reads four columns of row e
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* TrPtr;
  const int tr_e = (lane & 15) >> 2, tr_group = lane >> 4, tr_chunk0 = wave_n * kWaveN / 16;
  auto read_tr = [&](int elements) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((TrPtr)(smem + elements)); };
  const int tr_frag = BM * BK + (8 * tr_group + tr_e) * BN + (lane & 3) * 4 + (tr_chunk0 ^ ((tr_group & 1) * 4)) * 16;
  const int tr_d = BM * BK + (4 * tr_group + tr_e) * BN + (lane & 3) * 4 + (tr_chunk0 ^ ((tr_group >> 1) * 4)) * 16;
  static_assert(TN == 4, "a wave's column blocks are the low two bits of the chunk");
  auto read_q = [&](int stage, int kk, int j) {
    const int at = tr_frag + stage * kStageElems + kk * 32 * BN + ((j ^ tr_e) << 4);
    const s16x4 lo = read_tr(at), hi = read_tr(at + 4 * BN);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // 16x16x32 MFMA operands: lane l supplies row l % 16 of its 16-row block and the 8 k values of chunk l / 16 of
  // the 32 wide step.  (At equal peak rate this shape draws less power than 32x32x16 on operands with random
  // bits, and under sustained load the chip's clock is set by power: measured 2.0 against 1.8 PFLOP/s for bare
  // MFMA streams.)
  const int frag_row = lane & 15;
  const int frag_chunk = lane >> 4;

  // LDS offsets of this lane's fragment chunk for the k32 steps of a slab (the row part of the swizzle only
  // depends on frag_row: every 16-row block starts at a multiple of 16 rows)
  const __bf16* frag_p = smem + (wave_m * kWaveM + frag_row) * BK;
  const __bf16* frag_q = smem + BM * BK + (wave_n * kWaveN + frag_row) * BK;
  auto frag_off = [&](int stage, int kk) {
    return stage * kStageElems + (((kk * 4 + frag_chunk) ^ ((frag_row / kRowsPerSweep) % kChunks)) << 3);
  };
  // Software pipeline.  STAGES slabs are resident or in flight: the slab being multiplied and the next
  // STAGES - 1, streamed HBM -> LDS while the MFMAs run.  A k32 step runs as two half steps of TMH x TN MFMAs
  // (the upper and the lower tile rows of the wave).  Fragments: the Q side (all TN of a step) is double
  // buffered, the P side holds one buffer per half; the first half of a step reads the P fragments of its second
  // half, the second half reads the next step's Q fragments and first-half P fragments, so every 128-bit LDS read
  // has half a step of MFMAs to come back (it is waited for at the start of the next half step).  The one barrier
  // per slab sits before the slab's last half step: by then every wave has its last fragments of the current
  // stage in registers (the stage can be refilled with the slab STAGES ahead) and its share of the next slab has
  // landed, so the next slab's first fragments are fetched under this slab's last MFMAs.
  constexpr int kWaitLds = 0xC07F;  // s_waitcnt lgkmcnt(0), vmcnt / expcnt fields at their maxima
  // s_waitcnt lgkmcnt(0) vmcnt(N): loads return in order, so this leaves the N most recent ones in flight
  constexpr int kInFlight = (STAGES - 2) * kLoadsPerSlab;
  constexpr int kWaitNextSlab = 0x0070 | (kInFlight & 0xF) | ((kInFlight >> 4) << 14);
  bf16x8 fa_lo[TMH], fa_hi[TMH], fb0[TN], fb1[TN];
  // Loads are issued unconditionally, for a slab number clamped to the last one: past the end of the walk they
  // fetch the last slab once more into a stage nobody reads again.  (A branch around a load in the middle of the
  // MFMAs makes the register allocator spill the accumulators.)
  auto k0_clamped = [&](int i) { return k0_of(i < n_slabs ? i : n_slabs - 1); };
  if (n_slabs > 0) {
#pragma unroll
    for (int sidx = 0; sidx < STAGES; ++sidx) {
      stream_p(k0_clamped(sidx), sidx);
      if (sidx + 1 < STAGES) stream_q(k0_clamped(sidx), sidx);  // the Q rows of the last one go out under the first MFMAs
    }
    constexpr int kAfterFirst = (STAGES - 2) * kLoadsPerSlab + kLoadsP;
    __builtin_amdgcn_s_waitcnt(0x0F70 | (kAfterFirst & 0xF) | ((kAfterFirst >> 4) << 14));
    __syncthreads();
    const int off = frag_off(0, 0);
#pragma unroll
    for (int i = 0; i < TMH; ++i) fa_lo[i] = *reinterpret_cast<const bf16x8*>(frag_p + off + i * 16 * BK);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (kQColumns) fb0[j] = read_q(0, 0, j);
      else fb0[j] = *reinterpret_cast<const bf16x8*>(frag_q + off + j * 16 * BK);
    }
  }
  // One half step: the TMH x TN MFMAs on the fragments in hand (use_a for tile rows row0.., use_b), kReads LDS
  // reads (read(r), one behind each of the first MFMAs) and kLoads slab loads, interleaved instruction by
  // instruction: MFMA, LDS read, MFMA, LDS read, ..., slab load, ...  The matrix pipe is handed to the oldest wave
  // that has an MFMA ready, so whenever one of the two waves of a SIMD sits at the barrier the other runs alone,
  // and then every clump of other instructions between two MFMAs is a bubble in the pipe.
  // The first kPairs reads are two instructions each.
  auto half_step = [&](auto row0_tag, const bf16x8 (&use_a)[TMH], const bf16x8 (&use_b)[TN], auto reads_tag, auto pairs_tag, auto&& read,
                       auto loads_tag, auto&& load) {
    constexpr int kPairs = decltype(pairs_tag)::value;
    constexpr int kRow0 = decltype(row0_tag)::value;
    constexpr int kReads = decltype(reads_tag)::value;
    constexpr int kLoads = decltype(loads_tag)::value;
    constexpr int kMfma = TMH * TN;
    constexpr int kChunks_ = kLoads > 0 ? kLoads : 1;
    constexpr int kPer = kMfma / kChunks_;
    static_assert(kMfma % kChunks_ == 0 && kReads <= kMfma, "half step shape");
#pragma unroll
    for (int c = 0; c < kChunks_; ++c) {
#pragma unroll
      for (int n = c * kPer; n < (c + 1) * kPer; ++n) {
        if (n < kReads) read(n);
        acc[kRow0 + n / TN][n % TN] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(use_a[n / TN], use_b[n % TN], acc[kRow0 + n / TN][n % TN], 0, 0, 0);
      }
#pragma unroll
      for (int n = c * kPer; n < (c + 1) * kPer; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        if (n < kPairs) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        else if (n < kReads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kLoads > 0) {
        load(c);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  using Zero = std::integral_constant<int, 0>;
  using Upper = std::integral_constant<int, TMH>;
  // first half of step kk (fragments in fa_lo / use_b): reads the second half's P fragments
  auto first_half = [&](const bf16x8 (&use_b)[TN], int read_stage, int kk, auto loads_tag, auto&& load) {
    const int off = frag_off(read_stage, kk);
    half_step(Zero{}, fa_lo, use_b, std::integral_constant<int, TMH>{}, Zero{},
              [&](int r) { fa_hi[r] = *reinterpret_cast<const bf16x8*>(frag_p + off + (TMH + r) * 16 * BK); }, loads_tag, load);
  };
  // second half (fa_hi / use_b): reads the Q fragments and the first-half P fragments of the step after it
  auto second_half = [&](const bf16x8 (&use_b)[TN], bf16x8 (&next_b)[TN], int read_stage, int read_kk, auto loads_tag, auto&& load) {
    const int off = frag_off(read_stage, read_kk);
    half_step(Upper{}, fa_hi, use_b, std::integral_constant<int, TN + TMH>{}, std::integral_constant<int, kQColumns ? TN : 0>{},
              [&](int r) {
                // Q fragments first: the next step's first MFMAs need every one of them but only the first P fragment
                if (r < TN) {
                  if constexpr (kQColumns) next_b[r] = read_q(read_stage, read_kk, r);
                  else next_b[r] = *reinterpret_cast<const bf16x8*>(frag_q + off + r * 16 * BK);
                } else fa_lo[r - TN] = *reinterpret_cast<const bf16x8*>(frag_p + off + (r - TN) * 16 * BK);
              },
              loads_tag, load);
  };
  // D values out of a Q slab (see d_in_slabs above).  Slab q of the BM / BK slabs that hold the tile's D rows carries
  // the rows of kTilesPerSlab MFMA tile rows of the waves with wave_m == q / kSlabsPerWave; a lane's four rows of one
  // column are four consecutive k of one slab row: one 64-bit LDS read per MFMA tile, in two batches that are read at the
  // start of a half step and added at its end, so that every tile row gets its D between its two MFMAs of the slab.
  // The 256 and the 128 tiles therefore add in the same order: a result has the same bits in either (unless its K walk was
  // cut into pieces; the 64 tiles, whose waves share K and add D at the end, sum in an order of their own).
  constexpr int kTilesPerSlab = BK / 16;
  constexpr int kSlabsPerWave = kWaveM / BK;
  constexpr int kDSlabs = BM / BK;
  constexpr int kDPairs = kTilesPerSlab * TN, kDBatch = kDPairs / 2;
  static_assert(kWaveM % BK == 0 && TM == kSlabsPerWave * kTilesPerSlab && kSteps == 2 && TMH % (kTilesPerSlab / 2) == 0,
                "D slabs must divide over the waves and the half steps");
  const int d_base = BM * BK + lcol * BK + 4 * ((lane >> 4) & 1);  // slab row lcol (+ 16 j), first or second half of a chunk
  const int d_swizzle = (lcol / kRowsPerSweep) % kChunks;          // the same for lcol + 16 j
  u32x2 d_vals[kDBatch];
  auto d_read = [&](int stage, int batch) {
#pragma unroll
    for (int n = 0; n < kDBatch; ++n) {
      const int pair = batch * kDBatch + n, ii = pair / TN, j = pair % TN;
      if constexpr (kQColumns) {
        d_vals[n] = __builtin_bit_cast(u32x2, read_tr(tr_d + stage * kStageElems + ii * 16 * BN + ((j ^ tr_e) << 4)));
        continue;
      }
      const int chunk = (2 * ii + (lane >> 5)) ^ d_swizzle;
      d_vals[n] = *reinterpret_cast<const u32x2*>(smem + stage * kStageElems + d_base + j * 16 * BK + (chunk << 3));
    }
  };
  auto d_add = [&](auto qq_tag, int batch, float scale) {
    constexpr int kFirstTile = decltype(qq_tag)::value * kTilesPerSlab;
#pragma unroll
    for (int n = 0; n < kDBatch; ++n) {
      const int pair = batch * kDBatch + n, i = kFirstTile + pair / TN, j = pair % TN;
      acc[i][j][0] += scale * __uint_as_float(d_vals[n].x << 16);
      acc[i][j][1] += scale * __uint_as_float(d_vals[n].x & 0xffff0000u);
      acc[i][j][2] += scale * __uint_as_float(d_vals[n].y << 16);
      acc[i][j][3] += scale * __uint_as_float(d_vals[n].y & 0xffff0000u);
    }
  };
  int stage = 0;
  // One slab.  d_tag: -1, or which of the tile's D slabs this one is.
  auto slab = [&](int it, auto d_tag) {
    constexpr int kD = decltype(d_tag)::value;
    constexpr int kOwner = kD < 0 ? 0 : kD / kSlabsPerWave;
    using Part = std::integral_constant<int, kD < 0 ? 0 : kD % kSlabsPerWave>;
    // the half step the first D batch rides on: the slab's tile rows (its first two, in a tile whose slab rows span both
    // halves) meet their first MFMA there
    constexpr int kDHalf = kD < 0 ? -4 : (Part::value * kTilesPerSlab >= TMH ? 1 : 0);
    const float scale = (kD >= 0 && wave_m == kOwner) ? d_scale : 0.0f;  // the other waves add zero times a finite value
    auto d_before = [&](auto half_tag) {
      constexpr int kBatch = decltype(half_tag)::value - kDHalf;
      if constexpr (kBatch == 0 || kBatch == 1) {
        d_read(stage, kBatch);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto d_after = [&](auto half_tag) {
      constexpr int kBatch = decltype(half_tag)::value - kDHalf;
      if constexpr (kBatch == 0 || kBatch == 1) d_add(Part{}, kBatch, scale);
    };
    const int next_stage = stage + 1 == STAGES ? 0 : stage + 1;
    const int prev_stage = stage == 0 ? STAGES - 1 : stage - 1;
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    using H2 = std::integral_constant<int, 2>;
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    __builtin_amdgcn_sched_barrier(0);
    d_before(H0{});
    {
      // second half of the refill of the stage the previous slab's barrier released (its P rows went out there)
      const int k0 = k0_clamped(it - 1 + STAGES);
      first_half(fb0, stage, 0, std::integral_constant<int, kLoadsQ>{}, [&](int l) { load_q(k0, prev_stage, l); });
    }
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    __builtin_amdgcn_sched_barrier(0);
    d_after(H0{});
    d_before(H1{});
    second_half(fb0, fb1, stage, 1, Zero{}, [](int) {});
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    __builtin_amdgcn_sched_barrier(0);
    d_after(H1{});
    d_before(H2{});
    first_half(fb1, stage, 1, Zero{}, [](int) {});
    // last half step of the slab: the slab after it must have landed (the STAGES - 2 younger ones may be in
    // flight); behind the barrier this slab's stage is free and its refill starts with the P rows
    __builtin_amdgcn_s_waitcnt(kWaitNextSlab);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    d_after(H2{});
    if constexpr (kD >= 0) __builtin_amdgcn_sched_barrier(0);
    {
      const int k0 = k0_clamped(it + STAGES);
      second_half(fb1, fb0, next_stage, 0, std::integral_constant<int, kLoadsP>{}, [&](int l) { load_p(k0, stage, l); });
    }
    stage = next_stage;
  };
  using NoD = std::integral_constant<int, -1>;
  if (d_in_slabs) {
    // the slabs with k in [row0, row0 + BM) are peeled out of the walk (whole tiles walk all of K from slab 0)
    const int first_d = row0 / BK;
    for (int it = 0; it < first_d; ++it) slab(it, NoD{});
    auto d_slabs = [&](auto&& self, auto q_tag) -> void {
      constexpr int kQ = decltype(q_tag)::value;
      if (first_d + kQ < n_slabs) slab(first_d + kQ, q_tag);  // tile rows at or beyond K have no D (and no result)
      if constexpr (kQ + 1 < kDSlabs) self(self, std::integral_constant<int, kQ + 1>{});
    };
    d_slabs(d_slabs, Zero{});
    for (int it = first_d + kDSlabs; it < n_slabs; ++it) slab(it, NoD{});
  } else {
    for (int it = 0; it < n_slabs; ++it) slab(it, NoD{});
  }
  };  // walk
  if constexpr (BM == 256) {
    if (q_columns) walk(std::true_type{});
    else walk(std::false_type{});
  } else {  // without the code it never runs
    walk(std::false_type{});
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // the loads past the end of the walk have landed too; LDS is free

  // ---- K pieces: park the fp32 partial tile (row-major BM x BN); the fix-up kernel sums the pieces and
  // runs the epilogue.
  if (!whole) {
    float* mine = args.partials + (static_cast<int64_t>(a.partial_base) + piece_tile * a.splits + split) * (BM * BN);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(lrow + i * 16 + r) * BN + lcol + j * 16] = acc[i][j][r];
    return;
  }


  // ---- epilogue, staged through LDS so that HBM only sees whole 16-byte-per-lane, row-contiguous accesses.
  // Accumulator register r of lane l holds C[4*(l/16) + r][l%16] of its 16x16 tile: written
  // straight from registers that would be 2-byte stores for C and 8-byte stores scattered over 16 rows for
  // the transpose.  Instead: C tile -> LDS -> HBM, transposed tile -> LDS -> HBM.  (The D operand is already in the
  // accumulators.)
  uint16_t* __restrict__ C = static_cast<uint16_t*>(a.C);
  uint16_t* __restrict__ CT = static_cast<uint16_t*>(a.CT);
  int ldct = a.ldct;
  if (args.symmetric) {  // mirror the off-diagonal tile
    CT = tm != tn ? C : nullptr;
    ldct = a.ldc;
  }
  uint16_t* stage_c = reinterpret_cast<uint16_t*>(smem_raw);
  constexpr int kLdS = BN + 8;  // row pitch of the staged C tile (elements); +8 keeps rows 16-byte aligned and skews banks
  constexpr int kLdT = BM + 8;  // row pitch of the staged transposed tile
  constexpr int kRowChunks = BN / 8, kColChunks = BM / 8;
  __syncthreads();  // every wave is done reading the slab stages
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = args.alpha * acc[i][j][r];
  if (a.update_param != nullptr) {
    // the last product of a Muon step: the tile goes into the parameter (in the parameter's orientation) and nowhere else
    if (!(a.flags & kGemmUpdateTransposed)) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            stage_c[(lrow + i * 16 + r) * kLdS + lcol + j * 16] = __builtin_bit_cast(uint16_t, static_cast<__bf16>(acc[i][j][r]));
      __syncthreads();
      for (int c = tid; c < BM * kRowChunks; c += kThreads) {
        const int r = c / kRowChunks, cc = c - r * kRowChunks;
        update_param8(a, args.update_dtype, row0 + r, col0 + cc * 8, *reinterpret_cast<const u32x4*>(stage_c + r * kLdS + cc * 8));
      }
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          u32x2 four = {pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
          *reinterpret_cast<u32x2*>(stage_c + (lcol + j * 16) * kLdT + lrow + i * 16) = four;
        }
      __syncthreads();
      for (int c = tid; c < BN * kColChunks; c += kThreads) {
        const int r = c / kColChunks, cc = c - r * kColChunks;
        update_param8(a, args.update_dtype, col0 + r, row0 + cc * 8, *reinterpret_cast<const u32x4*>(stage_c + r * kLdT + cc * 8));
      }
    }
    return;
  }
  if (!(a.flags & kGemmSkipC)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          stage_c[(lrow + i * 16 + r) * kLdS + lcol + j * 16] = __builtin_bit_cast(uint16_t, static_cast<__bf16>(acc[i][j][r]));
    __syncthreads();
    for (int c = tid; c < BM * kRowChunks; c += kThreads) {
      const int r = c / kRowChunks, cc = c - r * kRowChunks;
      *reinterpret_cast<u32x4*>(C + static_cast<int64_t>(row0 + r) * a.ldc + col0 + cc * 8) =
          *reinterpret_cast<const u32x4*>(stage_c + r * kLdS + cc * 8);
    }
    if (CT == nullptr) return;
    __syncthreads();
  }
  if (CT == nullptr) return;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
    {
      // the four registers of a tile are four consecutive rows of one column: four consecutive elements of a transposed row
      u32x2 four = {pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
      *reinterpret_cast<u32x2*>(stage_c + (lcol + j * 16) * kLdT + lrow + i * 16) = four;
    }
  __syncthreads();
  for (int c = tid; c < BN * kColChunks; c += kThreads) {
    const int r = c / kColChunks, cc = c - r * kColChunks;
    *reinterpret_cast<u32x4*>(CT + static_cast<int64_t>(col0 + r) * ldct + row0 + cc * 8) =
        *reinterpret_cast<const u32x4*>(stage_c + r * kLdT + cc * 8);
  }
}

// Sums the K pieces of every split tile in split order and applies the epilogue of gemm_nt_kernel.  A workgroup of
// 1024 threads finishes a 64 x 64 block of a tile, thread t four consecutive columns of row t / 16; the transposed /
// mirrored copy goes through LDS so that both orientations leave in whole 16-byte, row-contiguous stores.
constexpr int kFixupThreads = 1024;
template <int BM, int BN, int N>
__global__ void __launch_bounds__(kFixupThreads)
splitk_fixup_kernel(LaunchArgs<N> args) {
  constexpr int kSub = 64;
  constexpr int kSubsPerTile = (BM / kSub) * (BN / kSub);
  __shared__ __attribute__((aligned(16))) uint16_t transposed[kSub][kSub + 8];
  const int split_tile = blockIdx.x / kSubsPerTile;
  const int sub = blockIdx.x % kSubsPerTile;
  const int problem = problem_of(args.split_begin, args.n, split_tile);
  const GemmProblem& a = args.problem[problem];
  const int tile = split_tile - args.split_begin[problem];
  const int full_tiles = args.tile_begin[problem + 1] - args.tile_begin[problem];
  const int sub_row0 = (sub / (BN / kSub)) * kSub, sub_col0 = (sub % (BN / kSub)) * kSub;
  int tm, tn;
  tile_coords(args.group_m, full_tiles + tile, (a.M + BM - 1) / BM, (a.N + BN - 1) / BN, args.symmetric != 0, &tm, &tn);
  const uint16_t* __restrict__ D = static_cast<const uint16_t*>(a.D);
  uint16_t* __restrict__ C = static_cast<uint16_t*>(a.C);
  uint16_t* __restrict__ CT = static_cast<uint16_t*>(a.CT);
  int ldct = a.ldct;
  if (args.symmetric) {  // mirror the off-diagonal tile
    CT = tm != tn ? C : nullptr;
    ldct = a.ldc;
  }
  const int t = threadIdx.x;
  const int r = t / 16, c = (t % 16) * 4;  // position inside the 64 x 64 block
  const int lrow = sub_row0 + r, lcol = sub_col0 + c;
  const float* base = args.partials + (static_cast<int64_t>(a.partial_base) + static_cast<int64_t>(tile) * a.splits) * (BM * BN) + lrow * BN + lcol;
  // four loads in flight at a time; the sum itself stays in split order
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  int s = 0;
  for (; s + 4 <= a.splits; s += 4) {
    f32x4 piece[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) piece[u] = *reinterpret_cast<const f32x4*>(base + static_cast<int64_t>(s + u) * (BM * BN));
#pragma unroll
    for (int u = 0; u < 4; ++u) sum += piece[u];
  }
  for (; s < a.splits; ++s) sum += *reinterpret_cast<const f32x4*>(base + static_cast<int64_t>(s) * (BM * BN));
  const int row = tm * BM + lrow, col = tn * BN + lcol;
  float v[4] = {args.alpha * sum.x, args.alpha * sum.y, args.alpha * sum.z, args.alpha * sum.w};
  if (D != nullptr) {
    const u32x2 d = *reinterpret_cast<const u32x2*>(D + static_cast<int64_t>(row) * a.ldd + col);
    v[0] += args.beta * bf16_bits_to_float(static_cast<uint16_t>(d.x));
    v[1] += args.beta * bf16_bits_to_float(static_cast<uint16_t>(d.x >> 16));
    v[2] += args.beta * bf16_bits_to_float(static_cast<uint16_t>(d.y));
    v[3] += args.beta * bf16_bits_to_float(static_cast<uint16_t>(d.y >> 16));
  }
  const uint32_t lo = pack_bf16x2(v[0], v[1]);
  const uint32_t hi = pack_bf16x2(v[2], v[3]);
  if (a.update_param != nullptr) {  // uniform over the grid: the parameter update in place of the stores (see gemm_nt_kernel)
    if (!(a.flags & kGemmUpdateTransposed)) {
      const u32x4 packed = {lo, hi, 0u, 0u};  // this thread's four columns
      update_param8(a, args.update_dtype, row, col, packed, 4);
      return;
    }
    transposed[c][r] = static_cast<uint16_t>(lo);
    transposed[c + 1][r] = static_cast<uint16_t>(lo >> 16);
    transposed[c + 2][r] = static_cast<uint16_t>(hi);
    transposed[c + 3][r] = static_cast<uint16_t>(hi >> 16);
    __syncthreads();
    if (t < kSub * 8) {
      const int tr = t / 8, chunk = t % 8;
      update_param8(a, args.update_dtype, tn * BN + sub_col0 + tr, tm * BM + sub_row0 + chunk * 8, *reinterpret_cast<const u32x4*>(&transposed[tr][chunk * 8]));
    }
    return;
  }
  if (!(a.flags & kGemmSkipC)) {
    const u32x2 packed = {lo, hi};
    *reinterpret_cast<u32x2*>(C + static_cast<int64_t>(row) * a.ldc + col) = packed;
  }
  if (CT == nullptr) return;  // uniform over the workgroup
  transposed[c][r] = static_cast<uint16_t>(lo);
  transposed[c + 1][r] = static_cast<uint16_t>(lo >> 16);
  transposed[c + 2][r] = static_cast<uint16_t>(hi);
  transposed[c + 3][r] = static_cast<uint16_t>(hi >> 16);
  __syncthreads();
  if (t < kSub * 8) {
    const int tr = t / 8, chunk = t % 8;  // row of the transposed block = column of the tile
    *reinterpret_cast<u32x4*>(CT + static_cast<int64_t>(tn * BN + sub_col0 + tr) * ldct + tm * BM + sub_row0 + chunk * 8) =
        *reinterpret_cast<const u32x4*>(&transposed[tr][chunk * 8]);
  }
}

// ---- 64 x 64 tiles for launches that leave most CUs idle otherwise.
// A chain of products of matrices of a few hundred rows is bound by the latency of each launch: with 128 x 128 tiles a
// handful of CUs walk all of K slab by slab, a load latency and a barrier per slab.  Here the eight waves of a workgroup
// cut K among themselves: each computes the whole 64 x 64 tile over its share, straight from global memory to registers
// (the loads of four k32 steps are in flight, no barrier in the walk), and the partial tiles are summed through LDS in a
// fixed order.  A tile moves four times the operand bytes of a 256 x 256 one per flop, so this pays only while the launch
// is latency bound.  Whole Muon step, 128 x 128 tiles -> these, us: 512x256 with 256x512 162 -> 124, 512x512 171 -> 142,
// two of 512x1536 220 -> 201, 1024x1024 251 -> 204, four of 64x256 117 -> 91.
template <int N>
struct SmallArgs {
  int begin[N];  // first workgroup of a problem; entries past the last problem are the end
  int symmetric;
  int group_m;
  int update_dtype;
  float alpha, beta;
  GemmProblem problem[N];
};
static_assert(sizeof(SmallArgs<kMaxGemmGroup>) <= 4096, "kernel arguments are limited to 4 KiB");

constexpr int kSmallTile = 64;
constexpr int kSmallWaves = 8;
constexpr int kSmallThreads = kSmallWaves * 64;
constexpr int kSmallPitch = kSmallTile + 4;  // floats per row of a partial tile in LDS: skews the banks of a lane's four rows

template <int N>
__global__ void __launch_bounds__(kSmallThreads, 2)
gemm_small_kernel(SmallArgs<N> args) {
  constexpr int kTiles = kSmallTile / 16;
  __shared__ __attribute__((aligned(16))) float sums[4 * kSmallTile * kSmallPitch];
  int problem = 0;
#pragma unroll
  for (int i = 1; i < N; ++i) problem += static_cast<int>(blockIdx.x) >= args.begin[i] ? 1 : 0;
  const GemmProblem a = args.problem[problem];  // a copy: all of its fields in one go instead of a scalar load at each use
  int tm, tn;
  tile_coords(args.group_m, blockIdx.x - args.begin[problem], (a.M + kSmallTile - 1) / kSmallTile, (a.N + kSmallTile - 1) / kSmallTile,
              args.symmetric != 0, &tm, &tn);
  const int row0 = tm * kSmallTile, col0 = tn * kSmallTile;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // D values of the epilogue (thread t: eight columns of row t / 8), fetched under the products
  const int orow = tid / 8, ocol = (tid % 8) * 8;
  u32x4 d = {0u, 0u, 0u, 0u};
  if (a.D != nullptr) d = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.D) + static_cast<int64_t>(row0 + orow) * a.ldd + col0 + ocol);

  // 16x16x32 MFMA operands: lane l supplies row l % 16 of a 16-row block and the 8 k values of chunk l / 16
  const int steps = a.K / 32;
  const int first = steps * wave / kSmallWaves, last = steps * (wave + 1) / kSmallWaves;
  const __bf16* __restrict__ P = static_cast<const __bf16*>(a.P) + static_cast<int64_t>(row0 + (lane & 15)) * a.ldp + (lane >> 4) * 8;
  const __bf16* __restrict__ Q = static_cast<const __bf16*>(a.Q) + static_cast<int64_t>(col0 + (lane & 15)) * a.ldq + (lane >> 4) * 8;
  const int64_t p_block = static_cast<int64_t>(16) * a.ldp, q_block = static_cast<int64_t>(16) * a.ldq;
  f32x4 acc[kTiles][kTiles];
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int j = 0; j < kTiles; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // kSteps k32 steps: every load is issued before the first product (left to itself the compiler sinks them to their uses
  // and waits out a memory latency for each)
  auto batch = [&](int step, auto steps_tag) {
    constexpr int kSteps = decltype(steps_tag)::value;
    bf16x8 fp[kSteps][kTiles], fq[kSteps][kTiles];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
#pragma unroll
      for (int i = 0; i < kTiles; ++i) fp[s][i] = *reinterpret_cast<const bf16x8*>(P + i * p_block + (step + s) * 32);
#pragma unroll
      for (int j = 0; j < kTiles; ++j) fq[s][j] = *reinterpret_cast<const bf16x8*>(Q + j * q_block + (step + s) * 32);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
#pragma unroll
      for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int j = 0; j < kTiles; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp[s][i], fq[s][j], acc[i][j], 0, 0, 0);
  };
  int step = first;
  for (; step + 4 <= last; step += 4) batch(step, std::integral_constant<int, 4>{});
  switch (last - step) {
    case 3: batch(step, std::integral_constant<int, 3>{}); break;
    case 2: batch(step, std::integral_constant<int, 2>{}); break;
    case 1: batch(step, std::integral_constant<int, 1>{}); break;
    default: break;
  }

  // ---- partial tiles: waves 4 .. 7 hand theirs to waves 0 .. 3 lane by lane, then every thread sums four
  f32x4* raw = reinterpret_cast<f32x4*>(sums);
  if (wave >= 4) {
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int j = 0; j < kTiles; ++j) raw[((wave - 4) * kTiles * kTiles + i * kTiles + j) * 64 + lane] = acc[i][j];
  }
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int j = 0; j < kTiles; ++j) acc[i][j] += raw[(wave * kTiles * kTiles + i * kTiles + j) * 64 + lane];
  }
  __syncthreads();
  if (wave < 4) {
    // accumulator register r of lane l holds C[4*(l/16) + r][l%16] of its 16x16 tile
    float* mine = sums + (wave * kSmallTile + (lane >> 4) * 4) * kSmallPitch + (lane & 15);
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int j = 0; j < kTiles; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(i * 16 + r) * kSmallPitch + j * 16] = acc[i][j][r];
  }
  __syncthreads();
  f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const f32x4* from = reinterpret_cast<const f32x4*>(sums + (w * kSmallTile + orow) * kSmallPitch + ocol);
    lo += from[0];
    hi += from[1];
  }
  u32x4 packed;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v0 = args.alpha * (e < 2 ? lo[2 * e] : hi[2 * e - 4]), v1 = args.alpha * (e < 2 ? lo[2 * e + 1] : hi[2 * e - 3]);
    if (a.D != nullptr) {
      v0 += args.beta * __uint_as_float(d[e] << 16);
      v1 += args.beta * __uint_as_float(d[e] & 0xffff0000u);
    }
    packed[e] = pack_bf16x2(v0, v1);
  }

  // ---- epilogue, as in gemm_nt_kernel: C, the transposed / mirrored tile, or the parameter
  uint16_t* __restrict__ C = static_cast<uint16_t*>(a.C);
  uint16_t* __restrict__ CT = static_cast<uint16_t*>(a.CT);
  int ldct = a.ldct;
  if (args.symmetric) {
    CT = tm != tn ? C : nullptr;
    ldct = a.ldc;
  }
  const bool update = a.update_param != nullptr, update_transposed = update && (a.flags & kGemmUpdateTransposed) != 0;
  if (update && !update_transposed) {
    update_param8(a, args.update_dtype, row0 + orow, col0 + ocol, packed);
    return;
  }
  if (!update) {
    if (!(a.flags & kGemmSkipC)) *reinterpret_cast<u32x4*>(C + static_cast<int64_t>(row0 + orow) * a.ldc + col0 + ocol) = packed;
    if (CT == nullptr) return;  // uniform over the workgroup
  }
  __syncthreads();  // every thread has read its sums
  constexpr int kLdT = kSmallTile + 8;
  uint16_t* transposed = reinterpret_cast<uint16_t*>(sums);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    transposed[(ocol + 2 * e) * kLdT + orow] = static_cast<uint16_t>(packed[e]);
    transposed[(ocol + 2 * e + 1) * kLdT + orow] = static_cast<uint16_t>(packed[e] >> 16);
  }
  __syncthreads();
  const u32x4 eight = *reinterpret_cast<const u32x4*>(transposed + orow * kLdT + ocol);  // column orow of the tile
  if (update_transposed) update_param8(a, args.update_dtype, col0 + orow, row0 + ocol, eight);
  else *reinterpret_cast<u32x4*>(CT + static_cast<int64_t>(col0 + orow) * ldct + row0 + ocol) = eight;
}

GemmTuning g_tuning;
std::mutex g_tuning_mutex;  // the setter may be called while other threads launch: every launch works on one snapshot

GemmTuning tuning_snapshot() {
  std::lock_guard<std::mutex> lock(g_tuning_mutex);
  return g_tuning;
}

// Tiles a product computes: every tile of a general product, the tiles on or below the diagonal of a symmetric one.
int tile_count(const GemmGroup& g, const GemmProblem& p, int tile) {
  const int tm = (p.M + tile - 1) / tile, tn = (p.N + tile - 1) / tile;
  return g.symmetric ? tm * (tm + 1) / 2 : tm * tn;
}

// Below this many slabs a tile is never cut: the pieces would be gone before the fix-up launch (4 us and more) has paid off.
constexpr int kMinSplitSlabs = 17;

// What a tile variant costs, in microseconds: one slab of a tile when few CUs are busy (lone_slab_us: for the variant with two
// workgroups per CU, while each has one of its own) and when the machine is full (slab_us: power and LDS shared by all; in
// between it grows with the workgroups of the launch), prologue and epilogue of a tile (tile_us).  The constants, and those of
// the fix-up launch below, follow 682 traced products: 25 matrices of 512 to 13824, both tiles, whole and cut into 2 to 16
// pieces (11 % rms; the plans they choose are 1.7 % slower than the best measured one in the mean.  With one rate for every
// launch beyond a workgroup per CU it was 23 % and 3.3 %, and the gram product of 2560 x 6912 was not cut: 69 us where two
// pieces take 55).  The tile they choose
// is the faster one on the groups measured (whole Muon step, symmetric / general products forced to 256 or 128):
// hidden4096 7.28 ms against 7.85 / 8.09 with small tiles, two hidden5120 matrices 11.0 against 12.1 / 12.8, five small ragged
// ones 0.344 against 0.427 / 0.406 with big ones, 24 of 1536 x 1024 1.23 against 1.27 / 1.29 with small ones.
constexpr int kSmallVariant = 4;
struct Variant {
  int tile, per_cu;
  double slab_us, lone_slab_us, tile_us;
};
constexpr Variant kVariants[5] = {{}, {256, 1, 1.35, 1.00, 8.6}, {128, 2, 0.86, 0.65, 4.7}, {}, {kSmallTile, 1, 0.45, 0.45, 4.6}};
constexpr double kFixupUs = 3.2, kFixupBytesPerUs = 3.0e6;  // of the fix-up launch: its partial tiles written and read again

// When the workgroups of a launch end, if each starts on the slot that is free first (as they do, in block order).
// Slots are kept as groups that are free at the same time; a launch of equal tiles costs a few steps per round.  Every call
// of add leaves at most one group more (a group is taken whole for each one that comes in, but for the last), so the groups
// of a launch's whole tiles and pieces fit an array.
class SlotTimes {
 public:
  explicit SlotTimes(int slots) : groups_{{0.0, slots}}, n_(1) {}
  void add(int workgroups, double us) {
    while (workgroups > 0) {
      const Slots busy{groups_[0].time + us, std::min(workgroups, groups_[0].count)};
      groups_[0].count -= busy.count;
      workgroups -= busy.count;
      if (groups_[0].count == 0) std::copy(groups_ + 1, groups_ + n_--, groups_);
      Slots* at = std::lower_bound(groups_, groups_ + n_, busy, [](const Slots& x, const Slots& y) { return x.time < y.time; });
      if (at != groups_ + n_ && at->time == busy.time) {
        at->count += busy.count;
      } else {
        std::copy_backward(at, groups_ + n_, groups_ + n_ + 1);
        *at = busy;
        ++n_;
      }
    }
  }
  double end() const { return groups_[n_ - 1].time; }

 private:
  struct Slots { double time; int count; };
  Slots groups_[2 * kMaxGemmGroup + 2];
  int n_;
};

GemmPlan make_plan(const GemmGroup& g, int variant, const GemmScratch& scratch, const GemmTuning& tuning) {
  const Variant& v = kVariants[variant];
  const int cus = device_cu_count(), slots = cus * v.per_cu;
  GemmPlan plan;
  plan.variant = variant;
  for (int i = 0; i < g.n; ++i) plan.order[i] = i;
  std::stable_sort(plan.order, plan.order + g.n, [&](int a, int b) { return g.problem[a].K > g.problem[b].K; });
  int tiles[kMaxGemmGroup], slabs[kMaxGemmGroup], total = 0;
  for (int i = 0; i < g.n; ++i) {
    tiles[i] = tile_count(g, g.problem[plan.order[i]], v.tile);
    slabs[i] = g.problem[plan.order[i]].K / kSlabK;
    total += tiles[i];
    plan.split_tiles[i] = 0;
    plan.splits[i] = 1;
  }
  // The last total % slots tiles (those with the shortest K) are the ones that may be cut: the others fill whole rounds.
  int rest[kMaxGemmGroup];
  for (int i = g.n - 1, left = total % slots; i >= 0; --i) {
    rest[i] = std::min(left, tiles[i]);
    left -= rest[i];
  }
  const double tile_bytes = static_cast<double>(v.tile) * v.tile * 4;
  // tries pieces of about `piece` slabs (0: nothing is cut) and keeps the plan if it is the fastest so far
  auto consider = [&](int piece) {
    int splits[kMaxGemmGroup], blocks = 0;
    int64_t partial = 0;
    for (int i = 0; i < g.n; ++i) {
      splits[i] = 1;
      if (piece > 0 && rest[i] > 0 && slabs[i] >= kMinSplitSlabs && 4 * slabs[i] > 5 * piece) splits[i] = std::min((slabs[i] + piece - 1) / piece, tuning.max_splits);
      if (splits[i] > 1) partial += static_cast<int64_t>(rest[i]) * splits[i];
      blocks += tiles[i] + rest[i] * (splits[i] - 1);
    }
    if (piece > 0 && (partial == 0 || partial > 0x7fffffff || partial * tile_bytes > static_cast<double>(scratch.partials_bytes))) return;
    const double full = std::min(1.0, std::max(0.0, static_cast<double>(blocks) / cus - (v.per_cu - 1)));
    const double slab_us = v.lone_slab_us + (v.slab_us - v.lone_slab_us) * full;
    SlotTimes times(slots);
    for (int i = 0; i < g.n; ++i) times.add(tiles[i] - (splits[i] > 1 ? rest[i] : 0), slabs[i] * slab_us + v.tile_us);
    for (int i = 0; i < g.n; ++i)
      if (splits[i] > 1) times.add(rest[i] * splits[i], (slabs[i] + splits[i] - 1) / splits[i] * slab_us + v.tile_us);
    const double us = times.end() + (partial > 0 ? kFixupUs + partial * tile_bytes / kFixupBytesPerUs : 0.0);
    if (piece > 0 && us >= plan.us) return;
    plan.us = us;
    for (int i = 0; i < g.n; ++i) {
      plan.splits[i] = splits[i];
      plan.split_tiles[i] = splits[i] > 1 ? rest[i] : 0;
    }
  };
  consider(0);
  if (variant == kSmallVariant || !tuning.split_remainder || scratch.partials == nullptr) return plan;
  // piece lengths worth a look: every fraction of the longest K that may be cut, and the other K themselves
  int longest = 0, tried = 0;
  for (int i = 0; i < g.n; ++i)
    if (rest[i] > 0 && slabs[i] >= kMinSplitSlabs) longest = std::max(longest, slabs[i]);
  for (int c = 2; longest > 0 && c <= tuning.max_splits; ++c) consider((longest + c - 1) / c);
  for (int i = 1; i < g.n && tried < 4; ++i)
    if (rest[i] > 0 && slabs[i] != slabs[i - 1] && slabs[i] < longest) {
      consider(slabs[i]);
      ++tried;
    }
  return plan;
}

template <int BM, int BN, int WM, int WN, int BK, int STAGES, int OCC, int N>
int launch(const GemmGroup& g, const GemmPlan& plan, const GemmScratch& scratch, const GemmTuning& tuning, hipStream_t stream) {
  LaunchArgs<N> args;
  args.n = g.n;
  args.symmetric = g.symmetric;
  args.group_m = std::max(1, tuning.group_m);
  args.round_tiles = std::max(kXcds, device_cu_count() * OCC / kXcds * kXcds);
  args.update_dtype = g.update_dtype;
  args.alpha = g.alpha;
  args.beta = g.beta;
  args.partials = static_cast<float*>(scratch.partials);
  int tile = 0, piece = 0, split = 0, partial = 0, classes = 0;
  for (int i = 0; i <= N; ++i) {
    args.tile_begin[i] = tile;
    args.split_begin[i] = split;
    args.piece_begin[i] = piece;
    if (i >= g.n) continue;
    GemmProblem& p = args.problem[i] = g.problem[plan.order[i]];
    if (i == 0 || p.K != args.problem[i - 1].K) args.class_begin[classes++] = tile;
    p.splits = plan.splits[i];
    p.partial_base = partial;
    tile += tile_count(g, p, BM) - plan.split_tiles[i];
    split += plan.split_tiles[i];
    piece += plan.split_tiles[i] * plan.splits[i];
    partial += plan.split_tiles[i] * plan.splits[i];
  }
  for (int i = 0; i <= N; ++i) args.piece_begin[i] += tile;  // block ids: behind the whole tiles
  for (int i = classes; i <= N; ++i) args.class_begin[i] = tile;
  constexpr size_t smem_loop = static_cast<size_t>(STAGES) * (BM + BN) * BK * sizeof(uint16_t);
  constexpr size_t smem_c = static_cast<size_t>(BM) * (BN + 8) * sizeof(uint16_t), smem_ct = static_cast<size_t>(BN) * (BM + 8) * sizeof(uint16_t);
  constexpr size_t smem_epilogue = smem_c > smem_ct ? smem_c : smem_ct;
  constexpr size_t smem = smem_loop > smem_epilogue ? smem_loop : smem_epilogue;
  auto kernel = gemm_nt_kernel<BM, BN, WM, WN, BK, STAGES, OCC, N>;
  {
    // raising the dynamic LDS limit is needed once per kernel and device
    static std::mutex mu;
    static bool configured[64] = {false};
    int dev = 0;
    MFSDP_HIP_TRY(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    if (dev < 0 || dev >= 64 || !configured[dev]) {
      MFSDP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(smem)));
      if (dev >= 0 && dev < 64) configured[dev] = true;
    }
  }
  hipLaunchKernelGGL(kernel, dim3(tile + piece), dim3(WM * WN * 64), smem, stream, args);
  MFSDP_CHECK_LAUNCH("gemm_nt_kernel");
  if (split > 0) {
    hipLaunchKernelGGL((splitk_fixup_kernel<BM, BN, N>), dim3(split * (BM / 64) * (BN / 64)), dim3(kFixupThreads), 0, stream, args);
    MFSDP_CHECK_LAUNCH("splitk_fixup_kernel");
  }
  return MFSDP_OK;
}

template <int N>
int launch_small(const GemmGroup& g, const GemmPlan& plan, const GemmTuning& tuning, hipStream_t stream) {
  SmallArgs<N> args;
  args.symmetric = g.symmetric;
  args.group_m = std::max(1, tuning.group_m);
  args.update_dtype = g.update_dtype;
  args.alpha = g.alpha;
  args.beta = g.beta;
  int tile = 0;
  for (int i = 0; i < g.n; ++i) {
    args.problem[i] = g.problem[plan.order[i]];
    args.begin[i] = tile;
    tile += tile_count(g, args.problem[i], kSmallTile);
  }
  for (int i = g.n; i < N; ++i) args.begin[i] = tile;
  hipLaunchKernelGGL(gemm_small_kernel<N>, dim3(tile), dim3(kSmallThreads), 0, stream, args);
  MFSDP_CHECK_LAUNCH("gemm_small_kernel");
  return MFSDP_OK;
}

}  // namespace

void set_gemm_tuning(const GemmTuning& t) {
  std::lock_guard<std::mutex> lock(g_tuning_mutex);
  g_tuning = t;
}
GemmTuning get_gemm_tuning() { return tuning_snapshot(); }

GemmPlan gemm_plan(const GemmGroup& g, const GemmScratch& scratch) {
  const GemmTuning tuning = tuning_snapshot();
  const int variant = g.symmetric ? tuning.symmetric_variant : tuning.general_variant;
  bool q_columns = false;
  for (int i = 0; i < g.n; ++i) q_columns = q_columns || (g.problem[i].flags & kGemmQColumns) != 0;
  if (q_columns) return make_plan(g, 1, scratch, tuning);
  if (variant == 1 || variant == 2 || variant == kSmallVariant) return make_plan(g, variant, scratch, tuning);
  const GemmPlan big = make_plan(g, 1, scratch, tuning);
  // On a machine shared with other matrices' kernels the CUs a part-filling triangle of big tiles leaves idle are
  // not lost, and a big tile moves fewer LDS bytes per flop.
  if (g.symmetric && g.shared && 4 * tile_count(g, g.problem[0], 256) >= device_cu_count()) return big;
  const GemmPlan small = make_plan(g, 2, scratch, tuning);
  const GemmPlan& better = big.us <= small.us ? big : small;
  // 64 x 64 tiles for one round at most: a second round costs as much as the first (1024 x 1536 update: 384 of them 279 us a
  // step against 241 with 128 x 128 tiles; eight matrices of 512 x 1536: 495 against 281).  Within a round the model decides;
  // K beyond about 2000 goes to 128 x 128 tiles cut along K (gram of 768 x 2304).
  int tiles = 0;
  for (int i = 0; i < g.n; ++i) tiles += tile_count(g, g.problem[i], kSmallTile);
  if (tiles > device_cu_count()) return better;
  const GemmPlan smallest = make_plan(g, kSmallVariant, scratch, tuning);
  return smallest.us < better.us ? smallest : better;
}

bool on_256_tiles(const GemmPlan& plan) { return kVariants[plan.variant].tile == 256; }

int64_t gemm_nt_executed_flops(const GemmGroup& g) {
  GemmScratch scratch;
  scratch.partials_bytes = kGemmPartialsBytes;
  scratch.partials = &scratch;  // only its presence counts
  const int tile = kVariants[gemm_plan(g, scratch).variant].tile;
  int64_t flops = 0;
  for (int i = 0; i < g.n; ++i) flops += 2 * static_cast<int64_t>(tile) * tile * g.problem[i].K * tile_count(g, g.problem[i], tile);
  return flops;
}

int gemm_nt_bf16(const GemmGroup& g, const GemmPlan& plan, const GemmScratch& scratch, hipStream_t stream) {
  if (g.n < 1 || g.n > kMaxGemmGroup) return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: %d problems in one launch", g.n);
  for (int i = 0; i < g.n; ++i) {
    const GemmProblem& a = g.problem[i];
    if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.K % kSlabK)
      return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: M=%d, N=%d must be positive and K=%d a multiple of %d", a.M, a.N, a.K, kSlabK);
    if (g.symmetric && a.M != a.N) return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: symmetric product needs M == N");
    if ((a.flags & kGemmSkipC) && (g.symmetric || !a.CT)) return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: skipping C needs a transposed output and a general product");
    if (!a.P || !a.Q || !a.C) return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: null operand");
    // tiles reach beyond M and N: rows up to the next multiple of 256 must exist (the caller's word), columns are checked
    const int mp = (a.M + 255) / 256 * 256, np = (a.N + 255) / 256 * 256;
    const bool q_columns = (a.flags & kGemmQColumns) != 0;
    if (q_columns && (g.symmetric || plan.variant != 1 || a.K < a.M || static_cast<int64_t>(mp) * a.ldq > kMaxQColumnsElements))
      return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: a Q of K rows needs a general product over M on 256 x 256 tiles and less than 2 GiB");
    if (a.ldp < a.K || a.ldq < (q_columns ? np : a.K) || a.ldc < np || (a.D && a.ldd < np) || (a.CT && a.ldct < mp))
      return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: leading dimension smaller than the padded row length");
    if ((a.ldp | a.ldq) % 8 || (reinterpret_cast<uintptr_t>(a.P) | reinterpret_cast<uintptr_t>(a.Q)) % 16)
      return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: operands must be 16-byte aligned with leading dimensions multiple of 8");
    if ((a.ldc % 8) || reinterpret_cast<uintptr_t>(a.C) % 16 || (a.D && ((a.ldd % 8) || reinterpret_cast<uintptr_t>(a.D) % 16)) ||
        (a.CT && ((a.ldct % 8) || reinterpret_cast<uintptr_t>(a.CT) % 16)))
      return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: C, D and the transposed output must be 16-byte aligned with leading dimensions multiple of 8");
    if (a.D && (a.K < a.M || g.alpha == 0.0f)) return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: a D operand needs K >= M and alpha != 0");
    if (a.ldp > kMaxGemmLeading || a.ldq > kMaxGemmLeading) return fail(MFSDP_ERR_UNSUPPORTED, "gemm_nt_bf16: leading dimensions beyond 2^22 elements");
    if (a.update_param != nullptr && (g.symmetric || (g.update_dtype != MFSDP_F32 && g.update_dtype != MFSDP_BF16) ||
                                      reinterpret_cast<uintptr_t>(a.update_param) % (g.update_dtype == MFSDP_F32 ? 4 : 2)))
      return fail(MFSDP_ERR_INVALID, "gemm_nt_bf16: parameter update needs a general product and an aligned f32 / bf16 parameter");
  }
  const GemmTuning tuning = tuning_snapshot();
  // Slabs of 32 (three to five deep) were measured too: each slab row is then half a 128-byte line, the vector
  // cache looks every line up twice, and the products run 15-25 % slower than with slabs of 64 two deep.
  if (plan.variant == kSmallVariant)
    return g.n <= 2   ? launch_small<2>(g, plan, tuning, stream)
           : g.n <= 8 ? launch_small<8>(g, plan, tuning, stream)
                      : launch_small<kMaxGemmGroup>(g, plan, tuning, stream);
  if (plan.variant == 2)  // 128x128 tile, 4 waves of 64x64, two workgroups per CU
    return g.n == 1  ? launch<128, 128, 2, 2, 64, 2, 2, 1>(g, plan, scratch, tuning, stream)
           : g.n <= 8 ? launch<128, 128, 2, 2, 64, 2, 2, 8>(g, plan, scratch, tuning, stream)
                      : launch<128, 128, 2, 2, 64, 2, 2, kMaxGemmGroup>(g, plan, scratch, tuning, stream);
  // 256x256 tile, 8 waves of 128x64, one workgroup per CU
  return g.n == 1  ? launch<256, 256, 2, 4, 64, 2, 1, 1>(g, plan, scratch, tuning, stream)
         : g.n <= 8 ? launch<256, 256, 2, 4, 64, 2, 1, 8>(g, plan, scratch, tuning, stream)
                    : launch<256, 256, 2, 4, 64, 2, 1, kMaxGemmGroup>(g, plan, scratch, tuning, stream);
}

}  // namespace mfsdp
