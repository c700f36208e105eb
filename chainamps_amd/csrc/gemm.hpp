// Grouped, persistent complex GEMM over uneven QN blocks.
//
// One launch covers a list of problems.  Problem p computes
//   C_p[m,n] (+)= sum_s op(A_s)[m,k] * op(B_s)[k,n]
// over its K-segments s (every QN-compatible block pair contributing to the
// same output block), optionally batched (strided) -- the sum over
// segments is accumulated in registers, so every output tile is written
// exactly once and no atomics are needed.  A is M-contiguous
// (A[m + k*csA]); B is either K-contiguous (B[k + n*csB]) or N-contiguous
// (B[k*rsB + n]); C is M-contiguous (C[m + n*csC]).  Complex values are
// interleaved (re,im); a complex multiply runs as three (Gauss) or four real
// MFMAs (v_mfma_f64_16x16x4 for FP64, v_mfma_f32_16x16x4 for FP32).
//
// The launch configuration of a plan -- product form, tile-shape policy, K chunk,
// persistent grid size and, for a small plan, its one-launch kernel -- is chosen
// by autotune(): candidates are timed with HIP events on the plan's own operands
// and the winner is cached under a signature of the plan's block-size histogram,
// so a later plan with the same histogram (the next iDMRG step at the same chi)
// reuses it.
#pragma once
#include <cstdint>
#include <vector>

#include "common.hpp"

namespace cam {

enum : int32_t {
  kSegConjA = 1,
  kSegConjB = 2,
  kSegBNContig = 4,   // B(k,n) at k*rsB + n   (else k + n*csB)
  kSegAKContig = 32,  // A(m,k) at k + m*csA   (else m + k*csA)
};

// Operand addressing: space 0 means the pointer field is an absolute
// address; space k > 0 means it is an element offset from the launch's
// bases.p[k].  Plans built with spaces are precision independent: the same
// plan runs on FP64 (double2) or FP32 (float2) copies of the operands.
constexpr int kMaxSpaces = 12;
struct GemmBases {
  const void* p[kMaxSpaces];
};
inline int32_t seg_spaces(int a, int b) { return (a << 8) | (b << 12); }

struct GemmSeg {
  const void* A;
  const void* B;
  int64_t csA;
  int64_t ldB;        // csB (K-contig) or rsB (N-contig)
  int64_t bsA, bsB;   // batch strides (elements)
  int32_t K;
  int32_t flags;
};

struct GemmProb {
  void* C;
  int64_t csC;
  int64_t bsC;
  int32_t M, N;
  int32_t seg0, nseg;
  int32_t batch;
  int32_t beta;       // 1: accumulate into C
  int32_t cspace;     // operand space of C
};

struct GemmTile {
  int32_t prob, batch, m0, n0;
};

// Row passes (see GemmPlan::rows).  A pass multiplies rows of `nin` input
// columns (the A columns of its problems' segments) with an nin x nout matrix
// (their B blocks) into `nout` output columns (the columns of its problems).
constexpr int kRowN = 16;       // columns of one problem
constexpr int kRowK = 32;       // K of one segment
constexpr int kRowIn = 192;     // input columns of a pass
constexpr int kRowOut = 64;     // output columns of a pass
constexpr int kRowB = 3072;     // elements of the padded matrix (LDS)

struct RowIn {                  // one input column
  int64_t off;                  // segment's A (address or offset, as GemmSeg::A)
  int64_t kcs, bs;              // column offset in it and batch stride (elements)
  int32_t seg, k;               // segment of the pass, column of the segment
};
struct RowOut {                 // one output column
  int64_t off, ncs, bs;
  int32_t prob, n;              // problem of the pass, column of the problem
};
struct RowBlk {                 // B block of (segment, problem)
  int64_t off;
  int32_t ld, flags;
};
struct RowItem {                // rows [.., + rows) of a pass, from row m0 of batch b0
  int32_t in0, out0, blk0;      // first entries in the tables
  int32_t nin, nout, nprob;
  int32_t M, batch0, m0, rows;
  int32_t aspace, bspace, cspace;
  int32_t conjA, beta;
};

constexpr int kDirectSegs = 64;    // segments of one problem of a small plan (see GemmPlan::direct)

// Tile shapes compiled into the kernels (TM x TN per workgroup).
struct TileShape { int tm, tn; };
constexpr int kNumTileShapes = 6;
constexpr TileShape kTileShapes[kNumTileShapes] = {{64, 64}, {32, 64}, {64, 32}, {128, 64}, {64, 128}, {128, 32}};
constexpr int kNumSmallShapes = 3;   // shapes of the policies 0-2

// Host-side grouped GEMM plan: problems + segments; tiles are generated by
// build_tiles() (LPT-sorted by cost) and everything is uploaded once.
enum { kAlgo4M = 0, kAlgo3M = 1 };

constexpr int kTileModes = 4;

// Launch configuration of a plan at one precision.
struct LaunchCfg {
  int algo = kAlgo3M;   // complex product: kAlgo4M or kAlgo3M real MFMAs
  int tile_mode = 1;    // 0: fixed 64x64; 1: min padded cost per problem;
                        // 2: narrow shapes only (32x64 / 64x32: more tiles);
                        // 3: min padded cost including 128-wide tiles
                        //    (fewer operand re-reads per flop)
  int wg_per_cu = 4;    // persistent grid = min(tiles, CUs * wg_per_cu)
  int kc = 16;          // K chunk per LDS stage: 16 or 8 (half the LDS)
  bool direct = true;   // small plans take the one-launch kernel (false: tiles)
};

struct GemmPlan {
  std::vector<GemmProb> probs;
  std::vector<GemmSeg> segs;
  std::vector<GemmTile> tiles[kTileModes][kNumTileShapes];
  double flops = 0.0;          // algorithmic 8*m*n*k
  // Device copies.  Whatever an upload finds missing goes up in one buffer
  // and one copy (a plan of a small tensor contraction lives for one launch,
  // and an allocation, a free and a copy cost some 1, 1 and 4 us: growth run of
  // the spin chain to chi=48 21.9 -> 20.1 ms, iTEBD to chi=32 7.8 -> 7.2).
  std::vector<DevBuf<char>> d_bufs;
  const GemmProb* d_probs = nullptr;
  const GemmSeg* d_segs = nullptr;
  const GemmTile* d_tiles[kTileModes][kNumTileShapes] = {};
  bool uploaded = false;                  // problems and segments
  bool built[kTileModes] = {false, false, false};
  bool tiles_uploaded[kTileModes] = {false, false, false};
  // Per precision (0 FP64, 1 FP32); plans below the tuning threshold keep the
  // defaults.  FP64 starts from chunks of 8 (more workgroups resident; stages
  // L, B, C, R with 16 and 8, us: chain d=64 chi=64 189 253 259 255 and 166 230
  // 233 241, chi=32 58 59 59 35 and 48 54 54 36, U(1) d=20 chi=300 L / R 164 218
  // and 131 194); in FP32 the two are level (107 138 143 139, 105 144 145 143).
  LaunchCfg cfg[2] = {{kAlgo3M, 1, 4, 8, true}, {}};
  bool tuned[2] = {false, false};
  // Problems with at most kRowN columns whose segments all have K <= kRowK
  // and an M-contiguous A (W stages and environments of small QN sectors: a
  // tile would be mostly padding) run as row passes: problems that read the
  // same input columns share a pass, and the rows of all batch members follow
  // one another.  Tables and items are built with the tiles.
  std::vector<RowIn> row_in;
  std::vector<RowOut> row_out;
  std::vector<RowBlk> row_blk;
  std::vector<RowItem> rows;
  int row_lds = 0;                        // largest padded matrix (elements)
  const RowIn* d_row_in = nullptr;
  const RowOut* d_row_out = nullptr;
  const RowBlk* d_row_blk = nullptr;
  const RowItem* d_rows = nullptr;
  bool rows_built = false, rows_uploaded = false;
  // Plans too small to fill the chip with tiles: one launch for all problems,
  // a workgroup per 16 x 16 outputs (empty: tiles and row passes).
  std::vector<GemmTile> direct;
  const GemmTile* d_direct = nullptr;
  bool direct_uploaded = false;
  // Per problem, a row group (-1: none).  Problems of one group read the
  // same A rows (one output per MPO channel from the same operand rows), so
  // their tiles of equal (batch, m0) are ordered next to each other and run
  // together on one XCD, which then fetches those rows from HBM once.
  std::vector<int64_t> group;

  int add_problem(void* C, int64_t csC, int M, int N, int batch, int64_t bsC, int beta,
                  int cspace = 0);
  void add_segment(int prob, const void* A, int64_t csA, int64_t bsA, const void* B, int64_t ldB,
                   int64_t bsB, int K, int flags);
  void set_group(int prob, int64_t g);
  // tile-shape policy for both precisions (see LaunchCfg::tile_mode)
  void choose_tiles(int mode);
  // a small plan's list, or the tiles of the selected policies, LPT-sorted
  void build_tiles();
  void build_tiles_mode(int mode);
  // the list of a small plan; false for any other
  bool build_direct();
  // tables and items of the row passes over the given problems
  void build_rows(const std::vector<int>& eligible);
  // Histogram signature: problems bucketed by (log2 M, log2 N, log2 K,
  // batched), weighted by flops (5% steps), plus the precision.
  uint64_t signature(int precision) const;
  // drops every list of a plan that is being added to
  void changed();
  // problems, segments and every built tile list to the device
  void upload(hipStream_t s);
  // what a launch at this precision runs: 1 tiles, 2 row passes, 4 the kernel
  // of small plans (summed)
  int route(int precision) const;
  // whether a launch at this precision finds all it needs on the device
  bool on_device(int precision) const;
  void clear();
};

// precision: 0 = FP64 (double2 data), 1 = FP32 (float2 data)
void launch_grouped_gemm(GemmPlan& plan, int precision, hipStream_t s, const GemmBases* bases = nullptr,
                         int grid_limit = 0);

int device_cu_count();

// Picks algo / tile_mode / wg_per_cu for `plan` at `precision` by timing the
// candidates on `stream` with the given operand bases (the plan's outputs
// are overwritten -- every problem must have beta = 0 -- and its inputs
// only read, so the last timed run leaves the correct result).  Plans below
// `min_flops` keep the defaults.  Disabled by CAM_AUTOTUNE=0.  Returns true
// when a configuration was timed or taken from the cache.
bool autotune(GemmPlan& plan, int precision, hipStream_t stream, const GemmBases* bases,
              double min_flops = 2e10);

}  // namespace cam
