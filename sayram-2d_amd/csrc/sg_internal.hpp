// sg_internal.hpp -- device-side data structures of the gfx950 PPFV step.
//
// One instance (one Solver in the reference, source/Solver.h:18-82) lives in
// one device slab. The 5-point operator is 5 bands and the multigrid levels are
// 9 bands, one value per cell each. Many instances of different sizes are
// processed by the same launches through per-level block/line maps.
//
// Device cell order. The reference numbers cells K = j*nx + i
// (source/Mesh.h:66-68). On the device every cell array of a level stores row
// j as its even-i cells followed by its odd-i cells:
//   slot(i, j) = j*nx + (i even ? i/2 : hx + i/2),   hx = (nx + 1) / 2.
// The zebra column sweeps solve every other column; in this order the columns
// of one colour are adjacent in memory, so their loads use whole cache lines
// (in the plain order every fetched line is half wasted). Rows stay two
// contiguous runs, and the coarse row J (the even points of fine row 2J) is
// exactly the first half of the fine row. Host arrays keep the reference's
// layouts; the conversion happens at upload and download.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace sg {

constexpr int kMaxLev = 16;
// partial sums per level-0 workgroup (the finalize pass uses all five)
constexpr int kNumPartials = 5;
// Cells per instance: every per-cell array then stays below 2 GiB, so kernels
// may address it with 32-bit byte offsets from its base.
constexpr long long kMaxCells = 1LL << 28;
constexpr int kBlock = 256;     // cells per workgroup in cell-parallel kernels
constexpr int kLightBlocks = 4; // map entries per workgroup of the lightest vector kernels
constexpr int kEnt = 4;         // map entries per workgroup of the multi-entry cell kernels
// Tile shapes of the line solves: L lines x S steps staged through LDS by a
// workgroup of NT threads, each thread owning 4 consecutive steps of a line in
// the solve:
//   0: 64 x 16 (256 threads)  short lines
//   1: 16 x 64 (256 threads)  medium rows; long columns of FP64 9-point levels
//   2:  4 x 256 (256 threads) long rows (a row is contiguous in memory)
//   3: 16 x 256 (1024 threads) long columns (16 columns of one colour are 64
//      contiguous bytes per row; 4x fewer serial tiles than shape 1)
//   4: 32 x 32 (256 threads) medium columns (32 columns of one colour are 128
//      contiguous bytes per row, so rows at any offset waste less of each
//      fetched line)
constexpr int kNumTileShapes = 5;
__host__ __device__ constexpr int tile_steps(int sh) {
  return sh == 0 ? 16 : sh == 1 ? 64 : sh == 4 ? 32 : 256;
}
__host__ __device__ constexpr int tile_lines(int sh) {
  return sh == 0 ? 64 : sh == 1 ? 16 : sh == 2 ? 4 : sh == 3 ? 16 : 32;
}
__host__ __device__ constexpr int tile_threads(int sh) { return sh == 3 ? 1024 : 256; }
// Rank of a shape by the length of the lines it takes (the longest lines are
// the critical path of a sweep).
__host__ __device__ constexpr int shape_rank(int sh) { return sh == 4 ? 1 : sh; }
// Tiles of the eliminated right-hand side d that a line sweep keeps in LDS
// (the last ones of each line; earlier tiles are parked in x and read back by
// the backward pass), for values of tbytes bytes and an nb-point operator.
// Sized so that the LDS of a workgroup does not lower the occupancy its
// registers allow, except for the 5-point 32 x 32 tiles: 9 tiles (288 steps)
// at 3 workgroups per CU measured faster than 6 at 4 (fewer parked tiles of the
// 512-cell columns). The 5-point long-line shapes (2, 3) hold one tile more
// than the 9-point ones, whose registers allow fewer workgroups.
__host__ __device__ constexpr int ring_tiles(int sh, int tbytes, int nb) {
  if (tbytes != 4) return sh == 3 ? 1 : 2;
  switch (sh) {
    case 0: return 2;
    case 2: return nb == 9 ? 4 : 5;
    case 3: return nb == 9 ? 6 : 7;
    case 4: return nb == 9 ? 8 : 9;
    default: return 4;
  }
}

// The sweeps with the lines in registers (sg_sweeps.hip), as further shapes of
// the sweep maps: 5 columns of at most 512 steps, 6 columns of at most 4096
// (another kernel: its runs need more registers), 7 rows of at most 2048, 8
// rows of at most 4096.
constexpr int kNumSweepShapes = 9;
constexpr int kColShape = 5, kColLongShape = 6, kRowShape = 7, kRowLongShape = 8;
constexpr int kColThreads = 512, kColMax = 512, kColLongMax = 4096;
constexpr int kRowThreads = 256, kRowMax = 2048, kRowLongMax = 4096;
// Columns per workgroup by line length n and value size: as many as leave a
// thread runs that its registers hold, so that a row's load is as long a
// piece of memory as can be.
__host__ __device__ constexpr int col_lines(int n, int tbytes) {
  if (n <= 64) return 32;
  if (n <= 512) return 16;
  if (tbytes == 4) return n <= 768 ? 16 : 8;
  return n <= 1024 ? 8 : 4;
}

// Rows per workgroup: as many as its four waves take, each a segment of the
// lanes that 8 (FP64 rows of at most 256: 4) steps per lane make, a power of
// two, at most 64; longer rows take 2 or 4 waves.
__host__ __device__ constexpr int row_lines(int n, int tbytes) {
  if (n > 1024) return 1;
  if (n > 512) return 2;
  const int k = tbytes == 8 && n <= 256 ? 4 : 8;
  int w = 1;
  while (w * k < n) w *= 2;
  return kRowThreads / w;
}

__host__ __device__ inline int half_x(int nx) { return (nx + 1) >> 1; }

// The prolongation fills only the lines the first post-smoothing sweep reads:
// odd rows before x-lines (1), odd columns before y-lines (2), else every
// point (0). `smoother` bits: 1/2 pre x/y, 4/8 post x/y.
__host__ __device__ inline int prolong_rows(int smoother) {
  return (smoother & 4) ? 1 : (smoother & 8) ? 2 : 0;
}
// After a pre-smoothing sweep of x-lines alone the odd rows (colour 1, solved
// last from the even rows' new values) satisfy their line equations, so the
// residual the restriction needs is that of the even rows only.
__host__ __device__ inline bool half_residual(int smoother) {
  return (smoother & 3) == 1;
}
// position of column i within its row
__host__ __device__ inline int xslot(int i, int hx) { return (i & 1) ? hx + (i >> 1) : (i >> 1); }
// column stored at position p of a row
__host__ __device__ inline int xcol(int p, int hx) { return p < hx ? 2 * p : 2 * (p - hx) + 1; }
__host__ __device__ inline size_t cell_slot(int i, int j, int nx) {
  return (size_t)j * nx + xslot(i, half_x(nx));
}

// The coarse end of a V-cycle runs in one workgroup per instance: the fused
// coarse cycle, from the first level that fits (fused_fits) and has at most
// fuse_cells cells. Sides of at most kFuseSide make lines of at most 16 lanes; a
// 64 x 48 level costs the cycle 12 us more and saves some nine launches of 4 us.
// Levels of at most kFuseLongCells cells may have sides of up to kFuseLong, lines of
// up to a wave: with a launch per level strips of two cells by 65 to 130 took up to
// 24% longer than fused, longer ones are no slower.
constexpr int kFuseCells = 4096;     // the largest level that fits (the default takes any)
constexpr int kFuseLimit64 = 1024;   // the largest limit FP64 V-cycles accept
constexpr int kFuseSide = 64, kFuseLong = 256, kFuseLongCells = 1024;
constexpr int kFuseThreads = 512;
__host__ __device__ constexpr bool fused_fits(int nx, int ny) {
  const int side = nx > ny ? nx : ny;
  return side <= kFuseSide || (side <= kFuseLong && nx * ny <= kFuseLongCells);
}
// Coarsening ends at the first level of at most kDense cells, which is solved by
// the inverse of its operator (one wave's lanes are the rows).
constexpr int kDense = 64;

// The lanes of a sweep colour in the fused cycle: a line of n cells is a segment
// of W = 1 << lw lanes, K steps each: one step while the line then has at most 16
// lanes and the colour fits the workgroup, else four. lanes counts whole waves.
struct LineLanes { int K, lw, nl, lanes; };
__host__ __device__ constexpr LineLanes line_lanes(int n, int np, int colour) {
  LineLanes a{1, 0, (np - colour + 1) >> 1, 0};
  while ((1 << a.lw) < n) ++a.lw;
  if (a.lw > 4 || (a.nl << a.lw) > kFuseThreads) {
    a.K = 4;
    a.lw = a.lw > 2 ? a.lw - 2 : 0;
  }
  a.lanes = ((a.nl << a.lw) + 63) & ~63;
  return a;
}
// (odd pitch: a column's stride then spreads over the LDS banks)
__host__ __device__ constexpr int fused_pitch(int nx) { return (nx + 2) | 1; }
// Its operator, packed per step in the order its lanes read it, one group of
// arrays per level and kind: rows and columns of either colour (9 arrays: -lo
// inv, inv, -up, and the couplings to the lines beside), the weights of the
// residual's restriction (rows of colour 0; 2 arrays, zeros, and the first of
// the couplings again) and of the prolongation (4, rows of colour 1). A phase
// reads the first 4 arrays of one group and, if it has couplings, arrays 4 to 8
// of a sweep's. Offsets in values from the level's start.
enum PackKind { PK_ROW0, PK_ROW1, PK_COL0, PK_COL1, PK_RES, PK_PRO, kNumPack };
__host__ __device__ constexpr int pack_arrays(int kind) {
  return kind < PK_RES ? 9 : 4;
}
__host__ __device__ constexpr LineLanes pack_lanes(int nx, int ny, int kind) {
  return kind == PK_COL0 || kind == PK_COL1
             ? line_lanes(ny, nx, kind == PK_COL1)
             : line_lanes(nx, ny, kind == PK_ROW1 || kind == PK_PRO);
}
__host__ __device__ constexpr int pack_offset(int nx, int ny, int kind) {
  int o = 0;
  for (int k = 0; k < kind; ++k) {
    const LineLanes a = pack_lanes(nx, ny, k);
    o += pack_arrays(k) * a.lanes * a.K;
  }
  return o;
}
// One phase of the cycle (built once per instance on the host): what it does,
// the lanes and lines it takes, and its places in LDS: x0 of the first line's
// step 0, sl and sp the strides along and across the lines; pack: its first 4
// arrays, pack2: its next 5 (negative: none); aux, pc: place and pitch in the next level (its b or x).
enum TaskKind { TK_ZERO, TK_SWEEP, TK_RES, TK_RESTB, TK_DENSE, TK_PRO, TK_PROALL, TK_END };
struct CoarseTask {
  int kind, K, lw, n, nl, lanes, x0, sl, sp, pack, aux, pc, lev, pack2, pad[2];
};
static_assert(sizeof(CoarseTask) == 64, "one scalar load");
constexpr int kMaxTasks = 64;

// band slots; level 0 uses the first five (the operator is 5-point), coarse
// Galerkin levels use all nine.
enum Band { BC = 0, BW = 1, BE = 2, BS = 3, BN = 4, BSW = 5, BSE = 6, BNW = 7, BNE = 8 };

// Krylov vector slots (precision of the Krylov iteration).
enum Vec { VR = 0, VRH, VP, VV, VS, VT, VPH, VSH, VXK, kNumVec };
// FP32 level-0 vectors of an FP64 Krylov solve with an FP32 V-cycle: the
// V-cycle input (p or s, scaled) and its outputs for p and s. Ids continue
// the Krylov slots, so a V-cycle addresses either kind by one index.
enum PcVec { PV_B = kNumVec, PV_P, PV_PH, PV_SH, PV_RH, kNumVecAll };

// solver status per instance
enum Status : int { ST_ACTIVE = 0, ST_HALF = 1, ST_DONE = 2, ST_FAIL = 3, ST_IDLE = 4 };

struct KScal {          // per-instance Krylov scalars, FP64 storage
  double rho, rho_old, alpha, omega, beta;
  double bnorm2, rnorm2, tol2;
  double scale;          // mixed: norm of the FP64 residual being corrected
  double pcs;            // FP32 V-cycle of an FP64 solve: scale of its input
                         // and output, the current residual norm
  double pcs_p;          // PC32: the scale the stored FP32 direction p was
                         // written with (pcs of the previous iteration)
  double onorm2, obnorm2, otol2;   // mixed: outer (FP64) residual norms
  double oprev2;         // mixed: residual norm^2 of the previous refinement
  double best2;          // smallest Krylov residual norm^2 of this solve
  int best_it;           // iteration at which it was reached
  int phase;             // step end: 0 solving, 1 finalized in this pass (f is
                         // written next), 2 finished in an earlier pass
  double true_rel;       // finalize: ||R - M x|| / ||R|| of the solution x
  double minf;           // finalize: min x (f before clamping)
  double theta;          // warm start: the next solve starts at f + theta df
  int iters, status;     // Krylov iteration count and status of this solve
  int ostatus, orefs;    // mixed: outer refinement status and count; every
                         // precision: ST_FAIL after finalize rejects the step
  int maxit, clamps;
  int omaxit, part;
  int titers;           // Krylov iterations summed over the refinements of a step
  int vcyc;             // level-0 V-cycles this instance ran in the step
  int nonfin;           // finalize: cells whose x is not finite
  int hist;             // 1: df holds the increment of an accepted step
};

struct Lev {            // one multigrid level of one instance
  int nx, ny;
  double *band64[9];    // FP64 operator (level 0: the 5 assembled bands)
  void *band[9];        // V-cycle precision copy (aliases band64 in FP64 mode)
  void *pw[4];          // prolongation weights to the next coarser level
  void *linv[2], *lup[2];   // LU factors of the row (0) and column (1) line
                            // matrices: 1/pivot and the eliminated upper entry
  void *x, *b, *cp, *dp;
  void *dinv;           // last level of at most kDense cells: inverse operator,
                        // entry (row r, column c) at c * cells + r, cells in
                        // row order (j nx + i)
};

struct InstDev {
  int nx, ny, nlev, bcmask;   // bcmask bit s set: side s Dirichlet
  int nblk0;                  // level-0 workgroups of this instance
  int prec;                   // sg_precision of the instance
  int noclamp;                // 1: f = x at the end of a step (no clamp at 0)
  int warm;                   // 1: the solve starts at f + theta df, 0: at f
  double dt;
  // geometry (source/Mesh.cc:36-65) and per-vertex interpolation weights of
  // fill_vertex_from_cells (source/Solver.cc:326-381), computed once
  const double *xe, *ye;
  const double *wx0, *wx1, *wy0, *wy1;
  const double *bcv[4];
  // Equation inputs, device cell order: G, D, 1/tau (the assembly forms
  // Lambda = G*D, source/Solver.cc:57-65, as it reads them)
  const double *G, *Dxx, *Dxy, *Dyy, *itau;
  // FP64 state
  double *f, *R, *x, *r64;
  float *df;                  // f^n - f^(n-1) of the last accepted step
                              // (valid when KScal::hist is 1)
  double *band64[5];
  void *kv[kNumVec];          // Krylov vectors (double, or float in MIXED)
  float *pv[kNumVecAll - kNumVec];   // PC32: FP32 V-cycle inputs (s, p) and outputs,
                                     // shadow residual
  double *partial;            // kNumPartials * nblk0
  unsigned int *ticket;       // 2 tickets
  KScal *sc;
  // fused coarse cycle: its phases, and the packed operator (V-cycle precision)
  const CoarseTask *tasks;
  void *pack;
  Lev lev[kMaxLev];
};

struct BlkMap { int inst; int k0; };      // cell-parallel: 256 cells of one instance
struct LineGrp { int inst; int first; int count; int step; };   // lines first + k*step, k < count
// lines first + k * step of one colour and direction of a level, by tile shape
struct FacGrp { int inst, first, count, step, lev, dir, shape, pad; };
// The instance table a kernel gets, with the statuses of the instances beside
// it (KScal::status and ostatus by compact index, mirrored by the kernels that
// change them): a workgroup reads its status and its instance's pointers in
// the same round trip instead of following the table to the scalars first.
// No kernel writes the table, so it is read through the constant address space: by
// scalar loads, also after a kernel's own stores, and free to be issued before them.
struct InstStat { int status, ostatus, phase, pad; };
typedef const __attribute__((address_space(4))) InstDev CInst;
typedef const __attribute__((address_space(4))) Lev CLev;
struct Insts {
  const InstDev *t;
  InstStat *st;
  __device__ __forceinline__ CInst &operator[](int k) const { return ((CInst *)t)[k]; }
};
struct PackMap { int inst, lev, kind, off; };   // off: of the kind's arrays in InstDev::pack
// an instance whose levels lev .. last run fused; rows: some of its lines take more
// than a row of 16 lanes
struct FuseMap { int inst, lev, last, rows; };

// Threads of the per-instance finish kernels (sums of the partials).
constexpr int kFinThreads = 1024;

}  // namespace sg
