// sg_coarse.hip -- the coarse end of the V-cycle: the dense inverse of the last
// level and the fused coarse cycle.
//
// Fused cycle: the levels of one instance from `lev` (its first level that fits,
// fused_fits, and has at most fuse_cells cells) down to its last and back, in one
// workgroup with LDS barriers between the phases, instead of several launches per
// level. Per level on the way down an optional pre-smoothing sweep of x-lines and
// the restriction of the residual (of b itself without pre-smoothing); the last
// level by the inverse of its operator, or as one line if it is a line of more
// than kDense cells; then per level the prolongation of the lines the first
// post-sweep reads and the zebra post-sweeps.
//
// Bound: latency of one workgroup, which walks 8 phases per level, each a few
// LDS accesses and some hundred instructions; bytes do not matter. A wave issues
// a dependent instruction every 8 to 10 cycles, taken branches and code run for
// the first time cost more. Hence:
//  * x and b of every level stay in LDS for the whole cycle, with a border of
//    zeros, so that no neighbour needs a test;
//  * a line of at most 64 cells is a segment of at most 16 lanes (one step per
//    lane, or four), so that both Thomas recurrences are scans of affine maps
//    inside one DPP row; the map at a line's first step has A = 0, which separates
//    the lines of a row without a mask. Lines of up to 256 cells (levels of at most
//    1024) take two or four rows, chained through v_readlane: against launches per
//    level 10 steps of 2048 x 32 FP64 18.8 -> 14.9 ms, of 64 grids of 256 x 4 MIXED
//    18.7 -> 12.8, a step of 66 x 2 MIXED 536 -> 422 us;
//  * the phases are one loop over a table built with the instance, and the
//    operator is packed once per step in the order the lanes read it, zero
//    where a lane has no cell: a phase's operands are a few vector loads from
//    one base, issued while the phase before runs;
//  * the hierarchy ends at kDense cells: the four levels that would follow an
//    8 x 8 level cost 32 phases, the product with its inverse one.
//  * the code is small: each piece of it runs a few times only, and cold.
// Measured per cycle (first level): 90 x 100 FP64 (45 x 50) 28 us, 32 with the
// operand loads inlined at nine places; a version with one thread per line
// took 69 from half the sides on, one with every level, direction and colour
// inlined (60 KB of code) 78.
#include "sg_device.hpp"
#include "sg_kernels.hpp"
#include "sg_scan.hpp"

namespace sg {

// ---------------------------------------------------------------------------
// Inverse of the last level's operator (FP64, stored in the V-cycle precision),
// once per step, by Gauss-Jordan. Wave w holds rows w + 16 r, one lane per
// column, in registers; the scaled pivot row goes through LDS, the pivot column
// comes from a lane of the wave itself: one barrier per pivot.
//
// Pivots: the Galerkin products are no M-matrices (on the log-normal test
// problems the weights have any sign and row sums of up to 380, a coarse
// off-diagonal is up to 2.9 times the diagonal and the smallest pivot of the
// natural order 7e-5 of it), so that order alone is not safe. It is tried
// first, every multiplier watched; if one exceeds 64 or is not finite the
// matrix is read again and inverted with partial pivoting. Measured at 90 x 100
// in FP64 (42 cells): 18.5 us unwatched, 23.0 watched, 40 with pivoting always
// (each pivot waits for two more LDS reads and a maximum over the waves). A
// singular operator gives an infinite inverse, which fails the solve at its first
// reduction.
// ---------------------------------------------------------------------------
// max over a row of 16 lanes, in each of them
__device__ __forceinline__ unsigned row_max(unsigned v) {
#define SG_ROR(N) v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 | N, 0xf, 0xf, true))
  SG_ROR(8); SG_ROR(4); SG_ROR(2); SG_ROR(1);
#undef SG_ROR
  return v;
}
// upper half of |v|: exponent and 20 bits, ordered as |v| is
__device__ __forceinline__ unsigned mag_bits(double v) {
  return (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32) & 0x7fffffffu;
}

template <typename T>
__global__ void __launch_bounds__(1024) k_dense_inverse(const Insts insts,
                                                        const FuseMap *__restrict__ map) {
  constexpr int R = kDense / 16;
  __shared__ double s_row[2][16][kDense];   // natural order: row 0; pivoting: the waves' candidates
  __shared__ unsigned s_key[2][16];
  __shared__ int s_at[kDense], s_of[kDense];   // pivot row of a column, column of a pivot row
  __shared__ int s_bad;
  CInst &I = insts[map[blockIdx.x].inst];
  if (ostatus_of(insts, map[blockIdx.x].inst) == ST_IDLE) return;
  CLev &L = I.lev[I.nlev - 1];
  const int nx = L.nx, ny = L.ny, n = nx * ny, hx = half_x(nx);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool nine = I.nlev > 1;
  double a[R];
  auto load = [&]() __attribute__((always_inline)) {
    const int cj = lane / nx, ci = lane - cj * nx;   // column: cell `lane` in row order
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int K = wave + 16 * r;
      a[r] = 0.0;
      if (K >= n || lane >= n) continue;
      const int j = K / nx, i = K - j * nx;
      const int di = ci - i, dj = cj - j;
      if (di < -1 || di > 1 || dj < -1 || dj > 1) continue;
      const int b = dj == 0 ? (di == 0 ? BC : di < 0 ? BW : BE)
                    : dj < 0 ? (di == 0 ? BS : di < 0 ? BSW : BSE)
                             : (di == 0 ? BN : di < 0 ? BNW : BNE);
      a[r] = (nine || b <= BN) ? gbl(L.band64[b])[j * nx + xslot(i, hx)] : 0.0;
    }
  };
  T *const out = ptr<T>(L.dinv);
  load();
  if (threadIdx.x == 0) s_bad = 0;   // (visible at the first barrier)
  unsigned long long bad = 0;
#pragma unroll
  for (int rp = 0; rp < R; ++rp) {
#pragma unroll 1
    for (int w = 0; w < 16; ++w) {
      const int p = w + 16 * rp;
      if (p >= n) break;   // uniform
      if (wave == w) {
        const double inv = 1.0 / rdlane(a[rp], p);
        a[rp] = lane == p ? inv : a[rp] * inv;
        s_row[p & 1][0][lane] = a[rp];
      }
      lds_barrier();
      const double rv = s_row[p & 1][0][lane];
      double below = 0.0;   // largest entry of the wave's rows below the pivot, column p
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double c = rdlane(a[r], p);
        if (r > rp || (r == rp && wave > w)) below = fmax(below, fabs(c));
        if (r != rp || wave != w) a[r] = (lane == p ? 0.0 : a[r]) - c * rv;
      }
      bad |= __ballot(!(below * fabs(rv) <= 64.0)) & 1ull << p;   // (lane p of rv: 1 / pivot)
    }
  }
  if (lane == 0 && bad) s_bad = 1;
  lds_barrier();
  if (!__builtin_amdgcn_readfirstlane(s_bad)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int K = wave + 16 * r;
      if (K < n && lane < n) st32(out, (uint32_t)(lane * n + K), (T)a[r]);
    }
    return;
  }
  load();
  // Rows do not move: the pivot of column p is the largest entry of that column
  // (to 14 bits) in a row that was no pivot yet. Each wave offers its own
  // candidate with the row scaled by it.
  unsigned rest = 0;   // bit r: row wave + 16 r was no pivot yet
#pragma unroll
  for (int r = 0; r < R; ++r) rest |= (wave + 16 * r < n ? 1u : 0u) << r;
#pragma unroll 1
  for (int p = 0; p < n; ++p) {
    double c[R], cand = a[0], piv = 1.0;
    unsigned key = 0;   // rows that were pivots, and rows past the matrix
#pragma unroll
    for (int r = 0; r < R; ++r) {
      c[r] = rdlane(a[r], p);
      const unsigned k = (rest >> r & 1)
          ? 0x80000000u | (mag_bits(c[r]) & ~63u) | (63 - (wave + 16 * r)) : 0u;
      if (k > key) { key = k; cand = a[r]; piv = c[r]; }
    }
    const double inv = 1.0 / piv;
    s_row[p & 1][wave][lane] = lane == p ? inv : cand * inv;
    if (lane == 0) s_key[p & 1][wave] = key;
    lds_barrier();
    const unsigned best = row_max(s_key[p & 1][lane & 15]);
    const int row = 63 - (int)(__builtin_amdgcn_readfirstlane((int)best) & 63);
    const double rv = s_row[p & 1][row & 15][lane];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool own = row == wave + 16 * r;
      a[r] = own ? rv : (lane == p ? 0.0 : a[r]) - c[r] * rv;
      if (own) rest &= ~(1u << r);
    }
    if (threadIdx.x == 0) { s_at[p] = row; s_of[row] = p; }
  }
  lds_barrier();
  // Row K now is row s_of[K] of the inverse, column p stands for column s_at[p].
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int K = wave + 16 * r;
    if (K < n && lane < n) st32(out, (uint32_t)(s_at[lane] * n + s_of[K]), (T)a[r]);
  }
}

// ---------------------------------------------------------------------------
// Packed operator of the fused levels, once per step: one workgroup per level
// and kind (PackKind) of an instance; a thread fills its lane's values.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(kFuseThreads) k_coarse_pack(const Insts insts,
                                                              const PackMap *__restrict__ map) {
  const PackMap pm = map[blockIdx.x];
  CInst &I = insts[pm.inst];
  if (ostatus_of(insts, pm.inst) == ST_IDLE) return;
  CLev &L = I.lev[pm.lev];
  const int nx = L.nx, ny = L.ny, hx = half_x(nx), kind = pm.kind;
  const LineLanes g = pack_lanes(nx, ny, kind);
  const bool col = kind == PK_COL0 || kind == PK_COL1, nine = pm.lev > 0;
  const int colour = kind == PK_ROW1 || kind == PK_COL1 || kind == PK_PRO;
  T *const out = ptr<T>(I.pack) + pm.off;
  const int n = col ? ny : nx, total = g.lanes * g.K, arrays = pack_arrays(kind);
  // neighbouring threads fill neighbouring values; all loads of a value's
  // arrays before their stores
  for (int idx = threadIdx.x; idx < total; idx += kFuseThreads) {
    const int ln = idx / g.K, t = g.K * (ln & ((1 << g.lw) - 1)) + idx % g.K, k = ln >> g.lw;
    const int li = colour + 2 * k;
    const bool on = k < g.nl && t < n;
    const int i = on ? (col ? li : t) : 0, j = on ? (col ? t : li) : 0;
    const uint32_t K = (uint32_t)(j * nx + xslot(i, hx));
    auto get = [&](const void *p) { return ld32(cptr<T>(p), K); };
    T v[9];
    if (kind == PK_RES || kind == PK_PRO) {   // the weights that are 0 or 1 are not stored
      v[0] = get(L.pw[0]);
      v[1] = get(L.pw[1]);
      v[2] = get(L.pw[2]);
      v[3] = get(L.pw[3]);
      v[1] = (t & 1) ? v[1] : T(0);
      v[3] = (t & 1) ? v[3] : T(0);
      if (kind == PK_RES) {
        v[0] = (t & 1) ? v[0] : T(0);
        v[2] = T(0);
        v[3] = get(L.band[BS]);   // the first coupling, as a sweep's v[3]
      }
    } else {
      v[0] = get(L.band[col ? BS : BW]);
      v[1] = get(L.linv[col]);
      v[2] = get(L.lup[col]);
      v[3] = get(L.band[col ? BW : BS]);
      v[4] = get(L.band[col ? BE : BN]);
      if (nine) {
        v[5] = get(L.band[BSW]);
        v[6] = get(L.band[col ? BNW : BSE]);
        v[7] = get(L.band[col ? BSE : BNW]);
        v[8] = get(L.band[BNE]);
      } else {
        v[5] = v[6] = v[7] = v[8] = T(0);
      }
      // nothing couples a line's first step to the one before, or its last to
      // the one after
      v[0] = t > 0 ? -v[0] * v[1] : T(0);
      v[2] = t < n - 1 ? -v[2] : T(0);
    }
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (q < arrays) st32(out, (uint32_t)(q * total + idx), on ? v[q] : T(0));
  }
}

// ---------------------------------------------------------------------------
// Fused coarse cycle
// ---------------------------------------------------------------------------
// LDS values of x (and as many of b): the sum over the levels of the bordered
// arrays, for the largest shapes, or what the lanes past the end of a level's
// columns may reach: up to 4 rows past its array.
constexpr int fused_elems_of(int nx, int ny) {
  int s = 0, most = 0;
  for (;; nx = (nx + 1) / 2, ny = (ny + 1) / 2) {
    const int p = fused_pitch(nx);
    s += p * (ny + 2);
    most = s + 4 * p > most ? s + 4 * p : most;
    if (nx == 1 || ny == 1 || nx * ny <= kDense) return most;
  }
}
constexpr int fused_elems(int cells) {
  int most = 0;
  for (int nx = 1; nx <= kFuseLong; ++nx)
    for (int ny = 1; ny <= kFuseLong && nx * ny <= cells && fused_fits(nx, ny); ++ny) {
      const int s = fused_elems_of(nx, ny);
      most = s > most ? s : most;
    }
  return most;
}
// (colour 0 has the most lines)
constexpr bool fused_lanes_fit() {
  for (int n = 1; n <= kFuseLong; ++n)
    for (int np = 1; np <= kFuseLong && fused_fits(n, np); ++np) {
      const LineLanes g = line_lanes(n, np, 0);
      if (n * np > kDense && (g.lanes > kFuseThreads || g.lw > 6)) return false;
    }
  return true;
}

// Arrays A0 .. A0 + N - 1 of a task's operands: K consecutive values of N packed
// arrays, `stride` values apart.
template <int K, int A0, int N, typename T>
__device__ __forceinline__ void load_pack(const T *p, uint32_t off, uint32_t stride, T (&v)[9][4]) {
  typedef T VT __attribute__((ext_vector_type(K)));
  using GC = const __attribute__((address_space(1))) char;
  using GV = const __attribute__((address_space(1))) VT;
#pragma unroll
  for (int a = 0; a < N; ++a) {
    const VT w = *(GV *)((GC *)p + (off + a * stride) * (uint32_t)sizeof(T));
#pragma unroll
    for (int e = 0; e < K; ++e) v[A0 + a][e] = w[e];
  }
}

// a task by scalar loads
__device__ __forceinline__ CoarseTask load_task(const CoarseTask *p, int it) {
  typedef const __attribute__((address_space(4))) int ConstInt;
  ConstInt *const q = (ConstInt *)(p + it);
  CoarseTask t;
  t.kind = q[0]; t.K = q[1]; t.lw = q[2]; t.n = q[3]; t.nl = q[4]; t.lanes = q[5]; t.x0 = q[6];
  t.sl = q[7]; t.sp = q[8]; t.pack = q[9]; t.aux = q[10]; t.pc = q[11]; t.lev = q[12]; t.pack2 = q[13];
  return t;
}

// What the cycle of an instance reads from its table (pinned: sg_device.hpp).
template <typename T> struct CycleIn {
  const CoarseTask *tasks;
  const T *pack, *bg, *dinv;
  T *xg;
  int lf, last, fx, fy, dx, dy;
};

// sx: x of the levels, bordered (XN values); sb: the dense level's b, then b in the
// places of x; sp: partial products of the dense level. ROWS: the instance has
// lines longer than a row of lanes.
template <typename T, int XN, bool ROWS>
__device__ __forceinline__ void coarse_cycle(CInst &I, const CycleIn<T> &C, T *const sx,
                                             T *const sb, T *const sp) {
  constexpr int NW = kFuseThreads / 64, DC = kDense / NW;
  const CoarseTask *const tasks = C.tasks;
  const T *const pack = C.pack, *const bg = C.bg, *const dinv = C.dinv;
  T *const xg = C.xg;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lf = C.lf, last = C.last, fx = C.fx, fy = C.fy, dx = C.dx, dy = C.dy;
  const int px = fused_pitch(fx), hxf = half_x(fx), dn = dinv ? dx * dy : 0;
  // this wave's columns of the last level's inverse, rows on the lanes
  T dv[DC];
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    const int col = wave * DC + c;
    dv[c] = col < dn && lane < dn ? ld32(dinv, (uint32_t)(col * dn + lane)) : T(0);
  }
  for (int k = tid; k < XN; k += kFuseThreads) { sx[k] = T(0); sb[kDense + k] = T(0); }
  lds_barrier();
  for (int c = tid; c < fx * fy; c += kFuseThreads) {
    const int j = c / fx, i = xcol(c - j * fx, hxf);
    const T v = ld32(bg, (uint32_t)c);
    sb[lf == last ? j * fx + i : kDense + (j + 1) * px + 1 + i] = v;
  }

  // Operands of a task, loaded while the one before runs: K steps of 4 or 9
  // arrays.
  T v[9][4];
  auto fetch = [&](const CoarseTask &t) __attribute__((always_inline)) {
    if ((tid & ~63) >= t.lanes) return;   // no line in this wave
    if (t.K == 4) {
      const uint32_t s = 4 * t.lanes;
      load_pack<4, 0, 4>(pack, t.pack + 4 * tid, s, v);
      if (t.pack2 >= 0) load_pack<4, 4, 5>(pack, t.pack2 + 4 * tid, s, v);
    } else {
      const uint32_t s = t.lanes;
      load_pack<1, 0, 4>(pack, t.pack + tid, s, v);
      if (t.pack2 >= 0) load_pack<1, 4, 5>(pack, t.pack2 + tid, s, v);
    }
  };
  // A task on lines runs in two parts, K steps per lane, between which the
  // operands of the next task are loaded into the registers the first part has
  // used up (one copy of the loads: code run for the first time is slow).
  T r[4], al[4], up[4];
  T *x;   // the lane's first step
  int k;  // its line
  auto first = [&](auto kc, const CoarseTask &t) __attribute__((always_inline)) {
    constexpr int K = decltype(kc)::value;
    const int u = tid & ((1 << t.lw) - 1);
    const int t0 = min(K * u, t.n);   // lanes past the end of the line stay near it
    const int sl = t.sl, sp_ = t.sp;
    k = tid >> t.lw;
    x = sx + t.x0 + 2 * min(k, t.nl - 1) * sp_ + t0 * sl;
    if (t.kind == TK_PRO) {   // odd rows, which alone are read before they are solved
      const T *const c = sx + t.aux + min(k, t.nl - 1) * t.pc + (t0 >> 1);
      T s[3], n[3];
#pragma unroll
      for (int e = 0; e < (K == 1 ? 2 : 3); ++e) { s[e] = c[e]; n[e] = c[t.pc + e]; }
#pragma unroll
      for (int e = 0; e < K; ++e) r[e] = x[e];
#pragma unroll
      for (int e = 0; e < K; ++e)
        r[e] += v[0][e] * s[e / 2] + v[1][e] * s[e / 2 + 1] + v[2][e] * n[e / 2] + v[3][e] * n[e / 2 + 1];
      return;
    }
    if (t.kind != TK_ZERO) {
      T xm[K + 2], xp[K + 2];
#pragma unroll
      for (int e = 0; e < K + 2; ++e) {
        xm[e] = x[(e - 1) * sl - sp_];
        xp[e] = x[(e - 1) * sl + sp_];
      }
#pragma unroll
      for (int e = 0; e < K; ++e) {
        T s = v[3][e] * xm[e + 1] + v[4][e] * xp[e + 1];
        s += v[5][e] * xm[e] + v[6][e] * xm[e + 2];
        s += v[7][e] * xp[e] + v[8][e] * xp[e + 2];
        r[e] = -s;
      }
    } else {
#pragma unroll
      for (int e = 0; e < K; ++e) r[e] = T(0);
    }
    if (t.kind == TK_RES) {
      // The even rows satisfy their equations with the odd rows at zero, so
      // after colour 1 their residual is what the odd rows contribute, r =
      // -(couplings to the odd rows) x; that of the odd rows vanishes. b of
      // the coarse point at an even column: the odd columns beside it send
      // their weighted residuals (a line's last column sends nothing on: its
      // weight is zero, so the lines of a row need no mask).
      if constexpr (K == 1) {
        r[0] = dpp0<kRowShr | 1>(v[1][0] * r[0]) + r[0] + dpp0<kRowShl | 1>(v[0][0] * r[0]);
      } else {
        const T west = dpp0<ROWS ? kWaveShr1 : kRowShr | 1>(v[1][3] * r[3]);
        r[0] = west + r[0] + v[0][1] * r[1];
        r[1] = v[1][1] * r[1] + r[2] + v[0][3] * r[3];
      }
      return;
    }
    // Gauss-Seidel on the lines: d_t = al d_{t-1} + (b_t + r_t) inv_t, then
    // x_t = nup x_{t+1} + d_t
    const T *const b = sb + kDense + (x - sx);
#pragma unroll
    for (int e = 0; e < K; ++e) {
      al[e] = v[0][e];
      up[e] = v[2][e];
      r[e] = (b[e * sl] + r[e]) * v[1][e];
    }
  };
  auto second = [&](auto kc, const CoarseTask &t) __attribute__((always_inline)) {
    constexpr int K = decltype(kc)::value;
    const int u = tid & ((1 << t.lw) - 1);
    const int t0 = min(K * u, t.n);
    const bool line = k < t.nl;
    if (t.kind == TK_RES) {
      T *const c = sb + t.aux + min(k, t.nl - 1) * t.pc + (t0 >> 1);
      if constexpr (K == 1) {
        if (line && u < t.n && !(u & 1)) c[0] = r[0];
      } else {
        if (line && K * u < t.n) c[0] = r[0];
        if (line && K * u + 2 < t.n) c[1] = r[1];
      }
      return;
    }
    if (t.kind != TK_PRO) {
      if constexpr (K == 1) {
        r[0] = scan_row0<true>(al[0], r[0]);
        r[0] = scan_row0<false>(up[0], r[0]);
      } else {
        T A = T(1), B = T(0);
#pragma unroll
        for (int e = 0; e < K; ++e) { B = al[e] * B + r[e]; A = e ? al[e] * A : al[e]; }
        const bool rows = ROWS && t.lw > 4;   // uniform
        T d = rows ? enter_rows0<true>(A, B) : enter_row0<true>(A, B);
#pragma unroll
        for (int e = 0; e < K; ++e) { d = al[e] * d + r[e]; r[e] = d; }
        B = T(0);
#pragma unroll
        for (int e = K - 1; e >= 0; --e) { B = up[e] * B + r[e]; A = e < K - 1 ? up[e] * A : up[e]; }
        T xv = rows ? enter_rows0<false>(A, B) : enter_row0<false>(A, B);
#pragma unroll
        for (int e = K - 1; e >= 0; --e) { xv = up[e] * xv + r[e]; r[e] = xv; }
      }
    }
    const int sl = t.sl;
#pragma unroll
    for (int e = 0; e < K; ++e)
      if (line && K * u + e < t.n) x[e * sl] = r[e];
  };

  CoarseTask t = load_task(tasks, 0);
  fetch(t);
#pragma unroll 1
  for (int it = 1; t.kind != TK_END; ++it) {
    const CoarseTask tn = load_task(tasks, it);
    lds_barrier();   // the task before is done
    const bool on = (tid & ~63) < t.lanes;   // the wave has a line (cell tasks: none)
    if (on) {
      if (t.K == 4) first(std::integral_constant<int, 4>(), t);
      else first(std::integral_constant<int, 1>(), t);
    }
    fetch(tn);
    if (on) {
      if (t.K == 4) second(std::integral_constant<int, 4>(), t);
      else second(std::integral_constant<int, 1>(), t);
    } else if (t.lanes == 0) {
      CLev &L = I.lev[t.lev];
      const int nx = L.nx, ny = L.ny, hx = half_x(nx);
      if (t.kind == TK_DENSE) {
        T s = T(0);
#pragma unroll
        for (int c = 0; c < DC; ++c) s += dv[c] * (wave * DC + c < dn ? sb[wave * DC + c] : T(0));
        sp[wave * kDense + lane] = s;
        lds_barrier();
        if (tid < dn) {
          T o = T(0);
#pragma unroll
          for (int w = 0; w < NW; ++w) o += sp[w * kDense + tid];
          const int j = tid / dx;
          sx[t.x0 + j * t.sp + tid - j * dx] = o;
        }
      } else if (t.kind == TK_RESTB) {   // x = 0: the restriction of b
        const int cx = (nx + 1) >> 1, cy = (ny + 1) >> 1;
        for (int c = tid; c < cx * cy; c += kFuseThreads) {
          const int J = c / cx, Ic = c - J * cx;
          // all loads first; points outside the grid weigh zero and have the
          // border's b
          T w[9];
#pragma unroll
          for (int m = 0; m < 9; ++m) {
            const int da = m % 3 - 1, db = m / 3 - 1, fi = 2 * Ic + da, fj = 2 * J + db;
            const bool in = fi >= 0 && fi < nx && fj >= 0 && fj < ny;
            const int slot = (da < 0 ? 1 : 0) + 2 * (db < 0 ? 1 : 0);
            const uint32_t K = in ? fj * nx + xslot(fi, hx) : 0;
            w[m] = m == 4 ? T(1) : ld32(cptr<T>(L.pw[slot]), K);
            w[m] = in ? w[m] : T(0);
          }
          T s = T(0);
          const T *const bf = sb + t.x0 + 2 * J * t.sp + 2 * Ic;
#pragma unroll
          for (int m = 0; m < 9; ++m) s += w[m] * bf[(m / 3 - 1) * t.sp + m % 3 - 1];
          sb[t.aux + J * t.pc + Ic] = s;
        }
      } else {   // TK_PROALL: x += P xc at every cell
        for (int c = tid; c < nx * ny; c += kFuseThreads) {
          const int j = c / nx, i = c - j * nx;
          const uint32_t K = j * nx + xslot(i, hx);
          const bool io = i & 1, jo = j & 1;
          const T *const xc = sx + t.aux + (j >> 1) * t.pc + (i >> 1);
          T e = xc[0];
          if (io || jo) e *= ld32(cptr<T>(L.pw[0]), K);
          if (io) e += ld32(cptr<T>(L.pw[1]), K) * xc[1];
          if (jo) e += ld32(cptr<T>(L.pw[2]), K) * xc[t.pc];
          if (io && jo) e += ld32(cptr<T>(L.pw[3]), K) * xc[t.pc + 1];
          sx[t.x0 + j * t.sp + i] += e;
        }
      }
    }
    t = tn;
  }
  lds_barrier();
  // x of the first level
  for (int c = tid; c < fx * fy; c += kFuseThreads) {
    const int j = c / fx, i = xcol(c - j * fx, hxf);
    st32(xg, (uint32_t)c, sx[(j + 1) * px + 1 + i]);
  }
}

// Instances with long lines run code of their own: with one copy for both the
// short lines' code is larger, and cold code is time (10 steps of 41 x 33 FP64 4.83
// ms with one copy, 4.70 with two).
template <typename T, int CAP>
__global__ void __launch_bounds__(kFuseThreads) k_coarse_cycle(const Insts insts,
                                                               const FuseMap *__restrict__ map,
                                                               int xid, int bid) {
  static_assert(fused_lanes_fit(), "every line of a colour has its lanes");
  constexpr int XN = fused_elems(CAP);
  __shared__ T sx[XN];
  __shared__ T sb[kDense + XN];
  __shared__ T sp[kFuseThreads / 64 * kDense];
  const FuseMap fm = map[blockIdx.x];
  CInst &I = insts[fm.inst];
  CycleIn<T> C;
  C.tasks = I.tasks;
  C.pack = cptr<T>(I.pack);
  C.lf = fm.lev;
  C.last = fm.last;
  level_xb<T>(I, C.lf, xid, bid, C.xg, C.bg);
  C.fx = I.lev[C.lf].nx; C.fy = I.lev[C.lf].ny;
  C.dx = I.lev[C.last].nx; C.dy = I.lev[C.last].ny;
  C.dinv = cptr<T>(I.lev[C.last].dinv);
  int st = status_of(insts, fm.inst);
  pin(C.tasks, C.pack, C.xg, C.bg, C.fx, C.fy, C.dx, C.dy, C.dinv, st);
  if (st != ST_ACTIVE) return;
  if (__builtin_expect(fm.rows == 0, 1)) coarse_cycle<T, XN, false>(I, C, sx, sb, sp);
  else coarse_cycle<T, XN, true>(I, C, sx, sb, sp);
}

void launch_dense_inverse(hipStream_t s, const Insts &d, const FuseMap *m, int n, bool h32) {
  if (!n) return;
  if (h32) k_dense_inverse<float><<<n, 1024, 0, s>>>(d, m);
  else k_dense_inverse<double><<<n, 1024, 0, s>>>(d, m);
}
void launch_coarse_pack(hipStream_t s, const Insts &d, const PackMap *m, int n, bool h32) {
  if (!n) return;
  if (h32) k_coarse_pack<float><<<n, kFuseThreads, 0, s>>>(d, m);
  else k_coarse_pack<double><<<n, kFuseThreads, 0, s>>>(d, m);
}

template <typename T>
void launch_coarse_cycle(hipStream_t s, const Insts &d, const FuseMap *m, int n, int xid, int bid,
                         int cap) {
  if (!n) return;
  if (cap <= 1024) k_coarse_cycle<T, 1024><<<n, kFuseThreads, 0, s>>>(d, m, xid, bid);
  else k_coarse_cycle<T, kFuseCells><<<n, kFuseThreads, 0, s>>>(d, m, xid, bid);
}
template void launch_coarse_cycle<double>(hipStream_t, const Insts &, const FuseMap *, int, int,
                                          int, int);
template void launch_coarse_cycle<float>(hipStream_t, const Insts &, const FuseMap *, int, int,
                                         int, int);

}  // namespace sg
