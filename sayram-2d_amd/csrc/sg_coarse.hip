// sg_coarse.hip -- the fused coarse cycle.
//
// The levels of one instance from `lev` (its first level that fits, see
// fused_fits) down to its coarsest and back, in one workgroup with LDS
// barriers between the phases, instead of several launches per level. The
// cycle is the per-level one: per level on the way down an optional
// pre-smoothing sweep of x-lines and the restriction of the residual (of b
// itself without pre-smoothing), the exact line solve of the coarsest level,
// then per level the prolongation of the lines the first post-sweep reads and
// the zebra post-sweeps.
//
// Bound: latency. One workgroup walks some 8 phases per level, each a few LDS
// accesses and a barrier, so the time is the sum of the phases' latencies,
// not bytes. Hence:
//  * x of every level (with a border of zeros, so that no neighbour needs a
//    test) and b of every level but the first stay in LDS for the whole cycle;
//  * a thread owns one cell per sweep colour (R rounds of 1024), with the lanes
//    of a wave along the line, and solves the line with wave scans of its
//    affine maps (sg_scan.hpp): one phase per colour. One thread per line
//    running the recurrences out of LDS took two phases and a chain of 2 n
//    dependent steps;
//  * the operator and factors of a cell are read straight into the owner's
//    registers, a whole level's in one round trip.
// Measured against one thread per line: 69.0 -> 30.5 us per cycle on a 90 x 100
// grid (FP64, first level 23 x 25), 76.0 -> 32.0 us at 1021 x 765 (FP32, 32 x
// 24), 104 -> 42 us for the 192 cycles of an FP64 batch in one launch.
#include "sg_device.hpp"
#include "sg_kernels.hpp"
#include "sg_scan.hpp"

namespace sg {

// LDS values of a fused cycle of R rounds: the sums over the levels of the
// bordered x (odd pitch: the stride of a column sweep then spreads over the
// banks) and of b below the first level, for the largest first level
// (fused_side_max x fused_side_max, at most 1024 R^2 cells).
__host__ __device__ constexpr int fused_pitch(int nx) { return (nx + 2) | 1; }
constexpr int fused_x_elems(int nx, int ny) {
  int s = 0;
  for (;;) {
    s += fused_pitch(nx) * (ny + 2);
    if (nx == 1 || ny == 1) return s;
    nx = (nx + 1) / 2; ny = (ny + 1) / 2;
  }
}
constexpr int fused_b_elems(int nx, int ny) {
  int s = 0;
  while (nx > 1 && ny > 1) {
    nx = (nx + 1) / 2; ny = (ny + 1) / 2;
    s += nx * ny;
  }
  return s;
}
constexpr int fused_rounds(int nx, int ny) {
  int most = 1;
  for (int d = 0; d < 2; ++d) {
    const int n = d ? ny : nx, lines = ((d ? nx : ny) + 1) / 2;
    int w = 1;
    while (w < n) w *= 2;
    const int r = (lines * w + kFuseThreads - 1) / kFuseThreads;
    most = r > most ? r : most;
  }
  return most;
}
struct FusedSize { int x, b, rounds; };
constexpr FusedSize fused_size(int cells) {
  FusedSize m{0, 0, 0};
  for (int nx = 1; nx <= kFuseSide; ++nx)
    for (int ny = 1; ny <= kFuseSide; ++ny) {
      if (nx * ny > cells) continue;
      const int x = fused_x_elems(nx, ny), b = fused_b_elems(nx, ny), r = fused_rounds(nx, ny);
      m.x = x > m.x ? x : m.x;
      m.b = b > m.b ? b : m.b;
      m.rounds = r > m.rounds ? r : m.rounds;
    }
  return m;
}

// One cell's row of its line's equations: the factors and the couplings to
// the lines beside (minus / plus side, at steps t - 1, t, t + 1); zero where
// there is no cell.
template <typename T> struct CellEq { T lo, inv, up, m0, p0, mm, mp, pm, pp; };

template <typename T, int DIR>
__device__ __forceinline__ CellEq<T> cell_eq(const Lev &L, bool nine, uint32_t K, bool on) {
  CellEq<T> q{};
  if (on) {
    q.lo = ld32(cptr<T>(L.band[DIR == 0 ? BW : BS]), K);
    q.inv = ld32(cptr<T>(L.linv[DIR]), K);
    q.up = ld32(cptr<T>(L.lup[DIR]), K);
    q.m0 = ld32(cptr<T>(L.band[DIR == 0 ? BS : BW]), K);
    q.p0 = ld32(cptr<T>(L.band[DIR == 0 ? BN : BE]), K);
    if (nine) {
      q.mm = ld32(cptr<T>(L.band[BSW]), K);
      q.mp = ld32(cptr<T>(L.band[DIR == 0 ? BSE : BNW]), K);
      q.pm = ld32(cptr<T>(L.band[DIR == 0 ? BNW : BSE]), K);
      q.pp = ld32(cptr<T>(L.band[BNE]), K);
    }
  }
  return q;
}

// The couplings of a cell to the lines beside it, applied to x in LDS (ix: its
// place, sl / sp: strides along and across the line).
template <typename T>
__device__ __forceinline__ T beside(const CellEq<T> &q, const T *x, int ix, int sl, int sp) {
  T s = q.m0 * x[ix - sp] + q.p0 * x[ix + sp];
  s += q.mm * x[ix - sp - sl] + q.mp * x[ix - sp + sl];
  s += q.pm * x[ix + sp - sl] + q.pp * x[ix + sp + sl];
  return s;
}

// Solution at step u of the line of this lane's segment with right-hand side
// r (zero at steps past the line's end, whose factors are zero too).
template <typename T>
__device__ __forceinline__ T solve_line(const CellEq<T> &q, T r, int u, int W) {
  T a = -q.lo * q.inv, d = r * q.inv;
  T A = a, B = d;
  scan_rows<true>(A, B, u, W);
  if (W > 16) {
    const RowMaps<T> m = row_maps<true>(A, B);
    B = a * enter<true>(A, B, m, u, W, T(0)) + d;
  }
  d = B;   // the eliminated right-hand side
  a = -q.up;
  A = a; B = d;
  scan_rows<false>(A, B, u, W);
  if (W > 16) {
    const RowMaps<T> m = row_maps<false>(A, B);
    B = a * enter<false>(A, B, m, u, W, T(0)) + d;
  }
  return B;
}

// smoother: the finest level's schedule in bits 0-3, the coarser levels' in
// bits 4-7 (post-smoothing bits and the x-line pre-smoothing bit)
template <typename T, int R>
__global__ void __launch_bounds__(kFuseThreads) k_coarse_cycle(const InstDev *__restrict__ insts,
                                                               const FuseMap *__restrict__ map,
                                                               int xid, int bid, int smoother) {
  constexpr FusedSize SZ = fused_size(R == 1 ? 1024 : kFuseCells32);
  static_assert(SZ.rounds <= R, "a thread owns R cells of a colour at most");
  __shared__ T sx[SZ.x];
  __shared__ T sb[SZ.b + 1];
  const FuseMap fm = map[blockIdx.x];
  const InstDev &I = insts[fm.inst];
  if (rsc(I)->status != ST_ACTIVE) return;
  const int tid = threadIdx.x;
  const int lf = fm.lev, last = I.nlev - 1;
  auto sched = [&](int m) { return m == 0 ? (smoother & 15) : (smoother >> 4); };
  T *xg; const T *bg;
  level_xb<T>(I, lf, xid, bid, xg, bg);
  int nx = I.lev[lf].nx, ny = I.lev[lf].ny;
  {
    int tot = 0, cx = nx, cy = ny;
    for (int m = lf;; ++m) {
      tot += fused_pitch(cx) * (cy + 2);
      if (m == last) break;
      cx = (cx + 1) >> 1; cy = (cy + 1) >> 1;
    }
    for (int k = tid; k < tot; k += kFuseThreads) sx[k] = T(0);
  }
  lds_barrier();
  int xo = 0, bo = 0;   // LDS offsets of the level's x and b (b of level lf is in global memory)

  // cell (i, j) of step u on line li
  auto place = [&](int dir, int li, int u, int &i, int &j) { i = dir ? li : u; j = dir ? u : li; };

  // One level's down-sweeps and restriction, up-sweeps; RR: rounds it needs.
  auto sweep = [&](auto dirc, auto rc, const Lev &L, bool nine, const CellEq<T> *q, int colour,
                   const T *b, bool zero) {
    constexpr int DIR = decltype(dirc)::value, RR = decltype(rc)::value;
    const int n = DIR == 0 ? nx : ny, np = DIR == 0 ? ny : nx;
    const int W = seg_width(n), lw = 31 - __builtin_clz(W), nl = (np - colour + 1) >> 1;
    const int px = fused_pitch(nx);
    T *const x = sx + xo + px + 1;
#pragma unroll
    for (int r = 0; r < RR; ++r) {
      const int idx = tid + r * kFuseThreads, u = idx & (W - 1), k = idx >> lw;
      if (((idx & ~63) >> lw) >= nl) continue;   // uniform over the wave
      const bool on = k < nl && u < n;
      int i, j;
      place(DIR, colour + 2 * k, u, i, j);
      const int ix = on ? j * px + i : 0;
      T rhs = b[r];
      if (!zero) rhs -= beside(q[r], x, ix, DIR == 0 ? 1 : px, DIR == 0 ? px : 1);
      const T v = solve_line(q[r], on ? rhs : T(0), u, W);
      if (on) x[ix] = v;
    }
    lds_barrier();
  };
  // equations and right-hand sides of one colour's cells
  auto load = [&](auto dirc, auto rc, const Lev &L, bool nine, bool first, CellEq<T> *q, T *b,
                  int colour) {
    constexpr int DIR = decltype(dirc)::value, RR = decltype(rc)::value;
    const int n = DIR == 0 ? nx : ny, np = DIR == 0 ? ny : nx, hx = half_x(nx);
    const int W = seg_width(n), lw = 31 - __builtin_clz(W), nl = (np - colour + 1) >> 1;
#pragma unroll
    for (int r = 0; r < RR; ++r) {
      const int idx = tid + r * kFuseThreads, u = idx & (W - 1), k = idx >> lw;
      const bool on = k < nl && u < n;
      int i, j;
      place(DIR, colour + 2 * k, u, i, j);
      const uint32_t K = on ? j * nx + xslot(i, hx) : 0;
      q[r] = cell_eq<T, DIR>(L, nine, K, on);
      b[r] = !on ? T(0) : first ? ld32(bg, K) : sb[bo + j * nx + i];
    }
  };
  std::integral_constant<int, 0> X;
  std::integral_constant<int, 1> Y;

  auto down = [&](auto rc, int m, bool first) {
    constexpr int RR = decltype(rc)::value;
    const Lev &L = I.lev[m];
    const bool nine = m > 0;
    const int hx = half_x(nx), px = fused_pitch(nx);
    const int cx = (nx + 1) >> 1, cy = (ny + 1) >> 1;
    T *const bc = sb + (first ? 0 : bo + nx * ny);
    if (sched(m) & 1) {
      // pre-smoothing with x-lines from x = 0: colour 0 from b alone; the
      // even rows then satisfy their equations with the odd rows at zero, so
      // after colour 1 their residual is what the odd rows contribute,
      // r = -(couplings to the odd rows) x, and that of the odd rows vanishes
      CellEq<T> q0[RR], q1[RR];
      T b0[RR], b1[RR], w0[RR], w1[RR];
      load(X, rc, L, nine, first, q0, b0, 0);
      load(X, rc, L, nine, first, q1, b1, 1);
      const int W = seg_width(nx), lw = 31 - __builtin_clz(W), nl = (ny + 1) >> 1;
#pragma unroll
      for (int r = 0; r < RR; ++r) {   // weights of the odd columns of the even rows
        const int idx = tid + r * kFuseThreads, u = idx & (W - 1), k = idx >> lw;
        const bool odd = k < nl && u < nx && (u & 1);
        const uint32_t K = 2 * k * nx + xslot(u, hx);
        w0[r] = odd ? ld32(cptr<T>(L.pw[0]), K) : T(0);
        w1[r] = odd ? ld32(cptr<T>(L.pw[1]), K) : T(0);
      }
      sweep(X, rc, L, nine, q0, 0, b0, true);
      sweep(X, rc, L, nine, q1, 1, b1, false);
      const T *const x = sx + xo + px + 1;
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        const int idx = tid + r * kFuseThreads, u = idx & (W - 1), k = idx >> lw;
        if (((idx & ~63) >> lw) >= nl) continue;
        const bool on = k < nl && u < nx;
        const T res = on ? -beside(q0[r], x, 2 * k * px + u, 1, px) : T(0);
        // b of the coarse point at column u (even): the odd columns beside it
        // send their weighted residuals
        const T east = __shfl_down(w0[r] * res, 1, W), west = __shfl_up(w1[r] * res, 1, W);
        if (on && !(u & 1)) {
          T s = u > 0 ? west : T(0);
          s += res;
          s += u + 1 < nx ? east : T(0);
          bc[k * cx + (u >> 1)] = s;
        }
      }
    } else {   // x = 0: b of the next level is the restriction of b
      for (int c = tid; c < cx * cy; c += kFuseThreads) {
        const int J = c / cx, Ic = c - J * cx;
        T s = T(0);
#pragma unroll
        for (int db = -1; db <= 1; ++db)
#pragma unroll
          for (int da = -1; da <= 1; ++da) {
            const int fi = 2 * Ic + da, fj = 2 * J + db;
            if (fi < 0 || fi >= nx || fj < 0 || fj >= ny) continue;
            const uint32_t K = fj * nx + xslot(fi, hx);
            const int slot = (da < 0 ? 1 : 0) + 2 * (db < 0 ? 1 : 0);
            const T w = da == 0 && db == 0 ? T(1) : ld32(cptr<T>(L.pw[slot]), K);
            s += w * (first ? ld32(bg, K) : sb[bo + fj * nx + fi]);
          }
        bc[c] = s;
      }
    }
    lds_barrier();
  };

  auto up = [&](auto rc, int m, bool first, int xc_off, int cx) {
    constexpr int RR = decltype(rc)::value;
    const Lev &L = I.lev[m];
    const bool nine = m > 0;
    const int hx = half_x(nx), px = fused_pitch(nx), pc = fused_pitch(cx);
    const int sml = sched(m);
    const bool post_x = sml & 4, post_y = sml & 8;
    T *const x = sx + xo + px + 1;
    const T *const xc = sx + xc_off + pc + 1;
    CellEq<T> q0[RR], q1[RR];
    T b0[RR], b1[RR];
    // x += P xc at cell (i, j); the weights that are 0 or 1 are not stored
    auto correct = [&](int i, int j) {
      const uint32_t K = j * nx + xslot(i, hx);
      const bool io = i & 1, jo = j & 1;
      const T *const c = xc + (j >> 1) * pc + (i >> 1);
      T w0 = T(1), w1 = T(0), w2 = T(0), w3 = T(0);
      if (io || jo) w0 = ld32(cptr<T>(L.pw[0]), K);
      if (io) w1 = ld32(cptr<T>(L.pw[1]), K);
      if (jo) w2 = ld32(cptr<T>(L.pw[2]), K);
      if (io && jo) w3 = ld32(cptr<T>(L.pw[3]), K);
      T e = w0 * c[0];
      e += w1 * c[1];
      e += w2 * c[pc];
      e += w3 * c[pc + 1];
      x[j * px + i] += e;
    };
    if (post_x) {
      load(X, rc, L, nine, first, q0, b0, 0);
      load(X, rc, L, nine, first, q1, b1, 1);
      // only the odd rows are read before they are solved
      for (int c = tid; c < nx * (ny >> 1); c += kFuseThreads) {
        const int k = c / nx;
        correct(c - k * nx, 2 * k + 1);
      }
      lds_barrier();
      sweep(X, rc, L, nine, q0, 0, b0, false);
      sweep(X, rc, L, nine, q1, 1, b1, false);
    } else {
      for (int c = tid; c < nx * ny; c += kFuseThreads) {
        const int j = c / nx;
        correct(c - j * nx, j);
      }
      lds_barrier();
    }
    if (post_y) {
      load(Y, rc, L, nine, first, q0, b0, 0);
      load(Y, rc, L, nine, first, q1, b1, 1);
      sweep(Y, rc, L, nine, q0, 0, b0, false);
      sweep(Y, rc, L, nine, q1, 1, b1, false);
    }
  };

  std::integral_constant<int, R> RF;
  std::integral_constant<int, 1> R1;
  for (int m = lf; m < last; ++m) {
    if (m == lf) down(RF, m, true); else down(R1, m, false);
    xo += fused_pitch(nx) * (ny + 2);
    if (m > lf) bo += nx * ny;
    nx = (nx + 1) >> 1; ny = (ny + 1) >> 1;
  }
  {   // exact solve of the coarsest level: one row or one column
    const Lev &L = I.lev[last];
    CellEq<T> q[1];
    T b[1];
    if (ny == 1) { load(X, R1, L, last > 0, last == lf, q, b, 0); sweep(X, R1, L, last > 0, q, 0, b, true); }
    else { load(Y, R1, L, last > 0, last == lf, q, b, 0); sweep(Y, R1, L, last > 0, q, 0, b, true); }
  }
  for (int m = last - 1; m >= lf; --m) {
    const int cx = nx, xc = xo;
    nx = I.lev[m].nx; ny = I.lev[m].ny;
    xo -= fused_pitch(nx) * (ny + 2);
    if (m > lf) bo -= nx * ny;
    if (m == lf) up(RF, m, true, xc, cx); else up(R1, m, false, xc, cx);
  }
  // x of the first level
  const int hx = half_x(nx), px = fused_pitch(nx);
  for (int c = tid; c < nx * ny; c += kFuseThreads) {
    const int j = c / nx, p = c - j * nx;
    st32(xg, (uint32_t)c, sx[(j + 1) * px + 1 + xcol(p, hx)]);
  }
}

template <typename T>
void launch_coarse_cycle(hipStream_t s, const InstDev *d, const FuseMap *m, int n, int xid, int bid,
                         int smoother, int cap) {
  if (!n) return;
  if (cap <= 1024) k_coarse_cycle<T, 1><<<n, kFuseThreads, 0, s>>>(d, m, xid, bid, smoother);
  else k_coarse_cycle<T, 2><<<n, kFuseThreads, 0, s>>>(d, m, xid, bid, smoother);
}
template void launch_coarse_cycle<double>(hipStream_t, const InstDev *, const FuseMap *, int, int,
                                          int, int, int);
template void launch_coarse_cycle<float>(hipStream_t, const InstDev *, const FuseMap *, int, int,
                                         int, int, int);

}  // namespace sg
