// sg_sweeps.hip -- zebra line sweeps with the lines held in registers.
//
// A sweep solves every line of one colour exactly with the precomputed
// factors, the off-line couplings moved to the right-hand side. Both Thomas
// recurrences are first-order affine maps (d_t = a_t d_{t-1} + b_t forward,
// x_t = d_t - u_t x_{t+1} backward): a thread takes a run of consecutive
// steps of one line into registers, composes their maps, the threads of the
// line combine the compositions (wave shuffles, then one LDS exchange
// between the waves), and each thread reruns its steps from the value that
// enters them. A line is solved in one pass over its data, with one barrier
// per recurrence, however long it is.
#include "sg_device.hpp"
#include "sg_kernels.hpp"
#include "sg_scan.hpp"

namespace sg {

// What a sweep of level l reads: its size, x, b, the line factors and the
// couplings along and across the lines (DIR 0: rows, 1: columns), read from the
// instance table together with the status (pinned: sg_device.hpp).
template <typename T, int NB, bool ZERO, int DIR> struct Lines {
  T *x;
  const T *b, *lo, *inv, *cu, *om, *op, *omm, *omp, *opm, *opp;
  int nx, ny, st;
  __device__ __forceinline__ Lines(const Insts &insts, int inst, int l, int xid, int bid) {
    CInst &I = insts[inst];
    CLev &L = I.lev[l];
    level_xb<T>(I, l, xid, bid, x, b);
    lo = cptr<T>(L.band[DIR == 0 ? BW : BS]);
    inv = cptr<T>(L.linv[DIR]);
    cu = cptr<T>(L.lup[DIR]);
    nx = L.nx; ny = L.ny;
    om = op = omm = omp = opm = opp = nullptr;
    if (!ZERO) {
      om = cptr<T>(L.band[DIR == 0 ? BS : BW]);
      op = cptr<T>(L.band[DIR == 0 ? BN : BE]);
      if (NB == 9) {
        omm = cptr<T>(L.band[BSW]); omp = cptr<T>(L.band[DIR == 0 ? BSE : BNW]);
        opm = cptr<T>(L.band[DIR == 0 ? BNW : BSE]); opp = cptr<T>(L.band[BNE]);
      }
    }
    st = status_of(insts, inst);
    pin(x, b, lo, inv, cu, nx, ny, st);
    if constexpr (!ZERO) pin(om, op);
    if constexpr (!ZERO && NB == 9) pin(omm, omp, opm, opp);
  }
};

// LDS values of a column sweep of L columns in C runs: the composed maps of
// every wave and column, forward and backward.
template <int L, int C> constexpr int col_lds() { return 4 * (L * C / 64) * L; }

// Columns. L columns of one colour (neighbouring lanes, so a step's loads are
// L contiguous values) times C runs of at most K steps; consecutive runs
// follow one another in a wave, then across the waves. The values of a thread's
// steps are loaded in one go, so a sweep costs about one memory round trip
// and the chip's bandwidth, where the tiled sweep (k_line) walked a line in
// serial tiles of a load, two scans and three barriers each. Measured, tiled
// against this, per launch of one colour: 765-step columns of a 1021 x 765
// grid (FP32) 56 -> 13.4 us, its coarser columns 18.8 -> 7.2; 4096 steps
// 131 -> 94 us; 2048 steps FP64 106 -> 41 us; the 9-point columns of a batch of
// 48 uneven grids 14.4 -> 6.8 us, its 5-point ones 34.5 -> 16.5.
// Run lengths: K steps of three values each are held in registers; 4096 steps
// as 8 columns x 64 runs of 64 took 94 us, as 4 columns x 128 runs of 32 (16
// byte pieces of a row) 158. A kernel holds every run length of its range in one
// body and so has the registers of the longest for all of them (9-point, not from
// zero): k_cols 127 VGPRs in FP32 (4 waves per SIMD) and 234 in FP64 (2, one
// workgroup per CU), where runs of 8 steps alone need 66 and 98; k_cols_long 256
// with 25 (FP32) and 32 (FP64) of them spilled to scratch, where no run length
// alone spills.
template <typename T, int NB, bool ZERO, int L, int C, int K>
__device__ __forceinline__ void col_sweep(const Lines<T, NB, ZERO, 1> &P, const LineGrp gr, T *lds) {
  constexpr int NW = L * C / 64;   // waves
  static_assert(L <= 64 && 64 % L == 0 && (L * C) % 64 == 0, "whole runs per wave");
  T *const s_a = lds, *const s_b = s_a + NW * L, *const r_a = s_b + NW * L, *const r_b = r_a + NW * L;
  const int nx = P.nx, n = P.ny, hx = half_x(nx);
  T *const x = P.x;
  const T *const b = P.b, *const lo = P.lo, *const inv = P.inv, *const cu = P.cu;
  const T *const om = P.om, *const op = P.op;
  const T *const omm = P.omm, *const omp = P.omp, *const opm = P.opm, *const opp = P.opp;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k = tid % L, c = tid / L;
  const int kc = (n + C - 1) / C;                  // steps per run (uniform, <= K)
  const int t0 = c * kc, cnt = min(kc, n - t0);    // this run's steps (cnt < 1: none)
  const bool on = k < gr.count;                    // lanes past the group repeat its last column
  const int li = gr.first + min(k, gr.count - 1) * gr.step;
  // Slots of the column and of its neighbours in a row. Couplings to columns
  // outside the grid are zero; such a neighbour is replaced by the one on the
  // other side, which holds a value of the other colour (this colour's own x
  // may never have been written, and 0 times a NaN is not 0).
  const int lm = li > 0 ? li - 1 : min(1, nx - 1), lp = li < nx - 1 ? li + 1 : max(nx - 2, 0);
  const uint32_t s0 = xslot(li, hx), sm = xslot(lm, hx), sp = xslot(lp, hx);
  auto row = [&](int t) -> uint32_t { return (uint32_t)(max(0, min(t, n - 1)) * nx); };
  // d_t = al d_{t-1} + be of every step; steps past the run are the identity
  T al[K], be[K], up[K];
  T xm0 = T(0), xm1 = T(0), xp0 = T(0), xp1 = T(0);   // x beside at steps t - 1 and t
  if (!ZERO && NB == 9) {
    xm0 = ld32(x, row(t0 - 1) + sm); xp0 = ld32(x, row(t0 - 1) + sp);
    xm1 = ld32(x, row(t0) + sm); xp1 = ld32(x, row(t0) + sp);
  }
#pragma unroll
  for (int e = 0; e < K; ++e) {
    const bool ok = e < cnt;
    const uint32_t q = row(t0 + e);
    T r = ld32(b, q + s0);
    const T v = ld32(inv, q + s0), w = ld32(lo, q + s0);
    up[e] = ld32(cu, q + s0);
    if (!ZERO) {
      if (NB == 9) {
        const uint32_t qn = row(t0 + e + 1);
        const T xm2 = ld32(x, qn + sm), xp2 = ld32(x, qn + sp);
        r = r - ld32(om, q + s0) * xm1 - ld32(op, q + s0) * xp1;
        r = r - ld32(omm, q + s0) * xm0 - ld32(omp, q + s0) * xm2;
        r = r - ld32(opm, q + s0) * xp0 - ld32(opp, q + s0) * xp2;
        xm0 = xm1; xm1 = xm2; xp0 = xp1; xp1 = xp2;
      } else {
        r = r - ld32(om, q + s0) * ld32(x, q + sm) - ld32(op, q + s0) * ld32(x, q + sp);
      }
    }
    al[e] = ok ? -w * v : T(1);
    be[e] = ok ? r * v : T(0);
  }
  T A = T(1), B = T(0);
#pragma unroll
  for (int e = 0; e < K; ++e) { B = al[e] * B + be[e]; A = al[e] * A; }
#pragma unroll
  for (int off = L; off < 64; off <<= 1) {
    const T Ap = __shfl_up(A, off, 64), Bp = __shfl_up(B, off, 64);
    if (lane >= off) { B = A * Bp + B; A = A * Ap; }
  }
  T Ae = T(1), Be = T(0);
  if (L < 64) {
    Ae = __shfl_up(A, L, 64); Be = __shfl_up(B, L, 64);
    if (lane < L) { Ae = T(1); Be = T(0); }
  }
  if (lane >= 64 - L) { s_a[wave * L + k] = A; s_b[wave * L + k] = B; }
  lds_barrier();
  T d = T(0);
#pragma unroll
  for (int w = 0; w < NW - 1; ++w) {
    const T a = s_a[w * L + k], bb = s_b[w * L + k];
    d = w < wave ? a * d + bb : d;
  }
  d = Ae * d + Be;
#pragma unroll
  for (int e = 0; e < K; ++e) {
    const bool ok = e < cnt;
    d = al[e] * d + be[e];
    be[e] = ok ? d : T(0);
    al[e] = ok ? -up[e] : T(1);
  }
  // backward: x_t = al x_{t+1} + be
  A = T(1); B = T(0);
#pragma unroll
  for (int e = K - 1; e >= 0; --e) { B = al[e] * B + be[e]; A = al[e] * A; }
#pragma unroll
  for (int off = L; off < 64; off <<= 1) {
    const T An = __shfl_down(A, off, 64), Bn = __shfl_down(B, off, 64);
    if (lane + off < 64) { B = A * Bn + B; A = A * An; }
  }
  Ae = T(1); Be = T(0);
  if (L < 64) {
    Ae = __shfl_down(A, L, 64); Be = __shfl_down(B, L, 64);
    if (lane >= 64 - L) { Ae = T(1); Be = T(0); }
  }
  if (lane < L) { r_a[wave * L + k] = A; r_b[wave * L + k] = B; }
  lds_barrier();
  T xv = T(0);
#pragma unroll
  for (int w = NW - 1; w > 0; --w) {
    const T a = r_a[w * L + k], bb = r_b[w * L + k];
    xv = w > wave ? a * xv + bb : xv;
  }
  xv = Ae * xv + Be;
#pragma unroll
  for (int e = K - 1; e >= 0; --e) {
    xv = al[e] * xv + be[e];
    if (on && e < cnt) st32(x, row(t0 + e) + s0, xv);
  }
}

template <typename T, int NB, bool ZERO>
__global__ void __launch_bounds__(kColThreads) k_cols(const Insts insts,
                                                      const LineGrp *__restrict__ map, int l,
                                                      int xid, int bid) {
  __shared__ T lds[col_lds<32, 16>()];
  const LineGrp gr = map[blockIdx.x];
  const Lines<T, NB, ZERO, 1> P(insts, gr.inst, l, xid, bid);
  if (P.st != ST_ACTIVE) return;
  const int n = P.ny;
  if (n <= 64) col_sweep<T, NB, ZERO, 32, 16, 4>(P, gr, lds);
  else if (n <= 128) col_sweep<T, NB, ZERO, 16, 32, 4>(P, gr, lds);
  else if (n <= 256) col_sweep<T, NB, ZERO, 16, 32, 8>(P, gr, lds);
  else if (n <= 384) col_sweep<T, NB, ZERO, 16, 32, 12>(P, gr, lds);
  else col_sweep<T, NB, ZERO, 16, 32, 16>(P, gr, lds);
}

template <typename T, int NB, bool ZERO>
__global__ void __launch_bounds__(kColThreads) k_cols_long(const Insts insts,
                                                           const LineGrp *__restrict__ map, int l,
                                                           int xid, int bid) {
  __shared__ T lds[col_lds<16, 32>()];
  const LineGrp gr = map[blockIdx.x];
  const Lines<T, NB, ZERO, 1> P(insts, gr.inst, l, xid, bid);
  if (P.st != ST_ACTIVE) return;
  const int n = P.ny;
  if constexpr (sizeof(T) == 4) {
    if (n <= 768) col_sweep<T, NB, ZERO, 16, 32, 24>(P, gr, lds);
    else if (n <= 1024) col_sweep<T, NB, ZERO, 8, 64, 16>(P, gr, lds);
    else if (n <= 2048) col_sweep<T, NB, ZERO, 8, 64, 32>(P, gr, lds);
    else col_sweep<T, NB, ZERO, 8, 64, 64>(P, gr, lds);
  } else {
    if (n <= 1024) col_sweep<T, NB, ZERO, 8, 64, 16>(P, gr, lds);
    else if (n <= 2048) col_sweep<T, NB, ZERO, 4, 128, 16>(P, gr, lds);
    else col_sweep<T, NB, ZERO, 4, 128, 32>(P, gr, lds);
  }
}

template <typename T>
void launch_cols(hipStream_t s, const Insts &d, const LineGrp *m, int ngroups, int l, bool is_long,
                 bool zero, int xid, int bid) {
  if (!ngroups) return;
#define SG_COLS(NB, Z)                                                                    \
  do {                                                                                    \
    if (is_long) k_cols_long<T, NB, Z><<<ngroups, kColThreads, 0, s>>>(d, m, l, xid, bid); \
    else k_cols<T, NB, Z><<<ngroups, kColThreads, 0, s>>>(d, m, l, xid, bid);              \
  } while (0)
  if (l > 0) { if (zero) SG_COLS(9, true); else SG_COLS(9, false); }
  else { if (zero) SG_COLS(5, true); else SG_COLS(5, false); }
#undef SG_COLS
}
template void launch_cols<double>(hipStream_t, const Insts &, const LineGrp *, int, int, bool,
                                  bool, int, int);
template void launch_cols<float>(hipStream_t, const Insts &, const LineGrp *, int, int, bool,
                                 bool, int, int);

// H consecutive values from slot on, in one load (global loads take any
// alignment of the element; a row's halves start at any slot).
template <typename T, int H>
__device__ __forceinline__ void ldv(const T *base, uint32_t slot, T (&v)[H]) {
  typedef T VT __attribute__((ext_vector_type(H), aligned(sizeof(T))));
  using GC = const __attribute__((address_space(1))) char;
  using GV = const __attribute__((address_space(1))) VT;
  const VT t = *(GV *)((GC *)base + slot * (uint32_t)sizeof(T));
#pragma unroll
  for (int e = 0; e < H; ++e) v[e] = t[e];
}
template <typename T, int H>
__device__ __forceinline__ void stv(T *base, uint32_t slot, const T (&v)[H]) {
  typedef T VT __attribute__((ext_vector_type(H), aligned(sizeof(T))));
  using GC = __attribute__((address_space(1))) char;
  using GV = __attribute__((address_space(1))) VT;
  VT t;
#pragma unroll
  for (int e = 0; e < H; ++e) t[e] = v[e];
  *(GV *)((GC *)base + slot * (uint32_t)sizeof(T)) = t;
}

// Rows. A lane takes K consecutive steps of a row, K/2 from each half of the
// split layout, as vector loads; WL = 1: a row is a segment of W lanes (64/W
// rows per wave) and nothing goes through LDS; WL > 1: a row is WL waves,
// chained through LDS. The last lane's vectors may reach up to K/2 values past
// the row (past the array for the last row, into the next array of the
// instance's slab; the slab ends with the last level's scratch, which no sweep
// reads): those values are never used.
// Measured per launch of one colour, tiled against this: the 9-point rows of a
// 1021 x 765 grid (FP32) 7.5 -> 4.1 us and its 5-point ones 12.2 -> 5.2;
// 2048 x 2048 FP64 12.5 -> 6.6 and 39 -> 27; 4096-step rows 62 -> 45 us (3.0
// TB/s); a batch of 48 uneven grids 8.9 -> 5.5 and 21 (two launches) -> 11.3.
template <typename T, int NB, bool ZERO, int K, int WL>
__device__ __forceinline__ void row_sweep(const Lines<T, NB, ZERO, 0> &P, const LineGrp gr, T *lds) {
  constexpr int H = K / 2;
  const int n = P.nx, ny = P.ny, hx = half_x(n);
  T *const x = P.x;
  const T *const b = P.b, *const lo = P.lo, *const inv = P.inv, *const cu = P.cu;
  const T *const om = P.om, *const op = P.op;
  const T *const omm = P.omm, *const omp = P.omp, *const opm = P.opm, *const opp = P.opp;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int W = WL > 1 ? 64 : seg_width((n + K - 1) / K);   // lanes per row in a wave
  const int u = lane & (W - 1);
  const int k = WL > 1 ? wave / WL : wave * (64 / W) + lane / W;   // row of the group
  const int q = WL > 1 ? (wave % WL) * 64 + lane : u;              // run of the row
  const bool on = k < gr.count;
  const int li = gr.first + min(k, gr.count - 1) * gr.step;
  // rows beside; outside the grid the couplings are zero and the row on the
  // other side stands in (it holds values of the other colour)
  const int lm = li > 0 ? li - 1 : min(1, ny - 1), lp = li < ny - 1 ? li + 1 : max(ny - 2, 0);
  const int t0 = q * K;                    // this lane's first step
  const int h0 = t0 < n ? q * H : 0;       // its place in each half
  const uint32_t r0 = (uint32_t)li * n, se = r0 + h0, so = r0 + hx + h0;
  // one array's K values in step order
  auto get = [&](const T *p, uint32_t a, uint32_t c, T (&v)[K]) {
    T ev[H], od[H];
    ldv<T, H>(p, a, ev);
    ldv<T, H>(p, c, od);
#pragma unroll
    for (int e = 0; e < H; ++e) { v[2 * e] = ev[e]; v[2 * e + 1] = od[e]; }
  };
  T al[K], be[K], up[K];
  {
    T vb[K], vl[K], vi[K];
    get(b, se, so, vb);
    get(lo, se, so, vl);
    get(inv, se, so, vi);
    get(cu, se, so, up);
    if (!ZERO) {
      // x of the row beside with its steps t0 - 1 and t0 + K (9-point), zero
      // past the end of the row
      auto beside = [&](int lj, const T *pc, const T *pm, const T *pp) {
        const uint32_t rj = (uint32_t)lj * n;
        T xv[K], c[K];
        get(x, rj + h0, rj + hx + h0, xv);
        get(pc, se, so, c);
        T xl = T(0), xr = T(0), cm[K], cp[K];
        if (NB == 9) {
          xl = ld32(x, rj + hx + max(h0 - 1, 0));
          xr = ld32(x, rj + min(h0 + H, hx - 1));
          get(pm, se, so, cm);
          get(pp, se, so, cp);
        }
#pragma unroll
        for (int e = 0; e < K; ++e) xv[e] = t0 + e < n ? xv[e] : T(0);
#pragma unroll
        for (int e = 0; e < K; ++e) {
          vb[e] -= c[e] * xv[e];
          if (NB == 9) {
            vb[e] -= cm[e] * (e > 0 ? xv[e - 1] : xl);
            vb[e] -= cp[e] * (e + 1 < K ? xv[e + 1] : xr);
          }
        }
      };
      beside(lm, om, omm, omp);
      beside(lp, op, opm, opp);
    }
#pragma unroll
    for (int e = 0; e < K; ++e) {
      const bool ok = t0 + e < n;
      al[e] = ok ? -vl[e] * vi[e] : T(1);
      be[e] = ok ? vb[e] * vi[e] : T(0);
    }
  }
  // the value entering this lane's steps, from the lanes (and waves) before
  auto carry = [&](auto fwdc, T A, T B, T *s) -> T {
    constexpr bool FWD = decltype(fwdc)::value;
    scan_rows<FWD>(A, B, u, W);
    RowMaps<T> m{};
    if (W > 16) m = row_maps<FWD>(A, B);
    T in = T(0);
    if (WL > 1) {
      T a, bb;
      wave_map<FWD>(m, a, bb);
      if (lane == 0) { s[2 * wave] = a; s[2 * wave + 1] = bb; }
      lds_barrier();
      const int w0 = wave - wave % WL;
#pragma unroll
      for (int w = 0; w < WL - 1; ++w) {
        const int ww = FWD ? w0 + w : w0 + WL - 1 - w;
        const T a2 = s[2 * ww], b2 = s[2 * ww + 1];
        in = (FWD ? ww < wave : ww > wave) ? a2 * in + b2 : in;
      }
    }
    return enter<FWD>(A, B, m, u, W, in);
  };
  T A = T(1), B = T(0);
#pragma unroll
  for (int e = 0; e < K; ++e) { B = al[e] * B + be[e]; A = al[e] * A; }
  T d = carry(std::true_type(), A, B, lds);
#pragma unroll
  for (int e = 0; e < K; ++e) {
    const bool ok = t0 + e < n;
    d = al[e] * d + be[e];
    be[e] = ok ? d : T(0);
    al[e] = ok ? -up[e] : T(1);
  }
  A = T(1); B = T(0);
#pragma unroll
  for (int e = K - 1; e >= 0; --e) { B = al[e] * B + be[e]; A = al[e] * A; }
  T xv = carry(std::false_type(), A, B, lds + 8);
  T ev[H], od[H];
#pragma unroll
  for (int e = K - 1; e >= 0; --e) {
    xv = al[e] * xv + be[e];
    if (e & 1) od[e / 2] = xv; else ev[e / 2] = xv;
  }
  if (!on) return;
  if (t0 + K <= n) {
    stv<T, H>(x, se, ev);
    stv<T, H>(x, so, od);
  } else {
#pragma unroll
    for (int e = 0; e < H; ++e) {
      if (t0 + 2 * e < n) st32(x, se + e, ev[e]);
      if (t0 + 2 * e + 1 < n) st32(x, so + e, od[e]);
    }
  }
}

template <typename T, int NB, bool ZERO>
__global__ void __launch_bounds__(kRowThreads) k_rows(const Insts insts,
                                                      const LineGrp *__restrict__ map, int l,
                                                      int xid, int bid) {
  __shared__ T lds[16];
  const LineGrp gr = map[blockIdx.x];
  const Lines<T, NB, ZERO, 0> P(insts, gr.inst, l, xid, bid);
  if (P.st != ST_ACTIVE) return;
  const int n = P.nx;
  if (sizeof(T) == 8 && n <= 256) row_sweep<T, NB, ZERO, 4, 1>(P, gr, lds);
  else if (n <= 512) row_sweep<T, NB, ZERO, 8, 1>(P, gr, lds);
  else if (n <= 1024) row_sweep<T, NB, ZERO, 8, 2>(P, gr, lds);
  else row_sweep<T, NB, ZERO, 8, 4>(P, gr, lds);
}
template <typename T, int NB, bool ZERO>
__global__ void __launch_bounds__(kRowThreads) k_rows_long(const Insts insts,
                                                           const LineGrp *__restrict__ map, int l,
                                                           int xid, int bid) {
  __shared__ T lds[16];
  const LineGrp gr = map[blockIdx.x];
  const Lines<T, NB, ZERO, 0> P(insts, gr.inst, l, xid, bid);
  if (P.st != ST_ACTIVE) return;
  row_sweep<T, NB, ZERO, 16, 4>(P, gr, lds);
}

template <typename T>
void launch_rows(hipStream_t s, const Insts &d, const LineGrp *m, int ngroups, int l, bool is_long,
                 bool zero, int xid, int bid) {
  if (!ngroups) return;
#define SG_ROWS(NB, Z)                                                                    \
  do {                                                                                    \
    if (is_long) k_rows_long<T, NB, Z><<<ngroups, kRowThreads, 0, s>>>(d, m, l, xid, bid); \
    else k_rows<T, NB, Z><<<ngroups, kRowThreads, 0, s>>>(d, m, l, xid, bid);              \
  } while (0)
  if (l > 0) { if (zero) SG_ROWS(9, true); else SG_ROWS(9, false); }
  else { if (zero) SG_ROWS(5, true); else SG_ROWS(5, false); }
#undef SG_ROWS
}
template void launch_rows<double>(hipStream_t, const Insts &, const LineGrp *, int, int, bool,
                                  bool, int, int);
template void launch_rows<float>(hipStream_t, const Insts &, const LineGrp *, int, int, bool,
                                 bool, int, int);

}  // namespace sg
