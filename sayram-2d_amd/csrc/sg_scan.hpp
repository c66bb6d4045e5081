// sg_scan.hpp -- wave-level scans of first-order affine maps.
//
// Both Thomas recurrences of a tridiagonal line are first-order affine maps
// y_t = a_t y_{t-1} + b_t (forward d_t, and backward x_t from the line's end).
// The threads of a line each compose the maps of their own steps into one map
// (A, B): y_out = A y_in + B. A segment of W lanes (a power of two, aligned in
// the wave) holds one line. The scans run on DPP lane moves inside the wave's
// rows of 16 lanes (a few cycles each; a bpermute through the LDS unit is an
// LDS round trip), and the rows are chained through v_readlane.
//
// Every lane of the wave must be active; W is uniform across the wave.
#pragma once
#include <hip/hip_runtime.h>

namespace sg {

// v moved between lanes by the DPP control CTRL; lanes without a source
// (across the ends of a row of 16) get `old`
template <int CTRL> __device__ __forceinline__ float dpp(float old, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old),
                                                               __builtin_bit_cast(int, v), CTRL,
                                                               0xf, 0xf, false));
}
template <int CTRL> __device__ __forceinline__ double dpp(double old, double v) {
  const long long o = __builtin_bit_cast(long long, old), s = __builtin_bit_cast(long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp((int)o, (int)s, CTRL, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(s >> 32), CTRL, 0xf, 0xf,
                                                  false);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
__device__ __forceinline__ float rdlane(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ double rdlane(double v, int l) {
  const long long s = __builtin_bit_cast(long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((int)s, l);
  const unsigned hi = __builtin_amdgcn_readlane((int)(s >> 32), l);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// DPP controls: lane i takes lane i - n / i + n of its row of 16
constexpr int kRowShr = 0x110, kRowShl = 0x100;
// lane i takes lane i - 1 of the wave
constexpr int kWaveShr1 = 0x138;

// Inclusive scan inside the rows: (A, B) of a lane becomes the composition of
// the maps of its row's (for W < 16: its segment's) lanes up to it, in order
// (FWD), or from it to the end (backward). u: the lane's position in its
// segment.
template <bool FWD, typename T>
__device__ __forceinline__ void scan_rows(T &A, T &B, int u, int W) {
  const int Wr = W < 16 ? W : 16, ur = u & (Wr - 1);
#define SG_ROUND(OFF)                                                             \
  if (W > OFF) {                                                                  \
    T Ap = dpp<(FWD ? kRowShr : kRowShl) | OFF>(T(1), A);                         \
    T Bp = dpp<(FWD ? kRowShr : kRowShl) | OFF>(T(0), B);                         \
    const bool in = FWD ? ur >= OFF : ur + OFF < Wr;                              \
    Ap = in ? Ap : T(1);                                                          \
    Bp = in ? Bp : T(0);                                                          \
    B = A * Bp + B;                                                               \
    A = A * Ap;                                                                   \
  }
  SG_ROUND(1) SG_ROUND(2) SG_ROUND(4) SG_ROUND(8)
#undef SG_ROUND
}

// The maps of the four rows of a wave, from the inclusive row scans (uniform).
template <typename T> struct RowMaps { T a[4], b[4]; };
template <bool FWD, typename T> __device__ __forceinline__ RowMaps<T> row_maps(T A, T B) {
  RowMaps<T> m;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m.a[r] = rdlane(A, FWD ? 16 * r + 15 : 16 * r);
    m.b[r] = rdlane(B, FWD ? 16 * r + 15 : 16 * r);
  }
  return m;
}
// The map of the whole wave (W = 64).
template <bool FWD, typename T>
__device__ __forceinline__ void wave_map(const RowMaps<T> &m, T &A, T &B) {
  A = T(1); B = T(0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = FWD ? k : 3 - k;
    B = m.a[r] * B + m.b[r];
    A = m.a[r] * A;
  }
}

// The value entering a lane's own map: after scan_rows, with `in` the value
// entering the segment (W = 64: the wave; shorter segments start from 0).
template <bool FWD, typename T>
__device__ __forceinline__ T enter(T A, T B, const RowMaps<T> &m, int u, int W, T in) {
  const int Wr = W < 16 ? W : 16, ur = u & (Wr - 1);
  T Ae = dpp<(FWD ? kRowShr : kRowShl) | 1>(T(1), A);
  T Be = dpp<(FWD ? kRowShr : kRowShl) | 1>(T(0), B);
  const bool first = FWD ? ur == 0 : ur == Wr - 1;
  Ae = first ? T(1) : Ae;
  Be = first ? T(0) : Be;
  if (W <= 16) return Be;
  const int row = (threadIdx.x >> 4) & 3;
  if (W == 32) {   // two rows per segment
    const T v = FWD ? (row == 1 ? m.b[0] : row == 3 ? m.b[2] : T(0))
                    : (row == 0 ? m.b[1] : row == 2 ? m.b[3] : T(0));
    return Ae * v + Be;
  }
  T v, w = in;
  v = w;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int r = FWD ? k : 3 - k;
    w = m.a[r] * w + m.b[r];
    v = row == (FWD ? k + 1 : 2 - k) ? w : v;
  }
  return Ae * v + Be;
}

// v moved by the DPP control CTRL inside the rows of 16 lanes; lanes without a
// source get 0
template <int CTRL> __device__ __forceinline__ float dpp0(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                               0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double dpp0(double v) {
  const long long s = __builtin_bit_cast(long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)s, CTRL, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(s >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// B of the inclusive scan over a row of 16 lanes that starts from 0, for
// segments whose first map has A = 0 (the recurrence starts anew there), so
// that no lane needs to know where its segment begins.
template <bool FWD, typename T> __device__ __forceinline__ T scan_row0(T A, T B) {
  constexpr int C = FWD ? kRowShr : kRowShl;
  B = A * dpp0<C | 1>(B) + B; A = A * dpp0<C | 1>(A);
  B = A * dpp0<C | 2>(B) + B; A = A * dpp0<C | 2>(A);
  B = A * dpp0<C | 4>(B) + B; A = A * dpp0<C | 4>(A);
  return A * dpp0<C | 8>(B) + B;
}

// The value entering a lane's map from the lanes before it, for segments of one
// row of 16 lanes (scan_row0), ...
template <bool FWD, typename T> __device__ __forceinline__ T enter_row0(T A, T B) {
  return dpp0<(FWD ? kRowShr : kRowShl) | 1>(scan_row0<FWD>(A, B));
}
// ... and of two or four rows: the rows are chained through v_readlane.
template <bool FWD, typename T> __device__ __forceinline__ T enter_rows0(T A, T B) {
  constexpr int C = FWD ? kRowShr : kRowShl;
  B = A * dpp0<C | 1>(B) + B; A = A * dpp<C | 1>(T(1), A);
  B = A * dpp0<C | 2>(B) + B; A = A * dpp<C | 2>(T(1), A);
  B = A * dpp0<C | 4>(B) + B; A = A * dpp<C | 4>(T(1), A);
  B = A * dpp0<C | 8>(B) + B; A = A * dpp<C | 8>(T(1), A);
  const RowMaps<T> m = row_maps<FWD>(A, B);
  const int row = (threadIdx.x >> 4) & 3;
  T v = T(0), w = T(0);   // w enters the next row, v this lane's
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int r = FWD ? k : 3 - k;
    w = m.a[r] * w + m.b[r];
    v = row == (FWD ? k + 1 : 2 - k) ? w : v;
  }
  const T e = dpp0<C | 1>(A * v + B);
  return (threadIdx.x & 15) == (FWD ? 0 : 15) ? v : e;
}

// smallest power of two >= n, at most 64
__device__ __forceinline__ int seg_width(int n) {
  return n <= 1 ? 1 : n >= 64 ? 64 : 1 << (32 - __builtin_clz(n - 1));
}

}  // namespace sg
