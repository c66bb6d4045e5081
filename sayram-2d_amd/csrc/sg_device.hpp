// sg_device.hpp -- device helpers shared by the kernel sources: address-space
// casts, slot arithmetic, workgroup barriers and level views.
#pragma once
#include "sg_internal.hpp"

namespace sg {

template <typename T> __device__ __forceinline__ T *ptr(void *p) { return static_cast<T *>(p); }

// Element `slot` of an array whose base is uniform across the workgroup, through
// a 32-bit byte offset in the global address space. The pointers of an
// instance are read from its table, so without the cast the compiler must use
// flat accesses, which also count against the LDS counter: every LDS wait would
// then wait for the global loads in flight too. Cast, the access is
// base + zext(offset), the scalar-base form of the global loads and stores, and
// one offset register serves every array of the same element type. Instances
// hold at most kMaxCells cells, so the offsets of FP64 arrays stay below 2^31.
template <typename T> __device__ __forceinline__ T ld32(const T *base, uint32_t slot) {
  using GC = const __attribute__((address_space(1))) char;
  using GT = const __attribute__((address_space(1))) T;
  return *(GT *)((GC *)base + slot * (uint32_t)sizeof(T));
}
template <typename T> __device__ __forceinline__ void st32(T *base, uint32_t slot, T v) {
  using GC = __attribute__((address_space(1))) char;
  using GT = __attribute__((address_space(1))) T;
  *(GT *)((GC *)base + slot * (uint32_t)sizeof(T)) = v;
}

// Global-address-space view of an array pointer read from the instance table
// (plain indexing of such a pointer compiles to flat accesses).
template <typename T> __device__ __forceinline__ __attribute__((address_space(1))) T *gbl(T *p) {
  return (__attribute__((address_space(1))) T *)p;
}

// Workgroup barrier for LDS data only: it waits for this thread's LDS
// accesses but not for its global loads, so tiles prefetched into registers
// stay in flight across it. Valid where threads exchange data through LDS
// only (a thread that reloads a global element is the one that stored it).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// (i, j) of storage slot K of a level with nx columns (hx = half_x(nx))
__device__ __forceinline__ void cell_ij(int K, int nx, int hx, int &i, int &j) {
  j = K / nx;
  i = xcol(K - j * nx, hx);
}
template <typename T> __device__ __forceinline__ const T *cptr(const void *p) {
  return static_cast<const T *>(p);
}

// Read-only view of an instance's scalars, for the kernels that do not write
// them (only the begin and finish kernels do). Through the constant address
// space the compiler reads these workgroup-uniform values with scalar loads
// instead of per-lane loads that every later load waits behind.
typedef const __attribute__((address_space(4))) KScal ConstKScal;
__device__ __forceinline__ ConstKScal *rsc(CInst &I) { return (ConstKScal *)I.sc; }

__device__ __forceinline__ int status_of(const Insts &insts, int k) {
  return ((const __attribute__((address_space(4))) InstStat *)insts.st)[k].status;
}
__device__ __forceinline__ int ostatus_of(const Insts &insts, int k) {
  return ((const __attribute__((address_space(4))) InstStat *)insts.st)[k].ostatus;
}

__device__ __forceinline__ int phase_of(const Insts &insts, int k) {
  return ((const __attribute__((address_space(4))) InstStat *)insts.st)[k].phase;
}

// Forces uniform values (pointers and sizes read from the instance table) to be
// in registers here. A dependent load costs about 0.8 us (the caches are cold
// when a kernel starts), and the compiler sinks the table's reads below a
// status test, one more round trip; pinned before the test, they are issued
// with the status read.
template <typename P> __device__ __forceinline__ void pin1(P &p) { asm volatile("" : "+s"(p)); }
template <typename... P> __device__ __forceinline__ void pin(P &...p) { (pin1(p), ...); }

// level-0 vector by id: a Krylov slot (Vec) or an FP32 V-cycle vector (PcVec)
__device__ __forceinline__ void *vec(CInst &I, int id) {
  return id < kNumVec ? I.kv[id] : (void *)I.pv[id - kNumVec];
}

template <typename T>
__device__ __forceinline__ void level_xb(CInst &I, int l, int xid, int bid, T *&x,
                                         const T *&b) {
  if (l == 0) { x = ptr<T>(vec(I, xid)); b = cptr<T>(vec(I, bid)); }
  else { x = ptr<T>(I.lev[l].x); b = cptr<T>(I.lev[l].b); }
}

}  // namespace sg
