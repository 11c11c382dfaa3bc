// ttg_gemm.h -- device pieces of the grouped GEMM kernels (gemm.hip): MFMA forms,
// k walk, operand loads.
#pragma once
#include "ttg_internal.h"
#include "ttg_plan.h"

namespace ttg {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

template <typename T>
struct MfmaOp;
template <>
struct MfmaOp<double> {
  typedef v4d acc_t;
  static __device__ __forceinline__ acc_t mac(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct MfmaOp<float> {
  typedef v4f acc_t;
  static __device__ __forceinline__ acc_t mac(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

__device__ __forceinline__ int64_t off2(int x, int e0, int64_t s0, int64_t s1) {
  return (int64_t)(x % e0) * s0 + (int64_t)(x / e0) * s1;
}
// the same in 32 bits: operand blocks are below 2^28 elements (checked by the
// planner), so element offsets and their byte offsets fit an unsigned
__device__ __forceinline__ unsigned off2u(int x, int e0, unsigned s0, unsigned s1) {
  return (unsigned)(x % e0) * s0 + (unsigned)(x / e0) * s1;
}

constexpr int kThreads = 256;

// k-walk state of one tile: task t, second k component k1, chunk start c
struct KWalk {
  int t, k1, c;
};
__device__ __forceinline__ void kwalk_next(KWalk& w, const GemmTask& g, int TK) {
  w.c += TK;
  if (w.c >= g.ek0) {
    w.c = 0;
    if (++w.k1 >= g.nk1) {
      w.k1 = 0;
      w.t++;
    }
  }
}
// position of k-tile kt of block cb's walk: the last task whose first k-tile
// is <= kt (tasks[t0..t1) hold ascending kt0), then (k1, chunk) inside it
__device__ __forceinline__ KWalk kwalk_start(const GemmTask* __restrict__ tasks, const CBlock& cb,
                                             int kt, int TK) {
  if (kt == 0) return KWalk{cb.t0, 0, 0};   // the walk's start (every item without split-K)
  int lo = cb.t0, hi = cb.t1;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (tasks[mid].kt0 <= kt) lo = mid;
    else hi = mid;
  }
  const int ek0 = tasks[lo].ek0, local = kt - tasks[lo].kt0;
  const int nch = (ek0 + TK - 1) / TK;
  return KWalk{lo, local / nch, (local % nch) * TK};
}

// ------------------------------------------------------------------ operand loads
// Raw buffer loads over one operand block: the resource's base is the block
// start, offsets are bytes, and an offset at or above 2^31 reads as zero.
// Row padding and the ragged end of a k chunk become such offsets, so the
// staging loop has no branches.  Blocks are below 2^31 bytes (checked by the
// planner), so a padding offset plus a k offset cannot wrap into range.
constexpr unsigned kOOB = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t block_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7FFFFFFF,
                                           0x00020000);
}
// `uni` is a uniform part of the offset (a scalar register: no vector add)
template <typename T>
__device__ __forceinline__ T buf_load(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned uni = 0) {
  if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, uni, 0));
  else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, uni, 0));
}

}  // namespace ttg
