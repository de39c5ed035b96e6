// Device helpers shared by the GEMM kernels (blr_gemm.hip, blr_gemm_mid.hip): where a result goes, and the fused output stage.
#pragma once
#include "blr_common.h"

namespace blr {

__device__ __forceinline__ int64_t epi_offset(const GemmArgs& g, int bt, int m, int n) {
  if (g.epi == EPI_MONARCH_SCATTER) {
    int dst_blk = n / g.per, j = n - dst_blk * g.per;
    return (int64_t)dst_blk * g.sL + (int64_t)m * g.ldc + (int64_t)bt * g.per + j;
  }
  return (int64_t)bt * g.sC + (int64_t)m * g.ldc + (int64_t)n * g.cn;
}

// Fused output stage (kernels instantiated with EP): bias (indexed by the element's offset inside its row of C) and
// activation are applied to the rounded result on its way out, like the separate kernels of the callers would.  The
// plain instantiations do not contain this code: it costs registers that the main loops need.
template <typename T>
__device__ __forceinline__ T ep_value(const GemmArgs& g, T r, int64_t in_row, int row) {
  float v = TypeTraits<T>::to_f32(r);
  if (g.bias) v += TypeTraits<T>::to_f32(reinterpret_cast<const T*>(g.bias)[in_row]);
  v = apply_act(v, g.act);
  if (g.gate || g.resid) {
    v = TypeTraits<T>::to_f32(TypeTraits<T>::from_f32(v));                    // what a separate gate / residual kernel would read
    if (g.gate) v *= TypeTraits<T>::to_f32(reinterpret_cast<const T*>(g.gate)[(int64_t)(row / g.gate_rows) * g.ld_gate + in_row]);
    if (g.resid) v += TypeTraits<T>::to_f32(reinterpret_cast<const T*>(g.resid)[(int64_t)row * g.ld_resid + in_row]);
  }
  return TypeTraits<T>::from_f32(v);
}

// eight consecutive outputs; their offset inside the row is a multiple of 8, so the bias comes as one 16-byte load
template <typename T>
__device__ __forceinline__ typename TypeTraits<T>::vec8 ep_vector(const GemmArgs& g, typename TypeTraits<T>::vec8 r, int64_t in_row, int row) {
  using V8 = typename TypeTraits<T>::vec8;
  V8 bv;
#pragma unroll
  for (int e = 0; e < 8; ++e) bv[e] = (T)0.0f;
  if (g.bias) bv = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.bias) + in_row);
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = TypeTraits<T>::from_f32(apply_act(TypeTraits<T>::to_f32(r[e]) + TypeTraits<T>::to_f32(bv[e]), g.act));
  if (g.gate || g.resid) {                      // one row of gate per group of gate_rows rows of C
    V8 gv, rv;
#pragma unroll
    for (int e = 0; e < 8; ++e) { gv[e] = (T)1.0f; rv[e] = (T)0.0f; }
    if (g.gate) gv = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.gate) + (int64_t)(row / g.gate_rows) * g.ld_gate + in_row);
    if (g.resid) rv = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.resid) + (int64_t)row * g.ld_resid + in_row);
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(r[e]) * TypeTraits<T>::to_f32(gv[e]) + TypeTraits<T>::to_f32(rv[e]));
  }
  return r;
}

// Second tile of a pair: (r + bias) rounded to T, times the first tile's result, which the same thread stored at `c` before.
template <typename T>
__device__ __forceinline__ typename TypeTraits<T>::vec8 ep_pair_up(const GemmArgs& g, typename TypeTraits<T>::vec8 r, int64_t in_row, const T* c) {
  using V8 = typename TypeTraits<T>::vec8;
  V8 bv;
#pragma unroll
  for (int e = 0; e < 8; ++e) bv[e] = (T)0.0f;
  if (g.bias) bv = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.bias) + in_row);
  const V8 gv = *reinterpret_cast<const V8*>(c);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const T up = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(r[e]) + TypeTraits<T>::to_f32(bv[e]));
    r[e] = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(gv[e]) * TypeTraits<T>::to_f32(up));
  }
  return r;
}

}  // namespace blr
