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

// U pieces of eight consecutive outputs; their offset inside the row is a multiple of 8, so bias, gate and residual come as 16-byte
// loads.  What bounds a write-out with an output stage is not its bytes: with one piece at a time a thread waits for a trip to the L2
// per piece (8 - 16 of them) and the values' exponentials follow one another.  So the operands of U pieces are asked for together,
// and the activation is chosen outside the loop over their values.  Pieces that are not stored carry positions inside the operands.
template <typename T, int U>
__device__ __forceinline__ void ep_vectors(const GemmArgs& g, typename TypeTraits<T>::vec8 (&r)[U], const int64_t (&in_row)[U], const int (&row)[U]) {
  using V8 = typename TypeTraits<T>::vec8;
  V8 bv[U], gv[U], rv[U];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) { bv[u][e] = (T)0.0f; gv[u][e] = (T)1.0f; rv[u][e] = (T)0.0f; }
  if (g.bias) {
#pragma unroll
    for (int u = 0; u < U; ++u) bv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.bias) + in_row[u]);
  }
  if (g.gate) {                                 // one row of gate per group of gate_rows rows of C
#pragma unroll
    for (int u = 0; u < U; ++u) gv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.gate) + (int64_t)(row[u] / g.gate_rows) * g.ld_gate + in_row[u]);
  }
  if (g.resid) {
#pragma unroll
    for (int u = 0; u < U; ++u) rv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.resid) + (int64_t)row[u] * g.ld_resid + in_row[u]);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = TypeTraits<T>::to_f32(r[u][e]) + TypeTraits<T>::to_f32(bv[u][e]);
    apply_act_n(v, g.act);
#pragma unroll
    for (int e = 0; e < 8; ++e) r[u][e] = TypeTraits<T>::from_f32(v[e]);
  }
  if (g.gate || g.resid) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) r[u][e] = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(r[u][e]) * TypeTraits<T>::to_f32(gv[u][e]) + TypeTraits<T>::to_f32(rv[u][e]));
  }
}
template <typename T>
__device__ __forceinline__ typename TypeTraits<T>::vec8 ep_vector(const GemmArgs& g, typename TypeTraits<T>::vec8 r, int64_t in_row, int row) {
  typename TypeTraits<T>::vec8 v[1] = {r};
  const int64_t at[1] = {in_row};
  const int rows[1] = {row};
  ep_vectors<T, 1>(g, v, at, rows);
  return v[0];
}

// Second tile of a pair: (r + bias) rounded to T, times the first tile's result, which the same thread stored at c[u] before.
template <typename T, int U>
__device__ __forceinline__ void ep_pair_up(const GemmArgs& g, typename TypeTraits<T>::vec8 (&r)[U], const int64_t (&in_row)[U], const T* const (&c)[U]) {
  using V8 = typename TypeTraits<T>::vec8;
  V8 bv[U], gv[U];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) bv[u][e] = (T)0.0f;
  if (g.bias) {
#pragma unroll
    for (int u = 0; u < U; ++u) bv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.bias) + in_row[u]);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) gv[u] = *reinterpret_cast<const V8*>(c[u]);
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const T up = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(r[u][e]) + TypeTraits<T>::to_f32(bv[u][e]));
      r[u][e] = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(gv[u][e]) * TypeTraits<T>::to_f32(up));
    }
}

}  // namespace blr
