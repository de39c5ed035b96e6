// What a transformer block does between its structured linears (DiT): adaLN's normalise-and-modulate.
#include "blr_common.h"

namespace blr {
namespace {

// ---- out = (1 + scale) * LayerNorm(x) + shift, no affine part (reference DiT/models.py:19-20, 120-121) ----------------------
// Memory bound: every row is read once and written once.  One wave takes a row and holds it in registers (NV pieces of 16 bytes
// a lane), so that mean and variance are two exact passes without another read; a workgroup is four rows, which share nothing.
// Statistics and result are fp32, rounded once at the end.  1152 columns x 4096 rows, fp16: layer norm 10.3, 1 + scale 4.7,
// multiply-add 8.9 us as three kernels, 6.7 us here (18.9 MB at 2.8 TB/s: start-up and two dependent reductions of one row a wave).
template <typename T, int NV>
__global__ __launch_bounds__(256) void ln_modulate_kernel(const T* __restrict__ x, const T* __restrict__ shift, int64_t ld_shift, const T* __restrict__ scale,
                                                          int64_t ld_scale, T* __restrict__ out, int rows, int C, int per, float eps) {
  using V8 = typename TypeTraits<T>::vec8;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* xr = x + (int64_t)row * C;
  const T* sh = shift + (int64_t)(row / per) * ld_shift;
  const T* sc = scale + (int64_t)(row / per) * ld_scale;
  V8 v[NV], a[NV], b[NV];
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (lane + 64 * i) * 8;
    if (c < C) {
      v[i] = ldg16<V8>(xr + c);
      a[i] = ldg16<V8>(sc + c);
      b[i] = ldg16<V8>(sh + c);
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if ((lane + 64 * i) * 8 < C)
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += TypeTraits<T>::to_f32(v[i][e]);
  const float mean = wave_sum(sum) / (float)C;
  float var = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if ((lane + 64 * i) * 8 < C)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = TypeTraits<T>::to_f32(v[i][e]) - mean;
        var += d * d;
      }
  const float rstd = rsqrtf(wave_sum(var) / (float)C + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (lane + 64 * i) * 8;
    if (c >= C) continue;
    V8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      o[e] = TypeTraits<T>::from_f32((TypeTraits<T>::to_f32(v[i][e]) - mean) * rstd * (1.0f + TypeTraits<T>::to_f32(a[i][e])) + TypeTraits<T>::to_f32(b[i][e]));
    *reinterpret_cast<V8*>(out + (int64_t)row * C + c) = o;
  }
}

template <typename T>
int ln_modulate(const void* x, const void* shift, int64_t ld_shift, const void* scale, int64_t ld_scale, void* out, int rows, int C, int per, float eps, hipStream_t st) {
  const dim3 grid((unsigned)cdiv(rows, 4));
#define GO(NV)                                                                                                                                     \
  hipLaunchKernelGGL((ln_modulate_kernel<T, NV>), grid, dim3(256), 0, st, (const T*)x, (const T*)shift, ld_shift, (const T*)scale, ld_scale, (T*)out, rows, C, per, eps)
  if (C <= 512) GO(1); else if (C <= 1024) GO(2); else if (C <= 1536) GO(3); else GO(4);
#undef GO
  BLR_CHECK_LAUNCH("ln_modulate");
  return BLR_OK;
}

}  // namespace
}  // namespace blr

using namespace blr;

extern "C" {

int blr_ln_modulate(const void* x, const void* shift, int64_t ld_shift, const void* scale, int64_t ld_scale, void* out, int rows, int cols, int rows_per_group,
                    float eps, int dtype, void* stream) {
  if (!x || !shift || !scale || !out) { set_error("ln_modulate: null pointer"); return BLR_ERR_BAD_ARG; }
  if (rows <= 0 || cols <= 0 || rows_per_group <= 0 || ld_shift < cols || ld_scale < cols) { set_error("ln_modulate: bad size"); return BLR_ERR_BAD_ARG; }
  if ((dtype != BLR_F16 && dtype != BLR_BF16) || cols % 8 || cols > 2048 || ld_shift % 8 || ld_scale % 8 || !aligned(x, 16) || !aligned(shift, 16) || !aligned(scale, 16) ||
      !aligned(out, 16)) {
    set_error("ln_modulate: needs f16 / bf16, at most 2048 columns in whole 16-byte pieces");
    return BLR_ERR_UNSUPPORTED;
  }
  return dtype == BLR_F16 ? ln_modulate<f16>(x, shift, ld_shift, scale, ld_scale, out, rows, cols, rows_per_group, eps, (hipStream_t)stream)
                          : ln_modulate<bf16>(x, shift, ld_shift, scale, ld_scale, out, rows, cols, rows_per_group, eps, (hipStream_t)stream);
}

}  // extern "C"
