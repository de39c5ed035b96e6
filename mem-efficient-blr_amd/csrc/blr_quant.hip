// Symmetric per-channel weight quantizer: max-abs over the reduced axis, scale = fp16(max / Qmax) (1 for a channel whose scale
// is zero), code = clamp(rne(w / scale), +-Qmax).  Memory bound: the weights are read twice (the maximum, then the codes), the
// second time out of the L2 or the Infinity Cache, and the codes written once.
#include "blr_common.h"

namespace blr {
namespace {

__device__ __forceinline__ float make_scale(float amax, float qmax) {
  const f16 s16 = (f16)__fdiv_rn(amax, qmax);
  return (float)s16 == 0.0f ? 1.0f : (float)s16;
}

// rne(w / s) clamped, for the correctly rounded quotient.  The product with 1 / s is within 2^-22 of it relatively (one rounding
// of the reciprocal, 1 ulp of v_rcp_f32, one of the product), at most 3.1e-5 where the clamp does not decide (|w / s| < 128), so
// both round to the same integer unless the product lies within 1e-4 of a half: only then is the division carried out.
__device__ __forceinline__ int quant_code(float w, float s, float inv, float qmax) {
  float q = w * inv;
  const float f = fabsf(q) - floorf(fabsf(q));
  if (fabsf(f - 0.5f) < 1e-4f) q = __fdiv_rn(w, s);
  q = fminf(fmaxf(rintf(q), -qmax), qmax);
  return (int)q;
}

// VEC consecutive elements as fp32 (four: 4 * sizeof(T)-byte aligned)
template <typename T, int VEC>
__device__ __forceinline__ void ld_vec(const T* p, float (&v)[VEC]) {
  typedef T vec __attribute__((ext_vector_type(VEC)));
  if constexpr (VEC < 4) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[e] = TypeTraits<T>::to_f32(p[e]);
  } else {
    const vec x = *reinterpret_cast<const vec*>(p);
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[e] = TypeTraits<T>::to_f32(x[e]);
  }
}

// inner == 1: one workgroup per channel row, max over the contiguous axis.
template <typename T>
__global__ __launch_bounds__(256) void quant_rows_kernel(const T* __restrict__ w, int64_t reduce, int bits,
                                                         uint8_t* __restrict__ codes, f16* __restrict__ scales) {
  __shared__ float s_max[4];
  const int64_t row = blockIdx.x;
  const T* wr = w + row * reduce;
  float amax = 0.0f;
  for (int64_t k = threadIdx.x; k < reduce; k += 256) amax = fmaxf(amax, fabsf(TypeTraits<T>::to_f32(wr[k])));
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = amax;
  __syncthreads();
  const float qmax = bits == 8 ? 127.0f : 7.0f;
  const float s = make_scale(fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3])), qmax), inv = __builtin_amdgcn_rcpf(s);
  if (threadIdx.x == 0) scales[row] = (f16)s;
  if (bits == 8) {
    int8_t* c = reinterpret_cast<int8_t*>(codes) + row * reduce;
    for (int64_t k = threadIdx.x; k < reduce; k += 256) c[k] = (int8_t)quant_code(TypeTraits<T>::to_f32(wr[k]), s, inv, qmax);
  } else {
    uint8_t* c = codes + row * (reduce / 2);
    for (int64_t k = threadIdx.x; k < reduce / 2; k += 256) {
      const int lo = quant_code(TypeTraits<T>::to_f32(wr[2 * k]), s, inv, qmax), hi = quant_code(TypeTraits<T>::to_f32(wr[2 * k + 1]), s, inv, qmax);
      c[k] = (uint8_t)((lo & 0xF) | ((hi & 0xF) << 4));
    }
  }
}

// inner > 1 (V (b, p, r)): a workgroup owns (1 << lg) pieces of VEC columns and all rows; its 256 >> lg row groups take every so
// many rows, meet in LDS for the maximum and go over the rows again for the codes.  One thread per column and a loop over all
// rows, as before, put 32 workgroups on the chip and waited out every load: 190 us for 16 blocks of 256 x 1024 in fp32, 10 us now
// (17 MB read twice, the second time from the L2).
template <typename T, int VEC, int BITS>
__global__ __launch_bounds__(256) void quant_cols_kernel(const T* __restrict__ w, int64_t reduce, int64_t inner, int lg,
                                                         uint8_t* __restrict__ codes, f16* __restrict__ scales) {
  __shared__ float s_max[256 * VEC];
  const int lane = threadIdx.x & ((1 << lg) - 1), g = threadIdx.x >> lg, ng = 256 >> lg;
  const int64_t o = blockIdx.y, c0 = (((int64_t)blockIdx.x << lg) + lane) * VEC;
  const bool in = c0 < inner;
  const T* wc = w + o * reduce * inner + (in ? c0 : 0);
  float amax[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) amax[e] = 0.0f;
  int64_t k = g;
  for (; k + 7 * ng < reduce; k += 8 * ng) {
    float v[8][VEC];
#pragma unroll
    for (int u = 0; u < 8; ++u) ld_vec<T, VEC>(wc + (k + u * ng) * inner, v[u]);
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < VEC; ++e) amax[e] = fmaxf(amax[e], fabsf(v[u][e]));
  }
  for (; k < reduce; k += ng) {
    float v[VEC];
    ld_vec<T, VEC>(wc + k * inner, v);
#pragma unroll
    for (int e = 0; e < VEC; ++e) amax[e] = fmaxf(amax[e], fabsf(v[e]));
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) s_max[threadIdx.x * VEC + e] = amax[e];
  __syncthreads();
  for (int h = ng >> 1; h > 0; h >>= 1) {
    if (g < h)
#pragma unroll
      for (int e = 0; e < VEC; ++e) s_max[threadIdx.x * VEC + e] = fmaxf(s_max[threadIdx.x * VEC + e], s_max[(threadIdx.x + (h << lg)) * VEC + e]);
    __syncthreads();
  }
  constexpr float qmax = BITS == 8 ? 127.0f : 7.0f;
  float s[VEC], inv[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    s[e] = make_scale(s_max[lane * VEC + e], qmax);
    inv[e] = __builtin_amdgcn_rcpf(s[e]);
  }
  if (!in) return;
  if (g == 0)
#pragma unroll
    for (int e = 0; e < VEC; ++e) scales[o * inner + c0 + e] = (f16)s[e];
  constexpr int CB = VEC * BITS / 8;                // bytes of codes per thread and row
  typedef uint8_t cvec __attribute__((ext_vector_type(CB > 1 ? CB : 2)));
  uint8_t* co = codes + ((o * reduce * inner + c0) * BITS) / 8;
  auto put = [&](int64_t row, const float (&v)[VEC]) {
    uint8_t c[CB];
#pragma unroll
    for (int e = 0; e < CB; ++e) {
      if constexpr (BITS == 8) c[e] = (uint8_t)quant_code(v[e], s[e], inv[e], qmax);
      else c[e] = (uint8_t)((quant_code(v[2 * e], s[2 * e], inv[2 * e], qmax) & 0xF) | ((quant_code(v[2 * e + 1], s[2 * e + 1], inv[2 * e + 1], qmax) & 0xF) << 4));
    }
    uint8_t* d = co + row * (inner * BITS / 8);
    if constexpr (CB == 1) *d = c[0];
    else {
      cvec x;
#pragma unroll
      for (int e = 0; e < CB; ++e) x[e] = c[e];
      *reinterpret_cast<cvec*>(d) = x;
    }
  };
  k = g;
  for (; k + 3 * ng < reduce; k += 4 * ng) {
    float v[4][VEC];
#pragma unroll
    for (int u = 0; u < 4; ++u) ld_vec<T, VEC>(wc + (k + u * ng) * inner, v[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) put(k + u * ng, v[u]);
  }
  for (; k < reduce; k += ng) {
    float v[VEC];
    ld_vec<T, VEC>(wc + k * inner, v);
    put(k, v);
  }
}

// Reduced axis contiguous, codes transposed (U (b, q, r) -> codes (b, r, q)).  First the scales: one wave per channel.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void quant_scale_kernel(const T* __restrict__ w, int64_t channels, int64_t reduce, float qmax, f16* __restrict__ scales) {
  const int64_t ch = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (ch >= channels) return;
  const int lane = threadIdx.x & 63;
  const T* wr = w + ch * reduce;
  float amax = 0.0f;
  int64_t k = lane * VEC;
  for (; k + 3 * 64 * VEC < reduce; k += 4 * 64 * VEC) {
    float v[4][VEC];
#pragma unroll
    for (int u = 0; u < 4; ++u) ld_vec<T, VEC>(wr + k + u * 64 * VEC, v[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < VEC; ++e) amax = fmaxf(amax, fabsf(v[u][e]));
  }
  for (; k < reduce; k += 64 * VEC) {
    float v[VEC];
    ld_vec<T, VEC>(wr + k, v);
#pragma unroll
    for (int e = 0; e < VEC; ++e) amax = fmaxf(amax, fabsf(v[e]));
  }
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
  if (lane == 0) scales[ch] = (f16)make_scale(amax, qmax);
}

// Then the codes: a workgroup turns a tile of 128 channels x 64 values.  A thread reads four values of four neighbouring channels
// (16 lanes cover a channel's 64 values), packs the four codes of each value into one dword of LDS, and the rows of the tile leave
// as 128 (int8) or 64 (int4) bytes each.  16 blocks of 1376 x 1024 in fp32: the transposed copy and the column kernel took 830 us,
// the two launches 17 + 26 us (90 MB each, at 5.2 and 3.9 TB/s with the codes).
template <typename T, int BITS>
__global__ __launch_bounds__(256) void quant_turn_kernel(const T* __restrict__ w, int64_t reduce, int64_t inner, int vec_ok, int words,
                                                         uint8_t* __restrict__ codes, const f16* __restrict__ scales) {
  __shared__ uint32_t s_codes[64][33];              // [value][channel / 4], padded: the 16 lanes of a channel meet 8 banks twice
  const int64_t o = blockIdx.z, q0 = (int64_t)blockIdx.x * 128, r0 = (int64_t)blockIdx.y * 64;
  const int l = threadIdx.x & 15, t16 = threadIdx.x >> 4;
  constexpr float qmax = BITS == 8 ? 127.0f : 7.0f;
  const T* wo = w + o * inner * reduce;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int qg = h * 16 + t16;                    // group of four channels
    float v[4][4];
    float s[4], inv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int64_t q = q0 + qg * 4 + c, r = r0 + l * 4;
      const bool in = q < inner;
      s[c] = in ? (float)scales[o * inner + q] : 1.0f;
      inv[c] = __builtin_amdgcn_rcpf(s[c]);
      const T* p = wo + q * reduce + r;
      if (in && vec_ok && r + 4 <= reduce) ld_vec<T, 4>(p, v[c]);
      else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[c][e] = in && r + e < reduce ? TypeTraits<T>::to_f32(p[e]) : 0.0f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t d = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t code = (uint32_t)quant_code(v[c][e], s[c], inv[c], qmax);
        d |= (code & (BITS == 8 ? 0xFFu : 0xFu)) << (c * BITS);
      }
      s_codes[l * 4 + e][qg] = d;                   // int4: two bytes of codes in the low half
    }
  }
  __syncthreads();
  const int64_t row_bytes = inner * BITS / 8;       // (inner even for int4)
  uint8_t* co = codes + o * reduce * row_bytes;
  constexpr int DW = BITS == 8 ? 32 : 16;           // dwords of a tile row
  for (int i = threadIdx.x; i < 64 * DW; i += 256) {
    const int rr = i / DW, d = i % DW;
    const int64_t r = r0 + rr, byte = (BITS == 8 ? q0 : q0 / 2) + d * 4;
    if (r >= reduce || byte >= row_bytes) continue;
    uint32_t x;
    if constexpr (BITS == 8) x = s_codes[rr][d];
    else x = (s_codes[rr][2 * d] & 0xFFFFu) | (s_codes[rr][2 * d + 1] << 16);
    uint8_t* p = co + r * row_bytes + byte;
    if (words) *reinterpret_cast<uint32_t*>(p) = x;
    else
      for (int e = 0; e < 4 && byte + e < row_bytes; ++e) p[e] = (uint8_t)(x >> (8 * e));
  }
}

template <typename T, int VEC>
int cols_launch(const T* w, int64_t outer, int64_t reduce, int64_t inner, int bits, uint8_t* codes, f16* scales, hipStream_t st) {
  // 64 columns a workgroup (whole lines of codes); down to pieces of 16 columns while that leaves compute units without one
  int lg = 4;
  while (lg > 2 && outer * cdiv(inner, (int64_t)VEC << lg) < 512) --lg;
  const dim3 grid((unsigned)cdiv(inner, (int64_t)VEC << lg), (unsigned)outer);
  if (bits == 8) hipLaunchKernelGGL((quant_cols_kernel<T, VEC, 8>), grid, dim3(256), 0, st, w, reduce, inner, lg, codes, scales);
  else hipLaunchKernelGGL((quant_cols_kernel<T, VEC < 2 ? 2 : VEC, 4>), grid, dim3(256), 0, st, w, reduce, inner, lg, codes, scales);
  BLR_CHECK_LAUNCH("quantize");
  return BLR_OK;
}

template <typename T>
int quantize_any(const T* w, int64_t outer, int64_t reduce, int64_t inner, int bits, uint8_t* codes, f16* scales, hipStream_t st) {
  if (inner == 1) {
    hipLaunchKernelGGL(quant_rows_kernel<T>, dim3((unsigned)outer), dim3(256), 0, st, w, reduce, bits, codes, scales);
    BLR_CHECK_LAUNCH("quantize");
    return BLR_OK;
  }
  // four columns a thread where rows of the weights and of the codes keep such pieces aligned
  if (inner % 4 == 0 && aligned(w, 4 * sizeof(T)) && aligned(codes, 4)) return cols_launch<T, 4>(w, outer, reduce, inner, bits, codes, scales, st);
  if (bits == 4) return cols_launch<T, 2>(w, outer, reduce, inner, bits, codes, scales, st);   // (inner is even)
  return cols_launch<T, 1>(w, outer, reduce, inner, bits, codes, scales, st);
}

template <typename T>
int quantize_turned(const T* w, int64_t outer, int64_t reduce, int64_t inner, int bits, uint8_t* codes, f16* scales, hipStream_t st) {
  const int64_t channels = outer * inner;
  const bool vec = reduce % 4 == 0 && aligned(w, 4 * sizeof(T));                     // loads of four values
  const bool words = (inner * bits / 8) % 4 == 0 && aligned(codes, 4);               // stores of four bytes of codes
  const float qmax = bits == 8 ? 127.0f : 7.0f;
  const dim3 g1((unsigned)cdiv(channels, 4));
  if (vec) hipLaunchKernelGGL((quant_scale_kernel<T, 4>), g1, dim3(256), 0, st, w, channels, reduce, qmax, scales);
  else hipLaunchKernelGGL((quant_scale_kernel<T, 1>), g1, dim3(256), 0, st, w, channels, reduce, qmax, scales);
  const dim3 g2((unsigned)cdiv(inner, 128), (unsigned)cdiv(reduce, 64), (unsigned)outer);
  if (bits == 8) hipLaunchKernelGGL((quant_turn_kernel<T, 8>), g2, dim3(256), 0, st, w, reduce, inner, (int)vec, (int)words, codes, (const f16*)scales);
  else hipLaunchKernelGGL((quant_turn_kernel<T, 4>), g2, dim3(256), 0, st, w, reduce, inner, (int)vec, (int)words, codes, (const f16*)scales);
  BLR_CHECK_LAUNCH("quantize");
  return BLR_OK;
}

}  // namespace

int quantize_launch(const void* w, int dtype, int64_t outer, int64_t reduce, int64_t inner, int bits, void* codes, void* scales, hipStream_t st) {
  uint8_t* c = (uint8_t*)codes; f16* s = (f16*)scales;
  if (dtype == BLR_F32) return quantize_any((const float*)w, outer, reduce, inner, bits, c, s, st);
  if (dtype == BLR_F16) return quantize_any((const f16*)w, outer, reduce, inner, bits, c, s, st);
  return quantize_any((const bf16*)w, outer, reduce, inner, bits, c, s, st);
}

int quantize_t_launch(const void* w, int dtype, int64_t outer, int64_t reduce, int64_t inner, int bits, void* codes, void* scales, hipStream_t st) {
  uint8_t* c = (uint8_t*)codes; f16* s = (f16*)scales;
  if (dtype == BLR_F32) return quantize_turned((const float*)w, outer, reduce, inner, bits, c, s, st);
  if (dtype == BLR_F16) return quantize_turned((const f16*)w, outer, reduce, inner, bits, c, s, st);
  return quantize_turned((const bf16*)w, outer, reduce, inner, bits, c, s, st);
}

}  // namespace blr
