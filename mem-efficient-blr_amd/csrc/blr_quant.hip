// Symmetric per-channel weight quantizer: max-abs over the reduced axis, scale = fp16(max / Qmax) (1 for a channel whose scale
// is zero), code = clamp(rne(w / scale), +-Qmax).  Memory bound.  quant_once_kernel reads the weights once and keeps them in registers
// between the maximum and the codes; the kernels before it read them twice and take what its pieces do not fit.
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

// Four codes at once, packed from the lowest bits up.  The clamped product is rounded by adding 1.5 x 2^23 (to nearest even; the code is then
// the low byte of the sum), and how far it lay from the rounded value says whether the division is needed (see quant_code): seven
// instructions a value and one branch for four, where quant_code takes sixteen and a branch for each.
template <int BITS>
__device__ __forceinline__ uint32_t quant_four(const float (&w)[4], const float (&s)[4], const float (&inv)[4]) {
  constexpr float qmax = BITS == 8 ? 127.0f : 7.0f, magic = 12582912.0f;
  float t[4], far = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float q = fminf(fmaxf(w[e] * inv[e], -qmax), qmax);
    t[e] = q + magic;
    far = fmaxf(far, fabsf(q - (t[e] - magic)));
  }
  if (far > 0.5f - 1e-4f) {
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = fminf(fmaxf(__fdiv_rn(w[e], s[e]), -qmax), qmax) + magic;
  }
  uint32_t d = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) d |= (__float_as_uint(t[e]) & (BITS == 8 ? 0xFFu : 0xFu)) << (e * BITS);
  return d;
}

// Both factors of a layer in one launch, every weight read once: a workgroup holds whole channels in the registers of its 512 threads
// (4 SZ pieces of four values each, all asked for at once), takes their maxima and writes the codes from the same registers.
//   Workgroups 0 .. nu-1, U (b, q, r) with the reduced axis contiguous and codes (b, r, q): 32 channels; a wave owns four of them, a lane four
//   neighbouring values per 256 (reduce <= 256 SZ).  The four channels' codes of a value make one dword (int4: two bytes) of LDS, placed so that
//   neither the lanes that write four rows apart nor those that read a row meet in a bank; rows leave in pieces of 16 bytes.  Runs of
//   workgroups go to one XCD (workgroup w runs on XCD w % 8), so that the 32 or 16 bytes that each adds to a row of codes meet in one L2.
//   The rest, V (b, p, r) with the reduced axis strided: (4 << lg) columns, 512 >> lg row groups (reduce <= 4 SZ (512 >> lg)).
//   What a piece lies outside of is replaced by the last one inside, which moves no maximum, so that no load stands under a branch (the
//   compiler waited for every second one there).
// Why: three launches that read the factors twice took 15 + 25 + 9 us for a 4096 -> 22016 layer of rank 1024 (107 MB fp32 to int4, the pass
// 47.3 us); now 26.2 us, the time of a copy of as many bytes (with a division test and a branch per value, and V's loads under
// conditions, 43).  11008 -> 4096 in fp16 to int8 36.5 -> 17.3; a small layer, bound by the host, 25.8 -> 15.4.
struct QuantSide { const void* w; int64_t outer, reduce, inner; uint8_t* codes; f16* scales; int words; };   // words: bytes that a store of codes may take (16, 4, 1)
constexpr int QO_NT = 512, QO_CH = 32, QO_MAX_REDUCE = 1024;

template <typename T, int BITS, int SZ>
__global__ __launch_bounds__(QO_NT, 4) void quant_once_kernel(QuantSide u, uint32_t nu, uint32_t u_chunks, uint32_t u_span, QuantSide v, uint32_t v_chunks, int lg) {
  __shared__ uint32_t lds[SZ * 256 * BITS + SZ * 64 > 512 ? SZ * 256 * BITS + SZ * 64 : 512];
  constexpr float qmax = BITS == 8 ? 127.0f : 7.0f;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (blockIdx.x < nu) {
    const uint32_t item = u_span ? (blockIdx.x & 7u) * u_span + (blockIdx.x >> 3) : blockIdx.x;
    const int64_t o = item / u_chunks, q0 = (int64_t)(item - (uint32_t)o * u_chunks) * QO_CH, q = q0 + wave * 4;
    const int reduce = (int)u.reduce;
    const T* wp = reinterpret_cast<const T*>(u.w) + o * u.inner * reduce;
    float x[SZ][4][4], s[4], inv[4];                       // [256 values][channel][value]
#pragma unroll
    for (int k = 0; k < SZ; ++k)
#pragma unroll
      for (int c = 0; c < 4; ++c)                          // (reduce is a multiple of 4)
        ld_vec<T, 4>(wp + min(q + c, u.inner - 1) * reduce + min(k * 256 + lane * 4, reduce - 4), x[k][c]);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float amax = 0.0f;
#pragma unroll
      for (int k = 0; k < SZ; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(x[k][c][e]));
      for (int h = 32; h > 0; h >>= 1) amax = fmaxf(amax, __shfl_xor(amax, h, 64));
      s[c] = make_scale(amax, qmax);
      inv[c] = __builtin_amdgcn_rcpf(s[c]);
      if (lane == 0 && q + c < u.inner) u.scales[o * u.inner + q + c] = (f16)s[c];
    }
#pragma unroll
    for (int k = 0; k < SZ; ++k) {
      if (k * 256 + lane * 4 >= reduce) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float w[4] = {x[k][0][e], x[k][1][e], x[k][2][e], x[k][3][e]};
        const uint32_t d = quant_four<BITS>(w, s, inv);
        const int r = k * 256 + lane * 4 + e;
        if constexpr (BITS == 8) lds[r * 8 + (r >> 2) + wave] = d;
        else reinterpret_cast<uint16_t*>(lds)[(r * 4 + (r >> 2)) * 2 + wave] = (uint16_t)d;
      }
    }
    __syncthreads();
    constexpr int RB = QO_CH * BITS / 8, PR = RB / 16;     // bytes and 16-byte pieces that the workgroup adds to a row of codes
    const int64_t row_bytes = u.inner * BITS / 8, b0 = q0 * BITS / 8;
    uint8_t* co = u.codes + o * reduce * row_bytes + b0;
    const int left = (int)(row_bytes - b0 < RB ? row_bytes - b0 : RB);
    for (int i = tid; i < reduce * PR; i += QO_NT) {
      const int r = i / PR, pc = i - r * PR;
      const uint32_t* sp = &lds[r * (RB / 4) + (r >> 2) + pc * 4];
      const u32x4 d = {sp[0], sp[1], sp[2], sp[3]};
      uint8_t* p = co + r * row_bytes + pc * 16;
      const int n = left - pc * 16;                        // bytes of the piece inside the row
      if (u.words == 16) { if (n > 0) *reinterpret_cast<u32x4*>(p) = d; }
      else if (u.words == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) if (4 * e < n) reinterpret_cast<uint32_t*>(p)[e] = d[e];
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) if (e < n) p[e] = (uint8_t)(d[e >> 2] >> (8 * (e & 3)));
      }
    }
    return;
  }
  const uint32_t item = blockIdx.x - nu;
  const int64_t o = item / v_chunks, reduce = v.reduce, inner = v.inner;
  const int cl = tid & ((1 << lg) - 1), g = tid >> lg, ng = QO_NT >> lg;
  const int64_t c0 = (((int64_t)(item - (uint32_t)o * v_chunks) << lg) + cl) * 4;
  const bool in = c0 < inner;                              // (inner is a multiple of 4)
  const T* wc = reinterpret_cast<const T*>(v.w) + o * reduce * inner + (in ? c0 : 0);
  float x[4 * SZ][4], amax[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int k = 0; k < 4 * SZ; ++k) ld_vec<T, 4>(wc + min((int64_t)(g + k * ng), reduce - 1) * inner, x[k]);
#pragma unroll
  for (int k = 0; k < 4 * SZ; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) amax[e] = fmaxf(amax[e], fabsf(x[k][e]));
  float* s_max = reinterpret_cast<float*>(lds);            // [wave][column]
  for (int h = 1 << lg; h < 64; h <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) amax[e] = fmaxf(amax[e], __shfl_xor(amax[e], h, 64));
  if (lane < (1 << lg))
#pragma unroll
    for (int e = 0; e < 4; ++e) s_max[((wave << lg) + cl) * 4 + e] = amax[e];
  __syncthreads();
  float s[4], inv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float m = 0.0f;
#pragma unroll
    for (int w = 0; w < QO_NT / 64; ++w) m = fmaxf(m, s_max[((w << lg) + cl) * 4 + e]);
    s[e] = make_scale(m, qmax);
    inv[e] = __builtin_amdgcn_rcpf(s[e]);
  }
  if (!in) return;
  if (g == 0)
#pragma unroll
    for (int e = 0; e < 4; ++e) v.scales[o * inner + c0 + e] = (f16)s[e];
  uint8_t* co = v.codes + ((o * reduce * inner + c0) * BITS) / 8;
#pragma unroll
  for (int k = 0; k < 4 * SZ; ++k) {
    const int64_t row = g + k * ng;
    if (row >= reduce) break;
    const uint32_t d = quant_four<BITS>(x[k], s, inv);
    uint8_t* p = co + row * (inner * BITS / 8);
    if constexpr (BITS == 8) *reinterpret_cast<uint32_t*>(p) = d;     // (codes are aligned to 4 bytes)
    else *reinterpret_cast<uint16_t*>(p) = (uint16_t)d;
  }
}

// The sides that quant_once_kernel takes: whole pieces of four values, channels that fit the registers, codes on four bytes for V.
template <typename T> bool once_u_ok(const QuantSide& u) {
  return u.reduce % 4 == 0 && u.reduce <= QO_MAX_REDUCE && aligned(u.w, 4 * sizeof(T)) && u.outer * cdiv(u.inner, QO_CH) < (int64_t)1 << 30;
}
template <typename T> bool once_v_ok(const QuantSide& v) {
  return v.inner > 1 && v.inner % 4 == 0 && v.reduce <= 16 * (QO_NT >> 2) && aligned(v.w, 4 * sizeof(T)) && aligned(v.codes, 4) && v.outer * cdiv(v.inner, 16) < (int64_t)1 << 30;
}
template <typename T>
int once_launch(QuantSide u, QuantSide v, int bits, hipStream_t st) {          // a side with w == null is left out
  uint32_t nu = 0, u_chunks = 1, u_span = 0, nv = 0, v_chunks = 1;
  int lg = 4;
  if (u.w) {
    u_chunks = (uint32_t)cdiv(u.inner, QO_CH);
    nu = (uint32_t)u.outer * u_chunks;
    u_span = nu % 8 == 0 ? nu / 8 : 0;
    const int64_t row_bytes = u.inner * bits / 8;
    u.words = row_bytes % 16 == 0 && aligned(u.codes, 16) ? 16 : row_bytes % 4 == 0 && aligned(u.codes, 4) ? 4 : 1;
  }
  int sz = 1;                                              // pieces per thread: what U's reduction needs, and V's with at least 16 columns a workgroup
  while (sz < 4 && ((u.w && u.reduce > 256 * sz) || (v.w && v.reduce > 4 * sz * (QO_NT >> 2)))) sz *= 2;
  if (v.w) {
    // 64 columns a workgroup (256-byte rows of fp32), fewer where that many row groups do not hold the rows or leaves compute units without work
    while (lg > 2 && (v.reduce > 4 * sz * (QO_NT >> lg) || v.outer * cdiv(v.inner, (int64_t)4 << lg) < 256)) --lg;
    v_chunks = (uint32_t)cdiv(v.inner, (int64_t)4 << lg);
    nv = (uint32_t)v.outer * v_chunks;
  }
#define BLR_QUANT_ONCE(BITS, SZ) hipLaunchKernelGGL((quant_once_kernel<T, BITS, SZ>), dim3(nu + nv), dim3(QO_NT), 0, st, u, nu, u_chunks, u_span, v, v_chunks, lg)
  if (bits == 8) { if (sz == 1) BLR_QUANT_ONCE(8, 1); else if (sz == 2) BLR_QUANT_ONCE(8, 2); else BLR_QUANT_ONCE(8, 4); }
  else { if (sz == 1) BLR_QUANT_ONCE(4, 1); else if (sz == 2) BLR_QUANT_ONCE(4, 2); else BLR_QUANT_ONCE(4, 4); }
#undef BLR_QUANT_ONCE
  BLR_CHECK_LAUNCH("quantize");
  return BLR_OK;
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
  const QuantSide v = {w, outer, reduce, inner, codes, scales, 0};
  if (once_v_ok<T>(v)) return once_launch<T>(QuantSide{}, v, bits, st);
  // four columns a thread where rows of the weights and of the codes keep such pieces aligned
  if (inner % 4 == 0 && aligned(w, 4 * sizeof(T)) && aligned(codes, 4)) return cols_launch<T, 4>(w, outer, reduce, inner, bits, codes, scales, st);
  if (bits == 4) return cols_launch<T, 2>(w, outer, reduce, inner, bits, codes, scales, st);   // (inner is even)
  return cols_launch<T, 1>(w, outer, reduce, inner, bits, codes, scales, st);
}

template <typename T>
int quantize_turned(const T* w, int64_t outer, int64_t reduce, int64_t inner, int bits, uint8_t* codes, f16* scales, hipStream_t st) {
  const QuantSide u = {w, outer, reduce, inner, codes, scales, 0};
  if (once_u_ok<T>(u)) return once_launch<T>(u, QuantSide{}, bits, st);
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

template <typename T>
int quantize_pair(const T* wu, const T* wv, int64_t b, int64_t q, int64_t p, int64_t r, int bits, uint8_t* cu, f16* su, uint8_t* cv, f16* sv, hipStream_t st) {
  const QuantSide u = {wu, b, r, q, cu, su, 0}, v = {wv, b, p, r, cv, sv, 0};
  if (once_u_ok<T>(u) && once_v_ok<T>(v)) return once_launch<T>(u, v, bits, st);
  const int rc = quantize_turned(wu, b, r, q, bits, cu, su, st);
  return rc ? rc : quantize_any(wv, b, p, r, bits, cv, sv, st);
}

}  // namespace

int quantize_pair_launch(const void* U, const void* V, int dtype, int64_t b, int64_t q, int64_t p, int64_t r, int bits,
                         void* u_codes, void* u_scales, void* v_codes, void* v_scales, hipStream_t st) {
  uint8_t* cu = (uint8_t*)u_codes; uint8_t* cv = (uint8_t*)v_codes; f16* su = (f16*)u_scales; f16* sv = (f16*)v_scales;
  if (dtype == BLR_F32) return quantize_pair((const float*)U, (const float*)V, b, q, p, r, bits, cu, su, cv, sv, st);
  if (dtype == BLR_F16) return quantize_pair((const f16*)U, (const f16*)V, b, q, p, r, bits, cu, su, cv, sv, st);
  return quantize_pair((const bf16*)U, (const bf16*)V, b, q, p, r, bits, cu, su, cv, sv, st);
}

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
