// What a transformer block does between its structured linears (DiT): adaLN's projection of the conditioning, its
// normalise-and-modulate, and attention.
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

// ---- out = softmax(q k^T / sqrt(D)) v over the packed result of the qkv linear (reference DiT/models.py:108, timm's Attention) ---
// qkv (image, token, 3, head, D) is read where the linear left it and out (image, token, head, D) written as the projection reads
// it, so nothing is permuted in memory.  Heads of 64 or 72 values over a few hundred tokens: the arithmetic is small (4.8 GFLOP at
// 16 images of 256 tokens), what counts is to have the chip full and little between the products.  A workgroup takes 128 queries
// of a head, 32 a wave, and walks the keys 64 at a time through LDS (the next 64 on their way into registers meanwhile).  Both
// products are turned, S^T = K Q^T and O^T = V^T P^T: a query then is one lane's column of the 32 x 32 results, so that maximum
// and sum are over a lane's own registers (and the lane 32 further), and the probabilities are the second product's operand as
// they lie.  The contraction over keys may take them in any order: the operand's slot j of half h is key 4 h + j (j < 4) or
// 8 + 4 h + j - 4 of its sixteen, the order in which the first product leaves them; V^T is read from LDS in the same order.
// D = 72 takes 80 (K) and 96 (V) padded values.  Probabilities go to the second product in T as in any flash attention; sums,
// maxima and results are fp32.  An XCD takes a contiguous run of workgroups, an image's heads one after the other: a head's 144
// (128) bytes of a token share cache lines with its neighbours', and an image's 1.8 MB stay in that XCD's L2, where heads dealt out over
// the XCDs fetched nearly twice the bytes.  16 images x 16 heads x 256 tokens x 72, fp16: 58 us in torch's
// kernel, 17.7 with heads dealt out, 16.2 us here (64 images 66.1 -> 62.8); one image alone takes 9.3: loads, exponentials and products of
// a step follow one another in a wave.
template <typename T, int D>
__global__ __launch_bounds__(256, 2) void attention_kernel(const T* __restrict__ qkv, T* __restrict__ out, int N, int H, int q_tiles, int per_xcd, int total, float scale_log2e) {
  using V8 = typename TypeTraits<T>::vec8;
  using V4 = typename TypeTraits<T>::vec4;
  constexpr int KT = 64, D8 = D / 8, DK = (D + 15) / 16, DT = (D + 31) / 32;
  constexpr int KS = D8 % 2 ? D : D + 8;           // row of K in LDS: an odd number of 16-byte pieces, sixteen rows cover all banks
  constexpr int VS = KT + 4;                       // row of V^T: 34 words, 32 rows of 8 bytes cover all banks
  constexpr int NK = (KT * D8 + 255) / 256, QUADS = KT / 4;
  static_assert(D % 8 == 0 && QUADS * D8 <= 256, "one piece of V a thread");
  __shared__ __align__(16) T ks[KT * KS];
  __shared__ __align__(16) T vt[DT * 32 * VS];     // (rows past D are read into results that nobody stores)
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
  const unsigned wg = (blockIdx.x & 7) * (unsigned)per_xcd + (blockIdx.x >> 3);
  if (wg >= (unsigned)total) return;
  const unsigned qt = wg % (unsigned)q_tiles, head = wg / (unsigned)q_tiles;
  const int h = (int)(head % (unsigned)H), img = (int)(head / (unsigned)H);
  const int q0 = (int)qt * 128 + (tid >> 6) * 32;
  const int64_t ld = (int64_t)3 * H * D;
  const T* base = qkv + (int64_t)img * N * ld + (int64_t)h * D;
  const bool live = q0 < N;                        // waves past the last query only help to load
  V8 zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero[e] = (T)0.0f;

  V8 q[DK];
  const T* qr = base + (int64_t)min(q0 + col, N - 1) * ld;
#pragma unroll
  for (int t = 0; t < DK; ++t) {
    const int d = 16 * t + 8 * half;
    q[t] = d < D ? ldg16<V8>(qr + (d < D ? d : 0)) : zero;
  }

  const int vq = tid / D8, vo = tid % D8;          // this thread's piece of V: four keys, eight values
  V8 kr[NK], vr[4];
  auto load = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int idx = tid + i * 256, key = idx / D8, o = idx % D8;
      kr[i] = zero;
      if (idx < KT * D8 && kt + key < N) kr[i] = ldg16<V8>(base + (int64_t)(kt + key) * ld + (int64_t)H * D + o * 8);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      vr[e] = zero;
      if (vq < QUADS && kt + 4 * vq + e < N) vr[e] = ldg16<V8>(base + (int64_t)(kt + 4 * vq + e) * ld + (int64_t)2 * H * D + vo * 8);
    }
  };

  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
  float m = -INFINITY, l = 0.0f;
  load(0);
  for (int kt = 0; kt < N; kt += KT) {
    __syncthreads();                               // the keys before these have been used
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int idx = tid + i * 256;
      if (idx < KT * D8) *reinterpret_cast<V8*>(ks + (idx / D8) * KS + (idx % D8) * 8) = kr[i];
    }
    if (vq < QUADS)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const V4 four = {vr[0][e], vr[1][e], vr[2][e], vr[3][e]};
        *reinterpret_cast<V4*>(vt + (vo * 8 + e) * VS + vq * 4) = four;
      }
    __syncthreads();
    if (kt + KT < N) load(kt + KT);
    if (!live) continue;

    f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = 0.0f;
#pragma unroll
      for (int t = 0; t < DK; ++t) {
        const int d = 16 * t + 8 * half;
        const V8 a = ldg16<V8>(ks + (kb * 32 + col) * KS + (d < D ? d : 0));
        s[kb] = TypeTraits<T>::mfma32(d < D ? a : zero, q[t], s[kb]);
      }
    }
    if (kt + KT > N)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (kt + kb * 32 + 8 * (i / 4) + 4 * half + i % 4 >= N) s[kb][i] = -INFINITY;
    float top = m;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) top = fmaxf(top, s[kb][i]);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float at = top == -INFINITY ? 0.0f : top * scale_log2e;      // (nothing but minus infinity so far: every term is 0)
    const float fade = __builtin_amdgcn_exp2f(m * scale_log2e - at);
    m = top;
    l *= fade;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[kb][i] = __builtin_amdgcn_exp2f(fmaf(s[kb][i], scale_log2e, -at));
        l += s[kb][i];
      }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] *= fade;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int ts = 0; ts < 2; ++ts) {
        V8 p;
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = TypeTraits<T>::from_f32(s[kb][8 * ts + j]);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const T* vp = vt + (dt * 32 + col) * VS + kb * 32 + 16 * ts + 4 * half;
          const V4 a = *reinterpret_cast<const V4*>(vp), b = *reinterpret_cast<const V4*>(vp + 8);
          o[dt] = TypeTraits<T>::mfma32(__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7), p, o[dt]);
        }
      }
  }
  l += __shfl_xor(l, 32, 64);
  if (q0 + col >= N) return;
  const float inv = 1.0f / l;
  T* orow = out + (((int64_t)img * N + q0 + col) * H + h) * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = dt * 32 + 8 * g;
      if (d >= D) continue;
      V4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = TypeTraits<T>::from_f32(o[dt][4 * g + i] * inv);
      *reinterpret_cast<V4*>(orow + d + 4 * half) = v;
    }
}

template <typename T>
int attention(const void* qkv, void* out, int images, int N, int H, int D, hipStream_t st) {
  const int q_tiles = (int)cdiv(N, 128);
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)D);
  const int total = (int)((int64_t)images * H * q_tiles), per_xcd = (int)cdiv(total, 8);
  const dim3 grid((unsigned)per_xcd * 8);
  if (D == 72) hipLaunchKernelGGL((attention_kernel<T, 72>), grid, dim3(256), 0, st, (const T*)qkv, (T*)out, N, H, q_tiles, per_xcd, total, scale_log2e);
  else hipLaunchKernelGGL((attention_kernel<T, 64>), grid, dim3(256), 0, st, (const T*)qkv, (T*)out, N, H, q_tiles, per_xcd, total, scale_log2e);
  BLR_CHECK_LAUNCH("attention");
  return BLR_OK;
}

// ---- out = silu(c) W^T + bias for the few rows of the conditioning (reference DiT/models.py:113-116: SiLU, then nn.Linear) -----
// Bound by the weights (1152 -> 6912 in fp16: 15.9 MB) and by latency, since nothing else is in flight beside it: 32 output columns
// a workgroup, so that 6912 columns are 216 workgroups, their reduction cut over eight waves that each have all their operands on
// the way (BATCH pieces of 32 values) before the first product.  16 rows of c are one matrix-core operand; silu is applied to it
// on the way in, rounded to T as the separate operator does, while the weights arrive (16 columns a workgroup and four waves do
// twice the exponentials for the same weights: 11.5 us); sums in fp32.  16 rows, fp16: silu 4.9 and
// the product 9.0 us as torch's two kernels, 8.8 us here.
template <typename T>
__global__ __launch_bounds__(512) void silu_linear_kernel(const T* __restrict__ c, int64_t ldc, const T* __restrict__ W, const T* __restrict__ bias, T* __restrict__ out,
                                                          int M, int N, int K) {
  using V8 = typename TypeTraits<T>::vec8;
  using V4 = typename TypeTraits<T>::vec4;
  constexpr int BATCH = 5, WAVES = 8;
  __shared__ f32x4 part[WAVES][2][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, quarter = lane >> 4;
  const int n0 = blockIdx.x * 32;
  const T* w0 = W + (int64_t)min(n0 + l16, N - 1) * K;
  const T* w1 = W + (int64_t)min(n0 + 16 + l16, N - 1) * K;
  const T* cr = c + (int64_t)min(l16, M - 1) * ldc;
  const int steps = (K + 31) / 32, each = (steps + WAVES - 1) / WAVES, first = wave * each, last = min(steps, first + each);
  V8 zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero[e] = (T)0.0f;
  f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
  for (int s0 = first; s0 < last; s0 += BATCH) {
    V8 x[BATCH], w[2][BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {              // (past the end: the row's start, not used)
      const int k = (s0 + i) * 32 + quarter * 8, at = s0 + i < last && k < K ? k : 0;
      x[i] = ldg16<V8>(cr + at);
      w[0][i] = ldg16<V8>(w0 + at);
      w[1][i] = ldg16<V8>(w1 + at);
    }
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const bool in = s0 + i < last && (s0 + i) * 32 + quarter * 8 < K;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[i][e] = TypeTraits<T>::from_f32(apply_act(TypeTraits<T>::to_f32(x[i][e]), BLR_ACT_SILU));
      x[i] = in ? x[i] : zero;
    }
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const bool in = s0 + i < last && (s0 + i) * 32 + quarter * 8 < K;
      acc[0] = TypeTraits<T>::mfma16(in ? w[0][i] : zero, x[i], acc[0]);
      acc[1] = TypeTraits<T>::mfma16(in ? w[1][i] : zero, x[i], acc[1]);
    }
  }
  part[wave][0][lane] = acc[0];
  part[wave][1][lane] = acc[1];
  __syncthreads();
  if (wave >= 2) return;
  f32x4 sum = part[0][wave][lane];
#pragma unroll
  for (int i = 1; i < WAVES; ++i) sum += part[i][wave][lane];
  const int n = n0 + 16 * wave + 4 * quarter;      // (N in whole quarters: a lane's four columns are inside or not)
  if (l16 >= M || n >= N) return;
  V4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = TypeTraits<T>::from_f32(sum[i] + (bias ? TypeTraits<T>::to_f32(bias[n + i]) : 0.0f));
  *reinterpret_cast<V4*>(out + (int64_t)l16 * N + n) = o;
}

template <typename T>
int silu_linear(const void* c, int64_t ldc, const void* W, const void* bias, void* out, int M, int N, int K, hipStream_t st) {
  hipLaunchKernelGGL((silu_linear_kernel<T>), dim3((unsigned)cdiv(N, 32)), dim3(512), 0, st, (const T*)c, ldc, (const T*)W, (const T*)bias, (T*)out, M, N, K);
  BLR_CHECK_LAUNCH("silu_linear");
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

int blr_attention_qkv(const void* qkv, void* out, int images, int tokens, int heads, int head_dim, int dtype, void* stream) {
  if (!qkv || !out) { set_error("attention: null pointer"); return BLR_ERR_BAD_ARG; }
  if (images <= 0 || tokens <= 0 || heads <= 0 || head_dim <= 0) { set_error("attention: bad size"); return BLR_ERR_BAD_ARG; }
  if ((dtype != BLR_F16 && dtype != BLR_BF16) || (head_dim != 64 && head_dim != 72) || tokens > (1 << 20) || !aligned(qkv, 16) || !aligned(out, 16) ||
      (double)images * heads * (double)cdiv(tokens, 128) > 2147483647.0) {
    set_error("attention: needs f16 / bf16, heads of 64 or 72 values, at most 2^20 tokens, 16-byte aligned operands");
    return BLR_ERR_UNSUPPORTED;
  }
  return dtype == BLR_F16 ? attention<f16>(qkv, out, images, tokens, heads, head_dim, (hipStream_t)stream)
                          : attention<bf16>(qkv, out, images, tokens, heads, head_dim, (hipStream_t)stream);
}

int blr_silu_linear(const void* c, int64_t ldc, const void* W, const void* bias, void* out, int rows, int out_f, int in_f, int dtype, void* stream) {
  if (!c || !W || !out) { set_error("silu_linear: null pointer"); return BLR_ERR_BAD_ARG; }
  if (rows <= 0 || out_f <= 0 || in_f <= 0 || ldc < in_f) { set_error("silu_linear: bad size"); return BLR_ERR_BAD_ARG; }
  if ((dtype != BLR_F16 && dtype != BLR_BF16) || rows > 16 || in_f % 8 || ldc % 8 || out_f % 4 || !aligned(c, 16) || !aligned(W, 16) || !aligned(out, 8)) {
    set_error("silu_linear: needs f16 / bf16, at most 16 rows, inputs in whole 16-byte pieces, outputs in whole 8-byte pieces");
    return BLR_ERR_UNSUPPORTED;
  }
  return dtype == BLR_F16 ? silu_linear<f16>(c, ldc, W, bias, out, rows, out_f, in_f, (hipStream_t)stream)
                          : silu_linear<bf16>(c, ldc, W, bias, out, rows, out_f, in_f, (hipStream_t)stream);
}

}  // extern "C"
