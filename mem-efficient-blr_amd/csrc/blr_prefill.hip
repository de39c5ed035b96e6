// BLAST above 16 rows: the kernels around the products.
//
//   Z[i][m][r] = sum_j S(i, j, r) * Y_j[m][r],      Y_j = x_j V_j   (x_j: columns j P .. (j+1) P of x, V_j (P, R)),      out_i = Z_i U_i
//
// For one rank r the mix is a 16 x 16 product over the input blocks, Z_r (i, m) = S_r (i, j) Y_r (j, m): one matrix instruction per rank and 16
// rows.  blast_mixm_kernel is the mix alone, blast_ymix_kernel forms Y_j in the compute unit for narrow input blocks, blast_ymixw_kernel for
// wide ones, blast_mixu_kernel continues with the product with U where output blocks are narrow, and blast_one_kernel does all three.
#include <hip/hip_runtime.h>
#include <cmath>
#include <type_traits>
#include "blr_common.h"
#include "blr_decode_dev.h"
#include "blr_ring_dev.h"

namespace blr {

namespace {
constexpr uint32_t YM_OOB = 0x80000000u;
}  // namespace

#ifdef BLR_TRACE
__device__ unsigned long long g_trace6[1024 * 16];
#define TR6(i) do { if (threadIdx.x == 0 && blockIdx.x < 1024) g_trace6[blockIdx.x * 16 + (i)] = wall_clock64(); } while (0)
#else
#define TR6(i) do {} while (0)
#endif

template <typename T> struct YmDot;
template <> struct YmDot<f16> {
  static __device__ __forceinline__ f32x4 mfma16(u32x2 a, u32x2 b, f32x4 c) {      // 16 x 16 x 16
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct YmDot<bf16> {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x4 mfma16(u32x2 a, u32x2 b, f32x4 c) {      // 16 x 16 x 16
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

template <typename T>
__device__ __forceinline__ uint32_t ym_pack(float lo, float hi) {
  typename TypeTraits<T>::vec4 v;      // (only two lanes used; a two-element vector of T has no common name here)
  v[0] = TypeTraits<T>::from_f32(lo); v[1] = TypeTraits<T>::from_f32(hi); v[2] = v[0]; v[3] = v[0];
  return __builtin_bit_cast(u32x2, v)[0];
}

// a barrier that orders LDS and leaves loads and stores of memory in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- the mix on its own: Z_i = sum_j S(i, j, r) Y_j for two-byte types, 4 / 8 / 12 / 16 blocks, ranks in pieces of eight -------------------------
// For one rank the mix is a b x b product with the rows: one 16 x 16 x 16 matrix instruction per rank and 16 rows, as in the kernels around it, which
// leaves the kernel to the memory: Y once in, Z once out.  (The kernels in blr_gemm.hip do it on the vector units, b x 8 multiply-adds per
// 16 bytes: with the arithmetic of bf16 in fp32 that was what bound them.)  A workgroup of eight waves takes 32 rows x 64 ranks of all blocks:
// whole 128-byte lines straight into LDS, 64 KB for 16 blocks, so two workgroups share a compute unit and one's loads run under the other's
// stores.  Wave w owns ranks 8 w .. 8 w + 7.  Lane (n, g) reads Y_j, j = 4 g .. 4 g + 3, of row n - 16 bytes are its eight ranks -, turns them
// into one operand per rank (byte permutes), and its products are Z_i, i = 4 g .. 4 g + 3, of the same row and ranks: they go back where
// the lane read Y.  Nothing crosses waves but the loads and the stores of whole rows on either side.  S is kept in registers along the row tiles
// that a workgroup walks; with the rank contiguous it comes through the same LDS, as (r, i, j) straight in operand order, and in any other order or off its
// boundary (MIXM_ANY) through LDS as well, an element at a time - once per rank tile.  Every size and every S is taken, so the sums are fp32 for all of them (the kernels in blr_gemm.hip sum in fp16 for fp16): whole calls
// with S one element off, there -> here, 4096 -> 4096, r = 512 at 1000 / 2048 rows 58.5 / 72.1 -> 35.6 / 53.8 us, 4096 -> 22016, r = 1024 in bf16 224 -> 152.
// 16 blocks, r = 1024 at 2048 rows (134 MB in and out): 32.9 -> 24.4 us = 5.5 TB/s, the rate of a device copy; bf16 24.6.
struct MixmParams {
  const void* Y; const void* S; void* Z;
  int M, b, R;
  int64_t s_si, s_sj, s_sr;     // strides of S (RIJ: not used)
  int nmt;                      // row tiles
  int items;                    // rank tiles x row tiles
};
// eight ranks x four blocks: v[t] = 8 ranks of block t -> one operand (four blocks) per rank
__device__ __forceinline__ void mixm_turn(const u32x4 (&v)[4], u32x2 (&o)[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
    o[q][0] = __builtin_amdgcn_perm(v[1][q >> 1], v[0][q >> 1], sel);
    o[q][1] = __builtin_amdgcn_perm(v[3][q >> 1], v[2][q >> 1], sel);
  }
}
enum { MIXM_RIJ = 0, MIXM_RUN, MIXM_ANY };
template <typename T, int ORDER>
__global__ __launch_bounds__(512, 4) void blast_mixm_kernel(MixmParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char mx_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4, b = p.b, M = p.M, R = p.R;
  const uint32_t wg = xcd_item(blockIdx.x, gridDim.x), G = gridDim.x;
  uint32_t item = (uint32_t)((uint64_t)wg * (uint32_t)p.items / G);
  const uint32_t item_end = (uint32_t)((uint64_t)(wg + 1) * (uint32_t)p.items / G);
  const uint32_t lds0 = ring_lds_addr(mx_lds);
  // piece c of row r (128 bytes) of a plane lies at c ^ ((r >> 1) & 7): 16 rows' pieces of one number then lie in different banks
  const int r8 = lane >> 3;                            // a load or store instruction of a wave: eight rows, eight lanes each
  const bool live = 4 * g < b;                         // (4 g + 3 < b as well: b is a multiple of four)
  u32x2 sa[8];
  bool fresh = true;                                   // S of this rank tile is not in registers yet
  int rt = (int)(item / (uint32_t)p.nmt), mt = (int)(item - (uint32_t)rt * (uint32_t)p.nmt);
  for (; item < item_end; ++item) {
    const int m0 = mt * 32, r0 = rt * 64;
    const int piece = r0 + wave * 8;
    if (fresh) {
      if constexpr (ORDER == MIXM_RIJ) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          sa[q] = u32x2{0u, 0u};
          if (live && n < b && piece < R) sa[q] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const T*>(p.S) + ((int64_t)(piece + q) * b + n) * b + 4 * g);
        }
      } else {                                         // rows (i, j) of the tile's 64 ranks, i b + j; b b is a multiple of 16
        for (int k = wave; k * 8 < b * b; k += 8) {
          const int row = k * 8 + r8, i = row / b, j = row - i * b, c = (lane & 7) ^ ((row >> 1) & 7);
          if constexpr (ORDER == MIXM_ANY) {
            const T* src = reinterpret_cast<const T*>(p.S) + i * p.s_si + j * p.s_sj + min(r0 + c * 8, R - 8) * p.s_sr;
            typename TypeTraits<T>::vec8 v;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[e * p.s_sr];
            *reinterpret_cast<typename TypeTraits<T>::vec8*>(mx_lds + k * 1024 + lane * 16) = v;
          } else {
            ring_load_lds(p.S, (uint32_t)((i * p.s_si + j * p.s_sj + min(r0 + c * 8, R - 8)) * 2), lds0 + k * 1024);
          }
        }
        __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));
        lds_barrier();
        u32x4 v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int row = n * b + 4 * g + t;
          v[t] = u32x4{0u, 0u, 0u, 0u};
          if (live && n < b) v[t] = *reinterpret_cast<const u32x4*>(mx_lds + row * 128 + ((wave ^ ((row >> 1) & 7)) << 4));
        }
        mixm_turn(v, sa);
        lds_barrier();                                 // read by every wave
      }
    }
    // in: four instructions a plane, a wave the same eight rows of every second plane
    {
      const int row = (wave & 3) * 8 + r8, c = (lane & 7) ^ ((row >> 1) & 7);
      const uint32_t off = (uint32_t)(min(row, M - 1 - m0) * R + min(c * 8, R - 8 - r0)) * 2u;
      const T* y = reinterpret_cast<const T*>(p.Y) + ((int64_t)(wave >> 2) * M + m0) * R + r0;
      for (int k = wave; k < 4 * b; k += 8, y += (int64_t)2 * M * R) ring_load_lds(y, off, lds0 + k * 1024);
    }
    __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));         // (S of this tile as well)
    lds_barrier();
#pragma unroll
    for (int mg = 0; mg < 2; ++mg) {
      unsigned char* const at = mx_lds + 4 * g * 4096 + (mg * 16 + n) * 128 + ((wave ^ ((n >> 1) & 7)) << 4);
      u32x4 v[4];
      u32x2 yb[8];
      f32x4 d[8];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        v[t] = u32x4{0u, 0u, 0u, 0u};
        if (live) v[t] = *reinterpret_cast<const u32x4*>(at + t * 4096);
      }
      mixm_turn(v, yb);
#pragma unroll
      for (int q = 0; q < 8; ++q) d[q] = YmDot<T>::mfma16(sa[q], yb[q], f32x4{0.f, 0.f, 0.f, 0.f});
      if (live) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          *reinterpret_cast<u32x4*>(at + t * 4096) = u32x4{ym_pack<T>(d[0][t], d[1][t]), ym_pack<T>(d[2][t], d[3][t]), ym_pack<T>(d[4][t], d[5][t]), ym_pack<T>(d[6][t], d[7][t])};
      }
    }
    lds_barrier();
    for (int k = wave; k < 4 * b; k += 8) {
      const int row = (k & 3) * 8 + r8, c = (lane & 7) ^ ((row >> 1) & 7);
      const u32x4 z = *reinterpret_cast<const u32x4*>(mx_lds + k * 1024 + lane * 16);
      if (m0 + row < M && r0 + c * 8 < R) *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(p.Z) + ((int64_t)(k >> 2) * M + m0 + row) * R + r0 + c * 8) = z;
    }
    lds_barrier();                                     // the rows have been read: the next tile may land
    fresh = ++mt == p.nmt;
    if (fresh) { mt = 0; ++rt; }
  }
}

// Returns BLR_OK, a negative blr_status, or 1 when the kernel does not take the operands.
int blast_mixm_launch(const void* Y, const void* S, void* Z, int M, int b, int R, int64_t s_si, int64_t s_sj, int64_t s_sr, int dtype, hipStream_t st) {
  if ((dtype != BLR_F16 && dtype != BLR_BF16) || b < 4 || b > 16 || b % 4 || R % 8 || !aligned(Y, 16) || !aligned(Z, 16)) return 1;
  const int64_t lim = (int64_t)1 << 31;
  const int nrt = (int)cdiv(R, 64), nmt = (int)cdiv(M, 32);
  if (R >= 1 << 25 || (int64_t)nrt * nmt >= lim) return 1;                         // (the rows of a tile lie within 32 bits)
  const bool rij = s_sj == 1 && s_si == b && s_sr == (int64_t)b * b && aligned(S, 8);
  const bool run = s_sr == 1 && s_si % 8 == 0 && s_sj % 8 == 0 && s_si >= 0 && s_sj >= 0 && aligned(S, 16) && ((b - 1) * (s_si + s_sj) + R) * 2 < lim;
  MixmParams p = {};
  p.Y = Y; p.S = S; p.Z = Z; p.M = M; p.b = b; p.R = R; p.s_si = s_si; p.s_sj = s_sj; p.s_sr = s_sr;
  p.nmt = nmt;
  p.items = nrt * nmt;
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const unsigned grid = (unsigned)(p.items < 2 * cus ? p.items : 2 * cus);
  void* const fns[6] = {(void*)blast_mixm_kernel<f16, MIXM_RIJ>, (void*)blast_mixm_kernel<f16, MIXM_RUN>, (void*)blast_mixm_kernel<f16, MIXM_ANY>,
                        (void*)blast_mixm_kernel<bf16, MIXM_RIJ>, (void*)blast_mixm_kernel<bf16, MIXM_RUN>, (void*)blast_mixm_kernel<bf16, MIXM_ANY>};
  void* args[] = {&p};
  const hipError_t e = hipLaunchKernel(fns[(dtype == BLR_F16 ? 0 : 3) + (rij ? MIXM_RIJ : run ? MIXM_RUN : MIXM_ANY)], dim3(grid), dim3(512), args, (size_t)b * 4096, st);
  if (e != hipSuccess) { set_error("blast_mixm: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  return BLR_OK;
}

// ---- Z = mix(S, x V) in one launch for narrow input blocks ----------------------------------------------------------------------------------------
// The tile and the mix of blast_mixm_kernel, with Y made on the spot: 32 rows (16 where that leaves compute units idle) x 64 ranks of all blocks.  Four waves, wave w makes Y_j for j = w, w + 4, ..:
// the block's 32 rows of x and its rows of V, at most 96 columns of the block at a time, come as whole lines into a piece of LDS of the wave's
// own and from there - V through transposing reads - into registers, whereupon the next block's loads go out under the products.  Nothing waits for
// another wave until all of Y is in registers (16 per block); then Y goes to LDS, over what the blocks came through, and the mix and the way out are
// those of blast_mixm_kernel.  64 - 80 KB of LDS: two workgroups share a compute unit and fill each other's waits.
// What bounds it: a wave's chain of trips to the L2, one per block, and the chip's write rate (4096 rows, 16 blocks of 72, r = 576: 75 MB out).  Before, a
// workgroup of eight waves held 32 rows x 96 - 128 ranks in 150 KB of LDS, read x and V straight into registers, 60 loads of half lines a
// wave and tile, and had its compute unit to itself.  Whole calls, before -> now: 1152 -> 4608, r = 576 at 2000 / 4096 rows 43.0 / 69.5 -> 38.4 / 63.4 us,
// 1024 -> 8192, r = 512 45.0 / 74.8 -> 37.4 / 64.0, 2048 -> 8192, r = 768 at 4096 127.1 -> 113.9, 768 -> 3072, r = 1000 99.4 -> 86.8, 512 -> 2048 in 4 blocks, r = 512
// 32.5 -> 28.2; 0.93 x in the mean over 49 calls of 12 layers at 150 .. 4096 rows, 1.05 x at worst (768 -> 3072, r = 1000 at 600 rows).
struct YmixParams {
  MixmParams m;                 // Y not used
  const void* x; int64_t ldx; const void* V;
  int P, PP;                    // columns of a block, and of a piece of it (a multiple of 8, at most 96)
  int slot;                     // bytes of LDS of a wave
  FastDiv cl;                   // chunks of a row of x in LDS
};
template <typename T, bool RIJ, int NB, int KS, int RX>   // NB = b / 4; KS: steps of 32 columns that cover a piece; RX: tiles of 16 RX rows
__global__ __launch_bounds__(256, 2) void blast_ymix_kernel(YmixParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char ym_lds[];
  using V8 = typename TypeTraits<T>::vec8;
  constexpr int b = 4 * NB, ROWS = 16 * RX, PLANE = ROWS * 128, NZ = 2 * RX * NB;   // PLANE: a block's Y in LDS; NZ: the pieces of Z that a wave stores
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int n = lane & 15, g = lane >> 4;
  const int M = p.m.M, R = p.m.R, P = p.P, PP = p.PP;
  const uint32_t wg = xcd_item(blockIdx.x, gridDim.x), G = gridDim.x;
  uint32_t item = (uint32_t)((uint64_t)wg * (uint32_t)p.m.items / G);
  const uint32_t item_end = (uint32_t)((uint64_t)(wg + 1) * (uint32_t)p.m.items / G);
  int r8 = lane >> 3;
  const bool live = g < NB;
  // x of a block: the rows' cl chunks of 16 bytes, cl odd (16 rows' chunks of one number then lie in different banks); V behind it as it lies,
  // chunk c of row k at c ^ (k & 2) << 1 ^ (k & 8) >> 2 (see the (k, n) stages of blr_gemm_wide.hip)
  const int cl = (PP / 8) | 1, xi = (RX * cl + 3) / 4;      // 16 RX cl chunks, in KiB
  unsigned char* const own = ym_lds + wave * p.slot;
  const uint32_t own0 = ring_lds_addr(own), lds0 = ring_lds_addr(ym_lds);
  u32x2 sa[2][8];
  uint32_t rt_have = ~0u;
  int m0, r0;
  constexpr int XI = RX * KS + 1;                      // (at most: 16 RX (4 KS + 1) chunks)
  uint32_t v_off[2], x_off[XI];                        // v_off: rows 0 .. 7 of an even and of an odd group of eight
  auto ask = [&](int j, int k0) {                      // columns k0 .. k0 + PP - 1 of block j
    const char* xb = reinterpret_cast<const char*>(p.x) + ((int64_t)m0 * p.ldx + (int64_t)j * P + k0) * 2;
    const char* vb = reinterpret_cast<const char*>(p.V) + ((int64_t)j * P + k0) * R * 2;
#pragma unroll
    for (int i = 0; i < XI; ++i)
      if (i < xi) ring_load_lds(xb, x_off[i], own0 + i * 1024);
#pragma clang loop unroll(disable)
    for (int i = 0; i * 8 < PP; ++i) ring_load_lds(vb + (int64_t)i * 16 * R, v_off[i & 1], own0 + (xi + i) * 1024);
  };
  auto begin = [&]() {                                 // a tile: S if its ranks are new, and the wave's first piece is asked for
    asm volatile("" : "+v"(n), "+v"(g), "+v"(r8));   // addresses are formed again for each tile: kept, they would not fit beside Y
    const uint32_t rt = item / (uint32_t)p.m.nmt;                            // (once a tile: any number of tiles, where the quick division has a limit)
    m0 = (int)(item - rt * (uint32_t)p.m.nmt) * ROWS;
    r0 = (int)rt * 64;
    if (rt != rt_have) {
      rt_have = rt;
      if constexpr (RIJ) {
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int r = r0 + (wave + 4 * cc) * 8 + q;
            sa[cc][q] = u32x2{0u, 0u};
            if (live && n < b && r < R) sa[cc][q] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const T*>(p.m.S) + ((int64_t)r * b + n) * b + 4 * g);
          }
      } else {
        for (int k = wave; k * 8 < b * b; k += 4) {
          const int row = k * 8 + r8, i = row / b, j = row - i * b, c = (lane & 7) ^ ((row >> 1) & 7);
          ring_load_lds(p.m.S, (uint32_t)((i * p.m.s_si + j * p.m.s_sj + min(r0 + c * 8, R - 8)) * 2), lds0 + k * 1024);
        }
        __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));
        lds_barrier();
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          u32x4 v[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int row = n * b + 4 * g + t;
            v[t] = u32x4{0u, 0u, 0u, 0u};
            if (live && n < b) v[t] = *reinterpret_cast<const u32x4*>(ym_lds + row * 128 + (((wave + 4 * cc) ^ ((row >> 1) & 7)) << 4));
          }
          mixm_turn(v, sa[cc]);
        }
        lds_barrier();
      }
    }
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const int c = (lane & 7) ^ ((r8 & 2) << 1 | o << 1);
      v_off[o] = (uint32_t)((r8 * R + min(r0 + c * 8, R - 8)) * 2);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const uint32_t L = min(i * 64 + r8 * 8 + (int)(lane & 7), ROWS * cl - 1), row = fd_div(L, p.cl);
      x_off[i] = (uint32_t)min((int)row, M - 1 - m0) * (uint32_t)(p.ldx * 2) + min(L - row * cl, (uint32_t)PP / 8 - 1) * 16;
      asm volatile("" : "+v"(x_off[i]));
    }
    ask(wave, 0);
  };
  if (item >= item_end) return;
  begin();
  int stores = 0;                                      // whether the NZ stores of the tile before are younger than the loads
  for (;;) {
    u32x2 y[NB][4][RX];
#pragma unroll
    for (int jb = 0; jb < NB; ++jb) {
      f32x4 acc[4][RX];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int x = 0; x < RX; ++x) acc[c][x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
      for (int at = 0; at < P; at += PP) {             // a last piece that would end past the block begins earlier: what the one before had of it is zero
        asm volatile("" : "+v"(n), "+v"(g));
        const int skip = max(at + PP - P, 0);
        V8 xf[KS][RX], vf[KS][4];
        ring_wait_loads<NZ>(stores);
        stores = 0;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const int kc = min(4 * s + g, PP / 8 - 1);                               // the lane's eight k, or the last ones there are
#pragma unroll
          for (int x = 0; x < RX; ++x) xf[s][x] = *reinterpret_cast<const V8*>(own + ((16 * x + n) * cl + kc) * 16);
          const int k = 8 * kc + (n >> 2), swz = (k & 2) << 1 | (k & 8) >> 2;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            union { V8 v; s16x4 h[2]; } w;
            const unsigned char* src = own + xi * 1024 + k * 128 + (((2 * c + ((n & 3) >> 1)) ^ swz) << 4) + (n & 1) * 8;
            w.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(src));
            w.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(src + 512));
            vf[s][c] = w.v;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        {                                              // the piece is in registers: the next one may come
          const int j = at + PP < P ? wave + 4 * jb : wave + 4 * (jb + 1);
          if (j < b) ask(j, at + PP < P ? min(at + PP, P - PP) : 0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          if (32 * s + 8 * g >= PP || 32 * s + 8 * g < skip) {                     // zero on both sides
#pragma unroll
            for (int x = 0; x < RX; ++x) xf[s][x] = V8{};
#pragma unroll
            for (int c = 0; c < 4; ++c) vf[s][c] = V8{};
          }
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int x = 0; x < RX; ++x) acc[c][x] = TypeTraits<T>::mfma16(vf[s][c], xf[s][x], acc[c][x]);
        }
      }
      // acc[c][x]: row 16 x + n, ranks 16 c + 4 g .. + 3
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int x = 0; x < RX; ++x) y[jb][c][x] = u32x2{ym_pack<T>(acc[c][x][0], acc[c][x][1]), ym_pack<T>(acc[c][x][2], acc[c][x][3])};
    }
    lds_barrier();                                     // nobody reads x and V any more
#pragma unroll
    for (int jb = 0; jb < NB; ++jb)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int x = 0; x < RX; ++x) {
          const int m = 16 * x + n;
          *reinterpret_cast<u32x2*>(ym_lds + (wave + 4 * jb) * PLANE + m * 128 + (((2 * c + (g >> 1)) ^ ((m >> 1) & 7)) << 4) + (g & 1) * 8) = y[jb][c][x];
        }
    lds_barrier();
    // ---- the mix and the way out, as above, with two pieces of eight ranks a wave ----
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int mg = 0; mg < RX; ++mg) {
        __builtin_amdgcn_sched_barrier(0);
        unsigned char* const at = ym_lds + 4 * g * PLANE + (mg * 16 + n) * 128 + (((wave + 4 * cc) ^ ((n >> 1) & 7)) << 4);
        u32x4 v[4];
        u32x2 yb[8];
        f32x4 d[8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          v[t] = u32x4{0u, 0u, 0u, 0u};
          if (live) v[t] = *reinterpret_cast<const u32x4*>(at + t * PLANE);
        }
        mixm_turn(v, yb);
#pragma unroll
        for (int q = 0; q < 8; ++q) d[q] = YmDot<T>::mfma16(sa[cc][q], yb[q], f32x4{0.f, 0.f, 0.f, 0.f});
        if (live) {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            *reinterpret_cast<u32x4*>(at + t * PLANE) = u32x4{ym_pack<T>(d[0][t], d[1][t]), ym_pack<T>(d[2][t], d[3][t]), ym_pack<T>(d[4][t], d[5][t]), ym_pack<T>(d[6][t], d[7][t])};
        }
      }
    lds_barrier();
    // the rows leave through registers, so that the next tile's first pieces are on their way before them
    u32x4 z[NZ];
#pragma unroll
    for (int i = 0; i < NZ; ++i) z[i] = *reinterpret_cast<const u32x4*>(ym_lds + (wave + 4 * i) * 1024 + lane * 16);
    lds_barrier();
    const int om0 = m0, or0 = r0;
    const bool more = ++item < item_end;
    if (more) begin();
#pragma unroll
    for (int i = 0; i < NZ; ++i) {                     // piece wave + 4 i: eight rows of block (wave + 4 i) / 2 RX
      const int row = (wave & (2 * RX - 1)) * 8 + r8, j = (wave + 4 * i) / (2 * RX), c = (lane & 7) ^ ((row >> 1) & 7);
      if (om0 + row < M && or0 + c * 8 < R) *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(p.m.Z) + ((int64_t)j * M + om0 + row) * R + or0 + c * 8) = z[i];
    }
    if (!more) break;
    stores = om0 + ROWS <= M && or0 + 64 <= R;
  }
}

// S(i, j, r) with any strides -> St[(r b + i) b + j]: one thread per (i, r), neighbouring threads on neighbouring ranks.
template <typename T>
__global__ __launch_bounds__(256) void ym_s_transpose_kernel(const T* __restrict__ S, T* __restrict__ St, int b, int R,
                                                              int64_t s_si, int64_t s_sj, int64_t s_sr) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= b * R) return;
  const int r = idx % R, i = idx / R;
  for (int j = 0; j < b; ++j) St[((int64_t)r * b + i) * b + j] = S[(int64_t)i * s_si + (int64_t)j * s_sj + (int64_t)r * s_sr];
}

// Z (b, M, R) of dtype = mix(S, x V).  scratch: room for S as (r, i, j) (b b R elements), used where S has neither that order nor its ranks
// contiguous on 16 bytes.  Returns BLR_OK, a negative blr_status, or 1 when the shape is not for this kernel (b not a multiple of
// 4 or above 16, rank or block width not a multiple of 8, unaligned operands, fp32, scratch too small).
int blast_ymix_launch(const void* x, int64_t ldx, const void* V, const void* S, void* Z, int M, int in_f, int b, int R,
                      int64_t s_si, int64_t s_sj, int64_t s_sr, int dtype, void* scratch, size_t scratch_bytes, hipStream_t st) {
  if ((dtype != BLR_F16 && dtype != BLR_BF16) || b < 4 || b > 16 || b % 4 || R % 8 || in_f % b || (in_f / b) % 8) return 1;
  if (ldx % 8 || !aligned(x, 16) || !aligned(V, 16) || !aligned(Z, 16)) return 1;
  const int64_t lim = (int64_t)1 << 31;
  if ((M < 32 ? M - 1 : 31) * ldx * 2 + 256 >= lim * 2 || (int64_t)8 * R * 2 >= lim) return 1;
  const int nrt = (int)cdiv(R, 64);
  int nmt = (int)cdiv(M, 32);
  if ((int64_t)nrt * nmt >= lim) return 1;
  bool rij = s_sj == 1 && s_si == b && s_sr == (int64_t)b * b && aligned(S, 8);
  const bool run = s_sr == 1 && s_si % 8 == 0 && s_sj % 8 == 0 && s_si >= 0 && s_sj >= 0 && aligned(S, 16) && ((b - 1) * (s_si + s_sj) + R) * 2 < lim;
  if (!rij && !run) {
    if (!scratch || scratch_bytes < (size_t)b * b * R * 2 || !aligned(scratch, 8)) return 1;
    const unsigned tg = (unsigned)cdiv((int64_t)b * R, 256);
    if (dtype == BLR_F16) hipLaunchKernelGGL(ym_s_transpose_kernel<f16>, dim3(tg), dim3(256), 0, st, (const f16*)S, (f16*)scratch, b, R, s_si, s_sj, s_sr);
    else hipLaunchKernelGGL(ym_s_transpose_kernel<bf16>, dim3(tg), dim3(256), 0, st, (const bf16*)S, (bf16*)scratch, b, R, s_si, s_sj, s_sr);
    BLR_CHECK_LAUNCH("ym_s_transpose");
    S = scratch;
    rij = true;
  }
  YmixParams p = {};
  p.m.S = S; p.m.Z = Z; p.m.M = M; p.m.b = b; p.m.R = R; p.m.s_si = s_si; p.m.s_sj = s_sj;
  p.x = x; p.ldx = ldx; p.V = V;
  p.P = in_f / b;
  const int pieces = (int)cdiv(p.P, 96);
  p.PP = (int)cdiv(p.P / 8, pieces) * 8;
  const int cl = (p.PP / 8) | 1;
  p.cl = fd_make((uint32_t)cl);
  const int cus = device_cus() > 0 ? device_cus() : 256;
  // Tiles of 16 rows where those of 32 give a compute unit at most one: twice the workgroups, each with half the products and the way out of half
  // the rows.  32 / 16 rows, whole calls: 2048 -> 2048 in 16 blocks, r = 256 at 500 / 1000 / 2048 rows 19.6 / 22.2 / 26.3 and 17.5 / 20.6 / 24.3 us, 512 -> 2048 in 4,
  // r = 512 at 500 / 1000 13.1 / 17.6 and 12.0 / 17.0; but past the line V is read twice as often for nothing: 1536 -> 3072 in 8, r = 256 at 3000 rows 28.8 and
  // 32.4, 2048 -> 8192, r = 512 at 2048 47.8 and 54.6.
  const int rx = nrt * nmt <= cus ? 1 : 2;
  if (rx == 1) nmt = (int)cdiv(M, 16);
  p.slot = (rx * cl + 3) / 4 * 1024 + p.PP * 128;
  p.m.nmt = nmt;
  p.m.items = nrt * nmt;
  size_t lds = (size_t)4 * p.slot;
  if (lds < (size_t)b * 2048 * rx) lds = (size_t)b * 2048 * rx;
  const unsigned grid = (unsigned)(p.m.items < 2 * cus ? p.m.items : 2 * cus);
  const int ks = (int)cdiv(p.PP, 32), fi = ((((dtype == BLR_F16 ? 0 : 1) * 2 + (rij ? 0 : 1)) * 4 + b / 4 - 1) * 3 + ks - 1) * 2 + rx - 1;
#define YN1(T, RIJ, NB, KS) (void*)blast_ymix_kernel<T, RIJ, NB, KS, 1>, (void*)blast_ymix_kernel<T, RIJ, NB, KS, 2>
#define YN3(T, RIJ, NB) YN1(T, RIJ, NB, 1), YN1(T, RIJ, NB, 2), YN1(T, RIJ, NB, 3)
#define YN(T, RIJ) YN3(T, RIJ, 1), YN3(T, RIJ, 2), YN3(T, RIJ, 3), YN3(T, RIJ, 4)
  void* const fns[96] = {YN(f16, true), YN(f16, false), YN(bf16, true), YN(bf16, false)};
#undef YN
#undef YN3
#undef YN1
  static bool attr_set[96] = {};
  if (!attr_set[fi]) {
    const hipError_t e = hipFuncSetAttribute(fns[fi], hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
    if (e != hipSuccess) { set_error("blast_ymix: cannot raise the LDS limit: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
    attr_set[fi] = true;
  }
  void* args[] = {&p};
  const hipError_t e = hipLaunchKernel(fns[fi], dim3(grid), dim3(256), args, lds, st);
  if (e != hipSuccess) { set_error("blast_ymix: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  return BLR_OK;
}

// ---- the same first half for wide input blocks: x V as one GEMM over all of x's columns, Y held in registers -------------------
//
// blast_ymix_kernel reads V once per 32 rows; from about 128 columns per input block on that costs more
// than the round trip of Y through memory that it saves.  (That round trip has become cheaper since: this kernel runs where the fused algorithm is asked for by name.)  Here a workgroup of four waves (one per SIMD, so a lane may hold some
// 250 registers) owns 64 rows x 64 ranks for all 16 input blocks.  x is (M, 16 P) and V (16 P, R), both contiguous over the
// blocks, so Y_0 .. Y_15 of the tile are one GEMM with a reduction over all 16 P columns whose accumulator is packed away and
// cleared every P columns: stages of 64 k of both operands go global -> LDS directly (whole 128-byte lines; the stage layouts
// and fragment reads of gemm_ring64_kernel), YW_NST stages deep, one barrier per stage; a wave's 32 x 32 block of Y_j leaves the
// accumulator as 8 dwords (two ranks each), 128 dwords for the sixteen blocks.  When the reduction is done the ring is no longer
// needed: Y goes to LDS as dwords (Y_2jp, Y_2jp+1) [jp][row][rank ^ f(row, jp)], and the mix runs as in blast_ymix_kernel (one
// 16 x 16 x 16 matrix instruction per rank and 16 rows), its rows of Z staged through LDS and stored as whole 128-byte lines.
namespace {
constexpr int YW_NT = 256, YW_NST = 8, YW_STG = 8192;      // threads; ring depth; bytes of a stage of one operand (64 x 64 elements)
constexpr size_t YW_LDS = 160 * 1024;                      // ring: 2 x 8 x 8 KiB + the tile's slice of S 32 KiB; afterwards Y 128 KiB + staged rows of Z 32 KiB
}

struct YmixwParams {
  const void* x; int64_t ldx;
  const void* V; const void* St; void* Z;
  int M, R, KT;                 // KT: stages of 64 k per input block (P / 64)
  FastDiv nrt;                  // rank tiles
  int s_stage;                  // 0: St is S as (r, i, j), read straight into the mix's operands; 1: S has the rank contiguous
  int64_t s_si, s_sj;           //    (strides of i and j in elements): the tile's slice goes through LDS
};

template <typename T>
__global__ __launch_bounds__(YW_NT, 1) void blast_ymixw_kernel(YmixwParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char yw_lds[];
  constexpr int NWV = 4, NST = YW_NST, BRING = NST * YW_STG, LT = 4, RB = 128;
  using V8 = typename TypeTraits<T>::vec8;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int M = p.M, R = p.R;
  // a run of items per XCD, rank tiles fastest: the workgroups of an XCD at any time share two tiles of rows of x in its L2
  const uint32_t item = xcd_item(blockIdx.x, gridDim.x);
  const uint32_t mt = fd_div(item, p.nrt), rt = item - mt * p.nrt.d;
  const int m0 = (int)mt * 64, r0 = (int)rt * 64;
  TR6(0);
  const int n = lane & 15, g = lane >> 4, rw = wave * 16;
  // ---------------------------------------------- phase 1: Y of the tile, in registers --------------------------------------
  // stage s covers columns 64 s .. 64 s + 63 of x and rows 64 s .. of V (all blocks).  K-contiguous stage (x): a load takes eight
  // 16-byte chunks of each of 8 rows, lane (r8, s8) chunk s8 ^ r8; (k, n) stage (V): a load takes 8 rows of 64 ranks, chunk c of
  // row k stored at c ^ ((k & 3) << 1).
  const int r8 = lane >> 3, s8 = lane & 7, c8 = s8 ^ r8;
  uint32_t a_off[2], b_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    a_off[i] = (uint32_t)(min(m0 + (i * NWV + wave) * 8 + r8, M - 1) * p.ldx * 2 + c8 * 16);
    const int krow = (i * NWV + wave) * 8 + r8;
    b_off[i] = (uint32_t)((krow * R + r0 + (s8 ^ ((krow & 3) << 1)) * 8) * 2);
  }
  const uint32_t lds0 = ring_lds_addr(yw_lds + wave * 1024);
  const char* Ab = reinterpret_cast<const char*>(p.x);
  const char* Bb = reinterpret_cast<const char*>(p.V);
  auto issue = [&](int s, int slot) {
    const char* ap = Ab + (int64_t)s * 128;
    const char* bp = Bb + (int64_t)s * 64 * R * 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) ring_load_lds(ap, a_off[i], lds0 + slot * YW_STG + i * (NWV * 1024));
#pragma unroll
    for (int i = 0; i < 2; ++i) ring_load_lds(bp, b_off[i], lds0 + BRING + slot * YW_STG + i * (NWV * 1024));
  };
  const int half = lane >> 5;
  const int rl = wm * 32 + (lane & 31);
  const uint32_t rowA = (uint32_t)(((rl >> 3) << 10) + ((rl & 7) << 7));
  uint32_t xo[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) xo[q] = (uint32_t)(((2 * q + half) ^ (lane & 7)) << 4);
  const int i16 = lane & 15;
  const int chunk0 = wn * 4 + (g & 1) * 2 + ((i16 & 3) >> 1);
  const uint32_t rowB = (uint32_t)(((g >> 1) * 8 + (i16 >> 2)) * RB + (i16 & 1) * 8 + ((chunk0 ^ ((i16 >> 2) << 1)) << 4));

  // Stage t lives in slot t % NST; NST - 1 stages are in flight.  A stage takes about 620 cycles here whatever the order of the
  // loop: the same with every workgroup of the launch on one and the same tile (all loads L2 hits), with a ring of ten stages,
  // with two accumulators taking the sub-steps in turn and with the fragments of stage s + 1 read under the products of stage s
  // (the blocks of Y pinned to accumulation registers to make room) - in-kernel cycle counts then show 29 % of a wave's loop in
  // the issue of its four loads: the compute unit's sixteen load instructions and 48 KiB of LDS traffic per stage are what a
  // 64 x 64 tile costs, and the tile cannot grow because Y of sixteen blocks has to stay in registers.  (Asking for every line a
  // first time twenty stages early, by a 4-byte load per line into a dump area, made it slower: 18.5 -> 28.9 us per tile at
  // P = 256, R = 512 - an instruction that touches 32 lines costs the address path as much as four that fetch them.)
  const int s_total = 16 * p.KT;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s) issue(min(s, s_total - 1), s);
  TR6(1);
  // S with the rank contiguous ((j, i, r) or (i, j, r)): the 256 rows (j, i) x 64 ranks of this tile go to LDS behind the ring,
  // where nothing else lives until the mix stages its rows of Z - by then the operands are in registers
  T* const s_t = reinterpret_cast<T*>(yw_lds + 2 * YW_NST * YW_STG);
  if (p.s_stage) {
    const T* Sg = reinterpret_cast<const T*>(p.St);
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int idx = it * YW_NT + tid, ji = idx >> 3, c = (idx & 7) * 8;
      *reinterpret_cast<V8*>(&s_t[ji * 64 + c]) = *reinterpret_cast<const V8*>(&Sg[(int64_t)(ji & 15) * p.s_si + (int64_t)(ji >> 4) * p.s_sj + r0 + c]);
    }
  }

  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  uint32_t yreg[16][8];
  int s = 0, slot = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    for (int kt = 0; kt < p.KT; ++kt, ++s) {
      __builtin_amdgcn_s_waitcnt(ring_vmcnt((NST - 2) * LT));   // this wave's part of stage s has landed
      __builtin_amdgcn_s_barrier();                             // everybody's has, and nobody reads stage s - 1 any more
      issue(min(s + NST - 1, s_total - 1), slot == 0 ? NST - 1 : slot - 1);   // (past the end: the last stage again, never read)
      const unsigned char* sta = yw_lds + slot * YW_STG;
      const unsigned char* stb = yw_lds + BRING + slot * YW_STG;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const V8 af = *reinterpret_cast<const V8*>(sta + rowA + xo[q]);
        union { V8 v; s16x4 h[2]; } w;
        w.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(stb + rowB + (q * 16) * RB));
        w.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(stb + rowB + (q * 16 + 4) * RB));
        acc = TypeTraits<T>::mfma32(w.v, af, acc);             // (ranks as rows: the product comes out transposed)
      }
      slot = slot + 1 == NST ? 0 : slot + 1;
    }
    // acc[4 q + e] is Y_j at row wm 32 + (lane & 31), rank wn 32 + 8 q + 4 half + e
#pragma unroll
    for (int d = 0; d < 8; ++d) yreg[j][d] = ym_pack<T>(acc[2 * d], acc[2 * d + 1]);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  }
  TR6(2);
  __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));                    // the repeats of the last stage have landed too: the ring is free
  __builtin_amdgcn_s_barrier();
  // the mix's S operands, asked for now (the loop had no registers to spare) and used after Y has gone to LDS.  Lane (n, g) of
  // wave w: S_r(i = n, j = 4 g .. 4 g + 3), r = r0 + 16 w ..
  u32x2 sa[16];
  if (p.s_stage) {                                              // (the barrier above is behind every wave's stores of the slice)
    const uint16_t* s16 = reinterpret_cast<const uint16_t*>(s_t);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      uint32_t v[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) v[jj] = s16[((4 * g + jj) * 16 + n) * 64 + rw + q];
      sa[q] = u32x2{v[0] | (v[1] << 16), v[2] | (v[3] << 16)};
    }
  } else {
    const __amdgpu_buffer_rsrc_t sbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.St), 0, (uint32_t)((int64_t)256 * R * 2), 0x00020000);
#pragma unroll
    for (int q = 0; q < 16; ++q)
      sa[q] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(sbuf, (uint32_t)(((r0 + rw + q) * 16 + n) * 16 + 4 * g) * 2u, 0, 0));
  }

  // Y -> LDS: dword (Y_2jp, Y_2jp+1) of (row m, rank r) at [jp][m][r ^ ((m & 15) + 16 (jp >> 1))] - the 64 lanes of a mix read
  // (16 rows x 4 pairs of planes, one rank) then hit 64 different banks.  Dword d of a block holds ranks ra, ra + 1 (ra even):
  // neighbours in LDS, in the order the row's parity gives.
  uint32_t* const y_s = reinterpret_cast<uint32_t*>(yw_lds);
  {
    const int m = wm * 32 + (lane & 31);
#pragma unroll
    for (int jp = 0; jp < 8; ++jp)
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const uint32_t h0 = yreg[2 * jp][d], h1 = yreg[2 * jp + 1][d];
        const uint32_t da = __builtin_amdgcn_perm(h1, h0, 0x05040100u), db = __builtin_amdgcn_perm(h1, h0, 0x07060302u);
        const int ra = wn * 32 + 8 * (d >> 1) + 4 * half + 2 * (d & 1);
        const int col = (ra ^ ((m & 15) + 16 * (jp >> 1))) & ~1;
        *reinterpret_cast<u32x2*>(&y_s[jp * 4096 + m * 64 + col]) = (m & 1) ? u32x2{db, da} : u32x2{da, db};
        if (d == 7) __builtin_amdgcn_sched_barrier(0);          // (one pair of blocks at a time: nothing to gain from more in flight)
      }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  TR6(3); TR6(4);

  // ---------------------------------------------- phase 2: the mix --------------------------------------------------------
  // lane (n, g): operand A = S_r(i = n, j = 4 g .. 4 g + 3), operand B = Y_r(j = 4 g .. 4 g + 3, m = 16 mg + n); the product's lane
  // holds Z_r(i = 4 g + t, m = 16 mg + n).  The 256 rows (i, m) of a group of 16 rows of the tile go through LDS (128 bytes each,
  // 16-byte slots XOR-ed with the row's low bits) and leave as whole lines.
  uint32_t* const z_st = y_s + 8 * 4096;
#pragma unroll 1
  for (int mg = 0; mg < 4; ++mg) {
    if (mg) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");     // the previous group's rows have been read
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 d[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int rr = rw + 8 * h + q;
        const uint32_t* src = &y_s[(2 * g) * 4096 + (16 * mg + n) * 64 + (rr ^ (n + 16 * g))];
        const u32x2 yb = {src[0], src[4096]};
        d[q] = YmDot<T>::mfma16(sa[8 * h + q], yb, f32x4{0.f, 0.f, 0.f, 0.f});
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        u32x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = ym_pack<T>(d[2 * q][t], d[2 * q + 1][t]);
        const int row = (4 * g + t) * 16 + n;
        *reinterpret_cast<u32x4*>(&z_st[row * 32 + (((wave * 2 + h) ^ (row & 7)) << 2)]) = o;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    {
      const int pc = tid & 7, rr = tid >> 3;               // 16-byte piece of a row; rows rr, rr + 32, ...
      u32x4 v[8];
#pragma unroll
      for (int it = 0; it < 8; ++it) v[it] = *reinterpret_cast<const u32x4*>(&z_st[(rr + 32 * it) * 32 + ((pc ^ (rr & 7)) << 2)]);
      const int m = m0 + 16 * mg + (rr & 15);
      if (m < M) {
#pragma unroll
        for (int it = 0; it < 8; ++it)
          *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(p.Z) + ((int64_t)(2 * it + (rr >> 4)) * M + m) * R + r0 + pc * 8) = v[it];
      }
    }
  }
  TR6(14);
}

// Z (16, M, R) of dtype = mix(S, x V) for 16 input blocks of a multiple of 64 columns and a rank that is a multiple of 64.
// scratch: room for S transposed to (r, i, j), used unless S already has that layout.  Returns BLR_OK, a negative blr_status, or
// 1 when the shape is not for this kernel.
int blast_ymixw_launch(const void* x, int64_t ldx, const void* V, const void* S, void* Z, int M, int in_f, int b, int R,
                       int64_t s_si, int64_t s_sj, int64_t s_sr, int s_layout, int dtype, void* scratch, size_t scratch_bytes,
                       hipStream_t st) {
  if (dtype != BLR_F16 && dtype != BLR_BF16) return 1;
  if (b != 16 || in_f % 16) return 1;
  const int P = in_f / 16;
  if (P % 64 || R % 64 || ldx % 8 || !aligned(x, 16) || !aligned(V, 16) || !aligned(Z, 16)) return 1;
  if (((int64_t)(M - 1) * ldx + in_f) * 2 >= ((int64_t)1 << 31) || (int64_t)64 * R * 2 >= ((int64_t)1 << 31) || (int64_t)256 * R * 2 >= ((int64_t)1 << 31)) return 1;
  // (A variant with 64 rows x 128 ranks on eight waves - two per SIMD, three quarters of the operand bytes per product, the tile's
  // two halves of 64 ranks mixed one after the other - passed the same tests and measured slower: a stage of its loop took 575 ns
  // against 270 ns, 4096 -> 22016 at 2048 rows 177 against 173 us for the call.  The same tile on four waves - a wave holding 32 rows
  // x 64 ranks, its 256 dwords of Y spilling over into the accumulation registers, a ring of four stages of 24 KiB, the mix a quarter
  // of the tile at a time - was no better: 39.2 us in the loop for twice the products of the 17.3 us here, 30 us in the mix against
  // 2 x 6.8, the call 177.5 against 171.7 us.  Fewer load instructions per product do not speed this loop up.)
  const int nmt = (int)cdiv(M, 64), nrt = R / 64;
  if ((int64_t)nmt * nrt >= 65536) return 1;
  YmixwParams p = {};
  p.x = x; p.ldx = ldx; p.V = V; p.Z = Z; p.M = M; p.R = R; p.KT = P / 64;
  p.nrt = fd_make((uint32_t)nrt);
  if (s_layout == BLR_S_RIJ && aligned(S, 8)) {
    p.St = S;
  } else if (s_sr == 1 && s_si % 8 == 0 && s_sj % 8 == 0 && aligned(S, 16)) {
    p.St = S; p.s_stage = 1; p.s_si = s_si; p.s_sj = s_sj;
  } else {
    if (!scratch || scratch_bytes < (size_t)256 * R * 2 || !aligned(scratch, 8)) return 1;
    const unsigned tg = (unsigned)cdiv((int64_t)16 * R, 256);
    if (dtype == BLR_F16) hipLaunchKernelGGL(ym_s_transpose_kernel<f16>, dim3(tg), dim3(256), 0, st, (const f16*)S, (f16*)scratch, 16, R, s_si, s_sj, s_sr);
    else hipLaunchKernelGGL(ym_s_transpose_kernel<bf16>, dim3(tg), dim3(256), 0, st, (const bf16*)S, (bf16*)scratch, 16, R, s_si, s_sj, s_sr);
    BLR_CHECK_LAUNCH("ym_s_transpose");
    p.St = scratch;
  }
  void* const fn = dtype == BLR_F16 ? (void*)blast_ymixw_kernel<f16> : (void*)blast_ymixw_kernel<bf16>;
  static bool attr_set[2] = {false, false};
  if (!attr_set[dtype == BLR_F16 ? 0 : 1]) {
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)YW_LDS);
    if (e != hipSuccess) { set_error("blast_ymixw: cannot raise the LDS limit: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
    attr_set[dtype == BLR_F16 ? 0 : 1] = true;
  }
  void* args[] = {&p};
  hipError_t e = hipLaunchKernel(fn, dim3((unsigned)(nmt * nrt)), dim3(YW_NT), args, YW_LDS, st);
  if (e != hipSuccess) { set_error("blast_ymixw: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  return BLR_OK;
}


// ---- second half for narrow output blocks: out_i = mix(S, Y)_i U_i in one launch, Z never written -------------------------
//
// When an output block is at most 80 columns wide, the results of ALL output blocks for a tile of 16 rows fit the registers of one
// workgroup (16 blocks x 16 rows x 80 columns of fp32 = 80 KB).  The workgroup then walks the rank in blocks of 64: it reads the
// block of Y for all input blocks once (the only pass over the intermediate), forms the block of every Z_i on the matrix cores
// (one 16 x 16 x 16 product per rank, as in the kernel above), hands it through LDS as T and multiplies it with the block of U_i.
// U (b, Q, R) has the rank contiguous, so 16 bytes of it are an operand as they stand - but the lanes of a matrix-core operand
// are its rows, and a load whose neighbouring lanes read different rows of U occupies the compute unit's memory pipeline for 64
// cycles instead of 16 (measured: 3 us per step with such loads, 0.5 us without any).  A small kernel therefore first re-lays U
// (1.3 MB at 4608 -> 1152, rank 576) and S in the order the lanes read them: U as (i, rank / 8, q, 8) - neighbouring lanes, i.e.
// neighbouring columns q, then read neighbouring 16-byte pieces - and S as (r / 2, j / 4, i, r % 2, 4), 16 bytes per lane and pair of ranks.
// A block of 64 ranks is two matrix-core steps of 32; step s takes the ranks 16 g + 8 s + e (g = 0..3 the lane group, e = 0..7 the
// element of the lane's 16 bytes).
//   wave w: four of the 32 load instructions that bring a block of Y (8 rows of 128 bytes each) into LDS; the mix of slots
//   4 w .. 4 w + 3 of a step (ranks 16 (w / 2) + 8 s + 4 (w % 2) + 0..3 of the block); output blocks 2 w, 2 w + 1.
// S and U of step c + 2 are asked for right after step c has used its registers, Y of the next block at the start of a block.
namespace {
constexpr int MU_NT = 512;
constexpr int MU_BM = 16;
constexpr int MU_RB = 64;       // ranks per block
constexpr int MU_LDY = 72;      // two-byte elements per LDS row of Y (64 ranks): 144 bytes keep 16-byte accesses aligned and rows apart
constexpr int MU_LDZ = 40;      // per LDS row of Z (the 32 slots of a step)
__device__ __forceinline__ void mu_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
}  // namespace

struct MixuParams {
  const void* Y; const void* Sp; const void* Ut; void* out; int64_t ldo;     // Sp (r / 2, j / 4, i, r % 2, 4), Ut (i, rank / 8, q, 8)
  int M, R, Q;
  uint32_t y_bytes;
  int rotate;
  const void* bias; int act;
  const void* gate; int gate_rows; int64_t ld_gate;
  const void* resid; int64_t ld_resid;
};

// The way out of blast_mixu_kernel and blast_one_kernel: stage() puts the tile (16 rows x 16 Q columns) into LDS as T, o_s[row][16 Q + 8];
// it leaves in whole rows, 16 bytes per lane, neighbouring lanes on neighbouring columns, through the output stage.  A thread has up to
// U = 5 pieces (Q <= 80) and asks for their bias, gate and residual together, ahead of the staging: one piece after another waited for up
// to three trips to memory each (DiT-XL/2's forward at sixteen images, 28 launches of either kernel: 8.83 -> 8.62 ms).
template <typename T, typename P, typename F>
__device__ __forceinline__ void mu_write_out(const P& p, const uint16_t* o_s, int m0, int tid, F&& stage) {
  using V8 = typename TypeTraits<T>::vec8;
  constexpr int U = 5;
  const int ppr = 2 * p.Q, OLD = 16 * p.Q + 8;                // 16-byte pieces per row
  int mr[U], col[U];
  bool live[U];
  V8 bv[U], gv[U], rv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int pi = tid + u * MU_NT, row = pi / ppr;
    live[u] = row < 16 && m0 + row < p.M;
    mr[u] = live[u] ? row : 0;                               // (the others carry the place of a piece inside, row 0 of the tile)
    col[u] = (pi - row * ppr) * 8;
  }
  if (p.bias) {
#pragma unroll
    for (int u = 0; u < U; ++u) bv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(p.bias) + col[u]);
  }
  if (p.gate) {
#pragma unroll
    for (int u = 0; u < U; ++u) gv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(p.gate) + (int64_t)((m0 + mr[u]) / p.gate_rows) * p.ld_gate + col[u]);
  }
  if (p.resid) {
#pragma unroll
    for (int u = 0; u < U; ++u) rv[u] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(p.resid) + (int64_t)(m0 + mr[u]) * p.ld_resid + col[u]);
  }
  stage();
  mu_barrier();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const V8 r = *reinterpret_cast<const V8*>(&o_s[mr[u] * OLD + col[u]]);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = TypeTraits<T>::to_f32(r[e]);
    if (p.bias) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += TypeTraits<T>::to_f32(bv[u][e]);
    }
    apply_act_n(v, p.act);
    if (p.gate || p.resid) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = TypeTraits<T>::to_f32(TypeTraits<T>::from_f32(v[e]));
      if (p.gate) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= TypeTraits<T>::to_f32(gv[u][e]);
      }
      if (p.resid) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += TypeTraits<T>::to_f32(rv[u][e]);
      }
    }
    V8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = TypeTraits<T>::from_f32(v[e]);
    if (live[u]) *reinterpret_cast<V8*>(reinterpret_cast<T*>(p.out) + (int64_t)(m0 + mr[u]) * p.ldo + col[u]) = o;
  }
}

template <typename T, int NTQ>
__global__ __launch_bounds__(MU_NT) void blast_mixu_kernel(MixuParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t mu_lds[256 * MU_LDY + 2 * 256 * MU_LDZ];
  uint16_t* const y_s = mu_lds;                              // [input block j][row m][rank of the block]
  uint16_t (*const z_s)[256 * MU_LDZ] = reinterpret_cast<uint16_t (*)[256 * MU_LDZ]>(mu_lds + 256 * MU_LDY);   // per step: [output block i][row m][slot]
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
  const int M = p.M, R = p.R, Q = p.Q;
  const int m0 = (int)blockIdx.x * MU_BM;
  const int NB = (R + MU_RB - 1) / MU_RB;             // the last block may hold 32 ranks: what lies past them is not asked for
  const bool half_u = (R % MU_RB) != 0 && g >= 2, half_y = (R % MU_RB) != 0 && (l & 7) >= 4;
  // Workgroups walk the blocks of ranks in turn from different starting points: all of them read the same ranks of U and S
  // otherwise, at the same moment, from the same lines of the eight L2s.  (The sum over the blocks is in fp32 and its order is
  // fixed per row tile.)
  const int rot = p.rotate ? (int)(blockIdx.x % (unsigned)NB) : 0;
  auto blk = [&](int k) { const int kk = k + rot; return kk >= NB ? kk - NB : kk; };
  TR6(0);
  const __amdgpu_buffer_rsrc_t ybuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Y), 0, p.y_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t sbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Sp), 0, (uint32_t)(256 * R * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t ubuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Ut), 0, (uint32_t)((int64_t)16 * Q * R * 2), 0x00020000);
  // Y: eight lanes fetch the 128 bytes of one (j, m); a load instruction covers eight rows m of one input block; the wave's four
  // loads are rows 0..7 and 8..15 of the input blocks 2 wv and 2 wv + 1.  Per-lane offsets are few (registers are short):
  // whatever is the same for all lanes goes into the scalar offset of the load.
  const int piece = l & 7, yrow = l >> 3;
  uint32_t yoff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    yoff[h] = m0 + 8 * h + yrow < M ? (uint32_t)(((int64_t)(2 * wv) * M + m0 + 8 * h + yrow) * R + piece * 8) * 2u : YM_OOB;
  const uint32_t yjs = (uint32_t)((int64_t)M * R * 2);           // from one input block to the next
  const int ypos = ((2 * wv) * 16 + yrow) * MU_LDY + piece * 8;
  // S_r(i = n, j = 4 g .. 4 g + 3) of the wave's four ranks of a step
  const int rk = 16 * (wv >> 1) + 4 * (wv & 1);                  // + 8 s + 64 k
  const uint32_t soff = (uint32_t)((rk >> 1) * 64 + l) * 16u;      // Sp: 16 bytes per lane and pair of ranks
  // U_i(q = 16 nt + n, ranks 16 g + 8 s .. + 7 of the block), i = 2 wv + ii: piece (i, 8 k + 2 g + s, q) of Ut
  const uint32_t uoff = (uint32_t)(((int64_t)(2 * wv) * (R / 8) + 2 * g) * Q + n) * 16u;
  const uint32_t uoff_last = 16 * (NTQ - 1) + n < Q ? uoff : YM_OOB;      // the last column tile of a block may be partly empty
  const uint32_t uis = (uint32_t)((R / 8) * Q) * 16u;            // from one output block to the next
  struct Regs { u32x4 s[2]; u32x4 u[2][NTQ]; };
  auto load_y = [&](u32x4 (&yr)[4], int k) {
    const bool cut = half_y && k == NB - 1;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      yr[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ybuf, cut ? YM_OOB : yoff[u & 1], (uint32_t)k * (MU_RB * 2u) + (uint32_t)(u >> 1) * yjs, 0));
  };
  auto store_y = [&](const u32x4 (&yr)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<u32x4*>(&y_s[ypos + ((u >> 1) * 16 + (u & 1) * 8) * MU_LDY]) = yr[u];
  };
  auto load_s = [&](Regs& r, int k, int s) {                 // rank 64 k + 8 s + rk + q
#pragma unroll
    for (int q = 0; q < 2; ++q) r.s[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(sbuf, soff + (uint32_t)q * 1024u, (uint32_t)(k * MU_RB + 8 * s) * 512u, 0));
  };
  auto load_u = [&](Regs& r, int k, int s) {
    const bool cut = half_u && k == NB - 1;
    const uint32_t v0 = cut ? YM_OOB : uoff, vl = cut ? YM_OOB : uoff_last;
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
      for (int nt = 0; nt < NTQ; ++nt)
        r.u[ii][nt] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ubuf, (nt == NTQ - 1 ? vl : v0) + (uint32_t)nt * 256u,
                                                                                        (uint32_t)((8 * k + s) * Q) * 16u + (uint32_t)ii * uis, 0));
  };
  f32x4 acc[2][NTQ];
#pragma unroll
  for (int ii = 0; ii < 2; ++ii)
#pragma unroll
    for (int nt = 0; nt < NTQ; ++nt) acc[ii][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // step s of block k on the register set `cur`.  No load sits under a condition (the compiler would then wait for everything in
  // flight where the paths meet): the last blocks ask again for the last block, which costs their turns in the memory pipeline
  // and nothing else.
  auto step = [&](int k, auto SS, Regs& cur) {
    constexpr int s = decltype(SS)::value;
    const int kn = blk(min(k + 1, NB - 1));
    // the mix of this wave's four ranks: operand B = Y_r(j = 4 g .. 4 g + 3, m = n), gathered from the four rows of its lane
    u32x2 yv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) yv[t] = *reinterpret_cast<const u32x2*>(&y_s[((4 * g + t) * 16 + n) * MU_LDY + rk + 8 * s]);
    f32x4 d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
      const u32x2 yb = {__builtin_amdgcn_perm(yv[1][q >> 1], yv[0][q >> 1], sel), __builtin_amdgcn_perm(yv[3][q >> 1], yv[2][q >> 1], sel)};
      d[q] = YmDot<T>::mfma16(u32x2{cur.s[q >> 1][2 * (q & 1)], cur.s[q >> 1][2 * (q & 1) + 1]}, yb, f32x4{0.f, 0.f, 0.f, 0.f});
    }
    load_s(cur, kn, s);
    // d[q][t] = Z_r(i = 4 g + t, m = n) of slot 4 wv + q
#pragma unroll
    for (int t = 0; t < 4; ++t)
      *reinterpret_cast<u32x2*>(&z_s[s][((4 * g + t) * 16 + n) * MU_LDZ + 4 * wv]) = u32x2{ym_pack<T>(d[0][t], d[1][t]), ym_pack<T>(d[2][t], d[3][t])};
    mu_barrier();                                   // Z of the step is whole (the other step's buffer was last read a barrier ago)
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
      const u32x4 zv = *reinterpret_cast<const u32x4*>(&z_s[s][((2 * wv + ii) * 16 + n) * MU_LDZ + 8 * g]);
#pragma unroll
      for (int nt = 0; nt < NTQ; ++nt) acc[ii][nt] = YmDot<T>::mfma(cur.u[ii][nt], zv, acc[ii][nt]);
    }
    load_u(cur, kn, s);
  };
  using S0 = std::integral_constant<int, 0>; using S1 = std::integral_constant<int, 1>;
  Regs ra, rb;
  // Block k asks for Y of block k + 2 into the registers `yl` that block k gave to LDS, and puts block k + 1 from `ys` into LDS at
  // its end.  (Loads return to a wave in the order it asked, and S and U are asked for one block ahead, so Y in effect has one
  // block's time as well; what bounds a step is the 112 KB per workgroup that 256 workgroups draw from L2 and memory, about
  // 1.4 us against 0.5 us for a step without loads.)
  auto block = [&](int k, u32x4 (&yl)[4], const u32x4 (&ys)[4]) {
    load_y(yl, blk(min(k + 2, NB - 1)));
    step(k, S0{}, ra);
    step(k, S1{}, rb);
    store_y(ys);                                    // every wave is past the barrier of the step: nobody reads this block of Y any more
    mu_barrier();                                   // Y of the next block is whole
  };

  u32x4 y0[4], y1[4];
  load_y(y0, blk(0)); load_s(ra, blk(0), 0); load_u(ra, blk(0), 0); load_s(rb, blk(0), 1); load_u(rb, blk(0), 1);
  load_y(y1, blk(min(1, NB - 1)));
  store_y(y0);
  mu_barrier();
  TR6(1);
  int k = 0;
  for (; k + 1 < NB; k += 2) {
    block(k, y0, y1);
    block(k + 1, y1, y0);
    TR6(2 + ((k >> 1) & 7));
  }
  if (k < NB) block(k, y0, y1);
  TR6(14);

  // acc[ii][nt][t] = out(m = m0 + n, column (2 wv + ii) Q + 16 nt + 4 g + t).  The tile (16 rows x 16 Q columns) goes through LDS
  // (over Y and the first Z buffer, which nobody reads any more: every wave is past the last step's barrier) so that it leaves
  // in whole rows: 16 bytes per lane, neighbouring lanes on neighbouring columns.
  using V4 = typename TypeTraits<T>::vec4;
  const int OLD = 16 * Q + 8;
  uint16_t* const o_s = mu_lds;
  mu_write_out<T>(p, o_s, m0, tid, [&] {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
      for (int nt = 0; nt < NTQ; ++nt) {
        const int q = 16 * nt + 4 * g;
        if (q < Q) {
          V4 o;
#pragma unroll
          for (int t = 0; t < 4; ++t) o[t] = TypeTraits<T>::from_f32(acc[ii][nt][t]);
          *reinterpret_cast<V4*>(&o_s[n * OLD + (2 * wv + ii) * Q + q]) = o;
        }
      }
  });
  TR6(15);
}

// The re-laying of U and S (side_prep_item) as a launch of its own: one thread per piece.
template <typename T>
__global__ __launch_bounds__(256) void mixu_prep_kernel(SidePrep s) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx < s.items) side_prep_item<T>(s, idx);
}

namespace {
template <typename T>
void* mixu_fn(int ntq) {
  switch (ntq) {
    case 1: return (void*)blast_mixu_kernel<T, 1>;
    case 2: return (void*)blast_mixu_kernel<T, 2>;
    case 3: return (void*)blast_mixu_kernel<T, 3>;
    case 4: return (void*)blast_mixu_kernel<T, 4>;
    case 5: return (void*)blast_mixu_kernel<T, 5>;
    default: return nullptr;
  }
}
}  // namespace

bool blast_mixu_plan(const void* Y, const void* S, const void* U, const void* out, int64_t ldo, const GemmArgs& ep, int M, int b, int R, int Q,
                     int64_t s_si, int64_t s_sj, int64_t s_sr, int dtype, void* scratch, size_t scratch_bytes, SidePrep* job, bool u_rq) {
  if (dtype != BLR_F16 && dtype != BLR_BF16) return false;
  if (b != 16 || Q % 8 || Q > 80 || Q < 8 || R % 32 || M < 1) return false;
  if (!aligned(Y, 16) || !aligned(U, 16) || !aligned(out, 16) || ldo % 8) return false;
  if ((ep.bias && !aligned(ep.bias, 16)) || (ep.gate && (!aligned(ep.gate, 16) || ep.ld_gate % 8 || ep.gate_rows < 1)) ||
      (ep.resid && (!aligned(ep.resid, 16) || ep.ld_resid % 8))) return false;
  const int64_t y_bytes = (int64_t)b * M * R * 2;
  if (y_bytes >= (int64_t)YM_OOB || (int64_t)b * Q * R * 2 >= (int64_t)YM_OOB || (int64_t)b * b * R * 2 >= (int64_t)YM_OOB) return false;
  if (cdiv(M, MU_BM) >= 2147483647LL) return false;
  if (!(dtype == BLR_F16 ? mixu_fn<f16>((int)cdiv(Q, 16)) : mixu_fn<bf16>((int)cdiv(Q, 16)))) return false;
  const size_t ut_bytes = align_up((size_t)b * Q * R * 2, 256), sp_bytes = (size_t)b * b * R * 2;
  if (!scratch || scratch_bytes < ut_bytes + sp_bytes || !aligned(scratch, 16)) return false;
  if (job) {
    job->U = U; job->S = S; job->Ut = scratch; job->Sp = reinterpret_cast<char*>(scratch) + ut_bytes;
    job->Q = Q; job->R = R; job->u_rq = u_rq ? 1 : 0; job->s_si = s_si; job->s_sj = s_sj; job->s_sr = s_sr;
    job->items = (int64_t)b * (R / 8) * Q + (int64_t)R * 64;
  }
  return true;
}

// out (M, b Q) = [mix(S, Y)_i U_i]_i with the fused output stage of `ep` (bias, act, gate, resid; its other members are not
// read).  Y (b, M, R), U (b, Q, R) of dtype.  scratch: room for U and S re-laid (b Q R + b b R elements, rounded up to 256
// bytes each); prepared: an earlier launch of the call has already put them there.  Returns BLR_OK, a negative blr_status, or 1
// when the shape is not for this kernel (b other than 16, blocks wider than 80 columns or not a multiple of 8, rank not a
// multiple of 32, unaligned operands, fp32).
int blast_mixu_launch(const void* Y, const void* S, const void* U, void* out, int64_t ldo, const GemmArgs& ep, int M, int b, int R, int Q,
                      int64_t s_si, int64_t s_sj, int64_t s_sr, int s_layout, int dtype, void* scratch, size_t scratch_bytes,
                      hipStream_t st, bool prepared, bool u_rq) {
  (void)s_layout;
  SidePrep job = {};
  if (!blast_mixu_plan(Y, S, U, out, ldo, ep, M, b, R, Q, s_si, s_sj, s_sr, dtype, scratch, scratch_bytes, &job, u_rq)) return 1;
  void* fn = dtype == BLR_F16 ? mixu_fn<f16>((int)cdiv(Q, 16)) : mixu_fn<bf16>((int)cdiv(Q, 16));
  MixuParams p = {};
  p.Y = Y; p.out = out; p.ldo = ldo; p.M = M; p.R = R; p.Q = Q; p.y_bytes = (uint32_t)((int64_t)b * M * R * 2);
  p.bias = ep.bias; p.act = ep.act; p.gate = ep.gate; p.gate_rows = ep.gate ? ep.gate_rows : 1; p.ld_gate = ep.ld_gate;
  p.resid = ep.resid; p.ld_resid = ep.ld_resid;
  p.Ut = job.Ut; p.Sp = job.Sp;
  p.rotate = 1;
  if (!prepared) {
    const unsigned tg = (unsigned)cdiv(job.items, 256);
    if (dtype == BLR_F16) hipLaunchKernelGGL(mixu_prep_kernel<f16>, dim3(tg), dim3(256), 0, st, job);
    else hipLaunchKernelGGL(mixu_prep_kernel<bf16>, dim3(tg), dim3(256), 0, st, job);
    BLR_CHECK_LAUNCH("mixu_prep");
  }
  void* args[] = {&p};
  hipError_t e = hipLaunchKernel(fn, dim3((unsigned)cdiv(M, MU_BM)), dim3(MU_NT), args, 0, st);
  if (e != hipSuccess) { set_error("blast_mixu: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  return BLR_OK;
}

// ---- narrow input AND output blocks: the whole call in one launch, neither Y nor Z in memory ------------------------------
//
// With input blocks of at most 96 columns the chunk of V that a step of blast_mixu_kernel's walk over the rank needs (16 input
// blocks x P x 32 ranks) is as small as its chunk of U, so the workgroup forms the step's Y itself instead of reading it: wave w
// keeps its rows of x for input blocks 2 w and 2 w + 1 in registers (operand B, 16 rows x P), loads the 32 ranks of V_2w and
// V_2w+1 (operand A: V re-laid like U, rank-major with k contiguous, in the order the lanes read it, k padded to 32 KS with
// zeros) and leaves Y^T (ranks x rows) as T in LDS - four consecutive ranks per lane.  The rest of the step is the step of
// blast_mixu_kernel: mix of four ranks per wave into Z (LDS), barrier, products with U_2w, U_2w+1 into the 16 x 16 Q results
// that stay in registers for the whole call.  Three barriers per step; Y and Z have one buffer each (every reader of a buffer is
// past the barrier that precedes its next writer in program order).
struct OneParams {
  const void* x; int64_t ldx; uint32_t x_bytes;
  const void* Vp; const void* Sp; const void* Ut; void* out; int64_t ldo;     // Vp (step, j, half, kstep, lane, 8), Sp, Ut as for blast_mixu_kernel
  int M, P, R, Q;
  const void* bias; int act;
  const void* gate; int gate_rows; int64_t ld_gate;
  const void* resid; int64_t ld_resid;
};

template <typename T, int NTQ, int KS>
__global__ __launch_bounds__(MU_NT) void blast_one_kernel(OneParams p) {
  constexpr int LDY = 40;                                    // two-byte elements per LDS row of Y and Z (32 ranks / slots + 8)
  constexpr int OSN = 16 * (16 * 80 + 8);                      // the tile on its way out: 16 rows of up to 16 x 80 columns (+ 8)
  __shared__ __attribute__((aligned(16))) uint16_t one_lds[2 * 256 * LDY > OSN ? 2 * 256 * LDY : OSN];
  uint16_t* const y_s = one_lds;                             // [input block j][row m][rank of the step]
  uint16_t* const z_s = one_lds + 256 * LDY;                 // [output block i][row m][slot]
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
  const int M = p.M, P = p.P, R = p.R, Q = p.Q;
  const int m0 = (int)blockIdx.x * MU_BM;
  const int NSTEP = R / 32;
  const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, p.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Vp), 0, (uint32_t)((int64_t)NSTEP * 16 * 2 * KS * 1024), 0x00020000);
  const __amdgpu_buffer_rsrc_t sbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Sp), 0, (uint32_t)(256 * R * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t ubuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.Ut), 0, (uint32_t)((int64_t)16 * Q * R * 2), 0x00020000);
  // the rows of x: operand B of the first products, lane (n, g) = row m0 + n, k = 32 ks + 8 g .. + 7 of input block 2 wv + jj
  u32x4 xr[2][KS];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k = 32 * ks + 8 * g;
      const uint32_t off = (m0 + n < M && k < P) ? (uint32_t)((int64_t)(m0 + n) * p.ldx + (int64_t)(2 * wv + jj) * P + k) * 2u : YM_OOB;
      xr[jj][ks] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, off, 0, 0));
    }
  const uint32_t voff = (uint32_t)((2 * wv) * 2 * KS * 1024 + l * 16);     // + ((jj 2 + nt) KS + ks) 1024; a step is 16 * 2 * KS KiB further
  // (k past P is not asked for: with P = 72 that is a quarter of V, 1152 -> 1152 at 4096 rows 29.8 -> 29.3 us; 640 -> 640 17.5 -> 16.9)
  const uint32_t voff_last = 32 * (KS - 1) + 8 * g < P ? voff : YM_OOB;
  const uint32_t soff = (uint32_t)((2 * wv) * 64 + l) * 16u;
  const uint32_t uoff = (uint32_t)(((int64_t)(2 * wv) * (R / 8) + g) * Q + n) * 16u;
  const uint32_t uoff_last = 16 * (NTQ - 1) + n < Q ? uoff : YM_OOB;
  const uint32_t uis = (uint32_t)((R / 8) * Q) * 16u;
  struct Regs { u32x4 s[2]; u32x4 u[2][NTQ]; };
  u32x4 vr[2][2][KS];
  auto load_v = [&](int s) {
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          vr[jj][nt][ks] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vbuf, (ks == KS - 1 ? voff_last : voff) + (uint32_t)(((jj * 2 + nt) * KS + ks) * 1024), (uint32_t)s * (uint32_t)(16 * 2 * KS * 1024), 0));
  };
  auto load_s = [&](Regs& r, int s) {                        // ranks 32 s + 4 wv + q
#pragma unroll
    for (int q = 0; q < 2; ++q) r.s[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(sbuf, soff + (uint32_t)q * 1024u, (uint32_t)(32 * s) * 512u, 0));
  };
  auto load_u = [&](Regs& r, int s) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
      for (int nt = 0; nt < NTQ; ++nt)
        r.u[ii][nt] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ubuf, (nt == NTQ - 1 ? uoff_last : uoff) + (uint32_t)nt * 256u,
                                                                                        (uint32_t)(4 * s * Q) * 16u + (uint32_t)ii * uis, 0));
  };
  f32x4 acc[2][NTQ];
#pragma unroll
  for (int ii = 0; ii < 2; ++ii)
#pragma unroll
    for (int nt = 0; nt < NTQ; ++nt) acc[ii][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Workgroups start at different steps (the fp32 sums keep a fixed order per row tile): they would otherwise all ask the L2s
  // for the same lines of V, U and S at the same moment.
  const int rot = (int)(blockIdx.x % (unsigned)NSTEP);
  auto stp = [&](int s) { const int v = s + rot; return v >= NSTEP ? v - NSTEP : v; };

  // No load sits under a condition (the compiler would then wait for everything in flight where the paths meet): the last steps
  // ask again for the last step, which costs their turns in the memory pipeline and nothing else.
  auto step = [&](int s, Regs& cur) {
    const int s1 = stp(min(s + 1, NSTEP - 1)), s2 = stp(min(s + 2, NSTEP - 1));
    // Y^T of the step: ranks 16 nt + 4 g + t of rows m = n, input blocks 2 wv and 2 wv + 1
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) y = YmDot<T>::mfma(vr[jj][nt][ks], xr[jj][ks], y);
        *reinterpret_cast<u32x2*>(&y_s[((2 * wv + jj) * 16 + n) * LDY + 16 * nt + 4 * g]) = u32x2{ym_pack<T>(y[0], y[1]), ym_pack<T>(y[2], y[3])};
      }
    load_v(s1);
    mu_barrier();                                   // Y of the step is whole
    // the mix of this wave's four ranks: operand B = Y_r(j = 4 g .. 4 g + 3, m = n), gathered from the four rows of its lane
    u32x2 yv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) yv[t] = *reinterpret_cast<const u32x2*>(&y_s[((4 * g + t) * 16 + n) * LDY + 4 * wv]);
    f32x4 d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
      const u32x2 yb = {__builtin_amdgcn_perm(yv[1][q >> 1], yv[0][q >> 1], sel), __builtin_amdgcn_perm(yv[3][q >> 1], yv[2][q >> 1], sel)};
      d[q] = YmDot<T>::mfma16(u32x2{cur.s[q >> 1][2 * (q & 1)], cur.s[q >> 1][2 * (q & 1) + 1]}, yb, f32x4{0.f, 0.f, 0.f, 0.f});
    }
    load_s(cur, s2);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      *reinterpret_cast<u32x2*>(&z_s[((4 * g + t) * 16 + n) * LDY + 4 * wv]) = u32x2{ym_pack<T>(d[0][t], d[1][t]), ym_pack<T>(d[2][t], d[3][t])};
    mu_barrier();                                   // Z of the step is whole; nobody reads this step's Y any more
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
      const u32x4 zv = *reinterpret_cast<const u32x4*>(&z_s[((2 * wv + ii) * 16 + n) * LDY + 8 * g]);
#pragma unroll
      for (int nt = 0; nt < NTQ; ++nt) acc[ii][nt] = YmDot<T>::mfma(cur.u[ii][nt], zv, acc[ii][nt]);
    }
    load_u(cur, s2);
  };
  Regs ra, rb;
  load_v(stp(0));
  load_s(ra, stp(0)); load_u(ra, stp(0));
  load_s(rb, stp(min(1, NSTEP - 1))); load_u(rb, stp(min(1, NSTEP - 1)));
  int s = 0;
  for (; s + 1 < NSTEP; s += 2) { step(s, ra); step(s + 1, rb); }
  if (s < NSTEP) step(s, ra);
  mu_barrier();                                     // every wave is through with Z: the tile may go over it

  // the tile (16 rows x 16 Q columns) leaves through LDS in whole rows, as in blast_mixu_kernel
  using V4 = typename TypeTraits<T>::vec4;
  const int OLD = 16 * Q + 8;
  uint16_t* const o_s = one_lds;
  mu_write_out<T>(p, o_s, m0, tid, [&] {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
      for (int nt = 0; nt < NTQ; ++nt) {
        const int q = 16 * nt + 4 * g;
        if (q < Q) {
          V4 o;
#pragma unroll
          for (int t = 0; t < 4; ++t) o[t] = TypeTraits<T>::from_f32(acc[ii][nt][t]);
          *reinterpret_cast<V4*>(&o_s[n * OLD + (2 * wv + ii) * Q + q]) = o;
        }
      }
  });
}

// V (16, P, R) -> Vp (step, j, half of the step's ranks, k step, lane (n, g), 8): element e of lane (n, g) is
// V_j[32 ks + 8 g + e][32 step + 16 half + n], zero past P; then U and S as side_prep_item lays them.  One thread per 16-byte piece.
template <typename T>
__global__ __launch_bounds__(256) void one_prep_kernel(const T* __restrict__ V, T* __restrict__ Vp, int P, int KS, SidePrep s) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t nv = (int64_t)(s.R / 32) * 16 * 2 * KS * 64;
  if (idx < nv) {
    const int l = (int)(idx & 63), n = l & 15, g = l >> 4;
    int64_t c = idx >> 6;
    const int ks = (int)(c % KS); c /= KS;
    const int half = (int)(c & 1); c >>= 1;
    const int j = (int)(c & 15), step = (int)(c >> 4);
    typename TypeTraits<T>::vec8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 32 * ks + 8 * g + e;
      o[e] = k < P ? V[((int64_t)j * P + k) * s.R + 32 * step + 16 * half + n] : (T)0.0f;
    }
    *reinterpret_cast<typename TypeTraits<T>::vec8*>(Vp + idx * 8) = o;
  } else if (idx - nv < s.items) {
    side_prep_item<T>(s, idx - nv);
  }
}

namespace {
template <typename T, int KS>
void* one_fn_ks(int Q) {
  return Q <= 48 ? (void*)blast_one_kernel<T, 3, KS> : (void*)blast_one_kernel<T, 5, KS>;
}
template <typename T>
void* one_fn(int Q, int ks) {
  switch (ks) {
    case 1: return one_fn_ks<T, 1>(Q);
    case 2: return one_fn_ks<T, 2>(Q);
    case 3: return one_fn_ks<T, 3>(Q);
    default: return nullptr;
  }
}
}  // namespace

// out = BLAST(x) for 16 input blocks of at most 96 columns and 16 output blocks of at most 80, U (b, Q, R) or (u_rq) (b, R, Q): one launch after the
// re-laying of V, U and S into scratch (b (32 ceil(P / 32) + Q + b) R elements, each part rounded up to 256 bytes).  The fused
// output stage is taken from `ep`.  Returns BLR_OK, a negative blr_status, or 1 when the shape is not for this kernel.
int blast_one_launch(const void* x, int64_t ldx, const void* U, const void* V, const void* S, void* out, int64_t ldo, const GemmArgs& ep,
                     int M, int in_f, int b, int R, int Q, int64_t s_si, int64_t s_sj, int64_t s_sr, int dtype,
                     void* scratch, size_t scratch_bytes, hipStream_t st, bool u_rq) {
  if (dtype != BLR_F16 && dtype != BLR_BF16) return 1;
  if (b != 16 || in_f % 16) return 1;
  const int P = in_f / 16, KS = (int)cdiv(P, 32);
  if (P % 8 || P > 96 || Q % 8 || Q > 80 || Q < 8 || R % 32 || M < 1) return 1;
  if (!aligned(x, 16) || ldx % 8 || !aligned(U, 16) || !aligned(V, 16) || !aligned(out, 16) || ldo % 8) return 1;
  if ((ep.bias && !aligned(ep.bias, 16)) || (ep.gate && (!aligned(ep.gate, 16) || ep.ld_gate % 8 || ep.gate_rows < 1)) ||
      (ep.resid && (!aligned(ep.resid, 16) || ep.ld_resid % 8))) return 1;
  const int64_t x_elems = (int64_t)(M - 1) * ldx + in_f;
  if (x_elems * 2 >= (int64_t)YM_OOB || (int64_t)b * Q * R * 2 >= (int64_t)YM_OOB || (int64_t)b * b * R * 2 >= (int64_t)YM_OOB ||
      (int64_t)b * 32 * KS * R * 2 >= (int64_t)YM_OOB || cdiv(M, MU_BM) >= 2147483647LL) return 1;
  const size_t vp_bytes = align_up((size_t)b * 32 * KS * R * 2, 256), ut_bytes = align_up((size_t)b * Q * R * 2, 256), sp_bytes = (size_t)b * b * R * 2;
  if (!scratch || scratch_bytes < vp_bytes + ut_bytes + sp_bytes || !aligned(scratch, 16)) return 1;
  void* fn = dtype == BLR_F16 ? one_fn<f16>(Q, KS) : one_fn<bf16>(Q, KS);
  if (!fn) return 1;
  char* sp = reinterpret_cast<char*>(scratch);
  SidePrep job = {};
  job.U = U; job.S = S; job.Ut = sp + vp_bytes; job.Sp = sp + vp_bytes + ut_bytes;
  job.Q = Q; job.R = R; job.u_rq = u_rq ? 1 : 0; job.s_si = s_si; job.s_sj = s_sj; job.s_sr = s_sr;
  job.items = (int64_t)b * (R / 8) * Q + (int64_t)R * 64;
  {
    const int64_t nv = (int64_t)(R / 32) * 16 * 2 * KS * 64;
    const unsigned tg = (unsigned)cdiv(nv + job.items, 256);
    if (dtype == BLR_F16) hipLaunchKernelGGL(one_prep_kernel<f16>, dim3(tg), dim3(256), 0, st, (const f16*)V, (f16*)sp, P, KS, job);
    else hipLaunchKernelGGL(one_prep_kernel<bf16>, dim3(tg), dim3(256), 0, st, (const bf16*)V, (bf16*)sp, P, KS, job);
    BLR_CHECK_LAUNCH("one_prep");
  }
  OneParams p = {};
  p.x = x; p.ldx = ldx; p.x_bytes = (uint32_t)(x_elems * 2); p.Vp = sp; p.Sp = job.Sp; p.Ut = job.Ut; p.out = out; p.ldo = ldo;
  p.M = M; p.P = P; p.R = R; p.Q = Q;
  p.bias = ep.bias; p.act = ep.act; p.gate = ep.gate; p.gate_rows = ep.gate ? ep.gate_rows : 1; p.ld_gate = ep.ld_gate;
  p.resid = ep.resid; p.ld_resid = ep.ld_resid;
  void* args[] = {&p};
  hipError_t e = hipLaunchKernel(fn, dim3((unsigned)cdiv(M, MU_BM)), dim3(MU_NT), args, 0, st);
  if (e != hipSuccess) { set_error("blast_one: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  return BLR_OK;
}

}  // namespace blr

#ifdef BLR_TRACE
extern "C" int blr_debug_trace6(unsigned long long* host, int n) {
  return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(blr::g_trace6), (size_t)n * 8, 0, hipMemcpyDeviceToHost);
}
#endif
