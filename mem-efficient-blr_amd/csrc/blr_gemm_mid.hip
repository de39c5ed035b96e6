// Batched GEMM for problems that do not fill the chip with the tiles of blr_gemm.hip: a few hundred rows, layers of a thousand
// columns, long reductions on few tiles.
//
// What bounds such a problem is the time one workgroup takes from its launch to its last store, not the chip's rate: with
// 128 x 128 tiles a 279 x 768 x 3072 product runs on 18 workgroups, each of which streams 1.5 MB through its compute unit's
// path from the L2 (about 110 B/ns) one stage after the other.  Here the tiles are small (32 x 64, 64 x 64, 64 x 128), so that
// there are several times as many workgroups with less to stream each, and the eight waves of a workgroup that a small tile does
// not need next to each other split its reduction: KG groups of waves own every KG-th stage of 64 k, each with a ring of its own
// in LDS (all groups together keep 128 - 144 KB of loads in flight), and meet in LDS once, at the end, in fp32 and in fixed order.
// Stages are filled by global_load_lds as in gemm_ring64_kernel, with the same layouts: a K-contiguous operand as 128 bytes of each
// of 8 rows per instruction, chunk c of row r at position c ^ (r & 7); a (k, n) operand as it lies, read back transposed.
#include <algorithm>
#include <mutex>
#include <set>
#include <type_traits>
#include "blr_common.h"
#include "blr_gemm_dev.h"
#include "blr_ring_dev.h"

namespace blr {
namespace {

// What differs between the 2-byte types and fp32: a stage is 128 bytes of k (64 or 32 values), a chunk 16 bytes (8 or 4).  fp32 runs
// on v_mfma_f32_32x32x2_f32 (fp32 products and sums; 256 flop per clock and compute unit, twice what the vector units do without
// packed instructions): product e of a sub-step takes value e of the lanes' chunks, so lane half h adds k = 4 (2 q + h) + e.
template <typename T> struct MidType {
  using V = typename TypeTraits<T>::vec8;
  static __device__ __forceinline__ f32x16 mul(V b, V a, f32x16 c) { return TypeTraits<T>::mfma32(b, a, c); }
};
template <> struct MidType<float> {
  using V = f32x4;
  static __device__ __forceinline__ f32x16 mul(V b, V a, f32x16 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(b[e], a[e], c, 0, 0, 0);
    return c;
  }
};

// (k, n) stage: position of 16-byte chunk c of row k is c ^ mid_swz(k): the four rows that a transposing read touches then lie in
// four different 32-byte groups of banks
// (fp32 reads single values, neighbouring lanes along n: nothing to spread)
template <typename T, int BN> __device__ __forceinline__ int mid_swz(int k) { return sizeof(T) == 4 ? 0 : BN == 32 ? ((k >> 1) & 1) << 1 : (k & 3) << 1; }

template <int BM, int BN, int KG, int NST>
constexpr size_t mid_lds_bytes() {
  size_t ring = (size_t)KG * NST * (BM + BN) * 128, red = (size_t)KG * BM * (BN + 4) * 4;
  return ring > red ? ring : red;
}

template <int LPW, int NST>
__device__ __forceinline__ void mid_wait(int later) {              // all but the loads of the `later` stages behind this one have landed
  if constexpr (NST >= 7) if (later >= 5) { __builtin_amdgcn_s_waitcnt(ring_vmcnt(5 * LPW)); return; }
  if constexpr (NST >= 6) if (later >= 4) { __builtin_amdgcn_s_waitcnt(ring_vmcnt(4 * LPW)); return; }
  if constexpr (NST >= 5) if (later >= 3) { __builtin_amdgcn_s_waitcnt(ring_vmcnt(3 * LPW)); return; }
  if constexpr (NST >= 4) if (later >= 2) { __builtin_amdgcn_s_waitcnt(ring_vmcnt(2 * LPW)); return; }
  if constexpr (NST >= 3) if (later >= 1) { __builtin_amdgcn_s_waitcnt(ring_vmcnt(LPW)); return; }
  __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));
}

// PARTIAL: the batch index counts slices of the reduction (g.kc values of k each); fp32 partial sums go to C.
template <typename T, bool B_KN, int BM, int BN, int TM, int TN, int KG, int NST, bool PIPE, bool EP, bool PARTIAL>
__global__ __launch_bounds__((BM / 32 / TM) * (BN / 32 / TN) * KG * 64) void gemm_mid_kernel(GemmArgs g, int tiles_m, int tiles_n, int per_xcd, int c_vec, int side_wgs) {
  constexpr int WGN = BN / 32 / TN, WPG = (BM / 32 / TM) * WGN, NT = WPG * KG * 64;
  constexpr int CH = TM * TN == 1 ? 2 : 1;                           // a single 32 x 32 block: even and odd sub-steps as two chains
  constexpr int GSTG = (BM + BN) * 128, LA = BM / 8, LPW = (LA + BN / 8) / WPG;
  constexpr int ES = sizeof(T), KS = 128 / ES, CE = 16 / ES;         // bytes of a value, k per stage, values per chunk
  constexpr int RB = BN * ES, CPR = RB / 16, RPI = 1024 / RB;        // (k, n) operand: bytes and chunks of a k row, rows per load
  using V8 = typename MidType<T>::V;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / WPG, w = wave % WPG, wm = w / WGN, wn = w % WGN;
  // an XCD gets a contiguous run of tiles, the row tiles of one column tile next to each other: they share its weights in the L2
  const int tiles = tiles_m * tiles_n;
  int u = blockIdx.x;
  if (u < side_wgs) {                                                // the first workgroups carry the side job, if there is one
    if constexpr (ES == 2)
      for (int64_t idx = (int64_t)u * NT + tid; idx < g.side.items; idx += (int64_t)side_wgs * NT) side_prep_item<T>(g.side, idx);
    return;
  }
  u -= side_wgs;
  u = (u & 7) * per_xcd + (u >> 3);
  if (u >= tiles * g.batch) return;
  const int bt = g.cn != 1 ? u % g.batch : u / tiles;                // interleaved columns: the batches of a tile fill each other's lines
  const int ut = g.cn != 1 ? u / g.batch : u - bt * tiles;
  const int m0 = (ut % tiles_m) * BM, n0 = (ut / tiles_m) * BN;

  const int Kloc = PARTIAL ? min(g.kc, g.K - bt * g.kc) : g.K;
  const int KT = (Kloc + KS - 1) / KS, ktail = Kloc % KS;             // a partial last stage holds ktail k, whole chunks
  const int mine = KT > kg ? (KT - kg + KG - 1) / KG : 0;            // stages of this group
  const int steps = (KT + KG - 1) / KG;

  const char* Ab0 = reinterpret_cast<const char*>(g.A) + (int64_t)bt * g.sA * ES;
  const char* Bb0 = reinterpret_cast<const char*>(g.B) + (int64_t)bt * g.sB * ES;
  T* C = reinterpret_cast<T*>(g.C);

  // load li of this wave: rows 8 idx .. of A for idx = li * WPG + w < LA, else instruction idx - LA of the B stage
  const int r8 = lane >> 3, c8 = (lane & 7) ^ r8;
  const int cmax = max(ktail / CE - 1, 0), rmax = max(ktail - 1, 0);
  const uint32_t tail_kc = (uint32_t)((c8 - min(c8, cmax)) * 16);    // what to step back by in a partial stage, to re-fetch valid values
  uint32_t off[LPW], tail[LPW];
#pragma unroll
  for (int li = 0; li < LPW; ++li) {
    const int idx = li * WPG + w;
    if (idx < LA) {
      off[li] = (uint32_t)(min(m0 + idx * 8 + r8, g.M - 1) * g.lda * ES + c8 * 16);
      tail[li] = tail_kc;
    } else if (B_KN) {
      const int krow = (idx - LA) * RPI + lane / CPR, chunk = (lane % CPR) ^ mid_swz<T, BN>(krow);
      off[li] = (uint32_t)(krow * g.ldb * ES + min(n0 + chunk * CE, g.N - CE) * ES);
      tail[li] = (uint32_t)((krow - min(krow, rmax)) * g.ldb * ES);
    } else {
      off[li] = (uint32_t)(min(n0 + (idx - LA) * 8 + r8, g.N - 1) * g.ldb * ES + c8 * 16);
      tail[li] = tail_kc;
    }
  }
  const uint32_t lds0 = ring_lds_addr(smem + kg * (NST * GSTG) + w * 1024);

  // fragment addresses inside a stage: see gemm_ring64_kernel
  const int half = lane >> 5;
  uint32_t rowA[TM], rowB[TN], xo[4];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int ra = (wm * TM + i) * 32 + (lane & 31);
    rowA[i] = (uint32_t)(((ra >> 3) << 10) + ((ra & 7) << 7));
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    if (B_KN && ES == 4) {
      rowB[j] = (uint32_t)(BM * 128 + half * 4 * RB + ((wn * TN + j) * 32 + (lane & 31)) * 4);
    } else if (B_KN) {
      const int g4 = lane >> 4, i16 = lane & 15, chunk = (wn * TN + j) * 4 + (g4 & 1) * 2 + ((i16 & 3) >> 1);
      rowB[j] = (uint32_t)(BM * 128 + ((g4 >> 1) * 8 + (i16 >> 2)) * RB + (i16 & 1) * 8 + ((chunk ^ mid_swz<T, BN>(i16 >> 2)) << 4));
    } else {
      const int rb = (wn * TN + j) * 32 + (lane & 31);
      rowB[j] = (uint32_t)(BM * 128 + ((rb >> 3) << 10) + ((rb & 7) << 7));
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) xo[q] = (uint32_t)(((2 * q + half) ^ (lane & 7)) << 4);

  constexpr int NV = (BM * BN / 8 + NT - 1) / NT;                    // 8-column pieces of the tile per thread
  typedef T out8 __attribute__((ext_vector_type(8)));
  out8 first[NV];                                                    // a pair: silu(first tile), kept for the second
  const int halves = (EP && !PARTIAL && g.pair) ? 2 : 1;
  for (int hf = 0; hf < halves; ++hf) {
    const char* Ab = Ab0 + (int64_t)hf * g.pair_dA * ES;
    const char* Bb = Bb0 + (int64_t)hf * g.pair_dB * ES;
    auto issue = [&](int step, int li) {                             // load li of this group's stage number `step`
      const int s = step * KG + kg, slot = step % NST;
      const bool partial = ktail && s == KT - 1, isA = li * WPG + w < LA;
      const char* base = isA ? Ab + (int64_t)s * 128 : Bb + (B_KN ? (int64_t)s * KS * g.ldb * ES : (int64_t)s * 128);
      ring_load_lds(base, off[li] - (partial ? tail[li] : 0u), lds0 + slot * GSTG + li * (WPG * 1024));
    };
    f32x16 acc[CH][TM][TN];
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[c][i][j][e] = 0.0f;
    constexpr int SETS = PIPE ? 2 : 1;
    V8 af[SETS][4][TM], bf[SETS][4][TN];                             // fragments of a stage (PIPE: of two), four sub-steps of 16 k each
    auto frags = [&](int step, int q, int set) {
      const unsigned char* st = smem + kg * (NST * GSTG) + (step % NST) * GSTG;
#pragma unroll
      for (int i = 0; i < TM; ++i) af[set][q][i] = *reinterpret_cast<const V8*>(st + rowA[i] + xo[q]);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (B_KN && ES == 4) {
#pragma unroll
          for (int e = 0; e < 4; ++e) bf[set][q][j][e] = *reinterpret_cast<const float*>(st + rowB[j] + (q * 8 + e) * RB);
        } else if constexpr (B_KN) {
          union { V8 v; s16x4 h[2]; } x;
          x.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(st + rowB[j] + (q * 16) * RB));
          x.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(st + rowB[j] + (q * 16 + 4) * RB));
          bf[set][q][j] = x.v;
        } else {
          bf[set][q][j] = *reinterpret_cast<const V8*>(st + rowB[j] + xo[q]);
        }
      }
    };
    auto zero_tail = [&](int t, int set) {                           // what a partial stage lacks is zero on both sides (one alone would make
      if (!(ktail && t * KG + kg == KT - 1)) return;                 // NaN of an infinity that was fetched again)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if ((2 * q + half) * CE >= ktail) {
#pragma unroll
          for (int e = 0; e < CE; ++e) {
#pragma unroll
            for (int i = 0; i < TM; ++i) af[set][q][i][e] = (T)0.0f;
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[set][q][j][e] = (T)0.0f;
          }
        }
    };
    auto products = [&](int q, int set) {                            // (operands swapped: a lane gets runs of four columns of a row)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[q % CH][i][j] = MidType<T>::mul(bf[set][q][j], af[set][q][i], acc[q % CH][i][j]);
    };
    constexpr int AHEAD = PIPE ? NST : NST - 1;                      // stages asked for before the loop
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
      if (s < mine)
#pragma unroll
        for (int li = 0; li < LPW; ++li) issue(s, li);
    if constexpr (!PIPE) {
      // One barrier per step: stage t has landed, stage t - 1 has been read by everybody and its slot may be filled again.  Short
      // reductions (a few steps per group) want this form: little code to fetch, and the tile is over before a pipeline would fill.
      for (int t = 0; t < steps; ++t) {
        if (t < mine) mid_wait<LPW, NST>(min(mine - 1 - t, NST - 2));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (WPG > 1) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (t + NST - 1 < mine)
#pragma unroll
          for (int li = 0; li < LPW; ++li) issue(t + NST - 1, li);
        if (t < mine) {
#pragma unroll
          for (int q = 0; q < 4; ++q) frags(t, q, 0);
          zero_tail(t, 0);
#pragma unroll
          for (int q = 0; q < 4; ++q) products(q, 0);
        }
      }
    } else {
      // Step t: the products of stage t, whose fragments are in registers, with the fragment reads of stage t + 1 and the loads of
      // stage t + NST between them; before them the step's one barrier: stage t + 1 has landed, stage t has been read by everybody.
      // MAIN: every group has all of these stages.
      auto step_body = [&](int t, auto main_c, auto set_c) {
        constexpr bool MAIN = decltype(main_c)::value;
        constexpr int set = decltype(set_c)::value;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (MAIN) __builtin_amdgcn_s_waitcnt(ring_vmcnt((NST - 2) * LPW));
        else if (t + 1 < mine) mid_wait<LPW, NST>(min(mine - 2 - t, NST - 2));
        if (WPG > 1) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const bool live = MAIN || t < mine, more = MAIN || t + NST < mine;
        if (!MAIN) zero_tail(t, set);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (more) {
#pragma unroll
            for (int li = q * LPW / 4; li < (q + 1) * LPW / 4; ++li) issue(t + NST, li);
          }
          __builtin_amdgcn_sched_barrier(0);
          frags(t + 1, q, set ^ 1);
          if (live) products(q, set);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      using std::false_type; using std::true_type;
      typedef std::integral_constant<int, 0> set0; typedef std::integral_constant<int, 1> set1;
      if (mine > 0) mid_wait<LPW, NST + 1>(min(mine - 1, NST - 1));
      if (WPG > 1) __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int q = 0; q < 4; ++q) frags(0, q, 0);
      int t = 0;
      for (; t + 2 + NST <= KT / KG; t += 2) {                         // (both steps' loads exist in every group)
        step_body(t, true_type{}, set0{});
        step_body(t + 1, true_type{}, set1{});
      }
      for (; t < steps; t += 2) {
        step_body(t, false_type{}, set0{});
        step_body(t + 1, false_type{}, set1{});
      }
    }
    // the groups' sums meet in LDS
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
    constexpr int LD = BN + 4;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = CH == 2 ? acc[0][i][j][4 * q + e] + acc[CH - 1][i][j][4 * q + e] : acc[0][i][j][4 * q + e];
          *reinterpret_cast<f32x4*>(&red[(kg * BM + (wm * TM + i) * 32 + (lane & 31)) * LD + (wn * TN + j) * 32 + q * 8 + half * 4]) = v;
        }
    __syncthreads();
    if (PARTIAL || c_vec) {
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const int v = tid + n * NT, row = v / (BN / 8), col = (v % (BN / 8)) * 8, gr = m0 + row, gc = n0 + col;
        if (v >= BM * BN / 8 || gr >= g.M || gc >= g.N) continue;
        f32x4 s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < KG; ++k) {
          s0 += *reinterpret_cast<const f32x4*>(&red[(k * BM + row) * LD + col]);
          s1 += *reinterpret_cast<const f32x4*>(&red[(k * BM + row) * LD + col + 4]);
        }
        if (PARTIAL) {
          float* P = reinterpret_cast<float*>(g.C) + (int64_t)bt * g.sC + (int64_t)gr * g.ldc + gc;
          *reinterpret_cast<f32x4*>(P) = s0;
          *reinterpret_cast<f32x4*>(P + 4) = s1;
          continue;
        }
        out8 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = TypeTraits<T>::from_f32(g.sat8 ? sat8_rne(s0[e]) : s0[e]);
          o[4 + e] = TypeTraits<T>::from_f32(g.sat8 ? sat8_rne(s1[e]) : s1[e]);
        }
        const int64_t in_row = (int64_t)bt * g.sC + gc;
        if constexpr (EP && ES == 2) {
          if (hf == 0) o = ep_vector<T>(g, o, in_row, gr);
          else {
            out8 up[1] = {o};
            const int64_t at[1] = {in_row + g.pair_dbias};
            const T* const c[1] = {reinterpret_cast<const T*>(&first[n])};
            ep_pair_up<T, 1>(g, up, at, c);
            o = up[0];
          }
          if (hf + 1 < halves) { first[n] = o; continue; }
        }
        if (g.epi == EPI_MONARCH_SCATTER) {
          const int d = gc / g.per;
          *reinterpret_cast<out8*>(&C[(int64_t)d * g.sL + (int64_t)gr * g.ldc + (int64_t)bt * g.per + (gc - d * g.per)]) = o;
        } else {
          *reinterpret_cast<out8*>(&C[in_row + (int64_t)gr * g.ldc]) = o;
        }
      }
    } else {
      for (int v = tid; v < BM * BN; v += NT) {                      // lanes along the columns
        const int row = v / BN, col = v % BN, gr = m0 + row, gc = n0 + col;
        if (gr >= g.M || gc >= g.N) continue;
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < KG; ++k) s += red[(k * BM + row) * LD + col];
        const int64_t o = epi_offset(g, bt, gr, gc);
        T r = TypeTraits<T>::from_f32(g.sat8 ? sat8_rne(s) : s);
        if (EP) r = ep_value<T>(g, r, o - (int64_t)gr * g.ldc, gr);
        C[o] = r;
      }
    }
    if (hf + 1 < halves) __syncthreads();                            // the sums have been read: the rings may be filled again
  }
}

template <typename T, int BM, int BN, int TM, int TN, int KG, int NST, bool PIPE, bool PARTIAL>
int launch_mid(const GemmArgs& g, hipStream_t st) {
  int tiles_m = (int)cdiv(g.M, BM), tiles_n = (int)cdiv(g.N, BN);
  const int64_t total = (int64_t)tiles_m * tiles_n * g.batch;
  if (total > (1ll << 30)) { set_error("gemm: too many tiles"); return BLR_ERR_UNSUPPORTED; }
  constexpr size_t lds = mid_lds_bytes<BM, BN, KG, NST>();
  constexpr int NT = (BM / 32 / TM) * (BN / 32 / TN) * KG * 64;
  const bool ep = g.bias || g.act || g.gate || g.resid;
  void* fn;
  if constexpr (PARTIAL) fn = g.b_kn ? (void*)gemm_mid_kernel<T, true, BM, BN, TM, TN, KG, NST, PIPE, false, true> : (void*)gemm_mid_kernel<T, false, BM, BN, TM, TN, KG, NST, PIPE, false, true>;
  else
    fn = ep ? (g.b_kn ? (void*)gemm_mid_kernel<T, true, BM, BN, TM, TN, KG, NST, PIPE, true, false> : (void*)gemm_mid_kernel<T, false, BM, BN, TM, TN, KG, NST, PIPE, true, false>)
            : (g.b_kn ? (void*)gemm_mid_kernel<T, true, BM, BN, TM, TN, KG, NST, PIPE, false, false> : (void*)gemm_mid_kernel<T, false, BM, BN, TM, TN, KG, NST, PIPE, false, false>);
  static std::mutex mu;
  static std::set<void*> raised;
  {
    std::lock_guard<std::mutex> lk(mu);
    if (!raised.count(fn)) {
      hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) { set_error("gemm: cannot raise LDS limit: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
      raised.insert(fn);
    }
  }
  // 8-column pieces of the result as one store
  int c_vec = (sizeof(T) == 2 || !ep) && g.cn == 1 && g.N % 8 == 0 && aligned(g.C, 8 * sizeof(T)) && g.ldc % 8 == 0 && g.sC % 8 == 0 &&
              (!g.bias || aligned(g.bias, 16)) && (!g.gate || (aligned(g.gate, 16) && g.ld_gate % 8 == 0)) && (!g.resid || (aligned(g.resid, 16) && g.ld_resid % 8 == 0)) &&
              (g.epi == EPI_PLAIN || (g.per % 8 == 0 && g.sL % 8 == 0));
  int per_xcd = (int)cdiv(total, 8), side_wgs = 0;
  if (!PARTIAL && sizeof(T) == 2 && g.side.items > 0 && g.side_taken) side_wgs = (int)std::min<int64_t>(cdiv(cdiv(g.side.items, NT), 8) * 8, 4096);
  GemmArgs ga = g;
  void* args[] = {&ga, &tiles_m, &tiles_n, &per_xcd, &c_vec, &side_wgs};
  hipError_t e = hipLaunchKernel(fn, dim3((unsigned)(per_xcd * 8 + side_wgs)), dim3(NT), args, lds, st);
  if (e != hipSuccess) { set_error("gemm_mid: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  if (side_wgs > 0) *g.side_taken = 1;
  return BLR_OK;
}

template <typename T, bool PARTIAL>
int mid_kind_launch(const GemmArgs& g, int kind, hipStream_t st) {
  switch (kind) {
    case MID_32_64: if constexpr (!PARTIAL) return launch_mid<T, 32, 64, 1, 1, 4, 2, false, false>(g, st); break;
    case MID_32_64_DEEP: return launch_mid<T, 32, 64, 1, 1, 4, 3, false, PARTIAL>(g, st);
    case MID_64_64: if constexpr (!PARTIAL) return launch_mid<T, 64, 64, 1, 1, 2, 2, false, false>(g, st); break;
    case MID_64_64_DEEP: return launch_mid<T, 64, 64, 1, 1, 2, 4, false, PARTIAL>(g, st);
    case MID_64_128: return launch_mid<T, 64, 128, 2, 1, 2, 3, true, PARTIAL>(g, st);
  }
  set_error("gemm_mid: no kernel for tile kind %d%s", kind, PARTIAL ? " in slices" : "");
  return BLR_ERR_UNSUPPORTED;
}

// What a launch of each kind takes, in microseconds: t = c0 + c1 k + (c2 + c3 k) min(f, o) + (c4 + c5 k) G, with k = thousands of k
// per slice, f = tiles * slices / compute units, o the workgroups that share a compute unit, G what is left after the first round
// of f / o (the mean of the whole rounds and the tiles it stands for); slices add c6 + c7 per million results for the launch
// that adds them up.  Fitted (non-negative, on relative errors) to HIP-graph timings of 210 products of 129 .. 4096 rows, 72 .. 8192
// columns and 64 .. 11008 k on every kind: 6 - 11 % rms each.  The kind with the smallest estimate was within 1 % of the best of
// all kinds in the mean (22 % at worst), and 1.73 x faster in the mean than 128 x 128 and 256 x 128 tiles with their old rule
// (768 x 768 at 279 rows 12.7 -> 4.9 us, 3072 x 768 19.2 -> 9.5, 2048 x 2048 at 1000 rows 26.5 -> 15.7; 80 columns of k = 8672 at
// 154 rows 20.5 -> 8.6 us).
struct MidModel { int bm, bn, occ, split; float c[8]; };
const MidModel kMidModel[MID_KINDS] = {
    {32, 64, 1, 0, {2.43f, 2.82f, 0.51f, 1.75f, 1.42f, 3.90f, 0.f, 0.f}},          // MID_32_64
    {32, 64, 1, 1, {2.94f, 2.52f, 0.52f, 0.96f, 1.73f, 3.23f, 2.37f, 1.68f}},      // MID_32_64_DEEP
    {64, 64, 2, 0, {2.24f, 4.70f, 1.00f, 1.56f, 0.70f, 4.09f, 0.f, 0.f}},          // MID_64_64
    {64, 64, 1, 1, {2.93f, 3.71f, 0.87f, 0.79f, 1.78f, 5.02f, 2.42f, 2.18f}},      // MID_64_64_DEEP
    {64, 128, 1, 1, {4.26f, 4.41f, 1.51f, 1.41f, 3.43f, 6.69f, 2.52f, 1.97f}},     // MID_64_128
    {128, 128, 1, 0, {4.65f, 6.41f, 1.09f, 2.17f, 4.43f, 10.41f, 0.f, 0.f}},       // MID_RING_128
    {128, 128, 2, 0, {3.42f, 8.89f, 1.66f, 4.26f, 1.95f, 5.93f, 0.f, 0.f}},        // MID_RING_128_TWO
    {256, 128, 1, 2, {7.44f, 13.55f, 1.53f, 1.98f, 0.f, 0.f, 0.f, 1.34f}},         // MID_RING_256_SLICES: fitted with its reduction, in slices only
};

float mid_estimate(int kind, int M, int N, int K, int batch, int slices, int cus) {
  const MidModel& m = kMidModel[kind];
  const float f = (float)(cdiv(M, m.bm) * cdiv(N, m.bn) * batch * slices) / cus, o = (float)m.occ;
  const float k = (float)(cdiv(cdiv(K, slices), 64) * 64) * 1e-3f, in = std::min(f, o);
  const float G = 0.5f * ((float)((int64_t)((f + o - 1e-4f) / o) - 1) * o + std::max(0.f, f - o));
  float t = m.c[0] + m.c[1] * k + (m.c[2] + m.c[3] * k) * in + (m.c[4] + m.c[5] * k) * std::max(0.f, G);
  if (slices > 1) t += m.c[6] + m.c[7] * (float)slices * M * N * 1e-6f;
  return t;
}

}  // namespace

// The kind of kernel and the number of slices of K for a product whose 128 x 128 tiles do not fill the chip; ring: whether the ring
// kernels take it, slices: whether the reduction may be cut (a plain single product with scratch for the partial sums).
MidPlan gemm_mid_plan(int M, int N, int K, int batch, bool ring, bool mid, bool slices) {
  const int cus = device_cus() > 0 ? device_cus() : 256;
  MidPlan best = {-1, 1, K};
  float t_best = 1e30f;
  for (int kind = 0; kind < MID_KINDS; ++kind) {
    const MidModel& m = kMidModel[kind];
    const bool is_ring = kind >= MID_RING_128;
    if (is_ring ? !ring : !mid) continue;
    for (int s = m.split == 2 ? 2 : 1; s <= (m.split && slices ? 12 : 1); ++s) {
      // slices of at least 192 k (ring: 512), no more of them than fill the compute units once
      if (s > 1 && (K / s < (is_ring ? 512 : 192) || cdiv(M, m.bm) * cdiv(N, m.bn) * s > cus)) break;
      if (is_ring && s > 8) break;
      const float t = mid_estimate(kind, M, N, K, batch, s, cus);
      if (t < t_best) { t_best = t; best = {kind, s, (int)(cdiv(cdiv(K, s), 64) * 64)}; }
    }
  }
  if (best.kind >= 0) best.slices = (int)cdiv(K, best.kc);           // (whole stages of 64 k may need fewer)
  return best;
}

bool gemm_mid_ok(const GemmArgs& g, int dtype) {
  const int es = dtype == BLR_F32 ? 4 : 2, ce = 16 / es;            // values per 16-byte chunk
  if (g.N < ce || g.K < ce || g.K % ce || (g.b_kn && g.N % ce)) return false;
  if (g.epi != EPI_PLAIN && (g.bias || g.act || g.gate || g.resid)) return false;
  if (!aligned(g.A, 16) || !aligned(g.B, 16) || g.lda % ce || g.sA % ce || g.ldb % ce || g.sB % ce) return false;
  if (g.pair && (es == 4 || g.cn != 1 || g.pair_dA % 8 || g.pair_dB % 8 || g.pair_dbias % 8 || g.N % 8 || !aligned(g.C, 16) || g.ldc % 8 || g.sC % 8 || (g.bias && !aligned(g.bias, 16)) || g.epi != EPI_PLAIN)) return false;
  const int64_t lim = (int64_t)1 << 32;                               // per-lane offsets are 32 bits
  return (int64_t)(g.M - 1) * g.lda * es + 128 < lim && (g.b_kn ? 63 * g.ldb * es + (int64_t)g.N * es < lim : (int64_t)(g.N - 1) * g.ldb * es + 128 < lim);
}

int gemm_mid_launch(const GemmArgs& g, int kind, bool partial, int dtype, hipStream_t st) {
  if (partial) return dtype == BLR_F16 ? mid_kind_launch<f16, true>(g, kind, st) : mid_kind_launch<bf16, true>(g, kind, st);
  return dtype == BLR_F16 ? mid_kind_launch<f16, false>(g, kind, st) : mid_kind_launch<bf16, false>(g, kind, st);
}

// fp32 at every size.  The matrix pipe bounds it: a compute unit adds 64 columns x 32 rows x 1000 k in 6.7 us, so a reduction on few
// tiles is cut into slices while that saves more than the launch that adds them costs.  Against the 64 x 64 kernel on the vector
// units that is still there for operands without 16-byte alignment: 128 x 128 x 192 25 -> 6 us, 35 x 768 x 3072 325 -> 11 us,
// 1024 x 22016 x 4096 3886 -> 1492 us (47 -> 124 TFLOP/s of the 154 that a library product of 8192 cubed reaches).
int gemm_mid_f32_slices(int M, int N, int K) {
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const int64_t tiles = cdiv(M, 32) * cdiv(N, 64);
  int best = 1;
  float t_best = 1e30f;
  for (int s = 1; s <= 16 && (s == 1 || (tiles * s <= cus && K / s >= 128)); ++s) {
    const float t = 6.7e-3f * K / s + (s > 1 ? 2.5f + 2.f * s * M * N * 1e-6f : 0.f);
    if (t < t_best) { t_best = t; best = s; }
  }
  return best > 1 ? (int)cdiv(K, cdiv(cdiv(K, best), 32) * 32) : 1;
}

int gemm_mid_f32_launch(const GemmArgs& g, bool partial, hipStream_t st) {
  if (partial) return launch_mid<float, 32, 64, 1, 1, 4, 3, false, true>(g, st);
  const int cus = device_cus() > 0 ? device_cus() : 256, mid = option_value(OPT_GEMM_MID, 1);
  // 64 x 64 tiles halve the operand traffic and run two workgroups per compute unit (1024 x 22016 x 4096: 124 TFLOP/s against 94);
  // with less than three for every four compute units the smaller tile spreads further (753 x 1152 x 1152, 216 tiles: 26.6 against
  // 30.8 us; 128 x 3072 x 768, 96 tiles: 18.6 against 12.3 us)
  if (mid == 3 || (mid == 1 && cdiv(g.M, 64) * cdiv(g.N, 64) * g.batch * 4 < 3 * cus)) return launch_mid<float, 32, 64, 1, 1, 4, 3, false, false>(g, st);
  return launch_mid<float, 64, 64, 1, 1, 2, 2, false, false>(g, st);
}

}  // namespace blr
