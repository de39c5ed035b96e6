// GEMM for products of more tiles than compute units: tiles of 256 rows x 96, 128, .. 352 columns, as wide as fits the output.
//
// The matrix pipe and the board's power limit bound the k loop of every tile here alike (256 x 256 x 64 on a compute unit 1.9 - 2.0 us with
// the whole chip at work, 1.4 us with half of it), and the rest of a product's time is what the tiles lose around it: columns and rows
// that pad a tile, a last round that leaves compute units idle, a tile's first loads (3 - 5 us when every compute unit asks at once) and its way
// out (4 - 5 us).  So:
//   * eleven widths less two: 288 columns are one tile of 288 instead of three of 96 (whose 768 tiles are a round and a half), 1376 are four of 352
//     instead of six of 256 that a ninth of the work pads;
//   * one workgroup of eight waves per compute unit, a wave = 32 rows x the tile's width: 16 TN accumulators, TN <= 11.  Stages of 64 k
//     (whole 128-byte lines, see gemm_ring64_kernel), two of them in LDS;
//   * v_mfma_f32_16x16x32: it reads and writes half the accumulators per product of a 32 x 32 x 16 one, and under the power limit that
//     is time: 4096 x 288 x 576 in 16 batches 34.6 -> 32.6 us, 2048 x 1376 x 1024 123.9 -> 117.7;
//   * fragments of B come out of LDS TN reads ahead of their products through a ring of registers, so nothing is read in bursts and one set is
//     enough;
//   * a workgroup walks its tiles: the last two steps of one load the first two stages of the next, and the way out needs no barrier
//     (a wave turns its own blocks in a piece of LDS beside the ring), so that the next tile's loads land under it: 4096 x 576 x 288 in 16
//     batches 46.8 -> 43.2 us.
// Measured against the 32-k and 64-k ring kernels with their rules, 1818 products of 260 .. 4096 rows, 64 .. 22000 columns, 72 .. 11008 k, 1 .. 16
// batches, weights from memory: 0.83 x the time in the mean (geometric), 0.5 at best, 1.17 at worst (gemm_wide_plan has more).  4096 x 288 x 576 in 16
// batches 49.4 -> 32.6 us (668 TFLOP/s), 2048 x 1024 x 2136 in 3 132.8 -> 76.9, 4096 x 576 x 1000 in 16 60.7 -> 41.4.
#include <mutex>
#include <set>
#include <type_traits>
#include <utility>
#include "blr_common.h"
#include "blr_gemm_dev.h"
#include "blr_ring_dev.h"

namespace blr {

namespace {

template <typename F, int... I> __device__ __forceinline__ void static_for_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void static_for(F&& f) { static_for_(f, std::make_integer_sequence<int, N>{}); }
constexpr int min2(int a, int b) { return a < b ? a : b; }

// ring_load_lds where go is not zero (wave-uniform): the branch stays inside the statement, so that the loop around it is one block
__device__ __forceinline__ void ring_load_lds_if(const void* base, uint32_t off, uint32_t lds, int go) {
  asm volatile("s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 .Lskip%=\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n.Lskip%=:" ::"s"(lds), "v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(go)) : "memory", "scc");
}

constexpr int WIDE_BM = 256;
// (k, n) stage: chunk c of row k lies at position c ^ wide_swz(k).  A transposing read takes 32 bytes of each of rows 8 g .. 8 g + 3, g = 0 .. 3: the four
// rows are to lie in different quarters of the 256 bytes of banks (rows of 64 TN bytes do so by themselves where TN is odd), and
// two of the four groups in the other half of their quarters.
template <int TN> __device__ constexpr int wide_quarter(int k) { return TN % 4 == 0 ? k & 3 : TN % 2 == 0 ? (k >> 1) & 1 : 0; }
template <int TN> __device__ constexpr int wide_swz(int k) { return wide_quarter<TN>(k) << 2 | ((k >> 3) & 1) << 1; }
template <int TN> constexpr int wide_frags() { return TN <= 9 ? TN : TN == 10 ? 5 : 4; }        // fragments of B on their way; divides 4 TN
// What a wave stages at a time on the way out, beside the ring: 32 rows of two 32-column blocks, of one, or 16 rows of one
template <int TN> constexpr int wide_cb() { return TN <= 8 ? 2 : 1; }
template <int TN> constexpr int wide_rows() { return TN <= 10 ? 32 : 16; }
template <int TN> constexpr int wide_out_bytes() { return wide_cb<TN>() * wide_rows<TN>() * 64; }
template <int TN> constexpr size_t wide_lds_bytes() { return 2 * (size_t)(WIDE_BM + 32 * TN) * 128 + 8 * wide_out_bytes<TN>(); }

template <typename T, bool B_KN, int TN, bool EP>
__global__ __launch_bounds__(512, 2) void gemm_wide_kernel(GemmArgs g, int tiles_m, int tiles_n, int per_xcd, int walkers, int side_wgs) {
  constexpr int W = 32 * TN, ASTG = WIDE_BM * 128, STG = ASTG + W * 128;
  constexpr int LA = 4, LB = (TN + 1) / 2, LT = LA + LB;      // 1 KiB loads per wave and stage (TN odd: waves 4..7 have one less)
  constexpr int RB = W * 2, CPR = W / 8;
  constexpr int NBF = wide_frags<TN>(), NS = 4 * TN;
  constexpr int BS = NS - NBF + (NBF > 5 ? 2 : 1), R = NS - BS;     // the step's barrier stands before product BS
  static_assert(NS % NBF == 0, "a stage starts at fragment register 0");
  using V8 = typename TypeTraits<T>::vec8;
  using V4 = typename TypeTraits<T>::vec4;
  typedef const unsigned char __attribute__((address_space(3)))* lds_ptr;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles = tiles_m * tiles_n;
  int u = blockIdx.x;
  if (side_wgs > 0) {
    if (u < side_wgs) {
      for (int64_t idx = (int64_t)u * 512 + tid; idx < g.side.items; idx += (int64_t)side_wgs * 512) side_prep_item<T>(g.side, idx);
      return;
    }
    u -= side_wgs;
  }
  // XCD x owns the tiles x per_xcd .. (x + 1) per_xcd - 1 and walks them with `walkers` workgroups; a pair is two tiles, one after the other
  const int halves = EP && g.pair ? 2 : 1;
  const int xcd = u & 7, t_end = min(per_xcd, tiles * g.batch - xcd * per_xcd);
  int it = u >> 3, hf = 0;                            // the tile whose operands are being asked for
  if (it >= t_end) return;

  T* C = reinterpret_cast<T*>(g.C);
  const int KF = g.K >> 6, ktail = g.K & 63, n = KF + (ktail ? 1 : 0);          // (n >= 2: the launcher checks)
  int bt, m0, n0;
  const char *Ab, *Bb;
  uint32_t a_off[LA], b_off[LB];
  // (lane numbers behind an empty statement: what only the way from one tile to the next needs is not to be kept in registers through the k loop)
  auto fresh_lane = [&]() { int l = lane; asm volatile("" : "+v"(l)); return l; };
  auto locate = [&]() {
    const int lane = fresh_lane();
    const int r8 = lane >> 3, c8 = (lane & 7) ^ r8;   // lane (r8, s8) of a K-contiguous load: row r8 of the instruction's eight, LDS position s8 of its 128 bytes, global chunk s8 ^ r8
    const int v = xcd * per_xcd + it;
    bt = v / tiles;
    const int ut = v - bt * tiles, strip = ut / (4 * tiles_n), rem = ut - strip * 4 * tiles_n, gm = min(4, tiles_m - strip * 4);
    m0 = (strip * 4 + rem % gm) * WIDE_BM;
    n0 = (rem / gm) * W;
    Ab = reinterpret_cast<const char*>(g.A) + ((int64_t)bt * g.sA + (EP ? hf * g.pair_dA : 0)) * 2;
    Bb = reinterpret_cast<const char*>(g.B) + ((int64_t)bt * g.sB + (EP ? hf * g.pair_dB : 0)) * 2;
#pragma unroll
    for (int i = 0; i < LA; ++i) a_off[i] = (uint32_t)(min(m0 + (i * 8 + wave) * 8 + r8, g.M - 1) * g.lda * 2 + c8 * 16);
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      if (B_KN) {
        const int L = (i * 8 + wave) * 64 + lane, krow = L / CPR, chunk = (L % CPR) ^ wide_swz<TN>(krow);
        b_off[i] = (uint32_t)(krow * g.ldb * 2 + min(n0 + chunk * 8, g.N - 8) * 2);
      } else {
        b_off[i] = (uint32_t)(min(n0 + (i * 8 + wave) * 8 + r8, g.N - 1) * g.ldb * 2 + c8 * 16);
      }
    }
#pragma unroll
    for (int i = 0; i < LA; ++i) asm volatile("" : "+v"(a_off[i]));               // (or it keeps the 64-bit products)
#pragma unroll
    for (int i = 0; i < LB; ++i) asm volatile("" : "+v"(b_off[i]));
  };
  const uint32_t lds0 = ring_lds_addr(smem + wave * 1024);
  const int last_b = TN % 2 == 0 || wave < 4 ? 1 : 0;

  const int g4 = lane >> 4, i16 = lane & 15;
  const uint32_t row_a = (uint32_t)((wave * 4 + (i16 >> 3)) * 1024 + (i16 & 7) * 128);
  const uint32_t row_b = B_KN ? 0 : (uint32_t)((i16 >> 3) * 1024 + (i16 & 7) * 128);
  constexpr int NKB = TN % 4 == 0 ? 8 : TN % 2 == 0 ? 4 : 2;
  uint32_t xo[2], kb[NKB];
#pragma unroll
  for (int q = 0; q < 2; ++q) xo[q] = (uint32_t)(((4 * q + g4) ^ (i16 & 7)) << 4);
#pragma unroll
  for (int c = 0; c < NKB; ++c)                       // (16-column block c lies where c ^ (low bits) of the row does)
    kb[c] = (uint32_t)((g4 * 8 + (i16 >> 2)) * RB + (i16 & 3) * 8 + 32 * ((c ^ (wide_quarter<TN>(i16 >> 2) << 1 | (g4 & 1))) - c));
  // A last stage of less than 64 k is the 64 k that end with K: the sub-steps that it shares with the stage before are left out.
  auto k_at = [&](int s) { return min(s * 64, g.K - 64); };
  auto issue = [&](int li, int koff, int slot, int go) {
    if (li < LA) {
      ring_load_lds_if(Ab + (int64_t)koff * 2, a_off[li], lds0 + slot * STG + li * 8192, go);
    } else {
      const char* Bp = B_KN ? Bb + (int64_t)koff * g.ldb * 2 : Bb + (int64_t)koff * 2;
      ring_load_lds_if(Bp, b_off[li - LA], lds0 + slot * STG + ASTG + (li - LA) * 8192, li - LA < LB - 1 ? go : go & last_b);
    }
  };
  f32x4 acc[2 * TN][2];                                // 16-column blocks x 16-row halves
  V8 af[2][2], bf[NBF];
  auto read_a = [&](const unsigned char* st, int q, int set) {
    af[set][0] = *reinterpret_cast<const V8*>(st + row_a + xo[q]);
    af[set][1] = *reinterpret_cast<const V8*>(st + row_a + xo[q] + 2048);
  };
  // (an offset of a (n, k) stage's reads is one register per sub-step and what the instruction holds; left to itself the compiler keeps one per few blocks)
  auto at_b = [&](const unsigned char* st, int q) {
    lds_ptr o = (lds_ptr)st + (ASTG + row_b);
    if (!B_KN) { o += xo[q]; asm volatile("" : "+v"(o)); }
    return o;
  };
  auto read_b = [&](lds_ptr o, int q, int c, int reg) {
    if (B_KN) {
      union { V8 v; s16x4 h[2]; } w;
      const lds_ptr p = o + kb[c % NKB] + (c * 32 + q * 32 * RB);
      w.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(p));
      w.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(p + 4 * RB));
      bf[reg] = w.v;
    } else {
      bf[reg] = *(const V8 __attribute__((address_space(3)))*)(o + c * 2048);
    }
  };
  auto first_frags = [&](const unsigned char* st) {
    read_a(st, 0, 0);
    const lds_ptr o = at_b(st, 0);
#pragma unroll
    for (int i = 0; i < NBF; ++i) read_b(o, 0, i, i);
  };
  auto handover = [&](int stores) {                    // this stage is in registers, the next one has landed
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_wait_loads<2 * TN>(stores);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // One stage.  Products in order of (32 k, 16-column block); fragment i of B sits in register i % NBF and is asked for as soon as product
  // i - NBF has used that register.  Before product BS the last fragments of the stage have been asked for: the step's barrier stands there, and
  // under the products that are left the next stage's first fragments are read and the loads of the stage after that go out into
  // this stage's place.
  auto step = [&](const unsigned char* cur, const unsigned char* nxt, int koff, int slot, int go, int stores) {
    // how many fragments of the next stage have been asked for, and loads of the one after it sent, once slot s is through
    constexpr auto asked = [](int s) { return s < BS ? 0 : s == NS - 1 ? NBF : min2(2 * (s - BS + 1), s - (NS - NBF) + 1); };
    constexpr auto sent = [](int s) { return s < BS ? 0 : ((s - BS + 1) * LT + R - 1) / R; };
    const lds_ptr ob[2] = {at_b(cur, 0), at_b(cur, 1)}, on = at_b(nxt, 0);
    static_for<NS>([&](auto S) {
      constexpr int s = decltype(S)::value, q = s / (2 * TN), c = s % (2 * TN);
      if constexpr (s == BS) handover(stores);
      acc[c][0] = TypeTraits<T>::mfma16(bf[s % NBF], af[q][0], acc[c][0]);
      acc[c][1] = TypeTraits<T>::mfma16(bf[s % NBF], af[q][1], acc[c][1]);
      if constexpr (s + NBF < NS) read_b(ob[(s + NBF) / (2 * TN)], (s + NBF) / (2 * TN), (s + NBF) % (2 * TN), s % NBF);
      if constexpr (c == TN && q == 0) read_a(cur, 1, 1);
      if constexpr (s >= BS) {
        if constexpr (s == BS) read_a(nxt, 0, 0);
        static_for<asked(s) - asked(s - 1)>([&](auto I) { constexpr int i = asked(s - 1) + decltype(I)::value; read_b(on, 0, i, i); });
        static_for<sent(s) - sent(s - 1)>([&](auto I) { issue(sent(s - 1) + decltype(I)::value, koff, slot, go); });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  locate();
#pragma unroll
  for (int li = 0; li < LT; ++li) issue(li, 0, 0, 1);
#pragma unroll
  for (int li = 0; li < LT; ++li) issue(li, k_at(1), 1, 1);
  if (last_b) __builtin_amdgcn_s_waitcnt(ring_vmcnt(LT));
  else __builtin_amdgcn_s_waitcnt(ring_vmcnt(LT - 1));
  __builtin_amdgcn_s_barrier();
  first_frags(smem);
  int slot = 0, stores = 0;
  for (;;) {                                           // tiles
#pragma unroll
    for (int c = 0; c < 2 * TN; ++c) acc[c][0] = acc[c][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int om0 = m0, on0 = n0, ohf = hf, obt = bt;
    const int64_t orow = (int64_t)bt * g.sC;
    int go = 1;
#pragma clang loop unroll(disable)
    for (int t = 0; t < KF; ++t) {
      if (t == n - 2) {                                // from here on the loads are the next tile's
        if (++hf == halves) { hf = 0; it += walkers; }
        go = it < t_end;
        if (go) locate();
      }
      step(smem + slot * STG, smem + (slot ^ 1) * STG, k_at(t < n - 2 ? t + 2 : t + 2 - n), slot, go, stores);
      slot ^= 1;
      stores = 0;
    }
    if (ktail) {
      const unsigned char* cur = smem + slot * STG;
      const int skip = 64 - ktail;                      // k of the last stage that the one before had: a multiple of 8
      static_for<2>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        if (q * 32 + 32 <= skip) return;
        const bool zero = q * 32 + g4 * 8 < skip;       // chunks that the stage before had are zero, on both sides
        read_a(cur, q, q);
        const lds_ptr o = at_b(cur, q);
        if (zero) af[q][0] = af[q][1] = V8{};
        static_for<2 * TN>([&](auto J) {
          constexpr int c = decltype(J)::value;
          read_b(o, q, c, c % NBF);
          if (zero) bf[c % NBF] = V8{};
          acc[c][0] = TypeTraits<T>::mfma16(bf[c % NBF], af[q][0], acc[c][0]);
          acc[c][1] = TypeTraits<T>::mfma16(bf[c % NBF], af[q][1], acc[c][1]);
          if constexpr (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);            // (a few reads ahead, not all of them)
        });
      });
      handover(0);
#pragma unroll
      for (int li = 0; li < LT; ++li) issue(li, k_at(1), slot, go);
      slot ^= 1;
      first_frags(smem + slot * STG);
    }

    // Out: a wave's 32 rows go through a piece of LDS of its own, one or two 32-column blocks at a time; nothing waits for the other waves, and
    // the next tile's first stages are on their way meanwhile.
    constexpr int CB = EP && TN > 6 ? 1 : wide_cb<TN>(), RH = wide_rows<TN>(), HP = 32 / RH;      // (an output stage needs registers)
    const int lane = fresh_lane();
    unsigned char* const cs = smem + 2 * STG + wave * wide_out_bytes<TN>();
    T* const crow = C + orow + (int64_t)(om0 + wave * 32) * g.ldc + on0;        // (wave-uniform; the rest of an address is 32 bits)
    constexpr int NP = (TN + CB - 1) / CB;
    constexpr bool EARLY = TN <= 6;
    constexpr int AHEAD = TN <= 10 ? 1 : 0;
    // A lane's pieces of a pass are the same eight columns of several rows, so their bias is one load, asked for a pass ahead; what differs from
    // row to row - gate, residual, the first half of a pair - is asked for before the pass turns its blocks, where registers are left.  (Everything asked for
    // when it was needed: 4096 x 216 x 288 in 16 batches with a bias 27.2 us, without 18.5.)
    V8 bias[1 + AHEAD] = {};
    auto ask_bias = [&](auto P) {
      constexpr int p = decltype(P)::value, j0 = p * CB, PR = 4 * (TN - j0 < CB ? TN - j0 : CB);
      if (g.bias) bias[p & AHEAD] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.bias) + orow + (ohf ? g.pair_dbias : 0) + min(on0 + j0 * 32 + (lane % PR) * 8, g.N - 8));
    };
    if constexpr (EP && AHEAD) ask_bias(std::integral_constant<int, 0>{});
    static_for<NP>([&](auto P) {
      constexpr int j0 = decltype(P)::value * CB, B = TN - j0 < CB ? TN - j0 : CB;
      constexpr int PR = 4 * B, U = RH * PR / 64;        // 16-byte pieces per row, and per lane
      if constexpr (EP && decltype(P)::value + AHEAD < NP) ask_bias(std::integral_constant<int, decltype(P)::value + AHEAD>{});
      // piece c of a row lies at c ^ f(row): both the writes (32 rows, 8 bytes each) and the reads (whole rows) meet every bank equally often
      auto place = [&](int row, int c) { return row * (PR * 16) + ((c ^ (B == 2 ? (row >> 1) & 7 : (row >> 2) & 3)) << 4); };
      static_for<HP>([&](auto H) {
        constexpr int h = decltype(H)::value;
        const int c = lane % PR, col = j0 * 32 + c * 8, row0 = h * RH + lane / PR;
        V8 gv[U], rv[U];                               // (positions outside the result take the operands of its last piece)
        auto ask_rows = [&]() {
#pragma unroll
          for (int x = 0; x < U; ++x)
#pragma unroll
            for (int e = 0; e < 8; ++e) { gv[x][e] = (T)1.0f; rv[x][e] = (T)0.0f; }
          const int64_t in_row = orow + min(on0 + col, g.N - 8);
          const int gr0 = om0 + wave * 32 + row0;
          if (g.gate) {                                // one row of gate per group of gate_rows rows of C
#pragma unroll
            for (int x = 0; x < U; ++x) gv[x] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.gate) + (int64_t)(min(gr0 + x * (64 / PR), g.M - 1) / g.gate_rows) * g.ld_gate + in_row);
          }
          if (g.resid) {
#pragma unroll
            for (int x = 0; x < U; ++x) rv[x] = *reinterpret_cast<const V8*>(reinterpret_cast<const T*>(g.resid) + (int64_t)min(gr0 + x * (64 / PR), g.M - 1) * g.ld_resid + in_row);
          }
          if (ohf) {
#pragma unroll
            for (int x = 0; x < U; ++x) gv[x] = *reinterpret_cast<const V8*>(C + (int64_t)min(gr0 + x * (64 / PR), g.M - 1) * g.ldc + in_row);
          }
        };
        if constexpr (EP && EARLY) ask_rows();
        // (acc[c][x]: row 16 x + (lane & 15), columns 16 c + 4 (lane >> 4) .. + 3)
#pragma unroll
        for (int c = 0; c < 2 * B; ++c)
#pragma unroll
          for (int x = h; x < h + RH / 16; ++x) {
            V4 v4;
#pragma unroll
            for (int e = 0; e < 4; ++e) v4[e] = TypeTraits<T>::from_f32(acc[2 * j0 + c][x][e]);
            *reinterpret_cast<V4*>(cs + place((lane & 15) + 16 * (x - h), 2 * c + (lane >> 5)) + ((lane >> 4) & 1) * 8) = v4;
          }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        V8 r[U];
#pragma unroll
        for (int x = 0; x < U; ++x) r[x] = *reinterpret_cast<const V8*>(cs + place(lane / PR + x * (64 / PR), c));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                          // read before the next blocks overwrite it
        if constexpr (EP) {
          float v[U][8];
#pragma unroll
          for (int x = 0; x < U; ++x)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[x][e] = TypeTraits<T>::to_f32(r[x][e]) + TypeTraits<T>::to_f32(bias[decltype(P)::value & AHEAD][e]);
          if (ohf == 0) {
#pragma unroll
            for (int x = 0; x < U; ++x) apply_act_n(v[x], g.act);
#pragma unroll
            for (int x = 0; x < U; ++x)
#pragma unroll
              for (int e = 0; e < 8; ++e) r[x][e] = TypeTraits<T>::from_f32(v[x][e]);
            if (g.gate || g.resid) {
              if constexpr (!EARLY) ask_rows();
#pragma unroll
              for (int x = 0; x < U; ++x)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                  r[x][e] = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(r[x][e]) * TypeTraits<T>::to_f32(gv[x][e]) + TypeTraits<T>::to_f32(rv[x][e]));
            }
          } else {                                     // the second tile of a pair is multiplied onto what this thread stored
            if constexpr (!EARLY) ask_rows();
#pragma unroll
            for (int x = 0; x < U; ++x)
#pragma unroll
              for (int e = 0; e < 8; ++e)
                r[x][e] = TypeTraits<T>::from_f32(TypeTraits<T>::to_f32(gv[x][e]) * TypeTraits<T>::to_f32(TypeTraits<T>::from_f32(v[x][e])));
          }
        }
#pragma unroll
        for (int x = 0; x < U; ++x) {
          const int row = row0 + x * (64 / PR);
          if (om0 + wave * 32 + row < g.M && on0 + col < g.N) {
            if (!EP && g.epi == EPI_MONARCH_SCATTER) {   // column c of entry bt -> block c / per, column bt * per + c % per
              const int gc = on0 + col, d = gc / g.per;
              *reinterpret_cast<V8*>(C + (int64_t)d * g.sL + (int64_t)(om0 + wave * 32 + row) * g.ldc + (int64_t)obt * g.per + (gc - d * g.per)) = r[x];
            } else {
              *reinterpret_cast<V8*>(crow + (uint32_t)(row * g.ldc + col)) = r[x];
            }
          }
        }
      });
    });
    if (!go) break;
    stores = om0 + WIDE_BM <= g.M && on0 + W <= g.N;   // every one of the 2 TN stores went out
  }  // tiles
}

template <typename T, int TN>
int launch_wide(const GemmArgs& g, hipStream_t st) {
  int tiles_m = (int)cdiv(g.M, WIDE_BM), tiles_n = (int)cdiv(g.N, 32 * TN);
  constexpr size_t lds = wide_lds_bytes<TN>();
  static_assert(lds <= 163840, "the ring and the way out fit one compute unit");
  const bool ep = g.bias || g.act || g.gate || g.resid || g.pair;
  void* fn = ep ? (g.b_kn ? (void*)gemm_wide_kernel<T, true, TN, true> : (void*)gemm_wide_kernel<T, false, TN, true>)
                : (g.b_kn ? (void*)gemm_wide_kernel<T, true, TN, false> : (void*)gemm_wide_kernel<T, false, TN, false>);
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
  const int64_t total = (int64_t)tiles_m * tiles_n * g.batch;
  if (total > (1ll << 30)) { set_error("gemm: too many tiles"); return BLR_ERR_UNSUPPORTED; }
  int per_xcd = (int)cdiv(total, 8), walkers = min2(per_xcd, (device_cus() > 0 ? device_cus() : 256) / 8), side_wgs = 0;
  if (g.side.items > 0 && g.side_taken) side_wgs = (int)(cdiv(cdiv(g.side.items, 512), 8) * 8);
  if (side_wgs > 4096) side_wgs = 4096;
  GemmArgs ga = g;
  void* args[] = {&ga, &tiles_m, &tiles_n, &per_xcd, &walkers, &side_wgs};
  hipError_t e = hipLaunchKernel(fn, dim3((unsigned)(walkers * 8 + side_wgs)), dim3(512), args, lds, st);
  if (e != hipSuccess) { set_error("gemm_wide: launch failed: %s", hipGetErrorString(e)); return BLR_ERR_LAUNCH; }
  if (side_wgs > 0) *g.side_taken = 1;
  return BLR_OK;
}

template <typename T>
int wide_width_launch(const GemmArgs& g, int tn, hipStream_t st) {
  switch (tn) {
    case 3: return launch_wide<T, 3>(g, st);
    case 4: return launch_wide<T, 4>(g, st);
    case 5: return launch_wide<T, 5>(g, st);
    case 6: return launch_wide<T, 6>(g, st);
    case 7: return launch_wide<T, 7>(g, st);
    case 8: return launch_wide<T, 8>(g, st);
    case 9: return launch_wide<T, 9>(g, st);
    case 10: return launch_wide<T, 10>(g, st);
    case 11: return launch_wide<T, 11>(g, st);
  }
  set_error("gemm_wide: no tile of %d columns", 32 * tn);
  return BLR_ERR_UNSUPPORTED;
}

// What a launch takes, in microseconds: t = c0 + (c1 R + c3 f) w + (c2 R + c4 f) w k, with k = stages of 64, w = the tile's size in units of
// 256 x 32, f = tiles / what the chip holds at a time, R = f rounded up.  Fitted (non-negative, on relative errors) to eager launches, 24 in a row over two copies of
// the operands, of 870 plain products of 129 .. 4096 rows, 64 .. 22000 columns, 72 .. 11008 k and 1 .. 16 batches on every kind: 7 - 12 % rms each.  An output stage
// costs every kind about the same: with bias and GELU 259 products chosen by these estimates take 0.82 x the time of the ring rules, 1.04 x at worst but for one.
struct WideModel { int bm, bn, occ; float c[5]; };
const WideModel kWideModel[12] = {
    {128, 128, 2, {3.424f, 0.050f, 0.202f, 2.019f, 0.406f}},           // the ring kernels with stages of 64 k
    {256, 128, 1, {1.821f, 0.828f, 0.120f, 0.576f, 0.148f}},
    {256, 256, 1, {1.895f, 0.608f, 0.127f, 0.419f, 0.098f}},
    {256, 96, 1, {3.138f, 0.241f, 0.220f, 0.305f, 0.139f}},            // tn = 3 ..
    {256, 128, 1, {3.127f, 0.229f, 0.180f, 0.326f, 0.115f}},
    {256, 160, 1, {3.449f, 0.173f, 0.167f, 0.407f, 0.097f}},
    {256, 192, 1, {3.448f, 0.196f, 0.157f, 0.369f, 0.088f}},
    {256, 224, 1, {3.670f, 0.208f, 0.157f, 0.358f, 0.075f}},
    {256, 256, 1, {3.547f, 0.212f, 0.151f, 0.362f, 0.071f}},
    {256, 288, 1, {3.389f, 0.263f, 0.152f, 0.350f, 0.065f}},
    {256, 320, 1, {2.830f, 0.351f, 0.149f, 0.269f, 0.058f}},
    {256, 352, 1, {2.486f, 0.399f, 0.152f, 0.273f, 0.055f}},
};

}  // namespace

bool gemm_wide_ok(const GemmArgs& g) {
  if (g.cn != 1 || g.sat8 || g.N < 8 || g.N % 8 || g.K % 8 || g.K <= 64) return false;
  const bool ep = g.bias || g.act || g.gate || g.resid || g.pair;
  if (g.epi == EPI_MONARCH_SCATTER ? (ep || g.per % 8 || g.sL % 8) : g.epi != EPI_PLAIN) return false;
  if (!aligned(g.A, 16) || !aligned(g.B, 16) || !aligned(g.C, 16) || g.lda % 8 || g.sA % 8 || g.ldb % 8 || g.sB % 8 || g.ldc % 8 || g.sC % 8) return false;
  if ((g.bias && !aligned(g.bias, 16)) || (g.gate && (!aligned(g.gate, 16) || g.ld_gate % 8)) || (g.resid && (!aligned(g.resid, 16) || g.ld_resid % 8))) return false;
  if (g.pair && (g.gate || g.resid || g.pair_dA % 8 || g.pair_dB % 8 || g.pair_dbias % 8)) return false;
  const int64_t lim = (int64_t)1 << 32;                               // per-lane offsets are 32 bits
  return (int64_t)(g.M - 1) * g.lda * 2 + 128 < lim && (g.b_kn ? 63 * g.ldb * 2 + (int64_t)g.N * 2 < lim : (int64_t)(g.N - 1) * g.ldb * 2 + 128 < lim) &&
         32 * g.ldc + g.N < lim / 2;
}

// Columns of the tile in units of 32, or 0, 1, 2 for the ring kernels with stages of 64 k on tiles of 128 x 128, 256 x 128 and 256 x 256, or -1 for the ring
// kernels by their own rules.  The estimates decide for short reductions.  For long ones they are too kind to the tiles here, whose ring is two stages deep, as soon
// as operands come from memory (they were fitted to warm ones): 4096 x 4096 x 11008 takes 287 us in 256 x 256 tiles of the ring kernel and 321 here, 2048 x 1024 x 2752
// in 4 batches with Monarch's scatter 49 and 52 - 59 (256 x 128).  So from 1536 k on a single product comes here where its estimate is 5 % better and one of
// several batches where it is 8 % better, and the others of several batches keep the rules that they had (2048 x 176 x 2088 in 16: 53 us, and 61 on the best of these
// tiles).  The 8 % are asked from 1024 k on where the batches share the rows of A, which then is the input of a call and not what the launch before left in the
// caches: Monarch 4096 -> 22016 at 2048 rows 168.7 -> 164.1 us, while Z U of BLAST 11008 -> 4096 stays (the call 113 us, 115 with the ring kernel).  A pair in four
// batches and more with less than 200 k and results for several rounds is two ways out for hardly any products: 2833 x 1952 x 120 in 4 43.5 us there, 51.0 here,
// 1548 x 832 x 192 in 8 26.4 and 28.0 (3838 x 584 x 144 the other way, 50.5 and 43.4).
// With weights from memory, against the ring rules alone: 660 products of 1024 .. 11008 k 0.866 x the time in the mean, nine 3 - 8 % longer (most of them the same kernel,
// timed twice); 1158 shorter ones, with scatter, output stage and pairs among them, 0.813 x, eight 4 - 17 % longer (the worst: 1528 x 768 x 88 in 16, scattered).
int gemm_wide_plan(const GemmArgs& g, bool ring) {
  const int cus = device_cus() > 0 ? device_cus() : 256, K = g.pair ? 2 * g.K : g.K;
  if (ring && g.pair && g.batch >= 4 && g.K < 200 && (int64_t)g.M * g.N * g.batch >= (int64_t)32768 * cus) return -1;
  int best[2] = {0, 3};                              // ring, wide
  float t_best[2] = {1e30f, 1e30f};
  for (int i = ring ? 0 : 3; i < 12; ++i) {
    const WideModel& m = kWideModel[i];
    const int64_t tiles = cdiv(g.M, m.bm) * cdiv(g.N, m.bn) * g.batch, holds = (int64_t)cus * m.occ;
    const float f = (float)tiles / holds, R = (float)cdiv(tiles, holds), w = (float)m.bm * m.bn / 8192.f, k = (float)K / 64.f;
    const float t = m.c[0] + (m.c[1] * R + m.c[3] * f) * w + (m.c[2] * R + m.c[4] * f) * w * k;
    if (t < t_best[i >= 3]) { t_best[i >= 3] = t; best[i >= 3] = i; }
  }
  const bool deep = g.K >= 1536, apart = g.K >= 1024 && g.batch > 1 && g.lda > g.K;
  if (t_best[1] < (!deep && !apart ? 1.0f : g.batch > 1 ? 0.92f : 0.95f) * t_best[0]) return best[1];
  return deep && g.batch > 1 ? -1 : best[0];
}

int gemm_wide_launch(const GemmArgs& g, int tn, int dtype, hipStream_t st) {
  return dtype == BLR_F16 ? wide_width_launch<f16>(g, tn, st) : wide_width_launch<bf16>(g, tn, st);
}

}  // namespace blr
