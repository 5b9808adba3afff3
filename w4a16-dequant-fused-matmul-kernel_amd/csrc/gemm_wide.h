// Prefill W4A16 GEMM on gfx950 matrix cores, one wave per SIMD, for tiles that
// give a wave up to 256 x 64 of Y (v_mfma_f32_16x16x32_f16, fp32 accumulation).
//
// Replaces the large-M regime of the reference's fused kernel
// (w4a16-kernel/src/w4a16/triton_kernel.py:62-128: fp16 dequant of the weight
// tile, tl.dot with fp32 accumulation, fp16 store).
//
// What bounds it: at prefill sizes the chip holds its power limit, so the time
// follows the energy of a multiply-add and not only the cycles.  Measured on
// MI355X in one process: registers alone, on N(0, 1) data, v_mfma_f32_16x16x32_f16
// sustains 1858 TFLOP/s and 32x32x16, with twice the accumulator traffic per
// multiply-add, 1601 (both about 2345 on zeros); M = N = K = 8192, G = 128:
//   * the two-waves-per-SIMD kernel of 128 x 64 per wave (gemm_stream.hip) 948 us;
//   * this kernel 780 us = 1410 TFLOP/s, matrix cores busy 77 % of the cycles;
//   * hipBLASLt's fp16 product of the dequantised weight 823.
// (The same scheme first built on 32x32x16 took as long as the streamed kernel: as
// busy, but at a clock 15 % lower.)
// Hence:
//   * a wave owns all rows of the tile and 64 columns (kMT m-tiles x 4 n-tiles),
//     so every weight is dequantised once per 256 rows (once per 128 rows with
//     128-row waves, which cost 2 % more at equal LDS reads saved);
//   * 256 accumulators in the accumulation registers, the rest in the other 256:
//     one wave per SIMD, so whatever runs beside the MFMAs is placed by hand, one
//     to two instructions behind each (the dequant of the next two halves, the
//     next fragments' LDS reads, the next panels' loads): 2.7 instructions per
//     MFMA against the four its 16 cycles leave room for;
//   * activations stream into four LDS buffers of 64 k by LDS-direct loads two
//     panels ahead (128-byte rows, octet slots XOR-swizzled by (row / 2) % 8: no
//     bank conflicts), weights, scales and zeros into registers three panels
//     ahead; one barrier per panel.
// Tiles of 32 and 64 rows wait on memory, not on the matrix cores: there the
// activations run three panels ahead and the weights four, and a step's wait
// leaves in flight all that the two newest steps issued (waiting for all but the
// last activations drained the weights each panel, a round trip to memory per 64
// k).  Measured on MI355X, 32 x 64 tiles with four k-slices, M = 17, us: K =
// 14336, N = 4096 unsplit / split 4 37.8 / 17.1 -> 29.0 / 14.6, 13.4 with the
// first panel's wait counted as well; K = 4096, N = 14336 14.5 -> 12.2 (a CU's activation lines bound it now: 64 x 64 tiles, twice
// the lines, gained 0-5 %, taller ones nothing and keep the depth they had).
// The `any` form holds a column's scale in a register each: joining two as they
// arrive would wait for each load in turn.  It is bound by the issue of its two-byte
// loads, 16 a panel, so it keeps two and three panels ahead: each panel further asks
// for one more past the end of k.  64 x 64 tiles, three / two ahead, us: M = 93, K =
// 2080, N = 1003, G = 32 12.9 / 11.5; M = 65, K = N = 1024 10.3 / 8.9; M = 300, K =
// 2048, N = 2047 14.5 / 12.2; M = 70, K = 28672, N = 1003 25.9 / 22.4.
// kKS = 2 or 4 k-slices per workgroup (waves along K instead of N) serve shapes
// with few tiles; the slices' sums meet in LDS in slice order.
// Scales and zeros have a buffer resource each: they may lie anywhere.
// Requirements (checked by the caller): G % 32 == 0, K % G == 0, 16-byte aligned
// x with ldx % 8 == 0, 4-byte aligned qweight, 2-byte aligned scales, zeros, y
// and bias, each operand below 2 GiB; any M, N.  Unless kAny also N % 4 == 0,
// ldy % 4 == 0, 16-byte aligned qweight and 8-byte aligned scales, zeros, y and
// bias (vector loads of the scales and zeros, vector stores of y).
#pragma once

#include "w4a16_device.h"
#include "w4a16_launch.h"

#include <type_traits>
#include <utility>

namespace w4a16 {
namespace {

constexpr int kBK = 64;        // k per panel
constexpr int kGroupM = 4;     // M-tiles per group of the tile order
constexpr int kWaves = 4;      // one per SIMD
constexpr int kNT = 4;         // 16-column MFMA tiles per wave: a lane's adjacent columns

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <class F, int... I>
__device__ __forceinline__ void static_for_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(f, std::make_integer_sequence<int, N>{});
}

// s_waitcnt operand that waits for all but the last n vector-memory operations.
constexpr int vmcnt_only(int n) { return (n & 15) | (n >> 4) << 14 | 0x0F70; }
constexpr int kLgkmcnt0 = 0xC07F;

// No memory access moves across this, in any pass of the compiler (a scheduling
// barrier holds only the scheduler).
__device__ __forceinline__ void pin_accesses() { asm volatile("" ::: "memory"); }

// A read-only argument; kPinned: loads through it stay on their side of
// pin_accesses() (through a `const __restrict__` one they may move).
template <class T, bool kPinned>
using In = std::conditional_t<kPinned, const T*, const T* __restrict__>;

// This wave's LDS accesses complete, then s_barrier (no wait for the LDS-direct
// loads in flight, as __syncthreads() would).
__device__ __forceinline__ void tile_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct WideArgs {
  const f16* X;
  const uint32_t* QW;
  const uint16_t *SC, *ZR;
  int M, N, K, G, ldx, ldy;
  uint32_t gmagic;
  int gshift;
  const f16* bias;
  f16* Y;
  float* part;   // fp32 partials [split][M][N], or nullptr
};

// Whether a tile keeps three panels of activations and four of weights in flight.
constexpr bool wide_deep(int mt, bool any) { return mt <= 4 && !any; }

// The tile at (m0, n0) of kBM = 16 kMT rows and kBN = 64 kWN columns, panels
// [p0, p0 + np) of split sp; As0 .. As3: kKS * kBM * 8 slots each.
template <int kMT, int kWN, int kKS, bool kSZ1, bool AZ, bool kAny>
__device__ __forceinline__ void wide_tile(const WideArgs& g, int m0, int n0, int sp, int p0, int np,
                                          uint4* As0, uint4* As1, uint4* As2, uint4* As3) {
  static_assert(kWN * kKS == kWaves, "four waves");
  static_assert(kMT == 16 || kMT == 8 || kMT == 4 || kMT == 2, "whole dequant units per slot");
  constexpr int kBM = 16 * kMT;
  constexpr int kRows = kBM / kWN;             // activation rows each wave streams
  constexpr int kAL = kRows / 8;               // its 8-row loads per panel
  static_assert(kRows % 16 == 0, "the swizzle's period");
  constexpr int kPanel = kKS * kBM * 8;
  // activations' and weights' panels ahead (256-row waves have no registers for more,
  // 128-row ones gain nothing by it, and the `any` form's many small loads cost more
  // than their latency)
  constexpr bool kDeep = wide_deep(kMT, kAny);
  constexpr int kXA = kDeep ? 3 : 2, kWA = kDeep ? 4 : 3;
  const int M = g.M, N = g.N, K = g.K;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slice = wave / kWN;                // k-slice
  const int wn = wave % kWN;                   // position along N
  const int l16 = lane & 15;
  const int oct = lane >> 4;                   // k-octet within a 32-k half
  const int ncol = n0 + wn * 16 * kNT + kNT * l16;   // this lane's 4 columns
  const bool nv = ncol < N;
  const int KP = K >> 3;
  // this slice's panels [KS0, KT); panels at or past KT load zeros
  const int KSL = np / kKS;
  const int KS0 = p0 + slice * KSL;
  const int KT = min((K + kBK - 1) / kBK, KS0 + KSL);
  const int NG = K / g.G;

  uint32_t magic_mix;
  asm volatile("v_mov_b32 %0, 0x54006400" : "=v"(magic_mix));
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc(g.X, ((uint32_t)(M - 1) * (uint32_t)g.ldx + (uint32_t)K) * 2u);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(g.QW, (uint32_t)KP * (uint32_t)N * 4u);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(g.SC, (uint32_t)NG * (uint32_t)N * 2u);
  const __amdgpu_buffer_rsrc_t rz = make_rsrc(g.ZR, (uint32_t)NG * (uint32_t)N * 2u);

  // Activation stream: wave wn of a slice fills rows kRows wn .. with kAL loads
  // of 8 rows; lane L writes row 8j + L/8, slot L%8, which holds octet
  // (L%8) ^ ((row/2)%8) = (L%8) ^ (L/16) ^ (4 if j is odd).  Rows at or past M
  // lie beyond the buffer range and read as zero.
  const uint32_t a_oct0 = (uint32_t)((lane & 7) ^ (lane >> 4));
  uint32_t a_off[kAL];
#pragma unroll
  for (int j = 0; j < kAL; ++j)
    a_off[j] = (uint32_t)(m0 + kRows * wn + 8 * j + (lane >> 3)) * (uint32_t)g.ldx * 2u +
               (a_oct0 ^ (j & 1 ? 4u : 0u)) * 16u;
  // A fragment of m-tile i, half h: row 16 i + l16, octet 4 h + oct
  int a_frag[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    a_frag[h] = slice * kBM * 8 + l16 * 8 + ((4 * h + oct) ^ ((l16 >> 1) & 7));
  // weight words of this lane: packed row 4 h + oct of a panel, columns ncol..+3
  // (kAny: the columns past N of a lane that has some inside hold the next
  // row's words, or zeros; nothing is stored for them)
  uint32_t b_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    b_off[h] = nv ? ((uint32_t)(4 * h + oct) * (uint32_t)N + (uint32_t)ncol) * 4u : kOobOffset;
  const uint32_t q_off = nv ? (uint32_t)ncol * 2u : kOobOffset;

  auto as = [&](auto bc) -> uint4* {
    constexpr int b = decltype(bc)::value % 4;
    if constexpr (b == 0) return As0;
    else if constexpr (b == 1) return As1;
    else if constexpr (b == 2) return As2;
    else return As3;
  };
  // One panel's words, scales and zeros.  kSZ1: G % 64 == 0, both halves of a
  // panel lie in one group.
  constexpr int kH = kSZ1 ? 1 : 2;
  // kAny: one column's 16 bits a register (joining two would wait for their loads)
  using Halves = std::conditional_t<kAny, u32x4, u32x2>;
  struct Panel {
    u32x4 w[2];
    Halves s[kH], z[kH];
  };
  // Vector loads of load_w, and what may be in flight where panel kt + 1's
  // activations must have landed.  Loads retire in order, so three panels ahead
  // all that steps kt - 1 and kt issued; two ahead step kt's activations.  The
  // former counts weights too, which must then be issued where they are written:
  // pin() keeps them from moving past a wait (they did, to where a loop first uses
  // them).  LDS-direct loads stay where they are: they write memory.
  constexpr int kWL = 2 + 2 * kH * (kAny ? kNT : 1);
  constexpr int kSince = 2 * (kAL + kWL);
  constexpr int kInFlight = kDeep ? kSince : kAL;
  auto pin = [] {
    if constexpr (kDeep) pin_accesses();
  };
  auto load_halves = [&](__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) -> Halves {
    if constexpr (kAny) {
      Halves v;
#pragma unroll
      for (int c = 0; c < kNT; ++c)
        v[c] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(
            r, (int)(voff + 2u * (uint32_t)c), (int)soff, 0);
      return v;
    } else {
      return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
    }
  };
  // column c's half, twice
  auto half2 = [&](const Halves& v, int c) {
    if constexpr (kAny) return as_h2(__builtin_amdgcn_perm(v[c], v[c], 0x01000100u));
    else return as_h2(__builtin_amdgcn_perm(v[c / 2], v[c / 2], c & 1 ? 0x03020302u : 0x01000100u));
  };
  auto load_w = [&](int kt, Panel& p) {
    const bool in = kt < KT;
    const uint32_t qo = in ? q_off : kOobOffset;
    const uint32_t wo = uniform(in ? (uint32_t)kt * 32u * (uint32_t)N : kOobOffset);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      p.w[h] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, (int)b_off[h], (int)wo, 0));
#pragma unroll
    for (int h = 0; h < kH; ++h) {
      const uint32_t gi = div_group((uint32_t)(kt * kBK + 32 * h), g.gmagic, g.gshift);
      const uint32_t go = uniform(gi * (uint32_t)N * 2u);
      p.s[h] = load_halves(rs, qo, go);
      p.z[h] = load_halves(rz, qo, go);
    }
  };
  // Loads [lo, hi) of panel kt's activations.  K % 64 == 32 (G % 64 != 0): the
  // last panel's second half lies past K, where a row's bytes may hold anything;
  // its octets read as zero.
  auto load_a = [&](auto bc, auto lo, auto hi, int kt) {
    uint4* a = as(bc) + slice * kBM * 8 + kRows * wn * 8;
    const uint32_t ao = uniform(kt < KT ? (uint32_t)kt * (uint32_t)(kBK * 2) : kOobOffset);
    const uint32_t lim = kt < KT ? (uint32_t)(KP - kt * 8) : 8u;   // octets inside K
#pragma unroll
    for (int j = decltype(lo)::value; j < decltype(hi)::value; ++j) {
      uint32_t vo = a_off[j];
      if constexpr (!kSZ1)
        vo = (a_oct0 ^ (j & 1 ? 4u : 0u)) < lim ? vo : kOobOffset;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(a + 64 * j), 16, (int)vo, (int)ao, 0,
                                               0);
    }
  };

  constexpr int kU = kMT / 2;   // m-tiles per sub-step
  auto read_a = [&](const uint4* A, int h, int u, int i) {
    return __builtin_bit_cast(f16x8, A[a_frag[h] + (u * kU + i) * 16 * 8]);
  };

  f32x4 acc[kMT][kNT];
#pragma unroll
  for (int i = 0; i < kMT; ++i)
#pragma unroll
    for (int c = 0; c < kNT; ++c) acc[i][c] = f32x4{};

  // Dequant (natural k order, as dq_word_nat of gemm_stream.hip): `prep` makes a
  // column's constants for one half (scale pair, zero pair), `diff` the exact
  // differences code - zero of two codes, and one sub-step later a
  // multiplication by the scale pair makes two weights (a packed multiply right
  // behind the subtraction it needs would wait a cycle).
  f16x2 dt[2][4], ds[2];       // differences and scales of two columns
  f16x2 pr_s[2], pr_z[2];      // the constants of the next two
  auto prep_s = [&](const Panel& p, int h, int c0, int c) {
    pr_s[c] = half2(p.s[kSZ1 ? 0 : h], c0 + c);
  };
  auto prep_z = [&](const Panel& p, int h, int c0, int c) {
    const f16x2 z2 = half2(p.z[kSZ1 ? 0 : h], c0 + c);
    pr_z[c] = AZ ? z2 : z2 + f16x2{(f16)1024.0f, (f16)64.0f};
  };
  auto diff = [&](uint32_t masked, int c) {
    const f16x2 p = as_h2(masked);
    return AZ ? (p - as_h2(magic_mix)) - pr_z[c] : p - pr_z[c];
  };

  Panel st[4];
  f16x8 a0[kU], a1[kU];
  u32x4 b0[kNT], b1[kNT];
  // One panel (buffer and register set s = kt % 4) in four sub-steps: half h of
  // its k by half u of the wave's m-tiles.  A sub-step is kU x 4 slots, each an
  // MFMA and its share of 32 units of other work (eight pairs of codes, four
  // phases each; phase t % 4 of the next few pairs in slot t, so that dependent
  // instructions lie apart); sched_barrier keeps the order written here.  The MFMAs are
  // inline asm so that the accumulators stay in the accumulation registers (the
  // allocator moved them to and fro, and spilled); the two wait states between a
  // VALU result and an MFMA that reads it are the s_nop at a sub-step's start
  // (weights are read from the sub-step after they were made).
  auto step = [&](auto sc, int kt) {
    constexpr int s = decltype(sc)::value;
    static_for<4>([&](auto qc) {
      constexpr int q = decltype(qc)::value, h = q / 2, u = q % 2;
      f16x8(&a)[kU] = u ? a1 : a0;
      f16x8(&an)[kU] = u ? a0 : a1;
      u32x4(&b)[kNT] = h ? b1 : b0;
      u32x4(&bn)[kNT] = h ? b0 : b1;
      __builtin_amdgcn_s_waitcnt(kLgkmcnt0);   // this sub-step's fragments
      asm volatile("s_nop 1");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (q == 3) {
        // this wave's activations of panel kt + 1 are there; then everyone's of
        // this slice
        pin();
        __builtin_amdgcn_s_waitcnt(vmcnt_only(kInFlight));
        pin();
        if constexpr (kWN > 1) tile_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      // unpacked here: columns 2, 3 of the next half (u = 0) or 0, 1 of the one
      // after it (u = 1); prepared: what the next sub-step unpacks
      constexpr int hn = h + 1 + u, c0 = u ? 0 : 2;
      constexpr int q2 = (q + 1) % 4, s2 = s + (q + 1) / 4, hn2 = q2 / 2 + 1 + q2 % 2;
      constexpr int c2 = q2 % 2 ? 0 : 2;
      const Panel& pu = st[(s + hn / 2) % 4];
      const Panel& pp = st[(s2 + hn2 / 2) % 4];
      const uint4* An = q < 3 ? as(sc) : as(std::integral_constant<int, s + 1>{});
      const f16x2 sc2[2] = {ds[0], ds[1]};
      constexpr int kSlots = kU * kNT, kUnits = 32 / kSlots;
      uint32_t tmp[kUnits];
      constexpr int kLd = kAL * (q + 1) / 3 - kAL * q / 3;   // activation loads (q < 3)
      static_for<kSlots>([&](auto tc) {
        constexpr int t = decltype(tc)::value, i = t / kNT, n = t % kNT;
        asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
            : "+a"(acc[u * kU + i][n])
            : "v"(a[i]), "v"(b[n]));
        static_for<kUnits>([&](auto vc) {
          constexpr int r = decltype(vc)::value, pair = t / 4 * kUnits + r, ph = t % 4;
          constexpr int c = pair / 4, e = pair % 4;          // codes 2e, 2e + 1 of column c
          if constexpr (ph == 0) {
            const uint32_t w = pu.w[hn % 2][c0 + c];
            tmp[r] = __builtin_amdgcn_perm(w, w, 0x01010101u * (uint32_t)e);
            bn[2 * u + c][e] = as_u32(dt[c][e] * sc2[c]);
          } else if constexpr (ph == 1) {
            tmp[r] = (tmp[r] & 0x00F0000Fu) | magic_mix;
            if constexpr (e == 3) ds[c] = pr_s[c];
          } else if constexpr (ph == 2) {
            dt[c][e] = diff(tmp[r], c);
          } else {
            if constexpr (pair == 3) prep_s(pp, hn2 % 2, c2, 0);
            if constexpr (pair == 4) prep_z(pp, hn2 % 2, c2, 0);
            if constexpr (pair == 7) prep_s(pp, hn2 % 2, c2, 1), prep_z(pp, hn2 % 2, c2, 1);
          }
        });
        constexpr int kGap = kU >= 4 ? kU / 2 : 1;
        // four ahead: into the set of panel kt, whose last words were unpacked in
        // sub-step 0
        if constexpr (q == (kDeep ? 1 : 3) && t == 1) load_w(kt + kWA, st[(s + kWA) % 4]);
        if constexpr (q < 3 && t % kGap == 1 % kGap && t / kGap < kLd)
          load_a(std::integral_constant<int, s + kXA>{},
                 std::integral_constant<int, kAL * q / 3 + t / kGap>{},
                 std::integral_constant<int, kAL * q / 3 + t / kGap + 1>{}, kt + kXA);
        // the next sub-step's fragments, early: they are there by its start
        if constexpr (t >= 1 && t - 1 < kU) an[t - 1] = read_a(An, (q + 1) / 2 % 2, (q + 1) % 2, t - 1);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };

  const std::integral_constant<int, 0> c0{};
  const std::integral_constant<int, 1> c1{};
  const std::integral_constant<int, 2> c2{};
  const std::integral_constant<int, 3> c3{};
  const std::integral_constant<int, kAL> call{};
  load_a(c0, c0, call, KS0);
  if constexpr (kDeep) {
    // no fewer loads behind each panel's activations than where the steps wait
    auto next = [&] {
      pin();
      __builtin_amdgcn_sched_barrier(0);
    };
    next();
    load_w(KS0, st[0]);
    load_w(KS0 + 1, st[1]);
    next();
    load_a(c1, c0, call, KS0 + 1);
    next();
    load_w(KS0 + 2, st[2]);
    next();
    load_a(c2, c0, call, KS0 + 2);
    next();
    load_w(KS0 + 3, st[3]);
    next();
  } else {
    load_w(KS0, st[0]);
    __builtin_amdgcn_sched_barrier(0);
    load_a(c1, c0, call, KS0 + 1);
    __builtin_amdgcn_sched_barrier(0);
    load_w(KS0 + 1, st[1]);
    load_w(KS0 + 2, st[2]);
  }
  // panel KS0's activations (the weights are waited for where they are used): so
  // many loads were issued behind them (two panels ahead, whether or not the
  // weights were).  64-row tiles wait for some of those too: with all of them in
  // flight the compiler puts waits of its own into the loop, and nothing is gained
  // (32-row tiles gain, M = 17, K = 14336, N = 4096 13.9 -> 13.4 us).
  constexpr int kSince0 = (kXA - 1) * kAL + (kMT == 2 ? kWA * kWL : 0);
  static_assert(kInFlight <= 63 && kSince0 <= 63, "s_waitcnt's counter");
  __builtin_amdgcn_s_waitcnt(vmcnt_only(kSince0));
  pin();
  tile_barrier();
#pragma unroll
  for (int i = 0; i < kU; ++i) a0[i] = read_a(As0, 0, 0, i);
  auto unpack2 = [&](const Panel& p, int h, int col) {
    prep_s(p, h, col, 0), prep_s(p, h, col, 1), prep_z(p, h, col, 0), prep_z(p, h, col, 1);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = p.w[h][col + c];
        dt[c][e] = diff((__builtin_amdgcn_perm(w, w, 0x01010101u * (uint32_t)e) & 0x00F0000Fu) | magic_mix, c);
      }
      ds[c] = pr_s[c];
    }
  };
#pragma unroll
  for (int col = 0; col < 4; col += 2) {
    unpack2(st[0], 0, col);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) b0[col + c][e] = as_u32(dt[c][e] * ds[c]);
  }
  unpack2(st[0], 1, 0);
  prep_s(st[0], 1, 2, 0), prep_s(st[0], 1, 2, 1), prep_z(st[0], 1, 2, 0), prep_z(st[0], 1, 2, 1);
  __builtin_amdgcn_sched_barrier(0);

  // one trip count for the whole workgroup: every wave reaches every barrier
  const int kend = kKS == 1 ? KT : KS0 + KSL;
  auto four = [&](int kt) {
    step(c0, kt);
    step(c1, kt + 1);
    step(c2, kt + 2);
    step(c3, kt + 3);
  };
  if constexpr (kDeep) {
    // entered at least once (kend > KS0): a guarded loop's entry would copy, and so
    // wait for, the loads in flight
    int kt = KS0;
    do {
      four(kt);
      kt += 4;
    } while (kt < kend);
  } else {
    for (int kt = KS0; kt < kend; kt += 4) four(kt);
  }
  // the last MFMAs' results (written by asm the compiler cannot see into)
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // kKS slices: each finishes kMT / kKS m-tiles, or (fewer m-tiles than slices)
  // kOwnR of the four rows of one.  The others' sums of them go through the
  // activation buffers (half a panel buffer per wave), once the loads in flight
  // (zeros past the range) have landed, and are added in slice order.
  static_assert(kMT % kKS == 0 || kKS % kMT == 0, "whole m-tiles or rows per slice");
  constexpr bool kByRow = kMT < kKS;
  constexpr int kOwn = kByRow ? 1 : kMT / kKS, kOwnR = kByRow ? 4 * kMT / kKS : 4;
  auto owns = [&](int i) { return kKS == 1 || (kByRow ? slice * kMT / kKS : slice) == i / kOwn; };
  const int r0 = kByRow ? slice % (kKS / kMT) * kOwnR : 0;
  if constexpr (kKS > 1) {
    static_assert((kByRow ? kMT : kMT - kOwn) * kNT * 64 <= kPanel / 2,
                  "a wave's hand-over fits half a buffer");
    auto region = [&](int w) { return (w < 2 ? As0 : As1) + (w & 1) * (kPanel / 2); };
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    tile_barrier();
    uint4* mine = region(wave);
#pragma unroll
    for (int i = 0; i < kMT; ++i)
      if (kByRow || !owns(i)) {
        const int at = kByRow || i < slice * kOwn ? i : i - kOwn;
#pragma unroll
        for (int c = 0; c < kNT; ++c)
          mine[(at * kNT + c) * 64 + lane] = __builtin_bit_cast(uint4, acc[i][c]);
      }
    tile_barrier();
#pragma unroll
    for (int i = 0; i < kMT; ++i)
      if (owns(i)) {
#pragma unroll
        for (int c = 0; c < kNT; ++c) {
          f32x4 v{};
#pragma unroll
          for (int o = 0; o < kKS; ++o) {
            f32x4 x = acc[i][c];
            if (kByRow || o != i / kOwn) {
              const int at = kByRow || i < o * kOwn ? i : i - kOwn;
              x = __builtin_bit_cast(f32x4, region(o * kWN + wn)[(at * kNT + c) * 64 + lane]);
            }
            v = o == 0 ? x : v + x;
          }
          acc[i][c] = v;
        }
      }
  }

  const int rbase = m0 + 4 * oct;
  if (!nv) return;
  // (256-row waves are never split along K: with a second way out the allocator
  // spilled accumulators)
  if (kMT < 16 && g.part) {
#pragma unroll
    for (int i = 0; i < kMT; ++i)
      if (owns(i)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = rbase + 16 * i + r;
          if (row < M && (!kByRow || (r >= r0 && r < r0 + kOwnR))) {
            float* p = g.part + ((size_t)sp * M + row) * N + ncol;
            if constexpr (kAny) {
#pragma unroll
              for (int c = 0; c < kNT; ++c)
                if (ncol + c < N) p[c] = acc[i][c][r];
            } else {
              *reinterpret_cast<float4*>(p) =
                  make_float4(acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]);
            }
          }
        }
      }
    return;
  }
  f16 bv[kNT] = {(f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f};
  if (g.bias) {
#pragma unroll
    for (int c = 0; c < kNT; ++c)
      if (!kAny || ncol + c < N) bv[c] = g.bias[ncol + c];
  }
#pragma unroll
  for (int i = 0; i < kMT; ++i)
    if (owns(i)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rbase + 16 * i + r;
        if (row < M && (!kByRow || (r >= r0 && r < r0 + kOwnR))) {
          f16x4 o;
          o.x = f32_to_f16(acc[i][0][r]);
          o.y = f32_to_f16(acc[i][1][r]);
          o.z = f32_to_f16(acc[i][2][r]);
          o.w = f32_to_f16(acc[i][3][r]);
          if (g.bias) {
            o.x = o.x + bv[0];
            o.y = o.y + bv[1];
            o.z = o.z + bv[2];
            o.w = o.w + bv[3];
          }
          f16* y = g.Y + (size_t)row * g.ldy + ncol;
          if constexpr (kAny) {
#pragma unroll
            for (int c = 0; c < kNT; ++c)
              if (ncol + c < N) y[c] = o[c];
          } else {
            __builtin_nontemporal_store(o, reinterpret_cast<f16x4*>(y));
          }
        }
      }
    }
}

// Grid: nb = tiles x splits workgroups; split sp owns panels [sp KTS, sp KTS +
// KTS).  kHalf: the tiles of 32 kMT rows from t0 on in their order, as two
// workgroups of 16 kMT rows each (unsplit).
//
// Arguments: the first fourteen SGPRs' worth, which the first loads need, are
// preloaded by the dispatch (-amdgpu-kernarg-preload-count).
template <int kMT, bool kHalf, int kWN, int kKS, bool kSZ1, bool AZ, bool kAny>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void wide_kernel(const f16* __restrict__ X, In<uint32_t, wide_deep(kMT, kAny)> QW, int M, int N,
                 int K, int KTS, int ldx, int nb, In<uint16_t, wide_deep(kMT, kAny)> SC,
                 In<uint16_t, wide_deep(kMT, kAny)> ZR, uint32_t gmagic, int gshift, int t0, int G,
                 int ldy, const f16* __restrict__ bias, f16* __restrict__ Y,
                 float* __restrict__ part) {
  constexpr int kBM = 16 * kMT * (kHalf ? 2 : 1), kBN = 16 * kNT * kWN;
  constexpr int kPanel = kKS * 16 * kMT * 8;
  __shared__ uint4 As0[kPanel], As1[kPanel], As2[kPanel], As3[kPanel];
  const WideArgs g{X, QW, SC, ZR, M, N, K, G, ldx, ldy, gmagic, gshift, bias, Y, part};

  // XCD-aware grouped tile order: the hardware deals workgroups to the 8 XCDs
  // round-robin; each XCD takes a contiguous run of an order that walks kGroupM
  // M-tiles x all N-tiles per group, so that concurrent tiles share activation
  // rows and weight columns in that XCD's L2.
  const int ntn = (N + kBN - 1) / kBN;
  const int ntm = (M + kBM - 1) / kBM;
  const int total = ntn * ntm;
  int B = (int)blockIdx.x;
  if ((nb & 7) == 0) B = (B & 7) * (nb >> 3) + (B >> 3);
  const int half = kHalf ? B & 1 : 0;
  if constexpr (kHalf) B = t0 + (B >> 1);
  const int sp = (int)uniform((uint32_t)(B / total));
  const int T = B - sp * total;
  const int group = (int)uniform((uint32_t)(T / (kGroupM * ntn)));
  const int first_m = group * kGroupM;
  const int gsz = min(ntm - first_m, kGroupM);
  const int rem = T - group * kGroupM * ntn;
  const int tn = (int)uniform((uint32_t)(rem / gsz));
  const int m0 = (first_m + rem - tn * gsz) * kBM + half * 16 * kMT;
  const int n0 = tn * kBN;
  if (kHalf && m0 >= M) return;
  wide_tile<kMT, kWN, kKS, kSZ1, AZ, kAny>(g, m0, n0, sp, sp * KTS, KTS, As0, As1, As2, As3);
}

// `nb` workgroups (x splits) from tile t0 on.
template <int kMT, bool kHalf, int kWN, int kKS, bool kSZ1, bool AZ, bool kAny>
hipError_t launch_wide_grid(const GemmArgs& a, int nb, int t0, int kts, float* part,
                            hipStream_t st) {
  const GroupDiv gd = group_div(a.G);
  hipLaunchKernelGGL((wide_kernel<kMT, kHalf, kWN, kKS, kSZ1, AZ, kAny>), dim3(nb), dim3(256), 0,
                     st, static_cast<const f16*>(a.x), reinterpret_cast<const uint32_t*>(a.qw),
                     a.M, a.N, a.K, kts, a.ldx, nb, static_cast<const uint16_t*>(a.sc),
                     static_cast<const uint16_t*>(a.zr), gd.magic, gd.shift, t0, a.G, a.ldy,
                     static_cast<const f16*>(a.bias), static_cast<f16*>(a.y), part);
  return hipGetLastError();
}

// kTail: where the last round of `cus` tiles would leave half the CUs or more
// idle, its tiles are done as halves (a second launch of half-height tiles,
// half a round).  Measured on MI355X, M = 4096, K = 4096, N = 14336 (896 tiles,
// three and a half rounds): 390 us in whole tiles, 362 so.
template <int kMT, bool kTail, int kWN, int kKS, bool kSZ1, bool AZ, bool kAny>
hipError_t launch_wide_kernel(const GemmArgs& a, int split, float* part, int cus, hipStream_t st) {
  constexpr int bm = 16 * kMT, bn = 16 * kNT * kWN;
  const int tiles = ((a.N + bn - 1) / bn) * ((a.M + bm - 1) / bm);
  const int kts = wide_split_panels(a.K, split, kKS);
  const int nsplit = split > 1 ? ((a.K + kBK - 1) / kBK + kts - 1) / kts : 1;
  hipError_t e;
  if (kMT == 16 && nsplit > 1) return hipErrorInvalidValue;
  if constexpr (kTail) {
    const int rem = tiles % cus;
    if (nsplit == 1 && tiles > cus && rem > 0 && 2 * rem <= cus) {
      e = launch_wide_grid<kMT, false, kWN, kKS, kSZ1, AZ, kAny>(a, tiles - rem, 0, kts, nullptr, st);
      if (e != hipSuccess) return e;
      return launch_wide_grid<kMT / 2, true, kWN, kKS, kSZ1, AZ, kAny>(a, 2 * rem, tiles - rem, kts,
                                                                       nullptr, st);
    }
  }
  e = launch_wide_grid<kMT, false, kWN, kKS, kSZ1, AZ, kAny>(a, tiles * nsplit, 0, kts,
                                                            nsplit > 1 ? part : nullptr, st);
  if (e != hipSuccess || nsplit == 1) return e;
  return launch_splitk_reduce(part, a.bias, a.y, a.M, a.N, a.ldy, nsplit, st);
}

// The forms of one tiling: by zero-points, group size and (kWithAny) alignment.
template <int kMT, bool kTail, int kWN, int kKS, bool kWithAny>
hipError_t launch_wide_tiling(const GemmArgs& a, bool any, int split, float* part, int cus,
                              hipStream_t st) {
  if (any) {
    if constexpr (kWithAny)
      return a.any_zeros
                 ? launch_wide_kernel<kMT, kTail, kWN, kKS, false, true, true>(a, split, part, cus, st)
                 : launch_wide_kernel<kMT, kTail, kWN, kKS, false, false, true>(a, split, part, cus, st);
    else
      return hipErrorInvalidValue;
  }
  if (a.G % 64 == 0)
    return a.any_zeros
               ? launch_wide_kernel<kMT, kTail, kWN, kKS, true, true, false>(a, split, part, cus, st)
               : launch_wide_kernel<kMT, kTail, kWN, kKS, true, false, false>(a, split, part, cus, st);
  return a.any_zeros
             ? launch_wide_kernel<kMT, kTail, kWN, kKS, false, true, false>(a, split, part, cus, st)
             : launch_wide_kernel<kMT, kTail, kWN, kKS, false, false, false>(a, split, part, cus, st);
}

}  // namespace
}  // namespace w4a16

