// Quantise / pack / unpack / dequantise kernels, bit-exact with the reference's
// PyTorch quantiser as torch evaluates it on the CPU
// (w4a16-kernel/src/w4a16/quant.py:45-178):
//   scale = (gmax - gmin) / 15        IEEE fp32 division (not a reciprocal multiply)
//   scale = scale > 0 ? scale : 1
//   zero  = clamp(rint(-gmin / scale), 0, 15)   compare-select clamp, -0.0 survives
//   q     = clamp(rint(W / scale) + zero, 0, 15) with the fp32 scale
//   scales, zeros -> fp16 (RNE); codes packed 8 per int32, row 8i+j in nibble j.
// rint is round-half-to-even (v_rndne_f32).  HIP divides fp32 with the correctly
// rounded sequence by default, and the build never enables fast-math, so the
// compare-selects are not folded into min/max (which could drop -0.0).
// Group minimum, as torch's CPU amin(dim=1) returns it when a group's minimum
// is a zero and the group holds both +0.0 and -0.0 (measured on torch's CPU
// reduction; the same on its DEFAULT, AVX2 and AVX512 code paths):
//  * N >= 2 (the reduced rows are strided): columns in whole blocks of 32
//    (n < 32 * (N / 32), the vectorised outer reduction) take the last zero in
//    k order (v <= min ? v : min), the N % 32 tail columns (its scalar loop) the
//    first (v < min ? v : min);
//  * N == 1 (the group's G values are contiguous): G < 32 takes the first zero;
//    G >= 32 follows the vectorised inner reduction (inner_zero_min below).
// Only the sign of the zero-point depends on it; the group maximum's zero sign
// reaches no output (gmax - gmin is the same for either zero, or the scale is
// replaced by 1).
#include "w4a16_device.h"
#include "w4a16_launch.h"

#include <type_traits>

namespace w4a16 {
namespace {

// Input element traits: fp16 weights arrive as raw bits, fp32 as floats.
struct InF16 {
  typedef uint16_t T;
  static __device__ __forceinline__ float val(T b) { return (float)as_h(b); }
  static __device__ __forceinline__ bool nonfinite(T b) { return (b & 0x7C00u) == 0x7C00u; }
};
struct InF32 {
  typedef float T;
  static __device__ __forceinline__ float val(T v) { return v; }
  static __device__ __forceinline__ bool nonfinite(T v) {
    return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) == 0x7F800000u;
  }
};

// Running group minimum; tie_last selects which of two equal values (only
// +0.0 / -0.0 differ in bits) is kept.
__device__ __forceinline__ float min_step(float v, float mn, bool tie_last) {
  return (v < mn || (tie_last && v == mn)) ? v : mn;
}

// N == 1, G >= 32, a group whose minimum is a zero: the zero torch's
// vectorised inner reduction returns.  It reduces the first 32 * (G / 32) values
// with 4 accumulators of 8 lanes (position p in lane p % 8 of accumulator
// (p / 8) % 4; a tie keeps the later value), folds accumulator 0 with 1, 2, 3 in
// turn (a tie keeps the later accumulator) and the lanes toward lane 0 (a tie
// keeps the lower lane), then scans the G % 32 tail values (a tie keeps the
// running minimum).  So among the zeros the lowest lane wins, then the highest
// accumulator, then the latest position; a tail zero only wins when no zero
// precedes the tail, and then the first one.  Only called when the group's
// minimum is a zero, so it rescans just those groups.
template <class IN>
__device__ float inner_zero_min(const typename IN::T* __restrict__ src, int G) {
  const int B = 32 * (G / 32);
  uint64_t best = ~0ull;
  float z = 0.0f;
  for (int p = 0; p < G; ++p) {
    const float v = IN::val(src[p]);
    if (v != 0.0f) continue;
    const int s = p & 31;
    // p >> 5 < 2^26 for any int G, so the chunk term fits its 28 bits
    const uint64_t key = p < B ? ((uint64_t)(s & 7) << 32) | ((uint64_t)(3 - (s >> 3)) << 28) |
                                     (uint64_t)(0x0FFFFFFF - (p >> 5))
                               : (8ull << 32) | (uint64_t)p;
    if (key < best) {
      best = key;
      z = v;
    }
  }
  return z;
}

__device__ __forceinline__ float clamp_q(float v) {
  v = (v < 0.0f) ? 0.0f : v;
  v = (v > 15.0f) ? 15.0f : v;
  return v;
}

// One group's column: fp32 scale s, r = the rounded 1 / s, zero-point z.
struct QCol {
  float s, r, z;
};

__device__ __forceinline__ QCol make_qcol(float mn, float mx) {
  QCol c;
  const float s = (mx - mn) / 15.0f;
  c.s = (s > 0.0f) ? s : 1.0f;
  c.r = 1.0f / c.s;
  c.z = clamp_q(__builtin_rintf(-mn / c.s));
  return c;
}

// Scales for which code_of's five-operation quotient is the IEEE one wherever
// its rounding can matter (|v / s| >= 1/4): there the reciprocal is normal and
// the residual v - q s, a multiple of 2^-48 s / 4, is not below the smallest
// subnormal.
__device__ __forceinline__ bool fast_scale(float s) { return s >= 0x1p-96f && s <= 0x1p120f; }

// clamp(rint(v / s) + z, 0, 15) as a whole float.  kDiv: by IEEE division,
// about ten instructions a weight, which bound the kernel (VALU-bound at 2.5
// TB/s of an achievable 5.1).  Else by Markstein's correction (P. Markstein,
// "Computation of elementary functions on the IBM RISC System/6000 processor",
// 1990): with r = RN(1 / s), one step from v r gives a faithful quotient and a
// second the correctly rounded one.  An fp16 v enters the fused operations
// unconverted (v_fma_mix_f32).
template <bool kDiv, class H>
__device__ __forceinline__ float code_of(H v, const QCol& c) {
  float q;
  if constexpr (kDiv) {
    q = (float)v / c.s;
  } else {
    q = __builtin_fmaf((float)v, c.r, 0.0f);
    q = __builtin_fmaf(__builtin_fmaf(-q, c.s, (float)v), c.r, q);
    q = __builtin_fmaf(__builtin_fmaf(-q, c.s, (float)v), c.r, q);
  }
  return __builtin_amdgcn_fmed3f(__builtin_rintf(q) + c.z, 0.0f, 15.0f);
}

// Eight codes (whole floats in [0, 15], row order) to a packed word: two exact
// sums below 2^16.
__device__ __forceinline__ uint32_t pack_codes(const float q[8]) {
  uint32_t half[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    half[h] = (uint32_t)__builtin_fmaf(
        q[4 * h + 3], 4096.0f,
        __builtin_fmaf(q[4 * h + 2], 256.0f, __builtin_fmaf(q[4 * h + 1], 16.0f, q[4 * h])));
  return half[0] | (half[1] << 16);
}

// Four columns' weights of one row, and their running minimum and maximum: four
// adjacent columns in one load of 8 (fp16) or 16 (fp32) bytes, or columns 64
// apart (`left` of them inside N, in each lane's order) in one load each.  minimum / maximum here are the IEEE 754
// ones (v_pk_minimum3_f16, v_minimum3_f32: two rows per instruction, for fp16
// of two columns): a NaN in any row survives to the end, and of two zeros the
// minimum is -0 whatever their order, so a zero minimum's sign is found again
// in row order (min_step).
template <class IN>
struct Row4;
template <>
struct Row4<InF16> {
  typedef f16 H;
  uint2 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const uint2*>(p); }
  __device__ __forceinline__ void load_apart(const uint16_t* p, int left) {
    const uint32_t a = left > 0 ? p[0] : 0u, b = left > 1 ? p[64] : 0u;
    const uint32_t c = left > 2 ? p[128] : 0u, d = left > 3 ? p[192] : 0u;
    v = make_uint2(a | (b << 16), c | (d << 16));
  }
  __device__ __forceinline__ H at(int c) const {
    const f16x2 h = as_h2(c < 2 ? v.x : v.y);
    return c & 1 ? h.y : h.x;
  }
};
template <>
struct Row4<InF32> {
  typedef float H;
  float4 v;
  __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ void load_apart(const float* p, int left) {
    v = make_float4(left > 0 ? p[0] : 0.0f, left > 1 ? p[64] : 0.0f, left > 2 ? p[128] : 0.0f,
                    left > 3 ? p[192] : 0.0f);
  }
  __device__ __forceinline__ H at(int c) const {
    return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
  }
};
template <class IN>
struct MinMax4;
template <>
struct MinMax4<InF16> {
  f16x2 mn[2], mx[2];
  __device__ __forceinline__ void first(const Row4<InF16>& r) {
    mn[0] = mx[0] = as_h2(r.v.x);
    mn[1] = mx[1] = as_h2(r.v.y);
  }
  __device__ __forceinline__ void add(const Row4<InF16>& r) {
    const f16x2 h[2] = {as_h2(r.v.x), as_h2(r.v.y)};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      mn[i] = __builtin_elementwise_minimum(mn[i], h[i]);
      mx[i] = __builtin_elementwise_maximum(mx[i], h[i]);
    }
  }
  __device__ __forceinline__ float lo(int c) const {
    return (float)(c & 1 ? mn[c >> 1].y : mn[c >> 1].x);
  }
  __device__ __forceinline__ float hi(int c) const {
    return (float)(c & 1 ? mx[c >> 1].y : mx[c >> 1].x);
  }
};
template <>
struct MinMax4<InF32> {
  float mn[4], mx[4];
  __device__ __forceinline__ void first(const Row4<InF32>& r) {
#pragma unroll
    for (int c = 0; c < 4; ++c) mn[c] = mx[c] = r.at(c);
  }
  __device__ __forceinline__ void add(const Row4<InF32>& r) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      mn[c] = __builtin_elementwise_minimum(mn[c], r.at(c));
      mx[c] = __builtin_elementwise_maximum(mx[c], r.at(c));
    }
  }
  __device__ __forceinline__ float lo(int c) const { return mn[c]; }
  __device__ __forceinline__ float hi(int c) const { return mx[c]; }
};

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) < __builtin_inff(); }

// One workgroup of 4 waves quantises 4 / WPG groups (G rows, G % 8 == 0) of 256
// columns: lane l of each wave owns columns 4l..4l+3 (VEC: N % 4 == 0 and
// aligned W and qweight) or l, l + 64, l + 128, l + 192, and the WPG waves of a
// group contiguous parts of its packed rows (octets), in k order.
// Every lane issues all of its rows' loads at once, the minima and maxima of a
// group's waves meet in LDS in wave (k) order, and the codes come from the rows
// still in registers (OPW > 0: at most OPW octets per wave) or from a second
// read of the group (OPW = 0, long groups; the tile is L2-resident).  The
// running minimum's tie rule (min_step) applied within a wave in k order and
// across the waves in k order gives the same zero as one scan in k order.
// Column blocks are the fast grid index: neighbouring workgroups read
// neighbouring 512-byte (fp16) pieces of the same rows.
//
// About ten VALU instructions a weight, where an IEEE division and an fp32
// comparison per weight (about 34) had made it VALU-bound; now neither the VALU (57
// % of the time at K = 4096, N = 14336, G = 128) nor memory (W read once, outputs
// written once, 22 of 34 us at 6.7 TB/s) bounds it alone: a workgroup loads, reduces
// and encodes in turn, and those beside it do not fill all of its waits.  Measured
// on MI355X, K = 4096, N = 14336, us: fp16 G = 128 / 64 / 32 61.2 / 55.7 / 55.3
// -> 34.0 / 32.9 / 32.8 (4.4-4.7 TB/s of W read and the outputs written; a large
// copy reaches 5.1), G = 4096 381 -> 171, fp32 G = 128 / 32 68.3 / 53.7 -> 47.4 /
// 45.9; K = 8192, N = 28672 197 -> 115 (5.2 TB/s); N = 1001 (one thread per
// column before) 30.8 -> 18.9.
template <class IN, int OPW, int WPG, bool VEC>
__global__ __launch_bounds__(256) void quantize_tile_kernel(const typename IN::T* __restrict__ W,
                                                            uint32_t* __restrict__ QW,
                                                            uint16_t* __restrict__ SC,
                                                            uint16_t* __restrict__ ZR, int K,
                                                            int N, int G,
                                                            int32_t* __restrict__ flag) {
  static_assert(WPG == 4 || (OPW > 0 && (WPG == 1 || WPG == 2)), "waves per group");
  constexpr int GPB = 4 / WPG;   // groups per workgroup
  __shared__ float smn[WPG > 1 ? 4 : 1][256], smx[WPG > 1 ? 4 : 1][256];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nblk = (N + 255) / 256;
  const int g = (int)(blockIdx.x / (unsigned)nblk) * GPB + wave / WPG;
  constexpr int kStep = VEC ? 1 : 64;   // between a lane's columns
  const int n = (int)(blockIdx.x % (unsigned)nblk) * 256 + (VEC ? 4 : 1) * lane;
  const int left = VEC ? 4 : (N - n + 63) / 64;   // of them inside N
  const int octs = G / 8;
  const int part = wave % WPG;
  const int per = (octs + WPG - 1) / WPG;
  const int o0 = min(octs, part * per), o1 = min(octs, o0 + per);
  const bool nv = n < N && g < K / G;
  bool tie_last[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) tie_last[c] = n + c * kStep < 32 * (N / 32);
  const typename IN::T* src = W + (size_t)g * G * N + n;

  MinMax4<IN> mm;
  float mn[4], mx[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    mn[c] = __builtin_inff();
    mx[c] = -__builtin_inff();
  }
  Row4<IN> keep[OPW > 0 ? OPW : 1][8];
  auto load8 = [&](Row4<IN>(&r)[8], int o) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const typename IN::T* p = src + (size_t)(o * 8 + j) * N;
      if constexpr (VEC) r[j].load(p);
      else r[j].load_apart(p, left);
    }
  };
  if constexpr (OPW > 0) {
#pragma unroll
    for (int i = 0; i < OPW; ++i)
      if (nv && o0 + i < o1) load8(keep[i], o0 + i);
  }
  if (nv && o0 < o1) {
    auto each = [&](auto&& f) {
      if constexpr (OPW > 0) {
#pragma unroll
        for (int i = 0; i < OPW; ++i)
          if (o0 + i < o1) f(keep[i], i == 0);
      } else {
        for (int o = o0; o < o1; ++o) {
          load8(keep[0], o);
          f(keep[0], o == o0);
        }
      }
    };
    each([&](const Row4<IN>(&r)[8], bool head) {
      if (head) mm.first(r[0]);
      else mm.add(r[0]);
#pragma unroll
      for (int j = 1; j < 8; ++j) mm.add(r[j]);
    });
    bool bad = false, zero = false;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      mn[c] = mm.lo(c);
      mx[c] = mm.hi(c);
      bad |= !finite(mn[c]) || !finite(mx[c]);
      zero |= mn[c] == 0.0f;
    }
    if (bad) *flag = 1;
    if (zero) {   // the sign of a zero minimum: the first or the last zero in k order
      float z[4] = {__builtin_inff(), __builtin_inff(), __builtin_inff(), __builtin_inff()};
      each([&](const Row4<IN>(&r)[8], bool) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int c = 0; c < 4; ++c) z[c] = min_step((float)r[j].at(c), z[c], tie_last[c]);
      });
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (mn[c] == 0.0f) mn[c] = z[c];
    }
  }
  if constexpr (WPG > 1) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      smn[wave][4 * lane + c] = mn[c];
      smx[wave][4 * lane + c] = mx[c];
    }
    __syncthreads();
    const int w0 = wave - part;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      mn[c] = smn[w0][4 * lane + c];
      mx[c] = smx[w0][4 * lane + c];
#pragma unroll
      for (int w = 1; w < WPG; ++w) {
        const float u = smx[w0 + w][4 * lane + c];
        mn[c] = min_step(smn[w0 + w][4 * lane + c], mn[c], tie_last[c]);
        mx[c] = (u >= mx[c]) ? u : mx[c];
      }
    }
  }
  if (!nv) return;
  if constexpr (!VEC) {
    if (N == 1 && G >= 32 && mn[0] == 0.0f) mn[0] = inner_zero_min<IN>(src, G);
  }
  QCol qc[4];
  bool fast = true;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    qc[c] = make_qcol(mn[c], mx[c]);
    fast &= fast_scale(qc[c].s);
  }
  auto codes = [&](auto div, const Row4<IN>(&r)[8], int o) {
    uint32_t word[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float q[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = code_of<decltype(div)::value>(r[j].at(c), qc[c]);
      word[c] = pack_codes(q);
    }
    uint32_t* dst = QW + (size_t)(g * octs + o) * N + n;
    if constexpr (VEC) {
      *reinterpret_cast<uint4*>(dst) = make_uint4(word[0], word[1], word[2], word[3]);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < left) dst[c * kStep] = word[c];
    }
  };
  auto all_codes = [&](auto div) {
    if constexpr (OPW > 0) {
#pragma unroll
      for (int i = 0; i < OPW; ++i)
        if (o0 + i < o1) codes(div, keep[i], o0 + i);
    } else {
      for (int o = o0; o < o1; ++o) {
        load8(keep[0], o);
        codes(div, keep[0], o);
      }
    }
  };
  if (__all(fast)) all_codes(std::false_type{});
  else all_codes(std::true_type{});
  if (part == 0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c < left) {
        SC[(size_t)g * N + n + c * kStep] = as_u16((f16)qc[c].s);
        ZR[(size_t)g * N + n + c * kStep] = as_u16((f16)qc[c].z);
      }
    }
  }
}

// v from another lane of the same group of L consecutive lanes, step D of a
// butterfly (D = 1, 2, 4, 8 by DPP: within quads, mirrored halves and rows of
// 16 lanes; 16 and 32 through the LDS crossbar).
template <int D>
__device__ __forceinline__ uint32_t lane_swap(uint32_t v) {
  if constexpr (D >= 16) {
    return (uint32_t)__shfl_xor((int)v, D);
  } else {
    constexpr int ctrl = D == 1 ? 0xB1 : D == 2 ? 0x4E : D == 4 ? 0x141 : 0x140;
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, 0xF, 0xF, false);
  }
}

// Eight consecutive k of one column (a packed word's worth): loads, minimum and
// maximum over L lanes (IEEE minimum / maximum, as MinMax4).
template <class IN>
struct Oct;
template <>
struct Oct<InF16> {
  uint4 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const uint4*>(p); }
  // keeps the compiler from carrying converted copies of the weights (twice
  // their registers) from one pass
  // over them to the next
  __device__ __forceinline__ void hide() { asm("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }
  __device__ __forceinline__ f16 at(int j) const {
    const f16x2 h = as_h2(j < 2 ? v.x : j < 4 ? v.y : j < 6 ? v.z : v.w);
    return j & 1 ? h.y : h.x;
  }
  template <int L>
  __device__ __forceinline__ void min_max(float& mn, float& mx) const {
    const f16x2 a = as_h2(v.x), b = as_h2(v.y), c = as_h2(v.z), d = as_h2(v.w);
    f16x2 lo = __builtin_elementwise_minimum(
        __builtin_elementwise_minimum(a, b), __builtin_elementwise_minimum(c, d));
    f16x2 hi = __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(a, b), __builtin_elementwise_maximum(c, d));
    auto fold = [&](auto step) {
      constexpr int D = decltype(step)::value;
      if constexpr (D < L) {
        lo = __builtin_elementwise_minimum(lo, as_h2(lane_swap<D>(as_u32(lo))));
        hi = __builtin_elementwise_maximum(hi, as_h2(lane_swap<D>(as_u32(hi))));
      }
    };
    fold(std::integral_constant<int, 1>{});
    fold(std::integral_constant<int, 2>{});
    fold(std::integral_constant<int, 4>{});
    fold(std::integral_constant<int, 8>{});
    fold(std::integral_constant<int, 16>{});
    fold(std::integral_constant<int, 32>{});
    mn = __builtin_elementwise_minimum((float)lo.x, (float)lo.y);
    mx = __builtin_elementwise_maximum((float)hi.x, (float)hi.y);
  }
};
template <>
struct Oct<InF32> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = reinterpret_cast<const float4*>(p)[0];
    b = reinterpret_cast<const float4*>(p)[1];
  }
  __device__ __forceinline__ void hide() {}
  __device__ __forceinline__ float at(int j) const {
    const float4 f = j < 4 ? a : b;
    return (j & 3) == 0 ? f.x : (j & 3) == 1 ? f.y : (j & 3) == 2 ? f.z : f.w;
  }
  template <int L>
  __device__ __forceinline__ void min_max(float& mn, float& mx) const {
    mn = mx = at(0);
#pragma unroll
    for (int j = 1; j < 8; ++j) {
      mn = __builtin_elementwise_minimum(mn, at(j));
      mx = __builtin_elementwise_maximum(mx, at(j));
    }
    auto fold = [&](auto step) {
      constexpr int D = decltype(step)::value;
      if constexpr (D < L) {
        mn = __builtin_elementwise_minimum(
            mn, __builtin_bit_cast(float, lane_swap<D>(__builtin_bit_cast(uint32_t, mn))));
        mx = __builtin_elementwise_maximum(
            mx, __builtin_bit_cast(float, lane_swap<D>(__builtin_bit_cast(uint32_t, mx))));
      }
    };
    fold(std::integral_constant<int, 1>{});
    fold(std::integral_constant<int, 2>{});
    fold(std::integral_constant<int, 4>{});
    fold(std::integral_constant<int, 8>{});
    fold(std::integral_constant<int, 16>{});
    fold(std::integral_constant<int, 32>{});
  }
};

// Quantise from the transposed weight: column n's K weights lie in a row of
// `ldw` elements (an nn.Linear weight [N, K]), so no transposed copy of W is
// made first.  G = 8 L, L a power of two from 4 to 64.  A workgroup of 4 waves
// takes 32 columns x 512 k: a wave reads one column's 512 k as one contiguous
// kilobyte (fp16), lane l holding the 8 k of one packed word; the L lanes of a
// group find its minimum and maximum by a butterfly, each of them finishes one
// column's (or several columns') scale and zero-point, and the words are turned
// round through LDS (rows padded by a word, no bank conflicts) so that they
// leave as runs of 32 adjacent words.  A zero minimum takes the sign of the
// first or last zero in k order (min_step), found from the wave's ballots.
// Bound as quantize_tile_kernel: VALU issue about two thirds of the time, bytes 17
// of 30 us.  Measured on MI355X, us, kernel alone: K = 4096, N = 11008 /
// 14336, G = 128 29.9 / 35.2 (4.2 TB/s), fp32 N = 14336 44.8 (6.0 TB/s), K =
// 8192, N = 28672 116.9; before, a transposing copy (292 at N = 11008) and the
// row-major quantiser.  16 columns a wave (runs of 64 words, 133 registers, three
// waves per SIMD) took 33.7 / 38.6.
constexpr int kNkCols = 8;   // columns per wave
template <class IN, int L>
__global__ __launch_bounds__(256) void quantize_nk_kernel(const typename IN::T* __restrict__ W,
                                                          int64_t ldw, uint32_t* __restrict__ QW,
                                                          uint16_t* __restrict__ SC,
                                                          uint16_t* __restrict__ ZR, int K, int N,
                                                          int32_t* __restrict__ flag) {
  static_assert(L >= 4 && L <= 64 && (L & (L - 1)) == 0, "a group is L lanes of a wave");
  constexpr int R = kNkCols, kCols = 4 * R;
  constexpr int kGrp = 64 / L;                     // groups in a wave's 512 k
  constexpr int kOwn = L >= R ? 1 : R / L;         // columns a lane finishes
  __shared__ uint32_t words[64][kCols + 1];
  __shared__ float4 stat[4][R][kGrp];              // s, r, z, fast_scale
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nkc = (K + 511) / 512;
  const int kc = (int)(blockIdx.x % (unsigned)nkc);
  const int n0 = (int)(blockIdx.x / (unsigned)nkc) * kCols;
  const int k = kc * 512 + 8 * lane;
  const bool kv = k < K;                           // whole groups: K % G == 0
  const int sub = lane % L, grp = lane / L;

  // Lanes past K and columns past N load in-range weights whose results go
  // nowhere: under a branch each load would be waited for before the next.
  Oct<IN> v[R];
#pragma unroll
  for (int i = 0; i < R; ++i)
    v[i].load(W + (size_t)min(N - 1, n0 + wave * R + i) * ldw + (kv ? k : 0));
  float omn[kOwn] = {}, omx[kOwn] = {};
  bool bad = false;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float mn, mx;
    v[i].template min_max<L>(mn, mx);
    bad |= !finite(mn) || !finite(mx);
    if (__any(mn == 0.0f)) {
      const bool last = n0 + wave * R + i < 32 * (N / 32);
      float z = __builtin_inff();
      v[i].hide();
#pragma unroll
      for (int j = 0; j < 8; ++j) z = min_step((float)v[i].at(j), z, last);
      const uint64_t has = __ballot(z == 0.0f);
      const uint64_t neg = __ballot(z == 0.0f && __builtin_signbit(z));
      const uint64_t mine = (has >> (grp * L)) & (L == 64 ? ~0ull : (1ull << (L % 64)) - 1ull);
      if (mn == 0.0f) {
        const int at = grp * L + (last ? 63 - __builtin_clzll(mine) : __builtin_ctzll(mine));
        mn = (neg >> at) & 1ull ? -0.0f : 0.0f;
      }
    }
    if (sub == i % L) {
      omn[i / L] = mn;
      omx[i / L] = mx;
    }
  }
  if (bad) *flag = 1;
#pragma unroll
  for (int o = 0; o < kOwn; ++o) {
    const int i = o * L + sub;
    if (i < R) {
      const QCol c = make_qcol(omn[o], omx[o]);
      stat[wave][i][grp] = make_float4(c.s, c.r, c.z, fast_scale(c.s) ? 1.0f : 0.0f);
      const int n = n0 + wave * R + i;
      if (kv && n < N) {
        const size_t at = (size_t)(kc * kGrp + grp) * N + n;
        SC[at] = as_u16((f16)c.s);
        ZR[at] = as_u16((f16)c.z);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < R; ++i) {
    v[i].hide();
    const float4 st = stat[wave][i][grp];
    const QCol c{st.x, st.y, st.z};
    float q[8];
    if (__all(st.w != 0.0f)) {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = code_of<false>(v[i].at(j), c);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = code_of<true>(v[i].at(j), c);
    }
    words[lane][wave * R + i] = pack_codes(q);
  }
  __syncthreads();
  constexpr int kRows = 256 / kCols;               // packed rows written at once
  const int wc = threadIdx.x % kCols, wr = threadIdx.x / kCols;
#pragma unroll
  for (int o = 0; o < 64; o += kRows) {
    const int row = kc * 64 + o + wr;
    if (row < K / 8 && n0 + wc < N) QW[(size_t)row * N + n0 + wc] = words[o + wr][wc];
  }
}

// Any G dividing K (G % 8 != 0 lets a packed word straddle groups): one thread
// per packed word; each row's group statistics are recomputed from the group's
// G values, and the thread that owns a group's first row writes its scale/zero.
struct GroupQ {
  float scale, zero;
  bool bad;
};

template <class IN>
__device__ GroupQ group_stats(const typename IN::T* __restrict__ W, int g, int G, int N, int n) {
  const typename IN::T* src = W + (size_t)g * G * N + n;
  typename IN::T b = src[0];
  bool bad = IN::nonfinite(b);
  float mn = IN::val(b), mx = mn;
  const bool tie_last = n < 32 * (N / 32);
  for (int r = 1; r < G; ++r) {
    b = src[(size_t)r * N];
    bad |= IN::nonfinite(b);
    const float v = IN::val(b);
    mn = min_step(v, mn, tie_last);
    mx = (v >= mx) ? v : mx;
  }
  if (N == 1 && G >= 32 && mn == 0.0f) mn = inner_zero_min<IN>(src, G);
  float s = (mx - mn) / 15.0f;
  s = (s > 0.0f) ? s : 1.0f;
  return GroupQ{s, clamp_q(__builtin_rintf(-mn / s)), bad};
}

template <class IN>
__global__ __launch_bounds__(256) void quantize_general_kernel(
    const typename IN::T* __restrict__ W, uint32_t* __restrict__ QW, uint16_t* __restrict__ SC,
    uint16_t* __restrict__ ZR, int K, int N, int G, int32_t* __restrict__ flag) {
  const int n = blockIdx.y * 256 + threadIdx.x;
  const int i = blockIdx.x;
  if (n >= N) return;
  uint32_t word = 0u;
  int gcur = -1;
  GroupQ gq{1.0f, 0.0f, false};
  bool bad = false;
  for (int j = 0; j < 8; ++j) {
    const int k = 8 * i + j;
    const int g = k / G;
    if (g != gcur) {
      gcur = g;
      gq = group_stats<IN>(W, g, G, N, n);
      bad |= gq.bad;
      if (k == g * G) {
        SC[(size_t)g * N + n] = as_u16((f16)gq.scale);
        ZR[(size_t)g * N + n] = as_u16((f16)gq.zero);
      }
    }
    const float q = clamp_q(__builtin_rintf(IN::val(W[(size_t)k * N + n]) / gq.scale) + gq.zero);
    word |= ((uint32_t)(int)q & 0xFu) << (4 * j);
  }
  if (bad) *flag = 1;
  QW[(size_t)i * N + n] = word;
}

// pack_int4: int32 codes [K, N] -> int32 [K/8, N]; flags values outside [0, 15].
__global__ __launch_bounds__(256) void pack_kernel(const int32_t* __restrict__ Q,
                                                   uint32_t* __restrict__ QW, int K, int N,
                                                   int32_t* __restrict__ flag) {
  const int n = blockIdx.y * 256 + threadIdx.x;
  const int i = blockIdx.x;
  if (n >= N) return;
  uint32_t word = 0u;
  bool bad = false;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int32_t v = Q[(size_t)(8 * i + j) * N + n];
    bad |= (v < 0) | (v > 15);
    word |= ((uint32_t)v & 0xFu) << (4 * j);
  }
  if (bad) *flag = 1;
  QW[(size_t)i * N + n] = word;
}

// unpack_int4: int32 [K/8, N] -> int32 codes [K, N].
__global__ __launch_bounds__(256) void unpack_kernel(const uint32_t* __restrict__ QW,
                                                     int32_t* __restrict__ Q, int K, int N) {
  const int n = blockIdx.y * 256 + threadIdx.x;
  const int i = blockIdx.x;
  if (n >= N) return;
  const uint32_t w = QW[(size_t)i * N + n];
#pragma unroll
  for (int j = 0; j < 8; ++j) Q[(size_t)(8 * i + j) * N + n] = (int32_t)((w >> (4 * j)) & 0xFu);
}

// dequantize_weight: fp16 (fp16(q) - z) * s for any fp16 zero-point.
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ QW,
                                                      const f16* __restrict__ SC,
                                                      const f16* __restrict__ ZR,
                                                      f16* __restrict__ Wd, int K, int N, int G) {
  const int n = blockIdx.y * 256 + threadIdx.x;
  const int i = blockIdx.x;
  if (n >= N) return;
  const uint32_t w = QW[(size_t)i * N + n];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int g = (8 * i + j) / G;
    const f16 s = SC[(size_t)g * N + n];
    const f16 z = ZR[(size_t)g * N + n];
    const f16 q = (f16)(float)((w >> (4 * j)) & 0xFu);
    Wd[(size_t)(8 * i + j) * N + n] = (q - z) * s;
  }
}

// dequantize_weight, C = 8 or 4 adjacent columns of one packed row per lane (G %
// 8 == 0: one group): 16-byte weight loads, and rows stored 2 C bytes per lane,
// so that a wave writes 1024 or 512 contiguous bytes of a row.  Two columns'
// codes of one row make a packed pair: byte b of both words (v_perm_b32) holds
// rows 2b and 2b + 1 as nibbles, which the magic words turn into the fp16 pairs
// 1024 + q and 64 + q; the magic is subtracted first (exact), then (q - z) * s is
// rounded as dequant_kernel rounds it.  Bound by memory, mostly by
// the stores, which are non-temporal (W is written once, and need not pass
// through L2).  Measured on MI355X with cold operands, us, one column a lane ->
// this with plain stores -> non-temporal: K = 4096, N = 11008 / 14336 42.7 / 54.0
// -> 25.4 / 28.8 -> 17.0 / 23.7 (6.3-6.7 TB/s); K = 8192, N = 28672 213 -> 104 ->
// 91.6; four columns, N = 11004 42.5 -> 27.6 -> 25.2.
template <int C>
__global__ __launch_bounds__(256) void dequant_vec_kernel(const uint32_t* __restrict__ QW,
                                                          const uint16_t* __restrict__ SC,
                                                          const uint16_t* __restrict__ ZR,
                                                          uint16_t* __restrict__ Wd, int N,
                                                          int octs) {
  static_assert(C == 4 || C == 8, "one or two 16-byte weight loads");
  typedef uint32_t Vec __attribute__((ext_vector_type(C / 2)));   // C halves
  const int nblk = (N + 256 * C - 1) / (256 * C);
  const int i = (int)(blockIdx.x / (unsigned)nblk);               // packed row
  const int n = ((int)(blockIdx.x % (unsigned)nblk) * 256 + (int)threadIdx.x) * C;
  if (n >= N) return;
  const size_t at = (size_t)(i / octs) * N + n;
  uint32_t w[C];
#pragma unroll
  for (int c = 0; c < C; c += 4) {
    const uint4 v = *reinterpret_cast<const uint4*>(QW + (size_t)i * N + n + c);
    w[c] = v.x, w[c + 1] = v.y, w[c + 2] = v.z, w[c + 3] = v.w;
  }
  const Vec s = *reinterpret_cast<const Vec*>(SC + at);
  const Vec z = *reinterpret_cast<const Vec*>(ZR + at);
  const MagicRegs mg = make_magic();
  uint16_t* dst = Wd + (size_t)i * 8 * N + n;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    Vec even, odd;
#pragma unroll
    for (int c = 0; c < C / 2; ++c) {
      // byte b of column 2c into byte 0, of column 2c + 1 into byte 2
      const uint32_t t = __builtin_amdgcn_perm(w[2 * c + 1], w[2 * c],
                                               0x0C040C00u + 0x00010001u * (uint32_t)b);
      const f16x2 lo = as_h2(and_or(t, 0x000F000Fu, mg.m1024)) - as_h2(mg.m1024);
      const f16x2 hi = as_h2(and_or(t, 0x00F000F0u, mg.m64)) - as_h2(mg.m64);
      even[c] = as_u32((lo - as_h2(z[c])) * as_h2(s[c]));
      odd[c] = as_u32((hi - as_h2(z[c])) * as_h2(s[c]));
    }
    __builtin_nontemporal_store(even, reinterpret_cast<Vec*>(dst + (size_t)(2 * b) * N));
    __builtin_nontemporal_store(odd, reinterpret_cast<Vec*>(dst + (size_t)(2 * b + 1) * N));
  }
}

// Zero-points outside the integer-zero kernels' domain (w4a16_device.h): any
// zero that is not an integer in [-1024, 1024] (NaN and infinities included)
// sets *flag.  Grid-stride over the n halves; every offending lane stores 1.
__global__ __launch_bounds__(256) void zeros_check_kernel(const f16* __restrict__ Z, int64_t n,
                                                          int32_t* __restrict__ flag) {
  bool bad = false;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    const float z = (float)Z[i];
    bad |= !(z == __builtin_rintf(z) && __builtin_fabsf(z) <= 1024.0f);
  }
  if (bad) *flag = 1;
}

template <class IN, bool VEC>
hipError_t quantize_tile_launch(const typename IN::T* w, uint32_t* q, uint16_t* s, uint16_t* z,
                                int K, int N, int G, int32_t* flag, hipStream_t st) {
  // Waves per group and octets per wave, so that a wave keeps about four
  // octets (32 rows) in registers whatever G: one wave per group up to G = 32,
  // two at 64, four beyond; more than 8 (fp16) / 4 (fp32) octets a wave are
  // read twice.  Four waves share a shorter group too where that is faster; `blocks4`
  // is the number of workgroups it makes.
  //  * None of the four without an octet (octs 4, 7, 8): below 1024 waves otherwise,
  //    fewer than SIMDs, where the time is one wave's own (G = 32, us, one wave a
  //    group -> four: K = 3712, N = 64 9.2 -> 3.7; K = 768, N = 320 7.6 -> 4.2; at 1024
  //    waves, K = 4096, N = 2048, 6.2 against 6.9).  With columns apart, whose loads a
  //    wave issues one by one, far beyond (fp16, N = 2045, K = 4096, G = 32 / 64 17.2 /
  //    17.5 -> 11.0 / 11.8; K = 4096, N = 14335, G = 64 63.8 -> 63.0); at G = 32 up to
  //    4096 (2688, N = 5121 30.9 -> 28.1; 7616, K = 14336, N = 4098 61.0 against 65.3).
  //  * Else (octs 2, 3, 5, 6) a wave idles through the workgroup's time: only while
  //    each CU gets one workgroup (fp16, K = 1000 / 4080, N = 1024, G = 40, 100 / 408
  //    workgroups 5.1 -> 4.3 / 5.4 against 5.8), with columns apart two (K = 4080,
  //    N = 1021 / 14335, 408 / 5712 workgroups 12.4 -> 10.9 / 68.6 against 87.2).
  const int octs = G / 8, per = (octs + 3) / 4;
  constexpr int kMaxKeep = sizeof(typename IN::T) == 2 ? 8 : 4;
  const int64_t blocks4 = (int64_t)(K / G) * ((N + 255) / 256);
  const bool four = octs > 1 && octs <= 8 &&
                    (octs <= 3 * per ? blocks4 <= (VEC ? 256 : 512)
                     : VEC           ? blocks4 * (octs <= 4 ? 1 : 2) < 1024
                                     : octs > 4 || blocks4 < 4096);
  const int gpb = four ? 1 : octs <= 4 ? 4 : octs <= 8 ? 2 : 1;   // groups per workgroup
  auto k = four        ? quantize_tile_kernel<IN, 4, 4, VEC>
           : octs <= 1 ? quantize_tile_kernel<IN, 1, 1, VEC>
           : octs <= 2 ? quantize_tile_kernel<IN, 2, 1, VEC>
           : octs <= 4 ? quantize_tile_kernel<IN, 4, 1, VEC>
           : octs <= 8 ? quantize_tile_kernel<IN, 4, 2, VEC>
           : per <= 4  ? quantize_tile_kernel<IN, 4, 4, VEC>
           : per <= kMaxKeep ? quantize_tile_kernel<IN, kMaxKeep, 4, VEC>
                             : quantize_tile_kernel<IN, 0, 4, VEC>;
  const unsigned blocks = (unsigned)((K / G + gpb - 1) / gpb) * (unsigned)((N + 255) / 256);
  hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, st, w, q, s, z, K, N, G, flag);
  return hipGetLastError();
}

template <class IN>
hipError_t quantize_launch(const void* W, int32_t* qw, void* sc, void* zr, int K, int N, int G,
                           int32_t* flag, hipStream_t st) {
  typedef typename IN::T T;
  const T* w = static_cast<const T*>(W);
  uint32_t* q = reinterpret_cast<uint32_t*>(qw);
  uint16_t* s = static_cast<uint16_t*>(sc);
  uint16_t* z = static_cast<uint16_t*>(zr);
  if (G % 8 != 0) {
    dim3 grid(K / 8, (N + 255) / 256);
    hipLaunchKernelGGL(quantize_general_kernel<IN>, grid, dim3(256), 0, st, w, q, s, z, K, N, G,
                       flag);
    return hipGetLastError();
  }
  const uintptr_t wa = 4 * sizeof(T);
  const bool vec = (N % 4 == 0) && ((reinterpret_cast<uintptr_t>(W) & (wa - 1)) == 0) &&
                   ((reinterpret_cast<uintptr_t>(qw) & 15) == 0);
  return vec ? quantize_tile_launch<IN, true>(w, q, s, z, K, N, G, flag, st)
             : quantize_tile_launch<IN, false>(w, q, s, z, K, N, G, flag, st);
}

template <class IN>
hipError_t quantize_nk_launch(const void* W, int64_t ldw, int32_t* qw, void* sc, void* zr, int K,
                              int N, int G, int32_t* flag, hipStream_t st) {
  auto k = G == 32    ? quantize_nk_kernel<IN, 4>
           : G == 64  ? quantize_nk_kernel<IN, 8>
           : G == 128 ? quantize_nk_kernel<IN, 16>
           : G == 256 ? quantize_nk_kernel<IN, 32>
                      : quantize_nk_kernel<IN, 64>;
  const unsigned blocks = (unsigned)((K + 511) / 512) * (unsigned)((N + 4 * kNkCols - 1) / (4 * kNkCols));
  hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, st, static_cast<const typename IN::T*>(W), ldw,
                     reinterpret_cast<uint32_t*>(qw), static_cast<uint16_t*>(sc),
                     static_cast<uint16_t*>(zr), K, N, flag);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_quantize_pack(const void* W, bool w_is_f32, int32_t* qw, void* sc, void* zr,
                                int K, int N, int G, int32_t* flag, hipStream_t st) {
  return w_is_f32 ? quantize_launch<InF32>(W, qw, sc, zr, K, N, G, flag, st)
                  : quantize_launch<InF16>(W, qw, sc, zr, K, N, G, flag, st);
}

bool quantize_nk_applicable(const void* W, bool w_is_f32, int64_t ldw, int K, int N, int G) {
  // rows of whole 16-byte loads; N == 1 has its own zero rule (inner_zero_min)
  const int64_t elems = w_is_f32 ? 4 : 8;
  return N >= 2 && ldw >= K && ldw % elems == 0 && K % 8 == 0 &&
         (reinterpret_cast<uintptr_t>(W) & 15) == 0 &&
         (G == 32 || G == 64 || G == 128 || G == 256 || G == 512) && K % G == 0;
}

hipError_t launch_quantize_pack_nk(const void* W, bool w_is_f32, int64_t ldw, int32_t* qw,
                                   void* sc, void* zr, int K, int N, int G, int32_t* flag,
                                   hipStream_t st) {
  return w_is_f32 ? quantize_nk_launch<InF32>(W, ldw, qw, sc, zr, K, N, G, flag, st)
                  : quantize_nk_launch<InF16>(W, ldw, qw, sc, zr, K, N, G, flag, st);
}

hipError_t launch_pack(const int32_t* q, int32_t* qw, int K, int N, int32_t* flag,
                       hipStream_t st) {
  dim3 grid(K / 8, (N + 255) / 256);
  hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, st, q, reinterpret_cast<uint32_t*>(qw), K,
                     N, flag);
  return hipGetLastError();
}

hipError_t launch_unpack(const int32_t* qw, int32_t* q, int K, int N, hipStream_t st) {
  dim3 grid(K / 8, (N + 255) / 256);
  hipLaunchKernelGGL(unpack_kernel, grid, dim3(256), 0, st,
                     reinterpret_cast<const uint32_t*>(qw), q, K, N);
  return hipGetLastError();
}

hipError_t launch_zeros_check(const void* zr, int64_t n, int32_t* flag, hipStream_t st) {
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(zeros_check_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256),
                     0, st, static_cast<const f16*>(zr), n, flag);
  return hipGetLastError();
}

hipError_t launch_dequant(const int32_t* qw, const void* sc, const void* zr, void* w, int K,
                          int N, int G, hipStream_t st) {
  // 8 columns a lane where rows and pointers allow its 16-byte accesses and a row
  // has 128 columns (N = 64, K = 4736 / 11520 2.5 / 3.0 us at 8 columns, 2.0 / 2.4 at
  // 4; N = 128 a tie), 4 where they allow 8-byte ones (N = 4, K = 8928 2.2 us against
  // 2.5 at one; N = 108, K = 4096 2.0 against 2.3); else, and where a packed row holds
  // two groups, one
  auto ok = [&](int c) {
    const uintptr_t m = 2 * (uintptr_t)c - 1;
    return N % c == 0 && (c == 4 || N >= 128) && G % 8 == 0 &&
           (((reinterpret_cast<uintptr_t>(sc) | reinterpret_cast<uintptr_t>(zr) |
              reinterpret_cast<uintptr_t>(w)) & m) |
            (reinterpret_cast<uintptr_t>(qw) & 15)) == 0;
  };
  const int c = ok(8) ? 8 : ok(4) ? 4 : 1;
  const unsigned blocks = (unsigned)(K / 8) * (unsigned)((N + 256 * c - 1) / (256 * c));
  if (c > 1) {
    hipLaunchKernelGGL((c == 8 ? dequant_vec_kernel<8> : dequant_vec_kernel<4>), dim3(blocks),
                       dim3(256), 0, st, reinterpret_cast<const uint32_t*>(qw),
                       static_cast<const uint16_t*>(sc), static_cast<const uint16_t*>(zr),
                       static_cast<uint16_t*>(w), N, G / 8);
    return hipGetLastError();
  }
  dim3 grid(K / 8, (N + 255) / 256);
  hipLaunchKernelGGL(dequant_kernel, grid, dim3(256), 0, st,
                     reinterpret_cast<const uint32_t*>(qw), static_cast<const f16*>(sc),
                     static_cast<const f16*>(zr), static_cast<f16*>(w), K, N, G);
  return hipGetLastError();
}

}  // namespace w4a16
