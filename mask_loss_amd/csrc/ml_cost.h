// Pairwise sigmoid-BCE / dice cost as an MFMA contraction (gfx950).  The kernels and
// their launches, by logit type; ml_cost_f32.hip, ml_cost_bf16.hip and ml_cost_f16.hip
// instantiate one type each (they compile side by side), ml_cost.hip picks among them.
//
// For one image b and query q, with per-cell planes A_neg = w an mn cn, A_pos =
// w ap mp cp, A_p = w p, A_w = w and the count n_g(cell) of GT column g:
//   bce_num(g) = sum A_neg (N2 - n_g) + A_pos n_g, I(g) = sum A_p n_g, T(g) = sum A_w n_g
// This is the reference's fused BCE+dice reduction (src/cuda/pw_mask.cu:52-308)
// as (Q x K)(K x G) products, its base + Delta of :300 regrouped so that both
// terms are non-negative (no cancellation); I and T as :270-271.  Class 0 (up to
// 31 non-empty GTs) sums these three, and a ones column (slot G, n = N2
// everywhere) gives the row sums P = sum N2 w p and S = sum N2 w (:140-141).
// The wide classes sum the four planes per slot instead,
//   N(s) = sum A_neg n_s, Pos(s) = sum A_pos n_s, I(s), T(s),
// slot G holding the pixels of no column, and finalize rebuilds the bce numerator of
// slot g as sum_{s != g} N(s) + Pos(g) and P, S as the sums of I and T over all
// slots: their right operands are zero outside the tiles that a K-step's cells
// touch, so those tiles' MFMAs are skipped.
//
// Operands are float16 where that loses nothing, else bf16.  A float16 plane is
// scaled by 2^lg (cost_form: the largest scale that keeps it finite) and split into
// two terms for float32 and float16 logits (22 bits), one for bf16 ones (11
// bits).  Below 2^-14 a scaled plane has absolute steps of 2^-24 instead: a plane is
// then up to 2^-25-lg off, 2e-12 at the operator's default weights and 3e-11 without
// weights.  The formulas are 6e-8 w off there themselves (1 + e^-|z| rounded to
// float32), but only as long as no factor makes the planes small: where a focal
// power does, or an uncertainty weight with a floor below 2^-6 (CostForm::wide), and
// where a range holds |z| > 60, the operands are bf16 terms (3, 2 or 1), which
// keep 24, 16 or 8 bits of any float32.
//
// The right operand is made of 16-bit integer ops: label codes of two
// labels differ by at least 0x100 under xor, so a saturating subtraction of the
// xor from 0x100 gives 0x100 (as a float16: 2^-16) where they agree and 0
// elsewhere; times a constant it is 2^-lg or a bf16 one.  The table kernels take
// the 2^-16 itself (the matrix cores align a subnormal factor's product without
// normalising it: that costs two of the plane's 11 bits).  A u8 count n under a
// float16 exponent whose last place is 2^-lg becomes 2^(10-lg) + 2^-lg n by one byte
// permute, then 2^-lg n.  Scales are powers of two, so no result depends on them
// but for the steps above.
//
// The kernels by formula are bound by vector-ALU issue (~25 ops and 3 transcendental
// per logit, a third of them the split), the widest class by latency at one wave per
// SIMD.  Float32 logits, bf16 operands throughout / float16 where they fit: 10 M in 32
// columns 28.1 / 22.2 us (focal gamma 2, bf16 operands by its rule: 29.8), 33.6 M
// against 4x targets 96 / 59, the 16- and 7-tile launches of 39 M 113 + 49 / 97 +
// 40.  A range that is redone costs its formula pass again: 40% of 10 M logits
// filled with -10^4, whole cost call 41.4 / 42.9 us (float16 logits 40.0 / 39.5; bf16
// ones, in the table's kernels, 45.0 / 43.4, against 4x targets 49.5 / 50.2).  Some logit
// beyond 60 in every K-step (20 M of sigma 24): 76.6 / 86.3 us, 66.8 / 77.6 and 76.5 / 74.0.
//
// Work decomposition: one wave = 16 query rows of one image over a
// contiguous range of 32-cell K-steps; each image is handled by the kernel
// instance whose column-tile count NT matches its number of non-empty GTs (+1
// slot), so accumulator registers are sized to the image, not to the padded
// GT width.
//
// Per-cell planes: bf16 logits take only 65536 values, so for them the four
// planes are read from a per-workgroup LDS table built with the same float32
// formulas (|z| in [2^-9, 64): one entry per bf16 value; |z| < 2^-9: the
// z = 0 entry, within 2^-9.5 of those; |z| >= 64, inf and nan read a NaN
// marker, and a wave whose sums come out NaN redoes its K-range with the
// formulas).  Other dtypes evaluate the formulas directly.
#pragma once

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "ml_internal.h"

namespace ml {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2_t as_u16x2(uint32_t v) { return __builtin_bit_cast(u16x2_t, v); }
__device__ __forceinline__ uint32_t as_u32(u16x2_t v) { return __builtin_bit_cast(uint32_t, v); }

// terms per plane: float16 operands, and bf16 ones
template <int DT>
struct InTraits;
template <>
struct InTraits<ML_F32> {
  static constexpr int kTerms = 2, kWide = 3;
};
template <>
struct InTraits<ML_BF16> {
  static constexpr int kTerms = 1, kWide = 1;
};
template <>
struct InTraits<ML_F16> {
  static constexpr int kTerms = 2, kWide = 2;
};

// ---- LUT geometry (bytes): positive block at 0, negative block at 32768 ----
constexpr uint32_t kLutBase = 118u << 7;         // bf16 magnitude bits of 2^-9
constexpr uint32_t kLutOver = 0x4280u;           // bf16 magnitude bits of 64.0
constexpr uint32_t kLutN = kLutOver - kLutBase;  // 1920 regular entries
constexpr uint32_t kLutSub = kLutBase - 1;       // idx = sat(m - kLutSub): 0 = tiny
constexpr uint32_t kLutBlock = kLutN + 2;        // tiny + regular + overflow slot
constexpr uint32_t kLutNegOff = 32768;
constexpr uint32_t kLutBytes = kLutNegOff + kLutBlock * 8;
constexpr float kNarrowMax = 60.f;               // of |z|: float16 operands by formula (see the top)
constexpr int kDepth = 4;  // K-steps of logits in flight per wave

__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
  f32x2_t f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2_t));
}
// v minus the low / high float16 of w, exactly rounded (one mixed-precision fma)
__device__ __forceinline__ float rem_lo(float v, uint32_t w) {
  float r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(v));
  return r;
}
__device__ __forceinline__ float rem_hi(float v, uint32_t w) {
  float r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(v));
  return r;
}

// ---- planes of one logit ---------------------------------------------------
// Which of the per-logit forms a call takes (chosen once per 8 logits, wave-uniform):
// 0 general; 1 no focal terms, weight H^1 (the operator's defaults); 2 no
// focal terms, no weights; 3 focal gamma 2 with or without weights H^1; 4 no focal
// terms, weight H^ug.
__device__ __forceinline__ int elem_mode(const ElemParams& ep) {
  const bool plain = ep.gamma_mode == 0 && ep.an == 1.f && ep.ap == 1.f;
  if (plain && ep.ug_mode == 1) return 1;
  if (plain && ep.ug_mode == 0) return 2;
  if (ep.gamma_mode == 2 && ep.ug_mode != 2) return 3;
  return plain ? 4 : 0;
}

// The planes of logit z scaled by sc (ug_sc: the scaled weight floor) and the
// unweighted terms of the unmatched-mask penalty.  With t = -|z| log2 e, e = 2^t, d = 1 + e:
// the entropy -(p ln p + q ln q) / ln 2 is log2 d + (e / d) |t| (both terms
// non-negative) and softplus(+-z) = ln 2 log2 d + max(+-z, 0), so the default
// form takes 3 transcendental and 15 other ops per logit.
template <int EM>
__device__ __forceinline__ void planes_of(float z, const ElemParams& ep, float sc, float ug_sc, float& neg,
                                          float& pos, float& wp, float& w, float& negu, float& pu) {
  if constexpr (EM == 0) {
    const Sig s = sig_terms(z);
    float mn, mp;
    focal_mods(s, ep, mn, mp);
    w = unc_weight(s, ep) * sc;
    negu = ep.an * mn * s.cn;
    pu = s.p;
    pos = w * (ep.ap * mp * s.cp);
  } else {
    const float t = -fabsf(z) * kLog2e;
    const float e = __builtin_amdgcn_exp2f(t);
    const float d = 1.f + e;
    const float r = __builtin_amdgcn_rcpf(d);
    const float l2 = __builtin_amdgcn_logf(d);  // log2
    const float er = e * r;
    const bool up = z >= 0.f;
    const float p = up ? r : er;
    float cn = __builtin_fmaf(l2, kLn2, fmaxf(z, 0.f)), cp = __builtin_fmaf(l2, kLn2, fmaxf(-z, 0.f));
    if constexpr (EM == 3) {
      const float q = up ? er : r;
      cn *= ep.an * (p * p);
      cp *= ep.ap * (q * q);
    }
    if (EM == 1 || EM == 4 || (EM == 3 && ep.ug_mode == 1)) {
      // (|z| beyond 2^127 / 1.44: 0 x inf here, and a NaN leaves the floor)
      float h = __builtin_fmaf(-er, t, l2);
      if constexpr (EM == 4) h = __builtin_amdgcn_exp2f(ep.ug * __builtin_amdgcn_logf(h));
      w = __builtin_amdgcn_fmed3f(h * sc, ug_sc, sc);
    } else {
      w = sc;
    }
    negu = cn;
    pu = p;
    pos = w * cp;
  }
  neg = w * negu;
  wp = w * pu;
}

// Operand types of the matrix instructions: float16, or bf16 (WIDE).
template <bool WIDE>
struct Ops {
  using v8 = f16x8_t;
  static __device__ __forceinline__ uint32_t pack(float a, float b) { return pack_f16x2(a, b); }
  static __device__ __forceinline__ f32x4_t mma16(v8 a, v8 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16_t mma32(v8 a, v8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Ops<true> {
  using v8 = bf16x8_t;
  static __device__ __forceinline__ uint32_t pack(float a, float b) { return pack_bf16x2(a, b); }
  static __device__ __forceinline__ f32x4_t mma16(v8 a, v8 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16_t mma32(v8 a, v8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

// Build the LUT in LDS (all threads of the workgroup): float16 planes scaled by
// 2^lg, or bf16 planes (WIDE).  The overflow slot holds NaN so that a wave whose
// sums come out NaN knows it met |z| >= 64, inf or nan (every other entry is finite).
template <bool WIDE>
__device__ void build_lut(unsigned char* lut, const ElemParams& ep, int lg) {
  const float sc = WIDE ? 1.f : __builtin_ldexpf(1.f, lg);
  for (uint32_t e = threadIdx.x; e < 2 * kLutBlock; e += blockDim.x) {
    const uint32_t sgn = e >= kLutBlock ? 1u : 0u;
    const uint32_t j = e - sgn * kLutBlock;
    uint2 v;
    if (j <= kLutN) {
      const uint32_t mag = j == 0 ? 0u : kLutSub + j;  // j == 0: |z| < 2^-9 -> z = 0
      const float z = __uint_as_float(((sgn << 15) | mag) << 16);
      float neg, pos, wp, w, nu, pu;
      planes_of<0>(z, ep, sc, 0.f, neg, pos, wp, w, nu, pu);
      v.x = Ops<WIDE>::pack(neg, pos);
      v.y = Ops<WIDE>::pack(wp, w);
    } else {
      v.x = WIDE ? 0x7FC07FC0u : 0x7E007E00u;  // NaN marker
      v.y = v.x;
    }
    *(uint2*)(lut + sgn * kLutNegOff + j * 8) = v;
  }
}

// 8 consecutive logits of one row as raw words.
template <int DT>
struct Raw8 {
  uint4 w[DT == ML_F32 ? 2 : 1];
};

// Rows of odd sizes start on element boundaries only: 16-byte loads all the
// same (global memory takes them at any alignment).
template <int DT>
__device__ __forceinline__ void load_raw8(const void* base, int64_t i, Raw8<DT>& r) {
  if constexpr (DT == ML_F32) __builtin_memcpy(&r, (const float*)base + i, 32);
  else __builtin_memcpy(&r, (const uint16_t*)base + i, 16);
}
// The first nvalid (any int64: <= 0 none, >= 8 all) of the 8 logits, the rest zero.
template <int DT>
__device__ __forceinline__ void load_raw8_part(const void* base, int64_t i, int64_t nvalid, Raw8<DT>& r) {
  if constexpr (DT == ML_F32) {
    uint32_t u[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k] = k < nvalid ? __float_as_uint(((const float*)base)[i + k]) : 0u;
    r.w[0] = make_uint4(u[0], u[1], u[2], u[3]);
    r.w[1] = make_uint4(u[4], u[5], u[6], u[7]);
  } else {
    uint32_t u[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k < nvalid) u[k >> 1] |= (uint32_t)((const uint16_t*)base)[i + k] << ((k & 1) * 16);
    r.w[0] = make_uint4(u[0], u[1], u[2], u[3]);
  }
}

template <int DT>
__device__ __forceinline__ void raw_to_f32(const Raw8<DT>& r, float z[8]) {
  if constexpr (DT == ML_F32) {
    const uint32_t u[8] = {r.w[0].x, r.w[0].y, r.w[0].z, r.w[0].w,
                           r.w[1].x, r.w[1].y, r.w[1].z, r.w[1].w};
#pragma unroll
    for (int k = 0; k < 8; ++k) z[k] = __uint_as_float(u[k]);
  } else {
    const uint32_t u[4] = {r.w[0].x, r.w[0].y, r.w[0].z, r.w[0].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (DT == ML_BF16) {
        z[2 * k] = bf16_lo(u[k]);
        z[2 * k + 1] = bf16_hi(u[k]);
      } else {
        z[2 * k] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u[k] & 0xFFFF));
        z[2 * k + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u[k] >> 16));
      }
    }
  }
}

// 8 float32 values as NT float16 terms (1 or 2) whose sum reproduces them.
template <int NT>
__device__ __forceinline__ void split_f16(const float v[8], f16x8_t out[NT]) {
  u32x4_t hi;
#pragma unroll
  for (int k = 0; k < 4; ++k) hi[k] = pack_f16x2(v[2 * k], v[2 * k + 1]);
  out[0] = __builtin_bit_cast(f16x8_t, hi);
  if constexpr (NT == 2) {
    u32x4_t lo;
#pragma unroll
    for (int k = 0; k < 4; ++k) lo[k] = pack_f16x2(rem_lo(v[2 * k], hi[k]), rem_hi(v[2 * k + 1], hi[k]));
    out[1] = __builtin_bit_cast(f16x8_t, lo);
  }
}
// ... and as NS bf16 terms.
template <int NS>
__device__ __forceinline__ void split_bf16(const float v[8], bf16x8_t out[NS]) {
  float rem[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) rem[k] = v[k];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    u32x4_t w;
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = pack_bf16x2(rem[2 * k], rem[2 * k + 1]);
    out[s] = __builtin_bit_cast(bf16x8_t, w);
    if (s + 1 < NS) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        rem[2 * k] -= bf16_lo(w[k]);
        rem[2 * k + 1] -= bf16_hi(w[k]);
      }
    }
  }
}

// The planes of one row's 8 cells, scaled by sc; with MASK, cells >= nvalid are
// zero.  ub, up: sums of the unweighted terms (unw).
template <bool MASK>
__device__ __forceinline__ void planes8(const float (&z)[8], const ElemParams& ep, float sc,
                                        int64_t nvalid, bool unw, float (&v)[4][8], float& ub, float& up) {
  const float ug_sc = ep.ug_min * sc;
  auto cells = [&](auto em) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      float neg, pos, wp, w, nu, pu;
      planes_of<decltype(em)::value>(z[k], ep, sc, ug_sc, neg, pos, wp, w, nu, pu);
      const bool ok = !MASK || k < nvalid;
      v[0][k] = ok ? neg : 0.f;
      v[1][k] = ok ? pos : 0.f;
      v[2][k] = ok ? wp : 0.f;
      v[3][k] = ok ? w : 0.f;
      if (unw) {
        ub += ok ? nu : 0.f;
        up += ok ? pu : 0.f;
      }
    }
  };
  switch (elem_mode(ep)) {
    case 1: cells(std::integral_constant<int, 1>()); break;
    case 2: cells(std::integral_constant<int, 2>()); break;
    case 3: cells(std::integral_constant<int, 3>()); break;
    case 4: cells(std::integral_constant<int, 4>()); break;
    default: cells(std::integral_constant<int, 0>()); break;
  }
}
// max(|a|, |b|, |c|), NaNs aside (written out: the compiler would quiet each operand first)
__device__ __forceinline__ float max_abs3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float max_abs8(const float (&z)[8], float m) {
#pragma unroll
  for (int k = 0; k < 8; k += 2) m = max_abs3(z[k], z[k + 1], m);
  return m;
}

// Table byte offsets (sign block included) of the two bf16 logits packed in
// u, in compiler-visible packed 16-bit ops (no inline assembly, so no hazard
// padding after each one): the clamped index times 8 stays below 2^15, so the
// sign bit ORs in without carry.
__device__ __forceinline__ uint32_t lut_addr_pair(uint32_t u) {
  const u16x2_t m = as_u16x2(u & 0x7FFF7FFFu);
  const u16x2_t idx = __builtin_elementwise_min(
      __builtin_elementwise_sub_sat(m, (u16x2_t){(unsigned short)kLutSub, (unsigned short)kLutSub}),
      (u16x2_t){(unsigned short)(kLutN + 1), (unsigned short)(kLutN + 1)});
  uint32_t addr = (u & 0x80008000u) | as_u32(idx << (u16x2_t){3, 3});
  // kept whole, so its two halves are one mask and one shift of it
  asm("" : "+v"(addr));
  return addr;
}

// Any of 8 bf16 logits beyond the table (|z| >= 64, inf, nan).
__device__ __forceinline__ bool lut_over8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const u16x2_t m = __builtin_elementwise_max(
      __builtin_elementwise_max(as_u16x2(a & 0x7FFF7FFFu), as_u16x2(b & 0x7FFF7FFFu)),
      __builtin_elementwise_max(as_u16x2(c & 0x7FFF7FFFu), as_u16x2(d & 0x7FFF7FFFu)));
  return m[0] >= kLutOver || m[1] >= kLutOver;
}

// Table entries of one row's 8 bf16 cells (LDS reads only; see lut_planes).
__device__ __forceinline__ void lut_lookup8(const uint4& x, const unsigned char* lut, uint2 E[8]) {
  const uint32_t u[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t addr = lut_addr_pair(u[i]);
    E[2 * i] = *(const uint2*)(lut + (addr & 0xFFFFu));
    E[2 * i + 1] = *(const uint2*)(lut + (addr >> 16));
  }
}

// The four A planes from the entries of 8 cells: (neg, pos) and (wp, w) of
// each cell regrouped into per-plane pairs of consecutive cells.
template <class V>
__device__ __forceinline__ void lut_planes(const uint2 E[8], V A[4]) {
  u32x4_t a[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint2 e0 = E[2 * i], e1 = E[2 * i + 1];
    a[0][i] = __builtin_amdgcn_perm(e1.x, e0.x, 0x05040100u);
    a[1][i] = __builtin_amdgcn_perm(e1.x, e0.x, 0x07060302u);
    a[2][i] = __builtin_amdgcn_perm(e1.y, e0.y, 0x05040100u);
    a[3][i] = __builtin_amdgcn_perm(e1.y, e0.y, 0x07060302u);
  }
#pragma unroll
  for (int pl = 0; pl < 4; ++pl) A[pl] = __builtin_bit_cast(V, a[pl]);
}

// ---- right operands ---------------------------------------------------------
// Counts of 8 cells: kHot where a label code equals the column's (a zero mask
// makes it the ones column), 0 elsewhere.
__device__ __forceinline__ u32x4_t hot8(const uint32_t (&L2)[4], uint32_t col, uint32_t mask = 0xFFFFFFFFu) {
  u32x4_t b;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    // (L ^ col) & mask in one three-input boolean op
    b[i] = as_u32(__builtin_elementwise_sub_sat((u16x2_t){kHot, kHot},
                                                as_u16x2(__builtin_amdgcn_bitop3_b32(L2[i], col, mask, 0x28))));
  return b;
}
// pair - n for 8 16-bit integers.
__device__ __forceinline__ u32x4_t isub8(uint32_t pair, const u32x4_t& n) {
  u32x4_t b;
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = as_u32(as_u16x2(pair) - as_u16x2(n[i]));
  return b;
}
// 8 integers times a constant.
__device__ __forceinline__ u32x4_t imul8(const u32x4_t& n, unsigned short c) {
  u32x4_t b;
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = as_u32(as_u16x2(n[i]) * (u16x2_t){c, c});
  return b;
}
// 8 u8 counts as 16-bit words with a byte of hi4 above each.
__device__ __forceinline__ u32x4_t widen8(uint32_t hi4, uint32_t x, uint32_t y) {
  constexpr uint32_t s0 = 0x04010400u, s1 = 0x04030402u;
  return u32x4_t{__builtin_amdgcn_perm(hi4, x, s0), __builtin_amdgcn_perm(hi4, x, s1),
                 __builtin_amdgcn_perm(hi4, y, s0), __builtin_amdgcn_perm(hi4, y, s1)};
}
// c + t and c - t for 8 float16 values, two per op (exact here: both are multiples
// of the same last place below 2^11 of them); c: the value twice.
template <bool NEG>
__device__ __forceinline__ u32x4_t hadd8(uint32_t c, const u32x4_t& t) {
  u32x4_t b;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (NEG) asm("v_pk_add_f16 %0, %1, %2 neg_lo:[0,1] neg_hi:[0,1]" : "=v"(b[i]) : "s"(c), "v"(t[i]));
    else asm("v_pk_add_f16 %0, %1, %2" : "=v"(b[i]) : "s"(c), "v"(t[i]));
  }
  return b;
}
// Operands n and N2 - n of one column tile.
struct Opnd {
  u32x4_t n, rest;
};
// float16 counts times 2^-lg (lg <= 14, N2 < 1024): wave-uniform constants.
struct RightF16 {
  uint32_t mul, one2;       // label compare: the factor of kHot, and the result twice
  uint32_t hi4, base, top;  // u8: bytes above a count, minus their value, their value + 2^-lg N2 (pairs)
  float inv;                // 2^-lg
};
__device__ __forceinline__ RightF16 right_f16(int lg, float N2) {
  const uint32_t one = (uint32_t)(15 - lg) << 10, e = (uint32_t)(25 - lg) << 10;
  return RightF16{one / kHot, one * 0x10001u, (e >> 8) * 0x01010101u, (e | 0x8000u) * 0x10001u,
                  (e + (uint32_t)N2) * 0x10001u, __builtin_ldexpf(1.f, -lg)};
}
template <bool REST>
__device__ __forceinline__ Opnd opnd_u8(uint32_t x, uint32_t y, const RightF16& c) {
  const u32x4_t t = widen8(c.hi4, x, y);
  Opnd o;
  o.n = hadd8<false>(c.base, t);
  if (REST) o.rest = hadd8<true>(c.top, t);
  return o;
}
// Label compare: `mul` times kHot is the value of a hit, one2 that value twice.
template <bool REST>
__device__ __forceinline__ Opnd opnd_hot(const u32x4_t& hot, uint32_t mul, uint32_t one2) {
  Opnd o;
  o.n = mul == 1u ? hot : imul8(hot, (unsigned short)mul);
  if (REST) o.rest = isub8(one2, o.n);
  return o;
}
// ... as the table kernels take it: 2^-16, or a bf16 0.5 (WIDE).
template <bool WIDE>
__device__ __forceinline__ Opnd opnd_tab(const u32x4_t& hot) {
  return WIDE ? opnd_hot<true>(hot, 0x3Fu, 0x3F003F00u) : opnd_hot<true>(hot, 1u, kHot * 0x10001u);
}
// Bits 0..10 (HIGH = 0) or 11..15 of 8 16-bit integers as float16, times inv.
template <bool HIGH>
__device__ __forceinline__ u32x4_t part8(const u32x4_t& w, float inv) {
  constexpr uint32_t m = HIGH ? 0xF800u : 0x07FFu;
  u32x4_t b;
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = pack_f16x2((float)(w[i] & m) * inv, (float)((w[i] >> 16) & m) * inv);
  return b;
}
// bf16 operands: a label hit as 1.0; a u8 count; and one byte of 16-bit integers,
// exact in 8 bits.
__device__ __forceinline__ u32x4_t wide_hot8(const u32x4_t& hot) {
  u32x4_t b = imul8(hot, 0x7Fu);
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = as_u32(as_u16x2(b[i]) >> (u16x2_t){1, 1});
  return b;
}
__device__ __forceinline__ Opnd wide_u8(uint32_t x, uint32_t y, float N2) {
  Opnd o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = i < 2 ? x : y;
    const float a = (float)((w >> (16 * (i & 1))) & 0xFFu), b = (float)((w >> (16 * (i & 1) + 8)) & 0xFFu);
    o.n[i] = pack_bf16x2(a, b);
    o.rest[i] = pack_bf16x2(N2 - a, N2 - b);
  }
  return o;
}
template <bool HIGH>
__device__ __forceinline__ u32x4_t wide_byte8(const u32x4_t& w) {
  constexpr uint32_t m = HIGH ? 0xFF00u : 0xFFu;
  u32x4_t b;
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = pack_bf16x2((float)(w[i] & m), (float)((w[i] >> 16) & m));
  return b;
}

// Pacing of the waves of one workgroup that share a CU: the SIMD arbiter
// issues the oldest ready wave first, so with equal work the younger waves
// fall behind and the CU ends the launch at part occupancy.  Every few
// K-steps a wave posts its progress in LDS and drops its issue priority while
// it is ahead of the slowest wave of the workgroup (progress values are
// approximate: no barrier, a stale read only delays the switch).
constexpr int kPaceSlack = 8;  // K-steps ahead of the slowest wave before yielding
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
// The workgroup has at most 16 waves, so lanes 0..15 (one DPP row) hold every
// wave's progress and four DPP swaps within the row give their minimum, with
// no LDS traffic.
__device__ __forceinline__ void pace(int* prog, int k) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  if (lane == 0) prog[wave] = k;
  int v = lane < nw ? prog[lane] : 0x7FFFFFFF;
  v = min(v, dpp_i<0xB1>(v));   // quad_perm [1,0,3,2]
  v = min(v, dpp_i<0x4E>(v));   // quad_perm [2,3,0,1]
  v = min(v, dpp_i<0x141>(v));  // row_half_mirror
  v = min(v, dpp_i<0x140>(v));  // row_mirror
  if (__builtin_amdgcn_readfirstlane(v) + kPaceSlack < k) __builtin_amdgcn_s_setprio(0);
  else __builtin_amdgcn_s_setprio(1);
}

// In-workgroup sum of R consecutive K-splits of one task (R a power of two):
// this wave is split r of its group grp of R waves.  buf: the workgroup's LDS
// exchange area for its writers, 2*NT float4 per lane each (two planes at a
// time); rsbuf: their row sums.  buf == null: no reduction.
struct SplitRed {
  f32x4_t* buf = nullptr;
  float2* rsbuf = nullptr;
  int R = 1, r = 0, grp = 0;
};
constexpr int kRedBarriers = 4;  // per level of the tree

// One wave's work: 16 query rows of task (lb, rtile) over the K-steps of
// split ks of KS; writes the partial sums to `out` ([NP][16][16*NT]) and,
// for unweighted penalties, the row sums to `rs` ([16][2]).  TAB:
// per-cell planes from the LDS table (bf16 only; WIDE: a table of bf16, label
// maps only).  If a table wave's sums come out non-finite (the marker), it redoes
// the range with the formulas and bf16 operands before writing.  `setup` (the
// workgroup's table build and barrier) is called exactly once on every path,
// after the first D K-steps of loads are issued, so their latency overlaps it.
// With red.buf, the R waves of the group add their sums in a fixed tree order
// (wave r takes wave r + h for h = R/2, ..., 1; kRedBarriers log2(R) barriers for
// every wave of the workgroup) and only wave 0 of the group writes.
// CNT: 0 label map, 1 u8 counts, 2 u16 counts.  In the wide classes (NT >= 7) a
// K-step's MFMAs run only for the column tiles its 32 cells touch (a coherent
// label map touches few of them).
template <int DT, int NT, int CNT, bool TAB, bool WIDE, class Setup>
__device__ __forceinline__ void cost_wave(const CostArgs& a, int64_t lb, int64_t rtile, int64_t ks, int64_t KS,
                                          const unsigned char* lut, float* out, float* rs_out, int* prog,
                                          Setup&& setup, const SplitRed& red = SplitRed(),
                                          uint32_t* klut = nullptr) {
  constexpr int NS = TAB ? 1 : InTraits<DT>::kTerms, NW = InTraits<DT>::kWide;
  using V = typename Ops<TAB && WIDE>::v8;  // the table's or the float16 operands
  // label maps in the wide classes: the label -> (slot | tile bit << 16) table
  // klut (this wave's, in LDS) gives each K-step's slots and touched tiles
  constexpr bool KEYS = CNT == 0 && NT >= 7;
  constexpr bool SUMS = NT >= 7;  // slot sums
  constexpr int NP = class_planes(SUMS ? 1 : 0);
  constexpr int D = TAB ? kDepth : 2;  // K-steps of logits and labels in flight
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g4 = lane >> 4;
  const ElemParams ep = a.ep;
  const bool unw = !TAB && rs_out != nullptr;
  const int64_t b = lb % a.B;
  const int G = __builtin_amdgcn_readfirstlane(a.ncols[b]);
  const int nt_used = (G + 1 + 15) >> 4;
  const int64_t q0 = rtile * 16;

  // Per tile: the lane's column code pair and compare mask (slot G: the ones
  // column; padding compares with label 0, its sums are never used), or its row
  // of the count tiles (slot G: the ones column or the pixels of no column;
  // padding reads that row too).
  uint32_t colL[KEYS ? 1 : NT], colM[KEYS ? 1 : NT];
  const uint8_t* cbase = nullptr;
  uint32_t crow[CNT ? NT : 1];
  const int64_t cstep = (int64_t)a.counts.rows * kCountCells * (CNT == 2 ? 2 : 1);  // bytes per block
  if constexpr (!KEYS) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int slot = nt * 16 + r;
      int act = -1;
      if (slot < G) {
        const int c = a.colmap[b * a.nslot + slot];
        act = c + (c >= a.bg ? 1 : 0);
      }
      if constexpr (CNT == 0) {
        colL[nt] = act >= 0 ? label_code(act) * 0x10001u : 0u;
        colM[nt] = slot == G ? 0u : 0xFFFFFFFFu;
        asm("" : "+v"(colM[nt]));  // a register, not a select at every use
      } else {
        const int rest = (int)a.GT_total + (SUMS ? 0 : 1);
        crow[nt] = ((uint32_t)(act >= 0 ? act : rest) * kCountCells + 8u * g4) * CNT;
      }
    }
    if constexpr (CNT != 0) cbase = a.counts.p + b * a.counts.nb * cstep;
  } else {
    // label (the code's high byte) -> key: every entry G first, then each
    // column's label its slot (one
    // wave's LDS writes land in issue order; the wait keeps the two rounds
    // apart all the same)
    const uint32_t eG = (uint32_t)G | (1u << (16 + (G >> 4)));
    for (int l = lane; l < 256; l += 64) klut[l] = eG;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (int sl = lane; sl < G; sl += 64) {
      const int c = a.colmap[b * a.nslot + sl];
      const int act = c + (c >= a.bg ? 1 : 0);
      klut[act & 255] = (uint32_t)sl | (1u << (16 + (sl >> 4)));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  f32x4_t acc[NP][NT];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[i][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  float ub = 0.f, up = 0.f;

  // this wave's K-steps: [s0, s1) of the full steps, plus the tail step
  const int64_t full = a.HW / kStep;
  const int64_t per = ceil_div(full, KS);
  const int64_t s0 = min(full, ks * per);
  const int64_t s1 = min(full, s0 + per);
  const bool has_tail = (a.HW % kStep) != 0 && ks == KS - 1;
  const int64_t rowoff = (lb * a.Q + min(q0 + r, a.Q - 1)) * a.HW + g4 * 8;  // rows >= Q: unused outputs
  const uint16_t* labp = a.lab16 + (CNT ? 0 : b * a.HWp + g4 * 8);

  // raw right operands of K-step st: labels, or the lane's 8 counts per tile
  struct BRaw {
    uint4 lab;
    uint32_t w[CNT ? NT : 1][CNT == 2 ? 4 : 2];
  };
  auto fetch_b = [&](BRaw& x, int64_t st) {
    if constexpr (CNT == 0) {
      x.lab = *(const uint4*)(labp + st * kStep);
    } else {
      const uint8_t* p = cbase + (st >> 1) * cstep + (st & 1) * (kStep * CNT);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if (nt >= nt_used) continue;
        if constexpr (CNT == 1) *(uint2*)x.w[nt] = *(const uint2*)(p + crow[nt]);
        else *(uint4*)x.w[nt] = *(const uint4*)(p + crow[nt]);
      }
    }
  };
  // slots of the lane's 8 cells as u16 pairs (like label codes), and the column tiles any of the
  // K-step's 32 cells falls in (the four lane groups hold different cells;
  // every lane ends with the same mask)
  auto keys_of = [&](const uint4& lv, uint32_t (&kp)[4]) -> uint32_t {
    const uint32_t L2[4] = {lv.x, lv.y, lv.z, lv.w};
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      e[2 * i] = klut[(L2[i] >> 8) & 0xFFu];
      e[2 * i + 1] = klut[L2[i] >> 24];
    }
    uint32_t t = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kp[i] = __builtin_amdgcn_perm(e[2 * i + 1], e[2 * i], 0x040C000Cu);  // slots in the high bytes
      t |= e[2 * i] | e[2 * i + 1];
    }
    t >>= 16;
    return __builtin_amdgcn_readlane(t, 0) | __builtin_amdgcn_readlane(t, 16) |
           __builtin_amdgcn_readlane(t, 32) | __builtin_amdgcn_readlane(t, 48);
  };
  // f(nt, raw 16-bit integers of tile nt: compare results or counts) for the
  // tiles the K-step touches; u8 counts stay packed in the first two words
  auto for_tiles = [&](const BRaw& x, const uint32_t (&kp)[4], uint32_t tmask, auto&& f) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt >= nt_used) continue;
      if constexpr (KEYS) {
        if (!((tmask >> nt) & 1u)) continue;
        f(nt, hot8(kp, (uint32_t)(nt * 16 + r) * 0x01000100u));
      } else if constexpr (CNT == 0) {
        const uint32_t L2[4] = {x.lab.x, x.lab.y, x.lab.z, x.lab.w};
        f(nt, hot8(L2, colL[nt], colM[nt]));
      } else {
        uint32_t any = 0u;
#pragma unroll
        for (int i = 0; i < 2 * CNT; ++i) any |= x.w[nt][i];
        if (SUMS && __ballot(any != 0u) == 0ull) continue;
        if constexpr (CNT == 1) f(nt, u32x4_t{x.w[nt][0], x.w[nt][1], 0u, 0u});
        else f(nt, u32x4_t{x.w[nt][0], x.w[nt][1], x.w[nt][2], x.w[nt][3]});
      }
    }
  };
  const uint32_t n2pair = (uint32_t)a.N2 * 0x10001u;
  // table sums carry the planes' scale, the others none
  const RightF16 rf = right_f16(TAB ? 0 : a.form.lg, a.N2);
  auto mul_tile = [&](auto ops, int nt, const auto& A, const Opnd& o) {
    using O = decltype(ops);
    constexpr int T = sizeof(A[0]) / sizeof(A[0][0]);
    auto mul = [&](int i, int pl, const u32x4_t& v) {
#pragma unroll
      for (int sp = 0; sp < T; ++sp)
        acc[i][nt] = O::mma16(A[pl][sp], __builtin_bit_cast(typename O::v8, v), acc[i][nt]);
    };
    if constexpr (SUMS) {
#pragma unroll
      for (int pl = 0; pl < 4; ++pl) mul(pl, pl, o.n);
    } else {
      mul(0, 0, o.rest);
      mul(1, 2, o.n);
      mul(2, 3, o.n);
      mul(0, 1, o.n);
    }
  };
  auto mma_step = [&](const V (&A)[4][NS], const BRaw& x, const uint32_t (&kp)[4], uint32_t tmask) {
    for_tiles(x, kp, tmask, [&](int nt, const u32x4_t& raw) {
      auto mul = [&](const Opnd& o) { mul_tile(Ops<TAB && WIDE>(), nt, A, o); };
      if constexpr (CNT == 0 && TAB) {
        mul(opnd_tab<WIDE>(raw));
      } else if constexpr (CNT == 0) {
        mul(opnd_hot<!SUMS>(raw, rf.mul, rf.one2));
      } else if constexpr (CNT == 1) {
        mul(opnd_u8<!SUMS>(raw[0], raw[1], rf));
      } else {  // integers up to 65025 as two exact float16 parts
        const u32x4_t rest = isub8(n2pair, raw);
        mul(Opnd{part8<false>(raw, rf.inv), part8<false>(rest, rf.inv)});
        mul(Opnd{part8<true>(raw, rf.inv), part8<true>(rest, rf.inv)});
      }
    });
  };
  // the same with bf16 operands from unscaled planes
  auto mma_wide = [&](const float (&v)[4][8], const BRaw& x, const uint32_t (&kp)[4], uint32_t tmask) {
    bf16x8_t A[4][NW];
#pragma unroll
    for (int pl = 0; pl < 4; ++pl) split_bf16<NW>(v[pl], A[pl]);
    for_tiles(x, kp, tmask, [&](int nt, const u32x4_t& raw) {
      auto mul = [&](const Opnd& o) { mul_tile(Ops<true>(), nt, A, o); };
      if constexpr (CNT == 0) {
        const u32x4_t n = wide_hot8(raw);
        mul(Opnd{n, isub8(0x3F803F80u, n)});
      } else if constexpr (CNT == 1) {
        mul(wide_u8(raw[0], raw[1], a.N2));
      } else {
        const u32x4_t rest = isub8(n2pair, raw);
        mul(Opnd{wide_byte8<false>(raw), wide_byte8<false>(rest)});
        mul(Opnd{wide_byte8<true>(raw), wide_byte8<true>(rest)});
      }
    });
  };
  // Software pipeline over this wave's nst steps: D steps of logits (and
  // labels) in flight, the count operands one step ahead.  Slot j holds step
  // k + j; it is turned into A operands first and then refilled with step
  // k + j + D (clamped to the last step, so the loads are unconditional).
  // Every branch here is wave-uniform.
  // step counters in 32 bits: their compares stay scalar (a wave has at most
  // HW / 32 < 2^31 steps)
  const int nst = (int)(s1 - s0);
  // steps summed; the bf16 loop below takes the rest.  A range that opens with
  // logits these operands do not take (a filled region) goes there whole, at once.
  int done = nst;
  float most = 0.f;  // of |z|, by formula
  if (nst > 0) {
    constexpr int DB = CNT ? 2 : D;  // right operands in flight
    Raw8<DT> buf[D];
    BRaw bb[DB];
    auto at = [&](int k) { return s0 + (k < nst ? k : nst - 1); };
#pragma unroll
    for (int j = 0; j < D; ++j) {
      load_raw8<DT>(a.logits, rowoff + at(j) * kStep, buf[j]);
      if (CNT == 0) fetch_b(bb[j % DB], at(j));
    }
    if constexpr (CNT != 0) fetch_b(bb[0], at(0));
    setup();
    int k = 0, nmain = nst;
    if constexpr (TAB) {
      const uint4 w = buf[0].w[0];
      if (__ballot(lut_over8(w.x, w.y, w.z, w.w)) != 0ull) nmain = done = 0;
      // software-pipelined one step deep: the table reads of step k + 1 are
      // issued before the right operands and MFMAs of step k, so their
      // latency hides behind that work
      uint2 E[8];
      lut_lookup8(buf[0].w[0], lut, E);
      auto step = [&](int j, int kj, bool refill) {
        V A[4][1];
        lut_planes(E, &A[0][0]);
        uint32_t kp[4] = {0u, 0u, 0u, 0u}, tm = 0;
        if constexpr (KEYS) tm = keys_of(bb[j % DB].lab, kp);
        lut_lookup8(buf[(j + 1) % D].w[0], lut, E);
        __builtin_amdgcn_sched_barrier(0);
        if (refill) load_raw8<DT>(a.logits, rowoff + at(kj + D) * kStep, buf[j]);
        if constexpr (CNT != 0) fetch_b(bb[(j + 1) % DB], at(kj + 1));
        mma_step(A, bb[j % DB], kp, tm);
        __builtin_amdgcn_sched_barrier(0);
        if (CNT == 0 && refill) fetch_b(bb[j % DB], at(kj + D));
      };
      for (; k + D <= nmain; k += D) {
        if (prog && (k & (2 * D - 1)) == 0) pace(prog, k);
#pragma unroll
        for (int j = 0; j < D; ++j) step(j, k + j, true);
      }
#pragma unroll
      for (int j = 0; j < D - 1; ++j)  // the last nst % D steps
        if (k + j < nmain) step(j, k + j, false);
    } else {
      const float sc = WIDE ? 1.f : __builtin_ldexpf(1.f, a.form.lg);
      if constexpr (!WIDE) {
        float z[8];
        raw_to_f32<DT>(buf[0], z);
        if (__ballot(max_abs8(z, 0.f) > kNarrowMax) != 0ull) nmain = done = 0;
      }
      auto step = [&](int j, int kj, bool refill) {
        // the key table reads go out before the plane work
        uint32_t kp[4] = {0u, 0u, 0u, 0u}, tm = 0;
        if constexpr (KEYS) tm = keys_of(bb[j % DB].lab, kp);
        if constexpr (CNT != 0) fetch_b(bb[(j + 1) % DB], at(kj + 1));
        float z[8], v[4][8];
        raw_to_f32<DT>(buf[j], z);
        if constexpr (!WIDE) most = max_abs8(z, most);
        planes8<false>(z, ep, sc, 8, unw, v, ub, up);
        // keep each refill below the last read of its slot, so that it reuses
        // the slot's registers instead of rotating the whole pipeline
        __builtin_amdgcn_sched_barrier(0);
        if (refill) load_raw8<DT>(a.logits, rowoff + at(kj + D) * kStep, buf[j]);
        if constexpr (WIDE) {
          mma_wide(v, bb[j % DB], kp, tm);
        } else {
          V A[4][NS];
#pragma unroll
          for (int pl = 0; pl < 4; ++pl) split_f16<NS>(v[pl], A[pl]);
          mma_step(A, bb[j % DB], kp, tm);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (CNT == 0 && refill) fetch_b(bb[j % DB], at(kj + D));
      };
      for (; k + D <= nmain; k += D) {
        if (prog && (k & (2 * D - 1)) == 0) pace(prog, k);
#pragma unroll
        for (int j = 0; j < D; ++j) step(j, k + j, true);
      }
#pragma unroll
      for (int j = 0; j < D - 1; ++j)  // the last nst % D steps
        if (k + j < nmain) step(j, k + j, false);
    }
  } else {
    setup();
  }

  if constexpr (TAB) {
    // the marker shows in the sums of A_neg and A_pos
    bool bad = false;
#pragma unroll
    for (int i = 0; i < (SUMS ? 2 : 1); ++i)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= !(fabsf(acc[i][nt][e]) < INFINITY);
    const float undo = WIDE ? 2.f : __builtin_ldexpf(1.f, (CNT == 0 ? 16 : 0) - a.form.lg);
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[i][nt] *= undo;
    if (__builtin_expect(__ballot(bad) != 0ull, 0)) {
      clear();
      done = 0;
    }
  } else if constexpr (!WIDE) {
    if (__builtin_expect(__ballot(most > kNarrowMax) != 0ull, 0)) {
      clear();
      ub = up = 0.f;
      done = 0;
    }
  }

  // Steps by the formulas with bf16 operands, the next one's loads in flight: the
  // last partial step, or a whole range (redone).
  // (Marked unlikely, so that it takes no registers from the loops above.)
  const int nall = nst + (has_tail ? 1 : 0);
  if (__builtin_expect(done < nall, 0)) {
    const int64_t tailn = a.HW - (full * kStep + g4 * 8);  // valid cells of the partial step
    Raw8<DT> raw, nraw;
    BRaw x, nx;
    auto fetch = [&](int k) {
      const int64_t st = k < nst ? s0 + k : full;
      if (k < nst) load_raw8<DT>(a.logits, rowoff + st * kStep, nraw);
      else load_raw8_part<DT>(a.logits, rowoff + st * kStep, tailn, nraw);
      fetch_b(nx, st);
    };
    fetch(done);
    for (int k = done; k < nall; ++k) {
      raw = nraw;
      x = nx;
      if (k + 1 < nall) fetch(k + 1);
      uint32_t kp[4] = {0u, 0u, 0u, 0u}, tm = 0;
      if constexpr (KEYS) tm = keys_of(x.lab, kp);
      float z[8], v[4][8];
      raw_to_f32<DT>(raw, z);
      if ((TAB || !WIDE) && k < nst) planes8<false>(z, ep, 1.f, 8, unw, v, ub, up);
      else planes8<true>(z, ep, 1.f, k < nst ? 8 : tailn, unw, v, ub, up);
      mma_wide(v, x, kp, tm);
    }
  }

  if constexpr (SUMS) if (red.buf) {
    constexpr int TW = 2 * NT;  // float4 per lane per writer
    for (int h = red.R >> 1; h >= 1; h >>= 1) {
      const int64_t slot = red.grp * (red.R >> 1) + (red.r & (h - 1));
      f32x4_t* d = red.buf + slot * TW * 64 + lane;
#pragma unroll
      for (int ph = 0; ph < 2; ++ph) {
        if (red.r >= h && red.r < 2 * h) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
              if (nt < nt_used) d[(i * NT + nt) * 64] = acc[2 * ph + i][nt];
          if (unw && ph == 0) red.rsbuf[slot * 64 + lane] = make_float2(ub, up);
        }
        __syncthreads();
        if (red.r < h) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
              if (nt < nt_used) acc[2 * ph + i][nt] += d[(i * NT + nt) * 64];
          if (unw && ph == 0) {
            const float2 v = red.rsbuf[slot * 64 + lane];
            ub += v.x;
            up += v.y;
          }
        }
        __syncthreads();
      }
    }
    if (red.r != 0) return;
  }

  // ---- write this wave's partial sums (only the tiles in use)
  constexpr int nslot = 16 * NT;
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt >= nt_used) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(i * 16 + g4 * 4 + e) * nslot + nt * 16 + r] = acc[i][nt][e];
    }
  if (unw) {
    // lanes r, r+16, r+32, r+48 hold the same row: fixed-order pair sums
    ub += __shfl_xor(ub, 16, 64);
    up += __shfl_xor(up, 16, 64);
    ub += __shfl_xor(ub, 32, 64);
    up += __shfl_xor(up, 32, 64);
    if (g4 == 0) {
      rs_out[r * 2] = ub;
      rs_out[r * 2 + 1] = up;
    }
  }
}

template <int NT>
constexpr int kClassOf = NT == 2 ? 0 : NT == 7 ? 1 : 2;

// One launch per column-tile class: wave w of the grid takes work item w of
// the class (item = split * n + task index), with the class's tasks, count
// and K-split read from the device schedule.  The grid has
// max(slots, tasks) waves, so every item has a wave.  Where the schedule sets
// R > 1 (classes 1 and 2), items are groups of R waves instead: item u of the
// grid's groups is task u % n at partial u / n, its R waves take R
// consecutive splits of the R * KS-way split and add their sums in LDS
// (n * KS * R <= slots, so the groups fit the grid).
template <int DT, int NT, int CNT, bool TAB, bool WIDE>
__global__ __launch_bounds__(64 * cost_waves(NT, TAB)) void cost_kernel(CostArgs a) {
  constexpr int CI = kClassOf<NT>;
  constexpr int WV = cost_waves(NT, TAB);
  constexpr bool kRed = CI > 0;  // classes whose splits the schedule may group
  constexpr bool KEYS = CNT == 0 && NT >= 7;
  __shared__ __align__(16) unsigned char lut_s[TAB ? kLutBytes : 16];
  __shared__ int prog_s[WV];
  __shared__ f32x4_t red_s[kRed ? (WV / 2) * 2 * NT * 64 : 1];
  __shared__ uint32_t klut_s[KEYS ? WV : 1][KEYS ? 260 : 1];
  __shared__ float2 red_rs[kRed ? (WV / 2) * 64 : 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n = __builtin_amdgcn_readfirstlane(a.sched[CI]);
  const int64_t KS = __builtin_amdgcn_readfirstlane(a.sched[kClasses + CI]);
  const int R = kRed ? __builtin_amdgcn_readfirstlane(a.sched[kSchedRed + CI]) : 1;
  const int64_t total = n * KS;
  // table build + barrier: once per wave, after its first loads are in flight
  auto setup = [&]() {
    if constexpr (TAB) build_lut<WIDE>(lut_s, a.ep, a.form.lg);
    __syncthreads();
  };
  constexpr int64_t tile = class_planes(CI) * 16 * 16 * NT;
  uint32_t* klut = KEYS ? &klut_s[KEYS ? wave : 0][0] : nullptr;
  if (kRed && R > 1) {
    const int gpw = WV / R;  // groups per workgroup
    const int grp = wave / R, r = wave - grp * R;
    const int64_t u0 = (int64_t)blockIdx.x * gpw;
    if (u0 >= total) return;  // the whole workgroup is idle
    const int64_t u = u0 + grp;
    if (u >= total) {  // an idle group still meets every barrier of the others
      setup();
      for (int h = R >> 1; h >= 1; h >>= 1)
        for (int k = 0; k < kRedBarriers; ++k) __syncthreads();
      return;
    }
    const int64_t i = u % n, kp = u / n;
    const int64_t task = __builtin_amdgcn_readfirstlane(a.sched[kSchedList + CI * a.plan.ntasks + i]);
    const int64_t lb = task / a.rtiles, rtile = task % a.rtiles;
    float* out = a.partials + a.plan.float_base[CI] + u * tile;
    float* rs = a.rowsum ? a.rowsum + (a.plan.slot_base[CI] + u) * 16 * 2 : nullptr;
    SplitRed red;
    red.buf = red_s;
    red.rsbuf = red_rs;
    red.R = R;
    red.r = r;
    red.grp = grp;
    cost_wave<DT, NT, CNT, TAB, WIDE>(a, lb, rtile, kp * R + r, KS * R, lut_s, out, rs, nullptr, setup, red, klut);
    return;
  }
  const int64_t w0 = (int64_t)blockIdx.x * WV;
  if (w0 >= total) return;  // the whole workgroup is idle
  if (threadIdx.x < WV) prog_s[threadIdx.x] = 0;
  const int64_t w = w0 + wave;
  if (w >= total) {
    setup();
    return;
  }
  const int64_t i = w % n, ks = w / n;
  const int64_t task = __builtin_amdgcn_readfirstlane(a.sched[kSchedList + CI * a.plan.ntasks + i]);
  const int64_t lb = task / a.rtiles, rtile = task % a.rtiles;
  float* out = a.partials + a.plan.float_base[CI] + w * tile;
  float* rs = a.rowsum ? a.rowsum + (a.plan.slot_base[CI] + w) * 16 * 2 : nullptr;
  // pace the waves only where many share the workgroup's CU
  cost_wave<DT, NT, CNT, TAB, WIDE>(a, lb, rtile, ks, KS, lut_s, out, rs, WV >= 16 ? prog_s : nullptr, setup,
                              SplitRed(), klut);
}

// ---- class 0 of bf16 table calls: row-tile pairs, 32x32x16 products ------------
// One wave takes 32 query rows (row tiles 2k and 2k + 1 of one image) and the
// 32 column slots of class 0 over its K-range, in K-steps of 16 cells: lane
// (r = lane & 31, h = lane >> 5) holds 8 cells of the step for query row r (A
// operand) and for column slot r (B operand), and its accumulators hold
// column r at rows 8 (v / 4) + 4 h + v % 4 of register v.
//
// HBM streams a row best in long runs, so the logits go through LDS: a group
// of 4 K-steps (32 rows x 64 cells, 4 KB) is fetched by four
// global_load_lds_dwordx4, each moving 1 KB as 8 rows x 128 contiguous bytes
// straight into the wave's LDS ring, and read back in the operand layout with
// one ds_read_b128 per K-step.  Instruction i has lane l load row R = 8 i +
// (l >> 3) at 16-byte chunk c = (l & 7) ^ (R & 7); the hardware stores lane l
// at ring slot 64 i + l = 8 R + (c ^ (R & 7)), so the 8 lanes of each read phase
// (8 consecutive rows, one chunk) touch 8 different bank groups.  The ring
// holds kRingGroups groups, so a group's fetch is in flight while the previous
// one is computed, without costing registers.
//
// Label maps: K-step s of a group holds cells 16 s + 8 h + (0 .. 7), and the
// labels are loaded a group ahead.  u8 counts: the K-steps of a group may hold its
// 64 cells in any order that both operands share, so K-step s holds cells 32 h +
// 8 s + (0 .. 7) and a lane's counts of the whole group are 32 consecutive bytes
// (two 16-byte loads, the wave's a run of 2 KB).
//
// A workgroup is 4 pairs x 4 adjacent K-splits (wave = 4 pair + split): the
// four splits of a pair are summed in LDS at the end, in the fixed order
// (s0 + s2) + (s1 + s3), and only that sum is written, so the partial sums
// that reach memory (and the finalize's reads of them) are a quarter of one
// tile per wave.  The schedule's class-0 split count is the number of such
// quads, KSq; the kernel runs 4 KSq K-ranges.
//
// Bound by vector-ALU issue (59 ops per K-step of 512 logits), LDS table reads and
// load latency at 4 waves per SIMD: 210 M logits against label maps 106 -> 100 us
// (traced; bf16 operands took 65 ops per K-step), 671 M against u8 counts of 4x targets
// 314 - 333 us (with the 7-tile class's 94 us; 886 + 208 us on the formula path).
//
// LDS map of the 16-wave workgroup: positive table block [0, 8 kLutBlock), the
// rings of waves 0 and 1 in the gap before the negative block at kLutNegOff,
// the negative block, then the rings of waves 2..15 (163,072 bytes).
constexpr int kGroupSteps = 4;            // K-steps per group
constexpr uint32_t kGroupBytes = 4096;    // 32 rows x 64 cells x 2 bytes
constexpr int kRingGroups = 2;
constexpr uint32_t kRingBytes = kRingGroups * kGroupBytes;
constexpr uint32_t kDmaWaves = 16;
constexpr uint32_t kLutBlockBytes = kLutBlock * 8;

static_assert(((kLutBlockBytes + 255) & ~255u) + 2 * kRingBytes <= kLutNegOff,
              "two rings fit between the table blocks");
constexpr uint32_t kDmaLds =
    ((kLutNegOff + kLutBlockBytes + 255) & ~255u) + (kDmaWaves - 2) * kRingBytes;
static_assert(kDmaLds <= 160 * 1024, "table and rings fit the LDS of one CU");

// Ring bases are 256-byte aligned, so a reader's address of K-step s is its
// step-0 address with bits of s flipped (see cost_wave_pair).
constexpr uint32_t kRingLo = (kLutBlockBytes + 255) & ~255u;
constexpr uint32_t kRingHi = (kLutNegOff + kLutBlockBytes + 255) & ~255u;
__device__ __forceinline__ uint32_t ring_base(int wave) {
  return wave < 2 ? kRingLo + wave * kRingBytes : kRingHi + (wave - 2) * kRingBytes;
}

typedef __attribute__((address_space(3))) void lds_void_t;

// One ds_read_b128 of the wave's ring, complete on return.  Written as
// assembly: the compiler would otherwise wait for every outstanding fetch
// before any LDS read, since it cannot tell which ring slot a
// global_load_lds writes.
__device__ __forceinline__ u32x4_t ring_read(uint32_t addr) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(addr) : "memory");
  return v;
}

// Table entries of 8 bf16 cells (as lut_lookup8) read with assembly, and the
// wait for them tied to their registers.  lut_base: the table's LDS address.
__device__ __forceinline__ void lut_lookup8_asm(const u32x4_t& x, uint32_t lut_base, uint64_t E[8]) {
  const uint32_t u[4] = {x[0], x[1], x[2], x[3]};
  uint32_t ad[4];  // the four words' chains side by side, then the reads
#pragma unroll
  for (int i = 0; i < 4; ++i) ad[i] = lut_addr_pair(u[i]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t addr = ad[i];
    asm volatile("ds_read_b64 %0, %1" : "=v"(E[2 * i]) : "v"(lut_base + (addr & 0xFFFFu)) : "memory");
    asm volatile("ds_read_b64 %0, %1" : "=v"(E[2 * i + 1]) : "v"(lut_base + (addr >> 16)) : "memory");
  }
}
// Wait for every outstanding LDS read; E (table entries) and x (ring words
// read earlier) are tied to it, so nothing that uses them moves above it.  Each
// is tied as the whole register group that its read writes: split into words, the
// compiler may copy them while the read is in flight.
__device__ __forceinline__ void lds_wait(uint64_t E[8], u32x4_t& x) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(E[0]), "+v"(E[1]), "+v"(E[2]), "+v"(E[3]), "+v"(E[4]), "+v"(E[5]), "+v"(E[6]),
                 "+v"(E[7]), "+v"(x));
}
// Wait for every outstanding LDS read at the end of a pipeline; the
// registers of reads nothing consumes are tied to it, so they stay reserved
// until the data has landed.
__device__ __forceinline__ void lds_drain(uint64_t E[8], u32x4_t (&x)[2]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(E[0]), "+v"(E[1]), "+v"(E[2]), "+v"(E[3]), "+v"(E[4]), "+v"(E[5]), "+v"(E[6]),
                 "+v"(E[7]), "+v"(x[0]), "+v"(x[1])
               :
               : "memory");
}
// One ds_read_b128 of the ring, not waited for (see lds_wait).
__device__ __forceinline__ u32x4_t ring_read_async(uint32_t addr) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr) : "memory");
  return v;
}
template <class V>
__device__ __forceinline__ void lut_planes64(const uint64_t E64[8], V A[4]) {
  uint2 E[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) E[i] = make_uint2((uint32_t)E64[i], (uint32_t)(E64[i] >> 32));
  lut_planes(E, A);
}
// 16 bytes of labels or counts from base + off + OFF, loaded with assembly (a
// wave-uniform base and a 32-bit lane offset: one address register);
// label_wait<N> waits until at most N vector-memory operations issued after it
// are outstanding.
template <int OFF>
__device__ __forceinline__ u32x4_t label_load(const void* base, uint32_t off) {
  // (a uniform value that the compiler keeps in vector registers would not fit
  // the scalar operand)
  const uint64_t u = (uint64_t)(uintptr_t)base;
  const uint64_t sb = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u) |
                      ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32)) << 32);
  u32x4_t v;
  asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(v) : "v"(off), "s"(sb), "n"(OFF) : "memory");
  return v;
}
template <int N>
__device__ __forceinline__ void label_wait(u32x4_t& v) {
  asm volatile("s_waitcnt vmcnt(%1)" : "+v"(v) : "n"(N));
}
// Drain every vector-memory operation; the operand registers are tied to it,
// so loads issued but never used (the pipeline's last ones) keep their
// registers until they have landed (an assembly load's destination would
// otherwise count as free at once and could be reused while it is in flight).
template <int N>
__device__ __forceinline__ void drain_loads(u32x4_t (&l)[N]) {
  if constexpr (N == 4)
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(l[0]), "+v"(l[1]), "+v"(l[2]), "+v"(l[3]) : : "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(l[0]), "+v"(l[1]) : : "memory");
}

constexpr int kPairStep = 16;                               // cells per K-step
constexpr int kPairGroupCells = kGroupSteps * kPairStep;    // 64 cells x 32 rows = 4 KB
constexpr int64_t kPairTile = 3 * 32 * 32;            // partial tile (floats)
static_assert(kPairGroupCells * 32 * 2 == (int)kGroupBytes, "a pair group fills one ring slot");
static_assert(kPairGroupCells == kCountCells, "a group's counts are one block");

// CNT: 0 label map, 1 u8 counts; WIDE: a table of bf16 (label maps only)
template <int CNT, bool WIDE, class Setup>
__device__ __forceinline__ void cost_wave_pair(const CostArgs& a, int64_t lb, int64_t q0, int64_t ks,
                                               int64_t KS, const unsigned char* lut, uint32_t ring,
                                               f32x16_t (&acc)[3], Setup&& setup) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, h = lane >> 5;
  const int64_t b = lb % a.B;
  const int G = __builtin_amdgcn_readfirstlane(a.ncols[b]);

  // the lane's column: its label pair and mask, or its row of the count tiles (see cost_wave)
  int act = -1;
  if (r < G) {
    const int c = a.colmap[b * a.nslot + r];
    act = c + (c >= a.bg ? 1 : 0);
  }
  const uint32_t colL = act >= 0 ? label_code(act) * 0x10001u : 0u;
  uint32_t colM = r == G ? 0u : 0xFFFFFFFFu;
  asm("" : "+v"(colM));  // a register, not a select at every use
  const int64_t cstep = (int64_t)a.counts.rows * kCountCells;  // bytes per block of counts
  const uint8_t* cimg = CNT ? a.counts.p + b * a.counts.nb * cstep : nullptr;
  const uint32_t crow = (uint32_t)(act >= 0 ? act : (int)a.GT_total + 1) * kCountCells;
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  };
  clear();

  using V = typename Ops<WIDE>::v8;
  RightF16 rf = right_f16(0, a.N2);
  rf.top = (uint32_t)__builtin_amdgcn_readfirstlane((int)rf.top);
  // full K-steps of this split (whole groups with counts), then the tail
  const int64_t full = CNT ? a.HW / kPairGroupCells * kGroupSteps : a.HW / kPairStep;
  const int64_t ngr = ceil_div(full, kGroupSteps);
  const int64_t gper = ceil_div(ngr, KS);
  const int64_t g0 = min(ngr, ks * gper), g1 = min(ngr, g0 + gper);
  const int64_t s0 = g0 * kGroupSteps;
  const int nst = (int)(min(full, g1 * kGroupSteps) - s0);
  const int64_t steps = ks == KS - 1 ? ceil_div(a.HW, kPairStep) : full;  // past `full`: this split's tail

  // fetch sources: rows past the last query read the last query's row
  // (never used); element offsets from zrow0 stay below 2^31 (host check)
  const uint16_t* zrow0 = (const uint16_t*)a.logits + (lb * a.Q + q0) * a.HW;
  const uint32_t HW32 = (uint32_t)a.HW, qlast = (uint32_t)(a.Q - 1 - q0);
  auto fetch_group = [&](int slot, int64_t g) {  // g in [g0, g1)
    const uint32_t cell0 = (uint32_t)(g * kPairGroupCells);
    const bool edge = cell0 + kPairGroupCells > HW32;  // wave-uniform
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t R = 8u * i + ((uint32_t)lane >> 3);
      uint32_t cell = cell0 + 8u * (((uint32_t)lane & 7u) ^ (R & 7u));
      if (edge) cell = min(cell, HW32 - 8u);  // past the row end: its last chunk (never used)
      // bytes below 2^32: a scalar base and a 32-bit lane offset
      const uint32_t off = (min(R, qlast) * HW32 + cell) * 2u;
      __builtin_amdgcn_global_load_lds((const void*)((const char*)zrow0 + off),
                                       (lds_void_t*)(size_t)(ring + slot * kGroupBytes + i * 1024), 16, 0, 0);
    }
  };
  // reader of K-step s of a group: ring + slot * kGroupBytes + 128 r + 16 (c ^ (r & 7))
  // for chunk c = 2 s + h (labels) or 4 h + s (counts); the ring is 256-byte
  // aligned, so that is the step-0 address with bits 5-6 or 4-5 flipped by s
  const uint32_t rd = ring + 128u * r + 16u * ((uint32_t)(CNT ? 4 * h : h) ^ ((uint32_t)r & 7u));
  auto step_addr = [&](int t) {
    const int s = t & (kGroupSteps - 1), slot = (t / kGroupSteps) & (kRingGroups - 1);
    return (rd ^ ((CNT ? 16u : 32u) * s)) + slot * kGroupBytes;
  };
  const uint16_t* labp = a.lab16 + (CNT ? 0 : b * a.HWp);
  u32x4_t lbuf[CNT ? 2 : kGroupSteps];  // labels of 4 K-steps, or counts of K-steps 0, 1 and 2, 3
  auto fetch_l = [&](int j, int t) {
    // t opaque: min(1, nst - 1) would become a vector select, and its readfirstlane
    // sit right before the load that uses it (a hazard inside assembly)
    asm("" : "+s"(t));
    const int64_t st = s0 + min(t, nst - 1);
    lbuf[j] = label_load<0>(labp + st * kPairStep, 16u * h);
  };
  auto fetch_c = [&](int j, int64_t g) {
    const uint8_t* p = cimg + min(g, g1 - 1) * cstep;
    lbuf[j] = j ? label_load<16>(p, crow + 32u * h) : label_load<0>(p, crow + 32u * h);
  };

  auto mma_ops = [&](auto ops, const auto& A, const Opnd& o) {
    using O = decltype(ops);
    const auto n = __builtin_bit_cast(typename O::v8, o.n), rest = __builtin_bit_cast(typename O::v8, o.rest);
    acc[0] = O::mma32(A[0], rest, acc[0]);
    acc[1] = O::mma32(A[2], n, acc[1]);
    acc[2] = O::mma32(A[3], n, acc[2]);
    acc[0] = O::mma32(A[1], n, acc[0]);
  };
  auto mma = [&](const V (&A)[4], const Opnd& o) { mma_ops(Ops<WIDE>(), A, o); };

  // Every load of the pipeline is issued in a fixed order, so the vmcnt waits
  // below are exact.
  //   Labels: labels of steps 0..3, groups 0 and 1; then per step t:
  //   [refill of this group's slot (s = 3)] [label of step t + 4].  The label
  //   of step t is then followed by exactly (near the start: at least) 7 later
  //   loads when it is used, and a group's fetch by at least 2 when its first
  //   step is read from the ring (two steps before that step).
  //   Counts: half 0 of group 0, groups 0 and 1, half 1 of group 0; then in group
  //   k: [half 0 of k + 1, after step 1 used it] [refill (s = 3)] [half 1 of
  //   k + 1, after step 3].  Half 0 is followed by 5 later loads when step 0
  //   uses it; half 1 by 1 when step 2 does, and group k + 1's fetch is older.
  // LDS reads run two steps ahead for the ring and one for the table: step t waits
  // for both (lds_wait), then issues the table reads of step t + 1 and the ring
  // read of step t + 2.
  int k = nst;  // steps summed by the table
  if (nst > 0) {
    const int ngl = (int)(g1 - g0);
    const uint32_t lut_base = (uint32_t)(size_t)(lds_void_t*)lut;
    if constexpr (CNT) {
      fetch_c(0, g0);
    } else {
#pragma unroll
      for (int j = 0; j < kGroupSteps; ++j) fetch_l(j, j);
    }
    fetch_group(0, g0);
    fetch_group(1, g0 + (ngl > 1 ? 1 : 0));
    if constexpr (CNT) fetch_c(1, g0);
    setup();
    // group 0 landed (group 1, and the counts' second half, may be in flight)
    if constexpr (CNT) __builtin_amdgcn_s_waitcnt(0x0F75);  // vmcnt(5)
    else __builtin_amdgcn_s_waitcnt(0x0F74);                // vmcnt(4)
    uint64_t E[8];
    u32x4_t xr[2];  // ring words of steps t + 1 (xr[(t + 1) & 1]) and t + 2
    const u32x4_t x0 = ring_read(step_addr(0));
    if (__ballot(lut_over8(x0[0], x0[1], x0[2], x0[3])) != 0ull) k = 0;  // a filled region: redone at once
    lut_lookup8_asm(x0, lut_base, E);
    xr[1] = nst > 1 ? ring_read_async(step_addr(1)) : u32x4_t{0u, 0u, 0u, 0u};
    for (int t0 = 0; t0 < k; t0 += kGroupSteps) {
#pragma unroll
      for (int s = 0; s < kGroupSteps; ++s) {  // s compile-time: lbuf and xr stay in registers
        const int t = t0 + s;
        if (CNT || t < nst) {  // with counts every group is whole
          u32x4_t& xn = xr[(s + 1) & 1];  // step t + 1
          u32x4_t& xnn = xr[s & 1];       // step t + 2
          lds_wait(E, xn);
          V A[4];
          lut_planes64(E, A);
          // E is consumed above the next lookups, which then reuse its
          // registers.  Past the last step the lookups and ring reads still
          // run (on stale ring words: table addresses stay in the table, ring
          // addresses in the ring), so no value depends on the step count;
          // lds_drain below waits for them.
          __builtin_amdgcn_sched_barrier(0);
          lut_lookup8_asm(xn, lut_base, E);
          if (s == kGroupSteps - 2) {  // step t + 2 opens the next group: its fetch has landed
            if constexpr (CNT) label_wait<1>(lbuf[1]);
            else __builtin_amdgcn_s_waitcnt(0x0F72);  // when at most 2 later loads are pending
          }
          xnn = ring_read_async(step_addr(t + 2));
          if (s == kGroupSteps - 1) {  // every step of this slot is read: refill it two groups on
            const int gk = t0 / kGroupSteps;
            fetch_group(gk & (kRingGroups - 1), g0 + min(gk + kRingGroups, ngl - 1));
          }
          Opnd o;
          if constexpr (CNT) {
            if (s == 0) label_wait<5>(lbuf[0]);
            o = opnd_u8<true>(lbuf[s >> 1][2 * (s & 1)], lbuf[s >> 1][2 * (s & 1) + 1], rf);
          } else {
            label_wait<7>(lbuf[s]);
            const uint32_t L2[4] = {lbuf[s][0], lbuf[s][1], lbuf[s][2], lbuf[s][3]};
            o = opnd_tab<WIDE>(hot8(L2, colL, colM));
          }
          __builtin_amdgcn_sched_barrier(0);
          mma(A, o);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (CNT) {
            if (s & 1) fetch_c(s >> 1, g0 + t0 / kGroupSteps + 1);
          } else {
            fetch_l(s, t + kGroupSteps);
          }
        }
      }
    }
    lds_drain(E, xr);
    drain_loads(lbuf);  // also: no fetch may land in LDS after the wave ends
  } else {
    setup();
  }

  // steps at natural cell order (16 st + 8 h + (0 .. 7)), guarded: the tail, and a redone range
  const ElemParams ep = a.ep;
  const int64_t rowoff = (lb * a.Q + min(q0 + r, a.Q - 1)) * a.HW + h * 8;
  // raw right operand of step st: compare results, or counts in the first two words
  auto counts_of = [&](int64_t st) -> u32x4_t {
    if constexpr (CNT) {
      const int64_t cell = st * kPairStep + h * 8;
      const uint2 c = *(const uint2*)(cimg + (cell >> 6) * cstep + crow + (cell & 63));
      return u32x4_t{c.x, c.y, 0u, 0u};
    } else {
      const uint4 lv = *(const uint4*)(labp + st * kPairStep + h * 8);
      const uint32_t L2[4] = {lv.x, lv.y, lv.z, lv.w};
      return hot8(L2, colL, colM);
    }
  };
  // |z| >= 64, inf or nan somewhere in the range (the table's marker): redone
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 16; ++e) bad |= !(fabsf(acc[0][e]) < INFINITY);
  const float undo = WIDE ? 2.f : __builtin_ldexpf(1.f, (CNT ? 0 : 16) - a.form.lg);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] *= undo;
  if (__builtin_expect(__ballot(bad) != 0ull, 0)) {
    clear();
    k = 0;
  }
  // the tail and a redone range: the formulas and bf16 operands, the next step's
  // loads in flight
  const int nall = nst + (int)(steps - full);
  if (__builtin_expect(k < nall, 0)) {
    auto nv_of = [&](int64_t st) { return a.HW - (st * kPairStep + h * 8); };
    Raw8<ML_BF16> raw, nraw;
    u32x4_t n, nn;
    auto fetch = [&](int k) {
      const int64_t st = k < nst ? s0 + k : full + (k - nst);
      if (k < nst) load_raw8<ML_BF16>(a.logits, rowoff + st * kPairStep, nraw);
      else load_raw8_part<ML_BF16>(a.logits, rowoff + st * kPairStep, nv_of(st), nraw);
      nn = counts_of(st);
    };
    fetch(k);
    for (; k < nall; ++k) {
      raw = nraw;
      n = nn;
      if (k + 1 < nall) fetch(k + 1);
      float z[8], v[4][8], ub = 0.f, up = 0.f;
      raw_to_f32<ML_BF16>(raw, z);
      if (k < nst) planes8<false>(z, ep, 1.f, 8, false, v, ub, up);
      else planes8<true>(z, ep, 1.f, nv_of(full + (k - nst)), false, v, ub, up);
      bf16x8_t A[4];
#pragma unroll
      for (int pl = 0; pl < 4; ++pl) split_bf16<1>(v[pl], &A[pl]);
      if constexpr (CNT) {
        mma_ops(Ops<true>(), A, wide_u8(n[0], n[1], a.N2));
      } else {
        const u32x4_t one = wide_hot8(n);
        mma_ops(Ops<true>(), A, Opnd{one, isub8(0x3F803F80u, one)});
      }
    }
  }
}

// One wave's accumulators in LDS (12 KB): 4 consecutive registers per lane
// as one 16-byte word, consecutive lanes at consecutive words.
__device__ __forceinline__ void acc_to_lds(float* buf, const f32x16_t (&acc)[3], int lane) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4)
      *(f32x4_t*)(buf + ((i * 4 + v4) * 64 + lane) * 4) =
          f32x4_t{acc[i][4 * v4], acc[i][4 * v4 + 1], acc[i][4 * v4 + 2], acc[i][4 * v4 + 3]};
}
__device__ __forceinline__ void acc_add_lds(f32x16_t (&acc)[3], const float* buf, int lane) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4) {
      const f32x4_t x = *(const f32x4_t*)(buf + ((i * 4 + v4) * 64 + lane) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][4 * v4 + e] += x[e];
    }
}

template <int CNT, bool WIDE>
__global__ __launch_bounds__(64 * kDmaWaves) void cost_pair_kernel(CostArgs a) {
  __shared__ __align__(16) unsigned char lds[kDmaLds];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t n = __builtin_amdgcn_readfirstlane(a.sched[0]);
  const int64_t KSq = __builtin_amdgcn_readfirstlane(a.sched[kClasses]);
  const int64_t rt = a.rtiles, prt = (rt + 1) >> 1;
  const int64_t np = (n / rt) * prt;  // class 0 holds whole images
  const int64_t npq = (np + 3) >> 2;
  // workgroup g: pairs 4 (g / KSq) .. + 3 at K-split quad g % KSq (split
  // quads fastest: measured faster than pair quads fastest on 512x512 maps)
  const int64_t g = blockIdx.x;
  if (g >= npq * KSq) return;  // the whole workgroup is idle
  const int64_t pq = g / KSq, ksq = g - pq * KSq, p = 4 * pq + (wave >> 2);
  const int kq = wave & 3;
  auto setup = [&]() {
    build_lut<WIDE>(lds, a.ep, a.form.lg);
    __syncthreads();
  };
  f32x16_t acc[3];
  int64_t lb = 0, rp = 0;
  if (p < np) {
    // pair p = row tiles 2 (p % prt) (+ 1) of the class's (p / prt)-th image
    const int64_t j = p / prt;
    rp = p - j * prt;
    const int64_t task = __builtin_amdgcn_readfirstlane(a.sched[kSchedList + j * rt + 2 * rp]);
    lb = task / rt;
    const uint32_t ring = (uint32_t)(size_t)(lds_void_t*)lds + ring_base(wave);
    cost_wave_pair<CNT, WIDE>(a, lb, 32 * rp, 4 * ksq + kq, 4 * KSq, lds, ring, acc, setup);
  } else {
    setup();
  }
  // sum the four splits of each pair: every wave has drained its loads, so
  // the table and the rings are free
  float* red = (float*)lds;
  constexpr int kAccFloats = 3 * 16 * 64;
  const int pp = wave >> 2;
  static_assert(8 * kAccFloats * 4 <= (int)kDmaLds, "eight waves' sums fit the LDS");
  __syncthreads();
  if (p < np && kq >= 2) acc_to_lds(red + (2 * pp + kq - 2) * kAccFloats, acc, lane);
  __syncthreads();
  if (p < np && kq < 2) acc_add_lds(acc, red + (2 * pp + kq) * kAccFloats, lane);
  __syncthreads();
  if (p < np && kq == 1) acc_to_lds(red + pp * kAccFloats, acc, lane);
  __syncthreads();
  if (p >= np || kq != 0) return;
  acc_add_lds(acc, red + pp * kAccFloats, lane);

  // item ksq * np + p: [3][32 rows][32 slots]; rows of the second tile only
  // for a real pair, slots up to G only (what the finalize reads)
  const int r = lane & 31, h = lane >> 5;
  const int G = __builtin_amdgcn_readfirstlane(a.ncols[lb % a.B]);
  const bool two = 2 * rp + 1 < rt;
  float* out = a.partials + a.plan.float_base[0] + (ksq * np + p) * kPairTile;
  if (r <= G) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = 8 * (v >> 2) + 4 * h + (v & 3);
        if (two || m < 16) out[(i * 32 + m) * 32 + r] = acc[i][v];
      }
  }
}

// ---- launch plan ---------------------------------------------------------------
// Resident waves of a kernel of `waves` waves per workgroup on the current
// device, cached per device in `cache`.
inline int occ_slots(std::atomic<int> (&cache)[64], const void* kernel, int waves) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int nb = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, 64 * waves, 0) != hipSuccess || nb < 1) nb = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
      cus = 256;
    v = nb * cus * waves;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}
template <int DT, int NT, int CNT, bool TAB, bool WIDE>
static int occ_slots_of() {
  static std::atomic<int> cache[64];
  return occ_slots(cache, (const void*)cost_kernel<DT, NT, CNT, TAB, WIDE>, cost_waves(NT, TAB));
}
template <int CNT, bool WIDE>
static int occ_slots_pair() {
  static std::atomic<int> cache[64];
  return occ_slots(cache, (const void*)cost_pair_kernel<CNT, WIDE>, (int)kDmaWaves);
}

// cnt: 0 label map, 1 u8 counts, 2 u16 counts
template <int DT, int NT>
static int occ_slots_for(int cnt, bool tab, bool wide) {
  constexpr bool kTab = DT == ML_BF16;
  if (kTab && tab)
    return cnt == 1   ? occ_slots_of<DT, NT, 1, kTab, false>()
           : cnt == 2 ? occ_slots_of<DT, NT, 2, kTab, false>()
           : wide     ? occ_slots_of<DT, NT, 0, kTab, true>()
                      : occ_slots_of<DT, NT, 0, kTab, false>();
  if (wide)
    return cnt == 1   ? occ_slots_of<DT, NT, 1, false, true>()
           : cnt == 2 ? occ_slots_of<DT, NT, 2, false, true>()
                      : occ_slots_of<DT, NT, 0, false, true>();
  return cnt == 1   ? occ_slots_of<DT, NT, 1, false, false>()
         : cnt == 2 ? occ_slots_of<DT, NT, 2, false, false>()
                    : occ_slots_of<DT, NT, 0, false, false>();
}

inline int cu_count() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v < 1) v = 256;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// With three classes the narrower ones leave `side` CUs' worth of waves free:
// their launches may run beside the widest class's assignment (one
// workgroup per image on the forward's side stream).
template <int DT>
void plan_slots(CostPlan& p, int cnt, bool tab, bool wide, int64_t side) {
  const int cus = cu_count();
  side = std::min<int64_t>(side, cus / 8);
  for (int ci = 0; ci < p.nclass; ++ci) {
    int v = 0;
    switch (ci) {
      case 0:
        if constexpr (DT == ML_BF16) {
          if (p.pair0) {
            v = cnt ? occ_slots_pair<1, false>() : wide ? occ_slots_pair<0, true>() : occ_slots_pair<0, false>();
            break;
          }
        }
        v = occ_slots_for<DT, 2>(cnt, tab, wide);
        break;
      case 1: v = occ_slots_for<DT, 7>(cnt, tab, wide); break;
      default: v = occ_slots_for<DT, 16>(cnt, tab, wide); break;
    }
    if (p.nclass == kClasses && ci < kClasses - 1) v -= (int)((int64_t)v * side / cus);
    p.slots[ci] = (int)std::min<int64_t>(std::max(v, 8), kCostSlots);
  }
}

template <int DT, int NT, bool TAB>
static void launch_cnt(const CostArgs& a, const Dims& d, hipStream_t st) {
  const int WV = cost_waves(NT, TAB);
  const dim3 grid((unsigned)ceil_div(std::max<int64_t>(a.plan.slots[kClassOf<NT>], a.plan.ntasks), WV)), blk(64 * WV);
  auto launch = [&](auto wide) {
    constexpr bool WIDE = decltype(wide)::value, COUNTS = !(TAB && WIDE);
    if (!COUNTS || !d.counts_mode) hipLaunchKernelGGL((cost_kernel<DT, NT, 0, TAB, WIDE>), grid, blk, 0, st, a);
    else if (d.cw == 1) hipLaunchKernelGGL((cost_kernel<DT, NT, COUNTS ? 1 : 0, TAB, WIDE>), grid, blk, 0, st, a);
    else hipLaunchKernelGGL((cost_kernel<DT, NT, COUNTS ? 2 : 0, TAB, WIDE>), grid, blk, 0, st, a);
  };
  if (a.form.wide) launch(std::true_type());
  else launch(std::false_type());
}

template <int DT, int NT>
static int launch_one(const CostArgs& a, const Dims& d, hipStream_t st) {
  constexpr int CI = kClassOf<NT>;
  if (NT == 2 && a.plan.pair0) {
    // the schedule's K-split was chosen for row-tile pairs
    if (DT != ML_BF16 || !a.form.tab || !d.pair_ok || d.rows != 16)
      return fail(ML_EINVAL, "internal: row-tile pair plan without the bf16 table path");
    // workgroups: ceil(np / 4) pair quads x KSq split quads, where np * 4 KSq
    // <= max(slots, np) unless KSq = 1 (then np <= L B ceil(rtiles / 2)), and
    // KSq <= ks_max / 4; surplus workgroups exit at once
    const int64_t np_max = d.LB * ((d.rtiles + 1) / 2);
    const int64_t wgs = ceil_div(a.plan.slots[CI], 16) + ceil_div(np_max, 4) + d.ks_max / 4 + 1;
    const dim3 grid((unsigned)wgs), blk(64 * kDmaWaves);
    if constexpr (DT == ML_BF16) {
      if (d.counts_mode) hipLaunchKernelGGL((cost_pair_kernel<1, false>), grid, blk, 0, st, a);
      else if (a.form.wide) hipLaunchKernelGGL((cost_pair_kernel<0, true>), grid, blk, 0, st, a);
      else hipLaunchKernelGGL((cost_pair_kernel<0, false>), grid, blk, 0, st, a);
    }
    return check_launch("pair_cost");
  }
  if (DT == ML_BF16 && a.form.tab) launch_cnt<DT, NT, DT == ML_BF16>(a, d, st);
  else launch_cnt<DT, NT, false>(a, d, st);
  return check_launch("pair_cost");
}

// One launch per column-tile class up to the padded width; each image is
// processed by exactly one of them.
template <int DT>
int launch_classes(const CostArgs& a, const Dims& d, unsigned classes, hipStream_t st) {
  int rc = 0;
  if (classes & 1u) rc = launch_one<DT, 2>(a, d, st);
  if (!rc && a.plan.nclass > 1 && (classes & 2u)) rc = launch_one<DT, 7>(a, d, st);
  if (!rc && a.plan.nclass > 2 && (classes & 4u)) rc = launch_one<DT, 16>(a, d, st);
  return rc;
}

#define ML_COST_TYPE(DT)                                                      \
  template void plan_slots<DT>(CostPlan&, int, bool, bool, int64_t);          \
  template int launch_classes<DT>(const CostArgs&, const Dims&, unsigned, hipStream_t);

}  // namespace ml
