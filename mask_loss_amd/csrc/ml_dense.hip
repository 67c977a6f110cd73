// Non-pairwise (per-class) losses over dense class logits (L, B, C, H, W)
// against an integer label map (B, Ht, Wt), counted per low-resolution cell:
//
//   sigmoid CE (src/cuda/sigmoid_ce.cu:13-332):
//     loss[l] = scale / (num_masks Ht Wt) * sum_{b,c,cell} ap mp cp n + an mn cn (N2 - n)
//     grad    = g[l] scale / (num_masks Ht Wt) *
//               ( -ap n mp (gamma p cp + 1-p) + an (N2-n) mn (gamma (1-p) cn + p) )
//   dice (src/cuda/dice_loss.cu:13-289):
//     I = sum p n, P = sum N2 p, T = sum n   per (l, b, c)
//     loss[l] = scale / num_masks * sum_{b,c} 1 - (2I + smooth) / (P + T + smooth)
//     grad    = -g[l] scale / num_masks * (2 n D - N2 (2I + smooth)) / D^2 * p (1-p),
//               D = P + T + smooth
//
// with n = count of class c inside the s x s target block of the cell.  The
// reference gives every low-resolution cell its own block of 64 threads and
// reads the C logits of that cell with stride H*W; here a workgroup streams a
// contiguous chunk of one (l, b, c) plane (coalesced 16-byte loads) against
// the compact targets (u16 labels for s == 1, u8 / u16 counts for s > 1) shared by
// all planes of the image, or (s > 1, dense_groups) counts its cells in LDS and
// streams all planes over them.  Sums are float64 per workgroup, combined in a
// fixed order by one small kernel, so results are deterministic (the
// reference's float / double atomics are not).
#include "ml_counts.h"
#include "ml_internal.h"

namespace ml {

constexpr int kDenseU = 4;                                 // 8-cell groups per thread
constexpr int64_t kDenseChunk = 256 * 8 * kDenseU;         // cells per workgroup

__device__ __forceinline__ void dense_load8(const void* base, int dt, int64_t i, int64_t nvalid,
                                            bool vec, float z[8]) {
  if (dt == ML_F32) {
    const float* p = (const float*)base + i;
    if (vec && nvalid >= 8) {
      const float4 v0 = *(const float4*)p;
      const float4 v1 = *(const float4*)(p + 4);
      z[0] = v0.x; z[1] = v0.y; z[2] = v0.z; z[3] = v0.w;
      z[4] = v1.x; z[5] = v1.y; z[6] = v1.z; z[7] = v1.w;
    } else {
      for (int k = 0; k < 8; ++k) z[k] = k < nvalid ? p[k] : 0.f;
    }
    return;
  }
  const uint16_t* p = (const uint16_t*)base + i;
  uint32_t w[4];
  if (vec && nvalid >= 8) {
    const uint4 v = *(const uint4*)p;
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
  } else {
    for (int k = 0; k < 4; ++k) {
      const uint32_t lo = 2 * k < nvalid ? p[2 * k] : 0u;
      const uint32_t hi = 2 * k + 1 < nvalid ? p[2 * k + 1] : 0u;
      w[k] = lo | (hi << 16);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (dt == ML_BF16) {
      z[2 * k] = bf16_lo(w[k]);
      z[2 * k + 1] = bf16_hi(w[k]);
    } else {
      z[2 * k] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[k] & 0xFFFF));
      z[2 * k + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[k] >> 16));
    }
  }
}

__device__ __forceinline__ void dense_store8(void* base, int dt, int64_t i, const float g[8],
                                             int64_t nvalid, bool vec) {
  if (dt == ML_F32) {
    float* p = (float*)base + i;
    if (vec && nvalid >= 8) {
      *(float4*)p = make_float4(g[0], g[1], g[2], g[3]);
      *(float4*)(p + 4) = make_float4(g[4], g[5], g[6], g[7]);
    } else {
      for (int k = 0; k < 8; ++k)
        if (k < nvalid) p[k] = g[k];
    }
    return;
  }
  uint16_t* p = (uint16_t*)base + i;
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (dt == ML_BF16) {
      w[k] = pack_bf16x2(g[2 * k], g[2 * k + 1]);
    } else {
      const uint16_t lo = __builtin_bit_cast(uint16_t, (_Float16)g[2 * k]);
      const uint16_t hi = __builtin_bit_cast(uint16_t, (_Float16)g[2 * k + 1]);
      w[k] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
  }
  if (vec && nvalid >= 8) {
    *(uint4*)p = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    for (int k = 0; k < 8; ++k)
      if (k < nvalid) p[k] = (uint16_t)(w[k >> 1] >> ((k & 1) * 16));
  }
}

// counts of class c for 8 cells starting at cell0
__device__ __forceinline__ void dense_count8(const DenseArgs& a, int64_t b, int64_t c,
                                             int64_t cell0, float n[8]) {
  if (a.counts.p == nullptr) {
    const uint4 lv = *(const uint4*)(a.lab16 + b * a.HWp + cell0);
    const uint32_t w[4] = {lv.x, lv.y, lv.z, lv.w};
    const uint32_t c32 = (uint32_t)c;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      n[2 * k] = (w[k] & 0xFFFFu) == c32 ? 1.f : 0.f;
      n[2 * k + 1] = (w[k] >> 16) == c32 ? 1.f : 0.f;
    }
  } else {
    counts8_f(a.counts.p, a.counts.cw, a.counts.at(b, c, cell0), n);
  }
}

__device__ __forceinline__ double block_sum_d(double v, double* sh) {
  v = wave_sum_d(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__device__ __forceinline__ float ce_elem(const ElemParams& ep, float N2, float z, float n) {
  const Sig sg = sig_terms(z);
  float mn, mp;
  focal_mods(sg, ep, mn, mp);
  const float lp = ep.ap * mp * sg.cp * n;
  const float ln = ep.an * mn * sg.cn * (N2 - n);
  return lp + ln;
}

// Gradient of one element with its plane's coefficients (reference: grad_out /
// (num_masks Ht Wt) in float, times scale; dice: -grad_out / num_masks times
// scale).
template <bool DICE>
struct DenseGrad {
  float coef, D = 1.f, num = 0.f, invD2 = 0.f;
  __device__ __forceinline__ void layer(const DenseArgs& a, int64_t l) {
    if constexpr (DICE) coef = (float)(-(double)a.grad_out[l] / a.num_masks) * a.scale;
    else coef = (float)((double)a.grad_out[l] / (a.num_masks * (double)a.HtWt)) * a.scale;
  }
  __device__ __forceinline__ void plane(const DenseArgs& a, int64_t o) {
    if constexpr (DICE) {
      D = a.P_in[o] + a.T_in[o] + a.smooth;
      num = 2.f * a.I_in[o] + a.smooth;
      invD2 = 1.f / (D * D);
    }
  }
  __device__ __forceinline__ float operator()(const DenseArgs& a, float z, float n) const {
    const Sig sg = sig_terms(z);
    if constexpr (DICE) return coef * ((2.f * n * D - a.N2 * num) * invD2) * (sg.p * sg.q1);
    float mn, mp;
    focal_mods(sg, a.ep, mn, mp);
    const float gm = a.ep.gamma;
    const float gp = -a.ep.ap * n * mp * (gm * sg.p * sg.cp + sg.q1);
    const float gn = a.ep.an * (a.N2 - n) * mn * (gm * sg.q1 * sg.cn + sg.p);
    return (gp + gn) * coef;
  }
};

// Forward partial sums of one chunk of one (l, b, c) plane.
// grid (nchunk, C, L*B); partials[(lb*C + c)*nchunk + chunk][np]
template <bool DICE>
__global__ __launch_bounds__(256) void dense_fwd_kernel(DenseArgs a, int64_t nchunk) {
  __shared__ double sh[3][4];
  const int64_t chunk = blockIdx.x, c = blockIdx.y, lb = blockIdx.z;
  const int64_t b = lb % a.B;
  const int64_t plane = (lb * a.C + c) * a.HW;
  const bool vec = a.dtype == ML_F32 ? (a.HW % 4 == 0) : (a.HW % 8 == 0);
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  const int64_t c0 = chunk * kDenseChunk + (int64_t)threadIdx.x * 8;
  float z[kDenseU][8], n[kDenseU][8];
#pragma unroll
  for (int u = 0; u < kDenseU; ++u) {
    const int64_t cell0 = c0 + u * 256 * 8;
    if (cell0 < a.HW) {
      dense_load8(a.logits, a.dtype, plane + cell0, a.HW - cell0, vec, z[u]);
      dense_count8(a, b, c, cell0, n[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < kDenseU; ++u) {
    const int64_t cell0 = c0 + u * 256 * 8;
    if (cell0 >= a.HW) continue;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (cell0 + k >= a.HW) continue;
      const float nk = n[u][k];
      if constexpr (DICE) {
        const Sig sg = sig_terms(z[u][k]);
        s0 += (double)(sg.p * nk);     // I
        s1 += (double)(a.N2 * sg.p);   // P
        s2 += (double)nk;              // T
      } else {
        s0 += (double)ce_elem(a.ep, a.N2, z[u][k], nk);
      }
    }
  }
  double* out = a.partials + ((lb * a.C + c) * nchunk + chunk) * (DICE ? 3 : 1);
  s0 = block_sum_d(s0, sh[0]);
  if constexpr (DICE) {
    s1 = block_sum_d(s1, sh[1]);
    s2 = block_sum_d(s2, sh[2]);
  }
  if (threadIdx.x == 0) {
    out[0] = s0;
    if constexpr (DICE) {
      out[1] = s1;
      out[2] = s2;
    }
  }
}

// Fixed-order reduction, one workgroup per layer.
//   sigmoid: loss[l] = scale * sum / (num_masks Ht Wt)
//   dice: I, P, T per (l, b, c) (float), loss[l] = scale / num_masks * sum (1 - dice)
template <bool DICE>
__global__ __launch_bounds__(256) void dense_reduce_kernel(DenseArgs a, int64_t planes, int64_t nchunk) {
  __shared__ double sh[4];
  const int64_t l = blockIdx.x;
  double acc = 0.0;
  if constexpr (DICE) {
    for (int64_t pl = threadIdx.x; pl < planes; pl += 256) {
      const double* src = a.partials + (l * planes + pl) * nchunk * 3;
      double I = 0.0, P = 0.0, T = 0.0;
      for (int64_t k = 0; k < nchunk; ++k) {
        I += src[3 * k];
        P += src[3 * k + 1];
        T += src[3 * k + 2];
      }
      const int64_t o = l * planes + pl;
      a.I_out[o] = (float)I;
      a.P_out[o] = (float)P;
      a.T_out[o] = (float)T;
      acc += 1.0 - (2.0 * I + a.smooth) / (P + T + a.smooth);
    }
  } else {
    const double* src = a.partials + l * planes * nchunk;
    for (int64_t i = threadIdx.x; i < planes * nchunk; i += 256) acc += src[i];
  }
  acc = block_sum_d(acc, sh);
  if (threadIdx.x == 0) {
    if constexpr (DICE) a.loss[l] = (float)(acc / a.num_masks * a.scale);
    else a.loss[l] = (float)(acc * a.scale / (a.num_masks * (double)a.HtWt));
  }
}

// Gradients, elementwise.  grid (nchunk, C, L*B)
template <bool DICE>
__global__ __launch_bounds__(256) void dense_bwd_kernel(DenseArgs a, int64_t nchunk) {
  const int64_t chunk = blockIdx.x, c = blockIdx.y, lb = blockIdx.z;
  const int64_t b = lb % a.B, l = lb / a.B;
  const int64_t plane = (lb * a.C + c) * a.HW;
  const bool vec = a.dtype == ML_F32 ? (a.HW % 4 == 0) : (a.HW % 8 == 0);
  const int64_t c0 = chunk * kDenseChunk + (int64_t)threadIdx.x * 8;
  DenseGrad<DICE> grad;
  grad.layer(a, l);
  grad.plane(a, lb * a.C + c);
  float z[kDenseU][8], n[kDenseU][8];
#pragma unroll
  for (int u = 0; u < kDenseU; ++u) {
    const int64_t cell0 = c0 + u * 256 * 8;
    if (cell0 < a.HW) {
      dense_load8(a.logits, a.dtype, plane + cell0, a.HW - cell0, vec, z[u]);
      dense_count8(a, b, c, cell0, n[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < kDenseU; ++u) {
    const int64_t cell0 = c0 + u * 256 * 8;
    if (cell0 >= a.HW) continue;
    float g[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] = grad(a, z[u][k], n[u][k]);
    dense_store8(a.grad, a.dtype, plane + cell0, g, a.HW - cell0, vec);
  }
}

// ---- s > 1: counts made where they are used --------------------------------
// One workgroup takes 256 cells and rc of the classes: it counts the cells'
// target pixels in LDS (ml_counts.h) and then streams the class planes of
// every layer over those cells, a wave per class row, 4 cells per lane.
//
// Bound by the logits (and the gradient).  Counting in a launch of its own
// costs another pass: at 4 images, 150 classes, 128 x 128, s = 4 that launch
// took 7.9 us and wrote 9.8 MB which this one reads back beside 39 MB of
// logits.  Figures there, launch of the counts included: CE forward 17.5 + 7.9 ->
// 16.0 us, CE gradient 23.4 + 7.9 -> 20.6 us (87 MB, 4.2 TB/s), dice gradient
// 18.4 + 7.9 -> 18.8 us.
enum { kDenseCe = 0, kDenseCeGrad = 1, kDenseDiceGrad = 2 };
constexpr int kFuseU = 4;  // class rows in flight per wave

template <bool F32>
__device__ __forceinline__ void dense_load4(uint32_t raw[4], const void* base, int64_t i, int64_t nvalid, bool vec) {
  if constexpr (F32) {
    const uint32_t* p = (const uint32_t*)base + i;
    if (vec && nvalid >= 4) {
      const uint4 v = *(const uint4*)p;
      raw[0] = v.x; raw[1] = v.y; raw[2] = v.z; raw[3] = v.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) raw[k] = k < nvalid ? p[k] : 0u;
    }
    return;
  }
  const uint16_t* p = (const uint16_t*)base + i;
  if (vec && nvalid >= 4) {
    const uint2 v = *(const uint2*)p;
    raw[0] = v.x; raw[1] = v.y;
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t lo = 2 * k < nvalid ? p[2 * k] : 0u, hi = 2 * k + 1 < nvalid ? p[2 * k + 1] : 0u;
      raw[k] = lo | (hi << 16);
    }
  }
  raw[2] = raw[3] = 0u;
}

template <bool F32>
__device__ __forceinline__ void dense_floats4(const uint32_t raw[4], int dt, float z[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (F32) z[k] = __builtin_bit_cast(float, raw[k]);
    else if (dt == ML_BF16) z[k] = k & 1 ? bf16_hi(raw[k >> 1]) : bf16_lo(raw[k >> 1]);
    else z[k] = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[k >> 1] >> (16 * (k & 1))));
  }
}

template <bool F32>
__device__ __forceinline__ void dense_store4(void* base, int dt, int64_t i, const float g[4], int64_t nvalid, bool vec) {
  if constexpr (F32) {
    float* p = (float*)base + i;
    if (vec && nvalid >= 4) {
      *(float4*)p = make_float4(g[0], g[1], g[2], g[3]);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < nvalid) p[k] = g[k];
    }
    return;
  }
  uint32_t w[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (dt == ML_BF16) {
      w[k] = pack_bf16x2(g[2 * k], g[2 * k + 1]);
    } else {
      const uint16_t lo = __builtin_bit_cast(uint16_t, (_Float16)g[2 * k]);
      const uint16_t hi = __builtin_bit_cast(uint16_t, (_Float16)g[2 * k + 1]);
      w[k] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
  }
  uint16_t* p = (uint16_t*)base + i;
  if (vec && nvalid >= 4) {
    *(uint2*)p = make_uint2(w[0], w[1]);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < nvalid) p[k] = (uint16_t)(w[k >> 1] >> ((k & 1) * 16));
  }
}

// grid (ceil(HW / 256), groups of rc classes, B); partials[l][b][group][block]
template <int KIND, int S, bool F32>
__global__ __launch_bounds__(kCntThreads) void dense_fused_kernel(DenseArgs a, int rc) {
  constexpr bool DICE = KIND == kDenseDiceGrad;
  __shared__ double sh[kCntThreads / 64];
  extern __shared__ __align__(16) unsigned char tile[];  // [4 blocks][rc][64]
  const int64_t b = blockIdx.z, r0 = (int64_t)blockIdx.y * rc;
  const int nr = (int)min((int64_t)rc, a.C - r0);
  const int tid = threadIdx.x, cl = tid >> 2, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t cell = (int64_t)blockIdx.x * kCntCells + lane * 4, left = a.HW - cell;
  const bool vec = a.HW % 4 == 0;
  CellLabels<S> px;
  px.load(a.targets, b, a.Ht, a.Wt, a.W, a.HW, a.s, (int64_t)blockIdx.x * kCntCells + cl, a.tvec != 0);
  uint32_t raw[kFuseU][4];
  auto load = [&](int64_t l, int r) {  // rows r, r + 16, ... of layer l
    const int64_t plane0 = ((l * a.B + b) * a.C + r0) * a.HW + cell;
#pragma unroll
    for (int u = 0; u < kFuseU; ++u)
      if (r + 16 * u < nr) dense_load4<F32>(raw[u], a.logits, plane0 + (r + 16 * u) * a.HW, left, vec);
  };
  load(0, wave);  // under the counting
  for (int i = tid; i < nr * (kCntCells / 16); i += kCntThreads) ((uint4*)tile)[i] = make_uint4(0u, 0u, 0u, 0u);
  px.settle();
  __syncthreads();
  px.runs([&](int64_t lab, uint32_t n, bool single) {
    const int64_t r = lab - r0;
    if (r >= 0 && r < nr) tile_add<1>(tile, nr, (int)r, cl, n, single);
  });
  __syncthreads();
  const unsigned char* cnt = tile + (lane >> 4) * nr * kCountCells + (lane & 15) * 4;
  for (int64_t l = 0; l < a.L; ++l) {
    double acc = 0.0;
    DenseGrad<DICE> grad;
    if constexpr (KIND != kDenseCe) grad.layer(a, l);
    const int64_t o0 = (l * a.B + b) * a.C + r0;
    for (int r = wave; r < nr; r += 16 * kFuseU) {
      if (l > 0 || r != wave) load(l, r);
#pragma unroll
      for (int u = 0; u < kFuseU; ++u) {
        const int ru = r + 16 * u;
        if (ru >= nr) continue;
        const uint32_t nw = *(const uint32_t*)(cnt + ru * kCountCells);
        float z[4], n[4];
        dense_floats4<F32>(raw[u], a.dtype, z);
#pragma unroll
        for (int k = 0; k < 4; ++k) n[k] = (float)((nw >> (8 * k)) & 0xFFu);
        if constexpr (KIND == kDenseCe) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float e = ce_elem(a.ep, a.N2, z[k], n[k]);
            if (k < left) acc += (double)e;
          }
        } else {
          float g[4];
          grad.plane(a, o0 + ru);
#pragma unroll
          for (int k = 0; k < 4; ++k) g[k] = grad(a, z[k], n[k]);
          dense_store4<F32>(a.grad, a.dtype, (o0 + ru) * a.HW + cell, g, left, vec);
        }
      }
    }
    if constexpr (KIND == kDenseCe) {
      acc = wave_sum_d(acc);
      __syncthreads();
      if (lane == 0) sh[wave] = acc;
      __syncthreads();
      if (tid == 0) {
        double v = 0.0;
        for (int k = 0; k < kCntThreads / 64; ++k) v += sh[k];
        a.partials[((l * a.B + b) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = v;
      }
    }
  }
}

// The class groups of a fused launch, or 0 where the counts are better made
// once in memory: sums of the dice forward are per class, which 256 cells are
// too few for; counts above 255 do not fit the tile; and where the LDS rows
// (kFuseRows) make more groups, each reads the labels (8 s^2 bytes a cell)
// again, against the 2 bytes per cell and class of storing and reading a count.
constexpr int64_t kFuseRows = 160;
// A wave takes a class row, so below 16 classes waves are idle while the labels
// of 256 cells wait: 2 classes of 8 maps of 512 x 512, s = 2: CE forward 71 us
// against 34 with the counts in memory, gradients 81 and 74 against 33 and 30;
// 19 classes of 6 x 2 maps of 256 x 256, s = 2: 28, 31 and 27 against 34, 38 and 31.
constexpr int64_t kFuseLeast = 16;
// The counts' launch saves a fixed time, and streaming 4 cells per lane under
// the labels' wait is slower per logit than the plane kernels (8 cells per
// lane), more so for 16-bit logits.  float32: 17 M logits 39, 48 and 43 us
// against 65, 71 and 63; 34 M 96, 127 and 123 against 67, 93 and 88.  bf16 /
// float16: 12.5 M 29, 26 and 22 against 31, 34 and 26; 16 M 40, 49 and 40
// against 29, 33 and 23; 84 M 126, 163 and 170 against 90, 133 and 91.
constexpr int64_t kFuseElems = 3 << 22;
// More groups than that only where the cells alone leave whole multiples of CUs (256
// on this card) without a workgroup: with 256 workgroups of 150 classes the three
// kernels below take 16.0, 20.6 and 18.8 us, with 512 of 75 classes 16.6, 24.9 and
// 23.3, with 1024 of 38 classes 21.6, 30.8 and 28.2; s = 8, 40 classes of one 200 x 200
// map in 157 workgroups 16, 15 and 14, in 314 27, 26 and 26 (23, 21 and 19 with the
// counts in memory).
constexpr int64_t kFuseBlocks = 256;
// ... and not where the groups' label reads add up: s = 12, 100 classes of one 128 x 128
// map in 4 groups (76 MB) 33, 32 and 31 us, in 2 (38 MB) 29, 28 and 27, with the
// counts in memory 30, 30 and 27; s = 10 in 4 groups (52 MB) 22, 21 and 20 against 25,
// 24 and 21.  Over 16 to 160 classes and 4,096 to 147,456 cells at s = 2, 4, 5, 8, 10, 12 and
// 15 the sum of the three is 1.65, 1.61, 1.50, 1.33, 1.23, 1.18 and 1.09 times as fast as with the
// counts in memory (the least 0.85: s = 15, 100 and more classes of one 64 x 64 map).
constexpr int64_t kFuseLabelBytes = (int64_t)56 << 20;
int64_t dense_groups(int64_t L, int64_t B, int64_t C, int64_t HW, int64_t s, bool f32, bool dice, bool backward) {
  if (s < 2 || s > 15 || (dice && !backward) || B < 1 || C < kFuseLeast || B > 65535) return 0;
  if (L * B * C * HW > kFuseElems * (f32 ? 2 : 1)) return 0;
  const int64_t least = ceil_div(C, kFuseRows);
  if ((least - 1) * 8 * s * s > 2 * C) return 0;
  const int64_t fill = std::min({kFuseBlocks / (ceil_div(HW, kCntCells) * B), kFuseLabelBytes / (8 * s * s * HW * B),
                                 ceil_div(C, 16)});
  const int64_t g = std::max({least, fill, (int64_t)1});
  return ceil_div(C, ceil_div(C, g));
}

template <int KIND, bool F32>
static void launch_fused_dt(const DenseArgs& a, int64_t groups, hipStream_t st) {
  const int rc = (int)ceil_div(a.C, groups);
  const dim3 grid((unsigned)ceil_div(a.HW, kCntCells), (unsigned)groups, (unsigned)a.B);
  const size_t lds = (size_t)rc * kCntCells;
  if (a.s == 4) hipLaunchKernelGGL((dense_fused_kernel<KIND, 4, F32>), grid, dim3(kCntThreads), lds, st, a, rc);
  else if (a.s == 2) hipLaunchKernelGGL((dense_fused_kernel<KIND, 2, F32>), grid, dim3(kCntThreads), lds, st, a, rc);
  else hipLaunchKernelGGL((dense_fused_kernel<KIND, 0, F32>), grid, dim3(kCntThreads), lds, st, a, rc);
}

template <int KIND>
static void launch_fused(const DenseArgs& a, int64_t groups, hipStream_t st) {
  if (a.dtype == ML_F32) launch_fused_dt<KIND, true>(a, groups, st);
  else launch_fused_dt<KIND, false>(a, groups, st);
}

int launch_dense(const DenseArgs& a, bool dice, bool backward, hipStream_t st) {
  const int64_t groups = a.groups;
  int64_t planes = a.B * a.C, nchunk = ceil_div(a.HW, kDenseChunk);
  if (a.L == 0) return ML_OK;
  if (a.C > 65535 || a.L * a.B > 65535 || nchunk > INT32_MAX)
    return fail(ML_EUNSUPPORTED, "dense loss: grid dimensions out of range");
  const dim3 grid((unsigned)nchunk, (unsigned)a.C, (unsigned)(a.L * a.B));
  const bool work = planes > 0 && a.HW > 0;
  ProfScope ps_(dice ? "dice" : "sigmoid_ce", st);
  if (backward) {
    if (!work) return ML_OK;
    if (groups && dice) launch_fused<kDenseDiceGrad>(a, groups, st);
    else if (groups) launch_fused<kDenseCeGrad>(a, groups, st);
    else if (dice) hipLaunchKernelGGL(dense_bwd_kernel<true>, grid, dim3(256), 0, st, a, nchunk);
    else hipLaunchKernelGGL(dense_bwd_kernel<false>, grid, dim3(256), 0, st, a, nchunk);
    return check_launch("dense backward");
  }
  if (work) {  // no planes: the reduction alone writes zero losses
    if (groups) {
      launch_fused<kDenseCe>(a, groups, st);
      planes = a.B * groups;
      nchunk = ceil_div(a.HW, kCntCells);
    } else if (dice) {
      hipLaunchKernelGGL(dense_fwd_kernel<true>, grid, dim3(256), 0, st, a, nchunk);
    } else {
      hipLaunchKernelGGL(dense_fwd_kernel<false>, grid, dim3(256), 0, st, a, nchunk);
    }
    int rc = check_launch("dense forward");
    if (rc) return rc;
  }
  const dim3 rgrid((unsigned)a.L);
  if (dice) hipLaunchKernelGGL(dense_reduce_kernel<true>, rgrid, dim3(256), 0, st, a, planes, nchunk);
  else hipLaunchKernelGGL(dense_reduce_kernel<false>, rgrid, dim3(256), 0, st, a, planes, nchunk);
  return check_launch("dense reduce");
}

size_t dense_partials_bytes(int64_t L, int64_t B, int64_t C, int64_t HW, int64_t groups, bool dice) {
  if (groups) return (size_t)(L * B * groups) * (size_t)ceil_div(HW, kCntCells) * 8;
  return (size_t)(L * B * C) * (size_t)ceil_div(HW, kDenseChunk) * (dice ? 3 : 1) * 8;
}

}  // namespace ml
