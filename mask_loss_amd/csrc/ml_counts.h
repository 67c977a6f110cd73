// The target pixels of one low-resolution cell, taken by T threads: the
// building block of the label-count kernels (s > 1).
#pragma once

#include "ml_internal.h"

namespace ml {

constexpr int kCntCells = 256;              // cells per workgroup: four 64-cell blocks
constexpr int kCntThreads = 4 * kCntCells;

// S = s for the unrolled forms 2 and 4, else 0.  Thread T c + k takes every
// T-th target row of cell c, from row k (T = 2 only for S = 2).
template <int S, int T = 4>
struct CellLabels {
  int64_t lab[S ? S : 1];
  const int64_t* src;  // the cell's first pixel
  int64_t Wt;
  int s, sub;
  bool in;             // a cell of the map
  bool whole = false;  // every pixel of the cell carries lab[0]
  bool first = true;   // ... and the wave's first cell does not carry that label all over, too

  // vec: the map starts on a 16-byte boundary (even s keeps pixel pairs there)
  __device__ __forceinline__ void load(const int64_t* targets, int64_t b, int64_t Ht, int64_t Wt_, int64_t W,
                                       int64_t HW, int64_t s_, int64_t cell, bool vec) {
    in = cell < HW;
    s = S ? S : (int)s_;
    sub = threadIdx.x & (T - 1);
    Wt = Wt_;
    const int64_t ci = in ? cell / W : 0, cj = in ? cell - ci * W : 0;
    src = targets + (b * Ht + ci * s) * Wt + cj * s;
    if constexpr (S != 0) {
      if (in && sub < S) {
        const int64_t* p = src + sub * Wt;
        if (vec) {
#pragma unroll
          for (int k = 0; k < S; k += 2) {
            const longlong2 v = *(const longlong2*)(p + k);
            lab[k] = v.x;
            lab[k + 1] = v.y;
          }
        } else {
#pragma unroll
          for (int k = 0; k < S; ++k) lab[k] = p[k];
        }
      }
    }
  }
  // after load, by the whole wave
  __device__ __forceinline__ void settle() {
    if constexpr (S != 0) {
      const int lane = threadIdx.x & 63;
      const bool act = in && sub < S;
      const int64_t l0 = __shfl(act ? lab[0] : 0, lane & ~(T - 1), 64);
      bool same = !act || lab[0] == l0;
#pragma unroll
      for (int k = 1; k < S; ++k) same = same && (!act || lab[k] == l0);
      const uint64_t m = __ballot(same);
      constexpr uint64_t all = (1u << T) - 1u;
      whole = in && ((m >> (lane & ~(T - 1))) & all) == all;
      const int64_t lw = __shfl(lab[0], 0, 64);
      first = lane == 0 || (m & all) != all || lab[0] != lw;
    }
  }
  // f(label, n, single): this thread's pixels as runs of one label; single:
  // the cell's only one
  template <class F>
  __device__ __forceinline__ void runs(F&& f) const {
    if constexpr (S != 0) {
      if (whole) {
        if (sub == 0) f(lab[0], (uint32_t)(S * S), true);
      } else if (in && sub < S) {
        uint32_t n = 1;
#pragma unroll
        for (int k = 1; k < S; ++k) {
          if (lab[k] != lab[k - 1]) {
            f(lab[k - 1], n, false);
            n = 0;
          }
          ++n;
        }
        f(lab[S - 1], n, false);
      }
    } else if (in) {
      for (int dy = sub; dy < s; dy += T) {
        const int64_t* p = src + dy * Wt;
        int64_t run = p[0];
        uint32_t n = 1;
        for (int dx = 1; dx < s; ++dx) {
          const int64_t v = p[dx];
          if (v != run) {
            f(run, n, false);
            run = v;
            n = 0;
          }
          ++n;
        }
        f(run, n, false);
      }
    }
  }
};

// Add n pixels of row r (of nr) to cell cl of the LDS tile [4][nr][64] of CW bytes each.
template <int CW>
__device__ __forceinline__ void tile_add(unsigned char* tile, int nr, int r, int cl, uint32_t n, bool single) {
  const uint32_t e = (uint32_t)(((cl >> 6) * nr + r) * kCountCells + (cl & (kCountCells - 1)));
  if (single) {
    if constexpr (CW == 1) tile[e] = (unsigned char)n;
    else ((uint16_t*)tile)[e] = (uint16_t)n;
  } else if constexpr (CW == 1) {
    atomicAdd((uint32_t*)tile + (e >> 2), n << ((e & 3u) * 8u));
  } else {
    atomicAdd((uint32_t*)tile + (e >> 1), n << ((e & 1u) * 16u));
  }
}

}  // namespace ml
