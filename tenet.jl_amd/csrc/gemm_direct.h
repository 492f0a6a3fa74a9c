// The contraction kernels' inner part: a complex gather-GEMM on MFMA whose
// operands go from memory straight into the matrix instructions' registers.
//
//   D(i, j) = sum_k X(i, k) Y(j, k)
//
// Lane l of a 16x16x4 MFMA holds X(i = l % 16, k = l / 16) and Y(j = l % 16,
// k = l / 16), so each lane gathers exactly the elements it feeds: no LDS
// tile, no barrier in the K loop, and every load of a K step is independent.
// A complex FP64 block step is four MFMAs of 64 cycles (FP32: 32), against
// one 16-byte (8-byte) load per lane and operand block, so the matrix cores
// stay the bound while the re-reads of X and Y by neighbouring waves hit L1
// and L2.  (Staged through LDS with a barrier pair per K step of 16, the
// same products ran at 12 TFLOP/s for complex128 512x512x512 and 42 at
// 2048^3; direct, 49 and 70, of 72 that a large real FP64 GEMM reaches.)
#pragma once
#include "internal.h"

namespace tenet {

typedef double d4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

template <typename R>
struct Acc4;
template <>
struct Acc4<double> {
  using T = d4v;
};
template <>
struct Acc4<float> {
  using T = f4v;
};

__device__ __forceinline__ d4v mfma16x16x4(double a, double b, d4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4v mfma16x16x4(float a, float b, f4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// TI x TJ MFMA blocks per wave (i, j); result register r of lane l holds
// D(i, j = l % 16) with i = 4 * (l / 16) + r for FP32 and 4 * r + l / 16 for
// FP64.
template <typename R, int TI, int TJ>
struct BlockAcc {
  using V4 = typename Acc4<R>::T;
  V4 r[TI][TJ], i[TI][TJ];
};

// The element offsets of one operand: row i (or column j), contracted index
// k, batch entry z.  AFF: each is index * stride, else it comes from a table.
template <bool AFF>
struct Offsets {
  const int64_t* table;
  int64_t stride;
  __device__ __forceinline__ int64_t operator[](int64_t i) const {
    if constexpr (AFF)
      return i * stride;
    else
      return table[i];
  }
};

// Two neighbouring entries of a complex64 operand, loaded at once (rows of odd
// length leave them 8-byte aligned).
typedef float f4pair __attribute__((ext_vector_type(4), aligned(8)));

// acc = sum over this wave's share of k in [k_lo, k_hi) for the blocks at
// rows i0.. (of I) and columns j0.. (of J): WK waves take the K steps of 4
// round robin (this one is number wk), U steps per load group, the next
// group's loads in flight during the current group's products.  Rows and
// columns past the edge read the last valid one (their results are never
// stored); k past the end contributes zeros.
//
// PX / PY (complex64): that operand's entries k, k + 1 (k even) are adjacent,
// and each lane takes them with one 16-byte load.  A lane group then covers
// k = 2 g, 2 g + 1 of a span of 8 instead of k = g of spans of 4; the sum does
// not care which lane group holds which k.  An operand read along its rows
// costs one cache-line access per row and load whatever the width, so this
// halves the accesses that bound it.
template <typename S2, typename R, int TI, int TJ, int WK, int U, bool AFF, bool PX, bool PY>
__device__ __forceinline__ void direct_accumulate(const S2* __restrict__ X, const S2* __restrict__ Y,
                                                  const Offsets<AFF>& rowX, const Offsets<AFF>& kX,
                                                  const Offsets<AFF>& rowY, const Offsets<AFF>& kY, int64_t i0,
                                                  int64_t I, int64_t j0, int64_t J, int64_t k_lo, int64_t k_hi,
                                                  int wk, bool conjX, bool conjY, BlockAcc<R, TI, TJ>& acc) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const S2* px[TI];
  const S2* py[TJ];
#pragma unroll
  for (int a = 0; a < TI; ++a) px[a] = X + rowX[min(i0 + 16 * a + l16, I - 1)];
#pragma unroll
  for (int b = 0; b < TJ; ++b) py[b] = Y + rowY[min(j0 + 16 * b + l16, J - 1)];
#pragma unroll
  for (int a = 0; a < TI; ++a)
#pragma unroll
    for (int b = 0; b < TJ; ++b) {
      acc.r[a][b] = typename BlockAcc<R, TI, TJ>::V4{0, 0, 0, 0};
      acc.i[a][b] = typename BlockAcc<R, TI, TJ>::V4{0, 0, 0, 0};
    }
  constexpr bool PAIR = PX || PY;
  static_assert(!PAIR || (U == 2 && sizeof(S2) == 8), "pairs: two steps per group, complex64");
  struct Group {
    S2 x[U][TI], y[U][TJ];
  };
  struct KOff {
    int64_t x[U], y[U];
  };
  constexpr int CK = 4 * WK * U;                               // k range of one group over the WK waves
  constexpr int KU = PAIR ? 1 : 4 * WK;                        // k distance of a lane's steps
  const int64_t kb = k_lo + (PAIR ? 8 * wk + 2 * g : 4 * wk + g);  // this lane's first k
  const int64_t k_last = k_hi - 1;
  auto offs = [&](int64_t c, KOff& o) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = c * CK + u * KU + kb;
      // a pair ends at the last entry: past it the second of the two is the
      // one wanted (tail)
      if (!PX || u == 0) o.x[u] = kX[min(k, PX ? k_last - 1 : k_last)];
      if (!PY || u == 0) o.y[u] = kY[min(k, PY ? k_last - 1 : k_last)];
      // opaque: otherwise every (block, step) address of the affine form
      // becomes a 64-bit induction variable of its own, 80 registers more
      // and half the resident waves
      if constexpr (AFF) {
        if (!PX || u == 0) asm("" : "+v"(o.x[u]));
        if (!PY || u == 0) asm("" : "+v"(o.y[u]));
      }
    }
  };
  auto load2 = [](const S2* q, S2& e0, S2& e1) {
    const f4pair v = *reinterpret_cast<const f4pair*>(q);
    e0.x = v[0];
    e0.y = v[1];
    e1.x = v[2];
    e1.y = v[3];
  };
  auto load = [&](const KOff& o, Group& f) {
    if constexpr (PX) {
#pragma unroll
      for (int a = 0; a < TI; ++a) load2(px[a] + o.x[0], f.x[0][a], f.x[U - 1][a]);
    }
    if constexpr (PY) {
#pragma unroll
      for (int b = 0; b < TJ; ++b) load2(py[b] + o.y[0], f.y[0][b], f.y[U - 1][b]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (!PX) {
#pragma unroll
        for (int a = 0; a < TI; ++a) f.x[u][a] = px[a][o.x[u]];
      }
      if constexpr (!PY) {
#pragma unroll
        for (int b = 0; b < TJ; ++b) f.y[u][b] = py[b][o.y[u]];
      }
    }
  };
  const R sx = conjX ? (R)-1 : (R)1, sy = conjY ? (R)-1 : (R)1;
  auto mul = [&](int64_t c, const Group& f, bool tail) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = c * CK + u * KU + kb;
      const bool in = !tail || k < k_hi;
      const bool second = PAIR && tail && u == 0 && k == k_last;  // the pair loaded was (k - 1, k)
      R xr[TI], xi[TI], yr[TJ], yi[TJ];
#pragma unroll
      for (int a = 0; a < TI; ++a) {
        const S2 v = PX && second ? f.x[U - 1][a] : f.x[u][a];
        xr[a] = in ? (R)v.x : (R)0;
        xi[a] = in ? sx * (R)v.y : (R)0;
      }
#pragma unroll
      for (int b = 0; b < TJ; ++b) {
        const S2 v = PY && second ? f.y[U - 1][b] : f.y[u][b];
        yr[b] = in ? (R)v.x : (R)0;
        yi[b] = in ? sy * (R)v.y : (R)0;
      }
#pragma unroll
      for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) acc.r[a][b] = mfma16x16x4(xr[a], yr[b], acc.r[a][b]);
#pragma unroll
      for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) acc.i[a][b] = mfma16x16x4(xr[a], yi[b], acc.i[a][b]);
#pragma unroll
      for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) acc.r[a][b] = mfma16x16x4(-xi[a], yi[b], acc.r[a][b]);
#pragma unroll
      for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) acc.i[a][b] = mfma16x16x4(xi[a], yr[b], acc.i[a][b]);
    }
  };
  const int64_t len = k_hi - k_lo;
  if (len <= 0) return;
  const int64_t nfull = len / CK, nc = (len + CK - 1) / CK;
  Group f0, f1;
  KOff o0, o1;
  offs(0, o0);
  offs(1, o1);
  load(o0, f0);
  int64_t c = 0;
  for (; c + 2 <= nfull; c += 2) {  // group c in f0, group c + 1's offsets in o1
    load(o1, f1);
    offs(c + 2, o0);
    mul(c, f0, false);
    load(o0, f0);
    offs(c + 3, o1);
    mul(c + 1, f1, false);
  }
  // at most one whole and one partial group are left
  if (c < nc) {
    const bool two = c + 1 < nc;
    if (two) load(o1, f1);
    mul(c, f0, true);
    if (two) mul(c + 1, f1, true);
  }
}

// Fold the sums of WK waves sharing one set of blocks into wave 0, pairwise
// in a fixed order through `red` (WK / 2 * TI * TJ * 512 values per set of
// waves).  All waves of the workgroup call this.
template <typename R, int TI, int TJ, int WK>
__device__ __forceinline__ void direct_fold(R* __restrict__ red, int wk, BlockAcc<R, TI, TJ>& acc) {
  constexpr int V = TI * TJ * 8 * 64;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = WK / 2; h >= 1; h /= 2) {
    R* o = red + (size_t)(wk % h) * V + lane;
    if (wk >= h && wk < 2 * h) {
#pragma unroll
      for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[((a * TJ + b) * 8 + r) * 64] = acc.r[a][b][r];
            o[((a * TJ + b) * 8 + 4 + r) * 64] = acc.i[a][b][r];
          }
    }
    __syncthreads();
    if (wk < h) {
#pragma unroll
      for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            acc.r[a][b][r] += o[((a * TJ + b) * 8 + r) * 64];
            acc.i[a][b][r] += o[((a * TJ + b) * 8 + 4 + r) * 64];
          }
    }
    __syncthreads();
  }
}

struct Scalars {
  double ar, ai, br, bi;  // C = alpha D + beta C
};

template <typename S2>
__device__ __forceinline__ void store_scaled(S2* __restrict__ o, double vr, double vi, const Scalars& sc) {
  double outr = sc.ar * vr - sc.ai * vi, outi = sc.ar * vi + sc.ai * vr;
  if (sc.br != 0.0 || sc.bi != 0.0) {
    const S2 old = *o;
    outr += sc.br * (double)old.x - sc.bi * (double)old.y;
    outi += sc.br * (double)old.y + sc.bi * (double)old.x;
  }
  S2 w;
  w.x = outr;
  w.y = outi;
  *o = w;
}

// C's entries of this wave's blocks; j runs over the lanes, so with C
// adjacent along j a store instruction writes 16 neighbours per row.
template <typename S2, typename R, int TI, int TJ, bool AFF>
__device__ __forceinline__ void direct_store(S2* __restrict__ C, const Offsets<AFF>& rowC, const Offsets<AFF>& colC,
                                             int64_t i0, int64_t I, int64_t j0, int64_t J, const Scalars& sc,
                                             const BlockAcc<R, TI, TJ>& acc) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int b = 0; b < TJ; ++b) {
    const int64_t j = j0 + 16 * b + l16;
    if (j >= J) continue;
    S2* Cj = C + colC[j];
#pragma unroll
    for (int a = 0; a < TI; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i = i0 + 16 * a + ((sizeof(R) == 8) ? (r * 4 + g) : (g * 4 + r));
        if (i < I) store_scaled<S2>(Cj + rowC[i], (double)acc.r[a][b][r], (double)acc.i[a][b][r], sc);
      }
  }
}

}  // namespace tenet
