// K1: pairwise tensor contraction as a gather-GEMM on CDNA4 MFMA.
//
// A binary contraction, once matricised, is a (batched) GEMM
//   C[m, n, z] = sum_k A[m, k, z] * B[k, n, z].
// The permutation that matricisation needs is never materialised: the host
// planner turns every label class into a table of element offsets
// (rowA[m], kA[k], bA[z], ...), and the kernels gather straight from the
// caller's strided tensors (gemm_direct.h).  Complex products run as four
// real MFMA products (no 3M trick: it cancels badly at the 1e-8 accuracy this
// path is held to).
#include "../../include/tenet_hip.h"
#include "internal.h"
#include "gemm_direct.h"

#include <algorithm>
#include <type_traits>

namespace tenet {

// ---- one contraction per launch -----------------------------------------------
// Workgroup shapes of the direct kernel: four waves, either all on the same
// TI x TJ blocks with the K steps dealt round robin (WK = 4: short chains and
// four times the waves where a product has few tiles), or side by side along
// j (WK = 1: a short K has no steps to deal).
struct DirectCfg {
  int ti, tj, wj, wk;
  double eff;  // share of its modelled rate that the shape reaches (fitted, see choose_direct)
};
enum { D16 = 0, D16x32, D32, D32x64, S32, S16, DIRECT_CFGS, ELEMENTS = DIRECT_CFGS };
static constexpr DirectCfg kDirect[DIRECT_CFGS] = {
    {1, 1, 1, 4, 0.65}, {1, 2, 1, 4, 0.75}, {2, 2, 1, 4, 0.75},
    {2, 4, 1, 4, 0.80}, {2, 2, 4, 1, 0.85}, {1, 2, 4, 1, 0.75}};

struct DirectArgs {
  const void* X;
  const void* Y;
  void* C;
  // offsets of rowX, kX, batchX, rowY, kY, batchY, rowC, colC, batchC
  const int64_t* tab[9];
  int64_t st[9];
  int64_t I, J, K;
  int64_t tiles_i, tiles_j;
  int conjX, conjY;
  Scalars sc;
};

// Map a physical workgroup id to a logical tile so that the tiles one XCD
// receives (ids congruent mod 8 are dispatched to the same XCD) are
// neighbours in the tile grid and share X / Y panels in that XCD's L2.
__device__ __forceinline__ int64_t xcd_remap(int64_t pid, int64_t total) {
  constexpr int64_t NXCD = 8;
  if (total % NXCD != 0) return pid;
  return (pid % NXCD) * (total / NXCD) + pid / NXCD;
}

template <typename S2, typename R, int TI, int TJ, int WJ, int WK, int U, bool AFF, bool PX, bool PY>
__global__ __launch_bounds__(256, 2) void gemm_direct_kernel(DirectArgs p) {
  static_assert(WJ * WK == 4, "four waves");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave % WK, wj = wave / WK;
  const int64_t total = gridDim.x, id = xcd_remap((int64_t)blockIdx.x, total);
  const int64_t per = p.tiles_i * p.tiles_j;
  const int64_t z = per == total ? 0 : id / per, t = id - z * per;
  const int64_t tj = t / p.tiles_i, ti = t - tj * p.tiles_i;
  const int64_t i0 = ti * (16 * TI), j0 = (tj * WJ + wj) * (16 * TJ);
  auto off = [&](int k) { return Offsets<AFF>{p.tab[k], p.st[k]}; };
  const S2* X = static_cast<const S2*>(p.X) + off(2)[z];
  const S2* Y = static_cast<const S2*>(p.Y) + off(5)[z];
  BlockAcc<R, TI, TJ> acc;
  direct_accumulate<S2, R, TI, TJ, WK, U, AFF, PX, PY>(X, Y, off(0), off(1), off(3), off(4), i0, p.I, j0, p.J, 0, p.K, wk,
                                               p.conjX != 0, p.conjY != 0, acc);
  if constexpr (WK > 1) {
    __shared__ R red[WK / 2 * TI * TJ * 512];
    direct_fold<R, TI, TJ, WK>(red, wk, acc);
    if (wk > 0) return;
  }
  direct_store<S2, R, TI, TJ, AFF>(static_cast<S2*>(p.C) + off(8)[z], off(6), off(7), i0, p.I, j0, p.J, p.sc, acc);
}

// One thread per output element, for products of so few terms that an MFMA
// block would be mostly padding (permutations, Hadamard scalings): consecutive
// threads take consecutive entries of the index class whose entries of C are
// closest (order 0: m, 1: n, 2: batch).
template <typename S2, typename R, typename IT>
__global__ __launch_bounds__(256) void gemm_elements_kernel(GemmTables t, const S2* __restrict__ A,
                                                            const S2* __restrict__ B, S2* __restrict__ C, IT total,
                                                            IT ext0, IT ext1, int K, int order, int conjA, int conjB,
                                                            Scalars sc) {
  const R sa = conjA ? (R)-1 : (R)1, sb = conjB ? (R)-1 : (R)1;
  for (IT e = (IT)blockIdx.x * 256 + threadIdx.x; e < total; e += (IT)gridDim.x * 256) {
    const IT rest = e / ext0, i0 = e - rest * ext0;
    const IT i2 = rest / ext1, i1 = rest - i2 * ext1;
    const int64_t m = order == 0 ? i0 : i1;
    const int64_t n = order == 0 ? i1 : (order == 1 ? i0 : i2);
    const int64_t z = order == 2 ? i0 : i2;
    const S2* a0 = A + (t.rowA[m] + t.bA[z]);
    const S2* b0 = B + (t.colB[n] + t.bB[z]);
    R cr = 0, ci = 0;
    for (int k = 0; k < K; ++k) {
      const S2 a = a0[t.kA[k]], b = b0[t.kB[k]];
      const R ar = (R)a.x, ai = sa * (R)a.y, br = (R)b.x, bi = sb * (R)b.y;
      cr += ar * br - ai * bi;
      ci += ar * bi + ai * br;
    }
    store_scaled<S2>(C + (t.rowC[m] + t.colC[n] + t.bC[z]), (double)cr, (double)ci, sc);
  }
}

// The workgroup shape with the least modelled time, in cycles of one CU: per
// K step the larger of its MFMAs (64 cycles each in FP64, 32 in FP32) and
// its operand loads (24 cycles of the CU's address unit per wave and block,
// twice that where 16 lanes read 16 rows instead of neighbours, one entry
// each), over the
// rounds the 256 CUs need, plus the epilogue of a tile.  On 45 measured shapes
// (K 4..3840, 24 x 38 to 590000 x 20, both types) the choice is 2% slower than
// the best of the six in the mean, 26% at worst (complex64 300 x 600 x 300,
// 11.8 against 9.4 us).  From K = 128 on the WK = 1 shapes never won.
static int choose_direct(double cyc, int64_t I, int64_t J, int64_t K, int64_t batch, bool x_adj, bool y_adj) {
  const double clx = x_adj ? 24 : 48, cly = y_adj ? 24 : 48;
  int best = 0;
  double best_t = 0.0;
  for (int c = 0; c < DIRECT_CFGS; ++c) {
    const DirectCfg& f = kDirect[c];
    if (f.wk == 1 && K >= 128) continue;
    const int64_t ei = 16 * f.ti, ej = 16 * f.tj * f.wj;
    const double tiles = (double)((I + ei - 1) / ei) * (double)((J + ej - 1) / ej) * (double)batch;
    const double rounds = tiles > 1024 ? tiles / 256 : std::ceil(tiles / 256);
    const double steps = (double)((K + 4 * f.wk - 1) / (4 * f.wk));
    const double step = std::max(4 * cyc * f.ti * f.tj, 4 * (f.ti * clx + f.tj * cly));
    const double t = rounds * (steps * step / f.eff + 200.0 * f.ti * f.tj);
    if (c == 0 || t < best_t) {
      best = c;
      best_t = t;
    }
  }
  return best;
}

// every entry pair (2 i, 2 i + 1) of a K table adjacent, and, with an odd
// length, the last two as well
bool k_pairs(const std::vector<int64_t>& t) {
  const size_t n = t.size();
  if (n < 2) return false;
  for (size_t k = 0; k + 1 < n; k += 2)
    if (t[k + 1] != t[k] + 1) return false;
  return n % 2 == 0 || t[n - 1] == t[n - 2] + 1;
}

void gemm_form(const std::vector<int64_t> v[9], int64_t M, int64_t N, int64_t K, int64_t batch, int dtype, int prec,
               GemmForm* f) {
  auto stride_of = [](const std::vector<int64_t>& t, int64_t* st) {
    *st = t.size() > 1 ? t[1] - t[0] : 0;
    for (size_t i = 0; i < t.size(); ++i)
      if (t[i] != (int64_t)i * *st) return false;
    return true;
  };
  f->affine = 1;
  for (int i = 0; i < 9; ++i)
    if (!stride_of(v[i], &f->st[i])) f->affine = 0;
  auto gap = [&](int i) { return v[i].size() > 1 ? std::llabs(v[i][1] - v[i][0]) : INT64_MAX; };
  const int64_t gm = gap(6), gn = gap(7), gz = gap(8);
  f->order = (gm <= gn && gm <= gz) ? 0 : (gn <= gz ? 1 : 2);
  f->j_is_m = gm <= gn ? 1 : 0;
  // up to two outputs per gathered row: 160000 x 8 by 8 x 2 in 9.4 us either
  // way, a Hadamard scaling of 51200 entries 2.1 us (MFMA blocks 4.5), a dot
  // of 8 terms per row over 4e6 rows 115 us (434); with three or more columns
  // the MFMA blocks win (160000 x 4 by 4 x 4: 7.4 against 11.8 us)
  if (K <= 8 && std::min(M, N) <= 2) {
    f->cfg = ELEMENTS;
    return;
  }
  f->pair_a = k_pairs(v[1]);
  f->pair_b = k_pairs(v[3]);
  const bool wide = dtype == TENET_C64;  // pairs of entries per load
  const bool a_adj = gap(0) == 1 || M == 1 || (wide && f->pair_a);
  const bool b_adj = gap(4) == 1 || N == 1 || (wide && f->pair_b);
  const double cyc = dtype == TENET_C128 && prec == TENET_PREC_NATIVE ? 64 : 32;
  if (f->j_is_m)
    f->cfg = choose_direct(cyc, N, M, K, batch, b_adj, a_adj);
  else
    f->cfg = choose_direct(cyc, M, N, K, batch, a_adj, b_adj);
}

template <typename S2, typename R, int TI, int TJ, int WJ, int WK, int U, bool PX, bool PY>
static int launch_direct_p(const DirectArgs& p, bool affine, unsigned total, hipStream_t s) {
  if (affine)
    hipLaunchKernelGGL((gemm_direct_kernel<S2, R, TI, TJ, WJ, WK, U, true, PX, PY>), dim3(total), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((gemm_direct_kernel<S2, R, TI, TJ, WJ, WK, U, false, PX, PY>), dim3(total), dim3(256), 0, s, p);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

template <typename S2, typename R, int TI, int TJ, int WJ, int WK, int U>
static int launch_direct(DirectArgs& p, const GemmLaunch& g, hipStream_t s) {
  p.tiles_i = (p.I + 16 * TI - 1) / (16 * TI);
  p.tiles_j = (p.J + 16 * TJ * WJ - 1) / (16 * TJ * WJ);
  const double total = (double)p.tiles_i * (double)p.tiles_j * (double)g.batch;
  if (total > 0x7fffffffLL) {
    set_error("contraction too large for one launch");
    return TENET_ERR_UNSUPPORTED;
  }
  const bool aff = g.form->affine != 0;
  const unsigned n = (unsigned)total;
  if constexpr (sizeof(S2) == 8) {
    const bool px = g.form->j_is_m ? g.form->pair_b : g.form->pair_a;
    const bool py = g.form->j_is_m ? g.form->pair_a : g.form->pair_b;
    if (px && py) return launch_direct_p<S2, R, TI, TJ, WJ, WK, 2, true, true>(p, aff, n, s);
    if (px) return launch_direct_p<S2, R, TI, TJ, WJ, WK, 2, true, false>(p, aff, n, s);
    if (py) return launch_direct_p<S2, R, TI, TJ, WJ, WK, 2, false, true>(p, aff, n, s);
  }
  return launch_direct_p<S2, R, TI, TJ, WJ, WK, U, false, false>(p, aff, n, s);
}

template <typename S2, typename R, typename IT>
static int launch_elements(const GemmLaunch& g, const Scalars& sc, hipStream_t s) {
  const int order = g.form->order;
  const int64_t total = g.M * g.N * g.batch;
  const int64_t ext0 = order == 0 ? g.M : (order == 1 ? g.N : g.batch), ext1 = order == 0 ? g.N : g.M;
  const int64_t blocks = std::min<int64_t>((total + 255) / 256, 1 << 20);
  hipLaunchKernelGGL((gemm_elements_kernel<S2, R, IT>), dim3((unsigned)blocks), dim3(256), 0, s, g.t,
                     (const S2*)g.A, (const S2*)g.B, (S2*)g.C, (IT)total, (IT)ext0, (IT)ext1, (int)g.K, order,
                     g.conjA, g.conjB, sc);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

template <typename S2, typename R>
static int launch_gemm_t(const GemmLaunch& g, hipStream_t s) {
  const Scalars sc{g.alpha_re, g.alpha_im, g.beta_re, g.beta_im};
  if (g.form->cfg == ELEMENTS) {
    if (g.M * g.N * g.batch <= (int64_t)INT32_MAX) return launch_elements<S2, R, uint32_t>(g, sc, s);
    return launch_elements<S2, R, int64_t>(g, sc, s);
  }
  // i and j are A's and B's free indices, or B's and A's when C's entries are
  // adjacent along m (a store instruction then writes neighbours)
  DirectArgs p{};
  p.C = g.C;
  p.K = g.K;
  p.sc = sc;
  const int64_t* tab[9] = {g.t.rowA, g.t.kA, g.t.bA, g.t.kB, g.t.colB, g.t.bB, g.t.rowC, g.t.colC, g.t.bC};
  static const int from[2][9] = {{0, 1, 2, 4, 3, 5, 6, 7, 8}, {4, 3, 5, 0, 1, 2, 7, 6, 8}};
  const int jm = g.form->j_is_m;
  for (int k = 0; k < 9; ++k) {
    p.tab[k] = tab[from[jm][k]];
    p.st[k] = g.form->st[from[jm][k]];
  }
  p.X = jm ? g.B : g.A;
  p.Y = jm ? g.A : g.B;
  p.conjX = jm ? g.conjB : g.conjA;
  p.conjY = jm ? g.conjA : g.conjB;
  p.I = jm ? g.N : g.M;
  p.J = jm ? g.M : g.N;
  switch (g.form->cfg) {
    case D16:
      return launch_direct<S2, R, 1, 1, 1, 4, 1>(p, g, s);
    case D16x32:
      return launch_direct<S2, R, 1, 2, 1, 4, 2>(p, g, s);
    case D32:
      return launch_direct<S2, R, 2, 2, 1, 4, 1>(p, g, s);
    case D32x64:
      return launch_direct<S2, R, 2, 4, 1, 4, 1>(p, g, s);
    case S32:
      return launch_direct<S2, R, 2, 2, 4, 1, 1>(p, g, s);
    default:
      return launch_direct<S2, R, 1, 2, 4, 1, 2>(p, g, s);
  }
}

int launch_split_gemm(const GemmLaunch& g, int dtype, int prec, hipStream_t s, void* ws, size_t ws_bytes);

int launch_gemm_c128(const GemmLaunch& g, int prec, hipStream_t s, void* ws, size_t ws_bytes) {
  if (g.M == 0 || g.N == 0 || g.batch == 0) return TENET_OK;
  switch (prec) {
    case TENET_PREC_NATIVE:
      return launch_gemm_t<double2, double>(g, s);
    case TENET_PREC_FP32:
      return launch_gemm_t<double2, float>(g, s);
    case TENET_PREC_SPLIT_BF16:
    case TENET_PREC_SPLIT_FP16:
      return launch_split_gemm(g, TENET_C128, prec, s, ws, ws_bytes);
    case TENET_PREC_SPLIT_I8:
    case TENET_PREC_SPLIT_I8_FAST:
      return launch_split8_gemm(g, TENET_C128, prec, s, ws, ws_bytes);
  }
  set_error("unknown precision");
  return TENET_ERR_ARG;
}

int launch_gemm_c64(const GemmLaunch& g, int prec, hipStream_t s, void* ws, size_t ws_bytes) {
  if (g.M == 0 || g.N == 0 || g.batch == 0) return TENET_OK;
  switch (prec) {
    case TENET_PREC_NATIVE:
    case TENET_PREC_FP32:
      return launch_gemm_t<float2, float>(g, s);
    case TENET_PREC_SPLIT_BF16:
    case TENET_PREC_SPLIT_FP16:
      return launch_split_gemm(g, TENET_C64, prec, s, ws, ws_bytes);
    case TENET_PREC_SPLIT_I8:
    case TENET_PREC_SPLIT_I8_FAST:
      return launch_split8_gemm(g, TENET_C64, prec, s, ws, ws_bytes);
  }
  set_error("unknown precision");
  return TENET_ERR_ARG;
}

// ---- grouped persistent launch ------------------------------------------------
// Work units (problem, tile, K chunk) are sorted by decreasing cost on the
// host; persistent workgroups take the next unit from a device counter, so
// the largest units start first and the tail is short (LPT order).  A tile
// whose K range is cut into chunks stores each chunk's partial tile, and a
// second kernel sums them in chunk order and writes C, so results do not
// depend on the schedule.
//
// A unit's workgroup shape: TI x TJ blocks per wave, the four waves in a
// W x W arrangement over the tile (WK = 1) or all on one tile, dealing its K
// steps (WK = 4).
template <int TI_, int TJ_, int W_, int WK_>
struct UnitCfg {
  static constexpr int TI = TI_, TJ = TJ_, W = W_, WK = WK_, EDGE = 16 * TI * W;
  static_assert(TI == TJ && W * W * WK == 4, "square tiles, four waves");
};
using Tile64 = UnitCfg<2, 2, 2, 1>;
using Tile32 = UnitCfg<2, 2, 1, 4>;
using Tile16 = UnitCfg<1, 1, 1, 4>;
// LDS values of the K-split fold of the largest tile whose waves deal K
// (WK / 2 * TI * TJ * 512)
constexpr int FOLD_VALUES = Tile32::WK / 2 * Tile32::TI * Tile32::TJ * 512;
static_assert(FOLD_VALUES >= Tile16::WK / 2 * Tile16::TI * Tile16::TJ * 512, "fold buffer");

// Split-K partials: a result-holding thread stores its registers at
// ((wave * TI + i) * TJ + j) * 4 + r) * 64 + lane, as (re, im) pairs
// (grouped_reduce_kernel reads them back).
template <typename R, typename Cfg>
__device__ __forceinline__ void partial_store(R* __restrict__ part, int wave,
                                              const BlockAcc<R, Cfg::TI, Cfg::TJ>& acc) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < Cfg::TI; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::TJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t e = ((((int64_t)wave * Cfg::TI + i) * Cfg::TJ + j) * 4 + r) * 64 + lane;
        part[2 * e] = acc.r[i][j][r];
        part[2 * e + 1] = acc.i[i][j][r];
      }
}

template <typename S2, typename R, typename Cfg>
__device__ __forceinline__ void grouped_unit(const GroupedProblem& q, const uint64_t* __restrict__ ptrs,
                                             const GroupedUnit& u, R* __restrict__ partials, R* __restrict__ red) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = Cfg::WK == 1 ? 0 : wave, wi = Cfg::WK == 1 ? wave % Cfg::W : 0, wj = Cfg::WK == 1 ? wave / Cfg::W : 0;
  const bool holds = wk == 0;  // this wave ends with results
  const int64_t per_batch = (int64_t)q.tiles_m * q.tiles_n;
  const int64_t z = u.tile / per_batch;
  const int64_t t = u.tile - z * per_batch;
  const int64_t tm = t % q.tiles_m, tn = t / q.tiles_m;
  const int64_t k_lo = (int64_t)u.chunk * q.kc;
  const int64_t k_hi = std::min<int64_t>(q.K, k_lo + q.kc);
  // i and j are A's and B's free indices, or B's and A's when C's entries are
  // adjacent along m
  const bool jm = q.j_is_m != 0;
  const S2* A = reinterpret_cast<const S2*>(ptrs[3 * u.prob]) + q.t.bA[z];
  const S2* B = reinterpret_cast<const S2*>(ptrs[3 * u.prob + 1]) + q.t.bB[z];
  S2* C = reinterpret_cast<S2*>(ptrs[3 * u.prob + 2]) + q.t.bC[z];
  using Off = Offsets<false>;
  const int64_t I = jm ? q.N : q.M, J = jm ? q.M : q.N;
  const int64_t i0 = (jm ? tn : tm) * Cfg::EDGE + wi * 16 * Cfg::TI, j0 = (jm ? tm : tn) * Cfg::EDGE + wj * 16 * Cfg::TJ;
  BlockAcc<R, Cfg::TI, Cfg::TJ> acc;
  const Off rowX{jm ? q.t.colB : q.t.rowA, 0}, kX{jm ? q.t.kB : q.t.kA, 0};
  const Off rowY{jm ? q.t.rowA : q.t.colB, 0}, kY{jm ? q.t.kA : q.t.kB, 0};
  const bool cx = (jm ? q.conjB : q.conjA) != 0, cy = (jm ? q.conjA : q.conjB) != 0;
  auto accumulate = [&](auto px, auto py) {
    constexpr int U = decltype(px)::value || decltype(py)::value ? 2 : 1;
    direct_accumulate<S2, R, Cfg::TI, Cfg::TJ, Cfg::WK, U, false, decltype(px)::value, decltype(py)::value>(
        jm ? B : A, jm ? A : B, rowX, kX, rowY, kY, i0, I, j0, J, k_lo, k_hi, wk, cx, cy, acc);
  };
  using No = std::integral_constant<bool, false>;
  using Yes = std::integral_constant<bool, true>;
  if constexpr (sizeof(S2) == 8) {
    // bit 0: A's K entries come in adjacent pairs, bit 1: B's
    const int pairs = jm ? ((q.pairs & 1) << 1 | q.pairs >> 1) : q.pairs;
    switch (pairs) {
      case 1:
        accumulate(Yes{}, No{});
        break;
      case 2:
        accumulate(No{}, Yes{});
        break;
      case 3:
        accumulate(Yes{}, Yes{});
        break;
      default:
        accumulate(No{}, No{});
        break;
    }
  } else {
    accumulate(No{}, No{});
  }
  if constexpr (Cfg::WK > 1) direct_fold<R, Cfg::TI, Cfg::TJ, Cfg::WK>(red, wk, acc);
  const Off rowC{jm ? q.t.colC : q.t.rowC, 0}, colC{jm ? q.t.rowC : q.t.colC, 0};
  const Scalars one{1.0, 0.0, 0.0, 0.0};
  if (q.kchunks == 1) {
    if (holds) direct_store<S2, R, Cfg::TI, Cfg::TJ, false>(C, rowC, colC, i0, I, j0, J, one, acc);
  } else {
    // chunks of K: partials through memory, summed by the kernel behind this
    // one (inside it, every chunk's device-scope release and acquire wrote back
    // and invalidated the XCD's L2: twice the chunks cost a 200-problem batch
    // 718 -> 1648 us)
    constexpr int64_t TILE = (int64_t)Cfg::EDGE * Cfg::EDGE;
    R* part = partials + 2 * (q.part_base + u.tile * q.kchunks * TILE);
    if (holds) partial_store<R, Cfg>(part + 2 * (int64_t)u.chunk * TILE, wave, acc);
  }
}

// Sum the chunk partials of one split tile (blockIdx.x) in chunk order and
// store C.
template <typename S2, typename R, typename Cfg>
__device__ __forceinline__ void reduce_tile(const GroupedProblem& q, S2* __restrict__ Call, const GroupedUnit& u,
                                            const R* __restrict__ partials) {
  constexpr int64_t TILE = (int64_t)Cfg::EDGE * Cfg::EDGE;
  const int64_t per_batch = (int64_t)q.tiles_m * q.tiles_n;
  const int64_t z = u.tile / per_batch;
  const int64_t t = u.tile - z * per_batch;
  const int64_t tm = t % q.tiles_m, tn = t / q.tiles_m;
  const bool jm = q.j_is_m != 0;
  const R* part = partials + 2 * (q.part_base + u.tile * q.kchunks * TILE);
  S2* C = Call + q.t.bC[z];
  for (int e = threadIdx.x; e < (int)TILE; e += 256) {
    const int lane = e & 63, r = (e >> 6) & 3, blk = e >> 8;
    const int j = blk % Cfg::TJ, i = (blk / Cfg::TJ) % Cfg::TI, wave = blk / (Cfg::TI * Cfg::TJ);
    const int wi = wave % Cfg::W, wj = wave / Cfg::W;
    const int rr = sizeof(R) == 8 ? r * 4 + (lane >> 4) : (lane >> 4) * 4 + r;
    const int64_t gi = (jm ? tn : tm) * Cfg::EDGE + (wi * Cfg::TI + i) * 16 + rr;
    const int64_t gj = (jm ? tm : tn) * Cfg::EDGE + (wj * Cfg::TJ + j) * 16 + (lane & 15);
    const int64_t m = jm ? gj : gi, n = jm ? gi : gj;
    if (m >= q.M || n >= q.N) continue;
    R sr = 0, si = 0;
#pragma unroll 8
    for (int c = 0; c < q.kchunks; ++c) {  // fixed order: deterministic
      sr += part[2 * (c * TILE + e)];
      si += part[2 * (c * TILE + e) + 1];
    }
    S2 o;
    o.x = sr;
    o.y = si;
    C[q.t.rowC[m] + q.t.colC[n]] = o;
  }
}

template <typename S2, typename R>
__global__ __launch_bounds__(256) void grouped_reduce_kernel(const GroupedProblem* __restrict__ probs,
                                                             const GroupedUnit* __restrict__ tiles,
                                                             const uint64_t* __restrict__ ptrs,
                                                             const R* __restrict__ partials) {
  const GroupedUnit u = tiles[blockIdx.x];
  const GroupedProblem& q = probs[u.prob];
  S2* C = reinterpret_cast<S2*>(ptrs[3 * u.prob + 2]);
  if (q.shape == GROUPED_TILE_16)
    reduce_tile<S2, R, Tile16>(q, C, u, partials);
  else if (q.shape == GROUPED_TILE_32)
    reduce_tile<S2, R, Tile32>(q, C, u, partials);
  else
    reduce_tile<S2, R, Tile64>(q, C, u, partials);
}

// A GROUPED_SMALLK unit: output elements [tile * SMALLK_ELEMS, +SMALLK_ELEMS)
// of the flattened (m, n, z) space, the class q.order varying fastest (the
// one with C's smallest stride, so consecutive threads write consecutive
// addresses); each thread sums its K <= 8 products directly.  The element
// index is decoded in 32-bit arithmetic when the problem's element count
// fits (a 64-bit division is a long software sequence on the GPU; the
// Vidal layer's gate contraction spent most of its time there).
template <typename S2, typename R, typename IT>
__device__ __forceinline__ void smallk_elems(const GroupedProblem& q, const S2* __restrict__ A,
                                             const S2* __restrict__ B, S2* __restrict__ C, IT e0, IT e1, IT ext0,
                                             IT ext1) {
  const R sa = q.conjA ? (R)-1 : (R)1, sb = q.conjB ? (R)-1 : (R)1;
  for (IT e = e0 + (IT)threadIdx.x; e < e1; e += (IT)blockDim.x) {
    const IT i0 = e % ext0, rest = e / ext0;
    const IT i1 = rest % ext1, i2 = rest / ext1;
    int64_t m, n, z;
    if (q.order == 0) {
      m = i0;
      n = i1;
      z = i2;
    } else if (q.order == 1) {
      n = i0;
      m = i1;
      z = i2;
    } else {
      z = i0;
      m = i1;
      n = i2;
    }
    const int64_t oa = q.t.rowA[m] + q.t.bA[z], ob = q.t.colB[n] + q.t.bB[z];
    R cr = 0, ci = 0;
    // K <= 8, unrolled: the element loop stays the only loop of the unit
    // (the persistent loop around it must keep a single nested level)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (k < q.K) {
        const S2 a = A[oa + q.t.kA[k]];
        const S2 b = B[ob + q.t.kB[k]];
        const R ar = (R)a.x, ai = sa * (R)a.y, br = (R)b.x, bi = sb * (R)b.y;
        cr += ar * br - ai * bi;
        ci += ar * bi + ai * br;
      }
    }
    S2 o;
    o.x = cr;
    o.y = ci;
    C[q.t.rowC[m] + q.t.colC[n] + q.t.bC[z]] = o;
  }
}

template <typename S2, typename R>
__device__ __forceinline__ void grouped_smallk_unit(const GroupedProblem& q, const uint64_t* __restrict__ ptrs,
                                                    const GroupedUnit& u) {
  const S2* __restrict__ A = reinterpret_cast<const S2*>(ptrs[3 * u.prob]);
  const S2* __restrict__ B = reinterpret_cast<const S2*>(ptrs[3 * u.prob + 1]);
  S2* __restrict__ C = reinterpret_cast<S2*>(ptrs[3 * u.prob + 2]);
  const int64_t total = q.M * q.N * q.batch;
  const int64_t e0 = u.tile * SMALLK_ELEMS;
  const int64_t e1 = std::min<int64_t>(total, e0 + SMALLK_ELEMS);
  // extents in decode order: fastest, middle, slowest
  const int64_t ext0 = q.order == 0 ? q.M : (q.order == 1 ? q.N : q.batch);
  const int64_t ext1 = q.order == 0 ? q.N : q.M;
  if (total <= (int64_t)INT32_MAX)
    smallk_elems<S2, R, uint32_t>(q, A, B, C, (uint32_t)e0, (uint32_t)e1, (uint32_t)ext0, (uint32_t)ext1);
  else
    smallk_elems<S2, R, int64_t>(q, A, B, C, e0, e1, ext0, ext1);
}

template <typename S2, typename R>
__device__ __forceinline__ void grouped_gemm_body(const GroupedProblem* __restrict__ probs,
                                                  const GroupedUnit* __restrict__ units, int64_t nunits,
                                                  const uint64_t* __restrict__ ptrs, R* __restrict__ partials,
                                                  uint32_t* __restrict__ queue) {
  __shared__ R red[FOLD_VALUES];
  __shared__ uint32_t next;
  // Every branch below depends only on values that are uniform across the
  // workgroup and are made scalar with readfirstlane, so the loop compiles to
  // scalar control flow: each iteration takes exactly one unit from the queue
  // and every workgroup leaves once the queue is drained.
  for (;;) {
    // The thread index is re-read through an opaque copy every iteration.
    // Otherwise the optimiser sees "thread 0" as loop-invariant and threads
    // the loop latch on it (thread 0 back to the queue fetch, every other
    // thread straight back to the first barrier), which splits the barrier
    // instances and never fetches a new unit for the other lanes.
    unsigned tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    if (tid == 0) next = __hip_atomic_fetch_add(queue, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int64_t ui = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)next);
    __syncthreads();
    if (ui >= nunits) {
      // every workgroup fetches exactly one number past the units, so the
      // largest comes after all other fetches: its taker readies the queue for
      // the next launch
      if (ui == nunits + (int64_t)gridDim.x - 1 && tid == 0) *queue = 0u;
      break;
    }
    const GroupedUnit u = units[ui];
    const GroupedProblem& q = probs[u.prob];
    switch (q.shape) {
      case GROUPED_SMALLK:
        grouped_smallk_unit<S2, R>(q, ptrs, u);
        break;
      case GROUPED_TILE_16:
        grouped_unit<S2, R, Tile16>(q, ptrs, u, partials, red);
        break;
      case GROUPED_TILE_32:
        grouped_unit<S2, R, Tile32>(q, ptrs, u, partials, red);
        break;
      default:
        grouped_unit<S2, R, Tile64>(q, ptrs, u, partials, red);
        break;
    }
  }
}

__global__ __launch_bounds__(256, 3) void grouped_gemm_c64_kernel(const GroupedProblem* __restrict__ probs,
                                                                  const GroupedUnit* __restrict__ units,
                                                                  int64_t nunits, const uint64_t* __restrict__ ptrs,
                                                                  float* __restrict__ partials,
                                                                  uint32_t* __restrict__ queue) {
  grouped_gemm_body<float2, float>(probs, units, nunits, ptrs, partials, queue);
}
__global__ __launch_bounds__(256, 2) void grouped_gemm_c128_kernel(const GroupedProblem* __restrict__ probs,
                                                                const GroupedUnit* __restrict__ units, int64_t nunits,
                                                                const uint64_t* __restrict__ ptrs,
                                                                double* __restrict__ partials,
                                                                uint32_t* __restrict__ queue) {
  grouped_gemm_body<double2, double>(probs, units, nunits, ptrs, partials, queue);
}

int grouped_occupancy(int dtype) {
  int blocks = 0;
  hipError_t e;
  if (dtype == TENET_C128)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, grouped_gemm_c128_kernel, 256, 0);
  else
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, grouped_gemm_c64_kernel, 256, 0);
  if (e != hipSuccess || blocks < 1) return 1;
  return std::min(blocks, 8);
}

int launch_grouped_gemm(const GroupedLaunch& g, hipStream_t s) {
  if (g.nunits <= 0) return TENET_OK;
  const int64_t grid = std::max<int64_t>(1, std::min<int64_t>(g.nunits, g.grid));
  if (g.dtype == TENET_C128)
    hipLaunchKernelGGL(grouped_gemm_c128_kernel, dim3((unsigned)grid), dim3(256), 0, s, g.probs,
                       g.units, g.nunits, g.ptrs, (double*)g.partials, g.queue);
  else
    hipLaunchKernelGGL(grouped_gemm_c64_kernel, dim3((unsigned)grid), dim3(256), 0, s, g.probs,
                       g.units, g.nunits, g.ptrs, (float*)g.partials, g.queue);
  TENET_HIP_CHECK(hipGetLastError());
  if (g.nsplit > 0) {
    if (g.dtype == TENET_C128)
      hipLaunchKernelGGL((grouped_reduce_kernel<double2, double>), dim3((unsigned)g.nsplit), dim3(256), 0, s, g.probs,
                         g.split, g.ptrs, (const double*)g.partials);
    else
      hipLaunchKernelGGL((grouped_reduce_kernel<float2, float>), dim3((unsigned)g.nsplit), dim3(256), 0, s, g.probs,
                         g.split, g.ptrs, (const float*)g.partials);
    TENET_HIP_CHECK(hipGetLastError());
  }
  return TENET_OK;
}

}  // namespace tenet
