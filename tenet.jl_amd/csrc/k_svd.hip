// K3: thin SVD by one-sided (Hestenes) block Jacobi in FP64, plus the
// truncation rule of Tenet's compress!/simple_update (compress.jl:46-59).
//
// The columns of the work matrix X (nr x ncols, nr >= ncols; a wide input is
// processed as A^H) are cut into blocks of b columns.  A sweep visits every
// block pair once in the round-robin ("circle") order, so the nblk/2 pairs
// of one round are independent.  For a pair (I, J) the 2b x 2b Gram matrix
// G = [X_I X_J]^H [X_I X_J] is diagonalised by cyclic two-sided Jacobi
// (Rutishauser's rotation formulas, complex form: Demmel & Veselic, SIAM J.
// Matrix Anal. Appl. 13 (1992)) in LDS, and the accumulated unitary W is
// applied to the pair's columns of X and V.  At convergence X = U diag(s),
// A = X V^H.  All rotations, Gram sums and norms are FP64.
//
// A round is one launch (phase 2): a pair is one workgroup, or q workgroups that
// each form its Gram, solve the same 2b x 2b problem and rotate their share of
// the rows.  One tall matrix (above 768 rows, or a single pair) takes two
// launches: partial Grams per row chunk (phase 0), then every workgroup of the
// pair sums the q partials in a fixed order, solves and rotates its own row
// chunk (phase 1).
#include <hip/hip_ext.h>

#include "../../include/tenet_hip.h"
#include "internal.h"

namespace tenet {

constexpr int SV_THREADS = 256;
// the round kernel: two waves per SIMD, the Gram, the inner solve and the
// rotation split so that each thread carries half the work of a 256-thread
// workgroup's thread
constexpr int SR_THREADS = 512;
constexpr int B2MAX = 32;  // 2b
constexpr int RS = 64;     // staged rows per LDS pass
constexpr int SORT_MAX = 4096;
constexpr int GT = 8;      // rows of a wave's Gram tile
constexpr int GT_LD = 34;  // its leading dimension: 16 lanes' 16-byte writes and reads meet in no LDS bank

__device__ __forceinline__ int circle_pos(int i, int r, int nb) {
  return i == 0 ? 0 : 1 + ((i - 1 + r) % (nb - 1));
}

struct SvSmem {
  double gr[B2MAX][B2MAX + 1];
  double gi[B2MAX][B2MAX + 1];
  double wr[B2MAX][B2MAX + 1];
  double wi[B2MAX][B2MAX + 1];
  union {
    struct {  // row staging (Gram accumulation, rotation of X and V)
      double xr[RS][B2MAX + 1];
      double xi[RS][B2MAX + 1];
    };
    double2 tile[SR_THREADS / 64][GT][GT_LD];  // per wave: rows of the pair on their way into MFMA operands
    struct {  // second Gram buffer of the inner solve
      double hr[B2MAX][B2MAX + 1];
      double hi[B2MAX][B2MAX + 1];
    };
  };
  // rotations by slot: [0..1] c, Re s, Im s (and d') by step parity, [2..3] the new diagonal
  double rcs[4][B2MAX / 2][4];
  int rpq[2][B2MAX / 2];  // rotation active
  int any_outer, any_big, need;
};

__device__ __forceinline__ int pair_col(int l, int I, int J, int b) { return l < b ? I * b + l : J * b + (l - b); }

// Stage rows [r0, r0+rows) of the pair's 2b columns of M (ld) into LDS.
// All of a thread's loads (64 x 32 / 512 = 4) are issued before any is
// written to LDS, so the staging costs one memory latency, not four.
constexpr int STAGE_PER = RS * B2MAX / SR_THREADS;
__device__ __forceinline__ void load_rows(double2 (&v)[STAGE_PER], const double* M, int64_t ld, int r0, int rows,
                                          int I, int J, int b) {
  const int n2 = 2 * b;
  const double2* M2 = reinterpret_cast<const double2*>(M);
#pragma unroll
  for (int u = 0; u < STAGE_PER; ++u) {
    const int e = threadIdx.x + u * SR_THREADS;
    const int r = e % RS, l = e / RS;
    v[u].x = 0.0;
    v[u].y = 0.0;
    if (l < n2 && r < rows) v[u] = M2[(size_t)pair_col(l, I, J, b) * ld + r0 + r];
  }
}

__device__ __forceinline__ void store_rows(SvSmem& sm, const double2 (&v)[STAGE_PER], int n2) {
#pragma unroll
  for (int u = 0; u < STAGE_PER; ++u) {
    const int e = threadIdx.x + u * SR_THREADS;
    const int r = e % RS, l = e / RS;
    if (l < n2) {
      sm.xr[r][l] = v[u].x;
      sm.xi[r][l] = v[u].y;
    }
  }
}

__device__ __forceinline__ void stage_rows(SvSmem& sm, const double* M, int64_t ld, int r0, int rows, int I, int J,
                                           int b) {
  double2 v[STAGE_PER];
  load_rows(v, M, ld, r0, rows, I, J, b);
  store_rows(sm, v, 2 * b);
}

// acc += staged^H staged for this thread's 2x2 block of the Gram matrix:
// slot t' = t % 256 < (n2/2)^2 owns rows {2i, 2i+1} x cols {2j, 2j+1},
// i = t' % (n2/2), j = t' / (n2/2); acc[0..3] = (2i,2j), (2i+1,2j),
// (2i,2j+1), (2i+1,2j+1).  Threads t < 256 take the staged rows [0, 32),
// threads t >= 256 the rows [32, 64); gram_combine adds the two halves.
constexpr int GE_PER_THREAD = 4;
constexpr int GRAM_SLOTS = 256;

__device__ __forceinline__ void gram_accum(SvSmem& sm, int n2, int rows, double* ar, double* ai) {
  const int h = n2 / 2;
  const int t = threadIdx.x % GRAM_SLOTS, half = threadIdx.x / GRAM_SLOTS;
  if (t >= h * h) return;
  const int i0 = 2 * (t % h), j0 = 2 * (t / h);
  const int rlo = half * (RS / 2), rhi = min(rows, rlo + RS / 2);
  double s0r = 0, s0i = 0, s1r = 0, s1i = 0, s2r = 0, s2i = 0, s3r = 0, s3i = 0;
  for (int r = rlo; r < rhi; ++r) {
    const double ar0 = sm.xr[r][i0], ai0 = sm.xi[r][i0];
    const double ar1 = sm.xr[r][i0 + 1], ai1 = sm.xi[r][i0 + 1];
    const double br0 = sm.xr[r][j0], bi0 = sm.xi[r][j0];
    const double br1 = sm.xr[r][j0 + 1], bi1 = sm.xi[r][j0 + 1];
    // conj(a) * b
    s0r += ar0 * br0 + ai0 * bi0;
    s0i += ar0 * bi0 - ai0 * br0;
    s1r += ar1 * br0 + ai1 * bi0;
    s1i += ar1 * bi0 - ai1 * br0;
    s2r += ar0 * br1 + ai0 * bi1;
    s2i += ar0 * bi1 - ai0 * br1;
    s3r += ar1 * br1 + ai1 * bi1;
    s3i += ar1 * bi1 - ai1 * br1;
  }
  ar[0] += s0r;
  ai[0] += s0i;
  ar[1] += s1r;
  ai[1] += s1i;
  ar[2] += s2r;
  ai[2] += s2i;
  ar[3] += s3r;
  ai[3] += s3i;
}

// Threads t < 256 end with the full sums: the upper half's partials pass
// through the (then idle) staging rows.
__device__ __forceinline__ void gram_combine(SvSmem& sm, int n2, double* ar, double* ai) {
  const int h = n2 / 2;
  const int t = threadIdx.x % GRAM_SLOTS, half = threadIdx.x / GRAM_SLOTS;
  double* buf = &sm.xr[0][0];
  __syncthreads();
  if (half == 1 && t < h * h) {
#pragma unroll
    for (int u = 0; u < GE_PER_THREAD; ++u) {
      buf[(2 * u) * GRAM_SLOTS + t] = ar[u];
      buf[(2 * u + 1) * GRAM_SLOTS + t] = ai[u];
    }
  }
  __syncthreads();
  if (half == 0 && t < h * h) {
#pragma unroll
    for (int u = 0; u < GE_PER_THREAD; ++u) {
      ar[u] += buf[(2 * u) * GRAM_SLOTS + t];
      ai[u] += buf[(2 * u + 1) * GRAM_SLOTS + t];
    }
  }
}

// Gram entry index (row, col) of this thread's slot t (0..3)
__device__ __forceinline__ void gram_slot(int n2, int slot, int& row, int& col) {
  const int h = n2 / 2;
  const int t = threadIdx.x;
  row = 2 * (t % h) + (slot & 1);
  col = 2 * (t / h) + (slot >> 1);
}

__device__ void gram_over_rows(SvSmem& sm, const double* X, int64_t ld, int r0, int r1, int I, int J, int b,
                               double* ar, double* ai) {
  const int n2 = 2 * b;
  for (int t = 0; t < GE_PER_THREAD; ++t) {
    ar[t] = 0.0;
    ai[t] = 0.0;
  }
  for (int rb = r0; rb < r1; rb += RS) {
    const int rows = min(RS, r1 - rb);
    __syncthreads();
    stage_rows(sm, X, ld, rb, rows, I, J, b);
    __syncthreads();
    gram_accum(sm, n2, rows, ar, ai);
  }
  gram_combine(sm, n2, ar, ai);
}

// Diagonalise the Hermitian Gram (n2 x n2, n2 <= 32) by one cyclic Jacobi
// sweep in the round-robin (circle) order over all n2 columns: n2 - 1
// steps, step s applies n2/2 disjoint rotations J_k (slot k pairs columns
// p_k < q_k), G <- J^H G J and W <- W J.  (The cross rounds, which pair only
// columns of different blocks, run jacobi_cross32 below.)
//
// One workgroup barrier per step, with the rotations formed one step ahead.
// G is double-buffered (the second buffer lies over the row-staging area,
// idle during the solve) and only its upper triangle is kept current
// (entries below it read as conjugated mirrors).  In the circle order the
// columns of slot k at step s + 1 come from two different slots k1, k2 of
// step s, so the entries step s + 1's rotation k needs are
//   G'[p'][p'], G'[q'][q'] = new diagonals of rotations k1, k2 of step s,
//   G'[p'][q']             = one entry of J_k1^H B J_k2, B the 2x2 block
//                            {p_k1, q_k1} x {p_k2, q_k2} of G before step s,
// all known from G_s and step s's rotations.  Wave 7 (one lane per slot)
// writes the (p, q) entries of step s's slots (closed form; G's diagonal
// passes through the rotation slots) and forms step s + 1's rotations while waves 0-1 update the off-diagonal 2 x 2 blocks (one thread
// per block: both output rows) and waves 2-6 rotate W with step s's
// rotations; the rotations (c, s and the new diagonal) pass through LDS
// slots double-buffered by step parity.
// columns of slot k at step s of the circle order
__device__ __forceinline__ void circle_pair(int k, int step, int n2, int& p, int& q) {
  // circle_pos without the modulo: i - 1 + r < 2 (n2 - 1)
  const int m = n2 - 1;
  const int i0 = k, i1 = n2 - 1 - k;
  int a0 = i0 - 1 + step, a1 = i1 - 1 + step;
  a0 = a0 >= m ? a0 - m : a0;
  a1 = a1 >= m ? a1 - m : a1;
  p = i0 == 0 ? 0 : 1 + a0;
  q = i1 == 0 ? 0 : 1 + a1;
  if (p > q) {
    const int t = p;
    p = q;
    q = t;
  }
}

typedef double GramRow[B2MAX + 1];

// 1/sqrt(x) for x > 0: hardware estimate and two Newton steps in correction
// form y <- y + y (1 - x y^2) / 2 (each squares the relative error; the
// estimate is good to ~2^-24, so two steps reach double precision).
__device__ __forceinline__ double rsqrt_nr(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
  y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
  return y;
}

// Rotation zeroing G[p][q] of [[a, g], [conj(g), d]].  With
// delta = (d - a) / 2 and r = sqrt(delta^2 + |g|^2) the angle has
// cos 2theta = |delta| / r and sin 2theta = |g| / r, so c = cos theta =
// sqrt((1 + |delta| / r) / 2) and s = sign(delta) g / (2 r c) (the
// smaller rotation of Rutishauser's formulas, tan theta = |g| / (|delta| + r)).
// The new diagonal is a - sign(delta) t |g|, d + sign(delta) t |g| with
// t |g| = |g|^2 / (|delta| + r) = |g|^2 / (2 r c^2).
// Identity when |g| <= tol sqrt(a d) or |g| <= abs_tol (compared squared).
// x of lane (l + 1) mod 16 within each 16-lane row (DPP row_ror:15, on the
// VALU; lanes 0-15 hold the slots of the cross-block inner solve)
__device__ __forceinline__ double from_next_lane(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), 0x12F, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x12F, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

struct Rot {
  double c, sr, si;  // J = [[c, s], [-conj(s), c]]
  double an, dn;     // new diagonal
  int act;
  int big;  // |g|^2 > big2 a d: the sweep has not converged (compared, not divided: a
            // reciprocal here would lengthen every step of the inner solve)
};

__device__ __forceinline__ Rot form_rotation(double ra, double rd, double rxr, double rxi, double tol2, double abs2,
                                             double big2) {
  Rot o;
  const double g2 = rxr * rxr + rxi * rxi;
  const double ad = fmax(ra, 0.0) * fmax(rd, 0.0);
  o.act = (g2 > tol2 * ad && g2 > abs2) ? 1 : 0;
  o.big = (g2 > big2 * ad && ad > 0.0) ? 1 : 0;
  o.c = 1.0;
  o.sr = 0.0;
  o.si = 0.0;
  o.an = ra;
  o.dn = rd;
  if (o.act) {
    const double dl = 0.5 * (rd - ra);
    const double ir = rsqrt_nr(fma(dl, dl, g2));    // 1 / r
    const double v = fma(0.5 * fabs(dl), ir, 0.5);  // c^2
    const double y = rsqrt_nr(v);                   // 1 / c
    o.c = v * y;
    const double sn = copysign(0.5 * ir * y, dl);
    const double tg = copysign((0.5 * g2) * (ir * (y * y)), dl);
    o.sr = sn * rxr;
    o.si = sn * rxi;
    o.an = ra - tg;
    o.dn = rd + tg;
  }
  return o;
}

// row H of B' = J_k^H B J_l for the 2x2 block B = [B0; B1] and the rotations
// J = [[c, e], [-conj(e), c]]: row 0 of T = J_k^H B is c_k B0 - e_k B1, row 1
// conj(e_k) B0 + c_k B1, and a row of B' is (c_l T0 - conj(e_l) T1,
// e_l T0 + c_l T1).
template <int H>
__device__ __forceinline__ void block_row(double ck, double ekr, double eki, double cl, double elr, double eli,
                                          const double (&b)[8], double& n0r, double& n0i, double& n1r, double& n1i) {
  // b = {B00 re, im, B01 re, im, B10 re, im, B11 re, im}
  double t[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const double xr = b[2 * j], xi = b[2 * j + 1], yr = b[4 + 2 * j], yi = b[5 + 2 * j];
    if (H == 0) {
      t[2 * j] = fma(ck, xr, fma(eki, yi, -(ekr * yr)));
      t[2 * j + 1] = fma(ck, xi, -fma(ekr, yi, eki * yr));
    } else {
      t[2 * j] = fma(ck, yr, fma(ekr, xr, eki * xi));
      t[2 * j + 1] = fma(ck, yi, fma(ekr, xi, -(eki * xr)));
    }
  }
  n0r = fma(cl, t[0], -fma(elr, t[2], eli * t[3]));
  n0i = fma(cl, t[1], fma(eli, t[2], -(elr * t[3])));
  n1r = fma(cl, t[2], fma(elr, t[0], -(eli * t[1])));
  n1i = fma(cl, t[3], fma(elr, t[1], eli * t[0]));
}

// G entry (r, c), r != c, from the upper triangle (an entry below it is the
// conjugate of its mirror), and the matching store
__device__ __forceinline__ void g_get(const GramRow* gr, const GramRow* gi, int r, int c, double& re, double& im) {
  const int lo = min(r, c), hi = max(r, c);
  re = gr[lo][hi];
  im = r < c ? gi[lo][hi] : -gi[lo][hi];
}
__device__ __forceinline__ void g_put(GramRow* gr, GramRow* gi, int r, int c, double re, double im) {
  const int lo = min(r, c), hi = max(r, c);
  gr[lo][hi] = re;
  gi[lo][hi] = r < c ? im : -im;
}

// Slot and side (0: p, 1: q) of column c at step s of the circle order over
// n2 columns (the inverse of circle_pair: the column at position i >= 1 is
// 1 + (i - 1 + s) mod (n2 - 1), position i belongs to slot min(i, n2 - 1 - i))
__device__ __forceinline__ void circle_slot(int c, int step, int n2, int& slot, int& side) {
  const int m = n2 - 1;
  int i = 0;
  if (c != 0) {
    int t = c - 1 - step;
    t = t < 0 ? t + m : t;
    i = 1 + t;
  }
  slot = min(i, n2 - 1 - i);
  int p, q;
  circle_pair(slot, step, n2, p, q);
  side = c == q ? 1 : 0;
}

constexpr int IROT_WAVE = 7;      // rotation wave of the full inner sweep
constexpr int IW_FIRST = 2 * 64;  // first W thread (waves 2-6)
constexpr int IW_THREADS = 5 * 64;

__device__ __forceinline__ void jacobi_inner(SvSmem& sm, int n2, double tol, double abs_tol) {
  const int tid = threadIdx.x, wave = tid >> 6, ln = tid & 63;
  const int npair = n2 / 2, nsteps = n2 - 1;
  // W = I on the pair's n2 columns and 0 elsewhere in the 32 x 32 block (the
  // MFMA rotation runs over all 32 columns)
  for (int e = tid; e < B2MAX * B2MAX; e += SR_THREADS) {
    const int i = e % B2MAX, c = e / B2MAX;
    sm.wr[i][c] = (i == c && i < n2) ? 1.0 : 0.0;
    sm.wi[i][c] = 0.0;
  }
  const double tol2 = tol * tol, abs2 = abs_tol * abs_tol, big2 = 0.25 * tol;
  const bool gwave = wave < 2, wwave = tid >= IW_FIRST && tid < IW_FIRST + IW_THREADS, rwave = wave == IROT_WAVE;
  // G: the npair (npair - 1) / 2 blocks bk < bl in row-major order, one thread each
  int bk = 0, bl = 1;
  bool gown = false;
  if (gwave) {
    gown = tid < npair * (npair - 1) / 2;
    int rem = gown ? tid : 0, k = 0;
    while (k < npair - 1 && rem >= npair - 1 - k) {
      rem -= npair - 1 - k;
      ++k;
    }
    bk = k;
    bl = k + 1 + rem;
  }
  // W: element e = (tid - IW_FIRST) + IW_THREADS u is (row e / npair, slot e % npair); npair n2 <= 512
  int wrow[2], wslot[2];
  bool wown[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int e = (tid - IW_FIRST) + IW_THREADS * u;
    wown[u] = wwave && e < npair * n2;
    const int ec = wown[u] ? e : 0;
    wrow[u] = ec / npair;
    wslot[u] = ec % npair;
  }
  // rotation wave: lane k < npair owns slot k
  const bool rown = rwave && ln < npair;
  const int k = rwave ? min(ln, npair - 1) : 0;
  Rot rt;
  double rgr = 0.0, rgi = 0.0;  // G[p_k][q_k] the current rotation was formed from
  int any = 0, big = 0;
  __syncthreads();
  if (rwave) {
    int p, q;
    circle_pair(k, 0, n2, p, q);
    rgr = sm.gr[p][q];
    rgi = sm.gi[p][q];
    rt = form_rotation(sm.gr[p][p], sm.gr[q][q], rgr, rgi, tol2, abs2, big2);
    if (rown) {
      sm.rcs[0][k][0] = rt.c;
      sm.rcs[0][k][1] = rt.sr;
      sm.rcs[0][k][2] = rt.si;
      sm.rcs[2][k][0] = rt.an;
      sm.rcs[2][k][1] = rt.dn;
      sm.rpq[0][k] = rt.act;
      big |= rt.big;
      any |= rt.act;
    }
  }
  __syncthreads();
  for (int step = 0; step < nsteps; ++step) {
    const int par = step & 1;
    const GramRow* cr = par ? sm.hr : sm.gr;
    const GramRow* ci = par ? sm.hi : sm.gi;
    GramRow* nr = par ? sm.gr : sm.hr;
    GramRow* ni = par ? sm.gi : sm.hi;
    if (gwave) {
      if (gown) {
        int p0, q0, p1, q1;
        circle_pair(bk, step, n2, p0, q0);
        circle_pair(bl, step, n2, p1, q1);
        double b[8];
        g_get(cr, ci, p0, p1, b[0], b[1]);
        g_get(cr, ci, p0, q1, b[2], b[3]);
        g_get(cr, ci, q0, p1, b[4], b[5]);
        g_get(cr, ci, q0, q1, b[6], b[7]);
        const double ck = sm.rcs[par][bk][0], ekr = sm.rcs[par][bk][1], eki = sm.rcs[par][bk][2];
        const double cl = sm.rcs[par][bl][0], elr = sm.rcs[par][bl][1], eli = sm.rcs[par][bl][2];
        double n0r, n0i, n1r, n1i;
        block_row<0>(ck, ekr, eki, cl, elr, eli, b, n0r, n0i, n1r, n1i);
        g_put(nr, ni, p0, p1, n0r, n0i);
        g_put(nr, ni, p0, q1, n1r, n1i);
        block_row<1>(ck, ekr, eki, cl, elr, eli, b, n0r, n0i, n1r, n1i);
        g_put(nr, ni, q0, p1, n0r, n0i);
        g_put(nr, ni, q0, q1, n1r, n1i);
      }
    } else if (wwave) {
      // W <- W J on this thread's elements
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int ks = wslot[u];
        if (!wown[u] || !sm.rpq[par][ks]) continue;
        int wp, wq;
        circle_pair(ks, step, n2, wp, wq);
        const int row = wrow[u];
        const double pr = sm.wr[row][wp], pi = sm.wi[row][wp], qr = sm.wr[row][wq], qi = sm.wi[row][wq];
        const double cw = sm.rcs[par][ks][0], er = sm.rcs[par][ks][1], ei = sm.rcs[par][ks][2];
        sm.wr[row][wp] = cw * pr - (er * qr + ei * qi);
        sm.wi[row][wp] = cw * pi - (er * qi - ei * qr);
        sm.wr[row][wq] = (er * pr - ei * pi) + cw * qr;
        sm.wi[row][wq] = (er * pi + ei * pr) + cw * qi;
      }
    } else if (rwave) {
      // the slots' off-diagonal entries of this step, then the next step's rotations
      if (rown) {
        int p, q;
        circle_pair(k, step, n2, p, q);
        nr[p][q] = rt.act ? 0.0 : rgr;
        ni[p][q] = rt.act ? 0.0 : rgi;
      }
      if (step + 1 < nsteps) {
        int pn, qn, k1, h1, k2, h2, pk1, qk1, pk2, qk2;
        circle_pair(k, step + 1, n2, pn, qn);
        circle_slot(pn, step, n2, k1, h1);
        circle_slot(qn, step, n2, k2, h2);
        circle_pair(k1, step, n2, pk1, qk1);
        circle_pair(k2, step, n2, pk2, qk2);
        double b[8];
        g_get(cr, ci, pk1, pk2, b[0], b[1]);
        g_get(cr, ci, pk1, qk2, b[2], b[3]);
        g_get(cr, ci, qk1, pk2, b[4], b[5]);
        g_get(cr, ci, qk1, qk2, b[6], b[7]);
        const double c1 = sm.rcs[par][k1][0], s1r = sm.rcs[par][k1][1], s1i = sm.rcs[par][k1][2];
        const double c2 = sm.rcs[par][k2][0], s2r = sm.rcs[par][k2][1], s2i = sm.rcs[par][k2][2];
        const double an = sm.rcs[2 + par][k1][h1], dn = sm.rcs[2 + par][k2][h2];
        double x0r, x0i, x1r, x1i, y0r, y0i, y1r, y1i;
        block_row<0>(c1, s1r, s1i, c2, s2r, s2i, b, x0r, x0i, x1r, x1i);
        block_row<1>(c1, s1r, s1i, c2, s2r, s2i, b, y0r, y0i, y1r, y1i);
        const double n0r = h1 ? y0r : x0r, n0i = h1 ? y0i : x0i;
        const double n1r = h1 ? y1r : x1r, n1i = h1 ? y1i : x1i;
        rgr = h2 ? n1r : n0r;
        rgi = h2 ? n1i : n0i;
        rt = form_rotation(an, dn, rgr, rgi, tol2, abs2, big2);
        if (rown) {
          sm.rcs[par ^ 1][k][0] = rt.c;
          sm.rcs[par ^ 1][k][1] = rt.sr;
          sm.rcs[par ^ 1][k][2] = rt.si;
          sm.rcs[2 + (par ^ 1)][k][0] = rt.an;
          sm.rcs[2 + (par ^ 1)][k][1] = rt.dn;
          sm.rpq[par ^ 1][k] = rt.act;
          big |= rt.big;
          any |= rt.act;
        }
      }
    }
    __syncthreads();
  }
  if (rown && any) sm.any_outer = 1;
  if (rown && big) sm.any_big = 1;
  __syncthreads();
}

// Inner solve for 2b = 32 (every round of a matrix of more than 30 columns), in
// levels H = h0, 2 h0, .. 16: at level H the 32 columns are 16 / H groups of
// 2H, and its H steps rotate every column of a group's first half with every
// one of its second half.  h0 = 16 is the cross-block solve of two 16-column
// blocks; h0 = 1 visits all 496 pairs once, within the blocks before across
// them.  Slot k (0..15), j = k mod H, pairs at step s
//   p_k = 2 (k - j) + j  and  q_k(s) = 2 (k - j) + H + (j + s) mod H,
// so p_k stays and q_k(s + 1) = q_n(s), n = k - j + (j + 1) mod H the group's
// next slot.  The entries rotation k of step s + 1 needs are therefore
//   G'[p][p]   = the new diagonal a'_k of rotation k of step s,
//   G'[q][q]   = the new diagonal d'_n of rotation n of step s,
//   G'[p][q_n] = row p, column q_n of J_k^H B J_n, B the 2x2 block
//                {p_k, q_k} x {p_n, q_n} of G before step s,
// all known from G_s and step s's rotations.  Wave 7 (lanes 0-15: one slot
// each) forms them and step s + 1's rotations while 120 threads of waves
// 0-1 update the G blocks above the diagonal (one 2 x 2 block each, read
// once; only G's upper triangle is kept, entries below it read as
// conjugated mirrors) and waves 4-6 rotate W, which they keep in registers,
// with step s's rotations; the rotations pass through LDS slots
// double-buffered by step parity, so a step takes one workgroup barrier.
// Wave 7 also writes the (p, q) entries of the step's slots (closed form); G's
// diagonal stays in its registers and goes to LDS between levels.
//
// The step is wave 7's dependent chain (LDS reads, one row of a block, two
// reciprocal square roots): ~1000 cycles; the circle order of jacobi_inner,
// whose slots change partners irregularly, takes 2500.
constexpr int XB = 16;         // slots
constexpr int XROT_WAVE = 7;   // rotation wave

// x of the next slot of the group (lanes of one 16-lane row)
__device__ __forceinline__ double from_next_slot(double x, int H, int lane) {
  return H == XB ? from_next_lane(x) : __shfl(x, lane, 64);
}

// The levels and steps of jacobi_levels.  Each role runs its own copy of these
// loops (so that its registers are its own), chosen by a scalar branch on the
// wave's number; every copy passes the same 1 + H barriers a level.
template <typename Init, typename Step, typename Done>
__device__ __forceinline__ void level_loops(int h0, Init init, Step step, Done done) {
  int par = 0;  // the G buffer and rotation slots of the coming step
#pragma unroll 1
  for (int H = h0; H <= XB; H <<= 1) {
    init(H, par);
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st < H; ++st) {
      step(H, st, par);
      par ^= 1;
      __syncthreads();
    }
    done(H);
  }
}

__device__ __forceinline__ void jacobi_levels(SvSmem& sm, int h0, double tol, double abs_tol) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = tid & 63;
  const int k = ln & (XB - 1);
  if (wave < 2) {
    // G: blocks bk < bl, one thread each (both output rows: the 2 x 2 block is
    // read once), sixteen threads at one distance d around the circle of slots
    // (d = 1..7, then half of d = 8): a wave's reads of G then meet in few LDS
    // banks (32 cycles for the eight reads of a step, 58 in row-major order)
    const bool own = tid < XB * (XB - 1) / 2;
    const int i = tid % XB, i2 = (i + 1 + tid / XB) % XB;
    const int bk = own ? min(i, i2) : 0, bl = own ? max(i, i2) : 1;
    int jk, jl, p0, p1, h0k, h0l;  // the blocks' columns p and the first of their groups' second halves
    level_loops(
        h0,
        [&](int H, int) {
          jk = bk & (H - 1);
          jl = bl & (H - 1);
          p0 = 2 * bk - jk;
          p1 = 2 * bl - jl;
          h0k = p0 - jk + H;
          h0l = p1 - jl + H;
        },
        [&](int H, int step, int par) {
          const GramRow* cr = par ? sm.hr : sm.gr;
          const GramRow* ci = par ? sm.hi : sm.gi;
          GramRow* nr = par ? sm.gr : sm.hr;
          GramRow* ni = par ? sm.gi : sm.hi;
          // only the upper triangle of G is kept up to date: an entry below the
          // diagonal is read as the conjugate of its mirror
          const int q0 = h0k + ((jk + step) & (H - 1)), q1 = h0l + ((jl + step) & (H - 1));
          const int qa = min(q0, q1), qb = max(q0, q1), ra = min(q0, p1), rb = max(q0, p1);
          double b[8];
          b[0] = cr[p0][p1];
          b[1] = ci[p0][p1];
          b[2] = cr[p0][q1];
          b[3] = ci[p0][q1];
          b[4] = cr[ra][rb];
          b[5] = ci[ra][rb];
          b[6] = cr[qa][qb];
          b[7] = ci[qa][qb];
          const double ck = sm.rcs[par][bk][0], ekr = sm.rcs[par][bk][1], eki = sm.rcs[par][bk][2];
          const double cl = sm.rcs[par][bl][0], elr = sm.rcs[par][bl][1], eli = sm.rcs[par][bl][2];
          b[5] = q0 <= p1 ? b[5] : -b[5];
          b[7] = q0 <= q1 ? b[7] : -b[7];
          if (own) {
            double n0r, n0i, n1r, n1i;
            block_row<0>(ck, ekr, eki, cl, elr, eli, b, n0r, n0i, n1r, n1i);
            nr[p0][p1] = n0r;
            ni[p0][p1] = n0i;
            nr[p0][q1] = n1r;
            ni[p0][q1] = n1i;
            block_row<1>(ck, ekr, eki, cl, elr, eli, b, n0r, n0i, n1r, n1i);
            nr[ra][rb] = n0r;
            ni[ra][rb] = q0 <= p1 ? n0i : -n0i;
            nr[qa][qb] = n1r;
            ni[qa][qb] = q0 <= q1 ? n1i : -n1i;
          }
        },
        [](int) {});
  } else if (wave >= 4 && wave < XROT_WAVE) {
    // W lives in the registers of waves 4-6: lane k of 16-lane row group wg
    // (0..11) holds, for rows wg, wg + 12 and wg + 24 (< 32), P = W[row][p_k]
    // and Q = W[row][q_k(step)]; Q moves one slot down between steps, and W
    // goes through LDS between levels.
    const int wg = (tid - 4 * 64) >> 4;
    double Pr[3], Pi[3], Qr[3], Qi[3];
    level_loops(
        h0,
        [&](int H, int) {
          const int p = 2 * k - (k & (H - 1));
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            const int row = wg + 12 * u, r = min(row, 2 * XB - 1);
            if (H == h0) {
              Pr[u] = row == p ? 1.0 : 0.0;
              Pi[u] = 0.0;
              Qr[u] = row == p + H ? 1.0 : 0.0;
              Qi[u] = 0.0;
            } else {  // written by this wave at the level before
              Pr[u] = sm.wr[r][p];
              Pi[u] = sm.wi[r][p];
              Qr[u] = sm.wr[r][p + H];
              Qi[u] = sm.wi[r][p + H];
            }
          }
        },
        [&](int H, int step, int par) {
          // an inactive rotation is c = 1, s = 0
          const double c = sm.rcs[par][k][0], er = sm.rcs[par][k][1], ei = sm.rcs[par][k][2];
          if (step > 0) {
            const int next = (ln & ~(H - 1)) | ((ln + 1) & (H - 1));
#pragma unroll
            for (int u = 0; u < 3; ++u) {
              Qr[u] = from_next_slot(Qr[u], H, next);
              Qi[u] = from_next_slot(Qi[u], H, next);
            }
          }
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            const double pr = Pr[u], pi = Pi[u], qr = Qr[u], qi = Qi[u];
            Pr[u] = c * pr - (er * qr + ei * qi);
            Pi[u] = c * pi - (er * qi - ei * qr);
            Qr[u] = (er * pr - ei * pi) + c * qr;
            Qi[u] = (er * pi + ei * pr) + c * qi;
          }
        },
        [&](int H) {
          const int j = k & (H - 1), p = 2 * k - j;
          const int q = p - j + H + ((j + H - 1) & (H - 1));  // q_k of the last step
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            const int row = wg + 12 * u;
            if (row < 2 * XB) {
              sm.wr[row][p] = Pr[u];
              sm.wi[row][p] = Pi[u];
              sm.wr[row][q] = Qr[u];
              sm.wi[row][q] = Qi[u];
            }
          }
        });
  } else if (wave == XROT_WAVE) {
    // lane k < 16 owns slot k
    const double tol2 = tol * tol, abs2 = abs_tol * abs_tol, big2 = 0.25 * tol;
    const bool own = ln < XB;
    int any = 0, big = 0;
    Rot rt;
    double gr, gi;  // G[p_k][q_k] the current rotation was formed from
    auto put = [&](int par) {
      if (!own) return;
      sm.rcs[par][k][0] = rt.c;
      sm.rcs[par][k][1] = rt.sr;
      sm.rcs[par][k][2] = rt.si;
      sm.rcs[par][k][3] = rt.dn;
      big |= rt.big;
      any |= rt.act;
    };
    level_loops(
        h0,
        [&](int H, int par) {
          const GramRow* cr = par ? sm.hr : sm.gr;
          const GramRow* ci = par ? sm.hi : sm.gi;
          const int p = 2 * k - (k & (H - 1)), q = p + H;
          gr = cr[p][q];
          gi = ci[p][q];
          rt = form_rotation(cr[p][p], cr[q][q], gr, gi, tol2, abs2, big2);
          put(par);
        },
        [&](int H, int step, int par) {
          const GramRow* cr = par ? sm.hr : sm.gr;
          const GramRow* ci = par ? sm.hi : sm.gi;
          GramRow* nr = par ? sm.gr : sm.hr;
          GramRow* ni = par ? sm.gi : sm.hi;
          const int j = k & (H - 1), jn = (j + 1) & (H - 1), base = 2 * (k - j), kn = k - j + jn;
          const int p = base + j, pn = base + jn;
          const int q = base + H + ((j + step) & (H - 1)), qn = base + H + ((j + 1 + step) & (H - 1));
          const int pa = min(p, pn), pb = max(p, pn), qa = min(q, qn), qb = max(q, qn);
          // (in a level's last step these feed nothing)
          double b[8];
          b[0] = cr[pa][pb];
          b[1] = ci[pa][pb];
          b[2] = cr[p][qn];
          b[3] = ci[p][qn];
          b[4] = cr[pn][q];
          b[5] = ci[pn][q];
          b[6] = cr[qa][qb];
          b[7] = ci[qa][qb];
          // the next slot's rotation and new diagonal d'
          const double cn = sm.rcs[par][kn][0], srn = sm.rcs[par][kn][1], sin_ = sm.rcs[par][kn][2];
          const double dnn = sm.rcs[par][kn][3];
          if (own) {
            nr[p][q] = rt.act ? 0.0 : gr;
            ni[p][q] = rt.act ? 0.0 : gi;
          }
          if (step + 1 < H) {
            b[1] = p > pn ? -b[1] : b[1];
            b[5] = -b[5];
            b[7] = q > qn ? -b[7] : b[7];
            double n0r, n0i;
            block_row<0>(rt.c, rt.sr, rt.si, cn, srn, sin_, b, n0r, n0i, gr, gi);
            rt = form_rotation(rt.an, dnn, gr, gi, tol2, abs2, big2);
            put(par ^ 1);
          } else if (own) {
            nr[p][p] = rt.an;
            nr[q][q] = rt.dn;
          }
        },
        [](int) {});
    if (own && any) sm.any_outer = 1;
    if (own && big) sm.any_big = 1;
  } else {
    level_loops(h0, [](int, int) {}, [](int, int, int) {}, [](int) {});
  }
  __syncthreads();
}

// The inner solve of a pair visit: a full sweep of its 2b columns (mode 0) or
// the cross-block rotations only (mode 1: always 2b = 32).  A pair none of
// whose entries asks for a rotation is left at once (nearly all pairs of the
// last sweep, where the solve would be half of the round).
__device__ __forceinline__ void inner_solve(SvSmem& sm, int n2, int mode, double tol, double abs_tol) {
  const double tol2 = tol * tol, abs2 = abs_tol * abs_tol;
  if (threadIdx.x == 0) sm.any_outer = sm.any_big = sm.need = 0;
  __syncthreads();
  const int h = n2 / 2;
  for (int e = threadIdx.x; e < (mode == 1 ? h * h : n2 * n2); e += SR_THREADS) {
    const int i = mode == 1 ? e % h : e % n2, j = mode == 1 ? h + e / h : e / n2;
    if (i >= j) continue;
    const double re = sm.gr[i][j], im = sm.gi[i][j], g2 = re * re + im * im;
    if (g2 > tol2 * (fmax(sm.gr[i][i], 0.0) * fmax(sm.gr[j][j], 0.0)) && g2 > abs2) sm.need = 1;
  }
  __syncthreads();
  if (!sm.need) return;
  if (n2 == B2MAX)
    jacobi_levels(sm, mode == 1 ? XB : 1, tol, abs_tol);
  else
    jacobi_inner(sm, n2, tol, abs_tol);
}

// The staged rows [rb, rb + rows) of the pair's columns of M <- M W.  Thread
// t: row t % 64 of the staged chunk and 4 consecutive output columns
// (group t / 64).
constexpr int APPLY_COLS = SR_THREADS / RS > 0 ? B2MAX / (SR_THREADS / RS) : B2MAX;
__device__ __forceinline__ void apply_staged(SvSmem& sm, double* M, int64_t ld, int rb, int rows, int I, int J,
                                             int b) {
  const int n2 = 2 * b;
  const int r = threadIdx.x % RS, cg = APPLY_COLS * (threadIdx.x / RS);
  if (r < rows && cg < n2) {
    double sr[APPLY_COLS], si[APPLY_COLS];
#pragma unroll
    for (int j = 0; j < APPLY_COLS; ++j) sr[j] = si[j] = 0.0;
    for (int t = 0; t < n2; ++t) {
      const double xr = sm.xr[r][t], xi = sm.xi[r][t];
#pragma unroll
      for (int j = 0; j < APPLY_COLS; ++j) {
        const double wr = sm.wr[t][cg + j], wi = sm.wi[t][cg + j];
        sr[j] += xr * wr - xi * wi;
        si[j] += xr * wi + xi * wr;
      }
    }
#pragma unroll
    for (int j = 0; j < APPLY_COLS; ++j) {
      if (cg + j < n2) {
        double2 v;
        v.x = sr[j];
        v.y = si[j];
        reinterpret_cast<double2*>(M)[(size_t)pair_col(cg + j, I, J, b) * ld + rb + r] = v;
      }
    }
  }
}

// rows [r0, r1) of the pair's columns of M <- M W, one staged chunk at a time
__device__ void apply_rows(SvSmem& sm, double* M, int64_t ld, int r0, int r1, int I, int J, int b) {
  for (int rb = r0; rb < r1; rb += RS) {
    const int rows = min(RS, r1 - rb);
    __syncthreads();
    stage_rows(sm, M, ld, rb, rows, I, J, b);
    __syncthreads();
    apply_staged(sm, M, ld, rb, rows, I, J, b);
  }
  __syncthreads();
}

// ---- FP64 MFMA forms of the Gram and of the rotation (v_mfma_f64_16x16x4_f64)
//
// Operand layout of the 16x16x4 FP64 product (lane l): A[i = l % 16][k = l / 16],
// B[k = l / 16][j = l % 16]; accumulator register r of lane l holds
// D[i = 4 r + l / 16][j = l % 16].  The pair's 2b <= 32 columns are two
// 16-column blocks (columns >= 2b staged as zeros).
typedef double svd_d4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ svd_d4v mfma_f64(double a, double b, svd_d4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Gram G = X^H X of the pair's columns over rows [r0, r1) into sm.gr / sm.gi.
// With P = Xr^T Xi:  Re G = Xr^T Xr + Xi^T Xi (symmetric), Im G = P - P^T.
// For a 4-row K step the A operand of X^T and the B operand of X are the same
// register (X[k = l / 16][c = l % 16]).  Every block takes fewer real
// products than the four of a complex one (errors O(eps |x_p| |x_q|), the
// order of a plain dot product's): a diagonal block two, S^T S with
// S = Xr + Xi and P, since Re G = S^T S - P - P^T; the off-diagonal block
// three (Gauss): T1 = Xr0^T Xr1, T2 = Xi0^T Xi1 and
// T3 = (Xr0 + Xi0)^T (Xr1 - Xi1) give Re G(0,1) = T1 + T2 and
// Im G(0,1) = T1 - T2 - T3.
//
// Wave w takes rows 8 w .. 8 w + 7 of each 64: it loads them with eight
// consecutive rows of a column in eight lanes (an MFMA operand wants sixteen
// columns in sixteen lanes, which as a load costs 76 cycles instead of 16),
// turns them round in an LDS tile of its own and forms all seven products, so
// no barrier falls into the loop; D loads are on their way while one is
// multiplied (they take 4000 cycles where other XCDs wrote the columns in the
// round before).  The waves' sums are added in LDS in a fixed order, halving
// the waves.  A chunk of 64 rows is bound by the products: 1800 cycles of the
// matrix cores.
//
// Returns false, with nothing formed, for a converged problem: its flag is
// looked at when the first loads are under way, not before them (FIRST: the
// caller has looked).
template <int D, bool FIRST>
__device__ __forceinline__ bool gram_mfma(SvSmem& sm, const double* X, int64_t ld, int r0, int r1, int I, int J, int b,
                                          int converged) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kr = lane >> 4, kc = lane & 15;
  const int n2 = 2 * b, tr = lane & (GT - 1), tc = lane / GT;
  const double2* X2 = reinterpret_cast<const double2*>(X);
  size_t col[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) col[u] = (size_t)pair_col(min(tc + GT * u, n2 - 1), I, J, b) * ld;
  double2(*tile)[GT_LD] = sm.tile[wave];
  svd_d4v a[7];
#pragma unroll
  for (int t = 0; t < 7; ++t) a[t] = svd_d4v{0, 0, 0, 0};
  double2 v[D][4];
  const int own = r0 + GT * wave + tr;
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (r0 + d * RS < r1)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[d][u] = X2[col[u] + min(own + d * RS, r1 - 1)];
  if (!FIRST && converged) return false;
  for (int r2 = r0; r2 < r1; r2 += D * RS) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int rb = r2 + d * RS, rn = rb + D * RS, row = own + rb - r0;
      if (rb >= r1) break;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = row < r1 && tc + GT * u < n2;
        double2 z = v[d][u];
        z.x = in ? z.x : 0.0;
        z.y = in ? z.y : 0.0;
        tile[tr][tc + GT * u] = z;
      }
      if (rn < r1)
#pragma unroll
        for (int u = 0; u < 4; ++u) v[d][u] = X2[col[u] + min(row + D * RS, r1 - 1)];
#pragma unroll
      for (int s = 0; s < GT / 4; ++s) {
        const double2 x0 = tile[4 * s + kr][kc], x1 = tile[4 * s + kr][16 + kc];
        const double s0 = x0.x + x0.y, s1 = x1.x + x1.y;
        a[0] = mfma_f64(s0, s0, a[0]);
        a[1] = mfma_f64(s1, s1, a[1]);
        a[2] = mfma_f64(x0.x, x0.y, a[2]);
        a[3] = mfma_f64(x1.x, x1.y, a[3]);
        a[4] = mfma_f64(x0.x, x1.x, a[4]);
        a[5] = mfma_f64(x0.y, x1.y, a[5]);
        a[6] = mfma_f64(s0, x1.x - x1.y, a[6]);
      }
    }
  }
  double* red = reinterpret_cast<double*>(&sm);
  static_assert(sizeof(SvSmem) >= (SR_THREADS / 128) * 28 * 64 * sizeof(double), "half the waves' sums fit");
#pragma unroll
  for (int half = SR_THREADS / 128; half > 0; half /= 2) {
    __syncthreads();
    if (wave >= half && wave < 2 * half)
#pragma unroll
      for (int i = 0; i < 28; ++i) red[((wave - half) * 28 + i) * 64 + lane] = a[i / 4][i % 4];
    __syncthreads();
    if (wave < half)
#pragma unroll
      for (int i = 0; i < 28; ++i) a[i / 4][i % 4] += red[(wave * 28 + i) * 64 + lane];
  }
  if (wave == 0) {
    // S^T S of the diagonal blocks and Re G(0,1) (mirrored) into gr, P into
    // wr (scratch until the inner solve sets W); the off-diagonal block of
    // Im G goes into wr above the diagonal (zeros below), so that
    // gi = wr - wr^T holds it and its mirror
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * r + kr, j = kc;
      sm.gr[i][j] = a[0][r];
      sm.gr[16 + i][16 + j] = a[1][r];
      sm.wr[i][j] = a[2][r];
      sm.wr[16 + i][16 + j] = a[3][r];
      sm.gr[i][16 + j] = a[4][r] + a[5][r];
      sm.gr[16 + j][i] = a[4][r] + a[5][r];
      sm.wr[i][16 + j] = a[4][r] - a[5][r] - a[6][r];
      sm.wr[16 + j][i] = 0.0;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < B2MAX * B2MAX; e += SR_THREADS) {
    const int i = e & (B2MAX - 1), j = e / B2MAX;
    const double pij = sm.wr[i][j], pji = sm.wr[j][i];
    sm.gi[i][j] = pij - pji;
    if ((i < 16) == (j < 16)) sm.gr[i][j] -= pij + pji;  // Re G = S^T S - P - P^T
  }
  __syncthreads();
  return true;
}

// M <- M W by MFMA, with no LDS staging, in strips of 16 rows: one wave takes a
// strip, X's operands straight from memory (lane l: row l % 16 of the strip,
// columns 4s + l / 16: 256 contiguous bytes per column and load) and W's from
// LDS.  The product is formed as W^T X^T, so that an accumulator register too
// holds sixteen rows of a column in sixteen lanes and is stored as it was
// loaded (as X W its lanes lie in sixteen columns, and the eight stores of a
// strip took 76 cycles each of the address unit, together nearly the time of
// the products).  The strips of X and then, where the rotations are
// accumulated, those of V are numbered through.
constexpr int STRIP = 16;

// A strip's first row in the pair's two 16-column blocks.  With b < 16 (one
// block pair: I = 0, J = 1) the pair's columns are 0 .. 2b - 1, the second block
// its columns from 16 on.  All members are uniform over the wave.
struct Strip {
  const char* src[2];
  char* dst[2];
  size_t ld;  // bytes from column to column
  int rows;     // rows of the strip inside the matrix (16 and more: all)
};

__device__ __forceinline__ int strip_count(const SvdProblem& P) {
  return (P.nr + STRIP - 1) / STRIP + (P.accum ? (P.ncp + STRIP - 1) / STRIP : 0);
}

// strip i of the (rows x n) matrix M going to D
__device__ __forceinline__ Strip strip_at(const double* M, double* D, int rows, int i, int I, int J, int b) {
  Strip t;
  const size_t c0 = (size_t)I * b, c1 = b == 16 ? (size_t)J * 16 : 16;
  const size_t o0 = (c0 * rows + (size_t)STRIP * i) * sizeof(double2), o1 = (c1 * rows + (size_t)STRIP * i) * sizeof(double2);
  t.src[0] = reinterpret_cast<const char*>(M) + o0;
  t.src[1] = reinterpret_cast<const char*>(M) + o1;
  t.dst[0] = reinterpret_cast<char*>(D) + o0;
  t.dst[1] = reinterpret_cast<char*>(D) + o1;
  t.ld = rows * sizeof(double2);
  t.rows = rows - STRIP * i;
  return t;
}

// X's strips may go from one buffer to another; V is rotated in place
__device__ __forceinline__ Strip strip_of(const SvdProblem& P, const double* Xs, double* Xd, int i, int I, int J) {
  const int sx = (P.nr + STRIP - 1) / STRIP;
  return i < sx ? strip_at(Xs, Xd, P.nr, i, I, J, P.b) : strip_at(P.V, P.V, P.ncp, i - sx, I, J, P.b);
}

// x[s]: row l % 16, column 4s + l / 16 (rows past the matrix: its last row
// again, never stored; columns past 2b: 0)
__device__ __forceinline__ void strip_load(double2 (&x)[B2MAX / 4], const Strip& t, int b) {
  const int lane = threadIdx.x & 63, kr = lane >> 4;
  const unsigned row = min(lane & 15, t.rows - 1) * (unsigned)sizeof(double2);
#pragma unroll
  for (int s = 0; s < B2MAX / 4; ++s) {
    const bool ok = 4 * s + kr < 2 * b;
    const size_t off = (ok ? (4 * (s & 3) + kr) * t.ld : 0) + row;
    const double2 v = *reinterpret_cast<const double2*>((ok ? t.src[s >> 2] : t.src[0]) + off);
    x[s].x = ok ? v.x : 0.0;
    x[s].y = ok ? v.y : 0.0;
  }
}

// The strip's output columns 16 cb .. 16 cb + 15, cb in [cb0, cb0 + NCB).
// Three real products per complex one (Gauss):
//   T1 = Xr Wr, T2 = Xi Wi, T3 = (Xr + Xi)(Wr + Wi);
//   Re Y = T1 - T2, Im Y = T3 - T1 - T2
// (W is unitary, so the cancellation in Im Y costs O(eps |X|))
template <int NCB>
__device__ __forceinline__ void strip_rotate(const SvSmem& sm, const double2 (&x)[B2MAX / 4], const Strip& t0, int cb0,
                                             int b) {
  const int lane = threadIdx.x & 63, kr = lane >> 4, kc = lane & 15;
  svd_d4v t[NCB][3];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int u = 0; u < 3; ++u) t[cb][u] = svd_d4v{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < B2MAX / 4; ++s) {
    const double xr = x[s].x, xi = x[s].y, xs = xr + xi;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      const int c = 16 * (cb0 + cb) + kc;
      const double wre = sm.wr[4 * s + kr][c], wim = sm.wi[4 * s + kr][c];
      t[cb][0] = mfma_f64(wre, xr, t[cb][0]);
      t[cb][1] = mfma_f64(wim, xi, t[cb][1]);
      t[cb][2] = mfma_f64(wre + wim, xs, t[cb][2]);
    }
  }
  if (kc >= t0.rows) return;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    char* dst = cb0 + cb ? t0.dst[1] : t0.dst[0];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (16 * (cb0 + cb) + 4 * r + kr < 2 * b) {
        double2 o;
        o.x = t[cb][0][r] - t[cb][1][r];
        o.y = t[cb][2][r] - t[cb][0][r] - t[cb][1][r];
        *reinterpret_cast<double2*>(dst + ((4 * r + kr) * t0.ld + kc * sizeof(double2))) = o;
      }
    }
  }
}

// strip t's rows of the pair's columns from one buffer to the other (an
// unrotated pair whose X changes buffers)
__device__ __forceinline__ void strip_copy(const Strip& t, int b) {
  const int lane = threadIdx.x & 63, kr = lane >> 4;
  if ((lane & 15) >= t.rows) return;
#pragma unroll 1
  for (int s = 0; s < B2MAX / 4; ++s) {
    const size_t off = (4 * (s & 3) + kr) * t.ld + (lane & 15) * sizeof(double2);
    if (4 * s + kr < 2 * b)
      *reinterpret_cast<double2*>(t.dst[s >> 2] + off) = *reinterpret_cast<const double2*>(t.src[s >> 2] + off);
  }
}

// Pair (I, J) of item p in round `round` (mode 0: the fixed pairs (2p, 2p+1);
// mode 1: the circle pairs).
__device__ __forceinline__ void round_pair(int p, int round, int mode, int nb, int& I, int& J) {
  I = 2 * p;
  J = 2 * p + 1;
  if (mode == 1) {
    I = circle_pos(p, round, nb);
    J = circle_pos(nb - 1 - p, round, nb);
    if (I > J) {
      const int t = I;
      I = J;
      J = t;
    }
  }
}

// One round in one launch: the Gram and the rotation of X (and of V when
// accumulated) on FP64 MFMA, the inner solve between them.
//
// A pair is one workgroup, in place, or q workgroups: each forms the whole
// Gram and solves the same inner problem (the same sums in the same order, so
// the same W), then rotates its own share of the strips.  As the others may
// still be reading X for their Gram, X then goes to the problem's second
// buffer; an unrotated pair is copied there.  The q workgroups of a pair lie
// eight apart in the grid: on one XCD, whose L2 holds the pair's columns for
// all of them.  With at most four strips per workgroup each strip goes to two
// waves, one per 16 output columns, loaded before the inner solve, whose
// barriers part those loads from the stores of the other wave.
//
// Why: with few pairs (one matrix, or the rounds that only the largest
// problems of a batch reach) a workgroup that rotates all rows of X and V is
// the whole round: 63 us at 512 rows of each, 30 us cut.  Such a round is a
// chain: launch 3 us, Gram 8 us at 256 rows (loads, then 2450 cycles per 64
// rows), inner solve 9 us (a sweep's first, fixed-pair round 17), rotation 2 us
// (one 256 x 256 matrix: 21.5 us a round; with two launches, the partial Grams
// on the VALU, it was 36).  With two workgroups on each CU (ALONE = false: 496
// pairs of 512 rows, 74 us in a whole sweep) a round fetches 193 MB of X, read
// twice, and writes 93 beyond the L2s (3.9 TB/s) at 24 TFLOP/s: neither is the
// bound, but the same chain, of which two workgroups hide a part of each other's.
// mode 0: full inner sweep on the fixed pairs; mode 1: cross-block inner steps.
//
// UNITS: a batch's unit list and problem table, else the one problem among the
// kernel's arguments (a choice at run time made every field a branch and a
// scalar load that the next one waited for).
// FIRST: the converged flag is waited for before the Gram's first loads go out,
// not while they are under way.  A captured run's fixed number of sweeps
// consists mostly of rounds over converged problems, whose loads (all of X at
// 256 rows) are then not made: the n = 64, chi = 256 Vidal sweep replayed from
// graphs 349 -> 326 ms, 31 captured 256 x 256 problems 8.2 -> 6.6 ms.
constexpr int NXCD = SVD_XCDS;
constexpr unsigned NCU = SVD_XCDS * SVD_XCD_CUS;

template <bool ALONE, bool UNITS, bool FIRST>
__global__ __launch_bounds__(SR_THREADS, ALONE ? 2 : 4) void svd_round_mfma_kernel(SvdBatch Bt, int round, int mode) {
  __shared__ SvSmem sm;
  int prob = 0, p, c, q, flip;
  if constexpr (UNITS) {
    const int4 u = Bt.units[blockIdx.x];
    if (u.x < 0) return;  // padding of the list
    prob = u.x;
    p = u.y;
    c = u.z & 0xffff;
    q = u.z >> 16;
    flip = u.w;
  } else {
    q = Bt.one.q;
    const int k = blockIdx.x / NXCD;
    p = blockIdx.x % NXCD + NXCD * (k / q);
    c = k % q;
    flip = q > 1 ? 2 : 0;
  }
  const SvdProblem& P = UNITS ? Bt.arr[prob] : Bt.one;
  const int converged = P.flag[1];
  if (FIRST && converged) return;
  const int nb = P.nblk;
  if (mode == 1 && (nb <= 2 || round >= nb - 1)) return;
  if (p >= nb / 2) return;
  int I, J;
  round_pair(p, round, mode, nb, I, J);
  const int b = P.b, n2 = 2 * b;
  const double* Xs = (flip & 1) ? P.X2 : P.X;
  double* Xd = (flip & 2) ? P.X2 : P.X;
  const double abs_tol = fmax(4.930380657631324e-32 * (*P.fro2), 1e-300), tol = P.tol;
  if (!gram_mfma<(ALONE ? 4 : 2), FIRST>(sm, Xs, P.nr, 0, P.nr, I, J, b, converged)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int S = strip_count(P);
  const int lo = (int)((int64_t)c * S / q), hi = (int)((int64_t)(c + 1) * S / q);
  const bool narrow = ALONE && q > 1 && hi - lo <= SR_THREADS / 128;
  double2 x[B2MAX / 4];
  if (narrow && lo + (wave >> 1) < hi) strip_load(x, strip_of(P, Xs, Xd, lo + (wave >> 1), I, J), b);
  inner_solve(sm, n2, mode, tol, abs_tol);
  if (threadIdx.x == 0 && c == 0) {
    if (sm.any_outer) P.flag[0] = 1;
    if (sm.any_big) P.flag[3] = 1;
  }
  const bool still = !sm.any_outer;  // pair already orthogonal: W = I (uniform)
  if (still) {
    if (Xs == Xd) return;
    for (int i = lo + wave; i < hi; i += SR_THREADS / 64) {
      const Strip t = strip_of(P, Xs, Xd, i, I, J);
      if (t.src[0] != t.dst[0]) strip_copy(t, b);
    }
    return;
  }
  if (narrow) {
    const int i = lo + (wave >> 1);
    if (i < hi) strip_rotate<1>(sm, x, strip_of(P, Xs, Xd, i, I, J), wave & 1, b);
    return;
  }
  for (int i = lo + wave; i < hi; i += SR_THREADS / 64) {
    const Strip t = strip_of(P, Xs, Xd, i, I, J);
    strip_load(x, t, b);
    strip_rotate<2>(sm, x, t, 0, b);
  }
}

// Rounds with each pair split over q workgroups by rows (phase 0: partial
// Grams; phase 1: reduce, inner solve, rotate the workgroup's row chunk), on
// the VALU with LDS staging.
// mode 0: full inner sweep on the fixed pairs (2p, 2p+1) (one such round per
// sweep); mode 1: cross-block inner steps on the circle pairs of `round`.
__global__ __launch_bounds__(SR_THREADS) void svd_round_kernel(SvdBatch Bt, int round, int phase, int mode) {
  __shared__ SvSmem sm;
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.y] : Bt.one;
  if (P.flag[1]) return;  // converged
  const int nb = P.nblk;
  // a single block pair (nb = 2) is swept whole in the mode-0 round; cross
  // rounds exist only for nb > 2, where every block is b = 16 wide
  if (mode == 1 && (nb <= 2 || round >= nb - 1)) return;
  const int q = P.q;
  const int item = blockIdx.x;
  const int p = item / q, c = item % q;
  if (p >= nb / 2) return;
  int I, J;
  round_pair(p, round, mode, nb, I, J);
  const int b = P.b, n2 = 2 * b;
  const int rcx = (P.nr + q - 1) / q;
  const int r0 = c * rcx, r1 = min(P.nr, r0 + rcx);
  double ar[GE_PER_THREAD], ai[GE_PER_THREAD];

  if (phase == 0) {
    gram_over_rows(sm, P.X, P.nr, r0, r1, I, J, b, ar, ai);
    double* out = P.Gpart + ((size_t)p * q + c) * (size_t)n2 * n2 * 2;
    if ((int)threadIdx.x < (n2 / 2) * (n2 / 2)) {
#pragma unroll
      for (int t = 0; t < GE_PER_THREAD; ++t) {
        int row, col;
        gram_slot(n2, t, row, col);
        const int e = col * n2 + row;
        out[2 * e] = ar[t];
        out[2 * e + 1] = ai[t];
      }
    }
    return;
  }
  {
    for (int t = 0; t < GE_PER_THREAD; ++t) {
      ar[t] = 0.0;
      ai[t] = 0.0;
    }
    // the q chunk partials in chunk order, four chunks' loads in flight at once
    if ((int)threadIdx.x < (n2 / 2) * (n2 / 2)) {
      int eo[GE_PER_THREAD];
#pragma unroll
      for (int t = 0; t < GE_PER_THREAD; ++t) {
        int row, col;
        gram_slot(n2, t, row, col);
        eo[t] = col * n2 + row;
      }
      const double2* base = reinterpret_cast<const double2*>(P.Gpart) + (size_t)p * q * n2 * n2;
      for (int cc = 0; cc < q; cc += 4) {
        double2 g[4][GE_PER_THREAD];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int t = 0; t < GE_PER_THREAD; ++t) {
            g[u][t].x = 0.0;
            g[u][t].y = 0.0;
            if (cc + u < q) g[u][t] = base[(size_t)(cc + u) * n2 * n2 + eo[t]];
          }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (cc + u < q)
#pragma unroll
            for (int t = 0; t < GE_PER_THREAD; ++t) {
              ar[t] += g[u][t].x;
              ai[t] += g[u][t].y;
            }
      }
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < (n2 / 2) * (n2 / 2)) {
#pragma unroll
    for (int t = 0; t < GE_PER_THREAD; ++t) {
      int row, col;
      gram_slot(n2, t, row, col);
      sm.gr[row][col] = ar[t];
      sm.gi[row][col] = ai[t];
    }
  }
  __syncthreads();
  // One cyclic sweep of the 2b x 2b problem per pair visit (the outer sweeps
  // converge regardless; a full inner diagonalisation costs ~5x more).  Rotations are skipped only below eps^2 ||A||_F^2: a larger
  // absolute floor (e.g. eps ||A||_F^2) stops the late small-angle rotations
  // that give one-sided Jacobi its accuracy on small singular values.
  const double abs_tol = fmax(4.930380657631324e-32 * (*P.fro2), 1e-300);
  inner_solve(sm, n2, mode, P.tol, abs_tol);
  if (threadIdx.x == 0 && c == 0) {
    if (sm.any_outer) P.flag[0] = 1;
    if (sm.any_big) P.flag[3] = 1;
  }
  if (!sm.any_outer) return;  // pair already orthogonal: W = I (uniform branch)
  apply_rows(sm, P.X, P.nr, r0, r1, I, J, b);
  if (!P.accum) return;
  const int rcv = (P.ncp + q - 1) / q;
  const int v0 = c * rcv;
  const int v1 = min(P.ncp, v0 + rcv);
  apply_rows(sm, P.V, P.ncp, v0, v1, I, J, b);
}

__global__ void svd_sweep_end_kernel(SvdBatch Bt, int64_t nprob) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nprob) return;
  const SvdProblem& P = Bt.arr ? Bt.arr[i] : Bt.one;
  if (P.flag[1]) return;
  // Converged when a sweep rotated nothing, or when no relative off-diagonal
  // of it was above sqrt(tol) / 2 (squared: tol / 4): one-sided
  // Jacobi converges quadratically, so after such a sweep every pair's
  // cosine is ~ that squared, below tol, and the verification sweep would
  // rotate nothing.
  if (P.flag[0] == 0 || P.flag[3] == 0) P.flag[1] = 1;
  P.flag[0] = 0;
  P.flag[2] += 1;
  P.flag[3] = 0;
}

// X (nr x ncp) from A or A^H with zero padding; V = I.
template <typename S2>
__global__ void svd_init_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.y] : Bt.one;
  const size_t nx = (size_t)P.nr * P.ncp, nv = (size_t)P.ncp * P.ncp;
  const S2* A = static_cast<const S2*>(P.A);
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < nx + nv; e += (size_t)gridDim.x * blockDim.x) {
    double2 v;
    v.x = 0.0;
    v.y = 0.0;
    if (e < nx) {
      const int r = (int)(e % P.nr), c = (int)(e / P.nr);
      if (c < P.ncols) {
        if (P.pre) {  // X = R^H, R the upper triangle of W (ld m)
          if (c <= r) {
            const double2 a = reinterpret_cast<const double2*>(P.W)[(size_t)r * P.m + c];
            v.x = a.x;
            v.y = -a.y;
          }
        } else if (!P.transposed) {
          const S2 a = A[(size_t)c * P.lda + r];
          v.x = a.x;
          v.y = a.y;
        } else {  // X = A^H : X[r][c] = conj(A[c][r])
          const S2 a = A[(size_t)r * P.lda + c];
          v.x = a.x;
          v.y = -(double)a.y;
        }
      }
      reinterpret_cast<double2*>(P.X)[e] = v;
    } else if (P.accum) {
      const size_t f = e - nx;
      const int r = (int)(f % P.ncp), c = (int)(f / P.ncp);
      v.x = (r == c) ? 1.0 : 0.0;
      reinterpret_cast<double2*>(P.V)[f] = v;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    P.flag[0] = 0;
    P.flag[1] = 0;
    P.flag[2] = 0;
    P.flag[3] = 0;
  }
}

// ||X||_F^2, one workgroup per problem, fixed summation order
// Column norms sqrt(sum_r |X[r][j]|^2) into sigma[j], one wave per column
// (grid.x covers ncp / 4 columns per problem).  Deterministic.
__global__ __launch_bounds__(SV_THREADS) void svd_colnorm_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.y] : Bt.one;
  const int lane = threadIdx.x & 63;
  const int j = blockIdx.x * (SV_THREADS / 64) + (threadIdx.x >> 6);
  if (j >= P.ncp) return;
  const double2* col = reinterpret_cast<const double2*>(P.X) + (size_t)j * P.nr;
  double s = 0.0;
  for (int r = lane; r < P.nr; r += 64) {
    const double2 v = col[r];
    s += v.x * v.x + v.y * v.y;
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) P.sigma[j] = sqrt(s);
}

// ||X||_F^2 from the column norms, one workgroup per problem, fixed order
__global__ __launch_bounds__(SV_THREADS) void svd_fro_kernel(SvdBatch Bt) {
  __shared__ double red[SV_THREADS / 64];
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.x] : Bt.one;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double s = 0.0;
  for (int j = tid; j < P.ncp; j += SV_THREADS) s += P.sigma[j] * P.sigma[j];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  if (tid == 0) *P.fro2 = red[0] + red[1] + red[2] + red[3];
}

// norms, descending sort, S, kept count and discarded weight
__global__ __launch_bounds__(SV_THREADS) void svd_sort_kernel(SvdBatch Bt) {
  __shared__ double key[SORT_MAX];
  __shared__ int idx[SORT_MAX];
  __shared__ double red[SV_THREADS / 64];
  __shared__ int cnt[SV_THREADS / 64];
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.x] : Bt.one;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ncp = P.ncp;
  int np2 = 1;
  while (np2 < ncp) np2 <<= 1;
  // column norms were written to sigma by svd_colnorm_kernel
  for (int j = tid; j < np2; j += SV_THREADS) {
    key[j] = (j < ncp) ? P.sigma[j] : -1.0;
    idx[j] = j;
  }
  __syncthreads();
  // bitonic sort, descending by key, ties by index
  for (int size = 2; size <= np2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < np2; i += SV_THREADS) {
        const int j = i ^ stride;
        if (j > i) {
          const bool desc = ((i & size) == 0);
          const double ki = key[i], kj = key[j];
          const int ii = idx[i], ij = idx[j];
          const bool i_first = (ki > kj) || (ki == kj && ii < ij);
          if (desc != i_first) {
            key[i] = kj;
            key[j] = ki;
            idx[i] = ij;
            idx[j] = ii;
          }
        }
      }
      __syncthreads();
    }
  }
  const int kmax = P.ncols;
  for (int j = tid; j < kmax; j += SV_THREADS) {
    P.sigma[j] = key[j];
    P.perm[j] = idx[j];
    if (P.S) {
      if (P.s_mode == 1) {
        reinterpret_cast<double2*>(P.S)[j] = make_double2(key[j], 0.0);
      } else if (P.s_mode == 2) {
        reinterpret_cast<float2*>(P.S)[j] = make_float2((float)key[j], 0.0f);
      } else {
        P.S[j] = key[j];
      }
    }
  }
  // kept count: min(maxdim, #(s > threshold)) -- a prefix since s descends
  int kcap = (P.maxdim > 0 && P.maxdim < kmax) ? (int)P.maxdim : kmax;
  int c = 0;
  for (int j = tid; j < kcap; j += SV_THREADS) c += (P.threshold > 0.0) ? (key[j] > P.threshold) : 1;
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
  if (lane == 0) cnt[wave] = c;
  __syncthreads();
  int k = 0;
  for (int w = 0; w < SV_THREADS / 64; ++w) k += cnt[w];
  double d = 0.0;
  for (int j = k + tid; j < kmax; j += SV_THREADS) d += key[j] * key[j];
  for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
  if (lane == 0) red[wave] = d;
  __syncthreads();
  if (tid == 0) {
    double disc = 0.0;
    for (int w = 0; w < SV_THREADS / 64; ++w) disc += red[w];
    if (P.k_dev) *P.k_dev = k;
    if (P.disc_dev) *P.disc_dev = disc;
  }
}

// QR preconditioning of the grouped problems with pre set: the column norms
// of A (one wave per column) into sigma (free until the Jacobi's own column
// norms), their descending order (ties by index) into cperm, and
// W[:, c] = A[:, cperm[c]] in complex128.  Sorting the columns first makes
// the unpivoted QR's R rows decrease in norm, as with column pivoting: on
// Vidal-gauge bond matrices the Jacobi on R^H then needs ~9 sweeps where the
// plain one needs ~14.
template <typename S2>
__global__ __launch_bounds__(SV_THREADS) void svd_pre_norm_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr[blockIdx.y];
  if (!P.pre) return;
  const int lane = threadIdx.x & 63;
  const int j = blockIdx.x * (SV_THREADS / 64) + (threadIdx.x >> 6);
  if (j >= P.n) return;
  const S2* col = static_cast<const S2*>(P.A) + (size_t)j * P.lda;
  double s = 0.0;
  for (int r = lane; r < P.m; r += 64) {
    const S2 v = col[r];
    s += (double)v.x * v.x + (double)v.y * v.y;
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) P.sigma[j] = s;
}

__global__ __launch_bounds__(SV_THREADS) void svd_pre_sort_kernel(SvdBatch Bt) {
  __shared__ double key[SORT_MAX];
  __shared__ int idx[SORT_MAX];
  const SvdProblem& P = Bt.arr[blockIdx.x];
  if (!P.pre) return;
  const int tid = threadIdx.x, n = P.n;
  int np2 = 1;
  while (np2 < n) np2 <<= 1;
  for (int j = tid; j < np2; j += SV_THREADS) {
    key[j] = (j < n) ? P.sigma[j] : -1.0;
    idx[j] = j;
  }
  __syncthreads();
  for (int size = 2; size <= np2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < np2; i += SV_THREADS) {
        const int j = i ^ stride;
        if (j > i) {
          const bool desc = ((i & size) == 0);
          const double ki = key[i], kj = key[j];
          const int ii = idx[i], ij = idx[j];
          const bool i_first = (ki > kj) || (ki == kj && ii < ij);
          if (desc != i_first) {
            key[i] = kj;
            key[j] = ki;
            idx[i] = ij;
            idx[j] = ii;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int j = tid; j < n; j += SV_THREADS) P.cperm[j] = idx[j];
}

template <typename S2>
__global__ void svd_pre_pack_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr[blockIdx.y];
  if (!P.pre) return;
  const size_t total = (size_t)P.m * P.n;
  const S2* A = static_cast<const S2*>(P.A);
  double2* W = reinterpret_cast<double2*>(P.W);
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(e % P.m), c = (int)(e / P.m);
    const S2 a = A[(size_t)P.cperm[c] * P.lda + r];
    W[e] = make_double2((double)a.x, (double)a.y);
  }
}

// U (m x kmax) and Vh (kmax x n) from X, V and the permutation.
template <typename S2>
__global__ void svd_write_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.y] : Bt.one;
  const int kmax = P.ncols;
  const size_t nu = (size_t)P.m * kmax, nvh = (size_t)kmax * P.n;
  const double2* X = reinterpret_cast<const double2*>(P.X);
  const double2* V = reinterpret_cast<const double2*>(P.V);
  S2* U = static_cast<S2*>(P.U);
  S2* Vh = static_cast<S2*>(P.Vh);
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < nu + nvh; e += (size_t)gridDim.x * blockDim.x) {
    S2 o;
    if (e < nu) {
      if (!U) continue;  // U not requested
      const int r = (int)(e % P.m), j = (int)(e / P.m);
      const int pj = P.perm[j];
      const double s = P.sigma[j];
      double vr, vi;
      if (!P.transposed) {
        const double2 x = X[(size_t)pj * P.nr + r];
        vr = s > 0.0 ? x.x / s : 0.0;
        vi = s > 0.0 ? x.y / s : 0.0;
      } else {
        const double2 x = V[(size_t)pj * P.ncp + r];
        vr = x.x;
        vi = x.y;
      }
      o.x = vr;
      o.y = vi;
      U[(size_t)j * P.ldu + r] = o;
    } else {
      const size_t f = e - nu;
      const int j = (int)(f % kmax), cidx = (int)(f / kmax);
      const int pj = P.perm[j];
      const double s = P.sigma[j];
      double vr, vi;
      if (!P.transposed) {
        const double2 x = V[(size_t)pj * P.ncp + cidx];
        vr = x.x;
        vi = -x.y;
      } else {
        const double2 x = X[(size_t)pj * P.nr + cidx];
        vr = s > 0.0 ? x.x / s : 0.0;
        vi = s > 0.0 ? -x.y / s : 0.0;
      }
      o.x = vr;
      o.y = vi;
      // preconditioned: X's row c belongs to A's column cperm[c]
      Vh[(size_t)(P.pre ? P.cperm[cidx] : cidx) * P.ldvh + j] = o;
    }
  }
}

// Orthonormal completion of the factor built as X_j / sigma_j (U, or V^H's
// rows when the Jacobi ran on A^H): for kept singular values (j < k of the
// truncation) at or below 1e-8 sigma_0 that column carries X's rounding
// noise, not an orthonormal direction (exactly zero sigma: a zero column).  Each such column j, in
// order, is projected off columns 0..j-1 twice (classical Gram-Schmidt with
// reorthogonalisation) and normalised; if too little of it survives (below
// 1e-3 of its length before), the unit vector e_t (t = j, j+1, ... mod L)
// is used instead.  The result is an orthonormal completion as LAPACK
// returns it; the product U diag(S) V^H changes by at most
// 1e-8 sigma_0 * O(eps) per column.  Such columns form the tail [j0, k) (sigma
// descends); their projections off the head [0, j0) run in parallel
// (svd_complete_head_kernel), the serial part is the tail alone
// (svd_complete_kernel, one workgroup per problem).  A problem without such
// columns returns at once.
constexpr int CP_THREADS = 256;
constexpr int CP_MAX_K = 4096;
constexpr int CP_HEAD_BLOCKS = 32;  // workgroups per problem projecting tail columns off the head

template <typename S2>
struct Fac {
  S2* p;
  int64_t ld;
  bool adj;  // column j of F is conj(row j of V^H)
  __device__ __forceinline__ double2 get(int64_t r, int64_t j) const {
    const S2 v = adj ? p[r * ld + j] : p[j * ld + r];
    double2 o;
    o.x = (double)v.x;
    o.y = adj ? -(double)v.y : (double)v.y;
    return o;
  }
  __device__ __forceinline__ void put(int64_t r, int64_t j, double re, double im) const {
    S2 o;
    o.x = re;
    o.y = adj ? -im : im;
    if (adj)
      p[r * ld + j] = o;
    else
      p[j * ld + r] = o;
  }
};

__device__ __forceinline__ double cp_wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ double cp_block_sum(double v, double* red) {
  v = cp_wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < CP_THREADS / 64; ++w) t += red[w];
  return t;
}

// The factor to complete and its extent: U (m rows) or, when the Jacobi ran
// on A^H, the rows of V^H (n entries each, read as columns of F).
template <typename S2>
__device__ __forceinline__ bool cp_setup(const SvdProblem& P, Fac<S2>& F, int64_t& L, int& klim, int& j0) {
  const int kmax = P.ncols;
  if (kmax > CP_MAX_K) return false;
  if (!P.transposed) {
    if (!P.U) return false;
    F.p = static_cast<S2*>(P.U);
    F.ld = P.ldu;
    F.adj = false;
    L = P.m;
  } else {
    F.p = static_cast<S2*>(P.Vh);
    F.ld = P.ldvh;
    F.adj = true;
    L = P.n;
  }
  // only the kept columns (the truncation's k, written by the sort kernel)
  // are completed: the caller drops the others (a TEBD bond matrix of rank
  // 256 in 512 columns would otherwise orthogonalise 256 discarded ones)
  klim = P.k_dev ? (int)min((int64_t)kmax, *P.k_dev) : kmax;
  // sigma descends: the columns to complete are the tail [j0, klim)
  const double tau = P.sigma[0] * 1e-8;
  int lo = 0, hi = klim;
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (P.sigma[mid] > tau)
      lo = mid + 1;
    else
      hi = mid;
  }
  j0 = lo;
  return j0 < klim;
}

// Two passes (classical Gram-Schmidt with reorthogonalisation) of column j
// against columns [lo, hi) of F.
template <typename S2>
__device__ __forceinline__ void cp_project(const Fac<S2>& F, int64_t L, int lo, int hi, int j, double* cr, double* ci) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int pass = 0; pass < 2; ++pass) {
    // c = F[:, lo:hi]^H v
    if (!F.adj) {
      // columns contiguous: one wave per column, lanes over rows
      for (int i = lo + wave; i < hi; i += CP_THREADS / 64) {
        double sr = 0.0, si = 0.0;
        for (int64_t r = lane; r < L; r += 64) {
          const double2 a = F.get(r, i), v = F.get(r, j);
          sr += a.x * v.x + a.y * v.y;
          si += a.x * v.y - a.y * v.x;
        }
        sr = cp_wave_sum(sr);
        si = cp_wave_sum(si);
        if (lane == 0) {
          cr[i] = sr;
          ci[i] = si;
        }
      }
    } else {
      // rows of V^H: F's column index is the contiguous one, so one
      // thread per column i walks the rows (v[r] is the same for all)
      for (int i = lo + tid; i < hi; i += CP_THREADS) {
        double sr = 0.0, si = 0.0;
        for (int64_t r = 0; r < L; ++r) {
          const double2 a = F.get(r, i), v = F.get(r, j);
          sr += a.x * v.x + a.y * v.y;
          si += a.x * v.y - a.y * v.x;
        }
        cr[i] = sr;
        ci[i] = si;
      }
    }
    __syncthreads();
    // v -= F[:, lo:hi] c (one thread per row; with V^H's rows each thread
    // walks contiguous memory)
    for (int64_t r = tid; r < L; r += CP_THREADS) {
      double2 v = F.get(r, j);
      for (int i = lo; i < hi; ++i) {
        const double2 a = F.get(r, i);
        v.x -= a.x * cr[i] - a.y * ci[i];
        v.y -= a.x * ci[i] + a.y * cr[i];
      }
      F.put(r, j, v.x, v.y);
    }
    __syncthreads();
  }
}

// Step 1, in parallel over the tail columns (grid.x workgroups per problem):
// each column's length before any projection goes to n0 (the Jacobi work
// matrix X, free once V^H and U are written), then the column is projected
// off the head columns [0, j0), which are orthonormal to working accuracy.
template <typename S2>
__global__ __launch_bounds__(CP_THREADS) void svd_complete_head_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.y] : Bt.one;
  Fac<S2> F;
  int64_t L;
  int klim, j0;
  if (!cp_setup(P, F, L, klim, j0)) return;
  __shared__ double cr[CP_MAX_K], ci[CP_MAX_K];
  __shared__ double red[CP_THREADS / 64];
  double* n0s = P.X;
  for (int j = j0 + blockIdx.x; j < klim; j += gridDim.x) {
    double n0 = 0.0;
    for (int64_t r = threadIdx.x; r < L; r += CP_THREADS) {
      const double2 v = F.get(r, j);
      n0 += v.x * v.x + v.y * v.y;
    }
    n0 = sqrt(cp_block_sum(n0, red));
    if (threadIdx.x == 0) n0s[j] = n0;
    if (n0 > 0.0 && j0 > 0) cp_project(F, L, 0, j0, j, cr, ci);
    __syncthreads();
  }
}

// Step 2, one workgroup per problem: each tail column in order is projected
// off the tail columns before it and normalised; if too little of it
// survives (below 1e-3 of its length before step 1), the unit vector e_t
// (t = j, j+1, ... mod L) is projected off every column before it instead.
template <typename S2>
__global__ __launch_bounds__(CP_THREADS) void svd_complete_kernel(SvdBatch Bt) {
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.y] : Bt.one;
  Fac<S2> F;
  int64_t L;
  int klim, j0;
  if (!cp_setup(P, F, L, klim, j0)) return;
  __shared__ double cr[CP_MAX_K], ci[CP_MAX_K];
  __shared__ double red[CP_THREADS / 64];
  const int tid = threadIdx.x;
  const double* n0s = P.X;
  int64_t next_unit = 0;
  for (int j = j0; j < klim; ++j) {
    const double n0 = n0s[j];
    bool unit = !(n0 > 0.0);
    if (!unit) cp_project(F, L, j0, j, j, cr, ci);
    for (int attempt = 0; attempt < 16; ++attempt) {
      if (unit) {
        // e_t, t taken in turn from the unit vectors not yet tried
        const int64_t t = (j + next_unit++) % L;
        for (int64_t r = tid; r < L; r += CP_THREADS) F.put(r, j, r == t ? 1.0 : 0.0, 0.0);
        __syncthreads();
        cp_project(F, L, 0, j, j, cr, ci);
      }
      double nn = 0.0;
      for (int64_t r = tid; r < L; r += CP_THREADS) {
        const double2 v = F.get(r, j);
        nn += v.x * v.x + v.y * v.y;
      }
      nn = sqrt(cp_block_sum(nn, red));
      if (nn > 1e-3 * (unit ? 1.0 : n0)) {
        const double inv = 1.0 / nn;
        for (int64_t r = tid; r < L; r += CP_THREADS) {
          const double2 v = F.get(r, j);
          F.put(r, j, v.x * inv, v.y * inv);
        }
        __syncthreads();
        break;
      }
      unit = true;
    }
  }
}

// After a fixed number of captured sweeps: bit 0 of *status is set for a
// problem whose sweeps did not converge (the graph's caller reads it).
__global__ void svd_status_kernel(SvdBatch Bt, int32_t* status) {
  const SvdProblem& P = Bt.arr ? Bt.arr[blockIdx.x] : Bt.one;
  if (threadIdx.x == 0 && !P.flag[1]) atomicOr(status, 1);
}

#define TRY_HIP_COLNORM(b, nprob, max_ncp, s)                                                             \
  do {                                                                                                    \
    hipLaunchKernelGGL(svd_colnorm_kernel, dim3((unsigned)(((max_ncp) + SV_THREADS / 64 - 1) / (SV_THREADS / 64)), \
                                                (unsigned)(nprob)),                                       \
                       dim3(SV_THREADS), 0, s, b);                                                        \
    TENET_HIP_CHECK(hipGetLastError());                                                                   \
  } while (0)

int launch_svd_init(const SvdBatch& b, int64_t nprob, int64_t max_elems, int max_ncp, int dtype, hipStream_t s) {
  const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>((max_elems + 255) / 256, 1024));
  if (dtype == TENET_C128)
    hipLaunchKernelGGL(svd_init_kernel<double2>, dim3(gx, (unsigned)nprob), dim3(256), 0, s, b);
  else
    hipLaunchKernelGGL(svd_init_kernel<float2>, dim3(gx, (unsigned)nprob), dim3(256), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  TRY_HIP_COLNORM(b, nprob, max_ncp, s);
  hipLaunchKernelGGL(svd_fro_kernel, dim3((unsigned)nprob), dim3(SV_THREADS), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

int launch_svd_round(const SvdBatch& b, int64_t nprob, int max_items, int round, int phase, int mode, bool flag_first,
                     hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  if (b.units && phase != 2) {
    set_error("SVD round: unit lists need the fused round kernel");
    return TENET_ERR_UNSUPPORTED;
  }
  // with a unit list, max_items is its length
  // one matrix in one launch: its pairs dealt over the XCDs, padded to whole rows of NXCD
  const int dealt = (max_items + NXCD - 1) / NXCD * NXCD * (phase == 2 && !b.arr ? b.one.q : 1);
  const dim3 grid = b.units ? dim3((unsigned)max_items)
                            : (phase == 2 ? dim3((unsigned)dealt) : dim3((unsigned)max_items, (unsigned)nprob));
  if (phase == 2) {
    // one matrix has at most one workgroup with work per CU (svd_row_shares)
    const auto pick = [&](auto first) {
      constexpr bool F = decltype(first)::value;
      return !b.units        ? svd_round_mfma_kernel<true, false, F>
             : grid.x <= NCU ? svd_round_mfma_kernel<true, true, F>
                             : svd_round_mfma_kernel<false, true, F>;
    };
    const auto kernel = flag_first ? pick(std::true_type{}) : pick(std::false_type{});
    if (ev0)
      hipExtLaunchKernelGGL(kernel, grid, dim3(SR_THREADS), 0, s, ev0, ev1, 0, b, round, mode);
    else
      hipLaunchKernelGGL(kernel, grid, dim3(SR_THREADS), 0, s, b, round, mode);
  } else if (ev0) {
    hipExtLaunchKernelGGL(svd_round_kernel, grid, dim3(SR_THREADS), 0, s, ev0, ev1, 0, b, round, phase, mode);
  } else {
    hipLaunchKernelGGL(svd_round_kernel, grid, dim3(SR_THREADS), 0, s, b, round, phase, mode);
  }
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

int launch_svd_sweep_end(const SvdBatch& b, int64_t nprob, hipStream_t s) {
  hipLaunchKernelGGL(svd_sweep_end_kernel, dim3((unsigned)((nprob + 255) / 256)), dim3(256), 0, s, b, nprob);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

int launch_svd_finalize(const SvdBatch& b, int64_t nprob, int max_ncp, int64_t max_elems, int dtype,
                        hipStream_t s) {
  if (max_ncp > SORT_MAX) {
    set_error("SVD: min(m, n) exceeds the sort limit (4096)");
    return TENET_ERR_UNSUPPORTED;
  }
  TRY_HIP_COLNORM(b, nprob, max_ncp, s);
  hipLaunchKernelGGL(svd_sort_kernel, dim3((unsigned)nprob), dim3(SV_THREADS), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>((max_elems + 255) / 256, 2048));
  if (dtype == TENET_C128)
    hipLaunchKernelGGL(svd_write_kernel<double2>, dim3(gx, (unsigned)nprob), dim3(256), 0, s, b);
  else
    hipLaunchKernelGGL(svd_write_kernel<float2>, dim3(gx, (unsigned)nprob), dim3(256), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  if (dtype == TENET_C128) {
    hipLaunchKernelGGL(svd_complete_head_kernel<double2>, dim3(CP_HEAD_BLOCKS, (unsigned)nprob), dim3(CP_THREADS), 0,
                       s, b);
    TENET_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(svd_complete_kernel<double2>, dim3(1, (unsigned)nprob), dim3(CP_THREADS), 0, s, b);
  } else {
    hipLaunchKernelGGL(svd_complete_head_kernel<float2>, dim3(CP_HEAD_BLOCKS, (unsigned)nprob), dim3(CP_THREADS), 0,
                       s, b);
    TENET_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(svd_complete_kernel<float2>, dim3(1, (unsigned)nprob), dim3(CP_THREADS), 0, s, b);
  }
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

int launch_svd_pre_pack(const SvdBatch& b, int64_t nprob, int max_n, int64_t max_elems, int dtype, hipStream_t s) {
  if (max_n > SORT_MAX) {
    set_error("SVD preconditioning: n exceeds the sort limit (4096)");
    return TENET_ERR_UNSUPPORTED;
  }
  const dim3 gn((unsigned)((max_n + SV_THREADS / 64 - 1) / (SV_THREADS / 64)), (unsigned)nprob);
  if (dtype == TENET_C128)
    hipLaunchKernelGGL(svd_pre_norm_kernel<double2>, gn, dim3(SV_THREADS), 0, s, b);
  else
    hipLaunchKernelGGL(svd_pre_norm_kernel<float2>, gn, dim3(SV_THREADS), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(svd_pre_sort_kernel, dim3((unsigned)nprob), dim3(SV_THREADS), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>((max_elems + 255) / 256, 1024));
  if (dtype == TENET_C128)
    hipLaunchKernelGGL(svd_pre_pack_kernel<double2>, dim3(gx, (unsigned)nprob), dim3(256), 0, s, b);
  else
    hipLaunchKernelGGL(svd_pre_pack_kernel<float2>, dim3(gx, (unsigned)nprob), dim3(256), 0, s, b);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

// Single-matrix form of the column ordering (tenet_svd_thin's preconditioned
// path): T = A (adj = 0, rows x cols = m x n) or A^H (adj = 1, n x m);
// norms of T's columns, their descending order (ties by index) into perm, and
// Tp = T[:, perm] in complex128 (rows x cols, ld rows).
template <typename S2>
__global__ __launch_bounds__(SV_THREADS) void pre1_norm_kernel(const S2* __restrict__ A, int64_t lda, int rows,
                                                                int cols, int adj, double* __restrict__ nrm) {
  const int lane = threadIdx.x & 63;
  const int j = blockIdx.x * (SV_THREADS / 64) + (threadIdx.x >> 6);
  if (j >= cols) return;
  double s = 0.0;
  for (int r = lane; r < rows; r += 64) {
    const S2 v = adj ? A[(size_t)r * lda + j] : A[(size_t)j * lda + r];
    s += (double)v.x * v.x + (double)v.y * v.y;
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) nrm[j] = s;
}

__global__ __launch_bounds__(SV_THREADS) void pre1_sort_kernel(const double* __restrict__ nrm, int cols,
                                                                int32_t* __restrict__ perm) {
  __shared__ double key[SORT_MAX];
  __shared__ int idx[SORT_MAX];
  const int tid = threadIdx.x;
  int np2 = 1;
  while (np2 < cols) np2 <<= 1;
  for (int j = tid; j < np2; j += SV_THREADS) {
    key[j] = (j < cols) ? nrm[j] : -1.0;
    idx[j] = j;
  }
  __syncthreads();
  for (int size = 2; size <= np2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < np2; i += SV_THREADS) {
        const int j = i ^ stride;
        if (j > i) {
          const bool desc = ((i & size) == 0);
          const double ki = key[i], kj = key[j];
          const int ii = idx[i], ij = idx[j];
          const bool i_first = (ki > kj) || (ki == kj && ii < ij);
          if (desc != i_first) {
            key[i] = kj;
            key[j] = ki;
            idx[i] = ij;
            idx[j] = ii;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int j = tid; j < cols; j += SV_THREADS) perm[j] = idx[j];
}

template <typename S2>
__global__ void pre1_pack_kernel(const S2* __restrict__ A, int64_t lda, int rows, int cols, int adj,
                                 const int32_t* __restrict__ perm, double2* __restrict__ Tp) {
  const size_t total = (size_t)rows * cols;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(e % rows), c = (int)(e / rows);
    const int pc = perm[c];
    const S2 v = adj ? A[(size_t)r * lda + pc] : A[(size_t)pc * lda + r];
    Tp[e] = make_double2((double)v.x, adj ? -(double)v.y : (double)v.y);
  }
}

// dst from src (complex128, rows x cols, ld lds) through the column order
// perm: mode 0 dst[:, perm[c]] = src[:, c] (ld ldd); mode 1 (conjugate
// transpose) dst[perm[c], r] = conj(src[r, c]).
__global__ void perm_scatter_kernel(const double2* __restrict__ src, int rows, int cols, int64_t lds,
                                    double2* __restrict__ dst, int64_t ldd, const int32_t* __restrict__ perm,
                                    int mode) {
  const size_t total = (size_t)rows * cols;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(e % rows), c = (int)(e / rows);
    const double2 v = src[(size_t)c * lds + r];
    if (mode == 0)
      dst[(size_t)perm[c] * ldd + r] = v;
    else
      dst[(size_t)r * ldd + perm[c]] = make_double2(v.x, -v.y);
  }
}

int launch_pre1_order_pack(const void* A, int64_t lda, int rows, int cols, int adj, int dtype, double* nrm,
                           int32_t* perm, double* Tp, hipStream_t s) {
  if (cols > SORT_MAX) {
    set_error("SVD preconditioning: more than 4096 columns to order");
    return TENET_ERR_UNSUPPORTED;
  }
  const dim3 gn((unsigned)((cols + SV_THREADS / 64 - 1) / (SV_THREADS / 64)));
  if (dtype == TENET_C128)
    hipLaunchKernelGGL(pre1_norm_kernel<double2>, gn, dim3(SV_THREADS), 0, s, (const double2*)A, lda, rows, cols,
                       adj, nrm);
  else
    hipLaunchKernelGGL(pre1_norm_kernel<float2>, gn, dim3(SV_THREADS), 0, s, (const float2*)A, lda, rows, cols, adj,
                       nrm);
  TENET_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(pre1_sort_kernel, dim3(1), dim3(SV_THREADS), 0, s, nrm, cols, perm);
  TENET_HIP_CHECK(hipGetLastError());
  const size_t total = (size_t)rows * cols;
  const unsigned g = (unsigned)std::max<size_t>(1, std::min<size_t>((total + 255) / 256, 2048));
  if (dtype == TENET_C128)
    hipLaunchKernelGGL(pre1_pack_kernel<double2>, dim3(g), dim3(256), 0, s, (const double2*)A, lda, rows, cols, adj,
                       perm, (double2*)Tp);
  else
    hipLaunchKernelGGL(pre1_pack_kernel<float2>, dim3(g), dim3(256), 0, s, (const float2*)A, lda, rows, cols, adj,
                       perm, (double2*)Tp);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

int launch_perm_scatter(const double* src, int rows, int cols, int64_t lds, double* dst, int64_t ldd,
                        const int32_t* perm, int mode, hipStream_t s) {
  const size_t total = (size_t)rows * cols;
  if (total == 0) return TENET_OK;
  const unsigned g = (unsigned)std::max<size_t>(1, std::min<size_t>((total + 255) / 256, 2048));
  hipLaunchKernelGGL(perm_scatter_kernel, dim3(g), dim3(256), 0, s, (const double2*)src, rows, cols, lds,
                     (double2*)dst, ldd, perm, mode);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

int launch_svd_status(const SvdBatch& b, int64_t nprob, int32_t* status, hipStream_t s) {
  hipLaunchKernelGGL(svd_status_kernel, dim3((unsigned)nprob), dim3(64), 0, s, b, status);
  TENET_HIP_CHECK(hipGetLastError());
  return TENET_OK;
}

}  // namespace tenet
