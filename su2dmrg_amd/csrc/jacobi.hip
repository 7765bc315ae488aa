// One-sided block Jacobi SVD, see jacobi.hpp.
#include "jacobi.hpp"

#include <algorithm>
#include <functional>
#include <map>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>
#include <type_traits>

#include "blas1.hpp"
#include "common.hpp"
#include "context.hpp"
#include "ops.hpp"
#include "precond.hpp"
#include "small_svd.hpp"

namespace su2 {

namespace {

constexpr int INNER_SWEEPS = 3; // most inner Jacobi sweeps per visit of a pair
constexpr int MAX_SLICES = 8;   // row slices per pair
constexpr int MIN_SLICE_ROWS = 64;
// A limit up to this many columns, the default among them, preconditions the
// smaller blocks as well: a 192 x 192 block takes 3.7 ms that way (13.3 ms in
// the plain iteration without).
constexpr int kPrecondDefault = 256;
constexpr double kTolAbs = 1e-14;   // rounding floor of a pair, relative to ||A||_F

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x4u __attribute__((ext_vector_type(4), aligned(8)));   // any 8-byte address
typedef double f64x2 __attribute__((ext_vector_type(2)));

struct BlockDesc {
  double* W;        // L x k, ld L
  double* V;        // k x k, ld k
  int L, k;
  double normF;     // Frobenius norm of the block (absolute floor scale)
};

struct PairJob {
  int blk;          // index into the block table
  int p0, bp;       // first column block
  int q0, bq;       // second column block (bq = 0: the first block alone)
  int P;            // row slices (workgroups) that share the pair's Gram matrix
  int full;         // rotate all its columns, not only those of p against q
};

// Threads of the launches that diagonalise a pair and apply its rotations: one
// wave that computes rotations and CB / 4 that apply them.
template <int CB>
struct SolveThreads {
  static constexpr int value = 64 + 16 * CB;
};

// Column of W (or V) of a pair's column c.
__device__ __forceinline__ int pair_column(const PairJob& J, int c) {
  return c < J.bp ? J.p0 + c : J.q0 + (c - J.bp);
}

// 1 / x and 1 / sqrt(x) for x > 0 (normal): the hardware estimates
// refined by two Newton-Raphson steps, y <- y (2 - x y) and
// y <- y (3 - x y^2) / 2, each of which squares the relative error.
__device__ __forceinline__ double recip_nr(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}
__device__ __forceinline__ double rsqrt_nr(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * fma(-hx * y, y, 1.5);
  return y * fma(-hx * y, y, 1.5);
}

// Scaled overlap of two columns from their Gram entries if it calls for a
// rotation, else 0: relative orthogonality, or the rounding floor of columns
// that carry absolute errors of order eps ||A||.  Columns at the rounding
// level of the block carry no direction (the SVD zeroes them) and do not hold
// the iteration open.
__device__ __forceinline__ double pair_overlap(double gab, double ga, double gb, double tol_rel,
                                               double tol_abs, double normF) {
  const double g = fabs(gab), na = sqrt(ga), nb = sqrt(gb);
  if (!(fmin(na, nb) > kNoiseRel * normF)) return 0.0;
  const double scale = na * nb;
  return g > fmax(tol_rel * scale, tol_abs * normF * (na + nb)) ? g / scale : 0.0;
}

// rows [lo, hi) of slice s when L rows are cut into P slices
__device__ __forceinline__ void slice_rows(int L, int P, int s, int& lo, int& hi) {
  const int per = (L + P - 1) / P;
  lo = min(L, s * per);
  hi = min(L, lo + per);
}

// Upper-triangle tile u (row-major over tr <= tc) of a TT x TT tile grid.
__device__ __forceinline__ void upper_tile(int u, int TT, int& tr, int& tc) {
  tr = 0;
  while (u >= TT - tr) {
    u -= TT - tr;
    ++tr;
  }
  tc = tr + u;
}

// ---- the plain iteration's two launches per round ----

constexpr int RCH = 32;         // rows per staged chunk

__device__ __forceinline__ int rr_p(int r, int k, int m) { return k == 0 ? m - 1 : (r + k) % (m - 1); }
__device__ __forceinline__ int rr_q(int r, int k, int m) {
  return k == 0 ? r : (r - k + (m - 1)) % (m - 1);
}

// Partial Gram matrix of one pair over one row slice of W, on the matrix
// cores.  RCH-row chunks of the pair's NP = 2 CB columns are staged in LDS
// (columns >= n zero).  The Gram matrix is symmetric, so only the
// TT (TT + 1) / 2 tiles of 16 x 16 on and above the diagonal (TT = NP / 16)
// are computed, spread over the waves, each a v_mfma_f64_16x16x4f64 chain:
// A = X^T fragment (lane l: X[r + l/16][16 tr + l%16]), B = X fragment (lane
// l: X[r + l/16][16 tc + l%16]), D lane l: G[16 tr + l/16 + 4 q][16 tc +
// l%16].  Each product X[r][a] X[r][b] is the same number either way round,
// so the mirrored tile is the one its own chain would give.  The NP x NP
// result goes row-major to gpart[blockIdx.x] (workgroup = job * pmax +
// slice).
template <int CB, int NT, int RCH>
__global__ __launch_bounds__(NT) void gram_partial_kernel(const BlockDesc* __restrict__ blocks,
                                                          const PairJob* __restrict__ jobs,
                                                          int pmax, double* __restrict__ gpart) {
  constexpr int NP = 2 * CB, TT = NP / 16, NU = TT * (TT + 1) / 2, NW = NT / 64;
  constexpr int TPW = (NU + NW - 1) / NW;   // tiles per wave (the last waves may hold none)
  static_assert(NW * 64 == NT, "whole waves");
  __shared__ double X[RCH][NP + 1];
  __shared__ int colmap[NP];
  const int job = blockIdx.x / pmax, slice = blockIdx.x - job * pmax;
  const PairJob J = jobs[job];
  if (slice >= J.P) return;
  const BlockDesc B = blocks[J.blk];
  const int n = J.bp + J.bq;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int c = t; c < n; c += NT) colmap[c] = c < J.bp ? J.p0 + c : J.q0 + (c - J.bp);
  int lo, hi;
  slice_rows(B.L, J.P, slice, lo, hi);
  int ttr[TPW], ttc[TPW];
#pragma unroll
  for (int j = 0; j < TPW; ++j) upper_tile(min(wave * TPW + j, NU - 1), TT, ttr[j], ttc[j]);
  f64x4 acc[TPW];
#pragma unroll
  for (int j = 0; j < TPW; ++j) acc[j] = f64x4{0.0, 0.0, 0.0, 0.0};
  // the next chunk's global loads are issued before the current chunk's MFMAs
  constexpr int LPT = RCH * NP / NT;
  static_assert(LPT * NT == RCH * NP, "chunk elements per thread");
  double pre[LPT];
  auto fetch = [&](int r0) {
    const int nr = min(RCH, hi - r0);
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int e = t + NT * i, rr = e % RCH, c = e / RCH;
      pre[i] = (rr < nr && c < n) ? B.W[(r0 + rr) + (long long)colmap[c] * B.L] : 0.0;
    }
  };
  __syncthreads();
  if (lo < hi) fetch(lo);
  for (int r0 = lo; r0 < hi; r0 += RCH) {
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int e = t + NT * i;
      X[e % RCH][e / RCH] = pre[i];
    }
    __syncthreads();
    if (r0 + RCH < hi) fetch(r0 + RCH);
#pragma unroll
    for (int k4 = 0; k4 < RCH; k4 += 4) {
      const int row = k4 + (lane >> 4);
#pragma unroll
      for (int j = 0; j < TPW; ++j)
        if (wave * TPW + j < NU)
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(X[row][16 * ttr[j] + (lane & 15)],
                                                        X[row][16 * ttc[j] + (lane & 15)], acc[j],
                                                        0, 0, 0);
    }
    __syncthreads();
  }
  double* out = gpart + (size_t)blockIdx.x * NP * NP;
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    if (wave * TPW + j >= NU) continue;
    const int tr = ttr[j], tc = ttc[j];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int a = 16 * tr + (lane >> 4) + 4 * q, b = 16 * tc + (lane & 15);
      out[a * NP + b] = acc[j][q];
      if (tr != tc) out[b * NP + a] = acc[j][q];
    }
  }
}

// Orthogonalise one pair of column blocks: every row slice of the pair sums
// the same partial Gram matrices in the same order, so the P workgroups of a
// pair hold bit-identical Gram matrices, convergence decisions and rotations;
// each then rotates its own rows of W and V.  Slice 0 records the pair's
// largest scaled off-diagonal Gram entry (before rotating) in off[blk] (as
// ordered bits of a non-negative double).
//
// The pair's Gram matrix is diagonalised in LDS by parallel cyclic Jacobi
// (round-robin rounds of disjoint rotations, inner_sweeps <= INNER_SWEEPS
// sweeps: the outer iteration revisits the pair; one inner sweep per visit
// costs a few more outer sweeps but the least time).  A round updates
// G <- J^T G J by 2 x 2 blocks, with the rotated entry set to zero and the diagonal
// moved by t g_pq; a rotation is skipped below max(tol_in sqrt(g_pp g_qq),
// 0.2 tol_abs ||A||_F sqrt(max(g_pp, g_qq))), about ten times below the
// outer test.  Round latency, not arithmetic, bounds this loop (a 32 x 32
// round costs about as much as a 64 x 64 one), so the rotation parameters
// avoid the correctly rounded square root and division sequences, and the
// 64 x 64 case runs 512 threads (two waves per SIMD) in two groups: the
// lower half updates G, then wave 0 computes the next round's rotations
// while the upper half updates R with this round's (double-buffered)
// parameters.
template <int CB, int NT>
__global__ __launch_bounds__(NT) void jacobi_rotate_kernel(const BlockDesc* __restrict__ blocks,
                                                           const PairJob* __restrict__ jobs,
                                                           int pmax,
                                                           const double* __restrict__ gpart,
                                                           double tol_rel, double tol_abs,
                                                           unsigned long long* __restrict__ off,
                                                           int inner_sweeps) {
  constexpr int NP = 2 * CB, HALF = NP / 2, TT = NP / 16, NW = NT / 64;
  // 512 and more threads: G and R are updated by separate halves
  constexpr bool SPLIT = NT >= 512;
  constexpr int NTG = SPLIT ? NT / 2 : NT, NTR = SPLIT ? NT / 2 : NT;
  constexpr int RT = RCH / 16, TPW = RT * TT / NW;
  static_assert(TPW * NW == RT * TT, "tiles must split evenly over the waves");
  static_assert(NT >= HALF && NT % NP == 0, "thread mapping");
  __shared__ double G[NP][NP + 1];
  __shared__ double R[NP][NP + 1];
  __shared__ double X[RCH][NP + 1];
  __shared__ double cs[2][HALF], sn[2][HALF], tn[2][HALF];
  __shared__ int pp[2][HALF], qq[2][HALF];
  __shared__ int colmap[NP];
  __shared__ double red[NT];
  __shared__ int rotated[INNER_SWEEPS];

  const int job = blockIdx.x / pmax, slice = blockIdx.x - job * pmax;
  const PairJob J = jobs[job];
  if (slice >= J.P) return;
  const BlockDesc B = blocks[J.blk];
  const int n = J.bp + J.bq;
  const int t = threadIdx.x;
  if (n < 2) return;
  for (int c = t; c < n; c += NT) colmap[c] = c < J.bp ? J.p0 + c : J.q0 + (c - J.bp);
  if (t < INNER_SWEEPS) rotated[t] = 0;
  {
    // the slices' partial Gram matrices, summed in slice order; all loads of
    // a thread are issued before the sums
    const double* gp = gpart + (size_t)job * pmax * NP * NP;
    constexpr int PER = NP * NP / NT, GRP = 4;
    static_assert(PER * NT == NP * NP && PER % GRP == 0, "Gram elements per thread");
    for (int i0 = 0; i0 < PER; i0 += GRP) {
      double part[GRP][MAX_SLICES];
#pragma unroll
      for (int i = 0; i < GRP; ++i)
#pragma unroll
        for (int s = 0; s < MAX_SLICES; ++s)
          part[i][s] = s < J.P ? gp[(size_t)s * NP * NP + t + NT * (i0 + i)] : 0.0;
#pragma unroll
      for (int i = 0; i < GRP; ++i) {
        const int e = t + NT * (i0 + i), a = e / NP, b = e % NP;
        double g = 0.0;
#pragma unroll
        for (int s = 0; s < MAX_SLICES; ++s)
          if (s < J.P) g += part[i][s];
        G[a][b] = g;
        R[a][b] = a == b ? 1.0 : 0.0;
      }
    }
  }
  __syncthreads();

  // ---- convergence measure of this pair ----
  double worst = 0.0;
  bool rotate = false;
  for (int e = t; e < n * n; e += NT) {
    const int a = e % n, b = e / n;
    if (a >= b) continue;
    const double g = fabs(G[a][b]);
    const double na = sqrt(G[a][a]), nb = sqrt(G[b][b]);
    // columns at the rounding level of the block carry no direction (the SVD
    // zeroes them); they do not hold the iteration open
    if (fmin(na, nb) <= kNoiseRel * B.normF) continue;
    const double scale = na * nb;
    // relative orthogonality, or the rounding floor of columns that carry
    // absolute errors of order eps ||A||
    const double floor_ab = tol_abs * B.normF * (na + nb);
    if (g > fmax(tol_rel * scale, floor_ab)) {
      rotate = true;
      worst = fmax(worst, g / scale);
    }
  }
  red[t] = worst + (rotate ? 4.0 : 0.0);   // +4 marks "needs a rotation" (ratios are <= 1)
  __syncthreads();
  for (int w = NT / 2; w > 0; w >>= 1) {
    if (t < w) red[t] = fmax(red[t], red[t + w]);
    __syncthreads();
  }
  const double top = red[0];
  if (t == 0 && slice == 0) {
    const double ratio = top >= 4.0 ? top - 4.0 : top;
    // a pair that still needs a rotation reports at least 2 (above any ratio)
    const double rep = top >= 4.0 ? 2.0 + ratio : ratio;
    atomicMax(off + J.blk, (unsigned long long)__double_as_longlong(rep));
  }
  if (top < 4.0) return;   // orthogonal to tolerance: nothing to rotate

  // ---- eigenvectors of G by parallel cyclic Jacobi ----
  const int m = n + (n & 1);   // index n (odd n) is a zero row and column
  const int npair = m / 2;
  const int nround = m - 1;
  const double tol_in = 1e-14;
  const double fl = 0.1 * tol_abs * B.normF;
  // Rotation of slot k in round r (into parameter buffer b): the
  // round-robin pair for k < npair, an identity on the spare indices
  // (2k, 2k+1) >= m otherwise, so that the HALF slots partition all NP
  // indices and every updating thread owns a fixed set of 2 x 2 blocks and R
  // entries with no branches.
  auto rotation = [&](int r, int k, int b, int sweep) {
    int p, q;
    double c = 1.0, s = 0.0, tt = 0.0;
    if (k < npair) {
      p = rr_p(r, k, m);
      q = rr_q(r, k, m);
      if (p < n && q < n) {
        const double apq = G[p][q];
        const double gpp = G[p][p], gqq = G[q][q];
        const double app = fabs(gpp), aqq = fabs(gqq);
        // skip test on squares (no square roots): |g_pq| against
        // tol_in sqrt(g_pp g_qq) and the rounding floor 2 fl sqrt(max g)
        const double a2 = apq * apq;
        if (a2 > tol_in * tol_in * (app * aqq) && a2 > 4.0 * fl * fl * fmax(app, aqq) &&
            fabs(apq) > 1e-300) {
          // t = tan(theta) of the smaller rotation angle,
          //   t = 2 g_pq sign(d) / (|d| + sqrt(d^2 + 4 g_pq^2)), d = g_qq - g_pp
          // (the textbook tau form without its division); c = 1 / sqrt(1 +
          // t^2) keeps the rotation orthogonal to rounding for any t, so
          // the reciprocals need not be correctly rounded
          const double d = gqq - gpp;
          const double h2 = d * d + 4.0 * a2;
          const double den = fabs(d) + h2 * rsqrt_nr(h2);
          tt = (d >= 0 ? 2.0 : -2.0) * apq * recip_nr(den);
          c = rsqrt_nr(1.0 + tt * tt);
          s = tt * c;
          rotated[sweep] = 1;
        }
      }
    } else {
      p = 2 * k;
      q = 2 * k + 1;
    }
    pp[b][k] = p;
    qq[b][k] = q;
    cs[b][k] = c;
    sn[b][k] = s;
    tn[b][k] = tt;
  };
  // G <- J^T G J on the 2 x 2 blocks (k, k2) of a full-square partition
  // (each element has one owner; identity rotations store their values back
  // unchanged) by NTG threads, tg < NTG.  All loads of a thread precede its
  // stores.
  auto update_g = [&](int b, int tg) {
    constexpr int KS = NTG / HALF, MB = HALF / KS;
    static_assert(MB * KS == HALF, "block partition");
    const int k = tg % HALF, kb = tg / HALF;
    const int p = pp[b][k], q = qq[b][k];
    const double c = cs[b][k], s = sn[b][k], tk = tn[b][k];
    double g[MB][4], c2v[MB], s2v[MB];
    int p2v[MB], q2v[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int k2 = kb + KS * i;
      p2v[i] = pp[b][k2];
      q2v[i] = qq[b][k2];
      c2v[i] = cs[b][k2];
      s2v[i] = sn[b][k2];
      g[i][0] = G[p][p2v[i]];
      g[i][1] = G[p][q2v[i]];
      g[i][2] = G[q][p2v[i]];
      g[i][3] = G[q][q2v[i]];
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const double c2 = c2v[i], s2 = s2v[i];
      const double t00 = c2 * g[i][0] - s2 * g[i][1], t01 = s2 * g[i][0] + c2 * g[i][1];
      const double t10 = c2 * g[i][2] - s2 * g[i][3], t11 = s2 * g[i][2] + c2 * g[i][3];
      double n00 = c * t00 - s * t10, n01 = c * t01 - s * t11;
      double n10 = s * t00 + c * t10, n11 = s * t01 + c * t11;
      // the rotated pair's own block: annihilated exactly, diagonal moved by t g_pq
      const bool own = (kb + KS * i == k) && s != 0.0;
      n00 = own ? g[i][0] - tk * g[i][1] : n00;
      n11 = own ? g[i][3] + tk * g[i][1] : n11;
      n01 = own ? 0.0 : n01;
      n10 = own ? 0.0 : n10;
      G[p][p2v[i]] = n00;
      G[p][q2v[i]] = n01;
      G[q][p2v[i]] = n10;
      G[q][q2v[i]] = n11;
    }
  };
  // R <- R J by NTR threads, tr < NTR, each on fixed rows and pair slots
  // (rows >= n hold zeros in the rotated columns)
  auto update_r = [&](int b, int tr) {
    constexpr int RS = NTR / NP, MR = HALF / RS;
    static_assert(MR * RS == HALF, "row partition");
    const int row = tr % NP, rb = tr / NP;
    double ru[MR], rv[MR], rc[MR], rsn[MR];
    int rp[MR], rq[MR];
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      const int kk = rb + RS * i;
      rp[i] = pp[b][kk];
      rq[i] = qq[b][kk];
      rc[i] = cs[b][kk];
      rsn[i] = sn[b][kk];
      ru[i] = R[row][rp[i]];
      rv[i] = R[row][rq[i]];
    }
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      R[row][rp[i]] = rc[i] * ru[i] - rsn[i] * rv[i];
      R[row][rq[i]] = rsn[i] * ru[i] + rc[i] * rv[i];
    }
  };
  if (!SPLIT) {
    // one group: rotations, barrier, G and R updates, barrier
    for (int sweep = 0; sweep < inner_sweeps; ++sweep) {
      for (int r = 0; r < nround; ++r) {
        if (t < HALF) rotation(r, t, 0, sweep);
        __syncthreads();
        update_g(0, t);
        update_r(0, t);
        __syncthreads();
      }
      if (!rotated[sweep]) break;
    }
  } else {
    // Two groups: threads below NTG update G; then, while wave 0 computes
    // the next round's rotations from the updated G, the other NTR threads
    // update R with this round's (double-buffered parameters).
    if (t < HALF) rotation(0, t, 0, 0);
    __syncthreads();
    int b = 0;
    for (int sweep = 0; sweep < inner_sweeps; ++sweep) {
      for (int r = 0; r < nround; ++r, b ^= 1) {
        if (t < NTG) update_g(b, t);
        __syncthreads();
        const bool last = r + 1 == nround;
        const int rn = last ? 0 : r + 1, sw = last ? sweep + 1 : sweep;
        if (t < HALF && sw < inner_sweeps) rotation(rn, t, b ^ 1, sw);
        if (t >= NTG) update_r(b, t - NTG);
        __syncthreads();
      }
      if (!rotated[sweep]) break;
    }
  }

  // ---- rotate this slice's rows: W[:, cols] <- W[:, cols] R, same for V ----
  // Y = X R per 32-row chunk on the matrix cores, the (RCH/16) x (NP/16)
  // output tiles spread over the waves: A = X fragment (lane l:
  // X[16 rt + l%16][k + l/16]), B = R fragment (lane l: R[k + l/16][16 ct + l%16]).
  // The result goes back through LDS so each column segment is written whole.
  // The W chunks of this slice and then its V chunks form one stream; the
  // next chunk's global loads are issued before the current chunk's MFMAs.
  const int lane = t & 63, wave = t >> 6;
  constexpr int LPT = RCH * NP / NT;   // elements of a chunk per thread
  int wlo, whi, vlo, vhi;
  slice_rows(B.L, J.P, slice, wlo, whi);
  slice_rows(B.k, J.P, slice, vlo, vhi);
  const int nw = (whi - wlo + RCH - 1) / RCH, nv = (vhi - vlo + RCH - 1) / RCH;
  auto chunk = [&](int ci, double*& M, long long& ld, int& r0, int& nr) {
    if (ci < nw) {
      M = B.W;
      ld = B.L;
      r0 = wlo + ci * RCH;
      nr = min(RCH, whi - r0);
    } else {
      M = B.V;
      ld = B.k;
      r0 = vlo + (ci - nw) * RCH;
      nr = min(RCH, vhi - r0);
    }
  };
  double pre[LPT];
  auto fetch = [&](int ci) {
    double* M;
    long long ld;
    int r0, nr;
    chunk(ci, M, ld, r0, nr);
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int e = t + NT * i, rr = e % RCH, c = e / RCH;
      pre[i] = (rr < nr && c < n) ? M[(r0 + rr) + (long long)colmap[c] * ld] : 0.0;
    }
  };
  if (nw + nv > 0) fetch(0);
  for (int ci = 0; ci < nw + nv; ++ci) {
    double* M;
    long long ld;
    int r0, nr;
    chunk(ci, M, ld, r0, nr);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int e = t + NT * i;
      X[e % RCH][e / RCH] = pre[i];
    }
    __syncthreads();
    if (ci + 1 < nw + nv) fetch(ci + 1);
    f64x4 y[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u) y[u] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NP; k += 4) {
#pragma unroll
      for (int u = 0; u < TPW; ++u) {
        const int tau = wave * TPW + u, rt = tau % RT, ct = tau / RT;
        y[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(X[16 * rt + (lane & 15)][k + (lane >> 4)],
                                                    R[k + (lane >> 4)][16 * ct + (lane & 15)],
                                                    y[u], 0, 0, 0);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      const int tau = wave * TPW + u, rt = tau % RT, ct = tau / RT;
#pragma unroll
      for (int q = 0; q < 4; ++q) X[16 * rt + (lane >> 4) + 4 * q][16 * ct + (lane & 15)] = y[u][q];
    }
    __syncthreads();
    for (int e = t; e < RCH * n; e += NT) {
      const int rr = e % RCH, c = e / RCH;
      if (rr < nr) M[(r0 + rr) + (long long)colmap[c] * ld] = X[rr][c];
    }
  }
}

// ---- the preconditioned iteration's launches ----

// Pairs of column blocks that share one round, merged over the blocks of a batch: workgroups of a
// launch find theirs by index.
//
// A visit of a pair takes three steps in as many launches (d = 2000 step, 34
// pairs: 12, 37 and 20 us; the two launches of the plain iteration 15 and 93): partial Gram matrices over row slices
// (gram_kernel), one workgroup per pair that sums them and diagonalises the pair's Gram matrix
// (the first workgroups of solve_kernel), and the pair's columns times the rotation it found
// (apply_rows), row tiles of W in a launch of their own.  V is not read before the sweep ends, so
// its row tiles ride in the next round's solve launch, whose few workgroups leave the chip idle.

// Partial Gram matrix of one pair over one row slice of W, on the matrix
// cores.  The TT (TT + 1) / 2 tiles of 16 x 16 on and above the diagonal are
// each a v_mfma_f64_16x16x4f64 chain over the rows: lane l holds rows 4 (l /
// 16) .. + 3 of a 16-row strip in column l % 16 of each tile column (the same
// assignment of rows to k for both operands, so any will do), which are 32
// contiguous bytes: the loads go straight from memory to the fragments, with
// no LDS pass and no barrier until the waves' sums meet.  Each wave takes
// every fourth strip, the next strip's loads in flight under the MFMAs.  The
// four partial sums are added in wave order; tile u's element of register q
// and lane l goes to gpart[u][q][l].
template <int CB>
__global__ __launch_bounds__(256) void gram_kernel(const BlockDesc* __restrict__ blocks,
                                                   const PairJob* __restrict__ jobs, int pmax,
                                                   double* __restrict__ gpart) {
  constexpr int NP = 2 * CB, TT = NP / 16, NU = TT * (TT + 1) / 2;
  __shared__ double red[4][NU * 256];
  const int job = blockIdx.x / pmax, slice = blockIdx.x - job * pmax;
  const PairJob J = jobs[job];
  if (slice >= J.P) return;
  const BlockDesc B = blocks[J.blk];
  const int n = J.bp + J.bq;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int lo, hi;
  slice_rows(B.L, J.P, slice, lo, hi);
  const double* col[TT];
  bool ok[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    const int c = 16 * i + (lane & 15);
    ok[i] = c < n;
    col[i] = B.W + (long long)pair_column(J, min(c, n - 1)) * B.L;
  }
  f64x4 acc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) acc[u] = f64x4{0.0, 0.0, 0.0, 0.0};
  f64x4 x[TT];
  auto fetch = [&](int r0) {
    const int r = r0 + 4 * (lane >> 4);
    if (r0 + 16 <= hi) {
#pragma unroll
      for (int i = 0; i < TT; ++i) x[i] = *(const f64x4u*)(col[i] + r);
    } else {
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[i][q] = r + q < hi ? col[i][r + q] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < TT; ++i)
      if (!ok[i]) x[i] = f64x4{0.0, 0.0, 0.0, 0.0};
  };
  if (lo + 16 * wave < hi) fetch(lo + 16 * wave);
  for (int r0 = lo + 16 * wave; r0 < hi; r0 += 64) {
    f64x4 y[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) y[i] = x[i];
    if (r0 + 64 < hi) fetch(r0 + 64);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int u = 0;
#pragma unroll
      for (int a = 0; a < TT; ++a)
#pragma unroll
        for (int b = a; b < TT; ++b, ++u)
          acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[a][q], y[b][q], acc[u], 0, 0, 0);
    }
  }
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave][256 * u + 64 * q + lane] = acc[u][q];
  __syncthreads();
  double* out = gpart + (size_t)blockIdx.x * NU * 256;
  for (int e = t; e < NU * 256; e += 256)
    out[e] = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
}

// LDS of one pair: G (upper triangle) and R[column][row], both NP x NP, cos
// and sin and tan of each slot (two buffers), whether a sweep rotated.
struct PairLds {
  double* G;
  double* R;
  f64x2* cs;
  double* tn;
  int* rotated;
};

// The inner sweeps of one pair of n columns; FULL: all of them against each
// other, else the first CB against the others.
template <int CB, bool FULL>
__device__ __forceinline__ void pair_sweeps(const PairLds& S, int n, double fl,
                                            int inner_sweeps) {
  constexpr int NP = 2 * CB, NT = SolveThreads<CB>::value;
  double* G = S.G;
  double* R = S.R;
  f64x2* cs = S.cs;
  double* tn = S.tn;
  int* rotated = S.rotated;
  const int t = threadIdx.x;
  const int m = n + (n & 1);   // index n (odd n) is a zero row and column
  const int nround = FULL ? m - 1 : CB;
  const double tol_in = 1e-14;
  // columns of slot k in round r: the round-robin pair in a full sweep
  // (identity slots (2k, 2k+1) past the last pair), else k and a q column
  auto slot = [&](int r, int k, int& p, int& q) {
    if (!FULL) {
      p = k;
      q = CB + ((k + r) & (CB - 1));
    } else if (k < m / 2) {
      p = k == 0 ? m - 1 : (r + k < m - 1 ? r + k : r + k - (m - 1));
      q = k == 0 ? r : (r >= k ? r - k : r - k + (m - 1));
    } else {
      p = 2 * k;
      q = 2 * k + 1;
    }
  };
  auto at = [&](int a, int b) { return min(a, b) * NP + max(a, b); };
  auto rotation = [&](int r, int k, int b, int sweep) {
    int p, q;
    slot(r, k, p, q);
    double c = 1.0, s = 0.0, tt = 0.0;
    if (p < n && q < n) {
      const double apq = G[at(p, q)], gpp = G[p * NP + p], gqq = G[q * NP + q];
      const double app = fabs(gpp), aqq = fabs(gqq), a2 = apq * apq;
      if (a2 > tol_in * tol_in * (app * aqq) && a2 > 4.0 * fl * fl * fmax(app, aqq) &&
          fabs(apq) > 1e-300) {
        // t = tan(theta) of the smaller rotation angle,
        //   t = 2 g_pq sign(d) / (|d| + sqrt(d^2 + 4 g_pq^2)), d = g_qq - g_pp;
        // c = 1 / sqrt(1 + t^2) keeps the rotation orthogonal to rounding for
        // any t, so the reciprocals need not be correctly rounded
        const double d = gqq - gpp, h2 = d * d + 4.0 * a2;
        const double den = fabs(d) + h2 * rsqrt_nr(h2);
        tt = (d >= 0 ? 2.0 : -2.0) * apq * recip_nr(den);
        c = rsqrt_nr(1.0 + tt * tt);
        s = tt * c;
        rotated[sweep] = 1;
      }
    }
    cs[b * CB + k] = f64x2{c, s};
    tn[b * CB + k] = tt;
  };
  // the 2 x 2 block of slots k and k2; a slot's own block (k == k2) has its
  // entry annihilated exactly and its diagonal moved by t g_pq
  auto mix = [&](int r, int b, int k, int k2) {
    int p, q, p2, q2;
    slot(r, k, p, q);
    slot(r, k2, p2, q2);
    const int e00 = at(p, p2), e01 = at(p, q2), e10 = at(q, p2), e11 = at(q, q2);
    const double g00 = G[e00], g01 = G[e01], g10 = G[e10], g11 = G[e11];
    const f64x2 x = cs[b * CB + k], y = cs[b * CB + k2];
    const double tt = tn[b * CB + k];
    const double t00 = y.x * g00 - y.y * g01, t01 = y.y * g00 + y.x * g01;
    const double t10 = y.x * g10 - y.y * g11, t11 = y.y * g10 + y.x * g11;
    const bool own = k == k2, hit = own && tt != 0.0;
    const double n01 = x.x * t01 - x.y * t11, n10 = x.y * t00 + x.x * t10;
    G[e00] = own ? g00 - tt * g01 : x.x * t00 - x.y * t10;
    G[e11] = own ? g11 + tt * g01 : x.y * t01 + x.x * t11;
    G[e01] = hit ? 0.0 : n01;
    G[e10] = hit ? 0.0 : own ? n01 : n10;
  };
  // G: threads (k, d), d = 1 .. CB/2 - 1, take slots k and k + d modulo CB;
  // then CB threads a slot's own block and CB / 2 the slots CB / 2 apart
  const int k = t % CB, d = t / CB + 1;
  constexpr int D = CB / 2;
  static_assert(CB * D + D <= NT, "threads of the G update");
  const int k2 = d < D ? (k + d) % CB : d == D ? k : (k + D) % CB;
  const bool mine = d <= D || (d == D + 1 && k < D);
  // R: four slots' elements of one row per thread.  In cross rounds a slot's
  // p column is always the same, so its element stays in a register.
  constexpr int NR = NT - 64, SL = CB * NP / NR;
  static_assert(SL * NR == CB * NP && NR % NP == 0, "slots per thread");
  const int row = (t - 64) % NP, k0 = (t - 64) / NP;
  double u[SL];
  if (!FULL && t >= 64) {
#pragma unroll
    for (int i = 0; i < SL; ++i) u[i] = R[(k0 + i * (NR / NP)) * NP + row];
  }
  if (t < CB) rotation(0, t, 0, 0);
  __syncthreads();
  int b = 0;
  for (int sweep = 0; sweep < inner_sweeps; ++sweep) {
    for (int r = 0; r < nround; ++r, b ^= 1) {
      if (mine) mix(r, b, k, k2);
      __syncthreads();
      const bool last = r + 1 == nround;
      const int sw = last ? sweep + 1 : sweep;
      if (t < 64) {
        if (t < CB && sw < inner_sweeps) rotation(last ? 0 : r + 1, t, b ^ 1, sw);
      } else {
        // R <- R J, all loads before the first store
        double v[SL];
        f64x2 x[SL];
        int p[SL], q[SL];
#pragma unroll
        for (int i = 0; i < SL; ++i) {
          const int kk = k0 + i * (NR / NP);
          x[i] = cs[b * CB + kk];
          slot(r, kk, p[i], q[i]);
          if (FULL) u[i] = R[p[i] * NP + row];
          v[i] = R[q[i] * NP + row];
        }
#pragma unroll
        for (int i = 0; i < SL; ++i) {
          const double w = x[i].x * u[i] - x[i].y * v[i];
          R[q[i] * NP + row] = x[i].y * u[i] + x[i].x * v[i];
          u[i] = w;
          if (FULL) R[p[i] * NP + row] = w;
        }
      }
      __syncthreads();
    }
    if (!rotated[sweep]) break;
  }
  if (!FULL && t >= 64) {
#pragma unroll
    for (int i = 0; i < SL; ++i) R[(k0 + i * (NR / NP)) * NP + row] = u[i];
  }
  __syncthreads();
}

// Diagonalises one pair's Gram matrix: the slices' partial sums in slice
// order, the convergence test, then inner_sweeps sweeps of parallel cyclic
// Jacobi in LDS, and the accumulated rotation to rot (column-major, NP rows).
// *active says whether the pair rotated at all; *moved is set if it did.
//
// A pair rotates its p columns against its q columns only (CB rounds of CB
// disjoint rotations): the pairs inside a block are rotated in the block's
// first visit of a sweep (J.full: 2 CB - 1 rounds over all its columns), so a
// sweep meets every pair of columns once.  A model of the iteration at k =
// 640 needed 908 such visits against 886 that rotate all pairs every time,
// each at half the rounds.
//
// G is symmetric, and only its upper triangle is kept: the rotations of slots
// k and k2 mix four elements, one thread's, at distinct places.  A round is
// two phases with a barrier each: every thread updates its 2 x 2 block (its
// LDS reads do not wait for the rotations' parameters); then wave 0 computes
// the next round's rotations while the other waves apply this round's to R
// (double-buffered parameters).  In cross rounds neighbouring threads' blocks
// lie NP + 1 apart, which spreads them over all LDS banks at a pitch of NP.
// Clock stamps of a cross round: 600 cycles of G, 1000 of R beside 700 of the
// rotations (2600 with the barriers; the plain launch takes 2900 for half the
// work of a round, being one group of threads after another).
// A rotation annihilates its entry exactly and moves the diagonal by t g_pq;
// it is skipped below max(tol_in sqrt(g_pp g_qq), 0.2 tol_abs ||A||_F
// sqrt(max(g_pp, g_qq))), about ten times below the outer test.
template <int CB>
__device__ __forceinline__ void solve_pair(const BlockDesc& B, const PairJob& J,
                                           const double* __restrict__ gp, double tol_rel,
                                           double tol_abs, int inner_sweeps, double* lds,
                                           double* __restrict__ rot, int* __restrict__ active,
                                           int* __restrict__ moved) {
  constexpr int NP = 2 * CB, TT = NP / 16, NU = TT * (TT + 1) / 2, NT = SolveThreads<CB>::value;
  double* G = lds;                       // NP x NP, upper triangle
  double* R = G + NP * NP;               // R[column][row]
  f64x2* cs = (f64x2*)(R + NP * NP);     // cos, sin of slot k: [2][CB]
  double* tn = (double*)(cs + 2 * CB);   // tan: [2][CB]
  int* rotated = (int*)(tn + 2 * CB);    // INNER_SWEEPS
  const int n = J.bp + J.bq, t = threadIdx.x;
  if (t < INNER_SWEEPS) rotated[t] = 0;
  for (int e = t; e < NP * NP; e += NT) R[e] = e / NP == e % NP ? 1.0 : 0.0;
  {
    // the slices' sums; all loads of a thread are in flight at once
    constexpr int PER = (NU * 256 + NT - 1) / NT;
    double part[PER][MAX_SLICES];
#pragma unroll
    for (int i = 0; i < PER; ++i)
#pragma unroll
      for (int s = 0; s < MAX_SLICES; ++s)
        part[i][s] = s < J.P ? gp[(size_t)s * NU * 256 + min(t + NT * i, NU * 256 - 1)] : 0.0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = t + NT * i;
      if (e >= NU * 256) break;
      double g = 0.0;
#pragma unroll
      for (int s = 0; s < MAX_SLICES; ++s)
        if (s < J.P) g += part[i][s];
      int tr, tc;
      upper_tile(e / 256, TT, tr, tc);
      const int l = e & 63, q = (e >> 6) & 3;
      G[(16 * tr + (l >> 4) + 4 * q) * NP + 16 * tc + (l & 15)] = g;
    }
  }
  __syncthreads();

  // ---- does the pair need a rotation? ----
  double* norm = tn;   // free until the rotations
  if (t < n) norm[t] = sqrt(G[t * NP + t]);
  __syncthreads();
  bool need = false;
  {
    const double noise = kNoiseRel * B.normF, ta = tol_abs * B.normF;
    const int ra = J.full ? n : J.bp;   // rows a of the entries looked at
    for (int e = t; e < ra * NP; e += NT) {
      const int a = e / NP, b = e % NP;
      if (b >= n || b <= a || (!J.full && b < J.bp)) continue;
      const double na = norm[a], nb = norm[b];
      need = need || (fmin(na, nb) > noise &&
                      fabs(G[a * NP + b]) > fmax(tol_rel * na * nb, ta * (na + nb)));
    }
  }
  const bool any = __syncthreads_or(need);
  if (t == 0) {
    *active = any;
    if (any) *moved = 1;
  }
  if (!any) return;

  PairLds L{G, R, cs, tn, rotated};
  const double fl = 0.1 * tol_abs * B.normF;
  if (J.full) pair_sweeps<CB, true>(L, n, fl, inner_sweeps);
  else pair_sweeps<CB, false>(L, n, fl, inner_sweeps);
  for (int e = t; e < NP * NP; e += NT) rot[e] = R[e];
}

// M[rows, cols] <- M[rows, cols] R for one row tile of W or V, 16 rows per
// wave.  R goes to LDS; a wave's 16 x NP strip goes straight from memory to its
// B fragments (lane l: row l % 16, column 4 s + l / 16, 128
// contiguous bytes per column), and Y^T = R^T X^T comes back with 16 rows of
// a column on neighbouring lanes, so it is stored as it is.  A wave owns its
// rows and reads them before it writes, so the update is in place.
template <int CB>
__device__ __forceinline__ void apply_rows(double* __restrict__ M, int rows, const PairJob& J,
                                           const double* __restrict__ rot, int tile,
                                           double* lds) {
  constexpr int NP = 2 * CB, TT = NP / 16, NT = SolveThreads<CB>::value, PR = NP + 1;
  const int n = J.bp + J.bq, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r0 = tile * (NT / 4) + wave * 16;
  const int row = min(r0 + (lane & 15), rows - 1);
  double x[NP / 4];
#pragma unroll
  for (int s = 0; s < NP / 4; ++s) {
    const int c = 4 * s + (lane >> 4);
    x[s] = M[row + (long long)pair_column(J, min(c, n - 1)) * rows];
  }
  for (int e = t; e < NP * NP; e += NT) lds[(e % NP) * PR + e / NP] = rot[e];
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NP / 4; ++s)
    if (4 * s + (lane >> 4) >= n) x[s] = 0.0;
  f64x4 y[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) y[i] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < NP / 4; ++s)
#pragma unroll
    for (int i = 0; i < TT; ++i)
      y[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(
          lds[(4 * s + (lane >> 4)) * PR + 16 * i + (lane & 15)], x[s], y[i], 0, 0, 0);
  if (r0 + (lane & 15) >= rows) return;
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 16 * i + (lane >> 4) + 4 * q;
      if (c < n) M[row + (long long)pair_column(J, c) * rows] = y[i][q];
    }
}

// The first nj workgroups diagonalise this round's pairs, the others apply
// the previous round's rotations to V's row tiles (nv of them per pair).
// moved: one flag per block of the batch, set where a pair rotated.
template <int CB>
__global__ __launch_bounds__(SolveThreads<CB>::value) void solve_kernel(
    const BlockDesc* __restrict__ blocks, const PairJob* __restrict__ jobs, int nj, int pmax,
    const double* __restrict__ gpart, double tol_rel, double tol_abs, int inner_sweeps,
    double* __restrict__ rot, int* __restrict__ active, int* __restrict__ moved,
    const PairJob* __restrict__ vjobs, int nv, const double* __restrict__ vrot,
    const int* __restrict__ vactive) {
  constexpr int NP = 2 * CB, NU = (NP / 16) * (NP / 16 + 1) / 2;
  __shared__ __align__(16) double lds[2 * NP * NP + 6 * CB + 2];
  const int i = blockIdx.x;
  if (i < nj) {
    const PairJob J = jobs[i];
    solve_pair<CB>(blocks[J.blk], J, gpart + (size_t)i * pmax * NU * 256, tol_rel, tol_abs,
                   inner_sweeps, lds, rot + (size_t)i * NP * NP, active + i, moved + J.blk);
    return;
  }
  const int job = (i - nj) / nv, tile = (i - nj) - job * nv;
  const PairJob J = vjobs[job];
  const BlockDesc B = blocks[J.blk];
  if (tile * (SolveThreads<CB>::value / 4) >= B.k || !vactive[job]) return;
  apply_rows<CB>(B.V, B.k, J, vrot + (size_t)job * NP * NP, tile, lds);
}

// This round's rotations on W's row tiles (ntile per pair).
template <int CB>
__global__ __launch_bounds__(SolveThreads<CB>::value) void apply_kernel(
    const BlockDesc* __restrict__ blocks, const PairJob* __restrict__ jobs, int ntile,
    const double* __restrict__ rot, const int* __restrict__ active) {
  constexpr int NP = 2 * CB;
  __shared__ double lds[NP * (NP + 1)];
  const int job = blockIdx.x / ntile, tile = blockIdx.x - job * ntile;
  const PairJob J = jobs[job];
  const BlockDesc B = blocks[J.blk];
  if (tile * (SolveThreads<CB>::value / 4) >= B.L || !active[job]) return;
  apply_rows<CB>(B.W, B.L, J, rot + (size_t)job * NP * NP, tile, lds);
}

// Largest overlap that calls for a rotation in each pair of column blocks (i
// <= j) of a block's kept columns, from their whole Gram matrix (0: none);
// workgroup = entry of the pair table.
struct FlagBlock {
  const double* G;   // kept x kept
  int kept, first;   // its pairs of column blocks (i <= j, row by row) from workgroup `first` on
  double normF;
};

__global__ __launch_bounds__(256) void pair_flags_kernel(const FlagBlock* __restrict__ blocks,
                                                         int nblocks, int cb, double tol_rel,
                                                         double tol_abs, double* __restrict__ out) {
  __shared__ double s[4];
  int b = nblocks - 1;
  while (b > 0 && blocks[b].first > (int)blockIdx.x) --b;
  const FlagBlock J = blocks[b];
  const int ncb = (J.kept + cb - 1) / cb;
  int i = 0, f = (int)blockIdx.x - J.first;
  while (f >= ncb - i) f -= ncb - i++;
  const int j = i + f;
  double worst = 0.0;
  for (int e = threadIdx.x; e < cb * cb; e += 256) {
    const int a = i * cb + e % cb, b = j * cb + e / cb;
    if (a >= b || b >= J.kept) continue;
    const double ga = J.G[a + (size_t)a * J.kept], gb = J.G[b + (size_t)b * J.kept];
    worst = fmax(worst, pair_overlap(J.G[a + (size_t)b * J.kept], ga, gb, tol_rel, tol_abs,
                                     J.normF));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) worst = fmax(worst, __shfl_xor(worst, o));
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = worst;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = fmax(fmax(s[0], s[1]), fmax(s[2], s[3]));
}

// Every block's start in one launch, blockIdx.y the block: W = A, or A^T where
// A is wider than tall (m x n, ld m), in 32 x 32 tiles, and V = 1 in the rest
// of the grid.
struct LoadJob {
  const double* A;
  double *W, *V;
  int m, n;
};
constexpr int kLoadsPerLaunch = 96;
struct LoadArgs {
  LoadJob j[kLoadsPerLaunch];
};

__global__ __launch_bounds__(256) void load_kernel(const LoadArgs args) {
  __shared__ double tile[32][33];
  const LoadJob J = args.j[blockIdx.y];
  const int m = J.m, n = J.n, tm = (m + 31) / 32, tn = (n + 31) / 32;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;   // 32 x 8
  if ((int)blockIdx.x >= tm * tn) {
    const int k = min(m, n);
    const long long e0 = ((long long)blockIdx.x - tm * tn) * 1024;
    for (long long e = e0 + threadIdx.x; e < min(e0 + 1024, (long long)k * k); e += 256)
      J.V[e] = (e % k) == (e / k) ? 1.0 : 0.0;
    return;
  }
  const int bx = (int)blockIdx.x % tm * 32, by = (int)blockIdx.x / tm * 32;
  if (m >= n) {
    for (int j = ty; j < 32; j += 8) {
      const int r = bx + tx, c = by + j;
      if (r < m && c < n) J.W[r + (long long)c * m] = J.A[r + (long long)c * m];
    }
    return;
  }
  // W (n x m) = A^T: read A tile (rows bx.., cols by..), write transposed
  for (int j = ty; j < 32; j += 8) {
    const int r = bx + tx, c = by + j;
    tile[j][tx] = (r < m && c < n) ? J.A[r + (long long)c * m] : 0.0;
  }
  __syncthreads();
  for (int j = ty; j < 32; j += 8) {
    const int wr = by + tx, wc = bx + j;   // W row = A column, W column = A row
    if (wr < n && wc < m) J.W[wr + (long long)wc * n] = tile[tx][j];
  }
}

__global__ void fill_u64_kernel(unsigned long long* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

// ---- batched helpers: one launch for every block of the batch ----

// block of global column gc (columns of all blocks concatenated)
__device__ __forceinline__ int col_block(const long long* __restrict__ noff, int nb, long long gc) {
  int lo = 0, hi = nb - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (noff[mid] <= gc) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// squared column norms of every block's current W into out[0, ncol) and of
// its V into out[ncol, 2 ncol) (one workgroup per column); every block's flag
// into out[2 ncol, 2 ncol + nb) and back to zero
__global__ __launch_bounds__(256) void colnorm_batched_kernel(const BlockDesc* __restrict__ desc,
                                                              const long long* __restrict__ noff,
                                                              int nb, long long ncol,
                                                              double* __restrict__ out,
                                                              int* __restrict__ moved) {
  __shared__ double s[2][256];
  const long long gc = blockIdx.x;
  const int b = col_block(noff, nb, gc);
  const BlockDesc B = desc[b];
  const double* col = B.W + (gc - noff[b]) * B.L;
  const double* vcol = B.V + (gc - noff[b]) * B.k;
  double a = 0.0, v = 0.0;
  for (int r = threadIdx.x; r < B.L; r += 256) a += col[r] * col[r];
  for (int r = threadIdx.x; r < B.k; r += 256) v += vcol[r] * vcol[r];
  s[0][threadIdx.x] = a;
  s[1][threadIdx.x] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s[0][threadIdx.x] += s[0][threadIdx.x + w];
      s[1][threadIdx.x] += s[1][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[gc] = s[0][0];
    out[ncol + gc] = s[1][0];
    if (gc == noff[b]) {
      out[2 * ncol + b] = moved[b] != 0;
      moved[b] = 0;
    }
  }
}

// dst[:, c] = sign[c] * src[:, perm[c]] for every job (perm and sign hold
// the batch's columns, a job's at its block's column offset)
struct PermJob {
  const double* src;
  double* dst;
  int rows, cols;
  long long elem_begin, col_off;
};

__global__ void permute_batched_kernel(const PermJob* __restrict__ jobs, int nj, long long total,
                                       const int* __restrict__ perm,
                                       const double* __restrict__ sign) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  int lo = 0, hi = nj - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].elem_begin <= e) lo = mid;
    else hi = mid - 1;
  }
  const PermJob J = jobs[lo];
  const long long i = e - J.elem_begin;
  const int r = (int)(i % J.rows), c = (int)(i / J.rows);
  const double v = J.src[r + (long long)perm[J.col_off + c] * J.rows];
  J.dst[i] = sign ? sign[J.col_off + c] * v : v;
}

// Sign of the first entry with |v| >= max|v|/2 of the columns perm[] of every
// block's V (desc[b].V, k x k), divided by
// the column's norm: the accumulated rotations leave V's columns off unit
// length by the rounding of every rotation applied (a few 1e-13 after tens of
// sweeps over hundreds of columns), and W = A V carries the same factor, so
// one scaling of both restores the triplet
__global__ __launch_bounds__(256) void col_sign_batched_kernel(const BlockDesc* __restrict__ desc,
                                                               const long long* __restrict__ noff,
                                                               int nb,
                                                               const int* __restrict__ perm,
                                                               double* __restrict__ sign) {
  __shared__ double sv[256];
  __shared__ int si[256];
  const long long gc = blockIdx.x;
  const int b = col_block(noff, nb, gc);
  const int rows = desc[b].k;
  const double* col = desc[b].V + (long long)perm[gc] * rows;
  double best = 0.0;
  for (int r = threadIdx.x; r < rows; r += 256) best = fmax(best, fabs(col[r]));
  sv[threadIdx.x] = best;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sv[threadIdx.x] = fmax(sv[threadIdx.x], sv[threadIdx.x + w]);
    __syncthreads();
  }
  const double half = 0.5 * sv[0];
  int first = 0x7fffffff;
  double n2 = 0.0;
  for (int r = threadIdx.x; r < rows; r += 256) {
    if (fabs(col[r]) >= half && r < first) first = r;
    n2 += col[r] * col[r];
  }
  si[threadIdx.x] = first;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) si[threadIdx.x] = min(si[threadIdx.x], si[threadIdx.x + w]);
    __syncthreads();
  }
  sv[threadIdx.x] = n2;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sv[threadIdx.x] += sv[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double inv = sv[0] > 0.0 ? 1.0 / sqrt(sv[0]) : 1.0;
    sign[gc] = (si[0] < rows && col[si[0]] < 0.0) ? -inv : inv;
  }
}

unsigned nblk(long long n, int t) { return (unsigned)std::max<long long>(1, (n + t - 1) / t); }

// device memory from the context's cache, returned on scope exit
struct DevMem {
  Context& c;
  void* p = nullptr;
  DevMem(Context& ctx, size_t bytes) : c(ctx), p(ctx.dev_alloc(bytes)) {}
  ~DevMem() { c.dev_free(p); }
  DevMem(const DevMem&) = delete;
  DevMem& operator=(const DevMem&) = delete;
};

}  // namespace

static int jacobi_svd_large(Context& c, const std::vector<JacobiBlock*>& blocks, double tol,
                            int max_sweeps, int block_cols, int inner_sweeps, double* worst_out,
                            int precondition_min_k, bool plain) {
  if (worst_out) *worst_out = 0.0;
  hipStream_t st = c.stream();
  const int nb = (int)blocks.size();
  if (nb == 0) return 0;
  SU2_CHECK(block_cols == 16 || block_cols == 32, kErrArgument, "jacobi: block width %d",
            block_cols);
  SU2_CHECK(inner_sweeps >= 1 && inner_sweeps <= INNER_SWEEPS, kErrArgument,
            "jacobi: inner sweeps %d", inner_sweeps);
  // pairs of 16-column blocks run one wave per workgroup (several per CU);
  // pairs of 32-column blocks run four waves
  const int CB = block_cols, NP = 2 * CB;
  const int slice_target = CB == 16 ? 1024 : 256;
  std::vector<int> L(nb), K(nb);
  std::vector<long long> noff(nb + 1, 0);
  for (int b = 0; b < nb; ++b) {
    SU2_CHECK(blocks[b]->m >= 1 && blocks[b]->n >= 1, kErrArgument, "jacobi: empty block");
    L[b] = std::max(blocks[b]->m, blocks[b]->n);
    K[b] = std::min(blocks[b]->m, blocks[b]->n);
    noff[b + 1] = noff[b] + K[b];
  }
  const long long ncol = noff[nb];
  SU2_CHECK(ncol < (1LL << 31), kErrCapacity, "jacobi: %lld columns", ncol);
  // second buffers: each sweep starts by moving the columns into descending
  // norm order (de Rijk's ordering; it cuts the sweep count severalfold)
  std::vector<std::unique_ptr<DevMem>> W2(nb), V2(nb);
  std::vector<double*> Wc(nb), Vc(nb), Wo(nb), Vo(nb);
  for (int b = 0; b < nb; ++b) {
    JacobiBlock& J = *blocks[b];
    W2[b].reset(new DevMem(c, sizeof(double) * (size_t)L[b] * K[b]));
    V2[b].reset(new DevMem(c, sizeof(double) * (size_t)K[b] * K[b]));
    Wc[b] = J.W;
    Vc[b] = J.V;
    Wo[b] = (double*)W2[b]->p;
    Vo[b] = (double*)V2[b]->p;
  }
  for (int b0 = 0; b0 < nb; b0 += kLoadsPerLaunch) {
    LoadArgs args;
    const int n = std::min(kLoadsPerLaunch, nb - b0);
    long long most = 1;
    for (int i = 0; i < n; ++i) {
      const JacobiBlock& J = *blocks[b0 + i];
      args.j[i] = LoadJob{J.A, J.W, J.V, J.m, J.n};
      const long long k = K[b0 + i];
      most = std::max(most, (long long)nblk(J.m, 32) * nblk(J.n, 32) + nblk(k * k, 1024));
    }
    hipLaunchKernelGGL(load_kernel, dim3((unsigned)most, n), dim3(256), 0, st, args);
    SU2_HIP(hipGetLastError());
  }
  // The tables that change from sweep to sweep, [permutation jobs | blocks |
  // flag blocks | permutation], in one device block and one upload.  A copy of
  // any size costs the host 3 us and the stream as much, and one back through
  // pageable memory 20 us with its wait, where a kernel that writes to pinned
  // memory needs 11: with one upload here, norms and flags written to pinned
  // memory, and descriptors as kernel arguments wherever a table goes to one
  // launch, a 6x4 lattice run up to d = 924 went from 310 to 262 ms, eight
  // small jobs from 341 to 262, a truncation at 64 multiplets from 0.47 to
  // 0.36 ms and one at 500 from 9.2 to 8.3.
  const size_t off_desc = sizeof(PermJob) * 2 * nb, off_flag = off_desc + sizeof(BlockDesc) * nb,
               off_perm = off_flag + sizeof(FlagBlock) * nb;
  DevMem dtab(c, off_perm + sizeof(int) * ncol), dsign(c, sizeof(double) * ncol),
      dnoff(c, sizeof(long long) * (nb + 1));
  std::vector<char> tab(off_perm + sizeof(int) * ncol, 0);
  PermJob* const hpj = (PermJob*)tab.data();
  FlagBlock* const hflag = (FlagBlock*)(tab.data() + off_flag);
  int* const hp = (int*)(tab.data() + off_perm);
  const PermJob* const dpj = (const PermJob*)dtab.p;
  const BlockDesc* const ddesc = (const BlockDesc*)((char*)dtab.p + off_desc);
  const FlagBlock* const dflagb = (const FlagBlock*)((char*)dtab.p + off_flag);
  const int* const dperm = (const int*)((char*)dtab.p + off_perm);
  std::vector<double> hn(2 * ncol);   // W then V squared column norms
  SU2_HIP(hipMemcpyAsync(dnoff.p, noff.data(), sizeof(long long) * (nb + 1), hipMemcpyHostToDevice,
                         st));
  std::vector<BlockDesc> desc(nb);
  auto upload = [&]() {
    for (int b = 0; b < nb; ++b) {
      desc[b].W = Wc[b];
      desc[b].V = Vc[b];
    }
    std::memcpy(tab.data() + off_desc, desc.data(), sizeof(BlockDesc) * nb);
    SU2_HIP(hipMemcpyAsync(dtab.p, tab.data(), tab.size(), hipMemcpyHostToDevice, st));
  };
  // squared column norms of the current W and V of every block, written to
  // pinned memory by the kernel, and whether any of a block's pairs rotated
  // since the last call (nothing before the first; every block has a column)
  DevMem dmoved(c, sizeof(int) * nb);
  std::vector<char> rotated(nb, 0);
  auto norms = [&]() {
    double* h = c.host_scratch(2 * ncol + nb);
    hipLaunchKernelGGL(colnorm_batched_kernel, dim3((unsigned)ncol), dim3(256), 0, st, ddesc,
                       (const long long*)dnoff.p, nb, (long long)ncol, h, (int*)dmoved.p);
    SU2_HIP(hipGetLastError());
    SU2_HIP(hipStreamSynchronize(st));
    std::memcpy(hn.data(), h, sizeof(double) * 2 * ncol);
    for (int b = 0; b < nb; ++b) rotated[b] = h[2 * ncol + b] != 0.0;
  };
  // src -> dst column moves of W and V: the first n jobs of the table
  // (prepare_permute before the upload, permute after it)
  long long perm_total = 0;
  auto prepare_permute = [&](const std::vector<PermJob>& pj) {
    perm_total = 0;
    for (size_t i = 0; i < pj.size(); ++i) {
      hpj[i] = pj[i];
      hpj[i].elem_begin = perm_total;
      perm_total += (long long)pj[i].rows * pj[i].cols;
    }
  };
  auto permute = [&](int n, const double* sign) {
    if (perm_total == 0) return;
    hipLaunchKernelGGL(permute_batched_kernel, dim3(nblk(perm_total, 256)), dim3(256), 0, st, dpj,
                       n, perm_total, dperm, sign);
    SU2_HIP(hipGetLastError());
  };
  for (int b = 0; b < nb; ++b) desc[b] = BlockDesc{Wc[b], Vc[b], L[b], K[b], 0.0};
  upload();
  norms();
  for (int b = 0; b < nb; ++b) {
    double g = 0;
    for (int i = 0; i < K[b]; ++i) g += hn[noff[b] + i];
    desc[b].normF = std::sqrt(g);
  }
  // descending column norms of every block (de Rijk's ordering), W and V
  // permuted alike
  // blocks still iterating: a block leaves after its first sweep without a
  // rotation (later sweeps would leave it unchanged: its columns stay in
  // order and no pair rotates), so converged blocks cost no further rounds
  std::vector<char> active(nb, 1);
  auto sort_permute = [&](const std::function<bool()>& tables) {
    std::vector<PermJob> pj;
    std::vector<char> moved(nb, 0);
    for (int b = 0; b < nb; ++b) {
      if (!active[b]) continue;
      int* p = hp + noff[b];
      const double* w = hn.data() + noff[b];
      std::iota(p, p + K[b], 0);
      std::stable_sort(p, p + K[b], [&](int x, int y) { return w[x] > w[y]; });
      moved[b] = !std::is_sorted(p, p + K[b]);
      if (!moved[b]) continue;
      // the norms follow their columns
      for (long long h : {noff[b], ncol + noff[b]}) {
        std::vector<double> old(hn.begin() + h, hn.begin() + h + K[b]);
        for (int i = 0; i < K[b]; ++i) hn[h + i] = old[p[i]];
      }
      pj.push_back(PermJob{Wc[b], Wo[b], L[b], K[b], 0, noff[b]});
      pj.push_back(PermJob{Vc[b], Vo[b], K[b], K[b], 0, noff[b]});
    }
    for (int b = 0; b < nb; ++b) {
      if (!moved[b]) continue;
      std::swap(Wc[b], Wo[b]);
      std::swap(Vc[b], Vo[b]);
    }
    // the caller's entries that follow from the order
    const bool more = tables && tables();
    if (pj.empty() && !more) return;
    prepare_permute(pj);
    upload();
    permute((int)pj.size(), nullptr);
  };
  // QR preconditioning (precond.hpp), one pass: a second one over the columns
  // at the Gram matrix's resolution empties a null space sooner (38 against 45 ms
  // at 2000 multiplets) but leaves its values ten times below those of other
  // sectors; while the cut went by them, runs that kept more multiplets than
  // their state has filled up with directions of the wrong sectors (first 16x8
  // sweeps up to 12 % above the usual energy).
  // Columns sorted, then W <- W P Q2 and V <- P Q2.  A block's own size and the
  // setting decide, so its bits do not depend on the rest of the batch (a block
  // left out is sorted here instead of at the first sweep: the same
  // permutation, and the first sweep's sort is then the identity).
  {
    std::vector<PrecondBlock> pb;
    std::vector<int> pre;
    for (int b = 0; b < nb; ++b)
      if (precondition_min_k > 0 && K[b] <= kPrecondMaxK &&
          (K[b] >= precondition_min_k || (!plain && precondition_min_k <= kPrecondDefault)))
        pre.push_back(b);
    if (!pre.empty()) {
      sort_permute(nullptr);
      for (int b : pre)
        pb.push_back(PrecondBlock{Wc[b], Vc[b], Wo[b], Vo[b], L[b], K[b], desc[b].normF});
      precondition_jacobi(c, pb, plain);
      for (int b : pre) {
        std::swap(Wc[b], Wo[b]);
        std::swap(Vc[b], Vo[b]);
      }
      upload();
      norms();
    }
  }
  // Deflation: the columns of a block above the rounding level, kept[b] of
  // them, lead the block after the descending sort, and only they are
  // scheduled.  A column at the rounding level is never rotated again (the
  // rotate launch skips its pairs), so kept[b] only falls; the QR
  // preconditioner puts a rank-deficient block's null directions into such
  // columns at once (a 16x8 D=2000 centre sector: 626 of 1383).  The count
  // comes from the block's own norms, so the bits do not depend on the batch.
  std::vector<int> kept(K.begin(), K.end());
  auto count_kept = [&]() {
    bool changed = false;
    for (int b = 0; b < nb; ++b) {
      if (!active[b]) continue;
      const double thr = kNoiseRel * desc[b].normF * (kNoiseRel * desc[b].normF);
      int k = 0;
      for (int i = 0; i < K[b]; ++i) k += hn[noff[b] + i] > thr;
      changed = changed || k != kept[b];
      kept[b] = k;
    }
    return changed;
  };
  count_kept();
  // the pairs of a sweep by round, and their launch order
  std::vector<std::vector<PairJob>> rounds;
  std::vector<int> round_off, round_pmax;
  std::vector<PairJob> all;
  auto slice_rounds = [&]() {
    all.clear();
    // Row slices: a group (the sectors of one wavefunction) with few pairs in
    // a round spreads each pair's Gram matrix over up to MAX_SLICES workgroups
    // (at least 64 rows each), about slice_target workgroups per group and
    // round, so that the round fills the chip.  The slice count of a pair
    // follows from its own group alone, never from the other groups of the
    // batch: the slices' partial Gram matrices are summed in slice order, so
    // the slicing decides the bits, and a wavefunction gets the same bits
    // alone and in a batch.
    round_off.assign(rounds.size() + 1, 0);
    round_pmax.assign(rounds.size(), 1);
    for (size_t r = 0; r < rounds.size(); ++r) {
      round_off[r] = (int)all.size();
      std::map<int, int> per_group;
      for (const PairJob& j : rounds[r]) per_group[blocks[j.blk]->group]++;
      int used = 1;
      for (PairJob& j : rounds[r]) {
        const int pmax =
            std::min(MAX_SLICES, std::max(1, slice_target / per_group[blocks[j.blk]->group]));
        j.P = std::max(1, std::min(pmax, L[j.blk] / MIN_SLICE_ROWS));
        used = std::max(used, j.P);
      }
      round_pmax[r] = used;
      all.insert(all.end(), rounds[r].begin(), rounds[r].end());
    }
    round_off[rounds.size()] = (int)all.size();
  };
  bool converged = false;
  double worst = 0;
  int sweeps_done = 0;
  if (plain) {
    // round-robin schedule of column-block pairs of the active blocks' kept
    // columns, merged across blocks by round
    auto build_schedule = [&]() {
      rounds.clear();
      all.clear();
      for (int b = 0; b < nb; ++b) {
        if (!active[b]) continue;
        const int kb = kept[b];
        const int ncb = (kb + CB - 1) / CB;
        auto width = [&](int i) { return i >= ncb ? 0 : std::min(CB, kb - i * CB); };
        if (ncb <= 1) {
          if (rounds.empty()) rounds.resize(1);
          if (kb >= 2) rounds[0].push_back(PairJob{b, 0, kb, 0, 0, 1, 0});
          continue;
        }
        const int mp = ncb + (ncb & 1);
        if ((int)rounds.size() < mp - 1) rounds.resize(mp - 1);
        for (int r = 0; r < mp - 1; ++r)
          for (int k = 0; k < mp / 2; ++k) {
            int P = (k == 0) ? mp - 1 : (r + k) % (mp - 1);
            int Q = (k == 0) ? r : (r - k + (mp - 1)) % (mp - 1);
            if (width(P) == 0) std::swap(P, Q);
            if (width(P) == 0) continue;
            rounds[r].push_back(PairJob{b, P * CB, width(P), width(Q) ? Q * CB : 0, width(Q), 1, 0});
          }
      }
      slice_rounds();
    };
    // the full schedule sizes the buffers; a smaller one replaces it in place
    // (a pair of a smaller schedule may take more slices, never more than
    // MAX_SLICES, and no round has more pairs than the full one's)
    build_schedule();
    size_t gpart_cap = 1;
    for (size_t r = 0; r + 1 < round_off.size(); ++r)
      gpart_cap = std::max(gpart_cap, (size_t)(round_off[r + 1] - round_off[r]) * MAX_SLICES);
    DevMem dgpart(c, sizeof(double) * NP * NP * gpart_cap);
    DevMem djobs(c, sizeof(PairJob) * std::max<size_t>(1, all.size())),
        doff(c, sizeof(unsigned long long) * nb);
    auto upload_jobs = [&]() {
      if (!all.empty())
        SU2_HIP(hipMemcpyAsync(djobs.p, all.data(), sizeof(PairJob) * all.size(),
                               hipMemcpyHostToDevice, st));
    };
    upload_jobs();
    std::vector<unsigned long long> hoff(nb);
    converged = all.empty();
    for (int sweep = 0; sweep < max_sweeps && !converged; ++sweep) {
      ++sweeps_done;
      // descending column norms (hn: read back with the previous sweep's
      // convergence counters, or before the first sweep)
      sort_permute(nullptr);
      hipLaunchKernelGGL(fill_u64_kernel, dim3(nblk(nb, 256)), dim3(256), 0, st,
                         (unsigned long long*)doff.p, nb);
      for (size_t r = 0; r < rounds.size(); ++r) {
        const int nj = round_off[r + 1] - round_off[r];
        if (nj == 0) continue;
        const int pm = round_pmax[r];
        const PairJob* jr = (const PairJob*)djobs.p + round_off[r];
        if (CB == 16) {
          hipLaunchKernelGGL((gram_partial_kernel<16, 64, RCH>), dim3(nj * pm), dim3(64), 0, st,
                             ddesc, jr, pm, (double*)dgpart.p);
          hipLaunchKernelGGL((jacobi_rotate_kernel<16, 64>), dim3(nj * pm), dim3(64), 0, st,
                             ddesc, jr, pm, (const double*)dgpart.p, tol,
                             kTolAbs,
                             (unsigned long long*)doff.p, inner_sweeps);
        } else {
          hipLaunchKernelGGL((gram_partial_kernel<32, 1024, 64>), dim3(nj * pm), dim3(1024), 0, st,
                             ddesc, jr, pm, (double*)dgpart.p);
          hipLaunchKernelGGL((jacobi_rotate_kernel<32, 512>), dim3(nj * pm), dim3(512), 0, st,
                             ddesc, jr, pm, (const double*)dgpart.p, tol,
                             kTolAbs,
                             (unsigned long long*)doff.p, inner_sweeps);
        }
      }
      SU2_HIP(hipGetLastError());
      SU2_HIP(hipMemcpyAsync(hoff.data(), doff.p, sizeof(unsigned long long) * nb,
                             hipMemcpyDeviceToHost, st));
      // the column norms for the next sweep's order (or the final one) come
      // back with the counters: one wait per sweep
      norms();
      converged = true;
      worst = 0;
      bool left = false;
      for (int b = 0; b < nb; ++b) {
        if (!active[b]) continue;
        double v;
        std::memcpy(&v, &hoff[b], sizeof v);
        if (v >= 2.0) {   // some pair still rotated this sweep
          converged = false;
          worst = std::max(worst, v - 2.0);
        } else {
          active[b] = 0;
          left = true;
        }
      }
      // columns that fell to the rounding level leave the schedule too
      const bool shrunk = count_kept();
      if ((left || shrunk) && !converged) {
        build_schedule();
        upload_jobs();
      }
    }
  } else {
    // The kept columns' pairs of column blocks that still need a rotation: at
    // the start of a sweep one Gram matrix of each block's kept columns says
    // which, and only those are scheduled, packed into as few rounds as their
    // blocks allow.  (The last sweeps rotate a few pairs among many.)  A block
    // without any has converged.  The schedule follows from the block alone.
    std::vector<std::unique_ptr<DevMem>> gram(nb);
    for (int b = 0; b < nb; ++b)
      gram[b].reset(new DevMem(c, sizeof(double) * (size_t)K[b] * K[b]));
    // flag blocks of the table: how many, their pairs, each block's first pair
    int nflag = 0, npair = 0;
    std::vector<size_t> f0(nb, 0);
    auto flag_blocks = [&]() {
      count_kept();
      nflag = npair = 0;
      for (int b = 0; b < nb; ++b) {
        f0[b] = npair;
        if (!active[b] || kept[b] < 2) continue;
        const int ncb = (kept[b] + CB - 1) / CB;
        hflag[nflag++] = FlagBlock{(const double*)gram[b]->p, kept[b], npair, desc[b].normF};
        npair += ncb * (ncb + 1) / 2;
      }
      return nflag > 0;
    };
    auto build_schedule = [&]() {
      rounds.clear();
      all.clear();
      GemmBatch g;
      for (int b = 0; b < nb; ++b) {
        const int kb = kept[b];
        if (!active[b] || kb < 2) continue;
        g.add((double*)gram[b]->p, kb, kb, kb, Wc[b], L[b], 1, Wc[b], L[b], 0, L[b]);
      }
      g.run(c);
      std::vector<double> flag(npair);
      if (npair > 0) {
        double* h = c.host_scratch(npair);
        hipLaunchKernelGGL(pair_flags_kernel, dim3((unsigned)npair), dim3(256), 0, st, dflagb, nflag,
                           CB, tol, kTolAbs, h);
        SU2_HIP(hipGetLastError());
        SU2_HIP(hipStreamSynchronize(st));
        std::memcpy(flag.data(), h, sizeof(double) * npair);
      }
      worst = 0;
      for (int b = 0; b < nb; ++b) {
        if (!active[b]) continue;
        const int kb = kept[b], ncb = (kb + CB - 1) / CB;
        auto width = [&](int i) { return std::min(CB, kb - i * CB); };
        // blocks whose own columns need rotations, and the pairs that do
        std::vector<char> self(ncb, 0);
        std::vector<std::pair<int, int>> pairs;
        std::vector<char> need((size_t)ncb * ncb, 0);
        if (kb >= 2) {
          size_t f = f0[b];
          for (int i = 0; i < ncb; ++i)
            for (int j = i; j < ncb; ++j, ++f) {
              worst = std::max(worst, flag[f]);
              if (!(flag[f] > 0.0)) continue;
              if (i == j) self[i] = 1;
              else need[(size_t)i * ncb + j] = 1;
            }
        }
        // round-robin order, which spreads a block's pairs over the rounds
        const int mp = ncb + (ncb & 1);
        for (int r = 0; r < mp - 1; ++r)
          for (int k = 0; k < mp / 2; ++k) {
            const int x = (k == 0) ? mp - 1 : (r + k) % (mp - 1);
            const int y = (k == 0) ? r : (r - k + (mp - 1)) % (mp - 1);
            const int i = std::min(x, y), j = std::max(x, y);
            if (j < ncb && need[(size_t)i * ncb + j]) pairs.push_back({i, j});
          }
        std::vector<std::vector<char>> used;   // used[round][column block]
        std::vector<char> seen(ncb, 0);
        auto place = [&](int i, int j) {
          size_t r = 0;
          for (; r < used.size(); ++r)
            if (!used[r][i] && !used[r][j]) break;
          if (r == used.size()) used.push_back(std::vector<char>(ncb, 0));
          used[r][i] = used[r][j] = 1;
          if (rounds.size() <= r) rounds.resize(r + 1);
          PairJob J{b, i * CB, width(i), 0, 0, 1, 0};
          if (j != i) {
            J.q0 = j * CB;
            J.bq = width(j);
          }
          rounds[r].push_back(J);
        };
        for (auto& pr : pairs) {
          place(pr.first, pr.second);
          seen[pr.first] = seen[pr.second] = 1;
        }
        // blocks in no pair: two by two, or alone
        int open = -1;
        for (int i = 0; i < ncb; ++i) {
          if (!self[i] || seen[i]) continue;
          if (open < 0) {
            open = i;
            continue;
          }
          place(open, i);
          seen[open] = seen[i] = 1;
          open = -1;
        }
        if (open >= 0) place(open, open);
        if (used.empty()) {
          active[b] = 0;
          continue;
        }
        // the first visit of a block whose own columns need rotations sweeps
        // all columns of its pair
        std::vector<char> done(ncb, 0);
        for (size_t r = 0; r < used.size(); ++r)
          for (PairJob& J : rounds[r]) {
            if (J.blk != b) continue;
            const int i = J.p0 / CB, j = J.bq ? J.q0 / CB : i;
            J.full = J.bq == 0 || (self[i] && !done[i]) || (self[j] && !done[j]);
            done[i] = done[j] = 1;
          }
      }
      slice_rounds();
    };
    // buffers for the most pairs a round can hold: half the column blocks of
    // every block (or one block alone)
    size_t pair_cap = 0;
    for (int b = 0; b < nb; ++b) pair_cap += std::max(1, ((K[b] + CB - 1) / CB + 1) / 2);
    const size_t gsz = (size_t)(NP / 16) * (NP / 16 + 1) / 2 * 256;
    DevMem dgpart(c, sizeof(double) * gsz * MAX_SLICES * pair_cap);
    DevMem drot(c, sizeof(double) * 2 * NP * NP * pair_cap), dact(c, sizeof(int) * 2 * pair_cap);
    int lmax = 0, kmax = 0;
    for (int b = 0; b < nb; ++b) {
      lmax = std::max(lmax, L[b]);
      kmax = std::max(kmax, K[b]);
    }
    const int rows_per_tile = (CB == 32 ? SolveThreads<32>::value : SolveThreads<16>::value) / 4;
    const int wt = (lmax + rows_per_tile - 1) / rows_per_tile;
    const int vt = (kmax + rows_per_tile - 1) / rows_per_tile;
    // each round's three launches, and a last one for V's rotations of the last round
    auto run_rounds = [&](auto cb) {
      constexpr int B = decltype(cb)::value;
      constexpr int NT = SolveThreads<B>::value;
      const BlockDesc* dd = ddesc;
      DevMem djobs(c, sizeof(PairJob) * all.size());
      SU2_HIP(hipMemcpyAsync(djobs.p, all.data(), sizeof(PairJob) * all.size(),
                             hipMemcpyHostToDevice, st));
      const PairJob* prev = nullptr;
      int nprev = 0;
      const double* prot = nullptr;
      const int* pact = nullptr;
      for (size_t r = 0; r <= rounds.size(); ++r) {
        const bool tail = r == rounds.size();
        const int nj = tail ? 0 : round_off[r + 1] - round_off[r];
        const int pm = tail ? 1 : round_pmax[r];
        const PairJob* jr = (const PairJob*)djobs.p + (tail ? 0 : round_off[r]);
        double* rot = (double*)drot.p + (r & 1) * (size_t)NP * NP * pair_cap;
        int* act = (int*)dact.p + (r & 1) * pair_cap;
        SU2_CHECK((size_t)nj <= pair_cap, kErrCapacity, "jacobi: %d pairs in a round", nj);
        if (nj > 0)
          hipLaunchKernelGGL(gram_kernel<B>, dim3(nj * pm), dim3(256), 0, st, dd, jr, pm,
                             (double*)dgpart.p);
        if (nj + nprev > 0)
          hipLaunchKernelGGL(solve_kernel<B>, dim3(nj + nprev * vt), dim3(NT), 0, st, dd, jr, nj,
                             pm, (const double*)dgpart.p, tol, kTolAbs, inner_sweeps, rot, act,
                             (int*)dmoved.p, prev, vt, prot, pact);
        if (nj > 0)
          hipLaunchKernelGGL(apply_kernel<B>, dim3(nj * wt), dim3(NT), 0, st, dd, jr, wt,
                             (const double*)rot, (const int*)act);
        prev = jr;
        nprev = nj;
        prot = rot;
        pact = act;
      }
      SU2_HIP(hipGetLastError());
    };
    for (int sweep = 0; sweep <= max_sweeps; ++sweep) {
      // descending column norms (hn: read back after the previous sweep)
      sort_permute(flag_blocks);
      build_schedule();
      converged = all.empty();
      if (converged || sweep == max_sweeps) break;
      ++sweeps_done;
      // The solve launches test every scheduled pair again, on Gram matrices
      // summed in another order.  A pair at the threshold can pass there, so a
      // block whose pairs all passed is done: nothing would change in the next
      // sweep, nor its flags.
      if (CB == 16) run_rounds(std::integral_constant<int, 16>{});
      else run_rounds(std::integral_constant<int, 32>{});
      norms();
      for (int b = 0; b < nb; ++b)
        if (!rotated[b]) active[b] = 0;
    }
  }
  // Out of sweeps: the columns are accepted when orthogonal to 1e-6 of their
  // norms -- the singular values then carry errors of order 1e-12 relative
  // (second order in the residual overlaps), harmless for a truncation --
  // and the shortfall is reported through *worst_out; beyond that it is an
  // error.
  SU2_CHECK(converged || worst <= 1e-6, kErrNumeric,
            "jacobi svd: no convergence after %d sweeps (worst |w_i.w_j|/|w_i||w_j| = %.2e)",
            max_sweeps, worst);
  if (worst_out) *worst_out = converged ? 0.0 : worst;

  // singular values in ascending order, sign convention on V (W follows),
  // results into the caller's buffers -- for every block in a few launches;
  // hn holds the final column norms
  for (int b = 0; b < nb; ++b) {
    JacobiBlock& J = *blocks[b];
    const int k = K[b];
    // s_i = |W e_i| / |V e_i|: the singular value of the normalised triplet
    std::vector<double> s2(k);
    for (int i = 0; i < k; ++i) {
      const double v2 = hn[ncol + noff[b] + i];
      s2[i] = v2 > 0.0 ? hn[noff[b] + i] / v2 : hn[noff[b] + i];
    }
    int* perm = hp + noff[b];
    std::iota(perm, perm + k, 0);
    std::stable_sort(perm, perm + k, [&](int x, int y) { return s2[x] < s2[y]; });
    J.s.resize(k);
    for (int i = 0; i < k; ++i) J.s[i] = std::sqrt(s2[perm[i]]);
  }
  // V and W in that order with V's signs into J.V and J.W, by way of the spare
  // buffer where those hold the source
  std::vector<PermJob> pj;
  std::vector<VecMove> moves;
  for (int b = 0; b < nb; ++b) {
    JacobiBlock& J = *blocks[b];
    double* vdst = J.V == Vc[b] ? Vo[b] : J.V;
    double* wdst = J.W == Wc[b] ? Wo[b] : J.W;
    pj.push_back(PermJob{Vc[b], vdst, K[b], K[b], 0, noff[b]});
    pj.push_back(PermJob{Wc[b], wdst, L[b], K[b], 0, noff[b]});
    if (wdst != J.W) moves.push_back(VecMove{wdst, J.W, (long long)L[b] * K[b], kMoveF64, 0});
    if (vdst != J.V) moves.push_back(VecMove{vdst, J.V, (long long)K[b] * K[b], kMoveF64, 0});
  }
  prepare_permute(pj);
  upload();
  hipLaunchKernelGGL(col_sign_batched_kernel, dim3((unsigned)ncol), dim3(256), 0, st, ddesc,
                     (const long long*)dnoff.p, nb, dperm, (double*)dsign.p);
  permute((int)pj.size(), (const double*)dsign.p);
  dev_moves(c, moves);
  // no wait: the outputs are used in stream order, and the host results (s)
  // are already on the host
  SU2_HIP(hipGetLastError());
  return sweeps_done;
}

int jacobi_svd_batched(Context& c, std::vector<JacobiBlock>& blocks, double tol, int max_sweeps,
                       int block_cols, int inner_sweeps, double* worst_out,
                       int precondition_min_k, bool plain) {
  // a block's own shape decides, so its bits do not depend on the rest of
  // the batch
  std::vector<JacobiBlock*> small, large, by_slices;
  for (JacobiBlock& b : blocks) {
    const int L = std::max(b.m, b.n), k = std::min(b.m, b.n);
    if (plain) by_slices.push_back(&b);
    else if (small_svd_fits(b.m, b.n)) small.push_back(&b);
    // the usual iteration takes the whole Gram matrix, and W Q2, from grouped
    // GEMMs, the plain one only row slices of W (2 000 000 x 20 does not fit,
    // nor about 23000 x 23000)
    else if (gemm_slice_fits(Prec::F64, k, k, L, L, 1, L, 0) &&
             gemm_slice_fits(Prec::F64, L, k, k, L, 0, k, 0)) large.push_back(&b);
    else by_slices.push_back(&b);
  }
  double w1 = 0.0, w2 = 0.0, w3 = 0.0;
  const int n1 = small_svd_batched(c, small, tol, kTolAbs, kNoiseRel, max_sweeps, &w1);
  const int n2 = jacobi_svd_large(c, large, tol, max_sweeps, block_cols, inner_sweeps, &w2,
                                  precondition_min_k, false);
  const int n3 = jacobi_svd_large(c, by_slices, tol, max_sweeps, block_cols, inner_sweeps, &w3,
                                  precondition_min_k, true);
  if (worst_out) *worst_out = std::max({w1, w2, w3});
  return std::max({n1, n2, n3});
}

}  // namespace su2
