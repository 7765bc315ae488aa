// One-sided Jacobi SVD in LDS, see small_svd.hpp.
//
// The columns of W (the block or its transpose, L x k with L >= k) and of V (k x k, from the
// identity) are stacked in LDS, longest columns first.  Then W is made lower trapezoidal by
// Householder reflectors from the right, each for the row with the largest remaining norm (W Q is
// then the transposed R factor of a QR with column pivoting of W^T, on which Jacobi converges fast
// after Drmac and Veselic; V becomes Q).  Last, pairs of columns are rotated until orthogonal
// (Hestenes): a sweep has k - 1 round-robin rounds of k / 2 disjoint pairs, a group of lanes owns a
// pair for one round, and one barrier separates two rounds.  Nothing else does: no launch, no Gram
// matrix, no host wait.
// Columns are never reordered between sweeps: after the reflectors they come in nearly descending
// order, and a model of the iteration took 7 sweeps without reordering at k = 44, 8 with it, 24
// without the reflectors (7, 9 and more than 20 at k = 120).
//
// A workgroup has one CU to itself, so a round is bound by the instructions one wave issues (4
// cycles each), not by LDS or arithmetic.  The workgroup is four waves, one per SIMD, and the lanes
// per pair are the most that still fit them (16 up to k = 32, 8 up to 64, 4 above): the rotation's
// scalar chain, the same on every lane of a pair, then serves 4, 8 or 16 pairs at once.  A lane
// holds two neighbouring rows at a time (16-byte LDS accesses); squared norms are carried from
// round to round and computed anew every sweep, which leaves one dot product per pair.  Measured at
// k = 42 (clock stamps): 4150 cycles per reflector, 7 sweeps of 41 rounds at 1620 cycles, of which
// 416 wait for the columns (LDS bandwidth: both columns of every pair pass through it each round),
// 75 form the dot product, 290 the rotation, the rest updates, drains and waits for the slowest
// wave.  The SVD call of a d = 64 step: 2.95 ms by pairs of 32-column blocks, 0.36 ms here.
#include "small_svd.hpp"

#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "context.hpp"
#include "jacobi.hpp"

namespace su2 {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxK = 128;
constexpr int kMaxL = 128;
constexpr int kColChunk = 8;      // columns a wave loads at once for a reflector
// 160 KB of LDS per CU, less the small arrays
constexpr int kLdsDoubles = 20480 - 2 * kThreads - 3 * kMaxK;
// elements of the block per thread (W is half of the LDS array at most)
constexpr int kElems = (kLdsDoubles / 2 + kThreads - 1) / kThreads;

typedef double f64x2 __attribute__((ext_vector_type(2)));

struct SmallDesc {
  const double* A;
  double* W;
  double* V;
  double* out;       // k squared singular values, then sweeps and worst squared overlap (pinned)
  int m, n, ld;
};

constexpr int kBlocksPerLaunch = 64;   // descriptors travel as kernel arguments
struct SmallArgs {
  SmallDesc d[kBlocksPerLaunch];
};

// Lanes per pair (see above).
__host__ __device__ inline int pair_lanes(int k) { return k <= 32 ? 16 : k <= 64 ? 8 : 4; }

// Row pairs per lane of a column's W part (its V part has as many), rounded up to a compiled
// unrolling: every value for 16 and 8 lanes, the even ones for 4.
__host__ __device__ inline int row_pairs(int L, int k) {
  const int g = pair_lanes(k), r = (L + 2 * g - 1) / (2 * g);
  return g == 4 ? (r + 1) / 2 * 2 : r;
}

// Column pitch: 2 G modulo 32 doubles, so that the 16-byte reads of neighbouring columns, which
// neighbouring pairs of a round hold, fall on different banks.
__host__ __device__ inline int column_pitch(int L, int k) {
  const int g = pair_lanes(k), rows = 4 * g * row_pairs(L, k);
  return rows + ((2 * g) % 32 - rows % 32 + 32) % 32;
}

template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  union {
    double d;
    int i[2];
  } u, v;
  u.d = x;
  v.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], CTRL, 0xf, 0xf, true);
  v.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], CTRL, 0xf, 0xf, true);
  return v.d;
}

// Sum over G neighbouring lanes, the same bits on each of them: quad swaps (1, 0, 3, 2) and (2, 3,
// 0, 1), then the half-row and row mirrors.
template <int G>
__device__ __forceinline__ double group_sum(double x) {
  x += dpp_move<0xB1>(x);
  x += dpp_move<0x4E>(x);
  if (G >= 8) x += dpp_move<0x141>(x);
  if (G >= 16) x += dpp_move<0x140>(x);
  return x;
}
__device__ __forceinline__ double max16(double x) {
  x = fmax(x, dpp_move<0xB1>(x));
  x = fmax(x, dpp_move<0x4E>(x));
  x = fmax(x, dpp_move<0x141>(x));
  return fmax(x, dpp_move<0x140>(x));
}
__device__ __forceinline__ int min16(int x) {
  x = min(x, __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true));
  x = min(x, __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true));
  x = min(x, __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true));
  return min(x, __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, true));
}

// x of lane l (the same l on every lane)
__device__ __forceinline__ double lane_value(double x, int l) {
  union {
    double d;
    int i[2];
  } u;
  u.d = x;
  u.i[0] = __builtin_amdgcn_readlane(u.i[0], l);
  u.i[1] = __builtin_amdgcn_readlane(u.i[1], l);
  return u.d;
}

// x >= 0 with its low bits replaced by a row (compares as x does, up to 2^-43 of it), and the row
__device__ __forceinline__ double tagged(double x, int row) {
  return __longlong_as_double((__double_as_longlong(x) & ~511ll) | (511 - row));
}
__device__ __forceinline__ int tag_of(double x) {
  return __builtin_amdgcn_readfirstlane(511 - (int)(__double_as_longlong(x) & 511ll));
}

// 1 / x and 1 / sqrt(x) for normal x > 0 from the hardware estimates (relative error about 2^-24):
// two Newton-Raphson steps, one third-order step
__device__ __forceinline__ double recip(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}
__device__ __forceinline__ double rsqrt_of(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double recip_signed(double x) { return copysign(recip(fabs(x)), x); }

// Constants of one workgroup.
struct Shape {
  int k, ld, mk, npair;
  double noise2, in2, out2, tol2;
};

// One round: group grp's pair of round r, the lane's rows from X + 2 g.  nrm: squared column norms.
// Returns the pair's squared overlap if the outer test calls for a further sweep, else 0.
template <int G, int NW>
__device__ __forceinline__ double rotate_pair(double* X, double* nrm, const Shape& S, int r,
                                              int grp) {
  int p = r + grp, q = r - grp;
  if (p >= S.mk - 1) p -= S.mk - 1;
  if (q < 0) q += S.mk - 1;
  if (grp == 0) p = S.mk - 1;
  if (p >= S.k || q >= S.k) return 0.0;
  f64x2* P = (f64x2*)(X + p * S.ld);
  f64x2* Q = (f64x2*)(X + q * S.ld);
  const double al = nrm[p], be = nrm[q];
  f64x2 x[NW], y[NW], u[NW], v[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    x[i] = P[G * i];
    y[i] = Q[G * i];
  }
  // with few rows per lane the V rows' loads run under the chain below
  constexpr bool kEager = NW <= 8;
  if (kEager) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      u[i] = P[G * (NW + i)];
      v[i] = Q[G * (NW + i)];
    }
  }
  double ga = 0.0, gb = 0.0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    ga = fma(x[i].x, y[i].x, ga);
    gb = fma(x[i].y, y[i].y, gb);
  }
  ga = group_sum<G>(ga + gb);
  // |g_pq| against 1e-14 sqrt(g_pp g_qq) and the rounding floor of columns that carry absolute
  // errors of order eps ||A||; columns at the rounding level of the block carry no direction and
  // are left alone
  const double g2 = ga * ga, ab = al * be;
  const bool rot = g2 > 1e-28 * ab && g2 > S.in2 * fmax(al, be) && fmin(al, be) > S.noise2 &&
                   g2 > 0.0;
  // tan of the smaller rotation angle, 2 g sign(d) / (|d| + sqrt(d^2 + 4 g^2)), from the hardware
  // estimates: what 2^-24 of it leaves of g is far below what the other rotations of the sweep
  // bring back, and c = 1 / sqrt(1 + t^2) keeps the rotation orthogonal to rounding for any t
  const double d = be - al, h2 = fma(d, d, 4.0 * g2);
  const double den = fma(h2, __builtin_amdgcn_rsq(h2), fabs(d));
  const double t = copysign(2.0, d) * ga * __builtin_amdgcn_rcp(den);
  const double c = rsqrt_of(fma(t, t, 1.0)), s = t * c;
  if (!rot) return 0.0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    P[G * i] = f64x2{fma(-s, y[i].x, c * x[i].x), fma(-s, y[i].y, c * x[i].y)};
    Q[G * i] = f64x2{fma(c, y[i].x, s * x[i].x), fma(c, y[i].y, s * x[i].y)};
  }
  if (!kEager) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      u[i] = P[G * (NW + i)];
      v[i] = Q[G * (NW + i)];
    }
  }
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    P[G * (NW + i)] = f64x2{fma(-s, v[i].x, c * u[i].x), fma(-s, v[i].y, c * u[i].y)};
    Q[G * (NW + i)] = f64x2{fma(c, v[i].x, s * u[i].x), fma(c, v[i].y, s * u[i].y)};
  }
  // every lane of the pair writes the same norms
  nrm[p] = fma(-t, ga, al);
  nrm[q] = fma(t, ga, be);
  return g2 > S.tol2 * ab && g2 > S.out2 * (al + be) ? g2 * __builtin_amdgcn_rcp(ab) : 0.0;
}

// Squared norms of every column over its row pairs i0 <= i < i1 of G lanes.
template <int G>
__device__ __forceinline__ void column_norms(const double* X, int k, int ld, int i0, int i1, int t,
                                             double* out) {
  const int g = t % G;
  for (int c = t / G; c < k; c += kThreads / G) {
    const f64x2* P = (const f64x2*)(X + c * ld + 2 * g);
    double a = 0.0;
    for (int i = i0; i < i1; ++i) {
      const f64x2 x = P[G * i];
      a = fma(x.x, x.x, fma(x.y, x.y, a));
    }
    a = group_sum<G>(a);
    if (g == 0) out[c] = a;
  }
}

// Sweeps until no pair needs a rotation; returns their number, *done whether they converged.
// s_worst: two slots in turn, the next sweep's cleared while this one's is read.
template <int G, int NW>
__device__ __forceinline__ int run_sweeps(double* X, double* nrm, const Shape& S, int t,
                                          int max_sweeps, unsigned long long* s_worst,
                                          bool* done) {
  const int grp = t / G;
  double* Xg = X + 2 * (t % G);
  int sweep = 0;
  *done = S.k < 2;
  for (; sweep < max_sweeps && !*done; ++sweep) {
    column_norms<G>(X, S.k, S.ld, 0, NW, t, nrm);
    __syncthreads();
    double worst = 0.0;
    for (int r = 0; r < S.mk - 1; ++r) {
      if (grp < S.npair) worst = fmax(worst, rotate_pair<G, NW>(Xg, nrm, S, r, grp));
      __syncthreads();
    }
    if (worst > 0.0)
      atomicMax(&s_worst[sweep & 1], (unsigned long long)__double_as_longlong(worst));
    __syncthreads();
    *done = s_worst[sweep & 1] == 0ull;
    if (t == 0 && !*done) s_worst[(sweep & 1) ^ 1] = 0ull;
    __syncthreads();
  }
  return sweep;
}

__global__ __launch_bounds__(kThreads, 1) void small_svd_kernel(const SmallArgs args,
                                                                double tol, double tol_abs,
                                                                double noise_rel,
                                                                int max_sweeps) {
  extern __shared__ __align__(16) double X[];
  __shared__ double s_y[kThreads], s_n[kThreads];
  __shared__ double s_norm[kMaxK], s_inv[kMaxK];
  double* const s_p = s_inv;   // the pivot row of a reflector
  __shared__ int s_pos[kMaxK];
  __shared__ unsigned long long s_worst[2];
  const SmallDesc D = args.d[blockIdx.x];
  const int L = max(D.m, D.n), k = min(D.m, D.n), ld = D.ld;
  const int G = pair_lanes(k), NW = row_pairs(L, k), Lp = 2 * G * NW, rows = 2 * Lp;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);

  // W (the block, transposed when it is wider than tall), V = 1, their columns in one order, zeros
  // in the padding
  for (int e = t; e < ld * k; e += kThreads) X[e] = 0.0;
  if (t < 2) s_worst[t] = 0ull;
  __syncthreads();
  // the block's elements, by way of registers (their order in LDS is not known yet)
  const int total = D.m * D.n;
  double a[kElems];
#pragma unroll
  for (int i = 0; i < kElems; ++i) {
    if (kThreads * i >= total) break;
    const int e = t + kThreads * i;
    a[i] = e < total ? D.A[e] : 0.0;
  }
  auto place = [&](auto column) {
    int r = t % D.m, c = t / D.m;
    const int dr = kThreads % D.m, dc = kThreads / D.m;
#pragma unroll
    for (int i = 0; i < kElems; ++i) {
      if (kThreads * i >= total) break;
      if (t + kThreads * i < total) {
        if (D.m >= D.n) X[column(c) * ld + r] = a[i];
        else X[column(r) * ld + c] = a[i];
      }
      r += dr;
      c += dc;
      if (r >= D.m) {
        r -= D.m;
        ++c;
      }
    }
  };
  // Columns by descending norm.  A Householder QR of W^T with pivoting (the reflectors below) is
  // then backward stable column by column of W as well, after Cox and Higham, and values far below
  // the largest keep their relative accuracy where W's columns span many decades: 48 shuffled
  // columns over six decades lost 2e-11 of the smallest values unsorted and lose 2e-15.
  place([](int c) { return c; });
  __syncthreads();
  column_norms<4>(X, k, ld, 0, Lp / 8, t, s_norm);
  __syncthreads();
  for (int c = t; c < k; c += kThreads) {
    const double v = s_norm[c];
    int pos = 0;   // ties by column, NaN first
    for (int d = 0; d < k; ++d) {
      const double u = s_norm[d];
      pos += u != u ? v == v || d < c : u > v || (u == v && d < c);
    }
    s_pos[c] = pos;
    X[pos * ld + Lp + c] = 1.0;
  }
  __syncthreads();
  place([&](int c) { return s_pos[c]; });
  __syncthreads();

  // ---- Householder reflectors from the right ----
  // Wave (rb, cg): rows 64 rb + lane of the columns cg, cg + ncg, ...  Every row's remaining squared
  // norm is kept as ncg partial sums in s_n, so each wave finds the pivot row (and its norm, which
  // the reflector needs) by itself; two barriers per reflector.
  const int nrb = (rows + 63) / 64, ncg = kWaves / nrb;
  const int rb = wave % nrb, cg = wave / nrb;
  const int row = 64 * rb + lane;
  const bool mine = cg < ncg && row < rows;
  bool alive = mine && row < L;   // a W row that no reflector has taken yet
  double* C = X + min(row, rows - 1);
  {
    double a = 0.0;
    if (alive)
      for (int j = cg; j < k; j += ncg) a = fma(C[j * ld], C[j * ld], a);
    s_n[t] = a;
  }
  __syncthreads();
  // the rows' norms, ncg partial sums each (rows past L and surplus waves hold zeros)
  auto row_norm = [&](int q) {
    if (ncg == 4)
      return q ? 0.0 : (s_n[lane] + s_n[64 + lane]) + (s_n[128 + lane] + s_n[192 + lane]);
    const double a = s_n[64 * q + lane];
    return ncg == 2 ? a + s_n[128 + 64 * q + lane] : a;
  };
  double fro;
  {
    const double a = group_sum<16>(row_norm(0) + row_norm(1));
    fro = sqrt((lane_value(a, 0) + lane_value(a, 16)) + (lane_value(a, 32) + lane_value(a, 48)));
  }
  const double noise2 = (noise_rel * fro) * (noise_rel * fro);
  for (int i = 0; i < k - 1; ++i) {
    // pivot: the row of W with the largest remaining norm, the same on every wave.  The search
    // compares norms whose low bits hold the row; the reflector takes the exact one.
    const double n0 = row_norm(0), n1 = row_norm(1);
    double best = max16(fmax(tagged(n0, lane), tagged(n1, 64 + lane)));
    best = fmax(fmax(lane_value(best, 0), lane_value(best, 16)),
                fmax(lane_value(best, 32), lane_value(best, 48)));
    // the remaining columns are at the rounding level of the block: nothing to order.  The exact
    // norm decides where that level underflows: the row in the low bits of `best` makes a norm of
    // zero positive, and the reciprocals below take normal numbers only.
    const int piv = tag_of(best);
    const double nn = lane_value(piv >= 64 ? n1 : n0, piv % 64);
    if (!(best > 1e-4 * noise2) || !(nn >= 0x1p-1022)) break;
    const double alpha = X[i * ld + piv];
    const double beta = -copysign(nn * rsqrt_of(nn), alpha);
    const double tau = (beta - alpha) * recip_signed(beta), scale = recip_signed(alpha - beta);
    // this wave's columns j0, j0 + ncg, ...; the reflector is v = (1, scale p_j), p the pivot row,
    // which every lane reads (one address: a broadcast) and the first row block saves, since the
    // update overwrites it
    const int im = i % ncg, j0 = i - im + cg + (cg < im ? ncg : 0);
    const int nj = cg < ncg && j0 < k ? (k - 1 - j0) / ncg + 1 : 0;
    const int cs = ncg * ld;
    double* Cj = C + j0 * ld;
    const double* Pj = X + piv + j0 * ld;
    const bool first = nj > 0 && j0 == i;
    // chunks of columns, the last one filled up with its last column
    double y = 0.0;
    for (int c = 0; c < nj; c += kColChunk) {
      double x[kColChunk], p[kColChunk];
#pragma unroll
      for (int u = 0; u < kColChunk; ++u) {
        const int o = min(c + u, nj - 1) * cs;
        x[u] = Cj[o];
        p[u] = Pj[o];
      }
#pragma unroll
      for (int u = 0; u < kColChunk; ++u) {
        if (c + u >= nj) break;
        y = fma(x[u], p[u], y);
        if (rb == 0) s_p[j0 + (c + u) * ncg] = p[u];
      }
    }
    // y = x_i + scale sum_{j > i} x_j p_j
    if (first) {
      const double x = Cj[0];
      y = fma(-x, alpha, y);
      s_y[t] = fma(scale, y, x);
    } else {
      s_y[t] = scale * y;
    }
    if (row == piv) alive = false;
    __syncthreads();
    const double* sy = s_y + 64 * rb + lane;
    y = ncg == 4 ? (sy[0] + sy[64]) + (sy[128] + sy[192]) : ncg == 2 ? sy[0] + sy[128] : sy[0];
    y = mine ? -tau * y : 0.0;
    const double ys = y * scale;
    // the update, and the rows' norms over the columns after i
    double nrm = 0.0;
    for (int c = 0; c < nj; c += kColChunk) {
      double x[kColChunk], p[kColChunk];
#pragma unroll
      for (int u = 0; u < kColChunk; ++u) {
        const int o = min(c + u, nj - 1);
        x[u] = Cj[o * cs];
        p[u] = s_p[j0 + o * ncg];
      }
#pragma unroll
      for (int u = 0; u < kColChunk; ++u) {
        if (c + u >= nj) break;
        const bool head = u == 0 && c == 0 && first;
        x[u] = head ? x[u] + y : fma(ys, p[u], x[u]);
        if (mine) Cj[(c + u) * cs] = x[u];
        if (!head) nrm = fma(x[u], x[u], nrm);
      }
    }
    s_n[t] = alive ? nrm : 0.0;
    __syncthreads();
  }
  __syncthreads();

  // ---- Jacobi ----
  Shape S;
  S.k = k;
  S.ld = ld;
  S.mk = k + (k & 1);
  S.npair = S.mk / 2;
  S.noise2 = noise2;
  S.in2 = (0.2 * tol_abs * fro) * (0.2 * tol_abs * fro);
  S.out2 = (tol_abs * fro) * (tol_abs * fro);
  S.tol2 = tol * tol;
  bool done = false;
  int sweep = 0;
  switch (100 * G + NW) {
#define SU2_CASE(G, N)                                                         \
  case 100 * G + N:                                                            \
    sweep = run_sweeps<G, N>(X, s_norm, S, t, max_sweeps, s_worst, &done);     \
    break;
    SU2_CASE(16, 1) SU2_CASE(16, 2) SU2_CASE(16, 3) SU2_CASE(16, 4)
    SU2_CASE(8, 3) SU2_CASE(8, 4) SU2_CASE(8, 5) SU2_CASE(8, 6) SU2_CASE(8, 7) SU2_CASE(8, 8)
    SU2_CASE(4, 10) SU2_CASE(4, 12) SU2_CASE(4, 14) SU2_CASE(4, 16)
#undef SU2_CASE
    default:
      break;
  }
  if (t == 0) {
    D.out[k] = (double)sweep;
    D.out[k + 1] = done ? 0.0 : __longlong_as_double((long long)s_worst[(sweep - 1) & 1]);
  }

  // s_i = |W e_i| / |V e_i|; the accumulated rotations leave V's columns off unit length by their
  // rounding, and W = A V carries the same factor
  column_norms<4>(X, k, ld, 0, Lp / 8, t, s_norm);
  column_norms<4>(X, k, ld, Lp / 8, 2 * Lp / 8, t, s_inv);
  __syncthreads();
  for (int c = t; c < k; c += kThreads)
    s_norm[c] = s_inv[c] > 0.0 ? s_norm[c] / s_inv[c] : s_norm[c];
  __syncthreads();
  // ascending order, ties by column (a NaN counts as the largest value)
  for (int c = t; c < k; c += kThreads) {
    const double v = s_norm[c];
    const bool vn = !(v == v);
    int pos = 0;
    for (int d = 0; d < k; ++d) {
      const double u = s_norm[d];
      const bool un = !(u == u);
      pos += (vn ? !un || d < c : !un && (u < v || (u == v && d < c)));
    }
    s_pos[c] = pos;
    D.out[pos] = v;
  }
  __syncthreads();
  // V's first entry of at least half its column's largest is positive, both columns over |V e_i|
  const int g = t % 16;
  for (int c = t / 16; c < k; c += kThreads / 16) {
    double best = 0.0;
    for (int i = g; i < k; i += 16) best = fmax(best, fabs(X[c * ld + Lp + i]));
    best = 0.5 * max16(best);
    int first = k;
    for (int i = g; i < k; i += 16)
      if (fabs(X[c * ld + Lp + i]) >= best) first = min(first, i);
    first = min16(first);
    const double inv = s_inv[c] > 0.0 ? 1.0 / sqrt(s_inv[c]) : 1.0;
    const double f = (first < k && X[c * ld + Lp + first] < 0.0) ? -inv : inv;
    const int pos = s_pos[c];
    for (int i = g; i < L; i += 16) D.W[(long long)pos * L + i] = f * X[c * ld + i];
    for (int i = g; i < k; i += 16) D.V[(long long)pos * k + i] = f * X[c * ld + Lp + i];
  }
}

}  // namespace

bool small_svd_fits(int m, int n) {
  const int L = std::max(m, n), k = std::min(m, n);
  return k <= kMaxK && L <= kMaxL && (long long)column_pitch(L, k) * k <= kLdsDoubles;
}

int small_svd_batched(Context& c, const std::vector<JacobiBlock*>& blocks, double tol,
                      double tol_abs, double noise_rel, int max_sweeps, double* worst) {
  if (worst) *worst = 0.0;
  const int nb = (int)blocks.size();
  if (nb == 0) return 0;
  hipStream_t st = c.stream();
  long long tot = 0;
  size_t lds = 0;
  std::vector<long long> off(nb);
  std::vector<SmallDesc> desc(nb);
  for (int i = 0; i < nb; ++i) {
    const JacobiBlock& b = *blocks[i];
    SU2_CHECK(b.m >= 1 && b.n >= 1 && small_svd_fits(b.m, b.n), kErrArgument,
              "small svd: block %d x %d", b.m, b.n);
    const int L = std::max(b.m, b.n), k = std::min(b.m, b.n);
    off[i] = tot;
    tot += k + 2;
    desc[i] = SmallDesc{b.A, b.W, b.V, nullptr, b.m, b.n, column_pitch(L, k)};
    lds = std::max(lds, sizeof(double) * (size_t)desc[i].ld * k);
  }
  double* host = c.host_scratch(tot);
  // the most any launch takes, and not this one's need: the attribute is the
  // kernel's, and another context's thread may set it before this launch
  SU2_HIP(hipFuncSetAttribute((const void*)small_svd_kernel,
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)(sizeof(double) * kLdsDoubles)));
  for (int i0 = 0; i0 < nb; i0 += kBlocksPerLaunch) {
    SmallArgs args;
    const int n = std::min(kBlocksPerLaunch, nb - i0);
    for (int i = 0; i < n; ++i) {
      args.d[i] = desc[i0 + i];
      args.d[i].out = host + off[i0 + i];
    }
    hipLaunchKernelGGL(small_svd_kernel, dim3(n), dim3(kThreads), lds, st, args, tol, tol_abs,
                       noise_rel, max_sweeps);
    SU2_HIP(hipGetLastError());
  }
  SU2_HIP(hipStreamSynchronize(st));
  int sweeps = 0;
  double w = 0.0;
  for (int i = 0; i < nb; ++i) {
    JacobiBlock& b = *blocks[i];
    const int k = std::min(b.m, b.n);
    const double* h = host + off[i];
    b.s.resize(k);
    for (int j = 0; j < k; ++j) b.s[j] = std::sqrt(h[j]);
    sweeps = std::max(sweeps, (int)h[k]);
    w = std::max(w, std::sqrt(h[k + 1]));
  }
  // out of sweeps: the columns are accepted when orthogonal to 1e-6 (as jacobi_svd_batched)
  SU2_CHECK(w <= 1e-6, kErrNumeric,
            "jacobi svd: no convergence after %d sweeps (worst |w_i.w_j|/|w_i||w_j| = %.2e)",
            max_sweeps, w);
  if (worst) *worst = w;
  return sweeps;
}

}  // namespace su2
