// Preconditioner of the one-sided Jacobi SVD, see precond.hpp.
#include "precond.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "context.hpp"
#include "ops.hpp"

namespace su2 {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int PB = 16;        // panel width
constexpr int PT = 1024;      // threads of the panel kernels
constexpr int PROWS = 2;      // rows (or columns) per thread of the panel kernels
static_assert(PT * PROWS == kPrecondMaxK, "panel register tile");

struct PDesc {
  double* G;   // K x K, column-major: Gram matrix, then the Cholesky factor Rc
               // (upper, zeros below).  Read row-major it is X = Rc^T (X[i][j]
               // at G[j + i K]), which the Householder QR then overwrites
               // with its vectors (below X's diagonal)
  double* Q;   // K x K, column-major: Q2
  double* T;   // 256 per panel: the panel's 16 x 16 upper triangular T (column-major)
  int K;
  int rk;      // rows of Rc up to its last nonzero pivot (X's later columns are zero)
  double tiny; // Cholesky pivot floor
};

// Compile-time loop: f(std::integral_constant<int, k>) for k = K0 .. K1-1, so
// that register arrays are indexed by constants only (a runtime index would
// send them to scratch memory).
template <int K0, int K1, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (K0 < K1) {
    f(std::integral_constant<int, K0>{});
    static_for<K0 + 1, K1>(f);
  }
}

// Lane `src`'s x on every lane, in scalar registers.
__device__ __forceinline__ double lane_value(double x, int src) {
  union { double d; int i[2]; } u, v;
  u.d = x;
  v.i[0] = __builtin_amdgcn_readlane(u.i[0], src);
  v.i[1] = __builtin_amdgcn_readlane(u.i[1], src);
  return v.d;
}

// Upper Cholesky of G by one 16-row panel: rows c0..c0+bp-1, columns c0..K-1.
// A pivot at or below tiny (or negative from rounding) gives a zero row.
// Bound by the 16 dependent pivots: every workgroup factors the 16 x 16
// diagonal block for itself in one wave, column c on lane c, without barriers,
// and then solves 256 further columns, one per thread.  The factor of the
// diagonal block goes to D.T (workgroups still read the block);
// rank_prefix_kernel puts it in place.  One workgroup for all columns with a
// barrier per pivot took 27 us a panel in the sectors of a D = 2000 bond where
// this takes 12, 16 against 8 on a 6x4 run's blocks.
constexpr int kCholCols = 256;

__global__ __launch_bounds__(kCholCols) void chol_panel_kernel(const PDesc* __restrict__ desc,
                                                               int p) {
  const PDesc D = desc[blockIdx.y];
  const int K = D.K, c0 = PB * p;
  if (c0 >= K) return;
  const int bp = min(PB, K - c0), nc = K - c0;
  const int j0 = PB + (int)blockIdx.x * kCholCols;
  if (blockIdx.x > 0 && j0 >= nc) return;
  const int t = threadIdx.x, j = j0 + t;
  // -R[k][i] / R[k][k]-scaled multipliers and the inverse pivots
  __shared__ double s_f[PB][PB], s_inv[PB];
  double w[PB];
  double* const gcol = D.G + (size_t)(c0 + min(j, nc - 1)) * K + c0;
#pragma unroll
  for (int i = 0; i < PB; ++i) w[i] = (j < nc && i < bp) ? gcol[i] : 0.0;
  if (t < 64) {
    const int c = t & 15;
    double d[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i)
      d[i] = (c < bp && i < bp) ? D.G[(size_t)(c0 + c) * K + c0 + i] : 0.0;
    static_for<0, PB>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const double dk = lane_value(d[k], k);
      const double inv = (k < bp && dk > D.tiny) ? 1.0 / sqrt(dk) : 0.0;
      const double rk = c >= k ? d[k] * inv : 0.0;
      // lane i's f multiplies row k into row i
      const double fi = -d[k] * inv;
      if (t < PB) s_f[k][t] = fi;
      if (t == 0) s_inv[k] = inv;
#pragma unroll
      for (int i = k + 1; i < PB; ++i) {
        const double f = lane_value(fi, i);
        if (i <= c) d[i] = fma(f, rk, d[i]);
      }
      d[k] = rk;
    });
    if (blockIdx.x == 0 && t < PB)
#pragma unroll
      for (int i = 0; i < PB; ++i)
        D.T[(size_t)p * PB * PB + i + PB * t] = i <= t ? d[i] : 0.0;
  }
  __syncthreads();
  if (j < nc) {
    static_for<0, PB>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      w[k] *= s_inv[k];
#pragma unroll
      for (int i = k + 1; i < PB; ++i) w[i] = fma(s_f[k][i], w[k], w[i]);
    });
#pragma unroll
    for (int i = 0; i < PB; ++i)
      if (i < bp) gcol[i] = w[i];
    // the panel's columns below its diagonal block: zero (Rc is upper
    // triangular, and read row-major they are X's entries above its diagonal)
    for (int i = 0; i < bp; ++i) D.G[(size_t)(c0 + j) + (size_t)(c0 + i) * K] = 0.0;
  }
}

// Trailing update of the Cholesky: G[i][j] -= sum_k R[c0+k][i] R[c0+k][j]
// for c1 <= i <= j (upper triangle only; the panel kernels read nothing
// below it).  64 x 64 tiles, k summed in order.
__global__ __launch_bounds__(256) void chol_trail_kernel(const PDesc* __restrict__ desc, int p) {
  const PDesc D = desc[blockIdx.z];
  const int K = D.K, c0 = PB * p, c1 = c0 + PB;
  if (c1 >= K) return;
  const int ti = blockIdx.x, tj = blockIdx.y;
  const int n = K - c1;
  if (ti > tj || ti * 64 >= n || tj * 64 >= n) return;
  __shared__ double Ri[PB][64], Rj[PB][64];
  const int t = threadIdx.x;
  for (int e = t; e < PB * 64; e += 256) {
    const int k = e / 64, x = e % 64;
    const int gi = c1 + ti * 64 + x, gj = c1 + tj * 64 + x;
    Ri[k][x] = gi < K ? D.G[(size_t)(c0 + k) + (size_t)gi * K] : 0.0;
    Rj[k][x] = gj < K ? D.G[(size_t)(c0 + k) + (size_t)gj * K] : 0.0;
  }
  __syncthreads();
  const int x = t % 64;                 // row within the tile (contiguous in memory)
  const int gi = c1 + ti * 64 + x;
  for (int s = 0; s < 16; ++s) {
    const int y = t / 64 + 4 * s;       // column within the tile
    const int gj = c1 + tj * 64 + y;
    if (gi < K && gj < K && gi <= gj) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < PB; ++k) acc = fma(Ri[k][x], Rj[k][y], acc);
      D.G[(size_t)gi + (size_t)gj * K] -= acc;
    }
  }
}

// Orthogonal factor of one 16-column panel of X (rows c0..K-1) in compact WY
// form, I - V T V^T = H_0 ... H_{b-1}.  A reflector needs inner products of the
// updated columns; the panel's Gram matrix X^T X does not change under the
// reflectors, so with it and the panel's first 16 rows one wave finds all 16 of
// them without another pass: the products over the rows below row j are
// (X^T X)_jc minus those over rows 0..j.  The same updates applied to an
// identity give M with V = X M below the first 16 rows.  The differences lose
// digits where a column nearly depends on those before it, so V need not
// annihilate exactly; T^-1 = striu(V^T V) + diag(V^T V) / 2, taken from the V
// that was stored, makes I - V T V^T orthogonal for any V, and only that counts
// for a preconditioner.  A column whose remainder is below kDepends of it gets
// no reflector.
//
// Three short phases on one workgroup, bound by the 16 dependent reflectors
// (about 5 us) and, from about 1000 rows, by the 12 MFMAs per 16 rows on the
// CU's four matrix cores.  Reducing every reflector's 16 products over the
// workgroup took 65 us a panel against 21 in the sectors of a D = 2000 bond (up to 1383), 51 against
// 14 on those of a 6x4 run up to d = 924.
constexpr double kDepends = 1e-13;

__global__ __launch_bounds__(PT) void wy_panel_kernel(const PDesc* __restrict__ desc, int p) {
  const PDesc D = desc[blockIdx.x];
  const int K = D.K, c0 = PB * p;
  // a panel of zero columns (past the last nonzero pivot) is the identity
  if (c0 >= D.rk) return;
  const int bp = min(PB, K - c0), m = K - c0;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  constexpr int NW = PT / 64;
  const int row4 = lane >> 4, col = lane & 15;
  __shared__ double s_part[NW][PB * PB];
  __shared__ double s_g[PB][PB + 1], s_m[PB][PB + 1], s_v[PB][PB + 1];
  static_assert(PB == 16, "16 x 16 x 4 MFMAs");
  double* const X = D.G + (size_t)c0 * K + c0;   // row r, column c at X[r K + c]

  // sum of the waves' 16 x 16 results (register r of lane l: row l/16 + 4 r, column l%16)
  auto gather = [&](const f64x4& acc) {
#pragma unroll
    for (int r = 0; r < 4; ++r) s_part[wave][(row4 + 4 * r) * PB + col] = acc[r];
    __syncthreads();
    if (t < PB * PB) {
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += s_part[w][t];
      s_g[t / PB][t % PB] = v;
    }
    __syncthreads();
  };

  // X^T X: four rows a step, the same register as both operands
  {
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int r0 = 4 * wave; r0 < m; r0 += 4 * NW) {
      const int r = r0 + row4;
      const double x = (r < m && col < bp) ? X[(size_t)r * K + col] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x, x, acc, 0, 0, 0);
    }
    gather(acc);
  }

  // the reflectors: lane c (of each 16) holds column c of the first 16 rows,
  // of the Gram matrix and of M
  unsigned used = 0;
  if (wave == 0) {
    double x[PB], g[PB], mm[PB];
#pragma unroll
    for (int r = 0; r < PB; ++r) {
      x[r] = (r < m && col < bp) ? X[(size_t)r * K + col] : 0.0;
      g[r] = s_g[r][col];
      mm[r] = (r == col && col < bp) ? 1.0 : 0.0;
    }
    static_for<0, PB>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j < bp) {
        // products over the rows below j
        double d = g[j];
#pragma unroll
        for (int r = 0; r <= j; ++r) d = fma(-lane_value(x[r], j), x[r], d);
        const double alpha = lane_value(x[j], j), sig2 = lane_value(d, j),
                     gjj = lane_value(g[j], j);
        double tau = 0.0, scale = 0.0;
        if (sig2 > kDepends * gjj) {
          const double beta = -copysign(sqrt(fma(alpha, alpha, sig2)), alpha);
          tau = (beta - alpha) / beta;
          scale = 1.0 / (alpha - beta);
          used |= 1u << j;
        }
        const double f = col > j ? -tau * fma(scale, d, x[j]) : 0.0;
        if (col > j) x[j] += f;
#pragma unroll
        for (int r = j + 1; r < PB; ++r) {
          const double v = lane_value(x[r], j) * scale;
          x[r] = col == j ? v : fma(f, v, x[r]);
        }
#pragma unroll
        for (int r = 0; r <= j; ++r) {
          const double v = lane_value(mm[r], j) * scale;
          mm[r] = col == j ? v : fma(f, v, mm[r]);
        }
      }
    });
    if (lane < PB) {
#pragma unroll
      for (int r = 0; r < PB; ++r) {
        if (r < m && col < bp) X[(size_t)r * K + col] = x[r];
        s_v[r][col] = (col >= bp || r < col) ? 0.0 : r == col ? 1.0 : x[r];
        s_m[r][col] = mm[r];
      }
    }
  }
  __syncthreads();

  // V = X M below them, 16 rows a step, and V^T V
  {
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    double b[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) b[s] = s_m[4 * s + row4][col];
    if (wave == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double v = s_v[row4 + 4 * r][col];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, acc, 0, 0, 0);
      }
    }
#pragma unroll 2
    for (int r0 = PB + PB * wave; r0 < m; r0 += PB * NW) {
      double a[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int r = r0 + col, c = 4 * s + row4;
        a[s] = (r < m && c < bp) ? X[(size_t)r * K + c] : 0.0;
      }
      f64x4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s) y = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], y, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = r0 + row4 + 4 * r;
        if (row < m && col < bp) X[(size_t)row * K + col] = y[r];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(y[r], y[r], acc, 0, 0, 0);
      }
    }
    gather(acc);
  }

  // T by back substitution, column c on lane c
  if (wave == 0) {
    const double inv = (used >> col & 1u) ? 2.0 / s_g[col][col] : 0.0;
    double tc[PB];
    static_for<0, PB>([&](auto ic) {
      constexpr int i = PB - 1 - decltype(ic)::value;
      double acc = i == col ? 1.0 : 0.0;
#pragma unroll
      for (int k = i + 1; k < PB; ++k) acc = fma(-s_g[i][k], tc[k], acc);
      tc[i] = acc * lane_value(inv, i);
    });
    if (lane < PB)
#pragma unroll
      for (int i = 0; i < PB; ++i) D.T[(size_t)p * PB * PB + i + PB * col] = tc[i];
  }
}

// Householder QR of one 16-column panel of X for the plain iteration, reflector
// by reflector (rows c0..K-1; row c0 + r on
// thread r % 1024, in registers).
// Column j becomes its Householder vector below the diagonal (the unit
// diagonal implicit); the panel's T factor of the compact WY form H_0 ...
// H_{b-1} = I - V T V^T goes to D.T.  Each step takes one block reduction of
// the 16 products d_c = sum_{r>j} x_j(r) x_c(r): with row j, they give
// sigma^2 = d_j, w_c = v_j^T x_c = x_c(j) + scale d_c (c > j) and
// y_c = v_c^T v_j = x_c(j) + scale d_c (c < j, for T).
__global__ __launch_bounds__(PT) void hh_panel_kernel(const PDesc* __restrict__ desc, int p) {
  const PDesc D = desc[blockIdx.x];
  const int K = D.K, c0 = PB * p;
  // a panel of zero columns (past the last nonzero pivot) is the identity
  if (c0 >= D.rk) return;
  const int bp = min(PB, K - c0), m = K - c0;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  __shared__ double s_red[2][PT / 64][PB + 1];
  __shared__ double s_row[2][PB];
  __shared__ double s_d[2][PB];
  __shared__ double s_T[PB][PB];
  double x[2][PB];
  double* xrow[PROWS];
#pragma unroll
  for (int s = 0; s < PROWS; ++s) {
    const int r = t + PT * s;
    xrow[s] = D.G + (size_t)(c0 + min(r, m - 1)) * K + c0;
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int r = t + PT * s;
#pragma unroll
    for (int c = 0; c < PB; ++c) x[s][c] = (r < m && c < bp) ? xrow[s][c] : 0.0;
  }
  if (t < PB * PB) s_T[t % PB][t / PB] = 0.0;
  static_for<0, PB>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    __builtin_amdgcn_sched_barrier(0);
    if (j < bp) {
      const int b = j & 1;
      // d_c over my rows below the diagonal, summed over each wave by a
      // reduce-scatter (lanes that differ in bit 32, 16, 8, 4 swap halves of
      // their 16, 8, 4, 2 sums, then the last sum is reduced over bits 2, 1):
      // 17 exchanges instead of 16 x 6
      double v[PB];
#pragma unroll
      for (int c = 0; c < PB; ++c) {
        v[c] = 0.0;
        if (c < bp) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const int r = t + PT * s;
            if (r > j && r < m) v[c] = fma(x[s][j], x[s][c], v[c]);
          }
        }
      }
      static_assert(PB == 16, "reduce-scatter of 16 sums over a 64-lane wave");
#pragma unroll
      for (int h = 8, o = 32; h >= 1; h >>= 1, o >>= 1) {
        // keep the upper h sums on lanes with bit o set, the lower h otherwise
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int i = 0; i < h; ++i) {
          const double send = up ? v[i] : v[h + i];
          const double keep = up ? v[h + i] : v[i];
          v[i] = keep + __shfl_xor(send, o);
        }
      }
      v[0] += __shfl_xor(v[0], 2);
      v[0] += __shfl_xor(v[0], 1);
      if ((lane & 3) == 0) {
        const int c = ((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 +
                      ((lane >> 2) & 1);
        s_red[b][wave][c] = v[0];
      }
      if (t == j) {
#pragma unroll
        for (int c = 0; c < PB; ++c) s_row[b][c] = x[0][c];
      }
      __syncthreads();
      if (t < PB) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < PT / 64; ++w) v += s_red[b][w][t];
        s_d[b][t] = v;
      }
      __syncthreads();
      // the reflector, computed alike on every thread
      const double alpha = s_row[b][j], sig2 = s_d[b][j];
      double tau = 0.0, scale = 0.0;
      if (sig2 != 0.0) {
        const double beta = -copysign(sqrt(fma(alpha, alpha, sig2)), alpha);
        tau = (beta - alpha) / beta;
        scale = 1.0 / (alpha - beta);
      }
      // T column j (T[t][k], k < j, was written by this same thread)
      if (t < j) {
        double acc = 0.0;
        for (int k = t; k < j; ++k) acc = fma(s_T[t][k], fma(scale, s_d[b][k], s_row[b][k]), acc);
        s_T[t][j] = -tau * acc;
      }
      if (t == j) s_T[j][j] = tau;
      // v_j into column j, H_j applied to the later columns (rows >= j);
      // w_c = v_j^T x_c read from LDS once for all rows
      double wc[PB];
#pragma unroll
      for (int c = j + 1; c < PB; ++c) wc[c] = fma(scale, s_d[b][c], s_row[b][c]);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int r = t + PT * s;
        if (r >= j && r < m) {
          const double vr = (r == j) ? 1.0 : x[s][j] * scale;
          if (r > j) x[s][j] = vr;
#pragma unroll
          for (int c = j + 1; c < PB; ++c)
            if (c < bp) x[s][c] = fma(-tau * vr, wc[c], x[s][c]);
        }
      }
    }
  });
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int r = t + PT * s;
    if (r >= m) continue;
#pragma unroll
    for (int c = 0; c < PB; ++c)
      if (c < bp) xrow[s][c] = x[s][c];
  }
  if (t < PB * PB) D.T[(size_t)p * PB * PB + t] = s_T[t % PB][t / PB];
}

// A <- A - V op(T) (V^T A) for 16 columns of A (rows c0..K-1): A = X from
// column c0 + bp (the QR's trailing columns, op(T) = T^T) or A = Q from
// column c0 (Q2's backward formation, op(T) = T).  One workgroup owns its 16
// columns over every row, so the products and the update need no other
// workgroup.  Each of the 16 waves takes every 16th tile of 16 rows: its tiles
// of A stay in registers between the two products (an accumulator's layout is
// that of a B operand), V comes from memory in the layout of either product,
// and the only exchange is the sum of the waves' V^T A in wave order.  Bound
// by the latency of its loads; staging V and A through LDS in 256-row chunks,
// two barriers each, took 27 us in the sectors of a D = 2000 bond where this
// takes 17, 8.6 against 6 on a 6x4 run's blocks.
__global__ __launch_bounds__(1024) void hh_apply_kernel(const PDesc* __restrict__ desc, int p,
                                                        int qr) {
  const PDesc D = desc[blockIdx.y];
  const int K = D.K, c0 = PB * p;
  if (c0 >= D.rk) return;   // identity reflectors
  const int bp = min(PB, K - c0), m = K - c0;
  // X's columns from rk on are zero and stay zero
  const int colstart = c0 + (qr ? bp : 0), ncols = (qr ? D.rk : K) - colstart;
  const int chunk = blockIdx.x * PB;
  if (chunk >= ncols) return;
  // A(row, col): X row-major (the QR's trailing columns) or Q column-major
  const size_t rs = qr ? (size_t)K : 1, cs = qr ? 1 : (size_t)K;
  double* const A = (qr ? D.G : D.Q) + (size_t)c0 * rs + (size_t)(colstart + chunk) * cs;
  const double* const X = D.G + (size_t)c0 * K + c0;   // row r, column c at X[r K + c]
  constexpr int NW = 16, TILES = kPrecondMaxK / (PB * NW);
  __shared__ double sp[NW][PB][PB + 1];   // the waves' partial V^T A
  __shared__ double sz[PB][PB + 1];
  static_assert(PB == 16 && TILES * PB * NW == kPrecondMaxK, "16 waves of 16-row tiles");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int row4 = lane >> 4, col = lane & 15;
  const bool mine = chunk + col < ncols;
  // Householder vector i at panel row r (the unit diagonal implicit)
  auto hh_v = [&](int i, int r) {
    const double v = (i < bp && r < m) ? X[(size_t)r * K + i] : 0.0;
    return i >= bp || r < i ? 0.0 : r == i ? 1.0 : v;
  };
  double a[TILES][4];
  f64x4 pacc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < TILES; ++q) {
    const int r0 = (q * NW + wave) * PB;
    if (r0 >= m) continue;
    // (V^T A)[i][c] += sum over 4 rows: lane l feeds V[row l/16][l%16] as
    // the A operand and A[row l/16][l%16] as the B operand
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int r = r0 + 4 * s + row4;
      a[q][s] = (r < m && mine) ? A[(size_t)r * rs + (size_t)col * cs] : 0.0;
      pacc = __builtin_amdgcn_mfma_f64_16x16x4f64(hh_v(col, r), a[q][s], pacc, 0, 0, 0);
    }
  }
  // result register r of lane l is row l/16 + 4 r, column l % 16
#pragma unroll
  for (int r = 0; r < 4; ++r) sp[wave][row4 + 4 * r][col] = pacc[r];
  __syncthreads();
  const int i = t / PB, c = t % PB;
  if (t < PB * PB) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += sp[w][i][c];
    sp[0][i][c] = v;   // row i of wave 0's block is read by this thread only
  }
  __syncthreads();
  if (t < PB * PB) {
    const double* T = D.T + (size_t)p * PB * PB;   // T[a][b] at a + 16 b
    double z = 0.0;
#pragma unroll
    for (int k = 0; k < PB; ++k) z = fma(qr ? T[k + PB * i] : T[i + PB * k], sp[0][k][c], z);
    sz[i][c] = (chunk + c < ncols) ? z : 0.0;
  }
  __syncthreads();
  // A -= V Z: lane l feeds V[row l%16][k] and Z[k][l%16], k = 4 s + l/16
#pragma unroll
  for (int q = 0; q < TILES; ++q) {
    const int r0 = (q * NW + wave) * PB;
    if (r0 >= m) continue;
    f64x4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = 4 * s + row4;
      y = __builtin_amdgcn_mfma_f64_16x16x4f64(hh_v(k, r0 + col), sz[k][col], y, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = r0 + row4 + 4 * r;
      if (row < m && mine) A[(size_t)row * rs + (size_t)col * cs] = a[q][r] - y[r];
    }
  }
}

// The Cholesky's diagonal blocks into place, and rk of every block: one past
// the last nonzero diagonal entry of Rc (a dropped pivot leaves its whole row
// exactly zero).
__global__ __launch_bounds__(256) void rank_prefix_kernel(PDesc* __restrict__ desc,
                                                          int* __restrict__ rk) {
  const PDesc D = desc[blockIdx.x];
  __shared__ int s[256];
  int last = -1;
  const int i = threadIdx.x % PB, j = threadIdx.x / PB;
  for (int c0 = 0; c0 < D.K; c0 += PB) {
    if (c0 + i >= D.K || c0 + j >= D.K) continue;
    const double v = D.T[(size_t)c0 * PB + i + PB * j];
    D.G[(size_t)(c0 + i) + (size_t)(c0 + j) * D.K] = v;
    if (i == j && v != 0.0) last = max(last, c0 + i);
  }
  s[threadIdx.x] = last;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] = max(s[threadIdx.x], s[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) desc[blockIdx.x].rk = rk[blockIdx.x] = s[0] + 1;
}

__global__ void eye_batched_kernel(const PDesc* __restrict__ desc) {
  const PDesc D = desc[blockIdx.y];
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long n = (long long)D.K * D.K;
  if (e < n) D.Q[e] = (e % D.K) == (e / D.K) ? 1.0 : 0.0;
}

unsigned cdiv(long long a, long long b) { return (unsigned)((a + b - 1) / b); }

}  // namespace

void precondition_jacobi(Context& c, std::vector<PrecondBlock>& blocks, bool plain) {
  const int nb = (int)blocks.size();
  if (nb == 0) return;
  SU2_CHECK(nb < 65536, kErrCapacity, "jacobi preconditioner: %d blocks", nb);
  hipStream_t st = c.stream();
  int kmax = 0;
  long long scratch = 0;
  for (auto& b : blocks) {
    SU2_CHECK(b.K >= 1 && b.K <= kPrecondMaxK && b.L >= b.K, kErrArgument,
              "jacobi preconditioner: block %d x %d", b.L, b.K);
    kmax = std::max(kmax, b.K);
    const long long np = (b.K + PB - 1) / PB;
    scratch += 2LL * b.K * b.K + np * PB * PB;
  }
  DevBuf work(c, scratch);
  std::vector<PDesc> hd(nb);
  long long off = 0;
  for (int i = 0; i < nb; ++i) {
    const PrecondBlock& b = blocks[i];
    const long long kk = (long long)b.K * b.K, np = (b.K + PB - 1) / PB;
    PDesc& d = hd[i];
    d.G = work.p + off;
    d.Q = d.G + kk;
    d.T = d.Q + kk;
    off += 2 * kk + np * PB * PB;
    d.K = b.K;
    d.rk = b.K;
    d.tiny = 1e-15 * b.normF * b.normF;
  }
  DevBuf ddesc(c, (long long)((sizeof(PDesc) * nb + 7) / 8));
  SU2_HIP(hipMemcpyAsync(ddesc.p, hd.data(), sizeof(PDesc) * nb, hipMemcpyHostToDevice, st));
  const PDesc* dd = (const PDesc*)ddesc.p;
  // Gram matrices
  {
    GemmBatch g;
    for (int i = 0; i < nb; ++i) {
      const PrecondBlock& b = blocks[i];
      g.add(hd[i].G, b.K, b.K, b.K, b.W, b.L, 1, b.W, b.L, 0, b.L);
    }
    g.run(c);
  }
  const int npmax = (kmax + PB - 1) / PB;
  // Cholesky by row panels
  for (int p = 0; p < npmax; ++p) {
    const int n = kmax - PB * (p + 1);
    hipLaunchKernelGGL(chol_panel_kernel, dim3(std::max(1u, cdiv(std::max(n, 0), kCholCols)), nb),
                       dim3(kCholCols), 0, st, dd, p);
    if (n > 0) {
      const unsigned nt = cdiv(n, 64);
      hipLaunchKernelGGL(chol_trail_kernel, dim3(nt, nt, nb), dim3(256), 0, st, dd, p);
    }
  }
  // Rc's rank prefix: X = Rc^T has zero columns from rk on (a rank-deficient
  // block, such as a two-site wavefunction sector, drops its last pivots),
  // whose panels are identity reflectors and whose updates change nothing;
  // one wait brings the counts back to bound the panel loops
  {
    int* rk = (int*)c.host_scratch((nb + 1) / 2);
    hipLaunchKernelGGL(rank_prefix_kernel, dim3(nb), dim3(256), 0, st, (PDesc*)ddesc.p, rk);
    SU2_HIP(hipGetLastError());
    SU2_HIP(hipStreamSynchronize(st));
    for (int i = 0; i < nb; ++i) hd[i].rk = rk[i];
  }
  int rkmax = 0;
  for (int i = 0; i < nb; ++i) rkmax = std::max(rkmax, hd[i].rk);
  const int npq = (rkmax + PB - 1) / PB;
  // Householder QR of Rc^T by column panels (trailing columns updated)
  for (int p = 0; p < npq; ++p) {
    hipLaunchKernelGGL(plain ? hh_panel_kernel : wy_panel_kernel, dim3(nb), dim3(PT), 0, st, dd, p);
    const int n = rkmax - PB * (p + 1);
    if (n > 0) {
      hipLaunchKernelGGL(hh_apply_kernel, dim3(cdiv(n, PB), nb), dim3(1024), 0, st, dd, p, 1);
    }
  }
  // Q2 = H_0 ... H_{np-1}, formed backwards from the identity
  hipLaunchKernelGGL(eye_batched_kernel, dim3(cdiv((long long)kmax * kmax, 256), nb), dim3(256),
                     0, st, dd);
  for (int p = npq - 1; p >= 0; --p) {
    const int n = kmax - PB * p;
    hipLaunchKernelGGL(hh_apply_kernel, dim3(cdiv(n, PB), nb), dim3(1024), 0, st, dd, p, 0);
  }
  SU2_HIP(hipGetLastError());
  // W Q2 and V Q2
  {
    GemmBatch g;
    for (int i = 0; i < nb; ++i) {
      const PrecondBlock& b = blocks[i];
      g.add(b.Wout, b.L, b.L, b.K, b.W, b.L, 0, hd[i].Q, b.K, 0, b.K);
      g.add(b.Vout, b.K, b.K, b.K, b.V, b.K, 0, hd[i].Q, b.K, 0, b.K);
    }
    g.run(c);
  }
}

}  // namespace su2
