// One-sided block Jacobi SVD (Hestenes) of many dense blocks at once.
//
// The reference obtains each sector's singular vectors from the Gram matrix
// with dsyev and then re-diagonalises the small-eigenvalue subspace again and
// again to recover their accuracy (tensor.cpp:1472-1529).  Here the columns
// of the block itself are rotated until mutually orthogonal: for a block A
// (m x n) with k = min(m, n) the working matrix W is A (m >= n) or A^T, and
// the accumulated rotation V (k x k) converges to the Gram eigenvectors, so
// that W = A V holds the reference's u = A v and the column norms of W are
// the singular values, accurate relative to each value rather than to the
// largest one.
//
// Blocks that fit one CU's LDS are decomposed there by one workgroup each
// (small_svd.hpp); the rest of this description is about the larger ones.
// Columns are cut into blocks of 16 (or 32), and before each sweep they are put
// in descending norm order.  Two iterations rotate them:
//
// The usual one starts from QR-preconditioned columns (precond.hpp; blocks from
// the caller's limit on, and with a limit up to 256 the smaller ones too).  A
// sweep begins with the Gram matrix of the columns above the rounding level,
// which says which pairs of column blocks still need a rotation; only those
// are visited, in rounds of disjoint pairs, with three launches per round:
// partial Gram matrices of the pairs over row slices of W, one workgroup per
// pair that diagonalises
// its (up to 64 x 64) Gram matrix in LDS by parallel cyclic Jacobi, p columns
// against q columns (all of them in a block's first visit), and the pairs'
// columns of W times the result (V's a round later, beside the next
// diagonalisations).  A block is done when no pair needs a rotation, or when
// every scheduled pair passed the launch's own test, on sums in another order.
//
// The plain one visits every pair once per sweep with two launches per round
// (Gram matrices, then every row slice diagonalises the whole pair for itself
// and rotates its rows of W and V), preconditioned from the caller's limit on
// only.  It is kept for uncut SVD calls (svd.hpp says why) and for blocks past
// the grouped GEMM's 4 GB of addresses.  Measured against
// it: svd call of a d = 500 step 20.6 -> 7.8 ms, d = 2000 84 -> 45 ms; a 192 x
// 192 block 13.3 -> 3.7 ms, 1390 x 1383 of rank 1106 66 -> 35 ms.
//
// Sweeps stop when every pair is orthogonal to
// |g_ij| <= max(tol * sqrt(g_ii g_jj), 1e-14 ||A||_F (sqrt g_ii + sqrt g_jj))
// (the absolute floor ends the iteration on columns that carry rounding
// errors of order eps ||A||); columns with norm <= kNoiseRel ||A||_F are left
// out of the test.
#pragma once

#include <vector>

namespace su2 {

class Context;

// Columns with norm at or below kNoiseRel ||A||_F are at the rounding level of
// the block: they carry no direction, no pair with one of them holds the
// iteration open, and the sweeps leave them as they are.
constexpr double kNoiseRel = 1e-13;

struct JacobiBlock {
  const double* A;   // m x n, column-major, leading dimension m (device)
  int m, n;
  double* W;         // out: L x k (L = max(m, n), k = min(m, n)), ld L, columns by
                     //      ascending singular value (device, caller-allocated)
  double* V;         // out: k x k, ld k, matching columns (device, caller-allocated)
  std::vector<double> s;   // out: k singular values, ascending
  int group = 0;           // blocks of one group (one wavefunction) share the
                           // row slicing of their pairs; groups never affect
                           // each other's bits
};

// Decomposes every block and returns the number of sweeps it took.  W and V
// columns are sorted ascending by singular value; each
// column of V has its first entry with |v| >= max|v|/2 made positive (the
// LAPACK routine the reference calls leaves signs open), W's columns follow.
// block_cols: 16 (pairs of 32 columns, one wave per pair) or 32 (pairs of 64
// columns, eight waves per pair); inner_sweeps: 1..3 inner Jacobi sweeps per
// visit of a pair.
// worst_out (nullable) receives 0 when every block converged, else the
// largest remaining |w_i.w_j| / |w_i||w_j| (accepted up to 1e-6, beyond it
// the call throws).
// precondition_min_k: QR-precondition the blocks with precondition_min_k <=
// min(m, n) <= kPrecondMaxK first (precond.hpp; 0: none); the results differ
// from the unpreconditioned iteration's by rounding only.
// plain: the plain iteration, for every block.
int jacobi_svd_batched(Context& c, std::vector<JacobiBlock>& blocks, double tol = 1e-13,
                       int max_sweeps = 60, int block_cols = 32, int inner_sweeps = 1,
                       double* worst_out = nullptr, int precondition_min_k = 0,
                       bool plain = false);

}  // namespace su2
