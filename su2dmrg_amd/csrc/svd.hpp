// Truncated SVD of a two-leg singlet wavefunction across its sectors
// (tensor_su2::svd, tensor_su2.cpp:1619-1758, with tensor::svd per sector,
// tensor.cpp:1472-1700).
//
// Per sector j with block A (m x n): a one-sided Jacobi SVD (jacobi.hpp) of its
// short side's columns, where the reference diagonalises the Gram matrix again
// and again (tensor.cpp:1498-1529); singular values count for w/w_max > 1e-100,
// w = s^2; kept columns are scaled by s^(p1-1)/s^p2 (or s^p1/s^(p2-1)).  The
// largest max_dcut values over all sectors survive, ordered by the reference's
// shell sort so ties at the cut fall the same way (sort2.f:76-111); values at
// the rounding level of their sector are ordered by its norm alone.
#pragma once

#include <memory>
#include <vector>

#include "structure.hpp"
#include "tensor.hpp"

namespace su2 {

struct SvdResult {
  Leg bond;                              // kept sectors (2j ascending), dir -1
  std::unique_ptr<Tensor> U;             // [psi leg 0, bond]
  std::unique_ptr<Tensor> V;             // [psi leg 1, bond]
  std::vector<std::vector<double>> kept; // ascending singular values per bond sector
  double discarded_weight = 0;           // sum of squares of the cut values
  // the reference's wout (tensor_su2.cpp:1707-1731): kept values sector by
  // sector, then the cut ones sector by sector, each ascending
  std::vector<double> wout;
  int jacobi_sweeps = 0;      // one-sided Jacobi sweeps the sectors took
  double t_jacobi = 0;        // seconds inside the Jacobi SVD
  double jacobi_worst = 0;    // 0, or the residual overlap accepted after the
                              // sweep ceiling (no convergence to 1e-13)
};

// keep_all_plain: where nothing can be cut (max_dcut >= the columns of all
// sectors together), use the plain Jacobi iteration (jacobi.hpp).  Such a
// result holds every direction down to the rounding level, where it is
// whatever the iteration leaves; the plain one is kept for callers that store
// or compare the factors, and gives them to rounding as it always has where
// the singular values determine them.  It is two to eight times slower (d =
// 2000 step 84 ms against 45, d = 64 step 2.95 against 0.36), and the DMRG
// solves never ask for it.  They keep null directions too, whenever they keep
// more multiplets than the state has, and grow into them: which ones those are
// changes the way of a run (its first sweep's energy by up to a percent on wide
// cylinders, with any kernel or tuning), not what it converges to.
SvdResult truncated_svd(Context& c, const Tensor& psi, double p1, double p2, int max_dcut,
                        bool keep_all_plain = false);

// Several wavefunctions at once: every sector of every one in one batched
// Jacobi SVD, then each one's keep rule and cut.  Each result equals the
// single call's (its blocks' rotations depend on those blocks alone).
struct SvdJob {
  const Tensor* psi;
  double p1, p2;
  int max_dcut;
  bool keep_all_plain = false;   // as truncated_svd
};
std::vector<SvdResult> truncated_svd_batch(Context& c, const std::vector<SvdJob>& jobs);

}  // namespace su2
