// Vector algebra of the Lanczos iteration (lanczos_su2.cpp:36-47, 125-195,
// 262-279, 320-332), whole steps of many solves at a time.
//
// Every sum is taken in the order of dev_dot (blas1.hpp): 512 x 256 strided
// lanes, a fixed tree inside each 256, a fixed tree over the 512, so a vector
// length always sums in the same order, on either path below.
#pragma once

#include <vector>

namespace su2 {

class Context;

enum KrylovKind : int {
  kKrylovNormalise,   // v[0] = psi / |psi|;                         slot b: <psi|psi>
  kKrylovFirst,       // v[1] -= <v0|v1> v0, then normalised;        slot a: |v1|^2, alpha
  kKrylovStep,        // v[m] -= <v[m-1]|v[m]> v[m-1] + beta v[m-2], then against v[0..m-1] one
                      // after the other, then normalised;           slot a: |v[m]|^2, alpha
  kKrylovOverlap,     // alpha: <v[m-1]|v[m]>
  kKrylovCheck,       // slot a: <tmp|tmp>, slot b: <tmp|psi>
};

// One job's next operation.  v[k] = base + k * ld; alpha, a and b are pinned
// host scalars, written before the stream reaches what is queued next.  A
// norm of zero (or NaN) leaves its vector as it is.
struct KrylovOp {
  int kind, m;
  double* base;
  long long ld, n;
  double* psi;
  double* tmp;
  double beta;
  double *alpha, *a, *b;
};

// psi = sum_j z[j] v[j] (in order, from zero), then, when normalise is set,
// psi /= |psi|, |psi|^2 into a.
struct KrylovRitz {
  double* base;
  long long ld, n;
  double* psi;
  std::vector<double> z;
  bool normalise;
  double* a;
};

// Partial sums of `jobs` concurrent operations, in doubles.
long long krylov_partials(int jobs);
// Queues the operations (different jobs: they touch disjoint vectors) on the
// context's stream; part holds krylov_partials(ops.size()) doubles.  No wait.
void krylov_run(Context& c, const std::vector<KrylovOp>& ops, double* part);
void krylov_ritz(Context& c, const std::vector<KrylovRitz>& jobs, double* part);

}  // namespace su2
