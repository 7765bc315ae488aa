// Small device building blocks shared by the SVD, environment and driver code.
#pragma once

#include <unordered_map>
#include <tuple>
#include <vector>

#include "blas1.hpp"
#include "gemm.hpp"

namespace su2 {

class Context;

// A batch of independent GEMMs launched as one grouped FP64 MFMA launch.
//   C = alpha op(A) op(B)        (C overwritten)
class GemmBatch {
 public:
  void add(double* C, long long ldc, int M, int N, const double* A, long long lda, int tA,
           const double* B, long long ldb, int tB, int K, double alpha = 1.0);
  // launch on the context stream (zero-fills problems with K == 0)
  void run(Context& c, int variant = -1);
  bool empty() const { return n_ == 0; }

 private:
  GroupedGemm g_;
  std::vector<std::pair<double*, std::pair<long long, std::pair<int, int>>>> zero_;
  int n_ = 0;
};

// Strided scale-adds (StridedAxpy) collected with a destination key.  Entries
// of one key are summed in the order of add(): those that write the same
// elements in the same layout one after the other in a thread, others in
// successive launches.  Entries of different keys write disjoint elements.
class ScatterBatch {
 public:
  void add(const void* key, const StridedAxpy& d);
  void run(Context& c);

 private:
  // entries in order of add(), each naming the next of its group (-1: the
  // last); one flat list, since a step adds thousands of them
  struct Entry {
    StridedAxpy d;
    int next;
  };
  struct Group {
    int first, last, count, launch;
  };
  std::vector<Entry> entries_;
  std::vector<Group> groups_;
  std::unordered_map<const void*, int> last_;   // key -> its last group
  int launches_ = 0;
};

// dst[:, j] = f[j] * src[:, j] for the cols columns of rows contiguous
// elements each, many matrices in a launch (descriptors as kernel arguments).
struct ScaledColumns {
  double* dst;
  const double* src;
  const double* f;
  int rows, cols;
};
void dev_scaled_columns(Context& c, const std::vector<ScaledColumns>& jobs);

}  // namespace su2
