// One-sided Jacobi SVD of blocks that fit one CU's LDS: one launch for every
// such block of a batch, one workgroup per block, no host round trip between
// sweeps.
#pragma once

#include <vector>

namespace su2 {

class Context;
struct JacobiBlock;

// Whether an m x n block is decomposed by small_svd_batched: its columns and
// its accumulated rotations fit the LDS of one CU (up to 96 x 96, or 128 rows
// and about 75 columns), the most the kernel takes.  There it is the faster
// one throughout (whole SVD call, 32 x 32: 0.24 ms against 2.06 ms by pairs
// of column blocks; 64 x 64: 0.61 against 3.8; 96 x 96: 1.73 against 7.9).
// Depends on the block's shape alone.
bool small_svd_fits(int m, int n);

// Decomposes the given blocks (every one small_svd_fits) as jacobi_svd_batched
// describes: W, V and s of each, ascending.  Returns the largest sweep count;
// *worst (nullable) as there.
int small_svd_batched(Context& c, const std::vector<JacobiBlock*>& blocks, double tol,
                      double tol_abs, double noise_rel, int max_sweeps, double* worst);

}  // namespace su2
