#include "ops.hpp"

#include <algorithm>

#include "common.hpp"
#include "context.hpp"

namespace su2 {

namespace {

constexpr int kScalesPerLaunch = 80;
struct ScaleArgs {
  ScaledColumns j[kScalesPerLaunch];
};

// blockIdx.y the matrix, 1024 elements per workgroup
__global__ __launch_bounds__(256) void scaled_columns_kernel(const ScaleArgs args) {
  const ScaledColumns J = args.j[blockIdx.y];
  const long long n = (long long)J.rows * J.cols;
  const long long e0 = (long long)blockIdx.x * 1024;
  for (long long e = e0 + threadIdx.x; e < min(e0 + 1024, n); e += 256)
    J.dst[e] = J.src[e] * J.f[e / J.rows];
}

}  // namespace

void GemmBatch::add(double* C, long long ldc, int M, int N, const double* A, long long lda, int tA,
                    const double* B, long long ldb, int tB, int K, double alpha) {
  if (M <= 0 || N <= 0) return;
  if (K <= 0) {
    zero_.push_back({C, {ldc, {M, N}}});
    return;
  }
  int p = g_.add_problem(C, ldc, M, N);
  g_.add_slice(p, A, lda, tA, B, ldb, tB, K, alpha);
  ++n_;
}

void GemmBatch::run(Context& c, int variant) {
  for (auto& z : zero_) {
    // a K == 0 product is a zero block; columns are contiguous of length M
    const long long ldc = z.second.first;
    const int M = z.second.second.first, N = z.second.second.second;
    if (ldc == M) dev_fill(c, z.first, (long long)M * N, 0.0);
    else
      for (int j = 0; j < N; ++j) dev_fill(c, z.first + (long long)j * ldc, M, 0.0);
  }
  if (n_ == 0) return;
  g_.finalize(c, 256, 64, variant);
  g_.launch(c.stream());
}

void ScatterBatch::add(const void* key, const StridedAxpy& d) {
  if (d.rows <= 0 || d.cols <= 0) return;
  auto it = last_.find(key);
  int launch = 0;
  if (it != last_.end()) {
    StridedSum& g = launches_[it->second.first][it->second.second];
    const StridedAxpy& h = g[0];
    if (h.dst == d.dst && h.rs == d.rs && h.cs == d.cs && h.rows == d.rows && h.cols == d.cols &&
        (h.src != nullptr) == (d.src != nullptr)) {
      g.push_back(d);
      return;
    }
    launch = it->second.first + 1;
  }
  if ((int)launches_.size() <= launch) launches_.resize(launch + 1);
  launches_[launch].push_back(StridedSum{d});
  last_[key] = {launch, (int)launches_[launch].size() - 1};
}

void ScatterBatch::run(Context& c) { dev_strided_axpy_launches(c, launches_); }

void dev_scaled_columns(Context& c, const std::vector<ScaledColumns>& jobs) {
  ScaleArgs args;
  for (size_t i0 = 0; i0 < jobs.size(); i0 += kScalesPerLaunch) {
    const int n = (int)std::min<size_t>(kScalesPerLaunch, jobs.size() - i0);
    long long most = 0;
    for (int i = 0; i < n; ++i) {
      args.j[i] = jobs[i0 + i];
      most = std::max(most, (long long)args.j[i].rows * args.j[i].cols);
    }
    if (most <= 0) continue;
    hipLaunchKernelGGL(scaled_columns_kernel, dim3((unsigned)((most + 1023) / 1024), n), dim3(256),
                       0, c.stream(), args);
    SU2_HIP(hipGetLastError());
  }
}

}  // namespace su2
