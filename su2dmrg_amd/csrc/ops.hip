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
  const int id = (int)entries_.size();
  entries_.push_back(Entry{d, -1});
  const auto it = last_.emplace(key, (int)groups_.size());
  int launch = 0;
  if (!it.second) {
    Group& g = groups_[it.first->second];
    const StridedAxpy& h = entries_[g.first].d;
    if (h.dst == d.dst && h.rs == d.rs && h.cs == d.cs && h.rows == d.rows && h.cols == d.cols &&
        (h.src != nullptr) == (d.src != nullptr)) {
      entries_[g.last].next = id;
      g.last = id;
      ++g.count;
      return;
    }
    launch = g.launch + 1;
    it.first->second = (int)groups_.size();
  }
  launches_ = std::max(launches_, launch + 1);
  groups_.push_back(Group{id, id, 1, launch});
}

void ScatterBatch::run(Context& c) {
  if (groups_.empty()) return;
  // the groups by launch, in the order they were opened
  std::vector<int> ends(launches_, 0);
  for (const Group& g : groups_) ++ends[g.launch];
  for (int i = 1; i < launches_; ++i) ends[i] += ends[i - 1];
  std::vector<int> at(launches_, 0);
  for (int i = 1; i < launches_; ++i) at[i] = ends[i - 1];
  std::vector<const Group*> order(groups_.size());
  for (const Group& g : groups_) order[at[g.launch]++] = &g;
  std::vector<StridedAxpy> desc;
  desc.reserve(entries_.size());
  std::vector<StridedSum> sums;
  sums.reserve(groups_.size());
  for (const Group* g : order) {
    sums.push_back(StridedSum{(int)desc.size(), g->count});
    for (int e = g->first; e >= 0; e = entries_[e].next) desc.push_back(entries_[e].d);
  }
  dev_strided_sums(c, desc, sums, ends);
}

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
