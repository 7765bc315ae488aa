#include "krylov.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "common.hpp"
#include "context.hpp"

namespace su2 {

namespace {

constexpr int kThreads = 256;     // threads of a grid-wide stage, and the leaves of a block sum
constexpr int kDotBlocks = 512;   // block sums of a dot product
constexpr int kMaxBatch = 16;     // jobs per launch (descriptors travel as kernel arguments)
constexpr int kMaxZ = 16;         // Ritz coefficients per launch and job

// x + its partner, six levels: every lane ends with the same tree sum as the
// halving tree over 64 leaves (addition commutes exactly)
__device__ __forceinline__ double wave_tree(double s) {
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w);
  return s;
}

// ---------------------------------------------------------------------------
// Short vectors: one workgroup takes a job's whole step.  v[m] stays in its
// registers from the first dot product to the normalisation, a wave sums whole
// blocks of 256, and a dot product costs one barrier.  What bounds it is the
// chain of 2 + m dependent sums; the next v[j] is on its way while a sum runs.

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / 64;

struct SmallOps {
  KrylovOp op[kMaxBatch];
};

template <int NB>
struct Vec {
  double e[NB][4];
};

// lane's elements of x: blocks wave, wave + 16, ... of 256, four per block
template <int NB>
__device__ __forceinline__ void load_vec(Vec<NB>& v, const double* __restrict__ x, int n, int wave,
                                         int lane) {
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = (q * kSmallWaves + wave) * 256 + k * 64 + lane;
      v.e[q][k] = i < n ? x[i] : 0.0;
    }
}

template <int NB>
__device__ __forceinline__ void store_vec(const Vec<NB>& v, double* __restrict__ x, int n, int wave,
                                          int lane) {
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = (q * kSmallWaves + wave) * 256 + k * 64 + lane;
      if (i < n) x[i] = v.e[q][k];
    }
}

// sh: two buffers of NB * 16 block sums, taken in turn (a wave is at most one
// barrier ahead of another, so it never writes what another still reads)
template <int NB>
__device__ __forceinline__ double dot_vec(const Vec<NB>& x, const Vec<NB>& y, double* sh, int& buf,
                                          int wave, int lane) {
  double* p = sh + buf * NB * kSmallWaves;
  buf ^= 1;
  double t[NB];
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    double s[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] = __builtin_fma(x.e[q][k], y.e[q][k], 0.0);
    t[q] = (s[0] + s[2]) + (s[1] + s[3]);
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1)
#pragma unroll
    for (int q = 0; q < NB; ++q) t[q] += __shfl_xor(t[q], w);
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < NB; ++q) p[q * kSmallWaves + wave] = t[q];
  __syncthreads();
  constexpr int nb = NB * kSmallWaves;
  double s = lane < nb ? p[lane] : 0.0;
  if (nb > 64) s += p[lane + 64];
  return wave_tree(s);
}

template <int NB>
__device__ __forceinline__ void axpy_vec(Vec<NB>& y, const Vec<NB>& x, double a) {
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) y.e[q][k] = __builtin_fma(a, x.e[q][k], y.e[q][k]);
}

template <int NB>
__device__ __forceinline__ void scale_vec(Vec<NB>& y, double norm2) {
  const double nrm = sqrt(norm2);
  if (!(nrm > 0)) return;
  const double a = 1.0 / nrm;
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) y.e[q][k] *= a;
}

template <int NB>
__global__ __launch_bounds__(kSmallThreads) void small_step_kernel(const SmallOps ops) {
  __shared__ double sh[2 * NB * kSmallWaves];
  const KrylovOp& o = ops.op[blockIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const int n = (int)o.n;
  int buf = 0;
  Vec<NB> y, x;
  const bool head = threadIdx.x == 0;
  switch (o.kind) {
    case kKrylovNormalise: {
      load_vec(y, o.psi, n, wave, lane);
      const double b = dot_vec(y, y, sh, buf, wave, lane);
      if (head) *o.b = b;
      scale_vec(y, b);
      store_vec(y, o.base, n, wave, lane);
      break;
    }
    case kKrylovFirst:
    case kKrylovStep: {
      const int m = o.kind == kKrylovFirst ? 1 : o.m;
      double* vm = o.base + m * o.ld;
      load_vec(y, vm, n, wave, lane);
      load_vec(x, o.base + (m - 1) * o.ld, n, wave, lane);
      const double al = dot_vec(y, x, sh, buf, wave, lane);
      if (head) *o.alpha = al;
      axpy_vec(y, x, -al);
      if (o.kind == kKrylovStep) {
        load_vec(x, o.base + (m - 2) * o.ld, n, wave, lane);
        axpy_vec(y, x, -o.beta);
        load_vec(x, o.base, n, wave, lane);
        for (int j = 0; j < m; ++j) {
          // the next v[j] loads during the sum, where registers allow
          Vec<NB> nx;
          if (NB < 4 && j + 1 < m) load_vec(nx, o.base + (j + 1) * o.ld, n, wave, lane);
          const double cj = dot_vec(y, x, sh, buf, wave, lane);
          axpy_vec(y, x, -cj);
          if (j + 1 < m) {
            if (NB < 4) x = nx;
            else load_vec(x, o.base + (j + 1) * o.ld, n, wave, lane);
          }
        }
      }
      const double a = dot_vec(y, y, sh, buf, wave, lane);
      if (head) *o.a = a;
      scale_vec(y, a);
      store_vec(y, vm, n, wave, lane);
      break;
    }
    case kKrylovOverlap: {
      load_vec(y, o.base + o.m * o.ld, n, wave, lane);
      load_vec(x, o.base + (o.m - 1) * o.ld, n, wave, lane);
      const double al = dot_vec(y, x, sh, buf, wave, lane);
      if (head) *o.alpha = al;
      break;
    }
    default: {   // kKrylovCheck
      load_vec(y, o.tmp, n, wave, lane);
      load_vec(x, o.psi, n, wave, lane);
      const double a = dot_vec(y, y, sh, buf, wave, lane);
      const double b = dot_vec(y, x, sh, buf, wave, lane);
      if (head) {
        *o.a = a;
        *o.b = b;
      }
      break;
    }
  }
}

struct RitzArg {
  const double* base;
  long long ld, n;
  double* psi;
  double* a;
  int m;              // coefficients of this launch
  bool first, norm;   // start from zero; end with the normalisation
  double z[kMaxZ];
};
struct RitzArgs {
  RitzArg r[kMaxBatch];
};

template <int NB>
__global__ __launch_bounds__(kSmallThreads) void small_ritz_kernel(const RitzArgs args) {
  __shared__ double sh[2 * NB * kSmallWaves];
  const RitzArg& o = args.r[blockIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const int n = (int)o.n;
  Vec<NB> y, x;
  load_vec(y, o.psi, o.first ? 0 : n, wave, lane);
  for (int j = 0; j < o.m; ++j) {
    load_vec(x, o.base + j * o.ld, n, wave, lane);
    axpy_vec(y, x, o.z[j]);
  }
  if (o.norm) {
    int buf = 0;
    const double a = dot_vec(y, y, sh, buf, wave, lane);
    if (threadIdx.x == 0) *o.a = a;
    scale_vec(y, a);
  }
  store_vec(y, o.psi, n, wave, lane);
}

// ---------------------------------------------------------------------------
// Long vectors: one launch per dependent sum.  Each stage finishes the sum of
// the stage before (every wave adds up the 512 block sums for itself), applies
// its coefficient to y and takes the block sums of the next product while y
// passes through, so y is read and written once per sum, and no launch is
// spent on a final reduction.

struct Stage {
  double* y;
  const double* src;    // the value of y comes from here (y itself unless normalising psi into v0)
  const double* u;      // y -= <previous sum> u
  const double* v2;     // then y += a2 v2
  const double* dv;     // then block sums of y * dv (y * y where dv == y)
  double* slot;         // the previous sum, for the host
  double a2;
  long long n;
  int part;             // which set of block sums
  int scale;            // y /= sqrt(previous sum)
};
struct Stages {
  Stage s[kMaxBatch];
};

__device__ __forceinline__ int dot_blocks(long long n) {
  const long long b = (n + kThreads - 1) / kThreads;
  return b < kDotBlocks ? (int)b : kDotBlocks;
}

// the tree over 512 block sums, in every wave for itself
__device__ __forceinline__ double sum_partials(const double* __restrict__ p, int nb, int lane) {
  double s[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) s[k] = lane + 64 * k < nb ? p[lane + 64 * k] : 0.0;
#pragma unroll
  for (int k = 0; k < 4; ++k) s[k] += s[k + 4];
  return wave_tree((s[0] + s[2]) + (s[1] + s[3]));
}

__device__ __forceinline__ void block_sum(double s, double* sh, double* __restrict__ out) {
  sh[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < 64) {
    const int l = threadIdx.x;
    const double t = wave_tree((sh[l] + sh[l + 128]) + (sh[l + 64] + sh[l + 192]));
    if (l == 0) out[blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kThreads) void stage_kernel(const Stages st,
                                                         const double* __restrict__ prev,
                                                         double* __restrict__ next) {
  __shared__ double sh[kThreads];
  const Stage& s = st.s[blockIdx.y];
  const int nb = dot_blocks(s.n);
  if ((int)blockIdx.x >= nb) return;
  double c = 0.0;
  if (s.slot || s.u || s.scale) {
    c = sum_partials(prev + (long long)s.part * kDotBlocks, nb, (int)threadIdx.x & 63);
    if (s.slot && blockIdx.x == 0 && threadIdx.x == 0) *s.slot = c;
  }
  const long long stride = (long long)kDotBlocks * kThreads;
  long long i = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (s.scale) {
    const double nrm = sqrt(c);
    const double a = nrm > 0 ? 1.0 / nrm : 1.0;
#pragma unroll 4
    for (; i < s.n; i += stride) s.y[i] = s.src[i] * a;
    return;
  }
  if (!s.dv) return;
  const bool self = s.dv == s.y;
  double acc = 0.0;
#pragma unroll 4
  for (; i < s.n; i += stride) {
    double y = s.src[i];
    if (s.u) {
      y = __builtin_fma(-c, s.u[i], y);
      if (s.v2) y = __builtin_fma(s.a2, s.v2[i], y);
      s.y[i] = y;
    }
    acc = __builtin_fma(y, self ? y : s.dv[i], acc);
  }
  block_sum(acc, sh, next + (long long)s.part * kDotBlocks);
}

__global__ __launch_bounds__(kThreads) void ritz_kernel(const RitzArgs args,
                                                        double* __restrict__ next) {
  __shared__ double sh[kThreads];
  const RitzArg& o = args.r[blockIdx.y];
  if ((int)blockIdx.x >= dot_blocks(o.n)) return;
  const long long stride = (long long)kDotBlocks * kThreads;
  double acc = 0.0;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < o.n; i += stride) {
    double y = o.first ? 0.0 : o.psi[i];
    for (int j = 0; j < o.m; ++j) y = __builtin_fma(o.z[j], o.base[j * o.ld + i], y);
    o.psi[i] = y;
    acc = __builtin_fma(y, y, acc);
  }
  if (o.norm) block_sum(acc, sh, next + (long long)blockIdx.y * kDotBlocks);
}

// ---------------------------------------------------------------------------

// Longest vector that one workgroup takes whole (16 registers a lane for v[m],
// 16 for v[j]).  A step with m = 4 takes 6.7 us on average up to here; in
// stages it is nine launches of 4 us.  Whole runs: a 6x4 lattice up to d = 924
// 311 ms against 319 with the line at 4096 and 318 with every vector in
// stages; with a launch per dot product, axpy and scaling it took 341, and
// eight small jobs 429 against 341.
constexpr long long kSmallMax = 16384;

// the number of 256-blocks per wave of the one-workgroup kernels
int small_nb(long long n) {
  if (n <= 4096) return 1;
  if (n <= 8192) return 2;
  return 4;
}

unsigned stage_grid(long long n) {
  const long long b = (n + kThreads - 1) / kThreads;
  return (unsigned)std::max(1LL, std::min<long long>(b, kDotBlocks));
}

// the stages of one operation, as parallel entries per launch
std::vector<std::vector<Stage>> stages(const KrylovOp& o) {
  std::vector<std::vector<Stage>> out;
  auto v = [&](int k) { return o.base + k * o.ld; };
  auto add = [&](double* y, const double* u, const double* dv, double* slot) -> Stage& {
    Stage s{};
    s.y = y;
    s.src = y;
    s.u = u;
    s.dv = dv;
    s.slot = slot;
    s.n = o.n;
    out.push_back({s});
    return out.back()[0];
  };
  auto second = [&](double* y, const double* dv, double* slot) {
    Stage s = out.back()[0];
    s.y = y;
    s.src = y;
    s.dv = dv;
    s.slot = slot;
    out.back().push_back(s);
  };
  switch (o.kind) {
    case kKrylovNormalise: {
      add(o.psi, nullptr, o.psi, nullptr);
      Stage& s = add(v(0), nullptr, nullptr, o.b);
      s.src = o.psi;
      s.scale = 1;
      break;
    }
    case kKrylovFirst:
      add(v(1), nullptr, v(0), nullptr);
      add(v(1), v(0), v(1), o.alpha);
      add(v(1), nullptr, nullptr, o.a).scale = 1;
      break;
    case kKrylovStep: {
      double* y = v(o.m);
      add(y, nullptr, v(o.m - 1), nullptr);
      Stage& s = add(y, v(o.m - 1), v(0), o.alpha);
      s.v2 = v(o.m - 2);
      s.a2 = -o.beta;
      for (int j = 1; j < o.m; ++j) add(y, v(j - 1), v(j), nullptr);
      add(y, v(o.m - 1), y, nullptr);
      add(y, nullptr, nullptr, o.a).scale = 1;
      break;
    }
    case kKrylovOverlap:
      add(v(o.m), nullptr, v(o.m - 1), nullptr);
      add(v(o.m), nullptr, nullptr, o.alpha);
      break;
    default:   // kKrylovCheck
      add(o.tmp, nullptr, o.tmp, nullptr);
      second(o.tmp, o.psi, nullptr);
      add(o.tmp, nullptr, nullptr, o.a);
      second(o.tmp, nullptr, o.b);
      break;
  }
  return out;
}

void launch_stage(Context& c, const std::vector<Stage>& st, const double* prev, double* next) {
  for (size_t i0 = 0; i0 < st.size(); i0 += kMaxBatch) {
    const int n = (int)std::min<size_t>(kMaxBatch, st.size() - i0);
    Stages arg{};
    long long longest = 1;
    bool vectors = false;
    for (int i = 0; i < n; ++i) {
      arg.s[i] = st[i0 + i];
      longest = std::max(longest, st[i0 + i].n);
      vectors = vectors || st[i0 + i].scale || st[i0 + i].dv;
    }
    // a stage that only reads sums back needs one workgroup
    hipLaunchKernelGGL(stage_kernel, dim3(vectors ? stage_grid(longest) : 1, n), dim3(kThreads), 0,
                       c.stream(), arg, prev, next);
    SU2_HIP(hipGetLastError());
  }
}

}  // namespace

long long krylov_partials(int jobs) { return 2LL * 2 * jobs * kDotBlocks; }

void krylov_run(Context& c, const std::vector<KrylovOp>& ops, double* part) {
  // one workgroup per short job
  for (int nb = 1; nb <= 4; nb *= 2) {
    SmallOps arg{};
    int n = 0;
    auto flush = [&] {
      if (n == 0) return;
      const auto fn = nb == 1 ? small_step_kernel<1>
                      : nb == 2 ? small_step_kernel<2> : small_step_kernel<4>;
      hipLaunchKernelGGL(fn, dim3(n), dim3(kSmallThreads), 0, c.stream(), arg);
      SU2_HIP(hipGetLastError());
      n = 0;
    };
    for (auto& o : ops) {
      if (o.n > kSmallMax || small_nb(o.n) != nb) continue;
      arg.op[n++] = o;
      if (n == kMaxBatch) flush();
    }
    flush();
  }
  // stage by stage over the long jobs
  std::vector<std::vector<std::vector<Stage>>> progs;
  size_t depth = 0;
  for (auto& o : ops) {
    if (o.n <= kSmallMax) continue;
    progs.push_back(stages(o));
    depth = std::max(depth, progs.back().size());
  }
  const long long half = 2LL * (long long)ops.size() * kDotBlocks;
  for (size_t d = 0; d < depth; ++d) {
    std::vector<Stage> st;
    for (size_t j = 0; j < progs.size(); ++j) {
      if (d >= progs[j].size()) continue;
      for (size_t e = 0; e < progs[j][d].size(); ++e) {
        Stage s = progs[j][d][e];
        s.part = (int)(2 * j + e);
        st.push_back(s);
      }
    }
    // the sums of stage d go to the half that stage d + 1 reads
    launch_stage(c, st, part + ((d + 1) & 1) * half, part + (d & 1) * half);
  }
}

void krylov_ritz(Context& c, const std::vector<KrylovRitz>& jobs, double* part) {
  for (int nb = 0; nb <= 4; nb = nb == 0 ? 1 : nb * 2) {   // 0: long vectors
    for (size_t i0 = 0; i0 < jobs.size();) {
      std::vector<const KrylovRitz*> grp;
      for (; i0 < jobs.size() && grp.size() < (size_t)kMaxBatch; ++i0) {
        const KrylovRitz& r = jobs[i0];
        if ((r.n > kSmallMax ? 0 : small_nb(r.n)) == nb) grp.push_back(&r);
      }
      if (grp.empty()) continue;
      size_t mmax = 0;
      long long longest = 1;
      for (auto r : grp) {
        mmax = std::max(mmax, r->z.size());
        longest = std::max(longest, r->n);
      }
      for (size_t j0 = 0; j0 < mmax; j0 += kMaxZ) {
        RitzArgs arg{};
        std::vector<Stage> fin;
        int n = 0;
        for (auto r : grp) {
          if (j0 >= r->z.size()) continue;
          RitzArg& a = arg.r[n];
          a.m = (int)std::min<size_t>(kMaxZ, r->z.size() - j0);
          a.base = r->base + (long long)j0 * r->ld;
          a.ld = r->ld;
          a.n = r->n;
          a.psi = r->psi;
          a.a = r->a;
          a.first = j0 == 0;
          a.norm = r->normalise && j0 + kMaxZ >= r->z.size();
          for (int j = 0; j < a.m; ++j) a.z[j] = r->z[j0 + j];
          if (a.norm) {
            Stage s{};
            s.y = r->psi;
            s.src = r->psi;
            s.slot = r->a;
            s.n = r->n;
            s.part = n;
            s.scale = 1;
            fin.push_back(s);
          }
          ++n;
        }
        if (nb == 0) {
          hipLaunchKernelGGL(ritz_kernel, dim3(stage_grid(longest), n), dim3(kThreads), 0,
                             c.stream(), arg, part);
          SU2_HIP(hipGetLastError());
          if (!fin.empty()) launch_stage(c, fin, part, nullptr);
        } else {
          const auto fn = nb == 1 ? small_ritz_kernel<1>
                          : nb == 2 ? small_ritz_kernel<2> : small_ritz_kernel<4>;
          hipLaunchKernelGGL(fn, dim3(n), dim3(kSmallThreads), 0, c.stream(), arg);
          SU2_HIP(hipGetLastError());
        }
      }
    }
  }
}

}  // namespace su2
