#include "lanczos.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>

#include "common.hpp"
#include "context.hpp"
#include "krylov.hpp"

namespace su2 {

void tridiag_eig(const std::vector<double>& d, const std::vector<double>& e,
                 std::vector<double>& w, std::vector<double>& z) {
  // cyclic Jacobi on the dense m x m matrix: m is at most the Krylov size
  const int m = (int)d.size();
  std::vector<double> a((size_t)m * m, 0.0);
  for (int i = 0; i < m; ++i) {
    a[i + (size_t)m * i] = d[i];
    if (i + 1 < m) {
      a[i + (size_t)m * (i + 1)] = e[i];
      a[i + 1 + (size_t)m * i] = e[i];
    }
  }
  z.assign((size_t)m * m, 0.0);
  for (int i = 0; i < m; ++i) z[i + (size_t)m * i] = 1.0;
  auto A = [&](int r, int c) -> double& { return a[r + (size_t)m * c]; };
  for (int sweep = 0; sweep < 100; ++sweep) {
    double off = 0;
    for (int p = 0; p < m; ++p)
      for (int q = p + 1; q < m; ++q) off += A(p, q) * A(p, q);
    if (off < 1e-300) break;
    for (int p = 0; p < m; ++p)
      for (int q = p + 1; q < m; ++q) {
        const double apq = A(p, q);
        if (std::fabs(apq) < 1e-300) continue;
        const double tau = (A(q, q) - A(p, p)) / (2 * apq);
        const double t = (tau >= 0 ? 1.0 : -1.0) / (std::fabs(tau) + std::sqrt(1 + tau * tau));
        const double cs = 1 / std::sqrt(1 + t * t), sn = t * cs;
        for (int r = 0; r < m; ++r) {
          const double x = A(r, p), y = A(r, q);
          A(r, p) = cs * x - sn * y;
          A(r, q) = sn * x + cs * y;
        }
        for (int col = 0; col < m; ++col) {
          const double x = A(p, col), y = A(q, col);
          A(p, col) = cs * x - sn * y;
          A(q, col) = sn * x + cs * y;
        }
        for (int r = 0; r < m; ++r) {
          const double x = z[r + (size_t)m * p], y = z[r + (size_t)m * q];
          z[r + (size_t)m * p] = cs * x - sn * y;
          z[r + (size_t)m * q] = sn * x + cs * y;
        }
      }
  }
  std::vector<int> perm(m);
  std::iota(perm.begin(), perm.end(), 0);
  std::stable_sort(perm.begin(), perm.end(), [&](int x, int y) { return A(x, x) < A(y, y); });
  w.resize(m);
  std::vector<double> zs((size_t)m * m);
  for (int i = 0; i < m; ++i) {
    w[i] = A(perm[i], perm[i]);
    for (int r = 0; r < m; ++r) zs[r + (size_t)m * i] = z[r + (size_t)m * perm[i]];
  }
  z.swap(zs);
}

// One solve through the batched state machine (a batch of one), so a single
// run and a batched one execute the same operations.
LanczosResult lanczos_ground(Context& c, const ApplyFn& apply, double* psi, long long n, int mlanc,
                             double tol, const ApplyFn* check_apply) {
  std::vector<LanczosJob> jobs(1);
  jobs[0].psi = psi;
  jobs[0].n = n;
  jobs[0].mlanc = mlanc;
  jobs[0].tol = tol;
  jobs[0].mixed = check_apply != nullptr;
  lanczos_batch(c, jobs, [&](const std::vector<LanczosReq>& reqs) {
    for (auto& r : reqs) (r.check && check_apply ? *check_apply : apply)(r.x, r.y);
  });
  return jobs[0].res;
}

// lanczos_batch: lanczos_ground's schedule as a state machine per job

namespace {

enum LzState { kStart, kAfterFirst, kM2Final, kLoop, kCheckCont, kCheckDone, kFinal, kDone };

struct LzJob {
  LanczosJob* job;
  int st = kStart;
  int m = 0;
  DevBuf ff;                // Krylov vectors 0..mlanc, ld apart
  long long ld = 0;
  DevBuf tmp;
  std::vector<double> aal, nnl;
  double* slots = nullptr;  // alpha, a, b (pinned)
  bool pending = false;     // has a matvec request this round
  const double* x = nullptr;
  double* y = nullptr;
  bool check = false;
  double* v(int k) const { return ff.p + k * ld; }
};

}  // namespace

void lanczos_batch(Context& c, std::vector<LanczosJob>& jobs, const BatchApply& apply) {
  const int nj = (int)jobs.size();
  if (nj == 0) return;
  // alpha, a and b of every job, written by the device into pinned memory (the
  // applies below leave the context's host scratch alone)
  double* host = c.host_scratch(3 * (size_t)nj);
  DevBuf part(c, krylov_partials(nj));
  std::vector<LzJob> L(nj);
  for (int i = 0; i < nj; ++i) {
    LzJob& s = L[i];
    s.job = &jobs[i];
    SU2_CHECK(s.job->mlanc >= 2, kErrArgument, "lanczos: mlanc=%d", s.job->mlanc);
    s.job->res = LanczosResult();
    const long long n = std::max<long long>(s.job->n, 1);
    s.ld = (n + 31) / 32 * 32;
    s.ff = DevBuf(c, s.ld * (s.job->mlanc + 1));
    s.tmp = DevBuf(c, n);
    s.aal.assign(s.job->mlanc, 0.0);
    s.nnl.assign(s.job->mlanc + 1, 0.0);
    s.slots = host + 3 * i;
  }
  auto request = [&](LzJob& s, const double* x, double* y, bool check) {
    s.pending = true;
    s.x = x;
    s.y = y;
    s.check = check;
    ++s.job->res.matvecs;
    if (check && s.job->mixed) ++s.job->res.check_matvecs;
  };
  // Ritz vector of the m x m tridiagonal into psi, then psi normalised on
  // the device (the check's normalisation, lanczos_su2.cpp:320-332); the
  // jobs of a round are queued together
  std::vector<KrylovRitz> ritzes;
  auto ritz = [&](LzJob& s, int m, bool normalise) {
    std::vector<double> d(s.aal.begin(), s.aal.begin() + m), e(s.nnl.begin() + 1, s.nnl.begin() + m),
        w, z;
    tridiag_eig(d, e, w, z);
    z.resize(m);
    if (z[0] < 0)   // Ritz vector with a positive overlap on the start vector
      for (int j = 0; j < m; ++j) z[j] = -z[j];
    ritzes.push_back(KrylovRitz{s.ff.p, s.ld, s.job->n, s.job->psi, z, normalise, s.slots + 1});
    s.job->res.ritz = s.job->res.energy = w[0];
  };
  auto check_request = [&](LzJob& s, int st) {
    ritz(s, s.m, true);
    request(s, s.job->psi, s.tmp.p, true);
    s.st = st;
  };
  // after iteration m: the next Krylov matvec, or the last one
  auto advance = [&](LzJob& s) {
    ++s.m;
    request(s, s.v(s.m - 1), s.v(s.m), false);
    s.st = s.m < s.job->mlanc ? kLoop : kFinal;
  };
  std::vector<KrylovOp> ops;
  auto queue = [&](LzJob& s, int kind, int m, double beta) {
    ops.push_back(KrylovOp{kind, m, s.ff.p, s.ld, s.job->n, s.job->psi, s.tmp.p, beta, s.slots,
                           s.slots + 1, s.slots + 2});
  };

  // start: v[0] = psi / |psi| (initialize_lanczos, lanczos_su2.cpp:36-47)
  for (auto& s : L) {
    queue(s, kKrylovNormalise, 0, 0.0);
    request(s, s.v(0), s.v(1), false);
    s.st = kAfterFirst;
  }
  krylov_run(c, ops, part.p);
  bool first = true;
  for (;;) {
    std::vector<LanczosReq> reqs;
    for (int i = 0; i < nj; ++i)
      if (L[i].pending) reqs.push_back(LanczosReq{i, L[i].x, L[i].y, L[i].check});
    if (reqs.empty()) break;
    apply(reqs);
    // each job's vector algebra after its matvec, scalars into its slots
    ops.clear();
    for (auto& s : L) {
      if (!s.pending) continue;
      s.pending = false;
      switch (s.st) {
        case kAfterFirst: queue(s, kKrylovFirst, 1, 0.0); break;
        case kM2Final: queue(s, kKrylovOverlap, 2, 0.0); break;
        case kLoop: queue(s, kKrylovStep, s.m, s.nnl[s.m - 1]); break;
        case kCheckCont:
        case kCheckDone: queue(s, kKrylovCheck, 0, 0.0); break;
        case kFinal: queue(s, kKrylovOverlap, s.job->mlanc, 0.0); break;
        default: break;
      }
    }
    krylov_run(c, ops, part.p);
    // one wait for the scalars of every job
    SU2_HIP(hipStreamSynchronize(c.stream()));
    for (auto& s : L) {
      if (s.st == kDone || s.pending) continue;
      const int mlanc = s.job->mlanc;
      const double alpha = s.slots[0], a = s.slots[1], b = s.slots[2];
      switch (s.st) {
        case kAfterFirst: {
          if (first) SU2_CHECK(b > 0, kErrNumeric, "lanczos: zero start vector");
          s.aal[0] = alpha;
          // an exactly invariant start vector (a 1-dim H_eff) leaves nnl = 0:
          // the unnormalised residual is then never read again
          s.nnl[1] = std::sqrt(a);
          if (mlanc == 2) {
            if (s.nnl[1] < s.job->tol) {
              ritz(s, 1, false);
              s.st = kDone;
            } else {
              request(s, s.v(1), s.v(2), false);
              s.st = kM2Final;
            }
          } else {
            s.m = 2;
            request(s, s.v(1), s.v(2), false);
            s.st = kLoop;
          }
          break;
        }
        case kM2Final:
          s.aal[1] = alpha;
          ritz(s, 2, true);
          s.st = kDone;
          break;
        case kLoop: {
          const int m = s.m;
          s.aal[m - 1] = alpha;
          s.nnl[m] = std::sqrt(a);
          if (s.nnl[m] < s.job->tol) check_request(s, kCheckDone);
          else if (m % 4 == 0) check_request(s, kCheckCont);
          else advance(s);
          break;
        }
        case kCheckCont:
        case kCheckDone: {
          const double prod = std::sqrt(a), rq = b;
          s.job->res.residual = std::sqrt(std::max(0.0, prod * prod - rq * rq));
          if (s.job->mixed) s.job->res.energy = rq;
          const double ov = std::fabs(rq / prod);
          if (s.st == kCheckDone || std::fabs(ov - 1.0) < 1e-8) s.st = kDone;
          else advance(s);
          break;
        }
        case kFinal:
          s.aal[mlanc - 1] = alpha;
          s.m = mlanc;
          check_request(s, kCheckDone);
          break;
        default:
          break;
      }
    }
    krylov_ritz(c, ritzes, part.p);
    ritzes.clear();
    first = false;
  }
  SU2_HIP(hipStreamSynchronize(c.stream()));
}

}  // namespace su2
