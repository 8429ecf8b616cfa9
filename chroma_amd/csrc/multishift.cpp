// Multishift CG (MInvCG2_a, minvcg2.cc:72-355; MdagMMultiSysSolverCG, multi_syssolver_mdagm_cg.h:58-100):
// (M^dag M + shifts[s]) psi[s] = chi for every shift with one Krylov space (Jegerlehner,
// hep-lat/9708029), in FP64 on the device.  Vectors and the shifted recurrences (z, bs, as) live there, so
// an iteration is nine launches with no host value between them; the host polls the stop flag every few
// iterations (two read-backs and three coefficient copies per iteration when the recurrences ran on the
// host left the device idle for 50 to 70 us of each 0.4 ms at 16^3x32).
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <vector>

#include "multishift.h"
#include "op.h"

namespace cmx {

namespace {

constexpr int MS_A = S_KRY;        // a, b of the p0 and r updates
constexpr int MS_B = S_KRY + 1;
constexpr int MS_C = S_KRY + 2;    // |chi|^2
constexpr int MS_SIG = S_KRY + 8;  // the shifts, for the residual checks
constexpr int MS_RES = MS_SIG + MS_MAX;  // |chi - (M^dag M + shift_s) psi_s|^2
static_assert(MS_RES + MS_MAX <= S_MR, "multishift slots overlap the MR slots");

}  // namespace

void solve_multishift(Op& op, const cmx_solver_params& p, int ns, const double* shifts, const double* rsd,
                      double* psi_h, const double* chi_h, cmx_solver_result* res) {
  CMX_REQUIRE(ns >= 1 && ns <= MS_MAX, CMX_ERR_ARG, "solve_multishift: 1.." + std::to_string(MS_MAX) + " shifts");
  CMX_REQUIRE(p.max_iter > 0, CMX_ERR_ARG, "solve_multishift: MaxIter must be positive");
  for (int s = 0; s < ns; ++s)
    CMX_REQUIRE(rsd[s] > 0 && std::isfinite(shifts[s]), CMX_ERR_ARG, "solve_multishift: bad shift or RsdCG");
  const auto t0 = std::chrono::steady_clock::now();
  const int n = op.subset_sites();
  const int nb = blas_blocks(n);
  Vec &chi = op.work(1, P64, n), &r = op.work(11, P64, n), &p0 = op.work(12, P64, n), &mp = op.work(13, P64, n),
      &mmp = op.work(14, P64, n);
  // p_s and psi_s of all shifts in one allocation
  const size_t vb = spinor_bytes(P64, n);
  DevScratch vecs(2 * vb * ns), state(sizeof(MsState));
  auto psi_of = [&](int s) {
    Vec v;
    v.prec = P64;
    v.n = n;
    v.buf.p = vecs.as<char>() + vb * (ns + s);
    v.buf.bytes = vb;
    v.buf.own = false;
    return v;
  };
  op.pack(chi_h, n, chi);
  hipEvent_t e0, e1;
  CMX_HIP(hipEventCreate(&e0));
  CMX_HIP(hipEventCreate(&e1));
  struct EvGuard {
    hipEvent_t a, b;
    ~EvGuard() {
      (void)hipEventDestroy(a);
      (void)hipEventDestroy(b);
    }
  } evg{e0, e1};
  CMX_HIP(hipEventRecord(e0, op.stream));

  // isz: the smallest shift decides the first convergence test (:99-104, :247)
  int isz = 0;
  for (int s = 1; s < ns; ++s)
    if (shifts[s] < shifts[isz]) isz = s;
  MsLaunch L;
  std::memset(&L, 0, sizeof(L));
  L.ne = 12L * n;
  L.ns = ns;
  L.isz = isz;
  L.max_iter = p.max_iter;
  L.st = state.as<MsState>();
  L.S = op.state_S.as<double>();
  L.F = op.state_F.as<int>();
  L.slot_a = MS_A;
  L.slot_b = MS_B;
  L.partials = op.partials.as<double>();
  L.r = r.buf.as<double2>();
  L.p0 = p0.buf.as<double2>();
  L.p = vecs.as<double2>();
  L.psi = vecs.as<double2>() + L.ne * ns;
  ms_init(L, chi.buf.as<double2>(), op.stream);  // r = p0 = p_s = chi, psi_s = 0 (:118-121, :161-175)
  op.blas(B_NORM2, {&chi});
  op.finalize(nb, 1, PG_STORE, MS_C);
  CMX_HIP(hipMemcpyAsync(op.hS + MS_C, static_cast<double*>(op.state_S.p) + MS_C, sizeof(double),
                         hipMemcpyDeviceToHost, op.stream));
  op.sync();
  const double chi_norm_sq = op.hS[MS_C];
  int n_count = 0;
  if (std::sqrt(chi_norm_sq) >= 1e-10) {  // a zero source returns the zero solutions (:133-153)
    MsState h;
    std::memset(&h, 0, sizeof(h));
    h.cp = chi_norm_sq;
    for (int s = 0; s < ns; ++s) h.sigma[s] = shifts[s], h.rsd_sq[s] = chi_norm_sq * rsd[s] * rsd[s];
    CMX_HIP(hipMemcpy(state.get(), &h, sizeof(h), hipMemcpyHostToDevice));
    std::memset(op.hF, 0, sizeof(int) * F_NFLAGS);
    CMX_HIP(hipMemcpyAsync(op.state_F.p, op.hF, sizeof(int) * F_NFLAGS, hipMemcpyHostToDevice, op.stream));
    op.sync();
    int* F = op.state_F.as<int>();
    // b = -|r|^2 / |M p0|^2 ; r += b M^dag M p0 ; c = |r|^2 and the recurrences (:179-217, :275-339)
    auto step = [&](int phase) {
      L.nb = op.apply(P64, mp.view(), p0.view(), +1, op.partials.as<double>(), F + F_DONE);
      ms_scalars(L, 1, op.stream);
      L.nb = op.apply(P64, r.view(), mp.view(), -1, op.partials.as<double>(), F + F_DONE, nullptr,
                      {TAIL_UPDATE, &r, op.state_S.as<double>() + MS_B});
      ms_scalars(L, phase, op.stream);
    };
    auto poll = [&]() {
      CMX_HIP(hipMemcpyAsync(op.hF, op.state_F.p, sizeof(int) * F_NFLAGS, hipMemcpyDeviceToHost, op.stream));
      if (p.verbose) CMX_HIP(hipMemcpyAsync(&h.c, &L.st->c, sizeof(double), hipMemcpyDeviceToHost, op.stream));
      op.sync();
      CMX_REQUIRE(op.hF[F_ERR] != CMX_ERR_BREAKDOWN, CMX_ERR_BREAKDOWN, "multishift CG: |M p| = 0 or not finite");
      return op.hF[F_CONV] != 0;
    };
    step(0);
    const int batch = p.verbose ? 1 : 6;
    for (long k = 0; !poll() && k <= (long)p.max_iter + batch; k += batch) {
      if (p.verbose && k > 0) std::printf("MInvCG2: k = %ld |r| = %g\n", k, std::sqrt(h.c));
      for (int j = 0; j < batch; ++j) {
        ms_update(L, op.stream);  // p0 = r + a p0 ; psi_s -= bs_s p_s ; p_s = z_s r + as_s p_s (:253-273, :312-322)
        step(2);
      }
    }
    n_count = op.hF[F_NCOUNT];
    if (p.verbose && n_count > 0) std::printf("MInvCG2: k = %d |r| = %g\n", n_count, std::sqrt(h.c));
    ms_finish(L, op.stream);
  }
  CMX_HIP(hipEventRecord(e1, op.stream));
  CMX_HIP(hipEventSynchronize(e1));
  float ms = 0;
  CMX_HIP(hipEventElapsedTime(&ms, e0, e1));
  // FP64 residual of every shifted system: |chi - (M^dag M + shift_s) psi_s|
  std::memcpy(op.hS + MS_SIG, shifts, sizeof(double) * ns);
  CMX_HIP(hipMemcpyAsync(static_cast<double*>(op.state_S.p) + MS_SIG, op.hS + MS_SIG, sizeof(double) * ns,
                         hipMemcpyHostToDevice, op.stream));
  for (int s = 0; s < ns; ++s) {
    const Vec x = psi_of(s);
    op.apply(P64, mp.view(), x.view(), +1, nullptr);
    op.apply(P64, mmp.view(), mp.view(), -1, nullptr);
    op.blas(B_AXPY, {&mmp, &x}, MS_SIG + s);
    op.blas(B_XMY_NORM, {&r, &chi, &mmp});
    op.finalize(nb, 1, PG_STORE, MS_RES + s);
  }
  CMX_HIP(hipMemcpyAsync(op.hS + MS_RES, static_cast<double*>(op.state_S.p) + MS_RES, sizeof(double) * ns,
                         hipMemcpyDeviceToHost, op.stream));
  op.sync();
  for (int s = 0; s < ns; ++s) {
    cmx_solver_result& q = res[s];
    std::memset(&q, 0, sizeof(q));
    q.n_count = n_count;
    q.resid = std::sqrt(op.hS[MS_RES + s]);
    q.rel_resid = chi_norm_sq > 0 ? q.resid / std::sqrt(chi_norm_sq) : q.resid;
    q.solve_seconds = ms * 1e-3;
    op.unpack(psi_h + (size_t)s * 24 * n, n, psi_of(s));
  }
  const double wall = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  for (int s = 0; s < ns; ++s) res[s].total_seconds = wall;
  if (n_count >= p.max_iter)  // QDP_error_exit("too many CG iterations") (:357-359)
    throw Error(CMX_ERR_NOCONV, "multishift CG: no convergence in " + std::to_string(p.max_iter) + " iterations");
}

}  // namespace cmx
