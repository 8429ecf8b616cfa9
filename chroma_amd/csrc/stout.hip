// Stout smearing on the device, in FP64: Stouting::smear_links (stout_utils.cc:936-962) with the
// parameters of StoutLinkSmearing (stout_link_smearing.cc:62-120): a set of smeared directions and
// rho(mu,nu) = rho for mu != nu both smeared, else 0.  Links of an unsmeared direction are copied, and
// only smeared directions contribute staples; the staple sum C and Q of getQsandCs (:105-180):
//   C_mu(x) = rho sum_{nu != mu} [ U_nu(x) U_mu(x+nu) U_nu^dag(x+mu) + U_nu^dag(x-nu) U_mu(x-nu) U_nu(x-nu+mu) ],
//   Omega = C U_mu^dag(x),  Q = (i/2) [ (Omega^dag - Omega) - tr(Omega^dag - Omega)/3 ],  U'_mu(x) = exp(iQ) U_mu(x).
// The reference evaluates exp(iQ) in closed form from the eigenvalues (getFsAndBs, :383-874); here it is a
// Taylor polynomial with scaling and squaring (Moler & Van Loan, "Nineteen dubious ways to compute the
// exponential of a matrix", method 3), reduced by Cayley-Hamilton to a combination of 1, Q and Q^2: exact to
// rounding with no small-eigenvalue special case.  The
// product is re-projected onto SU(3) (rows 0 and 1 orthonormalised, row 2 = conj(row0 x row1)), which
// moves it only at rounding level and keeps many steps from drifting off the group.
//
// Layout: the host gauge layout ([mu][site][3][3] complex, sites checkerboard-major, x fastest within a
// checkerboard) is transposed on the device into [mu][element][site], so that each of a lane's loads and
// stores is one 16 B element and a wave's 64 lanes touch 1 KiB of consecutive sites; the steps run in
// that layout and the result is transposed back.  One lane per (mu, site).  A step is bound by link traffic:
// each link is read by 13 lanes (its own, and as a staple leg of 12 others), 11.5 GB per step at 32^4 where the
// field has 0.6.  A work-group is the four directions of 64 sites, the two checkerboards of a region follow each
// other, and each XCD owns a contiguous eighth of the lattice, so that most of these reads are L1 and L2 hits.
// Per step, 16^3x32 and 32^4: one direction after another over the whole lattice 175 and 1610 us; this order
// 130 and 1000 us; with exp(iQ) from scalars instead of 14 matrix products 85 and 820 us.  A third wave per SIMD
// (168 instead of 210 registers) spills and loses: 166 and 1775 us in the first order.
#include <cmath>
#include <cstring>
#include <string>
#include <utility>

#include "op.h"

namespace cmx {

namespace {

struct M3 {
  double2 e[9];
};

__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {  // c + a b
  return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ double2 cfmac(double2 a, double2 b, double2 c) {  // c + a conj(b)
  return make_double2(fma(a.x, b.x, fma(a.y, b.y, c.x)), fma(a.y, b.x, fma(-a.x, b.y, c.y)));
}
__device__ __forceinline__ double2 cfmca(double2 a, double2 b, double2 c) {  // c + conj(a) b
  return make_double2(fma(a.x, b.x, fma(a.y, b.y, c.x)), fma(a.x, b.y, fma(-a.y, b.x, c.y)));
}

__device__ __forceinline__ M3 mul(const M3& a, const M3& b) {  // a b
  M3 c;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double2 t = make_double2(0, 0);
#pragma unroll
      for (int k = 0; k < 3; ++k) t = cfma(a.e[3 * i + k], b.e[3 * k + j], t);
      c.e[3 * i + j] = t;
    }
  return c;
}
__device__ __forceinline__ M3 mul_nd(const M3& a, const M3& b) {  // a b^dag
  M3 c;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double2 t = make_double2(0, 0);
#pragma unroll
      for (int k = 0; k < 3; ++k) t = cfmac(a.e[3 * i + k], b.e[3 * j + k], t);
      c.e[3 * i + j] = t;
    }
  return c;
}
// acc += a b c^dag and acc += a^dag b c, row by row: one row of the product a b is live at a time
__device__ __forceinline__ void add_abcd(M3& acc, const M3& a, const M3& b, const M3& c) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double2 t[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      t[j] = make_double2(0, 0);
#pragma unroll
      for (int k = 0; k < 3; ++k) t[j] = cfma(a.e[3 * i + k], b.e[3 * k + j], t[j]);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int k = 0; k < 3; ++k) acc.e[3 * i + j] = cfmac(t[k], c.e[3 * j + k], acc.e[3 * i + j]);
  }
}
__device__ __forceinline__ void add_adbc(M3& acc, const M3& a, const M3& b, const M3& c) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double2 t[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      t[j] = make_double2(0, 0);
#pragma unroll
      for (int k = 0; k < 3; ++k) t[j] = cfmca(a.e[3 * k + i], b.e[3 * k + j], t[j]);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int k = 0; k < 3; ++k) acc.e[3 * i + j] = cfma(t[k], c.e[3 * k + j], acc.e[3 * i + j]);
  }
}

struct StoutGeom {
  int L[4];
  long V, Vh;
};

__device__ __forceinline__ long site_of(const StoutGeom& g, const int (&x)[4]) {
  const int cb = (x[0] + x[1] + x[2] + x[3]) & 1;
  return cb * g.Vh + ((((long)x[3] * g.L[2] + x[2]) * g.L[1] + x[1]) * g.L[0] + x[0]) / 2;
}

// [mu][element][site] layout on the device
__device__ __forceinline__ M3 load(const double2* __restrict__ u, const StoutGeom& g, int mu, long s) {
  const double2* p = u + (size_t)mu * 9 * g.V + s;
  M3 m;
#pragma unroll
  for (int k = 0; k < 9; ++k) m.e[k] = p[(size_t)k * g.V];
  return m;
}

// host layout [mu][site][9] <-> device layout [mu][9][site], one lane per link
__global__ void __launch_bounds__(256) k_links_to_soa(long V, const double2* __restrict__ in, double2* __restrict__ out) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * V) return;
  const long mu = t / V, s = t - mu * V;
#pragma unroll
  for (int k = 0; k < 9; ++k) out[(mu * 9 + k) * V + s] = in[t * 9 + k];
}
__global__ void __launch_bounds__(256) k_links_from_soa(long V, const double2* __restrict__ in, double2* __restrict__ out) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * V) return;
  const long mu = t / V, s = t - mu * V;
#pragma unroll
  for (int k = 0; k < 9; ++k) out[t * 9 + k] = in[(mu * 9 + k) * V + s];
}

// exp(iQ) for a Hermitian traceless Q (diagonal q, upper triangle z01 z02 z12).  Q 2^-s with |Q 2^-s|_F <= 1,
// the degree-18 Taylor polynomial (truncation below 1e-17), then s squarings.  By Cayley-Hamilton
// Q^3 = c1 Q + c0 with c1 = tr Q^2 / 2 and c0 = det Q, so that Q^n = a + b Q + d Q^2 with real a, b, d that
// follow from those of Q^(n-1), and the polynomial costs one matrix square and scalar arithmetic (as a Horner
// scheme on matrices, degree 14 below norm 1/4, it was 14 to 16 of the 28 matrix products of a link).
__device__ M3 exp_i(const double (&q)[3], double2 z01, double2 z02, double2 z12) {
  auto sq = [](double2 z) { return fma(z.x, z.x, z.y * z.y); };
  double nrm = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + 2.0 * (sq(z01) + sq(z02) + sq(z12)));
  int s = 0;
  while (nrm > 1.0 && s < 60) {
    nrm *= 0.5;
    ++s;
  }
  const double sc = ldexp(1.0, -s);
  const double q0 = q[0] * sc, q1 = q[1] * sc, q2 = q[2] * sc;
  z01.x *= sc, z01.y *= sc, z02.x *= sc, z02.y *= sc, z12.x *= sc, z12.y *= sc;
  const double n01 = sq(z01), n02 = sq(z02), n12 = sq(z12);
  const double s0 = fma(q0, q0, n01 + n02), s1 = fma(q1, q1, n01 + n12), s2 = fma(q2, q2, n02 + n12);  // diag Q^2
  const double c1 = 0.5 * (s0 + s1 + s2);
  const double2 zz = cfma(z01, z12, make_double2(0, 0));
  const double c0 = q0 * q1 * q2 + 2.0 * fma(zz.x, z02.x, zz.y * z02.y) - q0 * n12 - q1 * n02 - q2 * n01;
  // f = sum i^n (a_n, b_n, d_n) / n! over n > 0; the 1 of n = 0 is added last, so that it is rounded once
  double a = 1, b = 0, d = 0, fr[3] = {0, 0, 0}, fi[3] = {0, 0, 0};
#pragma unroll
  for (int n = 1; n <= 18; ++n) {
    const double r = 1.0 / n, d0 = d * r;
    d = b * r;
    b = fma(c1, d0, a * r);
    a = c0 * d0;
    const double sg = (n >> 1) & 1 ? -1.0 : 1.0;
    double(&f)[3] = n & 1 ? fi : fr;
    f[0] = fma(sg, a, f[0]);
    f[1] = fma(sg, b, f[1]);
    f[2] = fma(sg, d, f[2]);
  }
  // E = 1 + f0 + f1 Q + f2 Q^2; E_ji has conj(Q_ij), conj((Q^2)_ij)
  M3 E;
  auto diag = [&](double x, double y) {
    return make_double2(1.0 + fma(fr[2], y, fma(fr[1], x, fr[0])), fma(fi[2], y, fma(fi[1], x, fi[0])));
  };
  auto off = [&](double2 x, double2 y) {  // f1 x + f2 y
    return make_double2(fma(fr[1], x.x, fma(-fi[1], x.y, fma(fr[2], y.x, -fi[2] * y.y))),
                        fma(fr[1], x.y, fma(fi[1], x.x, fma(fr[2], y.y, fi[2] * y.x))));
  };
  auto conj = [](double2 x) { return make_double2(x.x, -x.y); };
  const double2 w01 = cfmac(z02, z12, make_double2((q0 + q1) * z01.x, (q0 + q1) * z01.y));
  const double2 w02 = cfma(z01, z12, make_double2((q0 + q2) * z02.x, (q0 + q2) * z02.y));
  const double2 w12 = cfmca(z01, z02, make_double2((q1 + q2) * z12.x, (q1 + q2) * z12.y));
  E.e[0] = diag(q0, s0);
  E.e[4] = diag(q1, s1);
  E.e[8] = diag(q2, s2);
  E.e[1] = off(z01, w01);
  E.e[3] = off(conj(z01), conj(w01));
  E.e[2] = off(z02, w02);
  E.e[6] = off(conj(z02), conj(w02));
  E.e[5] = off(z12, w12);
  E.e[7] = off(conj(z12), conj(w12));
  for (int k = 0; k < s; ++k) E = mul(E, E);
  return E;
}

__device__ void reunit(M3& U) {
  double n0 = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) n0 += U.e[j].x * U.e[j].x + U.e[j].y * U.e[j].y;
  n0 = 1.0 / sqrt(n0);
#pragma unroll
  for (int j = 0; j < 3; ++j) U.e[j] = make_double2(U.e[j].x * n0, U.e[j].y * n0);
  double2 d = make_double2(0, 0);
#pragma unroll
  for (int j = 0; j < 3; ++j) d = cfmca(U.e[j], U.e[3 + j], d);  // <row0, row1>
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double2 p = cfma(d, U.e[j], make_double2(0, 0));
    U.e[3 + j] = make_double2(U.e[3 + j].x - p.x, U.e[3 + j].y - p.y);
  }
  double n1 = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) n1 += U.e[3 + j].x * U.e[3 + j].x + U.e[3 + j].y * U.e[3 + j].y;
  n1 = 1.0 / sqrt(n1);
#pragma unroll
  for (int j = 0; j < 3; ++j) U.e[3 + j] = make_double2(U.e[3 + j].x * n1, U.e[3 + j].y * n1);
#pragma unroll
  for (int k = 0; k < 3; ++k) {  // row2_k = conj(row0_a row1_b - row0_b row1_a)
    const int a = (k + 1) % 3, b = (k + 2) % 3;
    const double2 x = U.e[a], y = U.e[3 + b], z = U.e[b], w = U.e[3 + a];
    const double re = x.x * y.x - x.y * y.y - (z.x * w.x - z.y * w.y);
    const double im = x.x * y.y + x.y * y.x - (z.x * w.y + z.y * w.x);
    U.e[6 + k] = make_double2(re, -im);
  }
}

__global__ void __launch_bounds__(256) k_stout_step(StoutGeom g, const double2* __restrict__ cur,
                                                    double2* __restrict__ next, double rho, int dirs) {
  const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = xcd_range(blockIdx.x, gridDim.x);
  const long r0 = (long)(l >> 1) * 64 + (threadIdx.x & 63);
  if (r0 >= g.Vh) return;
  const int cb = l & 1;
  const long s = cb * g.Vh + r0;
  if (!(dirs >> mu & 1)) {  // next[mu] = current[mu]
    const double2* p = cur + (size_t)mu * 9 * g.V + s;
    double2* o = next + (size_t)mu * 9 * g.V + s;
#pragma unroll
    for (int k = 0; k < 9; ++k) o[(size_t)k * g.V] = p[(size_t)k * g.V];
    return;
  }
  int x[4];
  {
    long r = r0;
    const int Lxh = g.L[0] / 2;
    const int xh = (int)(r % Lxh);
    r /= Lxh;
    x[1] = (int)(r % g.L[1]);
    r /= g.L[1];
    x[2] = (int)(r % g.L[2]);
    x[3] = (int)(r / g.L[2]);
    x[0] = 2 * xh + ((cb + x[1] + x[2] + x[3]) & 1);
  }
  M3 C;
#pragma unroll
  for (int k = 0; k < 9; ++k) C.e[k] = make_double2(0, 0);
  for (int nu = 0; nu < 4; ++nu) {
    if (nu == mu || !(dirs >> nu & 1)) continue;
    int y[4] = {x[0], x[1], x[2], x[3]};
    y[mu] = x[mu] + 1 == g.L[mu] ? 0 : x[mu] + 1;
    const long xpm = site_of(g, y);
    y[nu] = x[nu] == 0 ? g.L[nu] - 1 : x[nu] - 1;
    const long xmnpm = site_of(g, y);
    y[mu] = x[mu];
    const long xmn = site_of(g, y);
    y[nu] = x[nu] + 1 == g.L[nu] ? 0 : x[nu] + 1;
    const long xpn = site_of(g, y);
    // forward staple U_nu(x) U_mu(x+nu) U_nu^dag(x+mu)
    add_abcd(C, load(cur, g, nu, s), load(cur, g, mu, xpn), load(cur, g, nu, xpm));
    // backward staple U_nu^dag(x-nu) U_mu(x-nu) U_nu(x-nu+mu)
    add_adbc(C, load(cur, g, nu, xmn), load(cur, g, mu, xmn), load(cur, g, nu, xmnpm));
  }
  const M3 U = load(cur, g, mu, s);
  const M3 Om = mul_nd(C, U);
  // Q = (i/2) T with T = (Omega^dag - Omega) - tr/3, Omega scaled by rho: Hermitian and traceless
  double q[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) q[i] = rho * Om.e[4 * i].y;
  const double tr = (q[0] + q[1] + q[2]) / 3.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) q[i] -= tr;
  auto up = [&](int i, int j) {  // (i/2) rho (conj(Omega_ji) - Omega_ij)
    const double2 a = Om.e[3 * j + i], c = Om.e[3 * i + j];
    return make_double2(0.5 * rho * (a.y + c.y), 0.5 * rho * (a.x - c.x));
  };
  M3 N = mul(exp_i(q, up(0, 1), up(0, 2), up(1, 2)), U);
  reunit(N);
  double2* o = next + (size_t)mu * 9 * g.V + s;
#pragma unroll
  for (int k = 0; k < 9; ++k) o[(size_t)k * g.V] = N.e[k];
}

}  // namespace

void stout_smear(const int dims[4], const double* in, double* out, int nstep, double rho, int dirs) {
  CMX_REQUIRE(dims && in && out, CMX_ERR_ARG, "gauge_stout_smear: null array");
  CMX_REQUIRE(dirs >= 0 && dirs <= 15, CMX_ERR_ARG, "gauge_stout_smear: smeared directions are a 4-bit mask");
  CMX_REQUIRE(nstep >= 0, CMX_ERR_ARG, "gauge_stout_smear: nstep must be >= 0");
  CMX_REQUIRE(std::isfinite(rho), CMX_ERR_ARG, "gauge_stout_smear: rho must be finite");
  StoutGeom g;
  g.V = 1;
  for (int m = 0; m < 4; ++m) {
    CMX_REQUIRE(dims[m] > 0 && dims[m] % 2 == 0, CMX_ERR_ARG, "gauge_stout_smear: extents must be even and positive");
    g.L[m] = dims[m];
    g.V *= dims[m];
  }
  g.Vh = g.V / 2;
  CMX_REQUIRE(4 * g.V <= (long)INT32_MAX * 256, CMX_ERR_ARG, "gauge_stout_smear: lattice too large for one grid");
  const size_t bytes = sizeof(double) * 18 * 4 * (size_t)g.V;
  if (nstep == 0) {
    if (out != in) std::memcpy(out, in, bytes);
    return;
  }
  DevScratch a(bytes), b(bytes);
  host_to_device(a.get(), in, bytes, 0);
  const dim3 grid((unsigned)((4 * g.V + 255) / 256));
  hipLaunchKernelGGL(k_links_to_soa, grid, dim3(256), 0, 0, g.V, a.as<double2>(), b.as<double2>());
  CMX_HIP(hipGetLastError());
  double2* cur = b.as<double2>();
  double2* nxt = a.as<double2>();
  for (int k = 0; k < nstep; ++k) {
    hipLaunchKernelGGL(k_stout_step, dim3((unsigned)(2 * ((g.Vh + 63) / 64))), dim3(256), 0, 0, g, cur, nxt, rho, dirs);
    CMX_HIP(hipGetLastError());
    std::swap(cur, nxt);
  }
  hipLaunchKernelGGL(k_links_from_soa, grid, dim3(256), 0, 0, g.V, cur, nxt);
  CMX_HIP(hipGetLastError());
  device_to_host(out, nxt, bytes, 0);
}

}  // namespace cmx
