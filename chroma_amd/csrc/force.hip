// Clover force terms on the device, in FP64 (CloverTermBase, clover_term_base_w.h:320-870), and the
// derivative of the even-odd clover operator (EvenOddPrecLogDetLinearOperator::deriv,
// eoprec_logdet_linop.h:114-157, with the pieces of eoprec_clover_linop_w.cc:192-260).
//
// For every plane mu < nu the insertion matrix Lambda lives on the sites of one checkerboard cb:
//   deriv:     Lambda(x) = -(1/8) c_munu traceSpin(outerProduct(gamma_mu gamma_nu psi, chi))(x)
//   derivTrLn: Lambda(x) = -(1/8) c_munu traceSpin(gamma_mu gamma_nu A^-1(x))   (triacntr, the inverted term)
// with c_munu the 1/2-scaled clover coefficient of the plane (clovCoeffT when nu is time).  The link
// derivative is the sum over the four clover leaves of the plane with Lambda inserted at each corner of
// cb (deriv_loops): per output link U_mu(x) two terms at x and two terms of the leaf below it (at
// x - nu), and per U_nu(x) two at x and two of the leaf to its left (at x - mu).  One lane evaluates
// those of the three planes of its link and writes that link's derivative only: no atomics, deterministic.  ds is [4][V][3][3] complex in the host site order (the layout
// of the C-ABI), accumulated as ds[mu] += ..., ds[nu] -= ... .
#include <cstring>

#include "op.h"
#include "su3_dev.h"

namespace cmx {

namespace {

// gamma_mu gamma_nu of the DeGrand-Rossi basis as a signed permutation: row s has its one entry ph[s]
// in column p[s]; it maps each chiral half (spins 0,1 / 2,3) onto itself
struct Gmn {
  int p[4];
  double re[4], im[4];
};

struct ForcePlanes {
  Gmn G[6];
  double f[6];  // -(1/8) c_munu
};

__device__ __forceinline__ int plane_index(int mu, int nu) { return mu == 0 ? nu - 1 : mu == 1 ? nu + 1 : 5; }

__device__ __forceinline__ M3 madd(const M3& A, const M3& B) {
  M3 C;
#pragma unroll
  for (int k = 0; k < 18; ++k) C.a[k] = A.a[k] + B.a[k];
  return C;
}

// Lambda for the six planes at site i of cb, from chi and psi (deriv) or the inverted clover (derivTrLn).
// Lam: [plane][9][Vh] double2
template <bool TRLN>
__global__ void __launch_bounds__(256) k_force_lambda(Geom g, ForcePlanes P, VRef chi, VRef psi,
                                                      const double2* __restrict__ clov, double2* __restrict__ Lam) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.Vh) return;
  double c[24], q[24];
  double Are[12][12], Aim[12][12];
  if constexpr (!TRLN) {
    SpinorIO<P64>::load(chi.v, chi.nrm, chi.stride, i, c);
    SpinorIO<P64>::load(psi.v, psi.nrm, psi.stride, i, q);
  } else {
    // the two chiral 6x6 blocks {diag[6], lower offd[15] complex} of the inverted term
#pragma unroll
    for (int r = 0; r < 12; ++r)
#pragma unroll
      for (int s = 0; s < 12; ++s) Are[r][s] = Aim[r][s] = 0;
    for (int b = 0; b < 2; ++b) {
      double t[36];
      for (int k = 0; k < 18; ++k) {
        const double2 v = clov[(size_t)(18 * b + k) * g.Vh + i];
        t[2 * k] = v.x;
        t[2 * k + 1] = v.y;
      }
      for (int r = 0; r < 6; ++r) Are[6 * b + r][6 * b + r] = t[r];
      for (int r = 1; r < 6; ++r)
        for (int s = 0; s < r; ++s) {
          const int e = r * (r - 1) / 2 + s;
          Are[6 * b + r][6 * b + s] = t[6 + 2 * e];
          Aim[6 * b + r][6 * b + s] = t[6 + 2 * e + 1];
          Are[6 * b + s][6 * b + r] = t[6 + 2 * e];
          Aim[6 * b + s][6 * b + r] = -t[6 + 2 * e + 1];
        }
    }
  }
  for (int pl = 0; pl < 6; ++pl) {
    const Gmn& G = P.G[pl];
    double2* L = Lam + (size_t)pl * 9 * g.Vh;
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) {
        double re = 0, im = 0;
        for (int s = 0; s < 4; ++s) {
          const int t = G.p[s];
          double xr, xi;  // deriv: (Gamma psi)_{s,a} conj(chi_{s,b});  derivTrLn: Gamma_{s,t} A_{(t,a),(s,b)}
          if constexpr (!TRLN) {
            const double pr = q[2 * (3 * t + a)], pi = q[2 * (3 * t + a) + 1];
            const double gr = G.re[s] * pr - G.im[s] * pi, gi = G.re[s] * pi + G.im[s] * pr;
            const double cr = c[2 * (3 * s + b)], ci = c[2 * (3 * s + b) + 1];
            xr = gr * cr + gi * ci;
            xi = gi * cr - gr * ci;
          } else {
            const double ar = Are[3 * t + a][3 * s + b], ai = Aim[3 * t + a][3 * s + b];
            xr = G.re[s] * ar - G.im[s] * ai;
            xi = G.re[s] * ai + G.im[s] * ar;
          }
          re += xr;
          im += xi;
        }
        L[(size_t)(3 * a + b) * g.Vh + i] = make_double2(P.f[pl] * re, P.f[pl] * im);
      }
  }
}

struct LoopCtx {
  Geom g;
  const double2* g64[2];
  const double2* Lam;  // [6 planes][9][Vh]
  int cb;
};

// conj-transposed if dag (the same in all lanes)
__device__ __forceinline__ M3 load_m3(const double2* b, size_t stride, bool dag) {
  M3 m;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const double2 v = b[(size_t)(dag ? 3 * (k % 3) + k / 3 : k) * stride];
    m.a[2 * k] = v.x;
    m.a[2 * k + 1] = dag ? -v.y : v.y;
  }
  return m;
}

// acc += f (one part of deriv_loops at site y (coordinates), Lambda on the sites of parity cb).
// part = 0: the ds_mu terms at y; 1: the tmp_mu terms (shifted to y + nu); 2: the ds_nu terms;
// 3: the tmp_nu terms (shifted to y + mu).  A part is a staple X Y Z of three links of the plaquette at y with
// Lambda inserted at the two of its corners that have parity cb: at the two ends of Y Z, X (P W + W Q) with
// W = Y Z, or of X Y, (P W + W Q) Z with W = X Y.  Y always enters conj-transposed.  Three links, two Lambda and
// four products, in place of four, two and five or six with each term by itself.
__device__ __forceinline__ void add_part(const LoopCtx& C, int mu, int nu, const int (&y)[4], int part, double f,
                                         M3& acc) {
  const Geom& g = C.g;
  int ym[4], yn[4], ymn[4];
  shiftc(g, y, mu, 1, ym);
  shiftc(g, y, nu, 1, yn);
  shiftc(g, ym, nu, 1, ymn);
  const int py = __builtin_amdgcn_readfirstlane(parity(y));
  const size_t Vh = g.Vh;
  auto link = [&](int q, int dir, int i) { return (q ? C.g64[1] : C.g64[0]) + (size_t)dir * 9 * Vh + i; };
  const int i0 = cb_index(g, y), im = cb_index(g, ym), in = cb_index(g, yn), imn = cb_index(g, ymn);
  const double2 *A = link(1 - py, nu, im), *G = link(1 - py, mu, in), *E = link(py, mu, i0), *F = link(py, nu, i0);
  const double2* Lam = C.Lam + (size_t)plane_index(mu, nu) * 9 * Vh;
  const bool odd = part & 1, low = part < 2, in_cb = py == C.cb, left = odd != in_cb;  // left: X (P W + W Q)
  const double2 *X = low ? A : G, *Y = low ? (odd ? E : G) : (odd ? F : A), *Z = low ? F : E;
  const double2 *P = Lam + (in_cb ? imn : (low ? im : in)), *Q = Lam + (in_cb ? i0 : (low ? in : im));
  const M3 W = mul(load_m3(left ? Y : X, Vh, left || odd), load_m3(left ? Z : Y, Vh, !left || !odd));
  const M3 T = madd(mul(load_m3(P, Vh, false), W), mul(W, load_m3(Q, Vh, false)));
  const M3 O = load_m3(left ? X : Z, Vh, left == odd);
  const M3 R = left ? mul(O, T) : mul(T, O);
#pragma unroll
  for (int k = 0; k < 18; ++k) acc.a[k] = fma(f, R.a[k], acc.a[k]);
}

// ds[mu](x) += scale sum over nu != mu of +- (ds_mu(x) - tmp_mu(x - nu)) of the plane (mu, nu), + for mu < nu.
// A work-group is the four directions of 64 sites of one checkerboard, so that mu and the insertion's corners are
// the same in all lanes of a wave and ds is read and written once; both checkerboards of a region follow each
// other on one XCD, whose L2 then serves most link and Lambda reads.  Bound by those reads and by two waves per
// SIMD (250 registers).  The six planes of one Lambda on 16^3x32: 156 us, where a launch per plane that kept all
// four parts of a site took 336.
__global__ void __launch_bounds__(256) k_force_loops(LoopCtx C, double scale, double2* __restrict__ ds) {
  const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = xcd_range(blockIdx.x, gridDim.x);
  const int i = (l >> 1) * 64 + (int)(threadIdx.x & 63);
  if (i >= C.g.Vh) return;
  const int p = l & 1;
  int x[4];
  cb_coords(C.g, p, i, x);
  double2* d = ds + ((size_t)mu * 2 * C.g.Vh + (size_t)p * C.g.Vh + i) * 9;
  M3 acc;
#pragma unroll
  for (int k = 0; k < 9; ++k) acc.a[2 * k] = d[k].x, acc.a[2 * k + 1] = d[k].y;
#pragma unroll 1
  for (int nu = 0; nu < 4; ++nu) {
    if (nu == mu) continue;
    const bool first = mu < nu;
    const int m = first ? mu : nu, n = first ? nu : mu;
    int xm[4];
    shiftc(C.g, x, nu, -1, xm);
    const double f = first ? scale : -scale;
    add_part(C, m, n, x, first ? 0 : 2, f, acc);
    add_part(C, m, n, xm, first ? 1 : 3, -f, acc);
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) d[k] = make_double2(acc.a[2 * k], acc.a[2 * k + 1]);
}

// ds_full[mu][cb*Vh + i] += f * ds_cb[mu][i]  (the hopping-term derivative's per-checkerboard layout)
__global__ void __launch_bounds__(256) k_force_axpy(long Vh, int cb, double f, const double2* __restrict__ src,
                                                    double2* __restrict__ dst) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * Vh * 9) return;
  const long k = t % 9, site = (t / 9) % Vh, mu = t / (9 * Vh);
  const double2 a = src[t];
  double2& b = dst[(mu * 2 * Vh + (long)cb * Vh + site) * 9 + k];
  b = make_double2(b.x + f * a.x, b.y + f * a.y);
}

ForcePlanes force_planes(const cmx_op_params& par) {
  // DeGrand-Rossi gamma_1..gamma_4 as signed permutations
  static const int perm[4][4] = {{3, 2, 1, 0}, {3, 2, 1, 0}, {2, 3, 0, 1}, {2, 3, 0, 1}};
  static const double gre[4][4] = {{0, 0, 0, 0}, {-1, 1, 1, -1}, {0, 0, 0, 0}, {1, 1, 1, 1}};
  static const double gim[4][4] = {{1, 1, -1, -1}, {0, 0, 0, 0}, {1, -1, -1, 1}, {0, 0, 0, 0}};
  ForcePlanes P;
  int pl = 0;
  for (int mu = 0; mu < 3; ++mu)
    for (int nu = mu + 1; nu < 4; ++nu, ++pl) {
      Gmn& G = P.G[pl];
      for (int s = 0; s < 4; ++s) {  // (gamma_mu gamma_nu)[s][p] = gmu[s][k] gnu[k][p], k = perm_mu[s]
        const int k = perm[mu][s];
        G.p[s] = perm[nu][k];
        G.re[s] = gre[mu][s] * gre[nu][k] - gim[mu][s] * gim[nu][k];
        G.im[s] = gre[mu][s] * gim[nu][k] + gim[mu][s] * gre[nu][k];
      }
      const double c = 0.5 * (nu == 3 ? par.clov_coeff_t : par.clov_coeff_r);  // getCloverCoeff
      P.f[pl] = -c / 8.0;
    }
  return P;
}

void launch_loops(Op& op, const double2* Lam, int cb, double scale, double2* ds) {
  LoopCtx C;
  C.g = op.g;
  C.g64[0] = op.gd->g64[0].as<double2>();
  C.g64[1] = op.gd->g64[1].as<double2>();
  C.Lam = Lam;
  C.cb = cb;
  hipLaunchKernelGGL(k_force_loops, dim3((unsigned)(2 * ((op.Vh + 63) / 64))), dim3(256), 0, op.stream, C, scale, ds);
  CMX_HIP(hipGetLastError());
}

}  // namespace

void clover_force(Op& op, bool trln, int cb, VRef chi, VRef psi, double scale, void* ds_full, void* lam_) {
  CMX_REQUIRE(op.clover(), CMX_ERR_ARG, "clover force: not a clover operator");
  CMX_REQUIRE(cb == 0 || cb == 1, CMX_ERR_ARG, "clover force: cb must be 0 or 1");
  CMX_REQUIRE(!trln || cb == 0, CMX_ERR_ARG, "clover force: derivTrLn of the inverted even-even term only");
  const ForcePlanes P = force_planes(op.par);
  double2* lam = static_cast<double2*>(lam_);
  const dim3 grid((unsigned)((op.Vh + 255) / 256));
  if (trln)
    hipLaunchKernelGGL(k_force_lambda<true>, grid, dim3(256), 0, op.stream, op.g, P, chi, psi,
                       op.clovinv_even[P64].as<double2>(), lam);
  else
    hipLaunchKernelGGL(k_force_lambda<false>, grid, dim3(256), 0, op.stream, op.g, P, chi, psi, nullptr,
                       lam);
  CMX_HIP(hipGetLastError());
  launch_loops(op, lam, cb, scale, static_cast<double2*>(ds_full));
}

void force_axpy(Op& op, int cb, double f, const void* ds_cb, void* ds_full) {
  const long n = 4 * op.Vh * 9;
  hipLaunchKernelGGL(k_force_axpy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, op.stream, op.Vh, cb, f,
                     static_cast<const double2*>(ds_cb), static_cast<double2*>(ds_full));
  CMX_HIP(hipGetLastError());
}

}  // namespace cmx
