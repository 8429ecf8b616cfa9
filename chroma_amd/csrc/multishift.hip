// Kernels of the multishift CG (MInvCG2_a, minvcg2.cc:72-355; Jegerlehner, hep-lat/9708029), FP64.
#include <cmath>

#include "multishift.h"

namespace cmx {

namespace {

// The scalar recurrences, one lane per shift, in the order the reference runs them (minvcg2.cc:179-339),
// after summing the preceding reduction's partials (fixed order, as the finalize kernel).
__global__ void __launch_bounds__(256) k_ms_scalars(MsLaunch L, int phase) {
  __shared__ double sh_sum;
  MsState* T = L.st;
  if (L.F[F_DONE]) return;
  double red[1] = {0};
  for (int k = threadIdx.x; k < L.nb; k += 256) red[0] += L.partials[k];
  block_sum<1>(red);
  if (threadIdx.x == 0) sh_sum = red[0];
  __syncthreads();
  const double sum = sh_sum;
  const int s = threadIdx.x;
  const bool mine = s < L.ns;
  if (phase == 1) {  // sum = |M p0|^2
    if (mine && T->conv[s] == 1) T->conv[s] = 2;  // ms_update has made its last psi_s update
    if (s == 0) {
      if (!(sum > 0.0) || !isfinite(sum)) {
        L.F[F_ERR] = CMX_ERR_BREAKDOWN;
        L.F[F_DONE] = L.F[F_CONV] = 1;
        return;
      }
      T->bp = T->b;
      T->b = -T->cp / sum;
      L.S[L.slot_b] = T->b;
    }
    return;
  }
  // sum = c = |r|^2
  const double c = sum, b = T->b, cp = T->cp;
  double z = 1.0;
  if (phase == 0) {
    if (mine) {
      z = 1.0 / (1.0 - T->sigma[s] * b);
      T->zp[s] = 1.0;
      T->zc[s] = z;
      T->bs[s] = b * z;
      T->conv[s] = 0;
    }
  } else {
    const double a = L.S[L.slot_a], bp = T->bp;
    if (mine && T->conv[s] == 0) {
      const double z0 = T->zc[s], z1 = T->zp[s];
      z = z0 * z1 * bp / (b * a * (z1 - z0) + z1 * bp * (1.0 - T->sigma[s] * b));
      T->zp[s] = z0;
      T->zc[s] = z;
      T->bs[s] = b * z / z0;
    }
  }
  const double a1 = c / cp;  // of the coming p0 = r + a p0
  bool conv = true;
  if (mine && T->conv[s] == 0) {
    // per-shift test on the shifted residual estimate c z_s^2 (:326-339); at the start the smallest
    // shift's target alone decides (:247)
    conv = phase == 0 ? c < T->rsd_sq[L.isz] : c * z * z < T->rsd_sq[s];
    if (conv && phase != 0) T->conv[s] = 1;
    T->zr[s] = T->zc[s];
    T->as[s] = a1 * T->zc[s] * T->bs[s] / (T->zp[s] * b);
  }
  const int all = __syncthreads_and(conv ? 1 : 0);
  if (s == 0) {
    L.S[L.slot_a] = a1;
    T->c = c;
    T->cp = c;
    const int k = phase == 0 ? 0 : L.F[F_K] + 1;
    L.F[F_K] = k;
    if (all) {
      L.F[F_DONE] = L.F[F_CONV] = 1;
      L.F[F_NCOUNT] = k;
    } else if (!isfinite(c) || k >= L.max_iter) {
      L.F[F_DONE] = L.F[F_CONV] = 1;
      L.F[F_NCOUNT] = L.max_iter;
    }
  }
}

__device__ __forceinline__ double2 lin(double a, double2 x, double b, double2 y) {  // a x + b y
  return make_double2(fma(a, x.x, b * y.x), fma(a, x.y, b * y.y));
}
__device__ __forceinline__ double2 axpy(double a, double2 x, double2 y) {  // y + a x
  return make_double2(fma(a, x.x, y.x), fma(a, x.y, y.y));
}

__global__ void __launch_bounds__(256) k_ms_init(MsLaunch L, const double2* __restrict__ chi) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= L.ne) return;
  const double2 x = chi[e];
  L.r[e] = x;
  L.p0[e] = x;
  for (int s = 0; s < L.ns; ++s) {
    L.p[s * L.ne + e] = x;
    L.psi[s * L.ne + e] = make_double2(0, 0);
  }
}

// Every shift in one pass over r, elementwise (all vectors share one layout): the psi_s update of the last
// iteration and the p_s update of this one read p_s once between them, so a shift costs four vector
// streams where the separate axpy and axpby passes took six, and r is read once for all shifts.
// 16^3x32, ten shifts: 8.5 + 7.1 us per shift and iteration as separate passes, 6.1 in this one (5 TB/s).
__global__ void __launch_bounds__(256) k_ms_update(MsLaunch L) {
  __shared__ int act[MS_MAX], nact, fin[MS_MAX];
  if (L.F[F_DONE]) return;
  const MsState* T = L.st;
  if (threadIdx.x == 0) {
    int n = 0;
    for (int s = 0; s < L.ns; ++s)
      if (T->conv[s] != 2) {
        fin[n] = T->conv[s];
        act[n++] = s;
      }
    nact = n;
  }
  __syncthreads();
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= L.ne) return;
  const double2 r = L.r[e];
  L.p0[e] = axpy(L.S[L.slot_a], L.p0[e], r);
  const int n = nact;
#pragma unroll 4
  for (int j = 0; j < n; ++j) {
    const int s = act[j];
    const double2 p = L.p[s * L.ne + e], x = L.psi[s * L.ne + e];
    L.psi[s * L.ne + e] = axpy(-T->bs[s], p, x);
    if (fin[j] == 0) L.p[s * L.ne + e] = lin(T->zr[s], r, T->as[s], p);
  }
}

__global__ void __launch_bounds__(256) k_ms_finish(MsLaunch L) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  const int s = blockIdx.y;
  if (e >= L.ne || L.st->conv[s] == 2) return;
  L.psi[s * L.ne + e] = axpy(-L.st->bs[s], L.p[s * L.ne + e], L.psi[s * L.ne + e]);
}

unsigned grid_of(long ne) { return (unsigned)((ne + 255) / 256); }

}  // namespace

void ms_init(const MsLaunch& L, const double2* chi, hipStream_t s) {
  hipLaunchKernelGGL(k_ms_init, dim3(grid_of(L.ne)), dim3(256), 0, s, L, chi);
}
void ms_scalars(const MsLaunch& L, int phase, hipStream_t s) {
  hipLaunchKernelGGL(k_ms_scalars, dim3(1), dim3(256), 0, s, L, phase);
}
void ms_update(const MsLaunch& L, hipStream_t s) {
  hipLaunchKernelGGL(k_ms_update, dim3(grid_of(L.ne)), dim3(256), 0, s, L);
}
void ms_finish(const MsLaunch& L, hipStream_t s) {
  hipLaunchKernelGGL(k_ms_finish, dim3(grid_of(L.ne), (unsigned)L.ns), dim3(256), 0, s, L);
}

}  // namespace cmx
