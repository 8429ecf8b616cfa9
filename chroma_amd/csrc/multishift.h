// Device side of the multishift CG (multishift.hip): the shifted recurrences and the update of every shift's
// vectors, so that an iteration needs no host value.
#pragma once
#include "blas.h"

namespace cmx {

constexpr int MS_MAX = 64;  // shifts per solve

// Scalars of one solve, on the device
struct MsState {
  double b, bp, c, cp;                 // b = -cp / |M p0|^2 and its predecessor; |r|^2 and its predecessor
  double zc[MS_MAX], zp[MS_MAX];       // z_s and its predecessor
  double bs[MS_MAX];                   // bs_s of the last iteration
  double zr[MS_MAX], as[MS_MAX];       // the coming p_s = zr_s r + as_s p_s
  double sigma[MS_MAX], rsd_sq[MS_MAX];
  int conv[MS_MAX];  // 0 running, 1 its estimate is below target (psi_s update pending), 2 finished
};

struct MsLaunch {
  long ne;                 // double2 elements per vector (12 per site)
  int ns, isz, max_iter;
  MsState* st;
  double* S;               // the operator's scalar array: S[slot_a], S[slot_b] for p0 and r
  int* F;                  // F_DONE, F_CONV, F_K, F_ERR of the operator
  int slot_a, slot_b;
  const double* partials;  // of the reduction that a scalar kernel finishes
  int nb;
  double2 *r, *p0;
  double2 *p, *psi;        // ns vectors of ne elements each
};

// r = p0 = p_s = chi, psi_s = 0
void ms_init(const MsLaunch& L, const double2* chi, hipStream_t s);
// z = 1, bs = b z and so on for the first step (phase 0); b from |M p0|^2 (phase 1); c = |r|^2, the shifted
// recurrences, the per-shift tests and the next coefficients (phase 2)
void ms_scalars(const MsLaunch& L, int phase, hipStream_t s);
// p0 = r + a p0; for every shift psi_s -= bs_s p_s, p_s = zr_s r + as_s p_s
void ms_update(const MsLaunch& L, hipStream_t s);
// the psi_s updates that no further iteration makes
void ms_finish(const MsLaunch& L, hipStream_t s);

}  // namespace cmx
