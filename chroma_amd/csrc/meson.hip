// Meson two-point functions on the device, in FP64: mesons() (mesons_w.cc:97-180) for the 16 gamma
// insertions Gamma(n) = gamma_1^n0 gamma_2^n1 gamma_3^n2 gamma_4^n3 (docs/notes/chroma_gamma_matrices.tex),
//   c_n(x) = tr[ adj(gamma_5 S_2(x) gamma_5) Gamma(n) S_1(x) Gamma(n) ]      (trace over spin and colour),
// then the sink-momentum projection of SftMom::sft (sftmom.cc:405-460, 520-530) over the spatial sites of
// each time slice, phase exp(i 2 pi sum_k n_k (x_k - origin_k) / L_k), with the time slice counted from
// the source, t_eff = (t - origin_t) mod L_t (mesons_w.cc:160-165).
//
// Every Gamma(n) and gamma_5 of the DeGrand-Rossi basis (docs/notes/gamma_conventions.tex:74-79) has one
// non-zero entry, a power of i, per row: gamma_5 is diagonal, and Gamma(n) maps spin a to spin a ^ k(n) with
// one of four masks k.  So the trace needs, for each of the 16 spin blocks (a, b) of S_2, the 3x3 colour
// products with the four blocks (a^k, b^k) of S_1, and every Gamma is a signed sum of those 64 numbers.
// Propagators: [site][sink spin*3 + colour][source spin*3 + colour] complex, sites in the host order.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <string>
#include <vector>

#include "op.h"

namespace cmx {

namespace {

// signed permutation: row a has its one non-zero entry ph[a] in column p[a]
struct SPerm {
  int p[4];
  double ph_re[4], ph_im[4];
};

SPerm sp_mul(const SPerm& A, const SPerm& B) {
  SPerm C;
  for (int a = 0; a < 4; ++a) {
    const int k = A.p[a];
    C.p[a] = B.p[k];
    C.ph_re[a] = A.ph_re[a] * B.ph_re[k] - A.ph_im[a] * B.ph_im[k];
    C.ph_im[a] = A.ph_re[a] * B.ph_im[k] + A.ph_im[a] * B.ph_re[k];
  }
  return C;
}

SPerm gamma_dr(int mu) {  // gamma_1..gamma_4 (mu = 0..3) of the DeGrand-Rossi basis
  static const int perm[4][4] = {{3, 2, 1, 0}, {3, 2, 1, 0}, {2, 3, 0, 1}, {2, 3, 0, 1}};
  static const double re[4][4] = {{0, 0, 0, 0}, {-1, 1, 1, -1}, {0, 0, 0, 0}, {1, 1, 1, 1}};
  static const double im[4][4] = {{1, 1, -1, -1}, {0, 0, 0, 0}, {1, -1, -1, 1}, {0, 0, 0, 0}};
  SPerm g;
  for (int a = 0; a < 4; ++a) g.p[a] = perm[mu][a], g.ph_re[a] = re[mu][a], g.ph_im[a] = im[mu][a];
  return g;
}

SPerm gamma_n(int n) {
  SPerm g;
  for (int a = 0; a < 4; ++a) g.p[a] = a, g.ph_re[a] = 1, g.ph_im[a] = 0;
  for (int mu = 0; mu < 4; ++mu)
    if (n >> mu & 1) g = sp_mul(g, gamma_dr(mu));
  return g;
}

// k(n): Gamma(n) maps spin a to a ^ k (gamma_1, gamma_2 flip with 3, gamma_3, gamma_4 with 2)
__host__ __device__ constexpr int meson_mask(int n) {
  return (((n ^ (n >> 1)) & 1) ? 3 : 0) ^ ((((n >> 2) ^ (n >> 3)) & 1) ? 2 : 0);
}

// c_n = sum_{a,b} coef[n][a][b] T_k(a,b), T_k(a,b) = sum_{ij} conj(S_2[(a,i),(b,j)]) S_1[(a^k,i),(b^k,j)]:
// anti_{(a,i),(b,j)} = g5ph[a] S_2[(a,i),(b,j)] g5ph[b] (gamma_5 diagonal) and
// (G S_1 G)_{(a,i),(b,j)} = Gph[a] S_1[(pG[a],i),(r,j)] Gph[r] where pG[r] = b.
std::vector<double2> meson_coefs() {
  const SPerm g5 = gamma_n(15);
  std::vector<double2> t;
  for (int n = 0; n < 16; ++n) {
    const SPerm G = gamma_n(n);
    const int k = meson_mask(n);
    for (int a = 0; a < 4; ++a)
      for (int b = 0; b < 4; ++b) {
        const int r = b ^ k;
        CMX_REQUIRE(g5.p[a] == a && G.p[a] == (a ^ k) && G.p[r] == b, CMX_ERR_STATE, "meson_2pt: gamma table");
        // conj(g5ph[a] g5ph[b]) Gph[a] Gph[r]
        const double ar = g5.ph_re[a] * g5.ph_re[b] - g5.ph_im[a] * g5.ph_im[b];
        const double ai = -(g5.ph_re[a] * g5.ph_im[b] + g5.ph_im[a] * g5.ph_re[b]);
        const double br = G.ph_re[a] * G.ph_re[r] - G.ph_im[a] * G.ph_im[r];
        const double bi = G.ph_re[a] * G.ph_im[r] + G.ph_im[a] * G.ph_re[r];
        t.push_back(make_double2(ar * br - ai * bi, ar * bi + ai * br));
      }
  }
  return t;
}

struct ProjGeom {
  int L[4];
  long V, Vh;
  int org[4];
};

// Contraction and projection in one pass over the propagators, which it reads once (HBM-bound: 2304 B per
// site and propagator against 4352 FP64 FMAs and 11.5 KB of LDS reads).  A work-group walks a range of one
// time slice MESON_SITES sites at a time: the sites go to LDS with direct loads (double-buffered: the next
// group is on its way while this one is contracted, and no registers hold it, which the 4 NM complex sums
// per lane need), lane (site, a, b) forms T_0..T_3 of its spin block and adds phase_m(x) T_k to its sums;
// Gamma and the momenta never meet per site.  At the end the lanes' sums are combined over sites and spins
// (fixed order) and the work-group writes its 16 x NM partial correlators.
// 24^3x48, 7 momenta, S_1 = S_2: two kernels that stored the 16 site correlators (one trace per lane and
// Gamma, 256 colour products per site) and read them back per momentum took 2.17 ms, this takes 0.33.
constexpr int MESON_SITES = 16;
constexpr int MESON_NM = 8;  // momenta per pass over the propagators
constexpr size_t MESON_SLAB = (size_t)1 << 30;  // bytes of a host propagator on the device at a time

struct MesonArgs {
  ProjGeom g;
  const double2 *s1, *s2, *coef;
  const int* moms;
  int nmom;    // momenta of this launch
  int tb, nt;  // the propagators hold the nt time slices from tb on
  int t0;      // first time slice of this launch
  int nchunk;  // work-groups per time slice
  int groups;  // groups of MESON_SITES sites per work-group
  double2* phase;  // [momentum][x, then y, then z]: exp(i 2 pi k (x - origin) / L) of each direction
  double2* part;   // [slice of this launch][chunk][momentum][n]
};

// The phase factors of each direction, from the product k (x - origin) reduced in integers: mod L, then to the
// nearest quarter turn, so that the argument of sincospi stays within 1/4 and its rounding does not show (the whole
// sum over a slice depends on the factor of one direction coherently).
__global__ void __launch_bounds__(256) k_meson_phase(MesonArgs A) {
  const int nx = A.g.L[0] + A.g.L[1] + A.g.L[2];
  const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x), m = blockIdx.y;
  if (q >= nx) return;
  const int d = q < A.g.L[0] ? 0 : (q < A.g.L[0] + A.g.L[1] ? 1 : 2);
  const int x = q - (d > 0 ? A.g.L[0] : 0) - (d > 1 ? A.g.L[1] : 0);
  const long L = A.g.L[d];
  const long k = (long)A.moms[3 * m + d] * (x - A.g.org[d]);
  long r = k == (int)k ? (int)k % (int)L : k % L;  // a 32-bit remainder takes a fraction of a 64-bit one's time
  if (r < 0) r += L;
  const int j = (int)(4.0f * (float)r * __builtin_amdgcn_rcpf((float)L) + 0.5f);  // off by one at a tie at most
  const long e = 4 * r - j * L;  // r / L = j / 4 + e / (4 L), |e| <= L / 2
  double s, c;
  sincospi((double)e / (double)(2 * L), &s, &c);
  A.phase[(size_t)m * nx + q] = (j & 1) ? ((j & 2) ? make_double2(s, -c) : make_double2(-s, c))
                                        : ((j & 2) ? make_double2(-c, -s) : make_double2(c, s));
}

__device__ __forceinline__ double2 cmul2(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}

// DIRECT: both propagators start on 16 bytes, as the direct loads' elements must; a caller's device arrays need only
// the 8 of a double, and otherwise pass through registers
template <int NM, bool SAME, bool DIRECT> __global__ void __launch_bounds__(256, 2) k_meson(MesonArgs A) {
  constexpr int SB = MESON_SITES * 144;  // 256 threads x 9 elements of 16 B
  __shared__ __align__(16) double2 stage[2][SAME ? 1 : 2][SB];
  __shared__ double2 shp[2][MESON_SITES * NM];
  static_assert(4 * NM * 4 * 16 <= SB, "the final combination re-uses a staging buffer");
  const int tid = threadIdx.x, ab = tid & 15, slot = tid >> 4, a = ab >> 2, b = ab & 3;
  const int t = A.t0 + (int)blockIdx.x / A.nchunk, chunk = (int)blockIdx.x % A.nchunk;
  const int m0 = (int)blockIdx.y * NM;
  const int Lxh = A.g.L[0] / 2, Ly = A.g.L[1];
  const int Vsh = Lxh * Ly * A.g.L[2];  // sites of the slice per checkerboard
  const int vbeg = chunk * A.groups * MESON_SITES;
  const int vend = min(2 * Vsh, vbeg + A.groups * MESON_SITES);
  const int nx = A.g.L[0] + A.g.L[1] + A.g.L[2];
  // stages the MESON_SITES sites from v0 (site v of the slice: even sites first, each checkerboard a
  // contiguous range of the host order).  Lanes past the range re-read its last site: their phase is zero.
  auto fetch = [&](int v0, int buf) {
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int q = tid + 256 * j, sl = q / 144, e = q - sl * 144;
      const int v = min(v0 + sl, vend - 1);
      const int cb = v >= Vsh ? 1 : 0;
      const size_t at = ((size_t)(cb * A.nt + (t - A.tb)) * Vsh + (v - cb * Vsh)) * 144 + e;
      if constexpr (DIRECT) {
        const int w = (tid & ~63) + 256 * j;  // a wave's 64 elements are consecutive in LDS
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(A.s1 + at),
                                         (__attribute__((address_space(3))) void*)&stage[buf][0][w], 16, 0, 0);
        if constexpr (!SAME)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(A.s2 + at),
                                           (__attribute__((address_space(3))) void*)&stage[buf][1][w], 16, 0, 0);
      } else {
        const double *d1 = reinterpret_cast<const double*>(A.s1), *d2 = reinterpret_cast<const double*>(A.s2);
        stage[buf][0][q] = make_double2(d1[2 * at], d1[2 * at + 1]);
        if constexpr (!SAME) stage[buf][1][q] = make_double2(d2[2 * at], d2[2 * at + 1]);
      }
    }
    if (tid < MESON_SITES * NM) {
      const int m = m0 + tid % NM, v = v0 + tid / NM;
      double2 p = make_double2(0, 0);
      if (v < vend && m < A.nmom) {
        const int cb = v >= Vsh ? 1 : 0;
        int r = v - cb * Vsh;
        const int xh = r % Lxh;
        r /= Lxh;
        const int y = r % Ly, z = r / Ly;
        const int x = 2 * xh + ((cb + y + z + t) & 1);
        const double2* f = A.phase + (size_t)m * nx;
        p = cmul2(cmul2(f[x], f[A.g.L[0] + y]), f[A.g.L[0] + Ly + z]);
      }
      shp[buf][tid] = p;  // [site][momentum]
    }
  };
  double2 acc[NM][4];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[m][k] = make_double2(0, 0);
  if (vbeg < vend) fetch(vbeg, 0);
  int buf = 0;
  for (int v0 = vbeg; v0 < vend; v0 += MESON_SITES, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's direct loads have reached LDS
    __syncthreads();
    if (v0 + MESON_SITES < vend) fetch(v0 + MESON_SITES, buf ^ 1);
    const double2* p1 = stage[buf][0] + slot * 144;
    const double2* p2 = stage[buf][SAME ? 0 : 1] + slot * 144 + a * 36 + b * 3;
    double2 x[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) x[3 * i + j] = p2[i * 12 + j];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double2* q = p1 + (a ^ k) * 36 + (b ^ k) * 3;
      double sr = 0, si = 0;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const double2 u = x[3 * i + j], w = q[i * 12 + j];
          sr = fma(u.x, w.x, fma(u.y, w.y, sr));
          si = fma(u.x, w.y, fma(-u.y, w.x, si));
        }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const double2 p = shp[buf][slot * NM + m];
        acc[m][k].x = fma(p.x, sr, fma(-p.y, si, acc[m][k].x));
        acc[m][k].y = fma(p.x, si, fma(p.y, sr, acc[m][k].y));
      }
    }
  }
  __syncthreads();
  double2* sh1 = stage[0][0];
  // over the wave's four sites, then the four waves and the spins
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
      for (int off = 16; off < 64; off <<= 1) {
        acc[m][k].x += __shfl_xor(acc[m][k].x, off, 64);
        acc[m][k].y += __shfl_xor(acc[m][k].y, off, 64);
      }
      if ((tid & 63) < 16) sh1[(((tid >> 6) * NM + m) * 4 + k) * 16 + ab] = acc[m][k];
    }
  __syncthreads();
  if (tid < 16 * NM) {
    const int n = tid & 15, m = tid >> 4, k = meson_mask(n);
    if (m0 + m < A.nmom) {
      double cr = 0, ci = 0;
      for (int s = 0; s < 16; ++s) {
        double2 z = make_double2(0, 0);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const double2 u = sh1[((w * NM + m) * 4 + k) * 16 + s];
          z.x += u.x;
          z.y += u.y;
        }
        const double2 c = A.coef[n * 16 + s];
        cr += c.x * z.x - c.y * z.y;
        ci += c.x * z.y + c.y * z.x;
      }
      A.part[((size_t)blockIdx.x * A.nmom + m0 + m) * 16 + n] = make_double2(cr, ci);
    }
  }
}

// s + z with the rounding error of the sum added to e
__device__ __forceinline__ void two_sum(double& s, double& e, double z) {
  const double t = s + z, b = t - s;
  e += (s - (t - b)) + (z - b);
  s = t;
}

// out[n][m0 + m][t_eff] = sum over the slice's chunks, in order (deterministic); one lane per (m, n) of a slice.
// The sum is compensated: the chunks of a coherent sum (the pion at zero momentum) are all alike, and the rounding of
// the plain sum over some forty of them was most of the result's error (8x10x6x8: 2.2e-16 of the correlators'
// norm, with it 0.7e-16).
__global__ void __launch_bounds__(256) k_meson_reduce(MesonArgs A, int m0, int nmom_all, double2* __restrict__ out) {
  const int t = A.t0 + (int)blockIdx.x, q = (int)(blockIdx.y * blockDim.x + threadIdx.x);
  if (q >= A.nmom * 16) return;
  const int m = q >> 4, n = q & 15;
  const double2* p = A.part + (size_t)blockIdx.x * A.nchunk * A.nmom * 16 + q;
  double2 s = make_double2(0, 0), e = make_double2(0, 0);
  for (int c = 0; c < A.nchunk; c += 8) {  // eight loads in flight, of few work-groups too
    double2 z[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      z[j] = c + j < A.nchunk ? p[(size_t)(c + j) * A.nmom * 16] : make_double2(0, 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      two_sum(s.x, e.x, z[j].x);
      two_sum(s.y, e.y, z[j].y);
    }
  }
  s.x += e.x;
  s.y += e.y;
  const int teff = (t - A.g.org[3] % A.g.L[3] + A.g.L[3]) % A.g.L[3];
  out[((size_t)n * nmom_all + m0 + m) * A.g.L[3] + teff] = s;
}

ProjGeom proj_geom(const int dims[4], const int origin[4]) {
  ProjGeom g;
  g.V = 1;
  for (int m = 0; m < 4; ++m) {
    CMX_REQUIRE(dims[m] > 0 && dims[m] % 2 == 0, CMX_ERR_ARG, "meson_2pt: extents must be even and positive");
    g.L[m] = dims[m];
    g.V *= dims[m];
    g.org[m] = origin ? origin[m] : 0;
    CMX_REQUIRE(g.org[m] >= 0 && g.org[m] < dims[m], CMX_ERR_ARG, "meson_2pt: origin outside the lattice");
  }
  g.Vh = g.V / 2;
  CMX_REQUIRE(g.V <= (long)INT32_MAX * 8, CMX_ERR_ARG, "meson_2pt: lattice too large for one grid");
  return g;
}

// The work-groups of a lattice: about 2048 in all (four rounds of the 512 that are resident), each with at
// least one group of sites.  They depend on the lattice alone, so the sums have one order whatever scratch
// they are cut to.
void meson_chunks(const ProjGeom& g, int& nchunk, int& groups) {
  const long Vs = (long)g.L[0] * g.L[1] * g.L[2], ng = (Vs + MESON_SITES - 1) / MESON_SITES;
  const long want = std::max<long>(1, std::min<long>(ng, (2048 + g.L[3] - 1) / g.L[3]));
  groups = (int)((ng + want - 1) / want);
  nchunk = (int)((ng + groups - 1) / groups);
}

// Scratch for nm momenta (the phase factors) and the partial correlators of nt slices
size_t meson_bytes(const ProjGeom& g, int nchunk, int nm, int nt) {
  return sizeof(double2) * (size_t)nm * ((size_t)(g.L[0] + g.L[1] + g.L[2]) + (size_t)16 * nchunk * nt);
}

template <int NM> void launch_meson(const MesonArgs& A, int nt, hipStream_t st) {
  const dim3 grid((unsigned)(nt * A.nchunk), (unsigned)((A.nmom + NM - 1) / NM));
  const bool direct = ((reinterpret_cast<uintptr_t>(A.s1) | reinterpret_cast<uintptr_t>(A.s2)) & 15) == 0;
  auto k = A.s1 == A.s2 ? (direct ? k_meson<NM, true, true> : k_meson<NM, true, false>)
                        : (direct ? k_meson<NM, false, true> : k_meson<NM, false, false>);
  hipLaunchKernelGGL(k, grid, dim3(256), 0, st, A);
}

// All momenta of the time slices tb .. tb + ntb - 1, which s1 and s2 hold (even sites, then odd sites, each by t), in passes
// whose partial correlators fit `bytes` of scratch
void run_meson(const ProjGeom& g, int tb, int ntb, const double2* s1, const double2* s2, const double2* coef,
               const int* moms, int nmom, double2* part, size_t bytes, double2* out, hipStream_t st) {
  MesonArgs A;
  A.g = g;
  A.tb = tb, A.nt = ntb;
  A.s1 = s1, A.s2 = s2, A.coef = coef;
  meson_chunks(g, A.nchunk, A.groups);
  const size_t slice = sizeof(double2) * 16 * (size_t)A.nchunk;  // per momentum
  // up to 64 momenta per pass (the grid's second index walks them by MESON_NM; fewer where the phases of a
  // very long lattice would fill the scratch), as many slices as fit
  const int nx = g.L[0] + g.L[1] + g.L[2];
  int mstep = std::min(nmom, 64);
  while (mstep > 1 && meson_bytes(g, A.nchunk, mstep, 1) > bytes) mstep = (mstep + 1) / 2;
  CMX_REQUIRE(meson_bytes(g, A.nchunk, mstep, 1) <= bytes, CMX_ERR_STATE, "meson_2pt: scratch too small");
  const size_t table = sizeof(double2) * (size_t)nx * mstep;
  const int tstep = (int)std::min<size_t>(ntb, (bytes - table) / (slice * mstep));
  A.phase = part, A.part = part + (size_t)nx * mstep;
  for (int m0 = 0; m0 < nmom; m0 += mstep) {
    A.moms = moms + 3 * m0;
    A.nmom = std::min(mstep, nmom - m0);
    A.t0 = tb;
    hipLaunchKernelGGL(k_meson_phase, dim3((unsigned)((nx + 255) / 256), (unsigned)A.nmom), dim3(256), 0, st, A);
    CMX_HIP(hipGetLastError());
    for (int t0 = tb; t0 < tb + ntb; t0 += tstep) {
      const int nt = std::min(tstep, tb + ntb - t0);
      A.t0 = t0;
      switch (A.nmom) {
        case 1: launch_meson<1>(A, nt, st); break;
        case 2: launch_meson<2>(A, nt, st); break;
        case 3: case 4: launch_meson<4>(A, nt, st); break;
        default: launch_meson<MESON_NM>(A, nt, st); break;
      }
      CMX_HIP(hipGetLastError());
      hipLaunchKernelGGL(k_meson_reduce, dim3((unsigned)nt, (unsigned)((A.nmom * 16 + 255) / 256)), dim3(256), 0, st, A,
                         m0, nmom, out);
      CMX_HIP(hipGetLastError());
    }
  }
}

// The allocation-free variant's scratch: the partial correlators of a pass (64 MiB), followed by the
// Gamma coefficients (written once per device at set-up, never overwritten).  Host code never uses this
// name as an address: it uses the per-device pointer that hipGetSymbolAddress returns.
constexpr long MESON_SCRATCH_SITES = 262144;  // 64^3: the largest spatial volume accepted
constexpr size_t MESON_SCRATCH_PART = (size_t)64 << 20;
constexpr size_t MESON_SCRATCH_BYTES = MESON_SCRATCH_PART + sizeof(double2) * 256;
static __device__ __align__(256) char scratch[MESON_SCRATCH_BYTES];

constexpr int MESON_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[MESON_MAX_DEVICES] = {};

}  // namespace

void meson_2pt(const int dims[4], const double* prop1, const double* prop2, const int origin[4], int nmom,
               const int* moms, double* corr) {
  CMX_REQUIRE(dims && prop1 && prop2 && corr, CMX_ERR_ARG, "meson_2pt: null array");
  CMX_REQUIRE(nmom >= 1 && nmom <= 4096 && moms, CMX_ERR_ARG, "meson_2pt: 1..4096 momenta");
  const ProjGeom g = proj_geom(dims, origin);
  const std::vector<double2> coefs = meson_coefs();
  // Host propagators pass through the device in ranges of time slices whose buffers the scratch cache holds: one of
  // 4.8 GB (32^3x64) was allocated and freed by every call, and hipMalloc then waited for the driver to clear what the
  // call before had freed (247 ms per call back to back, 103 without the wait).  A slice's sums do not depend on the range.
  const size_t slice = sizeof(double) * 288 * (size_t)g.L[0] * g.L[1] * g.L[2];
  const bool same = prop2 == prop1;
  const int nslab = (int)std::min<size_t>(g.L[3], std::max<size_t>(1, MESON_SLAB / slice));
  const size_t pbytes = slice * nslab;
  int nchunk, groups;
  meson_chunks(g, nchunk, groups);
  const size_t least = meson_bytes(g, nchunk, 1, 1), whole = meson_bytes(g, nchunk, std::min(nmom, 64), g.L[3]);
  DevScratch d1(pbytes), d2(same ? 0 : pbytes), dp(std::max(least, std::min(whole, MESON_SCRATCH_PART))), dt(sizeof(double2) * coefs.size()),
      dm(sizeof(int) * 3 * (size_t)nmom), dout(sizeof(double2) * 16 * (size_t)nmom * g.L[3]);
  CMX_HIP(hipMemcpy(dt.get(), coefs.data(), dt.bytes(), hipMemcpyHostToDevice));
  CMX_HIP(hipMemcpy(dm.get(), moms, dm.bytes(), hipMemcpyHostToDevice));
  for (int t = 0; t < g.L[3]; t += nslab) {
    const int nt = std::min(nslab, g.L[3] - t);
    const size_t half = slice / 2 * nt;  // a checkerboard's part, on the host and on the device
    auto up = [&](const DevScratch& d, const double* prop) {
      for (int cb = 0; cb < 2; ++cb)
        host_to_device(d.as<char>() + cb * half,
                       reinterpret_cast<const char*>(prop) + ((size_t)cb * g.L[3] + t) * (slice / 2), half, 0);
    };
    if (nt == g.L[3]) {
      host_to_device(d1.get(), prop1, 2 * half, 0);
      if (!same) host_to_device(d2.get(), prop2, 2 * half, 0);
    } else {
      up(d1, prop1);
      if (!same) up(d2, prop2);
    }
    run_meson(g, t, nt, d1.as<double2>(), same ? d1.as<double2>() : d2.as<double2>(), dt.as<double2>(), dm.as<int>(),
              nmom, dp.as<double2>(), dp.bytes(), dout.as<double2>(), 0);
  }
  CMX_HIP(hipMemcpy(corr, dout.get(), dout.bytes(), hipMemcpyDeviceToHost));
}

void meson_scratch_setup() {
  int dev = 0;
  CMX_HIP(hipGetDevice(&dev));
  CMX_REQUIRE(dev >= 0 && dev < MESON_MAX_DEVICES, CMX_ERR_UNSUPPORTED, "meson_2pt_noalloc: device index too large");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev]) return;
  void* ptr = nullptr;
  CMX_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  CMX_REQUIRE(ptr != nullptr, CMX_ERR_HIP, "meson_2pt_noalloc: no device address for the scratch array");
  const std::vector<double2> coefs = meson_coefs();
  CMX_HIP(hipMemcpy(static_cast<char*>(ptr) + MESON_SCRATCH_PART, coefs.data(), sizeof(double2) * coefs.size(),
                    hipMemcpyHostToDevice));
  g_scratch_ptr[dev] = ptr;
}

void meson_2pt_noalloc(const int dims[4], const double* prop1, const double* prop2, const int origin[4], int nmom,
                       const int* moms, double* corr, hipStream_t stream) {
  CMX_REQUIRE(dims && prop1 && prop2 && corr && moms, CMX_ERR_ARG, "meson_2pt_noalloc: null array");
  CMX_REQUIRE(nmom >= 1 && nmom <= 4096, CMX_ERR_ARG, "meson_2pt_noalloc: 1..4096 momenta");
  const ProjGeom g = proj_geom(dims, origin);
  const long Vs = (long)g.L[0] * g.L[1] * g.L[2];
  CMX_REQUIRE(Vs <= MESON_SCRATCH_SITES, CMX_ERR_ARG,
              "meson_2pt_noalloc: spatial volume above 262144 sites (64^3), the scratch array's limit");
  meson_scratch_setup();
  int dev = 0;
  CMX_HIP(hipGetDevice(&dev));
  char* base = static_cast<char*>(g_scratch_ptr[dev]);
  run_meson(g, 0, g.L[3], reinterpret_cast<const double2*>(prop1), reinterpret_cast<const double2*>(prop2),
            reinterpret_cast<const double2*>(base + MESON_SCRATCH_PART), moms, nmom, reinterpret_cast<double2*>(base),
            MESON_SCRATCH_PART, reinterpret_cast<double2*>(corr), stream);
}

}  // namespace cmx
