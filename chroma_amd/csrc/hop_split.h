// Hopping term for small lattices: the four directions of a site on four waves.
//
// A lattice of up to some 10^5 sites per checkerboard gives the one-lane-per-site kernels one wave per SIMD
// or less, and their time is the latency of eight dependent load-and-multiply steps.  Here a work-group of
// four waves owns 64 consecutive sites: wave mu forms the forward and backward term of direction mu for all
// of them (both steps' loads in flight together), the partial sums meet in LDS, and waves 0 and 1 finish one
// chiral half each (clover block, xpay, store).  Four times the waves and two steps instead of eight in a
// chain.  Same storage and admission as the plane-grid kernel (12-real links, real boundary phases, 32-bit
// offsets); the terms are summed per direction first, so results differ from it by rounding.
#pragma once
#include "hop_fast.h"

namespace cmx {

// one direction of one site, forward and backward, into acc
template <int P, int MU, int ISIGN>
__device__ __forceinline__ void split_dir(const HopLaunch& h, int i, int jf, int jb, bool lastf, bool lastb,
                                          typename FastReal<P>::T (&acc)[24]) {
  constexpr int SB = P == P16 ? 48 : (P == P32 ? 96 : 192);
  constexpr int LB = P == P16 ? 24 : (P == P32 ? 48 : 96);
  const int Vh = h.g.Vh;
  const __amdgpu_buffer_rsrc_t rin = make_rsrc(h.in, (unsigned)(SB * h.in_stride));
  const __amdgpu_buffer_rsrc_t rnin = make_rsrc(h.in_nrm, (unsigned)(4 * h.in_stride));
  const __amdgpu_buffer_rsrc_t rlf =
      make_rsrc(static_cast<const char*>(h.gauge[h.cb]) + (size_t)MU * LB * Vh, (unsigned)(LB * Vh));
  const __amdgpu_buffer_rsrc_t rlb =
      make_rsrc(static_cast<const char*>(h.gauge[1 - h.cb]) + (size_t)MU * LB * Vh, (unsigned)(LB * Vh));
  FastSpinor<P> sf, sb;
  FastLink<P> lf, lb;
  fast_load_spinor<P>(rin, rnin, h.in_stride, jf, sf);
  fast_load_link<P>(rlf, Vh, i, lf);
  fast_load_spinor<P>(rin, rnin, h.in_stride, jb, sb);
  fast_load_link<P>(rlb, Vh, jb, lb);
  const float gf = lastf ? h.sgn[MU][1] : h.sgn[MU][0], gb = lastb ? h.sgn[MU][1] : h.sgn[MU][0];
  if constexpr (P == P16) {
    fast_step_h<MU, true, ISIGN>(sf, lf, gf, acc);
    fast_step_h<MU, false, ISIGN>(sb, lb, gb, acc);
  } else {
    fast_step<P, MU, true, ISIGN>(sf, lf, gf, acc);
    fast_step<P, MU, false, ISIGN>(sb, lb, gb, acc);
  }
}

// Half of a fermion (chirality b: complex 6b .. 6b+5) of site i
template <int P, typename R>
__device__ __forceinline__ void half_load(const void* base, const float* nrm, int stride, int i, int b, R (&s)[12]) {
  if constexpr (P == P64) {
    const double2* q = static_cast<const double2*>(base);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const double2 v = q[(size_t)(6 * b + k) * stride + i];
      s[2 * k] = v.x, s[2 * k + 1] = v.y;
    }
  } else if constexpr (P == P32) {
    const float4* q = static_cast<const float4*>(base);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float4 v = q[(size_t)(3 * b + k) * stride + i];
      s[4 * k] = v.x, s[4 * k + 1] = v.y, s[4 * k + 2] = v.z, s[4 * k + 3] = v.w;
    }
  } else {  // chunk 2b (four complex) and half of chunk 1 (two complex); half 1 starts with the latter
    H8x w;
    H4x v;
    w.u = static_cast<const uint4*>(base)[(size_t)(2 * b) * stride + i];
    v.u = static_cast<const uint2*>(base)[2 * ((size_t)stride + i) + b];
    const float n = nrm[i];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float2 f = __half22float2(w.h[k]);
      s[(b ? 4 : 0) + 2 * k] = f.x * n, s[(b ? 4 : 0) + 2 * k + 1] = f.y * n;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float2 f = __half22float2(v.h[k]);
      s[(b ? 0 : 8) + 2 * k] = f.x * n, s[(b ? 0 : 8) + 2 * k + 1] = f.y * n;
    }
  }
}

// m: largest |component| of the whole site (FP16 storage)
template <int P, typename R>
__device__ __forceinline__ void half_store(void* base, float* nrm, int stride, int i, int b, const R (&s)[12], float m) {
  if constexpr (P == P64) {
    double2* q = static_cast<double2*>(base);
#pragma unroll
    for (int k = 0; k < 6; ++k) q[(size_t)(6 * b + k) * stride + i] = make_double2(s[2 * k], s[2 * k + 1]);
  } else if constexpr (P == P32) {
    float4* q = static_cast<float4*>(base);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      q[(size_t)(3 * b + k) * stride + i] = make_float4(s[4 * k], s[4 * k + 1], s[4 * k + 2], s[4 * k + 3]);
  } else {
    const bool keep = m >= __FLT_MIN__;  // as SpinorIO<P16>::store
    const float inv = keep ? 1.0f / m : 0.f;
    if (b == 0) nrm[i] = keep ? m : 0.f;
    H8x w;
    H4x v;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w.h[k] = __floats2half2_rn(s[(b ? 4 : 0) + 2 * k] * inv, s[(b ? 4 : 0) + 2 * k + 1] * inv);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      v.h[k] = __floats2half2_rn(s[(b ? 0 : 8) + 2 * k] * inv, s[(b ? 0 : 8) + 2 * k + 1] * inv);
    static_cast<uint4*>(base)[(size_t)(2 * b) * stride + i] = w.u;
    static_cast<uint2*>(base)[2 * ((size_t)stride + i) + b] = v.u;
  }
}

// out = (L + D + L^dag) in on one chiral block; c = {diag[6], offd[15] complex}
template <typename R> __device__ __forceinline__ void half_clover(const R (&c)[36], const R (&in)[12], R (&out)[12]) {
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    R re = c[i] * in[2 * i], im = c[i] * in[2 * i + 1];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      if (j == i) continue;
      const R pr = in[2 * j], pi = in[2 * j + 1];
      const int e = j < i ? 6 + 2 * (i * (i - 1) / 2 + j) : 6 + 2 * (j * (j - 1) / 2 + i);
      const R ci = j < i ? c[e + 1] : -c[e + 1];
      re += c[e] * pr - ci * pi;
      im += c[e] * pi + ci * pr;
    }
    out[2 * i] = re, out[2 * i + 1] = im;
  }
}

template <int P, int ISIGN, int EPI, int NORM>
__device__ __forceinline__ void hop_split_body(const HopLaunch& h, int blk, int nblk) {
  using R = typename FastReal<P>::T;
  __shared__ R part[4][24][64];
  __shared__ float mx[2][64];
  if (h.skip && *h.skip) return;
  if (h.run && !*h.run) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = xcd_range(blk, nblk) * 64 + lane;
  const bool in = i < h.g.Vh;
  R acc[24];
#pragma unroll
  for (int k = 0; k < 24; ++k) acc[k] = 0;
  if (in) {
    const int Lxh = h.g.Lxh, Ly = h.g.L[1], Lz = h.g.L[2], Lt = h.g.L[3];
    // Vh < 2^24: the float quotient is off by one at most
    auto div = [](int n, int d, float inv, int& rem) {
      int q = (int)((float)n * inv);
      rem = n - q * d;
      if (rem < 0) --q, rem += d;
      if (rem >= d) ++q, rem -= d;
      return q;
    };
    int xh, y, z;
    const int r0 = div(i, Lxh, h.inv_lxh, xh), r1 = div(r0, Ly, h.inv_ly, y), t = div(r1, Lz, h.inv_lz, z);
    const int x = 2 * xh + ((h.cb + y + z + t) & 1);
    const int Pl = Lxh * Ly;
    switch (w) {
      case 0: {
        const int xp = (x + 1 == 2 * Lxh) ? 0 : x + 1, xm = (x == 0) ? 2 * Lxh - 1 : x - 1;
        split_dir<P, 0, ISIGN>(h, i, i - xh + (xp >> 1), i - xh + (xm >> 1), x == 2 * Lxh - 1, x == 0, acc);
        break;
      }
      case 1:
        split_dir<P, 1, ISIGN>(h, i, i + (y + 1 == Ly ? -y : 1) * Lxh, i + (y == 0 ? Ly - 1 : -1) * Lxh, y == Ly - 1,
                               y == 0, acc);
        break;
      case 2:
        split_dir<P, 2, ISIGN>(h, i, i + (z + 1 == Lz ? -z : 1) * Pl, i + (z == 0 ? Lz - 1 : -1) * Pl, z == Lz - 1,
                               z == 0, acc);
        break;
      default:
        split_dir<P, 3, ISIGN>(h, i, i + (t + 1 == Lt ? -t : 1) * Lz * Pl, i + (t == 0 ? Lt - 1 : -1) * Lz * Pl,
                               t == Lt - 1, t == 0, acc);
        break;
    }
  }
#pragma unroll
  for (int k = 0; k < 24; ++k) part[w][k][lane] = acc[k];
  __syncthreads();
  double nsq = 0, dre = 0, dim = 0;
  const bool fin = in && w < 2;
  R out[12];
  if (fin) {
    R s[12];
#pragma unroll
    for (int k = 0; k < 12; ++k)
      s[k] = (R)h.b * ((part[0][12 * w + k][lane] + part[1][12 * w + k][lane]) +
                       (part[2][12 * w + k][lane] + part[3][12 * w + k][lane]));
    R c[36], xs[12];
    if constexpr (EPI == EPI_CLOV || EPI == EPI_CLOV_XPAY) CloverBlockIO<P>::load(h.clov, h.g.Vh, i, w, c);
    if constexpr (EPI == EPI_XPAY || EPI == EPI_CLOV_XPAY) half_load<P>(h.x, h.x_nrm, h.x_stride, i, w, xs);
    if constexpr (EPI == EPI_NONE) {
#pragma unroll
      for (int k = 0; k < 12; ++k) out[k] = s[k];
    } else if constexpr (EPI == EPI_CLOV) {
      half_clover<R>(c, s, out);
    } else if constexpr (EPI == EPI_XPAY) {
#pragma unroll
      for (int k = 0; k < 12; ++k) out[k] = fmar((R)h.a, xs[k], s[k]);
    } else {
      half_clover<R>(c, xs, out);
#pragma unroll
      for (int k = 0; k < 12; ++k) out[k] += s[k];
    }
    if constexpr (NORM) {
      auto dot = [&](const R(&u)[12], const R(&v)[12]) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          const double ur = u[2 * k], ui = u[2 * k + 1], vr = v[2 * k], vi = v[2 * k + 1];
          dre += ur * vr + ui * vi;
          dim += ur * vi - ui * vr;
        }
      };
      if constexpr (NORM == NORM_UPDATE) {  // as hop_finish, on half a site
        constexpr int PY = P == P64 ? P64 : P32;
        R y[12];
        const R cf = (R)*h.coef;
        half_load<PY>(h.y, nullptr, h.y_stride, i, w, y);
#pragma unroll
        for (int k = 0; k < 12; ++k) out[k] = y[k] + cf * out[k];
        half_store<PY>(h.y, nullptr, h.y_stride, i, w, out, 0.f);
      } else if constexpr (NORM == NORM_DOT_Y) {
        R y[12];
        half_load<P>(h.y, h.y_nrm, h.y_stride, i, w, y);
        dot(y, out);
      } else if constexpr (NORM == NORM_DOT_X) {
        dot(out, xs);
      }
#pragma unroll
      for (int k = 0; k < 12; ++k) nsq += (double)out[k] * (double)out[k];
    }
  }
  float m = 0;
  if constexpr (P == P16 && NORM != NORM_UPDATE) {
    if (fin) {
#pragma unroll
      for (int k = 0; k < 12; ++k) m = fmaxf(m, fabsf(out[k]));
      mx[w][lane] = m;
    }
    __syncthreads();
    if (fin) m = fmaxf(m, mx[1 - w][lane]);
  }
  if constexpr (NORM != NORM_UPDATE)
    if (fin) half_store<P>(h.out, h.out_nrm, h.out_stride, i, w, out, m);
  if constexpr (NORM) write_norm_partials<NORM>(h, blk, nsq, dre, dim);
}

template <int P, int ISIGN, int EPI, int NORM>
__global__ void __launch_bounds__(256) k_hop_split(HopLaunch h) {
  hop_split_body<P, ISIGN, EPI, NORM>(h, blockIdx.x, gridDim.x);
}
template <int P, int ISIGN, int EPI, int NORM>
__global__ void __launch_bounds__(256) k_hop_split_b(const HopLaunch* __restrict__ tab, const int4* __restrict__ map) {
  const int4 m = map[blockIdx.x];
  if (m.x < 0) return;  // alignment padding of the batched grid
  hop_split_body<P, ISIGN, EPI, NORM>(tab[m.x], m.y, m.z);
}

template <int P> void launch_hop_split_t(const HopLaunch& h, hipStream_t s, const BatchGrid* bg) {
  const dim3 grid((h.g.Vh + 63) / 64);
  const int norm = hop_norm(h);
#define CMX_HOPS_GO(IS, EP, NM)                                                                     \
  if (bg)                                                                                           \
    hipLaunchKernelGGL((k_hop_split_b<P, IS, EP, NM>), dim3(bg->nblocks), dim3(256), 0, s,          \
                       static_cast<const HopLaunch*>(bg->tab), bg->map);                            \
  else                                                                                              \
    hipLaunchKernelGGL((k_hop_split<P, IS, EP, NM>), grid, dim3(256), 0, s, h);
#define CMX_HOPS_CASE(IS, EP)                                                                       \
  if (h.isign == IS && h.epi == EP) {                                                               \
    if (norm == NORM_ONLY) {                                                                        \
      CMX_HOPS_GO(IS, EP, NORM_ONLY)                                                                \
    } else {                                                                                        \
      CMX_HOPS_GO(IS, EP, NORM_NONE)                                                                \
    }                                                                                               \
    return;                                                                                         \
  }
#define CMX_HOPS_TAIL(IS, EP, NM)                                                                   \
  if (h.isign == IS && h.epi == EP && norm == NM) {                                                 \
    CMX_HOPS_GO(IS, EP, NM)                                                                         \
    return;                                                                                         \
  }
  CMX_HOPS_TAIL(-1, EPI_XPAY, NORM_UPDATE)
  CMX_HOPS_TAIL(-1, EPI_CLOV_XPAY, NORM_UPDATE)
  CMX_HOPS_TAIL(1, EPI_XPAY, NORM_DOT_X)
  CMX_HOPS_TAIL(1, EPI_XPAY, NORM_DOT_Y)
  CMX_HOPS_TAIL(1, EPI_CLOV_XPAY, NORM_DOT_X)
  CMX_HOPS_TAIL(1, EPI_CLOV_XPAY, NORM_DOT_Y)
  CMX_HOPS_TAIL(-1, EPI_XPAY, NORM_DOT_X)
  CMX_HOPS_TAIL(-1, EPI_XPAY, NORM_DOT_Y)
  CMX_HOPS_TAIL(-1, EPI_CLOV_XPAY, NORM_DOT_X)
  CMX_HOPS_TAIL(-1, EPI_CLOV_XPAY, NORM_DOT_Y)
#undef CMX_HOPS_TAIL
  if (norm > NORM_ONLY) throw Error(CMX_ERR_ARG, "launch_hop_split: tail not instantiated");
  CMX_HOPS_CASE(1, EPI_NONE)
  CMX_HOPS_CASE(1, EPI_CLOV)
  CMX_HOPS_CASE(1, EPI_XPAY)
  CMX_HOPS_CASE(1, EPI_CLOV_XPAY)
  CMX_HOPS_CASE(-1, EPI_NONE)
  CMX_HOPS_CASE(-1, EPI_CLOV)
  CMX_HOPS_CASE(-1, EPI_XPAY)
  CMX_HOPS_CASE(-1, EPI_CLOV_XPAY)
#undef CMX_HOPS_CASE
#undef CMX_HOPS_GO
  throw Error(CMX_ERR_ARG, "launch_hop_split: bad isign/epilogue");
}

}  // namespace cmx
