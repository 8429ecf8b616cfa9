// Learned preconditioner, host side: weights and their initialisation, upload in the MFMA operand
// order, the forward application used by the flexible solver, the loss gradient, and training on
// (residual, error) pairs generated by the plain CG solver on the device.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <random>

#include "learned.h"
#include "op.h"

namespace cmx {

PtcBlock::PtcBlock()
    : W1((size_t)PTC_CH * 4 * PTC_PATHS * 4),
      W2((size_t)PTC_PATHS * 4 * PTC_CH * 4),
      W0(16),
      m1(2 * W1.size()), v1(2 * W1.size()),
      m2(2 * W2.size()), v2(2 * W2.size()),
      m0(2 * W0.size()), v0(2 * W0.size()) {}

std::vector<PtcBlock::cf> PtcBlock::contracted() const {
  const int R = PTC_PATHS * 4, K = PTC_CH * 4;  // 32, 64
  std::vector<cf> Wc((size_t)R * R, cf(0));
  for (int q = 0; q < R; ++q)
    for (int k = 0; k < K; ++k) {
      const cf a = W2[(size_t)q * K + k];
      if (a == cf(0)) continue;
      for (int p = 0; p < R; ++p) Wc[(size_t)q * R + p] += a * W1[(size_t)k * R + p];
    }
  return Wc;
}

void PtcBlock::reset_moments() {
  for (auto* m : {&m1, &v1, &m2, &v2, &m0, &v0}) std::fill(m->begin(), m->end(), 0.f);
}

namespace {

using cd = std::complex<double>;
using cf = std::complex<float>;

// DeGrand-Rossi gamma matrices (the spin basis of the fermion layout)
cd gamma_dr(int mu, int s, int t) {
  const cd I(0, 1);
  static const int pos[4][4] = {{3, 2, 1, 0}, {3, 2, 1, 0}, {2, 3, 0, 1}, {2, 3, 0, 1}};
  if (pos[mu][s] != t) return 0;
  switch (mu) {
    case 0: return (s < 2) ? I : -I;
    case 1: return (s == 0 || s == 3) ? cd(-1) : cd(1);
    case 2: return (s == 0 || s == 3) ? I : -I;
    default: return 1;
  }
}

// (1 + sigma_p gamma_mu) of path p (sigma = -1 forward, +1 backward): twice the path's projector
cd proj2(int p, int s, int t) {
  const int mu = p / 2;
  const double sg = (p % 2 == 0) ? -1.0 : 1.0;
  return (s == t ? cd(1) : cd(0)) + sg * gamma_dr(mu, s, t);
}

unsigned short bf16_rne(float x) {
  unsigned u;
  std::memcpy(&u, &x, 4);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

// Half-spinor coordinates of path p (mu = p / 2, sigma = -1 forward, +1 backward): the projector
// Pi_p = (1 + sigma gamma_mu)/2 = R_p Phat_p with Phat_p = (1/2)[1, sigma B] (2x4) and R_p = [1; sigma B^dag]
// (4x2), B the upper-right 2x2 block of gamma_mu
cd phat(int p, int sp, int s) {  // Phat_p[sp][s]
  const int mu = p / 2;
  const double sg = (p % 2 == 0) ? -1.0 : 1.0;
  if (s < 2) return s == sp ? cd(0.5) : cd(0);
  return 0.5 * sg * gamma_dr(mu, sp, s);
}
cd rrec(int p, int s, int sp) {  // R_p[s][sp]
  const int mu = p / 2;
  const double sg = (p % 2 == 0) ? -1.0 : 1.0;
  if (s < 2) return s == sp ? cd(1) : cd(0);
  return sg * std::conj(gamma_dr(mu, sp, s));  // (B^dag)[s-2][sp] = conj(B[sp][s-2])
}

// Wh = Phat_q Wc R_p (16 x 16, rows q*2+s', columns p*2+t') from Wc (32 x 32, rows q*4+s, columns p*4+t)
std::vector<cd> half_weights(const std::vector<cf>& Wc) {
  std::vector<cd> Wh(16 * 16, cd(0));
  for (int q = 0; q < 8; ++q)
    for (int p = 0; p < 8; ++p)
      for (int sq = 0; sq < 2; ++sq)
        for (int tp = 0; tp < 2; ++tp) {
          cd acc = 0;
          for (int s = 0; s < 4; ++s)
            for (int t = 0; t < 4; ++t)
              acc += phat(q, sq, s) * cd(Wc[(size_t)(q * 4 + s) * 32 + p * 4 + t]) * rrec(p, t, tp);
          Wh[(size_t)(q * 2 + sq) * 16 + p * 2 + tp] = acc;
        }
  return Wh;
}

struct PtcBuffers {
  DevBuf T, dT, G, gpart, w0part, S;
  DevBuf Afr[PTC_MAX_BLOCKS], W0[PTC_MAX_BLOCKS];    // each block's Wh (MFMA A operand) and W0
  DevBuf Afa[PTC_MAX_BLOCKS], W0a[PTC_MAX_BLOCKS];   // the adjoints: (1/2) Wh^dag and W0^dag
  std::unique_ptr<Vec> mid[3][2];                    // block outputs between blocks, per precision
  std::unique_ptr<Vec> u[3][PTC_MAX_BLOCKS];         // block inputs kept for the gradient
  std::unique_ptr<Vec> dprev[3];                     // the loss gradient carried back through a block
  // several sources at once: a mixed field per source, block outputs per source
  std::vector<DevBuf> Gb;
  std::vector<std::unique_ptr<Vec>> midb[3][2];
  int vh = 0;
  // inference path per precision: 0/1 fused (registers/LDS), 2 unfused, 3/4 fused with streamed links
  int variant[3] = {-1, -1, -1};
};

PtcBuffers& ptc_buffers(Op& op) {
  if (!op.ptc) op.ptc = std::shared_ptr<void>(new PtcBuffers(), [](void* q) { delete static_cast<PtcBuffers*>(q); });
  auto* pb = static_cast<PtcBuffers*>(op.ptc.get());
  if (pb->vh != op.Vh) {
    const size_t nblk = (op.Vh + 31) / 32;
    pb->T.alloc(nblk * 3 * 4 * 64 * 4 * 2);
    pb->dT.alloc(nblk * 3 * 4 * 64 * 4 * 2);
    pb->G.alloc((size_t)8 * 3 * op.Vh * 8);
    for (int k = 0; k < PTC_MAX_BLOCKS; ++k) {
      pb->Afr[k].alloc(4 * 64 * 4 * 2);
      pb->W0[k].alloc(32 * sizeof(float));
      pb->Afa[k].alloc(4 * 64 * 4 * 2);
      pb->W0a[k].alloc(32 * sizeof(float));
    }
    pb->gpart.alloc((size_t)ptc_waves() * 64 * 16 * sizeof(float));
    pb->w0part.alloc((size_t)((op.Vh + 255) / 256) * 32 * sizeof(double));
    pb->S.alloc(1024 * sizeof(double));
    // tiles beyond Vh (when Vh is not a multiple of 32) must read as zero in the gradient sum
    CMX_HIP(hipMemsetAsync(pb->T.p, 0, pb->T.bytes, op.stream));
    CMX_HIP(hipMemsetAsync(pb->dT.p, 0, pb->dT.bytes, op.stream));
    for (auto& v : pb->mid) v[0].reset(), v[1].reset();
    for (auto& v : pb->u)
      for (auto& w : v) w.reset();
    for (auto& v : pb->dprev) v.reset();
    pb->Gb.clear();
    for (auto& v : pb->midb) v[0].clear(), v[1].clear();
    pb->vh = (int)op.Vh;
  }
  return *pb;
}

Vec& scratch_vec(std::unique_ptr<Vec>& slot, int prec, int n) {
  if (!slot || slot->prec != prec || slot->n != n) slot.reset(new Vec(prec, n));
  return *slot;
}

// the MFMA A-operand order of the real embedding [[Wr, -Wi], [Wi, Wr]] of a 16x16 complex matrix
std::vector<unsigned short> a_operand(const std::vector<cd>& W) {
  auto A = [&](int r, int k) -> float {
    const cd w = W[(size_t)(r & 15) * 16 + (k & 15)];
    if (r < 16) return (float)(k < 16 ? w.real() : -w.imag());
    return (float)(k < 16 ? w.imag() : w.real());
  };
  std::vector<unsigned short> afr(4 * 64 * 4);
  for (int ks = 0; ks < 4; ++ks)
    for (int l = 0; l < 64; ++l)
      for (int j = 0; j < 4; ++j) afr[(ks * 64 + l) * 4 + j] = bf16_rne(A(l & 31, 8 * ks + 4 * (l >> 5) + j));
  return afr;
}

// Uploads every block's Wh (as the MFMA A operand) and W0, and their adjoints, when the network changed
// since the last upload
void ensure_weights(Op& op, PtcBuffers& b) {
  CMX_REQUIRE(op.net, CMX_ERR_ARG, "learned preconditioner: no network attached to the operator");
  if (op.net_version == op.net->version) return;
  const int nb = (int)op.net->blk.size();
  CMX_REQUIRE(nb >= 1 && nb <= PTC_MAX_BLOCKS, CMX_ERR_ARG, "learned preconditioner: 1..4 blocks");
  std::vector<std::vector<unsigned short>> keep;  // host copies alive until the copies have run
  std::vector<std::vector<float>> keepf;
  for (int k = 0; k < nb; ++k) {
    const PtcBlock& B = op.net->blk[k];
    const std::vector<cd> Wh = half_weights(B.contracted());
    std::vector<cd> Wa(16 * 16);
    for (int m = 0; m < 16; ++m)
      for (int j = 0; j < 16; ++j) Wa[(size_t)m * 16 + j] = 0.5 * std::conj(Wh[(size_t)j * 16 + m]);
    keep.push_back(a_operand(Wh));
    CMX_HIP(hipMemcpyAsync(b.Afr[k].p, keep.back().data(), keep.back().size() * 2, hipMemcpyHostToDevice, op.stream));
    keep.push_back(a_operand(Wa));
    CMX_HIP(hipMemcpyAsync(b.Afa[k].p, keep.back().data(), keep.back().size() * 2, hipMemcpyHostToDevice, op.stream));
    std::vector<float> w0(32), w0a(32);
    for (int s = 0; s < 4; ++s)
      for (int t = 0; t < 4; ++t) {
        const PtcBlock::cf w = B.W0[s * 4 + t], wt = std::conj(B.W0[t * 4 + s]);
        w0[2 * (s * 4 + t)] = w.real();
        w0[2 * (s * 4 + t) + 1] = w.imag();
        w0a[2 * (s * 4 + t)] = wt.real();
        w0a[2 * (s * 4 + t) + 1] = wt.imag();
      }
    keepf.push_back(w0);
    CMX_HIP(hipMemcpyAsync(b.W0[k].p, keepf.back().data(), 32 * 4, hipMemcpyHostToDevice, op.stream));
    keepf.push_back(w0a);
    CMX_HIP(hipMemcpyAsync(b.W0a[k].p, keepf.back().data(), 32 * 4, hipMemcpyHostToDevice, op.stream));
    op.sync();  // the host vectors may move when keep grows
  }
  op.net_version = op.net->version;
}

PtcLaunch ptc_base(Op& op, int prec, PtcBuffers& b, int blk = 0) {
  op.ensure_prec(prec);
  const HopLaunch h = op.hop_base(prec);
  PtcLaunch L;
  std::memset(&L, 0, sizeof(L));
  L.g = h.g;
  L.prec = prec;
  L.recon = h.recon;
  L.gauge[0] = h.gauge[0];
  L.gauge[1] = h.gauge[1];
  std::memcpy(L.ph, h.ph, sizeof(L.ph));
  L.T = b.T.as<unsigned short>();
  L.dT = b.dT.as<unsigned short>();
  L.G = b.G.as<unsigned short>();
  L.Afr = b.Afr[blk].as<unsigned short>();
  L.W0 = b.W0[blk].as<float>();
  L.gpart = b.gpart.as<float>();
  L.w0part = b.w0part.as<double>();
  return L;
}

// one block: out = B_blk(in)
void forward_block(Op& op, int prec, int blk, const Vec& in, Vec& out) {
  CMX_REQUIRE(in.prec == prec && out.prec == prec, CMX_ERR_ARG, "learned preconditioner: precision mismatch");
  CMX_REQUIRE(op.eo(), CMX_ERR_UNSUPPORTED, "learned preconditioner: even-odd operators only");
  PtcBuffers& b = ptc_buffers(op);
  ensure_weights(op, b);
  PtcLaunch L = ptc_base(op, prec, b, blk);
  const VRef vi = in.view(), vo = out.view();
  L.in = vi.v, L.in_nrm = vi.nrm, L.in_stride = vi.stride;
  L.out = vo.v, L.out_nrm = vo.nrm, L.out_stride = vo.stride;
  auto gather_mix = [&](int variant) {
    if (variant == 2) {
      launch_ptc_gather(L, false, op.stream);
      launch_ptc_mix(L, op.stream);
    } else {
      launch_ptc_gather_mix(L, variant, op.stream);
    }
  };
  auto block = [&](int variant) {  // gather + mix, then the scatter (links streamed in variants 3, 4)
    gather_mix(variant);
    launch_ptc_scatter(L, false, op.stream, variant >= 3);
  };
  int& var = b.variant[prec];
  if (var < 0) {  // first use at this precision: time the five inference paths, keep the fastest
    hipEvent_t e0, e1;
    CMX_HIP(hipEventCreate(&e0));
    CMX_HIP(hipEventCreate(&e1));
    float best = 1e30f;
    for (int v = 0; v < 5; ++v) {
      block(v);  // warm-up
      CMX_HIP(hipEventRecord(e0, op.stream));
      for (int k = 0; k < 3; ++k) block(v);
      CMX_HIP(hipEventRecord(e1, op.stream));
      CMX_HIP(hipEventSynchronize(e1));
      float ms = 0;
      CMX_HIP(hipEventElapsedTime(&ms, e0, e1));
      if (ms < best) best = ms, var = v;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  }
  block(var);
  CMX_HIP(hipGetLastError());
}

// out = P(in) = B_{n-1}(... B_0(in)); with keep_inputs every block's input stays in the buffers' u[prec][k]
// (u[prec][0] is not used: block 0's input is `in`)
void forward(Op& op, int prec, const Vec& in, Vec& out, bool keep_inputs = false) {
  CMX_REQUIRE(op.net, CMX_ERR_ARG, "learned preconditioner: no network attached to the operator");
  const int nb = (int)op.net->blk.size();
  const int n = op.subset_sites();
  PtcBuffers& b = ptc_buffers(op);
  const Vec* src = &in;
  for (int k = 0; k < nb; ++k) {
    Vec* dst = &out;
    if (k < nb - 1)
      dst = keep_inputs ? &scratch_vec(b.u[prec][k + 1], prec, n) : &scratch_vec(b.mid[prec][k & 1], prec, n);
    forward_block(op, prec, k, *src, *dst);
    src = dst;
  }
}

struct Grad {
  double loss = 0, enorm = 0;
  std::vector<std::vector<cd>> S;   // per block: 32 x 32, d loss / d conj(Wc)
  std::vector<std::vector<cd>> S0;  // per block: 4 x 4,  d loss / d conj(W0)
};

// The block's weight gradients from its input u and the loss gradient delta at its output:
// Sh = sum_{y,c} dgh th^dag (the transports of u against the adjoint scatter of delta) mapped to
// d/d conj(Wc), and sum_x delta u^dag for W0
void block_grad(Op& op, int prec, PtcBuffers& b, int blk, const Vec& u, const Vec& delta, std::vector<cd>& S,
                std::vector<cd>& S0) {
  PtcLaunch L = ptc_base(op, prec, b, blk);
  const VRef uv = u.view(), dv = delta.view();
  L.in = uv.v, L.in_nrm = uv.nrm, L.in_stride = uv.stride;  // th = transports of the block's input
  L.T = b.T.as<unsigned short>();
  launch_ptc_gather(L, false, op.stream);
  L.in = dv.v, L.in_nrm = dv.nrm, L.in_stride = dv.stride;  // dgh = adjoint scatter of delta
  L.T = b.dT.as<unsigned short>();
  launch_ptc_gather(L, true, op.stream);
  L.T = b.T.as<unsigned short>();
  L.dT = b.dT.as<unsigned short>();
  launch_ptc_grad(L, b.S.as<double>(), op.stream);
  L.in = uv.v, L.in_nrm = uv.nrm, L.in_stride = uv.stride;
  L.out = dv.v, L.out_nrm = dv.nrm, L.out_stride = dv.stride;
  const int nbw = launch_w0_grad(L, op.stream);
  launch_colsum(b.w0part.as<double>(), nbw, 32, op.state_S.as<double>() + S_KRY, 0, op.stream);
  CMX_HIP(hipGetLastError());
  std::vector<double> P(1024);
  CMX_HIP(hipMemcpyAsync(P.data(), b.S.p, 1024 * sizeof(double), hipMemcpyDeviceToHost, op.stream));
  CMX_HIP(hipMemcpyAsync(op.hS + S_KRY, static_cast<double*>(op.state_S.p) + S_KRY, 32 * sizeof(double),
                         hipMemcpyDeviceToHost, op.stream));
  op.sync();
  // Pm (32 x 32 real) from the MFMA accumulator layout, then Sh = d/d conj(Wh) (16 x 16 complex)
  std::vector<double> Pm(32 * 32);
  for (int l = 0; l < 64; ++l)
    for (int r = 0; r < 16; ++r) {
      const int row = 8 * (r / 4) + 4 * (l / 32) + (r % 4), col = l % 32;
      Pm[(size_t)row * 32 + col] = P[(size_t)l * 16 + r];
    }
  std::vector<cd> Sh(16 * 16);
  for (int m = 0; m < 16; ++m)
    for (int k = 0; k < 16; ++k) {
      const double re = Pm[(size_t)m * 32 + k] + Pm[(size_t)(16 + m) * 32 + 16 + k];
      const double im = Pm[(size_t)(16 + m) * 32 + k] - Pm[(size_t)m * 32 + 16 + k];
      Sh[(size_t)m * 16 + k] = cd(re, im);
    }
  // Wh = Phat_q Wc R_p, so d/d conj(Wc) = Phat_q^dag Sh R_p^dag
  S.assign(32 * 32, cd(0));
  for (int q = 0; q < 8; ++q)
    for (int p = 0; p < 8; ++p)
      for (int s = 0; s < 4; ++s)
        for (int t = 0; t < 4; ++t) {
          cd acc = 0;
          for (int sq = 0; sq < 2; ++sq)
            for (int tp = 0; tp < 2; ++tp)
              acc += std::conj(phat(q, sq, s)) * Sh[(size_t)(q * 2 + sq) * 16 + p * 2 + tp] * std::conj(rrec(p, t, tp));
          S[(size_t)(q * 4 + s) * 32 + p * 4 + t] = acc;
        }
  S0.resize(16);
  for (int k = 0; k < 16; ++k) S0[k] = cd(op.hS[S_KRY + 2 * k], op.hS[S_KRY + 2 * k + 1]);
}

// Loss and its gradients for every block; v, e, out, delta (and tmp) in precision prec (device vectors).
//   error norm    (tmp == nullptr): loss = |P v - e|^2,      normalisation |e|^2
//   residual norm (tmp != nullptr): loss = |M (P v - e)|^2,  normalisation |v|^2; with v = M e this is
//                                   |M P v - v|^2, and the output gradient is M^dag M (P v - e)
// Back-propagation: the gradient at block k's output is carried to its input by the block's adjoint
// B^dag d = W0^dag d + G^dag(Wh^dag S^dag d) (transports of the opposite paths, the same kernels).
Grad gradient(Op& op, int prec, const Vec& v, const Vec& e, Vec& out, Vec& delta, Vec* tmp = nullptr) {
  const int n = op.subset_sites();
  const int nb = blas_blocks(n);
  const int nblk = (int)op.net->blk.size();
  forward(op, prec, v, out, true);
  PtcBuffers& b = ptc_buffers(op);
  op.blas(B_XMY_NORM, {&delta, &out, &e});  // delta = P v - e
  op.finalize(nb, 1, PG_STORE, S_TR);
  if (tmp) {
    op.apply(prec, tmp->view(), delta.view(), +1, nullptr);   // M (P v - e)
    op.blas(B_NORM2, {tmp});
    op.finalize(nb, 1, PG_STORE, S_TR);
    op.apply(prec, delta.view(), tmp->view(), -1, nullptr);   // M^dag M (P v - e)
    op.blas(B_NORM2, {&v});
  } else {
    op.blas(B_NORM2, {&e});
  }
  op.finalize(nb, 1, PG_STORE, S_TR + 1);
  CMX_HIP(hipMemcpyAsync(op.hS + S_TR, static_cast<double*>(op.state_S.p) + S_TR, 2 * sizeof(double),
                         hipMemcpyDeviceToHost, op.stream));
  op.sync();
  Grad g;
  g.loss = op.hS[S_TR];
  g.enorm = op.hS[S_TR + 1];
  g.S.resize(nblk);
  g.S0.resize(nblk);
  Vec* d = &delta;
  Vec* d2 = &scratch_vec(b.dprev[prec], prec, n);
  for (int k = nblk - 1; k >= 0; --k) {
    const Vec& u = k == 0 ? v : *b.u[prec][k];
    block_grad(op, prec, b, k, u, *d, g.S[k], g.S0[k]);
    if (k > 0) {  // d <- B_k^dag d: mix the adjoint-scattered d (still in dT) with (1/2) Wh^dag, then G^dag
      PtcLaunch L = ptc_base(op, prec, b, k);
      L.Afr = b.Afa[k].as<unsigned short>();
      L.T = b.dT.as<unsigned short>();
      launch_ptc_mix(L, op.stream);
      L.W0 = b.W0a[k].as<float>();
      const VRef dv = d->view(), ov = d2->view();
      L.in = dv.v, L.in_nrm = dv.nrm, L.in_stride = dv.stride;
      L.out = ov.v, L.out_nrm = ov.nrm, L.out_stride = ov.stride;
      launch_ptc_scatter(L, true, op.stream);
      CMX_HIP(hipGetLastError());
      std::swap(d, d2);
    }
  }
  return g;
}

void adam(std::vector<cf>& w, std::vector<float>& m, std::vector<float>& v, const std::vector<cd>& grad, double lr,
          long t) {
  const double b1 = 0.9, b2 = 0.999, eps = 1e-12;
  const double c1 = 1.0 - std::pow(b1, (double)t), c2 = 1.0 - std::pow(b2, (double)t);
  for (size_t i = 0; i < w.size(); ++i) {
    double gg[2] = {grad[i].real(), grad[i].imag()};
    double x[2] = {w[i].real(), w[i].imag()};
    for (int k = 0; k < 2; ++k) {
      float& mm = m[2 * i + k];
      float& vv = v[2 * i + k];
      mm = (float)(b1 * mm + (1 - b1) * gg[k]);
      vv = (float)(b2 * vv + (1 - b2) * gg[k] * gg[k]);
      x[k] -= lr * (mm / c1) / (std::sqrt(vv / c2) + eps);
    }
    w[i] = cf((float)x[0], (float)x[1]);
  }
}

}  // namespace

void learned_precond_apply(Op& op, int prec, const Vec& in, Vec& out) { forward(op, prec, in, out); }

// the batch's mixed fields and block outputs of m sources
static void batch_buffers(Op& op, PtcBuffers& b, int prec, int m) {
  const size_t gbytes = (size_t)8 * 3 * op.Vh * 8;
  while ((int)b.Gb.size() < m) b.Gb.emplace_back(gbytes);
  auto &mid0 = b.midb[prec][0], &mid1 = b.midb[prec][1];
  while ((int)mid0.size() < m) mid0.emplace_back(), mid1.emplace_back();
  for (int k = 0; k + 1 < (int)op.net->blk.size(); ++k)
    for (int i = 0; i < m; ++i) scratch_vec((k & 1) ? mid1[i] : mid0[i], prec, op.subset_sites());
}

void learned_reserve_batch(Op& op, int prec, int ns) {
  if (!op.net || !op.eo() || ptc_buffers(op).variant[prec] == 2) return;
  batch_buffers(op, ptc_buffers(op), prec, std::min(ns, PTC_MAXSRC));
}

void learned_precond_apply_batch(Op& op, int prec, const std::vector<const Vec*>& in, const std::vector<Vec*>& out) {
  const int ns = (int)in.size();
  CMX_REQUIRE(ns == (int)out.size() && ns >= 1, CMX_ERR_ARG, "learned preconditioner: batch size mismatch");
  CMX_REQUIRE(op.net, CMX_ERR_ARG, "learned preconditioner: no network attached to the operator");
  CMX_REQUIRE(op.eo(), CMX_ERR_UNSUPPORTED, "learned preconditioner: even-odd operators only");
  PtcBuffers& b = ptc_buffers(op);
  ensure_weights(op, b);
  const int var = b.variant[prec];
  if (ns == 1 || var < 0 || var == 2) {  // the inference path not chosen yet, or the unfused one: per source
    for (int i = 0; i < ns; ++i) forward(op, prec, *in[i], *out[i]);
    return;
  }
  const int n = op.subset_sites();
  const int nb = (int)op.net->blk.size();
  for (int off = 0; off < ns; off += PTC_MAXSRC) {
    const int m = std::min(PTC_MAXSRC, ns - off);
    batch_buffers(op, b, prec, m);
    auto &mid0 = b.midb[prec][0], &mid1 = b.midb[prec][1];
    std::vector<const Vec*> src(m);
    for (int i = 0; i < m; ++i) src[i] = in[off + i];
    for (int k = 0; k < nb; ++k) {
      std::vector<Vec*> dst(m);
      for (int i = 0; i < m; ++i)
        dst[i] = k == nb - 1 ? out[off + i] : &scratch_vec((k & 1) ? mid1[i] : mid0[i], prec, n);
      PtcLaunch L = ptc_base(op, prec, b, k);
      PtcBatch B;
      std::memset(&B, 0, sizeof(B));
      B.ns = m;
      for (int i = 0; i < m; ++i) {
        CMX_REQUIRE(src[i]->prec == prec && dst[i]->prec == prec && src[i]->n == n && dst[i]->n == n, CMX_ERR_ARG,
                    "learned preconditioner: precision mismatch");
        const VRef vi = src[i]->view(), vo = dst[i]->view();
        B.in[i] = vi.v, B.in_nrm[i] = vi.nrm;
        B.out[i] = vo.v, B.out_nrm[i] = vo.nrm;
        B.G[i] = b.Gb[i].as<unsigned short>();
        L.in_stride = vi.stride, L.out_stride = vo.stride;
      }
      launch_ptc_gather_mix_batch(L, B, var, op.stream);
      launch_ptc_scatter_batch(L, B, var >= 3, op.stream);
      CMX_HIP(hipGetLastError());
      for (int i = 0; i < m; ++i) src[i] = dst[i];
    }
  }
}

void learned_share(Op& from, Op& to) {
  to.net = from.net;
  if (!from.net) return;
  PtcBuffers& b = ptc_buffers(from);
  ensure_weights(from, b);
  to.ptc = from.ptc;
  to.net_version = from.net_version;
}

void net_set_variant(Op& op, int prec, int variant) {
  CMX_REQUIRE(prec >= 0 && prec <= 2 && variant >= -1 && variant <= 4, CMX_ERR_ARG, "net variant: bad argument");
  ptc_buffers(op).variant[prec] = variant;
}

void PtcBlock::set_identity() {
  std::fill(W1.begin(), W1.end(), cf(0));
  std::fill(W2.begin(), W2.end(), cf(0));
  std::fill(W0.begin(), W0.end(), cf(0));
  for (int p = 0; p < PTC_PATHS; ++p)
    for (int s = 0; s < 4; ++s)
      for (int t = 0; t < 4; ++t) W1[(size_t)(p * 4 + s) * 32 + p * 4 + t] = cf(proj2(p, s, t));
  for (int s = 0; s < 4; ++s) W0[s * 4 + s] = cf(1.0f);
  reset_moments();
}

void net_init_neumann(LearnedNet& net, double diag) {
  // Block 0: P = 1/a + (1/(4 a^3)) D_oe D_eo, the first two terms of the Neumann series of the even-odd
  // operator a - (1/(4a)) D_oe D_eo with the clover term replaced by its diagonal a = Nd + m.
  // Channel c < 8 carries path c with the projector (1 - gamma_mu) (forward) / (1 + gamma_mu).
  // Further blocks start as the identity, so the network starts as this Neumann approximation.
  PtcBlock& B = net.blk[0];
  std::fill(B.W1.begin(), B.W1.end(), cf(0));
  std::fill(B.W2.begin(), B.W2.end(), cf(0));
  std::fill(B.W0.begin(), B.W0.end(), cf(0));
  // the factor 1/(4 a^3) is split evenly between the two layers, so that both start at the same
  // scale (Adam's steps are per-parameter and scale-free)
  const double c2 = std::sqrt(1.0 / (4.0 * std::fabs(diag * diag * diag)));
  const double c1 = (diag > 0 ? 1.0 : -1.0) * c2;
  for (int p = 0; p < PTC_PATHS; ++p)
    for (int s = 0; s < 4; ++s)
      for (int t = 0; t < 4; ++t) {
        B.W1[(size_t)(p * 4 + s) * 32 + p * 4 + t] = cf(c1 * proj2(p, s, t));
        for (int c = 0; c < PTC_PATHS; ++c) B.W2[(size_t)(p * 4 + s) * 64 + c * 4 + t] = cf(c2 * proj2(p, s, t));
      }
  for (int s = 0; s < 4; ++s) B.W0[s * 4 + s] = cf((float)(1.0 / diag));
  B.reset_moments();
  for (size_t k = 1; k < net.blk.size(); ++k) net.blk[k].set_identity();
  net.step = 0;
  net.version++;
}

void net_set_depth(LearnedNet& net, int nblocks) {
  CMX_REQUIRE(nblocks >= 1 && nblocks <= PTC_MAX_BLOCKS, CMX_ERR_ARG, "net: 1..4 blocks");
  const size_t old = net.blk.size();
  net.blk.resize(nblocks);
  for (size_t k = old; k < net.blk.size(); ++k) net.blk[k].set_identity();
  net.version++;
}

// Host-array entry points for tests: out = P(in); gradient of |P(v) - e|^2 (Wc and W0)
void net_apply_host(Op& op, int prec, double* out, const double* in) {
  const int n = op.subset_sites();
  Vec a(prec, n), b(prec, n);
  op.pack(in, n, a);
  forward(op, prec, a, b);
  op.unpack(out, n, b);
  op.sync();
}

void net_grad_host(Op& op, int prec, const double* v, const double* e, double* loss, double* gwc, double* gw0) {
  const int n = op.subset_sites();
  Vec a(prec, n), b(prec, n), o(prec, n), d(prec, n);
  op.pack(v, n, a);
  op.pack(e, n, b);
  Grad g = gradient(op, prec, a, b, o, d);
  *loss = g.loss;
  for (size_t blk = 0; blk < g.S.size(); ++blk) {
    for (int k = 0; k < 32 * 32; ++k) {
      gwc[2 * (blk * 1024 + k)] = g.S[blk][k].real();
      gwc[2 * (blk * 1024 + k) + 1] = g.S[blk][k].imag();
    }
    for (int k = 0; k < 16; ++k) {
      gw0[2 * (blk * 16 + k)] = g.S0[blk][k].real();
      gw0[2 * (blk * 16 + k) + 1] = g.S0[blk][k].imag();
    }
  }
}

// Training (cmx_net_train): pairs (r_k, e_k) = (b - M x_k, x* - x_k) from the iterates x_k of plain
// FP64 CGNE (invcg2.cc:70-232) on Gaussian sources, then Adam on the residual-norm loss
// |M (P(r_k) - e_k)|^2 / |r_k|^2, one pair per step.  The residual norm weights the error modes by
// M^dag M: a short-range network can represent M^-1 on the high modes, which this loss targets, and
// leaves the low modes to the Krylov solver (an error-norm loss is dominated by the low modes and
// drives the weights towards a poor compromise).
void net_train(Op& op, const cmx_train_params& tp, cmx_train_result& res) {
  CMX_REQUIRE(op.net, CMX_ERR_ARG, "net_train: no network attached");
  CMX_REQUIRE(tp.n_sources >= 1 && tp.snapshot_every >= 1 && tp.epochs >= 0 && tp.max_pairs >= 1, CMX_ERR_ARG,
              "net_train: bad parameters");
  const int prec = tp.prec;
  CMX_REQUIRE(prec == P32 || prec == P16, CMX_ERR_ARG, "net_train: precision must be single or half");
  const int n = op.subset_sites();
  const int nb = blas_blocks(n);
  LearnedNet& net = *op.net;
  std::memset(&res, 0, sizeof(res));
  auto t0 = std::chrono::steady_clock::now();
  std::mt19937_64 rng(tp.seed);
  std::normal_distribution<double> gauss(0.0, 1.0);
  std::vector<std::unique_ptr<Vec>> R, E;  // pairs, precision prec
  std::vector<double> host((size_t)24 * n);
  Vec bsrc(P64, n), x(P64, n), r(P64, n), p(P64, n), mp(P64, n), mmp(P64, n), chi_t(P64, n), t(P64, n);
  std::vector<std::unique_ptr<Vec>> snaps;
  int* F = op.state_F.as<int>();
  (void)F;
  for (int src = 0; src < tp.n_sources && (int)R.size() < tp.max_pairs; ++src) {
    for (auto& z : host) z = gauss(rng) * 0.70710678118654752;
    op.pack(host.data(), n, bsrc);
    // CGNE on M^dag M x = M^dag b from x = 0, snapshots of x every snapshot_every iterations
    op.apply(P64, chi_t.view(), bsrc.view(), -1, nullptr);
    op.blas(B_ZERO, {&x});
    op.blas(B_COPY, {&r, &chi_t});
    op.blas(B_COPY, {&p, &chi_t});
    op.blas(B_NORM2, {&chi_t});
    op.finalize(nb, 1, PG_STORE, S_TR);
    CMX_HIP(hipMemcpyAsync(op.hS + S_TR, static_cast<double*>(op.state_S.p) + S_TR, sizeof(double),
                           hipMemcpyDeviceToHost, op.stream));
    op.sync();
    double c = op.hS[S_TR];
    const double stop = tp.solve_rsd * tp.solve_rsd * c;
    snaps.clear();
    for (int k = 0; k < 100000 && c > stop; ++k) {
      if (k > 0 && k % tp.snapshot_every == 0 && (int)(R.size() + snaps.size()) < tp.max_pairs &&
          (tp.pairs_per_source <= 0 || (int)snaps.size() < tp.pairs_per_source)) {
        snaps.emplace_back(new Vec(P64, n));
        op.blas(B_COPY, {snaps.back().get(), &x});
      }
      op.apply(P64, mp.view(), p.view(), +1, nullptr);
      op.apply(P64, mmp.view(), mp.view(), -1, nullptr);
      op.blas(B_NORM2, {&mp});
      op.finalize(nb, 1, PG_STORE, S_TR);
      CMX_HIP(hipMemcpyAsync(op.hS + S_TR, static_cast<double*>(op.state_S.p) + S_TR, sizeof(double),
                             hipMemcpyDeviceToHost, op.stream));
      op.sync();
      const double a = c / op.hS[S_TR];
      op.hS[S_TR + 2] = a;
      op.hS[S_TR + 3] = -a;
      CMX_HIP(hipMemcpyAsync(static_cast<double*>(op.state_S.p) + S_TR + 2, op.hS + S_TR + 2, 2 * sizeof(double),
                             hipMemcpyHostToDevice, op.stream));
      op.blas(B_AXPY, {&x, &p}, S_TR + 2);
      op.blas(B_AXPY_NORM, {&r, &mmp}, S_TR + 3);
      op.finalize(nb, 1, PG_STORE, S_TR);
      CMX_HIP(hipMemcpyAsync(op.hS + S_TR, static_cast<double*>(op.state_S.p) + S_TR, sizeof(double),
                             hipMemcpyDeviceToHost, op.stream));
      op.sync();
      const double cp = op.hS[S_TR];
      op.hS[S_TR + 2] = cp / c;
      CMX_HIP(hipMemcpyAsync(static_cast<double*>(op.state_S.p) + S_TR + 2, op.hS + S_TR + 2, sizeof(double),
                             hipMemcpyHostToDevice, op.stream));
      op.blas(B_XPAY, {&p, &r}, S_TR + 2);  // p = r + b p
      c = cp;
    }
    // pairs: r_k = b - M x_k, e_k = x* - x_k
    for (auto& s : snaps) {
      op.apply(P64, t.view(), s->view(), +1, nullptr);
      R.emplace_back(new Vec(prec, n));
      E.emplace_back(new Vec(prec, n));
      op.blas(B_XMY_NORM, {&mp, &bsrc, &t});
      op.blas(B_COPY, {R.back().get(), &mp});
      op.blas(B_XMY_NORM, {&mmp, &x, s.get()});
      op.blas(B_COPY, {E.back().get(), &mmp});
    }
  }
  op.sync();
  res.n_pairs = (int)R.size();
  auto t1 = std::chrono::steady_clock::now();
  res.gen_seconds = std::chrono::duration<double>(t1 - t0).count();
  if (R.empty()) return;
  Vec o(prec, n), d(prec, n), tm(prec, n);
  double norm0 = 1.0;  // raw weighting: one common scale, 1 / max_k |r_k|^2
  if (!tp.normalize) {
    double mx = 0;
    for (auto& rv : R) {
      op.blas(B_NORM2, {rv.get()});
      op.finalize(nb, 1, PG_STORE, S_TR);
      CMX_HIP(hipMemcpyAsync(op.hS + S_TR, static_cast<double*>(op.state_S.p) + S_TR, sizeof(double),
                             hipMemcpyDeviceToHost, op.stream));
      op.sync();
      mx = std::max(mx, op.hS[S_TR]);
    }
    norm0 = mx > 0 ? 1.0 / mx : 1.0;
  }
  std::vector<int> order(R.size());
  std::iota(order.begin(), order.end(), 0);
  const int R32 = PTC_PATHS * 4, K64 = PTC_CH * 4;
  // the objective as optimised: mean over the pairs of the weighted loss
  auto objective = [&]() {
    double sum = 0;
    for (size_t k = 0; k < R.size(); ++k) {
      Grad g = gradient(op, prec, *R[k], *E[k], o, d, &tm);
      sum += g.loss * (tp.normalize ? (g.enorm > 0 ? 1.0 / g.enorm : 1.0) : norm0);
    }
    return sum / (double)R.size();
  };
  res.loss_first = objective();
  for (int ep = 0; ep < tp.epochs; ++ep) {
    std::shuffle(order.begin(), order.end(), rng);
    for (int idx : order) {
      Grad g = gradient(op, prec, *R[idx], *E[idx], o, d, &tm);
      const double scale = tp.normalize ? (g.enorm > 0 ? 1.0 / g.enorm : 1.0) : norm0;
      // chain rule through each block's Wc = W2 W1: dW1 = W2^H S, dW2 = S W1^H
      ++net.step;
      for (size_t blk = 0; blk < net.blk.size(); ++blk) {
        PtcBlock& B = net.blk[blk];
        const std::vector<cd>& S = g.S[blk];
        std::vector<cd> g1((size_t)K64 * R32, cd(0)), g2((size_t)R32 * K64, cd(0)), g0(16);
        for (int k = 0; k < K64; ++k)
          for (int q = 0; q < R32; ++q) {
            const cd w2c = std::conj(cd(B.W2[(size_t)q * K64 + k]));
            if (w2c == cd(0)) continue;
            for (int pp = 0; pp < R32; ++pp) g1[(size_t)k * R32 + pp] += w2c * S[(size_t)q * R32 + pp] * scale;
          }
        for (int q = 0; q < R32; ++q)
          for (int k = 0; k < K64; ++k) {
            cd sum = 0;
            for (int pp = 0; pp < R32; ++pp) sum += S[(size_t)q * R32 + pp] * std::conj(cd(B.W1[(size_t)k * R32 + pp]));
            g2[(size_t)q * K64 + k] = sum * scale;
          }
        for (int k = 0; k < 16; ++k) g0[k] = g.S0[blk][k] * scale;
        adam(B.W1, B.m1, B.v1, g1, tp.lr, net.step);
        adam(B.W2, B.m2, B.v2, g2, tp.lr, net.step);
        adam(B.W0, B.m0, B.v0, g0, tp.lr, net.step);
      }
      net.version++;
      ++res.n_steps;
    }
    if (tp.verbose) std::printf("net_train: epoch %d done (%d steps)\n", ep, res.n_steps);
  }
  res.loss_last = objective();
  res.train_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t1).count();
}

}  // namespace cmx
