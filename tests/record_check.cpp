// Host-only: the recorded launches of hopping kernels, and the kernels that a launch-shape request admits.
// Prints one line per case; tests/test_batch_record_cpu.py reads them.
#include <cstdio>
#include <cstring>

#include "batch.h"

int main() {
  double part = 0, coef = 0;
  for (int tail : {-1, (int)cmx::TAIL_NONE, (int)cmx::TAIL_DOT_X, (int)cmx::TAIL_DOT_Y, (int)cmx::TAIL_UPDATE}) {
    cmx::HopLaunch h;
    std::memset(&h, 0, sizeof(h));
    h.prec = cmx::P32;
    h.recon = 12;
    h.isign = -1;
    h.epi = cmx::EPI_XPAY;
    h.block = 64;
    h.g.Vh = 64;
    if (tail >= 0) {
      h.partials = &part;
      h.tail = tail;
      h.coef = &coef;
    }
    cmx::Recorder r;
    cmx::record_hop(r, h);
    std::printf("key %d", tail);
    for (int k : r.recs[0].key) std::printf(" %d", k);
    std::printf("\n");
  }
  const int lat[][4] = {{32, 32, 32, 64}, {36, 36, 36, 60}, {40, 40, 40, 60}, {48, 48, 48, 96}, {64, 64, 64, 48}, {16, 16, 16, 32}};
  for (const auto& L : lat)
    for (int prec : {(int)cmx::P64, (int)cmx::P32, (int)cmx::P16})
      for (int which : {0, 1}) {
        cmx::Geom g;
        std::memset(&g, 0, sizeof(g));
        for (int m = 0; m < 4; ++m) g.L[m] = L[m];
        g.Lxh = L[0] / 2;
        g.Vh = L[0] / 2 * L[1] * L[2] * L[3];
        const cmx::HopConfig c = cmx::hop_default_config(g, prec, true, which);
        std::printf("shape %d %d %d %d %d %d %d\n", L[0], L[3], prec, which, c.block, c.tiled, c.fast);
      }
  return 0;
}
