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
  return 0;
}
