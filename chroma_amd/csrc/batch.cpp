// Launch recording and batched replay (see batch.h).
#include "batch.h"

#include <algorithm>
#include <cstring>
#include <string>

namespace cmx {

Recorder*& active_recorder() {
  thread_local Recorder* r = nullptr;
  return r;
}

namespace {
template <typename T> LaunchRec make_rec(int kind, const T& v, int nblocks) {
  LaunchRec r;
  r.kind = kind;
  r.nblocks = nblocks;
  r.bytes.resize(sizeof(T));
  std::memcpy(r.bytes.data(), &v, sizeof(T));
  return r;
}
}  // namespace

void record_hop(Recorder& r, const HopLaunch& h) {
  LaunchRec x = make_rec(REC_HOP, h, hop_num_blocks(h));
  // everything that selects the kernel template (hop_norm: partials and tail) and the work-group size
  const int k[8] = {h.prec, h.recon, h.fast, h.prefetch, h.isign, h.epi, h.partials ? 1 + h.tail : 0, h.block};
  std::memcpy(x.key, k, sizeof(k));
  r.recs.push_back(std::move(x));
}

void record_blas(Recorder& r, int op, const BlasLaunch& b, const int prec[4]) {
  LaunchRec x = make_rec(REC_BLAS, b, blas_blocks(b.n));
  const int k[8] = {op, prec[0], prec[1], prec[2], prec[3], 0, 0, 0};
  std::memcpy(x.key, k, sizeof(k));
  r.recs.push_back(std::move(x));
}

static int fin_partials(const LaunchRec& r) {
  FinLaunch f;
  std::memcpy(&f, r.bytes.data(), sizeof(f));
  return f.nb;
}

void record_fin(Recorder& r, const FinLaunch& f) { r.recs.push_back(make_rec(REC_FIN, f, 1)); }

void BatchPlan::build(const std::vector<Recorder>& recs) {
  st_.clear();
  mem_.clear();
  CMX_REQUIRE(!recs.empty(), CMX_ERR_ARG, "batch: no problems");
  // problems whose launches select the same kernels share batched grids; others get their own
  std::vector<std::vector<Recorder>> groups;
  auto alike = [](const Recorder& a, const Recorder& b) {
    if (a.recs.size() != b.recs.size()) return false;
    for (size_t j = 0; j < a.recs.size(); ++j)
      if (a.recs[j].kind != b.recs[j].kind || std::memcmp(a.recs[j].key, b.recs[j].key, sizeof(a.recs[j].key)) != 0)
        return false;
    return true;
  };
  for (const Recorder& r : recs) {
    CMX_REQUIRE(r.recs.size() == recs[0].recs.size(), CMX_ERR_ARG,
                "batch: the problems' kernel sequences differ in length");
    size_t k = 0;
    while (k < groups.size() && !alike(groups[k][0], r)) ++k;
    if (k == groups.size()) groups.emplace_back();
    groups[k].push_back(r);
  }
  for (const auto& g : groups) add_group(g);
}

void BatchPlan::add_group(const std::vector<Recorder>& recs) {
  const size_t ns = recs[0].recs.size();
  const int np = (int)recs.size();
  // all stages' records and maps go to the device in one copy; stages with the same work-group counts share
  // a map
  std::vector<unsigned char> blob;
  auto place = [&](const void* p, size_t n) {
    const size_t at = (blob.size() + 255) & ~(size_t)255;
    blob.resize(at + n);
    std::memcpy(blob.data() + at, p, n);
    return at;
  };
  struct MapAt {
    bool hop;
    std::vector<int> nb;
    size_t at;
    int n;
  };
  std::vector<MapAt> maps;
  std::vector<size_t> tab_at(ns), map_at(ns, (size_t)-1);
  const size_t first = st_.size();
  for (size_t j = 0; j < ns; ++j) {
    const LaunchRec& r0 = recs[0].recs[j];
    Stage s;
    s.kind = r0.kind;
    s.nprob = np;
    s.rec0 = r0.bytes;
    std::memcpy(s.key, r0.key, sizeof(s.key));
    for (int p = 0; p < np; ++p) s.nb.push_back(recs[p].recs[j].nblocks);
    if (s.kind == REC_BLAS) {
      s.opc = r0.key[0];
      for (int k = 0; k < 4; ++k) s.prec[k] = r0.key[1 + k];
    }
    std::vector<unsigned char> tab;
    tab.reserve(r0.bytes.size() * np);
    std::vector<int4> map;
    const MapAt* known = nullptr;
    for (const MapAt& m : maps)
      if (s.kind != REC_FIN && m.hop == (s.kind == REC_HOP) && m.nb == s.nb) known = &m;
    int maxnb = 0;
    for (int p = 0; p < np; ++p) {
      const LaunchRec& r = recs[p].recs[j];
      CMX_REQUIRE(r.kind == r0.kind && std::memcmp(r.key, r0.key, sizeof(r.key)) == 0 && r.bytes.size() == r0.bytes.size(),
                  CMX_ERR_ARG,
                  "batch: stage " + std::to_string(j) + " selects a different kernel for problem " + std::to_string(p) +
                      " (launch shape, precision or epilogue)");
      tab.insert(tab.end(), r.bytes.begin(), r.bytes.end());
      if (s.kind == REC_BLAS && !known)
        for (int b = 0; b < r.nblocks; ++b) map.push_back(make_int4(p, b, r.nblocks, 0));
      maxnb = std::max(maxnb, r.nblocks);
    }
    if (s.kind == REC_HOP && !known) {
      // Hopping stages interleave the problems in runs of 8 work-groups: the work-groups of every
      // problem over the same 8 local blocks follow each other, and global work-group g lands on XCD
      // g mod 8 = local block mod 8.  Problems on one gauge field (the sources of a propagator) then
      // read the links and clover of a block from their XCD's L2 after the first problem brought
      // them in, and the plane kernel's XCD-aware tiling keeps its meaning.  Runs shorter than 8
      // are padded with idle entries (problem -1) to keep the alignment.
      for (int j8 = 0; j8 < maxnb; j8 += 8)
        for (int p = 0; p < np; ++p) {
          const int nbp = recs[p].recs[j].nblocks;
          if (j8 >= nbp) continue;
          for (int x = 0; x < 8; ++x) {
            const int b = j8 + x;
            map.push_back(b < nbp ? make_int4(p, b, nbp, 0) : make_int4(-1, 0, 0, 0));
          }
        }
    }
    tab_at[j] = place(tab.data(), tab.size());
    if (s.kind == REC_FIN) {
      s.nblocks = np;
      for (int p = 0; p < np; ++p) s.fin_nb = std::max(s.fin_nb, fin_partials(recs[p].recs[j]));
    } else if (known) {
      s.nblocks = known->n;
      map_at[j] = known->at;
    } else {
      s.nblocks = (int)map.size();
      map_at[j] = place(map.data(), sizeof(int4) * map.size());
      maps.push_back(MapAt{s.kind == REC_HOP, s.nb, map_at[j], s.nblocks});
    }
    st_.push_back(std::move(s));
  }
  mem_.emplace_back(new DevScratch(blob.size()));
  char* base = mem_.back()->as<char>();
  host_to_device(base, blob.data(), blob.size(), 0);
  CMX_HIP(hipStreamSynchronize(0));
  for (size_t j = 0; j < ns; ++j) {
    st_[first + j].tab = base + tab_at[j];
    if (map_at[j] != (size_t)-1) st_[first + j].map = reinterpret_cast<const int4*>(base + map_at[j]);
  }
}

void BatchPlan::refresh(const std::vector<Recorder>& recs, hipStream_t strm) {
  const int np = (int)recs.size();
  bool same = np >= 1 && !st_.empty();
  for (int p = 0; same && p < np; ++p) same = recs[p].recs.size() == st_.size();
  for (size_t j = 0; same && j < st_.size(); ++j) {
    const Stage& s = st_[j];
    same = s.nprob == np;
    for (int p = 0; same && p < np; ++p) {
      const LaunchRec& r = recs[p].recs[j];
      same = r.kind == s.kind && r.nblocks == s.nb[p] && std::memcmp(r.key, s.key, sizeof(s.key)) == 0 &&
             r.bytes.size() == s.rec0.size();
    }
  }
  if (!same) {
    build(recs);
    return;
  }
  for (size_t j = 0; j < st_.size(); ++j) {
    Stage& s = st_[j];
    const size_t rb = s.rec0.size(), bytes = rb * np;
    if (!s.htab) {
      void* h = nullptr;
      CMX_HIP(hipHostMalloc(&h, bytes, 0));
      s.htab = std::shared_ptr<void>(h, [](void* q) { (void)hipHostFree(q); });
    }
    unsigned char* h = static_cast<unsigned char*>(s.htab.get());
    for (int p = 0; p < np; ++p) std::memcpy(h + rb * p, recs[p].recs[j].bytes.data(), rb);
    s.rec0 = recs[0].recs[j].bytes;
    if (s.kind == REC_FIN) {
      s.fin_nb = 0;
      for (int p = 0; p < np; ++p) s.fin_nb = std::max(s.fin_nb, fin_partials(recs[p].recs[j]));
    }
    CMX_HIP(hipMemcpyAsync(s.tab, h, bytes, hipMemcpyHostToDevice, strm));
  }
}

long BatchPlan::blocks() const {
  long n = 0;
  for (const Stage& s : st_) n += s.nblocks;
  return n;
}

void BatchPlan::run(hipStream_t strm) const {
  CMX_REQUIRE(active_recorder() == nullptr, CMX_ERR_ARG, "batch: replay while recording");
  for (const Stage& s : st_) {
    const BatchGrid bg{s.tab, s.map, s.nblocks};
    switch (s.kind) {
      case REC_HOP: {
        HopLaunch h;
        std::memcpy(&h, s.rec0.data(), sizeof(h));
        launch_hop(h, strm, &bg);
        break;
      }
      case REC_BLAS: {
        BlasLaunch b;
        std::memcpy(&b, s.rec0.data(), sizeof(b));
        launch_blas(s.opc, b, s.prec, strm, &bg);
        break;
      }
      default:
        launch_finalize_batch(static_cast<const FinLaunch*>(s.tab), s.nprob, s.fin_nb, strm);
        break;
    }
  }
}

}  // namespace cmx
