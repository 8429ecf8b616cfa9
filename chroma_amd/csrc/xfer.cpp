// Pageable host memory reaches the device through pinned staging buffers: one to four threads each copy
// their own chunks (in turn) between the caller's array and two pinned slots, and queue the DMA of each
// slot on the caller's stream, so that the host copies of all threads, the page faults of fresh arrays and
// the DMA overlap.  The link runs at 57 GB/s each way; every DMA costs some 14 us beside its bytes, so
// slots are large (4 MB), and waking a thread costs 20 to 50 us, so small arrays use the calling thread
// alone, and below 1 MB the runtime's own staging is faster.  Measured (us, hipMemcpyAsync of pageable memory against
// this): up and down again, with buffers used before and in turn, 96 KB 43 / 52, 192 KB 52 / 82, 384 KB 69 / 96,
// 768 KB 102 / 126, 1152 KB 145 to 170 / 143 to 151, 1536 KB 169 to 194 / 157 to 168, into fresh pages 768 KB 253 / 266,
// 1152 KB 405 / 367; 2 MB down 137 / 98, 12 MB down into fresh pages 1177 / 462, 64 MB up 2199 / 1502, down 3784 / 1544,
// fresh 6183 / 1913, 256 MB up 8939 / 5821, fresh 25180 / 6322.  Chunks that hold only zero bits (an initial
// guess of zero, a point source) are cleared on the device instead of sent.
//
// The threads and slots live in a Lane; a call takes a free one, makes one if none is free (at most
// MAX_LANES per device), or falls back to hipMemcpy.  Any number of threads may call at once.
#include "xfer.h"

#include <sched.h>
#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace cmx {

namespace {

constexpr size_t SLOT = (size_t)4 << 20;     // bytes per pinned slot
constexpr size_t SMALL = (size_t)1 << 20;    // below this the runtime's own path is faster
constexpr size_t MIN_CHUNK = (size_t)128 << 10;
constexpr int MAX_WORKERS = 4, MAX_LANES = 2;

bool zero_bits(const void* p, size_t n) {
  const unsigned char* c = static_cast<const unsigned char*>(p);
  while (n >= 256) {  // 256 bytes between exits
    uint64_t w[32], o = 0;
    std::memcpy(w, c, 256);
    for (int k = 0; k < 32; ++k) o |= w[k];
    if (o) return false;
    c += 256, n -= 256;
  }
  for (size_t k = 0; k < n; ++k)
    if (c[k]) return false;
  return true;
}

class Lane {
 public:
  explicit Lane(int dev) : dev_(dev) {
    cpu_set_t set;
    CPU_ZERO(&set);
    int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    nw_ = std::max(1, std::min(MAX_WORKERS, cpus));
    CMX_HIP(hipHostMalloc(reinterpret_cast<void**>(&pin_), SLOT * 2 * nw_, 0));
    try {
      for (int k = 0; k < 2 * nw_; ++k) {
        hipEvent_t e = nullptr;
        CMX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        ev_.push_back(e);
      }
      busy_.assign(2 * nw_, 0);
      for (int w = 1; w < nw_; ++w) th_.emplace_back([this, w] { loop(w); });
    } catch (...) {
      close();
      throw;
    }
  }
  ~Lane() { close(); }
  int dev() const { return dev_; }

  void up(char* d, const char* h, size_t bytes, hipStream_t s) {
    const int nw = workers(bytes, (size_t)16 << 20);
    const size_t ch = chunk(bytes, nw);
    run(nw, [&](int w) {
      size_t turn = 0;
      for (size_t off = w * ch; off < bytes; off += ch * nw, ++turn) {
        const size_t n = std::min(ch, bytes - off);
        if (zero_bits(h + off, n)) {
          check(hipMemsetAsync(d + off, 0, n, s));
          continue;
        }
        const int k = 2 * w + (int)(turn & 1);
        wait(k);
        std::memcpy(pin_ + SLOT * k, h + off, n);
        check(hipMemcpyAsync(d + off, pin_ + SLOT * k, n, hipMemcpyHostToDevice, s));
        check(hipEventRecord(ev_[k], s));
        busy_[k] = 1;
      }
    });
  }

  void down(char* h, const char* d, size_t bytes, hipStream_t s) {
    const int nw = workers(bytes, (size_t)8 << 20);
    const size_t ch = chunk(bytes, nw);
    run(nw, [&](int w) {
      auto issue = [&](size_t off, int k) {
        wait(k);
        check(hipMemcpyAsync(pin_ + SLOT * k, d + off, std::min(ch, bytes - off), hipMemcpyDeviceToHost, s));
        check(hipEventRecord(ev_[k], s));
        busy_[k] = 1;
      };
      const size_t step = ch * nw;
      size_t off = w * ch;
      if (off < bytes) issue(off, 2 * w);
      for (int t = 0; off < bytes; off += step, t ^= 1) {
        if (off + step < bytes) issue(off + step, 2 * w + (t ^ 1));
        const int k = 2 * w + t;
        wait(k);
        std::memcpy(h + off, pin_ + SLOT * k, std::min(ch, bytes - off));
      }
    });
  }

 private:
  // one worker to 4 MB, all from `all` bytes, two between
  int workers(size_t bytes, size_t all) const {
    return std::min(nw_, bytes < ((size_t)4 << 20) ? 1 : (bytes < all ? 2 : MAX_WORKERS));
  }
  static size_t chunk(size_t bytes, int nw) {
    const size_t c = (bytes / (2 * nw) + 4095) & ~(size_t)4095;
    return std::max(MIN_CHUNK, std::min(SLOT, c));
  }
  static void check(hipError_t e) {
    if (e != hipSuccess) throw Error(CMX_ERR_HIP, std::string("host transfer: ") + hipGetErrorString(e));
  }
  void wait(int k) {  // the DMA that last used slot k
    if (!busy_[k]) return;
    check(hipEventSynchronize(ev_[k]));
    busy_[k] = 0;
  }
  // f(w) on nw workers, the calling thread as worker 0; the first error is rethrown after all have ended
  void run(int nw, const std::function<void(int)>& f) {
    if (nw == 1) {
      f(0);
      return;
    }
    {
      std::lock_guard<std::mutex> lk(m_);
      job_ = &f;
      left_ = nw - 1;
      use_ = nw;
      err_.clear();
      ++gen_;
    }
    go_.notify_all();
    work(0, f);
    std::unique_lock<std::mutex> lk(m_);
    done_.wait(lk, [&] { return left_ == 0; });
    job_ = nullptr;
    if (!err_.empty()) {
      const std::string e = err_;
      lk.unlock();
      throw Error(CMX_ERR_HIP, e);
    }
  }
  void work(int w, const std::function<void(int)>& f) {
    try {
      f(w);
    } catch (const std::exception& e) {
      std::lock_guard<std::mutex> lk(m_);
      if (err_.empty()) err_ = e.what();
    }
  }
  void loop(int w) {
    (void)hipSetDevice(dev_);
    long seen = 0;
    for (;;) {
      const std::function<void(int)>* f;
      {
        std::unique_lock<std::mutex> lk(m_);
        go_.wait(lk, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
        if (w >= use_ || !job_) continue;
        f = job_;
      }
      work(w, *f);
      std::lock_guard<std::mutex> lk(m_);
      if (--left_ == 0) done_.notify_one();
    }
  }
  void close() {
    {
      std::lock_guard<std::mutex> lk(m_);
      stop_ = true;
    }
    go_.notify_all();
    for (auto& t : th_) t.join();
    th_.clear();
    for (size_t k = 0; k < ev_.size(); ++k) {
      if (k < busy_.size() && busy_[k]) (void)hipEventSynchronize(ev_[k]);
      (void)hipEventDestroy(ev_[k]);
    }
    ev_.clear();
    if (pin_) (void)hipHostFree(pin_);
    pin_ = nullptr;
  }

  int dev_, nw_ = 1;
  char* pin_ = nullptr;
  std::vector<hipEvent_t> ev_;
  std::vector<char> busy_;  // slot k: touched by worker k / 2 alone
  std::vector<std::thread> th_;
  std::mutex m_;
  std::condition_variable go_, done_;
  const std::function<void(int)>* job_ = nullptr;
  long gen_ = 0;
  int left_ = 0, use_ = 0;
  bool stop_ = false;
  std::string err_;
};

struct Cached {
  void* p;
  size_t cap;
  int dev;
};
// device bytes and buffers the scratch cache keeps at most
constexpr size_t CACHE_MAX = (size_t)4 << 30, CACHE_ENTRIES = 1024;

struct Pool {
  std::mutex m;
  pid_t pid = 0;
  std::vector<Lane*> free_lanes;
  std::vector<int> made;  // lanes per device
  std::vector<Cached> cache;
  size_t cached = 0;
  std::vector<void*> pinned;
};
// never destroyed: its threads may outlive static destruction
Pool& pool() {
  static Pool* p = new Pool();
  return *p;
}

// a lane of the current device, or null
Lane* take_lane() {
  int dev = 0;
  CMX_HIP(hipGetDevice(&dev));
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.m);
  if (P.pid != getpid()) {  // a forked child has none of the parent's threads
    P.free_lanes.clear();
    P.made.clear();
    P.pid = getpid();
  }
  for (size_t k = 0; k < P.free_lanes.size(); ++k)
    if (P.free_lanes[k]->dev() == dev) {
      Lane* l = P.free_lanes[k];
      P.free_lanes.erase(P.free_lanes.begin() + (long)k);
      return l;
    }
  if ((int)P.made.size() <= dev) P.made.resize(dev + 1, 0);
  if (P.made[dev] >= MAX_LANES) return nullptr;
  Lane* l = nullptr;
  try {
    l = new Lane(dev);
  } catch (const std::exception&) {  // no pinned memory or threads to be had
    (void)hipGetLastError();
    return nullptr;
  }
  ++P.made[dev];
  return l;
}

struct LaneHold {
  Lane* l;
  LaneHold() : l(take_lane()) {}
  ~LaneHold() {
    if (!l) return;
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.m);
    P.free_lanes.push_back(l);
  }
};

}  // namespace

// Memory the runtime knows (pinned or managed by the caller) is copied directly
static bool pageable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

void host_to_device(void* dev, const void* host, size_t bytes, hipStream_t s) {
  if (bytes >= SMALL && pageable(host)) {
    LaneHold h;
    if (h.l) {
      h.l->up(static_cast<char*>(dev), static_cast<const char*>(host), bytes, s);
      return;
    }
  }
  if (bytes) CMX_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s));
}

void device_to_host(void* host, const void* dev, size_t bytes, hipStream_t s) {
  if (bytes >= SMALL && pageable(host)) {
    LaneHold h;
    if (h.l) {
      h.l->down(static_cast<char*>(host), static_cast<const char*>(dev), bytes, s);
      return;
    }
  }
  if (bytes) CMX_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
  CMX_HIP(hipStreamSynchronize(s));
}

void* scratch_take(size_t bytes, size_t& cap, int& dev) {
  CMX_HIP(hipGetDevice(&dev));
  cap = 0;
  if (!bytes) return nullptr;
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lk(P.m);
    size_t best = P.cache.size();
    for (size_t k = 0; k < P.cache.size(); ++k) {
      const Cached& c = P.cache[k];
      if (c.dev == dev && c.cap >= bytes && c.cap <= bytes + bytes / 4 + 65536 &&
          (best == P.cache.size() || c.cap < P.cache[best].cap))
        best = k;
    }
    if (best < P.cache.size()) {
      const Cached c = P.cache[best];
      cap = c.cap;
      P.cached -= cap;
      P.cache.erase(P.cache.begin() + (long)best);  // keeps the order of age
      return c.p;
    }
  }
  cap = bytes;
  void* p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  xfer_release();  // the cached buffers may be what is missing
  CMX_HIP(hipMalloc(&p, bytes));
  return p;
}

void scratch_give(void* p, size_t cap, int dev) {
  if (!p) return;
  // A full cache lets the buffers go that lay in it longest: they belong to sizes no longer in use, and refusing
  // the new ones instead made every later call allocate (12 batched solves: 34 -> 63 ms).
  std::vector<void*> out;
  if (cap > CACHE_MAX) {
    out.push_back(p);
  } else {
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.m);
    size_t n = 0;
    for (; n < P.cache.size() && (P.cached + cap > CACHE_MAX || P.cache.size() - n >= CACHE_ENTRIES); ++n) {
      out.push_back(P.cache[n].p);
      P.cached -= P.cache[n].cap;
    }
    P.cache.erase(P.cache.begin(), P.cache.begin() + (long)n);
    P.cache.push_back(Cached{p, cap, dev});
    P.cached += cap;
  }
  for (void* q : out) (void)hipFree(q);
}

void* pinned_take() {
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lk(P.m);
    if (!P.pinned.empty()) {
      void* p = P.pinned.back();
      P.pinned.pop_back();
      return p;
    }
  }
  void* p = nullptr;
  CMX_HIP(hipHostMalloc(&p, PINNED_BLOCK, 0));
  return p;
}

void pinned_give(void* p) {
  if (!p) return;
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lk(P.m);
    if (P.pinned.size() < 128) {
      P.pinned.push_back(p);
      return;
    }
  }
  (void)hipHostFree(p);
}

DevScratch::DevScratch(size_t bytes) : bytes_(bytes), throwing_(std::uncaught_exceptions()) {
  p_ = scratch_take(bytes, cap_, dev_);
}

DevScratch::~DevScratch() {
  if (!p_) return;
  if (std::uncaught_exceptions() == throwing_)
    scratch_give(p_, cap_, dev_);
  else
    (void)hipFree(p_);  // an error may leave work queued: hipFree waits for it
}

size_t scratch_cached() {
  int dev = 0;
  CMX_HIP(hipGetDevice(&dev));
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.m);
  size_t n = 0;
  for (const Cached& c : P.cache)
    if (c.dev == dev) n += c.cap;
  return n;
}

void xfer_release() {
  Pool& P = pool();
  std::vector<Lane*> lanes;
  std::vector<Cached> cache;
  std::vector<void*> pinned;
  {
    std::lock_guard<std::mutex> lk(P.m);
    if (P.pid == getpid()) {
      lanes.swap(P.free_lanes);
      for (Lane* l : lanes) --P.made[l->dev()];
    }
    cache.swap(P.cache);
    P.cached = 0;
    pinned.swap(P.pinned);
  }
  for (Lane* l : lanes) delete l;
  for (const Cached& c : cache) (void)hipFree(c.p);
  for (void* p : pinned) (void)hipHostFree(p);
}

}  // namespace cmx
