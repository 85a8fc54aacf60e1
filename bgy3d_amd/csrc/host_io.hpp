// What the solver keeps between calls for its traffic with the host: pinned
// memory, streams and twiddle tables, and the copies of large host arrays.
// rism3d_cache_release gives all of it back.
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <exception>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace rism {
namespace {

// Idle pinned blocks by size class (powers of two) and idle streams by
// device, handed out to one user at a time; those beyond the bounds are freed
// at once.  hipHostMalloc, hipHostFree and hipStreamCreate were 0.1 ms of the
// 0.5 ms of a call at 32^3.
struct HostPool {
  static constexpr size_t MOST_BYTES = (size_t)64 << 20;
  static constexpr size_t MOST_STREAMS = 32;
  std::mutex mu;
  std::multimap<size_t, void*> pinned;
  size_t pinned_bytes = 0;
  std::multimap<int, hipStream_t> streams;
};
HostPool& host_pool() {
  static HostPool p;
  return p;
}

// Pinned host memory, coherent: kernels and the host see each other's words
// while both run.
class Pinned {
 public:
  Pinned() = default;
  explicit Pinned(size_t need) {
    bytes_ = (size_t)1 << 16;
    while (bytes_ < need) bytes_ *= 2;
    HostPool& hp = host_pool();
    {
      std::lock_guard<std::mutex> lk(hp.mu);
      auto it = hp.pinned.find(bytes_);
      if (it != hp.pinned.end()) {
        p_ = it->second;
        hp.pinned.erase(it);
        hp.pinned_bytes -= bytes_;
        return;
      }
    }
    HIPCHK(hipHostMalloc(&p_, bytes_, hipHostMallocCoherent | hipHostMallocPortable));
  }
  Pinned(const Pinned&) = delete;
  Pinned& operator=(const Pinned&) = delete;
  Pinned(Pinned&& o) noexcept : p_(o.p_), bytes_(o.bytes_) { o.p_ = nullptr; }
  Pinned& operator=(Pinned&& o) noexcept {
    std::swap(p_, o.p_);
    std::swap(bytes_, o.bytes_);
    return *this;
  }
  // The owner frees it only when no kernel or copy uses it any more.
  ~Pinned() {
    if (!p_) return;
    HostPool& hp = host_pool();
    {
      std::lock_guard<std::mutex> lk(hp.mu);
      if (hp.pinned_bytes + bytes_ <= HostPool::MOST_BYTES) {
        hp.pinned.insert({bytes_, p_});
        hp.pinned_bytes += bytes_;
        return;
      }
    }
    (void)hipHostFree(p_);
  }
  explicit operator bool() const { return p_ != nullptr; }
  template <typename X> X* as(size_t offset = 0) const {
    return reinterpret_cast<X*>(static_cast<char*>(p_) + offset);
  }

 private:
  void* p_ = nullptr;
  size_t bytes_ = 0;
};

// A stream of the current device (default priority, non-blocking), idle when
// handed out; the user hands it back idle.
hipStream_t stream_take(int dev) {
  HostPool& hp = host_pool();
  {
    std::lock_guard<std::mutex> lk(hp.mu);
    auto it = hp.streams.find(dev);
    if (it != hp.streams.end()) {
      const hipStream_t s = it->second;
      hp.streams.erase(it);
      return s;
    }
  }
  hipStream_t s = nullptr;
  HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  return s;
}
void stream_give(int dev, hipStream_t s) {
  HostPool& hp = host_pool();
  // a stream that an error ended is not handed out again
  const bool ok = hipStreamSynchronize(s) == hipSuccess;
  {
    std::lock_guard<std::mutex> lk(hp.mu);
    if (ok && hp.streams.size() < HostPool::MOST_STREAMS) {
      hp.streams.insert({dev, s});
      return;
    }
  }
  (void)hipStreamDestroy(s);
}

// A stream for copies that are complete when the call returns.  Never the
// default stream: its copies fail, and void the capture, while another thread
// (a size class of rism3d_batch_solve_grids) records a graph.
struct OwnStream {
  int dev = 0;
  hipStream_t s = nullptr;
  OwnStream() {
    HIPCHK(hipGetDevice(&dev));
    s = stream_take(dev);
  }
  OwnStream(const OwnStream&) = delete;
  OwnStream& operator=(const OwnStream&) = delete;
  ~OwnStream() { stream_give(dev, s); }
};

void host_pool_empty() {
  HostPool& hp = host_pool();
  std::lock_guard<std::mutex> lk(hp.mu);
  for (auto& b : hp.pinned) (void)hipHostFree(b.second);
  for (auto& s : hp.streams) (void)hipStreamDestroy(s.second);
  hp.pinned.clear();
  hp.pinned_bytes = 0;
  hp.streams.clear();
}

// Large copies between device memory and the caller's pageable arrays.  The
// runtime stages them through one thread, which on the way out also meets
// every page of a fresh array for the first time: 10 GB/s into a new 50 MB
// array and 27 GB/s from one, of the link's 57.  Here several threads each
// take every n-th chunk through two pinned slots and a stream of their own, so
// that page faults, host copies and the link overlap: 35 GB/s into a new 50 MB
// array, 46 into 170 MB.  One such transfer at a time (the link is shared);
// arrays under COPY_MIN go through the runtime (0.1 ms of thread starts is not
// paid back), and so do those that the runtime knows (pinned by the caller):
// the link reaches them itself (one F of 3 sites with t and F in pinned arrays,
// staged and not: 96^3 1.15 and 0.91 ms, 128^3 2.40 and 2.00, 192^3 7.3 and 6.5).
constexpr size_t COPY_CHUNK = (size_t)2 << 20;
constexpr size_t COPY_MIN = (size_t)4 << 20;
constexpr int COPY_THREADS = 8;

struct HostCopy {
  void* host;
  void* dev;
  size_t bytes;
};

int copy_cpus() {
  cpu_set_t set;
  CPU_ZERO(&set);
  if (sched_getaffinity(0, sizeof set, &set) != 0) return 1;
  return std::max(1, CPU_COUNT(&set));
}

// The runtime allocated p (or shares it with the device).
bool runtime_memory(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeHost || a.type == hipMemoryTypeDevice ||
         a.type == hipMemoryTypeManaged;
}

// Every item copied, out (device to host) or in; the device data are ready
// (or the device buffers free) when it is called, and the copies complete
// when it returns.
void host_copies(const std::vector<HostCopy>& all, bool out) {
  std::vector<HostCopy> items, direct;
  for (const HostCopy& c : all)
    (c.bytes >= COPY_MIN && runtime_memory(c.host) ? direct : items).push_back(c);
  if (!direct.empty()) {
    const OwnStream s;
    for (const HostCopy& c : direct)
      HIPCHK(out ? hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDefault, s.s)
                 : hipMemcpyAsync(c.dev, c.host, c.bytes, hipMemcpyDefault, s.s));
    HIPCHK(hipStreamSynchronize(s.s));
  }
  if (items.empty()) return;
  struct Chunk {
    char *host, *dev;
    size_t bytes;
  };
  std::vector<Chunk> chunks;
  size_t total = 0;
  for (const HostCopy& c : items) {
    total += c.bytes;
    for (size_t o = 0; o < c.bytes; o += COPY_CHUNK)
      chunks.push_back({static_cast<char*>(c.host) + o, static_cast<char*>(c.dev) + o,
                        std::min(COPY_CHUNK, c.bytes - o)});
  }
  const int nt = (int)std::min({(size_t)COPY_THREADS, (size_t)copy_cpus(), chunks.size() / 2});
  if (total < COPY_MIN || nt < 2) {
    const OwnStream s;
    for (const HostCopy& c : items)
      if (c.bytes)
        HIPCHK(out ? hipMemcpyWithStream(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, s.s)
                   : hipMemcpyWithStream(c.dev, c.host, c.bytes, hipMemcpyHostToDevice, s.s));
    return;
  }
  static std::mutex one;
  std::lock_guard<std::mutex> lk(one);
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  struct Lane {
    Pinned slot;  // two chunks
    hipStream_t s = nullptr;
    hipEvent_t ev[2] = {};
    int dev = 0;
    ~Lane() {
      if (s) stream_give(dev, s);  // waits for its copies, before the slots go back
      for (hipEvent_t e : ev)
        if (e) (void)hipEventDestroy(e);
    }
  };
  std::vector<Lane> lanes(nt);
  for (Lane& l : lanes) {
    l.dev = dev;
    l.slot = Pinned(2 * COPY_CHUNK);
    l.s = stream_take(dev);
    for (hipEvent_t& e : l.ev) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  std::atomic<int> failed{(int)hipSuccess};
  auto work = [&](int t) {
    Lane& l = lanes[t];
    auto ok = [&](hipError_t e) {
      if (e != hipSuccess) failed = (int)e;
      return e == hipSuccess;
    };
    if (!ok(hipSetDevice(dev))) return;
    int k = 0;
    const Chunk* before = nullptr;  // out: in flight in the other slot
    for (size_t c = t; c < chunks.size(); c += nt, k ^= 1) {
      const Chunk& ch = chunks[c];
      char* slot = l.slot.as<char>(k * COPY_CHUNK);
      if (out) {
        if (!ok(hipMemcpyAsync(slot, ch.dev, ch.bytes, hipMemcpyDeviceToHost, l.s)) ||
            !ok(hipEventRecord(l.ev[k], l.s)))
          return;
        if (before) {
          if (!ok(hipEventSynchronize(l.ev[k ^ 1]))) return;
          std::memcpy(before->host, l.slot.as<char>((k ^ 1) * COPY_CHUNK), before->bytes);
        }
        before = &ch;
      } else {
        if (c >= (size_t)t + 2 * nt && !ok(hipEventSynchronize(l.ev[k]))) return;
        std::memcpy(slot, ch.host, ch.bytes);
        if (!ok(hipMemcpyAsync(ch.dev, slot, ch.bytes, hipMemcpyHostToDevice, l.s)) ||
            !ok(hipEventRecord(l.ev[k], l.s)))
          return;
      }
    }
    if (!ok(hipStreamSynchronize(l.s))) return;
    if (before) std::memcpy(before->host, l.slot.as<char>((k ^ 1) * COPY_CHUNK), before->bytes);
  };
  std::vector<std::thread> th;
  int started = 1;
  try {
    th.reserve(nt);
    for (; started < nt; ++started) th.emplace_back(work, started);
  } catch (const std::exception&) {  // no more threads: the rest of the lanes here
  }
  work(0);
  for (int t = started; t < nt; ++t) work(t);
  for (std::thread& t : th) t.join();
  HIPCHK((hipError_t)failed.load());
}

// exp(-2 pi i j / n) of a length on the current device, in FP64 and FP32,
// made on first use (ten lengths at most, 30 KB together).
struct TwiddleCache {
  std::mutex mu;
  std::map<std::pair<int, int>, std::pair<cpx<double>*, cpx<float>*>> tables;
};
TwiddleCache& twiddle_cache() {
  static TwiddleCache c;
  return c;
}
template <typename T>
std::vector<cpx<T>> twiddles(int n) {
  std::vector<cpx<T>> w(n);
  for (int j = 0; j < n; ++j) {
    const long double a = -2.0L * 3.14159265358979323846264338327950288L * j / n;
    w[j] = cpx<T>{(T)std::cos(a), (T)std::sin(a)};
  }
  return w;
}
std::pair<cpx<double>*, cpx<float>*> twiddles_on(int dev, int n) {
  TwiddleCache& c = twiddle_cache();
  std::lock_guard<std::mutex> lk(c.mu);
  auto it = c.tables.find({dev, n});
  if (it != c.tables.end()) return it->second;
  const auto wd = twiddles<double>(n);
  const auto wf = twiddles<float>(n);
  const OwnStream s;
  void* p = nullptr;
  HIPCHK(hipMalloc(&p, n * (sizeof(cpx<double>) + sizeof(cpx<float>))));
  cpx<double>* d = static_cast<cpx<double>*>(p);
  cpx<float>* f = reinterpret_cast<cpx<float>*>(d + n);
  hipError_t e =
      hipMemcpyWithStream(d, wd.data(), n * sizeof(cpx<double>), hipMemcpyHostToDevice, s.s);
  if (e == hipSuccess)
    e = hipMemcpyWithStream(f, wf.data(), n * sizeof(cpx<float>), hipMemcpyHostToDevice, s.s);
  if (e != hipSuccess) (void)hipFree(p);
  HIPCHK(e);
  return c.tables[{dev, n}] = {d, f};
}
void twiddles_empty() {
  TwiddleCache& c = twiddle_cache();
  std::lock_guard<std::mutex> lk(c.mu);
  for (auto& t : c.tables) (void)hipFree(t.second.first);
  c.tables.clear();
}

}  // namespace
}  // namespace rism
