// rhy_transfer.hip -- host transfers through pinned staging memory.
//
// A copy to or from pageable memory goes through the runtime's own staging
// with one host thread, which for a fresh destination also takes its page
// faults: 9 GB/s (a 256^3 snapshot of 537 MB: 58 ms beside 61 ms for the 60
// steps before it), against 55 GB/s of the link.  Large copies are cut into
// chunks that several threads take from a common counter: each keeps two
// chunks going, one on the link and one between staging and the caller's
// array, and widens or narrows the mixed form's values on the way.  Steps and
// snapshot of the 256^3 run: 119 -> 77 ms.
#include "rhy_transfer.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace rhy {
namespace {

constexpr size_t kChunk = (size_t)2 << 20;  // staging bytes of one chunk, at most
constexpr size_t kMinChunk = (size_t)256 << 10;
constexpr int kWorkers = 8;
constexpr int kSlots = 2 * kWorkers;

// Whether a copy of `bytes` device bytes is staged: from the size on where the
// threads give more than they cost (a queued copy and an event for each chunk,
// the helpers' wakes), by direction and conversion.  Direct against staged, us:
//   from the host      24 MiB 676 / 742   32 MiB 914 / 908    64 MiB 2304 / 1729
//   to the host         6 MiB 344 / 406    8 MiB 455 / 450    32 MiB 1885 / 946
//   narrowed (mixed)    6 MiB 365 / 383    8 MiB 476 / 427    32 MiB 3993 / 942
//   widened (mixed)     3 MiB 287 / 295    4 MiB 430 / 377    32 MiB 4655 / 1027
inline bool worth_staging(size_t bytes, bool as_double, bool to_host) {
  const size_t mib = as_double ? (to_host ? 4 : 8) : (to_host ? 8 : 32);
  return bytes >= mib << 20;
}

// The helpers of a copy: threads that wait for work(index), index 1 .. n.
// (Starting threads for each copy takes as long as a copy of 4 MB.)
struct Helpers {
  std::mutex lock;
  std::condition_variable wake, done;
  std::vector<std::thread> threads;
  const std::function<void(int)>* work = nullptr;  // of the copy going on
  int wanted = 0, running = 0;
  uint64_t round = 0;
  bool stop = false;

  Helpers() {
    threads.reserve(kWorkers - 1);
    for (int i = 1; i < kWorkers; ++i) {
      try {
        threads.emplace_back([this, i] { loop(i); });
      } catch (const std::exception&) {  // no thread or no memory for one
        break;  // the ones there are take the chunks
      }
    }
  }
  ~Helpers() {
    {
      std::lock_guard<std::mutex> hold(lock);
      stop = true;
    }
    wake.notify_all();
    for (std::thread& t : threads) t.join();
  }

  void loop(int index) {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> hold(lock);
    for (;;) {
      wake.wait(hold, [&] { return stop || round != seen; });
      if (stop) return;
      seen = round;
      if (index > wanted) continue;
      hold.unlock();
      (*work)(index);
      hold.lock();
      if (--running == 0) done.notify_all();
    }
  }

  // w(0) here and w(1) .. w(n) on the helpers, n at most their number;
  // returns once all have.
  void run(int n, const std::function<void(int)>& w) {
    n = std::min(n, (int)threads.size());
    {
      std::lock_guard<std::mutex> hold(lock);
      work = &w;
      wanted = running = n;
      ++round;
    }
    if (n > 0) wake.notify_all();
    w(0);
    std::unique_lock<std::mutex> hold(lock);
    done.wait(hold, [&] { return running == 0; });
  }
};

// One staging area (32 MB) and set of helpers per process, used by one copy at
// a time: a copy that finds them taken goes the direct way.  They go with the
// last box or batch; in a process that ends before, with the process.
//
// To pin the memory, start the threads and give both back is about 0.5 ms, which
// a program that makes a box, copies a little and drops it again would pay each
// time.  So the first copies of the objects alive go the direct way, until
// staging them would have saved that much: 29 us for each MiB to the host or
// converted, at least, and half of it from the host.
constexpr size_t kWorth = (size_t)32 << 20;
std::mutex g_lock;
unsigned char* g_staging = nullptr;
Helpers* g_helpers = nullptr;
bool g_taken = false, g_refused = false;
size_t g_missed = 0;  // what direct copies missed since the last giving back
int g_users = 0;

// saves: what staging saves a copy, in bytes to the host.
unsigned char* staging_take(size_t saves) {
  std::lock_guard<std::mutex> hold(g_lock);
  if (g_taken || g_refused) return nullptr;
  if (!g_staging) {
    g_missed += saves;
    if (g_missed < kWorth) return nullptr;
    try {
      if (!g_helpers) g_helpers = new Helpers;
    } catch (const std::bad_alloc&) {
      return nullptr;
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, kChunk * kSlots, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      g_refused = true;  // not asked for again until the last object has gone
      return nullptr;
    }
    g_staging = static_cast<unsigned char*>(p);
  }
  g_taken = true;
  return g_staging;
}

void staging_free_if_idle() {  // with g_lock held
  if (g_users > 0 || g_taken) return;
  if (g_staging) (void)hipHostFree(g_staging);
  g_staging = nullptr;
  delete g_helpers;
  g_helpers = nullptr;
  g_refused = false;
  g_missed = 0;
}

void staging_give() {
  std::lock_guard<std::mutex> hold(g_lock);
  g_taken = false;
  staging_free_if_idle();
}

struct StagingHold {
  unsigned char* staging;
  explicit StagingHold(size_t saves) : staging(saves ? staging_take(saves) : nullptr) {}
  ~StagingHold() {
    if (staging) staging_give();
  }
};

// Memory the runtime knows: it copies to and from it at the link's rate, 1.4 to
// 3.6 times as fast as through the staging area (128 MiB 2349 us against 3391).
bool pinned(const void* host) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// count values between staging (or a plain buffer) and the caller's array
void unload(const void* from, void* host, size_t count, size_t esz, bool as_double) {
  if (!as_double) {
    std::memcpy(host, from, count * esz);
    return;
  }
  const float* f = static_cast<const float*>(from);
  double* d = static_cast<double*>(host);
  for (size_t i = 0; i < count; ++i) d[i] = (double)f[i];
}

void fill(void* to, const void* host, size_t count, size_t esz, bool as_double) {
  if (!as_double) {
    std::memcpy(to, host, count * esz);
    return;
  }
  float* f = static_cast<float*>(to);
  const double* d = static_cast<const double*>(host);
  for (size_t i = 0; i < count; ++i) f[i] = (float)d[i];
}

// A span at a time through the runtime, converted in a host buffer.
hipError_t copy_direct(hipStream_t stream, const HostSpan* spans, int nspans, size_t esz,
                       bool as_double, bool to_host, bool wait) {
  std::vector<std::vector<float>> tmp(as_double ? (size_t)nspans : 0);
  for (int i = 0; as_double && i < nspans; ++i) tmp[i].resize(spans[i].count);
  for (int i = 0; i < nspans; ++i) {
    const HostSpan& s = spans[i];
    void* host = s.host;
    if (as_double) {
      host = tmp[i].data();
      if (!to_host) fill(host, s.host, s.count, esz, true);
    }
    const hipError_t e =
        to_host ? hipMemcpyAsync(host, s.dev, s.count * esz, hipMemcpyDeviceToHost, stream)
                : hipMemcpyAsync(s.dev, host, s.count * esz, hipMemcpyHostToDevice, stream);
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(stream);
      return e;
    }
  }
  if (!wait && !as_double) return hipSuccess;
  const hipError_t e = hipStreamSynchronize(stream);
  if (e == hipSuccess && as_double && to_host)
    for (int i = 0; i < nspans; ++i) unload(tmp[i].data(), spans[i].host, spans[i].count, esz, true);
  return e;
}

struct Job {
  hipStream_t stream;
  int device;
  size_t esz;
  bool as_double, to_host;
  unsigned char* staging;
  std::vector<HostSpan> chunks;
  std::atomic<size_t> next{0};
  std::atomic<int> error{(int)hipSuccess};

  // The chunks: two for each worker, within [kMinChunk, kChunk].
  void cut(const HostSpan* spans, int nspans, size_t bytes, size_t esz, bool as_double) {
    const size_t part = std::min(std::max(bytes / kSlots, kMinChunk), kChunk);
    const size_t per = part / esz, hsz = as_double ? sizeof(double) : esz;
    for (int i = 0; i < nspans; ++i)
      for (size_t at = 0; at < spans[i].count; at += per)
        chunks.push_back({static_cast<unsigned char*>(spans[i].dev) + at * esz,
                          static_cast<unsigned char*>(spans[i].host) + at * hsz,
                          std::min(spans[i].count - at, per)});
  }

  void fail(hipError_t e) {
    int ok = (int)hipSuccess;
    error.compare_exchange_strong(ok, (int)e);
  }
  bool failed() const { return error.load() != (int)hipSuccess; }

  // Takes chunks until none is left.  Copies still queued when it returns
  // are waited for by the caller before the staging memory is given back.
  void work(int w) {
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t e = hipSetDevice(device);
    for (int s = 0; s < 2 && e == hipSuccess; ++s)
      e = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming);
    if (e == hipSuccess) {
      if (to_host) drain(w, ev);
      else feed(w, ev);
    } else {
      fail(e);
    }
    for (int s = 0; s < 2; ++s)
      if (ev[s]) (void)hipEventDestroy(ev[s]);
  }

  unsigned char* slot(int w, int s) { return staging + kChunk * (size_t)(2 * w + s); }

  void drain(int w, hipEvent_t* ev) {
    const HostSpan* held[2] = {nullptr, nullptr};
    auto start = [&](int s) {
      held[s] = nullptr;
      if (failed()) return;
      const size_t i = next.fetch_add(1);
      if (i >= chunks.size()) return;
      const HostSpan& c = chunks[i];
      hipError_t e = hipMemcpyAsync(slot(w, s), c.dev, c.count * esz, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(ev[s], stream);
      if (e != hipSuccess) return fail(e);
      held[s] = &c;
    };
    start(0);
    start(1);
    for (int s = 0; held[s]; s ^= 1) {
      const hipError_t e = hipEventSynchronize(ev[s]);
      if (e != hipSuccess) return fail(e);
      unload(slot(w, s), held[s]->host, held[s]->count, esz, as_double);
      start(s);
    }
  }

  void feed(int w, hipEvent_t* ev) {
    for (int s = 0, n = 0; !failed(); s ^= 1, ++n) {
      const size_t i = next.fetch_add(1);
      if (i >= chunks.size()) return;
      const HostSpan& c = chunks[i];
      hipError_t e = n >= 2 ? hipEventSynchronize(ev[s]) : hipSuccess;  // the slot's last copy
      if (e == hipSuccess) {
        fill(slot(w, s), c.host, c.count, esz, as_double);
        e = hipMemcpyAsync(c.dev, slot(w, s), c.count * esz, hipMemcpyHostToDevice, stream);
      }
      if (e == hipSuccess) e = hipEventRecord(ev[s], stream);
      if (e != hipSuccess) return fail(e);
    }
  }
};

hipError_t copy(hipStream_t stream, const HostSpan* spans, int nspans, size_t esz, bool as_double,
                bool to_host, bool wait) {
  size_t bytes = 0;
  for (int i = 0; i < nspans; ++i) bytes += spans[i].count * esz;
  bool staged = worth_staging(bytes, as_double, to_host);
  for (int i = 0; i < nspans && staged && !as_double; ++i) staged = !pinned(spans[i].host);
  StagingHold held(!staged ? 0 : to_host || as_double ? bytes : bytes / 2);
  if (!held.staging) return copy_direct(stream, spans, nspans, esz, as_double, to_host, wait);
  Job job;
  try {
    job.cut(spans, nspans, bytes, esz, as_double);
  } catch (const std::bad_alloc&) {  // nothing has been queued by then
    return copy_direct(stream, spans, nspans, esz, as_double, to_host, wait);
  }
  // the workers' events belong to the stream's device, which need not be the
  // caller's current one
  int current = 0;
  hipError_t e = hipGetDevice(&current);
  if (e == hipSuccess) e = hipStreamGetDevice(stream, &job.device);
  if (e == hipSuccess) {
    job.stream = stream;
    job.esz = esz;
    job.as_double = as_double;
    job.to_host = to_host;
    job.staging = held.staging;
    const size_t half = (job.chunks.size() + 1) / 2;
    const int workers = half < (size_t)kWorkers ? (int)half : kWorkers;
    const std::function<void(int)> work = [&job](int w) { job.work(w); };
    g_helpers->run(workers - 1, work);
    e = (hipError_t)job.error.load();
    (void)hipSetDevice(current);  // worker 0 was this thread
    const hipError_t es = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = es;
  }
  return e;
}

}  // namespace

hipError_t copy_spans(hipStream_t stream, const HostSpan* spans, int nspans, size_t esz,
                      bool as_double, bool to_host, bool wait) {
  try {
    return copy(stream, spans, nspans, esz, as_double, to_host, wait);
  } catch (const std::bad_alloc&) {  // no copy has been queued by then
    return hipErrorOutOfMemory;
  }
}

void transfer_user_add() {
  std::lock_guard<std::mutex> hold(g_lock);
  ++g_users;
}

void transfer_user_drop() {
  std::lock_guard<std::mutex> hold(g_lock);
  --g_users;
  staging_free_if_idle();
}

}  // namespace rhy
