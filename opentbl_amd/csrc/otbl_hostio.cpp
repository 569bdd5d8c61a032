// Large fields of a mixed box read to the host as doubles.
//
// The FP32 values cross the host link and are widened by the host's threads:
// half the bytes of widening on the GPU first.  The copy through page-locked
// staging and the widening run side by side, chunk by chunk; the same doubles
// arrive either way.  Bound by the link, FP32 at 57 GB/s (23 ms for the 1.3 GB of
// a 1536 x 315 x 1024 field) unless the host's CPUs are busy.  Measured, ms per
// field, widened on the GPU -> here: 48.4 -> 31.5 there, in a program whose own 16
// threads spin between the reads on 16 CPUs.  Such a program waits 6 ms for its
// CPUs whatever the size, so smaller fields stay on the GPU's widening: 640 x 144
// x 160 1.6 -> 6.7 (1.0 with idle CPUs), 387 x 113 x 98 0.54 -> 6.3 (0.43).  From
// 2^27 values on the link's saving, 10 ms, is above that.
#include <emmintrin.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdio>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "otbl_internal.h"

namespace otbl {

// values per staging slot: copies of 8 MB (of 2 MB: 20% of the time between them)
static constexpr size_t STAGE = size_t(2) << 20;
// widening threads: about 6 GB/s each, and the host's memory is full at 10
static constexpr int THREADS = 10;
// fewest CPUs of the calling thread for which the threads are worth waking: ten of
// them bound to 1, 2, 4, 6 CPUs widen the largest field above (2.7 GB of doubles)
// in 180, 92, 61, 52 ms at best, the GPU's widening takes 48
static constexpr int MIN_CPUS = 6;

// CPUs that the calling thread may run on: its affinity mask, and the quota of
// its control group where there is one
static int usable_cpus() {
  static const int quota = [] {
    int n = 1 << 20;
    if (std::FILE *f = std::fopen("/sys/fs/cgroup/cpu.max", "r")) {
      long q = 0, p = 0; // "max 100000": no quota
      if (std::fscanf(f, "%ld %ld", &q, &p) == 2 && q > 0 && p > 0) n = (int)std::max(1L, q / p);
      std::fclose(f);
    }
    return n;
  }();
  const int most = 1 << 14; // CPUs in the mask
  cpu_set_t *set = CPU_ALLOC(most);
  if (!set) return 0;
  const size_t bytes = CPU_ALLOC_SIZE(most);
  const int n = sched_getaffinity(0, bytes, set) == 0 ? CPU_COUNT_S(bytes, set) : 0;
  CPU_FREE(set);
  return std::min(n, quota);
}

void free_stage(Box &b) {
  if (b.stage) (void)hipHostFree(b.stage);
  b.stage = nullptr;
  b.readers.reset();
  for (hipEvent_t &e : b.stage_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

// staging of this box, made at its first read; false where the host has no
// page-locked memory for it
static bool make_stage(Box &b) {
  if (b.stage) return true;
  for (hipEvent_t &e : b.stage_ev)
    if (!e) OTBL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (hipHostMalloc((void **)&b.stage, STAGE * STAGE_SLOTS * sizeof(float)) != hipSuccess) {
    (void)hipGetLastError();
    b.stage = nullptr;
    return false;
  }
  return true;
}

// out[0..n) = in, past the caches where out is 16-byte aligned (it is read later,
// if at all)
static void widen(const float *in, double *out, size_t n) {
  size_t i = 0;
  if (n && (reinterpret_cast<uintptr_t>(out) & 15)) out[0] = in[0], i = 1;
  if ((reinterpret_cast<uintptr_t>(out + i) & 15) == 0)
    for (; i + 4 <= n; i += 4) {
      const __m128 x = _mm_loadu_ps(in + i);
      _mm_stream_pd(out + i, _mm_cvtps_pd(x));
      _mm_stream_pd(out + i + 2, _mm_cvtps_pd(_mm_movehl_ps(x, x)));
    }
  for (; i < n; ++i) out[i] = in[i];
}

namespace {
// One read: its chunks, and how far the copies and the threads are.
struct Reader {
  const float *stage = nullptr;
  double *host = nullptr;
  size_t n = 0;
  HostMean mean;
  int workers = 0;
  std::atomic<size_t> ready{0}; // chunks in the staging
  std::atomic<bool> stop{false};
  std::unique_ptr<std::atomic<int>[]> done; // workers that widened a chunk

  size_t chunks() const { return (n + STAGE - 1) / STAGE; }
  // part w of the chunk, then the FP64 mean flow of the rows that start in it
  void part(size_t c, int w, int of) {
    const size_t o = c * STAGE, m = std::min(STAGE, n - o);
    const size_t a = o + m * w / of, e = o + m * (w + 1) / of;
    widen(stage + (c % STAGE_SLOTS) * STAGE + (a - o), host + a, e - a);
    if (mean.v)
      for (size_t r = (a + mean.row - 1) / mean.row; r * mean.row < e; ++r) host[r * mean.row] = mean.at(r);
    _mm_sfence();
  }
  void work(int w) {
    for (size_t c = 0; c < chunks(); ++c) {
      for (int k = 0; ready.load(std::memory_order_acquire) <= c; ++k) {
        if (stop) return;
        if (k > 100) std::this_thread::yield();
      }
      part(c, w, workers);
      done[c].fetch_add(1, std::memory_order_release);
    }
  }
};

// The widening threads, shared by the mixed boxes of the process: made by the
// first read that wants them, ended with the last box that read (a thread per
// read costs 6 ms to end: the driver follows every stack that is unmapped).
class Pool {
public:
  explicit Pool(int k) {
    try {
      for (int w = 0; w < k; ++w) th.emplace_back(&Pool::run, this, w);
    } catch (const std::system_error &) {
      // as many as there are
    }
  }
  ~Pool() {
    {
      std::lock_guard<std::mutex> l(mu);
      quit = true;
    }
    cv.notify_all();
    for (std::thread &t : th) t.join();
  }
  int size() const { return (int)th.size(); }
  std::mutex busy; // held by the read whose threads these are

  void start(Reader *r) {
    {
      std::lock_guard<std::mutex> l(mu);
      job = r;
      ++gen;
      active = r->workers;
    }
    cv.notify_all();
  }
  void finish() { // every worker has left the job
    std::unique_lock<std::mutex> l(mu);
    idle.wait(l, [&] { return active == 0; });
    job = nullptr;
  }

private:
  void run(int w) {
    unsigned long seen = 0;
    std::unique_lock<std::mutex> l(mu);
    for (;;) {
      cv.wait(l, [&] { return quit || (gen != seen && job); });
      if (quit) return;
      seen = gen;
      Reader *r = job;
      if (w >= r->workers) continue;
      l.unlock();
      r->work(w);
      l.lock();
      if (--active == 0) idle.notify_all();
    }
  }
  std::vector<std::thread> th;
  std::mutex mu;
  std::condition_variable cv, idle;
  Reader *job = nullptr;
  unsigned long gen = 0;
  int active = 0;
  bool quit = false;
};

std::mutex g_pool_mu;
std::weak_ptr<Pool> g_pool;

std::shared_ptr<Pool> the_pool() {
  std::lock_guard<std::mutex> l(g_pool_mu);
  std::shared_ptr<Pool> p = g_pool.lock();
  if (!p) g_pool = p = std::make_shared<Pool>(std::min(THREADS, usable_cpus() - 1));
  return p;
}
} // namespace

bool field_to_host(Box &b, const float *dev, double *host, size_t n, const HostMean &mean) {
  if (n < b.read_min || usable_cpus() < MIN_CPUS || !make_stage(b)) return false;
  if (!b.readers) b.readers = the_pool();
  Pool &pool = *static_cast<Pool *>(b.readers.get());
  std::unique_lock<std::mutex> mine(pool.busy, std::try_to_lock);
  if (!mine || pool.size() == 0) return false; // another read has them: widened on the GPU
  Reader r;
  r.stage = b.stage;
  r.host = host;
  r.n = n;
  r.mean = mean;
  r.workers = pool.size();
  const size_t nc = r.chunks();
  r.done.reset(new std::atomic<int>[nc]);
  for (size_t c = 0; c < nc; ++c) r.done[c] = 0;
  auto copy = [&](size_t c) {
    const size_t o = c * STAGE, m = std::min(STAGE, n - o);
    const int s = (int)(c % STAGE_SLOTS);
    OTBL_HIP(hipMemcpyAsync(b.stage + s * STAGE, dev + o, m * sizeof(float), hipMemcpyDeviceToHost, b.s));
    OTBL_HIP(hipEventRecord(b.stage_ev[s], b.s));
  };
  auto widened = [&](size_t c) {
    while (r.done[c].load(std::memory_order_acquire) < r.workers) std::this_thread::yield();
  };
  pool.start(&r);
  try {
    size_t next = 0;
    while (next < nc && next < (size_t)STAGE_SLOTS) copy(next++);
    for (size_t c = 0; c < nc; ++c) {
      OTBL_HIP(hipEventSynchronize(b.stage_ev[c % STAGE_SLOTS]));
      r.ready.store(c + 1, std::memory_order_release);
      if (next < nc) { // into chunk c's slot
        widened(c);
        copy(next++);
      }
    }
  } catch (...) {
    r.stop = true;
    pool.finish();
    (void)hipStreamSynchronize(b.s); // nothing lands in the staging after this
    throw;
  }
  pool.finish();
  return true;
}

} // namespace otbl
