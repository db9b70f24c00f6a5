// Many host arrays into one device buffer: kh_upload_many.
//
// An adapter that a loader process leaves in shared memory (load_lora_shm_multi.py:40-61) is some 1400 pageable float16 arrays.
// Copied one by one each costs a runtime call and the runtime's own staging (17 us apiece, 14 GB/s on the arrays of one
// 1280-wide transformer); here worker threads gather them into two pinned staging chunks in turn while the other chunk is on
// its way to the device, so the upload runs at the rate of the host's memory or of the link (57 GB/s from pinned memory).
// Merging a rank-64 float16 adapter into the 52 linears of a 1280-wide transformer of five blocks, the whole call: 2.1 -> 1.45 ms for
// matrices that have just been written, 1.95 -> 1.1 where the same host arrays are merged again (their lines are then in the CPU's
// caches; every call copies all bytes).  A rank-8 adapter of one 640-wide block 0.38 -> 0.30 and 0.30 -> 0.20.
#include "kh_common.h"
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace {

// Worker threads that live as long as the process, started by the first upload and shared by all: one job at a time, a
// second caller meanwhile copies on its own thread (try_lock).  Never destroyed: nothing runs in them at exit.
class Pool {
 public:
  static Pool& get() {
    static Pool* p = new Pool();
    return *p;
  }
  // fn(part, parts) on every worker and on the caller
  template <class F>
  void run(F fn) {
    std::unique_lock<std::mutex> one(busy_, std::try_to_lock);
    if (!one.owns_lock() || workers_ == 0) {
      fn(0, 1);
      return;
    }
    auto call = [](void* f, int part, int parts) { (*static_cast<F*>(f))(part, parts); };
    {
      std::lock_guard<std::mutex> l(m_);
      job_ = call;
      arg_ = &fn;
      left_ = workers_;
      ++serial_;
    }
    wake_.notify_all();
    fn(workers_, workers_ + 1);
    std::unique_lock<std::mutex> l(m_);
    done_.wait(l, [&] { return left_ == 0; });
  }

 private:
  Pool() {
    const unsigned hw = std::thread::hardware_concurrency();
    const int want = hw > 8 ? 7 : hw > 1 ? (int)hw - 1 : 0;
    for (int i = 0; i < want; ++i) {
      try {
        std::thread([this, i] { work(i); }).detach();
        ++workers_;
      } catch (...) {
        break;
      }
    }
  }
  void work(int part) {
    uint64_t seen = 0;
    for (;;) {
      void (*job)(void*, int, int);
      void* arg;
      int parts;
      {
        std::unique_lock<std::mutex> l(m_);
        wake_.wait(l, [&] { return serial_ != seen; });
        seen = serial_;
        job = job_; arg = arg_; parts = workers_ + 1;
      }
      job(arg, part, parts);
      {
        std::lock_guard<std::mutex> l(m_);
        if (--left_ == 0) done_.notify_one();
      }
    }
  }
  std::mutex busy_, m_;
  std::condition_variable wake_, done_;
  void (*job_)(void*, int, int) = nullptr;
  void* arg_ = nullptr;
  int workers_ = 0, left_ = 0;
  uint64_t serial_ = 0;
};

}  // namespace

// See include/katz_hip.h.
KH_EXPORT int kh_upload_many(const void* const* src, const int64_t* bytes, const int64_t* offset, int64_t n, void* dst, void* staging,
                             int64_t staging_bytes, void* stream) {
  if (!src || !bytes || !offset || n <= 0 || !dst || !staging || staging_bytes < 2 * 4096) return KH_ERR_INVALID_ARG;
  for (int64_t i = 0; i < n; ++i)
    if (!src[i] || bytes[i] < 0 || offset[i] < 0 || (i > 0 && offset[i] < offset[i - 1] + bytes[i - 1])) return KH_ERR_INVALID_ARG;
  const int64_t total = offset[n - 1] + bytes[n - 1], chunk = staging_bytes / 2 / 4096 * 4096;
  hipStream_t s = (hipStream_t)stream;
  hipEvent_t ev[2] = {nullptr, nullptr};
  hipError_t e = hipSuccess;
  for (int k = 0; k < 2 && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
  int64_t first = 0;                                   // the first array that reaches into the current chunk
  int used = 0;
  for (int64_t at = 0; at < total && e == hipSuccess; at += chunk, ++used) {
    char* stage = static_cast<char*>(staging) + (used & 1) * chunk;
    const int64_t end = at + chunk < total ? at + chunk : total;
    if (used >= 2) e = hipEventSynchronize(ev[used & 1]);   // that half has left for the device
    if (e != hipSuccess) break;
    while (first < n && offset[first] + bytes[first] <= at) ++first;
    // every thread takes an equal stretch of the chunk, whatever arrays that covers
    Pool::get().run([&](int part, int parts) {
      const int64_t len = end - at, lo = at + len * part / parts, hi = at + len * (part + 1) / parts;
      for (int64_t i = first; i < n && offset[i] < hi; ++i) {
        const int64_t a = offset[i] > lo ? offset[i] : lo, b = offset[i] + bytes[i] < hi ? offset[i] + bytes[i] : hi;
        if (a < b) std::memcpy(stage + (a - at), static_cast<const char*>(src[i]) + (a - offset[i]), (size_t)(b - a));
      }
    });
    e = hipMemcpyAsync(static_cast<char*>(dst) + at, stage, (size_t)(end - at), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipEventRecord(ev[used & 1], s);
  }
  // the staging memory is the caller's again when this returns
  for (int k = 0; k < 2; ++k) {
    if (e == hipSuccess && used > k) e = hipEventSynchronize(ev[k]);
    if (ev[k] != nullptr) (void)hipEventDestroy(ev[k]);
  }
  return e == hipSuccess ? KH_OK : (int)e;
}
