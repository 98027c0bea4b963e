// Copies between a caller's pageable arrays and the device.
//
// The runtime moves pageable memory at 15 (1.6 MB) to 29 GB/s (127 MB) up and
// 14 to 17 GB/s down; the link takes 56 GB/s from pinned memory in pieces of some MiB
// (21 GB/s in pieces of 512 KiB, 30 in 1 MiB).  Here the bytes go through
// pinned slots: a thread moves one piece between the caller's array and a slot
// while its other slot is on the link.  One thread copies 28
// GB/s, so a large copy takes two (three and four were no faster).  127 MB: 29
// -> 43 GB/s up, 17 -> 44 GB/s down; 25 MB: 32 -> 37 and 17 -> 32; 1.6 MB: 15 ->
// 18 and 14 -> 17.
#include "ii_internal.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>

namespace ii {

namespace {

constexpr int kPipeThreads = 2;                  // this one and a helper
constexpr size_t kPieceMax = (size_t)4 << 20;    // bytes of a slot
constexpr size_t kThreadBytes = (size_t)4 << 20; // the helper from twice that: it takes some
                                                 // tens of us to wake
// Smaller copies are the runtime's: its own staging has less latency than a
// slot and its event.  One Dhat on host arrays, us, through the runtime /
// through the slots, by the bytes each way: 72 KB 52 / 63, 243 KB 65 / 100,
// 768 KB 106 / 130, 1152 KB 165 / 152, 2.6 MB 287 / 260, 8.2 MB 632 / 620 (823
// before).
constexpr size_t kDirect = (size_t)1 << 20;
// A context pins a set of its own once it has moved this much by the runtime:
// pinning and freeing 16 MiB takes about 4 ms, what 400 MB up or 110 MB down
// gain.  Opening a context, uploading its links and closing it: 0.65 ms at
// 12x10x14x18 and 3.5 ms at 16^3x32, 4.9 and 6.3 ms with a set pinned at once.
constexpr size_t kPinAfter = (size_t)128 << 20;

}  // namespace

// A set of pinned slots, 16 MiB.  Pinning one takes time (kPinAfter), so the sets
// belong to the device and not to a context: a copy takes the set its context
// used last, else one with nothing in flight, else pins a new one.  So a copy
// never waits for another context's kernels or copies, its own stream orders
// the uses of a set in flight, and there are never more sets than contexts
// that copy: programs that use their contexts one after the other pin one.
//
// The helper thread belongs to the set and sleeps between copies.  It takes
// pieces while there are any; a copy waits only for pieces that it has taken,
// not for it to wake.  (A thread started and joined for each copy waited a time
// slice of 4 ms for a core while the caller's BLAS threads spun between calls:
// Dhat at 16^3x32 up to 3.9 ms, 0.9 alone.)
struct HostJob {
  virtual void run() = 0;
};
struct HostSet {
  char* pin = nullptr;
  hipEvent_t ev[2 * kPipeThreads] = {};
  ii_context* owner = nullptr;  // whose stream may have pieces in flight
  bool busy = false;            // a copy is running on it
  HostSet* next = nullptr;
  std::mutex jmu;
  std::condition_variable jcv;
  std::thread helper;
  bool tried = false, stop = false, active = false;
  HostJob* job = nullptr;
  // offers j to the helper
  void post(HostJob* j) {
    if (!tried) {
      tried = true;
      try {
        helper = std::thread([this] { serve(); });
      } catch (const std::exception&) {
        // no thread to be had: the callers take all the pieces
      }
    }
    std::lock_guard<std::mutex> l(jmu);
    job = j;
    jcv.notify_all();
  }
  // the job is not offered any more, and the helper is not in it
  void retract() {
    std::unique_lock<std::mutex> l(jmu);
    job = nullptr;
    jcv.wait(l, [&] { return !active; });
  }
  void serve() {
    std::unique_lock<std::mutex> l(jmu);
    for (;;) {
      jcv.wait(l, [&] { return stop || job; });
      if (stop) return;
      HostJob* j = job;
      job = nullptr;
      active = true;
      l.unlock();
      j->run();
      l.lock();
      active = false;
      jcv.notify_all();
    }
  }
  bool create() {
    bool ok = hipHostMalloc((void**)&pin, 2 * kPipeThreads * kPieceMax) == hipSuccess;
    for (auto& e : ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    return ok;
  }
  bool complete() const {
    for (auto& e : ev)
      if (hipEventQuery(e) != hipSuccess) {
        (void)hipGetLastError();  // not ready is no error of the caller's launches
        return false;
      }
    return true;
  }
  ~HostSet() {
    {
      std::lock_guard<std::mutex> l(jmu);
      stop = true;
      jcv.notify_all();
    }
    if (helper.joinable()) helper.join();
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (pin) (void)hipHostFree(pin);
  }
};
struct HostPipe {
  std::mutex mu;  // over the list, never held while a copy or a kernel runs
  HostSet* sets = nullptr;
  int nsets = 0, users = 0;  // users: contexts that have copied
};
constexpr int kPipeDevices = 64;  // as many as noalloc_setup lets a context be created on
static HostPipe g_pipe[kPipeDevices];

// The stream of a context that goes has been waited for.  Sets beyond the number
// of contexts that may use one are freed, outside the lock: freeing pinned
// memory may wait for the device.
void host_pipe_release(ii_context* ctx) {
  HostPipe* H = static_cast<HostPipe*>(ctx->host_pipe);
  if (!H) return;
  ctx->host_pipe = nullptr;
  HostSet* gone = nullptr;
  {
    std::lock_guard<std::mutex> lock(H->mu);
    for (HostSet* s = H->sets; s; s = s->next)
      if (s->owner == ctx) s->owner = nullptr;
    --H->users;
    for (HostSet** at = &H->sets; *at && H->nsets > H->users;) {
      HostSet* s = *at;
      if (s->busy || (s->owner && !s->complete())) {
        at = &s->next;
        continue;
      }
      *at = s->next;
      --H->nsets;
      s->next = gone;
      gone = s;
    }
  }
  while (gone) {
    HostSet* s = gone;
    gone = s->next;
    delete s;
  }
}

// a set for a copy of ctx of so many bytes; null if none is to be pinned for it
// yet, or none can be (the copy is the runtime's then)
static HostSet* take_set(ii_context* ctx, size_t bytes) {
  HostPipe* H = &g_pipe[ctx->device];
  HostSet* s = nullptr;
  {
    std::lock_guard<std::mutex> lock(H->mu);
    if (!ctx->host_pipe) {
      ++H->users;
      ctx->host_pipe = H;
    }
    for (s = H->sets; s && (s->busy || s->owner != ctx);) s = s->next;
    if (!s)
      for (s = H->sets; s && (s->busy || !s->complete());) s = s->next;
    if (s) {
      s->owner = ctx;
      s->busy = true;
      return s;
    }
  }
  ctx->host_moved += bytes;
  if (ctx->host_moved < kPinAfter) return nullptr;
  s = new (std::nothrow) HostSet();  // pinned outside the lock
  if (!s || !s->create()) {
    delete s;
    (void)hipGetLastError();
    return nullptr;
  }
  s->owner = ctx;
  s->busy = true;
  std::lock_guard<std::mutex> lock(H->mu);
  s->next = H->sets;
  H->sets = s;
  ++H->nsets;
  return s;
}
static void give_set(ii_context* ctx, HostSet* s) {
  std::lock_guard<std::mutex> lock(static_cast<HostPipe*>(ctx->host_pipe)->mu);
  s->busy = false;
}

// Runs work(t, take, e) on each thread t: take(&first, &bytes) hands out the
// pieces of [0, bytes) in order until none is left or a thread has failed, e is
// the thread's error.  After a failure nothing of the copy is left in flight.
template <typename Piece>
static ii_status run_pieces(ii_context* ctx, HostSet* H, size_t bytes, const Piece& work) {
  const int want = (int)std::max<size_t>(1, bytes / kThreadBytes);
  const int nthr = std::min(kPipeThreads, want);
  size_t piece = (bytes + 2 * nthr - 1) / (2 * nthr);
  piece = std::min(kPieceMax, (piece + 4095) / 4096 * 4096);
  const size_t n = (bytes + piece - 1) / piece;
  std::atomic<size_t> next{0};
  std::atomic<int> err{hipSuccess};
  auto pieces = [&](int t) {
    hipError_t e = t ? hipSetDevice(ctx->device) : hipSuccess;
    work(t, [&](size_t* first, size_t* len) {
      const size_t k = e == hipSuccess && err == hipSuccess ? next++ : n;
      if (k >= n) return false;
      *first = k * piece;
      *len = std::min(piece, bytes - *first);
      return true;
    }, e);
    if (e != hipSuccess) err = e;
  };
  struct Job final : HostJob {
    const decltype(pieces)& f;
    explicit Job(const decltype(pieces)& f) : f(f) {}
    void run() override { f(1); }
  } job(pieces);
  if (nthr > 1) H->post(&job);
  pieces(0);
  if (nthr > 1) H->retract();
  if (err != hipSuccess) {
    (void)hipStreamSynchronize(ctx->stream);
    return set_error(ctx, II_ERR_DEVICE,
                     std::string("host copy: ") + hipGetErrorString((hipError_t)err.load()));
  }
  return II_OK;
}

// Whether p is memory the runtime does not know.  Pinned memory goes straight
// to the link (53-57 GB/s, where the slots reach 37-44), and what else the
// runtime knows is its own to copy.
static bool pageable(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // "not known" may come as an error
  return true;
}

ii_status copy_to_device(ii_context* ctx, void* dst, const void* src, size_t bytes) {
  HostSet* H = bytes < kDirect || !pageable(src) ? nullptr : take_set(ctx, bytes);
  if (!H) {
    II_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    if (bytes >= kDirect) II_HIP(ctx, hipStreamSynchronize(ctx->stream));  // src has been read
    return II_OK;
  }
  const ii_status st = run_pieces(ctx, H, bytes, [&](int t, auto&& take, hipError_t& e) {
    size_t first = 0, len = 0;
    for (int i = 0; take(&first, &len); ++i) {
      const int slot = 2 * t + (i & 1);
      char* p = H->pin + slot * kPieceMax;
      if ((e = hipEventSynchronize(H->ev[slot])) != hipSuccess) return;
      std::memcpy(p, (const char*)src + first, len);
      if ((e = hipMemcpyAsync((char*)dst + first, p, len, hipMemcpyHostToDevice, ctx->stream)) !=
          hipSuccess)
        return;
      if ((e = hipEventRecord(H->ev[slot], ctx->stream)) != hipSuccess) return;
    }
  });
  give_set(ctx, H);
  return st;
}

ii_status copy_to_host(ii_context* ctx, void* dst, const void* src, size_t bytes) {
  HostSet* H = bytes < kDirect || !pageable(dst) ? nullptr : take_set(ctx, bytes);
  if (!H) {
    II_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    II_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return II_OK;
  }
  const ii_status st = run_pieces(ctx, H, bytes, [&](int t, auto&& take, hipError_t& e) {
    size_t first[2] = {0, 0}, len[2] = {0, 0};
    auto request = [&](int b) {
      const int slot = 2 * t + b;
      len[b] = 0;
      size_t f = 0, l = 0;
      if (!take(&f, &l)) return;
      first[b] = f;
      if ((e = hipMemcpyAsync(H->pin + slot * kPieceMax, (const char*)src + f, l,
                              hipMemcpyDeviceToHost, ctx->stream)) != hipSuccess)
        return;
      if ((e = hipEventRecord(H->ev[slot], ctx->stream)) == hipSuccess) len[b] = l;
    };
    request(0);
    for (int b = 0; len[b]; b ^= 1) {
      request(b ^ 1);
      const int slot = 2 * t + b;
      if (e != hipSuccess || (e = hipEventSynchronize(H->ev[slot])) != hipSuccess) return;
      std::memcpy((char*)dst + first[b], H->pin + slot * kPieceMax, len[b]);
    }
  });
  give_set(ctx, H);
  return st;
}

}  // namespace ii
