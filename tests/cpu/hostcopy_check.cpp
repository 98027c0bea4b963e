// The staged host copies (iroiro_amd/csrc/ii_hostcopy.hip), compiled unchanged
// for the host against a stand-in for the HIP calls they make: a stream is a
// thread that runs what was queued on it in order, and a copy moves its bytes
// when the stream reaches it, as the copy engines do.  What one context does
// must be right whatever another context of the device has in flight.
// Exits non-zero on the first violation.
#include "../../iroiro_amd/csrc/ii_hostcopy.hip"

#include <dlfcn.h>
#include <pthread.h>

#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <functional>
#include <memory>
#include <vector>

#define CHECK(c, ...)                                        \
  do {                                                       \
    if (!(c)) {                                              \
      std::fprintf(stderr, "hostcopy_check: " __VA_ARGS__); \
      std::fprintf(stderr, "\n");                            \
      std::_Exit(1);                                         \
    }                                                        \
  } while (0)

// ------------------------------------------------------------ the stand-in
namespace sim {

struct Stream {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  bool busy = false, stop = false;
  std::thread th{[this] { run(); }};
  void run() {
    std::unique_lock<std::mutex> l(mu);
    for (;;) {
      cv.wait(l, [&] { return stop || !q.empty(); });
      if (q.empty()) return;
      auto f = std::move(q.front());
      q.pop_front();
      busy = true;
      l.unlock();
      f();
      l.lock();
      busy = false;
      cv.notify_all();
    }
  }
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> l(mu);
    q.push_back(std::move(f));
    cv.notify_all();
  }
  bool idle() {
    std::lock_guard<std::mutex> l(mu);
    return q.empty() && !busy;
  }
  void sync() {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [&] { return q.empty() && !busy; });
  }
  ~Stream() {
    {
      std::lock_guard<std::mutex> l(mu);
      stop = true;
      cv.notify_all();
    }
    th.join();
  }
};

// a recorded point of a stream; never recorded: complete
struct Mark {
  std::mutex mu;
  std::condition_variable cv;
  bool done = false;
  void set() {
    std::lock_guard<std::mutex> l(mu);
    done = true;
    cv.notify_all();
  }
  void wait() {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [&] { return done; });
  }
};
struct Event {
  std::mutex mu;
  std::shared_ptr<Mark> m;
  std::shared_ptr<Mark> mark() {
    std::lock_guard<std::mutex> l(mu);
    return m;
  }
};

std::atomic<int> pins{0}, pin_calls{0}, fail_copy{-1}, copies{0};
std::atomic<bool> no_pins{false};
Mark* free_gate = nullptr;  // pinned memory is freed when the device lets go
const char *pinned_lo = nullptr, *pinned_hi = nullptr;  // the caller's pinned memory

Stream* of(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
Event* of(hipEvent_t e) { return reinterpret_cast<Event*>(e); }

}  // namespace sim

// threads started while `late` is set get no core for that many milliseconds
namespace sim {
std::atomic<int> late{0};
struct Start {
  void* (*f)(void*);
  void* arg;
  int ms;
};
void* late_start(void* v) {
  Start s = *static_cast<Start*>(v);
  delete static_cast<Start*>(v);
  std::this_thread::sleep_for(std::chrono::milliseconds(s.ms));
  return s.f(s.arg);
}
}  // namespace sim
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
  if (!sim::late) return real(t, a, f, arg);
  return real(t, a, sim::late_start, new sim::Start{f, arg, sim::late});
}

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (sim::no_pins) return hipErrorOutOfMemory;
  ++sim::pin_calls;
  *p = std::malloc(n);
  ++sim::pins;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  if (sim::free_gate) sim::free_gate->wait();
  std::free(p);
  --sim::pins;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new sim::Event());
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete sim::of(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  auto m = std::make_shared<sim::Mark>();
  {
    std::lock_guard<std::mutex> l(sim::of(e)->mu);
    sim::of(e)->m = m;
  }
  sim::of(s)->push([m] { m->set(); });
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (auto m = sim::of(e)->mark()) m->wait();
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  auto m = sim::of(e)->mark();
  if (!m) return hipSuccess;
  std::lock_guard<std::mutex> l(m->mu);
  return m->done ? hipSuccess : hipErrorNotReady;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (auto m = sim::of(e)->mark()) sim::of(s)->push([m] { m->wait(); });
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  sim::of(s)->sync();
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  if (sim::fail_copy >= 0 && sim::fail_copy-- == 0) return hipErrorUnknown;
  ++sim::copies;
  sim::of(st)->push([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  if (p < sim::pinned_lo || p >= sim::pinned_hi) return hipErrorInvalidValue;
  a->type = hipMemoryTypeHost;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
}

namespace ii {
ii_status set_error(ii_context* ctx, ii_status st, const std::string& msg) {
  if (ctx) ctx->err = msg;
  return st;
}
}  // namespace ii

using namespace ii;

// ------------------------------------------------------------ the checks
namespace {

struct Ctx {
  sim::Stream s;
  ii_context c;
  explicit Ctx(bool fresh = false) {
    c.stream = reinterpret_cast<hipStream_t>(&s);
    if (!fresh) c.host_moved = kPinAfter;  // a context that has copied a lot
  }
  // earlier work on the stream, ms long
  void kernel(int ms) {
    s.push([ms] { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); });
  }
  ~Ctx() {  // as ii_context_destroy
    s.sync();
    host_pipe_release(&c);
  }
};

std::vector<char> pattern(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i * 2654435761u >> 13) + seed * 97u + (i >> 12));
  return v;
}

void upload(Ctx& x, std::vector<char>& dev, const std::vector<char>& src) {
  CHECK(copy_to_device(&x.c, dev.data(), src.data(), src.size()) == II_OK, "upload failed");
}
void download(Ctx& x, std::vector<char>& dst, const std::vector<char>& dev) {
  CHECK(copy_to_host(&x.c, dst.data(), dev.data(), dev.size()) == II_OK, "download failed");
}

const size_t kSizes[] = {1 << 20, (1 << 20) + 8, 3 << 20, (8 << 20) + 24, 12 << 20, (37 << 20) + 8};

// one context: every byte both ways, the source free once the call returned
void round_trips() {
  Ctx a;
  for (size_t n : kSizes) {
    std::vector<char> src = pattern(n, 1), keep = src, dev(n), dst(n);
    a.kernel(2);
    upload(a, dev, src);
    std::fill(src.begin(), src.end(), 0);
    download(a, dst, dev);
    CHECK(dst == keep, "round trip of %zu bytes", n);
  }
}

// B downloads (or uploads) while A's upload is queued behind A's earlier work
void other_context() {
  Ctx a, b;
  for (size_t n : kSizes)
    for (int up = 0; up < 2; ++up) {
      std::vector<char> sa = pattern(n, 2), sb = pattern(n, 3), da(n), db(n), hb(n);
      a.kernel(20);
      upload(a, da, sa);
      if (up) {
        upload(b, db, sb);
        b.s.sync();
        CHECK(db == sb, "upload of %zu bytes beside another context's", n);
      } else {
        download(b, hb, sb);
        CHECK(hb == sb, "download of %zu bytes beside another context's upload", n);
      }
      a.s.sync();
      CHECK(da == sa, "upload of %zu bytes beside another context's %s", n,
            up ? "upload" : "download");
    }
}

// contexts in threads of their own, sizes and earlier work at random
void threads() {
  std::vector<std::thread> th;
  for (int t = 0; t < 3; ++t)
    th.emplace_back([t] {
      for (int round = 0; round < 2; ++round) {
        Ctx x;
        unsigned r = 12345u + 77u * t + round;
        for (int i = 0; i < 12; ++i) {
          r = r * 1664525u + 1013904223u;
          const size_t n = kSizes[(r >> 20) % 6];
          std::vector<char> src = pattern(n, r), keep = src, dev(n), dst(n);
          if (r & 0x10000) x.kernel(1 + (r >> 28));
          upload(x, dev, src);
          std::fill(src.begin(), src.end(), 0);
          download(x, dst, dev);
          CHECK(dst == keep, "thread %d, copy %d of %zu bytes", t, i, n);
        }
      }
    });
  for (auto& t : th) t.join();
}

// While A's stream is held by a kernel, with an upload queued behind it or a
// download waiting for it, B's copies run: none waits for another's kernels.
void no_waiting() {
  const size_t n = 12 << 20;
  for (int down = 0; down < 2; ++down) {
    Ctx a, b;
    sim::Mark gate, done;
    std::vector<char> src = pattern(n, 7), da(n), ha(n), db(n), hb(n);
    upload(b, db, src);
    upload(a, da, src);  // both have copied before
    a.s.push([&] { gate.wait(); });
    std::thread ta([&] {
      if (down) download(a, ha, da);
      else upload(a, da, src);
    });
    std::this_thread::sleep_for(std::chrono::milliseconds(20));
    std::thread tb([&] {
      upload(b, db, src);
      download(b, hb, db);
      done.set();
    });
    bool ok = false;
    {
      std::unique_lock<std::mutex> l(done.mu);
      ok = done.cv.wait_for(l, std::chrono::seconds(20), [&] { return done.done; });
    }
    CHECK(ok, "a context waits for another one's kernel (%s)", down ? "its download" : "its upload");
    CHECK(hb == src, "copies beside a held stream");
    gate.set();
    ta.join();
    tb.join();
    a.s.sync();
  }
}

// a context that goes, and waits for the device to give up its slots, holds up
// no other one's copies
void closing() {
  const size_t n = 12 << 20;
  std::vector<char> src = pattern(n, 12), da(n), db(n), hb(n);
  sim::Mark gate, done;
  Ctx b;
  auto a = std::make_unique<Ctx>();
  a->kernel(20);
  upload(*a, da, src);
  upload(b, db, src);  // a set of its own
  b.s.sync();
  sim::free_gate = &gate;
  std::thread ta([&] { a.reset(); });
  std::this_thread::sleep_for(std::chrono::milliseconds(100));
  std::thread tb([&] {
    upload(b, db, src);
    download(b, hb, db);
    done.set();
  });
  bool ok = false;
  {
    std::unique_lock<std::mutex> l(done.mu);
    ok = done.cv.wait_for(l, std::chrono::seconds(20), [&] { return done.done; });
  }
  CHECK(ok, "a context waits for another one that goes");
  CHECK(hb == src, "copies beside a context that goes");
  gate.set();
  ta.join();
  tb.join();
  sim::free_gate = nullptr;
}

// a caller's pinned memory: one copy each way, between it and the device
void pinned_memory() {
  Ctx a;
  for (size_t n : kSizes) {
    std::vector<char> src = pattern(n, 9), keep = src, dev(n);
    sim::pinned_lo = src.data();
    sim::pinned_hi = src.data() + n;
    a.kernel(2);
    const int before = sim::copies;
    upload(a, dev, src);
    std::fill(src.begin(), src.end(), 0);
    download(a, src, dev);
    CHECK(src == keep, "pinned round trip of %zu bytes", n);
    CHECK(sim::copies == before + 2, "%d copies of pinned memory", sim::copies - before);
    sim::pinned_lo = sim::pinned_hi = nullptr;
  }
}

// a context pins nothing before it has copied a lot, unless a set is idle
void short_lived() {
  const size_t n = 37 << 20;
  std::vector<char> src = pattern(n, 11), dev(n), dst(n);
  const int before = sim::pin_calls;
  {
    Ctx a(true);
    upload(a, dev, src);
    download(a, dst, dev);
    CHECK(dst == src && sim::pin_calls == before, "a short-lived context pinned a set");
    upload(a, dev, src);
    CHECK(sim::pin_calls == before, "pinned after 111 MiB");
    upload(a, dev, src);
    CHECK(sim::pin_calls == before + 1, "not pinned after 148 MiB");
    Ctx b(true);
    a.s.sync();
    const int copies = sim::copies;
    upload(b, dev, src);
    CHECK(sim::copies > copies + 1 && sim::pin_calls == before + 1, "an idle set is taken");
  }
  CHECK(sim::pins == 0, "%d pinned blocks left", (int)sim::pins);
}

// a copy does not wait for its helper thread to get a core
void late_helper() {
  const size_t n = 37 << 20;
  std::vector<char> src = pattern(n, 10), dev(n), dst(n);
  Ctx a;
  sim::late = 3000;
  const auto t0 = std::chrono::steady_clock::now();
  upload(a, dev, src);
  download(a, dst, dev);
  const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  sim::late = 0;
  CHECK(dst == src, "copies without a helper");
  CHECK(s < 1.5, "copies waited %.1f s for their helper", s);
}

// as many sets of slots as contexts with copies in flight, and one for
// contexts used in turn
void set_count() {
  const int before = sim::pin_calls;
  {
    Ctx a, b, c;
    std::vector<char> src = pattern(12 << 20, 8), dev(src.size()), dst(src.size());
    for (int i = 0; i < 3; ++i)
      for (Ctx* x : {&a, &b, &c}) {
        upload(*x, dev, src);
        download(*x, dst, dev);
      }
    CHECK(sim::pin_calls == before + 1, "contexts in turn pinned %d sets", sim::pin_calls - before);
    std::vector<char> devs[3] = {dev, dev, dev};
    int k = 0;
    for (Ctx* x : {&a, &b, &c}) {
      x->kernel(30);
      upload(*x, devs[k++], src);
    }
    for (Ctx* x : {&a, &b, &c}) x->s.sync();
    CHECK(sim::pins <= 3, "three contexts pinned %d sets", (int)sim::pins);
  }
  CHECK(sim::pins == 0, "%d pinned blocks left", (int)sim::pins);
}

// a copy that fails leaves nothing of its own in flight, and the next is right
void failures() {
  Ctx a, b;
  for (size_t n : kSizes)
    for (int down = 0; down < 2; ++down)
      for (int at = 0; at < 4; ++at) {
        std::vector<char> src = pattern(n, 5), dev(n), dst(n);
        a.kernel(5);
        sim::fail_copy = at;
        const ii_status st = down ? copy_to_host(&a.c, dst.data(), src.data(), n)
                                  : copy_to_device(&a.c, dev.data(), src.data(), n);
        sim::fail_copy = -1;
        CHECK(st == II_OK || a.s.idle(), "copy of %zu bytes failed at its piece %d with work left",
              n, at);
        a.s.sync();
        download(b, dst, src);
        CHECK(dst == src, "download of %zu bytes after another context's failure", n);
      }
}

}  // namespace

int main() {
  round_trips();
  other_context();
  threads();
  no_waiting();
  closing();
  pinned_memory();
  sim::no_pins = true;  // copies without slots are the runtime's
  round_trips();
  other_context();
  sim::no_pins = false;
  set_count();
  failures();
  late_helper();
  short_lived();
  CHECK(sim::pins == 0, "%d pinned blocks left", (int)sim::pins);
  round_trips();  // the slots come back after the last context gave them up
  CHECK(sim::pins == 0, "%d pinned blocks left", (int)sim::pins);
  std::printf("hostcopy_check: ok\n");
  return 0;
}
