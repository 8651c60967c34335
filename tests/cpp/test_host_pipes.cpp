// The pool of host pipes over a counting runtime with a limited amount of
// pinned memory: what idle pipes are kept, what gives them back, and that
// many callers at once do not make and unmake pipes.  Host code only.
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <stdexcept>
#include <thread>
#include <vector>

#include "host_pipes.hpp"

static int g_bad = 0;
#define EXPECT(x)                                                  \
  do {                                                             \
    if (!(x)) std::printf("line %d: %s\n", __LINE__, #x), ++g_bad; \
  } while (0)

struct Fake {
  using Stream = int*;
  using Error = int;
  static constexpr int kOk = 0;
  struct DeviceScope {
    explicit DeviceScope(int) {}
  };
  static inline std::mutex mu;
  static inline std::map<void*, size_t> live;
  static inline size_t pinned = 0, limit = ~size_t(0);
  static inline int streams = 0, streams_made = 0, bad_frees = 0;
  static void check(int e, const char* what) {
    if (e) throw std::runtime_error(what);
  }
  static int stream_create(int** s) {
    std::lock_guard<std::mutex> lk(mu);
    *s = new int;
    ++streams;
    ++streams_made;
    return 0;
  }
  static void stream_destroy(int* s) {
    std::lock_guard<std::mutex> lk(mu);
    delete s;
    --streams;
  }
  static int pinned_alloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    if (pinned + bytes > limit) return 2;
    *p = std::malloc(1);
    live[*p] = bytes;
    pinned += bytes;
    return 0;
  }
  static void pinned_free(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = live.find(p);
    if (it == live.end()) {
      ++bad_frees;
      return;
    }
    pinned -= it->second;
    live.erase(it);
    std::free(p);
  }
};

using namespace ecl::lib;
using Pool = PipePool<Fake>;
using Pipe = HostPipe<Fake>;
constexpr size_t MiB = size_t(1) << 20;

int main() {
  {  // a pipe comes back to the next caller of its device, with its buffers
    Pool pool;
    auto p = pool.take(3);
    p->reserve(pool, 2, 100, 3 * MiB);
    EXPECT(Fake::pinned == 2 * (MiB + 3 * MiB) && Fake::streams == 2);
    Pipe* was = p.get();
    pool.give(std::move(p));
    EXPECT(pool.take(4).get() != was);
    p = pool.take(3);
    EXPECT(p.get() == was && p->device == 3);
    p->reserve(pool, 2, 2 * MiB, 50);
    EXPECT(Fake::pinned == 2 * (2 * MiB + 3 * MiB) && Fake::streams == 2);
    pool.give(std::move(p));
    pool.release(4);
    EXPECT(Fake::streams == 2);
    pool.release(3);
    EXPECT(Fake::pinned == 0 && Fake::streams == 0);
    for (int odd : {-1, kPipeDevices, 1000}) {  // devices without a pool
      pool.give(pool.take(odd));
      pool.release(odd);
    }
  }
  EXPECT(Fake::pinned == 0 && Fake::streams == 0);
  {  // at most kIdlePipes are kept
    Pool pool;
    std::vector<std::unique_ptr<Pipe>> all;
    for (size_t i = 0; i < 2 * kIdlePipes; ++i) {
      all.push_back(pool.take(0));
      all.back()->reserve(pool, 1, 1, 1);
    }
    for (auto& p : all) pool.give(std::move(p));
    EXPECT(Fake::pinned == kIdlePipes * 2 * MiB);
  }
  EXPECT(Fake::pinned == 0 && Fake::streams == 0);
  {  // an allocation that would fail gets the idle pipes' memory, of every device
    Pool pool;
    std::vector<std::unique_ptr<Pipe>> all;
    for (int d = 0; d < 4; ++d) {
      all.push_back(pool.take(d));
      all.back()->reserve(pool, 1, MiB, MiB);
    }
    auto busy = std::move(all.back());
    all.pop_back();
    for (auto& p : all) pool.give(std::move(p));
    Fake::limit = 8 * MiB;
    busy->reserve(pool, 1, 7 * MiB, MiB);  // the 6 MiB of idle pipes are in its way
    EXPECT(Fake::pinned == 8 * MiB && busy->cap_in[0] == 7 * MiB);
    // and one that fails all the same leaves a pipe that can be used and freed
    bool threw = false;
    try {
      busy->reserve(pool, 3, 7 * MiB, MiB);
    } catch (const std::runtime_error&) {
      threw = true;
    }
    EXPECT(threw && busy->pin_in[1] == nullptr && busy->cap_in[1] == 0);
    threw = false;
    try {
      busy->reserve(pool, 1, 9 * MiB, MiB);
    } catch (const std::runtime_error&) {
      threw = true;
    }
    EXPECT(threw && busy->pin_in[0] == nullptr && busy->cap_in[0] == 0);
    busy->reserve(pool, 1, 2 * MiB, MiB);
    EXPECT(busy->cap_in[0] == 2 * MiB);
    Fake::limit = ~size_t(0);
  }
  EXPECT(Fake::pinned == 0 && Fake::streams == 0);
  {  // 16 callers at once, again and again: no pipe is made after the first round
    Pool pool;
    constexpr int kThreads = 16, kRounds = 50;
    std::mutex mu;
    std::condition_variable cv;
    int arrived = 0;
    int made_first = 0;
    auto barrier = [&](int round) {
      std::unique_lock<std::mutex> lk(mu);
      ++arrived;
      if (arrived == kThreads * round) cv.notify_all();
      cv.wait(lk, [&] { return arrived >= kThreads * round; });
    };
    Fake::streams_made = 0;
    std::vector<std::thread> th;
    for (int t = 0; t < kThreads; ++t)
      th.emplace_back([&, t] {
        for (int r = 0; r < kRounds; ++r) {
          auto p = pool.take(0);
          p->reserve(pool, 3, MiB, MiB);
          barrier(2 * r + 1);  // all of them hold one
          if (t == 0 && r == 0) made_first = Fake::streams_made;
          pool.give(std::move(p));
          barrier(2 * r + 2);
        }
      });
    for (auto& t : th) t.join();
    EXPECT(made_first == 3 * kThreads && Fake::streams_made == made_first);
  }
  EXPECT(Fake::pinned == 0 && Fake::streams == 0 && Fake::bad_frees == 0);
  std::printf(g_bad ? "FAILED\n" : "ALL OK\n");
  return g_bad != 0;
}
