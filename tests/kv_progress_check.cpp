// KvProgress (relay_amd/csrc/host/host_common.h) with threads, run by test_kv_progress.py. Every
// wait has a deadline; a check that fails prints its line and ends the program.
#include "host_common.h"

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <memory>
#include <thread>

using relay_hip_host::KvProgress;
using namespace std::chrono_literals;

#define CHECK(x)                                              \
  do {                                                        \
    if (!(x)) {                                               \
      std::printf("line %d: %s\n", __LINE__, #x);             \
      std::fflush(stdout);                                    \
      std::_Exit(1);                                          \
    }                                                         \
  } while (0)

static std::future<void> waiter(KvProgress& p, int layer) {
  auto f = std::async(std::launch::async, [&p, layer] { p.reach(layer); });
  std::this_thread::sleep_for(100ms);  // it has entered the wait, or returned
  return f;
}
static bool done(std::future<void>& f, std::chrono::milliseconds t) { return f.wait_for(t) == std::future_status::ready; }

int main() {
  {  // no pass: at once, and nothing is recorded for it
    KvProgress p(2);
    auto w = waiter(p, 1);
    CHECK(done(w, 2s) && !p.record() && !p.running());
  }
  {  // a pass with an observer: at once, also for a layer it has not reached; it records
    KvProgress p(2);
    KvProgress::Pass pass(p, true);
    CHECK(p.record() && p.running());
    auto w = waiter(p, 1);
    CHECK(done(w, 2s));
  }
  {  // without one: not before the pass is over, and a pass that follows at once does not prolong it
    KvProgress p(2);
    auto pass = std::make_unique<KvProgress::Pass>(p, false);
    CHECK(!p.record());
    auto w = waiter(p, 0);
    CHECK(!done(w, 0ms));
    for (int i = 0; i < 50; ++i) {
      pass.reset();
      pass = std::make_unique<KvProgress::Pass>(p, false);
    }
    CHECK(done(w, 2s));
    // From that wait on the passes record, and a wait ends with its layer.
    CHECK(p.record());
    auto a = waiter(p, 0), b = waiter(p, 1);
    CHECK(!done(a, 0ms));
    p.recorded(0);
    CHECK(done(a, 2s) && !done(b, 50ms));
    p.recorded(1);
    CHECK(done(b, 2s));
    auto c = waiter(p, 0);
    CHECK(done(c, 2s));
  }
  {  // the layers of a pass with an observer stay reachable while others run behind it
    KvProgress p(1);
    {
      KvProgress::Pass pass(p, true);
      p.recorded(0);
    }
    KvProgress::Pass next(p, false);
    CHECK(p.record());
    auto w = waiter(p, 0);
    p.recorded(0);
    CHECK(done(w, 2s));
  }
  {  // waiters beside back-to-back passes
    KvProgress p(4);
    std::atomic<bool> stop{false};
    std::thread run([&] {
      while (!stop) {
        KvProgress::Pass pass(p, false);
        for (int l = 0; l < 4; ++l)
          if (p.record()) p.recorded(l);
      }
    });
    std::vector<std::future<void>> w;
    for (int i = 0; i < 4; ++i)
      w.push_back(std::async(std::launch::async, [&p, i] {
        for (int k = 0; k < 2000; ++k) p.reach(i);
      }));
    for (auto& f : w) CHECK(done(f, 30s));
    stop = true;
    run.join();
    CHECK(!p.running());
  }
  std::puts("ok");
}
