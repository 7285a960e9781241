// The device-block cache (mrfmap_amd/csrc/block_cache.h) on a runtime made of
// counters.  Prints "ok" and exits 0, or says which check failed.
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <map>
#include <mutex>
#include <string>
#include <thread>

#include "../../mrfmap_amd/csrc/block_cache.h"

using namespace std::chrono_literals;

struct Fake {
  using Error = int;
  static std::mutex mu;
  static std::condition_variable cv;
  static bool busy, wait_ok;             // busy: the device's work does not end
  static int waiting;                    // threads in wait()
  static size_t memory, used, next;      // bytes of the device, in use, next address
  static std::map<void*, size_t> blocks;

  static int device() { return 0; }
  static int allocate(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    if (used + bytes > memory) return 2;
    used += bytes;
    *p = reinterpret_cast<void*>(next += 4096);
    blocks[*p] = bytes;
    return 0;
  }
  static void release(void* p) {
    std::lock_guard<std::mutex> lock(mu);
    used -= blocks.at(p);
    blocks.erase(p);
  }
  static bool wait(int) {
    std::unique_lock<std::mutex> lock(mu);
    ++waiting;
    cv.notify_all();
    cv.wait(lock, [] { return !busy; });
    --waiting;
    return wait_ok;
  }
  static size_t keep_limit() { return 3u << 20; }
  static void set_busy(bool b) {
    std::lock_guard<std::mutex> lock(mu);
    busy = b;
    cv.notify_all();
  }
  static void until_waiting(int n) {
    std::unique_lock<std::mutex> lock(mu);
    cv.wait(lock, [n] { return waiting >= n; });
  }
};
std::mutex Fake::mu;
std::condition_variable Fake::cv;
bool Fake::busy = false, Fake::wait_ok = true;
int Fake::waiting = 0;
size_t Fake::memory = size_t(1) << 30, Fake::used = 0, Fake::next = 0;
std::map<void*, size_t> Fake::blocks;

static void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::fflush(stdout);
  std::_Exit(1);
}

using Cache = mrf::BlockCache<Fake>;

static void* get(Cache& c, size_t bytes) {
  void* p = nullptr;
  check(c.allocate(&p, bytes) == 0 && p, "allocate");
  return p;
}

// a free that waits for the device holds up neither a new block, nor a kept
// one, nor another context's free
static void others_go_on() {
  Cache c;
  void *a = get(c, 5000), *b = get(c, 100000), *d = get(c, 70000);
  c.free(b);
  Fake::set_busy(true);
  std::thread t([&] { c.free(a); });
  Fake::until_waiting(1);
  auto fresh = std::async(std::launch::async, [&] { return get(c, 9000); });
  auto kept = std::async(std::launch::async, [&] { return get(c, 100000); });
  check(fresh.wait_for(10s) == std::future_status::ready, "a new block waits for another context's work");
  check(kept.wait_for(10s) == std::future_status::ready, "a kept block waits for another context's work");
  check(kept.get() == b, "the kept block");
  check(fresh.get() != a, "a block handed out before its last use ended");
  std::thread u([&] { c.free(d); });
  Fake::until_waiting(2);
  check(get(c, 5000) != a, "a block handed out before its last use ended");
  Fake::set_busy(false);
  t.join();
  u.join();
  check(get(c, 5000) == a, "the block once its last use has ended");
}

// a block whose last use cannot be waited for is not kept
static void failed_wait() {
  Cache c;
  void* a = get(c, 5000);
  Fake::wait_ok = false;
  c.free(a);
  check(Fake::blocks.count(a) == 0, "a block that may be in use is kept");
  Fake::wait_ok = true;
  check(get(c, 5000) != a, "a block that may be in use is handed out");
  check(!c.give_back(-1), "nothing is kept");
}

// an allocation that does not fit gets the memory of the kept blocks and of
// the frees under way
static void full_device() {
  Cache c;
  Fake::memory = 2u << 20;
  void *a = get(c, 1u << 20), *b = get(c, 512u << 10);
  c.free(b);
  Fake::set_busy(true);
  std::thread t([&] { c.free(a); });
  Fake::until_waiting(1);
  auto big = std::async(std::launch::async, [&] {
    void* p = nullptr;
    return c.allocate(&p, 2u << 20) == 0;
  });
  check(big.wait_for(200ms) != std::future_status::ready, "no memory is left while the device works");
  Fake::set_busy(false);
  t.join();
  check(big.get(), "the kept blocks' memory");
  void* p = nullptr;
  check(c.allocate(&p, 4096) != 0, "an allocation beyond the device's memory");
}

// blocks serve requests of 4/5 of their size to all of it; the rest goes back
static void sizes() {
  Cache c;
  void* a = get(c, 1u << 20);
  c.free(a);
  check(get(c, (1u << 20) + 1) != a, "a larger request");
  check(get(c, 700u << 10) != a, "a request below 4/5");
  check(get(c, 900u << 10) == a, "a request of 4/5 or more");
  void* big = get(c, 4u << 20);
  c.free(big);
  check(Fake::blocks.count(big) == 0, "a block beyond the limit is kept");
  c.free(a);
  check(c.give_back(0) && Fake::blocks.count(a) == 0, "the kept blocks go back");
}

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> tests = {
      {"others_go_on", others_go_on}, {"failed_wait", failed_wait}, {"full_device", full_device}, {"sizes", sizes}};
  if (argc != 2 || !tests.count(argv[1])) return 2;
  tests.at(argv[1])();
  std::printf("ok\n");
  return 0;
}
