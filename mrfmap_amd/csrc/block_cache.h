// Process-wide cache of device blocks.  A context makes some 25 allocations
// per camera and as many frees when it is closed or a camera is traversed
// again; hipMalloc takes 25-40 us and hipFree 80-180 us (4 x 160x120: 15 of
// the 18 ms of a map built from nothing; 13 x 640x480: 44 of 140 ms), and for
// lists of tens of GB the runtime takes seconds to provide the memory again
// (a 64-keyframe build: 0.86 s in a fresh process, 4.3-4.5 s after a context
// of that size was closed, whose frees took 2.4 s).  Blocks are therefore
// kept on free (after the device has finished with them) and handed out again
// for requests of up to their size and at least 4/5 of it.  Sizes below 32 MiB
// are rounded up to eighths of a power of two, so that slightly different
// requests share blocks; larger blocks keep their size, since lists may take
// most of the device.  The cache keeps at most R::keep_limit() bytes and gives
// everything back when an allocation fails.
//
// Several threads may allocate and free at once (a context each).  The lock
// covers the tables alone: the waits for the device and the runtime's own
// allocations and frees run outside it, so that one context's free, which may
// wait for another's queued iterations, holds up no third context.
//
// R, the runtime: Error (Error{} is success), device() the current device,
// allocate(p, bytes), release(p), wait(dev) until the device has ended all its
// work (false if that cannot be waited for: a stream of another library is
// being captured, say) and keep_limit().
#pragma once

#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace mrf {

inline size_t block_size(size_t bytes) {
  if (bytes >= size_t(32) << 20) return bytes;
  size_t step = 512;  // 4 KiB and below: multiples of 512 B
  while (step * 16 <= bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

template <class R>
class BlockCache {
 public:
  typename R::Error allocate(void** p, size_t bytes) {
    *p = nullptr;
    bytes = block_size(bytes);
    const int dev = R::device();
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = idle_.lower_bound({dev, bytes});
      if (it != idle_.end() && it->first.first == dev && it->first.second - it->first.second / 5 <= bytes) {
        *p = it->second;
        live_[*p] = {it->first.second, dev};
        kept_ -= it->first.second;
        idle_.erase(it);
        return typename R::Error{};
      }
    }
    typename R::Error e = R::allocate(p, bytes);
    if (e != typename R::Error{} && give_back(dev)) e = R::allocate(p, bytes);
    if (e == typename R::Error{}) {
      std::lock_guard<std::mutex> lock(mu_);
      live_[*p] = {bytes, dev};
    }
    return e;
  }

  void free(void* p) {
    if (!p) return;
    static const size_t limit = R::keep_limit();
    size_t bytes = 0;
    int dev = 0;
    bool keep = false;
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = live_.find(p);
      if (it != live_.end()) {
        bytes = it->second.first;
        dev = it->second.second;
        live_.erase(it);
        keep = kept_ + bytes <= limit;
        if (keep) {
          kept_ += bytes;
          ++begun_;
        }
      }
    }
    if (keep) {
      // the block's last uses end before another allocation can take it; where
      // that cannot be waited for, the block goes back to the runtime
      const bool ended = R::wait(dev);
      {
        std::lock_guard<std::mutex> lock(mu_);
        if (ended)
          idle_.insert({{dev, bytes}, p});
        else
          kept_ -= bytes;
        ++ended_;
      }
      freed_.notify_all();
      if (ended) return;
    }
    R::release(p);
  }

  // the kept blocks of device dev (all devices for dev < 0) back to the
  // runtime, those of the frees under way included; false if there were none
  bool give_back(int dev) {
    std::vector<void*> blocks;
    {
      std::unique_lock<std::mutex> lock(mu_);
      const uint64_t begun = begun_;
      freed_.wait(lock, [&] { return ended_ >= begun; });
      for (auto it = idle_.begin(); it != idle_.end();) {
        if (dev >= 0 && it->first.first != dev) {
          ++it;
          continue;
        }
        blocks.push_back(it->second);
        kept_ -= it->first.second;
        it = idle_.erase(it);
      }
    }
    for (void* b : blocks) R::release(b);
    return !blocks.empty();
  }

 private:
  std::mutex mu_;
  std::condition_variable freed_;
  std::unordered_map<void*, std::pair<size_t, int>> live_;  // blocks in use: bytes, device
  std::multimap<std::pair<int, size_t>, void*> idle_;        // (device, bytes) -> kept block
  size_t kept_ = 0;                                          // bytes of the idle blocks and of the frees under way
  uint64_t begun_ = 0, ended_ = 0;                           // frees that wait or have waited for the device
};

}  // namespace mrf
