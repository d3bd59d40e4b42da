// The pool of device memory behind resident results (host code, no device headers).
#pragma once
#include <algorithm>
#include <cstddef>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace tsr950 {

enum class PoolAlloc { kOk, kNoMemory, kFailed };
enum class PoolStatus { kOk, kForeign, kFailed };

// Device memory for results that a chain of default-stream calls allocates and drops (hipMalloc and hipFree
// cost about 65 us a pair and the free waits for the device: three of them were half the time of an attention
// block over 1000 tokens).  Blocks are kept by size class and device and handed out again
//   - at once, when only the library's own default-stream calls saw them: work on that stream runs in
//     order, so the block's next writer comes after its last reader.  An owner that wants such a block for other
//     streams calls `settle` first, which waits for the device where nothing has since the block was dropped;
//   - after the next synchronisation of the device, when the caller saw the address (`shared`) and may have work
//     on it in other streams: what hipFree itself would have waited for.  Where none comes, an allocation that
//     finds kWaitBlocks blocks of its class (or kWaitBytes of them) waiting makes one.
// At most kBytes are cached in a process; one block more, or an allocation anywhere in the library that finds no
// memory (`allocate`), gives all of them back.
//
// Api, static: bool device(int*), the current device; PoolAlloc malloc(void**, size_t); bool free(void*), which waits
// for the work that uses the block; bool synchronize(int dev).
template <class Api>
class DevicePool {
 public:
  static constexpr size_t kBytes = size_t(4) << 30;
  static constexpr size_t kWaitBlocks = 16, kWaitBytes = size_t(256) << 20;

  bool malloc(void** out, size_t bytes) {
    int dev = 0;
    if (!Api::device(&dev)) return false;
    const size_t size = size_class(bytes < 512 ? 512 : bytes);
    const Class cls{dev, size};
    std::unique_lock<std::mutex> lock(mu_);
    if (ready_[cls].empty()) {
      const size_t n = waiting_[cls].size();
      if (n >= kWaitBlocks || n * size >= kWaitBytes) {
        lock.unlock();
        if (!synchronize()) return false;
        lock.lock();
      }
    }
    auto& ready = ready_[cls];
    void* p = nullptr;
    unsigned long dropped = 0;
    if (!ready.empty()) {
      p = ready.back();
      ready.pop_back();
      dropped = kept_[p].dropped;
      kept_.erase(p);
      cached_ -= size;
    } else {
      PoolAlloc r = Api::malloc(&p, size);
      if (r == PoolAlloc::kNoMemory && !kept_.empty()) {
        (void)give_back_all();
        r = Api::malloc(&p, size);
      }
      if (r != PoolAlloc::kOk) return false;
    }
    live_[p] = Block{size, dev, ++clock_, dropped};
    *out = p;
    return true;
  }

  PoolStatus free(void* p, bool shared) {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = live_.find(p);
    if (it == live_.end()) return PoolStatus::kForeign;
    Block b = it->second;
    live_.erase(it);
    if (b.bytes > kBytes / 2) return Api::free(p) ? PoolStatus::kOk : PoolStatus::kFailed;
    bool ok = true;
    if (cached_ + b.bytes > kBytes) ok = give_back_all();
    b.dropped = ++clock_;
    kept_[p] = b;
    cached_ += b.bytes;
    if (shared) waiting_[{b.device, b.bytes}].push_back({p, b.id});
    else ready_[{b.device, b.bytes}].push_back(p);
    return ok ? PoolStatus::kOk : PoolStatus::kFailed;
  }

  // Makes a handed-out block safe for any stream: waits for its device where the block's last owner dropped it
  // after the latest synchronisation, so that work of that owner may still be queued on it.
  PoolStatus settle(void* p) {
    int dev = 0;
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = live_.find(p);
      if (it == live_.end()) return PoolStatus::kForeign;
      dev = it->second.device;
      if (it->second.dropped <= synced_[dev]) return PoolStatus::kOk;
    }
    return synchronize(dev) ? PoolStatus::kOk : PoolStatus::kFailed;
  }

  // Synchronises the current device; blocks that waited for that when it began are ready afterwards.
  bool synchronize() {
    int dev = 0;
    return Api::device(&dev) && synchronize(dev);
  }

  bool trim() {
    std::lock_guard<std::mutex> lock(mu_);
    return give_back_all();
  }

  // An allocation outside the pool: try_alloc() -> PoolAlloc; where it finds no memory, the pool's cached blocks are
  // given back and it is tried once more.
  template <class F>
  bool allocate(F try_alloc) {
    PoolAlloc r = try_alloc();
    if (r == PoolAlloc::kNoMemory) {
      std::lock_guard<std::mutex> lock(mu_);
      if (!kept_.empty()) {
        (void)give_back_all();
        r = try_alloc();
      }
    }
    return r == PoolAlloc::kOk;
  }

 private:
  struct Block { size_t bytes; int device; unsigned long id, dropped; };   // dropped: when its last owner did, 0 = none
  struct Waiting { void* p; unsigned long id; };
  using Class = std::pair<int, size_t>;                              // device, bytes

  bool synchronize(int dev) {
    std::vector<Waiting> before;
    unsigned long began = 0;
    {
      std::lock_guard<std::mutex> lock(mu_);
      began = clock_;
      for (auto& c : waiting_)
        if (c.first.first == dev) before.insert(before.end(), c.second.begin(), c.second.end());
    }
    if (!Api::synchronize(dev)) return false;
    std::lock_guard<std::mutex> lock(mu_);
    synced_[dev] = std::max(synced_[dev], began);
    for (const Waiting& w : before) {
      auto it = kept_.find(w.p);
      if (it == kept_.end() || it->second.id != w.id) continue;      // given back, or settled by another thread
      auto& waiting = waiting_[{dev, it->second.bytes}];
      auto at = std::find_if(waiting.begin(), waiting.end(), [&](const Waiting& x) { return x.id == w.id; });
      if (at == waiting.end()) continue;
      waiting.erase(at);
      ready_[{dev, it->second.bytes}].push_back(w.p);
    }
    return true;
  }

  // Eight classes per power of two: at most an eighth of a block is unused.
  static size_t size_class(size_t bytes) {
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
  }
  bool give_back_all() {                                             // (the caller holds the lock)
    bool ok = true;
    for (auto& b : kept_) ok &= Api::free(b.first);
    kept_.clear();
    ready_.clear();
    waiting_.clear();
    cached_ = 0;
    return ok;
  }

  std::mutex mu_;
  unsigned long clock_ = 0;                                          // one tick per hand-out and per drop
  std::map<int, unsigned long> synced_;                              // device: the tick up to which its work is done
  size_t cached_ = 0;
  std::map<void*, Block> live_;                                      // handed out
  std::map<void*, Block> kept_;                                      // ready or waiting
  std::map<Class, std::vector<void*>> ready_;
  std::map<Class, std::vector<Waiting>> waiting_;
};

}  // namespace tsr950
