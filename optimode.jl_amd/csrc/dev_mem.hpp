// Owning device allocations, and the blocks a call keeps between them.
#pragma once
#include <utility>
#include <vector>

#include "omx_common.hpp"
#include "omx_errors.hpp"

namespace omx {

// Device blocks that DevMem releases and takes while a scope of it is open on the thread: a call
// that makes a handle per grid reuses the first one's memory in the next (four grids up to
// 256 x 256, six problems: 225 hipMalloc and hipFree took 27 of 122 ms).  The blocks go back
// to the device with the scope, or when an allocation fails.  A block is kept only after the
// device is idle, as hipFree itself would wait, so whichever stream takes it next may use it.
class DevCache {
 public:
  DevCache() : outer_(current()) { current() = this; }
  ~DevCache() {
    current() = outer_;
    drop();
  }
  DevCache(const DevCache&) = delete;
  DevCache& operator=(const DevCache&) = delete;
  static DevCache*& current() {
    static thread_local DevCache* c = nullptr;
    return c;
  }
  // A kept block serves a request of at least an eighth of it, blocks up to 256 MiB any smaller
  // one too: a small buffer never sits on a large block that the next large one then has to
  // be allocated beside, and which dropping the kept blocks would not free.
  static bool serves(size_t cap, size_t bytes) {
    return cap >= bytes && (cap <= (size_t(256) << 20) || cap / 8 <= bytes);
  }
  // the smallest kept block that serves `bytes` (its size into cap), or nullptr
  void* take(size_t bytes, size_t& cap) {
    size_t best = blocks_.size();
    for (size_t j = 0; j < blocks_.size(); ++j)
      if (serves(blocks_[j].second, bytes) && (best == blocks_.size() || blocks_[j].second < blocks_[best].second)) best = j;
    if (best == blocks_.size()) return nullptr;
    void* p = blocks_[best].first;
    cap = blocks_[best].second;
    blocks_.erase(blocks_.begin() + long(best));
    return p;
  }
  bool put(void* p, size_t cap) noexcept {
    if (hipDeviceSynchronize() != hipSuccess) return false;
    try {
      blocks_.emplace_back(p, cap);
    } catch (...) {
      return false;
    }
    return true;
  }
  void drop() noexcept {
    for (auto& b : blocks_) (void)hipFree(b.first);
    blocks_.clear();
  }

 private:
  DevCache* outer_;
  std::vector<std::pair<void*, size_t>> blocks_;
};

// Owning device allocation.
class DevMem {
 public:
  DevMem() = default;
  explicit DevMem(size_t bytes) { alloc(bytes); }
  ~DevMem() { release(); }
  DevMem(const DevMem&) = delete;
  DevMem& operator=(const DevMem&) = delete;
  DevMem(DevMem&& o) noexcept : p_(o.p_), n_(o.n_), cap_(o.cap_) {
    o.p_ = nullptr;
    o.n_ = o.cap_ = 0;
  }
  DevMem& operator=(DevMem&& o) noexcept {
    if (this != &o) {
      release();
      p_ = o.p_;
      n_ = o.n_;
      cap_ = o.cap_;
      o.p_ = nullptr;
      o.n_ = o.cap_ = 0;
    }
    return *this;
  }
  void alloc(size_t bytes) {
    release();
    if (bytes) {
      DevCache* c = DevCache::current();
      if (c) p_ = c->take(bytes, cap_);
      if (!p_) {
        cap_ = bytes;
        if (c && hipMalloc(&p_, bytes) != hipSuccess) {
          (void)hipGetLastError();
          p_ = nullptr;
          c->drop();
        }
        if (!p_) OMX_HIP_CHECK(hipMalloc(&p_, bytes));
      }
    }
    n_ = bytes;
  }
  void ensure(size_t bytes) {
    if (bytes > n_) alloc(bytes);
  }
  void release() {
    if (p_ && !(DevCache::current() && DevCache::current()->put(p_, cap_))) (void)hipFree(p_);
    p_ = nullptr;
    n_ = cap_ = 0;
  }
  template <typename U> U* as() const { return static_cast<U*>(p_); }
  size_t size() const { return n_; }

 private:
  void* p_ = nullptr;
  size_t n_ = 0, cap_ = 0;  // bytes asked for; of the block
};

}  // namespace omx
