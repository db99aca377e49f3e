// Device memory lent for the length of one call. A multi-token call needs
// chunk buffers of up to 335 MB (a 35B model with matrix-core components);
// held by the session they stayed for its life, so a server paid them once per
// open conversation. Lent, they are paid once per call that runs at the same
// time. Host code only.
#pragma once

#include <cstddef>
#include <mutex>

namespace cq35 {

struct DeviceBlock {
  void* p = nullptr;
  size_t bytes = 0;
};

// Memory: static void* allocate(size_t bytes), null where there is none;
// static void release(void*). Safe from any thread; throws nothing.
template <typename Memory>
class BlockPool {
 public:
  static constexpr int kMostIdle = 8;  // blocks kept; more calls than that at once release theirs

  // The smallest idle block of at least `bytes`, or none.
  DeviceBlock idle(size_t bytes) {
    std::lock_guard<std::mutex> hold(lock_);
    int at = -1;
    for (int i = 0; i < count_; ++i)
      if (blocks_[i].bytes >= bytes && (at < 0 || blocks_[i].bytes < blocks_[at].bytes)) at = i;
    return remove(at);
  }

  // A new block, or none where there is no memory. The largest idle one makes
  // way for it if it is too small, all of them where memory is short.
  DeviceBlock allocate(size_t bytes) {
    DeviceBlock old;
    {
      std::lock_guard<std::mutex> hold(lock_);
      int at = count_ - 1;
      for (int i = 0; i < count_; ++i)
        if (blocks_[i].bytes > blocks_[at].bytes) at = i;
      if (at >= 0 && blocks_[at].bytes < bytes) old = remove(at);
    }
    if (old.p) Memory::release(old.p);
    void* p = Memory::allocate(bytes);
    if (!p && trim()) p = Memory::allocate(bytes);
    return p ? DeviceBlock{p, bytes} : DeviceBlock{};
  }

  // A block whose work has ended.
  void give(DeviceBlock block) {
    {
      std::lock_guard<std::mutex> hold(lock_);
      if (users_ > 0 && count_ < kMostIdle) {
        blocks_[count_++] = block;
        return;
      }
    }
    Memory::release(block.p);
  }

  // Releases the idle blocks; whether there were any.
  bool trim() {
    bool any = false;
    while (true) {
      DeviceBlock block;
      {
        std::lock_guard<std::mutex> hold(lock_);
        block = remove(count_ - 1);
      }
      if (!block.p) return any;
      any = true;
      Memory::release(block.p);
    }
  }

  // Models of the device: the last to go takes the idle blocks with it.
  void enter() {
    std::lock_guard<std::mutex> hold(lock_);
    ++users_;
  }
  void leave() {
    bool last;
    {
      std::lock_guard<std::mutex> hold(lock_);
      last = --users_ == 0;
    }
    if (last) trim();
  }

 private:
  DeviceBlock remove(int at) {
    if (at < 0) return {};
    const DeviceBlock b = blocks_[at];
    blocks_[at] = blocks_[--count_];
    return b;
  }

  std::mutex lock_;
  DeviceBlock blocks_[kMostIdle];
  int count_ = 0;
  int users_ = 0;
};

// A block of `pool` for *rows rows of bytes(rows), or for `few` of them where
// a new block would take an eighth of the free memory or is not to be had;
// *rows what it became. free_bytes() is asked for new blocks only.
template <typename Pool, typename Bytes, typename Free>
DeviceBlock lend_rows(Pool& pool, long* rows, long few, Bytes bytes, Free free_bytes) {
  DeviceBlock block = pool.idle(bytes(*rows));
  if (block.p) return block;
  if (bytes(*rows) > free_bytes() / 8 && few < *rows) {
    *rows = few;
    block = pool.idle(bytes(few));
  }
  if (!block.p) block = pool.allocate(bytes(*rows));
  if (!block.p && few < *rows) block = pool.allocate(bytes(*rows = few));
  return block;
}

}  // namespace cq35
