// slot_pool.hpp -- host memory blocks that the engines of a process share.
//
// Pinned memory costs about 0.5 ms a MB to make and is not for others while
// it is held, so the blocks that downloads pass through belong to the process:
// a call takes some and gives them back. Calls of several threads share kMax of
// them and never wait for each other: one that finds none left has a block
// made that goes again with it. The last engine to go gives the memory back.
#pragma once

#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

namespace mpm_engine {

// Memory: static uint8_t* make(size_t bytes) (null: none left), drop(uint8_t*).
// Blocks are made in steps of kStep bytes, so that calls whose size grows by
// little use one again.
template <class Memory, size_t kMax, size_t kStep>
class SlotPool {
 public:
  struct Slot {
    uint8_t* p;
    size_t bytes;
  };

  SlotPool() { idle_.reserve(kMax); }

  void attach() {
    std::lock_guard<std::mutex> lock(m_);
    ++users_;
  }
  void detach() {
    std::lock_guard<std::mutex> lock(m_);
    if (--users_ == 0) trim(0);
  }

  // 1 to `want` blocks of at least `bytes` into `out`, the number returned; 0
  // if there is no memory.
  size_t take(size_t want, size_t bytes, Slot* out) {
    std::lock_guard<std::mutex> lock(m_);
    size_t got = 0;
    while (got < want && (idle_block(bytes, &out[got]) || (room() && new_block(bytes, &out[got])))) ++got;
    if (got == 0 && new_block(bytes, &out[0])) got = 1;
    return got;
  }
  void give(const Slot* slots, size_t n) {
    std::lock_guard<std::mutex> lock(m_);
    for (size_t i = 0; i < n; ++i) {
      if (made_ > kMax || users_ == 0) drop(slots[i]);
      else idle_.push_back(slots[i]);
    }
  }

 private:
  // the last one given back that is large enough
  bool idle_block(size_t bytes, Slot* out) {
    for (size_t i = idle_.size(); i-- > 0;)
      if (idle_[i].bytes >= bytes) {
        *out = idle_[i];
        idle_.erase(idle_.begin() + (ptrdiff_t)i);
        return true;
      }
    return false;
  }
  // of kMax blocks; idle ones that were too small make way
  bool room() {
    if (made_ >= kMax && !idle_.empty()) trim(idle_.size() - 1);
    return made_ < kMax;
  }
  bool new_block(size_t bytes, Slot* out) {
    const size_t size = (bytes + kStep - 1) / kStep * kStep;
    *out = {Memory::make(size), size};
    if (out->p) ++made_;
    return out->p != nullptr;
  }
  void drop(const Slot& s) {
    Memory::drop(s.p);
    --made_;
  }
  void trim(size_t keep) {
    while (idle_.size() > keep) {
      drop(idle_.back());
      idle_.pop_back();
    }
  }

  std::mutex m_;
  std::vector<Slot> idle_;
  size_t made_ = 0;  // blocks there are, taken ones included
  int64_t users_ = 0;
};

}  // namespace mpm_engine
