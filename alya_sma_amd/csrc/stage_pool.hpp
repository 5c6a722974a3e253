// Idle stages (streams, events and a block of pinned memory each, made for one
// device) between the calls that use them.
#pragma once
#include <cstddef>
#include <mutex>

namespace sma_abi {

// Stage: `int device`, `size_t bytes` of its block, `Stage* next`, and
// `drop_block()`, which frees the block and leaves bytes 0.
// The pool grows with the callers that are in a call at once, up to `limit`
// idle stages for each device, so that a further round of the same callers makes
// nothing anew, and one device's stages take no other's place.  The idle blocks
// stay within `budget` bytes together: a stage that would go beyond it is kept
// without its block.  No allocation, so nothing to fail.
template <class Stage>
class StagePool {
  std::mutex mu_;
  Stage* idle_ = nullptr;          // the last one given first
  size_t bytes_ = 0;
  const size_t limit_, budget_;

 public:
  constexpr StagePool(size_t limit, size_t budget) : limit_(limit), budget_(budget) {}

  // An idle stage of the device, or null.
  Stage* take(int device) {
    std::lock_guard<std::mutex> lock(mu_);
    for (Stage** p = &idle_; *p; p = &(*p)->next)
      if ((*p)->device == device) {
        Stage* s = *p;
        *p = s->next;
        s->next = nullptr;
        bytes_ -= s->bytes;
        return s;
      }
    return nullptr;
  }

  // Keeps the stage (true) or leaves it to the caller to end (false).
  bool give(Stage* s) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (put(s)) return true;
      if (s->bytes == 0) return false;       // the device's limit, not the budget
    }
    s->drop_block();
    std::lock_guard<std::mutex> lock(mu_);
    return put(s);
  }

 private:
  bool put(Stage* s) {
    if (bytes_ + s->bytes > budget_) return false;
    size_t n = 0;
    for (const Stage* q = idle_; q; q = q->next) n += q->device == s->device;
    if (n >= limit_) return false;
    s->next = idle_;
    idle_ = s;
    bytes_ += s->bytes;
    return true;
  }
};

}  // namespace sma_abi
