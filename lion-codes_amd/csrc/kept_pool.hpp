// kept_pool.hpp -- buffers that idle owners leave for their next use.
//
// At most kSets sets and `limit` bytes in the whole process, one set per
// owner; the oldest make room for a new one.  Every call may come from any
// thread; sets are freed outside the lock.
#pragma once

#include <stdint.h>

#include <memory>
#include <mutex>
#include <utility>

namespace lufqhe {

template <class Buf>
class KeptPool {
 public:
  static constexpr int kSets = 16;
  explicit KeptPool(int64_t limit) : limit_(limit) {}

  // The owner's set, or null.
  std::unique_ptr<Buf> take(const void* owner) {
    std::lock_guard<std::mutex> lock(mu_);
    for (int i = 0; i < count_; ++i)
      if (sets_[i].owner == owner) return remove(i);
    return nullptr;
  }

  // Keeps the set, or frees it if it is larger than the limit.
  void put(const void* owner, std::unique_ptr<Buf> buf, int64_t bytes) {
    std::unique_ptr<Buf> drop[kSets + 1];
    int n = 0;
    std::lock_guard<std::mutex> lock(mu_);
    for (int i = 0; i < count_; ++i)
      if (sets_[i].owner == owner) {
        drop[n++] = remove(i);
        break;
      }
    if (bytes > limit_) {
      drop[n++] = std::move(buf);
      return;
    }
    while (count_ == kSets || bytes_ + bytes > limit_) drop[n++] = remove(0);
    sets_[count_].owner = owner;
    sets_[count_].buf = std::move(buf);
    sets_[count_].bytes = bytes;
    ++count_;
    bytes_ += bytes;
  }

  // Frees the owner's set, or every set if owner is null; whether there was one.
  bool release(const void* owner) {
    std::unique_ptr<Buf> drop[kSets];
    int n = 0;
    std::lock_guard<std::mutex> lock(mu_);
    for (int i = count_ - 1; i >= 0; --i)
      if (!owner || sets_[i].owner == owner) drop[n++] = remove(i);
    return n > 0;
  }

  // Bytes of the owner's set, or of all sets if owner is null.
  int64_t bytes(const void* owner) {
    std::lock_guard<std::mutex> lock(mu_);
    if (!owner) return bytes_;
    for (int i = 0; i < count_; ++i)
      if (sets_[i].owner == owner) return sets_[i].bytes;
    return 0;
  }

 private:
  struct Set {
    const void* owner = nullptr;
    std::unique_ptr<Buf> buf;
    int64_t bytes = 0;
  };

  std::unique_ptr<Buf> remove(int i) {
    std::unique_ptr<Buf> b = std::move(sets_[i].buf);
    bytes_ -= sets_[i].bytes;
    for (; i + 1 < count_; ++i) sets_[i] = std::move(sets_[i + 1]);
    --count_;
    return b;
  }

  const int64_t limit_;
  std::mutex mu_;
  Set sets_[kSets];  // oldest first
  int count_ = 0;
  int64_t bytes_ = 0;
};

}  // namespace lufqhe
