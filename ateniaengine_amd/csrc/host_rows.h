// What the host entry point does around its page-locked rows (moe_abi.hip), apart from the runtime's
// calls: plain C++, so that the CPU tests reach it.
#pragma once
#include <algorithm>
#include <cstddef>
#include <mutex>

namespace atenia_moe {

// Page-locked memory of one call: `bytes` each way and a tail.
struct HostRows {
  void* p = nullptr;
  size_t bytes = 0;
};
constexpr size_t kHostRowsTail = 256;

// The library's sets of them.  The handles of a model are called in turn, so they share: a call takes
// a set and gives it back, and as many exist as calls ran at once.  At most kMaxIdle lie idle, and
// with the last handle all are given back.  Any thread may call anything.
class HostRowsPool {
 public:
  static constexpr size_t kMaxIdle = 4;

  // alloc(n) returns n bytes or null, release(p) gives them back
  HostRowsPool(void* (*alloc)(size_t), void (*release)(void*)) : alloc_(alloc), release_(release) {}

  void attach() {  // a handle is made
    std::lock_guard<std::mutex> lock(mu_);
    ++handles_;
  }
  void detach() {  // and gone
    std::lock_guard<std::mutex> lock(mu_);
    if (--handles_ > 0) return;
    while (n_idle_ > 0) release_(remove(0).p);
    refused_ = 0;
  }

  // Room for `bytes` each way, in powers of two from 64 KiB on; p == null: not to be had.  A smaller set goes
  // only when the larger one is there, and a size that was refused is not asked for again: asking costs more than the
  // copies it would save.
  HostRows take(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu_);
    size_t best = n_idle_;
    for (size_t i = 0; i < n_idle_; ++i)
      if (idle_[i].bytes >= bytes && (best == n_idle_ || idle_[i].bytes < idle_[best].bytes)) best = i;
    if (best < n_idle_) return remove(best);
    HostRows r;
    size_t cap = (size_t)64 << 10;
    while (cap < bytes) cap *= 2;
    if (refused_ && cap >= refused_) return r;
    r.p = alloc_(2 * cap + kHostRowsTail);
    if (!r.p) {
      refused_ = cap;
      return r;
    }
    r.bytes = cap;
    if (n_idle_ > 0) release_(remove(0).p);
    return r;
  }
  void give(const HostRows& r) {
    if (!r.p) return;
    std::lock_guard<std::mutex> lock(mu_);
    if (handles_ <= 0) return release_(r.p);
    idle_[n_idle_++] = r;
    if (n_idle_ <= kMaxIdle) return;
    size_t least = 0;
    for (size_t i = 1; i < n_idle_; ++i)
      if (idle_[i].bytes < idle_[least].bytes) least = i;
    release_(remove(least).p);
  }

 private:
  HostRows remove(size_t i) {
    const HostRows r = idle_[i];
    idle_[i] = idle_[--n_idle_];
    return r;
  }

  void* (*alloc_)(size_t);
  void (*release_)(void*);
  std::mutex mu_;
  HostRows idle_[kMaxIdle + 1];
  size_t n_idle_ = 0;
  int handles_ = 0;
  size_t refused_ = 0;  // the smallest size that was not to be had; 0: none
};

// fetch(offset, bytes) copies one piece of the caller's rows into the page-locked ones and requests its
// way to the device; run() requests the forward; both return 0 or an error, and after an error nothing further is
// requested.  wait(rc) waits for what was, always, and returns rc or, if that is 0, its own error: on return
// nothing still reads or writes the rows, which the next call writes.
template <class Fetch, class Run, class Wait>
int through_host_rows(size_t bytes, size_t piece, Fetch fetch, Run run, Wait wait) {
  int rc = 0;
  for (size_t off = 0; off < bytes && !rc; off += piece) rc = fetch(off, std::min(piece, bytes - off));
  if (!rc) rc = run();
  return wait(rc);
}

}  // namespace atenia_moe
