// What the host entry point does around its page-locked rows (moe_abi.hip), apart from the runtime's
// calls: plain C++, so that the CPU tests reach it.
#pragma once
#include <algorithm>
#include <cstddef>

namespace atenia_moe {

// Page-locked memory of a handle: `bytes` each way and a tail.
struct HostRows {
  void* p = nullptr;
  size_t bytes = 0;
  size_t refused = 0;  // a size that was not to be had; 0: none
};
constexpr size_t kHostRowsTail = 256;

// Room for `bytes` each way, in powers of two from 64 KiB on; false: not to be had.  alloc(n) returns n bytes or
// null, release(p) gives them back.  The old memory goes only when the new is there, and a size that was
// refused once is not asked for again: asking costs more than the copies it would save.
template <class Alloc, class Release>
bool grow_host_rows(HostRows& r, size_t bytes, Alloc alloc, Release release) {
  if (bytes <= r.bytes) return true;
  size_t cap = (size_t)64 << 10;
  while (cap < bytes) cap *= 2;
  if (r.refused && cap >= r.refused) return false;
  void* p = alloc(2 * cap + kHostRowsTail);
  if (!p) {
    r.refused = cap;
    return false;
  }
  if (r.p) release(r.p);
  r.p = p;
  r.bytes = cap;
  return true;
}

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
