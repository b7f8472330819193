// What the host entry point does around its page-locked rows (moe_abi.hip), apart from the runtime's
// calls: plain C++, so that the CPU tests reach it.
#pragma once
#include <algorithm>
#include <cstddef>

namespace atenia_moe {

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
