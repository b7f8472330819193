// The order of the host entry point's steps around its page-locked rows (csrc/host_rows.h): pieces, the
// forward, the wait, with an error at each of them; and how that memory grows.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>

#include "../../ateniaengine_amd/csrc/host_rows.h"

using namespace atenia_moe;

static int g_failed = 0;
static void check(bool ok, const char* name, const std::string& got) {
  printf("%s %s%s%s\n", ok ? "ok  " : "FAIL", name, ok ? "" : ": ", ok ? "" : got.c_str());
  if (!ok) ++g_failed;
}

// The steps in order; step `bad` returns 7 (the wait: 9).
static std::string steps(size_t bytes, size_t piece, int bad) {
  std::string log;
  int n = 0;
  const int rc = through_host_rows(
      bytes, piece,
      [&](size_t off, size_t here) {
        log += "f" + std::to_string(off) + "+" + std::to_string(here) + " ";
        return n++ == bad ? 7 : 0;
      },
      [&] {
        log += "run ";
        return n++ == bad ? 7 : 0;
      },
      [&](int earlier) {
        log += "wait ";
        return earlier ? earlier : n++ == bad ? 9 : 0;
      });
  return log + "= " + std::to_string(rc);
}

// Growth with an allocator that has nothing of `limit` bytes and more.
static void growth() {
  HostRows r;
  std::set<void*> live;
  size_t limit = (size_t)1 << 30;
  int asked = 0;
  const auto grow = [&](size_t bytes) {
    return grow_host_rows(
        r, bytes,
        [&](size_t n) -> void* {
          ++asked;
          if (n >= limit) return nullptr;
          void* p = malloc(n);
          live.insert(p);
          return p;
        },
        [&](void* p) {
          live.erase(p);
          free(p);
        });
  };
  const auto state = [&](bool got) {
    return std::string(got ? "yes " : "no ") + std::to_string(r.bytes >> 10) + " KiB, " + std::to_string(live.size()) +
           " held, asked " + std::to_string(asked);
  };
  const auto expect = [&](const char* name, bool got, const char* want) { check(state(got) == want, name, state(got)); };
  expect("smallest", grow(1), "yes 64 KiB, 1 held, asked 1");
  expect("fits", grow(64 << 10), "yes 64 KiB, 1 held, asked 1");
  expect("grows_and_frees", grow((64 << 10) + 1), "yes 128 KiB, 1 held, asked 2");
  limit = (size_t)1 << 20;
  expect("refused_keeps_the_old", grow(600 << 10), "no 128 KiB, 1 held, asked 3");
  expect("what_fitted_still_fits", grow(128 << 10), "yes 128 KiB, 1 held, asked 3");
  expect("refused_size_is_not_asked_for_again", grow(1024 << 10), "no 128 KiB, 1 held, asked 3");
  expect("larger_ones_neither", grow(2 << 20), "no 128 KiB, 1 held, asked 3");
  expect("a_smaller_step_is", grow(200 << 10), "yes 256 KiB, 1 held, asked 4");
  for (void* p : live) free(p);
}

int main() {
  growth();
  const auto expect = [](const char* name, const std::string& got, const char* want) { check(got == want, name, got); };
  expect("pieces_and_rest", steps(10, 4, -1), "f0+4 f4+4 f8+2 run wait = 0");
  expect("one_whole_piece", steps(4, 4, -1), "f0+4 run wait = 0");
  expect("first_piece_fails", steps(10, 4, 0), "f0+4 wait = 7");
  expect("later_piece_fails_and_is_waited_for", steps(10, 4, 1), "f0+4 f4+4 wait = 7");
  expect("forward_fails_and_is_waited_for", steps(10, 4, 3), "f0+4 f4+4 f8+2 run wait = 7");
  expect("wait_fails", steps(10, 4, 4), "f0+4 f4+4 f8+2 run wait = 9");
  return g_failed != 0;
}
