// The order of the host entry point's steps around its page-locked rows (csrc/host_rows.h): pieces, the
// forward, the wait, with an error at each of them.
#include <cstdio>
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

int main() {
  const auto expect = [](const char* name, const std::string& got, const char* want) { check(got == want, name, got); };
  expect("pieces_and_rest", steps(10, 4, -1), "f0+4 f4+4 f8+2 run wait = 0");
  expect("one_whole_piece", steps(4, 4, -1), "f0+4 run wait = 0");
  expect("first_piece_fails", steps(10, 4, 0), "f0+4 wait = 7");
  expect("later_piece_fails_and_is_waited_for", steps(10, 4, 1), "f0+4 f4+4 wait = 7");
  expect("forward_fails_and_is_waited_for", steps(10, 4, 3), "f0+4 f4+4 f8+2 run wait = 7");
  expect("wait_fails", steps(10, 4, 4), "f0+4 f4+4 f8+2 run wait = 9");
  return g_failed != 0;
}
