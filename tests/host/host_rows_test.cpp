// The order of the host entry point's steps around its page-locked rows (csrc/host_rows.h): pieces, the
// forward, the wait, with an error at each of them; and the pool they come from.
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

// The pool with an allocator that has nothing of `g_limit` bytes and more.
static std::set<void*> g_live;
static size_t g_limit = (size_t)1 << 30;
static int g_asked = 0;
static void* take_bytes(size_t n) {
  ++g_asked;
  if (n >= g_limit) return nullptr;
  void* p = malloc(n);
  g_live.insert(p);
  return p;
}
static void free_bytes(void* p) {
  if (!g_live.erase(p)) check(false, "freed_twice", "");
  free(p);
}
static void pool() {
  HostRowsPool rows(take_bytes, free_bytes);
  const auto state = [&](const HostRows& r) {
    return std::to_string(r.bytes >> 10) + " KiB, " + std::to_string(g_live.size()) + " held, asked " +
           std::to_string(g_asked);
  };
  const auto expect = [&](const char* name, const HostRows& r, const char* want) {
    check(state(r) == want && (r.p != nullptr) == (r.bytes > 0), name, state(r));
    rows.give(r);
  };
  rows.attach();
  rows.attach();
  expect("smallest", rows.take(1), "64 KiB, 1 held, asked 1");
  expect("fits", rows.take(64 << 10), "64 KiB, 1 held, asked 1");
  expect("a_larger_set_takes_the_place", rows.take((64 << 10) + 1), "128 KiB, 1 held, asked 2");
  g_limit = (size_t)1 << 20;
  expect("refused_keeps_the_old", rows.take(600 << 10), "0 KiB, 1 held, asked 3");
  expect("what_fitted_still_fits", rows.take(128 << 10), "128 KiB, 1 held, asked 3");
  expect("refused_size_is_not_asked_for_again", rows.take(1024 << 10), "0 KiB, 1 held, asked 3");
  expect("larger_ones_neither", rows.take(2 << 20), "0 KiB, 1 held, asked 3");
  expect("a_smaller_step_is", rows.take(200 << 10), "256 KiB, 1 held, asked 4");
  HostRows out[7];
  for (HostRows& r : out) r = rows.take(64 << 10);
  check(g_live.size() == 7, "one_for_each_call_at_once", std::to_string(g_live.size()));
  bool apart = true;
  for (int i = 0; i < 7; ++i)
    for (int j = 0; j < i; ++j) apart = apart && out[i].p != out[j].p;
  check(apart, "none_taken_twice", "");
  for (const HostRows& r : out) rows.give(r);
  check(g_live.size() == HostRowsPool::kMaxIdle, "few_lie_idle", std::to_string(g_live.size()));
  expect("the_largest_of_them", rows.take(256 << 10), "256 KiB, 4 held, asked 10");
  rows.detach();
  check(g_live.size() == HostRowsPool::kMaxIdle, "kept_for_the_other_handle", std::to_string(g_live.size()));
  const HostRows late = rows.take(1);
  rows.detach();
  check(g_live.size() == 1, "given_back_with_the_last", std::to_string(g_live.size()));
  rows.give(late);
  check(g_live.empty(), "and_the_one_that_was_out", std::to_string(g_live.size()));
}

int main() {
  pool();
  const auto expect = [](const char* name, const std::string& got, const char* want) { check(got == want, name, got); };
  expect("pieces_and_rest", steps(10, 4, -1), "f0+4 f4+4 f8+2 run wait = 0");
  expect("one_whole_piece", steps(4, 4, -1), "f0+4 run wait = 0");
  expect("first_piece_fails", steps(10, 4, 0), "f0+4 wait = 7");
  expect("later_piece_fails_and_is_waited_for", steps(10, 4, 1), "f0+4 f4+4 wait = 7");
  expect("forward_fails_and_is_waited_for", steps(10, 4, 3), "f0+4 f4+4 f8+2 run wait = 7");
  expect("wait_fails", steps(10, 4, 4), "f0+4 f4+4 f8+2 run wait = 9");
  return g_failed != 0;
}
