// Waits of the LU-SGS sweeps (compiled and run by tests/test_plain_cpu.py).
// A wave polls for a neighbour's word that arrives after `need` of its polls;
// a clock beside it runs on while the queue is put aside.
#include <cstdio>

#include "ot2d_plain.h"

using ot2d::BoundedWait;

namespace {
double clock_s = 0.0;   // advances by a poll's time, and by the time aside

// the polls done, negative when the wait was given up
long wait_for(BoundedWait& w, long need, long aside_at, double aside_s, double poll_s) {
  w.start();
  for (long polls = 0;; ++polls) {
    if (polls >= need) return polls;
    clock_s += poll_s;
    if (polls == aside_at) clock_s += aside_s;
    if (w.over()) return -polls - 1;
  }
}

int failed = 0;
void check(bool ok, const char* what) {
  if (!ok) {
    std::printf("failed: %s\n", what);
    failed = 1;
  }
}
}  // namespace

int main() {
  BoundedWait w;
  check(wait_for(w, 200, -1, 0, 1e-6) == 200, "a wait of 200 polls ends");
  check(wait_for(w, 200, 3, 10.0, 1e-6) == 200, "put aside for 10 s in the middle");
  check(wait_for(w, 200, 0, 3600.0, 8e-8) == 200, "put aside for an hour at the first poll");
  check(wait_for(w, 1000000, 5, 10.0, 8e-8) == 1000000, "a million polls still to go after 10 s aside");
  // a neighbour that never answers: given up, the shortest poll not before
  // 0.3 s of running time, the longest not after 10 s
  for (int longest = 0; longest < 2; ++longest) {
    const double poll_s = longest ? 2e-6 : 8e-8, t0 = clock_s;
    check(wait_for(w, 1L << 40, -1, 0, poll_s) < 0, "a wait without an answer is given up");
    const double took = clock_s - t0;
    check(took > 0.3 && took < 10.0, "between 0.3 and 10 s of running time");
  }
  check(wait_for(w, 1L << 40, 10, 10.0, 1e-6) < 0, "given up after having been put aside too");
  check(wait_for(w, 1000000, -1, 0, 1e-6) == 1000000, "start() starts the count afresh");
  return failed;
}
