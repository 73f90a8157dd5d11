// The search's choice among timed launches (pick_launch), compiled and run by
// tests/test_plain_cpu.py.
#include <cstdio>
#include <random>
#include <vector>

#include "ot2d_plain.h"

using ot2d::pick_launch;

int main() {
  int failed = 0;
  auto check = [&](int got, int want, const char* what) {
    if (got != want) {
      std::printf("failed: %s: took %d\n", what, got);
      failed = 1;
    }
  };
  // three candidates, two rounds of three each; candidate 1 is the default
  const float noise[] = {99.8f, 103.f, 101.f, 100.f, 101.f, 102.f, 99.9f, 100.5f, 104.f};
  check(pick_launch(noise, 3, 3, 1), 1, "candidates within the rounds' spread");
  const float close[] = {99.5f, 99.5f, 99.5f, 100.f, 100.f, 100.f, 99.8f, 99.8f, 99.8f};
  check(pick_launch(close, 3, 3, 1), 1, "quiet candidates within 1 %");
  const float clear[] = {95.f, 95.2f, 95.1f, 100.f, 100.3f, 100.1f, 97.f, 97.1f, 97.2f};
  check(pick_launch(clear, 3, 3, 1), 0, "5 % faster");
  const float loud[] = {95.f, 130.f, 95.1f, 100.f, 100.3f, 100.1f, 97.f, 97.1f, 97.2f};
  check(pick_launch(loud, 3, 3, 1), 1, "faster by less than its own rounds differ");
  const float same[] = {100.f, 100.f, 100.f, 100.f};
  check(pick_launch(same, 4, 1, 2), 2, "all equal");
  const float one[] = {7.f};
  check(pick_launch(one, 1, 1, 0), 0, "one candidate");
  // six equal launches timed with 0.5 % of noise: the default stays, but for
  // 1 search in 100
  std::mt19937 g(1);
  std::normal_distribution<float> d(100.f, 0.5f);
  int off = 0;
  for (int t = 0; t < 20000; ++t) {
    std::vector<float> ms(18);
    for (float& v : ms) v = d(g);
    off += pick_launch(ms.data(), 6, 3, 1) != 1;
  }
  std::printf("equal launches: another one taken in %d of 20000 searches\n", off);
  if (off > 200) failed = 1;
  return failed;
}
