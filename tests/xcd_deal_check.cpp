// Tiles over the XCDs (xcd_deal), compiled and run by tests/test_plain_cpu.py.
// Workgroup (x, y) of a launch of (G, records) workgroups runs on XCD
// (y G + x) mod 8.
#include <cstdio>
#include <vector>

#include "ot2d_plain.h"

int main() {
  for (int G = 1; G <= 200; ++G)
    for (int n : {1, G / 3 + 1, G > 7 ? G - 7 : 1, G}) {
      long load[8] = {};
      for (int y = 0; y < 24; ++y) {
        std::vector<int> seen(n, 0), lo(8, n), hi(8, -1), cnt(8, 0);
        long empty = 0;
        for (int x = 0; x < G; ++x) {
          const int t = ot2d::xcd_deal(x, n), c = (int)(((long)y * G + x) % 8);
          if (t < 0) {
            ++empty;
            continue;
          }
          if (t >= n || seen[t]++) {
            std::printf("failed: G %d n %d record %d: workgroup %d takes tile %d\n", G, n, y, x, t);
            return 1;
          }
          ++load[c];
          ++cnt[c];
          lo[c] = t < lo[c] ? t : lo[c];
          hi[c] = t > hi[c] ? t : hi[c];
        }
        int bad = empty != G - n;
        for (int t = 0; t < n; ++t) bad |= seen[t] != 1;
        for (int c = 0; c < 8; ++c) bad |= cnt[c] > 0 && hi[c] - lo[c] + 1 != cnt[c];   // a run of neighbours
        long mn = load[0], mx = load[0];
        for (long l : load) {
          mn = l < mn ? l : mn;
          mx = l > mx ? l : mx;
        }
        if (bad || (n == G && mx - mn > 1)) {
          std::printf("failed: G %d n %d record %d: loads %ld to %ld\n", G, n, y, mn, mx);
          return 1;
        }
      }
    }
  return 0;
}
