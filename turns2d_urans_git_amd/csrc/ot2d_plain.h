// Rules and arithmetic on plain values, shared by the kernels and the CPU
// tests (which include this file alone, with the host compiler).
#pragma once
#if defined(__HIP__)
#define OT2D_PLAIN __host__ __device__ __forceinline__
#else
#define OT2D_PLAIN inline
#endif

namespace ot2d {

// Limit of a wait between the workgroups of one sweep launch, or between the
// waves of one of its workgroups: it is given up after POLLS polls that found
// nothing.  A normal wait is a few microseconds.  Polls and not time, for a
// clock runs on while the queue's waves are put aside for other processes'
// work, all of a launch together, and would end a sweep whose neighbour had
// no chance to run.  A poll of LDS takes upwards of 0.08 us of the wave's
// running time and one of memory about 1 us, so 2^22 of them are 0.3 to 5 s.
struct BoundedWait {
  static constexpr unsigned POLLS = 1u << 22;
  unsigned polls;
  OT2D_PLAIN void start() { polls = 0u; }
  // one more poll has found nothing: give up?
  OT2D_PLAIN bool over() { return ++polls > POLLS; }
};

// Tiles over the chip.  Workgroups go to the 8 XCDs in turn, so in a launch of
// (G, records) workgroups those of one record whose x agrees modulo 8 share
// an XCD.  Each of these 8 classes takes a run of neighbouring tiles, whose
// shared halos then come out of that XCD's L2: tile of workgroup x of a record
// of n <= G tiles, or -1.  A class of workgroups has as many members below n as
// its run has tiles, so G need not be a multiple of 8.  Filled up to one, 1000
// cases of 33x17 (2 tiles each) launched 6 empty workgroups in 8: viscous
// terms 114 us, 39 without them, SA right-hand side 88 and 35; 60 cases 1975
// and 1952 us a step.
OT2D_PLAIN int xcd_deal(int x, int n) {
  const int c = x & 7, len = n >> 3, more = n & 7;
  return x < n ? c * len + (c < more ? c : more) + (x >> 3) : -1;
}

// The launch choice a search keeps: n candidates timed in `rounds` rounds,
// candidate k's times at ms[k * rounds].  The fastest (by its best round) is
// taken over candidate `def` only if it wins by more than the rounds of
// both differ among themselves, and by more than 1 %: the choices of a
// class often lie closer than that (513x129 SA FP32: 263.3, 264.4, 264.8,
// 265.6, 268.6, 270.0 us a step), and by the best time alone a search took
// one that is slower than the default.
inline int pick_launch(const float* ms, int n, int rounds, int def) {
  auto low = [&](int k) {
    float v = ms[k * rounds];
    for (int r = 1; r < rounds; ++r) v = ms[k * rounds + r] < v ? ms[k * rounds + r] : v;
    return v;
  };
  auto spread = [&](int k) {
    float v = ms[k * rounds];
    for (int r = 1; r < rounds; ++r) v = ms[k * rounds + r] > v ? ms[k * rounds + r] : v;
    return v - low(k);
  };
  int best = def;
  for (int k = 0; k < n; ++k)
    if (low(k) < low(best)) best = k;
  const float both = spread(def) + spread(best), least = 0.01f * low(def), need = both > least ? both : least;
  return low(def) - low(best) > need ? best : def;
}

}  // namespace ot2d
