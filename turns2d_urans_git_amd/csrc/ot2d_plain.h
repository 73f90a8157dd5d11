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

}  // namespace ot2d
