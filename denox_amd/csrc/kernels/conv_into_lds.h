// Pieces that the persistent kernels with weights and halos straight into LDS share (conv3x3_mfma_dl.hip, conv3x3_upshare.hip).
#include "conv_common.h"

#ifndef NXCD
#define NXCD 8
#endif
#define NKT (KOUTP / KT)

// every memory instruction of this wave but the `n` newest has completed (they complete in issue order)
#define STEP_WAIT(n) __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")

// The lane's number as the compiler has not seen it yet.  What follows from it alone (slots, rows and columns of all vectors) is derived
// again where it is needed: kept from unit to unit (the compiler moves it out of the loop) it takes registers that the accumulators need.
__device__ DNX_INLINE int fresh_lane_of(int lane) {
  __asm__ volatile("" : "+v"(lane));
  return lane;
}

// Holds a step's matrix instructions in front of its barrier: they touch no memory, and in a block without branches the compiler
// otherwise collects several steps' worth behind it, their operands in scratch memory meanwhile.
__device__ DNX_INLINE void pin(float16v &v) { __asm__ volatile("" : "+v"(v)); }

// The units of work of one workgroup: unit, unit + NKT * SLOTS, ... below last.  Each XCD has a contiguous band of them.
struct UnitBand {
  int unit, last;
};
__device__ DNX_INLINE UnitBand unit_band(int units) {
  const int perXcd = (units + NXCD - 1) / NXCD;
  const int first = (int)(DNX_BID_X % NXCD) * perXcd;
  UnitBand b;
  b.last = first + perXcd < units ? first + perXcd : units;
  b.unit = first + (int)(DNX_BID_X / NXCD);
  return b;
}
