// gather.hip -- a chain of data-movement layers in one pass over memory: a source seen through a nearest upsample or a
// replicate pad, a concat of two such sources, an activation, a crop.
//   dst[h, w, :] = act(A[ya, xa, :] ++ B[yb, xb, :]),  (h + TOP, w + LEFT) mapped to each source's own coordinates:
//   divided by UPA / UPB, or moved by (AL, AT) / (BL, BT) and clamped into the source (PADA / PADB).
// The layers' own formulas are those of upsample.hip, pad.hip, copy_transform.hip, activation.hip and slice.hip; the values are
// theirs bit for bit (copies, and one element-wise binary16 operation).
// Definitions: CA, CB (0: no second source), UPA, UPB (1: none), [PADA], [PADB], ACT (0 none, 1 ReLU, 2 LeakyReLU), ALPHA, VEC, PQ.
//
// Bound: memory.  As separate dispatches every layer reads and writes the whole tensor (and concat sources written in place
// fill their lines in pieces); here each source is read once and the result written once.
// Pad, 2x2 pool, upsample, concat, leaky ReLU and crop of 1917 x 1077 x 9: 135 us as five dispatches, 48 us as two (pool.hip through
// the pad, then this one: 120 MB that have to move).
//
// VEC = 8 (whole 8-channel groups): one 16-byte vector per thread.  VEC = 1: a workgroup takes PQ consecutive pixels of one
// output row.  The pixels they come from are one contiguous run of one row in each source; both runs go into LDS with
// 16-byte loads, and the output run, contiguous as well, is written as aligned 4-byte words whose two halves are picked out of
// LDS (as in copy_transform.hip: consecutive lanes read consecutive halves, a store instruction covers 256 bytes).
// Run starts are 2-byte aligned in general; nothing outside a run is touched.  grid.y = output rows.
#include "common.h"
#ifndef KERNEL_NAME
#define KERNEL_NAME gather
#endif
struct PushConstants { unsigned int OUT_W, LEFT, TOP; int AW, AH, AL, AT, BW, BH, BL, BT; };

__device__ DNX_INLINE int clamped(int v, int n) { return v < 0 ? 0 : (v > n - 1 ? n - 1 : v); }
__device__ DNX_INLINE int map_a(unsigned v, int n, int pad) {
#ifdef PADA
  return clamped((int)v - pad, n);
#else
  return (int)(v / UPA);
#endif
}
#if CB
__device__ DNX_INLINE int map_b(unsigned v, int n, int pad) {
#ifdef PADB
  return clamped((int)v - pad, n);
#else
  return (int)(v / UPB);
#endif
}
#endif
__device__ DNX_INLINE _Float16 act1(_Float16 v) {
#if ACT == 1
  return v > (_Float16)0.0f ? v : (_Float16)0.0f;
#elif ACT == 2
  const _Float16 av = (_Float16)(ALPHA) * v;
  return v > av ? v : av;
#else
  return v;
#endif
}

#if VEC == 8
extern "C" __global__ DNX_LAUNCH_BOUNDS(WG) void KERNEL_NAME(const ushort_t *__restrict__ A,
#if CB
                                                             const ushort_t *__restrict__ B,
#endif
                                                             ushort_t *__restrict__ OUT, PushConstants pc) {
  constexpr unsigned CVA = CA / 8, CV = (CA + CB) / 8;
  const unsigned h = DNX_BID_Y;
  const unsigned i = DNX_ROW_INDEX();
  if (i >= pc.OUT_W * CV) return;
  const unsigned w = i / CV, cv = i - w * CV;
  const unsigned X = w + pc.LEFT, Y = h + pc.TOP;
  const ushort_t *p = A + ((size_t)map_a(Y, pc.AH, pc.AT) * pc.AW + map_a(X, pc.AW, pc.AL)) * CA + cv * 8;
#if CB
  const ushort_t *q = B + ((size_t)map_b(Y, pc.BH, pc.BT) * pc.BW + map_b(X, pc.BW, pc.BL)) * CB + (cv - CVA) * 8;
  p = cv < CVA ? p : q;
#endif
  half8 a = __builtin_bit_cast(half8, *reinterpret_cast<const uint4v *>(p));
#pragma unroll
  for (int e = 0; e < 8; ++e) a[e] = act1(a[e]);
  *reinterpret_cast<uint4v *>(OUT + ((size_t)h * pc.OUT_W + w) * (CA + CB) + cv * 8) = __builtin_bit_cast(uint4v, a);
}
#else
// n halves from src into LDS; the last, partial vector element by element
__device__ DNX_INLINE void stage_run(ushort_t *lds, const ushort_t *__restrict__ src, unsigned n) {
  for (unsigned e = (unsigned)DNX_TID * 8; e < n; e += WG * 8) {
    if (e + 8 <= n) *reinterpret_cast<uint4v *>(lds + e) = *reinterpret_cast<const uint4u *>(src + e);
    else
      for (unsigned k = e; k < n; ++k) lds[k] = src[k];
  }
}
extern "C" __global__ DNX_LAUNCH_BOUNDS(WG) void KERNEL_NAME(const ushort_t *__restrict__ A,
#if CB
                                                             const ushort_t *__restrict__ B,
#endif
                                                             ushort_t *__restrict__ OUT, PushConstants pc) {
  constexpr unsigned COUT = CA + CB;
  __shared__ __attribute__((aligned(16))) ushort_t sa[(PQ * CA + 7) / 8 * 8];
#if CB
  __shared__ __attribute__((aligned(16))) ushort_t sb[(PQ * CB + 7) / 8 * 8];
#endif
  const unsigned h = DNX_BID_Y, x0 = DNX_BID_X * PQ, tid = (unsigned)DNX_TID;
  const unsigned npix = pc.OUT_W - x0 < PQ ? pc.OUT_W - x0 : PQ; // (the grid has ceil(OUT_W / PQ) columns: at least one pixel)
  const unsigned X = x0 + pc.LEFT, Y = h + pc.TOP;
  const int a0 = map_a(X, pc.AW, pc.AL), a1 = map_a(X + npix - 1, pc.AW, pc.AL);
  stage_run(sa, A + ((size_t)map_a(Y, pc.AH, pc.AT) * pc.AW + a0) * CA, (unsigned)(a1 - a0 + 1) * CA);
#if CB
  const int b0 = map_b(X, pc.BW, pc.BL), b1 = map_b(X + npix - 1, pc.BW, pc.BL);
  stage_run(sb, B + ((size_t)map_b(Y, pc.BH, pc.BT) * pc.BW + b0) * CB, (unsigned)(b1 - b0 + 1) * CB);
#endif
  DNX_SYNC();
  ushort_t *dst = OUT + ((size_t)h * pc.OUT_W + x0) * COUT;
  const unsigned n = npix * COUT;
  auto pick = [&](unsigned p, unsigned c) {
    const ushort_t v =
#if CB
        c >= CA ? sb[(unsigned)(map_b(X + p, pc.BW, pc.BL) - b0) * CB + (c - CA)] :
#endif
                sa[(unsigned)(map_a(X + p, pc.AW, pc.AL) - a0) * CA + c];
    return __builtin_bit_cast(ushort_t, act1(__builtin_bit_cast(_Float16, v)));
  };
  const unsigned head = (unsigned)((size_t)dst >> 1) & 1u; // 1: the run starts in the middle of a word
  if (head && tid == 0) dst[0] = pick(0, 0);
  // (pixel, channel) of a lane's word advance by a constant per step: no division inside the loop
  constexpr unsigned STEP = 2 * WG, STEP_PIX = STEP / COUT, STEP_CH = STEP % COUT;
  unsigned e = 2 * tid + head, pix = e / COUT, ch = e - pix * COUT;
  for (; e < n; e += STEP) {
    const ushort_t v0 = pick(pix, ch);
    if (e + 1 < n) {
      const bool wrap = ch + 1 == COUT; // the word's second half is the next pixel's first channel
      const ushort_t v1 = pick(wrap ? pix + 1 : pix, wrap ? 0u : ch + 1);
      *reinterpret_cast<unsigned *>(dst + e) = (unsigned)v0 | ((unsigned)v1 << 16);
    } else dst[e] = v0;
    pix += STEP_PIX;
    ch += STEP_CH;
    if (ch >= COUT) {
      ch -= COUT;
      pix += 1;
    }
  }
}
#endif
