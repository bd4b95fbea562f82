// relayout.hip -- interface layout conversion between HWC, CHW and CHWC8
// (index formulas of common/src/denox/memory/tensor/ActivationLayout.hpp:37-66).
// The reference declares SSBO_CHW (dnx.fbs:86-95) but ships no shader that
// accepts it; this kernel is the missing conversion.
// Definitions: CH, SRC_LAYOUT, DST_LAYOUT (0 HWC, 1 CHW, 2 CHWC8).
//
// Four strategies, chosen at compile time:
//   * HWC <-> CHWC8 (CH % 8 == 0): both sides keep 8 channels contiguous, so one thread moves one
//     16-byte vector; 8 consecutive threads cover one pixel, a wave covers 128 contiguous bytes per plane.
//     Grid: ceil(H*W*CH/8 / WG) workgroups.
//   * HWC <-> CHW (CH % 8 == 0, CH <= 256): a workgroup transposes a tile of PX pixels x CH channels.  A thread owns blocks of
//     8 pixels x 8 channels: eight 16-byte accesses on the plane-major side (consecutive threads on consecutive pixels of a
//     plane, at least 128 contiguous bytes), an 8 x 8 transpose in registers, eight 16-byte vectors in LDS; the pixel-major side
//     is one flat run of 16-byte vectors.  LDS holds the tile pixel by pixel, the CH / 8 vectors of a pixel rotated by the
//     pixel's block, so that a wave's accesses spread over the banks.  Bound: memory.  Moving single halves (the strategy
//     below), takes the same time up to 64 channels; 1920 x 1080 x 128 took 215 us in and 270 out (205 and 205 so), and
//     960 x 1080 x 256, element by element in memory, 788 and 352 (218 and 207: 4.9 and 5.1 TB/s).  Grid: ceil(H*W / PX).
//   * HWC <-> CHW (other CH <= 128): a workgroup transposes WG pixels through LDS, so that the plane-major
//     side is accessed one plane at a time (coalesced across pixels) and the pixel-major side as a flat
//     run of 16-byte vectors.  Grid: ceil(H*W / WG) workgroups.
//   * anything else: one thread per pixel, element by element.  Grid: ceil(H*W / WG).
#include "prelude.h"
typedef unsigned short ushort_t;
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
#ifndef WG
#define WG 256
#endif
#ifndef KERNEL_NAME
#define KERNEL_NAME relayout
#endif
struct PushConstants { unsigned int W, H; };

#define IS_BLOCKY(l) ((l) == 0 || (l) == 2)
#if IS_BLOCKY(SRC_LAYOUT) && IS_BLOCKY(DST_LAYOUT) && (CH % 8 == 0)
#define MODE_VEC8 1
#elif ((SRC_LAYOUT == 0 && DST_LAYOUT == 1) || (SRC_LAYOUT == 1 && DST_LAYOUT == 0)) && (CH <= 128)
#if CH % 8 == 0
#define MODE_BLOCK 1
#else
#define MODE_LDS 1
#endif
#elif ((SRC_LAYOUT == 0 && DST_LAYOUT == 1) || (SRC_LAYOUT == 1 && DST_LAYOUT == 0)) && CH % 8 == 0 && CH <= 256
#define MODE_BLOCK 1
#endif
#ifdef MODE_BLOCK
// pixels per workgroup: about one 8 x 8 block per thread and at most 32 KB of LDS (the host sizes the grid with the same rule)
#define PX (CH <= 32 ? 512 : CH <= 64 ? 256 : CH <= 128 ? 128 : 64)
typedef uint4v uint4u __attribute__((aligned(2)));
typedef unsigned short ushort8 __attribute__((ext_vector_type(8)));
#endif

__device__ DNX_INLINE size_t lidx(int layout, size_t HW, size_t pix, unsigned c) {
  if (layout == 0) return pix * CH + c;
  if (layout == 1) return (size_t)c * HW + pix;
  return (size_t)(c >> 3) * (HW * 8) + pix * 8 + (c & 7);
}

extern "C" __global__ DNX_LAUNCH_BOUNDS(WG) void KERNEL_NAME(
    const ushort_t *__restrict__ IN, ushort_t *__restrict__ OUT, PushConstants pc) {
  const size_t HW = (size_t)pc.W * pc.H;
#if defined(MODE_VEC8)
  constexpr unsigned CV = CH / 8;
  const size_t i = (size_t)DNX_BID_X * WG + DNX_TID;
  if (i >= HW * CV) return;
  const size_t pix = i / CV;
  const unsigned c = (unsigned)(i - pix * CV) * 8;
  *reinterpret_cast<uint4v *>(OUT + lidx(DST_LAYOUT, HW, pix, c)) = *reinterpret_cast<const uint4v *>(IN + lidx(SRC_LAYOUT, HW, pix, c));
#elif defined(MODE_BLOCK)
  constexpr unsigned G = CH / 8, PB = PX / 8;
  __shared__ uint4v tile[PX * G];
  const size_t pix0 = (size_t)DNX_BID_X * PX;
  const unsigned t = DNX_TID;
  const size_t left = HW - pix0;
  const unsigned npix = left < PX ? (unsigned)left : PX; // pixels of this tile
  auto slot = [](unsigned p, unsigned g) { return p * G + (g + (p >> 3)) % G; };
  // The pixel-major run starts at pixel pix0, a multiple of 8: aligned like the tensor.
#if SRC_LAYOUT == 1 // CHW -> HWC
  for (unsigned b = t; b < PB * G; b += WG) {
    const unsigned p = b % PB * 8, g = b / PB; // (PB is a power of two)
    if (p >= npix) continue;
    const ushort_t *src = IN + (size_t)g * 8 * HW + pix0 + p;
    ushort8 v[8];
    if (p + 8 <= npix) {
#pragma unroll
      for (unsigned c = 0; c < 8; ++c) v[c] = __builtin_bit_cast(ushort8, *reinterpret_cast<const uint4u *>(src + (size_t)c * HW));
    } else {
#pragma unroll
      for (unsigned c = 0; c < 8; ++c)
#pragma unroll
        for (unsigned j = 0; j < 8; ++j) v[c][j] = p + j < npix ? src[(size_t)c * HW + j] : (ushort_t)0;
    }
#pragma unroll
    for (unsigned j = 0; j < 8; ++j) {
      ushort8 o;
#pragma unroll
      for (unsigned c = 0; c < 8; ++c) o[c] = v[c][j];
      tile[slot(p + j, g)] = __builtin_bit_cast(uint4v, o);
    }
  }
  DNX_SYNC();
  uint4v *dst = reinterpret_cast<uint4v *>(OUT + pix0 * CH);
  for (unsigned i = t; i < npix * G; i += WG) dst[i] = tile[slot(i / G, i % G)];
#else // HWC -> CHW
  const uint4v *src = reinterpret_cast<const uint4v *>(IN + pix0 * CH);
  for (unsigned i = t; i < npix * G; i += WG) tile[slot(i / G, i % G)] = src[i];
  DNX_SYNC();
  for (unsigned b = t; b < PB * G; b += WG) {
    const unsigned p = b % PB * 8, g = b / PB;
    if (p >= npix) continue;
    ushort_t *dst = OUT + (size_t)g * 8 * HW + pix0 + p;
    ushort8 v[8];
#pragma unroll
    for (unsigned j = 0; j < 8; ++j) v[j] = __builtin_bit_cast(ushort8, tile[slot(p + j, g)]); // (past npix: never stored)
    if (p + 8 <= npix) {
#pragma unroll
      for (unsigned c = 0; c < 8; ++c) {
        ushort8 o;
#pragma unroll
        for (unsigned j = 0; j < 8; ++j) o[j] = v[j][c];
        *reinterpret_cast<uint4u *>(dst + (size_t)c * HW) = __builtin_bit_cast(uint4v, o);
      }
    } else {
#pragma unroll
      for (unsigned c = 0; c < 8; ++c)
#pragma unroll
        for (unsigned j = 0; j < 8; ++j)
          if (p + j < npix) dst[(size_t)c * HW + j] = v[j][c];
    }
  }
#endif
#elif defined(MODE_LDS)
  __shared__ __attribute__((aligned(16))) ushort_t tile[WG * CH];
  const size_t pix0 = (size_t)DNX_BID_X * WG;
  const unsigned t = DNX_TID;
  const size_t left = HW - pix0;
  const unsigned npix = left < WG ? (unsigned)left : WG; // pixels of this tile
  const unsigned nelem = npix * CH;
  // The pixel-major run of this tile starts at element pix0 * CH: a multiple of WG * CH * 2 bytes, so 16-byte aligned.
#if SRC_LAYOUT == 1 // CHW -> HWC
  if (t < npix)
#pragma unroll 8
    for (unsigned c = 0; c < CH; ++c) tile[t * CH + c] = IN[(size_t)c * HW + pix0 + t];
  DNX_SYNC();
  ushort_t *dst = OUT + pix0 * CH;
  for (unsigned e = t * 8; e < nelem; e += WG * 8) {
    if (e + 8 <= nelem) *reinterpret_cast<uint4v *>(dst + e) = *reinterpret_cast<const uint4v *>(tile + e);
    else for (unsigned k = e; k < nelem; ++k) dst[k] = tile[k];
  }
#else // HWC -> CHW
  const ushort_t *src = IN + pix0 * CH;
  for (unsigned e = t * 8; e < nelem; e += WG * 8) {
    if (e + 8 <= nelem) *reinterpret_cast<uint4v *>(tile + e) = *reinterpret_cast<const uint4v *>(src + e);
    else for (unsigned k = e; k < nelem; ++k) tile[k] = src[k];
  }
  DNX_SYNC();
  if (t < npix)
#pragma unroll 8
    for (unsigned c = 0; c < CH; ++c) OUT[(size_t)c * HW + pix0 + t] = tile[t * CH + c];
#endif
#else
  const size_t pix = (size_t)DNX_BID_X * WG + DNX_TID;
  if (pix >= HW) return;
#pragma unroll 8
  for (unsigned c = 0; c < CH; ++c)
    OUT[lidx(DST_LAYOUT, HW, pix, c)] = IN[lidx(SRC_LAYOUT, HW, pix, c)];
#endif
}
