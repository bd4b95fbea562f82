// conv3x3_upshare.hip -- 3x3 convolution over concat(upsample2x(A), B) that multiplies every low-resolution pixel of A once per tap.
//
// Nearest-neighbour upsampling repeats a pixel in a 2x2 block, so along one axis the taps (w0, w1, w2) of output 2y + 1 read the source
// pixels (y, y, y + 1) and those of output 2y (y - 1, y, y).  With
//     M(y) = w1 a[y]          E(y) = w0 a[y] + w2 a[y + 1]      (E belongs to the edge between y and y + 1)
// both are one addition away from shared products: out(2y) = M(y) + E(y - 1), out(2y + 1) = M(y) + E(y).  In two dimensions four
// accumulators per source pixel -- MM (1 tap), ME (2: an edge in x), EM (2: an edge in y), EE (4) -- hold 9 products per source pixel
// where the convolution's definition takes 36 and weights folded by parity class (conv3x3_upfold.hip) take 16, and no weight is
// summed or rounded: the arithmetic is the definition's with its binary32 sums in another order.
//     C_b(y) = MM(y) + ME(y, x - 1 + b)   R_b(y) = EM(y) + EE(y, x - 1 + b)   out(2y + a, 2x + b) = C_b(y) + R_b(y - 1 + a)
// The edge left of a pixel belongs to the neighbouring lane (a DPP operand of the addition).  B keeps its 9 taps per output pixel.
//
// Mapping (v_mfma_f32_32x32x16_f16, weights as the M operand).  A wave computes 32 output channels for RPW edges: the 2 RPW
// output rows around them, from RPW + 1 rows of C and RPW rows of R, over 32 consecutive source pixels; the first lane only supplies
// the left edge of the second, so 31 pixels = 62 output columns are stored.  RPW = 2: 10 accumulators, 21 matrix instructions
// per 16 channels of A for 4 x 62 outputs of 32 channels.  The WAVES waves of a workgroup are KB = KT / 32 channel blocks x RG row
// groups that share a halo and the weights.
//
// All channels come in steps -- CKA channels of A, then 16 of B -- with the step's weights and halo in one of two LDS buffers.  The other
// buffer is filled meanwhile straight from memory (buffer_load ... lds): the weights lie in memory in the order of the fragments
// (1 KiB each, lane by lane), so their copy is linear and their reads conflict-free; a halo pixel takes CKA / 8 slots of 16 bytes whose
// order is rotated by the pixel's column, so that 16 lanes reading the same channels of 16 consecutive pixels hit 16 different
// bank groups.  One barrier per step.  A source whose channels are not whole vectors goes through registers.
//
// What bounds it: the LDS-fed matrix rate and, beside it, loads and stores that overlap it only in part.  64 + 9 -> 64 channels at
// 1920 x 1088: 71 us with neither, 82 with stores, 90 with loads, 105 - 112 with both (memory alone: 371 MB, 73).  Microseconds a launch inside
// frames of the U-Nets by estimates, the other exact kernels before: that layer 160 and 109, 96 + 32 -> 64 at 960 x 544 80 and 50, 112 + 48 -> 96 at 480 x 272
// 39 and 35, 192 + 64 -> 128 at 960 x 544 259 and 143, 128 + 9 -> 128 at 1920 x 1088 619 and 273.  Back to back, caches warm, small
// images take less: 112 + 48 -> 96 25, 96 + 32 -> 64 45.  Four waves to a workgroup (one per SIMD) are slower on every layer measured.
//
// Launch: persistent, NXCD * NKT * SLOTS workgroups; a unit of work is (tile, slice of KT output channels), each XCD has a contiguous band.
// Definitions: as conv_common.h (UPA = 1), plus CKA and SLOTS.
#include "conv_into_lds.h"

#ifndef KERNEL_NAME
#define KERNEL_NAME conv3x3_upshare
#endif
static_assert(UPA == 1 && MF == 32 && !POOL && !CROP && !PADA && KR == 3 && KS == 3 && PY == 1 && PX == 1 && SY == 1 && SX == 1 && PW == 0, "upsampled source A, plain 3 x 3");
static_assert(CA % 8 == 0 && (CB == 0 || CB >= 8), "whole vectors of A; B with at least one");
static_assert(KOUT % 8 == 0 && OPITCH % 8 == 0 && OVEC, "two 16-byte stores per accumulator: the wait for a step's loads counts them");

#define RG (WAVES / KB)
static_assert(KOUTP % KT == 0 && WAVES % KB == 0, "whole slices and row groups");
#define CAP ((CA + 15) / 16 * 16)
#define CBP ((CB + 15) / 16 * 16)
#define NA (CAP / CKA)
#define NB (CBP / 16)
static_assert(CAP % CKA == 0 && (CKA == 16 || CKA == 32 || CKA == 64), "whole steps of a power of two of vectors");
#define GA (CKA / 8)                  // slots per halo pixel of A
#define AROWS (RG * RPW + 1)
#define ACOLS 33
#define BROWS (2 * RG * RPW + 2)
#define BCOLS 33                      // per column parity
#define WAFRAGS (9 * KB * (CKA / 16)) // weight fragments of a step
#define WBFRAGS (9 * KB)
#define AGROUPS ((AROWS * ACOLS * GA + 63) / 64) // halo loads of one wave's 64 lanes
#define BGROUPS ((BROWS * BCOLS * 2 * 2 + 63) / 64)
#define CMAX(a, b) ((a) > (b) ? (a) : (b))
#define BUF_SLOTS (64 * CMAX(WAFRAGS + AGROUPS, CB > 0 ? WBFRAGS + BGROUPS : 0))
#define BDMA (CB % 8 == 0)            // B straight into LDS as well
#define NVA ((AGROUPS + WAVES - 1) / WAVES)
#define NVB ((BGROUPS + WAVES - 1) / WAVES)
#define AITEMS (NVA + (WAFRAGS + WAVES - 1) / WAVES) // load instructions of a wave per step
#define BITEMS (NVB + (WBFRAGS + WAVES - 1) / WAVES)
#define OUT_ROWS (2 * RPW)
#define NSTORES (OUT_ROWS * 4)        // store instructions of a wave per tile
static_assert(NSTORES <= 63, "the wait's counter");

// Between LDS accesses of one wave whose lanes read what other lanes wrote: the hardware serves them in order, and here the compiler
// keeps that order too (it reasons lane by lane and may exchange accesses that never meet in one lane).  No instruction comes of it.
__device__ DNX_INLINE void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x - 1's value: lane i receives lane i - 1's (lanes 0 and 32 hold the pixel that only supplies its edge)
__device__ DNX_INLINE float from_prev_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true)); // wave_shr:1
}

extern "C" __global__ DNX_LAUNCH_BOUNDS(NT) void KERNEL_NAME(
    const _Float16 *__restrict__ A,
#if CB > 0
    const _Float16 *__restrict__ B,
#endif
    _Float16 *__restrict__ OUT, const _Float16 *__restrict__ FILT,
#if HAS_BIAS
    const _Float16 *__restrict__ BIAS,
#endif
    PushConstants pc) {
  // One LDS object: beside a second one the compiler waits for every load into LDS in front of every LDS read.
  __shared__ uint4v sBuf[2 * BUF_SLOTS + KOUTP / 4 + WAVES * 256];
  bias_t *const sBias = (bias_t *)(sBuf + 2 * BUF_SLOTS);
  uint4v *const sRow = sBuf + 2 * BUF_SLOTS + KOUTP / 4; // an output row of each wave on its way to memory
#if CB == 0
  const _Float16 *B = nullptr;
#endif
  const int tid = DNX_TID;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int kb = wv % KB, rg = wv / KB; // this wave's channel block and row group
  const OutBuf out = out_buffer(OUT, pc);
  const Sources srcs = make_sources(A, B, pc);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(A), 0, (int)srcs.bytesA, 0x00020000);
#if CB > 0
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(B), 0, (int)srcs.bytesB, 0x00020000);
#endif
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(FILT), 0, KOUTP * 9 * (CAP + CBP) * 2, 0x00020000);

  const int WL = (int)(pc.IN_W >> 1), HL = (int)(pc.IN_H >> 1);
  const int tilesX = (WL + 30) / 31, tilesY = (2 * HL + OUT_ROWS * RG) / (OUT_ROWS * RG); // the first output row of the first tile is row -1
  const int units = HL > 0 ? tilesX * tilesY * NKT : 0;
  const UnitBand band = unit_band(units);
  const int last = band.last;
  int unit = band.unit;
  if (unit >= last)
    return; // uniform for the workgroup
  const bool rev = (pc.FLAGS & 1u) != 0;
  struct Geo { int kt, x0, y0; }; // slice; source column of lane 0 and source row of the first C row
  auto geometry = [&](int u) {
    Geo g;
    g.kt = u % NKT;
    int t = u / NKT;
    t = rev ? tilesX * tilesY - 1 - t : t;
    const int ty = t / tilesX;
    g.x0 = (t - ty * tilesX) * 31 - 1;
    g.y0 = ty * (RG * RPW) - 1;
    return g;
  };

#if HAS_BIAS
  for (int i = tid; i < KOUTP; i += NT) sBias[i] = (float)BIAS[i];
#endif

  // ---- loads of a step into a buffer ----
  auto fresh_lane = [&]() { return fresh_lane_of(lane); };
  // A step's loads are items, a wave's share of one load instruction per 64 slots each, which the matrix loops issue one by one between their
  // instructions: a memory instruction waits for room in the memory pipeline, and all of a step's in front of its matrix work left
  // the matrix cores idle for that time.  No branch: a wave without an item left repeats the last one (the same bytes to the same place).
  auto weights_item = [&](int buf, int frag0, int N, int q) { // of N fragments of the packed weights from frag0 on
    const int f = wv + q * WAVES < N ? wv + q * WAVES : N - 1;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void_t *)(sBuf + buf * BUF_SLOTS + f * 64), 16, fresh_lane() * 16, (frag0 + f) * 1024, 0, 0);
  };
  // Byte offsets of this lane's halo vectors in their source at the step's first channel 0; NO_LOAD outside the image (reads as zero).
  // From one unit to the next they move by the same amount where both halos lie inside the image; only at its borders every vector is
  // looked at (20 - 40 vector instructions each, beside matrix instructions that wait for the same issue slots).
  unsigned aoff[NVA];
  auto a_group = [&](int i) { return wv + i * WAVES < AGROUPS ? wv + i * WAVES : AGROUPS - 1; };
  // slot i of A's halo: pixel (row, column) and the channel group that belongs there; past the halo its last row again
  auto a_slot = [&](unsigned i, unsigned &hy, unsigned &hx, unsigned &grp) {
    const unsigned pix = i / GA;
    hy = pix / ACOLS;
    hx = pix - hy * ACOLS;
    hy = hy < AROWS ? hy : AROWS - 1;
    grp = (i - hx / (16 / GA)) & (GA - 1);
  };
  auto a_inside = [&](const Geo &g) { return (g.y0 >= 0) & (g.y0 + AROWS <= HL) & (g.x0 >= 0) & (g.x0 + ACOLS <= WL); };
  auto aim_a = [&](const Geo &g) {
    const unsigned ln = (unsigned)fresh_lane();
#pragma unroll
    for (int i = 0; i < NVA; ++i) {
      unsigned hy, hx, grp;
      a_slot((unsigned)a_group(i) * 64 + ln, hy, hx, grp);
      const int y = g.y0 + (int)hy, x = g.x0 + (int)hx;
      const unsigned p = (unsigned)(y * WL + x);
      aoff[i] = (((unsigned)y < (unsigned)HL) & ((unsigned)x < (unsigned)WL)) ? (LAYIN ? p * 16u + grp * srcs.planeA : p * (CA * 2u) + grp * 16u) : NO_LOAD;
    }
  };
  auto move_a = [&](const Geo &from, const Geo &to) {
    if (a_inside(from) & a_inside(to)) {
      const unsigned d = (unsigned)((to.y0 - from.y0) * WL + to.x0 - from.x0) * (LAYIN ? 16u : CA * 2u);
#pragma unroll
      for (int i = 0; i < NVA; ++i) aoff[i] += d;
    } else
      aim_a(to);
  };
  auto item_a = [&](int buf, const Geo &g, int k, int i) { // item i of the step with the channels from k * CKA on
    if (i < NVA) {
      bool ok = aoff[i] != NO_LOAD;
      if (CA % 16 != 0) { // channels past CA are staged as zeros: their weights are zero, but 0 * NaN is NaN
        unsigned hy, hx, grp;
        a_slot((unsigned)(a_group(i) * 64 + fresh_lane()), hy, hx, grp);
        ok = ok & (k * CKA + (int)grp * 8 < CA);
      }
      const unsigned off = aoff[i] + (LAYIN ? (unsigned)(k * GA) * srcs.planeA : (unsigned)(k * CKA * 2));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t *)(sBuf + buf * BUF_SLOTS + (WAFRAGS + a_group(i)) * 64), 16, ok ? off : NO_LOAD, 0, 0, LOAD_AUX);
    } else
      weights_item(buf, g.kt * (9 * KB * ((CAP + CBP) / 16)) + k * WAFRAGS, WAFRAGS, i - NVA);
  };
#if CB > 0
  // Slots of B's halo: two per pixel, pixels by row, column parity and column pair; the channel groups of 8 pixels with the same slots
  // modulo 16 as the 8 before them change places.  Straight into LDS, the slot belongs to the lane and the group follows (as for A);
  // through registers, the lane takes group lane % 2 and writes it where it belongs.
  unsigned boff[NVB];
  auto b_group = [&](int i) { return wv + i * WAVES < BGROUPS ? wv + i * WAVES : BGROUPS - 1; };
  auto b_slot = [&](unsigned i, unsigned &hy, unsigned &col, unsigned &grp, unsigned &slot) {
    const unsigned pix = i >> 1;
    hy = pix / (2 * BCOLS);
    const unsigned rem = pix - hy * (2 * BCOLS), par = rem >= BCOLS ? 1 : 0, idx = rem - par * BCOLS;
    col = 2 * idx + par;
    grp = BDMA ? (i - (idx >> 3)) & 1 : i & 1;
    slot = BDMA ? i : pix * 2 + ((i + (idx >> 3)) & 1);
    hy = hy < BROWS ? hy : BROWS - 1; // past the halo: its last row again
  };
#if PADB
  auto b_inside = [&](const Geo &g) {
    const int y = 2 * g.y0, x = 2 * g.x0 - 1;
    return (y >= (int)pc.PAD_T) & (y + BROWS <= (int)(pc.PAD_T + pc.SRC_H)) & (x >= (int)pc.PAD_L) & (x + 2 * BCOLS <= (int)(pc.PAD_L + pc.SRC_W));
  };
  const int pitchB = (int)pc.SRC_W;
#else
  auto b_inside = [&](const Geo &g) {
    const int y = 2 * g.y0, x = 2 * g.x0 - 1;
    return (y >= 0) & (y + BROWS <= (int)pc.IN_H) & (x >= 0) & (x + 2 * BCOLS <= (int)pc.IN_W);
  };
  const int pitchB = (int)pc.IN_W;
#endif
  auto aim_b = [&](const Geo &g) {
    const unsigned ln = (unsigned)fresh_lane();
#pragma unroll
    for (int i = 0; i < NVB; ++i) {
      unsigned hy, col, grp, slot;
      b_slot((unsigned)b_group(i) * 64 + ln, hy, col, grp, slot);
      const int y = 2 * g.y0 + (int)hy, x = 2 * g.x0 - 1 + (int)col;
#if PADB
      const int sy = clampi(y - (int)pc.PAD_T, 0, (int)pc.SRC_H - 1), sx = clampi(x - (int)pc.PAD_L, 0, (int)pc.SRC_W - 1);
#else
      const int sy = y, sx = x;
#endif
      const unsigned p = (unsigned)(sy * pitchB + sx);
      boff[i] = (((unsigned)y < pc.IN_H) & ((unsigned)x < pc.IN_W)) ? (LAYIN ? p * 16u + grp * srcs.planeB : p * (CB * 2u) + grp * 16u) : NO_LOAD;
    }
  };
  auto move_b = [&](const Geo &from, const Geo &to) {
    if (b_inside(from) & b_inside(to)) {
      const unsigned d = (unsigned)(2 * (to.y0 - from.y0) * pitchB + 2 * (to.x0 - from.x0)) * (LAYIN ? 16u : CB * 2u);
#pragma unroll
      for (int i = 0; i < NVB; ++i) boff[i] += d;
    } else
      aim_b(to);
  };
  uint4v breg[BDMA ? 1 : NVB];
  auto item_b = [&](int buf, const Geo &g, int j, int i) {
    if (i < NVB) {
      const bool ok = boff[i] != NO_LOAD;
#if BDMA
      const unsigned off = boff[i] + (LAYIN ? (unsigned)(2 * j) * srcs.planeB : (unsigned)(j * 32));
      const bool beyond = CB % 16 != 0 && j == NB - 1; // 8 channels in the last step: the second group is staged as zeros
      unsigned hy, col, grp = 0, slot;
      if (beyond) b_slot((unsigned)(b_group(i) * 64 + fresh_lane()), hy, col, grp, slot);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void_t *)(sBuf + buf * BUF_SLOTS + (WBFRAGS + b_group(i)) * 64), 16, (ok & !(beyond & (grp == 1))) ? off : NO_LOAD, 0, 0, LOAD_AUX);
#else
      // the partial last vector is fetched so that it ends at the pixel's last channel and shifted down when it is written to LDS
      constexpr int REM = CB - (NB - 1) * 16; // channels of the last step
      unsigned off = boff[i] + (unsigned)(j * 32);
      const bool odd = (fresh_lane() & 1) != 0;
      if (j == NB - 1) {
        if (REM < 8) off = odd ? NO_LOAD : off - (8 - REM) * 2u;
        else off -= odd ? (16 - REM) * 2u : 0u;
      }
      breg[i] = __builtin_amdgcn_raw_buffer_load_b128(rb, ok ? off : NO_LOAD, 0, LOAD_AUX);
#endif
    } else
      weights_item(buf, g.kt * (9 * KB * ((CAP + CBP) / 16)) + 9 * KB * (CAP / 16) + j * WBFRAGS, WBFRAGS, i - NVB);
  };
  auto commit_b = [&](int buf, int j) {
#if !BDMA
    const bool part = j == NB - 1 && (fresh_lane() & 1) == (CB % 16 > 8 ? 1 : 0); // this lane's vectors are the partial ones
    typedef __attribute__((address_space(3))) uint4v lds_slot_t;
    lds_slot_t *dst = (lds_slot_t *)(__attribute__((address_space(3))) void *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + WBFRAGS * 64));
#pragma unroll
    for (int i = 0; i < NVB; ++i) {
      const uint4v sh = shr_halves<(8 - CB % 8) % 8>(breg[i]);
      uint4v v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = part ? sh[e] : breg[i][e];
      unsigned hy, col, grp, slot;
      b_slot((unsigned)(b_group(i) * 64 + fresh_lane()), hy, col, grp, slot);
      dst[slot] = v;
    }
#endif
  };
#endif

  // ---- matrix work ----
  float16v mm[RPW + 1], me[RPW + 1], em[RPW], ee[RPW];
  auto step_a = [&](int buf, auto item, const int nitems) { // item(i): item i of the loads for the next step
    const int KS_ = CKA / 16;
    typedef __attribute__((address_space(3))) const char lds_char_t;
    const int ln = fresh_lane(), l32 = ln & 31, kh = ln >> 5;
    lds_char_t *wb, *pb[2][CKA / 16];
    wb = (lds_char_t *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + (kb * KS_) * 64 + ln));
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int ks = 0; ks < CKA / 16; ++ks) {
        const int x = l32 + cc;
        pb[cc][ks] = (lds_char_t *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + WAFRAGS * 64 + (rg * RPW * ACOLS + x) * GA + ((2 * ks + kh + x / (16 / GA)) & (GA - 1))));
      }
    // Per 16 channels 9 units, one per tap: a weight fragment and the 2 or 3 matrix instructions per RPW = 2 that use it -- first
    // the taps that read column x, then those that read x + 1, so that either column's pixel fragments are replaced while the
    // other's are multiplied.  Reads run two units ahead; scheduling barriers keep the order.
    constexpr int taps[9] = {4, 1, 7, 3, 0, 6, 5, 2, 8}; // r * 3 + s
    half8 wf[3], px[2][RPW + 1];
    auto read_w = [&](int u) {
      const int ks = u / 9, tap = taps[u % 9];
      wf[u % 3] = *(__attribute__((address_space(3))) const half8 *)(wb + (tap * KB * KS_ + ks) * 1024);
    };
    auto read_p = [&](int cc, int ks) {
#pragma unroll
      for (int t = 0; t <= RPW; ++t)
        px[cc][t] = *(__attribute__((address_space(3))) const half8 *)(pb[cc][ks] + t * (ACOLS * GA * 16));
    };
    read_p(0, 0);
    read_w(0);
    read_w(1);
#pragma unroll
    for (int u = 0; u < 9 * (CKA / 16); ++u) {
      if (u + 2 < 9 * (CKA / 16)) read_w(u + 2);
      if (u % 9 == 3) read_p(1, u / 9);
      if (u % 9 == 6 && u / 9 + 1 < CKA / 16) read_p(0, u / 9 + 1);
      {
        constexpr int UNITS = 9 * (CKA / 16);
#pragma unroll
        for (int i = u * nitems / UNITS; i < (u + 1) * nitems / UNITS; ++i) item(i);
      }
      __builtin_amdgcn_sched_barrier(0);
      const half8 w = wf[u % 3];
      const int tap = taps[u % 9], r = tap / 3, s = tap % 3, cc = s == 2 ? 1 : 0;
      if (r == 1) {
#pragma unroll
        for (int t = 0; t <= RPW; ++t) {
          if (s == 1) mm[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, px[cc][t], mm[t], 0, 0, 0);
          else me[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, px[cc][t], me[t], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int t = 0; t < RPW; ++t) {
          const int row = t + (r == 2 ? 1 : 0);
          if (s == 1) em[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, px[cc][row], em[t], 0, 0, 0);
          else ee[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, px[cc][row], ee[t], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  auto pin_a = [&]() {
#pragma unroll
    for (int t = 0; t <= RPW; ++t) {
      pin(mm[t]);
      pin(me[t]);
      if (t < RPW) { pin(em[t]); pin(ee[t]); }
    }
  };

  // An output row of this wave, 64 pixels x 32 channels: activation, rounding, and through LDS of its own into the order in which 64 lanes
  // store consecutive 16-byte pieces -- whole 64-byte channel ranges of 16 pixels, or 64 pixels of one 8-channel plane.  (Stored from the
  // accumulators' lanes, every piece lies in another line and an instruction takes four times as long.)  Pixel p, 8-channel group c of 4
  // goes to slot (4 p + c) of 16-slot rows, XOR-ed with the row: conflict-free both ways.
  unsigned ooff[4]; // byte offsets of this lane's four pieces inside an output row of the unit; NO_STORE where there is nothing to store
  auto aim_out = [&](const Geo &g) {
    const int ln = fresh_lane(), ch0 = g.kt * KT + kb * 32;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int p = LAYOUT_OUT ? ln : q * 16 + (ln >> 2), c = LAYOUT_OUT ? q : ln & 3, x = 2 * g.x0 + p;
      const unsigned off = LAYOUT_OUT ? (unsigned)((ch0 >> 3) + c) * out_plane_bytes(pc) + (unsigned)x * 16u : ((unsigned)x * OPITCH + (unsigned)(ch0 + c * 8)) * 2u;
      // (pixels 0 and 1 belong to the lane that only supplies its edge)
      ooff[q] = ((p >= 2) & (x < (int)pc.IN_W) & (ch0 + c * 8 < KOUT)) ? off : NO_STORE;
    }
  };
  // A result that fills most of the memory-side cache (256 MB) is stored past it: little of it would be left there for its reader, and what
  // it displaces are this kernel's own halos.  267 MB 112 -> 102 us, 535 MB 273 -> 250; 134 MB (192 + 64 -> 128 at 960 x 544) 134 -> 139.
  const bool streamed = (unsigned long long)pc.IN_W * pc.IN_H * (OPITCH * 2u) > 192ull << 20;
  const OutBuf nowhere = __builtin_amdgcn_make_buffer_rsrc(OUT, 0, 0, 0x00020000); // a row outside the image: the hardware drops the stores
  auto finish_row = [&](const Geo &g, int r, const float16v &acc0, const float16v &acc1) {
    const int ln = fresh_lane(), l32 = ln & 31;
    typedef __attribute__((address_space(3))) uint4v lds_slot_t;
    typedef __attribute__((address_space(3))) char lds_byte_t;
    const unsigned row = (unsigned)(size_t)(lds_byte_t *)(__attribute__((address_space(3))) void *)(sRow + wv * 256);
    // byte address of pixel 2 l32, group 2 (lane / 32); pixel 2 l32 + b and group + e are at its XOR with 64 b + 16 e
    const unsigned wr = (unsigned)((l32 >> 1) * 256 + ((((l32 & 1) * 8 + (ln >> 5) * 2) ^ (l32 >> 1)) * 16));
    wave_lds_order(); // the row before has been read
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = b ? acc1[i] : acc0[i];
      const half8 h[2] = {finish8(v), finish8(v + 8)};
#pragma unroll
      for (int e = 0; e < 2; ++e) *(lds_slot_t *)(size_t)(row + (wr ^ (b * 64u + e * 16u))) = __builtin_bit_cast(uint4v, h[e]);
    }
    wave_lds_order();
    // piece q: pixel 16 q + lane / 4, group lane % 4, or pixel lane, group q
    const unsigned rd = LAYOUT_OUT ? (unsigned)((ln >> 2) * 256 + (((ln & 3) * 4) ^ (ln >> 2)) * 16) : (unsigned)((ln >> 4) * 256 + ((ln & 15) ^ (ln >> 4)) * 16);
    const int y = 2 * (g.y0 + rg * RPW) + 1 + r;
    // (no scalar offset outside either: a range check of `size - scalar offset` would wrap for a size of 0)
    const bool inside = (unsigned)y < pc.IN_H;
    const OutBuf to = inside ? out : nowhere;
    const int rowBytes = inside ? (int)((unsigned)y * pc.IN_W * (LAYOUT_OUT ? 16u : OPITCH * 2u)) : 0;
    uint4v v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = *(lds_slot_t *)(size_t)(row + (LAYOUT_OUT ? rd ^ (q * 16u) : (rd ^ (q * 64u)) + q * 1024u));
    if (streamed) {
#pragma unroll
      for (int q = 0; q < 4; ++q) __builtin_amdgcn_raw_buffer_store_b128(v[q], to, ooff[q], rowBytes, 2);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) __builtin_amdgcn_raw_buffer_store_b128(v[q], to, ooff[q], rowBytes, 0);
    }
  };

  int buf = 0;
  Geo g = geometry(unit);
  aim_a(g);
#if CB > 0
  aim_b(g);
#endif
#pragma unroll
  for (int i = 0; i < AITEMS; ++i) item_a(0, g, 0, i);
  STEP_WAIT(0);
  DNX_SYNC();
  for (;;) {
    const int next = unit + NKT * SLOTS;
    const bool more = next < last;
    const int hsel = fresh_lane() >> 5;
    const Geo gn = geometry(more ? next : unit); // (behind the last unit its own first step is loaded once more and not used)
#pragma unroll
    for (int t = 0; t <= RPW; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        mm[t][i] = HAS_BIAS ? sBias[g.kt * KT + kb * 32 + hsel * 16 + i] : 0.0f;
        me[t][i] = 0.0f;
        if (t < RPW) { em[t][i] = 0.0f; ee[t][i] = 0.0f; }
      }
    for (int k = 0; k < NA - 1; ++k) {
      step_a(buf, [&](int i) { item_a(buf ^ 1, g, k + 1, i); }, AITEMS);
      pin_a();
      STEP_WAIT(0);
      DNX_SYNC();
      buf ^= 1;
    }
#if CB > 0
    step_a(buf, [&](int i) { item_b(buf ^ 1, g, 0, i); }, BITEMS);
    commit_b(buf ^ 1, 0);
#else
    move_a(g, gn);
    step_a(buf, [&](int i) { item_a(buf ^ 1, gn, 0, i); }, AITEMS);
#endif
    pin_a();
    // A's part of the outputs: row i of the wave's 2 RPW output rows is a = (i + 1) % 2 of source row (i + 1) / 2, edge i / 2.  In place: row
    // 2 t takes the registers of C(t), row 2 t + 1 those of R(t).
    auto combine = [&]() {
#pragma unroll
      for (int t = 0; t <= RPW; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float m = mm[t][i], e = me[t][i];
          mm[t][i] = m + from_prev_lane(e);
          me[t][i] = m + e;
        }
        pin(mm[t]);
        pin(me[t]);
        if (t < RPW) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float m = em[t][i], e = ee[t][i];
            em[t][i] = m + from_prev_lane(e);
            ee[t][i] = m + e;
          }
          pin(em[t]);
          pin(ee[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < RPW; ++t) {
        mm[t] += em[t];
        me[t] += ee[t];
        pin(mm[t]);
        pin(me[t]);
        em[t] += mm[t + 1];
        ee[t] += me[t + 1];
        pin(em[t]);
        pin(ee[t]);
      }
    };
    auto out_acc = [&](int r, int b) -> float16v & { return r % 2 ? (b ? ee[r / 2] : em[r / 2]) : (b ? me[r / 2] : mm[r / 2]); };
#if CB > 0
    // 16 channels of B, 9 taps: output row r, column parity b, tap (tr, ts) reads halo row r + tr, column 2 l + b + ts.  Halo row by halo
    // row: its 4 pixel fragments feed every output row that reads it (1, 2 or 3 of them), the next row's are read meanwhile.
    // FINAL: output row r, complete after halo row r + 2, is stored behind the next halo row's matrix instructions.
    auto step_b = [&](int buf, auto item, const int nitems, const bool FINAL) {
      typedef __attribute__((address_space(3))) const char lds_char_t;
      typedef __attribute__((address_space(3))) const half8 *lds_frag;
      const int ln = fresh_lane(), l32 = ln & 31, kh = ln >> 5;
      lds_char_t *wb = (lds_char_t *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + kb * 64 + ln));
      lds_char_t *pb[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int x = l32 + h;
        pb[h] = (lds_char_t *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + WBFRAGS * 64 + (rg * OUT_ROWS * 2 * BCOLS + x) * 2 + ((kh + (x >> 3)) & 1)));
      }
      half8 w[9], px[2][4];
      auto read_row = [&](int h) {
#pragma unroll
        for (int cc = 0; cc < 4; ++cc)
          px[h & 1][cc] = *(lds_frag)(pb[cc >> 1] + (h * 2 + (cc & 1)) * (BCOLS * 32));
      };
      read_row(0);
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) w[tap] = *(lds_frag)(wb + tap * KB * 1024);
#pragma unroll
      for (int h = 0; h < OUT_ROWS + 2; ++h) {
        if (h + 1 < OUT_ROWS + 2) read_row(h + 1);
#pragma unroll
        for (int i = h * nitems / 3; i < (h + 1) * nitems / 3 && i < nitems; ++i) item(i); // (in front of every store: see the wait behind the last step)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ts = 0; ts < 3; ++ts)
#pragma unroll
          for (int r = h - 2; r <= h; ++r) {
            if (r < 0 || r >= OUT_ROWS) continue;
#pragma unroll
            for (int b = 0; b < 2; ++b)
              out_acc(r, b) = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[(h - r) * 3 + ts], px[h & 1][b + ts], out_acc(r, b), 0, 0, 0);
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < OUT_ROWS; ++r) {
          if (r < h - 2 || r > h) continue;
          pin(out_acc(r, 0));
          pin(out_acc(r, 1));
        }
        if (FINAL && h >= 3) {
          finish_row(g, h - 3, out_acc(h - 3, 0), out_acc(h - 3, 1));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (FINAL) finish_row(g, OUT_ROWS - 1, out_acc(OUT_ROWS - 1, 0), out_acc(OUT_ROWS - 1, 1));
    };
    // The two waves of a SIMD add up at different times, one in front of the barrier and one behind it, each beside the other's matrix
    // instructions (the older wave is served first).
    if (wv < WAVES / 2) combine();
    STEP_WAIT(0);
    DNX_SYNC();
    if (wv >= WAVES / 2) combine();
    buf ^= 1;
    move_a(g, gn);
    if (NB == 1) move_b(g, gn);
    for (int j = 0; j < NB - 1; ++j) {
      step_b(buf, [&](int i) { item_b(buf ^ 1, g, j + 1, i); }, BITEMS, false);
      commit_b(buf ^ 1, j + 1);
      STEP_WAIT(0);
      DNX_SYNC();
      buf ^= 1;
    }
    if (NB > 1) move_b(g, gn);
    aim_out(g);
    step_b(buf, [&](int i) { item_a(buf ^ 1, gn, 0, i); }, AITEMS, true);
#else
    combine();
    aim_out(g);
#pragma unroll
    for (int r = 0; r < OUT_ROWS; ++r) finish_row(g, r, out_acc(r, 0), out_acc(r, 1));
#endif
    STEP_WAIT(NSTORES); // the next unit's first step has landed (before the end too: no wave leaves loads into LDS behind); the stores may still be on their way
    if (!more)
      break;
    DNX_SYNC();
    buf ^= 1;
    unit = next;
    g = gn;
  }
}
