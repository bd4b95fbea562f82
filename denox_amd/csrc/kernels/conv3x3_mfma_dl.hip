// conv3x3_mfma_dl.hip -- convolution of one plain source with weights and halos streamed straight into LDS (any filter with a tap in
// every phase, as the other kernels whose name says 3x3).
//
// The streaming kernel (conv3x3_mfma.hip) loads a step's weights and halo into registers, writes them to LDS and lets every wave wait at
// two barriers per step.  Here both go from memory into one of two LDS buffers (buffer_load ... lds) while the other is
// multiplied: no registers, no LDS writes, one barrier per step, and a persistent workgroup asks for the next tile's first step
// during the last step of the one before.  The loads are issued one by one between the matrix instructions (a memory instruction waits
// for room in the memory pipeline; all of a step's at once leave the matrix cores idle), a finished tile is stored in portions during
// the steps of the next.
//
// Mapping: as conv3x3_mfma.hip -- WAVES waves, each RPW rows of 32 pixels for all KT output channels of the workgroup.  The weights lie in
// memory in the order of the fragments (1 KiB each, lane by lane): their copy is linear and their reads are conflict-free.  A halo pixel
// takes CK / 8 slots of 16 bytes whose order is rotated by the pixel's column, so that 16 lanes reading the same channels of
// 16 consecutive pixels hit 16 different bank groups.
//
// What bounds it: the LDS-fed matrix rate of the part under load, loads and stores overlapping it only in part (128 -> 64 channels at
// 1920 x 1088: 257 us, 215 with neither loads nor stores, 800 MB of memory traffic are 156).  Tiles of 32 rows (RPW = 4, two blocks) halve the
// LDS reads per matrix instruction of tiles of 16, which need steps of 16 channels to fit; those fetch a pixel-major source's lines
// twice or more, so the large tiles pay on block-major sources (128 -> 64 257 us, pixel-major 313 and with 32-channel steps 277).
// (These are back to back.)  Microseconds a launch inside frames of the U-Nets by estimates, the other kernels before: 96 -> 96 at 480 x 272 27 and 23,
// 192 -> 192 there 79 and 68, 64 -> 96 pooled at 960 x 544 62 and 51, 128 -> 128 there 159 and 126, 128 -> 64 at 1920 x 1088 330 and 236.
//
// Strides.  Tap r of output row y reads input row y SY + r - PY = (y + d) SY + a: the taps fall into SY phases a, each of which is a
// convolution of stride 1 over every SY-th row with consecutive offsets d (columns alike).  A step is one phase and CK channels: its
// halo is staged as an image of its own, so a strided layer's matrix loop is that of a plain one -- consecutive lanes read consecutive
// slots, a pixel fragment serves all of its rows -- where the other kernels read every SY-th pixel of one large halo.  5 x 5, stride 2:
// phases of 9, 6, 6 and 4 taps.  Microseconds a launch, back to back, resident weights and one large halo before: 32 -> 64 at 1920 x 1080, pixel-major, 86 to 93
// and 65 to 76 (dense signed values in buffers that take turns: 91 and 81; a card at its power limit: 93 both), first pass on new buffers
// 126 and 105; 64 -> 64 at 960 x 544 (weights that do not stay in LDS): 38.  Of a 16-channel step each phase fetches 32 bytes of every
// 128: 78, so those suit block-major sources (121 and 65).
//
// Launch: persistent, NXCD * NKT * SLOTS workgroups; a unit of work is (tile, slice of KT output channels), each XCD has a contiguous band.
#include "conv_into_lds.h"

#ifndef KERNEL_NAME
#define KERNEL_NAME conv3x3_mfma_dl
#endif
static_assert(CB == 0 && !UPA && !PADA && !CROP && MF == 32 && PW == 0 && SY <= 2 && SX <= 2, "one plain source, strides up to 2");
static_assert(KR >= SY && KS >= SX, "a tap in every phase");
static_assert(CA % CK == 0 && (CK == 16 || CK == 32 || CK == 64), "whole steps of a power of two of vectors");
static_assert(KOUT % 8 == 0 && OPITCH % 8 == 0 && OVEC, "two 16-byte stores per pixel and block: the wait for a step's loads counts them");

// phase a of n taps with padding p and stride s: taps r = PH_FIRST, PH_FIRST + s, ...; the first one's offset d = (r - p - a) / s
#define PH_FIRST(a, p, s) ((((a) + (p)) % (s)))
#define PH_TAPS(a, n, p, s) (((n) - PH_FIRST(a, p, s) + (s) - 1) / (s))
#define PH_OFFSET(a, p, s) ((PH_FIRST(a, p, s) - (p) - (a)) / (s))
#define MAXTAPS(n, s) (((n) + (s) - 1) / (s))
#define PHASES (SY * SX)
#define NR MAXTAPS(KR, SY) // filter rows and columns of the largest phase
#define NC MAXTAPS(KS, SX)
#define HH (TH + NR - 1)   // staged halo of a phase (smaller phases leave its last row or column unused)
#define HW (TW + NC - 1)
#define G8 (CK / 8)                      // slots per halo pixel
#define WFRAGS (NR * NC * KB * (CK / 16)) // weight fragments of a step of the largest phase
#define HGROUPS ((HH * HW * G8 + 63) / 64) // halo loads of one wave's 64 lanes
#define BUF_SLOTS (64 * (WFRAGS + HGROUPS))
#define NVH ((HGROUPS + WAVES - 1) / WAVES)
#define DEFER (KB * RPW <= 4)            // the registers hold a converted tile beside the next one's accumulators
#define NSTORES (KB * OROWS * 2)        // store instructions of a wave per tile
#define ITEMS (NVH + (WFRAGS + WAVES - 1) / WAVES) // load instructions of a wave per step

extern "C" __global__ DNX_LAUNCH_BOUNDS(NT) void KERNEL_NAME(
    const _Float16 *__restrict__ A, _Float16 *__restrict__ OUT, const _Float16 *__restrict__ FILT,
#if HAS_BIAS
    const _Float16 *__restrict__ BIAS,
#endif
    PushConstants pc) {
  // One LDS object: beside a second one the compiler waits for every load into LDS in front of every LDS read.
  __shared__ uint4v sBuf[2 * BUF_SLOTS + KOUTP / 4];
  bias_t *const sBias = (bias_t *)(sBuf + 2 * BUF_SLOTS);
  const int tid = DNX_TID;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const OutBuf out = out_buffer(OUT, pc);
  const Sources srcs = make_sources(A, nullptr, pc);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(A), 0, (int)srcs.bytesA, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(FILT), 0, KOUTP * NTAPS * CA * 2, 0x00020000);
  const int W = (int)pc.IN_W, H = (int)pc.IN_H;

  const int tilesX = ((int)CONV_OUT_W(pc) + TW - 1) / TW, tilesY = ((int)CONV_OUT_H(pc) + TH - 1) / TH;
  const int units = tilesX * tilesY * NKT;
  const UnitBand band = unit_band(units);
  const int last = band.last;
  int unit = band.unit;
  if (unit >= last)
    return; // uniform for the workgroup
  const bool rev = (pc.FLAGS & 1u) != 0;
  struct Geo { int kt, x0, y0; };
  auto geometry = [&](int u) {
    Geo g;
    g.kt = u % NKT;
    int t = u / NKT;
    t = rev ? tilesX * tilesY - 1 - t : t;
    const int ty = t / tilesX;
    g.x0 = (t - ty * tilesX) * TW;
    g.y0 = ty * TH;
    return g;
  };

#if HAS_BIAS
  for (int i = tid; i < KOUTP; i += NT) sBias[i] = (float)BIAS[i];
#endif

  auto fresh_lane = [&]() { return fresh_lane_of(lane); };
  // Byte offsets of this lane's halo vectors in the source at channel 0, for one unit and phase; NO_LOAD outside the image (reads as
  // zero).  From one to the next they move by the same amount where both halos lie inside the image.
  unsigned hoff[NVH];
  auto group = [&](int i) { return wv + i * WAVES < HGROUPS ? wv + i * WAVES : HGROUPS - 1; }; // a wave without one left repeats the last
  auto row0 = [&](const Geo &g, int ph) { return (g.y0 + PH_OFFSET(ph / SX, PY, SY)) * SY + ph / SX; }; // source position of the halo's first pixel
  auto col0 = [&](const Geo &g, int ph) { return (g.x0 + PH_OFFSET(ph % SX, PX, SX)) * SX + ph % SX; };
  auto inside = [&](int y, int x) { return (y >= 0) & (y + (HH - 1) * SY < H) & (x >= 0) & (x + (HW - 1) * SX < W); };
  auto aim = [&](const Geo &g, int ph) {
    const unsigned ln = (unsigned)fresh_lane();
#pragma unroll
    for (int i = 0; i < NVH; ++i) {
      const unsigned slot = (unsigned)group(i) * 64 + ln, pix = slot / G8;
      unsigned hy = pix / HW;
      const unsigned hx = pix - hy * HW, grp = (slot - hx / (16 / G8)) & (G8 - 1); // the channel group that belongs into this slot
      hy = hy < HH ? hy : HH - 1;                                                  // past the halo: its last row again
      const int y = row0(g, ph) + (int)hy * SY, x = col0(g, ph) + (int)hx * SX;
      const unsigned p = (unsigned)(y * W + x);
      hoff[i] = (((unsigned)y < (unsigned)H) & ((unsigned)x < (unsigned)W)) ? (LAYIN ? p * 16u + grp * srcs.planeA : p * (CA * 2u) + grp * 16u) : NO_LOAD;
    }
  };
  auto move = [&](const Geo &from, int fph, const Geo &to, int tph) {
    const int y = row0(from, fph), x = col0(from, fph), ty = row0(to, tph), tx = col0(to, tph);
    if (inside(y, x) & inside(ty, tx)) {
      const unsigned d = (unsigned)((ty - y) * W + tx - x) * (LAYIN ? 16u : CA * 2u);
#pragma unroll
      for (int i = 0; i < NVH; ++i) hoff[i] += d;
    } else
      aim(to, tph);
  };
  // first weight fragment of (phase, step of channels) inside a slice; a phase's steps follow one another
  auto first_frag = [](int ph, int k) constexpr {
    int f = 0;
    for (int q = 0; q < ph; ++q) f += PH_TAPS(q / SX, KR, PY, SY) * PH_TAPS(q % SX, KS, PX, SX) * KB * (CA / 16);
    return f + k * PH_TAPS(ph / SX, KR, PY, SY) * PH_TAPS(ph % SX, KS, PX, SX) * KB * (CK / 16);
  };
  auto item = [&](int buf, int kt, const int ph, int k, int i) { // item i of the loads of the step of phase ph with the channels from k * CK on
    if (i < NVH) {
      const unsigned off = hoff[i] + (LAYIN ? (unsigned)(k * G8) * srcs.planeA : (unsigned)(k * CK * 2));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t *)(sBuf + buf * BUF_SLOTS + (WFRAGS + group(i)) * 64), 16, hoff[i] != NO_LOAD ? off : NO_LOAD, 0, 0, LOAD_AUX);
    } else {
      const int n = PH_TAPS(ph / SX, KR, PY, SY) * PH_TAPS(ph % SX, KS, PX, SX) * KB * (CK / 16);
      const int q = wv + (i - NVH) * WAVES, f = q < n ? q : n - 1;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void_t *)(sBuf + buf * BUF_SLOTS + f * 64), 16, fresh_lane() * 16, (kt * (NTAPS * KB * (CA / 16)) + first_frag(ph, k) + f) * 1024, 0, 0);
    }
  };

  Acc acc;
  auto step = [&](int buf, const int ph, auto load) { // load(i): item i of the loads for the next step
    typedef __attribute__((address_space(3))) const char lds_char_t;
    typedef __attribute__((address_space(3))) const half8 *lds_frag;
    constexpr int KSN = CK / 16;
    const int nr = PH_TAPS(ph / SX, KR, PY, SY), nc = PH_TAPS(ph % SX, KS, PX, SX), NG = nc * KSN, UNITS = nr * NG;
    const int ln = fresh_lane(), l32 = ln & 31, kh = ln >> 5;
    lds_char_t *wb = (lds_char_t *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + ln)), *pb[NC][KSN];
#pragma unroll
    for (int s = 0; s < NC; ++s)
#pragma unroll
      for (int ks = 0; ks < KSN; ++ks) {
        const int x = l32 + s;
        pb[s][ks] = (lds_char_t *)lds_opaque((const _Float16 *)(sBuf + buf * BUF_SLOTS + WFRAGS * 64 + (wv * RPW * HW + x) * G8 + ((2 * ks + kh + x / (16 / G8)) & (G8 - 1))));
      }
    // A group is a filter column s of one 16-channel slice: RPW + nr - 1 pixel fragments; its units (one per filter row) read KB weight
    // fragments each and feed KB * RPW matrix instructions.  Weights are read one or two units ahead, a group's pixels during the group before.
    constexpr int WR = KB <= 2 ? 3 : 2; // weight sets: the one in use and those under way
    half8 px[2][RPW + NR - 1], w[WR][KB];
    auto read_w = [&](int u) {
      const int gr = u / nr, r = u % nr, s = gr / KSN, ks = gr % KSN;
#pragma unroll
      for (int b = 0; b < KB; ++b) w[u % WR][b] = *(lds_frag)(wb + (((r * nc + s) * KB + b) * KSN + ks) * 1024);
    };
    auto read_p = [&](int gr, int t) {
      const int s = gr / KSN, ks = gr % KSN;
      px[gr & 1][t] = *(lds_frag)(pb[s][ks] + t * (HW * G8 * 16));
    };
#pragma unroll
    for (int t = 0; t < RPW + nr - 1; ++t) read_p(0, t);
#pragma unroll
    for (int u = 0; u < WR - 1; ++u) read_w(u);
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int gr = u / nr, r = u % nr;
      if (u + WR - 1 < UNITS) read_w(u + WR - 1);
      if (gr + 1 < NG) {
#pragma unroll
        for (int t = r * (RPW + nr - 1) / nr; t < (r + 1) * (RPW + nr - 1) / nr; ++t) read_p(gr + 1, t);
      }
#pragma unroll
      for (int i = u * ITEMS / UNITS; i < (u + 1) * ITEMS / UNITS; ++i) load(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int j = 0; j < RPW; ++j) acc.v[b][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u % WR][b], px[gr & 1][j + r], acc.v[b][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int j = 0; j < RPW; ++j) pin(acc.v[b][j]);
  };

  int buf = 0;
  Geo g = geometry(unit);
#if DEFER
  Geo gd = g;
#endif
  aim(g, 0);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) item(0, g.kt, 0, 0, i);
  STEP_WAIT(0);
  DNX_SYNC();
#if DEFER
  // The finished tile, converted; its stores go out in NPARTS portions in front of the next tile's steps (whole output rows: a line filled
  // in two portions far apart in time is written to memory twice).
  constexpr int NPARTS = PHASES * NCHUNK < OROWS ? PHASES * NCHUNK : OROWS;
  Packed done;
  bool pend = false;
  auto store_part = [&](int part) {
#pragma unroll
    for (int p = 0; p < NPARTS; ++p)
      if (part == p) store_packed(done, out, gd.y0, gd.x0, gd.kt, wv, fresh_lane(), pc, p, NPARTS);
  };
#endif
  for (;;) {
    const int next = unit + NKT * SLOTS;
    const bool more = next < last;
    const Geo gn = geometry(more ? next : unit); // (behind the last unit its own first step is loaded once more and not used)
#if HAS_BIAS
    const int hsel = fresh_lane() >> 5;
#endif
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int j = 0; j < RPW; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#if HAS_BIAS
          acc.v[b][j][i] = sBias[g.kt * KT + b * 32 + hsel * 16 + i];
#else
          acc.v[b][j][i] = 0.0f;
#endif
#pragma unroll
    for (int ph = 0; ph < PHASES; ++ph) {
      for (int k = 0; k < NCHUNK - 1; ++k) {
#if DEFER
        if (pend & (ph * NCHUNK + k < NPARTS)) store_part(ph * NCHUNK + k);
#endif
        step(buf, ph, [&](int i) { item(buf ^ 1, g.kt, ph, k + 1, i); });
        STEP_WAIT(0); // the next step's loads; the stores in front of them have had the step's matrix work to complete
        DNX_SYNC();
        buf ^= 1;
      }
#if DEFER
      if (pend & (ph * NCHUNK + NCHUNK - 1 < NPARTS)) store_part(ph * NCHUNK + NCHUNK - 1);
#endif
      if (ph < PHASES - 1) {
        move(g, ph, g, ph + 1);
        step(buf, ph, [&](int i) { item(buf ^ 1, g.kt, ph + 1, 0, i); });
        STEP_WAIT(0);
        DNX_SYNC();
        buf ^= 1;
      }
    }
    move(g, PHASES - 1, gn, 0);
    step(buf, PHASES - 1, [&](int i) { item(buf ^ 1, gn.kt, 0, 0, i); });
#if DEFER
    pack_tile(acc, done);
    STEP_WAIT(0);
#else
    store_tile(acc, out, g.y0, g.x0, g.kt, wv, fresh_lane(), pc);
    STEP_WAIT(NSTORES); // the next unit's first step has landed; the stores behind its loads may still be on their way
#endif
    DNX_SYNC();
    buf ^= 1;
#if DEFER
    gd = g;
    pend = true;
#endif
    if (!more)
      break;
    unit = next;
    g = gn;
  }
#if DEFER
#pragma unroll
  for (int p = 0; p < NPARTS; ++p) store_part(p);
#endif
}
