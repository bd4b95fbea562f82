// Why an estimate per configuration: a bytes-and-FLOP bound is the same for every configuration of a layer, so a schedule
// without a timing table used one configuration (the first of the table) for every layer.  A frame of the 1920 x 1080 U-Net took
// 690 us so, 592 with estimates and 578 with a measured table (none of them with folded weights); at 251 x 187 185, 96 and 95; with
// doubled widths at 1917 x 1077 2530, 2037 and 2000.  With the kernels that load straight into LDS, estimates and table: 496 and 510, 96 and 94,
// 1390 and 1375 (denox_amd/conv_estimates.py).
//
// The form is the kernels' own: what the busiest compute unit does -- matrix instructions, halo staging and its memory round
// trips, weight slices, stores -- against what the whole launch moves through memory; the parts that overlap combine as the root of
// their squares.  The constants are fitted (least squares on the logarithm, near-best candidates weighted up) to the
// latencies of 53 000 candidate dispatches measured on one MI355X, as Db::populate, Db::bench and the table's CSV give them: every
// candidate of the U-Net at eight extents from 180 x 108 to 3840 x 2160 and at two widths, of the small U-Net, and of 16 single
// convolutions (1 x 1 to 5 x 5, stride 1 and 2, 3 to 256 channels) at five extents.  denox_amd/conv_estimates.py measures how far
// they are from a GPU, per configuration, and what a changed or new kernel's entry in kFactor should be.  On layers that are not among
// those of the fit the measured time is 1.07 times the estimate in the median, 0.99 - 1.18 for half of the candidates; the schedules picked take
// 0.97 - 1.07 times as long as measured ones.  A timing table, where there is one, still decides.
#include "conv_cost.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>

namespace denox::compiler {

namespace {

struct KernelFit {
  float matrix;  // time of a computing wave's matrix instructions over their issue time at 2 GHz
  float step;    // us per LDS step: the round trip of a halo load that nothing hides
  float vector;  // us per 16-byte vector a staging thread moves in a step
  float barrier; // us per step that nothing overlaps
  float spill;   // growth of matrix and staging time once the registers a wave needs exceed 55 % of its share
  float crowded; // ... and beyond 80 %
};
const KernelFit kFit[] = {
    /* Streamed   */ {0.824f, 0.0337f, 0.0865f, 0.0209f, 0.441f, 0.08f},
    /* Resident   */ {1.467f, 0.0965f, 0.1360f, 0.0246f, 0.924f, 3.06f},
    /* Staged     */ {1.191f, 0.0288f, 0.0759f, 0.0096f, 0.539f, 5.74f},
    /* StagedTile */ {1.373f, 0.0333f, 0.0806f, 0.0252f, 0.510f, 5.00f},
    /* TwoPhase   */ {1.634f, 0.0598f, 0.2382f, 0.0203f, 3.940f, 3.29f},
    /* Fold       */ {1.388f, 0.5124f, 0.1078f, 0.0299f, 0.000f, 0.00f},
    /* FoldStaged */ {2.886f, 0.2374f, 0.0641f, 0.0286f, 0.000f, 0.00f},
    /* Pair       */ {1.122f, 0.1087f, 0.0748f, 0.0273f, 0.000f, 0.00f},
    /* PairStaged */ {1.296f, 0.4625f, 0.0629f, 0.0305f, 0.000f, 0.00f},
};
// what is left to the configuration itself, as a factor
const struct { const char *name; float factor; } kFactor[] = {
    {"c4r2k16m", 0.81f}, {"c4r2k16n", 0.85f}, {"c4r2k32n", 0.80f}, {"d4r2k64", 0.88f}, {"e8r1", 1.00f}, {"e8r2", 1.00f}, {"f4r1", 0.78f}, {"f4r2", 0.76f}, {"f8r1", 0.84f},
    {"g4r1", 0.57f}, {"g4r1k32", 0.58f}, {"g4r1k32n", 0.54f}, {"g4r1n", 0.55f}, {"g4r1p", 0.52f}, {"h4r2", 0.57f}, {"h4r2k32n", 0.53f},
    {"h4r2k32p", 0.53f}, {"h4r2n", 0.53f}, {"h4r2p", 0.51f}, {"l8k16", 1.00f}, {"l8k32", 1.00f}, {"m2r1k32x1n", 0.79f}, {"m4r1k32x2", 1.01f}, {"m4r1kfx1n", 1.01f}, {"m4r1kfx2", 1.24f},
    {"m4r2k32x1", 1.01f}, {"m4r2k32x1n", 1.11f}, {"m4r2k32x2", 1.09f}, {"m4r2k32x2n", 1.18f}, {"m4r2k64x2", 1.11f}, {"m4r2kfx1", 1.14f},
    {"m4r2kfx1n", 1.10f}, {"m4r4k32x1", 1.09f}, {"m8r2k32x2", 1.19f}, {"p16r1k16", 1.05f}, {"p16r1k32", 0.95f}, {"p16r2k16", 0.98f},
    {"p4r1k32", 0.93f}, {"p4r1k32n", 0.84f}, {"p4r2k32", 0.96f}, {"p4r2k32n", 0.92f}, {"p4r4k16", 0.91f}, {"p4r4k32", 0.84f}, {"p8r1k16", 0.99f},
    {"p8r1k32", 0.97f}, {"p8r2k16", 0.97f}, {"p8r2k32", 0.94f}, {"p8r2k32s", 0.87f}, {"p8r4k16", 1.02f}, {"q4r2k32x1n", 0.93f}, {"q4r2k32x2", 0.86f},
    {"q8r1k32x2", 1.02f}, {"q8r2k32x1", 0.97f}, {"q8r2k32x2", 0.98f}, {"r4r1k16n", 0.87f}, {"r4r2k16", 0.89f}, {"r4r2k16n", 0.85f},
    {"r4r2k32n", 0.85f}, {"r8r1k16n", 0.90f}, {"s12r1k16", 1.03f}, {"s8r2k16", 0.95f}, {"s8r2k16s", 0.99f}, {"s8r2k32s", 1.37f}, {"t16r1k16", 1.01f},
    {"t16r1k32", 0.95f}, {"t16r2k16", 1.06f}, {"t4r2k32", 0.86f}, {"t8r1k16", 0.91f}, {"t8r2k16", 0.85f}, {"t8r2k32", 0.81f}, {"t8r4k16", 0.89f},
    {"u16r1k32x2", 1.01f}, {"u4r2k32", 0.77f}, {"u8r2k32x2", 0.75f}, {"v4r2k16", 0.85f}, {"v4r2k64", 0.80f}, {"w2r1k16n", 0.82f}, {"w2r2k16n", 0.98f},
    {"w2r2k32", 0.89f}, {"w2r2k32n", 0.86f}, {"w2r2kfn", 1.09f}, {"w4r1k16", 1.01f}, {"w4r1k32", 0.95f}, {"w4r1k32n", 1.03f}, {"w4r1kfm", 0.99f},
    {"w4r1kfn", 1.00f}, {"w4r1khn", 1.04f}, {"w4r2k16", 1.25f}, {"w4r2k16s", 1.15f}, {"w4r2k32", 1.13f}, {"w4r2k32n", 1.19f}, {"w4r2k32s", 1.06f},
    {"w4r2k64", 1.11f}, {"w4r2kfn", 1.22f}, {"w4r2khn", 1.36f}, {"w4r4k16", 1.41f}, {"w4r4k32", 1.24f}, {"w8r1k16", 1.25f}, {"w8r2k16", 1.40f},
    {"w8r2k32", 1.30f}, {"x4r2k16", 1.33f}, {"x4r2k32", 1.07f}, {"x4r4k16", 1.22f}, {"x8r2k16", 1.12f}, {"y4r2k32", 0.81f}, {"z4r2k64", 0.82f},
};

float factorOf(const char *name) {
  for (const auto &f : kFactor) if (std::strcmp(f.name, name) == 0) return f.factor;
  return 1.2f; // a configuration without a measurement: behind those that have one
}

double cdiv(double a, double b) { return std::ceil(a / b); }

// Kernels that share the products of an upsampled source (conv3x3_upshare.hip), one form for all of its configurations: a workgroup's units of
// work one after the other -- the matrix instructions of the two waves of a SIMD at 2 GHz, 0.5 us per step (its barrier, the first
// fragments behind it, loads that arrive late), the result's way out -- against the launch's memory traffic.  Fitted to 614 launches
// of 12 layers (32 to 224 upsampled, 0 to 128 other channels, 16 to 224 outputs) at 96 x 64 to 1920 x 1088 in all layouts, back to back: measured
// over estimated, without the start, 0.89 - 1.16 for nine of ten, median 1.00.
// The start is what a frame adds to a launch that the same kernel did not precede (64 + 9 -> 64 at 256 x 192: 12.6 us inside the U-Net, 11.0
// back to back).  Whole frames of 37 networks and extents (the U-Net and twice its width at 96 x 96 to 1920 x 1080, the small U-Net), schedules by
// estimates with starts of 0 to 2.2: 1.2 to 2.0 choose the same but for two frames (1 % either way), without one the frames at 512 x 512
// and 640 x 360 are 2 % slower, with 2.2 the one at 1280 x 720.
constexpr double kShareStartUs = 1.6;
double share_cost_us(const ConvCost &c, double ow, double oh, double bytes, unsigned xcds) {
  const double cap = cdiv(c.CA, 16) * 16, cbp = cdiv(c.CB, 16) * 16, rows = c.waves / (c.KT / 32) * c.rpw, slices = cdiv(cdiv(c.K, 32) * 32, c.KT);
  const double units = cdiv(ow, 62) * cdiv(oh + 1, 2 * rows) * slices, rounds = cdiv(cdiv(units, xcds), c.slots * slices);
  const double mfma = cap / 16 * (9 * c.rpw + 3) + cbp / 16 * 36 * c.rpw, steps = cap / c.ck + cbp / 16, tileKB = 2 * rows * 62 * c.KT * 2 / 1024;
  const double work = rounds * (1.03 * mfma * 2 * 32 / 2000 + 0.506 * steps + 0.0142 * tileKB), memory = bytes / 5.183e6;
  return kLaunchUs + factorOf(c.config) * (kShareStartUs + std::sqrt(work * work + memory * memory));
}

// Streaming kernels whose weights and halos go straight into LDS (conv3x3_mfma_dl.hip), one form as well: matrix instructions, LDS reads and
// loads of a unit of work overlap, a pixel-major result leaves the lanes in short pieces, and steps of 16 channels fetch a
// pixel-major source's lines more than once.  Fitted to 1632 launches of 15 layers (16 to 256 channels, with and without a pool) at
// 96 x 64 to 1920 x 1088 in all layouts: measured over estimated 0.88 - 1.14 for nine of ten, median 1.00.  (5 x 5 with stride 2, 32 and 64 -> 64 channels at
// 480 x 270 to 1920 x 1080: 0.92 - 1.27; the price of short pieces is four times as high there, every pixel lies in a phase of its own.)
// The figures are back to back and without the start, which is fitted as above: with none the small U-Net takes the kernel for 16 -> 32 channels
// and is slower than without it (760 x 448: 44.5 us a frame against 43.3, 960 x 540: 49.8 and 48.8), with 0.5 it does not, and seven frames
// of the U-Nets gain 0.1 - 2 % (one loses 0.7); 0.3 leaves half of that, 0.8 and more lose in three.
constexpr double kStreamedLdsStartUs = 0.5;
double streamed_lds_cost_us(const ConvCost &c, double ow, double oh, double bytesRead, double bytesWritten, unsigned xcds) {
  const double kb = c.KT / 32, rows = 8.0 * c.rpw, slices = cdiv(cdiv(c.K, 32) * 32, c.KT), groups = c.CA / 16.0;
  const double rounds = cdiv(cdiv(cdiv(ow, 32) * cdiv(oh, rows) * slices, xcds), c.slots * slices);
  // (a strided layer's taps fall into phases that each stage a halo of their own)
  const double taps = c.R * c.S, phases = c.SY * c.SX, nr = cdiv(c.R, c.SY), nc = cdiv(c.S, c.SX);
  const double matrix = 0.865 * taps * groups * kb * c.rpw * 2 * 32 / 2000, lds = 3.235e-3 * 8 * groups * (c.S * c.SY * (c.rpw - 1 + c.R / static_cast<double>(c.SY)) + taps * kb);
  const double haloKB = phases * (rows + nr - 1) * (32 + nc - 1) * c.CA * 2 / 1024, loads = 2.035e-2 * (haloKB + taps * c.KT * c.CA * 2 / 1024);
  const double stored = bytesWritten / std::max(1.0, 2 * ow * oh * c.K), tileKB = rows * 32 * c.KT * 2 / 1024 * stored; // (a pooled tile is a quarter)
  const double unit = std::sqrt(matrix * matrix + lds * lds + loads * loads) + 0.0371 * phases * c.CA / c.ck + (c.ck == 16 && !c.blockedIn ? (phases > 1 ? 0.0144 : 0.0036) * haloKB : 0) + (c.blockedOut ? 0 : 0.0141 * tileKB);
  const double memory = (bytesRead + bytesWritten) / 5.712e6;
  return kLaunchUs + factorOf(c.config) * (kStreamedLdsStartUs + std::pow(std::pow(rounds * unit, 1.2) + std::pow(memory, 1.2), 1 / 1.2));
}

} // namespace

double conv_cost_us(const ConvCost &c, uint64_t outWidth, uint64_t outHeight, double bytesRead, double bytesWritten, unsigned xcds, unsigned cus, unsigned ldsBytes) {
  const double ow = static_cast<double>(outWidth), oh = static_cast<double>(outHeight);
  if (c.kernel == ConvKernel::Share) return share_cost_us(c, ow, oh, bytesRead + bytesWritten, xcds);
  if (c.kernel == ConvKernel::StreamedLds) return streamed_lds_cost_us(c, ow, oh, bytesRead, bytesWritten, xcds);
  const KernelFit &f = kFit[static_cast<int>(c.kernel)];
  const double W = c.waves, RPW = c.rpw, KT = c.KT, CK = c.ck, stagers = (c.pw ? c.pw : c.waves) * 64.0, wavesPerSimd = std::max(1.0, W / 4.0);
  const bool pair = c.kernel == ConvKernel::Pair || c.kernel == ConvKernel::PairStaged, fold = c.kernel == ConvKernel::Fold || c.kernel == ConvKernel::FoldStaged;
  // per compute unit: rounds of tiles, LDS steps, matrix cycles of a wave, LDS reads; per step: halo bytes; per launch: resident weights
  double rounds, steps, cycles, ldsReads, halo, haloSteps, resident = 0, tileBytes, overfetch, weightStep = 0, over = 0, groups = 0, rereads = 1;
  if (pair) {
    const double cpad = cdiv(c.CA + c.CB, 16) * 16, ck = std::min(CK, cpad), chunks = cdiv(cpad, ck), rowsPerStep = W * RPW, strips = cdiv(ow, 30);
    const double wanted = std::max(1.0, std::floor(cus / strips));
    const double rows = cdiv(cdiv(oh, wanted) + 2, rowsPerStep) * rowsPerStep, segments = cdiv(oh, rows - 2); // as conv3x3_pair.hip cuts the image
    rounds = (rows / rowsPerStep + 1) * cdiv(strips * segments, cus);
    const double mfma = 9 * (cpad / 16) * RPW + (c.tapm ? RPW * 6 : RPW * 18);
    steps = haloSteps = rounds * chunks;
    halo = (rowsPerStep + 2) * 34 * ck * 2;
    resident = 9 * 32 * cpad * 2;
    tileBytes = rowsPerStep * 32 * 32 * 2;
    overfetch = 34 * (rowsPerStep + 2) / (30 * rowsPerStep);
    cycles = mfma * 32 * wavesPerSimd * rounds;
    ldsReads = rounds * W * (mfma + 9 * (cpad / 16));
  } else if (fold) {
    const bool staged = c.kernel == ConvKernel::FoldStaged;
    const double cap = cdiv(c.CA, 16) * 16, cbp = c.CB ? cdiv(c.CB, 16) * 16 : 0, rows = W / c.ksplit * RPW, kbw = KT / 32 / c.ksplit;
    const double slices = cdiv(cdiv(c.K, 32) * 32, KT), classes = staged ? 2 : 4, cols = staged ? 2 : 1;
    const double tiles = cdiv(cdiv(ow, 2), 32) * cdiv(cdiv(oh, 2), rows), walkers = std::max(1.0, std::floor(cus / (xcds * classes * slices))) * xcds;
    rounds = cdiv(tiles, walkers);
    const double mfma = (4 * cap / 16 + 9 * cbp / 16) * kbw * RPW * cols, stepsA = staged ? std::floor(cap / c.cka) : 1, perTile = stepsA + (c.CB ? 1 : 0);
    steps = haloSteps = rounds * perTile;
    halo = ((rows + 1) * 34 * cap + (2 * rows + 1) * 66 * cbp) * 2 / perTile;
    resident = (4 * cols * cap + 9 * cbp) * KT * 2;
    tileBytes = rows * 32 * cols * KT * 2;
    overfetch = 1.15 * classes * slices;
    cycles = mfma * 32 * wavesPerSimd * rounds;
    ldsReads = rounds * W * mfma * (1 + 1 / RPW);
  } else {
    const double kstep = c.mf == 32 ? 16 : 32, cpad = cdiv(c.CA + c.CB, kstep) * kstep, chunks = cdiv(cpad, CK), taps = c.R * c.S, xb = c.mf == 32 ? 1 : c.xb;
    const double tw = c.mf == 32 ? 32 : 16 * xb, th = W * RPW, kb = KT / c.mf, slices = cdiv(cdiv(c.K, c.mf) * c.mf, KT), tiles = cdiv(ow, tw) * cdiv(oh, th);
    const double haloPix = ((th - 1) * c.SY + c.R) * ((tw - 1) * c.SX + c.S), mfma = cpad / kstep * taps * kb * RPW * xb;
    const double shared = c.SY > 1 || c.R == 1 ? 1.0 : (RPW + c.R - 1) / (RPW * c.R); // pixel fragments reused across vertical taps
    const double accRegs = c.mf == 32 ? kb * RPW * 16 : kb * RPW * xb * 4, haloRegs = 4 * cdiv(std::floor(haloPix * CK * 2 / 16), stagers);
    const double fragRegs = c.swp ? 8 * kb * c.R + 8 * (RPW + 2) : 4 * kb + 4 * ((RPW - 1) * c.SY + c.R) * xb;
    halo = haloPix * CK * 2;
    tileBytes = th * tw * KT * 2;
    overfetch = haloPix / (th * tw * c.SY * c.SX);
    double regs;
    if (c.kernel == ConvKernel::Streamed) {
      const double weights = taps * KT * CK, lds = (haloPix * (c.hrot ? CK : CK + 8) + taps * KT * (CK + 8)) * 2 + KT * 4;
      const double weightRegs = 4 * cdiv(std::floor(weights / 8), W * 64);
      const double perWave = std::min(512.0, accRegs + haloRegs + weightRegs + 64), simdWaves = std::floor(512 / perWave) * 4;
      const double resident_ = std::max(1.0, std::min({std::floor(ldsBytes / lds), std::floor(simdWaves / W), 8.0})); // workgroups of one compute unit at a time
      rounds = cdiv(tiles * slices, cus);
      groups = rounds;
      rereads = 1 + 0.530 * (slices - 1); // every slice of output channels walks the image again
      steps = chunks * cdiv(rounds, std::min(resident_, rounds));
      haloSteps = chunks * rounds;
      weightStep = weights * 2;
      regs = accRegs + haloRegs + weightRegs + fragRegs;
    } else {
      rounds = cdiv(tiles, static_cast<double>(c.slots) * xcds);
      rereads = 1 + 0.628 * (slices - 1);
      steps = haloSteps = rounds * chunks;
      resident = taps * KT * cpad * 2;
      regs = std::max(accRegs + fragRegs, c.pw ? 2 * haloRegs : 0) + (c.pw ? 0 : 2 * haloRegs);
    }
    over = regs / std::min(256.0, 512.0 / cdiv(W + c.pw, 4));
    cycles = mfma * (c.mf == 32 ? 32 : 16) * wavesPerSimd * rounds;
    ldsReads = cpad / kstep * taps * (kb + RPW * xb * shared) * W * rounds;
  }
  const double spill = std::exp(f.spill * std::max(0.0, over - 0.55) + f.crowded * std::max(0.0, over - 0.8));
  const double matrix = cycles / 2000.0 * f.matrix * (c.mf == 16 ? 1.325 : 1) * (c.swp ? 1.008 : 1) * spill;
  const double lds = ldsReads * 0.556e-3;
  const bool ragged = c.CA % 8 || c.CB % 8;
  const double staging = steps * (f.step + halo / 16 / stagers * f.vector * (ragged ? 2.373 : 1)) * spill * (c.blockedIn ? 0.862 : 1);
  const double weights = haloSteps * weightStep * 31.095e-6;
  // 8-byte pieces where a 16-channel block has no partner; a block-major result leaves the lanes in longer runs
  const double stores = rounds * tileBytes * 2.149e-5 * (c.blockedOut ? 0.659 : 1) * (c.ntStore ? 0.749 : 1) * (c.mf == 16 && (c.KT / 16) % 2 ? 3.851 : 1);
  const double memory = (bytesRead * std::min(overfetch, 4.0) * rereads + bytesWritten) / 5.661e6;
  const double moved = staging + weights + stores;
  const double start = (resident > 0 ? 0.795 + resident * 1.064e-5 : 0) + (c.weightsInRegisters ? 1.154 : 0);
  // Fewer than 8 channels are read in pieces, which the persistent kernels' long-lived loaders feel more than the streaming ones'
  // (medians of measured over estimated time above 10 us: 1.3 and, with staging waves, 1.55 against 0.97).
  const bool persistent = !pair && !fold && c.kernel != ConvKernel::Streamed;
  const double few = persistent && c.CA < 8 ? (c.pw ? 1.55 : 1.3) : 1;
  return kLaunchUs + start + few * factorOf(c.config) * (std::sqrt(matrix * matrix + memory * memory + moved * moved + lds * lds) + steps * f.barrier + groups * 0.0139);
}

} // namespace denox::compiler
