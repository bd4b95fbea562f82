// Estimated run time of a convolution dispatch, for schedules that are selected without a timing table.
#pragma once
#include "../common/sym.hpp"
#include <cstdint>

namespace denox::compiler {

enum class ConvKernel : uint8_t { Streamed, Resident, Staged, StagedTile, TwoPhase, Fold, FoldStaged, Pair, PairStaged, Share, StreamedLds };

// What the estimate needs to know about a dispatch; the extents are those of the convolution's result before a fused pool or crop.
struct ConvCost {
  bool valid = false;
  ConvKernel kernel = ConvKernel::Streamed;
  const char *config = "";      // name in the configuration tables
  unsigned waves = 0, pw = 0, rpw = 0, ck = 0, mf = 32, xb = 1, KT = 0, K = 0, CA = 0, CB = 0;
  unsigned R = 3, S = 3, SY = 1, SX = 1;
  unsigned slots = 0;           // workgroups per XCD and slice of output channels (persistent kernels)
  unsigned cka = 0, ksplit = 1; // upsample-folding kernels: channels of the upsampled source per step; waves sharing a row
  bool hrot = false, swp = false, ntStore = false, blockedIn = false, blockedOut = false, tapm = false, weightsInRegisters = false;
  Sym outWidth, outHeight;
};

// Microseconds on an MI355X, launch included.
double conv_cost_us(const ConvCost &c, uint64_t outWidth, uint64_t outHeight, double bytesRead, double bytesWritten, unsigned xcds, unsigned computeUnits, unsigned ldsBytes);

// what any dispatch costs before its work: the launch, as a pair of events around it sees it
constexpr double kLaunchUs = 5.56;

} // namespace denox::compiler
