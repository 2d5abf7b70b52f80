// The deep convolution kernel (deep.h) as the other launch code sees it: which launches it takes, on which tile.
#pragma once

#include "conv_common.h"

namespace fim {

constexpr int DEEP_TAPS = 25;  // filter taps the kernel's per-row validity masks hold (with the K tail's taps, below 32)

// 32-channel blocks of an MX input: the kernel keeps their scales in LDS
constexpr int DEEP_CBLOCKS = 256;

// The tile of a deep launch: WN wavefronts across 64-channel columns (tile width 64 WN), mbw blocks of rows per
// wavefront; rag: Cin or Cout not a multiple of 16. wn 0: the deep kernel does not take the launch.
struct DeepPlan {
  int wn, mbw;
  bool rag, two;  // two: 128 x 128 tiles, two workgroups per CU
};

int launch_deep_int8(const ConvArgs& a, DeepPlan p, hipStream_t stream);
int launch_deep_mx(const ConvArgs& a, DeepPlan p, hipStream_t stream);

constexpr int DEEP_BR = 32;  // rows per block
constexpr int deep_min_mbw(int wn) { return wn == 4 ? 4 : 2; }
constexpr int deep_max_mbw(int wn) { return wn == 4 ? 8 : 5; }

// LDS stages of a bm x bn tile: three where they fit in the 160 KB beside the epilogue operands, tap offsets and MX
// scales.
constexpr int deep_stages(bool mx, int bm, int bn) {
  return 3 * (bm + bn) * KC + (mx ? 3 * bn * 4 + 128 + DEEP_CBLOCKS + 16 : 2 * bn * 4 + 128 + 24) <= 163840 ? 3 : 2;
}

DeepPlan deep_plan(const ConvArgs& a, int kind);

}  // namespace fim
