// Launches of the deep convolution kernel, one translation unit per operand format.
#pragma once

#include "deep.h"
#include "deep_plan.h"

namespace fim {

inline void magic_divisor(int d, uint32_t& mul, int& shift) {
  if (d <= 1) {
    mul = 0;
    shift = -1;
    return;
  }
  int s = 1;
  while ((1LL << s) < d) ++s;
  mul = (uint32_t)((((uint64_t)1 << (31 + s)) + d - 1) / d);
  shift = s - 1;
}

inline DeepArgs deep_args(const ConvArgs& a, int bm, int bn) {
  DeepArgs d;
  d.c = a;
  d.c.n_tiles = (int)cdiv((int64_t)a.Cout, bn);
  d.c.m_tiles = (int)cdiv((int64_t)a.M, bm);
  magic_divisor(a.Wo, d.wo_mul, d.wo_shift);
  magic_divisor(a.Ho, d.ho_mul, d.ho_shift);
  d.segs = (a.Cin + 15) / 16;
  d.adv_tap = 8 / d.segs;
  d.adv_seg = 8 % d.segs;
  d.nk = (int)cdiv((int64_t)a.kh * a.kw * d.segs, 8);
  return d;
}

template <int KIND, int OUT, int WN, int MBW, bool RAG, bool TWO = false>
inline int launch_deep_tile(const ConvArgs& a, hipStream_t stream) {
  const DeepArgs d = deep_args(a, (4 / WN) * MBW * DEEP_BR, WN * 64);
  const dim3 grid((unsigned)(cdiv((int64_t)d.c.n_tiles * d.c.m_tiles, 8) * 8));
  conv_deep_kernel<KIND, OUT, WN, MBW, RAG, TWO><<<grid, dim3(256), 0, stream>>>(d);
  return launch_status();
}

}  // namespace fim
