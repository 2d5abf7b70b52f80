// Which launches the deep convolution kernel takes, and on which tile.
#include "deep_plan.h"

namespace fim {

// Estimated clocks of one K step of a bm x bn tile: the MFMAs (bm bn / 32 clocks) at 78% of their issue rate, the LDS
// traffic (operand reads and staging) at 90%, and the loads into LDS at 47 bytes per clock, which with two stages have to
// land within the step. Measured (MI355X, random data): 160 x 256 1570 (INT8) to 1640 (MXFP8), 256 x 256 2460, 256 x 128
// 1310 to 1470, 320 x 128 2100, 128 x 128 830.
static double step_clocks(int wn, int bm, int bn, bool three_stages) {
  const double mfma = bm * bn / 32.0 * 1.28, lds = (wn * bm + 256 + bm + bn) * 1.12;
  const double load = (bm + bn) * 128 / 47.0 + (three_stages ? 0 : 900);
  const double c = mfma > lds ? mfma : lds;
  return (c > load ? c : load) + 60;
}

// Whether, and on which tile, the deep kernel takes this launch: of its tiles the one with the least estimated time,
// where that is below the estimate for the 128-row kernels, which run without its prologue and epilogue costs (about
// 8 us a round of tiles, one workgroup per CU) but at half its rate. Their time, in clocks of 1.85 GHz, is 4 us and per
// 128-byte K step 1.65 us a round of 512 tiles (0.45 to 1.5 us for launches of fewer than 256, which run as 64 x 64
// tiles; 13.5 us a round, at least 6, where Cin is no multiple of 16: byte loads). Measured, deep against 128-row: INT8
// 512 -> 512 at 112 x 150 41 to 45 / 75 us, MXFP8 256 -> 256 at 224 x 300 46 to 49 / 67 us, INT8 196 -> 128 at 448 x 600
// 108 to 118 / 970 us; one-step 1 x 1 layers the other way round (64 -> 256 at 233 x 286 23 / 21 us).
// The 128-row kernels are the only alternative that is estimated, also where the wide kernel would take the launch instead
// of them; 1 x 1 launches that fit the pointwise kernels never come here (those kernels are asked first). Cout up to 64
// fills half of the narrowest tile at most, and a Cin below 36 was not tried (the walk needs two segments a tap, more than
// 16 channels): both stay with the 128-row kernels, on byte loads where ragged.
DeepPlan deep_plan(const ConvArgs& a, int kind) {
  const DeepPlan none = {0, 0, false, false};
  const bool mx = kind == KIND_MX;
  if (a.x_swz != nullptr || a.pool_out != nullptr || a.a_scale_rows != nullptr || a.gelu || a.Cout <= 64) return none;
  if (a.out_mode == (mx ? OUT_INT8 : OUT_E4M3)) return none;
  const int taps = a.kh * a.kw;
  if (taps > DEEP_TAPS || a.Cin < 36 || a.out_ld != a.Cout || (uintptr_t)a.out % 16 != 0) return none;
  if (mx && (a.w_expo_e8m0 || taps * a.Cin < 128 || a.Cin / 32 > DEEP_CBLOCKS)) return none;
  const uintptr_t both = (uintptr_t)a.x | (uintptr_t)a.w;
  const bool rag_in = a.Cin % 16 != 0, rag = rag_in || a.Cout % 16 != 0;
  if (mx ? rag || both % 16 != 0 : a.Cin % 4 != 0 || a.Cout % 4 != 0 || both % (rag_in ? 4 : 16) != 0) return none;
  // 32-bit offsets into buffers below 2 GiB, the residual laid out as the output
  if ((int64_t)a.B * a.H * a.W * a.Cin >= (1LL << 31) - 16 || (int64_t)a.Cout * taps * a.Cin >= (1LL << 31) - 16)
    return none;
  if ((int64_t)a.M * a.Cout * (a.residual != nullptr || a.out_mode == OUT_BF16 ? 2 : 1) >= (int64_t)0x7fffffff) return none;
  if (a.residual != nullptr &&
      !(a.res_dtype == FIM_BF16 && a.res_channels == a.Cout && a.rs_c == 1 && a.rs_w == a.Cout &&
        a.rs_h == (int64_t)a.Wo * a.Cout && a.rs_b == (int64_t)a.Ho * a.Wo * a.Cout && (uintptr_t)a.residual % 8 == 0))
    return none;
  constexpr double US = 1850;  // clocks
  const int64_t cus = device_cus();
  const double rounds128 = (double)(cdiv((int64_t)a.M, 128) * cdiv((int64_t)a.Cout, 128)) / (2.0 * cus);
  const double step16 = rounds128 >= 0.5 ? (1.65 * rounds128 > 1.3 ? 1.65 * rounds128 : 1.3)
                                         : (3.0 * rounds128 > 0.45 ? 3.0 * rounds128 : 0.45);
  const double step128 = !rag_in ? step16 : 13.5 * rounds128 > 6 ? 13.5 * rounds128 : 6;
  double best = (4 + taps * cdiv((int64_t)a.Cin, 128) * step128) * US;
  DeepPlan p = none;
  for (int wn = 2; wn <= 4; wn += 2)
    for (int mbw = deep_min_mbw(wn); mbw <= deep_max_mbw(wn); ++mbw) {
      const int bm = (4 / wn) * mbw * DEEP_BR, bn = 64 * wn;
      const int nst = deep_stages(mx, bm, bn);
      const int64_t rounds = cdiv(cdiv((int64_t)a.M, bm) * cdiv((int64_t)a.Cout, bn), cus);
      const int64_t nk = cdiv(cdiv((int64_t)taps * cdiv((int64_t)a.Cin, 16), 8), nst) * nst;
      const double epilogue = bm * bn * ((a.out_mode == OUT_INT8 ? 0.33 : 0.19) + (rag ? 0.12 : 0));
      const double mask = rag_in ? 300.0 * bm / 256 : 0;
      const double t = 2 * US + rounds * (nk * (step_clocks(wn, bm, bn, nst == 3) + mask) + 7500 + epilogue);
      if (t < best) {
        best = t;
        p = {wn, mbw, rag, false};
      }
    }
  // two 128 x 128 workgroups per CU: a pair's step is slower than a large tile's, but the round's prologue and epilogue
  // are half covered, which pays where several rounds of few steps run (INT8 196 -> 320 1 x 1 at 2 x 111 x 177 27 -> 21 us)
  const int64_t pairs = cdiv(cdiv((int64_t)a.M, 128) * cdiv((int64_t)a.Cout, 128), 2 * cus);
  const int64_t nk2 = cdiv(cdiv((int64_t)taps * cdiv((int64_t)a.Cin, 16), 8), 2) * 2;
  if (2 * US + pairs * (nk2 * (rag_in ? 1850 : 1700) + 11500) < best) p = {2, 2, rag, true};
  return p;
}

}  // namespace fim
