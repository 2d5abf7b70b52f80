// Shared by the implicit-GEMM convolution kernels (igemm.hip, deep.h): the launch arguments, masked segment loads, the
// GEMM row order and the epilogues.
#pragma once

#include <type_traits>

#include "common.h"

namespace fim {

enum { KIND_INT8 = 0, KIND_MX = 1 };
enum { OUT_BF16 = 0, OUT_INT8 = 1, OUT_E4M3 = 2 };

struct ConvArgs {
  const uint8_t* x;        // [B, H, W, Cin] int8 / e4m3
  const uint8_t* w;        // [Cout, T*Cin]
  const int8_t* x_expo;    // MX: [Cin / 32]
  const int8_t* w_expo;    // MX: [Cout, T*Cin / 32]
  int w_expo_e8m0;         // MX: w_expo holds E8M0 bytes (exponent + 127) instead of signed exponents
  const uint8_t* x_swz;    // MX, per-row scales (XS = 1): E8M0 bytes of x in the 128x4 swizzled layout
  int x_swz_tiles_k;       //   ceil((Cin / 32) / 4)
  const float* a_scale_rows;  // INT8: per-row activation scales [M] (null: the per-tensor a_scale)
  const float* a_scale;    // INT8: scalar
  const float* w_scale;    // INT8: [Cout]
  const void* bias;        // [Cout] or null
  int bias_dtype;          // FIM_F32 / FIM_BF16
  const void* residual;    // [B, Ho, Wo, res_channels] with strides, or null
  int res_dtype;
  int64_t res_channels, rs_b, rs_h, rs_w, rs_c;
  const float* out_scale;  // OUT_INT8
  const int8_t* out_expo;  // OUT_E4M3: [Cout / 32]
  void* out;               // [B, Ho, Wo, Cout]: pixel rows out_ld elements apart (out_ld >= Cout)
  int64_t out_ld;
  int8_t* pool_out;        // POOL: [B, Ho/2, Wo/2, Cout] int8, the 2x2 max pool of out quantized with out_scale
  int out_mode, relu_pre, relu_post, gelu;  // ReLU before the BF16 rounding / after the residual add
  int B, H, W, Cin, Ho, Wo, Cout;
  int kh, kw, sh, sw, ph, pw, dh, dw;
  int M;                   // output pixels (< 2^31)
  int kchunks;             // ceil(Cin / 128)
  int tps;                 // taps per 128-byte K step of the packed-tap kernels (PACK): 128 / Cin for Cin 16, 32, 64
  int n_tiles, m_tiles;
  int m_base;              // first GEMM row of this launch (a split launch runs its last rows as a second launch)
};

// The MFMA scale byte (E8M0: exponent + 127) of a weight exponent entry read as int8: signed exponents get + 127,
// E8M0 bytes pass through; (v + add) & 0xff covers both (an E8M0 byte above 127 reads as v - 256).
__device__ __forceinline__ int w_scale_byte(const ConvArgs& a, int v) { return (v + (a.w_expo_e8m0 ? 0 : 127)) & 0xff; }


constexpr int BM_MAIN = 128;  // pixel rows per tile (the tail of a launch may use 64-row tiles)
constexpr int KC = 128;          // bytes of K per step


// 16 bytes of one row segment, channel-masked. LW = widest load the layout allows (16: Cin % 16 == 0; else 1).
// 16 zero bytes in device memory: masked lanes (padding pixels, channel tails, rows past the tile) load from here, so
// every 16-byte segment load is unconditional and branch-free.
static __device__ __attribute__((aligned(16))) uint4 fim_zero_segment[1];

template <int LW>
__device__ __forceinline__ uint4 load_seg(const uint8_t* p, bool row_ok, int cvalid) {
  if (LW == 16) {
    const uint8_t* src = (row_ok && cvalid > 0) ? p : reinterpret_cast<const uint8_t*>(fim_zero_segment);
    return *reinterpret_cast<const uint4*>(src);
  }
  uint4 v = make_uint4(0, 0, 0, 0);
  if (!row_ok || cvalid <= 0) return v;
  if (LW == 4) {
    uint32_t t[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * i < cvalid) t[i] = reinterpret_cast<const uint32_t*>(p)[i];
    v = make_uint4(t[0], t[1], t[2], t[3]);
  } else {
    uint32_t t[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (i < cvalid) t[i >> 2] |= (uint32_t)p[i] << (8 * (i & 3));
    v = make_uint4(t[0], t[1], t[2], t[3]);
  }
  return v;
}

// GEMM row m -> output pixel index (img * Ho + oh) * Wo + ow. Plain order is the identity; the pool order (POOL, Ho and
// Wo even) puts the 4 pixels of each 2x2 pool window on 4 consecutive rows, windows in (img, oh / 2, ow / 2) order:
// m = 4 * window + 2 * dy + dx.
template <int POOL>
__device__ __forceinline__ int pixel_of_row(const ConvArgs& a, int m, int& img, int& oh, int& ow) {
  if (POOL) {
    const int wo2 = a.Wo >> 1, ho2 = a.Ho >> 1;
    const int win = m >> 2;
    const int q = win / wo2;
    ow = 2 * (win - q * wo2) + (m & 1);
    img = q / ho2;
    oh = 2 * (q - img * ho2) + ((m >> 1) & 1);
    return (img * a.Ho + oh) * a.Wo + ow;
  }
  ow = m % a.Wo;
  const int q = m / a.Wo;
  img = q / a.Ho;
  oh = q - img * a.Ho;
  return m;
}

// Epilogue of one wavefront's MB x NB blocks of 16 x 16 outputs, straight from the accumulators: D[n][m] with
// lane = pixel (lane & 15) of a 16-pixel block and 4 consecutive channels 4 (lane >> 4) + v of a 16-channel block, so
// each store writes 4 channels of one pixel. mrow[j]: this lane's GEMM row in block j (M or more: no output);
// n_tile0: the tile's first channel; nl0:
// the wave's first channel within the tile (index into the per-channel operands ep_* staged in LDS).
// Branch-free epilogue for the common case (no residual, no pooling, Cout % 16 == 0, output below 2 GiB): per
// 16-pixel row block, all NB x 4 values of the lane are computed (their chains, GELU's above all, interleave) and then
// stored, so the stores stream out while the next block is computed, each burst covering whole lines; outputs past M
// or Cout are dropped by the buffer store's range check instead of per-lane branches. Same arithmetic, in the same
// order per value, as the general epilogue below.
// RES: a BF16 residual laid out as the output ([M, Cout] dense, so its element offset is the output's), added after
// the activation with the conv semantics relu(y + r) (ops/conv.py:198-203): loaded per row block with the same
// out-of-range handling as the stores.
// The lane's per-channel epilogue operands: for each of its NB channel blocks, the scale and bias of its 4 channels
// and their output scale (the lane's 4 channels, aligned by 4, share one 32-channel scale block).
template <int NB>
struct EpiChannels {
  float cs[NB][4], cb[NB][4], osc[NB];
};

// CB: channels per block, i.e. the accumulators' layout: 16 (16 x 16 MFMA: 4 consecutive channels per 16-lane group) or
// 8 (32 x 32 MFMA: lane = pixel (lane & 31), 4 consecutive channels 4 (lane >> 5) of each 8).
template <int NB, int CB = 16>
__device__ __forceinline__ EpiChannels<NB> epi_channels(int nl0, const float* ep_scale, const float* ep_bias,
                                                        const float* ep_osc) {
  const int g = (threadIdx.x & 63) >> (CB == 16 ? 4 : 5);
  EpiChannels<NB> ch;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int nl = nl0 + i * CB + 4 * g;
    const float4 cs4 = *reinterpret_cast<const float4*>(&ep_scale[nl]);
    const float4 cb4 = *reinterpret_cast<const float4*>(&ep_bias[nl]);
    ch.cs[i][0] = cs4.x; ch.cs[i][1] = cs4.y; ch.cs[i][2] = cs4.z; ch.cs[i][3] = cs4.w;
    ch.cb[i][0] = cb4.x; ch.cb[i][1] = cb4.y; ch.cb[i][2] = cb4.z; ch.cb[i][3] = cb4.w;
    ch.osc[i] = ep_osc[nl];
  }
  return ch;
}

// Staged output: the values go to an LDS tile instead of global memory, row (tile pixel) spix[j] of STAGE_RB bytes per
// pixel, 16-byte slot s of row p at slot s ^ stage_swz(p) (the caller writes the tile out in whole lines).
__device__ __forceinline__ int stage_swz(int p) { return (p >> 1) & 7; }

// GELU: 0 none (ReLU or the identity as one IEEE maximum), 1 GELU without ReLU (no maximum), 2 ReLU then GELU.
// CB: see epi_channels. RAG: Cout % 4 == 0 only, so the channel test is the lane's own instead of the block's.
template <int KIND, int OUT, int MB, int NB, int GELU, bool RES = false, int STAGE_RB = 0, int CB = 16,
          bool RAG = false>
__device__ __forceinline__ void conv_epilogue_fast(const ConvArgs& a, const v4i (&acc_i)[NB][MB],
                                                   const v4f (&acc_f)[NB][MB], const int (&mrow)[MB], int n_tile0,
                                                   int nl0, const EpiChannels<NB>& ch, uint8_t* stage = nullptr,
                                                   const int* spix = nullptr) {
  constexpr int ESZ = OUT == OUT_BF16 ? 2 : 1;
  const int lane = threadIdx.x & 63;
  const int g = lane >> (CB == 16 ? 4 : 5);
  const float out_scale = OUT == OUT_INT8 ? *a.out_scale : 1.0f;
  const float out_inv = OUT == OUT_INT8 ? __fdiv_rn(1.0f, out_scale) : 1.0f;
  // ReLU as IEEE maximum against 0 (on) or -inf (off: the identity, NaN kept): one operation, no select
  float relu_lo = a.relu_pre != 0 ? 0.0f : -__builtin_inff();
  asm("" : "+v"(relu_lo));  // opaque: otherwise the compiler folds the bound back into a per-value select
  const bool row_scales = KIND == KIND_INT8 && a.a_scale_rows != nullptr;
  // descriptor operands through readfirstlane: provably uniform, so the descriptor stays in SGPRs (a descriptor the
  // compiler cannot prove uniform turns every store into a readfirstlane loop)
  const int nbytes = __builtin_amdgcn_readfirstlane((int)((uint32_t)a.M * (uint32_t)a.out_ld * ESZ));
  const uint64_t out_addr = (uint64_t)a.out;
  const uint64_t out_u = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(out_addr >> 32)) << 32) |
                         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)out_addr);
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(out_u), (short)0, nbytes, 0x00020000);
  __amdgpu_buffer_rsrc_t res_rsrc = rsrc;
  float relu_post_lo = -__builtin_inff();
  if constexpr (RES) {
    const uint64_t res_addr = (uint64_t)a.residual;
    const uint64_t res_u = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(res_addr >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)res_addr);
    res_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(res_u), (short)0,
        __builtin_amdgcn_readfirstlane((int)((uint32_t)a.M * (uint32_t)a.Cout * 2)), 0x00020000);
    relu_post_lo = a.relu_post != 0 ? 0.0f : -__builtin_inff();
    asm("" : "+v"(relu_post_lo));
  }
  float arow[MB];
#pragma unroll
  for (int j = 0; j < MB; ++j) arow[j] = row_scales ? a.a_scale_rows[min(mrow[j], a.M - 1)] : 1.f;
  const auto& cs = ch.cs;
  const auto& cb = ch.cb;
  const auto& osc = ch.osc;
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int m = mrow[j];
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    u32x2 rv[NB];
    if constexpr (RES) {  // this row block's residual, in flight while its values are computed
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const bool nvalid = n_tile0 + nl0 + i * CB + (RAG ? 4 * g : 0) < a.Cout;
        const uint32_t roff =
            nvalid ? ((uint32_t)m * (uint32_t)a.Cout + (uint32_t)(n_tile0 + nl0 + i * CB + 4 * g)) * 2 : 0x80000000u;
        rv[i] = __builtin_amdgcn_raw_buffer_load_b64(res_rsrc, (int)roff, 0, 0);
      }
    }
    float y[NB][4];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      float* v = y[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t;
        if (KIND == KIND_INT8)
          t = row_scales ? __fmul_rn((float)acc_i[i][j][e], __fmul_rn(arow[j], cs[i][e]))
                         : __fmul_rn((float)acc_i[i][j][e], cs[i][e]);
        else
          t = acc_f[i][j][e];
        t = __fadd_rn(t, cb[i][e]);  // the staged bias is -0 when there is none
        v[e] = GELU == 1 ? t : __builtin_elementwise_maximum(t, relu_lo);
      }
      round_bf16x2(v[0], v[1]);
      round_bf16x2(v[2], v[3]);
      if (GELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_erf(v[e]);
        if (RES || OUT == OUT_INT8) {  // a BF16 store's pack and the E4M3 conversion round the same way
          round_bf16x2(v[0], v[1]);
          round_bf16x2(v[2], v[3]);
        }
      }
      if constexpr (RES) {  // relu(y + r) in FP32, then BF16 (a BF16 store's pack rounds)
        v[0] = __builtin_elementwise_maximum(__fadd_rn(v[0], u2f(rv[i][0] << 16)), relu_post_lo);
        v[1] = __builtin_elementwise_maximum(__fadd_rn(v[1], u2f(rv[i][0] & 0xffff0000u)), relu_post_lo);
        v[2] = __builtin_elementwise_maximum(__fadd_rn(v[2], u2f(rv[i][1] << 16)), relu_post_lo);
        v[3] = __builtin_elementwise_maximum(__fadd_rn(v[3], u2f(rv[i][1] & 0xffff0000u)), relu_post_lo);
        if (OUT == OUT_INT8) {
          round_bf16x2(v[0], v[1]);
          round_bf16x2(v[2], v[3]);
        }
      }
    }
    uint32_t codes[NB];
    if constexpr (OUT == OUT_INT8) {
      // NQ values share one near-tie test (one wave-uniform branch): 4 where another wavefront of the SIMD covers the
      // branch's latency, 16 in the one-wavefront kernel (deep.h: its 160 x 256 INT8 epilogue 15.9k -> 13.7k clocks)
      constexpr int NQ = CB == 16 ? 1 : 4;
#pragma unroll
      for (int i = 0; i < NB; i += NQ) {
        float vq[4 * NQ];
        int qi[4 * NQ];
#pragma unroll
        for (int e = 0; e < 4 * NQ; ++e) vq[e] = y[i + (e >> 2)][e & 3];
        quantize_int8_fast_n<4 * NQ>(vq, out_scale, out_inv, qi);
#pragma unroll
        for (int e = 0; e < NQ; ++e)
          codes[i + e] = (uint32_t)(qi[4 * e] & 0xff) | ((uint32_t)(qi[4 * e + 1] & 0xff) << 8) |
                         ((uint32_t)(qi[4 * e + 2] & 0xff) << 16) | ((uint32_t)qi[4 * e + 3] << 24);
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const float* v = y[i];
      const int nbase = n_tile0 + nl0 + i * CB + 4 * g;
      const bool nvalid = n_tile0 + nl0 + i * CB + (RAG ? 4 * g : 0) < a.Cout;  // whole block in or out (not RAG)
      // rows past M land past the buffer's end; invalid channel blocks are sent there too
      const uint32_t off = nvalid ? ((uint32_t)m * (uint32_t)a.out_ld + (uint32_t)nbase) * ESZ : 0x80000000u;
      uint8_t* sd = nullptr;
      if constexpr (STAGE_RB > 0) {
        const int cb = (nl0 + i * CB + 4 * g) * ESZ;  // the lane's bytes within the staged row
        const int sl = ((cb >> 4) ^ stage_swz(spix[j])) & (STAGE_RB / 16 - 1);
        sd = stage + spix[j] * STAGE_RB + sl * 16 + (cb & 15);
      }
      if (OUT == OUT_BF16) {
        const uint32_t lo = pack_bf16x2(v[0], v[1]), hi = pack_bf16x2(v[2], v[3]);
        if constexpr (STAGE_RB > 0)
          *reinterpret_cast<u32x2*>(sd) = u32x2{lo, hi};
        else
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{lo, hi}, rsrc, (int)off, 0, 0);
      } else {
        uint32_t pk;
        if (OUT == OUT_INT8) {
          pk = codes[i];
        } else {
          pk = e4m3x4_of_bf16(v[0], v[1], v[2], v[3], osc[i], 448.0f * osc[i]);  // rounds to BF16 first
        }
        if constexpr (STAGE_RB > 0)
          *reinterpret_cast<uint32_t*>(sd) = pk;
        else
          __builtin_amdgcn_raw_buffer_store_b32(pk, rsrc, (int)off, 0, 0);
      }
    }
    // this row block's stores (all NB x 16 channels of 16 pixels: whole 128-byte lines of a BF16 output) go out before
    // the next block is computed, so the writes stream during the epilogue and each line is written in one burst
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The fast epilogue's variants (GELU with or without a ReLU before it, dense residual) for lane rows mrow, into global
// memory (STAGE_RB = 0) or an LDS staging tile (see conv_epilogue_fast's STAGE_RB); the caller has checked
// conv_fast_ok.
template <int KIND, int OUT, int MB, int NB, int STAGE_RB = 0>
__device__ __forceinline__ void conv_epilogue_any(const ConvArgs& a, const v4i (&acc_i)[NB][MB],
                                                  const v4f (&acc_f)[NB][MB], const int (&mrow)[MB], int n_tile0,
                                                  int nl0, const EpiChannels<NB>& ch, uint8_t* stage = nullptr,
                                                  const int* spix = nullptr) {
#define FIM_EPI(G, R) \
  conv_epilogue_fast<KIND, OUT, MB, NB, G, R, STAGE_RB>(a, acc_i, acc_f, mrow, n_tile0, nl0, ch, stage, spix)
  const int act = a.gelu ? (a.relu_pre ? 2 : 1) : 0;
  if (a.residual != nullptr) {
    if (act == 1) FIM_EPI(1, true);
    else if (act == 2) FIM_EPI(2, true);
    else FIM_EPI(0, true);
  } else {
    if (act == 1) FIM_EPI(1, false);
    else if (act == 2) FIM_EPI(2, false);
    else FIM_EPI(0, false);
  }
#undef FIM_EPI
}

// Calls f(integral_constant<int, GELU>, integral_constant<bool, RES>) with the fast epilogue's variant for this launch:
// kernels whose epilogue is a loop of calls select the variant once, outside the loop, so the loop body holds one
// variant and unrolls (with the selection inside, the body holds all six and the compiler stops unrolling, which turns
// the accumulator indexing dynamic and puts the accumulators in scratch memory).
template <typename F>
__device__ __forceinline__ void with_epilogue_variant(const ConvArgs& a, F&& f) {
  using G0 = std::integral_constant<int, 0>;
  using G1 = std::integral_constant<int, 1>;
  using G2 = std::integral_constant<int, 2>;
  using RY = std::integral_constant<bool, true>;
  using RN = std::integral_constant<bool, false>;
  const int act = a.gelu ? (a.relu_pre ? 2 : 1) : 0;
  if (a.residual != nullptr) {
    if (act == 1) f(G1{}, RY{});
    else if (act == 2) f(G2{}, RY{});
    else f(G0{}, RY{});
  } else {
    if (act == 1) f(G1{}, RN{});
    else if (act == 2) f(G2{}, RN{});
    else f(G0{}, RN{});
  }
}

template <int KIND, int OUT, int MB, int NB>
__device__ __forceinline__ void conv_epilogue_rows(const ConvArgs& a, const v4i (&acc_i)[NB][MB],
                                                   const v4f (&acc_f)[NB][MB], const int (&mrow)[MB], int n_tile0,
                                                   int nl0, const EpiChannels<NB>& ch) {
  conv_epilogue_any<KIND, OUT, MB, NB>(a, acc_i, acc_f, mrow, n_tile0, nl0, ch);
}

template <int KIND, int OUT, int MB, int NB>
__device__ __forceinline__ void conv_epilogue_rows(const ConvArgs& a, const v4i (&acc_i)[NB][MB],
                                                   const v4f (&acc_f)[NB][MB], const int (&mrow)[MB], int n_tile0,
                                                   int nl0, const float* ep_scale, const float* ep_bias,
                                                   const float* ep_osc) {
  conv_epilogue_rows<KIND, OUT, MB, NB>(a, acc_i, acc_f, mrow, n_tile0, nl0,
                                        epi_channels<NB>(nl0, ep_scale, ep_bias, ep_osc));
}

// Whether the fast epilogue applies: no residual or a BF16 residual laid out as the output (the refiner blocks'
// contract convs), no pooling, Cout % 16 == 0, the output below 2 GiB.
template <int OUT>
__host__ __device__ __forceinline__ bool conv_fast_ok(const ConvArgs& a) {
  const bool res_dense = a.residual != nullptr && a.res_dtype == FIM_BF16 && a.res_channels == a.Cout && a.rs_c == 1 &&
                         a.rs_w == a.Cout && a.rs_h == (int64_t)a.Wo * a.Cout &&
                         a.rs_b == (int64_t)a.Ho * a.Wo * a.Cout && ((uintptr_t)a.residual & 7) == 0 &&
                         (int64_t)a.M * a.Cout * 2 < (int64_t)0x7fffffff;
  return a.pool_out == nullptr && (a.residual == nullptr || res_dense) && (a.Cout & 15) == 0 &&
         (int64_t)a.M * a.out_ld * (OUT == OUT_BF16 ? 2 : 1) < (int64_t)0x7fffffff;
}

template <int KIND, int OUT, int POOL, int MB, int NB>
__device__ __forceinline__ void conv_epilogue(const ConvArgs& a, const v4i (&acc_i)[NB][MB], const v4f (&acc_f)[NB][MB],
                                              int row0, int n_tile0, int nl0, const float* ep_scale,
                                              const float* ep_bias, const float* ep_osc) {
  if (!POOL && conv_fast_ok<OUT>(a)) {
    int mrow[MB];
#pragma unroll
    for (int j = 0; j < MB; ++j) mrow[j] = row0 + j * 16 + (threadIdx.x & 15);
    conv_epilogue_rows<KIND, OUT, MB, NB>(a, acc_i, acc_f, mrow, n_tile0, nl0, ep_scale, ep_bias, ep_osc);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  // flags are uniform (scalar branches); the output format is a template parameter
  const float out_scale = (OUT == OUT_INT8 || POOL) ? *a.out_scale : 1.0f;
  const float out_inv = (OUT == OUT_INT8 || POOL) ? __fdiv_rn(1.0f, out_scale) : 1.0f;
  const bool has_bias = a.bias != nullptr;
  const bool res = a.residual != nullptr;
  const bool relu_pre = a.relu_pre != 0;
  const bool relu_post = a.relu_post != 0;
  const bool res_vec = res && a.res_dtype == FIM_BF16 && a.rs_c == 1 && (((uintptr_t)a.residual) & 7) == 0 &&
                       (a.rs_w % 4) == 0 && (a.rs_h % 4) == 0 && (a.rs_b % 4) == 0;
  const bool out_vec = (a.Cout % 4) == 0;
  int pm[MB], px[MB];
  int64_t roff[MB];
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int m = row0 + j * 16 + (lane & 15);
    pm[j] = m;
    roff[j] = 0;
    int img, oh, ow;
    px[j] = pixel_of_row<POOL>(a, m < a.M ? m : 0, img, oh, ow);
    if (res) roff[j] = (int64_t)img * a.rs_b + (int64_t)oh * a.rs_h + (int64_t)ow * a.rs_w;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int nl = nl0 + i * 16 + 4 * g;
    const int nbase = n_tile0 + nl;
    const float4 cs4 = *reinterpret_cast<const float4*>(&ep_scale[nl]);
    const float4 cb4 = *reinterpret_cast<const float4*>(&ep_bias[nl]);
    const float osc = ep_osc[nl];  // E4M3 output scale of the lane's 4 channels (one 32-channel block)
    const float cs[4] = {cs4.x, cs4.y, cs4.z, cs4.w};
    const float cb[4] = {cb4.x, cb4.y, cb4.z, cb4.w};
    const bool full = nbase + 4 <= a.Cout;
    const bool any = nbase < a.Cout;
    const bool res_full = res_vec && nbase + 4 <= a.res_channels;
#pragma unroll
    for (int j = 0; j < MB; ++j) {
      const int m = pm[j];
      if (!any || m >= a.M) continue;
      float y[4];
      if (KIND == KIND_INT8 && a.a_scale_rows != nullptr) {
        const float arow = a.a_scale_rows[m];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = __fmul_rn((float)acc_i[i][j][v], __fmul_rn(arow, cs[v]));
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = KIND == KIND_INT8 ? __fmul_rn((float)acc_i[i][j][v], cs[v]) : acc_f[i][j][v];
      }
      if (has_bias) {
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = __fadd_rn(y[v], cb[v]);
      }
      if (relu_pre) {
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = fmaxf(y[v], 0.0f);
      }
      round_bf16x2(y[0], y[1]);
      round_bf16x2(y[2], y[3]);
      if (a.gelu) {
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = gelu_erf(y[v]);
        round_bf16x2(y[0], y[1]);
        round_bf16x2(y[2], y[3]);
      }
      if (res) {
        float rv[4] = {0.f, 0.f, 0.f, 0.f};
        if (res_full) {
          const uint2 pk = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.residual) + roff[j] + nbase);
          rv[0] = u2f(pk.x << 16);
          rv[1] = u2f(pk.x & 0xffff0000u);
          rv[2] = u2f(pk.y << 16);
          rv[3] = u2f(pk.y & 0xffff0000u);
#pragma unroll
          for (int v = 0; v < 4; ++v) y[v] = __fadd_rn(y[v], rv[v]);
          if (relu_post) {
#pragma unroll
            for (int v = 0; v < 4; ++v) y[v] = fmaxf(y[v], 0.0f);
          }
          round_bf16x2(y[0], y[1]);
          round_bf16x2(y[2], y[3]);
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int n = nbase + v;
            if (n < a.res_channels) {
              const int64_t off = roff[j] + (int64_t)n * a.rs_c;
              const float r = a.res_dtype == FIM_BF16 ? bf16_to_f32(static_cast<const uint16_t*>(a.residual)[off])
                                                      : static_cast<const float*>(a.residual)[off];
              float t = __fadd_rn(y[v], r);
              if (relu_post) t = fmaxf(t, 0.0f);
              y[v] = round_bf16_hw(t);
            } else if (relu_post) {
              y[v] = fmaxf(y[v], 0.0f);
            }
          }
        }
      }
      const int64_t o = (int64_t)px[j] * a.out_ld + nbase;
      if (POOL) {
        // the window's 4 pixels sit on lanes 4k .. 4k + 3 of this 16-lane group (rows m = 4 * window + 0..3), all
        // valid or all past M together: max across them, quantize (monotonic, so equal to quantizing the max of the
        // quantized values), one 4-channel store per window
        float p[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          p[v] = fmaxf(y[v], __shfl_xor(y[v], 1));
          p[v] = fmaxf(p[v], __shfl_xor(p[v], 2));
        }
        if ((lane & 3) == 0) {
          uint32_t pk = 0;
#pragma unroll
          for (int v = 0; v < 4; ++v) pk |= (uint32_t)(uint8_t)quantize_int8_fast(p[v], out_scale, out_inv) << (8 * v);
          uint8_t* pdst = reinterpret_cast<uint8_t*>(a.pool_out) + (int64_t)(m >> 2) * a.Cout + nbase;
          if (out_vec && full) {
            *reinterpret_cast<uint32_t*>(pdst) = pk;
          } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
              if (nbase + v < a.Cout) pdst[v] = (uint8_t)(pk >> (8 * v));
          }
        }
      }
      if (OUT == OUT_BF16) {
        uint16_t* dst = static_cast<uint16_t*>(a.out) + o;
        const uint32_t lo = pack_bf16x2(y[0], y[1]), hi = pack_bf16x2(y[2], y[3]);
        if (out_vec && full) {
          *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
        } else {
          const uint16_t h[4] = {(uint16_t)lo, (uint16_t)(lo >> 16), (uint16_t)hi, (uint16_t)(hi >> 16)};
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (nbase + v < a.Cout) dst[v] = h[v];
        }
      } else {
        uint32_t pk;
        if (OUT == OUT_INT8) {
          pk = 0;
#pragma unroll
          for (int v = 0; v < 4; ++v) pk |= (uint32_t)(uint8_t)quantize_int8_fast(y[v], out_scale, out_inv) << (8 * v);
        } else {
          pk = e4m3x4_of_bf16(y[0], y[1], y[2], y[3], osc, 448.0f * osc);
        }
        uint8_t* dst = static_cast<uint8_t*>(a.out) + o;
        if (out_vec && full) {
          *reinterpret_cast<uint32_t*>(dst) = pk;
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (nbase + v < a.Cout) dst[v] = (uint8_t)(pk >> (8 * v));
        }
      }
    }
  }
}

typedef __attribute__((address_space(3))) void lds_void_t;

// s_waitcnt immediate (gfx9 encoding) for at most `vm` outstanding vector memory operations and no LDS/scalar ones:
// vmcnt in bits 3:0 and 15:14, expcnt (7: no wait) in 6:4, lgkmcnt (0) in 11:8. Issued through the builtin, so the
// compiler's own wait counting sees it.
constexpr int waitcnt_vm_lgkm0(int vm) { return (vm & 0xF) | (0x7 << 4) | (((vm >> 4) & 0x3) << 14); }

}  // namespace fim
