// Deep implicit-GEMM convolution: launches of several K steps (3 x 3 and 5 x 5 convs, wide 1 x 1 ones), INT8 and MXFP8.
// One workgroup of four wavefronts per CU, one wavefront per SIMD with the whole register file, over a tile of 128 x 128
// to 256 x 256 or 320 x 128 outputs; each wavefront 32 mbw rows x 64 channels on 32 x 32 MFMAs.
//
// What bounds the 128-row kernel on these launches is LDS traffic: a wavefront's 64 x 64 outputs take as many clocks of
// operand reads as of MFMAs, and two workgroups per CU stage the same weights twice. Here the accumulators take up to
// 256 registers, so an operand read feeds twice to three times the MFMAs. With one wavefront per SIMD nothing else covers
// its waits, so they are taken out of the K loop: loads go to LDS two steps ahead (one for the tiles whose three stages
// do not fit), operands are read one block ahead, the last blocks' MFMAs run past the step's barrier, and reads and loads
// sit between the MFMAs. K is walked in 16-byte segments across the taps, so only the last step is padded (a Cin of 160
// takes 12 steps of a 3 x 3 filter instead of 18), and INT8 channel counts may be any multiple of 4 (from 36 in and 68
// out on).
// Measured (MI355X): a 160 x 256 step 1570 clocks for 1280 of MFMA issue, at the 1.75 to 1.9 GHz that the matrix cores'
// power draw leaves; prologue 3.3 us, epilogue 3 to 6 us. INT8 512 -> 512 3 x 3 at 112 x 150 75 -> 41 to 45 us (160 x 256
// tiles), MXFP8 256 -> 256 at 224 x 300 67 -> 46 to 49 us (the same), INT8 196 -> 128 at 448 x 600 970 -> 108 to 118 us
// (two 128 x 128 workgroups per CU; it ran on byte loads).
#pragma once

#include "deep_plan.h"

namespace fim {

// What the host adds to the launch arguments: division by Wo and Ho as a multiply and a shift (exact for rows below
// 2^31), and the K walk in 16-byte segments.
struct DeepArgs {
  ConvArgs c;
  uint32_t wo_mul, ho_mul;
  int wo_shift, ho_shift;
  int segs;              // 16-byte K segments per tap: ceil(Cin / 16)
  int adv_tap, adv_seg;  // 8 segments (one K step) on: 8 / segs taps and 8 % segs segments
  int nk;                // K steps: ceil(taps * segs / 8)
};

__device__ __forceinline__ int div_magic(int n, uint32_t mul, int shift) {
  return shift < 0 ? n : (int)(__umulhi((uint32_t)n, mul) >> shift);
}

// TWO: two workgroups per CU (128 x 128 tiles in two stages), which cover each other's prologues, epilogues and waits.
template <int KIND, int OUT, int WN, int MBW, bool RAG, bool TWO = false>
__global__ __launch_bounds__(256, TWO ? 2 : 1) void conv_deep_kernel(const DeepArgs d) {
  constexpr int WM = 4 / WN, BR = DEEP_BR;
  constexpr int BM = WM * MBW * BR, BN = WN * 64;
  // a stage: the weight rows, then the activation rows, in 8-row chunks (one wave-wide 16-byte-per-lane load each);
  // wavefront w loads chunks w, w + 4, ... of each
  constexpr int NW = BN / 32, NA = BM / 32, CHUNKS = NW + NA;
  constexpr int STAGE = (BM + BN) * KC;
  constexpr int NST = TWO ? 2 : deep_stages(KIND == KIND_MX, BM, BN);
  // The software pipeline over a step's 32-row blocks: a block's operands are read during the block before it, and the
  // last L blocks' MFMAs run after the barrier that ends the step, while the next step's first operands are read. The
  // reads and the next stage's loads are placed one by one between the MFMAs (a load issued behind another waits for
  // the address unit, 64 clocks for the four wavefronts, and the MFMAs behind it in the wavefront wait with it).
  constexpr int L = MBW > 3 ? 2 : 1, MAIN = MBW - L;
  static_assert(MAIN >= 1, "a block before the tail");
  constexpr int SL = KIND == KIND_MX ? 4 : 8;  // MFMAs per block and step
  constexpr int SPAN = NST == 3 ? MAIN * SL : (MAIN * SL * 5 + 7) / 8;  // MFMA slots that the loads are spread over
  const ConvArgs& a = d.c;

  __shared__ __attribute__((aligned(16))) uint8_t st0[STAGE];
  __shared__ __attribute__((aligned(16))) uint8_t st1[STAGE];
  __shared__ __attribute__((aligned(16))) uint8_t st2[NST == 3 ? STAGE : 16];
  __shared__ __attribute__((aligned(16))) float ep_bias[BN], ep_scale[KIND == KIND_INT8 ? BN : 4];
  __shared__ int tap_off[32];
  __shared__ uint32_t ex_w[KIND == KIND_MX ? 2 * BN : 1];
  __shared__ uint8_t ex_x[KIND == KIND_MX ? DEEP_CBLOCKS : 4];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = wave / WN;

  const int per_xcd = gridDim.x >> 3;
  const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (t >= a.n_tiles * a.m_tiles) return;
  const int n0 = (t % a.n_tiles) * BN;
  const int m0 = (t / a.n_tiles) * BM;
  const int taps = a.kh * a.kw;

  if (tid < BN) {
    const int n = n0 + tid;
    const bool nok = n < a.Cout;
    if (KIND == KIND_INT8) ep_scale[tid] = nok ? *a.a_scale * a.w_scale[n] : 1.0f;
    float bias = -0.0f;  // x + (-0) == x for every x, -0 included: the fast epilogue adds it unconditionally
    if (a.bias != nullptr && nok)
      bias = a.bias_dtype == FIM_BF16 ? bf16_to_f32(static_cast<const uint16_t*>(a.bias)[n])
                                      : static_cast<const float*>(a.bias)[n];
    ep_bias[tid] = bias;
  }
  if (tid >= 224) {
    const int tap = tid - 224, ky = tap < taps ? tap / a.kw : 0, kx = tap < taps ? tap - ky * a.kw : 0;
    tap_off[tap] = (ky * a.dh * a.W + kx * a.dw) * a.Cin;
  }

  const int wrow = taps * a.Cin;
  const int x_nrec = __builtin_amdgcn_readfirstlane((int)((int64_t)a.B * a.H * a.W * a.Cin));
  const int w_nrec = __builtin_amdgcn_readfirstlane(a.Cout * wrow);
  constexpr uint32_t OOB = 0x80000000u;  // past both buffers: reads as zero

  // staged rows of this lane: chunk c holds rows 8 c + lane / 8; LDS slot lane % 8 of row r holds K segment
  // (lane % 8) ^ ((r / 2) % 8), the same for all of this wavefront's chunks (they have one parity)
  const int seg = (lane & 7) ^ (lane >> 4) ^ (4 * (wave & 1));
  int x_base[NA];
  uint32_t x_dead[NA];  // bit t: tap t of this row lies outside the image (or past the filter)
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int m = m0 + 8 * (wave + 4 * i) + (lane >> 3);
    const int mc = m < a.M ? m : 0;
    const int q = div_magic(mc, d.wo_mul, d.wo_shift);
    const int ow = mc - q * a.Wo;
    const int img = div_magic(q, d.ho_mul, d.ho_shift);
    const int oh = q - img * a.Ho;
    const int ih = oh * a.sh - a.ph, iw = ow * a.sw - a.pw;
    x_base[i] = ((img * a.H + ih) * a.W + iw) * a.Cin;
    uint32_t cols = 0, live = 0;
    for (int kx = 0; kx < a.kw; ++kx) cols |= (uint32_t)((unsigned)(iw + kx * a.dw) < (unsigned)a.W) << kx;
    for (int ky = 0; ky < a.kh; ++ky)
      live |= ((unsigned)(ih + ky * a.dh) < (unsigned)a.H ? cols : 0u) << (ky * a.kw);
    x_dead[i] = m < a.M ? ~live : ~0u;
  }
  uint32_t w_base[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int n = n0 + 8 * (wave + 4 * i) + (lane >> 3);
    w_base[i] = n < a.Cout ? (uint32_t)(n * wrow) : OOB;
  }
  __syncthreads();  // tap_off (the epilogue operands too)

  // K walk of the next step to load: segment index over all taps, its tap and its segment within the tap
  int ld_flat = seg, ld_tap = seg / d.segs, ld_cs = seg % d.segs;
  const int total_segs = taps * d.segs;
  int xk, xsh, wk;  // per step: offset within x, mask shift, offset within a weight row
  uint32_t wdead;
  auto load_step = [&]() __attribute__((always_inline)) {
    const bool live = ld_flat < total_segs;
    const int tap = live ? ld_tap : 31;  // bit 31 of a row's mask is set: past the end every load reads zero
    xk = tap_off[tap] + ld_cs * 16;
    xsh = 31 - tap;
    wk = RAG ? tap * a.Cin + ld_cs * 16 : ld_flat * 16;
    wdead = live ? 0u : OOB;
    ld_flat += 8;
    ld_tap += d.adv_tap;
    ld_cs += d.adv_seg;
    const bool wrap = ld_cs >= d.segs;
    ld_cs -= wrap ? d.segs : 0;
    ld_tap += wrap ? 1 : 0;
  };
  // chunk i of the step into LDS stage st: first the weights (i < NW), then the activations
  auto issue = [&](uint8_t* st, int i) __attribute__((always_inline)) {
    if (i < NW) {
      const uint32_t off = (w_base[i] + (uint32_t)wk) | wdead;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.w), (short)0, w_nrec, 0x00020000),
          (lds_void_t*)(st + (wave + 4 * i) * 1024), 16, off, 0, 0, 0);
    } else if (i < CHUNKS) {
      const uint32_t off = (uint32_t)(x_base[i - NW] + xk) | ((x_dead[i - NW] << xsh) & OOB);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.x), (short)0, x_nrec, 0x00020000),
          (lds_void_t*)(st + (BN / 8 + wave + 4 * (i - NW)) * 1024), 16, off, 0, 0, 0);
    }
  };

  // MX scales, as MFMA scale bytes (exponent + 127) in LDS: thread tid loads the step's four weight exponents of tile row
  // tid % BN in one load, two steps ahead, and the lanes pick theirs from LDS. (A byte load per lane
  // and 16-channel block, the lanes of an instruction on 16 rows, keeps the address unit busy for 64 clocks: five of
  // them a step and wavefront took longer than the step's MFMAs.) The activations' scales, one per 32 channels for all
  // rows, are staged once.
  const int h = lane >> 5;
  const int cblocks = a.Cin >> 5, wblocks = taps * cblocks;
  int ex_blk = 0;           // first K block of the step to load
  uint32_t ex_raw = 0;
  int ex_shift = 0;
  const int8_t* ex_row = nullptr;
  if constexpr (KIND == KIND_MX) {
    const int n = n0 + (tid & (BN - 1));
    ex_row = a.w_expo + (int64_t)(n < a.Cout ? n : 0) * wblocks;
    for (int i = tid; i < cblocks; i += 256) ex_x[i] = (uint8_t)(a.x_expo[i] + 127);
  }
  auto load_exponents = [&]() __attribute__((always_inline)) {
    if constexpr (KIND == KIND_MX) {
      // the row's last blocks: its last four, shifted (blocks past the row get scale 2^-127 on zero data)
      const int over = ex_blk + 4 - wblocks;
      __builtin_memcpy(&ex_raw, ex_row + (over > 0 ? wblocks - 4 : ex_blk), 4);
      ex_shift = over > 0 && over < 4 ? 8 * over : 0;
      ex_blk += 4;
    }
  };
  // into the slot of the odd or even steps
  int ex_slot = 0;
  auto store_exponents = [&]() __attribute__((always_inline)) {
    if constexpr (KIND == KIND_MX) {
      // per byte exponent + 128 - 1, without borrows between the bytes
      const uint32_t H = 0x80808080u, v = ex_raw ^ H;
      ex_w[ex_slot + (tid & (BN - 1))] = (((v | H) - 0x01010101u) ^ (~v & H)) >> ex_shift;
    }
  };
  // K blocks h and 2 + h of the step are this lane's in its two MFMA steps of 64 K bytes (h = lane / 32)
  int exb0 = KIND == KIND_MX ? h % cblocks : 0, exb1 = KIND == KIND_MX ? (2 + h) % cblocks : 0;
  const int eadv = KIND == KIND_MX ? 4 % cblocks : 0;
  int sx[NST][2], sw[NST][2];
  auto read_scales = [&](int slot) __attribute__((always_inline)) {
    if constexpr (KIND == KIND_MX) {
      sx[slot][0] = ex_x[exb0];
      sx[slot][1] = ex_x[exb1];
#pragma unroll
      for (int i = 0; i < 2; ++i) sw[slot][i] = (int)ex_w[ex_slot + wn * 64 + i * 32 + (lane & 31)];
      exb0 += eadv;
      exb0 -= exb0 >= cblocks ? cblocks : 0;
      exb1 += eadv;
      exb1 -= exb1 >= cblocks ? cblocks : 0;
    }
  };

  // operand fragments of 32 rows: lane l holds row l % 32, K pieces 2 k + h (16 bytes each), k = 0..3. MXFP8 takes pieces
  // 2 kk and 2 kk + 1 as the MFMA's K bytes [16 h, + 16) and [32 + 16 h, + 16) of 64, INT8 one piece per MFMA
  struct Frag { v4i p[4]; };
  const int frow = lane & 31;
  int fo[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) fo[k] = frow * KC + (((2 * k + h) ^ ((frow >> 1) & 7)) << 4);
  const int fx0 = (BN + wm * MBW * BR) * KC, fw0 = wn * 64 * KC;
  auto piece = [&](const uint8_t* st, int base, int blk, int k) __attribute__((always_inline)) {
    return *reinterpret_cast<const v4i*>(st + base + fo[k] + blk * BR * KC);
  };
  // RAG: a tap's last segment holds Cin % 16 channels, then the next tap's bytes: zero in the weights
  int rag_cs = RAG ? h : 0;  // segment of piece 0 within its tap, walked like ld_cs
  const int rag_last = d.segs - 1, rag_words = RAG ? (a.Cin & 15) >> 2 : 4;
  auto mask_w = [&](Frag (&f)[2]) __attribute__((always_inline)) {
    if constexpr (RAG) {
      int cs = rag_cs;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool tail = cs == rag_last && rag_words != 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int keep = tail && e >= rag_words ? 0 : -1;
#pragma unroll
          for (int i = 0; i < 2; ++i) f[i].p[k][e] &= keep;
        }
        cs += 2;
        while (cs >= d.segs) cs -= d.segs;
      }
      rag_cs += 8 % d.segs;
      rag_cs -= rag_cs >= d.segs ? d.segs : 0;
    }
  };

  typedef typename std::conditional<KIND == KIND_MX, v16f, v16i>::type Acc;
  Acc acc[2][MBW];
#pragma unroll
  for (int j = 0; j < MBW; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

  // the MFMAs of x block j with operand set s, side(k) after the k-th of SL
  auto mfma_block = [&](int j, const Frag& x, const Frag (&w)[2], int s, auto&& side) __attribute__((always_inline)) {
    if constexpr (KIND == KIND_MX) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const v8i xv = __builtin_shufflevector(x.p[2 * kk], x.p[2 * kk + 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const v8i wv = __builtin_shufflevector(w[i].p[2 * kk], w[i].p[2 * kk + 1], 0, 1, 2, 3, 4, 5, 6, 7);
          // the weights' scale: byte 2 kk of the row's four, shifted by 8 h
          if (kk == 0)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv, xv, acc[i][j], 0, 0, 0, sw[s][i], 0, sx[s][0]);
          else
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv, xv, acc[i][j], 0, 0, 2, sw[s][i], 0, sx[s][1]);
          side(2 * kk + i);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[i].p[k], x.p[k], acc[i][j], 0, 0, 0);
          side(2 * k + i);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  };

  Frag xr[2], xt[L], wf[NST][2];
  // read n of the next step's first operands (8 weight pieces, then x block 0), from stage nxt into set s
  constexpr int FIRST_READS = 8 + 4;
  auto first_read = [&](const uint8_t* nxt, int s, int n) __attribute__((always_inline)) {
    if (n < 8)
      wf[s][n >> 2].p[n & 3] = piece(nxt, fw0, n >> 2, n & 3);
    else
      xr[0].p[n - 8] = piece(nxt, fx0, 0, n - 8);
  };
  // one K step from stage cur (operand set s, whose first reads are under way); the loads of NST - 1 steps on into `fill`;
  // then the barrier and, from stage nxt, the next step's first operands
  auto step = [&](const uint8_t* cur, const uint8_t* nxt, uint8_t* fill, int s) __attribute__((always_inline)) {
    const int s1 = (s + 1) % NST;
    if constexpr (KIND == KIND_MX) {
#pragma unroll
      for (int i = 0; i < 2; ++i) sw[s][i] = (int)((uint32_t)sw[s][i] >> (8 * h));
    }
    mask_w(wf[s]);
    ex_slot ^= BN;
    store_exponents();
    load_exponents();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < MAIN; ++j) {
      mfma_block(j, xr[j & 1], wf[s], s, [&](int k) __attribute__((always_inline)) {
        // the block(s) read during this one: the next, at the last main block all of the tail
        const int nread = j + 1 < MAIN ? 4 : 4 * L;
#pragma unroll
        for (int q = 0; q < 4 * L; ++q)
          if (q < nread && q * SL / nread == k) {
            Frag& f = j + 1 < MAIN ? xr[(j + 1) & 1] : xt[q >> 2];
            f.p[q & 3] = piece(cur, fx0, j + 1 + (q >> 2), q & 3);
          }
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
          if (c * SPAN / CHUNKS == j * SL + k) {
            issue(fill, c);
            if (c == CHUNKS - 1) load_step();
          }
      });
    }
    // the next step's stage landed: with two stages every load, with three all but this step's
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(NST == 3 ? CHUNKS + (KIND == KIND_MX ? 1 : 0) : 0));
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int j = 0; j < L; ++j)
      mfma_block(MAIN + j, xt[j], wf[s], s, [&](int k) __attribute__((always_inline)) {
        if (j == 0) {  // (past the last step: zeros, unused)
          constexpr int PER = 16 / SL;
#pragma unroll
          for (int n = PER * k; n < PER * k + PER; ++n)
            if (n < FIRST_READS) first_read(nxt, s1, n);
          if (k == SL - 1) read_scales(s1);
        }
      });
  };

  load_exponents();
  store_exponents();
  load_exponents();
  load_step();
#pragma unroll
  for (int i = 0; i < CHUNKS; ++i) issue(st0, i);
  if (NST == 3) {
    load_step();
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) issue(st1, i);
  }
  load_step();
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(NST == 3 ? CHUNKS : 0));
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int n = 0; n < FIRST_READS; ++n) first_read(st0, 0, n);
  read_scales(0);

  // whole rounds of the stages: a loop with one exit (with exits between the steps the compiler keeps several copies of
  // the accumulators and spills); the steps past the last multiply zeros
  for (int kt = 0; kt < d.nk; kt += NST) {
    if constexpr (NST == 3) {
      step(st0, st1, st2, 0);
      step(st1, st2, st0, 1);
      step(st2, st0, st1, 2);
    } else {
      step(st0, st1, st1, 0);
      step(st1, st0, st0, 1);
    }
  }

  // Epilogue, 64 pixels at a time: the wavefront's 64 channels staged in its own part of the (consumed) first stage and
  // written out as whole 128-byte (BF16) or 64-byte rows, once every load (of zeros, past the last step) and every read
  // of a stage is done.
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
  asm volatile("s_barrier" ::: "memory");
  constexpr int ESZ = OUT == OUT_BF16 ? 2 : 1, RB = 64 * ESZ, LPP = RB / 16, PPC = 64 / LPP;
  constexpr int CB = 8, NBE = 64 / CB, GB = 64 / BR;  // channel blocks of 8, row blocks per 64 pixels
  static_assert(STAGE >= 4 * 64 * RB, "the wavefronts' staging areas lie in the first stage");
  uint8_t* my_stage = st0 + wave * 64 * RB;
  const int out_nrec = __builtin_amdgcn_readfirstlane((int)((uint32_t)a.M * (uint32_t)a.out_ld * ESZ));
  const __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc(a.out, (short)0, out_nrec, 0x00020000);
  const float* ep_s = KIND == KIND_INT8 ? ep_scale : ep_bias;
  EpiChannels<NBE> ch = epi_channels<NBE, CB>(wn * 64, ep_s, ep_bias, ep_bias);
  if constexpr (OUT == OUT_E4M3) {  // E4M3 output scales 2^e, one per 32 channels
#pragma unroll
    for (int i = 0; i < NBE; ++i) {
      const int n = n0 + wn * 64 + i * CB;
      ch.osc[i] = exp2_int((int)a.out_expo[(n < a.Cout ? n : 0) >> 5]);
    }
  }
  const int mw = m0 + wm * MBW * BR, nw = n0 + wn * 64;
  auto group = [&](auto jc, auto res, auto staged) __attribute__((always_inline)) {
    constexpr int J0 = decltype(jc)::value, NJ = MBW - J0 < GB ? MBW - J0 : GB;
    constexpr bool RES = decltype(res)::value, STG = decltype(staged)::value;
    v4i ai[NBE][NJ];
    v4f af[NBE][NJ];
    int mrow[NJ], spix[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      spix[j] = j * BR + frow;
      const int m = mw + J0 * BR + spix[j];
      mrow[j] = m < a.M ? m : a.M;
#pragma unroll
      for (int i = 0; i < NBE; ++i) {
        const Acc& s = acc[i >> 2][J0 + j];
        const int q = 4 * (i & 3);
        if constexpr (KIND == KIND_MX)
          af[i][j] = v4f{s[q], s[q + 1], s[q + 2], s[q + 3]};
        else
          ai[i][j] = v4i{s[q], s[q + 1], s[q + 2], s[q + 3]};
      }
    }
    if constexpr (STG) {
      conv_epilogue_fast<KIND, OUT, NJ, NBE, 0, RES, RB, CB>(a, ai, af, mrow, nw, 0, ch, my_stage, spix);
      __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
      const int sl = lane % LPP;
      const bool cvalid = nw + sl * (16 / ESZ) < a.Cout;
#pragma unroll
      for (int c = 0; c < NJ * BR / PPC; ++c) {
        typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
        const int pl = c * PPC + lane / LPP;
        const u32x4 v = *reinterpret_cast<const u32x4*>(my_stage + pl * RB + ((sl ^ stage_swz(pl)) & (LPP - 1)) * 16);
        const int m = mw + J0 * BR + pl;
        const uint32_t off =
            cvalid && m < a.M ? ((uint32_t)m * (uint32_t)a.out_ld + (uint32_t)nw) * ESZ + sl * 16 : OOB;
        __builtin_amdgcn_raw_buffer_store_b128(v, orsrc, (int)off, 0, 0);
      }
      __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
    } else {
      conv_epilogue_fast<KIND, OUT, NJ, NBE, 0, RES, 0, CB, true>(a, ai, af, mrow, nw, 0, ch);
    }
  };
  auto groups = [&](auto res, auto staged) __attribute__((always_inline)) {
    group(std::integral_constant<int, 0>{}, res, staged);
    if constexpr (MBW > GB) group(std::integral_constant<int, GB>{}, res, staged);
    if constexpr (MBW > 2 * GB) group(std::integral_constant<int, 2 * GB>{}, res, staged);
    if constexpr (MBW > 3 * GB) group(std::integral_constant<int, 3 * GB>{}, res, staged);
    static_assert(MBW <= 4 * GB, "four groups");
  };
  using Y = std::integral_constant<bool, true>;
  using N = std::integral_constant<bool, false>;
  if (RAG && a.Cout % 16 != 0) {
    if (a.residual != nullptr) groups(Y{}, N{});
    else groups(N{}, N{});
  } else {
    if (a.residual != nullptr) groups(Y{}, Y{});
    else groups(N{}, Y{});
  }
}

}  // namespace fim
