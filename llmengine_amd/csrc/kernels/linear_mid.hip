// linear_mid.hip -- Q8_0 Linear for a serving batch or a short prompt (17-128
// tokens) on bf16 MFMA for gfx950, every weight byte read once per launch.
//
// y[m, n] = sum_k x[m, k] * d[n, k/32] * q[n, k]  (+ bias[n]), as
// cpu::sgemm_nt(const float*, const uint8_t*, ...) computes it
// (src/runtime/kernels/cpu_kernels.cpp:208-218).
//
// Below 64 tokens (PARTS 3) the activations are split exactly into three bf16 parts
// and the binary16 scale is applied in fp32 to each 32-wide block's sum, acc =
// fma(d, s, acc), the arithmetic of the MFMA decode.  From 64 tokens (PARTS 1) they
// are rounded once to bf16 and v = d * q is formed in fp32 and rounded once to bf16,
// the arithmetic of the prefill GEMM.
//
// Work split.  A workgroup of 4 x 2 waves owns 64 RG weight rows, all tokens and one
// K split.  K is walked in phases of 4 blocks: the phase's activations are loaded
// row by row, converted to MFMA fragments in LDS (two buffers, one barrier a phase)
// and shared by the 4 row waves; the 2 K waves take one block pair each and stream
// their RG row groups' quants straight into registers, two phases ahead.  The MFMA
// (16 x 16 x 32) takes the activations as its A operand and the weights as B, so a
// lane's accumulators belong to one weight row and need one scale.  The K waves add
// their sums in LDS; the K splits of a tile meet as in the MFMA decode (device-scope
// partials, completion wait, counter, read-back in split order: deterministic).
// The number of K splits follows K, the token tiles and, for vocabulary-sized weights
// and very long rows, the output's own row groups (linear_mid_pick).  Raw and tiled
// weights split alike; a fused launch below 64 tokens takes the splits that its outputs
// take alone, in a second launch where they differ, so that it adds in the same order.
//
// What bounds it: the vector ALUs (activation split, int8 -> bf16, scale FMAs; the
// MFMAs run beside them) and, on K = 4096, a fixed ~7 us of launch, first loads and
// split hand-off.  Loading the activations a lane a token (16 cache lines per
// quarter-wave) cost 0.9 us a phase at 64 tokens; deeper load rings (3-4 phases)
// measured 5-15% slower than 2, 8-block phases 3-10%.
//
// Measured (MI355X, rotated weights, us; before: 16-token chunks of the MFMA decode,
// the GEMM from 64 tokens):
//   tiled  M = 32 / 63 / 64:  12288 x 4096  33.7 / 66.5 / 27.2 -> 21.5 / 31.8 / GEMM
//                              4096 x 4096  16.5 / 32.9 / 18.2 -> 11.4 / 16.4 / 13.4
//                             4096 x 11008  38.9 / 77.0 / 29.1 -> 20.7 / 30.6 / 24.9
//                              896 x 4864   17.4 / 34.6 / 17.4 ->  9.1 / 12.6 / 11.2
//   raw                       12288 x 4096  41.6 / 79.8 / 29.9 -> 26.4 / 34.7 / GEMM
//                              4096 x 4096  21.3 / 41.5 / 18.8 -> 12.9 / 17.8 / 14.1
//   SwiGLU 2 x 11008 x 4096, tiled, M = 32 / 63:  61.6 / 122.8 -> 33.9 / 51.0
#include <algorithm>

#include "../launch.hpp"
#include "../q8_0_device.hpp"

namespace mle {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWN = 4;  // waves along the rows
constexpr int kWK = 2;  // waves along K
constexpr int kNT = 64 * kWN * kWK;

// The parts of 4 activations as packed bf16 (two dwords a part).  PARTS 3: hi / mid
// / lo by truncation, exact for every finite x (Inf carried in hi, NaN in all), as
// the MFMA decode splits them; PARTS 1: one rounding to nearest even.
template <int PARTS>
__device__ __forceinline__ void split_x(const f32x4 x, u32x2 (&out)[PARTS]) {
  const float v[4] = {x.x, x.y, x.z, x.w};
  if constexpr (PARTS == 1) {
    out[0].x = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[0], v[1]}, bf16x2));
    out[0].y = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2], v[3]}, bf16x2));
  } else {
    uint32_t rb[4], lb[4];
    bool finite = true;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float r = v[j] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v[j]) & 0xffff0000u);
      rb[j] = __builtin_bit_cast(uint32_t, r);
      lb[j] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, rb[j] & 0xffff0000u));
      finite &= !__builtin_amdgcn_class(v[j], 0x207);  // NaN, +-Inf
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite) != 0, 0)) {  // uniform
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float h = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v[j]) & 0xffff0000u);
        const float r = (v[j] == h) ? 0.0f : v[j] - h;
        rb[j] = __builtin_bit_cast(uint32_t, r);
        lb[j] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, rb[j] & 0xffff0000u));
      }
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      out[0][p] = top_halves(__builtin_bit_cast(uint32_t, v[2 * p]),
                             __builtin_bit_cast(uint32_t, v[2 * p + 1]));
      out[1][p] = top_halves(rb[2 * p], rb[2 * p + 1]);
      out[2][p] = top_halves(lb[2 * p], lb[2 * p + 1]);
    }
  }
}

// Output segments of a launch: segment i owns the 16-row groups
// [grp_end[i-1], grp_end[i]) (SwiGLU: segment 0's groups; seg[1] is the up
// weight of the same rows).
struct MidArgs {
  LinearSeg seg[3];
  unsigned grp_end[3];
  int count;
  int swiglu;
  unsigned tile0;  // first tile of this launch
};

constexpr int kPhaseBlocks = 4;  // K blocks per phase
constexpr int kStages = 2;       // phases of loads in flight

template <int TT, int PARTS, int RG, int LAYOUT>
__global__ __launch_bounds__(kNT, 2) void linear_mid_kernel(const float* __restrict__ x,
                                                            const MidArgs args, int M, int K,
                                                            int phases_per_split,
                                                            float* __restrict__ partials,
                                                            uint32_t* __restrict__ counters) {
  constexpr int CB = kPhaseBlocks, D = kStages;
  constexpr int BUF = CB * TT * PARTS * 1024;  // fragment bytes of one phase
  constexpr int PW = CB / (2 * kWK);  // block pairs per wave per phase
  static_assert(PW >= 1 && CB == 2 * kWK * PW, "whole pairs per wave");
  constexpr bool kTiled = LAYOUT == int(WeightLayout::kTiled);
  static_assert(CB == 4, "half a wave reads a token's 4 blocks");
  constexpr int RED = kWN * RG * TT * 1024;  // the wave reduction shares the area
  __shared__ __attribute__((aligned(16))) uint8_t frag[RED > 2 * BUF ? RED : 2 * BUF];
  constexpr int kRawBytes = 1024 + 64;  // one row group's pair of blocks
  __shared__ __attribute__((aligned(16))) uint8_t rawbuf[kTiled ? 16 : kWN * kWK * PW * RG * kRawBytes];
  __shared__ uint32_t arrived;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave / kWK, wk = wave % kWK;
  const int g = lane >> 4, r16 = lane & 15;
  const int KB = K / kBlockElems, KP = (KB + 1) >> 1;
  constexpr bool kPairs = PARTS == 3 && RG % 2 == 0;  // what a SwiGLU launch takes
  const bool swi = kPairs && args.swiglu != 0;
  const int ph0 = blockIdx.y * phases_per_split;
  // Blocks [ph0 CB, KBE) are this split's; blocks past KBE read as zero
  // activations and zero scales.
  const int KBE = min(KB, (ph0 + phases_per_split) * CB);
  const int steps = (KBE - ph0 * CB + CB - 1) / CB;
  const unsigned grp_total = args.count == 1 ? args.grp_end[0]
                             : args.count == 2 ? args.grp_end[1]
                                               : args.grp_end[2];
  const int RGO = swi ? RG / 2 : RG;  // output groups per wave
  const unsigned wgrp0 = ((args.tile0 + blockIdx.x) * kWN + wn) * RGO;
  auto group_of = [&](int rg) {  // output group of this wave's row group rg
    return wgrp0 + (unsigned)(swi ? (rg >= RG / 2 ? rg - RG / 2 : rg) : rg);
  };
  auto seg_of = [&](unsigned grp) {
    return (args.count > 1 && grp >= args.grp_end[0])
               ? ((args.count > 2 && grp >= args.grp_end[1]) ? 2 : 1)
               : 0;
  };
  auto grp_begin = [&](int si) {
    return si == 0 ? 0u : si == 1 ? args.grp_end[0] : args.grp_end[1];
  };

  // Activations of one phase: for token tile t, half h of wave w loads the phase's
  // 128 values of token 16 t + 2 w + h, 16 bytes a lane (512 contiguous bytes), and
  // writes their parts to the fragments, 8 bytes a lane.  Slot (g, r) of block b's
  // fragment (16 bytes: quarter g of token r) lies at g * 16 + (r ^ swz(b, g)), so
  // that one token's 16 slots of a phase spread over the banks.  Tokens past M and
  // blocks past KBE are zero.  (Loading whole fragments, a lane a token, costs a
  // cache line lookup per lane: 64 tokens' phases took 0.9 us each, MI355X.)
  auto swz = [](int b, int q) { return (q | (b << 2)) & 7; };
  const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(x, (uint32_t)((int64_t)M * K * 4));
  const int xr = 2 * wave + (lane >> 5), xb = (lane >> 3) & 3, xq = (lane >> 1) & 3;
  const uint32_t xslot = (uint32_t)((xq * 16 + (xr ^ swz(xb, xq))) * 16 + (lane & 1) * 8);
  struct XStage {
    f32x4 v[TT];
  };
  auto load_x = [&](int ph, XStage& st) {
    const bool live = ph * CB + xb < KBE;
    const uint32_t base = live ? (uint32_t)(xr * K + ph * (CB * kBlockElems)) * 4 + (lane & 31) * 16
                               : 0x80000000u;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      // A dead offset (2^31) stays past the buffer with the tile's offset added.
      uint32_t off = 16 * t + xr < M ? base + (uint32_t)(16 * t * K) * 4 : 0x80000000u;
      asm volatile("" : "+v"(off));  // one load for live and dead lanes, no branch
      st.v[t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 0, 0));
    }
  };
  auto split_phase = [&](int buf, const XStage& st) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      u32x2 parts[PARTS];
      split_x<PARTS>(st.v[t], parts);
#pragma unroll
      for (int p = 0; p < PARTS; ++p)
        *reinterpret_cast<u32x2*>(frag + buf * BUF + ((xb * TT + t) * PARTS + p) * 1024 + xslot) =
            parts[p];
    }
  };

  // Weights of this wave's row groups.
  // Groups past the last read group 0 (their sums are never written); pairs past
  // K re-read the last pair, with zero scales.
  const uint8_t* qptr[RG];  // tiled: the group's quant pieces; raw: this lane's row
  const uint8_t* sptr[RG];  // tiled: the group's scale pieces
#pragma unroll
  for (int rg = 0; rg < RG; ++rg) {
    const unsigned grp = group_of(rg);
    const bool live = grp < grp_total;
    const int si = swi ? (rg >= RG / 2 ? 1 : 0) : seg_of(grp);
    const uint8_t* w = si == 0 ? args.seg[0].w : si == 1 ? args.seg[1].w : args.seg[2].w;
    const int N = si == 0 ? args.seg[0].N : si == 1 ? args.seg[1].N : args.seg[2].N;
    const int64_t lg = live ? (int64_t)(grp - (swi ? 0u : grp_begin(si))) : 0;
    if constexpr (kTiled) {
      const int64_t G = ((int64_t)N + kTileRows - 1) / kTileRows;
      qptr[rg] = w + lg * KP * kTilePieceBytes;
      sptr[rg] = w + G * KP * kTilePieceBytes + lg * KP * kTileScaleBytes;
    } else {
      const int64_t n = min(lg * kTileRows + (lane >> 2), (int64_t)N - 1);
      qptr[rg] = w + n * (int64_t)KB * kBlockBytes;
    }
  }
  struct WStage {
    u32x4 q[PW][RG];
    uint32_t s[PW][RG];
  };
  auto load_w = [&](int ph, WStage& st) {
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const int pr = ph * (CB / 2) + wk * PW + j;
      if constexpr (kTiled) {
        const int pc = min(pr, KP - 1);
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          st.q[j][rg] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
              qptr[rg] + (int64_t)pc * kTilePieceBytes + (uint32_t)lane * 16));
          st.s[j][rg] = *reinterpret_cast<const uint32_t*>(
              sptr[rg] + (int64_t)pc * kTileScaleBytes + (uint32_t)r16 * 4);
        }
      } else {
        // Lane (row l / 4, block (l / 2) % 2 of the pair, half l % 2): 16 quants and
        // the block's scale; the 4 lanes of a row read 68 contiguous bytes.
        const uint32_t o = (uint32_t)min(2 * pr + ((lane >> 1) & 1), KB - 1) * kBlockBytes;
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          __builtin_memcpy(&st.q[j][rg],
                           __builtin_assume_aligned(qptr[rg] + o + 2 + 16 * (lane & 1), 2), 16);
          st.s[j][rg] = *reinterpret_cast<const uint16_t*>(qptr[rg] + o);
        }
      }
    }
  };

  f32x4 acc[RG][TT];
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[rg][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // One phase: (block, row group) products in sequence.  Product q's MFMAs are
  // interleaved with product q + 1's int8 -> bf16 conversion and product q - 1's
  // scale FMAs, so both pipes work; the fences keep the compiler from holding the
  // MFMA results of a whole phase.
  auto compute = [&](int ph, int buf, WStage& st) {
    if constexpr (!kTiled) {
      // Raw: the loaded halves of a row's two blocks pass through wave-private LDS
      // into the tiled layout's lanes (lane (g, r16): quarter g of both blocks).
      uint8_t* const rb = rawbuf + wave * (PW * RG * kRawBytes);
      const int row = lane >> 2, slot = lane & 3;
#pragma unroll
      for (int i = 0; i < PW * RG; ++i) {
        uint8_t* const b = rb + i * kRawBytes;
        *reinterpret_cast<u32x4*>(b + row * 64 + (slot ^ ((row >> 1) & 3)) * 16) = st.q[i / RG][i % RG];
        *reinterpret_cast<uint16_t*>(b + 1024 + row * 4 + (slot & 2)) = (uint16_t)st.s[i / RG][i % RG];
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < PW * RG; ++i) {
        const uint8_t* const b = rb + i * kRawBytes;
        const int sw = (r16 >> 1) & 3;
        const u32x2 lo = *reinterpret_cast<const u32x2*>(b + r16 * 64 + ((g >> 1) ^ sw) * 16 + (g & 1) * 8);
        const u32x2 hi = *reinterpret_cast<const u32x2*>(b + r16 * 64 + ((2 + (g >> 1)) ^ sw) * 16 + (g & 1) * 8);
        st.q[i / RG][i % RG] = u32x4{lo.x, lo.y, hi.x, hi.y};
        st.s[i / RG][i % RG] = *reinterpret_cast<const uint32_t*>(b + 1024 + r16 * 4);
      }
      __builtin_amdgcn_wave_barrier();  // the next phase's writes stay below these reads
    }
    constexpr int NQ = PW * 2 * RG;
    constexpr bool kFold = PARTS == 1;  // scale folded into the weight operand
    constexpr int VALU = kFold ? 22 : 15 + 4 * TT;
    constexpr int VPM = (VALU + PARTS * TT - 1) / (PARTS * TT);  // VALU per MFMA
    bf16x8 wf[2];
    float d[2];
    f32x4 s[2][kFold ? 1 : TT];
    bf16x8 xf[TT][PARTS];
    auto weight = [&](int q) {  // operand and scale of product q
      const int j = q / (2 * RG), h = q / RG % 2, rg = q % RG;
      const u32x4 w = st.q[j][rg];
      const uint32_t q0 = h ? w.z : w.x, q1 = h ? w.w : w.y;
      const uint32_t sb = h ? st.s[j][rg] >> 16 : st.s[j][rg];
      const bool live = ph * CB + (wk * PW + j) * 2 + h < KBE;  // uniform
      const float dd = scale_to_f32_fast(live ? sb & 0xffffu : 0u);
      if constexpr (kFold) {
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = __builtin_bit_cast(
              uint32_t, __builtin_convertvector(f32x2{dd * q_at(i < 2 ? q0 : q1, 2 * (i & 1)),
                                                      dd * q_at(i < 2 ? q0 : q1, 2 * (i & 1) + 1)},
                                                bf16x2));
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(o[i]));  // converted here
        wf[q & 1] = __builtin_bit_cast(bf16x8, o);
      } else {
        wf[q & 1] = quants_to_bf16(q0, q1);
        d[q & 1] = dd;
      }
    };
    __builtin_amdgcn_sched_barrier(0);
    weight(0);
#pragma unroll
    for (int q = 0; q <= NQ; ++q) {
      if (q < NQ) {
        if (q % RG == 0) {
          const int bl = (wk * PW + q / (2 * RG)) * 2 + q / RG % 2;  // block of the phase
          const uint8_t* fb = frag + buf * BUF + bl * TT * PARTS * 1024 +
                              (g * 16 + (r16 ^ swz(bl, g))) * 16;
#pragma unroll
          for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
              xf[t][p] = *reinterpret_cast<const bf16x8*>(fb + (t * PARTS + p) * 1024);
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kFold) {
#pragma unroll
          for (int t = 0; t < TT; ++t)
            acc[q % RG][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[t][0], wf[q & 1],
                                                                     acc[q % RG][t], 0, 0, 0);
        } else {
#pragma unroll
          for (int p = 0; p < PARTS; ++p)
#pragma unroll
            for (int t = 0; t < TT; ++t)
              s[q & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  xf[t][p], wf[q & 1], p == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[q & 1][t], 0, 0, 0);
        }
      }
      if (!kFold && q > 0) {
        const float dd = d[(q - 1) & 1];
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          const f32x4 v = s[(q - 1) & 1][kFold ? 0 : t];
          f32x4& a = acc[(q - 1) % RG][t];
          a.x = __builtin_fmaf(dd, v.x, a.x);
          a.y = __builtin_fmaf(dd, v.y, a.y);
          a.z = __builtin_fmaf(dd, v.z, a.z);
          a.w = __builtin_fmaf(dd, v.w, a.w);
          asm volatile("" : "+v"(a));  // the sum is formed here, not sunk past the phase
        }
      }
      if (q + 1 < NQ) weight(q + 1);
      if (q < NQ) {
#pragma unroll
        for (int i = 0; i < PARTS * TT; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);  // VALU
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Step i (phase ph0 + i) splits the next phase's activations into the other
  // buffer, multiplies its own, and refills the register stages it emptied, D
  // phases ahead.  A step issues its loads in the order X(i + 1 + D), W(i + D), so
  // the wait for X(i + 1) leaves the weights of D - 1 later phases in flight.
  XStage xs[D];
  WStage ws[D];
  load_x(ph0, xs[0]);
#pragma unroll
  for (int i = 0; i + 1 < D; ++i) {
    load_x(ph0 + i + 1, xs[i + 1]);
    __builtin_amdgcn_sched_barrier(0);
    load_w(ph0 + i, ws[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  split_phase(0, xs[0]);
  __builtin_amdgcn_sched_barrier(0);
  load_x(ph0 + D, xs[0]);
  __builtin_amdgcn_sched_barrier(0);
  load_w(ph0 + D - 1, ws[D - 1]);
  __syncthreads();
  int buf = 0;
  for (int i = 0;;) {
    bool done = false;
#pragma unroll
    for (int u = 0; u < D; ++u) {
      split_phase(buf ^ 1, xs[(u + 1) % D]);
      load_x(ph0 + i + 1 + D, xs[(u + 1) % D]);
      compute(ph0 + i, buf, ws[u]);
      load_w(ph0 + i + D, ws[u]);
      __syncthreads();
      buf ^= 1;
      if (++i == steps) {
        done = true;
        break;
      }
    }
    if (done) break;
  }

  // The K waves add their sums in LDS.
  f32x4* red = reinterpret_cast<f32x4*>(frag);
  if (wk == 1) {
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int t = 0; t < TT; ++t) red[((wn * RG + rg) * TT + t) * 64 + lane] = acc[rg][t];
  }
  __syncthreads();
  // Output column of an output group's row r16: its pointer and bias.
  struct Out {
    float* y;  // y + n, or null past the last row
    int64_t N;
    float bias;
    bool has_bias;
  };
  auto out_of = [&](unsigned grp) {
    const int si = swi ? 0 : seg_of(grp);
    float* y = si == 0 ? args.seg[0].y : si == 1 ? args.seg[1].y : args.seg[2].y;
    const int N = si == 0 ? args.seg[0].N : si == 1 ? args.seg[1].N : args.seg[2].N;
    const void* bias = si == 0 ? args.seg[0].bias : si == 1 ? args.seg[1].bias : args.seg[2].bias;
    const int bias_bf16 =
        si == 0 ? args.seg[0].bias_bf16 : si == 1 ? args.seg[1].bias_bf16 : args.seg[2].bias_bf16;
    const int64_t n = (int64_t)(grp - (swi ? 0u : grp_begin(si))) * kTileRows + r16;
    Out o;
    const bool live = grp < grp_total && n < N;
    o.y = live ? y + n : nullptr;
    o.N = N;
    o.has_bias = bias != nullptr && !swi;
    o.bias = o.has_bias && live ? bias_at(bias, bias_bf16, n) : 0.0f;
    return o;
  };
  auto write4 = [&](const Out& o, int t, f32x4 v) {  // tokens 16 t + 4 g .. + 3
    if (o.y == nullptr) return;
    if (o.has_bias) v += f32x4{o.bias, o.bias, o.bias, o.bias};
    const int m = 16 * t + 4 * g;
    float* p = o.y + m * o.N;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (m + e < M) p[e * o.N] = v[e];
  };
  auto silu4 = [&](f32x4 a, f32x4 b) {
    return f32x4{silu_mul(a.x, b.x), silu_mul(a.y, b.y), silu_mul(a.z, b.z), silu_mul(a.w, b.w)};
  };
  constexpr int SC1 = 16;  // cache-policy bit: device scope
  const unsigned nspl = gridDim.y;
  constexpr uint32_t REGION = kWN * RG * TT * 1024;  // bytes of one workgroup's partials
  if (nspl == 1) {
    if (wk != 0) return;
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int t = 0; t < TT; ++t) acc[rg][t] += red[((wn * RG + rg) * TT + t) * 64 + lane];
    if (swi) {
      if constexpr (kPairs) {
#pragma unroll
        for (int rg = 0; rg < RG / 2; ++rg) {
          const Out o = out_of(group_of(rg));
#pragma unroll
          for (int t = 0; t < TT; ++t) write4(o, t, silu4(acc[rg][t], acc[rg + RG / 2][t]));
        }
      }
    } else {
#pragma unroll
      for (int rg = 0; rg < RG; ++rg) {
        const Out o = out_of(group_of(rg));
#pragma unroll
        for (int t = 0; t < TT; ++t) write4(o, t, acc[rg][t]);
      }
    }
    return;
  }

  // Split K: partials by device-scope stores, their completion, the tile's
  // counter; the last workgroup resets the counter and adds the splits in order.
  const __amdgpu_buffer_rsrc_t prs =
      buffer_rsrc(reinterpret_cast<uint8_t*>(partials) + (int64_t)blockIdx.x * nspl * REGION, nspl * REGION);
  if (wk == 0) {
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const int slot = (wn * RG + rg) * TT + t;
        acc[rg][t] += red[slot * 64 + lane];
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[rg][t]), prs,
                                               blockIdx.y * REGION + (uint32_t)(slot * 64 + lane) * 16,
                                               0, SC1);
      }
  }
  uint32_t* const counter = counters + (size_t)blockIdx.x * kCounterStride;
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);  // every partial has reached the coherence point
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  if (tid == 0)
    arrived = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  if (arrived != nspl - 1) return;
  if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // Item i = (output group, token tile) goes to K wave i % kWK; all of a wave's
  // items of four splits are in flight at once.
  constexpr int IT = kPairs ? 2 * ((RG / 2 * TT + 1) / 2) : (RG * TT + 1) / 2;
  static_assert(kWK == 2, "two K waves share the items");
  const int items = RGO * TT;
  f32x4 sum[IT];
#pragma unroll
  for (int u = 0; u < IT; ++u) sum[u] = f32x4{0.f, 0.f, 0.f, 0.f};
  // SwiGLU: load u is item u / 2 of this wave, its gate (even u) or up (odd u) sum.
  auto slot_of = [&](int u) {
    const int i = swi ? (u >> 1) * kWK + wk : u * kWK + wk;
    if (i >= items) return -1;
    const int rg = i / TT, t = i % TT;
    return (wn * RG + rg + (swi && (u & 1) ? RG / 2 : 0)) * TT + t;
  };
  for (unsigned sp = 0; sp < nspl; sp += 4) {
    f32x4 v[4][IT];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < IT; ++u) {
        const int slot = slot_of(u);
        v[j][u] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       prs,
                       sp + j < nspl && slot >= 0
                           ? (sp + j) * REGION + (uint32_t)(slot * 64 + lane) * 16
                           : 0x80000000u,
                       0, SC1));
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < IT; ++u) sum[u] += v[j][u];
  }
  if (swi) {
    if constexpr (kPairs) {
#pragma unroll
      for (int u = 0; u + 1 < IT; u += 2) {
        const int i = (u >> 1) * kWK + wk;
        if (i < items) write4(out_of(group_of(i / TT)), i % TT, silu4(sum[u], sum[u + 1]));
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < IT; ++u) {
      const int i = u * kWK + wk;
      if (i < items) write4(out_of(group_of(i / TT)), i % TT, sum[u]);
    }
  }
}

MidArgs mid_args(const LinearSegs& s) {
  MidArgs a{};
  a.swiglu = s.mode == Epilogue::kSwiGLU ? 1 : 0;
  unsigned end = 0;
  for (int i = 0; i < 3; ++i) {
    a.seg[i] = s.seg[i];
    if (i < (a.swiglu ? 1 : s.count)) end += (unsigned)((s.seg[i].N + kTileRows - 1) / kTileRows);
    a.grp_end[i] = end;
  }
  if (a.swiglu) a.seg[1].N = s.seg[0].N;
  a.count = a.swiglu ? 1 : s.count;
  return a;
}

// Row groups per wave: all that fit the registers without spills below 64 tokens, from 64
// on all that the pick's bounds on the row groups ask for.
constexpr int max_rg(int tt, int parts) { return parts == 3 ? 4 : tt <= 6 ? 2 : 1; }

struct MidGrid {
  unsigned tiles, splits;
  unsigned tiles_per_launch;
  int phases_per_split;
  MidArgs args;
};
// Phases of a K split, and the K splits a launch makes of them (fewer than asked for where
// whole phases do not fill them).
int mid_phases_per_split(const MidConfig& c, int K) {
  const int phases = (K / kBlockElems + kPhaseBlocks - 1) / kPhaseBlocks;
  return (phases + c.splits - 1) / c.splits;
}
int mid_splits(const MidConfig& c, int K) {
  const int phases = (K / kBlockElems + kPhaseBlocks - 1) / kPhaseBlocks;
  const int per = mid_phases_per_split(c, K);
  return (phases + per - 1) / per;
}

MidGrid mid_grid(const MidConfig& c, const LinearSegs& s, int K) {
  MidGrid gr{};
  gr.args = mid_args(s);
  const unsigned groups = gr.args.grp_end[gr.args.count - 1];
  const unsigned per = kWN * (gr.args.swiglu ? c.rg / 2 : c.rg);
  gr.tiles = (groups + per - 1) / per;
  gr.tiles_per_launch = c.tiles_per_launch > 0 ? std::min(gr.tiles, (unsigned)c.tiles_per_launch)
                                               : gr.tiles;
  gr.phases_per_split = mid_phases_per_split(c, K);
  gr.splits = (unsigned)mid_splits(c, K);
  return gr;
}

template <int TT, int PARTS, int RG>
hipError_t launch_mid_k(MidGrid gr, WeightLayout layout, const float* x, int M, int K,
                        const SplitKWorkspace& ws, hipStream_t stream) {
  const dim3 block(kNT);
  for (unsigned t0 = 0; t0 < gr.tiles; t0 += gr.tiles_per_launch) {
    const dim3 grid(std::min(gr.tiles - t0, gr.tiles_per_launch), gr.splits);
    gr.args.tile0 = t0;
    if (layout == WeightLayout::kTiled)
      hipLaunchKernelGGL((linear_mid_kernel<TT, PARTS, RG, int(WeightLayout::kTiled)>), grid,
                         block, 0, stream, x, gr.args, M, K, gr.phases_per_split, ws.partials,
                         ws.counters);
    else
      hipLaunchKernelGGL((linear_mid_kernel<TT, PARTS, RG, int(WeightLayout::kRaw)>), grid, block,
                         0, stream, x, gr.args, M, K, gr.phases_per_split, ws.partials,
                         ws.counters);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

template <int TT, int PARTS>
hipError_t launch_mid_rg(const MidConfig& c, const MidGrid& gr, WeightLayout layout,
                         const float* x, int M, int K, const SplitKWorkspace& ws,
                         hipStream_t stream) {
  switch (c.rg) {
    case 1: return launch_mid_k<TT, PARTS, 1>(gr, layout, x, M, K, ws, stream);
    case 2:
      if constexpr (max_rg(TT, PARTS) >= 2)
        return launch_mid_k<TT, PARTS, 2>(gr, layout, x, M, K, ws, stream);
      break;
    case 3:
      if constexpr (max_rg(TT, PARTS) >= 3)
        return launch_mid_k<TT, PARTS, 3>(gr, layout, x, M, K, ws, stream);
      break;
    case 4:
      if constexpr (max_rg(TT, PARTS) >= 4)
        return launch_mid_k<TT, PARTS, 4>(gr, layout, x, M, K, ws, stream);
      break;
  }
  return hipErrorInvalidValue;
}

}  // namespace

// Whether a launch takes this kernel, and its shape (tt == 0: it does not).
//
// Tokens: 17-63 always (1.2-2.7 times as fast as 16-token chunks on every shape
// measured, raw and tiled).  Not 9-16, where one launch of the decode reads the weights
// once as well: rows of 672-1024 elements take 0.8x its time here on up to 256 row groups,
// but up to 1.5x on 400 and more (16384 x 896 raw at 16 tokens: 12.2 us vs 9.0), and the
// kernel cannot follow the groups, since a fused launch has to keep the bits of its outputs'
// own launches.  From 64 tokens the GEMM reuses each dequantised weight more:
//   * of rows of up to 4096 elements it keeps launches of more than 512 row groups up to 80
//     tokens (12288 x 4096 at 77: 28.0 vs 27.8 us), 288 up to 96 (4864 x 896 from 84 tokens
//     on 1.04-1.07x its time here, 4864 x 4096 tiled 1.04) and 256 beyond;
//   * longer rows' 8 K splits fill the GPU from fewer groups: it keeps more than 256 up to
//     80 tokens (4864 x 5120 at 80 1.08x its time here, 8192 x 11008 1.07-1.17x), 128 up to
//     96 (4096 x 6400 1.05-1.09x, 4864 x 11008 1.42x) and 64 beyond (4096 x 11008 at 128 34.9
//     vs 31.6);
//   * and SwiGLU pairs (11008 x 4096 at 64: 40.5 vs 39.8).
//
// K splits: about 32 blocks each, none up to 16 blocks, where the 16-token decode needs no
// workspace either (8 splits past 4096 elements: 896 x 4864 at 32 tokens 9.1 us vs 12.0
// with 4; 7 at three token tiles, as fast as 8, whose partials stay within the 16-token
// decode's); one split for weights whose rows alone fill the GPU several times over (3072
// groups).  Rows past 11264 elements of few groups: twice as many while the workgroups are
// at most one a CU and a split keeps 16 blocks (32 x 65536 raw at 18 tokens 54.3 us with 8,
// 16.5 with 64, 23.1 in two 16-token launches).  Shorter rows keep one count for every number of
// groups, so that a fused launch and its outputs' own split alike (run_mid forms the launch
// of outputs that do not by groups that do).  A SwiGLU pair, which no single launch has to
// match, doubles them from any K while a split keeps 12 blocks (24 past 32 splits), and
// halves them until its grid fits the CUs.
// Row groups per wave (which no bits depend on).
//   * Up to two token tiles: the fewest groups of one to three that keep the grid within
//     one workgroup a CU (304 with one group, 4864 x 896 runs as well so as with two, and
//     with two in splits of up to 3 phases), else two, which are resident twice a CU and
//     hide each other's start.  288 workgroups leave a last round of 32 (9216 x 5120 raw at
//     17 tokens 39.1 us, 27.6 with three groups), and four groups in two rounds of 384 or 512
//     take 1.2-1.5x the time of two (49136 x 768 raw 32.7 -> 24.5, 50880 x 4096 raw 124 -> 78).
//   * More tiles are resident once a CU.  Splits of up to 3 phases are over before a second
//     round costs much: the fewest groups within 304 workgroups (of the splits asked for).
//     Longer ones: the fewest rounds (a second one of up to 64 workgroups counts 0.6), a
//     workgroup costing its groups and one more for the activations (13824 x 4096 at 48
//     tokens: 4 groups in 216 workgroups 0.51x the chunks' time, 3 in 288 0.71x; 4864 x
//     1024 at 33: 1 in 304 0.46x, 2 in 152 0.55x).
static int mid_row_groups(const MidConfig& c, int64_t G, int K) {
  const int rg_max = max_rg(c.tt, c.parts);
  const int splits = mid_splits(c, K);
  const bool brief = mid_phases_per_split(c, K) <= 3;
  auto grid = [&](int rg) { return (G + kWN * rg - 1) / (kWN * rg) * splits; };
  if (c.tt <= 2) {
    for (int rg = 1; rg <= 3; ++rg)
      if (grid(rg) <= (rg == 1 || (rg == 2 && brief) ? 304 : 256)) return rg;
    return 2;
  }
  int best = 1;
  if (brief) {
    while (best < rg_max && (G + kWN * best - 1) / (kWN * best) * c.splits > 304) ++best;
    return best;
  }
  auto cost = [&](int rg) {  // in fifths of a round
    const int64_t wgs = grid(rg);
    return (wgs > 256 && wgs <= 320 ? 8 : (wgs + 255) / 256 * 5) * (rg + 1);
  };
  for (int rg = 2; rg <= rg_max; ++rg)
    if (cost(rg) <= cost(best)) best = rg;
  return best;
}

MidConfig linear_mid_pick(int M, const LinearSegs& s, int K, int splits) {
  MidConfig c;
  if (M < 17 || M > 128 || s.layout == WeightLayout::kKN) return c;
  const MidArgs a = mid_args(s);
  const bool swi = a.swiglu != 0;
  const int64_t G = a.grp_end[a.count - 1];  // output row groups
  const int KB = K / kBlockElems;
  if (M >= 64) {
    const int most = K <= 4096 ? (M <= 80 ? 512 : M <= 96 ? 288 : 256) : M <= 80 ? 256 : M <= 96 ? 128 : 64;
    if (swi || G > most) return c;
  }
  c.parts = M < 64 ? 3 : 1;
  c.tt = M < 64 ? (M + 15) / 16 : M <= 64 ? 4 : M <= 80 ? 5 : M <= 96 ? 6 : 8;
  auto grid = [&](int rg) { return (G + kWN * rg - 1) / (kWN * rg) * c.splits; };
  c.splits = G >= 3072 || KB <= 16 ? 1 : KB <= 128 ? 4 : c.tt == 3 ? 7 : 8;
  if (c.parts == 3 && c.splits > 1 && (swi || KB > 352)) {
    const int least = swi ? 12 : 16;
    while (grid(1) * 2 <= 256 && c.splits <= 32 &&
           KB >= 2 * c.splits * (swi && c.splits >= 32 ? 24 : least))
      c.splits *= 2;
  }
  if (splits > 0) c.splits = splits;
  if (swi) {
    c.rg = grid(1) <= 304 ? 2 : 4;  // half of each weight
    while (c.splits > 1 && grid(c.rg / 2) > 304) c.splits /= 2;
  } else {
    c.rg = mid_row_groups(c, G, K);
  }
  return c;
}

// 32-bit offsets of the activations.
bool linear_mid_fits(int M, int K) { return (int64_t)M * K * 4 < (int64_t(1) << 31); }

SplitKNeed linear_mid_workspace(const MidConfig& c, const LinearSegs& s, int K) {
  const MidGrid gr = mid_grid(c, s, K);
  SplitKNeed need;
  need.splits = (int)gr.splits;
  if (gr.splits > 1) {
    need.partial_floats = (size_t)gr.tiles_per_launch * gr.splits * kWN * c.rg * c.tt * 256;
    need.counters = (size_t)gr.tiles_per_launch * kCounterStride;
  }
  return need;
}

hipError_t launch_linear_mid(const MidConfig& c, const float* x, const LinearSegs& s, int M, int K,
                             const SplitKWorkspace& ws, hipStream_t stream) {
  if (M > 16 * c.tt) return hipErrorInvalidValue;
  const MidGrid gr = mid_grid(c, s, K);
  if (c.parts == 3) {
    switch (c.tt) {
      case 2: return launch_mid_rg<2, 3>(c, gr, s.layout, x, M, K, ws, stream);
      case 3: return launch_mid_rg<3, 3>(c, gr, s.layout, x, M, K, ws, stream);
      case 4: return launch_mid_rg<4, 3>(c, gr, s.layout, x, M, K, ws, stream);
    }
  } else {
    switch (c.tt) {
      case 4: return launch_mid_rg<4, 1>(c, gr, s.layout, x, M, K, ws, stream);
      case 5: return launch_mid_rg<5, 1>(c, gr, s.layout, x, M, K, ws, stream);
      case 6: return launch_mid_rg<6, 1>(c, gr, s.layout, x, M, K, ws, stream);
      case 8: return launch_mid_rg<8, 1>(c, gr, s.layout, x, M, K, ws, stream);
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace mle
