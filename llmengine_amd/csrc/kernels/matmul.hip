// matmul.hip -- Q8_0 MatMul C[M,N] = A[M,K] . B[K,N] for gfx950.
//
// B is one Q8_0 stream in row-major [K, N] order, so element (k, n) is flat
// index k*N + n and blocks run along N (reference
// src/runtime/kernels/cpu_kernels.cpp:116-130, cuda_kernels.cu:296-331).  The
// reference forms v = d * q in fp32 and sums a * v.  The half-block kernel does so in
// fp32 FMA chains; the MFMA kernel rounds a * d to fp32 instead (q is exact beside it)
// and sums on the matrix cores.  Both split the K sum into fixed pieces added in a fixed
// order, so the result is deterministic and within fp32 rounding of the reference's
// sequential sum (relative L2 ~1e-7), as the reference's own device kernel is
// (it splits K over 8 warps and adds their partials).
//
// Kernels (from 64 rows of A, 16-byte aligned, the MatMul runs the bf16 MFMA GEMM
// instead):
//   * one or two rows of A, and three on few columns of long K: the half-block kernel
//     below, lanes reading 16-byte pieces of whole blocks along a B row, fp32 FMAs;
//   * more: the MFMA kernel below, B read once per tile of up to 64 rows.
// Where column tiles alone leave the GPU's 256 CUs short of work, K is spread over S
// workgroups per tile.  Up to 8 rows of A they meet through a tile counter (a second
// launch costs the host as much as such a call takes: 4 x 1632 x 2272 10.6 us a call with
// it, 7.8 without); for more rows the MFMA kernel writes [S][M][N] partials, which a second
// launch adds in fixed runs of splits.
#include "../launch.hpp"
#include "../q8_0_device.hpp"

namespace mle {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int v2i __attribute__((ext_vector_type(2)));

// MFMA kernel (3 and more rows of A, up to 64 a workgroup), fp32-exact operands.
//
// A block of B holds 32 columns of one k, so its scale cannot leave the K sum; it goes
// into the activations instead: for one 32-column block, c[m, n] = sum_k (a[m, k]
// d[k]) q[k, n].  The fp32 product a * d (one rounding, as the FMA chain rounds each
// sum) is split exactly into three bf16 parts by truncation, the quants are exact in
// bf16, and v_mfma_f32_16x16x32_bf16 forms the products exactly with fp32 sums.  The
// matrix cores take parts below 2^-126 as zero, so the sums are formed 2^40 times too
// large (exact) and brought back at the end: what is lost stays below fp32's smallest
// value (unscaled, activations of 1e-36 gave a relative error of 4e-3, of 1e-40 zeros).
// From the first K step of a wave that holds a non-finite scale or an activation past
// 2^40 (whose scaled sums could overflow) it sums by fp32 FMAs instead, unscaled, v = d *
// q first, as the reference does.
//
// A workgroup owns NBW 32-column blocks and one K split; its 8 waves take 32-row K
// steps in turn and add their sums in LDS.  Per step a wave reads its 32 B rows as
// whole half blocks (2 NBW lanes a row, 34 NBW contiguous bytes) and its 16 TT x 32
// activations (8 lanes a row), passes both through wave-private LDS, and takes the
// quants back transposed, 8 consecutive k of one column a lane, with ds_read_b64_tr_b8.
// The next step's loads are in flight while one is multiplied.
//
// Bound by the vector ALUs (8 products, the split of 8 values and 16 int8 -> bf16
// conversions a lane for 6 TT MFMAs).  Measured (MI355X, rotated B, us, against fp32
// FMAs on up to 8 rows at a time): 4096 x 4096 at M = 4 / 8 / 16 / 63 14.1 / 27.4 /
// 40.7 / 121 -> 11.7 / 11.5 / 12.4 / 21.6; 11008 x 4096 21.2 / 38.7 / 103 / 371 -> 21.1
// / 20.7 / 22.6 / 51.4; [896, 151936] 49.3 / 90.6 / 293 / 1029 -> 43.9 / 43.7 / 45.1 /
// 147.  256-column wave tiles (one workgroup a CU) were 1.1-1.5x slower.
constexpr int kMfWaves = 8;
constexpr int kMfNT = 64 * kMfWaves;

struct MfGrid {
  unsigned tiles, splits, row_tiles;
  int tt, nbw, steps_per_split;
};

// Whether the K splits meet inside the launch (else in a second one).
bool mf_handoff(int M) { return M <= 8; }

MfGrid mf_grid(int M, int N, int K) {
  MfGrid g;
  g.tt = (M + 15) / 16;
  if (g.tt > 4) g.tt = 4;
  g.nbw = g.tt <= 2 ? 4 : 2;
  g.tiles = (unsigned)((N / kBlockElems + g.nbw - 1) / g.nbw);
  // More than 64 rows (an A that is not 16-byte aligned, or past the GEMM's offsets): all
  // row tiles in one launch.  A launch a tile took 4055 x 224 x 160 418 us against 28 on
  // fp32 FMAs; in one it takes 7.4 (2048 x 4096 x 4096 704 -> 450, MI355X).
  g.row_tiles = (unsigned)((M + 16 * g.tt - 1) / (16 * g.tt));
  const int steps = K / kBlockElems;
  // At most two workgroups a CU at one token tile (126 registers), else one; each wave
  // at least one K step.  Rounded down: a third round for a few workgroups costs more
  // (11008 x 4096 at 16 rows: 22.6 us with 5 splits, 25.7 with 6).
  int s = (int)((g.tt == 1 ? 512 : 256) / ((int64_t)g.tiles * g.row_tiles));
  if (s > steps / kMfWaves) s = steps / kMfWaves;
  // A tile's last workgroup adds its splits alone: few columns of very long K are faster
  // with fewer (4 x 480 x 32608 18.9 us with 127, 15.2 with 48; 16 take 21).
  if (mf_handoff(M) && s > 48) s = 48;
  // Many rows over few columns stay without a workspace, so that a capture that reserved
  // none is accepted: from 512 tiles of 8 rows x 256 columns on, as many as fill the GPU
  // with one split on the fp32 kernel that took these calls first.
  if (M > 64 && (int64_t)((N + 255) / 256) * ((M + 7) / 8) >= 512) s = 1;
  if (s < 1) s = 1;
  g.steps_per_split = (steps + s - 1) / s;
  g.splits = (unsigned)((steps + g.steps_per_split - 1) / g.steps_per_split);
  return g;
}

template <int TT, int NBW>
__global__ __launch_bounds__(kMfNT, 2) void matmul_q8_0_mfma_kernel(
    const float* __restrict__ a, const uint8_t* __restrict__ b, float* __restrict__ out, int M,
    int N, int K, int steps_per_split, float* __restrict__ partials,
    uint32_t* __restrict__ counters) {
  constexpr int QS = NBW * 32 + 16;    // LDS bytes of a B row (16-byte pieces, banks spread)
  constexpr int AS = 36;               // LDS floats of an activation row
  constexpr int LPR = 2 * NBW;         // lanes a B row
  constexpr int RPI = 64 / LPR;        // B rows per load instruction
  constexpr int BL = 32 / RPI;         // B load instructions per step
  constexpr int Q_BYTES = 32 * QS, S_BYTES = NBW * 64, A_BYTES = 16 * TT * AS * 4;
  constexpr int WAVE_BYTES = Q_BYTES + S_BYTES + A_BYTES;
  constexpr int SLOTS = 2 * NBW * TT;  // 16 x 16 output tiles
  constexpr int RED_BYTES = 4 * SLOTS * 1024;
  constexpr int LDS = kMfWaves * WAVE_BYTES > RED_BYTES ? kMfWaves * WAVE_BYTES : RED_BYTES;
  static_assert(WAVE_BYTES % 16 == 0, "16-byte wave areas");
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];
  __shared__ uint32_t arrived;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int64_t NB = N / kBlockElems;
  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous run of (split, column
  // tile) pairs, so the 128-byte lines that neighbouring tiles share are fetched into
  // one L2 (0.93-0.97x).
  const unsigned total = gridDim.x * gridDim.y, lin = blockIdx.y * gridDim.x + blockIdx.x;
  const unsigned q8 = total / 8, r8 = total % 8, xcd = lin % 8, ix = lin / 8;
  const unsigned nid = xcd * q8 + min(xcd, r8) + ix;
  const unsigned by = nid / gridDim.x, bx = nid % gridDim.x;
  const int64_t blk0 = (int64_t)bx * NBW;
  const int s0 = by * steps_per_split;
  const int s1 = min(s0 + steps_per_split, K / kBlockElems);
  uint8_t* const qs = lds + wave * WAVE_BYTES;
  uint16_t* const ss = reinterpret_cast<uint16_t*>(qs + Q_BYTES);
  float* const as = reinterpret_cast<float*>(qs + Q_BYTES + S_BYTES);

  // This lane's half block of a B row (columns past N re-read the last block) and its
  // 4 activations of a row (rows past M re-read row M - 1); neither is ever stored.
  const int brow = lane / LPR, bcol = lane % LPR;
  const uint8_t* const bp = b + ((int64_t)brow * NB + min(blk0 + (bcol >> 1), NB - 1)) * kBlockBytes;
  const int arow = lane >> 3, acol = lane & 7;
  const int m0 = blockIdx.z * 16 * TT;
  const float* ap[2 * TT];
#pragma unroll
  for (int i = 0; i < 2 * TT; ++i) ap[i] = a + (int64_t)min(m0 + arow + 8 * i, M - 1) * K + 4 * acol;
  struct Stage {
    u32x4 q[BL];
    uint16_t s[BL];
    f32x4 x[2 * TT];
  };
  auto load = [&](int step, Stage& st) {
    const uint8_t* p = bp + (int64_t)step * kBlockElems * NB * kBlockBytes;
#pragma unroll
    for (int i = 0; i < BL; ++i) {
      const uint8_t* r = p + (int64_t)(i * RPI) * NB * kBlockBytes;
      __builtin_memcpy(&st.q[i], __builtin_assume_aligned(r + 2 + 16 * (bcol & 1), 2), 16);
      st.s[i] = *reinterpret_cast<const uint16_t*>(r);
    }
#pragma unroll
    for (int i = 0; i < 2 * TT; ++i)
      __builtin_memcpy(&st.x[i], __builtin_assume_aligned(ap[i] + (int64_t)step * kBlockElems, 4), 16);
  };

  f32x4 acc[NBW][2][TT];
#pragma unroll
  for (int n = 0; n < NBW; ++n)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < TT; ++t) acc[n][j][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  bool scaled = true;  // uniform: the sums are kUp times too large
  constexpr float kUp = 0x1p40f;
  auto unscale = [&] {
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) acc[i / (2 * TT)][i / TT % 2][i % TT] *= 1.0f / kUp;
  };
  // Registers -> wave-private LDS; the first step that is not all finite and small ends
  // the scaled sums.
  auto stage = [&](const Stage& st) {
    bool fine = true;
#pragma unroll
    for (int i = 0; i < BL; ++i) {
      const int row = i * RPI + brow;
      *reinterpret_cast<u32x4*>(qs + row * QS + bcol * 16) = st.q[i];
      ss[(bcol >> 1) * 32 + row] = st.s[i];
      fine &= (st.s[i] & 0x7c00u) != 0x7c00u;
    }
#pragma unroll
    for (int i = 0; i < 2 * TT; ++i) {
      *reinterpret_cast<f32x4*>(as + (arow + 8 * i) * AS + 4 * acol) = st.x[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) fine &= __builtin_fabsf(st.x[i][e]) < 0x1p40f;  // false on NaN
    }
    if (scaled && __builtin_amdgcn_ballot_w64(!fine) != 0) {
      scaled = false;
      unscale();
    }
  };
  auto multiply = [&] {
    float x[TT][8];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const f32x4 lo = *reinterpret_cast<const f32x4*>(as + (16 * t + r16) * AS + 8 * g);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(as + (16 * t + r16) * AS + 8 * g + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[t][e] = lo[e];
        x[t][4 + e] = hi[e];
      }
    }
#pragma unroll
    for (int n = 0; n < NBW; ++n) {
      const u32x4 sc = *reinterpret_cast<const u32x4*>(ss + n * 32 + 8 * g);
      float d[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)  // one v_fma_mix_f32 each: the scaling is free
        d[e] = __builtin_fmaf(
            scale_to_f32_fast(e & 1 ? sc[e >> 1] >> 16 : sc[e >> 1] & 0xffffu), kUp, 0.0f);
      bf16x8 wf[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        typedef __attribute__((address_space(3))) v2i lds_v2i;
        const v2i q = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (lds_v2i*)(qs + (8 * g + (r16 >> 1)) * QS + n * 32 + j * 16 + (r16 & 1) * 8));
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = (uint32_t)(e < 2 ? q.x : q.y);
          o[e] = top_halves(__builtin_bit_cast(uint32_t, q_at(w, 2 * (e & 1))),
                            __builtin_bit_cast(uint32_t, q_at(w, 2 * (e & 1) + 1)));
        }
        wf[j] = __builtin_bit_cast(bf16x8, o);
      }
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        u32x4 part[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t hb[2], rb[2], lb[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const float v = x[t][2 * e + u] * d[2 * e + u];
            hb[u] = __builtin_bit_cast(uint32_t, v);
            const float r = v - __builtin_bit_cast(float, hb[u] & 0xffff0000u);
            rb[u] = __builtin_bit_cast(uint32_t, r);
            lb[u] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, rb[u] & 0xffff0000u));
          }
          part[0][e] = top_halves(hb[0], hb[1]);
          part[1][e] = top_halves(rb[0], rb[1]);
          part[2][e] = top_halves(lb[0], lb[1]);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[n][j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, part[p]), wf[j], acc[n][j][t], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // The same sums by fp32 FMAs, v = d * q first (rare: see above).
  auto multiply_fp32 = [&] {
    for (int k = 0; k < 32; ++k)
#pragma unroll
      for (int n = 0; n < NBW; ++n)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float v = scale_to_f32(ss[n * 32 + k]) *
                          (float)(int8_t)qs[k * QS + n * 32 + j * 16 + r16];
#pragma unroll
          for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[n][j][t][e] =
                  __builtin_fmaf(as[(16 * t + 4 * g + e) * AS + k], v, acc[n][j][t][e]);
        }
  };

  Stage st;
  int step = s0 + wave;
  if (step < s1) {
    load(step, st);
    for (; step < s1; step += kMfWaves) {
      stage(st);
      wave_sync();
      if (step + kMfWaves < s1) load(step + kMfWaves, st);
      if (scaled)
        multiply();
      else
        multiply_fp32();
      wave_sync();  // the step's LDS reads come before the next one's writes
    }
  }

  if (scaled) unscale();

  // Waves w and w + 4 add first, then the four pairs' sums in order.
  __syncthreads();
  f32x4* const red = reinterpret_cast<f32x4*>(lds);
  if (wave >= 4) {
#pragma unroll
    for (int i = 0; i < SLOTS; ++i)
      red[((wave - 4) * SLOTS + i) * 64 + lane] = acc[i / (2 * TT)][i / TT % 2][i % TT];
  }
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      f32x4& slot = red[(wave * SLOTS + i) * 64 + lane];
      slot = acc[i / (2 * TT)][i / TT % 2][i % TT] + slot;
    }
  }
  __syncthreads();
  // Output tile i of the workgroup: rows 4 g .. + 3 of its token tile, column r16.
  auto store = [&](float* dst, int i, const f32x4 v) {
    const int n = i / (2 * TT), j = i / TT % 2, t = i % TT;
    const int m = m0 + 16 * t + 4 * g;
    const int64_t col = (blk0 + n) * kBlockElems + j * 16 + r16;
    if (blk0 + n >= NB) return;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (m + e < M) dst[(int64_t)(m + e) * N + col] = v[e];
  };
  auto sum_of = [&](int i) {
    f32x4 v = red[i * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) v += red[(w * SLOTS + i) * 64 + lane];
    return v;
  };
  if (counters == nullptr) {
    float* const dst = out + (int64_t)by * M * N;
#pragma unroll
    for (int u = 0; u < (SLOTS + kMfWaves - 1) / kMfWaves; ++u) {
      const int i = u * kMfWaves + wave;
      if (SLOTS % kMfWaves == 0 || i < SLOTS) store(dst, i, sum_of(i));
    }
    return;
  }
  if constexpr (SLOTS == kMfWaves) {  // one output tile a wave
    // The splits of a tile meet: partials by device-scope stores, their completion,
    // the tile's counter; the last workgroup resets it and adds them in split order.
    constexpr int SC1 = 16;  // cache-policy bit: device scope
    constexpr uint32_t REGION = SLOTS * 1024;
    const unsigned nspl = gridDim.y;
    const uint32_t mine = (uint32_t)(wave * 64 + lane) * 16;
    const __amdgpu_buffer_rsrc_t prs =
        buffer_rsrc(reinterpret_cast<uint8_t*>(partials) + (int64_t)bx * nspl * REGION, nspl * REGION);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum_of(wave)), prs,
                                           by * REGION + mine, 0, SC1);
    uint32_t* const counter = counters + (size_t)bx * kCounterStride;
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
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (unsigned sp = 0; sp < nspl; sp += 8) {
      f32x4 p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        p[j] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       prs, sp + j < nspl ? (sp + j) * REGION + mine : 0x80000000u, 0, SC1));
#pragma unroll
      for (int j = 0; j < 8; ++j) v += p[j];
    }
    store(out, wave, v);
  }
}

// Half-block kernel (M <= 2, and 3 on few columns).  A workgroup owns a tile of 256 output columns (8
// blocks of a B row) for MR token rows and a run of K.  Lane c of a 16-lane group
// takes 16 columns, half h = c % 2 of block c / 2 of the tile, of one B row per
// step, so a group reads the tile's 272 contiguous bytes of a row and a wave four
// rows.  Per row a lane issues one 16-byte load and one 2-byte load, both inside
// its block:
//   h = 0, block 4-aligned: 16 bytes at the block (scale, q0 .. q13), 2 at +16;
//   h = 0, block 2 mod 4:   16 bytes at +2 (q0 .. q15), the scale at +0;
//   h = 1, block 4-aligned: 16 bytes at +16 (q14 .. q29), 2 at +32 (q30, q31);
//   h = 1, block 2 mod 4:   16 bytes at +18 (q16 .. q31), 2 at +16 (not used);
// and the h = 1 lane takes the scale from its h = 0 neighbour.  Loads go through
// buffer resources, so rows of B past K and activations past M or K read as
// zeros.  A lane issues the loads of U rows (a batch) and of their MR activations
// each before using any.  Values are formed as the reference forms them,
// v = d * q in fp32 (exact: an 11-bit by 8-bit significand product), and folded
// into per-token fp32 accumulators, acc = fma(a, v, acc).  The
// workgroup's 32 row phases (8 waves x 4 rows) are then added in LDS in a fixed
// order, one token at a time.  When K is spread over S workgroups per tile, each
// stores its sums to the workspace by device-scope stores, waits for their
// completion and bumps the tile's counter; the last to arrive resets the counter
// and adds the S partials of every output in fixed runs of consecutive splits, the
// runs' sums in run order (deterministic).
constexpr int kLnWaves = 8;                              // waves per workgroup
constexpr int kLnNT = 64 * kLnWaves;
constexpr int kLnLanes = 16;                             // lanes per B row
constexpr int kLnRows = 64 / kLnLanes;                   // B rows per wave step
constexpr int kLnCols = kLnLanes / 2 * kBlockElems;      // 256 columns per tile
constexpr int kLnMaxSplits = 64;

struct LnGrid {
  unsigned col_tiles, row_tiles, splits;
  int batches_per_split, mr, unroll;
};

LnGrid ln_grid(int M, int N, int K) {
  LnGrid g;
  const int NB = N / kBlockElems;
  g.mr = M >= 2 ? 2 : 1;
  g.unroll = 8;
  g.col_tiles = (unsigned)((NB + kLnLanes / 2 - 1) / (kLnLanes / 2));
  g.row_tiles = (unsigned)((M + g.mr - 1) / g.mr);
  const int batch = g.unroll * kLnWaves * kLnRows;
  const int batches = (K + batch - 1) / batch;
  const int64_t tiles = (int64_t)g.col_tiles * g.row_tiles;
  int s = (int)((512 + tiles - 1) / tiles);  // about two workgroups per CU
  if (s > batches) s = batches;
  if (s > kLnMaxSplits) s = kLnMaxSplits;
  if (s < 1) s = 1;
  g.batches_per_split = (batches + s - 1) / s;
  g.splits = (unsigned)((batches + g.batches_per_split - 1) / g.batches_per_split);
  return g;
}

template <int MR, int U>
__global__ __launch_bounds__(kLnNT) void matmul_q8_0_half_kernel(
    const float* __restrict__ a, const uint8_t* __restrict__ b, float* __restrict__ c,
    int M, int N, int K, int batches_per_split, float* __restrict__ partials,
    uint32_t* __restrict__ counters) {
  constexpr int BATCH = U * kLnWaves * kLnRows;  // B rows per batch
  constexpr int SC1 = 16;                        // cache-policy bit: device scope
  __shared__ __attribute__((aligned(16))) float red[kLnWaves * 64 * 16];
  __shared__ uint32_t arrived;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane % kLnLanes, rsub = lane / kLnLanes, h = c16 & 1;
  const int NB = N / kBlockElems;
  const uint32_t row_bytes = (uint32_t)NB * kBlockBytes;
  const int jb = blockIdx.x * (kLnLanes / 2) + (c16 >> 1);
  const uint32_t cb = (uint32_t)(jb < NB ? jb : NB - 1) * kBlockBytes;  // columns past N: dead
  // A lane's rows all have the parity of rsub, so its blocks' 4-byte phase is fixed.
  const uint32_t mis =
      (uint32_t)(((uintptr_t)b + cb + ((rsub & 1) ? row_bytes : 0u)) & 2u);
  const uint32_t offx = cb + 16 * h + mis;
  const uint32_t offu = cb + 16 * h + (mis ? 0u : 16u);
  // Buffer resources: B rows past K and A entries past M or K read as zeros.
  const __amdgpu_buffer_rsrc_t brs = buffer_rsrc(b, (uint32_t)K * row_bytes);
  const __amdgpu_buffer_rsrc_t ars = buffer_rsrc(a, (uint32_t)M * (uint32_t)K * 4u);
  const int m0 = blockIdx.z * MR;
  const int nbatches = (K + BATCH - 1) / BATCH;
  const int bt0 = blockIdx.y * batches_per_split;
  const int bt1 = min(bt0 + batches_per_split, nbatches);

  float acc[MR][16];
#pragma unroll
  for (int r = 0; r < MR; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.0f;

  // One batch: U rows of B per lane (16 + 2 bytes each) and their activations.
  // The 2-byte loads stay 16 bits wide until used, so no instruction placed with
  // the loads waits for them.
  struct Batch {
    u32x4 q4[U];
    uint16_t u2[U];
    float x[U][MR];
  };
  auto load = [&](Batch& t, int bt) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = bt * BATCH + (u * kLnWaves + wave) * kLnRows + rsub;
      const bool kv = k < K;
      const uint32_t ro = kv ? (uint32_t)k * row_bytes : 0x80000000u;
      t.q4[u] = __builtin_amdgcn_raw_buffer_load_b128(brs, ro + offx, 0, 0);
      t.u2[u] = __builtin_amdgcn_raw_buffer_load_b16(brs, ro + offu, 0, 0);
#pragma unroll
      for (int r = 0; r < MR; ++r)
        t.x[u][r] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(
                       ars, kv && m0 + r < M ? ((uint32_t)(m0 + r) * (uint32_t)K + k) * 4u
                                             : 0x80000000u,
                       0, 0));
    }
  };
  auto consume = [&](const Batch& t) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t w[5] = {t.q4[u].x, t.q4[u].y, t.q4[u].z, t.q4[u].w, (uint32_t)t.u2[u]};
      uint32_t q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = mis ? w[i] : __builtin_amdgcn_alignbyte(w[i + 1], w[i], 2);
      const uint32_t own = mis ? w[4] : (w[0] & 0xffffu);  // the scale, on h = 0 lanes
      const uint32_t other = (uint32_t)__shfl_xor((int)own, 1);
      const float d = scale_to_f32(h ? other : own);
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = d * q_at(q[i >> 2], i & 3);
#pragma unroll
      for (int r = 0; r < MR; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][i] = __builtin_fmaf(t.x[u][r], v[i], acc[r][i]);
    }
  };

  // Every load of a batch is issued before the first use of any.  (Issuing the
  // next batch's loads before using the current one, in a second register set,
  // measured no faster: the extra registers halve the workgroups per CU.)
  for (int bt = bt0; bt < bt1; ++bt) {
    Batch t;
    load(t, bt);
    __builtin_amdgcn_sched_barrier(0);
    consume(t);
  }

  // Per token: every lane's 16 sums to LDS, then each column's 32 row-phase sums in
  // (wave, row) order.
  const unsigned tile = blockIdx.z * gridDim.x + blockIdx.x;
  const int n = blockIdx.x * kLnCols + (tid % kLnCols);
  const bool split = gridDim.y > 1;
  const uint32_t region = MR * kLnCols;  // floats of one workgroup's partial sums
  const __amdgpu_buffer_rsrc_t prs =
      buffer_rsrc(partials, split ? (uint32_t)((tile + 1) * gridDim.y * region * 4) : 0u);
#pragma unroll
  for (int r = 0; r < MR; ++r) {
    float* mine = red + (wave * 64 + lane) * 16;
#pragma unroll
    for (int i = 0; i < 16; i += 4)
      *reinterpret_cast<f32x4*>(mine + i) = f32x4{acc[r][i], acc[r][i + 1], acc[r][i + 2],
                                                  acc[r][i + 3]};
    __syncthreads();
    if (tid < kLnCols) {
      const int cc = tid / 16, i = tid % 16;  // lane of the group, column within its half
      float s = 0.0f;
#pragma unroll
      for (int w = 0; w < kLnWaves; ++w)
#pragma unroll
        for (int p = 0; p < kLnRows; ++p) s += red[(w * 64 + p * kLnLanes + cc) * 16 + i];
      const int m = m0 + r;
      if (!split) {
        if (m < M && n < N) c[(int64_t)m * N + n] = s;
      } else {
        __builtin_amdgcn_raw_buffer_store_b32(
            __builtin_bit_cast(uint32_t, s), prs,
            (uint32_t)(((tile * gridDim.y + blockIdx.y) * region + r * kLnCols + tid) * 4), 0,
            SC1);
      }
    }
    __syncthreads();
  }
  if (!split) return;

  uint32_t* const counter = counters + (size_t)tile * kCounterStride;
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);  // every partial has reached the coherence point
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  if (tid == 0)
    arrived = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  if (arrived != gridDim.y - 1) return;
  if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // The last workgroup adds the S partials of every output: the region's 16-byte
  // pieces are split over the threads as (piece, run of consecutive splits); each
  // thread sums its run in split order with the loads of 8 splits issued together,
  // then the runs' sums of a piece are added in run order in LDS.
  constexpr int PIECES = MR * kLnCols / 4;
  constexpr int RUNS = kLnNT / PIECES;  // 8 or 4 for MR = 1, 2
  const unsigned nspl = gridDim.y, per = (nspl + RUNS - 1) / RUNS;
  const int pc = tid % PIECES, run = tid / PIECES;
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  const unsigned s0 = run * per, s1 = min(nspl, s0 + per);
  for (unsigned sp = s0; sp < s1; sp += 8) {
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     prs, sp + j < s1 ? (uint32_t)(((tile * nspl + sp + j) * region + 4 * pc) * 4)
                                      : 0x80000000u,
                     0, SC1));
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (sp + j < s1) sum += v[j];
  }
  f32x4* const runs = reinterpret_cast<f32x4*>(red);  // [RUNS][PIECES]
  runs[run * PIECES + pc] = sum;
  __syncthreads();
  if (run == 0) {
    f32x4 t = runs[pc];
    for (int q = 1; q < RUNS; ++q) t += runs[q * PIECES + pc];
    const int r = (4 * pc) / kLnCols, m = m0 + r;
    const int nn = blockIdx.x * kLnCols + (4 * pc) % kLnCols;  // N % 32 == 0: 4 columns in or out
    if (m < M && nn < N) *reinterpret_cast<f32x4*>(c + (int64_t)m * N + nn) = t;
  }
}

// out[m, n] = sum over s of part[s][m][n], four columns a thread: the splits are
// taken in kSpGroups runs of consecutive splits, each run summed in split order by
// its own thread (their loads in flight together), and the runs' sums added in run
// order, so the grouping is fixed and the result deterministic.
constexpr int kSpGroups = 8;
constexpr int kSpCols = 256 / kSpGroups;  // float4 columns per workgroup

__global__ __launch_bounds__(256) void matmul_splits_kernel(const float* __restrict__ part,
                                                           float* __restrict__ c, int64_t mn4,
                                                           int splits) {
  __shared__ f32x4 run[kSpGroups][kSpCols];
  const int col = threadIdx.x % kSpCols, g = threadIdx.x / kSpCols;
  const int64_t i = (int64_t)blockIdx.x * kSpCols + col;
  const int per = (splits + kSpGroups - 1) / kSpGroups;
  const int s0 = g * per, s1 = min(s0 + per, splits);
  const f32x4* p = reinterpret_cast<const f32x4*>(part);
  f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
  if (i < mn4 && s0 < s1) {
    s = p[(int64_t)s0 * mn4 + i];
#pragma unroll 8
    for (int sp = s0 + 1; sp < s1; ++sp) s += p[(int64_t)sp * mn4 + i];
  }
  run[g][col] = s;
  __syncthreads();
  if (g == 0 && i < mn4) {
    f32x4 t = run[0][col];
    for (int r = 1; r < kSpGroups && r * per < splits; ++r) t += run[r][col];
    reinterpret_cast<f32x4*>(c)[i] = t;
  }
}

template <int TT, int NBW>
void launch_mf(const MfGrid& g, const float* a, const uint8_t* b, float* dst, int M, int N, int K,
               float* partials, uint32_t* counters, hipStream_t stream) {
  hipLaunchKernelGGL((matmul_q8_0_mfma_kernel<TT, NBW>), dim3(g.tiles, g.splits, g.row_tiles),
                     dim3(kMfNT), 0, stream, a, b, dst, M, N, K, g.steps_per_split, partials, counters);
}

template <int MR, int U>
void launch_ln(const LnGrid& g, const float* a, const uint8_t* b, float* c, int M, int N, int K,
               float* partials, uint32_t* counters, hipStream_t stream) {
  hipLaunchKernelGGL((matmul_q8_0_half_kernel<MR, U>), dim3(g.col_tiles, g.splits, g.row_tiles),
                     dim3(kLnNT), 0, stream, a, b, c, M, N, K, g.batches_per_split, partials,
                     counters);
}

// The half-block kernel's calls: up to two rows of A (MI355X, two rows: 4096 x 4096
// 10.6 us vs 11.2 on the MFMA kernel, 11008 x 4096 20.3 vs 21.3; three and four rows
// 13.9-14.5 vs 11.8, 21-28 vs 21.4), three where K is long over few columns, whose 16-row
// MFMA tiles stay mostly empty (two row tiles read B twice, from the L2: 3 x 480 x 32608
// 12.0 us vs 14.9, 3 x 1024 x 8192 1.24x, 3 x 2048 x 4096 1.11x; above 8.6 million elements
// of B on more than 512 columns the MFMA kernel wins, 2048 x 5120 0.93x), and B below 2 GiB
// (32-bit buffer offsets).
bool use_half(int M, int N, int K) {
  const int64_t elems = (int64_t)N * K;
  const bool three = M == 3 && ((N <= 512 && K >= 8192) ||
                                (K >= 3072 && elems >= 5000000 && elems <= 8600000));
  return (M <= 2 || three) && (int64_t)K * (N / kBlockElems) * kBlockBytes < (int64_t(1) << 31) &&
         (int64_t)M * K * 4 < (int64_t(1) << 31);
}

}  // namespace

MatmulNeed matmul_workspace(int M, int N, int K) {
  MatmulNeed need;
  if (M <= 0 || N <= 0 || K <= 0) return need;
  if (use_half(M, N, K)) {
    const LnGrid g = ln_grid(M, N, K);
    if (g.splits > 1) {
      const size_t tiles = (size_t)g.col_tiles * g.row_tiles;
      need.partial_floats = tiles * g.splits * g.mr * kLnCols;
      need.counters = tiles * kCounterStride;
    }
    return need;
  }
  const MfGrid g = mf_grid(M, N, K);
  if (g.splits > 1) need.partial_floats = (size_t)g.splits * M * N;
  if (g.splits > 1 && mf_handoff(M)) {
    need.partial_floats = (size_t)g.tiles * g.splits * kMfWaves * 256;
    need.counters = (size_t)g.tiles * kCounterStride;
  }
  return need;
}

hipError_t launch_matmul(const float* a, const uint8_t* b, float* c, int M, int N, int K,
                         float* partials, uint32_t* counters, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
  if (N % kBlockElems != 0 || K % kBlockElems != 0) return hipErrorInvalidValue;
  if (use_half(M, N, K)) {
    const LnGrid g = ln_grid(M, N, K);
    if (g.row_tiles > 65535 || g.splits > 65535) return hipErrorInvalidValue;
    if (g.splits > 1) {
      const int64_t bytes = (int64_t)g.col_tiles * g.row_tiles * g.splits * g.mr * kLnCols * 4;
      if (partials == nullptr || counters == nullptr || bytes >= (int64_t(1) << 32))
        return hipErrorInvalidValue;
    }
    switch (g.mr) {
      case 1: launch_ln<1, 8>(g, a, b, c, M, N, K, partials, counters, stream); break;
      default: launch_ln<2, 8>(g, a, b, c, M, N, K, partials, counters, stream); break;
    }
    return hipGetLastError();
  }
  const MfGrid g = mf_grid(M, N, K);
  if (g.row_tiles > 65535 || g.splits > 65535) return hipErrorInvalidValue;
  if (g.splits > 1 && partials == nullptr) return hipErrorInvalidValue;
  const bool handoff = g.splits > 1 && mf_handoff(M);
  if (handoff && counters == nullptr) return hipErrorInvalidValue;
  if (!handoff) counters = nullptr;
  float* dst = g.splits > 1 && !handoff ? partials : c;
  switch (g.tt) {
    case 1: launch_mf<1, 4>(g, a, b, dst, M, N, K, partials, counters, stream); break;
    case 2: launch_mf<2, 4>(g, a, b, dst, M, N, K, partials, counters, stream); break;
    case 3: launch_mf<3, 2>(g, a, b, dst, M, N, K, partials, counters, stream); break;
    default: launch_mf<4, 2>(g, a, b, dst, M, N, K, partials, counters, stream); break;
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || g.splits == 1 || handoff) return err;
  const int64_t mn4 = (int64_t)M * N / 4;
  hipLaunchKernelGGL(matmul_splits_kernel, dim3((unsigned)((mn4 + kSpCols - 1) / kSpCols)),
                     dim3(256), 0, stream, partials, c, mn4, (int)g.splits);
  return hipGetLastError();
}

}  // namespace mle
