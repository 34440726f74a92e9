// argmax.hip -- greedy-decode argmax of lm_head logits on the device.
//
// idx[r] = the first index of the largest value of logits[r, 0:n] (ties go to
// the lower index, as the reference's greedy pick does: it scans candidates in
// index order and replaces the best only on a strictly larger value,
// src/runtime/sampler.cpp:108-118; -0 and +0 compare equal).  NaN entries are
// ignored; a row of NaN only gives index 0 and value NaN.  Replaces the
// per-token device-to-host copy of the whole logits row that the reference's
// CUDA generator makes before sampling on the host
// (examples/generate_cuda.cpp:81-94, 305-314).
//
// A workgroup (grid chunks x rows) reduces a chunk of a row to one 64-bit key.  key =
// (order(v) << 32) | ~index, where order() maps float bits to unsigned integers in
// value order, so the largest key is the largest value with the smallest index:
// deterministic in any order of reduction.  Up to kArgRows rows of kArgMeetPieces pieces
// the chunks' keys meet by an atomic maximum beside the row's counter in the workspace,
// and the row's last workgroup decodes the winner; more rows (whose counters a default
// workspace does not hold) and longer ones write the keys, which a second launch reduces.
//
// Bound by latency (152k logits are 0.6 MB): a thread's 8 values are loaded at once
// (one by one in a loop, each load waited for, and with a second launch for every call, the
// [1, 151936] pick behind its [151936, 896] Linear took 29.3 us a pair on MI355X; this
// takes 27.1).  A row's chunks take turns at its counter, so at most kArgChunks of them
// meet, two pieces each where there are more pieces (300000 logits: 5.3 us, 6.1 with a
// chunk a piece, 5.9 in two launches), and rows past two pieces a chunk take two launches
// (524288 logits: 5.8 us, 6.0 with 96 chunks meeting, 9.0 with 256).
#include <algorithm>

#include "../launch.hpp"

namespace mle {
namespace {

constexpr int kArgThreads = 256;
constexpr int kArgVecs = 2;                              // 4-value loads a thread
constexpr int kArgPiece = 4 * kArgVecs * kArgThreads;    // 2048 values
constexpr int kArgRows = 4096 / kCounterStride;          // a default workspace's counters
constexpr int kArgChunks = 96;                           // of a row that meet
constexpr int kArgMeetPieces = 2 * kArgChunks;

__device__ __forceinline__ uint64_t arg_key(float v, uint32_t i) {
  if (v != v) return 0;  // NaN: never selected
  if (v == 0.0f) v = 0.0f;  // -0 -> +0
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ((uint64_t)u << 32) | (uint32_t)~i;
}

__device__ __forceinline__ uint64_t wave_max(uint64_t k) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)k, off, 64);
    const uint32_t hi = __shfl_xor((uint32_t)(k >> 32), off, 64);
    const uint64_t o = ((uint64_t)hi << 32) | lo;
    k = o > k ? o : k;
  }
  return k;
}

__device__ __forceinline__ uint64_t block_max(uint64_t k) {
  __shared__ uint64_t part[kArgThreads / 64];
  k = wave_max(k);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) part[wave] = k;
  __syncthreads();
  uint64_t r = part[0];
#pragma unroll
  for (int i = 1; i < kArgThreads / 64; ++i) r = part[i] > r ? part[i] : r;
  return r;
}

__device__ __forceinline__ void write_winner(uint64_t k, int64_t r, int32_t* __restrict__ idx,
                                             float* __restrict__ val) {
  if (k == 0) {  // NaN only
    idx[r] = 0;
    if (val) val[r] = __builtin_nanf("");
    return;
  }
  idx[r] = (int32_t)~(uint32_t)k;
  if (val) {
    uint32_t u = (uint32_t)(k >> 32);
    u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
    val[r] = __builtin_bit_cast(float, u);
  }
}

// Workgroup (c, r) reduces logits[r, c*chunk : (c+1)*chunk), chunk a multiple of
// kArgPiece.  MEET: the chunks meet in counters[r * kCounterStride] (dwords 0-1 the
// largest key, 2 the arrivals; zero before and after), else each writes its key.
template <bool MEET>
__global__ __launch_bounds__(kArgThreads) void argmax_chunks_kernel(
    const float* __restrict__ x, int64_t n, int64_t chunk, uint64_t* __restrict__ keys,
    uint32_t* __restrict__ counters, int32_t* __restrict__ idx, float* __restrict__ val) {
  const int64_t r = blockIdx.y;
  const int64_t b = (int64_t)blockIdx.x * chunk;
  const int64_t e = b + chunk < n ? b + chunk : n;
  const float* row = x + r * n;
  uint64_t k = 0;
  for (int64_t p = b; p < e; p += kArgPiece) {
    const int64_t i0 = p + 4 * threadIdx.x;
    float v[kArgVecs][4];
    if (p + kArgPiece <= e) {  // rows are 4-byte aligned only
#pragma unroll
      for (int j = 0; j < kArgVecs; ++j)
        __builtin_memcpy(v[j], __builtin_assume_aligned(row + i0 + j * 4 * kArgThreads, 4), 16);
    } else {
#pragma unroll
      for (int j = 0; j < kArgVecs; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int64_t i = i0 + j * 4 * kArgThreads + c;
          const float u = row[i < e ? i : e - 1];
          v[j][c] = i < e ? u : __builtin_nanf("");
        }
    }
#pragma unroll
    for (int j = 0; j < kArgVecs; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint64_t key = arg_key(v[j][c], (uint32_t)(i0 + j * 4 * kArgThreads + c));
        k = key > k ? key : k;
      }
  }
  k = block_max(k);
  if (threadIdx.x != 0) return;
  if constexpr (!MEET) {
    keys[r * gridDim.x + blockIdx.x] = k;
  } else {
    uint32_t* const count = counters + r * kCounterStride + 2;
    uint64_t* const best = reinterpret_cast<uint64_t*>(counters + r * kCounterStride);
    (void)__hip_atomic_fetch_max(best, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);  // the maximum is in before the arrival counts
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (__hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
        gridDim.x - 1)
      return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    k = __hip_atomic_exchange(best, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    write_winner(k, r, idx, val);
  }
}

// More rows: one workgroup per row over its `chunks` keys.
__global__ __launch_bounds__(kArgThreads) void argmax_final_kernel(
    const uint64_t* __restrict__ keys, int chunks, int32_t* __restrict__ idx,
    float* __restrict__ val) {
  const int64_t r = blockIdx.x;
  uint64_t k = 0;
  for (int i = threadIdx.x; i < chunks; i += kArgThreads) {
    const uint64_t c = keys[r * chunks + i];
    k = c > k ? c : k;
  }
  k = block_max(k);
  if (threadIdx.x == 0) write_winner(k, r, idx, val);
}

}  // namespace

int argmax_chunks(int64_t n) {
  // Chunks of at least 2048 values, at most 256 per row.
  const int64_t c = (n + 2047) / 2048;
  return (int)(c < 1 ? 1 : c > 256 ? 256 : c);
}

size_t argmax_counters(int rows, int64_t n) {
  return rows <= kArgRows && n <= (int64_t)kArgMeetPieces * kArgPiece ? (size_t)rows * kCounterStride
                                                                      : 0;
}

hipError_t launch_argmax(const float* x, int rows, int64_t n, int32_t* idx, float* val,
                         uint64_t* keys, uint32_t* counters, hipStream_t stream) {
  if (rows <= 0 || n <= 0 || n > 0x7fffffff || rows > 65535) return hipErrorInvalidValue;
  const int chunks = counters != nullptr ? std::min(argmax_chunks(n), kArgChunks) : argmax_chunks(n);
  const int64_t pieces = (n + kArgPiece - 1) / kArgPiece;
  const int64_t chunk = (pieces + chunks - 1) / chunks * kArgPiece;
  const dim3 grid((unsigned)chunks, (unsigned)rows);
  if (counters != nullptr) {
    hipLaunchKernelGGL(argmax_chunks_kernel<true>, grid, dim3(kArgThreads), 0, stream, x, n, chunk,
                       keys, counters, idx, val);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(argmax_chunks_kernel<false>, grid, dim3(kArgThreads), 0, stream, x, n, chunk,
                     keys, counters, idx, val);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(argmax_final_kernel, dim3((unsigned)rows), dim3(kArgThreads), 0, stream,
                     keys, chunks, idx, val);
  return hipGetLastError();
}

}  // namespace mle
