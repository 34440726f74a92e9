// topk.hip -- the top-n tokens of logits rows with their softmax probabilities.
//
// For each row r of n logits: scaled = logits * (1 / temperature) when
// temperature > 0 and != 1 (else the logits as they are); p = softmax(scaled),
// computed as exp(scaled - max) / sum (the sum and the quotient in fp64); ids[r, j],
// probs[r, j] for j < min(top_n, n) are the top_n tokens by probability, largest
// first, ties to the lower index.  A row whose maximum is not finite, whose sum is not
// finite or not positive, or that holds a NaN gives the uniform distribution
// 1 / n, i.e. ids 0, 1, 2, ... .  This is Sampler::get_top_tokens
// (src/runtime/sampler.cpp:141-197; the same softmax as Sampler::sample,
// :31-63) on the device: the reference's generator copies the whole logits
// row to the host per token instead (examples/generate_cuda.cpp:81-94).  Where
// the reference leaves the order of equal probabilities to std::partial_sort,
// the order here is the logit, then the index.
//
// Two launches.  Pass 1 (grid chunks x rows, 256 threads) streams a 2048-value chunk:
// its maximum (+Inf where it holds a NaN), its sum of exp(value - maximum), and the maxima of its
// groups of 64 values (1024 / top_n for fewer than 16 tokens, so that the workspace
// stays within 2 top_n floats a chunk).  Pass 2 (one 1024-thread workgroup per row)
// merges the chunk statistics in a fixed order (max, then the sum of sum_c *
// exp(max_c - max)) and works on whole groups: the top_n tokens lie in the top_n
// groups of largest maximum (ties to the lower group), so it picks groups, re-reads
// only their values and picks among those.
//   * Groups: one histogram over the distance of the group maxima from the row's
//     maximum, in floating-point bins (5 mantissa bits), gives a distance within which
//     at least top_n groups lie; usually a few more do, all of them are taken.  Where
//     that is too many values (massive ties), the exact top_n groups are selected.
//   * Values within that distance are ranked by counting the larger keys (64-bit:
//     order(value) << 32 | ~index, all distinct); more than 256 go through the
//     radix select.
// Selection (exact): a radix select over the keys (8-bit digit histograms in LDS, most
// significant first) narrows a prefix until at most 256 keys reach it; those are gathered
// and sorted by one wave in registers (bitonic network, lane shuffles, no barriers), and
// the first top_n are the result.  Rows of few distinct values need the index's digits
// too; sorting all 16384 keys in LDS there took 157 us for a constant row at top_n 3
// (MI355X), the digits 31.  Results are deterministic: the keys are distinct, so
// neither the ranks nor the sorted order depend on the order of gathering.
//
// Latency bounds it, not bytes (8 rows x 152k logits are 4.9 MB).  Selecting top_n keys
// in every chunk instead (a radix select per chunk, then one over 75 x top_n
// candidates) took 31.6 us for 8 rows at top_n 40 (MI355X); this takes 12.3.  Pass 2
// issues all its loads of a stage before it uses one, and a NaN travels as an infinite
// maximum instead of through a reduction of its own (13.7 us otherwise).
#include "../launch.hpp"

namespace mle {
namespace {

constexpr int kChunk = 2048;           // values per pass-1 workgroup
constexpr int kGroup = 64;             // values per group (top_n >= 16)
constexpr int kP1Threads = 256;
constexpr int kP2Threads = 1024;
constexpr int kP2Keys = 16384;         // values of the picked groups (16 a thread)
constexpr int kP2Groups = 8192;        // groups of a row that pass 2 picks from
constexpr int kBins = 8192;            // distance bins: 8 exponent and 5 mantissa bits

// Group maxima a pass-1 chunk writes for top k: at most 2 k, whole powers of two.
__host__ __device__ constexpr int chunk_groups(int k) {
  int c = kChunk / kGroup;
  while (c > 2 * k) c >>= 1;
  return c;
}

__device__ __forceinline__ uint64_t topk_key(float v, uint32_t i) {
  if (v != v) return 0;      // NaN (the row becomes uniform anyway)
  if (v == 0.0f) v = 0.0f;   // -0 -> +0
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ((uint64_t)u << 32) | (uint32_t)~i;
}

__device__ __forceinline__ float key_value(uint64_t k) {
  uint32_t u = (uint32_t)(k >> 32);
  u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
  return __builtin_bit_cast(float, u);
}

template <int NT, typename T, typename Op>
__device__ T block_reduce(T v, Op op, T* part) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();  // part[] may still be read from an earlier reduction
  if (lane == 0) part[wave] = v;
  __syncthreads();
  T r = part[0];
#pragma unroll
  for (int i = 1; i < NT / 64; ++i) r = op(r, part[i]);
  return r;
}

struct SelectLds {
  uint32_t hist[256];
  uint64_t cand[256];
  uint32_t digit, above, eq, total, ncand;
};

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
  const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, m, 64);
  const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m, 64);
  return ((uint64_t)hi << 32) | lo;
}

// Descending bitonic sort of 256 keys held by one wave, 4 per lane (element
// 4 lane + j), in registers.
__device__ void wave_sort256_desc(uint64_t (&v)[4]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int size = 2; size <= 256; size <<= 1)
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int e = 4 * lane + j;
          const uint64_t o = shfl_xor64(v[j], stride >> 2);
          const bool lower = (e & stride) == 0;
          const bool keep_max = lower == ((e & size) == 0);
          v[j] = keep_max ? (o > v[j] ? o : v[j]) : (o < v[j] ? o : v[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j & stride) continue;  // handle each in-lane pair once, from its lower element
          const int e = 4 * lane + j;
          const bool desc = (e & size) == 0;
          const uint64_t a = v[j], c = v[j + stride];
          const bool swap = desc ? a < c : a > c;
          v[j] = swap ? c : a;
          v[j + stride] = swap ? a : c;
        }
      }
    }
}

// hist[bin] += 1 for every lane with `in`.  Lanes that all name one bin (ties, the leading
// digits) add once: 16384 single adds to one LDS word took 7 us a digit (MI355X).
__device__ __forceinline__ void count_bin(uint32_t* hist, uint32_t bin, bool in) {
  const uint64_t lanes = __builtin_amdgcn_ballot_w64(in);
  if (lanes == 0) return;  // uniform
  const int first = __builtin_ctzll(lanes);
  const uint32_t one = (uint32_t)__builtin_amdgcn_readlane((int)bin, first);
  if (__builtin_amdgcn_ballot_w64(in && bin == one) == lanes) {
    if ((int)(threadIdx.x & 63) == first) atomicAdd(&hist[one], (uint32_t)__builtin_popcountll(lanes));
  } else if (in) {
    atomicAdd(&hist[bin], 1u);
  }
}

// Top k (k <= kTopTokensMax) of the distinct keys held E per thread by NT threads
// (0 = no key), written sorted descending to out[0, k) (zeros past the number
// of keys).
template <int NT, int E>
__device__ void select_top(const uint64_t (&key)[E], int k, uint64_t* __restrict__ out,
                           SelectLds& sm) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint64_t prefix = 0, mask = 0;
  int need = k;
  bool all = false;  // fewer keys than k: every key is a candidate
  // Digits from the top until at most 256 keys reach the prefix: values' digits first,
  // the index's too where more than 256 keys tie at the value.
  for (int shift = 56; shift >= 0; shift -= 8) {
    for (int i = tid; i < 256; i += NT) sm.hist[i] = 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e)
      count_bin(sm.hist, (uint32_t)(key[e] >> shift) & 255u,
                key[e] != 0 && (key[e] & mask) == prefix);
    __syncthreads();
    if (wave == 0) {
      uint32_t h[4], local = 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        h[t] = sm.hist[255 - (4 * lane + t)];
        local += h[t];
      }
      uint32_t incl = local;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, off, 64);
        if (lane >= off) incl += o;
      }
      uint32_t run = incl - local;  // keys in the bins above this lane's first bin
      if (lane == 63) sm.total = incl;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (run < (uint32_t)need && (uint32_t)need <= run + h[t]) {
          sm.digit = 255u - (uint32_t)(4 * lane + t);
          sm.above = run;
          sm.eq = h[t];
        }
        run += h[t];
      }
    }
    __syncthreads();
    if (shift == 56 && sm.total <= (uint32_t)k) {
      all = true;
      break;
    }
    need -= (int)sm.above;
    prefix |= (uint64_t)sm.digit << shift;
    mask |= (uint64_t)255u << shift;
    if ((uint32_t)(k - need) + sm.eq <= 256u) break;  // always so once the key is whole
  }
  // Candidates: every key (all) or the keys from the prefix up.
  __syncthreads();
  if (tid == 0) sm.ncand = 0;
  for (int i = tid; i < 256; i += NT) sm.cand[i] = 0;
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (key[e] != 0 && (all || key[e] >= prefix)) sm.cand[atomicAdd(&sm.ncand, 1u)] = key[e];
  __syncthreads();
  if (wave == 0) {
    uint64_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = sm.cand[4 * lane + j];
    wave_sort256_desc(v);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * lane + j < k) out[4 * lane + j] = v[j];
  }
  __syncthreads();
}

// A logit under the temperature, rounded once.  Never contracted with what uses it: both
// passes have to see the same value, or a row's own maximum could lie above its maximum.
__device__ __forceinline__ float scaled_logit(float v, float inv_temp) {
#pragma clang fp contract(off)
  return v * inv_temp;
}

// Distance bin of a value not above the row's finite maximum (0: at it, +Inf: 8160).  The
// sign goes: a maximum held as -0 beside a +0 is at distance -0.
__device__ __forceinline__ uint32_t dist_bin(float mx, float v) {
  return __builtin_bit_cast(uint32_t, __builtin_fabsf(mx - v)) >> 18;
}

// Pass 1: workgroup (c, r) over logits[r, c * kChunk : (c + 1) * kChunk).
// maxima: [row][chunk][gpc] group maxima; stats: [row][chunk] x {max (+Inf beside a
// NaN), sum, rest of the sum, 0}.
typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));  // rows are 4-byte aligned

__global__ __launch_bounds__(kP1Threads) void topk_chunks_kernel(
    const float* __restrict__ x, int64_t n, int gpc, float inv_temp, int scale,
    float* __restrict__ maxima, float* __restrict__ stats) {
  __shared__ float gmax[kChunk / kGroup];
  __shared__ float fpart[kP1Threads / 64];
  __shared__ double dpart[kP1Threads / 64];
  const int64_t r = blockIdx.y;
  const int64_t b = (int64_t)blockIdx.x * kChunk;
  const float* row = x + r * n;
  constexpr int PER = kChunk / kP1Threads, Q = PER / 4;
  static_assert(kGroup == 64, "16 lanes x 4 values are a group");
  float v[PER];
  float mx = -__builtin_inff();
  bool nan = false;
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const int64_t i = b + 4 * ((int)threadIdx.x + kP1Threads * j);
    f4 t = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
    if (i + 4 <= n) {
      t = *reinterpret_cast<const f4*>(row + i);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < n) t[e] = row[i + e];
    }
    float g = -__builtin_inff();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float u = scale && i + e < n ? scaled_logit(t[e], inv_temp) : t[e];
      v[4 * j + e] = u;
      nan |= u != u;
      g = fmaxf(g, u);  // ignores NaN
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) g = fmaxf(g, __shfl_xor(g, off, 64));
    if ((threadIdx.x & 15) == 0) gmax[threadIdx.x / 16 + kP1Threads / 16 * j] = g;
    mx = fmaxf(mx, g);
  }
  if (nan) mx = __builtin_inff();  // the row is uniform either way
  mx = block_reduce<kP1Threads>(mx, [](float a, float c) { return fmaxf(a, c); }, fpart);
  double sum = 0.0;  // one chunk can hold most of the row's sum: its rounding is the row's
  if (mx > -__builtin_inff() && mx < __builtin_inff()) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (v[j] == v[j]) sum += expf(v[j] - mx);
  }
  sum = block_reduce<kP1Threads>(sum, [](double a, double c) { return a + c; }, dpart);
  const int64_t slot = r * gridDim.x + blockIdx.x;
  if ((int)threadIdx.x < gpc) {
    const int f = kChunk / kGroup / gpc;  // 64-value groups per written maximum
    float g = gmax[threadIdx.x * f];
    for (int i = 1; i < f; ++i) g = fmaxf(g, gmax[threadIdx.x * f + i]);
    maxima[slot * gpc + threadIdx.x] = g;
  }
  if (threadIdx.x == 0) {
    stats[slot * 4 + 0] = mx;
    stats[slot * 4 + 1] = (float)sum;
    stats[slot * 4 + 2] = (float)(sum - (float)sum);
    stats[slot * 4 + 3] = 0.0f;
  }
}

// Pass 2: one workgroup per row over its chunks' statistics and group maxima.  A group
// here is `gm` consecutive written maxima (a power of two; 1 up to kP2Groups maxima),
// 2^gshift values; the kk groups' values fit kP2Keys for every accepted n.
__global__ __launch_bounds__(kP2Threads) void topk_final_kernel(
    const float* __restrict__ x, const float* __restrict__ maxima,
    const float* __restrict__ stats, int chunks, int gpc, int gm, int gshift, int64_t n, int kk,
    float inv_temp, int scale, int32_t* __restrict__ ids, float* __restrict__ probs) {
  __shared__ __attribute__((aligned(16))) uint32_t hist[kBins];
  __shared__ SelectLds sm;
  __shared__ uint64_t top[kTopTokensMax];
  __shared__ int list[kP2Keys / kGroup];
  __shared__ float fpart[kP2Threads / 64];
  __shared__ double dpart[kP2Threads / 64];
  __shared__ uint32_t wsum[kP2Threads / 64];
  __shared__ uint32_t bin_at, groups_in, nlist;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t r = blockIdx.x;
  const float* st = stats + r * chunks * 4;
  // The group maxima first: nothing below waits for more than they do.
  constexpr int GPT = kP2Groups / kP2Threads;
  const int total_max = chunks * gpc;  // per row
  const int groups = (int)((n + ((int64_t)1 << gshift) - 1) >> gshift);
  const float* mrow = maxima + r * (int64_t)total_max;
  float gv[GPT];
  if (gm == 1) {  // all loads in flight
#pragma unroll
    for (int e = 0; e < GPT; ++e) gv[e] = mrow[min(tid + kP2Threads * e, groups - 1)];
  } else {
#pragma unroll
    for (int e = 0; e < GPT; ++e) {
      const int gi = tid + kP2Threads * e;
      float g = -__builtin_inff();
      if (gi < groups)
        for (int j = 0; j < gm && gi * gm + j < total_max; ++j) g = fmaxf(g, mrow[gi * gm + j]);
      gv[e] = g;
    }
  }
  const f4 st0 = *reinterpret_cast<const f4*>(st + 4 * min(tid, chunks - 1));
  float mx = st0.x;
  for (int c = tid + kP2Threads; c < chunks; c += kP2Threads) mx = fmaxf(mx, st[c * 4]);
  for (int i = tid; i < kBins / 4; i += kP2Threads)
    reinterpret_cast<uint4*>(hist)[i] = uint4{0u, 0u, 0u, 0u};
  if (tid == 0) {
    bin_at = kBins - 1;
    groups_in = (uint32_t)groups;
    nlist = 0;
    sm.ncand = 0;
  }
  mx = block_reduce<kP2Threads>(mx, [](float a, float c) { return fmaxf(a, c); }, fpart);
  double sum = 0.0;
  const bool finite_max = mx > -__builtin_inff() && mx < __builtin_inff();
  if (finite_max) {
    // The first bin B at which kk groups have a maximum within it (scanned below).
#pragma unroll
    for (int e = 0; e < GPT; ++e)
      count_bin(hist, dist_bin(mx, gv[e]), tid + kP2Threads * e < groups);
    auto add = [&](const f4 c) {
      if (c.x > -__builtin_inff()) sum += ((double)c.y + c.z) * exp((double)c.x - (double)mx);
    };
    if (tid < chunks) add(st0);
    for (int c = tid + kP2Threads; c < chunks; c += kP2Threads)
      add(*reinterpret_cast<const f4*>(st + c * 4));
  }
  sum = block_reduce<kP2Threads>(sum, [](double a, double c) { return a + c; }, dpart);
  const bool uniform = !finite_max || !(sum > 0.0) || !(sum < __builtin_inf());
  int32_t* oid = ids + r * kk;
  float* opr = probs + r * kk;
  if (uniform) {
    const float u = 1.0f / (float)n;
    for (int j = tid; j < kk; j += kP2Threads) {
      oid[j] = j;
      opr[j] = u;
    }
    return;
  }
  {
    constexpr int BPT = kBins / kP2Threads;
    uint32_t h[BPT], local = 0;
#pragma unroll
    for (int t = 0; t < BPT; ++t) local += h[t] = hist[tid * BPT + t];
    uint32_t incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t o = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += o;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    for (int w = 0; w < wave; ++w) before += wsum[w];
    uint32_t run = before + incl - local;
#pragma unroll
    for (int t = 0; t < BPT; ++t) {
      if (run < (uint32_t)kk && (uint32_t)kk <= run + h[t]) {
        bin_at = (uint32_t)(tid * BPT + t);
        groups_in = run + h[t];
      }
      run += h[t];
    }
  }
  __syncthreads();
  uint32_t bin = bin_at;
  uint32_t ngroups = groups_in;
  if (((int64_t)ngroups << gshift) <= kP2Keys) {
#pragma unroll
    for (int e = 0; e < GPT; ++e) {
      const int gi = tid + kP2Threads * e;
      if (gi < groups && dist_bin(mx, gv[e]) <= bin) list[atomicAdd(&nlist, 1u)] = gi;
    }
    __syncthreads();
  } else {
    // Massive ties: the kk groups of largest maximum, ties to the lower group.
    uint64_t gk[GPT];
#pragma unroll
    for (int e = 0; e < GPT; ++e) {
      const int gi = tid + kP2Threads * e;
      gk[e] = gi < groups ? topk_key(gv[e], (uint32_t)gi) : 0;
    }
    select_top<kP2Threads, GPT>(gk, kk, top, sm);
    ngroups = (uint32_t)(kk < groups ? kk : groups);
    for (int j = tid; j < (int)ngroups; j += kP2Threads) list[j] = (int)~(uint32_t)top[j];
    if (tid == 0) sm.ncand = 0;
    __syncthreads();
  }
  // Their values; those within the bin are candidates (all kk winners are).
  constexpr int PER = kP2Keys / kP2Threads;
  const int total = (int)(ngroups << gshift);
  const float* row = x + r * n;
  auto index_of = [&](int j) {
    return ((int64_t)list[j >> gshift] << gshift) + (j & ((1 << gshift) - 1));
  };
  uint64_t key[PER];
  float val[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) {  // all loads in flight
    val[e] = 0.0f;
    if (kP2Threads * e < total) val[e] = row[min(index_of(min(tid + kP2Threads * e, total - 1)), n - 1)];
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int j = tid + kP2Threads * e;
    key[e] = 0;
    if (j < total) {
      const int64_t i = index_of(j);
      if (i < n) {
        float t = val[e];
        if (scale) t = scaled_logit(t, inv_temp);
        if (dist_bin(mx, t) <= bin) {
          key[e] = topk_key(t, (uint32_t)i);
          const uint32_t slot = atomicAdd(&sm.ncand, 1u);
          if (slot < 256u) sm.cand[slot] = key[e];
        }
      }
    }
  }
  __syncthreads();
  const uint32_t ncand = sm.ncand;
  if (ncand <= 256u) {
    // 4 threads a candidate count the larger keys: its rank.
    const int c = tid >> 2;
    const uint64_t mine = c < (int)ncand ? sm.cand[c] : 0;
    int rank = 0;
    if (mine != 0)
      for (int j = tid & 3; j < (int)ncand; j += 4) rank += sm.cand[j] > mine;
    rank += __shfl_xor(rank, 1, 64);
    rank += __shfl_xor(rank, 2, 64);
    if (mine != 0 && (tid & 3) == 0 && rank < kk) top[rank] = mine;
    __syncthreads();
  } else {
    select_top<kP2Threads, PER>(key, kk, top, sm);
  }
  for (int j = tid; j < kk; j += kP2Threads) {
    const uint64_t kv = top[j];
    oid[j] = (int32_t)~(uint32_t)kv;
    opr[j] = (float)(exp((double)key_value(kv) - (double)mx) / sum);
  }
}

}  // namespace

int topk_chunks(int64_t n) { return (int)((n + kChunk - 1) / kChunk); }

int topk_max_n(int k) {
  // The values of k groups must fit pass 2's registers; kept at chunks * k <= kP2Keys.
  return k <= 0 ? 0 : (kP2Keys / k) * kChunk;
}

hipError_t launch_top_tokens(const float* x, int rows, int64_t n, int top_n, float temperature,
                             int32_t* ids, float* probs, float* workspace, hipStream_t stream) {
  const int kk = (int)(top_n < n ? top_n : n);
  if (rows <= 0 || rows > 65535 || n <= 0 || top_n <= 0 || top_n > kTopTokensMax ||
      n > topk_max_n(kk))
    return hipErrorInvalidValue;
  const int chunks = topk_chunks(n);
  const int gpc = chunk_groups(kk);
  // Pass 2 groups: gm written maxima each, at most kP2Groups (n / (2048 / gpc) is at
  // most 4 kP2Groups for an accepted n, so kk groups hold at most kP2Keys values).
  int gm = 1, gshift = 0;
  while ((int64_t)chunks * gpc > (int64_t)gm * kP2Groups) gm <<= 1;
  while ((1 << gshift) < kChunk / gpc * gm) ++gshift;
  if (((int64_t)kk << gshift) > kP2Keys) return hipErrorInvalidValue;
  float* maxima = workspace;
  float* stats = workspace + (size_t)rows * chunks * gpc;
  const bool scale = temperature > 0.0f && temperature != 1.0f;
  const float inv_temp = scale ? 1.0f / temperature : 1.0f;
  hipLaunchKernelGGL(topk_chunks_kernel, dim3((unsigned)chunks, (unsigned)rows), dim3(kP1Threads),
                     0, stream, x, n, gpc, inv_temp, scale ? 1 : 0, maxima, stats);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(topk_final_kernel, dim3((unsigned)rows), dim3(kP2Threads), 0, stream, x,
                     maxima, stats, chunks, gpc, gm, gshift, n, kk, inv_temp, scale ? 1 : 0, ids,
                     probs);
  return hipGetLastError();
}

size_t top_tokens_workspace_floats(int rows, int64_t n, int top_n) {
  const int kk = (int)(top_n < n ? top_n : n);
  return (size_t)rows * topk_chunks(n) * (size_t)(chunk_groups(kk) + 4);
}

}  // namespace mle
