// LSD radix sort kernels (device code), shared by radix.hip and the
// tuning probes. See radix.hip for the pipeline description.
#pragma once

#include "device_common.hpp"

namespace msv {

constexpr int kRadixIpt = 16;     // keys per thread in a pass tile
constexpr int kLookbackBatch = 4;  // predecessors a onesweep look-back step reads
constexpr int kRadixBins = 256;   // 8-bit digits

// Element moved by the passes: the key (1 or 2 dwords) followed by the value
// (0, 1 or 2 dwords). Between passes elements are kept interleaved (AoS), so
// each pass reorders one array and writes one stream of runs; the first pass
// reads the caller's separate key/value arrays and the last writes them.
template <int EW>
struct alignas(4) Elem {
  uint32_t w[EW];
};

template <typename K, int EW>
__device__ inline K elem_key(const Elem<EW>& e) {
  if constexpr (sizeof(K) == 4) return bit_cast<K>(e.w[0]);
  else return bit_cast<K>(((uint64_t)e.w[1] << 32) | e.w[0]);
}

struct RadixPass {
  uint32_t active;
  uint32_t shift;  // a multiple of 8
  uint32_t in_aos;   // source is an element array (else separate keys/values)
  uint32_t out_aos;  // destination is an element array
  const void* src_k;
  const void* src_v;
  void* dst_k;
  void* dst_v;
};

// Lanes of the wave holding a valid digit equal to ours (the low DBITS bits of
// d). One ballot per digit bit; a lane differs from us where its ballot bit
// differs from our own bit, so the differences are collected with 32-bit
// XOR/OR against our bit spread to 0 / all-ones (signed bit extract).
template <int DBITS>
__device__ inline uint64_t match_digit(uint32_t d, bool valid) {
  uint32_t diff_lo = 0, diff_hi = 0;
#pragma unroll
  for (int b = 0; b < DBITS; ++b) {
    const uint32_t s = (uint32_t)__builtin_amdgcn_sbfe((int)d, b, 1);
    const uint64_t m = ballot(s != 0);
    diff_lo |= (uint32_t)m ^ s;
    diff_hi |= (uint32_t)(m >> 32) ^ s;
  }
  return ballot(valid) & ~(((uint64_t)diff_hi << 32) | diff_lo);
}

static __global__ void fill_u32_kernel(uint32_t* p, uint32_t n, uint32_t v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// 1. First upsweep (pass 0's digit counts, see 3a) from the caller's keys,
//    which also records per tile the OR and the AND of the keys' order
//    words: a digit position on which OR ^ AND is zero holds one value for
//    every key, and its pass is skipped. (An all-digit histogram would need
//    one LDS atomic per key per digit; two bitwise reductions per tile do.)
template <typename K, int MODE, int BLOCK, int IPT = kRadixIpt>
__global__ __launch_bounds__(BLOCK) void radix_upsweep0_kernel(const K* __restrict__ keys,
                                                              uint32_t n, uint32_t ntiles,
                                                              uint32_t* __restrict__ counts,
                                                              uint64_t* __restrict__ orand) {
  using U = typename Bits<K>::U;
  constexpr int NW = BLOCK / kWave;
  constexpr uint32_t TILE = (uint32_t)BLOCK * IPT;
  __shared__ uint32_t s_cnt[NW][kRadixBins];
  __shared__ uint64_t s_or[NW], s_and[NW];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid / 64u;
  for (uint32_t i = tid; i < NW * kRadixBins; i += BLOCK) (&s_cnt[0][0])[i] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * TILE;
  uint64_t o = 0, a = ~0ull;
  uint32_t dig[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const size_t i = base + (size_t)j * BLOCK + tid;
    const U w = order_bits<K, MODE>(keys[i < n ? i : (size_t)n - 1]);
    const bool ok = i < n;
    o |= ok ? (uint64_t)w : 0ull;
    a &= ok ? (uint64_t)w : ~0ull;
    dig[j] = ok ? ((uint32_t)w & 0xffu) : 0x100u;
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (dig[j] < 0x100u) atomicAdd(&s_cnt[wid][dig[j]], 1u);
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    o |= __shfl_xor(o, m);
    a &= __shfl_xor(a, m);
  }
  if (lane == 0) {
    s_or[wid] = o;
    s_and[wid] = a;
  }
  __syncthreads();
  for (uint32_t d = tid; d < (uint32_t)kRadixBins; d += BLOCK) {
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) c += s_cnt[w][d];
    counts[(size_t)d * ntiles + blockIdx.x] = c;
  }
  if (tid == 0) {
    uint64_t ro = 0, ra = ~0ull;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      ro |= s_or[w];
      ra &= s_and[w];
    }
    orand[2 * (size_t)blockIdx.x] = ro;
    orand[2 * (size_t)blockIdx.x + 1] = ra;
  }
}

// 2. Pass plan: which digit positions need a pass (a position on which the
//    OR and the AND of all order words agree is skipped) and the source and
//    destination of each remaining pass: caller arrays -> element buffer A0
//    -> A1 -> A0 ... -> caller arrays. `orand` holds (OR, AND) per tile of
//    the first upsweep.
template <int P, bool SOA = false>
__global__ __launch_bounds__(kRadixBins) void radix_plan_kernel(
    const uint64_t* __restrict__ orand, uint32_t ntiles, uint32_t n, RadixPass* __restrict__ table,
    const void* in_k, const void* in_v, void* out_k, void* out_v, void* aos0, void* aos1) {
  __shared__ uint32_t s_trivial[P];
  __shared__ uint64_t s_or[kRadixBins / kWave], s_and[kRadixBins / kWave];
  const uint32_t t = threadIdx.x, lane = t & 63u, wid = t >> 6;
  uint64_t o = 0, a = ~0ull;
  for (uint32_t q = t; q < ntiles; q += kRadixBins) {
    o |= orand[2 * (size_t)q];
    a &= orand[2 * (size_t)q + 1];
  }
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    o |= __shfl_xor(o, m);
    a &= __shfl_xor(a, m);
  }
  if (lane == 0) {
    s_or[wid] = o;
    s_and[wid] = a;
  }
  __syncthreads();
  if (t == 0) {
    uint64_t ro = 0, ra = ~0ull;
    for (int w = 0; w < kRadixBins / kWave; ++w) {
      ro |= s_or[w];
      ra &= s_and[w];
    }
    const uint64_t varying = ro ^ ra;
    for (int p = 0; p < P; ++p) s_trivial[p] = ((varying >> (8 * p)) & 0xffu) == 0 ? 1u : 0u;
  }
  __syncthreads();
  if (t == 0) {
    int active = 0;
    for (int p = 0; p < P; ++p) active += s_trivial[p] ? 0 : 1;
    // All digits constant (all keys equal): one pass still moves the data.
    const bool force_last = active == 0;
    if (force_last) active = 1;
    int j = 0;
    for (int p = 0; p < P; ++p) {
      RadixPass rp;
      rp.shift = 8u * (uint32_t)p;
      rp.active = (!s_trivial[p] || (force_last && p == P - 1)) ? 1u : 0u;
      rp.in_aos = rp.out_aos = 0;
      rp.src_k = rp.src_v = nullptr;
      rp.dst_k = rp.dst_v = nullptr;
      if (rp.active) {
        // SOA: an intermediate buffer holds the n keys followed by the values.
        rp.in_aos = !SOA && j > 0;
        rp.out_aos = !SOA && j < active - 1;
        if (j == 0) {
          rp.src_k = in_k;
          rp.src_v = in_v;
        } else {
          char* b = (char*)(((j - 1) & 1) ? aos1 : aos0);
          rp.src_k = b;
          rp.src_v = SOA ? b + (size_t)n * P : nullptr;
        }
        if (j == active - 1) {
          rp.dst_k = out_k;
          rp.dst_v = out_v;
        } else {
          char* b = (char*)((j & 1) ? aos1 : aos0);
          rp.dst_k = b;
          rp.dst_v = SOA ? b + (size_t)n * P : nullptr;
        }
        ++j;
      }
      table[p] = rp;
    }
  }
}

template <typename K, int EW>
__device__ inline K load_key(const RadixPass& rp, size_t i) {
  if (rp.in_aos) return elem_key<K, EW>(((const Elem<EW>*)rp.src_k)[i]);
  return ((const K*)rp.src_k)[i];
}

template <typename K, int EW>
__device__ inline Elem<EW> load_elem(const RadixPass& rp, size_t i) {
  if (rp.in_aos) return ((const Elem<EW>*)rp.src_k)[i];
  Elem<EW> e;
  const K k = ((const K*)rp.src_k)[i];
  if constexpr (sizeof(K) == 4) {
    e.w[0] = bit_cast<uint32_t>(k);
  } else {
    const uint64_t u = bit_cast<uint64_t>(k);
    e.w[0] = (uint32_t)u;
    e.w[1] = (uint32_t)(u >> 32);
  }
  constexpr int KW = sizeof(K) / 4;
#pragma unroll
  for (int v = 0; v < EW - KW; ++v) e.w[KW + v] = ((const uint32_t*)rp.src_v)[i * (EW - KW) + v];
  return e;
}

template <typename K, int EW>
__device__ inline void store_elem(const RadixPass& rp, size_t i, const Elem<EW>& e) {
  if (rp.out_aos) {
    ((Elem<EW>*)rp.dst_k)[i] = e;
    return;
  }
  constexpr int KW = sizeof(K) / 4;
  ((K*)rp.dst_k)[i] = elem_key<K, EW>(e);
#pragma unroll
  for (int v = 0; v < EW - KW; ++v) ((uint32_t*)rp.dst_v)[i * (EW - KW) + v] = e.w[KW + v];
}

// 3. Per-pass reduce-then-scan over tiles of BLOCK * IPT keys.
//  3a. upsweep: digit counts of every tile, digit-major
//      (counts[d * ntiles + tile]), so that one exclusive scan of `counts`
//      yields the global position of each (digit, tile) run.
template <typename K, int MODE, int EW, int BLOCK, int IPT = kRadixIpt>
__global__ __launch_bounds__(BLOCK) void radix_upsweep_kernel(const RadixPass* __restrict__ table,
                                                             int pass, uint32_t n, uint32_t ntiles,
                                                             uint32_t* __restrict__ counts) {
  constexpr int NW = BLOCK / kWave;
  constexpr uint32_t TILE = (uint32_t)BLOCK * IPT;
  constexpr int KW = sizeof(K) / 4;
  static_assert(IPT % 4 == 0, "groups of 4 elements");
  __shared__ uint32_t s_cnt[NW][kRadixBins];
  const RadixPass rp = table[pass];
  if (!rp.active) return;
  const uint32_t tid = threadIdx.x, wid = tid / 64u;
  for (uint32_t i = tid; i < NW * kRadixBins; i += BLOCK) (&s_cnt[0][0])[i] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * TILE;
  const uint32_t shift = rp.shift;
  const bool full = base + TILE <= n;
  // A full tile whose source is 16-byte aligned is read as groups of 4 whole
  // elements (EW dwordx4 loads for an element array, KW for a key array);
  // counting does not depend on the order in which keys are seen.
  const bool vec = full && (((uintptr_t)rp.src_k & 15u) == 0);
  uint32_t dig[IPT];
  if (vec) {
#pragma unroll
    for (int r = 0; r < IPT / 4; ++r) {
      const size_t g = base / 4 + (size_t)r * BLOCK + tid;  // group of elements 4g .. 4g+3
      uint32_t w[4 * (EW > KW ? EW : KW)];
      const int QW = rp.in_aos ? EW : KW;  // dwordx4 loads per group
      const uint4* q = (const uint4*)rp.src_k + g * (size_t)QW;
#pragma unroll
      for (int t = 0; t < (EW > KW ? EW : KW); ++t) {
        if (t < QW) {
          const uint4 v = q[t];
          w[4 * t] = v.x;
          w[4 * t + 1] = v.y;
          w[4 * t + 2] = v.z;
          w[4 * t + 3] = v.w;
        }
      }
      const int stride = rp.in_aos ? EW : KW;  // dwords per element in the group
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        K k;
        if constexpr (KW == 1) {
          k = bit_cast<K>(w[m * stride]);
        } else {
          k = bit_cast<K>(((uint64_t)w[m * stride + 1] << 32) | w[m * stride]);
        }
        dig[4 * r + m] = (uint32_t)(order_bits<K, MODE>(k) >> shift) & 0xffu;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const size_t i = base + (size_t)j * BLOCK + tid;
      dig[j] = i < n ? ((uint32_t)(order_bits<K, MODE>(load_key<K, EW>(rp, i)) >> shift) & 0xffu)
                     : 0x100u;
    }
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (dig[j] < 0x100u) atomicAdd(&s_cnt[wid][dig[j]], 1u);
  __syncthreads();
  for (uint32_t d = tid; d < (uint32_t)kRadixBins; d += BLOCK) {
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) c += s_cnt[w][d];
    counts[(size_t)d * ntiles + blockIdx.x] = c;
  }
}

//  3b. downsweep: rank the tile's keys stably, reorder the elements through
//      LDS into digit-sorted runs, and write the runs to their offsets
//      (offsets[d * ntiles + tile], the exclusive scan of `counts`).
template <typename K, int MODE, int EW, int BLOCK, int IPT = kRadixIpt>
__global__ __launch_bounds__(BLOCK) void radix_downsweep_kernel(
    const RadixPass* __restrict__ table, int pass, const uint32_t* __restrict__ offsets,
    uint32_t n, uint32_t ntiles) {
  constexpr int NW = BLOCK / kWave;
  constexpr uint32_t TILE = (uint32_t)BLOCK * IPT;
  __shared__ Elem<EW> s_el[TILE];
  __shared__ uint32_t s_hist[NW][kRadixBins];     // per-wave counts, then wave offsets
  __shared__ uint32_t s_tile_start[kRadixBins];   // in-tile start of each digit
  __shared__ uint32_t s_goff[kRadixBins];         // global position - in-tile position
  __shared__ uint32_t s_wsum[kRadixBins / kWave];

  const RadixPass rp = table[pass];
  if (!rp.active) return;

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid / 64u;
  const bool digit_thread = tid < (uint32_t)kRadixBins;
  for (uint32_t i = tid; i < NW * kRadixBins; i += BLOCK) (&s_hist[0][0])[i] = 0;
  __syncthreads();
  const uint32_t tile = blockIdx.x;
  const size_t base = (size_t)tile * TILE + (size_t)wid * (kWave * IPT);
  const uint32_t shift = rp.shift;

  Elem<EW> el[IPT];
  uint32_t dig[IPT];
  uint32_t rank[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const size_t i = base + (size_t)j * kWave + lane;
    if (i < n) {
      el[j] = load_elem<K, EW>(rp, i);
      dig[j] = (uint32_t)(order_bits<K, MODE>(elem_key<K, EW>(el[j])) >> shift) & 0xffu;
    } else {
      dig[j] = 0x100u;
    }
  }
  uint32_t goff = 0;
  if (digit_thread) goff = offsets[(size_t)tid * ntiles + tile];

  // Wave-level multi-split: rank each key among the wave's earlier keys with
  // the same digit (input order: j-major, lane-minor).
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t d = dig[j];
    const bool valid = d < 0x100u;
    const uint64_t peers = match_digit<8>(d, valid);
    uint32_t before = 0;
    if (valid) before = s_hist[wid][d];
    const uint32_t below = (uint32_t)__builtin_popcountll(peers & lt);
    if (valid && below == 0) s_hist[wid][d] = before + (uint32_t)__builtin_popcountll(peers);
    rank[j] = before + below;
  }
  __syncthreads();

  // Per digit (thread t <-> digit t): wave offsets, tile count, tile start.
  uint32_t cnt = 0;
  if (digit_thread) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const uint32_t c = s_hist[w][tid];
      s_hist[w][tid] = cnt;
      cnt += c;
    }
  }
  uint32_t incl = 0;
  if (digit_thread) {
    incl = wave_inclusive_scan<uint32_t, OP_ADD>(cnt);
    if (lane == 63) s_wsum[wid] = incl;
  }
  __syncthreads();
  if (digit_thread) {
    uint32_t woff = 0;
    for (uint32_t k = 0; k < wid; ++k) woff += s_wsum[k];
    const uint32_t tstart = woff + incl - cnt;
    s_tile_start[tid] = tstart;
    s_goff[tid] = goff - tstart;
  }
  __syncthreads();

  // Reorder elements into digit-sorted runs in LDS, then write the runs out.
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (dig[j] < 0x100u) s_el[s_tile_start[dig[j]] + s_hist[wid][dig[j]] + rank[j]] = el[j];
  __syncthreads();
  const uint32_t tile_n = (uint32_t)min((size_t)TILE, (size_t)n - (size_t)tile * TILE);
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const uint32_t i = tid + (uint32_t)q * BLOCK;
    if (i < tile_n) {
      const Elem<EW> e = s_el[i];
      const uint32_t d = (uint32_t)(order_bits<K, MODE>(elem_key<K, EW>(e)) >> shift) & 0xffu;
      store_elem<K, EW>(rp, (size_t)s_goff[d] + i, e);
    }
  }
}


// ---- onesweep: one histogram pass, then one pass per digit ---------------------
// How a long sort of 8-byte keys goes (9).
struct RadixRepair {
  uint32_t low;   // passes run from this digit; 0: all of them do
  uint32_t redo;  // the repair gave up: every digit's pass runs
  uint32_t near;  // 8 - the highest digit in which a key differs from a hot key that
                  // it shares the digits from the looked-at one on with; 0: none does
};
constexpr uint32_t kSample = 8192, kSamples = 16;  // keys of a sample (most), samples
constexpr uint32_t kHots = 128;                    // most hot keys of a sample
constexpr uint32_t kLows = 5;                      // digits 0 .. 4 are looked at (at least 4 get a pass)
struct RadixSample {
  uint32_t clash[kLows][kSamples];  // [low]: pairs of different keys that share the digits from low on
  uint32_t varying[kSamples];   // bit p: digit p varies
  uint32_t most[kSamples];      // how often the most frequent key is there
  uint32_t hots[kSamples];      // keys that are there at least 4 times (kHots at most),
  uint32_t heavy[kSamples];     // and first those that are there 16 times (all of them counted)
  uint64_t hot[kSamples][kHots];
};
constexpr int kFirstPasses = 7;  // most digits that get a pass before a repair
// Keys of a sample of n keys (a quarter of them are looked at in 9 us, all in 30),
// and the pairs that may clash in all samples.
__device__ inline uint32_t sample_size(uint32_t n) { return n >= 1u << 25 ? kSample : kSample / 4; }
__device__ inline uint32_t clash_limit(uint32_t n) {
  const uint32_t size = sample_size(n), pairs = kSamples * (size / 2) * size;
  return n >= 1u << 29 ? 0u : max(1u, pairs / 4 / n);
}

// The digit that the passes of n keys start from, or 0, by the rules of (9).
__device__ inline uint32_t choose_low(uint32_t n, uint32_t varying, bool hot, const uint32_t* clash) {
  const uint32_t bits = 4 + 32 - (uint32_t)__builtin_clz(n - 1);
  uint32_t want = (bits + 7) / 8 + (hot ? 1 : 0), low = 8;
  while (low > 0 && want > 0) want -= varying >> --low & 1u;
  const uint32_t limit = clash_limit(n);
  for (; low > 0; --low)
    if ((varying >> (low - 1) & 1u) && clash[low] <= limit) break;
  return low;
}

// The samples' sums (all threads of the block call; s_sum: kLows + 2 words).
__device__ inline void sum_samples(const RadixSample* __restrict__ sample, uint32_t* s_sum) {
  const uint32_t tid = threadIdx.x;
  if (tid < kLows + 2) s_sum[tid] = 0;
  __syncthreads();
  if (tid < kLows * kSamples) atomicAdd(&s_sum[tid / kSamples], (&sample->clash[0][0])[tid]);
  if (tid < kSamples) {
    atomicOr(&s_sum[kLows], sample->varying[tid]);
    atomicMax(&s_sum[kLows + 1], sample->most[tid]);
  }
  __syncthreads();
}
__device__ inline uint32_t sampled_low(uint32_t n, const uint32_t* s_sum) {
  return choose_low(n, s_sum[kLows], s_sum[kLows + 1] > sample_size(n) / 64, s_sum);
}

// The samples' hot keys in LDS, two to a bucket of the digits that the passes
// may start from. Returns 8 times that digit, or 0 when there is nothing to look
// at; *lost: a heavy key has no room (others are just not looked at). An empty
// place holds the first hot key: what shares its digits is near a hot key in any
// case.
constexpr uint32_t kHotBuckets = 256;  // (with 512 a CU holds three blocks of the histogram, not four)
__device__ inline uint32_t hot_bucket(uint64_t word, uint32_t shift) {  // shift in 8 .. 32
  const uint32_t high = (uint32_t)(word >> 32), rest = shift < 32 ? (uint32_t)word >> (shift & 31u) : 0u;
  return ((high ^ rest ^ (rest << 13)) * 2654435761u) >> 24;
}
template <int BLOCK>
__device__ inline uint32_t hot_table(const RadixSample* __restrict__ sample, uint32_t n, uint64_t* s_hot,
                                     bool* lost) {
  constexpr int PER = (int)(kSamples * kHots / BLOCK);
  static_assert(BLOCK % kHots == 0 && PER > 0, "a thread's keys are of one place in their samples");
  __shared__ uint32_t s_sum[kLows + 2], s_hots[kSamples], s_heavy[kSamples], s_first;
  const uint32_t at = threadIdx.x % kHots, sub = threadIdx.x / kHots;
  uint64_t word[PER];  // (those past a sample's hot keys are not used)
#pragma unroll
  for (int j = 0; j < PER; ++j) word[j] = sample->hot[sub + j * (BLOCK / kHots)][at];
  if (threadIdx.x < kSamples) {
    s_hots[threadIdx.x] = sample->hots[threadIdx.x];
    s_heavy[threadIdx.x] = sample->heavy[threadIdx.x];
  }
  if (threadIdx.x == 0) s_first = kSamples;
  sum_samples(sample, s_sum);
  if (threadIdx.x < kSamples && s_hots[threadIdx.x] > 0) atomicMin(&s_first, threadIdx.x);
  __syncthreads();
  const uint32_t shift = 8 * sampled_low(n, s_sum), first = s_first;
  *lost = false;
  if (shift == 0 || first == kSamples) return 0;
  const uint64_t empty = sample->hot[first][0];
  for (uint32_t i = threadIdx.x; i < 2 * kHotBuckets; i += BLOCK) s_hot[i] = empty;
  __syncthreads();
  for (int light = 0; light < 2; ++light) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t s = sub + j * (BLOCK / kHots);
      *lost = *lost || s_heavy[s] > kHots;
      if (at >= s_hots[s] || (at >= s_heavy[s]) != (light == 1)) continue;
      const uint64_t w = word[j];
      unsigned long long* to = (unsigned long long*)&s_hot[2 * hot_bucket(w, shift)];
      uint64_t was = atomicCAS(to, (unsigned long long)empty, (unsigned long long)w);
      if (was != empty && was != w) was = atomicCAS(to + 1, (unsigned long long)empty, (unsigned long long)w);
      *lost = *lost || (was != empty && was != w && light == 0);
    }
    __syncthreads();
  }
  return shift;
}

// 5. Global digit histograms of every digit position in one read of the keys:
//    hist[p * 256 + d] = number of keys whose digit p is d. Each thread reads
//    16 keys per step with 16-byte loads (all in flight before the first is
//    counted), each wave counts into its own LDS histogram, then the block adds
//    its counts to the global histogram. On a full step the wave ORs every
//    key's difference from its first key once (a wave reduction), and a digit
//    position that is constant over the step's 1024 keys (constant bytes are
//    common: small keys, a constant top byte) is counted by one add; the other
//    positions take one LDS add per key and no per-key test (per key and
//    position, a uniformity test had cost more instructions than the add).
//    (Its last block making the plan, to save that launch, gained 0-2 us.)
//    SAMPLE: a long sort of 8-byte keys (9), whose hot keys every key is
//    compared with on the way.
template <typename K, int MODE, int BLOCK, bool SAMPLE = false>
__global__ __launch_bounds__(BLOCK) void radix_hist_kernel(const K* __restrict__ keys, uint32_t n,
                                                          uint32_t* __restrict__ hist,
                                                          const RadixSample* __restrict__ sample,
                                                          RadixRepair* __restrict__ rep) {
  using U = typename Bits<K>::U;
  constexpr int P = sizeof(K);
  constexpr int KPT = 16;                   // keys per thread per step
  constexpr int V = 16 / sizeof(K);         // keys per 16-byte load
  constexpr int NW = BLOCK / kWave;
  __shared__ uint32_t s_hw[NW][P * kRadixBins];  // per-wave histograms
  const uint32_t tid = threadIdx.x;
  uint32_t* s_h = s_hw[tid / kWave];
  for (uint32_t i = tid; i < (uint32_t)(NW * P * kRadixBins); i += BLOCK) (&s_hw[0][0])[i] = 0;
  __syncthreads();
  uint32_t shift = 0, near = 0;  // shift 0: no hot keys to compare with
  __shared__ __align__(16) uint64_t s_hot[SAMPLE ? 2 * kHotBuckets : 2];
  if constexpr (SAMPLE) {
    bool lost;
    shift = hot_table<BLOCK>(sample, n, s_hot, &lost);
    if (lost) near = 8;
  }
  auto compare = [&](U word) {
    if constexpr (SAMPLE) {
      const uint32_t b = hot_bucket((uint64_t)word, shift);
      const uint4 hot = *reinterpret_cast<const uint4*>(s_hot + 2 * b);
      const uint32_t low_word = (uint32_t)word, high = (uint32_t)((uint64_t)word >> 32);
      // The same digits from shift (8 .. 32) on, but not the same key: the
      // difference is in [1, 2^shift).
      const uint32_t x0 = low_word ^ hot.x, x1 = low_word ^ hot.z, span = 0xffffffffu >> (32 - shift);
      if (high == hot.y && x0 - 1 < span) near = max(near, (32 + (uint32_t)__builtin_clz(x0)) / 8 + 1);
      if (high == hot.w && x1 - 1 < span) near = max(near, (32 + (uint32_t)__builtin_clz(x1)) / 8 + 1);
    }
  };
  const bool aligned = ((uintptr_t)keys & 15u) == 0;
  const size_t step = (size_t)gridDim.x * BLOCK * KPT;
  for (size_t b0 = (size_t)blockIdx.x * BLOCK * KPT; b0 < n; b0 += step) {
    U w[KPT];
    bool ok[KPT];
    // Row-striped: load r of thread t covers keys b0 + (r * BLOCK + t) * V ...
    if (aligned && b0 + (size_t)BLOCK * KPT <= n) {
#pragma unroll
      for (int r = 0; r < KPT / V; ++r) {
        const uint4 q = *reinterpret_cast<const uint4*>(keys + b0 + ((size_t)r * BLOCK + tid) * V);
        const uint32_t qq[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < V; ++k) {
          K key;
          if constexpr (sizeof(K) == 4) key = bit_cast<K>(qq[k]);
          else key = bit_cast<K>(((uint64_t)qq[2 * k + 1] << 32) | qq[2 * k]);
          w[r * V + k] = order_bits<K, MODE>(key);
        }
      }
      if (SAMPLE && shift != 0) {
#pragma unroll
        for (int j = 0; j < KPT; ++j) compare(w[j]);
      }
      // Bytes in which some key of the wave's step differs from its first key.
      uint32_t lo0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)w[0]);
      uint32_t hi0 = 0, xlo = 0, xhi = 0;
      if constexpr (sizeof(U) == 8)
        hi0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)w[0] >> 32));
#pragma unroll
      for (int j = 0; j < KPT; ++j) {
        xlo |= (uint32_t)w[j] ^ lo0;
        if constexpr (sizeof(U) == 8) xhi |= (uint32_t)((uint64_t)w[j] >> 32) ^ hi0;
      }
#pragma unroll
      for (int k = 1; k < kWave; k <<= 1) {
        xlo |= (uint32_t)__shfl_xor((int)xlo, k);
        if constexpr (sizeof(U) == 8) xhi |= (uint32_t)__shfl_xor((int)xhi, k);
      }
      xlo = (uint32_t)__builtin_amdgcn_readfirstlane((int)xlo);
      xhi = (uint32_t)__builtin_amdgcn_readfirstlane((int)xhi);
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const uint32_t sh = 8u * (uint32_t)(p & 3);
        const uint32_t diff = ((p < 4 ? xlo : xhi) >> sh) & 0xffu;
        if (diff == 0) {
          const uint32_t d0 = ((p < 4 ? lo0 : hi0) >> sh) & 0xffu;
          if (__lane_id() == 0) atomicAdd(&s_h[p * kRadixBins + d0], (uint32_t)(kWave * KPT));
        } else {
#pragma unroll
          for (int j = 0; j < KPT; ++j)
            atomicAdd(&s_h[p * kRadixBins + ((uint32_t)(w[j] >> (8 * p)) & 0xffu)], 1u);
        }
      }
      continue;
    } else {
#pragma unroll
      for (int r = 0; r < KPT / V; ++r)
#pragma unroll
        for (int k = 0; k < V; ++k) {
          const size_t i = b0 + ((size_t)r * BLOCK + tid) * V + k;
          ok[r * V + k] = i < n;
          w[r * V + k] = i < n ? order_bits<K, MODE>(keys[i]) : (U)0;
        }
    }
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      if (SAMPLE && shift != 0 && ok[j]) compare(w[j]);
      const uint64_t valid = ballot(ok[j]);
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const uint32_t d = (uint32_t)(w[j] >> (8 * p)) & 0xffu;
        const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
        if (ballot(ok[j] && d != d0) == 0) {
          if (__lane_id() == 0 && valid) atomicAdd(&s_h[p * kRadixBins + d0], (uint32_t)__builtin_popcountll(valid));
        } else if (ok[j]) {
          atomicAdd(&s_h[p * kRadixBins + d], 1u);
        }
      }
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < (uint32_t)(P * kRadixBins); i += BLOCK) {
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) c += s_hw[w][i];
    if (c) atomicAdd(&hist[i], c);
  }
  if constexpr (SAMPLE) {
    near = wave_reduce<uint32_t, OP_MAX>(near);
    if (near && (tid & 63u) == 0) atomicMax(&rep->near, near);
  }
}

// What the local sort (8) does after the first pass: sorts every run of equal
// digits `top` by the digits below it.
struct RadixLocal {
  uint32_t on;
  uint32_t top;
  RadixPass pass;  // its source and destination
};

// 6. Onesweep plan (one block of 256 threads): the exclusive scan of every
//    digit position's histogram (the global start of each digit in that
//    pass), which positions need a pass (a position whose histogram puts all
//    n keys in one bin is skipped), the pass table (the passes to run first;
//    sources and destinations as in the reduce-then-scan plan) and zeroed tile
//    counters.
//    local_max > 0: when at least three positions need a pass and no digit of
//    the highest holds more than local_max keys, only that position gets a
//    pass, and `local` the rest.
//    sample: the passes may start at a higher digit (9), chosen here into rep; a
//    second table then has the passes over every digit, for when the repair
//    gives up. These read what the first passes left in the output (equal keys
//    still in input order): the caller's arrays may have been written by then,
//    when a job sorts its keys or its values in place. (At least four digits are
//    passed over before a repair, so they are five or more.)
//    vofs = 0: the intermediate buffers hold interleaved elements; else each
//    holds the keys and, vofs bytes in, the values (the two-phase passes).
struct RadixPlan {
  const uint32_t* hist;     // [P][256]
  RadixPass* table;         // [P], or [2 P] with a sample
  uint32_t* gbase;          // [P][256]
  uint32_t* tile_counters;  // one to a launch of the passes, `launches` of them
  uint32_t launches;
  RadixLocal* local;
  uint32_t local_max;
  const RadixSample* sample;  // null: the passes start at digit 0
  RadixRepair* rep;
  const void *in_k, *in_v;
  void *out_k, *out_v, *aos0, *aos1;
  size_t vofs;
};

template <int P>
__global__ __launch_bounds__(kRadixBins) void radix_onesweep_plan_kernel(RadixPlan q, uint32_t n) {
  __shared__ uint32_t s_most[P], s_sum[kLows + 2];
  __shared__ uint32_t s_wsum[P][kRadixBins / kWave];
  const uint32_t t = threadIdx.x, lane = t & 63u, wid = t >> 6;
  if (t < (uint32_t)P) s_most[t] = 0;
  if (t < q.launches) q.tile_counters[t] = 0;
  if (P == 8 && q.sample) sum_samples(q.sample, s_sum);
  uint32_t c[P], incl[P];
#pragma unroll
  for (int p = 0; p < P; ++p) c[p] = q.hist[p * kRadixBins + t];
  __syncthreads();
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const uint32_t most = wave_reduce<uint32_t, OP_MAX>(c[p]);
    if (lane == 0) atomicMax(&s_most[p], most);
    incl[p] = wave_inclusive_scan<uint32_t, OP_ADD>(c[p]);
    if (lane == 63) s_wsum[p][wid] = incl[p];
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < P; ++p) {
    uint32_t woff = 0;
    for (uint32_t k = 0; k < wid; ++k) woff += s_wsum[p][k];
    q.gbase[p * kRadixBins + t] = woff + incl[p] - c[p];
  }
  // The first P threads write an entry of the table each, the next P of the second.
  if (t >= 2 * P) return;
  uint32_t varying = 0, hot = n, low = 0;
  for (int p = 0; p < P; ++p) {
    varying |= (s_most[p] < n ? 1u : 0u) << p;
    hot = min(hot, s_most[p]);
  }
  if (P == 8 && q.sample) {
    low = min(choose_low(n, varying, hot > n / 64, s_sum), sampled_low(n, s_sum));
    low = min(low, 8 - q.rep->near);
    const int passes = __builtin_popcount(varying >> low);
    if ((varying & ((1u << low) - 1)) == 0 || passes < 4 || passes > kFirstPasses) low = 0;
    if (t == 0) q.rep->low = low;
  } else if (t >= P) {
    return;
  }
  const bool split = q.vofs != 0, again = t >= P;
  const int active = __builtin_popcount(varying >> low), top = 31 - __builtin_clz(varying | 1u);
  const bool use_local = q.local_max > 0 && active >= 3 && s_most[top] <= q.local_max;
  if (t == 0) {
    q.local->on = use_local ? 1u : 0u;
    q.local->top = (uint32_t)top;
    q.local->pass = RadixPass{1u, 0u, split ? 0u : 1u, 0u,
                              q.aos0, split ? (char*)q.aos0 + q.vofs : nullptr, q.out_k, q.out_v};
  }
  uint32_t digits = again ? varying : (use_local ? 1u << top : (varying >> low << low));
  if (digits == 0) digits = 1u << (P - 1);  // all keys equal: one pass still moves the data
  const int passes = __builtin_popcount(digits), p = (int)(t % P);
  RadixPass* table = q.table + (again ? P : 0);
  if (p >= passes) table[p].active = 0;
  if (!(digits >> p & 1u)) return;
  const int j = __builtin_popcount(digits & ((1u << p) - 1));
  const bool to_out = j == passes - 1 && !use_local;
  char* src = (char*)(((j - 1) & 1) ? q.aos1 : q.aos0);
  char* dst = (char*)((j & 1) ? q.aos1 : q.aos0);
  RadixPass rp;
  rp.active = 1;
  rp.shift = 8u * (uint32_t)p;
  rp.in_aos = j > 0 && !split;
  rp.out_aos = !to_out && !split;
  rp.src_k = j == 0 ? (again ? q.out_k : q.in_k) : src;
  rp.src_v = j == 0 ? (again ? q.out_v : q.in_v) : (split ? src + q.vofs : nullptr);
  rp.dst_k = to_out ? q.out_k : dst;
  rp.dst_v = to_out ? q.out_v : (split ? dst + q.vofs : nullptr);
  table[j] = rp;
}

// Whether a onesweep pass over EW-word elements reorders keys and values in
// two phases (and keeps them in separate arrays between passes).
constexpr bool radix_split(int EW) { return EW >= 3; }

// 7. Onesweep pass: a block claims the next tile id from the pass's counter
//    (so every predecessor of a tile is already running), ranks its keys as
//    the downsweep does, publishes its per-digit counts as an aggregate, and
//    one thread per digit walks back over the predecessors' statuses (adding
//    aggregates until it meets an inclusive prefix), publishes its own
//    inclusive prefix and places the digit's run at
//    global start + prefix. A tile publishes its aggregate before it waits on
//    anything, so every walk ends.
//    What bounds it: the status rows that the look-back reads (2 KB per
//    predecessor, through the Infinity Cache), the partial lines at the ends of
//    the runs, and how far two blocks' phases overlap per CU. All shrink with
//    the tile, so a key takes as few as it can of the 64 registers per lane
//    that two 1024-thread blocks leave: the digit is taken from the key again
//    wherever it is used (held per key it cost a third of the tile), the
//    per-wave counts are 16-bit in LDS, and elements of 12 or 16 bytes hold
//    only their keys while they are ranked: they are reordered through LDS in
//    two phases, the keys and then the values, which are loaded in between.
//    Per pass, before -> now: 2^28 u32 + u32 1.75 (6144-key tiles) -> 1.32 ms
//    (8192), 2^27 u64 + u32 1.13 (5120) -> 0.86 ms (8192). Counting after the
//    ranking instead of by one LDS atomic per key before it: 1.38 and 0.91
//    (predecessors' counts come too late); 2, 6 or 8 predecessors a step: 1.36,
//    1.45, 2.44; keys and values of 8-byte elements in two phases (10240-key
//    tiles): 1.35.
template <typename K, int MODE, int EW, int BLOCK, int IPT = kRadixIpt>
__global__ __launch_bounds__(BLOCK, 8) void radix_onesweep_kernel(
    const RadixPass* __restrict__ table, int pass, int again, const RadixRepair* __restrict__ rep,
    const uint32_t* __restrict__ gbase, uint32_t* __restrict__ tile_counter,
    uint64_t* __restrict__ status, uint32_t gen, uint32_t n) {
  constexpr int NW = BLOCK / kWave;
  constexpr uint32_t TILE = (uint32_t)BLOCK * IPT;
  constexpr int KW = (int)sizeof(K) / 4, VW = EW - KW;
  static_assert(TILE <= 65535, "16-bit counts");
  using V = typename std::conditional<VW == 2, uint64_t, uint32_t>::type;
  constexpr bool kSplit = radix_split(EW);
  constexpr int MW = kSplit ? (KW > VW ? KW : VW) : EW;  // LDS words per element
  __shared__ __align__(16) uint32_t s_part[TILE * MW];
  __shared__ uint16_t s_hist[NW][kRadixBins];     // per-wave counts, then wave offsets
  __shared__ uint32_t s_tile_start[kRadixBins];   // in-tile start of each digit
  __shared__ uint32_t s_goff[kRadixBins];         // global position - in-tile position
  __shared__ uint32_t s_wsum[kRadixBins / kWave];
  __shared__ uint32_t s_cnt[kRadixBins];          // the tile's digit counts (early)
  __shared__ uint32_t s_tile;

  // After a repair (rep): pass `again` when it gave up, else `pass`, if any.
  if (rep && rep->redo) pass = again;
  if (pass < 0) return;
  const RadixPass rp = table[pass];
  if (!rp.active) return;

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid / 64u;
  const bool digit_thread = tid < (uint32_t)kRadixBins;
  for (uint32_t i = tid; i < NW * kRadixBins / 2; i += BLOCK)
    reinterpret_cast<uint32_t*>(&s_hist[0][0])[i] = 0;
  if (digit_thread) s_cnt[tid] = 0;
  if (tid == 0) s_tile = atomicAdd(tile_counter, 1u);
  __syncthreads();
  const uint32_t tile = s_tile;
  const size_t base = (size_t)tile * TILE + (size_t)wid * (kWave * IPT);
  const uint32_t shift = rp.shift;

  // The wave's keys are [base, base + left); key j of a lane is the lane's of
  // row j.
  const uint32_t left = base < n ? (uint32_t)min((size_t)n - base, (size_t)kWave * IPT) : 0u;
  auto valid = [&](int j) { return (uint32_t)j * kWave + lane < left; };
  auto digit = [&](const auto& e) {
    return (uint32_t)(order_bits<K, MODE>(elem_key<K, sizeof(e) / 4>(e)) >> shift) & 0xffu;
  };
  // Two phases: the keys only.
  constexpr int HW = kSplit ? KW : EW;
  Elem<HW> el[IPT];
  uint32_t rank[IPT];
  const K* src_k = (const K*)rp.src_k + base + lane;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    if (!valid(j)) continue;
    if constexpr (kSplit) el[j] = bit_cast<Elem<HW>>(src_k[j * kWave]);
    else el[j] = load_elem<K, EW>(rp, base + (size_t)j * kWave + lane);
  }
  uint32_t gstart = 0;
  if (digit_thread) gstart = gbase[shift / 8 * kRadixBins + tid];

  // The tile's digit counts first (LDS atomics), published at once as its
  // aggregate: successors walking back meet an aggregate instead of waiting
  // for this tile's ranking.
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (valid(j)) atomicAdd(&s_cnt[digit(el[j])], 1u);
  __syncthreads();
  uint64_t* my_status = status + (size_t)tile * kRadixBins + tid;
  uint32_t cnt = 0;
  if (digit_thread) {
    cnt = s_cnt[tid];
    st_agent(my_status, pack_status(gen, tile == 0 ? kFlagInc : kFlagAgg, 0, cnt));
  }

  // Wave-level multi-split, as in the downsweep. (The empty asm makes the
  // compiler form the digit again instead of keeping all of them.)
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    asm volatile("" : "+v"(el[j].w[0]));
    const uint32_t d = digit(el[j]);
    const uint64_t peers = match_digit<8>(d, valid(j));
    uint32_t before = 0;
    if (valid(j)) before = s_hist[wid][d];
    const uint32_t below = (uint32_t)__builtin_popcountll(peers & lt);
    if (valid(j) && below == 0)
      s_hist[wid][d] = (uint16_t)(before + (uint32_t)__builtin_popcountll(peers));
    rank[j] = before + below;
  }
  __syncthreads();

  // Per digit (thread t <-> digit t): wave offsets (their sum is cnt).
  if (digit_thread) {
    uint32_t acc = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const uint32_t c = s_hist[w][tid];
      s_hist[w][tid] = (uint16_t)acc;
      acc += c;
    }
  }
  uint32_t incl = 0;
  if (digit_thread) {
    incl = wave_inclusive_scan<uint32_t, OP_ADD>(cnt);
    if (lane == 63) s_wsum[wid] = incl;
  }
  __syncthreads();
  if (digit_thread) {
    uint32_t woff = 0;
    for (uint32_t k = 0; k < wid; ++k) woff += s_wsum[k];
    const uint32_t tstart = woff + incl - cnt;
    s_tile_start[tid] = tstart;
    // Look back: the number of keys with this digit in all earlier tiles,
    // reading kLookbackBatch predecessors per step (loads in flight
    // together); an unpublished predecessor is polled again from there.
    uint32_t prefix = 0;
    if (tile > 0) {
      constexpr int B = kLookbackBatch;
      int64_t q = (int64_t)tile - 1;  // nearest predecessor not yet added
      for (;;) {
        uint64_t w[B];
#pragma unroll
        for (int k = 0; k < B; ++k)
          w[k] = q - k >= 0 ? ld_agent(status + (size_t)(q - k) * kRadixBins + tid) : 0ull;
        int used = 0;
        bool done = false;
#pragma unroll
        for (int k = 0; k < B; ++k) {
          if (done || used < k) continue;
          const uint32_t f = status_flag(w[k], gen);
          if (f == 0) continue;  // not published yet (tile 0 always is)
          prefix += (uint32_t)w[k];
          used = k + 1;
          done = f == kFlagInc;
        }
        if (done) break;
        q -= used;
        if (used == 0) __builtin_amdgcn_s_sleep(1);
      }
      st_agent(my_status, pack_status(gen, kFlagInc, 0, prefix + cnt));
    }
    s_goff[tid] = gstart + prefix - tstart;
  }
  __syncthreads();

  // Reorder into digit-sorted runs in LDS, then write the runs out (two
  // phases: the keys first, each output position's digit kept for the values,
  // then the values).
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    if (!valid(j)) continue;
    asm volatile("" : "+v"(el[j].w[0]));
    const uint32_t d = digit(el[j]);
    rank[j] += s_tile_start[d] + s_hist[wid][d];
  }
  const uint32_t tile_n = (uint32_t)min((size_t)TILE, (size_t)n - (size_t)tile * TILE);
  if constexpr (!kSplit) {
    Elem<EW>* s_el = reinterpret_cast<Elem<EW>*>(s_part);
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if (valid(j)) s_el[rank[j]] = el[j];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const uint32_t i = tid + (uint32_t)q * BLOCK;
      if (i < tile_n) {
        const Elem<EW> e = s_el[i];
        store_elem<K, EW>(rp, (size_t)s_goff[digit(e)] + i, e);
      }
    }
    return;
  }
  Elem<KW>* s_key = reinterpret_cast<Elem<KW>*>(s_part);
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (valid(j)) s_key[rank[j]] = bit_cast<Elem<KW>>(elem_key<K, HW>(el[j]));
  V val[IPT];
  const V* src_v = (const V*)rp.src_v + base + lane;
  if constexpr (VW > 0) {
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if (valid(j)) val[j] = src_v[j * kWave];
  }
  __syncthreads();
  uint32_t dq[(IPT + 3) / 4] = {};  // four digits each
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const uint32_t i = tid + (uint32_t)q * BLOCK;
    if (i < tile_n) {
      const Elem<KW> k = s_key[i];
      const uint32_t d = digit(k);
      dq[q / 4] |= d << (8 * (q & 3));
      ((K*)rp.dst_k)[(size_t)s_goff[d] + i] = bit_cast<K>(k);
    }
  }
  if constexpr (VW == 0) return;
  __syncthreads();  // every key read out before the values overwrite them
  V* s_val = reinterpret_cast<V*>(s_part);
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (valid(j)) s_val[rank[j]] = val[j];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const uint32_t i = tid + (uint32_t)q * BLOCK;
    if (i < tile_n)
      ((V*)rp.dst_v)[(size_t)s_goff[(dq[q / 4] >> (8 * (q & 3))) & 0xffu] + i] = s_val[i];
  }
}

// 8. Local sort: one block sorts up to TILE elements stably in LDS, by the
//    digits [0, top) of which some vary. Each digit is ranked as a pass ranks
//    it (no counts before, no look-back); elements stay in registers between
//    digits and go through LDS whole. A digit costs about 7 us (its chain of
//    ranks, barriers and LDS round trips), so only the highest DIGITS varying
//    ones are sorted by (more where these vary in too few bits to tell the
//    elements apart: 65536 u32 keys of four digits with 10 values each, two
//    digits and then all again 88.7 us, at once 48), and runs that these leave
//    equal are put in order by insertion, one thread a run. Runs longer than
//    kLocalRun that are out of order (keys far from uniform) send the block
//    through all its digits.
//    Two uses: a sort of at most TILE elements is one launch of one block
//    (src/dst in `only`), and after the first pass of a short sort block g
//    sorts the run of digit g (`local`, gbase: where the runs start).
constexpr uint32_t kLocalRun = 16;

template <typename K, int MODE, int EW, int BLOCK, int IPT, int DIGITS>
__global__ __launch_bounds__(BLOCK, 8) void radix_local_kernel(
    const RadixLocal* __restrict__ local, const uint32_t* __restrict__ gbase, RadixPass only,
    uint32_t n) {
  constexpr int NW = BLOCK / kWave;
  constexpr uint32_t TILE = (uint32_t)BLOCK * IPT;
  constexpr int P = (int)sizeof(K);
  __shared__ __align__(16) uint32_t s_part[TILE * EW];
  __shared__ uint16_t s_hist[NW][kRadixBins];
  __shared__ uint32_t s_start[kRadixBins];
  __shared__ uint32_t s_wsum[kRadixBins / kWave];
  __shared__ uint32_t s_diff[2];
  uint32_t start = 0, cnt = n, top = P;
  RadixPass rp = only;
  if (local) {
    if (!local->on) return;
    rp = local->pass;
    top = local->top;
    const uint32_t* runs = gbase + top * kRadixBins;
    start = runs[blockIdx.x];
    cnt = (blockIdx.x + 1 < (uint32_t)kRadixBins ? runs[blockIdx.x + 1] : n) - start;
  }
  if (cnt == 0) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid / 64u;
  const bool digit_thread = tid < (uint32_t)kRadixBins;
  // Rows the elements need, and this wave's: [base, base + left).
  const uint32_t rows = (cnt + BLOCK - 1) / BLOCK;
  const uint32_t base = wid * kWave * rows;
  const uint32_t left = base < cnt ? min(cnt - base, kWave * rows) : 0u;
  auto valid = [&](int j) { return (uint32_t)j * kWave + lane < left; };
  auto word = [&](const Elem<EW>& e) { return order_bits<K, MODE>(elem_key<K, EW>(e)); };
  Elem<EW>* s_el = reinterpret_cast<Elem<EW>*>(s_part);
  Elem<EW> el[IPT];
  if (tid < 2) s_diff[tid] = 0;
  __syncthreads();
  const auto first = order_bits<K, MODE>(load_key<K, EW>(rp, start));
  uint32_t xlo = 0, xhi = 0;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    if (!valid(j)) continue;
    el[j] = load_elem<K, EW>(rp, (size_t)start + base + (uint32_t)j * kWave + lane);
    const auto x = word(el[j]) ^ first;
    xlo |= (uint32_t)x;
    if constexpr (sizeof(K) == 8) xhi |= (uint32_t)(x >> 32);
  }
  if (xlo) atomicOr(&s_diff[0], xlo);
  if (xhi) atomicOr(&s_diff[1], xhi);
  __syncthreads();
  const uint32_t diff[2] = {(uint32_t)__builtin_amdgcn_readfirstlane((int)s_diff[0]),
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)s_diff[1])};
  auto varies = [&](uint32_t p) { return ((diff[p / 4] >> (8 * (p & 3))) & 0xffu) != 0; };
  // The lowest of the DIGITS highest varying digits, or of as many as have two
  // varying bits more than the elements need, and whether any below varies.
  uint32_t low = DIGITS >= P ? 0u : top;
  bool below_varies = false;
  if constexpr (DIGITS < P) {
    const int need = 32 - __builtin_clz(cnt) + 2;
    int digits = 0, bits = 0;
#pragma unroll
    for (int p = P - 1; p >= 0; --p) {
      const uint32_t varying = (diff[p / 4] >> (8 * (p & 3))) & 0xffu;
      if (varying == 0 || (uint32_t)p >= top) continue;
      if (digits >= DIGITS && bits >= need) {
        below_varies = true;
      } else {
        ++digits;
        bits += __builtin_popcount(varying);
        low = (uint32_t)p;
      }
    }
  }
  const uint64_t lt = lanemask_lt();
  bool in_lds = false;
  for (uint32_t from = low;;) {
    for (uint32_t p = from; p < top; ++p) {
      if (!varies(p)) continue;
      if (in_lds) {
#pragma unroll
        for (int j = 0; j < IPT; ++j)
          if (valid(j)) el[j] = s_el[base + (uint32_t)j * kWave + lane];
      }
      for (uint32_t i = tid; i < NW * kRadixBins / 2; i += BLOCK)
        reinterpret_cast<uint32_t*>(&s_hist[0][0])[i] = 0;
      __syncthreads();
      uint32_t rank[IPT];
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        if ((uint32_t)j >= rows) break;
        asm volatile("" : "+v"(el[j].w[0]));
        const uint32_t d = (uint32_t)(word(el[j]) >> (8 * p)) & 0xffu;
        const uint64_t peers = match_digit<8>(d, valid(j));
        uint32_t before = 0;
        if (valid(j)) before = s_hist[wid][d];
        const uint32_t below = (uint32_t)__builtin_popcountll(peers & lt);
        if (valid(j) && below == 0)
          s_hist[wid][d] = (uint16_t)(before + (uint32_t)__builtin_popcountll(peers));
        rank[j] = before + below;
      }
      __syncthreads();
      uint32_t sum = 0, incl = 0;
      if (digit_thread) {
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const uint32_t c = s_hist[w][tid];
          s_hist[w][tid] = (uint16_t)sum;
          sum += c;
        }
        incl = wave_inclusive_scan<uint32_t, OP_ADD>(sum);
        if (lane == 63) s_wsum[wid] = incl;
      }
      __syncthreads();
      if (digit_thread) {
        uint32_t woff = 0;
        for (uint32_t k = 0; k < wid; ++k) woff += s_wsum[k];
        s_start[tid] = woff + incl - sum;
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        if (!valid(j)) continue;
        asm volatile("" : "+v"(el[j].w[0]));
        const uint32_t d = (uint32_t)(word(el[j]) >> (8 * p)) & 0xffu;
        s_el[s_start[d] + s_hist[wid][d] + rank[j]] = el[j];
      }
      in_lds = true;
      __syncthreads();
    }
    if (from == 0 || !below_varies) break;
    // Repair: thread t looks at positions t + q * BLOCK. An element below its
    // predecessor is in one run with it; the first such one of a run speaks
    // for the run. (Prefixes do not change while runs are put in order.)
    const uint32_t shift = 8 * low;
    auto at = [&](uint32_t i) { return word(s_el[i]); };
    if (tid == 0) s_diff[0] = 0;
    uint32_t mine = 0;
#pragma unroll 1
    for (uint32_t i = tid, q = 0; i < cnt; i += BLOCK, ++q)
      if (i > 0 && at(i - 1) > at(i)) mine |= 1u << q;
    __syncthreads();
#pragma unroll 1
    for (uint32_t left_out = mine; left_out; left_out &= left_out - 1) {
      const uint32_t q = (uint32_t)__builtin_ctz(left_out), i = tid + q * BLOCK;
      const auto prefix = at(i) >> shift;
      uint32_t b = i - 1, e = i + 1;
      bool first = true;
      while (b > 0 && i - b < kLocalRun && at(b - 1) >> shift == prefix) {
        if (at(b - 1) > at(b)) first = false;
        --b;
      }
      while (e < cnt && e - b <= kLocalRun && at(e) >> shift == prefix) ++e;
      if (i - b >= kLocalRun || e - b > kLocalRun) s_diff[0] = 1;
      if (!first) mine &= ~(1u << q);
    }
    __syncthreads();
    if (s_diff[0]) {
      from = 0;
      continue;
    }
#pragma unroll 1
    for (; mine; mine &= mine - 1) {
      const uint32_t i = tid + (uint32_t)__builtin_ctz(mine) * BLOCK;
      const auto prefix = at(i) >> shift;
      uint32_t b = i - 1, e = i + 1;
      while (b > 0 && at(b - 1) >> shift == prefix) --b;
      while (e < cnt && at(e) >> shift == prefix) ++e;
      for (uint32_t k = b + 1; k < e; ++k) {
        const Elem<EW> x = s_el[k];
        uint32_t h = k;
        for (; h > b && at(h - 1) > word(x); --h) s_el[h] = s_el[h - 1];
        s_el[h] = x;
      }
    }
    __syncthreads();
    break;
  }
  if (!in_lds) {
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if (valid(j)) store_elem<K, EW>(rp, (size_t)start + base + (uint32_t)j * kWave + lane, el[j]);
    return;
  }
  for (uint32_t i = tid; i < cnt; i += BLOCK) store_elem<K, EW>(rp, (size_t)start + i, s_el[i]);
}

// 9. Long sorts of 8-byte keys by their highest digits only. n keys that are
//    spread at all differ from most others in not many more than log2(n) of
//    their highest varying bits, so the passes stop at digit `low` and a repair
//    orders what they left equal: a pass moves every element once (24 bytes of
//    traffic for u64 + u32), the look of the repair reads 8 of them.
//     * radix_begin_kernel looks at some samples of kSample keys: for every
//       digit, how many pairs of different keys share the digits from there on.
//     * low: at least log2(n) + 4 bits of varying digits, one digit more when some
//       key may hold over 1/64 of the input, and lower until the samples' pairs
//       say that at most a quarter of the keys share these digits with another
//       one (n / 16 runs to repair: 2^27 keys of 100 values to a digit have n / 3,
//       which took 2.4 ms, more than two passes; 16 samples hold 2^29 pairs, so one
//       may clash at 2^27).
//       16 keys of a sample with the same digits that are not all equal are a long
//       run, which counts as any number of pairs.
//     * Keys that a sample has 4 times (a share of 2^-12 is found nearly always)
//       are hot: their runs are too long to repair when any other key shares
//       their digits, however rare. radix_hist_kernel compares every key with
//       them, and low goes down to the highest digit that tells all apart.
//     * radix_repair_find_kernel lists the runs of equal digits that have an
//       element below its predecessor, radix_repair_kernel orders them.
//     * When that is too much (many long runs), the passes start over with every
//       digit. Any input is sorted; the choice only decides how soon.
//    2^27 u64 + u32, eight passes -> now: uniform 7.0 -> 4.50 ms (four passes),
//    zipf with hot keys 7.2 -> 5.12 (five); the samples 34 us (uniform 47), the
//    comparison with hot keys 50 us, the look 0.22 ms (4.7 TB/s; with 64 consecutive
//    bytes per thread 0.46; uniform, with 2 million runs to list, 0.34), ordering the
//    runs 5 us (uniform 0.27 ms), passes left out 14 us each. Digits of
//    100 values 4.6, of 32 values 5.6, groups of two keys that differ in the lowest
//    bytes 6.7 (10.2, 10.4 and 11.4 when digits counted 8 bits each and the passes
//    then started over). 2^25 with half the keys equal and 1e-5 of them off in the
//    low digits 2.3 (3.5 when only a sample looked).
// Keys: 2^21 + 100000 uniform u64 + u32 223 -> 171 us. What the samples and the
// launches that find nothing to do cost shows where few digits vary: two digits 81
// -> 111 us there, 183 -> 219 at 8 million, 299 -> 344 at 16 million.
constexpr uint32_t kRepairMin = 1u << 21;
constexpr uint32_t kRepairRun = 32;         // Elements one thread orders,
constexpr uint32_t kRepairLong = 1u << 15;  // elements of a run that a block orders,
constexpr uint32_t kRepairSum = 1u << 16;   // and of all that one block does,
constexpr uint32_t kRepairLongs = 64;       // and how many

// The first kLows blocks to a sample look at it: block b at sample b / kLows, from
// digit b % kLows on (0: whole keys). The others zero words.
template <typename K, int MODE>
__global__ __launch_bounds__(1024) void radix_begin_kernel(const K* __restrict__ keys, uint32_t n,
                                                           RadixSample* __restrict__ sample,
                                                           uint32_t* __restrict__ zero, uint32_t words) {
  // A slot: the number of its first key, from 1; whether another one differs; how
  // many more share its digits.
  constexpr uint32_t kFirst = 0x3fffu, kDiffers = 0x8000u, kMore = 0x10000u;
  constexpr uint32_t kLongRun = 16, kAny = 1u << 20;
  __shared__ uint64_t s_word[kSample];
  __shared__ uint32_t s_slot[2 * kSample];
  __shared__ uint32_t s_sum, s_most, s_heavy;
  __shared__ unsigned long long s_xor;
  constexpr int PER = (int)(kSample / 1024);  // most keys of a thread
  constexpr uint32_t looks = kSamples * kLows;
  const uint32_t tid = threadIdx.x;
  if (blockIdx.x >= looks) {
    const uint32_t step = (gridDim.x - looks) * 1024u;
    for (size_t i = (blockIdx.x - looks) * 1024u + tid; i < words; i += step) zero[i] = 0;
    return;
  }
  const uint32_t low = blockIdx.x % kLows, sub = blockIdx.x / kLows;
  const uint32_t size = sample_size(n), slots = 2 * size;
  // Positions spread by an odd multiplier.
  uint64_t word[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t i = sub * size + j * 1024 + tid;
    if (j * 1024u < size) word[j] = (uint64_t)order_bits<K, MODE>(keys[(uint64_t)(i * 2654435761u) * n >> 32]);
  }
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (j * 1024u < size) s_word[j * 1024 + tid] = word[j];
  for (uint32_t i = tid; i < slots; i += 1024) s_slot[i] = 0;
  if (tid == 0) {
    s_sum = s_most = s_heavy = 0;
    s_xor = 0;
  }
  __syncthreads();
  uint64_t x = 0;
#pragma unroll 1
  for (uint32_t j = 0; j < size / 1024; ++j) {
    const uint32_t i = j * 1024 + tid;
    const uint64_t mine = s_word[i], prefix = mine >> (8 * low);
    x |= mine ^ s_word[0];
    uint32_t h = (uint32_t)((prefix * 0x9E3779B97F4A7C15ull) >> 40) % slots;
    for (;;) {
      uint32_t other = s_slot[h];  // (a hot key: one read for all)
      if (other == 0) other = atomicCAS(&s_slot[h], 0u, i + 1);
      if (other == 0) break;
      const uint64_t w = s_word[(other & kFirst) - 1];
      if (w >> (8 * low) == prefix) {
        const uint64_t same = ballot(true);  // the lanes that are here at once
        if (ballot(h != (uint32_t)__builtin_amdgcn_readfirstlane((int)h)) != 0) atomicAdd(&s_slot[h], kMore);
        else if (__builtin_ctzll(same) == (int)(tid & 63u)) atomicAdd(&s_slot[h], kMore * (uint32_t)__builtin_popcountll(same));
        if (w != mine && !(other & kDiffers)) atomicOr(&s_slot[h], kDiffers);
        break;
      }
      h = (h + 1) % slots;
    }
  }
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) x |= __shfl_xor(x, m);
  if (x && (tid & 63u) == 0) atomicOr(&s_xor, (unsigned long long)x);
  __syncthreads();
  if (low > 0) {
    uint32_t pairs = 0;
    for (uint32_t i = tid; i < slots; i += 1024) {
      const uint32_t more = s_slot[i] / kMore;
      if (s_slot[i] & kDiffers) pairs += more + 1 >= kLongRun ? kAny : more;
    }
    if (pairs) atomicAdd(&s_sum, min(pairs, kAny));
    __syncthreads();
    if (tid == 0) sample->clash[low][sub] = min(s_sum, kAny);
    return;
  }
  // The hot keys, the most frequent ones first.
  for (uint32_t least : {16u, 4u}) {
    for (uint32_t i = tid; i < slots; i += 1024) {
      const uint32_t count = s_slot[i] / kMore + 1;
      if (count < least || (least == 4 && count >= 16)) continue;
      atomicMax(&s_most, count);
      const uint32_t k = atomicAdd(&s_sum, 1u);
      if (k < kHots) sample->hot[sub][k] = s_word[(s_slot[i] & kFirst) - 1];
    }
    __syncthreads();
    if (least == 16 && tid == 0) s_heavy = s_sum;
    __syncthreads();
  }
  if (tid == 0) {
    uint32_t varying = 0;
    for (int p = 0; p < 8; ++p) varying |= (s_xor >> (8 * p) & 0xffu ? 1u : 0u) << p;
    sample->clash[0][sub] = 0;
    sample->varying[sub] = varying;
    sample->most[sub] = s_most;
    sample->hots[sub] = min(s_sum, kHots);
    sample->heavy[sub] = s_heavy;
  }
}

// The end of the run of equal words >> shift that i is in (the first index
// after it), or its start.
template <typename K, int MODE>
__device__ inline uint32_t run_end(const K* __restrict__ keys, uint32_t n, uint32_t i, uint32_t shift) {
  const auto prefix = order_bits<K, MODE>(keys[i]) >> shift;
  uint64_t step = 1, in = i;
  while (in + step < n && order_bits<K, MODE>(keys[in + step]) >> shift == prefix) {
    in += step;
    step *= 2;
  }
  uint64_t lo = in + 1, hi = min((uint64_t)n, in + step);
  while (lo < hi) {
    const uint64_t mid = (lo + hi) / 2;
    if (order_bits<K, MODE>(keys[mid]) >> shift == prefix) lo = mid + 1;
    else hi = mid;
  }
  return (uint32_t)lo;
}
template <typename K, int MODE>
__device__ inline uint32_t run_start(const K* __restrict__ keys, uint32_t i, uint32_t shift) {
  const auto prefix = order_bits<K, MODE>(keys[i]) >> shift;
  int64_t step = 1, in = i;
  while (in - step >= 0 && order_bits<K, MODE>(keys[in - step]) >> shift == prefix) {
    in -= step;
    step *= 2;
  }
  int64_t lo = in - step < 0 ? 0 : in - step, hi = in;
  while (lo < hi) {
    const int64_t mid = (lo + hi) / 2;
    if (order_bits<K, MODE>(keys[mid]) >> shift == prefix) hi = mid;
    else lo = mid + 1;
  }
  return (uint32_t)lo;
}

// Block b looks at elements [b * chunk, (b + 1) * chunk) and lists runs in
// list[b * (chunk / 2 + 1)...] (each has an element below its predecessor in
// the chunk, so there are no more), counts[b] of them. chunk is a multiple of
// 2048.
template <typename K, int MODE>
__global__ __launch_bounds__(256) void radix_repair_find_kernel(const K* __restrict__ keys, uint32_t n,
                                                                uint32_t chunk, bool aligned,
                                                                RadixRepair* __restrict__ rep,
                                                                uint32_t* __restrict__ marks,
                                                                uint32_t* __restrict__ list,
                                                                uint32_t* __restrict__ counts) {
  static_assert(sizeof(K) == 8, "8-byte keys");
  constexpr int ROWS = 4;  // rows of 256 threads x 2 keys
  __shared__ uint32_t s_count;
  if (rep->low == 0) return;
  const uint32_t shift = 8 * rep->low, lane = threadIdx.x & 63u;
  list += (size_t)blockIdx.x * (chunk / 2 + 1);
  if (threadIdx.x == 0) s_count = 0;
  __syncthreads();
  const size_t end = min((size_t)n, (size_t)(blockIdx.x + 1) * chunk);
  for (size_t base = (size_t)blockIdx.x * chunk; base < end; base += 256 * 2 * ROWS) {
    uint64_t w[ROWS][2], left[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const size_t i = base + (j * 256 + threadIdx.x) * 2;
      K x[2] = {};
      if (aligned && i + 2 <= n) {
        const uint4 q = *reinterpret_cast<const uint4*>(keys + i);
        x[0] = bit_cast<K>((uint64_t)q.y << 32 | q.x);
        x[1] = bit_cast<K>((uint64_t)q.w << 32 | q.z);
      } else {
        if (i < n) x[0] = keys[i];
        if (i + 1 < n) x[1] = keys[i + 1];
      }
      if (lane == 0 && i < n) left[j] = order_bits<K, MODE>(keys[i > 0 ? i - 1 : 0]);
      w[j][0] = order_bits<K, MODE>(x[0]);
      w[j][1] = order_bits<K, MODE>(x[1]);
    }
#pragma unroll
    for (int h = 0; h < 2 * ROWS; ++h) {
      const int j = h / 2, k = h % 2;
      const uint64_t word = w[j][k];
      const uint64_t up = __shfl_up(w[j][1], 1);
      const uint64_t before = k == 1 ? w[j][0] : (lane == 0 ? left[j] : up);
      const size_t at = base + (j * 256 + threadIdx.x) * 2 + k;
      const uint32_t i = (uint32_t)at;
      if (at < n && before > word) {
        // The run's first such element lists it. One that sees neither the
        // run's start nor another before it within kRepairRun elements may be
        // the first; the mark at the start decides.
        const uint64_t prefix = word >> shift;
        uint64_t cur = before;
        uint32_t s = i - 1;
        bool first = true;
        while (s > 0) {
          const uint64_t p = order_bits<K, MODE>(keys[s - 1]);
          if (p >> shift != prefix) break;
          if (p > cur) {
            first = false;
            break;
          }
          if (i - s >= kRepairRun) {
            s = run_start<K, MODE>(keys, s, shift);
            break;
          }
          cur = p;
          --s;
        }
        if (first && !(atomicOr(&marks[s / 32], 1u << (s % 32)) >> (s % 32) & 1u)) list[atomicAdd(&s_count, 1u)] = s;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = s_count;
}

// Block b orders the runs that block b of the find listed: a thread each run of
// up to kRepairRun elements by insertion, the block each longer one by stable
// LSD passes over its varying digits below low, 1024 elements at a time,
// between the run and the same places of tmp. What is too much for that leaves
// redo set. VW: 4-byte words of a value (0: none).
template <typename K, int MODE, int VW>
__global__ __launch_bounds__(1024) void radix_repair_kernel(K* keys, uint32_t* vals, K* tmp_k,
                                                            uint32_t* tmp_v, uint32_t n, uint32_t chunk,
                                                            RadixRepair* rep,
                                                            const uint32_t* __restrict__ list,
                                                            const uint32_t* __restrict__ counts) {
  constexpr int NW = 1024 / kWave;
  __shared__ uint32_t s_base[kRadixBins];
  __shared__ uint16_t s_hist[NW][kRadixBins];
  __shared__ uint32_t s_wsum[kRadixBins / kWave], s_diff[2];
  __shared__ uint32_t s_start[kRepairLongs], s_end[kRepairLongs], s_longs, s_sum;
  const uint32_t low = rep->low;
  if (low == 0) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid / 64u, shift = 8 * low;
  const uint32_t runs = counts[blockIdx.x];
  list += (size_t)blockIdx.x * (chunk / 2 + 1);
  if (tid == 0) s_longs = s_sum = 0;
  __syncthreads();
  for (uint32_t r = tid; r < runs; r += 1024) {
    const uint32_t s = list[r];
    const auto prefix = order_bits<K, MODE>(keys[s]) >> shift;
    uint32_t e = s + 1;
    while (e < n && e - s <= kRepairRun && order_bits<K, MODE>(keys[e]) >> shift == prefix) ++e;
    if (e - s > kRepairRun) {
      const uint32_t j = atomicAdd(&s_longs, 1u);
      if (j < kRepairLongs) {
        e = run_end<K, MODE>(keys, n, s, shift);
        s_start[j] = s;
        s_end[j] = e;
        atomicAdd(&s_sum, min(e - s, 2 * kRepairSum));
        if (e - s > kRepairLong) atomicAdd(&s_sum, kRepairSum);
      }
      continue;
    }
    for (uint32_t k = s + 1; k < e; ++k) {
      const K x = keys[k];
      const auto w = order_bits<K, MODE>(x);
      uint32_t h = k;
      if (order_bits<K, MODE>(keys[h - 1]) <= w) continue;
      uint32_t v[VW > 0 ? VW : 1];
#pragma unroll
      for (int c = 0; c < VW; ++c) v[c] = vals[(size_t)k * VW + c];
      for (; h > s && order_bits<K, MODE>(keys[h - 1]) > w; --h) {
        keys[h] = keys[h - 1];
#pragma unroll
        for (int c = 0; c < VW; ++c) vals[(size_t)h * VW + c] = vals[(size_t)(h - 1) * VW + c];
      }
      keys[h] = x;
#pragma unroll
      for (int c = 0; c < VW; ++c) vals[(size_t)h * VW + c] = v[c];
    }
  }
  __syncthreads();
  const uint32_t longs = s_longs;
  if (longs > kRepairLongs || s_sum > kRepairSum) {
    if (tid == 0) rep->redo = 1;
    return;
  }
  const bool digit_thread = tid < (uint32_t)kRadixBins;
  const uint64_t lt = lanemask_lt();
  for (uint32_t r = 0; r < longs; ++r) {
    // Indices count from the run's start (beside 2^32 elements, start + index +
    // stride does not fit 32 bits).
    const uint32_t s = s_start[r], cnt = s_end[r] - s;
    __syncthreads();
    if (tid < 2) s_diff[tid] = 0;
    __syncthreads();
    const uint64_t word = order_bits<K, MODE>(keys[s]);
    uint64_t x = 0;
    for (uint32_t i = tid; i < cnt; i += 1024) x |= order_bits<K, MODE>(keys[s + i]) ^ word;
    if (x) {
      atomicOr(&s_diff[0], (uint32_t)x);
      atomicOr(&s_diff[1], (uint32_t)(x >> 32));
    }
    __syncthreads();
    const uint64_t diff = (uint64_t)s_diff[1] << 32 | s_diff[0];
    K *src_k = keys + s, *dst_k = tmp_k + s;
    uint32_t *src_v = vals + (size_t)s * VW, *dst_v = tmp_v + (size_t)s * VW;
    for (uint32_t p = 0; p < low; ++p) {
      if ((diff >> (8 * p) & 0xffu) == 0) continue;
      auto digit = [&](K k) { return (uint32_t)(order_bits<K, MODE>(k) >> (8 * p)) & 0xffu; };
      if (digit_thread) s_base[tid] = 0;
      __syncthreads();
      for (uint32_t i = tid; i < cnt; i += 1024) atomicAdd(&s_base[digit(src_k[i])], 1u);
      __syncthreads();
      uint32_t c = 0, incl = 0;
      if (digit_thread) {
        c = s_base[tid];
        incl = wave_inclusive_scan<uint32_t, OP_ADD>(c);
        if (lane == 63) s_wsum[wid] = incl;
      }
      __syncthreads();
      if (digit_thread) {
        uint32_t off = incl - c;
        for (uint32_t w = 0; w < wid; ++w) off += s_wsum[w];
        s_base[tid] = off;
      }
      for (uint32_t c0 = 0; c0 < cnt; c0 += 1024) {
        for (uint32_t i = tid; i < NW * kRadixBins / 2; i += 1024)
          reinterpret_cast<uint32_t*>(&s_hist[0][0])[i] = 0;
        __syncthreads();
        const uint32_t i = c0 + tid;
        const bool valid = i < cnt;
        const K k = src_k[valid ? i : 0];
        const uint32_t d = digit(k);
        const uint64_t peers = match_digit<8>(d, valid);
        const uint32_t below = (uint32_t)__builtin_popcountll(peers & lt);
        if (valid && below == 0) s_hist[wid][d] = (uint16_t)__builtin_popcountll(peers);
        __syncthreads();
        uint32_t total = 0;
        if (digit_thread) {
#pragma unroll
          for (int w = 0; w < NW; ++w) {
            const uint32_t h = s_hist[w][tid];
            s_hist[w][tid] = (uint16_t)total;
            total += h;
          }
        }
        __syncthreads();
        if (valid) {
          const uint32_t o = s_base[d] + s_hist[wid][d] + below;
          dst_k[o] = k;
#pragma unroll
          for (int q = 0; q < VW; ++q) dst_v[(size_t)o * VW + q] = src_v[(size_t)i * VW + q];
        }
        __syncthreads();
        if (digit_thread) s_base[tid] += total;
      }
      __syncthreads();
      K* const tk = src_k;
      src_k = dst_k;
      dst_k = tk;
      uint32_t* const tv = src_v;
      src_v = dst_v;
      dst_v = tv;
    }
    if (src_k != keys + s) {
      for (uint32_t i = tid; i < cnt; i += 1024) {
        dst_k[i] = src_k[i];
#pragma unroll
        for (int q = 0; q < VW; ++q) dst_v[(size_t)i * VW + q] = src_v[(size_t)i * VW + q];
      }
    }
  }
}

}  // namespace msv
