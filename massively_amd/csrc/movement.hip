// vector::gather / scatter and seeded synthetic inputs for gfx950.
//
// gather: out[i] = values[idx[i]]   (massively/src/core/indexed.rs:16-196)
// scatter: out[idx[i]] = values[i]  (massively/src/core/scatter.rs:8-21)
// Each thread owns ROWS 16-byte index vectors laid out row-striped like the
// scan tiles, so index loads and the sequential-side stores are full-wave
// dwordx4 accesses and each thread keeps 16 independent random accesses in
// flight. Large tables with indices in no order take the binned forms of
// bin_kernels.hpp. The reference leaves out-of-range indices undefined; here a gather
// reads zero for them and a scatter drops them, so no index can fault.
#include <algorithm>

#include "bin_kernels.hpp"
#include "msv_internal.hpp"

namespace msv {

constexpr int kMoveBlock = 256;
constexpr int kMoveRows = 4;  // 4 x uint4 of indices = 16 indices per thread
constexpr uint32_t kMoveTile = kMoveBlock * kMoveRows * 4;

// With `looks` (see gather_look_kernel), the first `binned` positions are done by
// the binned form when the looks say so.
template <typename T>
__global__ __launch_bounds__(kMoveBlock) void gather_kernel(const T* __restrict__ values,
                                                            uint32_t vlen,
                                                            const uint32_t* __restrict__ idx,
                                                            T* __restrict__ out, uint32_t n,
                                                            bool aligned,
                                                            const uint32_t* __restrict__ looks,
                                                            uint32_t binned) {
  const uint32_t tid = threadIdx.x;
  const size_t base = (size_t)blockIdx.x * kMoveTile;
  if (looks && base < binned && look_binned(looks)) return;
  const bool full = aligned && base + kMoveTile <= n;
  uint32_t ix[kMoveRows][4];
  if (full) {
#pragma unroll
    for (int r = 0; r < kMoveRows; ++r) {
      const uint4 q = *reinterpret_cast<const uint4*>(idx + base + ((size_t)r * kMoveBlock + tid) * 4);
      ix[r][0] = q.x; ix[r][1] = q.y; ix[r][2] = q.z; ix[r][3] = q.w;
    }
  } else {
#pragma unroll
    for (int r = 0; r < kMoveRows; ++r)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const size_t i = base + ((size_t)r * kMoveBlock + tid) * 4 + k;
        ix[r][k] = i < n ? idx[i] : 0xffffffffu;
      }
  }
  T v[kMoveRows][4];
#pragma unroll
  for (int r = 0; r < kMoveRows; ++r)
#pragma unroll
    for (int k = 0; k < 4; ++k) v[r][k] = ix[r][k] < vlen ? values[ix[r][k]] : (T)0;
#pragma unroll
  for (int r = 0; r < kMoveRows; ++r) {
    const size_t o = base + ((size_t)r * kMoveBlock + tid) * 4;
    if (full) {
      if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<uint4*>(out + o) =
            make_uint4(bit_cast<uint32_t>(v[r][0]), bit_cast<uint32_t>(v[r][1]),
                       bit_cast<uint32_t>(v[r][2]), bit_cast<uint32_t>(v[r][3]));
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) out[o + k] = v[r][k];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (o + k < n) out[o + k] = v[r][k];
    }
  }
}

// Sorted indices: consecutive lanes take consecutive positions of their wave's
// 256 in a row, so that a store of the wave has whole lines (2^22 u32, one to 64:
// 172 -> 140 us, one to 4: 55 -> 23).
template <typename T>
__global__ __launch_bounds__(kMoveBlock) void scatter_kernel(const T* __restrict__ values,
                                                             const uint32_t* __restrict__ idx,
                                                             uint32_t n, T* __restrict__ out,
                                                             uint32_t olen) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const size_t base = (size_t)blockIdx.x * kMoveTile + (size_t)tid * 4;
  uint32_t d[kMoveRows][4];
#pragma unroll
  for (int r = 0; r < kMoveRows; ++r)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const size_t i = base + (size_t)r * kMoveBlock * 4 + k;
      d[r][k] = i < n ? idx[i] : 0xffffffffu;
    }
  const bool lanes = ordered_wave(d[0][0], d[0][1], d[0][2], d[0][3], 3, 3 * 64);
  if (lanes) {
#pragma unroll
    for (int r = 0; r < kMoveRows; ++r)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const size_t i = base - 3 * lane + (size_t)r * kMoveBlock * 4 + k * kWave;
        d[r][k] = i < n ? idx[i] : 0xffffffffu;
      }
  }
#pragma unroll
  for (int r = 0; r < kMoveRows; ++r)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const size_t i = base + (size_t)r * kMoveBlock * 4 + (lanes ? (size_t)k * kWave - 3 * lane : (size_t)k);
      if (d[r][k] < olen) out[d[r][k]] = values[i];
    }
}

// ---- seeded streams (massively/src/api/util/random.rs:12-22,331-396) ------
// pcg_hash32 and seed_key: msv_internal.hpp.

__global__ void uniform_u32_kernel(uint32_t* __restrict__ out, uint32_t n, uint32_t start,
                                   uint32_t key, uint32_t lo, uint32_t span) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t v = pcg_hash32((start + i) ^ key);
  out[i] = (span == 0xffffffffu) ? v : lo + v % (span + 1u);
}

__global__ void uniform_u64_kernel(uint64_t* __restrict__ out, uint32_t n, uint32_t start,
                                   uint32_t key, uint64_t lo, uint64_t span) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = start + i;
  const uint64_t v = (uint64_t)pcg_hash32(p ^ key) | ((uint64_t)pcg_hash32(p ^ key ^ 0x9e3779b9u) << 32);
  out[i] = (span == ~0ull) ? v : lo + v % (span + 1ull);
}

__global__ void iota_u32_kernel(uint32_t* __restrict__ out, uint32_t n, uint32_t start) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = start + i;
}

// ---- host ------------------------------------------------------------------
template <typename T>
static msv_status direct_gather(Ctx& c, const T* values, uint32_t vlen, const uint32_t* idx, T* out,
                                uint32_t n, const uint32_t* looks = nullptr, uint32_t binned = 0) {
  const bool aligned = (((uintptr_t)idx | (uintptr_t)out) & 15u) == 0;
  hipLaunchKernelGGL(gather_kernel<T>, dim3(div_up(n, kMoveTile)), dim3(kMoveBlock), 0, c.stream(),
                     values, vlen, idx, out, n, aligned, looks, binned);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

template <typename T>
static msv_status direct_scatter(Ctx& c, const T* values, const uint32_t* idx, uint32_t n, T* out,
                                 uint32_t olen) {
  hipLaunchKernelGGL(scatter_kernel<T>, dim3(div_up(n, kMoveTile)), dim3(kMoveBlock), 0, c.stream(),
                     values, idx, n, out, olen);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

// How a table of tlen elements and n indices are cut (see BinPlan).
static BinPlan bin_plan(uint32_t tlen, uint32_t n, uint32_t tile, uint32_t leaf_shift,
                        uint32_t sub_shift) {
  BinPlan p = {};
  p.leaf_shift = leaf_shift;
  p.sub_shift = sub_shift;
  p.subs = 1u << sub_shift;
  p.windows = ((tlen - 1) >> (leaf_shift + sub_shift)) + 1;
  p.tile_row = (p.windows + 8) & ~7u;
  p.chunk_row = (p.subs + 8) & ~7u;
  p.tiles = n / tile;
  // A chunk is filled to 7/8 by indices spread evenly over the windows. (A tile
  // has at most 4 times the mean in a window.)
  p.group = std::min(kBinMost, std::max(1u, (uint32_t)((uint64_t)kBinChunk * 7 / 8 * p.windows / tile)));
  p.groups = div_up(p.tiles, p.group);
  p.cap = p.groups * div_up((uint64_t)p.group * (4 * tile / p.windows), kBinChunk);
  return p;
}

static msv_status binned_gather(Ctx& c, const uint32_t* values, uint32_t vlen, const uint32_t* idx,
                                uint32_t* out, uint32_t n) {
  // Tiles of 32768 positions, so that a run in one of 512 windows is 64 indices.
  constexpr int IPT = 32;
  constexpr uint32_t TILE = (uint32_t)kBinBlock * IPT;
  uint32_t shift = 18;  // windows of 1 MiB, larger ones past 512 MiB
  while (((vlen - 1) >> shift) >= kBinMost) ++shift;
  const BinPlan p = bin_plan(vlen, n, TILE, shift, 0);
  uint32_t* pidx = (uint32_t*)c.scratch(sizeof(uint32_t) * (size_t)p.tiles * TILE);
  uint16_t* ppos = (uint16_t*)c.scratch(sizeof(uint16_t) * (size_t)p.tiles * TILE);
  uint16_t* starts = (uint16_t*)c.scratch(sizeof(uint16_t) * (size_t)p.tiles * p.tile_row);
  uint32_t* looks = (uint32_t*)c.scratch(kLooks);
  if (!pidx || !ppos || !starts || !looks) {
    clear_error();
    return direct_gather(c, values, vlen, idx, out, n);
  }
  const bool aligned = (((uintptr_t)idx | (uintptr_t)out) & 15u) == 0;
  const uint32_t cus = (uint32_t)c.num_cus();
  static_assert(TILE % kMoveTile == 0, "a tile is whole direct tiles");
  hipLaunchKernelGGL(gather_look_kernel, dim3(kLooks), dim3(kBinBlock), 0, c.stream(), idx, n, p,
                     aligned, (uint8_t*)looks);
  MSV_TRY(direct_gather(c, values, vlen, idx, out, n, looks, p.tiles * TILE));
  hipLaunchKernelGGL((bin_tiles_kernel<uint32_t, IPT, false>), dim3(std::min(p.tiles, cus)),
                     dim3(kBinBlock), 0, c.stream(), const_cast<uint32_t*>(values), vlen, idx, out, n,
                     p, aligned, looks, pidx, ppos, (uint32_t*)nullptr, starts, BinChunks{}, (uint64_t*)nullptr, 0u);
  // The values replace the indices in place.
  hipLaunchKernelGGL((gather_window_kernel<uint32_t, TILE, 8>), dim3(div_up(cus, kXcds) * kXcds),
                     dim3(256), 0, c.stream(), values, vlen, p, pidx, pidx, starts, looks);
  hipLaunchKernelGGL((unbin_tiles_kernel<uint32_t, IPT>), dim3(std::min(p.tiles, 4 * cus)),
                     dim3(kBinBlock), 0, c.stream(), p, pidx, ppos, starts, out, aligned, looks);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

template <typename T>
static msv_status binned_scatter(Ctx& c, const T* values, const uint32_t* idx, uint32_t n, T* out,
                                 uint32_t olen) {
  constexpr int IPT = 16;
  constexpr uint32_t TILE = (uint32_t)kBinBlock * IPT;
  constexpr uint32_t leaf_shift = sizeof(T) == 4 ? 14 : 13;
  static_assert((sizeof(T) << leaf_shift) == kLeafBytes, "leaf");
  // As many leaves per window as windows.
  const uint32_t leaves = ((olen - 1) >> leaf_shift) + 1;
  uint32_t bits = 0;
  while ((1u << bits) < leaves) ++bits;
  const BinPlan p = bin_plan(olen, n, TILE, leaf_shift, (bits + 1) / 2);
  // Room for the elements, for rounding each chunk to 8 of them and for less than
  // a chunk left over in each part.
  const size_t most = (size_t)p.tiles * TILE / kBinChunk + (size_t)p.windows * p.groups;
  BinChunks chunks = {};
  chunks.shard = (uint32_t)(((size_t)p.tiles * TILE / 8 + most) / kShards + 1 + kBinChunk / 8);
  const size_t slots = (size_t)chunks.shard * 8 * kShards;
  uint32_t* pidx = (uint32_t*)c.scratch(sizeof(uint32_t) * (size_t)p.tiles * TILE);
  T* pval = (T*)c.scratch(sizeof(T) * (size_t)p.tiles * TILE);
  uint16_t* starts = (uint16_t*)c.scratch(sizeof(uint16_t) * (size_t)p.tiles * p.tile_row);
  uint16_t* cidx = (uint16_t*)c.scratch(sizeof(uint16_t) * slots);
  T* cval = (T*)c.scratch(sizeof(T) * slots);
  uint16_t* rows = (uint16_t*)c.scratch(sizeof(uint16_t) * (size_t)p.windows * p.cap * p.chunk_row);
  chunks.used = (uint32_t*)c.scratch(sizeof(uint32_t) * kShards * kShardStep);
  chunks.counts = (uint32_t*)c.scratch(sizeof(uint32_t) * p.windows);
  chunks.at = (uint32_t*)c.scratch(sizeof(uint32_t) * (size_t)p.windows * p.cap);
  if (!pidx || !pval || !starts || !cidx || !cval || !rows || !chunks.used || !chunks.counts ||
      !chunks.at) {
    clear_error();
    return direct_scatter(c, values, idx, n, out, olen);
  }
  uint64_t *counter, *status;
  uint32_t gen;
  MSV_TRY(c.lookback(1, &counter, &status, &gen));
  const bool aligned = (((uintptr_t)idx | (uintptr_t)values) & 15u) == 0;
  const uint32_t cus = (uint32_t)c.num_cus();
  hipLaunchKernelGGL((bin_tiles_kernel<T, IPT, true>), dim3(div_up(n, TILE)), dim3(kBinBlock), 0,
                     c.stream(), out, olen, idx, const_cast<T*>(values), n, p, aligned,
                     (const uint32_t*)nullptr, pidx, (uint16_t*)nullptr, pval, starts, chunks, status, gen);
  hipLaunchKernelGGL((bin_leaves_kernel<T, TILE>), dim3(std::min(p.windows * p.groups, 2 * cus)),
                     dim3(kBinBlock), 0, c.stream(), p, pidx, pval, starts, cidx, cval, rows, chunks,
                     status, gen);
  hipLaunchKernelGGL(leaf_scatter_kernel<T>, dim3(std::min(leaves, 2 * cus)), dim3(kBinBlock), 0,
                     c.stream(), out, olen, p, ((uintptr_t)out & 15u) == 0, cidx, cval, rows, chunks,
                     status, gen);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

// The binned gather: 4-byte elements (8-byte ones gained 16% at 2^27), at least
// 2^27 indices (random 2.54 -> 1.57 ms; the look and the launches that find
// nothing to do add 15 us to any other, 5% to a sorted gather there) and at most
// 16 table elements to an index, since every window is read once.
static bool gather_binned(msv_dtype dt, uint32_t n, uint32_t vlen) {
  return dtype_size(dt) == 4 && n >= (1u << 27) && vlen / 16 <= n && vlen >= (1u << 24);
}

// The binned scatter: from 2^23 indices and 32 MiB of output (u32 random 0.122
// -> 0.094 ms, reversed 0.038 -> 0.029; at 2^22 u64 random 0.072 -> 0.085), at
// most 16 output elements to an index, since every leaf is walked, and an
// output that 512 x 512 leaves cover.
constexpr uint64_t kBinScatterMinBytes = 32ull << 20;

bool scatter_binned(msv_dtype dt, uint32_t n, uint32_t olen) {
  return (uint64_t)olen * dtype_size(dt) >= kBinScatterMinBytes && n >= (1u << 23) && olen / 16 <= n &&
         (uint64_t)olen * dtype_size(dt) <= (uint64_t)kLeafBytes * kBinMost * kBinMost;
}

template <typename T>
static msv_status scatter_typed(Ctx& c, msv_dtype dt, const T* values, const uint32_t* idx,
                                uint32_t n, T* out, uint32_t olen) {
  return scatter_binned(dt, n, olen) ? binned_scatter(c, values, idx, n, out, olen)
                                     : direct_scatter(c, values, idx, n, out, olen);
}

msv_status gather_run(Ctx& c, msv_dtype dt, const void* values, uint32_t vlen,
                      const uint32_t* idx, void* out, uint32_t n) {
  if (n == 0) return MSV_OK;
  if (gather_binned(dt, n, vlen))
    return binned_gather(c, (const uint32_t*)values, vlen, idx, (uint32_t*)out, n);
  if (dtype_size(dt) == 4)
    return direct_gather(c, (const uint32_t*)values, vlen, idx, (uint32_t*)out, n);
  return direct_gather(c, (const uint64_t*)values, vlen, idx, (uint64_t*)out, n);
}

msv_status scatter_run(Ctx& c, msv_dtype dt, const void* values, const uint32_t* idx,
                       uint32_t n, void* out, uint32_t olen) {
  if (n == 0) return MSV_OK;
  if (dtype_size(dt) == 4)
    return scatter_typed(c, dt, (const uint32_t*)values, idx, n, (uint32_t*)out, olen);
  return scatter_typed(c, dt, (const uint64_t*)values, idx, n, (uint64_t*)out, olen);
}

msv_status uniform_run(Ctx& c, msv_dtype dt, void* out, uint32_t n, uint64_t seed) {
  if (n == 0) return MSV_OK;
  const dim3 grid((n + 255) / 256), block(256);
  switch (dt) {
    case MSV_U32:
    case MSV_I32:
      hipLaunchKernelGGL(uniform_u32_kernel, grid, block, 0, c.stream(), (uint32_t*)out, n, 0u,
                         seed_key(seed), 0u, 0xffffffffu);
      break;
    case MSV_F32:  // bit patterns of [0.5, 1)
      hipLaunchKernelGGL(uniform_u32_kernel, grid, block, 0, c.stream(), (uint32_t*)out, n, 0u,
                         seed_key(seed), 0x3F000000u, 0x007FFFFFu);
      break;
    case MSV_U64:
    case MSV_I64:
      hipLaunchKernelGGL(uniform_u64_kernel, grid, block, 0, c.stream(), (uint64_t*)out, n, 0u,
                         seed_key(seed), 0ull, ~0ull);
      break;
    case MSV_F64:  // bit patterns of [0.5, 1)
      hipLaunchKernelGGL(uniform_u64_kernel, grid, block, 0, c.stream(), (uint64_t*)out, n, 0u,
                         seed_key(seed), 0x3FE0000000000000ull, 0x000FFFFFFFFFFFFFull);
      break;
  }
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

msv_status iota_run(Ctx& c, uint32_t* out, uint32_t n, uint32_t start) {
  if (n == 0) return MSV_OK;
  hipLaunchKernelGGL(iota_u32_kernel, dim3((n + 255) / 256), dim3(256), 0, c.stream(), out, n,
                     start);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}


// ---- vector::scatter_reduce ----------------------------------------------------
// out[d] = op(out[d], init (+) the values whose index is d), for destinations
// present in `indices` (api/algorithm/scatter.rs:337-420; the reference sorts
// the proposals by index, reduces each run and combines each result with its
// destination, core/scatter_reduce.rs:19-150). `init` must be op's identity,
// as the reference requires. Integers: one pass of device-scope atomics, exact
// whatever the order. Floats: the reference's shape (stable radix sort of
// (index, value), reduce_by_key, one combine per destination), so results are
// reproducible bit for bit.
template <typename T, int OP>
__device__ inline void atomic_combine(T* p, T v) {
  if constexpr (OP == OP_ADD) {
    if constexpr (sizeof(T) == 4) atomicAdd((unsigned int*)p, (unsigned int)v);
    else atomicAdd((unsigned long long*)p, (unsigned long long)v);
  } else if constexpr (OP == OP_XOR) {
    if constexpr (sizeof(T) == 4) atomicXor((unsigned int*)p, (unsigned int)v);
    else atomicXor((unsigned long long*)p, (unsigned long long)v);
  } else if constexpr (OP == OP_MIN) {
    if constexpr (std::is_same<T, int64_t>::value) atomicMin((long long*)p, (long long)v);
    else if constexpr (std::is_same<T, uint64_t>::value) atomicMin((unsigned long long*)p, (unsigned long long)v);
    else atomicMin(p, v);
  } else {
    if constexpr (std::is_same<T, int64_t>::value) atomicMax((long long*)p, (long long)v);
    else if constexpr (std::is_same<T, uint64_t>::value) atomicMax((unsigned long long*)p, (unsigned long long)v);
    else atomicMax(p, v);
  }
}

template <typename T, int OP>
__global__ __launch_bounds__(256) void scatter_reduce_atomic_kernel(const T* __restrict__ vals,
                                                                    const uint32_t* __restrict__ idx,
                                                                    uint32_t n, T* out,
                                                                    uint32_t out_len, bool aligned) {
  const size_t groups = ((size_t)n + 3) / 4;
  for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < groups;
       g += (size_t)gridDim.x * blockDim.x) {
    const bool full = aligned && g * 4 + 4 <= n;
    uint32_t d[4];
    T v[4];
    load4<uint32_t>(idx, g * 4, n, full, d);
    load4<T>(vals, g * 4, n, full, v);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (g * 4 + k < n && d[k] < out_len) atomic_combine<T, OP>(out + d[k], v[k]);
  }
}

// One proposal per destination (keys distinct): out[d] = op(out[d], proposal).
template <typename T, int OP>
__global__ void scatter_combine_kernel(const uint32_t* __restrict__ keys, const T* __restrict__ vals,
                                       const uint32_t* __restrict__ count, T* __restrict__ out,
                                       uint32_t out_len) {
  const uint32_t m = *count;
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < m; j += gridDim.x * blockDim.x) {
    const uint32_t d = keys[j];
    if (d < out_len) out[d] = Combine<T, OP>::apply(out[d], vals[j]);
  }
}

template <typename T, int OP>
static msv_status scatter_reduce_typed(Ctx& c, msv_dtype dt, msv_op op, const void* vals,
                                       const uint32_t* idx, uint32_t n, const void* init,
                                       void* out, uint32_t out_len) {
  if (n == 0 || out_len == 0) return MSV_OK;
  if constexpr (!IsFloat<T>::value) {
    (void)dt;
    (void)op;
    (void)init;
    const bool aligned = (((uintptr_t)vals | (uintptr_t)idx) & 15u) == 0;
    const uint32_t groups = (n + 3) / 4;
    const uint32_t blocks = min((groups + 255) / 256, 8192u);
    hipLaunchKernelGGL((scatter_reduce_atomic_kernel<T, OP>), dim3(blocks), dim3(256), 0,
                       c.stream(), (const T*)vals, idx, n, (T*)out, out_len, aligned);
    MSV_HIP(hipGetLastError());
    return MSV_OK;
  } else {
    uint32_t* sk = (uint32_t*)c.scratch((size_t)n * 4);
    T* sv = (T*)c.scratch((size_t)n * sizeof(T));
    uint32_t* rk = (uint32_t*)c.scratch((size_t)n * 4);
    T* rv = (T*)c.scratch((size_t)n * sizeof(T));
    uint32_t* cnt = (uint32_t*)c.scratch(8);
    if (!sk || !sv || !rk || !rv || !cnt) return MSV_ERR_OUT_OF_MEMORY;
    MSV_TRY(radix_sort_run(c, MSV_U32, 0, sizeof(T), idx, vals, n, sk, sv));
    MSV_TRY(runs_scan_run(c, MSV_U32, sk, dt, op, RUNS_REDUCE, sv, n, rv, init, rk, cnt, cnt + 1));
    const uint32_t blocks = min((n + 255) / 256, 8192u);
    hipLaunchKernelGGL((scatter_combine_kernel<T, OP>), dim3(blocks), dim3(256), 0, c.stream(), rk,
                       rv, cnt, (T*)out, out_len);
    MSV_HIP(hipGetLastError());
    return MSV_OK;
  }
}

template <typename T>
static msv_status scatter_reduce_by_op(Ctx& c, msv_dtype dt, msv_op op, const void* vals,
                                       const uint32_t* idx, uint32_t n, const void* init,
                                       void* out, uint32_t out_len) {
  switch (op) {
    case MSV_OP_ADD: return scatter_reduce_typed<T, OP_ADD>(c, dt, op, vals, idx, n, init, out, out_len);
    case MSV_OP_MIN: return scatter_reduce_typed<T, OP_MIN>(c, dt, op, vals, idx, n, init, out, out_len);
    case MSV_OP_MAX: return scatter_reduce_typed<T, OP_MAX>(c, dt, op, vals, idx, n, init, out, out_len);
    case MSV_OP_XOR:
      if constexpr (!IsFloat<T>::value)
        return scatter_reduce_typed<T, OP_XOR>(c, dt, op, vals, idx, n, init, out, out_len);
      break;
  }
  set_error(MSV_ERR_INVALID_ARGUMENT, 0, 0, "operator %d is not defined for this dtype", (int)op);
  return MSV_ERR_INVALID_ARGUMENT;
}

}  // namespace msv

using namespace msv;

static msv_status check_index_slice(const View& v) {
  if (v.dtype != MSV_U32) {
    set_error(MSV_ERR_INVALID_ARGUMENT, 0, 0, "indices must be u32 (MIndex)");
    return MSV_ERR_INVALID_ARGUMENT;
  }
  return MSV_OK;
}

extern "C" {

msv_status msv_gather(msv_executor* ex, msv_slice values, msv_slice indices, msv_vec** out) {
  clear_error();
  View v, ix;
  MSV_TRY(resolve(ex, values, &v));
  MSV_TRY(resolve(ex, indices, &ix));
  MSV_TRY(check_index_slice(ix));
  MSV_TRY(new_vec(ex, v.dtype, ix.len, false, out));
  Ctx c(ex);
  msv_status s = gather_run(c, v.dtype, v.ptr, v.len, (const uint32_t*)ix.ptr, (*out)->ptr, ix.len);
  if (s != MSV_OK) {
    msv_vec_release(*out);
    *out = nullptr;
  }
  return s;
}

msv_status msv_scatter(msv_executor* ex, msv_slice values, msv_slice indices, msv_slice output) {
  clear_error();
  View v, ix, o;
  MSV_TRY(resolve(ex, values, &v));
  MSV_TRY(resolve(ex, indices, &ix));
  MSV_TRY(resolve(ex, output, &o));
  MSV_TRY(check_index_slice(ix));
  if (v.len != ix.len) {
    set_error(MSV_ERR_LENGTH_MISMATCH, v.len, ix.len, "input lengths differ: %u != %u", v.len,
              ix.len);
    return MSV_ERR_LENGTH_MISMATCH;
  }
  if (o.dtype != v.dtype) {
    set_error(MSV_ERR_INVALID_ARGUMENT, 0, 0, "output dtype differs from values");
    return MSV_ERR_INVALID_ARGUMENT;
  }
  Ctx c(ex);
  return scatter_run(c, v.dtype, v.ptr, (const uint32_t*)ix.ptr, v.len, o.ptr, o.len);
}

msv_status msv_scatter_reduce(msv_executor* ex, msv_slice values, msv_slice indices,
                              const void* init, msv_op op, msv_slice output) {
  clear_error();
  View v, ix, o;
  MSV_TRY(resolve(ex, values, &v));
  MSV_TRY(resolve(ex, indices, &ix));
  MSV_TRY(resolve(ex, output, &o));
  MSV_TRY(check_index_slice(ix));
  if (v.len != ix.len) {
    set_error(MSV_ERR_LENGTH_MISMATCH, v.len, ix.len, "input lengths differ: %u != %u", v.len,
              ix.len);
    return MSV_ERR_LENGTH_MISMATCH;
  }
  if (o.dtype != v.dtype || !init) {
    set_error(MSV_ERR_INVALID_ARGUMENT, 0, 0, "output dtype differs from values, or null init");
    return MSV_ERR_INVALID_ARGUMENT;
  }
  Ctx c(ex);
  const uint32_t* idx = (const uint32_t*)ix.ptr;
  switch (v.dtype) {
    case MSV_U32: return scatter_reduce_by_op<uint32_t>(c, v.dtype, op, v.ptr, idx, v.len, init, o.ptr, o.len);
    case MSV_I32: return scatter_reduce_by_op<int32_t>(c, v.dtype, op, v.ptr, idx, v.len, init, o.ptr, o.len);
    case MSV_F32: return scatter_reduce_by_op<float>(c, v.dtype, op, v.ptr, idx, v.len, init, o.ptr, o.len);
    case MSV_U64: return scatter_reduce_by_op<uint64_t>(c, v.dtype, op, v.ptr, idx, v.len, init, o.ptr, o.len);
    case MSV_I64: return scatter_reduce_by_op<int64_t>(c, v.dtype, op, v.ptr, idx, v.len, init, o.ptr, o.len);
    case MSV_F64: return scatter_reduce_by_op<double>(c, v.dtype, op, v.ptr, idx, v.len, init, o.ptr, o.len);
  }
  set_error(MSV_ERR_INVALID_ARGUMENT, 0, 0, "bad dtype");
  return MSV_ERR_INVALID_ARGUMENT;
}

msv_status msv_random_uniform_u32(msv_executor* ex, uint32_t min, uint32_t max, uint64_t seed,
                                  msv_slice out) {
  clear_error();
  View o;
  MSV_TRY(resolve(ex, out, &o));
  if (o.dtype != MSV_U32 || min > max) {
    set_error(MSV_ERR_LAUNCH, 0, 0, "random distribution range must satisfy min <= max (u32 out)");
    return MSV_ERR_LAUNCH;
  }
  if (o.len == 0) return MSV_OK;
  Ctx c(ex);
  hipLaunchKernelGGL(uniform_u32_kernel, dim3((o.len + 255) / 256), dim3(256), 0, c.stream(),
                     (uint32_t*)o.ptr, o.len, 0u, seed_key(seed), min, max - min);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

msv_status msv_random_uniform_u64(msv_executor* ex, uint64_t min, uint64_t max, uint64_t seed,
                                  msv_slice out) {
  clear_error();
  View o;
  MSV_TRY(resolve(ex, out, &o));
  if (o.dtype != MSV_U64 || min > max) {
    set_error(MSV_ERR_LAUNCH, 0, 0, "random distribution range must satisfy min <= max (u64 out)");
    return MSV_ERR_LAUNCH;
  }
  if (o.len == 0) return MSV_OK;
  Ctx c(ex);
  hipLaunchKernelGGL(uniform_u64_kernel, dim3((o.len + 255) / 256), dim3(256), 0, c.stream(),
                     (uint64_t*)o.ptr, o.len, 0u, seed_key(seed), min, max - min);
  MSV_HIP(hipGetLastError());
  return MSV_OK;
}

msv_status msv_iota_u32(msv_executor* ex, uint32_t start, msv_slice out) {
  clear_error();
  View o;
  MSV_TRY(resolve(ex, out, &o));
  if (o.dtype != MSV_U32) {
    set_error(MSV_ERR_INVALID_ARGUMENT, 0, 0, "iota output must be u32");
    return MSV_ERR_INVALID_ARGUMENT;
  }
  Ctx c(ex);
  return iota_run(c, (uint32_t*)o.ptr, o.len, start);
}

}  // extern "C"
