// Binned gather and scatter for gfx950: random indices into a table far larger
// than an XCD's 4 MiB L2.
//
// A direct random access moves a whole line for one element (48 G/s at 2^28
// u32). Both binned forms begin with bin_tiles_kernel, which sorts every tile
// of consecutive positions by table window in LDS; the order and the windows'
// starts stay tile-local, so there is no scan or look-back over tiles, and
// every later pass reads and writes runs of consecutive elements.
//  * gather: gather_look_kernel looks at some tiles, and the whole call goes
//    directly or this way. gather_window_kernel walks the table window by window
//    while it stays in one L2, and unbin_tiles_kernel undoes the sort through
//    LDS with the 16-bit source positions the sort kept (2^28 u32: 0.65 + 2.07 +
//    0.43 ms and 0.03 for the look and the direct kernel, which ends at once; 5.56
//    directly; the L2s serve about 130 G random reads/s).
//  * scatter: an L2 takes random 4-byte stores at about the same rate and lets
//    them go as partial lines, so it ends in LDS instead. bin_leaves_kernel
//    takes a window's runs from a group of tiles (a chunk of at most kBinChunk
//    elements; more of them where the window has more) and sorts them by leaf
//    (64 KiB of the table), chunk-local; leaf_scatter_kernel collects a leaf in
//    LDS and writes whole lines (2^28 u32: 0.76 + 0.93 + 0.52 ms, from 6.0 with one look-back
//    partition into 256 windows and random stores from L2).
// Each tile decides for itself as well: one whose indices stay near each other
// (sorted, reversed, clustered, rows of elements) is gathered or scattered
// directly by bin_tiles_kernel.
#pragma once

#include "device_common.hpp"

namespace msv {

constexpr int kBinBlock = 1024;
constexpr uint32_t kBinMost = 512;           // most windows, and most leaves per window
constexpr uint32_t kLeafBytes = 64u << 10;
constexpr uint32_t kBinChunk = 16384;        // elements of a chunk, at most
constexpr int kChunkIpt = kBinChunk / kBinBlock;
constexpr uint32_t kNoPlace = 0xffffffffu;   // an element a scatter drops
constexpr uint32_t kXcds = 8;

// How a table is cut: leaf = index >> leaf_shift; window = leaf >> sub_shift.
// A row of starts holds one entry per bin and the end, padded.
struct BinPlan {
  uint32_t leaf_shift, sub_shift;
  uint32_t windows, subs;      // subs = 1 << sub_shift
  uint32_t tile_row, chunk_row;
  uint32_t tiles, group, groups;  // full tiles; tiles of a group; groups
  uint32_t cap;                   // chunks a window can have
};

// What bin_leaves_kernel hands to leaf_scatter_kernel. Chunk c of window w has row
// w * cap + c of leaf starts. Elements are placed as blocks come, in one of
// kShards parts of the memory, a part to neighbouring windows (one counter for
// all blocks cost 8 us when 512 blocks begin at once, and chunks of a window all
// over the memory 5% of the collecting step); windows with more than their share
// go on in other parts.
constexpr uint32_t kShards = 64, kShardStep = 16;
struct BinChunks {
  uint32_t* used;    // elements / 8 of each part, kShardStep words apart
  uint32_t* counts;  // chunks of each window
  uint32_t* at;      // a chunk's first element / 8
  uint32_t shard;    // elements / 8 of a part
};

// Room for cnt elements (their first / 8), in two steps: the first only asks, so
// that the answer can come while the block does other work. A part that has run
// out leaves less than a chunk unused, which the parts' size allows for, so one
// of them has room. (A part that is seen to have none is not asked: its counter
// stays far from 2^32.)
__device__ inline uint32_t ask_room(const BinChunks& c, uint32_t part, uint32_t cnt) {
  return atomicAdd(&c.used[part * kShardStep], (cnt + 7) / 8);
}
// `other`: where this block found room the last time that a window's own part had none.
__device__ inline uint32_t take_room(const BinChunks& c, uint32_t part, uint32_t cnt, uint32_t asked,
                                     uint32_t& other) {
  const uint32_t units = (cnt + 7) / 8;
  while (asked + units > c.shard) {
    part = other;
    asked = __hip_atomic_load(&c.used[part * kShardStep], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (asked + units <= c.shard) asked = ask_room(c, part, cnt);
    if (asked + units > c.shard) other = (other * 13 + 11) % kShards;  // (goes through all of them)
  }
  return part * c.shard + asked;
}

// Exclusive scan of s_cnt[0, kBinMost) into s_start, by the first kBinMost
// threads; s_start[kBinMost] is the total, *s_most (zero before) the largest.
__device__ inline void bin_scan(const uint32_t* s_cnt, uint32_t* s_start, uint32_t* s_wsum,
                                uint32_t* s_most = nullptr) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6;
  uint32_t cnt = 0, incl = 0;
  if (tid < kBinMost) {
    cnt = s_cnt[tid];
    incl = wave_inclusive_scan<uint32_t, OP_ADD>(cnt);
    if (lane == 63) s_wsum[wid] = incl;
    if (s_most) {
      const uint32_t most = wave_reduce<uint32_t, OP_MAX>(cnt);
      if (lane == 0) atomicMax(s_most, most);
    }
  }
  __syncthreads();
  if (tid < kBinMost) {
    uint32_t off = 0;
    for (uint32_t w = 0; w < wid; ++w) off += s_wsum[w];
    s_start[tid] = off + incl - cnt;
    if (tid == kBinMost - 1) s_start[kBinMost] = off + incl;
  }
  __syncthreads();
}

template <typename T>
__device__ inline void store4(T* p, const T (&v)[4]) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<uint4*>(p) = make_uint4(bit_cast<uint32_t>(v[0]), bit_cast<uint32_t>(v[1]),
                                              bit_cast<uint32_t>(v[2]), bit_cast<uint32_t>(v[3]));
  } else {
    reinterpret_cast<ulonglong2*>(p)[0] = make_ulonglong2(bit_cast<uint64_t>(v[0]), bit_cast<uint64_t>(v[1]));
    reinterpret_cast<ulonglong2*>(p)[1] = make_ulonglong2(bit_cast<uint64_t>(v[2]), bit_cast<uint64_t>(v[3]));
  }
}

// Copies cnt elements of LDS (16-byte aligned) to global memory (16-byte
// aligned) as 16-byte stores; the last store may write past cnt (the
// destination is padded).
template <typename E>
__device__ inline void copy_out16(const E* s, E* g, uint32_t cnt) {
  constexpr uint32_t V = 16 / sizeof(E);
  for (uint32_t i = threadIdx.x * V; i < cnt; i += kBinBlock * V)
    *reinterpret_cast<uint4*>(g + i) = *reinterpret_cast<const uint4*>(s + i);
}

// How many indices lie outside the table window of their wave's first one,
// summed over the block (all threads call).
template <int N>
__device__ inline uint32_t count_far(const uint32_t (&ix)[N], uint32_t shift, uint32_t* s_far) {
  const uint32_t w0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(ix[0] >> shift));
  uint32_t far = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) far += (uint32_t)__builtin_popcountll(ballot((ix[j] >> shift) != w0));
  if ((threadIdx.x & 63u) == 0) atomicAdd(s_far, far);
  __syncthreads();
  return *s_far;
}

// Gather, step 1: whether the binned form pays, from kLooks looks at kLookTile
// indices, spread over all of them. A look votes for it when its indices touch
// lines of the table that no other of them touches (5/8 of them; rows of a few elements, a permutation back
// from a partition and strides along a matrix share lines, which a direct
// gather then finds in L2), do not go on by equal steps, and meet no window
// often (4 times the mean: indices near each other or a few hot ones, which a
// cache holds). 3/4 of the votes decide, since a tile that should have gone
// the other way costs more in the binned form. The look and the three launches
// that then find nothing to do add 15 us to a direct gather. Times at 2^28 u32, direct and
// binned (ms): random 5.56, 3.1; rows of 64 elements 0.57, 1.9; 256 interleaved
// sorted streams 1.19, 2.7; columns of a matrix 1.84, 2.8; random within a
// window of 2^20 that moves along 2.2, 4.7; Zipf 2.2, 2.2.
constexpr uint32_t kLooks = 64, kLookTile = 16384;
constexpr int kLineShift = 5;  // 4-byte elements of a 128-byte line

// The verdict of the looks (a byte each, 0 or 1).
__device__ inline bool look_binned(const uint32_t* __restrict__ looks) {
  uint32_t votes = 0;
#pragma unroll
  for (uint32_t i = 0; i < kLooks / 4; ++i) votes += (uint32_t)__builtin_popcount(looks[i]);
  return votes * 4 >= kLooks * 3;
}

static __global__ __launch_bounds__(kBinBlock) void gather_look_kernel(
    const uint32_t* __restrict__ idx, uint32_t n, BinPlan p, bool aligned, uint8_t* __restrict__ looks) {
  constexpr uint32_t TILE = kLookTile;
  constexpr int ROWS = (int)(TILE / kBinBlock / 4);
  constexpr uint32_t BITS = 17;  // of the lines' hash
  __shared__ uint32_t s_lines[(1u << BITS) / 32], s_cnt[kBinMost];
  __shared__ uint32_t s_new, s_regular, s_most;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t shift = p.leaf_shift + p.sub_shift;
  const size_t base = (size_t)((uint64_t)blockIdx.x * (n / TILE) / kLooks) * TILE;
  for (uint32_t i = tid; i < (1u << BITS) / 32; i += kBinBlock) s_lines[i] = 0;
  if (tid < kBinMost) s_cnt[tid] = 0;
  if (tid == 0) s_new = s_regular = s_most = 0;
  uint32_t ix[ROWS][4];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
    load4<uint32_t>(idx, base + ((size_t)r * kBinBlock + tid) * 4, 0xffffffffu, aligned, ix[r]);
  __syncthreads();
  uint32_t regular = 0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const uint32_t step = ix[r][1] - ix[r][0];
    regular += ix[r][2] - ix[r][1] == step && ix[r][3] - ix[r][2] == step ? 1 : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t line = ix[r][k] >> kLineShift;
      if (k == 0 || line != ix[r][k - 1] >> kLineShift) {
        const uint32_t h = (line * 2654435761u) >> (32 - BITS);
        atomicOr(&s_lines[h >> 5], 1u << (h & 31u));
      }
      // A wave in one window adds once (an index past the table counts for the last).
      const uint32_t w = min(ix[r][k] >> shift, p.windows - 1);
      const uint32_t w0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
      if (ballot(w != w0) != 0) atomicAdd(&s_cnt[w], 1u);
      else if (lane == 0) atomicAdd(&s_cnt[w0], (uint32_t)kWave);
    }
  }
  regular = wave_reduce<uint32_t, OP_ADD>(regular);
  if (lane == 0) atomicAdd(&s_regular, regular);
  __syncthreads();
  uint32_t lines = 0;
  for (uint32_t i = tid; i < (1u << BITS) / 32; i += kBinBlock) lines += (uint32_t)__builtin_popcount(s_lines[i]);
  lines = wave_reduce<uint32_t, OP_ADD>(lines);
  const uint32_t most = wave_reduce<uint32_t, OP_MAX>(tid < p.windows ? s_cnt[tid] : 0u);
  if (lane == 0) {
    atomicAdd(&s_new, lines);
    atomicMax(&s_most, most);
  }
  __syncthreads();
  if (tid == 0)
    looks[blockIdx.x] = s_new * 8 >= TILE * 5 && s_regular * 2 < TILE / 4 && s_most * p.windows <= 4 * TILE;
}

// Whether most lanes' four indices go up or down, from `least` to `most` between
// the first and the last.
__device__ inline bool ordered_wave(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t least,
                                    uint32_t most) {
  const bool up = a < b && b < c && c < d && d - a >= least && d - a <= most;
  const bool down = a > b && b > c && c > d && a - d >= least && a - d <= most;
  return __builtin_popcountll(ballot(up || down)) >= 3 * kWave / 4;
}

// Keeps one element of those of a tile with the same index (most of the time: not
// where another index has the same hash) and marks the others kNoPlace. All of
// them meet in one leaf, which one block collects: 2^24 u32 with Zipf indices
// (7% of them one index) 1.29 ms, now 0.13; 2^28 3.8 -> 1.93. s_slot: a word to
// an element.
template <int IPT>
__device__ inline void drop_repeats(uint32_t (&ix)[IPT], uint32_t tlen, uint32_t* s_slot) {
  constexpr uint32_t SLOTS = (uint32_t)kBinBlock * IPT;
  static_assert((SLOTS & (SLOTS - 1)) == 0 && IPT <= 32, "slots");
  auto slot = [](uint32_t i) { return (i * 2654435761u) >> (32 - __builtin_ctz(SLOTS)); };
  uint32_t mine = 0;  // elements whose index has its slot
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (ix[j] < tlen) s_slot[slot(ix[j])] = ix[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j) mine |= (ix[j] < tlen && s_slot[slot(ix[j])] == ix[j] ? 1u : 0u) << j;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (mine >> j & 1u) s_slot[slot(ix[j])] = threadIdx.x * IPT + j;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((mine >> j & 1u) && s_slot[slot(ix[j])] != threadIdx.x * IPT + j) ix[j] = kNoPlace;
  __syncthreads();
}

// The sort of one tile by window. table: the gather's values or the scatter's
// output, of tlen elements; io: the gather's output or the scatter's values,
// by position. pidx: the tile's indices in window order; ppos (gather): their
// in-tile positions; pval (scatter): their values. A row of zeros in `starts`:
// the tile was done directly. The gather takes the full tiles, and none unless
// the looks say so; the scatter takes every tile (the last, partial one
// directly), and a block that binned one says so in the launch's status word,
// for the later steps (looking at it first: 65536 stores to one word took 2.3 ms).
template <typename T, int IPT, bool SCATTER>
__global__ __launch_bounds__(kBinBlock, IPT * (SCATTER ? sizeof(T) : 4) == 64 ? 8 : 4) void bin_tiles_kernel(
    T* __restrict__ table, uint32_t tlen, const uint32_t* __restrict__ idx, T* __restrict__ io,
    uint32_t n, BinPlan p, bool aligned, const uint32_t* __restrict__ looks,
    uint32_t* __restrict__ pidx, uint16_t* __restrict__ ppos, T* __restrict__ pval,
    uint16_t* __restrict__ starts, BinChunks chunks, uint64_t* __restrict__ status, uint32_t gen) {
  constexpr uint32_t TILE = (uint32_t)kBinBlock * IPT;
  constexpr int ROWS = IPT / 4;
  constexpr uint32_t W = SCATTER ? sizeof(T) : 4;
  static_assert(TILE <= 32768 && IPT % 8 == 0, "tile");
  __shared__ __align__(16) unsigned char s_mem[TILE * W];
  __shared__ uint32_t s_cnt[kBinMost], s_start[kBinMost + 1];
  __shared__ uint32_t s_far, s_joined, s_out, s_most, s_wsum[kBinMost / kWave];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t shift = p.leaf_shift + p.sub_shift;
  uint32_t tile = blockIdx.x;
  if constexpr (!SCATTER) {
    if (!look_binned(looks)) return;
  } else if (tile == 0) {  // for the next step
    if (tid < p.windows) chunks.counts[tid] = 0;
    if (tid < kShards) chunks.used[tid * kShardStep] = 0;
  }
  do {
    const size_t base = (size_t)tile * TILE;
    const bool full = base + TILE <= n;
    uint16_t* row = starts + (size_t)tile * p.tile_row;
    __syncthreads();
    if (tid < kBinMost) s_cnt[tid] = 0;
    if (tid == 0) s_far = s_joined = s_out = s_most = 0;
    __syncthreads();

    // Element 4 r + k of a thread is position (r * kBinBlock + tid) * 4 + k.
    uint32_t ix[IPT];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const size_t i = base + ((size_t)r * kBinBlock + tid) * 4;
      if (full && aligned) {
        const uint4 q = load16_nt(idx + i);
        ix[4 * r] = q.x; ix[4 * r + 1] = q.y; ix[4 * r + 2] = q.z; ix[4 * r + 3] = q.w;
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) ix[4 * r + k] = i + k < n ? idx[i + k] : 0xffffffffu;
      }
    }
    if constexpr (SCATTER) {
      // Lanes whose first index shares its line with the one before it.
      constexpr int LINE = sizeof(T) == 4 ? kLineShift : kLineShift - 1;
      uint32_t joined = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t before = (uint32_t)__shfl_up((int)ix[4 * r + 3], 1);
        joined += (uint32_t)__builtin_popcountll(ballot(lane > 0 && before >> LINE == ix[4 * r] >> LINE));
      }
      if (lane == 0) atomicAdd(&s_joined, joined);
    }
    // Counted in registers first: the counts below would serialise on one
    // LDS word for a tile that stays in a window or two. Rows of some elements
    // are written directly as well (half of the lanes go on in a line): 2^28 u32
    // in rows of 64 3.5 -> 0.65 ms, of 16 2.7 -> 0.95; rows of 4 stay (2.6).
    bool spread = full && count_far(ix, shift, &s_far) * 2 >= TILE;
    if constexpr (SCATTER) spread = spread && s_joined * 2 < TILE / 4;
    if constexpr (!SCATTER) {
      bool out = false;
#pragma unroll
      for (int j = 0; j < IPT; ++j) out = out || ix[j] >= tlen;
      if (ballot(out)) s_out = 1;
      __syncthreads();
      spread = spread && s_out == 0;
    }
    uint32_t at[IPT];
    auto count = [&]() {
      // A scatter drops an index past the table; a gather reads 0 there, and
      // its tile is done directly.
#pragma unroll
      for (int j = 0; j < IPT; ++j)
        at[j] = !SCATTER || ix[j] < tlen ? atomicAdd(&s_cnt[ix[j] >> shift], 1u) : kNoPlace;
      __syncthreads();
      bin_scan(s_cnt, s_start, s_wsum, &s_most);
      spread = s_most * p.windows <= 4 * TILE;
    };
    if (spread) count();
    if constexpr (SCATTER) {
      // A window with far more than its share (6 standard deviations) may come
      // from an index that is there many times (then it also follows itself):
      // only one of its values stays.
      const int32_t over = (int32_t)s_most - (int32_t)(TILE / p.windows);
      bool twins = false;
      if (over > 0 && (uint32_t)(over * over) > 36 * (TILE / p.windows)) {
#pragma unroll
        for (int j = 1; j < IPT; ++j) twins = twins || ((j & 3) && ix[j] == ix[j - 1] && ix[j] < tlen);
        twins = __syncthreads_or(twins);
      }
      if (twins) {
        drop_repeats<IPT>(ix, tlen, reinterpret_cast<uint32_t*>(s_mem));
        if (tid < kBinMost) s_cnt[tid] = 0;
        if (tid == 0) s_most = 0;
        __syncthreads();
        count();
      }
    }
    if (!spread) {
      if (full && tid <= p.windows) row[tid] = 0;
      // Sorted indices some elements apart: consecutive lanes take consecutive
      // positions, so that a store of the wave has whole lines (2^24 u32, one to
      // 16: 750 -> 494 us; indices without gaps 157 -> 234 at 2^26).
      const bool lanes = SCATTER && ordered_wave(ix[0], ix[1], ix[2], ix[3], 4, 3 * 64);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const size_t o = base + ((size_t)r * kBinBlock + tid) * 4;
        T x[4];
        if constexpr (SCATTER) {
          if (lanes) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const size_t i = o - 3 * lane + k * kWave;
              const uint32_t d = i < n ? idx[i] : kNoPlace;
              if (d < tlen) table[d] = io[i];
            }
            continue;
          }
          load4<T, true>(io, o, n, full && aligned, x);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (ix[4 * r + k] < tlen) table[ix[4 * r + k]] = x[k];
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) x[k] = ix[4 * r + k] < tlen ? table[ix[4 * r + k]] : (T)0;
#pragma unroll
          for (int k = 0; k < 4; ++k) io[o + k] = x[k];
        }
      }
      if (SCATTER) return;
      continue;
    }

    // Recompute the windows below instead of keeping them in registers.
#pragma unroll
    for (int j = 0; j < IPT; ++j) asm volatile("" : "+v"(ix[j]));
    const uint32_t total = s_start[kBinMost];
    if constexpr (SCATTER) {
      if (tid == 0 && status_flag(ld_agent(status), gen) == 0)
        st_agent(status, pack_status(gen, kFlagInc, 0, 0));
    }
    if (tid < p.windows) row[tid] = (uint16_t)s_start[tid];
    if (tid == kBinMost) row[p.windows] = (uint16_t)total;
    uint32_t* s_idx = reinterpret_cast<uint32_t*>(s_mem);
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if (!SCATTER || at[j] != kNoPlace) {
        at[j] += s_start[ix[j] >> shift];
        s_idx[at[j]] = ix[j];
      }
    }
    __syncthreads();
    copy_out16(s_idx, pidx + base, total);
    __syncthreads();
    if constexpr (SCATTER) {
      T* s_val = reinterpret_cast<T*>(s_mem);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        T x[4];
        load4<T, true>(io, base + ((size_t)r * kBinBlock + tid) * 4, n, aligned, x);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (at[4 * r + k] != kNoPlace) s_val[at[4 * r + k]] = x[k];
      }
      __syncthreads();
      copy_out16(s_val, pval + base, total);
    } else {
      uint16_t* s_pos = reinterpret_cast<uint16_t*>(s_mem);
#pragma unroll
      for (int j = 0; j < IPT; ++j)
        s_pos[at[j]] = (uint16_t)(((uint32_t)(j / 4) * kBinBlock + tid) * 4 + (j & 3));
      __syncthreads();
      copy_out16(s_pos, ppos + base, total);
    }
  } while (!SCATTER && (tile += gridDim.x) < p.tiles);
}

// Gather, step 2: replaces the indices of the binned tiles by their values,
// window by window (pval may be pidx). Block b works on the windows w with
// w % 8 == b % 8, which the round-robin of workgroups keeps on one XCD, in
// order, so one or two windows are live in each L2. A group of 16 lanes reads
// the run of one tile, U elements a lane in flight. One block of four waves a
// CU and 2 MiB windows: 2.07 ms at 2^28 u32 (130 G reads/s); two blocks
// 2.35, eight 4.0 (more windows at once than an L2 holds), 4 MiB windows 2.5.
template <typename T, uint32_t TILE, int U>
__global__ __launch_bounds__(256) void gather_window_kernel(
    const T* __restrict__ table, uint32_t tlen, BinPlan p, const uint32_t* pidx, T* pval,
    const uint16_t* __restrict__ starts, const uint32_t* __restrict__ looks) {
  if (!look_binned(looks)) return;
  constexpr uint32_t kTilesPerWave = 16, kTilesPerBlock = 4 * kTilesPerWave;
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  const uint32_t g = blockIdx.x % kXcds;
  const uint32_t mine = p.windows > g ? (p.windows - g + kXcds - 1) / kXcds : 0u;
  const uint32_t chunks = (p.tiles + kTilesPerBlock - 1) / kTilesPerBlock;
  for (uint32_t q = blockIdx.x / kXcds; q < mine * chunks; q += gridDim.x / kXcds) {
    const uint32_t w = g + kXcds * (q / chunks);
    const uint32_t t0 = (q % chunks) * kTilesPerBlock + wid * kTilesPerWave;
    uint32_t s = 0, e = 0;
    if (lane < kTilesPerWave && t0 + lane < p.tiles) {
      const uint16_t* row = starts + (size_t)(t0 + lane) * p.tile_row + w;
      s = row[0];
      e = row[1];
    }
#pragma unroll
    for (uint32_t r = 0; r < kTilesPerWave / 4; ++r) {
      const uint32_t t = r * 4 + (lane >> 4);
      const uint32_t len = (uint32_t)__shfl((int)(e - s), (int)t);
      const size_t at = (size_t)(t0 + t) * TILE + (uint32_t)__shfl((int)s, (int)t);
      for (uint32_t k0 = lane & 15u; k0 < len; k0 += 16 * U) {
        uint32_t ix[U];
        T v[U];
        // The runs are read and written once: non-temporal, so the window stays.
#pragma unroll
        for (int k = 0; k < U; ++k)
          ix[k] = k0 + 16 * k < len ? __builtin_nontemporal_load(pidx + at + k0 + 16 * k) : tlen;
#pragma unroll
        for (int k = 0; k < U; ++k) v[k] = ix[k] < tlen ? table[ix[k]] : (T)0;
#pragma unroll
        for (int k = 0; k < U; ++k)
          if (k0 + 16 * k < len) __builtin_nontemporal_store(v[k], pval + at + k0 + 16 * k);
      }
    }
  }
}

// Copies the elements [lo, hi) of a sequence of runs of E (s_src: their first
// elements, s_off: their places in the sequence) to LDS, 32 lanes a run, four
// loads of a lane in flight.
template <typename E>
__device__ inline void load_runs(const E* __restrict__ from, const uint32_t* s_src,
                                 const uint32_t* s_off, uint32_t runs, uint32_t lo, uint32_t hi,
                                 E* s_to) {
  constexpr int U = 4;
  for (uint32_t r = threadIdx.x / 32; r < runs; r += kBinBlock / 32) {
    const uint32_t o = s_off[r], e = min(s_off[r + 1], hi);
    const E* src = from + s_src[r];
    for (uint32_t k0 = max(o, lo) + (threadIdx.x & 31u); k0 < e; k0 += 32 * U) {
      E d[U];
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + 32 * k < e) d[k] = src[k0 + 32 * k - o];
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + 32 * k < e) s_to[k0 + 32 * k - lo] = d[k];
    }
  }
}

// Scatter, step 2: the runs of one window in one group of tiles at a time, in as
// many chunks of equal length as they fill. cidx: the elements' places in their
// leaf, in leaf order; cval: their values. Where indices are spread evenly a
// group fills 7/8 of a chunk; a window with up to four times its share (a tile
// with more does not get here) takes up to four. (Chunks of fixed places, one to
// a window and group, with what did not fit scattered directly: 2^28 u32 into
// half of the output 9.0 ms, now 2.8.) Concurrent blocks take the
// windows of one group of tiles, so the runs they read are neighbours (a
// window at a time over all tiles was 8% slower: 1 KiB pieces of 1 GiB).
// 64 registers and 64 KiB of LDS: two blocks a CU (one: 1.12 ms at 2^28 u32, two
// then 0.86, and 0.93 with the chunks' places asked for).
template <typename T, uint32_t TILE>
__global__ __launch_bounds__(kBinBlock, sizeof(T) == 4 ? 8 : 4) void bin_leaves_kernel(
    BinPlan p, const uint32_t* __restrict__ pidx, const T* __restrict__ pval,
    const uint16_t* __restrict__ starts, uint16_t* __restrict__ cidx, T* __restrict__ cval,
    uint16_t* __restrict__ rows, BinChunks chunks, const uint64_t* __restrict__ status, uint32_t gen) {
  if (status_flag(ld_agent(status), gen) == 0) return;
  __shared__ __align__(16) T s_val[kBinChunk];
  __shared__ uint32_t s_cnt[kBinMost], s_off[kBinMost + 1], s_src[kBinMost];
  __shared__ uint32_t s_wsum[kBinMost / kWave];
  __shared__ uint32_t s_at, s_place;
  const uint32_t tid = threadIdx.x;
  uint32_t* s_idx = reinterpret_cast<uint32_t*>(s_val);
  uint16_t* s_16 = reinterpret_cast<uint16_t*>(s_val);
  uint32_t other = (kShards - 1 - blockIdx.x) % kShards;
  for (uint32_t q = blockIdx.x; q < p.windows * p.groups; q += gridDim.x) {
    const uint32_t w = q % p.windows, g = q / p.windows, part = w * kShards / p.windows;
    // The window's runs in the group's tiles: where each begins, and its place
    // among them.
    const uint32_t t0 = g * p.group, runs = min(p.group, p.tiles - t0);
    if (tid < kBinMost) {
      uint32_t s = 0, e = 0;
      if (tid < runs) {
        const uint16_t* r = starts + (size_t)(t0 + tid) * p.tile_row + w;
        s = r[0];
        e = r[1];
        s_src[tid] = (t0 + tid) * TILE + s;
      }
      s_cnt[tid] = e - s;
    }
    __syncthreads();
    bin_scan(s_cnt, s_off, s_wsum);
    const uint32_t total = s_off[kBinMost];
    const uint32_t pieces = (total + kBinChunk - 1) / kBinChunk;
    for (uint32_t c = 0; c < pieces; ++c) {
      const uint32_t lo = (uint32_t)((uint64_t)total * c / pieces);
      const uint32_t hi = (uint32_t)((uint64_t)total * (c + 1) / pieces), cnt = hi - lo;
      load_runs(pidx, s_src, s_off, runs, lo, hi, s_idx);
      if (tid < kBinMost) s_cnt[tid] = 0;
      __syncthreads();
      uint32_t place = 0, asked = 0;
      if (tid == kBinBlock - 1) {
        place = atomicAdd(&chunks.counts[w], 1u);
        asked = ask_room(chunks, part, cnt);
      }
      uint32_t ix[kChunkIpt], at[kChunkIpt];
#pragma unroll
      for (int j = 0; j < kChunkIpt; ++j) {
        const uint32_t i = tid + (uint32_t)j * kBinBlock;
        ix[j] = s_idx[i];
        at[j] = i < cnt ? atomicAdd(&s_cnt[(ix[j] >> p.leaf_shift) & (p.subs - 1)], 1u) : kNoPlace;
      }
      // Recompute the leaf numbers below instead of keeping them in registers.
#pragma unroll
      for (int j = 0; j < kChunkIpt; ++j) asm volatile("" : "+v"(ix[j]));
      __syncthreads();
      // The leaves' starts (over their counts: s_off still holds the runs' places).
      uint32_t n_leaf = 0, incl = 0;
      if (tid < kBinMost) {
        n_leaf = s_cnt[tid];
        incl = wave_inclusive_scan<uint32_t, OP_ADD>(n_leaf);
        if ((tid & 63u) == 63u) s_wsum[tid >> 6] = incl;
      }
      if (tid == kBinBlock - 1) {
        s_place = w * p.cap + place;
        s_at = take_room(chunks, part, cnt, asked, other);
        chunks.at[s_place] = s_at;
      }
      __syncthreads();
      uint16_t* row = rows + (size_t)s_place * p.chunk_row;
      const size_t first = (size_t)s_at * 8;
      if (tid < kBinMost) {
        uint32_t start = incl - n_leaf;
        for (uint32_t v = 0; v < (tid >> 6); ++v) start += s_wsum[v];
        s_cnt[tid] = start;
        if (tid < p.subs) row[tid] = (uint16_t)start;
      }
      if (tid == kBinMost) row[p.subs] = (uint16_t)cnt;
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kChunkIpt; ++j) {
        if (at[j] != kNoPlace) {
          at[j] += s_cnt[(ix[j] >> p.leaf_shift) & (p.subs - 1)];
          s_16[at[j]] = (uint16_t)(ix[j] & ((1u << p.leaf_shift) - 1));
        }
      }
      __syncthreads();
      copy_out16(s_16, cidx + first, cnt);
      __syncthreads();
      // The values the same way: runs into LDS, then from chunk to leaf order.
      load_runs(pval, s_src, s_off, runs, lo, hi, s_val);
      __syncthreads();
      T v[kChunkIpt];
#pragma unroll
      for (int j = 0; j < kChunkIpt; ++j) v[j] = s_val[tid + (uint32_t)j * kBinBlock];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kChunkIpt; ++j)
        if (at[j] != kNoPlace) s_val[at[j]] = v[j];
      __syncthreads();
      copy_out16(s_val, cval + first, cnt);
      __syncthreads();
    }
  }
}

// Scatter, step 3: one leaf a block at a time. The leaf's elements meet in LDS and leave as whole lines;
// a bitmap keeps what no index names unwritten.
template <typename T>
__global__ __launch_bounds__(kBinBlock) void leaf_scatter_kernel(
    T* __restrict__ table, uint32_t tlen, BinPlan p, bool aligned,
    const uint16_t* __restrict__ cidx, const T* __restrict__ cval,
    const uint16_t* __restrict__ rows, BinChunks chunks, const uint64_t* __restrict__ status, uint32_t gen) {
  if (status_flag(ld_agent(status), gen) == 0) return;
  constexpr uint32_t LEAF = kLeafBytes / sizeof(T);
  constexpr int U = 4;
  // Rows of so many elements (indices that follow each other in this leaf, as
  // behind a partition) are left for the whole block: 2^28 u32 in 256 streams
  // 3.25 -> 2.82 ms.
  constexpr uint32_t kLongRow = 1024, kLongRows = 64;
  __shared__ __align__(16) T s_leaf[LEAF];
  __shared__ uint32_t s_set[LEAF / 32];
  __shared__ uint3 s_long[kLongRows];
  __shared__ uint32_t s_longs;
  // Elements [i0, b) of the chunk at c, `step` apart.
  auto collect = [&](size_t c, uint32_t i0, uint32_t b, uint32_t step) {
    for (; i0 < b; i0 += step * U) {
      uint32_t d[U];
      T v[U];
#pragma unroll
      for (int q = 0; q < U; ++q)
        if (i0 + step * q < b) {
          d[q] = cidx[c + i0 + step * q];
          v[q] = cval[c + i0 + step * q];
        }
#pragma unroll
      for (int q = 0; q < U; ++q)
        if (i0 + step * q < b) {
          s_leaf[d[q]] = v[q];
          atomicOr(&s_set[d[q] >> 5], 1u << (d[q] & 31u));
        }
    }
  };
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6;
  const uint32_t leaves = (tlen - 1) / LEAF + 1;  // (tlen + LEAF may not fit 32 bits)
  for (uint32_t leaf = blockIdx.x; leaf < leaves; leaf += gridDim.x) {
    const uint32_t w = leaf >> p.sub_shift, sub = leaf & (p.subs - 1);
    const size_t l0 = (size_t)leaf * LEAF;
    if (tid == 0) s_longs = 0;
    for (uint32_t i = tid; i < LEAF / 32; i += kBinBlock) s_set[i] = 0;
    __syncthreads();
    const uint32_t mine = chunks.counts[w];
    for (uint32_t g0 = wid; g0 < mine; g0 += 16 * kWave) {
      uint32_t s = 0, e = 0, at = 0;
      const uint32_t g = g0 + 16 * lane;
      if (g < mine) {
        const uint32_t c = w * p.cap + g;
        const uint16_t* row = rows + (size_t)c * p.chunk_row + sub;
        at = chunks.at[c];
        s = row[0];
        e = row[1];
      }
      const uint32_t many = min((uint32_t)kWave, (mine - g0 + 15) / 16);
      for (uint32_t k = 0; k < many; ++k) {
        const uint32_t a = readlane(s, (int)k), b = readlane(e, (int)k);
        const uint32_t c = readlane(at, (int)k);
        if (b - a >= kLongRow) {
          uint32_t j = 0;
          if (lane == 0) j = atomicAdd(&s_longs, 1u);
          j = (uint32_t)__builtin_amdgcn_readfirstlane((int)j);
          if (j < kLongRows) {
            if (lane == 0) s_long[j] = make_uint3(c, a, b);
            continue;
          }
        }
        collect((size_t)c * 8, a + lane, b, kWave);
      }
    }
    __syncthreads();
    for (uint32_t j = 0; j < min(s_longs, kLongRows); ++j)
      collect((size_t)s_long[j].x * 8, s_long[j].y + tid, s_long[j].z, kBinBlock);
    __syncthreads();
    for (uint32_t i = tid * 4; i < LEAF; i += kBinBlock * 4) {
      const uint32_t m = (s_set[i >> 5] >> (i & 31u)) & 15u;
      if (m == 15u && aligned) {
        const T x[4] = {s_leaf[i], s_leaf[i + 1], s_leaf[i + 2], s_leaf[i + 3]};
        store4(table + l0 + i, x);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (m >> k & 1u) table[l0 + i + k] = s_leaf[i + k];
      }
    }
    __syncthreads();
  }
}

// Gather, step 3: a tile's values from window order back to positions.
template <typename T, int IPT>
__global__ __launch_bounds__(kBinBlock, IPT * sizeof(T) == 64 ? 8 : 4) void unbin_tiles_kernel(
    BinPlan p, const T* __restrict__ pval, const uint16_t* __restrict__ ppos,
    const uint16_t* __restrict__ starts, T* __restrict__ out, bool aligned,
    const uint32_t* __restrict__ looks) {
  if (!look_binned(looks)) return;
  constexpr uint32_t TILE = (uint32_t)kBinBlock * IPT;
  constexpr int V = 16 / sizeof(T);
  __shared__ __align__(16) T s_val[TILE];
  const uint32_t tid = threadIdx.x;
  for (uint32_t tile = blockIdx.x; tile < p.tiles; tile += gridDim.x) {
    if (starts[(size_t)tile * p.tile_row + p.windows] == 0) continue;
    const size_t base = (size_t)tile * TILE;
#pragma unroll
    for (int r = 0; r < IPT / 8; ++r) {
      const uint32_t i = ((uint32_t)r * kBinBlock + tid) * 8;
      const uint4 q = load16_nt(ppos + base + i);
      const uint32_t pw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int h = 0; h < 8; h += 4) {
        T x[4];
        load4<T, true>(pval + base, i + h, 0, true, x);
#pragma unroll
        for (int k = 0; k < 4; ++k) s_val[(pw[(h + k) / 2] >> (16 * (k & 1))) & 0xffffu] = x[k];
      }
    }
    __syncthreads();
    if (aligned) {
#pragma unroll
      for (int r = 0; r < IPT / V; ++r) {
        const uint32_t i = ((uint32_t)r * kBinBlock + tid) * V;
        *reinterpret_cast<uint4*>(out + base + i) = *reinterpret_cast<const uint4*>(s_val + i);
      }
    } else {
#pragma unroll
      for (int r = 0; r < IPT; ++r) out[base + (uint32_t)r * kBinBlock + tid] = s_val[r * kBinBlock + tid];
    }
    __syncthreads();
  }
}

}  // namespace msv
