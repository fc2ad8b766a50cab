// Expert histogram, offset scans and the stable token->expert counting sort.
//
// count:  one launch. Waves privatise the histogram (ballot/popcount counters in registers for <= 8 bins, LDS copies up to 1,024 bins,
//         one copy for the block beyond), blocks merge into a zero-initialised global accumulator, and the last block to finish (ticket
//         counters) scans the bins, writes counts / inclusive ends / exclusive starts and puts the accumulator back to
//         zero.
// sort:   up to 4,096 ids one launch of one block (sort_small_kernel), beyond that two. (1) every block histograms its
//         contiguous segment of the ids into its row of a table. (2) every block sums the table's columns, which with a scan
//         over the bins is the destination of its first id of every bin in a stable sort, and ranks its ids 64 at a time
//         with bit-ballots; block 0 writes counts / offsets / tile-aligned segment starts.
#include <stdlib.h>

#include "ck_common.h"

namespace ck {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kMaxCountBins = 16384;
constexpr int kMaxSortBins = 4096;
// The sort's table of counts holds at most this many words (bins * blocks). Half as many: 524,288 ids over 128 experts 1 %
// slower, 32,768 over 513 1.26 times, 131,072 over 4,096 1.66 times.
constexpr int kSortTableWords = 32768;
constexpr int kSortMaxBlocks = 256;            // one per CU
constexpr int64_t kSortIdsPerBlock = 1024;     // 2,048: 32,768 ids over 64 experts 7 % slower, 65,536 over 128 14 %

// Exclusive scan, in place, of data[0..n) (LDS) by a block of BLOCK threads. Returns the total. tmp: BLOCK / kWave words.
template <int BLOCK = kBlock>
__device__ uint32_t block_exclusive_scan(uint32_t* data, int n, uint32_t* tmp) {
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const int per = (n + BLOCK - 1) / BLOCK;
  const int b = min(n, t * per), e = min(n, b + per);
  uint32_t s = 0;
  for (int i = b; i < e; ++i) s += data[i];
  uint32_t incl = s;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t v = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += v;
  }
  __syncthreads();
  if (lane == kWave - 1) tmp[wave] = incl;
  __syncthreads();
  uint32_t wave_off = 0, total = 0;
#pragma unroll
  for (int w = 0; w < BLOCK / kWave; ++w) {
    const uint32_t v = tmp[w];
    if (w < wave) wave_off += v;
    total += v;
  }
  uint32_t run = wave_off + incl - s;
  for (int i = b; i < e; ++i) {
    const uint32_t v = data[i];
    data[i] = run;
    run += v;
  }
  __syncthreads();
  return total;
}

// Returns true in every thread of exactly one block: the last one to arrive. Blocks must have made their global writes before
// calling; the caller may read other blocks' writes after a true return. Blocks publish their data only through device-scope
// atomics, which are coherent across the XCDs by themselves: the L2 write-back + invalidate of a full fence (about 0.2 us per
// block, serialised) is not needed. Their completion is: an atomic that returns nothing is on its way to an L2 channel of its
// own when the wave goes on, and __syncthreads() waits for LDS only. So every wave waits for its own (vmcnt) ahead of
// the barrier behind which the block takes its ticket, or the last block could read an accumulator that an addition
// has yet to reach.
// Atomics on one address follow each other at about 9 ns, so the blocks take tickets of `groups` groups, each kTicketWords
// apart, and only the last of a group one of the launch (groups = 0: all of the launch). tickets: 1 word, or (1 + groups) *
// kTicketWords words, zero on entry and again when the last block has returned.
constexpr int kTicketWords = 16;
__device__ bool last_block_ticket(uint32_t* tickets, int groups, uint32_t* lds_flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t arrivals = gridDim.x;  // at the launch's ticket
    bool at_launch = true;
    if (groups > 0) {
      const uint32_t g = (uint32_t)groups, group = blockIdx.x % g, members = (gridDim.x - group + g - 1) / g;
      uint32_t* mine = tickets + (1 + group) * kTicketWords;
      arrivals = min(g, gridDim.x);
      at_launch = atomicAdd(mine, 1u) == members - 1;
      // nobody else of the group comes
      if (at_launch) __hip_atomic_store(mine, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool last = at_launch && atomicAdd(tickets, 1u) == arrivals - 1;
    if (last) __hip_atomic_store(tickets, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *lds_flag = last ? 1u : 0u;
  }
  __syncthreads();
  return *lds_flag != 0u;
}

template <typename id_t>
__device__ inline int load_id(const id_t* p) {
  const id_t v = *p;
  // ids outside int32 are out of range by definition; map them to -1
  if constexpr (sizeof(id_t) == 8) return (v >= 0 && v < (id_t)0x7fffffff) ? (int)v : -1;
  return (int)v;
}

// ------------------------------------------------------------------------------------------------------------
// count
// ------------------------------------------------------------------------------------------------------------
// What a count launch does with its workspace of 1 + bins * replicas words: tickets, then global accumulators.
struct CountLayout {
  int replicas;  // of the accumulator
  int groups;    // of tickets (last_block_ticket)
  int acc;       // first word of the accumulators
};

template <int REG_BINS>
struct RegCounters {
  uint32_t c[REG_BINS];
  __device__ RegCounters() {
#pragma unroll
    for (int i = 0; i < REG_BINS; ++i) c[i] = 0;
  }
  __device__ inline void add(int id) {
#pragma unroll
    for (int e = 0; e < REG_BINS; ++e) c[e] += (uint32_t)__popcll(__ballot(id == e));
  }
};

// REG_BINS > 0: wave-uniform register counters via ballot (num_bins <= REG_BINS): a handful of bins would make every
//               lane of an LDS atomic hit the same few addresses.
// REG_BINS == 0: LDS atomics on per-wave copies of the histogram.
template <typename id_t, int REG_BINS, int BLOCK>
__global__ __launch_bounds__(BLOCK) void count_kernel(const id_t* __restrict__ ids, int64_t n, int num_bins,
                                                        int lds_copies, CountLayout layout, uint32_t* __restrict__ counts,
                                                        uint32_t* __restrict__ ends, uint32_t* __restrict__ starts,
                                                        uint32_t* __restrict__ ws) {
  extern __shared__ uint32_t lds[];  // [lds_copies][num_bins] then (BLOCK / kWave) + 1 words of scan scratch
  uint32_t* hist = lds;
  uint32_t* tmp = lds + (size_t)lds_copies * num_bins;
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;

  for (int i = t; i < lds_copies * num_bins; i += BLOCK) hist[i] = 0;
  __syncthreads();
  uint32_t* my_hist = hist + (size_t)(lds_copies > 1 ? wave % lds_copies : 0) * num_bins;

  constexpr int VEC = 16 / sizeof(id_t);
  // scalar head up to the first 16-byte boundary, vector body, scalar tail
  const uintptr_t addr = reinterpret_cast<uintptr_t>(ids);
  int64_t head = ((16 - (addr & 15)) & 15) / sizeof(id_t);
  if (head > n) head = n;
  const int64_t nvec = (n - head) / VEC;
  const int64_t tail_begin = head + nvec * VEC;

  RegCounters<(REG_BINS > 0 ? REG_BINS : 1)> rc;
  auto tally = [&](int id) {
    if constexpr (REG_BINS > 0) {
      rc.add(id);
    } else {
      if ((unsigned)id < (unsigned)num_bins) atomicAdd(&my_hist[id], 1u);
    }
  };

  const id_t* body = ids + head;
  const int64_t gthreads = (int64_t)gridDim.x * BLOCK;
  const int64_t gtid = (int64_t)blockIdx.x * BLOCK + t;
  constexpr int UNROLL = 4;
  // every wave runs the same number of iterations so that ballots see whole waves
  const int64_t iters = (nvec + gthreads * UNROLL - 1) / (gthreads * UNROLL);
  for (int64_t it = 0; it < iters; ++it) {
    vec16 v[UNROLL];
    bool ok[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int64_t vi = (it * UNROLL + u) * gthreads + gtid;
      ok[u] = vi < nvec;
      v[u] = ok[u] ? load16_nt(body + vi * VEC) : zero16();  // ids are read once
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if constexpr (sizeof(id_t) == 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) tally(ok[u] ? (int)v[u].w[j] : -1);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int64_t x = (int64_t)(((uint64_t)v[u].w[2 * j + 1] << 32) | v[u].w[2 * j]);
          tally((ok[u] && x >= 0 && x < 0x7fffffff) ? (int)x : -1);
        }
      }
    }
  }
  if (blockIdx.x == 0) {  // ragged ends, at most VEC-1 ids each; whole waves participate (ballot)
    const int64_t ragged = head + (n - tail_begin);
    for (int64_t base = 0; base < ragged; base += BLOCK) {
      const int64_t r = base + t;
      int id = -1;
      if (r < ragged) id = load_id(ids + (r < head ? r : tail_begin + (r - head)));
      tally(id);
    }
  }

  if constexpr (REG_BINS > 0) {
    if (lane == 0) {
#pragma unroll
      for (int e = 0; e < REG_BINS; ++e)
        if (e < num_bins && rc.c[e]) atomicAdd(&hist[e], rc.c[e]);
    }
  }
  __syncthreads();
  if (lds_copies > 1) {
    for (int e = t; e < num_bins; e += BLOCK) {
      uint32_t s = 0;
      for (int c = 0; c < lds_copies; ++c) s += hist[(size_t)c * num_bins + e];
      hist[e] = s;  // copy 0 row becomes the block total; other rows are not read again
    }
    __syncthreads();
  }

  // Blocks merge into one of several global accumulators (thousands of atomics on one cache line would serialise in a
  // single L2 channel); the last block adds the replicas up and puts them back to zero.
  uint32_t* acc = ws + layout.acc;
  if (gridDim.x > 1) {
    uint32_t* my_acc = acc + (size_t)(blockIdx.x % layout.replicas) * num_bins;
    for (int e = t; e < num_bins; e += BLOCK)
      if (hist[e]) atomicAdd(&my_acc[e], hist[e]);
    const int used = min(layout.replicas, (int)gridDim.x);
    if (!last_block_ticket(ws, layout.groups, tmp + (BLOCK / kWave))) return;
    // Sum the replicas that were used and put them back to zero. Device-scope atomic loads read the values where the
    // other blocks' atomics left them; the loads of one thread are independent, so their latencies overlap.
    for (int e = t; e < num_bins; e += BLOCK) hist[e] = 0;
    __syncthreads();
    for (int idx = t; idx < used * num_bins; idx += BLOCK) {  // (replica, bin) pairs spread over the whole block
      const uint32_t v = __hip_atomic_load(&acc[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      acc[idx] = 0u;  // visible to the next launch at the kernel boundary; nobody reads it before
      if (v) atomicAdd(&hist[idx % num_bins], v);
    }
    __syncthreads();
  }
  // hist[0..num_bins) now holds the global counts
  for (int e = t; e < num_bins; e += BLOCK) counts[e] = hist[e];
  if (ends != nullptr || starts != nullptr) {
    __syncthreads();
    block_exclusive_scan<BLOCK>(hist, num_bins, tmp);
    for (int e = t; e < num_bins; e += BLOCK) {
      const uint32_t s = hist[e];
      if (starts) starts[e] = s;
      if (ends) ends[e] = s + counts[e];  // counts[e] was written by this same thread above
    }
  }
}

// ------------------------------------------------------------------------------------------------------------
// sort
// ------------------------------------------------------------------------------------------------------------
// Blocks of the two-launch sort. Up to kSmallBins bins a block has 16 waves; beyond, 4, as its counters are one word per bin
// and wave in LDS. Every block of the second launch reads the whole table of per-block counts: E * blocks words.
constexpr int kSortPer = 4;  // ids a lane holds in registers
constexpr int kWideWaves = 16, kNarrowWaves = 4;
constexpr int kSmallBins = 512;

struct SortPlan {
  int blocks;
  int64_t seg_len;  // ids of one block: a multiple of 64 per wave
};

SortPlan make_sort_plan(int64_t R, int E) {
  const int64_t unit = (int64_t)(E <= kSmallBins ? kWideWaves : kNarrowWaves) * kWave;
  int64_t cap = kSortTableWords / (E > 0 ? E : 1);
  if (cap > kSortMaxBlocks) cap = kSortMaxBlocks;
  if (cap < 1) cap = 1;
  const int64_t want = ceil_div(R > 0 ? R : 1, kSortIdsPerBlock);
  SortPlan p;
  p.blocks = (int)(want < cap ? want : cap);
  p.seg_len = round_up(ceil_div(R > 0 ? R : 1, p.blocks), unit);
  return p;
}

// tile_expert[tile]: the expert whose padded segment holds the tile's rows, -1 past the last one. padded: [E + 1] starts (LDS)
__device__ inline void write_tile_experts(const uint32_t* padded, int E, uint32_t padded_total, int align, int64_t max_tiles,
                                          int32_t* __restrict__ tile_expert, int64_t t, int64_t threads) {
  for (int64_t tile = t; tile < max_tiles; tile += threads) {
    const uint32_t row = (uint32_t)(tile * align);
    int32_t owner = -1;
    if (row < padded_total) {
      // last e with padded[e] <= row; empty experts share a start with their successor and are skipped by "last"
      int lo = 0, hi = E - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (padded[mid] <= row) lo = mid; else hi = mid - 1;
      }
      owner = lo;
    }
    tile_expert[tile] = owner;
  }
}

// ranks of 64 ids (one per lane): the lanes of the wave that hold the same id
__device__ inline uint64_t lanes_with_same_id(int id, bool valid, int id_bits) {
  uint64_t peers = __ballot(valid);
  for (int b = 0; b < id_bits; ++b) {
    const bool bit = (id >> b) & 1;
    const uint64_t m = __ballot(bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

// First launch of the sort: table[block][bin] = how often the bin occurs in the block's contiguous segment of the ids.
template <typename id_t, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void sort_hist_kernel(const id_t* __restrict__ ids, int64_t R, int E, int64_t seg_len,
                                                                  uint32_t* __restrict__ table) {
  constexpr int BLOCK = WAVES * kWave;
  extern __shared__ uint32_t lds[];  // [WAVES][E]: a wave's own counters, so that few bins do not serialise the whole block
  const int t = threadIdx.x, wave = t / kWave;
  for (int i = t; i < WAVES * E; i += BLOCK) lds[i] = 0;
  const int64_t begin = (int64_t)blockIdx.x * seg_len;
  const int64_t end = min(R, begin + seg_len);
  bool cleared = false;
  for (int64_t base = begin + t; base - t < end; base += kSortPer * BLOCK) {
    int id[kSortPer];
#pragma unroll
    for (int u = 0; u < kSortPer; ++u) {
      const int64_t i = base + u * BLOCK;
      id[u] = i < end ? load_id(ids + i) : -1;
    }
    if (!cleared) __syncthreads();  // block-uniform; the first ids are under way meanwhile
    cleared = true;
#pragma unroll
    for (int u = 0; u < kSortPer; ++u)
      if ((unsigned)id[u] < (unsigned)E) atomicAdd(&lds[wave * E + id[u]], 1u);
  }
  __syncthreads();
  for (int e = t; e < E; e += BLOCK) {
    uint32_t n = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) n += lds[w * E + e];
    table[(int64_t)blockIdx.x * E + e] = n;
  }
}

// Second launch: every block sums the table's columns (all blocks, and those ahead of it), scans the bins, ranks its ids 64
// at a time with bit-ballots and writes them to their places; the outputs per bin come from block 0, the tiles' experts
// from all blocks.
// What bounds the sort: latency. In the form before, one block scanned the table of all waves' counts behind a device-wide
// fence and ticket, and wrote it back for the second launch; here the launch boundary is the only wait between blocks, the
// table has one row per block instead of per wave, and reading all of it takes a block less time than the hand-over did.
// The blocks' number is free of that one block's scan, so that a wave ranks 64 to 256 ids instead of 1,024 to 4,096.
// Measured, both launches, 50 sorts in a replayed graph (no host time), before -> now: 8,192 ids over 64 experts 17.7 -> 9.2 us,
// 32,768 over 64 21.2 -> 9.8, 32,768 over 512 64 -> 12.6, 65,536 over 128 39.9 -> 10.6, 524,288 over 128 99 -> 18.1, 2,000,003
// over 60 150 -> 35, 131,072 over 4,096 494 -> 96.
template <typename id_t, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void sort_scatter_kernel(
    const id_t* __restrict__ ids, int64_t R, int E, int64_t seg_len, int id_bits, int align, int64_t max_tiles,
    const uint32_t* __restrict__ table, int32_t* __restrict__ sorted_expert_idxs, int32_t* __restrict__ sorted_scattered_idxs,
    uint32_t* __restrict__ counts, uint32_t* __restrict__ ends, uint32_t* __restrict__ starts, int32_t* __restrict__ seg_starts,
    int32_t* __restrict__ row_slot, int32_t* __restrict__ tile_expert) {
  constexpr int BLOCK = WAVES * kWave, STRIDE = WAVES + 1;  // a spare word per bin (always zero) spreads the bins over the banks
  extern __shared__ uint32_t lds[];  // next [E][STRIDE], ahead [E], start [E], padded [E + 1], scan scratch [WAVES]
  uint32_t *next = lds, *ahead = lds + STRIDE * E, *start = ahead + E, *padded = start + E, *tmp = padded + E + 1;
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const int S = gridDim.x, me = blockIdx.x;
  const int64_t per_wave = seg_len / WAVES;
  const int64_t begin = (int64_t)me * seg_len + wave * per_wave, end = min(R, begin + per_wave);
  constexpr int kRound = kSortPer * kWave;  // ids of a wave per round trip
  int id[kSortPer];
  auto fetch = [&](int64_t base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kSortPer; ++u) {
      const int64_t i = base + u * kWave + lane;
      id[u] = i < end ? load_id(ids + i) : -1;
    }
  };
  fetch(begin);
  for (int i = t; i < (STRIDE + 2) * E; i += BLOCK) lds[i] = 0;  // next, ahead, start
  __syncthreads();

  // ---- column sums: BLOCK / E threads share a bin where there are fewer bins than threads
  const int parts = E < BLOCK ? BLOCK / E : 1, part = E < BLOCK ? t / E : 0;
  if (part < parts) {
    for (int e = t - part * E; e < E; e += BLOCK) {
      uint32_t all = 0, before = 0;
#pragma unroll 8
      for (int s = part; s < S; s += parts) {
        const uint32_t n = table[(int64_t)s * E + e];
        all += n;
        if (s < me) before += n;
      }
      atomicAdd(&start[e], all);
      atomicAdd(&ahead[e], before);
    }
  }
  // ---- this block's ids by bin and wave
  for (int64_t base = begin; base < end; base += kRound) {
    if (base > begin) fetch(base);
#pragma unroll
    for (int u = 0; u < kSortPer; ++u)
      if ((unsigned)id[u] < (unsigned)E) atomicAdd(&next[id[u] * STRIDE + wave], 1u);
  }
  __syncthreads();
  for (int e = t; e < E; e += BLOCK) {
    const uint32_t c = start[e];
    padded[e] = (c + (uint32_t)align - 1) / (uint32_t)align * (uint32_t)align;
    if (me == 0) counts[e] = c;
  }
  __syncthreads();
  block_exclusive_scan<BLOCK>(start, E, tmp);
  const uint32_t padded_total = block_exclusive_scan<BLOCK>(padded, E, tmp);
  block_exclusive_scan<BLOCK>(next, E * STRIDE, tmp);
  if (me == 0) {
    for (int e = t; e < E; e += BLOCK) {
      starts[e] = start[e];
      ends[e] = start[e] + counts[e];  // counts[e] was written by this same thread above
      seg_starts[e] = (int32_t)padded[e];
    }
    if (t == 0) seg_starts[E] = (int32_t)padded_total;
  }
  // next[e][w] counts from the block's first id on: to the bin's place among all blocks
  for (int e = t; e < E; e += BLOCK) ahead[e] += start[e] - next[e * STRIDE];
  __syncthreads();
  write_tile_experts(padded, E, padded_total, align, max_tiles, tile_expert, (int64_t)me * BLOCK + t, (int64_t)S * BLOCK);
  const uint64_t lanes_below = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
  const bool again = per_wave > kRound;  // more than the registers hold: read once more, out of L2
  for (int64_t base = begin; base < end; base += kRound) {
    if (again) fetch(base);
#pragma unroll
    for (int u = 0; u < kSortPer; ++u) {
      if (base + u * kWave >= end) break;
      const bool valid = (unsigned)id[u] < (unsigned)E;
      const uint64_t peers = lanes_with_same_id(id[u], valid, id_bits);
      if (valid) {
        uint32_t* mine = &next[id[u] * STRIDE + wave];  // this wave's word alone; its LDS operations keep their order
        const uint32_t local = *mine + (uint32_t)__popcll(peers & lanes_below);
        if ((peers >> lane) == 1ull) *mine = local + 1;  // the highest lane of the group advances the bin
        const uint32_t pos = ahead[id[u]] + local;
        const int32_t i = (int32_t)(base + u * kWave + lane);
        sorted_expert_idxs[pos] = id[u];
        sorted_scattered_idxs[pos] = i;
        row_slot[padded[id[u]] + (pos - start[id[u]])] = i;
      }
    }
  }
}

// Exclusive scan over the bins as a wave holds them: lane l bins l, 64 + l, ..
template <int NB>
__device__ inline void bins_exclusive_scan(const uint32_t (&v)[NB], uint32_t (&before)[NB], int lane) {
  uint32_t total = 0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    uint32_t incl = v[b];
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t u = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += u;
    }
    before[b] = total + incl - v[b];
    total += __shfl(incl, kWave - 1, kWave);
  }
}

// The sort over up to 64 NB experts: the whole of it in one block (SMALL: the ids fit its registers) or the second of two launches.
// What bounds it is latency, and most of that was the block's barriers: three block-wide scans of two or three barriers each
// beside four more. With a bin (or two) per lane every wave scans all bins in its own registers, and sums over the waves as it
// reads them: one barrier, behind which no wave waits for another. 50 sorts in a replayed graph, the kernels for any number of
// experts -> these: 16 ids over 64 experts 4.6 -> 3.3 us, 512 over 64 4.75 -> 3.45, 1,024 over 128 5.4 -> 4.7, 4,096 over 64 8.9 -> 7.0, in
// two launches 8,192 over 64 9.3 -> 7.05, 32,768 over 64 9.9 -> 7.6, over 128 10.9 -> 9.15, 65,536 over 64 10.6 -> 7.7, 524,288 over
// 128 18.3 -> 16.9, 2,000,003 over 60 34.5 -> 30.4.
constexpr int kLaneWaves = 16, kLaneBins = 2 * kWave;
constexpr int kLaneIds = kLaneWaves * kWave * kSortPer;  // R up to which one block sorts
template <typename id_t, int NB, bool SMALL>
__global__ __launch_bounds__(kLaneWaves * kWave) void sort_lanes_kernel(
    const id_t* __restrict__ ids, int64_t R, int E, int64_t seg_len, int id_bits, int align, int64_t max_tiles,
    const uint32_t* __restrict__ table, int32_t* __restrict__ sorted_expert_idxs, int32_t* __restrict__ sorted_scattered_idxs,
    uint32_t* __restrict__ counts, uint32_t* __restrict__ ends, uint32_t* __restrict__ starts, int32_t* __restrict__ seg_starts,
    int32_t* __restrict__ row_slot, int32_t* __restrict__ tile_expert) {
  constexpr int W = kLaneWaves, BINS = NB * kWave;
  __shared__ uint32_t hist[W][BINS];                                 // a wave's own ids by bin
  __shared__ uint32_t all[SMALL ? 1 : W][BINS], before[SMALL ? 1 : W][BINS];  // a wave's share of the table: of all blocks, of those ahead
  __shared__ uint32_t next[W][BINS], padded[W][BINS + 1];            // a wave's own: the bins' next places; their padded starts
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave, me = blockIdx.x;
  const int64_t per_wave = seg_len / W, begin = (int64_t)me * seg_len + wave * per_wave, end = min(R, begin + per_wave);
  constexpr int kRound = kSortPer * kWave;
  int id[kSortPer];
  auto fetch = [&](int64_t base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kSortPer; ++u) {
      const int64_t i = base + u * kWave + lane;
      id[u] = u * kWave < per_wave && i < end ? load_id(ids + i) : -1;
    }
  };
  fetch(begin);
#pragma unroll
  for (int b = 0; b < NB; ++b) hist[wave][b * kWave + lane] = 0;
  if constexpr (!SMALL) {
    uint32_t a[NB] = {}, n_before[NB] = {};
#pragma unroll 4
    for (int s = wave; s < (int)gridDim.x; s += W)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint32_t n = b * kWave + lane < E ? table[(int64_t)s * E + b * kWave + lane] : 0;
        a[b] += n;
        if (s < me) n_before[b] += n;
      }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      all[wave][b * kWave + lane] = a[b];
      before[wave][b * kWave + lane] = n_before[b];
    }
  }
  for (int64_t base = begin; base < end; base += kRound) {
    if (base > begin) fetch(base);
#pragma unroll
    for (int u = 0; u < kSortPer; ++u)
      if ((unsigned)id[u] < (unsigned)E) atomicAdd(&hist[wave][id[u]], 1u);
  }
  __syncthreads();

  // ---- every wave for itself: the bins' counts, starts and padded starts, and how many ids of a bin lie ahead of its own
  uint32_t count[NB] = {}, ahead[NB] = {}, start[NB], size[NB], pad[NB];
#pragma unroll
  for (int w = 0; w < W; ++w)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t mine = hist[w][b * kWave + lane];
      if constexpr (SMALL) {
        count[b] += mine;
      } else {
        count[b] += all[w][b * kWave + lane];
        ahead[b] += before[w][b * kWave + lane];
      }
      if (w < wave) ahead[b] += mine;
    }
  bins_exclusive_scan<NB>(count, start, lane);
#pragma unroll
  for (int b = 0; b < NB; ++b) size[b] = (count[b] + (uint32_t)align - 1) / (uint32_t)align * (uint32_t)align;
  bins_exclusive_scan<NB>(size, pad, lane);
  uint32_t padded_total = __shfl(pad[NB - 1] + size[NB - 1], kWave - 1, kWave);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int e = b * kWave + lane;
    next[wave][e] = start[b] + ahead[b];
    padded[wave][e] = pad[b];
    if (me == 0 && wave == 0 && e < E) {
      counts[e] = count[b];
      starts[e] = start[b];
      ends[e] = start[b] + count[b];
      seg_starts[e] = (int32_t)pad[b];
      if (e == E - 1) seg_starts[E] = (int32_t)padded_total;
    }
  }
  __builtin_amdgcn_wave_barrier();  // the wave's own LDS words, in order
  write_tile_experts(padded[wave], E, padded_total, align, max_tiles, tile_expert, (int64_t)me * W * kWave + t, (int64_t)gridDim.x * W * kWave);
  const uint64_t lanes_below = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
  const bool again = per_wave > kRound;  // more than the registers hold: read once more, out of L2
  for (int64_t base = begin; base < end; base += kRound) {
    if (again) fetch(base);
#pragma unroll
    for (int u = 0; u < kSortPer; ++u) {
      if (u * kWave >= per_wave || base + u * kWave >= end) break;
      const bool valid = (unsigned)id[u] < (unsigned)E;
      const uint64_t peers = lanes_with_same_id(id[u], valid, id_bits);
      const int bin = valid ? id[u] : 0;
      uint32_t shift = 0;  // padded start less start of the id's bin
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint32_t v = __shfl(pad[b] - start[b], bin & (kWave - 1), kWave);
        if (bin / kWave == b) shift = v;
      }
      if (valid) {
        uint32_t* mine = &next[wave][bin];  // this wave's word alone; its LDS operations keep their order
        const uint32_t pos = *mine + (uint32_t)__popcll(peers & lanes_below);
        if ((peers >> lane) == 1ull) *mine = pos + 1;  // the highest lane of the group advances the bin
        const int32_t i = (int32_t)(base + u * kWave + lane);
        sorted_expert_idxs[pos] = bin;
        sorted_scattered_idxs[pos] = i;
        row_slot[pos + shift] = i;
      }
    }
  }
}

// The whole sort in one block and one launch, for few ids over more than kLaneBins experts. What bounds it: latency.
// An id is read once and stays in registers, and the table in LDS; the second launch and the way of the table through memory
// go. Measured, 40 sorts in a replayed graph, one launch against two: 8 / 512 / 2,048 / 3,500 / 4,096 ids over 129 experts 4.9 / 5.1
// / 6.9 / 9.0 / 9.9 against 8.2 / 8.5 / 9.2 / 9.6 / 9.6 us, over 384 5.7 / 6.1 / 7.8 / 10.5 / 11.1 against 9.0 / 9.7 / 10.5 / 11.0 / 10.8;
// over 512 3,000 / 3,500 / 4,096 ids 11.2 / 12.2 / 13.2 against 11.1 / 11.3 / 11.4. The line lies where the two meet: past it one
// block's rounds of 64, and its scan of a word per expert and wave, take longer than launches that spread them over the chip.
constexpr int kSmallBlock = 1024, kSmallWaves = kSmallBlock / kWave;
constexpr int kSmallPer = 4;                                  // ids per lane
constexpr int kSmallIds = kSmallBlock * kSmallPer;            // R up to which the one-block sort runs, up to kSmallBins bins
constexpr int small_ids(int E) { return E <= 384 ? kSmallIds : kSmallIds * 3 / 4; }

template <typename id_t>
__global__ __launch_bounds__(kSmallBlock) void sort_small_kernel(const id_t* __restrict__ ids, int R, int E, int align, int64_t max_tiles,
                                                                  int id_bits, int32_t* __restrict__ sorted_expert_idxs,
                                                                  int32_t* __restrict__ sorted_scattered_idxs, uint32_t* __restrict__ counts,
                                                                  uint32_t* __restrict__ ends, uint32_t* __restrict__ starts,
                                                                  int32_t* __restrict__ seg_starts, int32_t* __restrict__ row_slot,
                                                                  int32_t* __restrict__ tile_expert) {
  extern __shared__ uint32_t lds[];  // table [E][waves], start [E], padded [E + 1], scan scratch [waves]
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const int words = E * kSmallWaves;
  uint32_t *table = lds, *start = lds + words, *padded = start + E, *tmp = padded + E + 1;
  // a wave's ids are neighbours and the waves are in order, so that the flattened table, scanned, is a stable sort's first
  // destination of every (id, wave)
  const int per_wave = (R + kSmallBlock - 1) / kSmallBlock * kWave;
  int id[kSmallPer];
#pragma unroll
  for (int u = 0; u < kSmallPer; ++u) {
    const int i = wave * per_wave + u * kWave + lane;
    id[u] = u * kWave < per_wave && i < R ? load_id(ids + i) : -1;
  }
  for (int i = t; i < words; i += kSmallBlock) table[i] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSmallPer; ++u)
    if ((unsigned)id[u] < (unsigned)E) atomicAdd(&table[id[u] * kSmallWaves + wave], 1u);
  __syncthreads();
  const uint32_t total = block_exclusive_scan<kSmallBlock>(table, words, tmp);
  for (int e = t; e < E; e += kSmallBlock) {
    const uint32_t s = table[e * kSmallWaves], nxt = e + 1 < E ? table[(e + 1) * kSmallWaves] : total;
    start[e] = s;
    counts[e] = nxt - s;
    starts[e] = s;
    ends[e] = nxt;
    padded[e] = (nxt - s + (uint32_t)align - 1) / (uint32_t)align * (uint32_t)align;
  }
  __syncthreads();
  const uint32_t padded_total = block_exclusive_scan<kSmallBlock>(padded, E, tmp);
  if (t == 0) padded[E] = padded_total;
  __syncthreads();
  for (int e = t; e <= E; e += kSmallBlock) seg_starts[e] = (int32_t)padded[e];
  write_tile_experts(padded, E, padded_total, align, max_tiles, tile_expert, t, kSmallBlock);
  const uint64_t lanes_below = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
#pragma unroll
  for (int u = 0; u < kSmallPer; ++u) {
    if (u * kWave >= per_wave) break;
    const bool valid = (unsigned)id[u] < (unsigned)E;
    const uint64_t peers = lanes_with_same_id(id[u], valid, id_bits);
    if (valid) {
      uint32_t* next = &table[id[u] * kSmallWaves + wave];  // this wave's word alone; its LDS operations keep their order
      const uint32_t pos = *next + (uint32_t)__popcll(peers & lanes_below);
      if ((peers >> lane) == 1ull) *next = pos + 1;  // the highest lane of the group advances the bin
      const int i = wave * per_wave + u * kWave + lane;
      sorted_expert_idxs[pos] = id[u];
      sorted_scattered_idxs[pos] = i;
      row_slot[padded[id[u]] + (pos - start[id[u]])] = i;
    }
  }
}

}  // namespace
}  // namespace ck

using namespace ck;

// global accumulators that the workspace holds beside one word: as many as fit in 16384 words, at most 32
static int count_replicas(int num_bins) {
  int r = kMaxCountBins / (num_bins > 0 ? num_bins : 1);
  return r < 1 ? 1 : (r > 32 ? 32 : r);
}

namespace {
constexpr int kNarrowCount = 512, kWideCount = 1024;  // threads of a block
constexpr int64_t kMaxCountBlocks = 512;

// Half of the accumulators' words are enough for as many blocks as there are; the tickets of up to 16 groups take what they
// need of the rest, where there is room for two groups or more.
CountLayout count_layout(int num_bins) {
  const int replicas = count_replicas(num_bins), half = replicas / 2;
  const int groups = half >= 1 ? min(16, (1 + num_bins * (replicas - half)) / kTicketWords - 1) : 0;
  if (groups < 2) return {replicas, 0, 1};
  return {half, groups, (1 + groups) * kTicketWords};
}
}  // namespace

extern "C" int64_t ck_count_workspace_words(int32_t num_bins) {
  return 1 + (int64_t)(num_bins > 0 ? num_bins : 0) * count_replicas(num_bins);
}

namespace ck {
namespace {

// Validates the arguments and launches count_kernel on `workspace` (zero on entry, zero again on exit).
int launch_count(const char* name, const void* ids, int32_t ids_are_i64, int64_t n, int32_t num_bins, uint32_t* counts,
                 uint32_t* ends, uint32_t* starts, uint32_t* workspace, hipStream_t s) {
  CK_REQUIRE(num_bins >= 1 && num_bins <= kMaxCountBins, "%s: num_bins=%d outside [1, %d]", name, num_bins, kMaxCountBins);
  CK_REQUIRE(n >= 0, "%s: n=%lld is negative", name, (long long)n);
  CK_REQUIRE(counts != nullptr && workspace != nullptr, "%s: counts and workspace are required", name);
  CK_REQUIRE(n == 0 || ids != nullptr, "%s: ids is NULL", name);
  const size_t esz = ids_are_i64 ? 8 : 4;
  CK_REQUIRE((reinterpret_cast<uintptr_t>(ids) & (esz - 1)) == 0, "%s: ids is not element-aligned", name);

  const int64_t vec = 16 / (int64_t)esz;
  // up to 8 bins: ballot counters in registers (LDS atomics on so few addresses serialise); more bins: LDS atomics (16 register
  // counters measured half as fast)
  const int reg_bins = num_bins <= 8 ? 8 : 0;
  // A thread starts with 4 vectors (64 bytes) and goes round only once the launch is as large as the chip takes at once:
  // 512 blocks of 16 waves. Figures are us a launch, with all three outputs, in a captured graph of 50 of them. With 4 trips from
  // the start and at most 512 blocks of 4 waves, int32 / int64 ids over 64 experts, now / then: 65,536 ids 5.7 / 6.5 and 6.4 / 8.1,
  // 2^20 6.8 / 9.6 and 6.7 / 11.5, 2^22 7.1 / 12.1 and 8.5 / 16.3, 2^26 45.5 / 50.0 and 80.7 / 161.8 (a wave's wait for its additions
  // ahead of the ticket is 0.3 to 0.4 of each). Small inputs want blocks of 8 waves, whose barriers and merge are shorter (1,024
  // ids over 64 experts 3.1 against 3.7), as long as that makes few blocks -- up to 16, or 512 where a block's merge is short
  // (32 bins or fewer: 2^20 int32 ids over 16 experts 6.5 against 7.6; over 64 and 128 the two are within 10 % of each other up
  // to there, over 512 11.5 against 9.8). What two of them would share fits one wide block, which merges nothing: 16,384
  // int32 ids over 64 / 2,048 / 16,384 bins 4.5 / 4.8 / 18.5 against 5.3 / 10.2 / 49.4.
  const int64_t narrow = ceil_div(n, (int64_t)kNarrowCount * vec * 4);
  const bool wide = narrow == kWideCount / kNarrowCount || narrow > (num_bins <= 32 ? 512 : 16);
  const int threads = wide ? kWideCount : kNarrowCount;
  int64_t blocks = wide ? ceil_div(n, (int64_t)kWideCount * vec * 4) : narrow;
  blocks = blocks < 1 ? 1 : blocks > kMaxCountBlocks ? kMaxCountBlocks : blocks;
  // copies of the histogram in LDS: one a wave up to 1,024 bins, at most 32 KiB of them; beyond, waves seldom meet in a bin, and
  // clearing and adding up copies costs more than it saves (1,024 ids over 4,096 bins 6.1 with one, 7.6 with two; 2^20 11.8
  // and 12.3)
  int copies = reg_bins > 0 || num_bins > 1024 ? 1 : kMaxCountBins / 2 / num_bins;
  copies = copies > threads / kWave ? threads / kWave : copies;
  const size_t lds_bytes = ((size_t)copies * num_bins + threads / kWave + 2) * sizeof(uint32_t);
  const CountLayout layout = count_layout(num_bins);
#define CK_LAUNCH_COUNT_W(ID_T, RB, THREADS)                                                                              \
  hipLaunchKernelGGL((count_kernel<ID_T, RB, THREADS>), dim3((unsigned)blocks), dim3(THREADS), lds_bytes, s,             \
                     static_cast<const ID_T*>(ids), n, (int)num_bins, copies, layout, counts, ends, starts, workspace)
#define CK_LAUNCH_COUNT(ID_T, RB)                          \
  do {                                                     \
    if (wide) CK_LAUNCH_COUNT_W(ID_T, RB, kWideCount);     \
    else CK_LAUNCH_COUNT_W(ID_T, RB, kNarrowCount);        \
  } while (0)
  if (ids_are_i64) {
    if (reg_bins == 8) CK_LAUNCH_COUNT(int64_t, 8);
    else CK_LAUNCH_COUNT(int64_t, 0);
  } else {
    if (reg_bins == 8) CK_LAUNCH_COUNT(int32_t, 8);
    else CK_LAUNCH_COUNT(int32_t, 0);
  }
#undef CK_LAUNCH_COUNT
#undef CK_LAUNCH_COUNT_W
  CK_CHECK_LAUNCH(name);
  return CK_OK;
}

// ---- the entry point that allocates nothing ---------------------------------------------------------------------
// The count kernel's workspace (ticket + replicated global accumulators: at most 1 + 16384 words) lives in this
// file-scope device array instead of a caller's buffer. Every GPU holds its own copy at its own address until the
// process ends. In host code the array's name is only a handle for hipGetSymbolAddress: the address a kernel may use is
// looked up once per device, with that device current, and kept in g_scratch_ptr.
constexpr int kScratchWords = 1 + kMaxCountBins;
static __device__ __align__(256) uint32_t scratch[kScratchWords];

constexpr int kMaxScratchDevices = 64;
uint32_t* g_scratch_ptr[kMaxScratchDevices] = {};

int scratch_for_current_device(const char* name, uint32_t** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxScratchDevices) {
    set_error("%s: cannot tell the current device (%s, device %d)", name, hipGetErrorString(e), dev);
    return CK_ERR_LAUNCH;
  }
  uint32_t* p = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (p == nullptr) {  // first call on this device; a race between host threads only repeats the same lookup
    void* sym = nullptr;
    e = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));
    if (e != hipSuccess || sym == nullptr) {
      set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", name, dev, hipGetErrorString(e));
      return CK_ERR_LAUNCH;
    }
    p = static_cast<uint32_t*>(sym);
    __atomic_store_n(&g_scratch_ptr[dev], p, __ATOMIC_RELEASE);
  }
  *out = p;
  return CK_OK;
}

__global__ __launch_bounds__(kBlock) void zero_words_kernel(uint32_t* __restrict__ p, int words) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < words) p[i] = 0u;
}

}  // namespace
}  // namespace ck

extern "C" int ck_count_offsets(const void* ids, int32_t ids_are_i64, int64_t n, int32_t num_bins, uint32_t* counts,
                                uint32_t* ends, uint32_t* starts, uint32_t* workspace, void* stream) {
  return launch_count("ck_count_offsets", ids, ids_are_i64, n, num_bins, counts, ends, starts, workspace,
                      static_cast<hipStream_t>(stream));
}

extern "C" int ck_count_offsets_static(const void* ids, int32_t ids_are_i64, int64_t n, int32_t num_bins, uint32_t* counts,
                                       uint32_t* ends, uint32_t* starts, void* stream) {
  const char* name = "ck_count_offsets_static";
  CK_REQUIRE(num_bins >= 1 && num_bins <= kMaxCountBins,
             "%s: num_bins=%d outside [1, %d] (the built-in workspace holds %d words)", name, num_bins, kMaxCountBins,
             kScratchWords);
  const int64_t words = ck_count_workspace_words(num_bins);
  CK_REQUIRE(words <= kScratchWords, "%s: num_bins=%d needs %lld workspace words, the built-in workspace holds %d", name,
             num_bins, (long long)words, kScratchWords);
  uint32_t* ws = nullptr;
  if (int rc = scratch_for_current_device(name, &ws)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // The array keeps whatever the last call on this GPU left (zeros after a completed call, anything after one that was
  // cut short): the words this call uses are cleared first, by a kernel, so that the sequence can be captured in a graph.
  hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)ceil_div(words, kBlock)), dim3(kBlock), 0, s, ws, (int)words);
  CK_CHECK_LAUNCH(name);
  return launch_count(name, ids, ids_are_i64, n, num_bins, counts, ends, starts, ws, s);
}

// The padded grouped layout from a sort somebody else did (torch.sort + bincount + cumsum in the reference's own layer):
// every block derives the tile-aligned segment starts from the inclusive offsets (E is small), block 0 writes the tables,
// and every sorted position p of expert e goes to padded row seg_starts[e] + (p - starts[e]).
template <typename id_t, typename off_t>
__global__ __launch_bounds__(kBlock) void segments_from_sorted_kernel(
    const id_t* __restrict__ sorted_expert_idxs, const id_t* __restrict__ sorted_scattered_idxs,
    const off_t* __restrict__ ends, int64_t R, int E, int align, int64_t max_tiles, uint32_t* __restrict__ counts,
    int32_t* __restrict__ seg_starts, int32_t* __restrict__ row_slot, int32_t* __restrict__ row_pos,
    int32_t* __restrict__ tile_expert) {
  extern __shared__ uint32_t lds[];  // padded[E + 1], starts[E], count[E], scan scratch
  uint32_t* padded = lds;
  uint32_t* first = lds + E + 1;
  uint32_t* count = first + E;
  uint32_t* tmp = count + E;
  const int t = threadIdx.x;
  for (int e = t; e < E; e += kBlock) {
    const uint32_t end = (uint32_t)ends[e], begin = e > 0 ? (uint32_t)ends[e - 1] : 0u;
    const uint32_t c = end >= begin ? end - begin : 0u;
    first[e] = begin;
    count[e] = c;
    padded[e] = (c + (uint32_t)align - 1) / (uint32_t)align * (uint32_t)align;
  }
  __syncthreads();
  const uint32_t padded_total = block_exclusive_scan(padded, E, tmp);
  if (t == 0) padded[E] = padded_total;
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int e = t; e < E; e += kBlock) counts[e] = count[e];
    for (int e = t; e <= E; e += kBlock) seg_starts[e] = (int32_t)padded[e];
    for (int64_t tile = t; tile < max_tiles; tile += kBlock) {
      const uint32_t row = (uint32_t)(tile * align);
      int32_t owner = -1;
      if (row < padded_total) {  // last e with padded[e] <= row (empty experts share a start with their successor)
        int lo = 0, hi = E - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (padded[mid] <= row) lo = mid; else hi = mid - 1;
        }
        owner = lo;
      }
      tile_expert[tile] = owner;
    }
  }
  for (int64_t p = (int64_t)blockIdx.x * kBlock + t; p < R; p += (int64_t)gridDim.x * kBlock) {
    const int e = load_id(sorted_expert_idxs + p);
    if ((unsigned)e >= (unsigned)E) continue;
    const int64_t j = p - (int64_t)first[e];
    if (j < 0 || j >= (int64_t)count[e]) continue;  // offsets that do not describe these ids: the row stays unowned
    const int64_t dst = (int64_t)padded[e] + j;
    row_slot[dst] = load_id(sorted_scattered_idxs + p);
    row_pos[dst] = (int32_t)p;
  }
}

extern "C" int ck_segments_from_sorted(const void* sorted_expert_idxs, const void* sorted_scattered_idxs,
                                       int32_t idxs_are_i64, const void* expert_offsets, int32_t offsets_are_i64,
                                       int64_t R, int32_t E, int32_t align, uint32_t* counts, int32_t* seg_starts,
                                       int32_t* row_slot, int32_t* row_pos, int32_t* tile_expert, void* stream) {
  const char* name = "ck_segments_from_sorted";
  CK_REQUIRE(E >= 1 && E <= kMaxSortBins, "%s: E=%d outside [1, %d]", name, E, kMaxSortBins);
  CK_REQUIRE(align >= 1, "%s: align=%d must be positive", name, align);
  CK_REQUIRE(R >= 0 && R < (int64_t)0x7fffffff - (int64_t)E * align, "%s: R=%lld out of range", name, (long long)R);
  CK_REQUIRE(expert_offsets && counts && seg_starts && row_slot && row_pos && tile_expert, "%s: NULL argument", name);
  CK_REQUIRE(R == 0 || (sorted_expert_idxs && sorted_scattered_idxs), "%s: NULL index tensor", name);
  const int64_t max_tiles = ck_sort_max_rows(R, E, align) / align;
  int64_t blocks = ceil_div(R > 0 ? R : 1, (int64_t)kBlock * 4);
  if (blocks > 1024) blocks = 1024;
  const size_t lds_bytes = ((size_t)3 * E + 1 + kWavesPerBlock) * sizeof(uint32_t);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CK_LAUNCH_SEGMENTS(ID_T, OFF_T)                                                                               \
  hipLaunchKernelGGL((segments_from_sorted_kernel<ID_T, OFF_T>), dim3((unsigned)blocks), dim3(kBlock), lds_bytes, s, \
                     static_cast<const ID_T*>(sorted_expert_idxs), static_cast<const ID_T*>(sorted_scattered_idxs),   \
                     static_cast<const OFF_T*>(expert_offsets), R, (int)E, (int)align, max_tiles, counts, seg_starts, \
                     row_slot, row_pos, tile_expert)
  if (idxs_are_i64) {
    if (offsets_are_i64) CK_LAUNCH_SEGMENTS(int64_t, int64_t);
    else CK_LAUNCH_SEGMENTS(int64_t, int32_t);
  } else {
    if (offsets_are_i64) CK_LAUNCH_SEGMENTS(int32_t, int64_t);
    else CK_LAUNCH_SEGMENTS(int32_t, int32_t);
  }
#undef CK_LAUNCH_SEGMENTS
  CK_CHECK_LAUNCH(name);
  return CK_OK;
}

extern "C" int64_t ck_sort_max_rows(int64_t R, int32_t E, int32_t align) {
  if (R < 0 || E < 1 || align < 1) return 0;
  // sum_e round_up(c_e, align) <= R + E * (align - 1); round to whole tiles
  return round_up(R + (int64_t)E * (align - 1), align);
}

extern "C" int64_t ck_sort_workspace_words(int64_t R, int32_t E) {
  if (E < 1) return 1;
  const SortPlan p = make_sort_plan(R, E);
  return 1 + (int64_t)E * p.blocks;
}

extern "C" int ck_sort_by_expert(const void* expert_ids, int32_t ids_are_i64, int64_t R, int32_t E, int32_t align,
                                 int32_t* sorted_expert_idxs, int32_t* sorted_scattered_idxs, uint32_t* counts,
                                 uint32_t* ends, uint32_t* starts, int32_t* seg_starts, int32_t* row_slot,
                                 int32_t* tile_expert, uint32_t* workspace, void* stream) {
  CK_REQUIRE(E >= 1 && E <= kMaxSortBins, "ck_sort_by_expert: E=%d outside [1, %d]", E, kMaxSortBins);
  CK_REQUIRE(R >= 0 && R < (int64_t)0x7fffffff - (int64_t)E * align, "ck_sort_by_expert: R=%lld out of range",
             (long long)R);
  CK_REQUIRE(align >= 1, "ck_sort_by_expert: align=%d must be positive", align);
  CK_REQUIRE(R == 0 || expert_ids != nullptr, "ck_sort_by_expert: expert_ids is NULL");
  CK_REQUIRE(sorted_expert_idxs && sorted_scattered_idxs && counts && ends && starts && seg_starts && row_slot &&
                 tile_expert && workspace,
             "ck_sort_by_expert: every output and the workspace are required");
  const int64_t max_tiles = ck_sort_max_rows(R, E, align) / align;
  int id_bits = 0;
  while ((1 << id_bits) < E) ++id_bits;
#define CK_LAUNCH_LANES(ID_T, NB, SMALL, BLOCKS, SEG_LEN, TABLE)                                                              \
  hipLaunchKernelGGL((sort_lanes_kernel<ID_T, NB, SMALL>), dim3(BLOCKS), dim3(kLaneWaves * kWave), 0, static_cast<hipStream_t>(stream), \
                     static_cast<const ID_T*>(expert_ids), R, (int)E, (int64_t)(SEG_LEN), id_bits, (int)align, max_tiles, TABLE,         \
                     sorted_expert_idxs, sorted_scattered_idxs, counts, ends, starts, seg_starts, row_slot, tile_expert)
#define CK_LAUNCH_LANES_OF(ID_T, SMALL, BLOCKS, SEG_LEN, TABLE)                        \
  do {                                                                                 \
    if (E <= kWave) CK_LAUNCH_LANES(ID_T, 1, SMALL, BLOCKS, SEG_LEN, TABLE);           \
    else CK_LAUNCH_LANES(ID_T, 2, SMALL, BLOCKS, SEG_LEN, TABLE);                      \
  } while (0)
  if (R <= kLaneIds && E <= kLaneBins) {
    const int64_t seg_len = round_up(R > 0 ? R : 1, (int64_t)kLaneWaves * kWave);
    const uint32_t* none = nullptr;
    if (ids_are_i64) CK_LAUNCH_LANES_OF(int64_t, true, 1, seg_len, none);
    else CK_LAUNCH_LANES_OF(int32_t, true, 1, seg_len, none);
    CK_CHECK_LAUNCH("ck_sort_by_expert");
    return CK_OK;
  }
  if (E <= kSmallBins && R <= small_ids(E)) {
    const size_t lds = ((size_t)E * (kSmallWaves + 2) + 1 + kSmallWaves) * sizeof(uint32_t);
#define CK_LAUNCH_SMALL(ID_T)                                                                                                \
  hipLaunchKernelGGL((sort_small_kernel<ID_T>), dim3(1), dim3(kSmallBlock), lds, static_cast<hipStream_t>(stream),           \
                     static_cast<const ID_T*>(expert_ids), (int)R, (int)E, (int)align, max_tiles, id_bits, sorted_expert_idxs, \
                     sorted_scattered_idxs, counts, ends, starts, seg_starts, row_slot, tile_expert)
    if (ids_are_i64) CK_LAUNCH_SMALL(int64_t);
    else CK_LAUNCH_SMALL(int32_t);
#undef CK_LAUNCH_SMALL
    CK_CHECK_LAUNCH("ck_sort_by_expert");
    return CK_OK;
  }
  const SortPlan p = make_sort_plan(R, E);
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint32_t* table = workspace + 1;  // word 0 is left alone
#define CK_LAUNCH_SORT(ID_T, WAVES)                                                                                            \
  do {                                                                                                                         \
    const ID_T* ids = static_cast<const ID_T*>(expert_ids);                                                                    \
    const size_t hist_words = (size_t)WAVES * E, words = (size_t)(WAVES + 4) * E + 1 + WAVES;                                  \
    hipLaunchKernelGGL((sort_hist_kernel<ID_T, WAVES>), dim3(p.blocks), dim3(WAVES * kWave), hist_words * sizeof(uint32_t), s, \
                       ids, R, (int)E, p.seg_len, table);                                                                      \
    if (E <= kLaneBins) {                                                                                                      \
      CK_LAUNCH_LANES_OF(ID_T, false, p.blocks, p.seg_len, table);                                                             \
      break;                                                                                                                   \
    }                                                                                                                          \
    hipLaunchKernelGGL((sort_scatter_kernel<ID_T, WAVES>), dim3(p.blocks), dim3(WAVES * kWave), words * sizeof(uint32_t), s,   \
                       ids, R, (int)E, p.seg_len, id_bits, (int)align, max_tiles, table, sorted_expert_idxs,                   \
                       sorted_scattered_idxs, counts, ends, starts, seg_starts, row_slot, tile_expert);                        \
  } while (0)
  if (E <= kSmallBins) {
    if (ids_are_i64) CK_LAUNCH_SORT(int64_t, kWideWaves);
    else CK_LAUNCH_SORT(int32_t, kWideWaves);
  } else {
    if (ids_are_i64) CK_LAUNCH_SORT(int64_t, kNarrowWaves);
    else CK_LAUNCH_SORT(int32_t, kNarrowWaves);
  }
#undef CK_LAUNCH_SORT
#undef CK_LAUNCH_LANES_OF
#undef CK_LAUNCH_LANES
  CK_CHECK_LAUNCH("ck_sort_by_expert");
  return CK_OK;
}
