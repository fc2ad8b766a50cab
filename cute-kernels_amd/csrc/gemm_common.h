// Pieces shared by the grouped GEMM kernels (bf16 / f16 in grouped_gemm.hip, fp8 e4m3 in grouped_gemm_fp8.hip).
#pragma once

#include <type_traits>

#include "ck_common.h"

namespace ck {

constexpr int kXcds = 8;

enum Mode { kGrouped = CK_EPI_GROUPED, kScatter = CK_EPI_SCATTER, kSwiglu = CK_EPI_SWIGLU, kSwigluBwd = CK_EPI_SWIGLU_BWD, kDw = 4 };

struct GemmParams {
  const void* a;      // forward modes: [*, K]; dW: a_t [M, ld_t]
  const void* w;      // forward modes: [E, N, K]; dW: b_t [N, ld_t]
  int64_t lda;        // row stride of a (elements)
  int64_t ldw;        // row stride of w (elements)
  int64_t w_expert_stride;
  int a_gather_div;   // > 0: A row p comes from a[row_slot[p] / div]
  int M;              // dW only: rows of a_t
  int N;              // output columns of the GEMM (2I for kSwiglu)
  int K;              // contraction length (forward modes)
  int I;              // kSwiglu / kSwigluBwd: intermediate size
  int n_tiles;        // tiles along N
  int m_tiles;        // dW only: tiles along M
  int align;          // rows per M tile (== BM) in the padded layout
  int num_experts;
  const int32_t* seg_starts;
  const uint32_t* counts;
  const int32_t* tile_expert;
  const int32_t* row_slot;      // padded row -> index of the A row it reads (gathered input)
  const int32_t* row_slot_out;  // padded row -> output row of the scatter epilogue (ck_segments::row_slot_out, else row_slot)
  void* y;
  void* y_t;
  int64_t ld_t;
  void* aux;
  const void* aux_in;
  const float* a_scale;  // fp8 only: per-row dequantisation scale of a (indexed like the rows of a)
  const float* w_scale;  // fp8 only: per-output-channel scale of w, [E, N]
  int act_kind;          // kSwiglu epilogue: CK_ACT_SWIGLU (up * gate * sigmoid(gate)) or CK_ACT_GLU (up * sigmoid(gate));
                         // kGrouped epilogue with aux: CK_ACT_GELU_TANH (aux = gelu(y), second output)
  void* trace;           // measurement builds only (CK_STAMP): per-wave cycle counts, 8 x uint64 each, else NULL
  // Split contraction for the last, partial round of tiles (128-byte-row kernel, all forward epilogues):
  // split_ws = [tiles][parts][4 waves][64 blocks][64 lanes] f32x4 partial accumulators (at most kSplitMaxTail tiles in
  // kSplitParts parts or twice as many in half as many parts), followed by 2 * kSplitMaxTail 64-bit arrival words; NULL =
  // never split. split_base = the launch's grid without the extra workgroups (they are blockIdx split_base ..).
  // An arrival word holds (launch tag << 4) | parts arrived. A part that finds another tag in the word starts the
  // count afresh, so the words need no initial value: whatever another launch, one that was cut short or the memory's former
  // owner left behind reads as "nobody has arrived yet". The last part to arrive puts the word to 0 (no launch's tag): a
  // launch in a captured graph has the same tag in every replay. split_tag: 60 bits, never 0.
  float* split_ws;
  int split_base;
  uint64_t split_tag;
};
uint64_t next_split_tag();  // grouped_gemm.hip
constexpr int kSplitParts = 4, kSplitMaxTail = 64, kSplitMaxRounds = 64;
// K steps that splitting has to take off the last round. A step of a 256 x 256 tile takes 1.5 to 1.7 us with all CUs at work and 1.1
// to 1.3 with few (the chip's power is shared by fewer), and the exchange of the parts' accumulators 25 to 40 us: launches of 24 and
// 32 steps that save 16 to 24 of them gain nothing (-5 to 0 us), of 64 that save 48 gain 14 to 16, of 128 that save 64 gain 37, of
// 224 that save 168 gain 160.
constexpr int kSplitMinSaved = 40;
constexpr bool split_pays(int k_steps, int parts) { return k_steps - (k_steps + parts - 1) / parts >= kSplitMinSaved; }
constexpr int64_t kSplitPartFloats = 4 * 64 * 64 * 4;  // one workgroup's 256 x 256 fp32 tile
constexpr int64_t kSplitWorkspaceBytes = kSplitMaxTail * kSplitParts * kSplitPartFloats * 4 + 2 * kSplitMaxTail * 8;

// The 16-bit kernel with 128-byte LDS rows (grouped_gemm_line.hip): 256 x bn tiles, bn = 256 or 384, contraction length a
// multiple of 64, modes kGrouped, kScatter, kSwiglu, kDw. The caller fills `prm` for these tile dimensions (n_tiles,
// m_tiles) and sizes the grid accordingly.
constexpr int kLineBM = 256, kLineK = 64;
// bt: the weight operand is [E, contraction, columns] (contraction-strided) instead of [E, columns, contraction];
// grouped and scatter epilogues only, prm.ldw = its row length.
int launch_line(const GemmParams& prm, int mode, int bn, bool bt, int dtype, unsigned blocks, hipStream_t stream,
                const char* name);

// Weight gradients from row-major operands on 128 x 256 tiles, two workgroups per compute unit (grouped_gemm_dw.hip); sets
// prm's tile counts itself.
int launch_dw_short(const GemmParams& prm, int dtype, hipStream_t stream, const char* name);

// Tiles of 16, 32 or 64 rows (grouped_gemm_skinny.hip): forward GEMMs of inference batches with few rows per expert, modes
// kGrouped, kScatter, kSwiglu, 16-bit or e4m3 operands; prm.align is the tile height.
inline bool skinny_align(int align) { return align == 16 || align == 32 || align == 64; }
int launch_skinny(const GemmParams& prm, int mode, int64_t max_rows, bool fp8, int dtype, hipStream_t stream, const char* name);

namespace {

// The dynamic-LDS limit of a kernel is a per-device attribute: set it once per (instantiation, device). `done` is the
// instantiation's own table; the call is idempotent, so a race between host threads only repeats it.
constexpr int kMaxDevices = 64;
inline int reserve_lds(const void* kernel, size_t bytes, bool (&done)[kMaxDevices], const char* name) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = -1;
  if (dev >= 0 && done[dev]) return CK_OK;
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess) {
    set_error("%s: cannot reserve %zu bytes of LDS: %s", name, bytes, hipGetErrorString(e));
    return CK_ERR_LAUNCH;
  }
  if (dev >= 0) done[dev] = true;
  return CK_OK;
}

template <typename T>
struct Mfma;
template <>
struct Mfma<bf16_t> {
  typedef bf16x8 frag;
  __device__ static inline f32x16 run(const frag& a, const frag& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<f16_t> {
  typedef f16x8 frag;
  __device__ static inline f32x16 run(const frag& a, const frag& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// v_mfma_f32_16x16x32: A lane l holds row l % 16, contraction values 8 (l / 16) .. + 7; B likewise for column l % 16; the
// result register s of lane l is row 4 (l / 16) + s, column l % 16. On N(0,1) operands a register-only loop of this
// shape sustains about 2.0 PFLOP/s where the 32x32x16 shape sustains 1.7 (the clock is power-managed), hence its use in
// the 128-byte-row kernel.
template <typename T>
struct Mfma16;
// run_acc: the same instruction with the accumulator pinned to the accumulation registers (AGPRs) and updated in place.
// With one wave per SIMD a kernel has 256 of them next to its 256 vector registers; left to choose, the register
// allocator spreads 256 accumulator values over both files and shuffles them at every loop boundary. The instruction is
// opaque to the compiler's hazard checks: a caller that reads the accumulators with vector instructions afterwards
// waits out the MFMA write latency itself (mfma_drain).
template <>
struct Mfma16<bf16_t> {
  typedef bf16x8 frag;
  __device__ static inline f32x4 run(const frag& a, const frag& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static inline void run_acc(const frag& a, const frag& b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  // the first product of a tile: c = a * b + 0 (the constant as the third operand), so that nothing has to zero the
  // accumulators first -- 256 v_accvgpr_write per wave, which the compiler also re-materialised in front of the loop
  __device__ static inline void run_acc_first(const frag& a, const frag& b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
};
template <>
struct Mfma16<f16_t> {
  typedef f16x8 frag;
  __device__ static inline f32x4 run(const frag& a, const frag& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  __device__ static inline void run_acc(const frag& a, const frag& b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  __device__ static inline void run_acc_first(const frag& a, const frag& b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
};
// The lane's number, counted anew: what an epilogue derives from it needs no register while the products are under way.
__device__ inline int lane_again() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// After the last run_acc, before anything else reads the accumulators: longer than any MFMA's result latency. The wait
// alone is not enough: nothing ties the compiler's own reads of the accumulators (v_accvgpr_read, spills) to it, and the
// scheduler is free to hoist them above the wait, right behind the MFMA that writes them (it did: a few stale values
// per tile). mfma_fence(c) makes c a result of an empty asm statement placed behind the wait; volatile asm statements
// keep their order, so every later read of c stays behind the wait. Call it for every accumulator.
__device__ inline void mfma_drain() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }
__device__ inline void mfma_fence(f32x4& c) { asm volatile("" : "+a"(c)); }

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): a loop whose index is a constant expression
template <int N, typename F>
__device__ inline void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

template <typename T>
__device__ inline uint16_t bits16(T v) {
  union {
    T t;
    uint16_t u;
  } c;
  c.t = v;
  return c.u;
}

// two fp32 values rounded (to nearest even) and packed into one register: one v_cvt_pk instruction
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2_t;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 f16x2_t;
template <typename T>
__device__ inline uint32_t pack_pair(float a, float b);
template <>
__device__ inline uint32_t pack_pair<bf16_t>(float a, float b) {
  const f32x2_t v = {a, b};
  union {
    bf16x2_t h;
    uint32_t u;
  } c;
  c.h = __builtin_convertvector(v, bf16x2_t);
  return c.u;
}
template <>
__device__ inline uint32_t pack_pair<f16_t>(float a, float b) {
  const f32x2_t v = {a, b};
  union {
    f16x2_t h;
    uint32_t u;
  } c;
  c.h = __builtin_convertvector(v, f16x2_t);
  return c.u;
}

// 4 consecutive 16-bit values as one 8-byte store
template <typename T>
__device__ inline void store4(T* p, T v0, T v1, T v2, T v3) {
  uint2 u;
  u.x = (uint32_t)bits16(v0) | ((uint32_t)bits16(v1) << 16);
  u.y = (uint32_t)bits16(v2) | ((uint32_t)bits16(v3) << 16);
  *reinterpret_cast<uint2*>(p) = u;
}

// Tile order inside a run of tiles: groups of at most 8 along `a` (the side with a_count tiles), then `b`, with `a` fastest
// inside a group -- 32 consecutive tiles form an 8 x 4 block that shares 8 + 4 operand panels.
// (measured at 4 / 8 / 16 / 32 tiles per group on the Mixtral-shape and fine-grained layers: 8 is fastest on both)
// The groups are of even height (9 tiles are 5 + 4): a last group of one tile would share 1 + 32 panels.
template <int GROUP = 8>
__device__ inline void grouped_order(int r, int a_count, int b_count, int& a, int& b) {
  const int groups = (a_count + GROUP - 1) / GROUP;
  const int low = a_count / groups, taller = a_count - low * groups;  // `taller` groups of low + 1, then groups of low
  const int taller_tiles = taller * (low + 1) * b_count;
  int height = low, first = taller * (low + 1), q = r - taller_tiles;
  if (q < 0) {
    height = low + 1;
    first = 0;
    q = r;
  }
  const int group_sz = height * b_count;
  const int g = q / group_sz;
  q -= g * group_sz;
  b = q / height;
  a = first + g * height + (q - b * height);
}

// Tile `pid` of a forward launch's (m tiles x n_tiles) live tiles. Each XCD takes a contiguous run of them (workgroups are
// dealt round-robin to the XCDs; the ragged end keeps its order), and the run goes expert by expert, each in groups
// of its own m tiles: the 32 tiles an XCD computes at a time read one expert's weights where groups over all m tiles read
// those of every expert the 8 m tiles belong to (4 tiles per expert: 4 + 8 operand panels against 8 + 8). 64 experts of
// 2,048 x 1,408 at 1,024 rows each: 357 -> 346 us; 16 of 14,336 x 4,096: 1,557 -> 1,518, input gradients 1,537 -> 1,497.
// ACROSS (the general kernel, whose tiles are mostly 128 rows): with fewer than two m tiles per expert there is nothing to share,
// and the groups, of 8 and a rest, go over all m tiles. Over 67 such launches expert by expert is 2 % faster on average, but
// which XCD gets which tiles is luck then, and a few lose much: 16 experts of 5,088 x 3,552 with Zipf(1.0) loads at 12 / 13 rows
// 147 / 137 us across, 170 / 168 expert by expert.
template <bool ACROSS = false>
__device__ inline void forward_tile(const GemmParams& prm, int pid, int total, int& mt, int& nt, int& expert) {
  const int per_xcd = total / kXcds;
  if (pid < per_xcd * kXcds) pid = (pid % kXcds) * per_xcd + pid / kXcds;
  if constexpr (ACROSS) {
    const int live_m = total / prm.n_tiles;
    if (live_m < 2 * prm.num_experts) {
      const int g = pid / (8 * prm.n_tiles), height = min(8, live_m - 8 * g);
      nt = (pid - g * 8 * prm.n_tiles) / height;
      mt = 8 * g + pid - g * 8 * prm.n_tiles - nt * height;
      expert = prm.tile_expert[mt];
      return;
    }
  }
  expert = prm.tile_expert[pid / prm.n_tiles];  // an expert's tiles are consecutive: n_tiles for each of its m tiles
  const int first = prm.seg_starts[expert] / prm.align, end = prm.seg_starts[expert + 1] / prm.align;
  grouped_order(pid - first * prm.n_tiles, end - first, prm.n_tiles, mt, nt);
  mt += first;
}

// Tile `pid` of a weight-gradient launch: `position` of its expert in the launch's order of experts, and its place in that
// expert's m_tiles x n_tiles grid. Experts differ in contraction length, and which XCD computes a workgroup is fixed by its
// index, so every XCD has to get its share of every length.
// Slices: every expert's grid is cut in 8 along its longer side, which makes the shares equal.
// Chunks: runs of consecutive tiles (blocks of one expert's) go out over the XCDs and back; the experts are sorted by length,
// so that turning back evens the shares out, unless experts end in the middle of a round of the XCDs and have few rounds:
// half of the XCDs then get a chunk more of the longest expert than the others.
// Which of the two, by the slice's tiles along the longer side:
//   none (no multiple of 8) or 1: chunks of 16, 4 x 4 blocks (8 + 8 operand panels for the 32 tiles an XCD computes at a time);
//     slices would leave an XCD one row of an expert's tiles, or every eighth tile: 36 panels for 32 tiles of 11 x 8 per
//     expert. 64 experts of 2,816 x 2,048 at 400 / 1,024 / 2,048 rows each: 496 / 806 / 1,398 us -> 481 / 777 / 1,329, with
//     Zipf(0.8) loads 484 / 860 / 1,462 -> 457 / 820 / 1,393. Chunks of 8 and 12 were slower, chunks of 32 (8 x 4) 1 % faster at
//     even loads and 5 to 10 % slower at Zipf(0.8): too few of them to even out. At 8 x 6 tiles per expert (3 rounds of half
//     the XCDs) chunks are 4 to 5 % faster than slices at even loads, and at 600 / 1,500 rows with Zipf(0.8) 4 / 2 % faster,
//     with Zipf(1.0) equal / 3 % slower, with Zipf(1.2) 6 % slower / 3 % faster; at 6,144 rows 5 to 9 % slower at Zipf(1.0).
//   2 or 3: the same chunks where they deal the experts evenly or below 2,048 rows per expert. 64 of 4,096 x 2,048 (one whole
//     round) 1 to 2 % faster than slices at every load from Zipf(0) to Zipf(1.2); 128 of 3,072 x 4,096 (1.5 rounds) at 1,024 rows
//     3.5 % faster up to Zipf(1.0), at 1,500 rows with Zipf(0) / (0.8) / (1.0) / (1.2) 3 % faster, equal, 3 and 4 % slower, at
//     4,096 rows 10,211 / 10,484 / 10,592 / 10,759 us in slices and 10,262 / 10,830 / 11,100 / 11,469 in chunks.
//   4 or more (4 + 8 panels in slices): chunks of 32 from 4,096 rows per expert on, where they deal the experts evenly. All XCDs
//     together then read 16 + 16 panels where slices read 64 + 4, and the contraction is long enough for that to count.
//     8 experts of 28,672 x 4,096, slices / chunks at 1,024, 2,048, 3,072, 4,096, 6,144 rows each: 1,801 / 1,881, 3,234 / 3,300,
//     4,655 / 4,702, 6,126 / 6,093, 9,073 / 8,990 us; Zipf(1.0) 1,847 / 1,922, 3,303 / 3,291, 4,800 / 4,724, 6,299 / 6,176, 9,160 /
//     9,105. 64 of 8,192 x 3,072 (1.5 rounds) at 4,096 rows with the four loads 10,005 / 10,319 / 10,369 / 10,474 in slices and
//     9,878 / 10,412 / 10,667 / 11,003 in chunks; 32 of 10,240 x 4,096 (2.5 rounds) equal within 1 %; 16 of 14,336 x 4,096 (3.5
//     rounds) 1.5 to 3 % faster in chunks.
template <int CHUNK, int HEIGHT>
__device__ inline void dw_chunk_tile(int pid, int major, int minor, int num_experts, int& position, int& a, int& b) {
  const int per_expert = major * minor, total = per_expert * num_experts;
  if (pid < total / (kXcds * CHUNK) * (kXcds * CHUNK)) {  // the last, partial round keeps its order
    const int xcd = pid % kXcds, j = pid / kXcds, round = j / CHUNK;
    pid = (round * kXcds + ((round & 1) ? kXcds - 1 - xcd : xcd)) * CHUNK + j % CHUNK;
  }
  position = pid / per_expert;
  grouped_order<HEIGHT>(pid - position * per_expert, major, minor, a, b);
}
__device__ inline void dw_tile(const GemmParams& prm, int pid, int& position, int& mt, int& nt) {
  const bool m_major = prm.m_tiles >= prm.n_tiles;
  const int major = m_major ? prm.m_tiles : prm.n_tiles, minor = m_major ? prm.n_tiles : prm.m_tiles;
  int a, b;
  const int per_expert = major * minor, slice = major % kXcds == 0 ? major / kXcds : 0;
  const int rows = prm.seg_starts[prm.num_experts] / prm.num_experts;  // of an expert, on average
  const auto even = [&](int chunk) { return per_expert % (kXcds * chunk) == 0 || per_expert >= 3 * kXcds * chunk; };
  if (slice < 2 || (slice < 4 && (rows < 2048 || even(16)))) {
    dw_chunk_tile<16, 4>(pid, major, minor, prm.num_experts, position, a, b);
  } else if (slice >= 4 && rows >= 4096 && even(32)) {
    dw_chunk_tile<32, 8>(pid, major, minor, prm.num_experts, position, a, b);
  } else {
    const int per_slice = slice * minor, j = pid / kXcds;
    position = j / per_slice;
    grouped_order(j - position * per_slice, slice, minor, a, b);
    a += pid % kXcds * slice;
  }
  mt = m_major ? a : b;
  nt = m_major ? b : a;
}
// The same for tiles of half the height (grouped_gemm_dw.hip; 64 at a time on an XCD): blocks of 8 m tiles x 4 n tiles.
__device__ inline void dw_rows_first_tile(const GemmParams& prm, int pid, int& position, int& mt, int& nt) {
  if (prm.m_tiles % kXcds == 0 && prm.m_tiles / kXcds >= 8) {
    const int slice = prm.m_tiles / kXcds, per_slice = slice * prm.n_tiles, j = pid / kXcds;
    position = j / per_slice;
    grouped_order(j - position * per_slice, slice, prm.n_tiles, mt, nt);
    mt += pid % kXcds * slice;
  } else {
    dw_chunk_tile<32, 8>(pid, prm.m_tiles, prm.n_tiles, prm.num_experts, position, mt, nt);
  }
}

// The expert with the position-th largest count, ties by index: the longest contractions go first (the hardware hands tiles
// out in block order), so that the tiles still running when the grid drains are the short ones. One thread ranks one
// expert against the counts parked in LDS (sh: THREADS + 1 words, free again on return); more experts than threads keep
// their order.
template <int THREADS>
__device__ inline int longest_first(const GemmParams& prm, int position, int* sh) {
  const int E = prm.num_experts, t = threadIdx.x;
  if (E > THREADS) return position;
  if (t < E) sh[t] = (int)prm.counts[t];
  __syncthreads();
  if (t < E) {
    const int c = sh[t];
    int rank = 0;
    for (int i = 0; i < E; ++i) {
      const int ci = sh[i];
      rank += (ci > c || (ci == c && i < t)) ? 1 : 0;
    }
    if (rank == position) sh[THREADS] = t;
  }
  __syncthreads();
  const int expert = sh[THREADS];
  __syncthreads();  // everyone holds its expert before the first loads land there
  return expert;
}


// XOR swizzle of the 64-byte LDS rows of the direct-to-LDS pipeline: 16-byte chunk c of row r sits in slot
// c ^ lds_swizzle(r). Found by exhaustive search: fragment reads (32 consecutive rows, same chunk) are free of bank
// conflicts both for 8 lanes over 32 banks and for 16 lanes over 64 banks.
__device__ inline int lds_swizzle(int row) { return ((row >> 2) & 1) | ((((row >> 1) ^ (row >> 3)) & 1) << 1); }

inline int check_segments(const ck_segments* seg, const char* name, bool small_tiles = false) {
  CK_REQUIRE(seg != nullptr, "%s: seg is NULL", name);
  CK_REQUIRE(seg->seg_starts && seg->counts && seg->tile_expert && seg->row_slot, "%s: NULL table in seg", name);
  CK_REQUIRE(seg->align == 128 || seg->align == 256 || (small_tiles && skinny_align(seg->align)), "%s: align=%d must be %s128 or 256",
             name, seg->align, small_tiles ? "16, 32, 64, " : "");
  CK_REQUIRE(seg->num_experts >= 1, "%s: num_experts=%d", name, seg->num_experts);
  CK_REQUIRE(seg->max_rows >= 0 && seg->max_rows % seg->align == 0, "%s: max_rows=%lld is not a multiple of align", name,
             (long long)seg->max_rows);
  return CK_OK;
}

}  // namespace
}  // namespace ck
