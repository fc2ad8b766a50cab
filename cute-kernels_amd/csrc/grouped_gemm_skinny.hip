// Grouped GEMM for few rows per expert (inference with small batches): 16-, 32- or 64-row tiles, bf16 / f16 or fp8 e4m3
// operands, fp32 accumulation.
//
// What bounds it: the stream of expert weights out of HBM. A decoding step reads nearly every expert's matrices for a
// handful of rows each, 2 to 64 multiply-adds per weight, far below what the matrix cores need to matter. So the kernel is
// built around the weight stream and nothing else:
//  * weights go straight from memory into MFMA operand registers: no LDS stage and no barrier in the main loop. A load
//    takes whole 128-byte lines, of 8 columns, and two loads become the two operands of a step by 8 moves between lanes
//    (to_operands); v_mfma_f32_16x16x32 takes 8 contraction values a lane and operand, v_mfma_f32_16x16x128_f8f6f4 both pieces
//    at once, 32 values. Because a line is used up by one load, the loads can be non-temporal, and memory then delivers more: bare
//    reads of 369 to 1,611 MB in this kernel's pattern 6.6 to 7.0 TB/s, of plain loads 5.9 to 6.2 whatever the pattern. With
//    half lines (16 columns a load) non-temporal loads fetch lines twice, 5 to 20 % slower, and so they do where a row's pitch or
//    the first row is off a 128-byte boundary: plain loads there (non-temporal 10 to 28 % slower at 200 MB and more);
//  * the four waves of a workgroup share the output tile and split the contraction, a quarter of every row each, in steps
//    of one 128-byte line per row; no weight is read twice. The four partial tiles meet once, in LDS, in front of the
//    epilogue (a fixed order of additions). Waves that take every fourth line instead measured equal in bf16 and 2 to 8 %
//    slower in fp8;
//  * a wave keeps the next step's loads in flight under the current step's MFMAs (two register sets); with 2 to 4
//    workgroups per CU that is 64 to 128 KiB of weights in flight per CU (eight waves per workgroup: 0 to 10 % slower,
//    128-column tiles: equal);
//  * the workgroups in flight read one stretch of memory, expert by expert (column tiles of all experts in turn: 2 to 6 %
//    slower);
//  * the activations, a few hundred KiB for the whole launch, are re-read by every column tile from L2.
// An expert with more rows than a tile has several tiles; they are neighbours in launch order on one XCD, so that the
// second reads the weights from that XCD's L2.
// Measured (kernel trace, all experts with as many rows; the rate is the weights' bytes by the time; before: plain loads of half lines,
// column tile by column tile): 8 experts of 28,672 x 4,096 with 2 rows each 308 -> 271 us = 6.9 TB/s, 4,096 x 14,336 163 -> 152 = 6.2,
// 64 of 2,816 x 2,048 with 8 rows 130 -> 116 = 6.4, 2,048 x 1,408 69 -> 58.5 = 6.3, e4m3, 128 of 3,072 x 4,096 with 8 rows 281 -> 237 =
// 6.8, 4,096 x 1,536 157 -> 141 = 5.7 with two workgroups per CU, three now (see the kernel). That launch's waves have three steps each, so
// start and reduction weigh most; several column tiles a workgroup, the next one's first loads ahead of the reduction, made it 2 % faster
// with two workgroups, but take the registers that a third one has now, and were slower with more tiles and in other launches.
// The memory reads 1.000 to 1.007 times the weights' bytes (1.01 to 1.13 before). 224 launches of 4 to 128
// experts, 4 MB to 2.1 GB of weights, 0.3 to 60 rows each, even and uneven loads: 26 % less time on average, none slower than by the
// spread of a 10 us launch; 181 with odd row pitches 17 % less.
#include "gemm_common.h"

namespace ck {
namespace {

constexpr int kNT = 256, kWaves = kNT / kWave;
constexpr int kStepBytes = 128;  // one cache line of every operand row per wave and step
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));

struct fp8_t {};  // e4m3 operand bytes

template <typename TI>
struct Operand {
  static constexpr int kBytes = 2;
};
template <>
struct Operand<fp8_t> {
  static constexpr int kBytes = 1;
};

// one step: 64 contraction values of 16 columns x 16 rows as two 16-bit MFMAs, or 128 values as one fp8 MFMA; the two
// pieces are the lane's quarter of the row's line, 32 bytes; which contraction values those are does not matter as long as
// both operands hold the same
template <typename TI>
__device__ inline void multiply(const vec16 (&w)[2], const vec16 (&a)[2], f32x4& c) {
  if constexpr (std::is_same_v<TI, fp8_t>) {
    union {
      vec16 v[2];
      i32x8_t f;
    } uw, ua;
    uw.v[0] = w[0];
    uw.v[1] = w[1];
    ua.v[0] = a[0];
    ua.v[1] = a[1];
    // both operands e4m3 (cbsz = blgp = 0), block scales 2^0 (127)
    c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(uw.f, ua.f, c, 0, 0, 0, 127, 0, 127);
  } else {
    union {
      vec16 v;
      typename Mfma16<TI>::frag f;
    } uw, ua;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uw.v = w[h];
      ua.v = a[h];
      c = Mfma16<TI>::run(uw.f, ua.f, c);
    }
  }
}

// The two loads of a column block (columns 0 to 7 and 8 to 15, lane l: piece l / 8 of column l % 8) as the two operands of a step:
// lane l: pieces 2 (l / 16) and 2 (l / 16) + 1 of column l % 16. The lanes whose bit 3 is the piece's lowest bit in one order and the
// column's highest in the other change places, 8 lanes apart within a row of 16.
__device__ inline void to_operands(const vec16 (&lines)[2], vec16 (&w)[2]) {
  constexpr int kRowRor8 = 0x128, kLow = 0x3, kHigh = 0xc;  // banks of 4 lanes: lanes 0 to 7 / 8 to 15 of a row
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int low = (int)lines[0].w[d], high = (int)lines[1].w[d];
    w[0].w[d] = (uint32_t)__builtin_amdgcn_update_dpp(low, high, kRowRor8, 0xf, kHigh, false);
    w[1].w[d] = (uint32_t)__builtin_amdgcn_update_dpp(high, low, kRowRor8, 0xf, kLow, false);
  }
}

// TI: operand type, TO: output type; MB: row blocks of 16 per tile, NB: column blocks of 16 per tile. kSwiglu: half of the
// column blocks are up columns, the other half the gate columns of the same outputs; of one block, the first and the last 8 columns.
// LINES: every row of the weights starts on a 128-byte boundary. The tile of rows m0.. and outputs n0..
template <typename TI, typename TO, int MODE, int MB, int NB, bool LINES>
__device__ __attribute__((always_inline)) inline void skinny_tile(const GemmParams& prm, f32x4 (*red)[kWave], int expert, int m0, int n0) {
  constexpr int kEl = Operand<TI>::kBytes;
  constexpr bool kPair = MODE == kSwiglu && NB == 1;              // up and gate columns share a block
  constexpr int NH = MODE == kSwiglu && !kPair ? NB / 2 : NB;  // column blocks of outputs per tile
  static_assert(MODE != kSwiglu || kPair || NB % 2 == 0, "whole up / gate block pairs");
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lrow = lane & 15, lq = lane >> 4;
  const int valid_end = prm.seg_starts[expert] + (int)prm.counts[expert];

  // ---- operand rows of this lane, as 32-bit byte offsets from a uniform base (the host checks that they fit)
  const char* w_base = static_cast<const char*>(prm.w) + (int64_t)expert * prm.w_expert_stride * kEl;
  const char* a_base = static_cast<const char*>(prm.a);
  if (prm.a_gather_div <= 0) a_base += (int64_t)m0 * prm.lda * kEl;
  uint32_t w_off[NB][2], a_off[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int p = min(m0 + i * 16 + lrow, valid_end - 1);  // pad rows re-read a valid row; their results are never stored
    const int row = prm.a_gather_div > 0 ? prm.row_slot[p] / prm.a_gather_div : p - m0;
    a_off[i] = (uint32_t)row * (uint32_t)(prm.lda * kEl) + lq * 32;
  }
  // weights: a load takes the whole lines of 8 columns, lane l 16-byte piece l / 8 of column l % 8; two loads are a column block
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = 8 * h + (lane & 7);
      int n;
      if constexpr (kPair) n = h * prm.I + min(n0 + (lane & 7), prm.I - 1);
      else if constexpr (MODE == kSwiglu) n = (j / NH) * prm.I + min(n0 + (j % NH) * 16 + c, prm.I - 1);
      else n = min(n0 + j * 16 + c, prm.N - 1);
      w_off[j][h] = (uint32_t)n * (uint32_t)(prm.ldw * kEl) + (lane >> 3) * 16;
    }

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Set {
    vec16 w[NB][2], a[MB][2];
  };
  auto fetch = [&](Set& s, int step) __attribute__((always_inline)) {
    const char* wp = w_base + (int64_t)step * kStepBytes;
    const char* ap = a_base + (int64_t)step * kStepBytes;
    // As 32-bit values that it knows nothing of, the offsets stay one register each, behind a scalar base. Otherwise the compiler
    // widens them ahead of the loop, to pairs of which one is zero, and has 2 others in scratch for it.
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) asm("" : "+v"(w_off[j][h]));
#pragma unroll
    for (int i = 0; i < MB; ++i) asm("" : "+v"(a_off[i]));
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) s.w[j][h] = LINES ? load16_nt(wp + w_off[j][h]) : load16(wp + w_off[j][h]);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) s.a[i][h] = load16(ap + a_off[i] + h * 16);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay in front of the products they overlap with
  };
  auto step_products = [&](const Set& s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      vec16 w[2];
      to_operands(s.w[j], w);
#pragma unroll
      for (int i = 0; i < MB; ++i) multiply<TI>(w, s.a[i], acc[i][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  const int row_bytes = prm.K * kEl;
  const int full = row_bytes / kStepBytes;  // whole steps; the rest of a row, if any, is one partial step
  const int mine = __builtin_amdgcn_readfirstlane(full * (wave + 1) / kWaves - full * wave / kWaves);  // steps of this wave
  const int first = __builtin_amdgcn_readfirstlane(full * wave / kWaves);
  Set s0, s1;
  if (mine > 0) {
    fetch(s0, first);
    int t = 0;
    for (; t + 2 < mine; t += 2) {
      fetch(s1, first + t + 1);
      step_products(s0);
      fetch(s0, first + t + 2);
      step_products(s1);
    }
    if (mine - t == 2) {
      fetch(s1, first + t + 1);
      step_products(s0);
      step_products(s1);
    } else {
      step_products(s0);
    }
  }
  if (row_bytes % kStepBytes != 0 && wave == full % kWaves) {  // the partial step: pieces past the end of a row are zero
    const int left = row_bytes - full * kStepBytes;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool in = (2 * lq + h) * 16 < left, in_w = (lane >> 3) * 16 < left;
#pragma unroll
      for (int j = 0; j < NB; ++j) s0.w[j][h] = in_w ? load16(w_base + (int64_t)full * kStepBytes + w_off[j][h]) : zero16();
#pragma unroll
      for (int i = 0; i < MB; ++i) s0.a[i][h] = in ? load16(a_base + (int64_t)full * kStepBytes + a_off[i] + h * 16) : zero16();
    }
    step_products(s0);
  }

  // ---- the four partial tiles meet in LDS; the weight operand is the MFMA's first, so a lane holds 4 consecutive output
  // columns (16 j + 4 (lane / 16) ..) of tile row 16 i + lane % 16
  const int out_lane = lane_again(), out_row = out_lane & 15, out_q = out_lane >> 4;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) red[wave * MB * NB + i * NB + j][out_lane] = acc[i][j];
  __syncthreads();
  auto total_of = [&](int b, int l) {
    f32x4 v = red[b][l];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v += red[w * MB * NB + b][l];
    return v;
  };
  constexpr int kItems = MB * NH * kWave;
  constexpr bool kFp8 = std::is_same_v<TI, fp8_t>;
#pragma unroll
  for (int it = wave * kWave + out_lane; it < kItems; it += kNT) {
    const int b = it / kWave, i = b / NH, j = b % NH;  // lane of the item: this thread's (kNT is a multiple of kWave)
    const int p = m0 + i * 16 + out_row;
    const int n = n0 + j * 16 + 4 * out_q;  // first of 4 columns; widths are multiples of 8, so all 4 exist or none
    const bool inside = p < valid_end && n < (MODE == kSwiglu ? prm.I : prm.N) && (!kPair || out_q < 2);
    f32x4 v = total_of(i * NB + j, out_lane);
    [[maybe_unused]] f32x4 g = v;
    if constexpr (MODE == kSwiglu) g = kPair ? total_of(i, out_lane ^ 32) : total_of(i * NB + j + NH, out_lane);
    if (!inside) continue;
    if constexpr (kFp8) {
      const float rs = prm.a_scale[prm.a_gather_div > 0 ? prm.row_slot[p] / prm.a_gather_div : p];
      const float4 cs = *reinterpret_cast<const float4*>(prm.w_scale + (int64_t)expert * prm.N + n);
      v = f32x4{v[0] * rs * cs.x, v[1] * rs * cs.y, v[2] * rs * cs.z, v[3] * rs * cs.w};
      if constexpr (MODE == kSwiglu) {
        const float4 cg = *reinterpret_cast<const float4*>(prm.w_scale + (int64_t)expert * prm.N + prm.I + n);
        g = f32x4{g[0] * rs * cg.x, g[1] * rs * cg.y, g[2] * rs * cg.z, g[3] * rs * cg.w};
      }
    } else if constexpr (MODE != kSwiglu) {
      if (prm.aux_in != nullptr) {  // per-expert bias: joins the fp32 sum, one rounding
        const TO* bias = static_cast<const TO*>(prm.aux_in) + (int64_t)expert * prm.N + n;
#pragma unroll
        for (int s = 0; s < 4; ++s) v[s] += Elem<TO>::up(bias[s]);
      }
    }
    TO o[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) o[s] = Elem<TO>::down(v[s]);
    if constexpr (MODE == kSwiglu) {  // from the rounded pre-activation, as if it had been a tensor
      TO og[4], oa[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        og[s] = Elem<TO>::down(g[s]);
        const float gf = Elem<TO>::up(og[s]), sg = sigmoid_fast(gf);
        oa[s] = Elem<TO>::down(prm.act_kind == CK_ACT_GLU ? Elem<TO>::up(o[s]) * sg : Elem<TO>::up(o[s]) * gf * sg);
      }
      store4(static_cast<TO*>(prm.aux) + (int64_t)p * prm.I + n, oa[0], oa[1], oa[2], oa[3]);
      if (prm.y != nullptr) {
        TO* pre = static_cast<TO*>(prm.y) + (int64_t)p * 2 * prm.I + n;
        store4(pre, o[0], o[1], o[2], o[3]);
        store4(pre + prm.I, og[0], og[1], og[2], og[3]);
      }
    } else {
      const int64_t row = MODE == kScatter ? prm.row_slot_out[p] : p;
      if (MODE == kScatter || prm.y != nullptr) store4(static_cast<TO*>(prm.y) + row * prm.N + n, o[0], o[1], o[2], o[3]);
      if constexpr (MODE == kGrouped && !kFp8) {
        if (prm.aux != nullptr) {  // CK_ACT_GELU_TANH: the activation of the rounded output
          TO oa[4];
#pragma unroll
          for (int s = 0; s < 4; ++s) oa[s] = Elem<TO>::down(gelu_tanh_fast(Elem<TO>::up(o[s])));
          store4(static_cast<TO*>(prm.aux) + row * prm.N + n, oa[0], oa[1], oa[2], oa[3]);
        }
      }
    }
  }
}

// Narrow weights of few experts are few tiles, and a compute unit streams 28 bytes a ns however many it holds (256 of them: what
// memory gives), so that a launch takes as long as the unit with the most tiles: 128, 256, 384, ... tiles of 32 x 14,336 took 37, 40, 69,
// 73, 102, 107 and 136 us. Where the last round of one tile per unit is at most half full, its tiles go out in two halves of the columns
// therefore: 28, 41, 59, 74, 93, 107 and 125 us (a half's single wave per SIMD does not get the full rate out of its unit, so halves
// are no better for a fuller round). No sum changes. SwiGLU tiles likewise, 4 experts of 2,000 x 3,072 with a row or two in all 11.8 ->
// 10.1 us; where more than a dozen rounds go by, the units are out of step anyway and a last one is worth 1 % or nothing. Of 265 launches
// in all (4 to 128 experts, 4 MB to 2.1 GB) 2 to 3 % less time on average; 3 % of a 10 us launch more for the longer program.
constexpr int kCus = 256;

// Workgroups per compute unit: three of 32-row tiles. Left to itself the compiler takes 174 registers for e4m3 operands, for
// which there is room twice: 128 experts of 4,096 x 1,536 with 8 rows on average, Zipf(0.8), 150 us and now 133, 64 gated ones of 11,264
// x 1,024 176 and 156.
template <typename TI, typename TO, int MODE, int MB, int NB, bool LINES>
__global__ __launch_bounds__(kNT, MB == 1 ? 4 : MB == 2 ? 3 : 2) void grouped_gemm_skinny_kernel(const GemmParams prm) {
  constexpr int BM = 16 * MB, kColumns = 16 * (MODE == kSwiglu ? NB / 2 : NB);
  __shared__ f32x4 red[kWaves * MB * NB][kWave];

  // ---- which tile: expert by expert, column tile by column tile, the row tiles of one column tile in a row; chunks of kChunk
  // consecutive tiles go out over the XCDs, so that the chip reads one stretch of memory at a time
  const int live_m = prm.seg_starts[prm.num_experts] / BM;
  const int total = live_m * prm.n_tiles;
  constexpr int kChunk = 32;
  static_assert(kXcds * kChunk == kCus, "the partial round of the chunks is that of the compute units");
  const int whole = total / kCus * kCus;
  int pid = blockIdx.x, half = -1;
  if (pid < whole) {
    const int j = pid / kXcds;
    pid = (j / kChunk * kXcds + pid % kXcds) * kChunk + j % kChunk;
  } else if (total - whole <= kCus / 2) {
    half = (pid - whole) % 2;
    pid = whole + (pid - whole) / 2;
  }
  if (pid >= total) return;
  const int expert = __builtin_amdgcn_readfirstlane(prm.tile_expert[pid / prm.n_tiles]);
  const int first_m = prm.seg_starts[expert] / BM, expert_m = prm.seg_starts[expert + 1] / BM - first_m;
  const int local = pid - first_m * prm.n_tiles, nt = local / expert_m, mt = first_m + local - nt * expert_m;
  if (half >= 0) return skinny_tile<TI, TO, MODE, MB, NB / 2, LINES>(prm, red, expert, mt * BM, nt * kColumns + half * (kColumns / 2));
  skinny_tile<TI, TO, MODE, MB, NB, LINES>(prm, red, expert, mt * BM, nt * kColumns);
}

template <typename TI, typename TO, int MODE, int MB, int NB>
int launch_tile(const GemmParams& prm_in, int64_t m_tiles, int out_cols, hipStream_t s, const char* name) {
  GemmParams prm = prm_in;
  prm.n_tiles = (int)ceil_div(out_cols, 16 * (MODE == kSwiglu ? NB / 2 : NB));
  const int64_t blocks = m_tiles * prm.n_tiles + kCus / 2;  // where a last round has halves, each of them
  CK_REQUIRE(blocks < (int64_t)0x7fffffff, "%s: grid too large", name);
  constexpr int64_t kLine = 128;
  const bool lines = prm.ldw * Operand<TI>::kBytes % kLine == 0 && reinterpret_cast<uintptr_t>(prm.w) % kLine == 0;
  auto kernel = lines ? grouped_gemm_skinny_kernel<TI, TO, MODE, MB, NB, true> : grouped_gemm_skinny_kernel<TI, TO, MODE, MB, NB, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kNT), 0, s, prm);
  CK_CHECK_LAUNCH(name);
  return CK_OK;
}

template <typename TI, typename TO, int MODE>
int launch_mode(const GemmParams& prm, int64_t rows, int64_t m_tiles, hipStream_t s, const char* name) {
  const int out_cols = MODE == kSwiglu ? prm.I : prm.N;
  switch (prm.align) {
    case 16: {
      // narrow column tiles while the launch would not fill the chip (256 CUs x 4 workgroups) with wide ones; the number of
      // row tiles with work is at most one per row
      const int64_t live = rows < m_tiles ? rows : m_tiles;
      const bool narrow = live * ceil_div(out_cols, MODE == kSwiglu ? 32 : 64) < 1024;
      if (narrow) return launch_tile<TI, TO, MODE, 1, 2>(prm, m_tiles, out_cols, s, name);
      return launch_tile<TI, TO, MODE, 1, 4>(prm, m_tiles, out_cols, s, name);
    }
    case 32: return launch_tile<TI, TO, MODE, 2, 4>(prm, m_tiles, out_cols, s, name);
    case 64: return launch_tile<TI, TO, MODE, 4, 4>(prm, m_tiles, out_cols, s, name);
    default: set_error("%s: no small-row kernel for %d-row tiles", name, prm.align); return CK_ERR_ARG;
  }
}

template <typename TI, typename TO>
int launch_types(const GemmParams& prm, int mode, int64_t rows, int64_t m_tiles, hipStream_t s, const char* name) {
  switch (mode) {
    case kGrouped: return launch_mode<TI, TO, kGrouped>(prm, rows, m_tiles, s, name);
    case kScatter: return launch_mode<TI, TO, kScatter>(prm, rows, m_tiles, s, name);
    case kSwiglu: return launch_mode<TI, TO, kSwiglu>(prm, rows, m_tiles, s, name);
    default: set_error("%s: the small-row kernel has no epilogue %d", name, mode); return CK_ERR_ARG;
  }
}

}  // namespace

int launch_skinny(const GemmParams& prm, int mode, int64_t max_rows, bool fp8, int dtype, hipStream_t stream, const char* name) {
  const int64_t m_tiles = max_rows / prm.align;
  // the padded layout holds at most max_rows - num_experts * (align - 1) rows (ck_sort_max_rows)
  int64_t rows = max_rows - (int64_t)prm.num_experts * (prm.align - 1);
  if (rows < 1) rows = 1;
  CK_DISPATCH_HALF(dtype, name, {
    if (fp8) return launch_types<fp8_t, scalar_t>(prm, mode, rows, m_tiles, stream, name);
    return launch_types<scalar_t, scalar_t>(prm, mode, rows, m_tiles, stream, name);
  });
  return CK_ERR_ARG;
}

}  // namespace ck
