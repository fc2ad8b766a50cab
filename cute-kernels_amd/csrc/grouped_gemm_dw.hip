// Weight gradients from row-major operands, for contractions too short for the 256 x 256 kernel: dw[e] = a[rows of e]^T @
// b[rows of e], bf16 / f16, fp32 accumulation on v_mfma_f32_16x16x32.
//
// What bounds it: a weight-gradient tile contracts over one expert's rows, a few hundred to a few thousand. On the kernel with
// 128-byte LDS rows (grouped_gemm_line.hip: one workgroup per compute unit, all registers and 128 KiB of LDS) a 256 x 256 tile
// of 400 rows takes 22 us (128 experts of 4,096 x 1,536: 48 rounds in 1,056 us), of which its MFMAs are 8: the dependent loads
// of the segment tables, the first operands' latency and the output stores have nothing to run under them. Here a tile is 128 x 256 and two workgroups share
// a compute unit, so that one multiplies while the other starts up or stores. Per FLOP that reads half as much again from L2
// and LDS, which is what a long contraction is bound by.
//
// Workgroup = 4 waves in a 2 x 2 grid, wave tile 64 x 128 (4 x 8 blocks). A K step is 32 contraction rows of both operands
// (24 KiB): the rows are contraction-strided, so a short step still reads whole 256- and 512-byte row pieces, and fragments
// come out of LDS through ds_read_b64_tr_b16. Three stages: the loads of step kt + 2 go out behind the one barrier of step kt,
// which says that step kt has landed and that step kt - 1 is read. (Wave priority over the MFMAs measured nothing.)
#include "gemm_common.h"

namespace ck {
namespace {

constexpr int TM = 128, TN = 256, BK = 32, kStages = 3;
constexpr int kThreads = 256;
constexpr int kARow = TM * 2, kBRow = TN * 2;  // bytes of a contraction row in LDS
constexpr int kAStage = BK * kARow, kStage = BK * (kARow + kBRow);
constexpr int A_LD = kAStage / 4096, B_LD = (kStage - kAStage) / 4096;  // 1 KiB loads per wave and step
constexpr int kLoads = A_LD + B_LD;
constexpr int MI = 4, NI = 8;
static_assert(2 * kStages * kStage <= 160 * 1024, "two workgroups per compute unit");

// 32-byte window q (16 columns) of contraction row n sits at window position swap02(q) ^ tr_swz(n) of its row: the 4 rows x 32
// bytes that a 16-lane group of a transposing read touches fill one 128-byte block, and the neighbouring group (the same
// columns 8 rows further down) falls into the other half of the banks.
__device__ inline int swap02(int w) { return (w & ~5) | ((w & 1) << 2) | ((w >> 2) & 1); }
__device__ inline int tr_swz(int n) { return (n & 3) | (((n >> 3) & 1) << 2); }

template <typename T>
__global__ __launch_bounds__(kThreads, 2) void grouped_gemm_dw_kernel(const GemmParams prm) {
  __shared__ __attribute__((aligned(1024))) char lds[kStages * kStage];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave >> 1, wn = wave & 1;

  int expert, mt, nt;
  dw_rows_first_tile(prm, blockIdx.x, expert, mt, nt);
  expert = longest_first<kThreads>(prm, expert, reinterpret_cast<int*>(lds));
  const int count = (int)prm.counts[expert];
  const int64_t k_begin = prm.seg_starts[expert], m0 = (int64_t)mt * TM, n0 = (int64_t)nt * TN;
  const int nk = __builtin_amdgcn_readfirstlane((count + BK - 1) / BK);

  auto uniform = [](const char* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<char*>(((uint64_t)hi << 32) | lo);
  };
  const char* a_base = uniform(static_cast<const char*>(prm.a) + k_begin * prm.lda * 2);
  const char* b_base = uniform(static_cast<const char*>(prm.w) + k_begin * prm.ldw * 2);
  // lane offsets of a wave's loads: byte pos of the stage <- the chunk that belongs there. Columns past the matrix re-read the
  // tile's first ones; what they produce is not stored.
  uint32_t off[kLoads];
#pragma unroll
  for (int t = 0; t < kLoads; ++t) {
    const bool is_a = t < A_LD;
    const int row_bytes = is_a ? kARow : kBRow;
    const int pos = (is_a ? wave * A_LD + t : wave * B_LD + t - A_LD) * 1024 + lane * 16;
    const int n = pos / row_bytes, slot16 = (pos % row_bytes) / 16;
    const int q = swap02((slot16 >> 1) ^ tr_swz(n));
    const int64_t first = is_a ? m0 : n0, width = is_a ? prm.M : prm.N;
    int64_t col = first + (2 * q + (slot16 & 1)) * 8;
    if (col >= width) col = first;
    off[t] = (uint32_t)(((int64_t)n * (is_a ? prm.lda : prm.ldw) + col) * 2);
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const uint32_t wave_a = __builtin_amdgcn_readfirstlane(lds_base + wave * A_LD * 1024);
  const uint32_t wave_b = __builtin_amdgcn_readfirstlane(lds_base + kAStage + wave * B_LD * 1024);
  auto load = [&](int step, int stage, int t) __attribute__((always_inline)) {
    const uint32_t to = (t < A_LD ? wave_a + t * 1024 : wave_b + (t - A_LD) * 1024) + (uint32_t)(stage * kStage);
    const char* base = t < A_LD ? a_base + (int64_t)step * BK * prm.lda * 2 : b_base + (int64_t)step * BK * prm.ldw * 2;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(off[t]), "s"(base)
                 : "m0", "memory");
  };
  // rows past the expert's last one hold whatever the buffers hold: every lane zeroes the slots of such rows that its own loads
  // filled, behind those loads and ahead of the barrier that publishes them (both operands: no 0 * Inf)
  auto zero_pad_rows = [&](int step, int stage) {
    const int rows_here = count - step * BK;
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const bool is_a = t < A_LD;
      const int pos = (is_a ? wave * A_LD + t : wave * B_LD + t - A_LD) * 1024 + lane * 16;
      if (pos / (is_a ? kARow : kBRow) >= rows_here) *reinterpret_cast<vec16*>(lds + stage * kStage + (is_a ? 0 : kAStage) + pos) = zero16();
    }
  };

  typedef typename Mfma16<T>::frag frag_t;
  typedef __attribute__((__vector_size__(4 * sizeof(short)))) short tr16x4;
  const int g = lane >> 4, i4 = lane & 15, n_low = i4 >> 2;
  int a_off[MI], b_off[NI];
#pragma unroll
  for (int i = 0; i < MI; ++i) a_off[i] = (8 * g + n_low) * kARow + (swap02(wm * 4 + i) ^ (n_low | ((g & 1) << 2))) * 32 + 8 * (i4 & 3);
#pragma unroll
  for (int j = 0; j < NI; ++j)
    b_off[j] = kAStage + (8 * g + n_low) * kBRow + (swap02(wn * 8 + j) ^ (n_low | ((g & 1) << 2))) * 32 + 8 * (i4 & 3);
  auto read = [&](const char* p, int row_bytes) {
    union {
      tr16x4 h[2];
      frag_t f;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr16x4 __attribute__((address_space(3)))*)(p));
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr16x4 __attribute__((address_space(3)))*)(p + 4 * row_bytes));
    return u.f;
  };

  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto issue = [&](int step, int stage) {
#pragma unroll
    for (int t = 0; t < kLoads; ++t) load(step, stage, t);
  };
  if (nk > 0) issue(0, 0);
  if (nk > 1) issue(1, 1);
  int stage = 0;
  // One K step. fetch: the loads of step kt + 2 go out between the groups of MFMAs, into the stage of step kt - 1. Issued ahead
  // of the MFMAs they hold up the first ones.
  auto step = [&](int kt, auto fetch) __attribute__((always_inline)) {
    const char* st = lds + stage * kStage;
    frag_t fa[MI], fb[NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[i] = read(st + a_off[i], kARow);
#pragma unroll
    for (int j = 0; j < NI; ++j) fb[j] = read(st + b_off[j], kBRow);
    const int behind = stage == 0 ? kStages - 1 : stage - 1;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
      for (int i = 0; i < MI; ++i) acc[i][j] = Mfma16<T>::run(fb[j], fa[i], acc[i][j]);  // 4 consecutive columns of one row per lane
      if constexpr (decltype(fetch)::value) {
        __builtin_amdgcn_sched_barrier(0);
        if (j < kLoads) load(kt + 2, behind, j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    stage = stage == kStages - 1 ? 0 : stage + 1;
  };
  auto landed = [&]() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoads) : "memory"); };
  int kt = 0;
  for (; kt + 2 < nk; ++kt) {
    landed();
    step(kt, std::true_type{});
  }
  if (kt + 1 < nk) {
    landed();
    step(kt, std::false_type{});
    ++kt;
  }
  if (kt < nk) {  // the last step: its loads are the only ones left
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    zero_pad_rows(kt, stage);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    step(kt, std::false_type{});
  }

  // ---- epilogue straight from the accumulators, as in grouped_gemm_line.hip: pairs of column blocks regrouped into 8
  // consecutive columns per lane, 16-byte stores from a uniform base
  const bool odd_group = (g & 1) != 0;
  const int64_t row0 = m0 + wm * 64, col0 = n0 + wn * 128;
  char* base = uniform(reinterpret_cast<char*>(static_cast<T*>(prm.y) + (int64_t)expert * prm.M * prm.N + row0 * prm.N + col0));
  const uint32_t pitch = (uint32_t)prm.N * 2u;
  const int rows_left = (int)min((int64_t)64, (int64_t)prm.M - row0), cols_left = (int)min((int64_t)128, (int64_t)prm.N - col0);
  uint32_t row_off = (uint32_t)i4 * pitch;
  static_for<MI>([&](auto i) {
    static_for<NI / 2>([&](auto jp) {
      const f32x4 p = acc[i][2 * jp], q = acc[i][2 * jp + 1];
      const auto s0 = __builtin_amdgcn_permlane16_swap(pack_pair<T>(p[0], p[1]), pack_pair<T>(q[0], q[1]), false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(pack_pair<T>(p[2], p[3]), pack_pair<T>(q[2], q[3]), false, false);
      vec16 v;
      v.w[0] = s0[0];
      v.w[1] = s1[0];
      v.w[2] = s0[1];
      v.w[3] = s1[1];
      const int col = (2 * jp + (odd_group ? 1 : 0)) * 16 + 4 * (g & ~1);
      if (i * 16 + i4 < rows_left && col < cols_left) store16(base + (row_off + (uint32_t)col * 2u), v);
    });
    row_off += 16u * pitch;
  });
}

}  // namespace

int launch_dw_short(const GemmParams& prm_in, int dtype, hipStream_t s, const char* name) {
  GemmParams prm = prm_in;
  prm.m_tiles = (int)ceil_div(prm.M, TM);
  prm.n_tiles = (int)ceil_div(prm.N, TN);
  const int64_t blocks = (int64_t)prm.m_tiles * prm.n_tiles * prm.num_experts;
  CK_REQUIRE(blocks < (int64_t)0x7fffffff, "%s: grid too large", name);
  CK_DISPATCH_HALF(dtype, name, {
    hipLaunchKernelGGL((grouped_gemm_dw_kernel<scalar_t>), dim3((unsigned)blocks), dim3(kThreads), 0, s, prm);
  });
  CK_CHECK_LAUNCH(name);
  return CK_OK;
}

}  // namespace ck
