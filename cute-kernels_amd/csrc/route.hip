// Router: top-k over the logits of one token + softmax over the k selected logits, and its backward.
//
// A token is owned by a group of G lanes (a power of two, chosen on the host); each lane keeps ceil(E / G) logits in registers as
// integer keys (order-preserving float bits in the high half, ~expert index in the low half), so "largest value, lowest
// expert index on ties" is a plain integer max that a butterfly over the lanes reduces in log2(G) steps. A 16-bit logit and
// its index fit one 32-bit key, whose butterfly inside 16 lanes is one v_max with a DPP operand per step; fp32 logits take
// 64-bit keys and two shuffles per step.
#include "ck_common.h"

namespace ck {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxPerLane = 16;  // E <= 64 * 16
constexpr int kMaxTopK = 32;

// Key<T>: the sort key of a logit with its expert, the logit and the expert of a key. A key is never 0 (a real expert index is
// below the low half's maximum).
template <typename T>
struct Key {  // 16-bit logits
  typedef uint32_t type;
  __device__ static type make(T value, int e) {
    const float v = Elem<T>::up(value);
    uint32_t u = (uint32_t)__builtin_bit_cast(unsigned short, value);
    if (u == 0x8000u) u = 0;                                // -0.0 -> +0.0 so that the two zeros tie
    u = (u & 0x8000u) ? (~u & 0xffffu) : (u | 0x8000u);
    if (v != v) u = 0xffffu;                                // NaN sorts above everything, as torch does
    return (u << 16) | (0xffffu - (uint32_t)e);
  }
  __device__ static float value(type key) {  // -0.0 comes back as +0.0
    const uint32_t u = key >> 16;
    return Elem<T>::up(__builtin_bit_cast(T, (unsigned short)((u & 0x8000u) ? (u & 0x7fffu) : (~u & 0xffffu))));
  }
  __device__ static uint32_t expert(type key) { return 0xffffu - (key & 0xffffu); }
};
template <>
struct Key<float> {
  typedef uint64_t type;
  __device__ static type make(float v, int e) {
    uint32_t u = 0xffffffffu;
    if (v == v) {
      u = __float_as_uint(v + 0.0f);
      u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    }
    return ((uint64_t)u << 32) | (uint32_t)(0xffffffffu - (uint32_t)e);
  }
  __device__ static float value(type key) {
    const uint32_t u = (uint32_t)(key >> 32);
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
  }
  __device__ static uint32_t expert(type key) { return 0xffffffffu - (uint32_t)key; }
};

// the largest key of a group of G consecutive lanes, in all of them
__device__ inline uint64_t group_max(uint64_t best, int G) {
  for (int off = G >> 1; off > 0; off >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)best, off, kWave);
    const uint32_t hi = __shfl_xor((uint32_t)(best >> 32), off, kWave);
    const uint64_t other = ((uint64_t)hi << 32) | lo;
    best = other > best ? other : best;
  }
  return best;
}
template <int CTRL>
__device__ inline uint32_t max_dpp(uint32_t v) {
  const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
  return other > v ? other : v;
}
__device__ inline uint32_t group_max(uint32_t best, int G) {
  // lanes that differ in bit 0, bit 1, then the mirror images inside 8 and 16 lanes (whose halves are uniform by then)
  if (G > 1) best = max_dpp<0xB1>(best);   // quad_perm 1 0 3 2
  if (G > 2) best = max_dpp<0x4E>(best);   // quad_perm 2 3 0 1
  if (G > 4) best = max_dpp<0x141>(best);  // row_half_mirror
  if (G > 8) best = max_dpp<0x140>(best);  // row_mirror
  for (int off = 16; off < G; off <<= 1) {
    const uint32_t other = __shfl_xor(best, off, kWave);
    best = other > best ? other : best;
  }
  return best;
}

// What bounds it: latency. A token's k selections depend on each other, so everything inside one is kept short: the selected
// logit comes back out of its key (a second read of the row was a memory round trip per selection) and the exponentials
// stay in registers until the denominator is known (KMAX of them; the group's lanes all hold them). Every output a caller
// wants is written here, the 16-bit gates and 64-bit ids included: each was a launch of its own behind this one.
// KMAX: upper bound of k in this instantiation.
// BY_LANE: the group has k lanes or more, and lane j writes selection j, so that a store instruction takes whole groups; in
// smaller groups lane 0 writes them all. Not a branch inside: fp32 logits of 16 experts in groups of 2, top-16 and top-8 of 16,384
// tokens, took 10.8 and 7.5 us with both forms in one loop, 10.1 and 6.5 with lane 0's alone.
template <typename T, int PER, int KMAX, bool BY_LANE>
__global__ __launch_bounds__(kBlock) void route_topk_softmax_kernel(const T* __restrict__ logits, int64_t T_tokens,
                                                                     int E, int k, int G, int32_t* __restrict__ selected,
                                                                     int64_t* __restrict__ selected_long,
                                                                     float* __restrict__ gates, T* __restrict__ gates_rounded,
                                                                     T* __restrict__ topk_values) {
  const int lane_in_group = threadIdx.x & (G - 1);
  const int64_t token = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / G;
  const bool live = token < T_tokens;
  const T* row = logits + (live ? token : 0) * (int64_t)E;

  typedef typename Key<T>::type key_t;
  key_t key[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int e = p * G + lane_in_group;  // consecutive lanes read consecutive experts
    key[p] = 0;                           // below every real key
    if (live && e < E) key[p] = Key<T>::make(row[e], e);
  }

  float vmax = 0.f, denom = 0.f, ex[KMAX];
  [[maybe_unused]] uint32_t my_expert = 0;
  [[maybe_unused]] float my_ex = 0.f;
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    if (j >= k) break;
    key_t best = 0;
#pragma unroll
    for (int p = 0; p < PER; ++p) best = key[p] > best ? key[p] : best;
    best = group_max(best, G);
#pragma unroll
    for (int p = 0; p < PER; ++p)
      if (key[p] == best) key[p] = 0;  // keys are unique (they embed the expert index)
    const uint32_t e = Key<T>::expert(best);
    const float v = live ? Key<T>::value(best) : 0.f;
    if (j == 0) vmax = v;
    ex[j] = expf(v - vmax);
    denom += ex[j];
    if constexpr (BY_LANE) {
      if (lane_in_group == j) {
        my_expert = e;
        my_ex = ex[j];
      }
    } else if (live && lane_in_group == 0) {
      if (selected) selected[token * k + j] = (int32_t)e;
      if (selected_long) selected_long[token * k + j] = (int64_t)e;
      if (topk_values) topk_values[token * k + j] = row[e < (uint32_t)E ? e : 0];  // as stored: keeps the sign of a zero
    }
  }
  if (!live) return;
  if constexpr (BY_LANE) {
    if (lane_in_group >= k) return;
    const int64_t at = token * k + lane_in_group;
    const float g = my_ex / denom;
    if (selected) selected[at] = (int32_t)my_expert;
    if (selected_long) selected_long[at] = (int64_t)my_expert;
    if (topk_values) topk_values[at] = row[my_expert < (uint32_t)E ? my_expert : 0];
    if (gates) gates[at] = g;
    if (gates_rounded) gates_rounded[at] = Elem<T>::down(g);
  } else if (lane_in_group == 0) {
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      if (j >= k) break;
      const float g = ex[j] / denom;
      if (gates) gates[token * k + j] = g;
      if (gates_rounded) gates_rounded[token * k + j] = Elem<T>::down(g);
    }
  }
}

// d_values = g * (d_g - sum_i g_i d_g_i); scattered into an otherwise zero row of d_logits. One group of G lanes per token.
// d_gates_rounded (optional): the gradient as it arrived in the 16-bit type. Where it is d_gates rounded to that type,
// the unrounded d_gates is used, elsewhere (something scaled or replaced the gradient on its way) the value that arrived.
template <typename T>
__global__ __launch_bounds__(kBlock) void route_bwd_kernel(const float* __restrict__ gates, const float* __restrict__ d_gates,
                                                            const T* __restrict__ d_gates_rounded,
                                                            const int32_t* __restrict__ selected, int64_t T_tokens, int E,
                                                            int k, T* __restrict__ d_logits) {
  const int64_t token = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  if (token >= T_tokens) return;
  const int lane = threadIdx.x & (kWave - 1);
  auto d_gate = [&](int j) {
    const float exact = d_gates[token * k + j];
    if (d_gates_rounded == nullptr) return exact;
    const float arrived = Elem<T>::up(d_gates_rounded[token * k + j]);
    return Elem<T>::up(Elem<T>::down(exact)) == arrived ? exact : arrived;
  };
  float dot = 0.f;
  for (int j = 0; j < k; ++j) dot += gates[token * k + j] * d_gate(j);
  for (int e = lane; e < E; e += kWave) {
    float d = 0.f;
    for (int j = 0; j < k; ++j) {
      if (selected[token * k + j] == e) {
        const float g = gates[token * k + j];
        d += g * (d_gate(j) - dot);
      }
    }
    d_logits[token * (int64_t)E + e] = Elem<T>::down(d);
  }
}

}  // namespace
}  // namespace ck

using namespace ck;

static int route_impl(const char* name, const void* logits, int32_t dtype, int64_t T, int32_t E, int32_t k,
                      int32_t* selected, int64_t* selected_long, float* gates, void* gates_rounded, void* topk_values,
                      void* stream) {
  CK_REQUIRE(E >= 1 && E <= kWave * kMaxPerLane, "%s: E=%d outside [1, %d]", name, E, kWave * kMaxPerLane);
  CK_REQUIRE(k >= 1 && k <= E && k <= kMaxTopK, "%s: k=%d outside [1, min(E, %d)]", name, k, kMaxTopK);
  CK_REQUIRE(T >= 0, "%s: T is negative", name);
  if (T == 0) return CK_OK;
  CK_REQUIRE(logits && (selected || selected_long) && (gates || gates_rounded),
             "%s: logits, the selection and the gates are required", name);
  // Lanes per token: as few as keep at most 8 logits per lane (fewer lanes = fewer shuffle rounds per selection and more
  // tokens per wave; measured at T = 65,536, E = 128, k = 8: 85 us with a whole wave per token). Wide rows fall back to
  // whole waves with up to 16 logits per lane.
  int G = 1;
  while (G < kWave && (E + G - 1) / G > 8) G <<= 1;
  const int per = (E + G - 1) / G;
  const int64_t blocks = ceil_div(T * G, kBlock);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CK_LAUNCH_ROUTE_FORM(PER, KMAX, BY_LANE)                                                                           \
  hipLaunchKernelGGL((route_topk_softmax_kernel<scalar_t, PER, KMAX, BY_LANE>), dim3((unsigned)blocks), dim3(kBlock), 0, s, \
                     static_cast<const scalar_t*>(logits), T, (int)E, (int)k, G, selected, selected_long, gates,           \
                     static_cast<scalar_t*>(gates_rounded), static_cast<scalar_t*>(topk_values))
#define CK_LAUNCH_ROUTE(PER, KMAX)                      \
  do {                                                  \
    if (G >= k) CK_LAUNCH_ROUTE_FORM(PER, KMAX, true);  \
    else CK_LAUNCH_ROUTE_FORM(PER, KMAX, false);        \
  } while (0)
#define CK_LAUNCH_ROUTE_K(PER)                                       \
  do {                                                               \
    if (k <= 2) CK_LAUNCH_ROUTE(PER, 2);                             \
    else if (k <= 8) CK_LAUNCH_ROUTE(PER, 8);                        \
    else CK_LAUNCH_ROUTE(PER, kMaxTopK);                             \
  } while (0)
  CK_DISPATCH_FLOAT(dtype, name, {
    if (per <= 4) CK_LAUNCH_ROUTE_K(4);
    else if (per <= 8) CK_LAUNCH_ROUTE_K(8);
    else CK_LAUNCH_ROUTE_K(16);
  });
#undef CK_LAUNCH_ROUTE_K
#undef CK_LAUNCH_ROUTE
#undef CK_LAUNCH_ROUTE_FORM
  CK_CHECK_LAUNCH(name);
  return CK_OK;
}

extern "C" int ck_route_topk_softmax(const void* logits, int32_t dtype, int64_t T, int32_t E, int32_t k,
                                     int32_t* selected, float* gates, void* topk_values, void* stream) {
  return route_impl("ck_route_topk_softmax", logits, dtype, T, E, k, selected, nullptr, gates, nullptr, topk_values, stream);
}

extern "C" int ck_route_topk_softmax_all(const void* logits, int32_t dtype, int64_t T, int32_t E, int32_t k,
                                         int32_t* selected, int64_t* selected_long, float* gates, void* gates_rounded,
                                         void* stream) {
  return route_impl("ck_route_topk_softmax_all", logits, dtype, T, E, k, selected, selected_long, gates, gates_rounded,
                    nullptr, stream);
}

static int route_bwd_impl(const char* name, const float* gates, const float* d_gates, const void* d_gates_rounded,
                          const int32_t* selected, int64_t T, int32_t E, int32_t k, void* d_logits, int32_t dtype,
                          void* stream) {
  CK_REQUIRE(E >= 1 && k >= 1 && k <= E && T >= 0, "%s: bad sizes T=%lld E=%d k=%d", name, (long long)T, E, k);
  if (T == 0) return CK_OK;
  CK_REQUIRE(gates && d_gates && selected && d_logits, "%s: NULL argument", name);
  const int64_t blocks = ceil_div(T, kBlock / kWave);
  hipStream_t s = static_cast<hipStream_t>(stream);
  CK_DISPATCH_FLOAT(dtype, name, {
    hipLaunchKernelGGL((route_bwd_kernel<scalar_t>), dim3((unsigned)blocks), dim3(kBlock), 0, s, gates, d_gates,
                       static_cast<const scalar_t*>(d_gates_rounded), selected, T, (int)E, (int)k,
                       static_cast<scalar_t*>(d_logits));
  });
  CK_CHECK_LAUNCH(name);
  return CK_OK;
}

extern "C" int ck_route_topk_softmax_bwd(const float* gates, const float* d_gates, const int32_t* selected, int64_t T,
                                         int32_t E, int32_t k, void* d_logits, int32_t dtype, void* stream) {
  return route_bwd_impl("ck_route_topk_softmax_bwd", gates, d_gates, nullptr, selected, T, E, k, d_logits, dtype, stream);
}

extern "C" int ck_route_topk_softmax_bwd_exact(const float* gates, const float* d_gates_exact, const void* d_gates,
                                               const int32_t* selected, int64_t T, int32_t E, int32_t k, void* d_logits,
                                               int32_t dtype, void* stream) {
  const char* name = "ck_route_topk_softmax_bwd_exact";
  CK_REQUIRE(T == 0 || d_gates != nullptr, "%s: d_gates is required", name);
  CK_REQUIRE(dtype != CK_F32, "%s: d_gates of a 16-bit type (fp32 gradients go to ck_route_topk_softmax_bwd)", name);
  return route_bwd_impl(name, gates, d_gates_exact, d_gates, selected, T, E, k, d_logits, dtype, stream);
}
