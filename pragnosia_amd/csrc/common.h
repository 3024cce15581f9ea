// Shared definitions for the carrier-path HIP kernels (gfx950 / CDNA4 only).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include <mutex>
#include <set>
#include <utility>

#include "../../include/pragnosia_hip.h"

// Raise a kernel's dynamic LDS limit to `bytes` on the current device, once per (kernel, device). Safe to call from
// several host threads at once (the entry points promise that calls on distinct streams are independent).
inline hipError_t pgn_lds_limit(const void* fn, size_t bytes) {
  static std::mutex mu;
  static std::set<std::pair<const void*, int>> done;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  if (done.count({fn, dev})) return hipSuccess;
  e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) done.insert({fn, dev});
  return e;
}

#define PGN_DEVICE __device__ __forceinline__

// Phase stamps, for the instrumented build only (compiled with -DPRAGNOSIA_PHASE_STAMPS into a separate library; the
// product library has none). A translation unit declares its stamp buffer with PGN_STAMP_UNIT(name), which also
// exports `pragnosia_stamps_set_<name>(void* buffer)` to set it (NULL: no stamps). PGN_STAMP(i) has the wave write
// the low 32 bits of the shader clock (s_memtime) to entry i of the buffer (32-bit entries: differences over a
// kernel's duration do not wrap); PGN_STAMP_CLOCKS(i) writes the shader clock and the constant 100 MHz clock
// (s_memrealtime) to entries i and i + 1, from which the shader clock's rate follows. `i` is wave-uniform: every
// lane stores the same (scalar) value to the same entry, so no branch splits the kernel's scheduled blocks.
#ifdef PRAGNOSIA_PHASE_STAMPS
// The buffer pointer lives in constant memory (one scalar load, hoisted out of the kernels' loops) and points to
// global memory (plain global stores: no wait on the kernel's outstanding loads, stores or LDS traffic).
typedef __attribute__((address_space(1))) unsigned int pgn_stamp_t;
#define PGN_STAMP_UNIT(name)                                                                        \
  static __constant__ pgn_stamp_t* pgn_stamps;                                                      \
  static __constant__ pgn_stamp_t* pgn_stamps_aux;                                                  \
  extern "C" int pragnosia_stamps_set_##name(void* buffer) {                                        \
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(pgn_stamps), &buffer, sizeof(buffer));                 \
  }                                                                                                 \
  extern "C" int pragnosia_stamps_set_##name##_aux(void* buffer) {                                  \
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(pgn_stamps_aux), &buffer, sizeof(buffer));             \
  }
#define PGN_STAMP(i)                                                                                \
  do {                                                                                              \
    pgn_stamp_t* const pgn_b_ = pgn_stamps;                                                         \
    if (pgn_b_ != nullptr) pgn_b_[(i)] = (unsigned int)__builtin_amdgcn_s_memtime();                \
  } while (0)
#define PGN_STAMP_CLOCKS(i)                                                                         \
  do {                                                                                              \
    pgn_stamp_t* const pgn_b_ = pgn_stamps;                                                         \
    if (pgn_b_ != nullptr) {                                                                        \
      pgn_b_[(i)] = (unsigned int)__builtin_amdgcn_s_memtime();                                     \
      pgn_b_[(i) + 1] = (unsigned int)__builtin_amdgcn_s_memrealtime();                             \
    }                                                                                               \
  } while (0)
// The second buffer of a unit (`pragnosia_stamps_set_<name>_aux`), for a kernel launched beside the one stamping the
// first: the shader clock to entry i (PGN_STAMP_AUX), or the shader and 100 MHz clocks to i, i + 1.
#define PGN_STAMP_AUX(i)                                                                            \
  do {                                                                                              \
    pgn_stamp_t* const pgn_b_ = pgn_stamps_aux;                                                     \
    if (pgn_b_ != nullptr) pgn_b_[(i)] = (unsigned int)__builtin_amdgcn_s_memtime();                \
  } while (0)
#define PGN_STAMP_CLOCKS_AUX(i)                                                                     \
  do {                                                                                              \
    pgn_stamp_t* const pgn_b_ = pgn_stamps_aux;                                                     \
    if (pgn_b_ != nullptr) {                                                                        \
      pgn_b_[(i)] = (unsigned int)__builtin_amdgcn_s_memtime();                                     \
      pgn_b_[(i) + 1] = (unsigned int)__builtin_amdgcn_s_memrealtime();                             \
    }                                                                                               \
  } while (0)
#else
#define PGN_STAMP_UNIT(name)
#define PGN_STAMP(i) ((void)0)
#define PGN_STAMP_CLOCKS(i) ((void)0)
#define PGN_STAMP_AUX(i) ((void)0)
#define PGN_STAMP_CLOCKS_AUX(i) ((void)0)
#endif

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(2 * sizeof(int)))) int i32x2;
typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4;

// Launch-time argument failures are reported with negative codes (hipError_t values are non-negative).
#define PGN_CHECK_ARG(cond)                                   \
  do {                                                        \
    if (!(cond)) return PRAGNOSIA_ERR_INVALID_ARGUMENT;       \
  } while (0)

#define PGN_RETURN_LAUNCH()                                   \
  do {                                                        \
    hipError_t e_ = hipGetLastError();                        \
    return e_ == hipSuccess ? PRAGNOSIA_OK : (int)e_;         \
  } while (0)

PGN_DEVICE float pgn_exp(float x) { return __expf(x); }

// GELU, erf form (torch's default F.gelu): 0.5 x (1 + erf(x / sqrt 2)).
PGN_DEVICE float pgn_gelu_erf(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }

// Lane exchanges in the vector unit: DPP row operations within a row of 16 lanes, v_permlane16_swap and
// v_permlane32_swap across rows. __shfl_xor goes through the LDS permute unit, a wait of about 100 cycles a step where
// these take a few cycles, and a decode layer's LayerNorm + GEMV runs three 64-lane sums in series.
template <int CTRL>
PGN_DEVICE float dpp_move(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// With O = 16 or 32 and bit O of the lane number clear: a of the lane plus a of the lane O above; set: b of the lane
// plus b of the lane O below (the swap leaves a's lower and b's lower halves in one register, the upper in the other).
template <int O>
PGN_DEVICE float swap_add(float a, float b) {
  static_assert(O == 16 || O == 32, "");
  const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
  const auto r = O == 16 ? __builtin_amdgcn_permlane16_swap(ua, ub, false, false)
                         : __builtin_amdgcn_permlane32_swap(ua, ub, false, false);
  const unsigned lo = r[0], hi = r[1];  // copied out: a bit cast of a vector's element reads its first one
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}

// Sum over each aligned group of N lanes, in every lane of it: the pairs of a butterfly over lane bits 0, 1, ... (the
// mirrors are exchanges of bits 2 and 3 once the 4 and 8 lanes below hold equal sums). The lanes of a row of 16 must
// all be active, those of the wave for N > 16.
template <int N>
PGN_DEVICE float group_sum(float x) {
  if constexpr (N >= 2) x += dpp_move<0xB1>(x);   // quad_perm [1, 0, 3, 2]
  if constexpr (N >= 4) x += dpp_move<0x4E>(x);   // quad_perm [2, 3, 0, 1]
  if constexpr (N >= 8) x += dpp_move<0x141>(x);  // row_half_mirror
  if constexpr (N >= 16) x += dpp_move<0x140>(x);  // row_mirror
  if constexpr (N >= 32) x = swap_add<16>(x, x);
  if constexpr (N >= 64) x = swap_add<32>(x, x);
  return x;
}

// Sum over the 64 lanes of a wave of NV values per lane (NV a power of two <= 16): the lanes exchange halves, so the
// sums take 6 + NV - 1 exchanges instead of 6 NV. Lane l ends with the sum of value l >> (6 - log2 NV) in v[0].
template <int NV>
PGN_DEVICE void wave_sum_many(float (&v)[NV], int l) {
  if constexpr (NV == 1) {
    v[0] = group_sum<64>(v[0]);
  } else {
#pragma unroll
    for (int m = 0; m < NV / 2; ++m) v[m] = swap_add<32>(v[m], v[m + NV / 2]);
    if constexpr (NV >= 4) {
#pragma unroll
      for (int m = 0; m < NV / 4; ++m) v[m] = swap_add<16>(v[m], v[m + NV / 4]);
    } else {
      v[0] = swap_add<16>(v[0], v[0]);
    }
    if constexpr (NV >= 8) {  // lane bit 3: the lane 8 away keeps the other half
      const bool hi = (l & 8) != 0;
#pragma unroll
      for (int m = 0; m < NV / 8; ++m) {
        const float send = hi ? v[m] : v[m + NV / 8], keep = hi ? v[m + NV / 8] : v[m];
        v[m] = keep + dpp_move<0x128>(send);  // row_ror:8
      }
    }
    if constexpr (NV >= 16) {
      const bool hi = (l & 4) != 0;
      const float send = hi ? v[0] : v[1], keep = hi ? v[1] : v[0];
      v[0] = keep + __shfl_xor(send, 4);
    }
    constexpr int rest = 64 / NV;
    if constexpr (rest == 32) {  // lane bits 0..3 left (bit 4 summed above)
      v[0] = group_sum<16>(v[0]);
    } else {
      v[0] = group_sum<rest>(v[0]);
    }
  }
}

template <int NV>
constexpr int log2_of() { return NV == 1 ? 0 : NV == 2 ? 1 : NV == 4 ? 2 : NV == 8 ? 3 : 4; }

// sin and cos of x. The hardware sine/cosine (through __sincosf) take the argument in revolutions: scaling x to
// revolutions in fp32 costs about |x| * 2^-24 rad of absolute angle error, so they are used for |x| < 64 rad (at
// most ~4e-6 rad; measured 1.3e-6 relative on the diagonal scan's outputs for angles in [-pi, pi]) and the precise
// library routine beyond.
PGN_DEVICE void pgn_sincos(float x, float* s, float* c) {
  if (fabsf(x) < 64.f)
    __sincosf(x, s, c);
  else
    sincosf(x, s, c);
}

// Round-to-nearest-even fp32 -> bf16 (finite inputs).
PGN_DEVICE __bf16 pgn_bf16(float x) { return (__bf16)x; }
PGN_DEVICE float pgn_f32(__bf16 x) { return (float)x; }

// One 16x16x32 bf16 MFMA step: acc += A(16x32) B(32x16).
PGN_DEVICE f32x4 pgn_mfma(bf16x8 a, bf16x8 b, f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
