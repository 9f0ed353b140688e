// Device helpers shared by the matrix-core decode kernels (attention_mfma.hip,
// attention_rows.h): operand types, wave and workgroup exchanges, and the
// agent-coherent accesses of the in-kernel split merge.
#pragma once

#include <math.h>

#include "attention_internal.h"

namespace smaq {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// s_waitcnt operand that waits for LDS and scalar loads only (lgkmcnt 0,
// vmcnt and expcnt at their maxima)
constexpr int kWaitLdsOnly = 0xC07F;
// s_waitcnt operand that waits for vector memory operations only (vmcnt 0,
// expcnt and lgkmcnt at their maxima)
constexpr int kWaitVmemOnly = 0x0F70;

__device__ __forceinline__ uint32_t f16_bits(_Float16 h) { return (uint32_t)__builtin_bit_cast(uint16_t, h); }

__device__ __forceinline__ f16x8 as_f16x8(u32x4 v) { return __builtin_bit_cast(f16x8, v); }
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// exponent e with |x| in [2^e, 2^(e+1)); 0 for x == 0
__device__ __forceinline__ int exponent_of(float x) {
  if (!(x > 0.0f)) return 0;
  int e;
  frexpf(x, &e);
  return e - 1;
}

// Workgroup barrier that waits for this wave's LDS operations only (global
// loads stay in flight).  The compiler barriers on both sides of the wait
// keep every LDS access of the code around it on its side: the wait
// intrinsic itself does not order memory operations.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(kWaitLdsOnly);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Orders this wave's LDS writes before its later LDS reads of other lanes'
// data (a wave-local exchange; the workgroup's waves run independent tiles).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave-uniform 64-bit value, moved to SGPRs.
__device__ __forceinline__ int64_t uniform64(int64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)x >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// 2^x on the transcendental unit (v_exp_f32); denormal results flush to 0,
// which is harmless for softmax weights.
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Lanes of the banks (4-lane groups of a 16-lane row) in BANKS take `src` from
// the lane the DPP control CTRL names (row_shr:k = lane i - k); the others keep
// `old`.
template <int CTRL, int BANKS>
__device__ __forceinline__ float dpp_bank_move(float old, float src) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, src),
                                                               CTRL, 0xf, BANKS, false));
}

// Rotation within each 16-lane row (CTRL = row_ror:k); fuses into the
// consuming max / add.
template <int CTRL>
__device__ __forceinline__ float dpp_row_ror(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// Two output elements (o0, o1) at element offset oi of the output.
__device__ __forceinline__ void store_out2(const smaq_attn_params& p, int64_t oi, float o0, float o1) {
  switch (p.out_dtype) {
    case SMAQ_F32: {
      float* o = (float*)p.out + oi;
      o[0] = o0;
      o[1] = o1;
    } break;
    case SMAQ_F16: {
      _Float16* o = (_Float16*)p.out + oi;
      o[0] = Num<_Float16>::from_f(o0);
      o[1] = Num<_Float16>::from_f(o1);
    } break;
    default: {
      bf16* o = (bf16*)p.out + oi;
      o[0] = Num<bf16>::from_f(o0);
      o[1] = Num<bf16>::from_f(o1);
    } break;
  }
}

// NaN test on the bits: attention_mfma.hip is built with -fno-honor-nans,
// under which a floating-point self-comparison folds to false.
__device__ __forceinline__ bool is_nan_bits(float x) {
  return (__builtin_bit_cast(uint32_t, x) & 0x7fffffffu) > 0x7f800000u;
}
constexpr float kQuietNaN = __builtin_bit_cast(float, 0x7fc00000u);

// x rounded to the output dtype (kept in fp32).
__device__ __forceinline__ float round_out(const smaq_attn_params& p, float x) {
  switch (p.out_dtype) {
    case SMAQ_F32: return x;
    case SMAQ_F16: return Num<_Float16>::round(x);
    default: return Num<bf16>::round(x);
  }
}

// Agent-coherent (device-scope relaxed atomic) stores and loads: on gfx950
// they carry the sc1 cache policy, so a store is written through the XCD's
// L2 and a load misses a stale L2 line, without cache-wide maintenance.
__device__ __forceinline__ void store_agent(float* a, float v) {
  __hip_atomic_store((uint32_t*)a, __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_agent(float* a, f32x2 v) {
  __hip_atomic_store((uint64_t*)a, __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_agent(const float* a) {
  return __builtin_bit_cast(float, __hip_atomic_load((const uint32_t*)a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ f32x2 load_agent2(const float* a) {
  return __builtin_bit_cast(f32x2, __hip_atomic_load((const uint64_t*)a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

}  // namespace smaq
