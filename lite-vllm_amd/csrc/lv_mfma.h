// MFMA operand types and the 32x32x16 bf16/fp16 matrix instruction used by
// the chunk-attention and linear kernels.
//
// v_mfma_f32_32x32x16_{bf16,f16} (wave64), operand layouts:
//   A[i][k] (32 x 16): lane i % 32 + 32 * (k / 8), element k % 8
//   B[k][j] (16 x 32): lane j % 32 + 32 * (k / 8), element k % 8
//   D[i][j] (32 x 32, fp32): lane j + 32 * ((i / 4) % 2), element 4 * (i / 8) + i % 4
// so a lane's A or B operand is 8 consecutive k of one row: one 16-byte load
// from a k-contiguous matrix.
#pragma once
#include "lv_common.h"

namespace lv {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef short i16x8_t __attribute__((ext_vector_type(8)));


template <typename T> struct Mfma32;
template <> struct Mfma32<bf16> {
  using v8 = bf16x8_t;
  __device__ __forceinline__ static f32x16_t run(v8 a, v8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // Two fp32 values -> packed pair, round to nearest even (v_cvt_pk_bf16_f32).
  __device__ __forceinline__ static uint32_t pack2(float a, float b) {
    return float_to_bf16_pair(a, b);
  }
};
template <> struct Mfma32<f16> {
  using v8 = f16x8_t;
  __device__ __forceinline__ static f32x16_t run(v8 a, v8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static uint32_t pack2(float a, float b) {
    return (uint32_t)float_to_f16_bits(a) | ((uint32_t)float_to_f16_bits(b) << 16);
  }
};

// 16 x 16 instructions (the matrix-core decode kernel).  Layouts:
//   A[i][k]: lane i + 16 * (k / E), element k % E    (E = 8: K = 32; E = 4: K = 16)
//   B[k][j]: lane j + 16 * (k / E), element k % E
//   D[i][j]: lane j + 16 * (i / 4), element i % 4
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma16;
template <> struct Mfma16<bf16> {
  __device__ __forceinline__ static f32x4_t run32(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static f32x4_t run16(i16x4_t a, i16x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
  // The leading bits of x that T holds (truncated; x - head(x) is exact).
  __device__ __forceinline__ static float head(float x) {
    return __uint_as_float(__float_as_uint(x) & 0xffff0000u);
  }
  __device__ __forceinline__ static uint16_t head_bits(float x) {
    return (uint16_t)(__float_as_uint(x) >> 16);
  }
};
template <> struct Mfma16<f16> {
  __device__ __forceinline__ static f32x4_t run32(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static f32x4_t run16(i16x4_t a, i16x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, a),
                                                 __builtin_bit_cast(f16x4_t, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static float head(float x) { return (float)(_Float16)x; }
  __device__ __forceinline__ static uint16_t head_bits(float x) { return float_to_f16_bits(x); }
};

// 16 bytes per lane from global memory into LDS at byte address lds + 16 lane
// (global_load_lds_dwordx4), issued from inline assembly: the compiler does
// not track it, so nothing waits for it but a wait on the vector-memory count
// (its own tracking of loads into LDS would wait for all of them before the
// first LDS read of a loop's next iteration).  lds is the same in every lane.
// The load takes its LDS address from M0.  The hardware needs one wait state
// between a scalar write of M0 and a load that reads it, and the compiler's
// hazard pass does not look into inline assembly: s_nop 0 is that state.  M0
// is not on the clobber lists: the compiler allocates no value to it and
// writes it itself only ahead of instructions of its own that read it
// (load_lds16 below), so a kernel uses either these loads or load_lds16.
#define LV_SET_M0(ARG) "s_mov_b32 m0, " ARG "\n\ts_nop 0\n\t"
// Any address per lane.
__device__ __forceinline__ void load_lds16_async(const void* g, uint32_t lds) {
  asm volatile(LV_SET_M0("%1") "global_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds) : "memory");
}
// base (the same in every lane) + the lane's byte offset; read once, so not
// kept in the caches.
__device__ __forceinline__ void load_lds16_stream(uint64_t base, uint32_t offset, uint32_t lds) {
  asm volatile(LV_SET_M0("%1") "global_load_lds_dwordx4 %0, %2 nt" ::"v"(offset), "s"(lds),
               "s"(base)
               : "memory");
}
#undef LV_SET_M0

// Waits until at most N of the wavefront's vector-memory operations are
// outstanding; loads complete in order.
template <int N>
__device__ __forceinline__ void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Waits until all of the wavefront's LDS operations are done.
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// 16 bytes per lane from global memory straight into LDS at wave base + 16 lane.
__device__ __forceinline__ void load_lds16(const void* g, uint16_t* lds_wave_base) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds_wave_base, 16,
                                   0, 0);
}

}  // namespace lv
