// The GEMM's activation operand (te_gemm.hip): fp32 values as hi + lo bf16 in
// the order the MFMA operand is held in, shared by the kernels that produce it.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Stored values are x * kActScale; the weights' scales carry kActUnscale.
constexpr float kActScale = 0x1p-13f;
constexpr float kActUnscale = 0x1p13f;

// The operand's first byte: the buffer's first 16-byte boundary
// (act_buffer_bytes has room for it).
inline unsigned char *act_base(void *act) {
    return reinterpret_cast<unsigned char *>(((uintptr_t)act + 15) & ~(uintptr_t)15);
}

// Byte offset of values col .. col + 7 (col % 8 == 0) of `row`, hi part (the
// lo part is 2048 bytes on); nb = K / 32.
__device__ __forceinline__ size_t act_off(size_t row, int nb, int col) {
    return (((row >> 5) * (size_t)nb + (size_t)(col >> 5)) << 12) + ((col >> 4) & 1) * 1024 + ((col >> 3) & 1) * 512 +
           (row & 31) * 16;
}

// hi = RNE(x), lo = RNE(x - hi) of a pair.  An infinity or NaN leaves a NaN in
// lo, so its row's products are NaN.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t &hi, uint32_t &lo) {
    const f32x2 x = {x0 * kActScale, x1 * kActScale};
    const bf16x2 h = __builtin_convertvector(x, bf16x2);
    const f32x2 hf = __builtin_convertvector(h, f32x2);
    const f32x2 rest = {x[0] - hf[0], x[1] - hf[1]};
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2));
}

// One value: hi | lo << 16.
__device__ __forceinline__ uint32_t split_pack(float x) {
    uint32_t hi, lo;
    split_pair(x, 0.0f, hi, lo);
    return (hi & 0xffffu) | lo << 16;
}

__device__ __forceinline__ void split_store8(const float (&v)[8], size_t row, int nb, int col,
                                             unsigned char *__restrict__ act) {
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        split_pair(v[2 * j], v[2 * j + 1], hi[j], lo[j]);
    }
    const size_t o = act_off(row, nb, col);
    *reinterpret_cast<uint4 *>(act + o) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4 *>(act + o + 2048) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}
