// silu(gate) * up of bfloat16 numbers in float32, for the epilogues of the products that hold both (gemm_block.hip,
// gemm_pair.hip).
#pragma once
#include <hip/hip_runtime.h>

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32;
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// silu(g) * u of bfloat16 numbers below SILU_WIDE in magnitude.  Their product is exact and comes first; exp(-g) is a
// power of two whose argument's rounding is put back; the quotient is by a reciprocal and one Newton step.  No step
// leaves the normal range (87 log2(e) < 126).  Over all gates and eight factors, in ulp of float32, root mean square
// 0.204; g / (1 + expf(-g)) * u, the other kernels' form, 0.222; neither is further off than 2.5 at worst.  That form in its
// place, microseconds of the many-row product at 8,192 rows: 24,576 x 4,096 1,158 against 1,117, 6,144 x 1,024 99 against 90.
#define SILU_WIDE 87.f
#define SILU_WIDE_BITS 0x42ae  // as bfloat16
__device__ __forceinline__ float silu_times(float g, float u) {
    const float t = g * -1.44269502162933349609375f;  // -log2(e), its high part
    const float r = fmaf(g, -1.925963033500011079e-8f, fmaf(g, -1.44269502162933349609375f, -t));
    const float p = __builtin_amdgcn_exp2f(t);
    const float d = 1.f + fmaf(p, r * 0.693147182464599609375f, p);
    const float y = __builtin_amdgcn_rcpf(d), n = g * u, q = n * y;
    return fmaf(fmaf(-d, q, n), y, q);
}
// the same for any two, by the numbers alone (never by what stands beside them)
__device__ __forceinline__ float silu_times_any(float g, float u) {
    return fmaxf(fabsf(g), fabsf(u)) < SILU_WIDE ? silu_times(g, u) : g / (1.f + expf(-g)) * u;
}

// four numbers rounded to bfloat16, two an instruction; `most` keeps the largest magnitudes' bits (NaN above infinity)
__device__ __forceinline__ f32x4 rounded(f32x4 v, u16x2& most) {
    const u32 a = __builtin_bit_cast(u32, __builtin_convertvector(__builtin_shufflevector(v, v, 0, 1), bf16x2));
    const u32 b = __builtin_bit_cast(u32, __builtin_convertvector(__builtin_shufflevector(v, v, 2, 3), bf16x2));
    most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, a & 0x7fff7fffu));
    most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, b & 0x7fff7fffu));
    return __builtin_bit_cast(f32x4, (u32x4){a << 16, a & 0xffff0000u, b << 16, b & 0xffff0000u});
}
