// An fp32 operand as three bf16 parts whose sum it is exactly (gfx950): what the matrix-core kernels multiply.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace sddmm {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float vec4f __attribute__((ext_vector_type(4)));  // (a plain vector type: stays in registers)
typedef float vec2f __attribute__((ext_vector_type(2)));
typedef uint32_t vec4w __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Eight floats as three bf16 parts each: part 0 is x rounded to 8 significant bits, part 1 what is
// left rounded to 8, part 2 the rest, so x = p0 + p1 + p2 exactly.  `lost` collects the bits below
// part 2, which are nonzero only where x is so small that they lie under bf16's smallest subnormal.
// An infinity or a NaN leaves a NaN in part 1, a value that rounds beyond the range an infinity.
__device__ __forceinline__ void split8(const vec4f lo4, const vec4f hi4, vec4w (&part)[3], uint32_t &lost)
{
    const float x[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        vec2f v = {x[2 * e], x[2 * e + 1]};
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            if (p == 2) lost |= __float_as_uint(v.x) | __float_as_uint(v.y);
            const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
            part[p][e] = b;
            v.x -= __uint_as_float(b << 16);
            v.y -= __uint_as_float(b & 0xffff0000u);
        }
    }
}

// The sum of 16 products per result, by eight of the nine products of parts (the one left out is at most 2^-34 of the
// product): the matrix instruction does not round its sums to nearest, so the products of the first parts, exact for one
// alone, are added up apart from the seven small ones, and vector instructions, which round to nearest, add the two.
__device__ __forceinline__ void add_products(floatx16 &sum, const vec4w (&a)[3], const vec4w (&b)[3])
{
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    constexpr int pp[7] = {1, 2, 0, 1, 2, 0, 1}, qq[7] = {2, 1, 2, 1, 0, 1, 0};
    floatx16 low = zero;  // small ones first
#pragma unroll
    for (int k = 0; k < 7; ++k)
        low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[pp[k]]), __builtin_bit_cast(bf16x8, b[qq[k]]), low, 0, 0, 0);
    const floatx16 high = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[0]), __builtin_bit_cast(bf16x8, b[0]), zero, 0, 0, 0);
    sum += high + low;
    asm volatile("" : "+v"(sum));  // (added here: left alone the compiler sinks it to where the sums are read)
}

}  // namespace sddmm
