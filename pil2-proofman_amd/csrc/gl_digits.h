// Field constants times words on the matrix cores: a word is eight bytes, a constant
// times 2^(8a) mod p eight signed digits of 8 bits, and the int32 sums over byte products
// of v_mfma_i32_*_i8 are put together to a word again.
//
// Bytes are signed in the instruction: a word enters as w ^ 0x8080808080808080, whose
// bytes are those of w minus 128, and 128 * (sum of a result's coefficients) *
// 0x0101010101010101 is part of the addend of the result.
#pragma once
#include "p2_arith.h"

namespace glc {

constexpr uint64_t add(uint64_t a, uint64_t b) { return a >= GL_P - b ? a - (GL_P - b) : a + b; }
constexpr uint64_t mul(uint64_t a, uint64_t b) { return (uint64_t)((unsigned __int128)a * b % GL_P); }
constexpr uint64_t pow(uint64_t b, uint64_t e)
{
    uint64_t r = 1;
    for (; e; e >>= 1, b = mul(b, b))
        if (e & 1) r = mul(r, b);
    return r;
}
constexpr uint64_t kBytes = 0x0101010101010101ULL % GL_P;

// Digit t (0 .. 7) of c: c = sum_t d_t 2^(8t) mod p with d_t in -128 .. 127. c or c - p
// lies in the range of eight such digits.
struct Digits {
    int8_t d[8];
    constexpr explicit Digits(uint64_t c) : d{}
    {
        uint64_t x = c > 0x7F7F7F7F7F7F7F7FULL ? c - GL_P : c;
        for (int t = 0; t < 8; t++) {
            int64_t v = (int64_t)(int8_t)(x & 255);  // byte or byte - 256
            d[t] = (int8_t)v;
            x = (uint64_t)((int64_t)(x - (uint64_t)v) >> 8);
        }
    }
};

// The constant v of a result as the two 64-bit addends of the halves form, with 2^47 in
// each half, which makes the sums non-negative
constexpr void addends(uint64_t v, uint64_t *k)
{
    const uint64_t bias = 1ULL << 47, off = add(bias, mul(bias, 1ULL << 32));
    uint64_t d = add(v, GL_P - off);
    k[0] = bias + (uint32_t)d;
    k[1] = bias + (d >> 32);
}
struct Addend {
    uint64_t k[2];
    constexpr explicit Addend(uint64_t v) : k{} { addends(v, k); }
};
}  // namespace glc

typedef int gl_v4i __attribute__((ext_vector_type(4)));
typedef int gl_v16i __attribute__((ext_vector_type(16)));

#if defined(__HIP_DEVICE_COMPILE__)
// Bytes of a word as the signed bytes of half an operand
__device__ __forceinline__ void gl_put_word(gl_v4i &v, int half, uint64_t w)
{
    v[2 * half] = (int)((uint32_t)w ^ 0x80808080u);
    v[2 * half + 1] = (int)((uint32_t)(w >> 32) ^ 0x80808080u);
}

__device__ __forceinline__ void gl_mac16(gl_v4i &acc, const gl_v4i &a, const gl_v4i &in)
{
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, in, acc, 0, 0, 0);
}

// The result whose digit sums (absolute values < 2^22) are a (digits 0 .. 3) and b (4 ..
// 7), with addends k0, k1 of the lane's own or (SK) in scalar registers
template <bool SK>
__device__ __forceinline__ hz gl_digit_sums(const gl_v4i &a, const gl_v4i &b, uint64_t k0, uint64_t k1)
{
    const uint32_t c16 = 65536;
    uint32_t e0 = ((uint32_t)a[1] << 8) + (uint32_t)a[0], e1 = ((uint32_t)a[3] << 8) + (uint32_t)a[2];
    uint32_t e2 = ((uint32_t)b[1] << 8) + (uint32_t)b[0], e3 = ((uint32_t)b[3] << 8) + (uint32_t)b[2];
    uint64_t l, h, d0, d1;
    if constexpr (SK)
        asm("v_mad_i64_i32 %0, %2, %4, %6, %7\n\t"
            "v_mad_i64_i32 %1, %3, %5, %6, %8"
            : "=&v"(l), "=&v"(h), "=&s"(d0), "=&s"(d1)
            : "v"(e1), "v"(e3), "v"(c16), "s"(k0), "s"(k1));
    else
        asm("v_mad_i64_i32 %0, %2, %4, %6, %7\n\t"
            "v_mad_i64_i32 %1, %3, %5, %6, %8"
            : "=&v"(l), "=&v"(h), "=&s"(d0), "=&s"(d1)
            : "v"(e1), "v"(e3), "v"(c16), "v"(k0), "v"(k1));
    hz r;
    asm("v_mad_i64_i32 %0, %2, %4, 1, %6\n\t"
        "v_mad_i64_i32 %1, %3, %5, 1, %7"
        : "=&v"(r.lo), "=&v"(r.hi), "=&s"(d0), "=&s"(d1)
        : "v"(e0), "v"(e2), "v"(l), "v"(h));
    return r;
}
#endif
