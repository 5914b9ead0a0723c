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

// Wait states. A register that a matrix instruction reads or writes may be written by a
// VALU instruction only some instructions later (its SrcC after 3 at four passes and 7 at
// eight, its result after 8 and 12, also where nobody reads it). The compiler sees to that
// for the instructions it knows, not for those in inline assembly, and it gives a register
// that is free to the assembly's outputs at once. Assembly near matrix instructions thus
// writes only registers that an instruction of the compiler's has written before: its
// vector outputs start as operands ("+v"), and a value that starts anew is a product in C.
// tests/test_isa_hazards.py looks for early accesses in the built code. (Time against outputs of the assembly's own: LDE of
// 2^22 x 128 to 2^24 30.8 -> 30.6 ms, 2^19 x 64 to 2^20 1,015 -> 1,026 us, commits the same.)

// e 2^16 + k (the factor is hidden from the compiler: shifts and adds take two more), k
// a lane's own or (SK) in scalar registers. An instruction takes one scalar operand: with
// the factor in the other kind of register k stays where it is (a scalar factor for both
// kinds: constants k held in vector registers, 60 of 128 spilled in block passes).
template <bool SK> __device__ __forceinline__ uint64_t gl_mad_64k(int e, uint64_t k)
{
    int c16 = 65536;
    if constexpr (SK)
        asm("" : "+v"(c16));
    else
        asm volatile("" : "+s"(c16));
    return (uint64_t)((int64_t)e * c16) + k;
}
// e + k
__device__ __forceinline__ uint64_t gl_mad_one(int e, uint64_t k)
{
    uint64_t d;
    asm("v_mad_i64_i32 %0, %1, %2, 1, %0" : "+v"(k), "=s"(d) : "v"(e));
    return k;
}

// The result whose digit sums (absolute values < 2^22) are a (digits 0 .. 3) and b (4 ..
// 7), with the addends k0, k1
template <bool SK>
__device__ __forceinline__ hz gl_digit_sums(const gl_v4i &a, const gl_v4i &b, uint64_t k0, uint64_t k1)
{
    int e0 = (int)(((uint32_t)a[1] << 8) + (uint32_t)a[0]), e1 = (int)(((uint32_t)a[3] << 8) + (uint32_t)a[2]);
    int e2 = (int)(((uint32_t)b[1] << 8) + (uint32_t)b[0]), e3 = (int)(((uint32_t)b[3] << 8) + (uint32_t)b[2]);
    return {gl_mad_one(e0, gl_mad_64k<SK>(e1, k0)), gl_mad_one(e2, gl_mad_64k<SK>(e3, k1))};
}
#endif
