// The Poseidon2 partial rounds as linear maps on the matrix cores (gfx950).
//
// A partial round is s0 <- (s0 + rc)^7, s <- diag(d) s + sum(s). Between S-boxes
// everything is linear, so over a segment of P2_SEG rounds the inputs u_1, u_2, ... of
// the later S-boxes and the state after the segment are fixed linear forms of the
// words s_1 .. s_{W-1} before it and the S-box outputs y_0, y_1, ... of its rounds
// (22 rounds = 2 segments with the same forms). Only the S-boxes stay on the VALU:
// 44 + 12 instructions a round instead of 44 + 11 (W + 1) and the state sum.
//
// A form's terms c * word are sums over bytes: word = sum_a 2^(8a) byte_a, and
// c 2^(8a) mod p as eight signed digits of 8 bits gives, per result, eight int32
// sums of products of bytes: v_mfma_i32_32x32x32_i8. Its B operand holds 16 bytes
// (two words) of column l % 32 in each of lanes l and l + 32, its D operand 16 rows
// of the column in each. With A block diagonal over the two lane halves every lane
// multiplies its own two words: a lane keeps its own permutation, one instruction
// gives four word products for each of the 64 lanes, and the matrix cores run beside
// the VALU work of the other waves. (A holds zeros in half of its lanes; spreading a
// permutation over two lanes would use them, but the S-boxes need it in one.)
//
// Bytes are signed in the instruction: words enter as w ^ 0x8080808080808080, i.e.
// byte - 128, and 128 * (sum of the coefficients) * 0x0101010101010101 goes into the
// result's constant together with the round constant that follows it.
#pragma once
#include "p2_arith.h"
#include "p2_constants.h"

#define P2_SEG 11  // rounds per segment (odd: y_1 .. y_10 fill whole operands)
#define P2_SEGS 2  // 22 partial rounds

namespace p2c {

constexpr uint64_t add(uint64_t a, uint64_t b) { return a >= GL_P - b ? a - (GL_P - b) : a + b; }
constexpr uint64_t mul(uint64_t a, uint64_t b) { return (uint64_t)((unsigned __int128)a * b % GL_P); }

constexpr uint64_t rc8[86] = P2_RC8_INIT, rc12[118] = P2_RC12_INIT, rc16[150] = P2_RC16_INIT;
constexpr uint64_t d8[8] = P2_DIAG8_INIT, d12[12] = P2_DIAG12_INIT, d16[16] = P2_DIAG16_INIT;
constexpr uint64_t rc(int w, int i) { return w == 8 ? rc8[i] : w == 12 ? rc12[i] : rc16[i]; }
constexpr uint64_t diag(int w, int i) { return w == 8 ? d8[i] : w == 12 ? d12[i] : d16[i]; }

// The forms of one segment: in-words 0 .. W-2 are s_1 .. s_{W-1}, then y_0 .. y_10;
// out-words 0 .. 9 are u_1 .. u_10 (without round constants), then the W state words.
template <int W> struct Forms {
    static constexpr int NIN = W - 1 + P2_SEG, NOUT = P2_SEG - 1 + W;
    uint64_t c[NOUT][NIN];
    constexpr Forms() : c{}
    {
        uint64_t w[W][NIN] = {};
        for (int i = 1; i < W; i++) w[i][i - 1] = 1;
        for (int r = 0; r < P2_SEG; r++) {
            for (int k = 0; k < NIN; k++) w[0][k] = 0;
            w[0][W - 1 + r] = 1;
            for (int k = 0; k < NIN; k++) {
                uint64_t sum = 0;
                for (int i = 0; i < W; i++) sum = add(sum, w[i][k]);
                for (int i = 0; i < W; i++) w[i][k] = w[i][k] ? add(mul(w[i][k], diag(W, i)), sum) : sum;
            }
            for (int k = 0; k < NIN && r + 1 < P2_SEG; k++) c[r][k] = w[0][k];
        }
        for (int i = 0; i < W; i++)
            for (int k = 0; k < NIN; k++) c[P2_SEG - 1 + i][k] = w[i][k];
    }
};
template <int W> inline constexpr Forms<W> forms{};

// The A operands in the order they are used. In-words go in pairs (s_1, s_2), ...,
// (s_{W-1}, y_0), (y_1, y_2), ..., out-words in pairs too. The pair (u_{2p+1}, u_{2p+2})
// takes every in-pair up to (y_{2p-1}, y_{2p}) and then (y_{2p+1}, -) for its second
// word; the state pairs take all of them. All in-pairs of the next out-pair but its last
// come before that (y_{2p+1}, -). An operand is 16 rows (out-word, digit) of 16 bytes
// (in-word, byte) and a 17th row of zeros, which the lanes off the diagonal read.
template <int W> struct Operands {
    static constexpr int NS = W / 2, NY = (P2_SEG - 1) / 2;  // in-pairs: NS, then NY
    static constexpr int NU = (P2_SEG - 1) / 2;              // pairs of u, then W / 2 of the state
    static constexpr int COUNT = NU * NS + NU * (NU - 1) / 2 + NU + (W / 2) * (NS + NY);
    static constexpr int STRIDE = 17 * 16;
    static_assert(Forms<W>::NIN * 8 * 128 * 128 < 1 << 22, "digit sums (p2_digits)");
    alignas(16) int8_t b[COUNT * STRIDE];
    constexpr void put(int n, int out0, int in0, bool half)
    {
        for (int o = 0; o < 2; o++)
            for (int i = 0; i < (half ? 1 : 2); i++) {
                uint64_t v = half && o == 0 ? 0 : forms<W>.c[out0 + o][in0 + i];
                for (int a = 0; a < 8; a++, v = mul(v, 256)) {
                    // v or v - p in the range of eight digits -128 .. 127; digit = byte or byte - 256
                    uint64_t x = v > 0x7F7F7F7F7F7F7F7FULL ? v - GL_P : v;
                    for (int t = 0; t < 8; t++) {
                        int64_t d = (int64_t)(int8_t)(x & 255);
                        b[n * STRIDE + (o * 8 + t) * 16 + i * 8 + a] = (int8_t)d;
                        x = (uint64_t)((int64_t)(x - (uint64_t)d) >> 8);
                    }
                }
            }
    }
    constexpr Operands() : b{}
    {
        int n = 0;
        for (int t = 0; t < NS; t++) put(n++, 0, 2 * t, false);
        for (int p = 0; p < NU; p++) {
            for (int t = 0; t < NS + p; t++) put(n++, 2 * p + 2, 2 * t, false);
            put(n++, 2 * p, 2 * (NS + p), true);
            put(n++, 2 * p + 2, 2 * (NS + p), false);
        }
        for (int p = NU + 1; p < NU + W / 2; p++)
            for (int t = 0; t < NS + NY; t++) put(n++, 2 * p, 2 * t, false);
    }
};

// Per segment and out-word the constant of its result, as the two 64-bit addends of
// the halves form: the correction for the signed bytes, the round constant added to
// the word next, and 2^47 in each half, which makes the sums non-negative.
template <int W> struct Addends {
    static constexpr int NOUT = Forms<W>::NOUT;
    uint64_t k[P2_SEGS][NOUT][2];
    constexpr Addends() : k{}
    {
        for (int g = 0; g < P2_SEGS; g++)
            for (int o = 0; o < NOUT; o++) {
                uint64_t s = 0;
                for (int i = 0; i < Forms<W>::NIN; i++) s = add(s, forms<W>.c[o][i]);
                uint64_t v = mul(mul(s, 128), 0x0101010101010101ULL % GL_P);
                int r = g * P2_SEG + o + 1;  // the partial round whose S-box takes out-word o (o = 10: w_0)
                if (o < P2_SEG && r < P2_SEG * P2_SEGS) v = add(v, rc(W, 4 * W + r) % GL_P);
                // after the last segment the first of the closing full rounds follows
                if (o >= P2_SEG - 1 && g == P2_SEGS - 1) v = add(v, rc(W, 4 * W + 22 + o - (P2_SEG - 1)) % GL_P);
                const uint64_t bias = 1ULL << 47, off = add(bias, mul(bias, 1ULL << 32));
                uint64_t d = add(v, GL_P - off);
                k[g][o][0] = bias + (uint32_t)d;
                k[g][o][1] = bias + (d >> 32);
            }
    }
};

// The round constants added after full round r (of 8): the next full round's, the first
// partial round's after round 3, none after the last.
template <int W> struct NextRc {
    uint64_t k[8][W];
    constexpr NextRc() : k{}
    {
        for (int r = 0; r < 7; r++)
            for (int i = 0; i < W; i++)
                k[r][i] = r == 3 ? (i == 0 ? rc(W, 4 * W) : 0) : rc(W, (r < 3 ? (r + 1) * W : 4 * W + 22 + (r - 3) * W) + i);
    }
};
}  // namespace p2c

template <int W> __constant__ const p2c::NextRc<W> c_p2_next_rc{};
template <int W> __device__ const p2c::Operands<W> c_p2_operands{};
template <int W> __constant__ const p2c::Addends<W> c_p2_addends{};

typedef int p2_v4i __attribute__((ext_vector_type(4)));
typedef int p2_v16i __attribute__((ext_vector_type(16)));

#if defined(__HIP_DEVICE_COMPILE__)

// Copies the operands of width W into a block's LDS (every thread; the caller syncs).
template <int W>
__device__ __forceinline__ void p2_operands_load(p2_v4i *s)
{
    const p2_v4i *g = (const p2_v4i *)c_p2_operands<W>.b;
    for (uint32_t i = threadIdx.x; i < sizeof(p2c::Operands<W>::b) / 16; i += blockDim.x) s[i] = g[i];
}

// The lane's first A row in LDS: row l % 32 of the operand for k-half l / 32; its data
// row is 4 (row / 8) + row % 4 if the row belongs to that half, else the zero row.
__device__ __forceinline__ const p2_v4i *p2_operand_row(const p2_v4i *s)
{
    uint32_t l = __lane_id(), row = l & 31;
    return s + (((row >> 2) & 1) == (l >> 5) ? 4 * (row >> 3) + (row & 3) : 16);
}

// The result whose eight digit sums (absolute values < 2^22) start at acc[at]: lo + 2^32 hi
// plus the addends
__device__ __forceinline__ hz p2_digits(const p2_v16i &acc, int at, const uint64_t *k, uint32_t c16)
{
    uint32_t a[8];
#pragma unroll
    for (int i = 0; i < 8; i++) a[i] = (uint32_t)acc[at + i];
    uint32_t e0 = (a[1] << 8) + a[0], e1 = (a[3] << 8) + a[2];
    uint32_t e2 = (a[5] << 8) + a[4], e3 = (a[7] << 8) + a[6];
    uint64_t l, h, d0, d1;
    asm("v_mad_i64_i32 %0, %2, %4, %6, %7\n\t"
        "v_mad_i64_i32 %1, %3, %5, %6, %8"
        : "=&v"(l), "=&v"(h), "=&s"(d0), "=&s"(d1)
        : "v"(e1), "v"(e3), "v"(c16), "s"(k[0]), "s"(k[1]));
    hz r;
    asm("v_mad_i64_i32 %0, %2, %4, 1, %6\n\t"
        "v_mad_i64_i32 %1, %3, %5, 1, %7"
        : "=&v"(r.lo), "=&v"(r.hi), "=&s"(d0), "=&s"(d1)
        : "v"(e0), "v"(e2), "v"(l), "v"(h));
    return r;
}

// Bytes of a word as the signed bytes of half an operand
__device__ __forceinline__ void p2_put_word(p2_v4i &v, int half, uint64_t w)
{
    v[2 * half] = (int)((uint32_t)w ^ 0x80808080u);
    v[2 * half + 1] = (int)((uint32_t)(w >> 32) ^ 0x80808080u);
}

// The A operands on their way from LDS, P2_AHEAD of them (1 to 5 measure the same within
// 2 %; more than 2 pushes width 16 over 128 VGPRs).
#define P2_AHEAD 2
template <int W> struct p2_stream {
    const p2_v4i *ops;
    p2_v4i a[P2_AHEAD];
    int n;
    __device__ __forceinline__ void start(const p2_v4i *o)
    {
        ops = o;
        n = 0;
#pragma unroll
        for (int i = 0; i < P2_AHEAD; i++) a[i] = ops[i * 17];
        asm volatile("" ::: "memory");
    }
    // acc += operand n * in; operand n + P2_AHEAD is read
    __device__ __forceinline__ void mac(p2_v16i &acc, const p2_v4i &in)
    {
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[n % P2_AHEAD], in, acc, 0, 0, 0);
        if (n + P2_AHEAD < p2c::Operands<W>::COUNT) a[n % P2_AHEAD] = ops[(n + P2_AHEAD) * 17];
        asm volatile("" ::: "memory");
        n++;
    }
};

// One segment on the state s, where s[0] already holds its round constant; s[0] (and
// after the last segment every word) comes out with the next one. All 64 lanes of the
// wave must be active: the A operands are spread over them. While an S-box runs, the
// products of the next out-pair that do not wait for it are under way.
template <int W>
__device__ __forceinline__ void p2_segment(uint64_t *s, const p2_v4i *ops, int g)
{
    using Op = p2c::Operands<W>;
    constexpr int NS = Op::NS, NY = Op::NY, NU = Op::NU;
    const uint64_t(*k)[2] = c_p2_addends<W>.k[g];
    const uint32_t c16 = 65536;
    p2_v4i in[NS + NY];
    p2_stream<W> st;
    st.start(ops);
#pragma unroll
    for (int i = 1; i < W; i++) p2_put_word(in[(i - 1) / 2], (i - 1) % 2, s[i]);
    p2_v16i acc = {}, nxt;
#pragma unroll
    for (int t = 0; t < NS - 1; t++) st.mac(acc, in[t]);
    p2_put_word(in[NS - 1], 1, pow7(s[0]));
    st.mac(acc, in[NS - 1]);
#pragma unroll
    for (int p = 0; p < NU; p++) {
        hz u = p2_digits(acc, 0, k[2 * p], c16);
        nxt = (p2_v16i){};
#pragma unroll
        for (int t = 0; t < NS + p; t++) st.mac(nxt, in[t]);
        uint64_t y = pow7(hz_fold(u));
        p2_put_word(in[NS + p], 0, y);
        p2_put_word(in[NS + p], 1, y);  // any value: its coefficients in the next operand are zero
        st.mac(acc, in[NS + p]);
        u = p2_digits(acc, 8, k[2 * p + 1], c16);
        // the first word's sums are written again by the second product: they stay
        // reserved until its results have been read
        asm volatile("" : "+v"(u.lo) : "v"(acc));
        p2_put_word(in[NS + p], 1, pow7(hz_fold(u)));
        st.mac(nxt, in[NS + p]);
        acc = nxt;
    }
#pragma unroll
    for (int p = 0; p < W / 2; p++) {
        if (p + 1 < W / 2) {
            nxt = (p2_v16i){};
#pragma unroll
            for (int t = 0; t < NS + NY; t++) st.mac(nxt, in[t]);
        }
        s[2 * p] = hz_fold(p2_digits(acc, 0, k[P2_SEG - 1 + 2 * p], c16));
        s[2 * p + 1] = hz_fold(p2_digits(acc, 8, k[P2_SEG + 2 * p], c16));
        acc = nxt;
    }
}
#else  // host pass: declarations only (the kernels are compiled for the device)
template <int W> __device__ void p2_operands_load(p2_v4i *s);
__device__ const p2_v4i *p2_operand_row(const p2_v4i *s);
template <int W> __device__ void p2_segment(uint64_t *s, const p2_v4i *ops, int g);
#endif
