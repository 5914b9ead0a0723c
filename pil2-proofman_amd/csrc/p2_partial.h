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
// the VALU work of the other waves. A holds zeros in half of its lanes then; the state
// after the segment, which no S-box waits for, is computed with words exchanged between
// lanes l and l + 32 and whole operands (111 -> 81 products a segment at width 12, leaves
// of 2^20 x 128 rows 4.37 -> 4.10 ms).
//
// (Bytes, digits and addends: gl_digits.h. The addend of a result carries the round
// constant that is added to it next.)
#pragma once
#include "gl_digits.h"
#include "p2_constants.h"

#define P2_SEG 11  // rounds per segment (odd: y_1 .. y_10 fill whole operands)
#define P2_SEGS 2  // 22 partial rounds

namespace p2c {

using glc::add;
using glc::addends;
using glc::mul;

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
// (s_{W-1}, y_0), (y_1, y_2), ..., and the u in pairs too: (u_{2p+1}, u_{2p+2}) takes
// every in-pair up to (y_{2p-1}, y_{2p}) and then (y_{2p+1}, -) for its second word. All
// in-pairs of the next pair but its last come before that (y_{2p+1}, -). These operands
// are 16 rows (out-word, digit) of 16 bytes (in-word, byte) and a 17th row of zeros,
// which the lanes off the diagonal read.
//
// The state after the segment takes no part in that chain, so its products use the
// whole operand: lanes l and l + 32 exchange words (v_permlane32_swap), after which one
// B operand holds four words of the lower lane's permutation and another four of the
// upper one's, and one D operand four words of the result, two in each lane. That takes
// half the products: four out-words of 2 in-pairs are 2 x 2 instead of 2 x 4. In-pairs
// 2t and 2t + 1 give operand t (an odd last pair is paired with nothing), out-words 4m,
// 4m + 1 are in lane l, 4m + 2 and 4m + 3 in lane l + 32; 32 rows of 32 bytes.
template <int W> struct Operands {
    static constexpr int NS = W / 2, NY = (P2_SEG - 1) / 2;  // in-pairs: NS, then NY
    static constexpr int NU = (P2_SEG - 1) / 2;              // pairs of u
    static constexpr int COUNT = NS + NU * NS + NU * (NU - 1) / 2 + 2 * NU - NS - NY;  // operands of the u
    static constexpr int STRIDE = 17 * 16;
    static constexpr int NK = (NS + NY + 1) / 2, NM = W / 4;  // state operands: NM rows of NK
    static constexpr int STATE = COUNT * STRIDE;              // where they start
    static_assert(Forms<W>::NIN * 8 * 128 * 128 < 1 << 22, "digit sums (p2_digits)");
    alignas(16) int8_t b[STATE + NM * NK * 1024];
    // the digits of coefficient c times 2^(8a), a < 8: row t, byte a at b[at + t * 16 + a]
    constexpr void digits(int at, uint64_t c)
    {
        uint64_t v = c;
        for (int a = 0; a < 8; a++, v = mul(v, 256)) {
            const glc::Digits d(v);
            for (int t = 0; t < 8; t++) b[at + t * 16 + a] = d.d[t];
        }
    }
    constexpr void put(int n, int out0, int in0, bool half)
    {
        for (int o = 0; o < 2; o++)
            for (int i = 0; i < (half ? 1 : 2); i++)
                digits(n * STRIDE + o * 8 * 16 + i * 8, half && o == 0 ? 0 : forms<W>.c[out0 + o][in0 + i]);
    }
    constexpr Operands() : b{}
    {
        int n = 0;
        for (int t = 0; t < NS; t++) put(n++, 0, 2 * t, false);
        for (int p = 0; p < NU; p++) {
            for (int t = 0; t < NS + p && p + 1 < NU; t++) put(n++, 2 * p + 2, 2 * t, false);
            put(n++, 2 * p, 2 * (NS + p), true);
            if (p + 1 < NU) put(n++, 2 * p + 2, 2 * (NS + p), false);
        }
        // 16-byte pieces: k-half kh of the 16 rows of row half oh at ((kh * 2 + oh) * 16 + row) * 16
        for (int m = 0; m < NM; m++)
            for (int k = 0; k < NK; k++)
                for (int oh = 0; oh < 2; oh++)
                    for (int o = 0; o < 2; o++)
                        for (int kh = 0; kh < 2; kh++)
                            for (int i = 0; i < 2; i++) {
                                int in = 4 * k + 2 * kh + i;
                                if (in < Forms<W>::NIN)
                                    digits(STATE + (m * NK + k) * 1024 + ((kh * 2 + oh) * 16 + o * 8) * 16 + i * 8,
                                           forms<W>.c[P2_SEG - 1 + 4 * m + 2 * oh + o][in]);
                            }
    }
};

// Per segment and out-word the addends of its result: the correction for the signed
// bytes and the round constant added to the word next.
template <int W> struct Addends {
    static constexpr int NOUT = Forms<W>::NOUT;
    uint64_t k[P2_SEGS][NOUT][2];
    constexpr Addends() : k{}
    {
        for (int g = 0; g < P2_SEGS; g++)
            for (int o = 0; o < NOUT; o++) {
                uint64_t s = 0;
                for (int i = 0; i < Forms<W>::NIN; i++) s = add(s, forms<W>.c[o][i]);
                uint64_t v = mul(mul(s, 128), glc::kBytes);
                int r = g * P2_SEG + o + 1;  // the partial round whose S-box takes out-word o (o = 10: w_0)
                if (o < P2_SEG && r < P2_SEG * P2_SEGS) v = add(v, rc(W, 4 * W + r) % GL_P);
                // after the last segment the first of the closing full rounds follows
                if (o >= P2_SEG - 1 && g == P2_SEGS - 1) v = add(v, rc(W, 4 * W + 22 + o - (P2_SEG - 1)) % GL_P);
                addends(v, k[g][o]);
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

typedef gl_v4i p2_v4i;
typedef gl_v16i p2_v16i;

#if defined(__HIP_DEVICE_COMPILE__)

// Copies the operands of width W into a block's LDS (every thread; the caller syncs).
template <int W>
__device__ __forceinline__ void p2_operands_load(p2_v4i *s)
{
    const p2_v4i *g = (const p2_v4i *)c_p2_operands<W>.b;
    for (uint32_t i = threadIdx.x; i < sizeof(p2c::Operands<W>::b) / 16; i += blockDim.x) s[i] = g[i];
}

// Where the lane's row l % 32 of the A operands is in LDS, for k-half l / 32: D row
// 8q + 4h + j is row 4q + j of lane half h. u: the 16 rows of a diagonal operand, for
// lanes whose row belongs to the other half the zero row; w: of a state operand.
struct p2_rows {
    const p2_v4i *u, *w;
};
template <int W>
__device__ __forceinline__ p2_rows p2_operand_rows(const p2_v4i *s)
{
    uint32_t l = __lane_id(), row = l & 31, kh = l >> 5, oh = (row >> 2) & 1, i = 4 * (row >> 3) + (row & 3);
    return {s + (oh == kh ? i : 16), s + p2c::Operands<W>::STATE / 16 + (kh * 2 + oh) * 16 + i};
}

// The result whose eight digit sums (absolute values < 2^22) start at acc[at]: lo + 2^32 hi
// plus the addends k, the same for the wave (SK) or each lane's own
template <bool SK>
__device__ __forceinline__ hz p2_digits(const p2_v16i &acc, int at, const uint64_t *k)
{
    const gl_v4i a = {acc[at], acc[at + 1], acc[at + 2], acc[at + 3]};
    const gl_v4i b = {acc[at + 4], acc[at + 5], acc[at + 6], acc[at + 7]};
    return gl_digit_sums<SK>(a, b, k[0], k[1]);
}

// The A operands on their way from LDS, P2_AHEAD of them (1 and 2 measure the same within
// 2 %; more pushes width 16 further over 128 VGPRs). First those of the u, then the state's.
#define P2_AHEAD 2
template <int W> struct p2_stream {
    using Op = p2c::Operands<W>;
    p2_rows ops;
    p2_v4i a[P2_AHEAD];
    int n;
    __device__ __forceinline__ void fetch(int i)
    {
        if (i < Op::COUNT)
            a[i % P2_AHEAD] = ops.u[i * 17];
        else if (i < Op::COUNT + Op::NM * Op::NK)
            a[i % P2_AHEAD] = ops.w[(i - Op::COUNT) * 64];
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void start(const p2_rows &o)
    {
        ops = o;
        n = 0;
#pragma unroll
        for (int i = 0; i < P2_AHEAD; i++) fetch(i);
    }
    // acc += operand n * in
    __device__ __forceinline__ void mac(p2_v16i &acc, const p2_v4i &in)
    {
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[n % P2_AHEAD], in, acc, 0, 0, 0);
        fetch(n + P2_AHEAD);
        n++;
    }
    // acc0 += operand n * in0, acc1 += operand n * in1
    __device__ __forceinline__ void mac2(p2_v16i &acc0, const p2_v4i &in0, p2_v16i &acc1, const p2_v4i &in1)
    {
        acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[n % P2_AHEAD], in0, acc0, 0, 0, 0);
        mac(acc1, in1);
    }
};

// x of lanes 32 .. 63 and y of lanes 0 .. 31 change places
__device__ __forceinline__ void p2_swap32(int &x, int &y)
{
    auto r = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    x = (int)r[0];
    y = (int)r[1];
}

// One segment on the state s, where s[0] already holds its round constant; s[0] (and
// after the last segment every word) comes out with the next one. All 64 lanes of the
// wave must be active: the A operands are spread over them. While an S-box runs, the
// products of the next pair of u that do not wait for it are under way.
template <int W>
__device__ __forceinline__ void p2_segment(uint64_t *s, const p2_rows &ops, int g)
{
    using Op = p2c::Operands<W>;
    constexpr int NS = Op::NS, NY = Op::NY, NU = Op::NU;
    const uint64_t(*k)[2] = c_p2_addends<W>.k[g];
    p2_v4i in[2 * Op::NK];
    p2_stream<W> st;
    st.start(ops);
#pragma unroll
    for (int i = 1; i < W; i++) gl_put_word(in[(i - 1) / 2], (i - 1) % 2, s[i]);
    p2_v16i acc = {}, nxt;
#pragma unroll
    for (int t = 0; t < NS - 1; t++) st.mac(acc, in[t]);
    gl_put_word(in[NS - 1], 1, pow7(s[0]));
    st.mac(acc, in[NS - 1]);
#pragma unroll
    for (int p = 0; p < NU; p++) {
        hz u = p2_digits<true>(acc, 0, k[2 * p]);
        nxt = (p2_v16i){};
#pragma unroll
        for (int t = 0; t < NS + p && p + 1 < NU; t++) st.mac(nxt, in[t]);
        uint64_t y = pow7(hz_fold(u));
        gl_put_word(in[NS + p], 0, y);
        gl_put_word(in[NS + p], 1, y);  // any value: its coefficients in the next operand are zero
        st.mac(acc, in[NS + p]);
        u = p2_digits<true>(acc, 8, k[2 * p + 1]);
        // the first word's sums are written again by the second product: they stay
        // reserved until its results have been read
        asm volatile("" : "+v"(u.lo) : "v"(acc));
        gl_put_word(in[NS + p], 1, pow7(hz_fold(u)));
        if (p + 1 < NU) st.mac(nxt, in[NS + p]);
        acc = nxt;
    }
    if ((NS + NY) % 2) in[NS + NY] = in[NS + NY - 1];  // any value: its coefficients are zero
#pragma unroll
    for (int t = 0; t < Op::NK; t++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            int x = in[2 * t][i], y = in[2 * t + 1][i];
            p2_swap32(x, y);
            in[2 * t][i] = x;
            in[2 * t + 1][i] = y;
        }
    }
    // the state words' addends, those of lane half h at k[.. + 2h]
    const uint64_t(*kh)[2] = k + P2_SEG - 1 + 2 * (__lane_id() >> 5);
#pragma unroll
    for (int m = 0; m < Op::NM; m++) {
        acc = nxt = (p2_v16i){};
#pragma unroll
        for (int t = 0; t < Op::NK; t++) st.mac2(acc, in[2 * t], nxt, in[2 * t + 1]);
#pragma unroll
        for (int o = 0; o < 2; o++) {
            uint64_t x = hz_fold(p2_digits<false>(acc, 8 * o, kh[4 * m + o]));
            uint64_t y = hz_fold(p2_digits<false>(nxt, 8 * o, kh[4 * m + o]));
            asm volatile("s_nop 1" : "+v"(x), "+v"(y));  // the exchange reads what inline assembly wrote
            int x0 = (int)(uint32_t)x, x1 = (int)(x >> 32), y0 = (int)(uint32_t)y, y1 = (int)(y >> 32);
            p2_swap32(x0, y0);
            p2_swap32(x1, y1);
            s[4 * m + o] = gl_pack((uint32_t)x0, (uint32_t)x1);
            s[4 * m + 2 + o] = gl_pack((uint32_t)y0, (uint32_t)y1);
        }
    }
}
#else  // host pass: declarations only (the kernels are compiled for the device)
template <int W> __device__ void p2_operands_load(p2_v4i *s);
struct p2_rows {
    const p2_v4i *u, *w;
};
template <int W> __device__ p2_rows p2_operand_rows(const p2_v4i *s);
template <int W> __device__ void p2_segment(uint64_t *s, const p2_rows &ops, int g);
#endif
