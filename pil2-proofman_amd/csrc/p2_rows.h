// One Poseidon2 permutation on 16 lanes, for levels too short to fill the GPU with one
// permutation a lane: their time is the latency of a permutation, so what counts is the
// length of its chain of instructions.
//
// Lane l of a wave is (g, n) = (l / 16, l % 16): permutation n / 4 of the wave, word
// 4q + g with q = n % 4 (words W and above are zero). These are the lane groups of
// v_mfma_i32_16x16x64_i8: B holds 16 bytes (two words) of column n from each of the four
// g, D four rows of the column for each g, so a product sums over the eight words that
// the four lanes of a column hold (bytes and digits as in p2_partial.h).
//   external layer   a lane gathers its quad's other words by DPP, own word first; the
//                    layer is M4 (2 x_own + x_other + ...), 4 products and 12 instructions
//   partial rounds   the forms of a segment (p2_partial.h): every lane gets every u (its
//                    rows repeat for each g) and runs the S-box, whose output each g in
//                    turn keeps as one of its in-words: 2 products and 12 instructions
//                    beside the S-box instead of a row sum, a diagonal product and two folds
// In the partial rounds' S-box the lanes are redundant: even ones compute x^3, odd ones
// x^4, and neighbours multiply.
#pragma once
#include "p2_partial.h"

namespace p2c {

// In-words of a segment: slot s of lane group g holds state word 4s + g (s < W / 4, word
// 0 replaced by y_0), then y_{1 + 4 (s - W/4) + g}; slots 2t and 2t + 1 are operand t.
template <int W> struct RowOps {
    static constexpr int NQ = W / 4;
    static constexpr int slot_y(int e) { return e == 0 ? 0 : NQ + (e - 1) / 4; }
    // operands that u_{e+1} takes: up to y_e's, and the state's
    static constexpr int tiles(int e) { return (slot_y(e) > NQ - 1 ? slot_y(e) : NQ - 1) / 2 + 1; }
    static constexpr int NT = tiles(P2_SEG - 1);
    // u_{e+1}, digits 4h .. 4h + 3, operand t: 4 rows for each of 4 k-groups, 256 bytes
    static constexpr int u_at(int e, int h, int t)
    {
        int n = 0;
        for (int i = 0; i < e; i++) n += 2 * tiles(i);
        return (n + h * tiles(e) + t) * 256;
    }
    static constexpr int STATE = u_at(P2_SEG - 1, 0, 0);
    // state words 4q + g, digits 4h .. 4h + 3, operand t: 16 rows for each k-group, 1 KB
    static constexpr int s_at(int q, int h, int t) { return STATE + ((q * 2 + h) * NT + t) * 1024; }
    static constexpr int BYTES = s_at(NQ, 0, 0);
    alignas(16) int8_t b[BYTES];
    static constexpr int in_word(int s, int g)
    {
        if (s < NQ) return 4 * s + g == 0 ? W - 1 : 4 * s + g - 1;
        int e = 1 + 4 * (s - NQ) + g;
        return e < P2_SEG ? W - 1 + e : -1;
    }
    // byte column (slot, a) of row `row` of k-group kg in an operand of `rows` rows
    constexpr void digits(int at0, int at1, int rows, int kg, int row, int slot, uint64_t c)
    {
        uint64_t v = c;
        for (int a = 0; a < 8; a++, v = mul(v, 256)) {
            const glc::Digits d(v);
            for (int t = 0; t < 8; t++) b[(t < 4 ? at0 : at1) + (kg * rows + row + t % 4) * 16 + slot * 8 + a] = d.d[t];
        }
    }
    constexpr RowOps() : b{}
    {
        for (int s = 0; s < 2 * NT; s++)
            for (int kg = 0; kg < 4; kg++) {
                int in = in_word(s, kg), t = s / 2;
                if (in < 0) continue;
                for (int e = 0; e + 1 < P2_SEG; e++)
                    if (t < tiles(e)) digits(u_at(e, 0, t), u_at(e, 1, t), 4, kg, 0, s % 2, forms<W>.c[e][in]);
                for (int q = 0; q < NQ; q++)
                    for (int g = 0; g < 4; g++)
                        digits(s_at(q, 0, t), s_at(q, 1, t), 16, kg, 4 * g, s % 2, forms<W>.c[P2_SEG - 1 + 4 * q + g][in]);
            }
    }
};

constexpr int m4[4][4] = {{5, 7, 1, 3}, {4, 6, 1, 1}, {1, 3, 5, 7}, {1, 1, 4, 6}};

// The external layer's operands: digits 4h .. 4h + 3 of M4 (2 slot_0 + slot_1) and of
// M4 (slot_2 + slot_3); digit t takes byte t only, the entries being below 128.
struct RowExt {
    alignas(16) int8_t b[2][2][4][16][16];  // h, operand, k-group, row, byte column
    constexpr RowExt() : b{}
    {
        for (int h = 0; h < 2; h++)
            for (int t = 0; t < 2; t++)
                for (int kg = 0; kg < 4; kg++)
                    for (int r = 0; r < 16; r++)
                        for (int s = 0; s < 2; s++)
                            b[h][t][kg][r][s * 8 + 4 * h + r % 4] = (int8_t)(m4[r / 4][kg] * (t == 0 && s == 0 ? 2 : 1));
    }
};

// Addends of the external layers (the initial one, then after full rounds 0 .. 7) and of
// the state after a segment, by word 4q + g: see Addends
template <int W> struct RowAddends {
    uint64_t ext[9][16][2], state[P2_SEGS][16][2];
    constexpr RowAddends() : ext{}, state{}
    {
        const Addends<W> seg{};
        const NextRc<W> next{};
        for (int w = 0; w < W; w++) {
            int m = m4[w % 4][0] + m4[w % 4][1] + m4[w % 4][2] + m4[w % 4][3];
            for (int r = 0; r < 9; r++) {
                uint64_t v = mul(128 * 5 * (uint64_t)m, glc::kBytes);
                v = add(v, (r == 0 ? rc(W, w) : next.k[r - 1][w]) % GL_P);
                addends(v, ext[r][w]);
            }
            for (int g = 0; g < P2_SEGS; g++)
                for (int i = 0; i < 2; i++) state[g][w][i] = seg.k[g][P2_SEG - 1 + w][i];
        }
    }
};
}  // namespace p2c

template <int W> __device__ const p2c::RowOps<W> c_p2_row_ops{};
template <int W> __device__ const p2c::RowAddends<W> c_p2_row_addends{};
__device__ const p2c::RowExt c_p2_row_ext{};

#define P2_ROW_THREADS 256
template <int W> constexpr int p2_row_pieces() { return p2c::RowOps<W>::BYTES / 16; }

#if defined(__HIP_DEVICE_COMPILE__)

template <int CTRL>
__device__ __forceinline__ int p2_dpp(int v)
{
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, false);
}

// What was loaded in program order before is requested before what follows from x
__device__ __forceinline__ void p2_loads_first(uint64_t &x) { asm volatile("" : "+v"(x) : : "memory"); }

// x^7 where lanes l and l ^ 1 hold the same x
__device__ __forceinline__ uint64_t p2_pow7_pair(uint64_t x)
{
    uint64_t x2 = p2_mul(x, x);
    uint64_t z = p2_mul(x2, (__lane_id() & 1) ? x2 : x);
    asm("s_nop 1" : "+v"(z));  // DPP reads two wait states after the write
    uint64_t o = gl_pack((uint32_t)p2_dpp<0xB1>((int)(uint32_t)z), (uint32_t)p2_dpp<0xB1>((int)(z >> 32)));
    return p2_mul(z, o);
}

// What a lane keeps through its permutations. The segment operands are read from global
// memory at the start (start), written to LDS when they are first needed (stage), and
// read from there, each before the S-box that it follows.
template <int W> struct p2_row {
    using Op = p2c::RowOps<W>;
    static constexpr int PIECES = p2_row_pieces<W>(), EACH = (PIECES + P2_ROW_THREADS - 1) / P2_ROW_THREADS;
    p2_v4i ext[4], pre[EACH];
    p2_v4i *lds;
    uint32_t g, q, word;
    __device__ __forceinline__ void start(p2_v4i *s)
    {
        const uint32_t l = __lane_id();
        lds = s;
        g = l >> 4;
        q = l & 3;
        word = 4 * q + g;
        const p2_v4i *e = (const p2_v4i *)c_p2_row_ext.b + g * 16 + (l & 15);
#pragma unroll
        for (int i = 0; i < 4; i++) ext[i] = e[i * 64];
        const p2_v4i *o = (const p2_v4i *)c_p2_row_ops<W>.b;
#pragma unroll
        for (int i = 0; i < EACH; i++) {
            uint32_t at = threadIdx.x + i * P2_ROW_THREADS;
            pre[i] = o[at < (uint32_t)PIECES ? at : 0];
        }
    }
    __device__ __forceinline__ void stage()
    {
#pragma unroll
        for (int i = 0; i < EACH; i++) {
            uint32_t at = threadIdx.x + i * P2_ROW_THREADS;
            if (at < (uint32_t)PIECES) lds[at] = pre[i];
        }
        __syncthreads();
    }
    // M_E of the row's words x (zero in lanes without a word), plus the addends k
    __device__ __forceinline__ uint64_t external(uint64_t x, uint64_t k0, uint64_t k1) const
    {
        int lo = (int)((uint32_t)x ^ 0x80808080u), hi = (int)((uint32_t)(x >> 32) ^ 0x80808080u);
        p2_v4i b0 = {lo, hi, p2_dpp<0xB1>(lo), p2_dpp<0xB1>(hi)};
        p2_v4i b1 = {p2_dpp<0x4E>(lo), p2_dpp<0x4E>(hi), p2_dpp<0x1B>(lo), p2_dpp<0x1B>(hi)};
        p2_v4i a = {}, b = {};
        gl_mac16(a, ext[0], b0);
        gl_mac16(b, ext[2], b0);
        gl_mac16(a, ext[1], b1);
        gl_mac16(b, ext[3], b1);
        return hz_fold(gl_digit_sums<false>(a, b, k0, k1));
    }
    // full rounds r .. r + 3: S-box, external layer, next constants
    __device__ __forceinline__ uint64_t full(uint64_t x, int r0) const
    {
        const uint64_t *k = c_p2_row_addends<W>.ext[r0 + 1][word];
#pragma unroll 1
        for (int r = 0; r < 4; r++, k += 32) {
            const uint64_t k0 = k[0], k1 = k[1];
            p2_loads_first(x);
            x = pow7(x);
            x = external(word < (uint32_t)W ? x : 0, k0, k1);
        }
        return x;
    }
    // operands of u_{e+1} (e < 10) or of state words 4 (e - 11) + g
    __device__ __forceinline__ void operands(p2_v4i (&o)[2][Op::NT], int e) const
    {
        const uint32_t l = __lane_id();
        const p2_v4i *ou = lds + g * 4 + (l & 3), *os = lds + g * 16 + (l & 15);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int t = 0; t < Op::NT; t++) {
                if (e < P2_SEG - 1) {
                    if (t < Op::tiles(e)) o[h][t] = ou[Op::u_at(e, h, t) / 16];
                } else {
                    o[h][t] = os[Op::s_at(e - (P2_SEG - 1), h, t) / 16];
                }
            }
    }
    // 11 partial rounds; word 0 comes with its round constant
    __device__ __forceinline__ uint64_t segment(uint64_t x, int sg) const
    {
        constexpr int NQ = Op::NQ, NT = Op::NT;
        const uint32_t l = __lane_id();
        p2_v4i cur[2][NT], nxt[2][NT];
        operands(cur, 0);
        uint64_t k[P2_SEG - 1][2];
#pragma unroll
        for (int e = 0; e + 1 < P2_SEG; e++) {
            k[e][0] = c_p2_addends<W>.k[sg][e][0];
            k[e][1] = c_p2_addends<W>.k[sg][e][1];
            asm volatile("" : "+s"(k[e][0]), "+s"(k[e][1]));
        }
        const uint64_t *ks = c_p2_row_addends<W>.state[sg][word];
        const uint64_t ks0 = ks[0], ks1 = ks[1];
        asm volatile("s_nop 1" : "+v"(x) : : "memory");
        uint64_t u = gl_pack((uint32_t)__shfl((int)(uint32_t)x, l & 12), (uint32_t)__shfl((int)(x >> 32), l & 12));
        int lo = (int)((uint32_t)x ^ 0x80808080u), hi = (int)((uint32_t)(x >> 32) ^ 0x80808080u);
        p2_v4i in[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) in[t] = (p2_v4i){};
#pragma unroll
        for (int s = 0; s < NQ; s++) {
            in[s / 2][s % 2 * 2] = s == 0   ? p2_dpp<0x00>(lo)
                                   : s == 1 ? p2_dpp<0x55>(lo)
                                   : s == 2 ? p2_dpp<0xAA>(lo)
                                            : p2_dpp<0xFF>(lo);
            in[s / 2][s % 2 * 2 + 1] = s == 0   ? p2_dpp<0x00>(hi)
                                       : s == 1 ? p2_dpp<0x55>(hi)
                                       : s == 2 ? p2_dpp<0xAA>(hi)
                                                : p2_dpp<0xFF>(hi);
        }
#pragma unroll
        for (int e = 0; e < P2_SEG; e++) {
            const int s = Op::slot_y(e), tn = s / 2, gn = e == 0 ? 0 : (e - 1) % 4;
            p2_v4i a = {}, b = {};
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (e + 1 < P2_SEG && t < Op::tiles(e) && t != tn) {
                    gl_mac16(a, cur[0][t], in[t]);
                    gl_mac16(b, cur[1][t], in[t]);
                }
            if (e + 1 < P2_SEG) operands(nxt, e + 1);
            p2_loads_first(u);
            uint64_t y = p2_pow7_pair(u);
            in[tn][s % 2 * 2] = g == (uint32_t)gn ? (int)((uint32_t)y ^ 0x80808080u) : in[tn][s % 2 * 2];
            in[tn][s % 2 * 2 + 1] = g == (uint32_t)gn ? (int)((uint32_t)(y >> 32) ^ 0x80808080u) : in[tn][s % 2 * 2 + 1];
            if (e + 1 < P2_SEG) {
                gl_mac16(a, cur[0][tn], in[tn]);
                gl_mac16(b, cur[1][tn], in[tn]);
                u = hz_fold(gl_digit_sums<true>(a, b, k[e][0], k[e][1]));
#pragma unroll
                for (int t = 0; t < NT; t++) cur[0][t] = nxt[0][t], cur[1][t] = nxt[1][t];
            }
        }
        p2_v4i a, b;
#pragma unroll
        for (int w = 0; w < NQ; w++) {
            p2_v4i sa = {}, sb = {};
#pragma unroll
            for (int t = 0; t < NT; t++) cur[0][t] = nxt[0][t], cur[1][t] = nxt[1][t];
            if (w + 1 < NQ) {
                operands(nxt, P2_SEG + w);
                asm volatile("" : : : "memory");
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                gl_mac16(sa, cur[0][t], in[t]);
                gl_mac16(sb, cur[1][t], in[t]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                a[i] = w == 0 || q == (uint32_t)w ? sa[i] : a[i];
                b[i] = w == 0 || q == (uint32_t)w ? sb[i] : b[i];
            }
        }
        return hz_fold(gl_digit_sums<false>(a, b, ks0, ks1));
    }
    // The permutation: word `word` in and out. need_stage (the same for the block, whose
    // threads then all call it): no stage() yet since start().
    __device__ __forceinline__ uint64_t permute(uint64_t x, bool need_stage)
    {
        const uint64_t *k = c_p2_row_addends<W>.ext[0][word];
        x = external(word < (uint32_t)W ? x : 0, k[0], k[1]);
        x = full(x, 0);
        if (need_stage) stage();
#pragma unroll 1
        for (int sg = 0; sg < P2_SEGS; sg++) x = segment(x, sg);
        return full(x, 4);
    }
};

#else  // host pass: declarations only
template <int W> struct p2_row {
    uint32_t g, q, word;
    __device__ void start(p2_v4i *s);
    __device__ void stage();
    __device__ uint64_t permute(uint64_t x, bool need_stage);
};
template <int CTRL> __device__ int p2_dpp(int v);
#endif
