// NTT rounds of four index bits on the matrix cores (included by ntt_kernels.hip).
//
// A round's 16-point transform is a constant 16 x 16 matrix of roots, in bytes and digits
// (gl_digits.h) a 128 x 128 matrix of int8: 16 v_mfma_i32_16x16x64_i8 for the 16 groups of
// a wave. Lane (g, n) = (l / 16, l % 16) holds the values j = g + 4i, i < 4, of group n
// before and after, so a round reads four words a lane, transforms and writes them back
// to the same places. That leaves 12 VALU instructions a word for the transform (putting
// the digits together) instead of the 38 of four butterfly stages, and any 64-bit words
// may come in: only a result that leaves the transform is made canonical.
//
// A round over r < 4 bits takes the matrix with 16 / 2^r blocks: value j stands for index
// j mod 2^r of transform j / 2^r. The first round of a DIT pass and the last one of a DIF
// pass are the short ones; they are the rounds without twiddles.
//
// What bounds the passes (2^22 x 128 columns to 2^24, kernel times before, with the rounds
// on the VALU, and now): block pass 19.3 -> 15.4 ms, strided forward 13.1 -> 11.0 ms,
// strided inverse 3.8 -> 3.2 ms; at 75 columns 2^18 -> 2^20 the forward pass moves 4.4 TB/s of
// the 4.8 that a large copy reaches. VALU instructions fell by 40 percent, the matrix cores
// are 20 percent busy; waiting (LDS, twiddles, barriers) is what is left, so registers are
// held to 128 for four waves a SIMD: with 256 and two waves the same rounds took 16.8,
// 14.3 and 4.1 ms. Each value spilled at 128 is 256 bytes of memory traffic a wave; the
// fences below keep the pieces of an unrolled round apart for that reason. What still
// spills: 6 to 12 registers a line in the block pass of blowup 4, 4 to 8 of blowup 8, and in
// the strided inverse of 2^8 points 8, of the matrix.
#pragma once
#include "gl_digits.h"

namespace nttc {

constexpr uint64_t root16(int r)  // w_{2^r} = 2^(192 / 2^r)
{
    return glc::pow(2, 192 >> r);
}
constexpr int bitrev(int x, int bits)
{
    int y = 0;
    for (int i = 0; i < bits; i++) y |= ((x >> i) & 1) << (bits - 1 - i);
    return y;
}

enum { DIT = 0, DIT_INV = 1, DIF_INV = 2 };  // roots: forward, inverse, inverse

// 2^(-s / 2): 2^24 - 2^72 is a root of 2
constexpr uint64_t kRoot2 = glc::add(1 << 24, GL_P - glc::pow(2, 72));
static_assert(glc::mul(kRoot2, kRoot2) == 2, "root of 2");
constexpr uint64_t half_pow(int s) { return glc::pow(kRoot2, 384 - s); }

// Operand x = 4i + 2h + t of lane 16 kg + row, row = 4g + d: digits 4h + d of out-value
// g + 4i, bytes of in-values kg + 4 (2t) and kg + 4 (2t + 1). All times 2^(-S / 2).
template <int KIND, int R, int S> struct Mat {
    alignas(16) int8_t b[16][64][16];
    constexpr Mat() : b{}
    {
        const uint64_t w = KIND == DIT ? root16(R) : glc::pow(root16(R), (1 << R) - 1);
        const uint64_t scale = half_pow(S);
        const int m = (1 << R) - 1;
        for (int k = 0; k < 16; k++)
            for (int j = 0; j < 16; j++) {
                if (k >> R != j >> R) continue;
                uint64_t c = glc::mul(scale, glc::pow(w, KIND == DIF_INV ? (j & m) * bitrev(k & m, R)
                                                                         : (k & m) * bitrev(j & m, R)));
                for (int a = 0; a < 8; a++, c = glc::mul(c, 256)) {
                    const glc::Digits d(c);
                    const int i = k / 4, g = k % 4, kg = j % 4, t = j / 8, half = j / 4 % 2;
                    for (int x = 0; x < 8; x++) b[4 * i + 2 * (x / 4) + t][16 * kg + 4 * g + x % 4][half * 8 + a] = d.d[x];
                }
            }
    }
};
// The addends: the coefficients of an out-value sum to 2^r times the scale if it is index
// 0 of its transform, else to 0
constexpr glc::Addend kZero(0);
template <int R, int S> constexpr glc::Addend kFirst = glc::Addend(glc::mul(half_pow(S), glc::mul(128 << R, glc::kBytes)));
}  // namespace nttc

template <int KIND, int R, int S> __device__ const nttc::Mat<KIND, R, S> c_ntt_mat{};

// A wave holds MX_PIECES pieces of 16 groups of 16 values: four waves a SIMD with up to
// 128 registers, of which the matrix takes 64.
#define MX_PIECES 4
#define MX_LOG_THREAD 4  // log2 values of a thread

// A wave's place: group n of its pieces, values g + 4i. Piece c has the groups gi + c *
// step, gi < step: their indices have no bits in common, so an address is a lane's part
// for gi plus a scalar part for c.
struct MxLane {
    uint32_t g, gi, first, step;  // first: the wave's gi (scalar)
};

// Shapes of the strided passes and of the block pass (below)
struct MxStrided {
    uint64_t cs;
    uint32_t L1, log_n2, lt, tiles_log, tiles;  // tiles a column, of all columns
};
struct MxBlock {
    uint64_t cs_in, cs_out, ncols;
    uint32_t L1, L2, per;  // per: columns of a block
};

#if defined(__HIP_DEVICE_COMPILE__)

// Every phase derives its own (the compiler is kept from sharing it): lane constants held
// through the whole kernel would not fit beside a matrix.
__device__ __forceinline__ uint32_t mx_lane_id()
{
    uint32_t l = __lane_id();
    asm volatile("" : "+v"(l));
    return l;
}
__device__ __forceinline__ MxLane mx_lane()
{
    const uint32_t l = mx_lane_id(), g = l >> 4;
    uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    return {g, wave * 16 + (l & 15), wave * 16, (blockDim.x >> 6) * 16};
}

// The group's bits gi of a round over index bits [q, q + 4) of a tile with 2^lt lines: the
// tile index of its value 0, and the index bits below the round
__device__ __forceinline__ uint32_t mx_pos(uint32_t gi, uint32_t q, uint32_t lt)
{
    uint32_t rest = gi >> lt;
    return ((((rest >> q) << (q + 4)) | (rest & ((1u << q) - 1))) << lt) | (gi & ((1u << lt) - 1));
}
__device__ __forceinline__ uint32_t mx_low(uint32_t gi, uint32_t q, uint32_t lt) { return (gi >> lt) & ((1u << q) - 1); }

// Words by a scalar base and a 32-bit byte offset
__device__ __forceinline__ uint64_t mx_ld(const uint64_t *b, uint32_t off) { return *(const uint64_t *)((const char *)b + off); }
__device__ __forceinline__ uint64_t mx_ld_nt(const uint64_t *b, uint32_t off)
{
    return __builtin_nontemporal_load((const uint64_t *)((const char *)b + off));
}
__device__ __forceinline__ void mx_st(uint64_t *b, uint32_t off, uint64_t v) { *(uint64_t *)((char *)b + off) = v; }

// Nothing is moved across: unrolled pieces that overlap need more registers than there are
__device__ __forceinline__ void mx_fence()
{
    asm volatile("" : : : "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void mx_sync()
{
    mx_fence();
    __syncthreads();
    mx_fence();
}

// S: by default 2^-R with DIF_INV, 1 otherwise
template <int KIND, int R, int S = (KIND == nttc::DIF_INV ? 2 * R : 0)> struct MxDft {
    gl_v4i a[16];
    uint64_t k0, k1;  // of a lane's values that may be index 0
    __device__ __forceinline__ void load()
    {
        const uint32_t l = mx_lane_id(), off = l * 16;
        const char *m = (const char *)c_ntt_mat<KIND, R, S>.b;
#pragma unroll
        for (int x = 0; x < 16; x++) a[x] = *(const gl_v4i *)(m + off + x * 1024);
        const bool first = R == 1 ? (l & 16) == 0 : l < 16;
        k0 = first ? nttc::kFirst<R, S>.k[0] : nttc::kZero.k[0];
        k1 = first ? nttc::kFirst<R, S>.k[1] : nttc::kZero.k[1];
    }
    // the transform of a lane's four values (any words in and out)
    __device__ __forceinline__ void apply(uint64_t *v) const
    {
        gl_v4i b0, b1;
        gl_put_word(b0, 0, v[0]);
        gl_put_word(b0, 1, v[1]);
        gl_put_word(b1, 0, v[2]);
        gl_put_word(b1, 1, v[3]);
#pragma unroll
        for (int p = 0; p < 2; p++) {
            hz h[2];
#pragma unroll
            for (int o = 0; o < 2; o++) {
                const int i = 2 * p + o;
                gl_v4i x = {}, y = {};
                gl_mac16(x, a[4 * i], b0);
                gl_mac16(y, a[4 * i + 2], b0);
                gl_mac16(x, a[4 * i + 1], b1);
                gl_mac16(y, a[4 * i + 3], b1);
                if (i == 0 || R < 3 || (R == 3 && i == 2))
                    h[o] = gl_digit_sums<false>(x, y, k0, k1);
                else
                    h[o] = gl_digit_sums<true>(x, y, nttc::kZero.k[0], nttc::kZero.k[1]);
            }
            hz_fold2(h, v + 2 * p);
        }
    }
};

__device__ __forceinline__ void mx_mul4(uint64_t *v, const uint64_t *w)
{
    gl_mulk2(v, w, v);
    gl_mulk2(v + 2, w + 2, v + 2);
}
__device__ __forceinline__ void mx_canon4(uint64_t *v)
{
    gl_canon2(v);
    gl_canon2(v + 2);
}

// w[i] = w^(o * bitrev4(g + 4i)), o < 2^q, w of order 2^(q + 4): the round table t has them
// at the values' places, so that a wave reads runs (by exponent, 16 lanes with consecutive
// o read up to 16 lines, and of a table larger than the L1 cache one word of each: block
// pass of 2^22 x 128 to 2^24 16.0 ms instead of 15.4, INTT of 2^21 x 24 405 us instead of 385)
__device__ __forceinline__ void mx_twiddles(uint64_t *w, const uint64_t *t, uint32_t o, uint32_t q, const MxLane &L)
{
    const uint32_t off = 8 * ((L.g << q) | o);
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) w[i] = mx_ld(t + ((4 * i) << q), off);
}

// The same by exponent, from the powers t of w: for the strided passes, whose lanes have few
// different o and whose tables the L1 cache holds; it takes fewer registers
__device__ __forceinline__ void mx_powers(uint64_t *w, const uint64_t *t, uint32_t o, const MxLane &L)
{
    const uint32_t o8 = o * 8, b = __umul24(o8, 4 * ((L.g & 1) * 2 + (L.g >> 1)));
    w[0] = mx_ld(t, b);
    w[1] = mx_ld(t, b + 2 * o8);
    w[2] = mx_ld(t, b + o8);
    w[3] = mx_ld(t, b + 3 * o8);
}

// A round over index bits [q, q + 4) of a tile in LDS: where a lane's values are
struct MxTile {
    uint32_t q, lt, at, s1, s2;  // byte offset of value 0 of piece 0, steps to values 1 and 2
    __device__ __forceinline__ MxTile(uint32_t q_, uint32_t lt_, const MxLane &L) : q(q_), lt(lt_)
    {
        at = 8 * lds_addr(mx_pos(L.gi, q, lt) | (L.g << (q + lt)));
        s1 = 8 * lds_addr(4u << (q + lt));
        s2 = 8 * lds_addr(8u << (q + lt));
    }
    __device__ __forceinline__ uint32_t piece(uint32_t c, const MxLane &L) const
    {
        return at + 8 * lds_addr(mx_pos(c * L.step, q, lt));
    }
    __device__ __forceinline__ uint32_t low(uint32_t c, const MxLane &L) const
    {
        return mx_low(L.gi, q, lt) + mx_low(c * L.step, q, lt);
    }
    __device__ __forceinline__ void read(uint64_t *v, const uint64_t *s, uint32_t a) const
    {
        v[0] = mx_ld(s, a);
        v[1] = mx_ld(s, a + s1);
        v[2] = mx_ld(s, a + s2);
        v[3] = mx_ld(s, a + s1 + s2);
    }
    __device__ __forceinline__ void write(uint64_t *s, uint32_t a, const uint64_t *v) const
    {
        mx_st(s, a, v[0]);
        mx_st(s, a + s1, v[1]);
        mx_st(s, a + s2, v[2]);
        mx_st(s, a + s1 + s2, v[3]);
    }
};

// A full round in LDS (t: its table of 2^(q + 4) words, by place or by exponent): DIT twiddles before
// the transform, DIF after it.
template <int PIECES, bool PLACE = true, int KIND, int S>
__device__ __forceinline__ void mx_round(uint64_t *__restrict__ s, const MxDft<KIND, 4, S> &d, uint32_t q, uint32_t lt,
                                         const uint64_t *t)
{
    const MxLane L = mx_lane();
    const MxTile T(q, lt, L);
#pragma unroll 1
    for (uint32_t c = 0; c < PIECES; c++) {
        uint64_t v[4], w[4];
        const uint32_t a = T.piece(c, L);
        T.read(v, s, a);
        if (PLACE)
            mx_twiddles(w, t, T.low(c, L), q, L);
        else
            mx_powers(w, t, T.low(c, L), L);
        if (KIND != nttc::DIF_INV) mx_mul4(v, w);
        d.apply(v);
        if (KIND == nttc::DIF_INV) mx_mul4(v, w);
        T.write(s, a, v);
    }
}

// ------------------------------------------------------ strided passes ----
// As k_ntt_strided_inv and k_ntt_strided_fwd for one launch of L1 = 4 .. 10 bits of m: the
// first round reads global memory and the last one writes it, both in runs of 2^lt words,
// the rounds between them are in LDS. The short round of L1 % 4 bits is on the VALU: about
// the instructions a word of a matrix round, without a second matrix to read (2^18 x 75
// forward, two bits: 313 us with a matrix, 292 without). L1 = 4: one round and no LDS; a
// block keeps its matrix and works on every gridDim.x-th tile of all columns.
__device__ __forceinline__ uint64_t *mx_tile(uint64_t *data, const MxStrided &p, uint32_t tile)
{
    const uint32_t bx = tile & ((1u << p.tiles_log) - 1);
    return data + (uint64_t)(tile >> p.tiles_log) * p.cs + ((uint64_t)bx << p.lt);
}

// A lane's words of a round's values in a tile of global memory: byte offset of the lane's
// part of tile index x, scalar base of the other part
__device__ __forceinline__ uint32_t mx_goff(uint32_t x, const MxStrided &p)
{
    return (((x >> p.lt) << p.log_n2) + (x & ((1u << p.lt) - 1))) * 8;
}
__device__ __forceinline__ uint64_t *mx_gbase(uint64_t *col, uint32_t x, const MxStrided &p)
{
    return col + (((uint64_t)(x >> p.lt) << p.log_n2) + (x & ((1u << p.lt) - 1)));
}

// Short round: thread t has the groups j < 16 >> R of 2^R neighbouring m: tile index of
// value 0, the thread's part (t < blockDim.x) or the scalar part (t = j blockDim.x)
template <int R> __device__ __forceinline__ uint32_t mx_short(uint32_t t, uint32_t lt)
{
    return ((t >> lt) << (lt + R)) | (t & ((1u << lt) - 1));
}
__device__ __forceinline__ uint32_t mx_thread()
{
    return __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u) + mx_lane_id();
}

// Root e of the split tables
__device__ __forceinline__ uint64_t mx_split_root(const uint64_t *tl, const uint64_t *th, uint32_t e, const NttTables &tb)
{
    return gl_mul_nc(mx_ld(tl, tw_lo(e, tb) * 8), mx_ld(th, tw_hi(e, tb) * 8));
}

// iNTT pass 1, times 2^-L1, L1 = 4 (NR - 1) + R. The short round is the last one (no
// twiddles in it); results take w_N^-(line * bitrev(m)). A lane's m of a step differ in
// bits that are the same in every step and its line stays the same, so it takes one
// root a step and the ratios to the others once a tile from the split tables (random 8-byte
// reads of 32 KB tables). Two reads for every word: 4.1 ms for 2^22 x 128 instead of 3.4. (L1 = 4:
// m stays the same and the lines grow by a constant, and so the roots by a factor.)
template <int L1>
__global__ __launch_bounds__(1024, 4) void k_ntt_strided_inv_mx(uint64_t *__restrict__ data, MxStrided p, NttTables tb)
{
    extern __shared__ uint64_t s[];
    constexpr int NR = (L1 + 3) / 4, R = L1 - 4 * (NR - 1);
    constexpr uint32_t top = L1 - 4;
    constexpr int FULL = R == 4 ? NR : NR - 1;  // rounds with a matrix, which share the scale
    static_assert(2 * L1 % FULL == 0, "scale");
    const uint32_t lt = p.lt, shift_n = 2 * tb.bits - (L1 + p.log_n2);
    MxDft<nttc::DIF_INV, 4, 2 * L1 / FULL> d;
    if (NR == 1) d.load();
    uint32_t tile = blockIdx.x;
    do {
        uint64_t *col = mx_tile(data, p, tile);
        const uint32_t line_t = (uint32_t)((col - data) & ((1ull << p.log_n2) - 1));
        if constexpr (NR > 1) {
            const MxLane L = mx_lane();
            uint64_t v[2][4];
            const uint32_t off = mx_goff(mx_pos(L.gi, top, lt) | (L.g << (top + lt)), p);
            auto load = [&](uint32_t c) {
#pragma unroll
                for (uint32_t i = 0; i < 4; i++)
                    v[c & 1][i] = mx_ld_nt(mx_gbase(col, mx_pos(c * L.step, top, lt) | ((4 * i) << (top + lt)), p), off);
                mx_fence();
            };
            d.load();
            mx_fence();
            load(0);
            load(1);
            const MxTile F(top, lt, L);
#pragma unroll
            for (uint32_t c = 0; c < MX_PIECES; c++) {
                uint64_t w[4], *x = v[c & 1];
                d.apply(x);
                mx_fence();
                mx_powers(w, tb.tki + (1u << L1), F.low(c, L), L);
                mx_mul4(x, w);
                F.write(s, F.piece(c, L), x);
                mx_fence();
                if (c + 2 < MX_PIECES) load(c + 2);
            }
            mx_sync();
            if constexpr (NR == 3) {
                mx_round<MX_PIECES, false>(s, d, top - 4, lt, tb.tki + (1u << top));
                mx_sync();
            }
        }
        // a step's N values: tile index x0 | xc | (i D << lt), m = (x0 | xc) >> lt | i D
        constexpr uint32_t N = R == 4 ? 4 : 1 << R, D = R == 4 ? 4 : 1;
        const MxLane L = mx_lane();
        const uint32_t x0 = R == 4 ? mx_pos(L.gi, 0, lt) | (L.g << lt) : mx_short<R>(mx_thread(), lt);
        const uint32_t line = line_t + (x0 & ((1u << lt) - 1)), br0 = bitrev32(x0 >> lt, L1), at = mx_goff(x0, p);
        uint64_t ratio[N], w[N];
#pragma unroll
        for (uint32_t i = L1 == 4 ? 0 : 1; i < N; i++) {
            if (L1 == 4) w[i] = mx_split_root(tb.twl_i, tb.twh_i, (line * (br0 + bitrev32(i * D, L1))) << shift_n, tb);
            const uint32_t e = L1 == 4 ? L.step * (br0 + bitrev32(i * D, L1)) : line * bitrev32(i * D, L1);
            ratio[i] = mx_split_root(tb.twl_i, tb.twh_i, e << shift_n, tb);
        }
#pragma unroll 1
        for (uint32_t c = 0; c < 16 / N; c++) {
            const uint32_t xc = R == 4 ? mx_pos(c * L.step, 0, lt) : mx_short<R>(c * blockDim.x, lt);
            uint64_t v[N];
            if (L1 > 4) w[0] = mx_split_root(tb.twl_i, tb.twh_i, (line * (br0 + bitrev32(xc >> lt, L1))) << shift_n, tb);
#pragma unroll
            for (uint32_t i = 0; i < N; i++)
                v[i] = NR == 1 ? mx_ld_nt(mx_gbase(col, xc | ((i * D) << lt), p), at)
                               : mx_ld(s, 8 * (lds_addr(x0) + lds_addr(xc) + lds_addr((i * D) << lt)));
            if constexpr (R == 4) {
                d.apply(v);
            } else {
#pragma unroll
                for (uint32_t i = 0; i < N; i += 2) gl_canon2(v + i);
                dft_dif<N, true>(v);
            }
            if (L1 > 4) {
#pragma unroll
                for (uint32_t i = 1; i < N; i++) w[i] = gl_mul_nc(w[0], ratio[i]);
            }
#pragma unroll
            for (uint32_t i = 0; i < N; i += 2) {
                gl_mulk2(v + i, w + i, v + i);
                if (L1 == 4) gl_mulk2(w + i, ratio + i, w + i);
            }
#pragma unroll
            for (uint32_t i = 0; i < N; i++) mx_st(mx_gbase(col, xc | ((i * D) << lt), p), at, v[i]);
        }
    } while (NR == 1 && (tile += gridDim.x) < p.tiles);
}

// NTT pass 3. The short round is the first one; the result is canonical.
template <bool INV, int L1>
__global__ __launch_bounds__(1024, 4) void k_ntt_strided_fwd_mx(uint64_t *__restrict__ data, MxStrided p, NttTables tb)
{
    extern __shared__ uint64_t s[];
    constexpr int KIND = INV ? nttc::DIT_INV : nttc::DIT, NR = (L1 + 3) / 4, R = L1 - 4 * (NR - 1);
    constexpr uint32_t q = L1 - 4;
    const uint32_t lt = p.lt;
    const uint64_t *tk = INV ? tb.dti : tb.dtf;
    MxDft<KIND, 4> d;
    if (R == 4) d.load();
    uint32_t tile = blockIdx.x;
    do {
        uint64_t *col = mx_tile(data, p, tile);
        if constexpr (R == 4) {
            const MxLane L = mx_lane();
            const uint32_t x0 = mx_pos(L.gi, 0, lt) | (L.g << lt), off = mx_goff(x0, p), a0 = 8 * lds_addr(x0);
            uint64_t v[2][4];
            auto load = [&](uint32_t c) {
#pragma unroll
                for (uint32_t i = 0; i < 4; i++)
                    v[c & 1][i] = mx_ld(mx_gbase(col, mx_pos(c * L.step, 0, lt) | ((4 * i) << lt), p), off);
                mx_fence();
            };
            load(0);
            load(1);
#pragma unroll
            for (uint32_t c = 0; c < MX_PIECES; c++) {
                const uint32_t xc = mx_pos(c * L.step, 0, lt);
                uint64_t *x = v[c & 1];
                d.apply(x);
                if (NR == 1) mx_canon4(x);
#pragma unroll
                for (uint32_t i = 0; i < 4; i++)
                    if (NR > 1)
                        mx_st(s, a0 + 8 * lds_addr(xc) + 8 * lds_addr((4 * i) << lt), x[i]);
                    else
                        mx_st(mx_gbase(col, xc | ((4 * i) << lt), p), off, x[i]);
                mx_fence();
                if (c + 2 < MX_PIECES) load(c + 2);
            }
        } else {
            constexpr uint32_t N = 1 << R;
            const uint32_t x0 = mx_short<R>(mx_thread(), lt), off = mx_goff(x0, p), a0 = 8 * lds_addr(x0);
            uint64_t v[16 / N][N];
#pragma unroll
            for (uint32_t j = 0; j < 16 / N; j++)
#pragma unroll
                for (uint32_t i = 0; i < N; i++)
                    v[j][i] = mx_ld(mx_gbase(col, mx_short<R>(j * blockDim.x, lt) | (i << lt), p), off);
#pragma unroll
            for (uint32_t j = 0; j < 16 / N; j++) {
                const uint32_t xc = mx_short<R>(j * blockDim.x, lt);
#pragma unroll
                for (uint32_t i = 0; i < N; i += 2) gl_canon2(v[j] + i);
                dft_dit<N, INV>(v[j]);
#pragma unroll
                for (uint32_t i = 0; i < N; i++) mx_st(s, a0 + 8 * lds_addr(xc) + 8 * lds_addr(i << lt), v[j][i]);
                mx_fence();
            }
            mx_fence();
            d.load();
        }
        if constexpr (NR > 1) {
            mx_sync();
            if constexpr (NR == 3) {
                mx_round<MX_PIECES>(s, d, R, lt, tk + (1u << (R + 4)));
                mx_sync();
            }
            const MxLane L = mx_lane();
            const MxTile T(q, lt, L);
            const uint32_t off = mx_goff(mx_pos(L.gi, q, lt) | (L.g << (q + lt)), p);
#pragma unroll 1
            for (uint32_t c = 0; c < MX_PIECES; c++) {
                uint64_t v[4], w[4];
                T.read(v, s, T.piece(c, L));
                mx_twiddles(w, tk + (1u << L1), T.low(c, L), q, L);
                mx_mul4(v, w);
                d.apply(v);
                mx_canon4(v);
                const uint32_t xc = mx_pos(c * L.step, q, lt);
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) mx_st(mx_gbase(col, xc | ((4 * i) << (q + lt)), p), off, v[i]);
            }
        }
    } while (NR == 1 && (tile += gridDim.x) < p.tiles);
}

// ----------------------------------------------------------- block pass ----
// As k_lde_block for 2^L2 coefficients a line (L2 >= 8), blowup 2^LOGB <= 8, n2 * B / 16
// threads. Phase 1 has TP pieces a wave over LINES lines of the column's line m (blowups 4
// and 8 take two columns, so that every wave has work between two barriers); its results
// stay in registers until every wave has read its last round's values, then a line's go to
// the places of the spread array where copy 0 stands. The first round of phase 2 reads
// copy 0 for every copy: the copies of a coefficient are neighbouring groups of one piece,
// so they are read before the same wave writes them. COEF_IN: the line holds coefficients
// already; INV: inverse roots in phase 2.

// The last round of phase 1 (2^R points, no twiddles), scaled by 7^e, e = bitrev(m 2^L2 +
// k); kept in `held`, or (IN_PLACE) written back. A lane's four k differ in the same two
// bits in every piece, so it takes one power a piece and the ratios once.
template <int R, int TP, bool IN_PLACE, bool PARTIAL>
__device__ __forceinline__ void mx_block_coef(uint64_t *__restrict__ s, const MxDft<nttc::DIF_INV, R> &d,
                                              uint64_t (&held)[TP][4], uint32_t m, uint32_t L2, uint32_t log_n,
                                              uint32_t end, const NttTables &tb)
{
    const MxLane L = mx_lane();
    const MxTile T(0, 0, L);
    const uint32_t mask = (1u << L2) - 1, k0 = mx_pos(L.gi, 0, 0) | L.g;
    const uint32_t e0 = bitrev32((m << L2) | (k0 & mask), log_n);
    uint64_t ratio[4];  // of k + 4i: scalar
#pragma unroll
    for (uint32_t i = 1; i < 4; i++) ratio[i] = mx_split_root(tb.shl, tb.shh, bitrev32(4 * i, log_n), tb);
#pragma unroll
    for (uint32_t c = 0; c < TP; c++) {
        if (PARTIAL && L.first + c * L.step >= end) break;
        uint64_t v[4], w[4];
        w[0] = mx_split_root(tb.shl, tb.shh, e0 + bitrev32(mx_pos(c * L.step, 0, 0) & mask, log_n), tb);
        T.read(v, s, T.piece(c, L));
        d.apply(v);
        mx_fence();
#pragma unroll
        for (uint32_t i = 1; i < 4; i++) w[i] = gl_mul_nc(w[0], ratio[i]);
        mx_mul4(v, w);
        if constexpr (IN_PLACE) {
            T.write(s, T.piece(c, L), v);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) held[c][i] = v[i];
        }
        mx_fence();
    }
}

// The first round of phase 2: 2^R points at bits [LOGB, LOGB + R) of the spread array. The
// lane's group is (coefficients gi >> LOGB, copy gi mod 2^LOGB).
template <int KIND, int R, int LOGB>
__device__ __forceinline__ void mx_block_spread(uint64_t *__restrict__ s, const MxDft<KIND, R> &d, const NttTables &tb)
{
    const MxLane L = mx_lane();
    const MxTile T(LOGB, 0, L);
    const uint32_t o = L.gi & ((1u << LOGB) - 1), copy0 = 8 * lds_addr(o);
    uint64_t w[4];
    if (LOGB > 0) {  // copy o: w_{2^(LOGB + R)}^(o bitrev(j)), the same for every piece
        const uint64_t *t = (KIND == nttc::DIT ? tb.tkf : tb.tki) + (1u << (LOGB + R));
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) w[i] = t[o * bitrev32((L.g + 4 * i) & ((1u << R) - 1), R)];
    }
#pragma unroll 1
    for (uint32_t c = 0; c < MX_PIECES; c++) {
        uint64_t v[4];
        const uint32_t a = T.piece(c, L);
        T.read(v, s, a - copy0);
        if (LOGB > 0) mx_mul4(v, w);
        d.apply(v);
        T.write(s, a, v);
    }
}

// The same for R <= 2 on the VALU: a lane has groups of all 2^R values, and the block reads
// one matrix less (2^18 x 75 to 2^20: block pass 537 -> 511 us). COEF_IN: they are read from
// global memory (each copy reads them), not from where copy 0 stands, which saves a barrier;
// with a matrix that would be reads of 32 bytes (2^15 x 50 NTT: 21.8 us instead of 17.7).
template <bool INV, int R, int LOGB, bool COEF_IN>
__device__ __forceinline__ void mx_block_spread_short(uint64_t *__restrict__ s, const uint64_t *__restrict__ src,
                                                      const NttTables &tb)
{
    constexpr uint32_t N = 1 << R;
    const uint32_t t = mx_thread(), o = t & ((1u << LOGB) - 1), grp = t >> LOGB;
    const uint32_t at = 8 * lds_addr(grp << (R + LOGB)), copy = 8 * lds_addr(o);
    uint64_t w[N];
    if (LOGB > 0) {
        const uint64_t *tk = (INV ? tb.tki : tb.tkf) + (1u << (LOGB + R));
#pragma unroll
        for (uint32_t i = 1; i < N; i++) w[i] = tk[o * bitrev32(i, R)];
    }
    uint64_t v[16 / N][N];
#pragma unroll
    for (uint32_t j = 0; j < 16 / N; j++) {
        const uint32_t gj = (j * blockDim.x) >> LOGB;
#pragma unroll
        for (uint32_t i = 0; i < N; i++)
            v[j][i] = COEF_IN ? mx_ld(src + (gj << R) + i, (grp << R) * 8)
                              : mx_ld(s, at + 8 * (lds_addr(gj << (R + LOGB)) + lds_addr(i << LOGB)));
    }
    mx_fence();
#pragma unroll
    for (uint32_t j = 0; j < 16 / N; j++) {
        const uint32_t gj = (j * blockDim.x) >> LOGB;
        if (LOGB > 0) {
            v[j][0] = gl_canon(v[j][0]);
            gl_mul_v<N - 1>(v[j] + 1, v[j] + 1, w + 1);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < N; i += 2) gl_canon2(v[j] + i);
        }
        dft_dit<N, INV>(v[j]);
#pragma unroll
        for (uint32_t i = 0; i < N; i++)
            mx_st(s, at + copy + 8 * (lds_addr(gj << (R + LOGB)) + lds_addr(i << LOGB)), v[j][i]);
        mx_fence();
    }
}

template <bool COEF_IN, bool INV, int LOGB, int R>
__global__ __launch_bounds__(1024, 4) void k_lde_block_mx(const uint64_t *__restrict__ in, uint64_t *__restrict__ out,
                                                          MxBlock p, NttTables tb)
{
    extern __shared__ uint64_t s[];
    constexpr int KIND = INV ? nttc::DIT_INV : nttc::DIT;
    constexpr int LINES = !COEF_IN && LOGB >= 2 ? 2 : 1;
    constexpr int TP = COEF_IN ? 1 : (MX_PIECES * LINES) >> LOGB;
    const uint32_t L1 = p.L1, L2 = p.L2, log_n = L1 + L2, top = L2 + LOGB;
    const uint32_t per_line = 1u << (L2 - 4);  // groups of a line
    // the wave's first group and the distance of its pieces
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 16, step = blockDim.x / 4;
    const uint32_t m = blockIdx.x;
    const uint64_t c0 = (uint64_t)blockIdx.y * p.per;
    const uint32_t lines = LINES == 2 && p.per == 2 && c0 + 1 < p.ncols ? 2 : 1;  // an odd last column is alone
    const uint64_t *src = in + c0 * p.cs_in + ((uint64_t)m << L2);
    uint64_t held[TP][4];
    if constexpr (COEF_IN && R >= 3) {
        constexpr uint32_t N = (1u << MX_LOG_THREAD) >> LOGB;
        uint64_t x[N];
#pragma unroll
        for (uint32_t i = 0; i < N; i++) x[i] = __builtin_nontemporal_load(&src[threadIdx.x + i * blockDim.x]);
#pragma unroll
        for (uint32_t i = 0; i < N; i++) s[lds_addr((threadIdx.x + i * blockDim.x) << LOGB)] = x[i];
        mx_sync();
    } else if constexpr (!COEF_IN) {
        const uint32_t q = L2 - 4, end = lines * per_line;
        const bool busy = LOGB < 2 || first < end;  // (without pairs every piece has a line)
        const MxLane L = mx_lane();
        const MxTile T(q, 0, L);  // (the line is the group's bits above the round's)
        MxDft<nttc::DIF_INV, 4> D;
        if (busy) {
            D.load();
            mx_fence();
            // a wave's 16 groups are of one line
            const uint32_t off = ((L.g << q) | mx_low(L.gi, q, 0)) * 8;
            const uint64_t *line = src + (first >> q) * p.cs_in;
            auto load = [&](uint32_t c) {
                if (LOGB >= 2 && first + c * step >= end) return;
                const uint64_t *b = line + ((c * L.step) >> q) * p.cs_in + mx_low(c * L.step, q, 0);
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) held[c][i] = mx_ld_nt(b + ((4 * i) << q), off);
                mx_fence();
            };
            load(0);
            if (TP > 1) load(1);
#pragma unroll
            for (uint32_t c = 0; c < TP; c++) {
                if (LOGB >= 2 && first + c * step >= end) break;
                uint64_t w[4];
                D.apply(held[c]);
                mx_fence();
                mx_twiddles(w, tb.dti + (1u << L2), T.low(c, L), q, L);
                mx_mul4(held[c], w);
                T.write(s, T.piece(c, L), held[c]);
                mx_fence();
                if (c + 2 < TP) load(c + 2);
            }
        }
        mx_sync();
        for (uint32_t qk = q; qk >= 4 + R;) {
            qk -= 4;
            if (busy) {
                if (LINES == 1 || TP == 1 || first + (TP - 1) * step < end)
                    mx_round<TP>(s, D, qk, 0, tb.dti + (1u << (qk + 4)));
                else
                    mx_round<(TP + 1) / 2>(s, D, qk, 0, tb.dti + (1u << (qk + 4)));
            }
            mx_sync();
        }
        if (busy) {
            MxDft<nttc::DIF_INV, R> e;
            if constexpr (R == 4)
                e = D;
            else
                e.load();
            mx_block_coef<R, TP, LOGB == 0, (LOGB >= 2)>(s, e, held, m, L2, log_n, end, tb);
        }
        mx_sync();
    }
    const uint32_t e1 = bitrev32(m, L1), shift_e = 2 * tb.bits - (log_n + LOGB);
    const uint64_t *tl = INV ? tb.twl_i : tb.twl_f, *th = INV ? tb.twh_i : tb.twh_f;
    const uint64_t *tk = INV ? tb.dti : tb.dtf;
#pragma unroll 1
    for (uint32_t l = 0; l < lines; l++) {
        if constexpr (!COEF_IN && LOGB > 0) {
            if (l) mx_sync();  // the values that the coefficients replace have been read
            const MxLane L = mx_lane();
            constexpr uint32_t HELD = LINES == 2 && TP > 1 ? TP / 2 : TP;  // of one line
#pragma unroll
            for (uint32_t c = 0; c < HELD; c++) {
                const uint32_t gr = first + (l * (TP - HELD) + c) * step;
                if (gr >> (L2 - 4) != l) continue;
                // coefficient position k of the line at k 2^LOGB
                const uint32_t k = (((gr & (per_line - 1)) + (L.gi & 15)) << 4) | L.g;
                const uint32_t a = 8 * lds_addr(k << LOGB);
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) mx_st(s, a + 8 * lds_addr((4 * i) << LOGB), held[c][i]);
            }
            if constexpr (HELD < TP) {
#pragma unroll
                for (uint32_t c = 0; c < HELD; c++)
#pragma unroll
                    for (uint32_t i = 0; i < 4; i++) held[c][i] = held[c + HELD][i];
            }
            mx_sync();
        }
        MxDft<KIND, 4> F;
        if constexpr (R <= 2) {
            mx_block_spread_short<INV, R, LOGB, COEF_IN>(s, src, tb);
            F.load();
        } else if constexpr (R == 3) {
            MxDft<KIND, R> e;
            e.load();
            mx_block_spread<KIND, R, LOGB>(s, e, tb);
            F.load();
        } else {
            F.load();
            mx_block_spread<KIND, R, LOGB>(s, F, tb);
        }
        mx_sync();
        uint32_t q = LOGB + R;
        for (; q + 4 < top; q += 4) {
            mx_round<MX_PIECES>(s, F, q, 0, tk + (1u << (q + 4)));
            mx_sync();
        }
        // last round: position P = (g + 4i) 2^q + o of line m times w_NExt^(e1 P). From piece
        // to piece o grows by `step`, and the factors by the same power of w.
        const MxLane L = mx_lane();
        uint64_t *dst = out + (c0 + l) * p.cs_out + ((uint64_t)m << top);
        uint64_t tw[4], ws[2];
        if (L1) {
            uint64_t hi[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t e = (e1 * (((L.g + 4 * i) << q) + L.gi)) << shift_e;
                tw[i] = tl[tw_lo(e, tb)];
                hi[i] = th[tw_hi(e, tb)];
            }
            mx_mul4(tw, hi);
            const uint32_t e = (e1 * L.step) << shift_e;
            ws[0] = ws[1] = gl_mul_nc(tl[tw_lo(e, tb)], th[tw_hi(e, tb)]);
        }
        const MxTile T(q, 0, L);
        const uint32_t off = ((L.g << q) | L.gi) * 8;
#pragma unroll 1
        for (uint32_t c = 0; c < MX_PIECES; c++) {
            uint64_t v[4], w[4];
            T.read(v, s, T.piece(c, L));
            mx_twiddles(w, tk + (1u << top), T.low(c, L), q, L);
            mx_mul4(v, w);
            F.apply(v);
            if (L1) {  // the strided pass takes any words
                mx_mul4(v, tw);
                gl_mulk2(tw, ws, tw);
                gl_mulk2(tw + 2, ws, tw + 2);
            } else {
                mx_canon4(v);
            }
#pragma unroll
            for (uint32_t i = 0; i < 4; i++)
                __builtin_nontemporal_store(v[i], (uint64_t *)((char *)(dst + c * L.step + ((4 * i) << q)) + off));
        }
    }
}

#else  // host pass: only the launch stubs
template <int L1> __global__ void k_ntt_strided_inv_mx(uint64_t *, MxStrided, NttTables) {}
template <bool INV, int L1> __global__ void k_ntt_strided_fwd_mx(uint64_t *, MxStrided, NttTables) {}
template <bool COEF_IN, bool INV, int LOGB, int R>
__global__ void k_lde_block_mx(const uint64_t *, uint64_t *, MxBlock, NttTables)
{
}
#endif
