// FRI fold and FRI-layer regrouping kernels for gfx950.
//
// k_fri_fold restates FRI::fold (pil2-stark/src/starkpil/fri/fri.hpp:32-99) with
// polMulAxi (:178-186) and evalPol (:189-206): for each folded index g in
// [0, 2^cur), gather the nX = 2^(prev-cur) cubic values pol[i*2^cur + g], the values
// of a polynomial of degree below nX at the points w_nX^i / sinv_g with
// sinv_g = (7^(2^(nBitsExt-prev)) * w_{2^prev}^g)^-1, and evaluate it at the challenge.
//
// k_fri_transpose restates getTransposed (fri.hpp:209-226): aux[i*h + j] =
// pol[j*w + i] for w = 2^nextBits, h = 2^cur / w (elements of 3 words).
#include "gl_field.h"
#include "fri_kernels.h"
#include "ntt_kernels.h"

// lanes of a fold that still takes several a group: two waves on each of 1,024 SIMDs
#define FRI_LANES_MAX (1ull << 17)

// w^-e for the roots of one split table pair (lo[e mod 2^bits] * hi[e >> bits]);
// e is a coset index already scaled to the tables' domain. Without tables
// (lo == nullptr), w_inv^e0 by squaring and multiplying.
struct RootTab {
    const uint64_t *lo, *hi;
    uint32_t bits, shift;  // e = e0 << shift
};
__device__ __forceinline__ uint64_t root_pow(const RootTab &t, uint64_t w_inv, uint64_t e0)
{
    if (t.lo) {
        uint64_t e = e0 << t.shift;
        return gl_mul(t.lo[e & ((1ull << t.bits) - 1)], t.hi[e >> t.bits]);
    }
    return gl_pow(w_inv, e0);
}

// A cubic factor with the sums that its Karatsuba products share
struct Gl3Factor {
    uint64_t v[3], s[3];  // v0 + v1, v0 + v2, v1 + v2
};
__device__ __forceinline__ Gl3Factor gl3_factor(const uint64_t *v)
{
    Gl3Factor f;
    const uint64_t a[3] = {v[0], v[0], v[1]}, b[3] = {v[1], v[2], v[2]};
#pragma unroll
    for (int k = 0; k < 3; k++) f.v[k] = v[k];
    gl_add_v<3>(f.s, a, b);
    return f;
}

// out = add + d * x in the cubic extension (the product of gl3_mul), three lanes a step
__device__ __forceinline__ void gl3_mul_add(uint64_t *out, const uint64_t *d, const Gl3Factor &x, const uint64_t *add)
{
    uint64_t m[6], n[6];
    const uint64_t a[3] = {d[0], d[0], d[1]}, b[3] = {d[1], d[2], d[2]};
    gl_add_v<3>(m, a, b);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        m[3 + k] = d[k];
        n[k] = x.s[k];
        n[3 + k] = x.v[k];
    }
    gl_mul_v<6>(m, m, n);  // A, B, C, D, E, F of gl3_mul
    const uint64_t G = gl_sub(m[3], m[4]), H = gl_add(m[3], m[4]);
    const uint64_t p[3] = {m[2], m[0], m[1]}, q[3] = {G, m[2], m[4]}, r[3] = {m[5], m[4], m[3]};
    uint64_t t[3], u[3] = {add[0], gl_sub(add[1], H), add[2]};
    gl_add_v<3>(t, p, q);  // C + D - E, A + C, B + E
    gl_sub_v<3>(t, t, r);  // ... - F, - E (and D + E with add), - D
    gl_add_v<3>(out, t, u);
}

// The fold of a group from its NX = 2^LOGX cubic values a[k][i] (component k of
// pol[i*2^cur + g], canonical) is p(x), p the interpolant of the values at the points
// z_i = z w_NX^i, z = 1 / sinv. It halves the points at each step: with p(z) =
// e(z^2) + z o(z^2), the polynomial q(z^2) = e + x o has q(x^2) = p(x), and its value
// at z_i^2 is (v_i + v_{i+h}) / 2 + (x / z_i) (v_i - v_{i+h}) / 2, h = NX / 2. The
// halves are left to one factor 1/NX at the end, and the powers of w_NX in 1 / z_i are
// powers of two (w_32 = 2^6). That is NX - 1 cubic products against an inverse DFT, the
// scaling of its coefficients and NX - 1 products one after another by Horner (ratio 16:
// 29 -> 9 us for the latency of one group).
template <int LOGX, int T, int I>
__device__ __forceinline__ void fold_pairs(uint64_t (&a)[3][1 << LOGX], const Gl3Factor &x)
{
    constexpr int H = 1 << (LOGX - 1 - T);
    if constexpr (I < H) {
        uint64_t u[3], v[3], d[3], sum[3];
#pragma unroll
        for (int k = 0; k < 3; k++) u[k] = a[k][I], v[k] = a[k][I + H];
        gl_add_v<3>(sum, u, v);
        if constexpr (I == 0) {
            gl_sub_v<3>(d, u, v);
        } else {  // w_2H^-I = -2^(96 - 96 I / H)
            constexpr int S = 96 - 96 / H * I;
            gl_sub_v<3>(d, v, u);
            gl_mul_pow2_3<S, S, S>(d, d);
        }
        gl3_mul_add(d, d, x, sum);
#pragma unroll
        for (int k = 0; k < 3; k++) a[k][I] = d[k];
        fold_pairs<LOGX, T, I + 1>(a, x);
    }
}
template <int LOGX, int T>
__device__ __forceinline__ void fold_halves(uint64_t (&a)[3][1 << LOGX], const Gl3Factor &x)
{
    fold_pairs<LOGX, T, 0>(a, x);
    if constexpr (T + 1 < LOGX) {
        const uint64_t zero[3] = {0, 0, 0};
        uint64_t sq[3];
        gl3_mul_add(sq, x.v, x, zero);
        fold_halves<LOGX, T + 1>(a, gl3_factor(sq));
    }
}

template <int LOGX>
__device__ __forceinline__ gl3 fold_group(uint64_t (&a)[3][1 << LOGX], uint64_t sinv, gl3 x, uint64_t nx_inv)
{
    const uint64_t s[3] = {sinv, sinv, sinv}, n[3] = {nx_inv, nx_inv, nx_inv};
    uint64_t xs[3];
    gl_mul_v<3>(xs, x.v, s);
    fold_halves<LOGX, 0>(a, gl3_factor(xs));
    const uint64_t c[3] = {a[0][0], a[1][0], a[2][0]};
    gl3 r;
    gl_mul_v<3>(r.v, c, n);
    return r;
}

// The same fold on NX / 2 lanes, lane i of them (lanes i and i + j are j * stride apart)
// with u = value i and v = value i + NX / 2: every lane halves its pair, then lanes h
// apart exchange. Twice the products and shorter by the NX - 1 of them in a row; every
// lane of the group ends with the result.
template <int LOGX>
__device__ __forceinline__ gl3 fold_group_lanes(const uint64_t *u0, const uint64_t *v0, uint32_t i, uint32_t stride,
                                                uint64_t sinv, gl3 x, uint64_t nx_inv)
{
    const uint64_t s[3] = {sinv, sinv, sinv}, n[3] = {nx_inv, nx_inv, nx_inv};
    uint64_t u[3] = {u0[0], u0[1], u0[2]}, v[3] = {v0[0], v0[1], v0[2]}, xs[3], q[3];
    gl_mul_v<3>(xs, x.v, s);
    Gl3Factor f = gl3_factor(xs);
#pragma unroll
    for (int t = 0; t < LOGX; t++) {
        const uint32_t h = 1u << (LOGX - 1 - t), j = i & (h - 1), e = 96 - 96 / h * j;
        // w_2h^-j
        const uint64_t pw = e < 64 ? 1ull << e : GL_EPS << (e - 64), w = j ? GL_P - pw : 1;
        const uint64_t ws[3] = {w, w, w};
        uint64_t d[3], sum[3];
        gl_add_v<3>(sum, u, v);
        gl_sub_v<3>(d, u, v);
        gl_mul_v<3>(d, d, ws);
        gl3_mul_add(q, d, f, sum);
        if (t + 1 < LOGX) {
            const bool up = i & (h >> 1);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                uint64_t o = __shfl_xor((unsigned long long)q[k], (int)((h >> 1) * stride));
                u[k] = up ? o : q[k];
                v[k] = up ? q[k] : o;
            }
            const uint64_t zero[3] = {0, 0, 0};
            gl3_mul_add(xs, f.v, f, zero);
            f = gl3_factor(xs);
        }
    }
    gl3 r;
    gl_mul_v<3>(r.v, q, n);
    return r;
}

// Loads group g's values pol[i*n2 + g], i < 2^LOGX.
template <int LOGX>
__device__ __forceinline__ void load_group(uint64_t (&a)[3][1 << LOGX], const uint64_t *__restrict__ pol, uint64_t n2,
                                           uint64_t g)
{
#pragma unroll
    for (int i = 0; i < (1 << LOGX); i++) {
#pragma unroll
        for (int k = 0; k < 3; k++) a[k][i] = gl_canon(pol[((uint64_t)i * n2 + g) * 3 + k]);
    }
}

__device__ __forceinline__ gl3 load_challenge(uint64_t ch0, uint64_t ch1, uint64_t ch2, const uint64_t *chp)
{
    if (chp) return {{gl_canon(chp[0]), gl_canon(chp[1]), gl_canon(chp[2])}};
    return {{ch0, ch1, ch2}};
}

// Where value g of the folded layer goes: out, and with aux also to its place in the
// regrouped source of the layer's tree (getTransposed with 2^t_bits rows of 2^h_bits).
struct FoldOut {
    uint64_t *out, *aux;
    uint32_t t_bits, h_bits;
};
__device__ __forceinline__ void store_fold(const FoldOut &o, uint64_t g, const gl3 &r)
{
#pragma unroll
    for (int k = 0; k < 3; k++) o.out[g * 3 + k] = r.v[k];
    if (o.aux) {
        uint64_t d = ((g & ((1ull << o.t_bits) - 1)) << o.h_bits) + (g >> o.t_bits);
#pragma unroll
        for (int k = 0; k < 3; k++) o.aux[d * 3 + k] = r.v[k];
    }
}

// The challenge is (ch0, ch1, ch2), or the three words at chp when chp is not
// null (device memory read at run time, so a captured graph folds with the
// buffer's current contents).
template <int LOGX>
__global__ __launch_bounds__(256) void k_fri_fold(FoldOut out, const uint64_t *pol, uint32_t cur_bits,
                                                  uint64_t shift_inv, uint64_t w_inv, uint64_t ch0, uint64_t ch1,
                                                  uint64_t ch2, const uint64_t *__restrict__ chp, uint64_t nx_inv,
                                                  RootTab rt)
{
    uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t n2 = 1ull << cur_bits;
    if (g >= n2) return;
    gl3 x = load_challenge(ch0, ch1, ch2, chp);
    uint64_t a[3][1 << LOGX];
    load_group<LOGX>(a, pol, n2, g);
    // sinv_g = shift_inv * w_inv^g
    store_fold(out, g, fold_group<LOGX>(a, gl_mul(shift_inv, root_pow(rt, w_inv, g)), x, nx_inv));
}

// NX / 2 lanes a group, 64 / (NX / 2) neighbouring groups a wave. Groups past the last
// one work on it again: the exchanges want every lane. Each group's reads of pol come
// before the write of out[g], in the same wave, so out may equal pol.
template <int LOGX>
__global__ __launch_bounds__(64) void k_fri_fold_lanes(FoldOut out, const uint64_t *pol, uint32_t cur_bits,
                                                       uint64_t shift_inv, uint64_t w_inv, uint64_t ch0, uint64_t ch1,
                                                       uint64_t ch2, const uint64_t *__restrict__ chp, uint64_t nx_inv,
                                                       RootTab rt)
{
    constexpr uint32_t L = 1u << (LOGX - 1), G = 64 / L;
    const uint64_t n2 = 1ull << cur_bits, g0 = (uint64_t)blockIdx.x * G + threadIdx.x % G;
    const uint64_t g = g0 < n2 ? g0 : n2 - 1;
    const uint32_t i = threadIdx.x / G;
    gl3 x = load_challenge(ch0, ch1, ch2, chp);
    uint64_t u[3], v[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        u[k] = gl_canon(pol[((uint64_t)i * n2 + g) * 3 + k]);
        v[k] = gl_canon(pol[((uint64_t)(i + L) * n2 + g) * 3 + k]);
    }
    gl3 r = fold_group_lanes<LOGX>(u, v, i, G, gl_mul(shift_inv, root_pow(rt, w_inv, g)), x, nx_inv);
    if (i == 0 && g0 < n2) store_fold(out, g, r);
}

// Fold ratios 2^6 .. 2^10 as two folds in one kernel. With x^nX = (x^32)^(nX/32),
// the FRI fold of ratio nX at challenge c equals a fold of ratio 32 at c
// (prev -> prev-5 bits, on the coset shift s and w_{2^prev}) followed by a fold of
// ratio nB = nX/32 at c^32 (prev-5 -> cur bits, on the coset s^32 and
// w_{2^(prev-5)}): the polynomial sum_i c^i f_i(y) regrouped as i = j + 32 l. A
// block handles GB = 256/nB consecutive groups g: its 256 lanes first fold the
// ratio-32 groups h = l*2^cur + g (l < nB) of the intermediate layer into LDS,
// then GB lanes fold each g's nB intermediate values. Every read of pol comes
// before the block's writes of out[g], and other blocks read only other g's
// groups, so out may equal pol (in place, as the reference folds).
template <int LOGB>
__global__ __launch_bounds__(256) void k_fri_fold_big(FoldOut out, const uint64_t *pol, uint32_t cur_bits,
                                                      uint64_t shift_inv1, uint64_t w_inv1,
                                                      uint64_t shift_inv2, uint64_t w_inv2, uint64_t ch0, uint64_t ch1,
                                                      uint64_t ch2, const uint64_t *__restrict__ chp,
                                                      uint64_t n32_inv, uint64_t nb_inv, RootTab rt1, RootTab rt2)
{
    constexpr int NB = 1 << LOGB, GB = 256 / NB;
    __shared__ uint64_t mid[3][256];  // [k][l*GB + gl]
    uint64_t n2 = 1ull << cur_bits, n1 = n2 << LOGB;  // intermediate layer: 2^(cur+LOGB) values
    gl3 c = load_challenge(ch0, ch1, ch2, chp);
    uint32_t t = threadIdx.x, l = t / GB, gl = t % GB;
    uint64_t g = (uint64_t)blockIdx.x * GB + gl;
    if (g < n2) {
        uint64_t h = (uint64_t)l * n2 + g;
        uint64_t a[3][32];
        load_group<5>(a, pol, n1, h);
        gl3 r = fold_group<5>(a, gl_mul(shift_inv1, root_pow(rt1, w_inv1, h)), c, n32_inv);
#pragma unroll
        for (int k = 0; k < 3; k++) mid[k][t] = r.v[k];
    }
    __syncthreads();
    if (t < (uint32_t)GB && g < n2) {
        gl3 c32 = c;
#pragma unroll
        for (int q = 0; q < 5; q++) c32 = gl3_mul(c32, c32);
        uint64_t a[3][NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
#pragma unroll
            for (int k = 0; k < 3; k++) a[k][i] = mid[k][i * GB + t];
        }
        store_fold(out, g, fold_group<LOGB>(a, gl_mul(shift_inv2, root_pow(rt2, w_inv2, g)), c32, nb_inv));
    }
}

__global__ __launch_bounds__(256) void k_fri_transpose(uint64_t *__restrict__ aux, const uint64_t *__restrict__ pol,
                                                       uint64_t degree, uint32_t t_bits)
{
    uint64_t d = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;  // destination element index i*h + j
    if (d >= degree) return;
    uint64_t w = 1ull << t_bits, h = degree >> t_bits;
    uint64_t i = d / h, j = d - i * h;
    uint64_t s = j * w + i;
#pragma unroll
    for (int k = 0; k < 3; k++) aux[d * 3 + k] = pol[s * 3 + k];
}

extern "C" int fri_launch_fold(uint64_t *out, const uint64_t *pol, const uint64_t *challenge, uint64_t n_bits_ext,
                               uint64_t prev_bits, uint64_t cur_bits, const NttTablesHost *tw, hipStream_t st)
{
    return fri_launch_fold2(out, pol, challenge, nullptr, n_bits_ext, prev_bits, cur_bits, tw, nullptr, 0, st);
}

// The inverse split tables of the smallest NTT domain (2^24 or 2^28) holding
// 2^log_w points, scaled so that e0 indexes w_{2^log_w}^-e0; none above 2^28.
static RootTab root_tab(const NttTablesHost *tw, uint64_t log_w)
{
    if (!tw || log_w > 28) return {nullptr, nullptr, 0, 0};
    const NttSplitTables &S = tw->split[log_w > 24 ? 1 : 0];
    return {S.twl_i, S.twh_i, S.bits, (uint32_t)(2 * S.bits - log_w)};
}

extern "C" int fri_launch_fold2(uint64_t *out, const uint64_t *pol, const uint64_t *challenge,
                                const uint64_t *d_challenge, uint64_t n_bits_ext, uint64_t prev_bits,
                                uint64_t cur_bits, const NttTablesHost *tw, uint64_t *aux, uint64_t t_bits,
                                hipStream_t st)
{
    FoldOut fo = {out, aux, (uint32_t)t_bits, (uint32_t)(cur_bits - t_bits)};
    if (cur_bits > prev_bits || prev_bits > n_bits_ext || prev_bits > 32) return -1;
    uint32_t logx = (uint32_t)(prev_bits - cur_bits);
    uint64_t shift = 7;
    for (uint64_t j = 0; j < n_bits_ext - prev_bits; j++) shift = gl_mul(shift, shift);
    uint64_t shift_inv = gl_inv(shift);
    static const uint64_t W[33] = {
        0x1ULL, 18446744069414584320ULL, 281474976710656ULL, 16777216ULL, 4096ULL, 64ULL, 8ULL,
        2198989700608ULL, 4404853092538523347ULL, 6434636298004421797ULL, 4255134452441852017ULL,
        9113133275150391358ULL, 4355325209153869931ULL, 4308460244895131701ULL,
        7126024226993609386ULL, 1873558160482552414ULL, 8167150655112846419ULL,
        5718075921287398682ULL, 3411401055030829696ULL, 8982441859486529725ULL,
        1971462654193939361ULL, 6553637399136210105ULL, 8124823329697072476ULL,
        5936499541590631774ULL, 2709866199236980323ULL, 8877499657461974390ULL,
        3757607247483852735ULL, 4969973714567017225ULL, 2147253751702802259ULL,
        2530564950562219707ULL, 1905180297017055339ULL, 3524815499551269279ULL,
        7277203076849721926ULL};
    uint64_t w_inv = gl_inv(W[prev_bits]);
    uint64_t c0 = 0, c1 = 0, c2 = 0;
    if (!d_challenge) c0 = gl_canon(challenge[0]), c1 = gl_canon(challenge[1]), c2 = gl_canon(challenge[2]);
    uint64_t n2 = 1ull << cur_bits;
    if (logx > 5) {
        // two-stage fold: ratio 32 (prev -> prev-5) at c, then ratio 2^(logx-5) at c^32
        uint32_t logb = logx - 5;
        uint64_t shift2 = shift;
        for (int q = 0; q < 5; q++) shift2 = gl_mul(shift2, shift2);
        uint64_t groups = 256u >> logb, blocks = (n2 + groups - 1) / groups;
        dim3 gb((unsigned)blocks);
        uint64_t n32_inv = gl_inv(32);
        uint64_t nb_inv = gl_inv(1ull << logb), w_inv2 = gl_inv(W[prev_bits - 5]), shift_inv2 = gl_inv(shift2);
#define FOLD_BIG(L)                                                                                              \
    case L:                                                                                                      \
        hipLaunchKernelGGL(k_fri_fold_big<L>, gb, dim3(256), 0, st, fo, pol, (uint32_t)cur_bits, shift_inv,      \
                           w_inv, shift_inv2, w_inv2, c0, c1, c2, d_challenge, n32_inv, nb_inv,                  \
                           root_tab(tw, prev_bits), root_tab(tw, prev_bits - 5));                                \
        break;
        switch (logb) {
            FOLD_BIG(1)
            FOLD_BIG(2)
            FOLD_BIG(3)
            FOLD_BIG(4)
            FOLD_BIG(5)
        default: return -2;
        }
#undef FOLD_BIG
        return (int)hipGetLastError();
    }
    uint64_t nx_inv = gl_inv((1ull << logx) % GL_P);
    // one lane a group, or 2^(logx-1) of them while that makes at most two waves a SIMD: a
    // group's chain of products is what short layers wait for
    const bool lanes = logx >= 2 && (n2 << (logx - 1)) <= FRI_LANES_MAX;
    const uint64_t per = 128u >> logx;  // groups of a wave with 2^(logx-1) lanes each
    dim3 g((unsigned)(lanes ? (n2 + per - 1) / per : (n2 + 255) / 256)), b(lanes ? 64 : 256);
#define FOLD_CASE(L)                                                                                                \
    case L:                                                                                                         \
        if (lanes)                                                                                                  \
            hipLaunchKernelGGL(k_fri_fold_lanes<L>, g, b, 0, st, fo, pol, (uint32_t)cur_bits, shift_inv, w_inv, c0, \
                               c1, c2, d_challenge, nx_inv, root_tab(tw, prev_bits));                               \
        else                                                                                                        \
            hipLaunchKernelGGL(k_fri_fold<L>, g, b, 0, st, fo, pol, (uint32_t)cur_bits, shift_inv, w_inv, c0, c1,   \
                               c2, d_challenge, nx_inv, root_tab(tw, prev_bits));                                   \
        break;
    switch (logx) {
    case 1:
        hipLaunchKernelGGL(k_fri_fold<1>, g, b, 0, st, fo, pol, (uint32_t)cur_bits, shift_inv, w_inv, c0, c1, c2,
                           d_challenge, nx_inv, root_tab(tw, prev_bits));
        break;
        FOLD_CASE(2)
        FOLD_CASE(3)
        FOLD_CASE(4)
        FOLD_CASE(5)
    default: return -2;
    }
#undef FOLD_CASE
    return (int)hipGetLastError();
}

extern "C" int fri_launch_transpose(uint64_t *aux, const uint64_t *pol, uint64_t degree, uint32_t t_bits,
                                    hipStream_t st)
{
    if (degree == 0) return 0;
    dim3 g((unsigned)((degree + 255) / 256));
    hipLaunchKernelGGL(k_fri_transpose, g, dim3(256), 0, st, aux, pol, degree, t_bits);
    return (int)hipGetLastError();
}

// ------------------------------------------------------- field self-check ----
// Element-wise field operations on device (op 0 add, 1 sub, 2 mul, 3 canonical
// reduce of a 128-bit value (a = low word, b = high word)). Exposed so the GPU
// tests can pin the device arithmetic on edge values against exact integers.
__global__ __launch_bounds__(256) void k_gl_binop(uint64_t *__restrict__ out, const uint64_t *__restrict__ a,
                                                  const uint64_t *__restrict__ b, uint64_t n, int op)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t x = a[i], y = b[i];
    uint64_t r;
    if (op == 0) r = gl_add(gl_canon(x), gl_canon(y));
    else if (op == 1) r = gl_sub(gl_canon(x), gl_canon(y));
    else if (op == 2) r = gl_mul(x, y);
    else r = gl_reduce128_canon(x, y);
    out[i] = r;
}

extern "C" int fri_launch_gl_binop(uint64_t *out, const uint64_t *a, const uint64_t *b, uint64_t n, int op,
                                   hipStream_t st)
{
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_gl_binop, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, out, a, b, n, op);
    return (int)hipGetLastError();
}
