// flare_wave_bwd.h -- backward of the chunked causal FLARE forward with wave-private latents
// (equal head dims, M <= 256).  Per (b, h), latent m and token t, with s the encoder score,
// D_t the running sum of e^s, alpha_t the decoder softmax, g = dY and U_t the running sum of
// e^s v (z_t = U_t / D_t):
//   gz_t  = g_t . U_t / D_t                 da_t = alpha_t (gz_t - g_t . y_t)
//   X_tau = sum_{t >= tau} (alpha_t / D_t) g_t      Y_tau = sum_{t >= tau} (alpha_t / D_t) gz_t
//   ds_tau = e^{s_tau} (v_tau . X_tau - Y_tau)      dv_tau = sum_m e^{s_tau} X_tau
// and dQ, dK (dQ_dec, dK_dec) are contractions of ds + da (ds, da).
//
// Two walks over the forward's own kind of chunks replace per-token statistics in memory:
//   wave_gz   forward over a chunk from its exclusive prefix (max, den, U): writes gz, the
//             (max, den) at each 16-token tile's start, and the chunk's share of X and Y;
//   wave_ds   backward over a chunk from the X, Y after it (a reverse scan over chunks):
//             recomputes a tile's weights from the stored (max, den), writes ds and dv.
// Between them only gz (fp32) travels per token and latent; scores, weights, decoder softmax
// and running sums are formed again from K, Q and one (max, den) pair per 16 tokens.
// g . y: for fp32 inputs the sum of alpha gz over the latents, from the very gz it is subtracted
// from (gz - g . y cancels, and the saved output carries its own rounding: with it the fp32
// gradients of the block-causal layer were up to 1.4 times as far off).  16-bit inputs take it
// from the saved output, whose rounding their results have anyway (in the walk it cost 30 us
// against 16 for its own kernel at B 4, N 4096, H 16, M 128, D 64).
//
// Layout: the tile's score-like matrices are C tiles with tokens as rows (lane (g, c):
// tokens 4g + i, latent c), U and X are kept transposed (rows = value columns, lane column =
// latent).  g . U, v . X, U += , X += and the in-tile sums then need no data movement; only
// dv (a sum over latents) needs e, w and X the other way round, through wave-private LDS.
// A latent is one lane column, so its reference max and its moves are per-lane scalars.
//
// Products.  fp32 inputs: fp32 MFMA (16x16x4).  16-bit inputs: every fp32 factor enters the
// bf16 MFMA as a sum of P bf16 parts, each the nearest to what the parts before it leave; two
// parts lie side by side in the contraction index of the 16x16x32 instruction (16 tokens or
// latents of the first, the same 16 of the second).  P = 3 holds all 24 bits, P = 2 is within
// 2^-18.  Two parts serve the banks whose states always met the matrix units as two parts (M
// 128 and 256, D 64 and 128), three the banks whose kernels were all fp32 (three_parts).  Share
// of dV entries that are not the rounded 64-bit value, against those kernels, fp16, N 1531: M 64,
// D 32 0.16 -> 0.13% (0.7% with two parts), M 128, D 64 0.73 -> 0.52% (1.1% with two of which
// the first is cut off and not rounded); dK of separate decoder weights at M 64, D 32 1.75 -> 0.18%.
//
// Numerics.  Weights inside a tile are relative to the latents' max after the tile, X and Y
// to the max of the tile they were last used in (factors <= 1 as the walk goes back).  A tile
// in which a max rises by more than kTileJump runs token by token with each token's own max.
//
// Bound by vector issue and the latency of a tile's chain at two to three waves a SIMD (some
// 60% of the issue slots are used, 12% of the matrix pipe's).  What is read the other way round
// (V, g, X and the e / w tiles of 16-bit kernels) comes through transposing LDS reads, X, e and w
// already split into bf16 hi + lo: splitting after the read took a third more instructions
// (1,691 against 1,114 in the backward walk at D = 128; 677 -> 515 us at N 16384, M 256, the hi
// parts cut off).
// Measured, forward and backward, against per-token statistics and one state per 32 tokens in
// memory (MI355X):
//   bf16 B 4, N 4096, H 16, M 128, D 64    1525 -> 529 us (wave_gz 124, wave_ds 166 of it)
//   bf16 N 16384, H 16, M 256, D 128       3807 -> 1445 us (wave_gz 405, wave_ds 517)
//   bf16 B 4, N 2011, H 16, M 64, D 32     2946 -> 213 us (wave_gz 37, wave_ds 48)
//   fp32 B 2, N 1024, H 8, M 64, D 64, decoder weights of its own   1171 -> 216 us
#pragma once

#include <type_traits>

#include "flare_internal.h"
#include "flare_wave.h"

namespace flare {
namespace wave {

using mfma::bf16x4;
using mfma::f16x8;
typedef short s16x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Value columns.  Lane c (or C row c) of column tile dt is value column walk_col(dt, c).  fp32
// kernels keep the pieces of col_of (several tiles' columns side by side, so that a lane reads
// 16 bytes); 16-bit ones (FLAT) take column 16 dt + c, the order of the transposing LDS reads.
// ---------------------------------------------------------------------------
template <int DT, bool FLAT>
__host__ __device__ constexpr int walk_piece(int dt) { return FLAT ? 1 : piece_of<DT>(dt); }
// column tiles taken at a time: two where each has a read of its own (four held 16 registers more
// and spilled at D = 64: 130 against 119 us for the forward walk)
template <typename T, int DT>
__host__ __device__ constexpr int step_of(int dt) { return sizeof(T) == 2 ? (dt + 2 <= DT ? 2 : 1) : piece_of<DT>(dt); }
// these by number, and the most tiles a step has (see pieces: loops over them have to unroll)
template <int DT, bool FLAT>
__host__ __device__ constexpr int walk_pieces() { return FLAT ? DT : pieces<DT>(); }
template <int DT, bool FLAT>
__host__ __device__ constexpr int walk_start(int p) { return FLAT ? p : piece_start<DT>(p); }
template <typename T, int DT>
__host__ __device__ constexpr int steps() { return sizeof(T) == 2 ? (DT + 1) / 2 : pieces<DT>(); }
template <typename T, int DT>
__host__ __device__ constexpr int step_start(int s) { return sizeof(T) == 2 ? 2 * s : piece_start<DT>(s); }
template <typename T>
__host__ __device__ constexpr int step_most() { return sizeof(T) == 2 ? 2 : 4; }
template <int DT, bool FLAT>
__device__ __forceinline__ int walk_col(int dt, int c) { return FLAT ? 16 * dt + c : col_of<DT>(dt, c); }

// ---------------------------------------------------------------------------
// A row of D = 16 DT values, split over the lane groups as the C rows of a transposed state
// are: lane group g holds value column walk_col(dt, 4g + i) for every dt, i.  Within a piece
// these are 4 P consecutive columns.
// ---------------------------------------------------------------------------
template <int DT, bool FLAT>
__host__ __device__ constexpr int list_at(int dt, int i) {    // position of (dt, i) in the lane's list
    return FLAT ? 4 * dt + i : 4 * piece_off<DT>(dt) + i * piece_of<DT>(dt) + (dt - piece_off<DT>(dt));
}

template <typename T, int DT, bool FLAT = false>
struct GroupRow {
    static constexpr int W = sizeof(T) == 4 ? 4 * DT : 2 * DT;
    static constexpr int S = (DT + 1) / 2;                    // steps of 8 values (32 over the groups)
    unsigned w[W];
    __device__ __forceinline__ void load(const T* row, int g) {
#pragma unroll
        for (int pc = 0, dt = 0; pc < walk_pieces<DT, FLAT>(); dt = walk_start<DT, FLAT>(++pc)) {
            const int P = walk_piece<DT, FLAT>(dt);
            const T* p = row + 16 * dt + 4 * g * P;
            // 4 P values
            const int at = (sizeof(T) == 4 ? 4 : 2) * dt, words = (sizeof(T) == 4 ? 4 : 2) * P;
            if (words == 2) {
                const u32x2 x = *reinterpret_cast<const u32x2*>(p);
                w[at] = x[0];
                w[at + 1] = x[1];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * j < words) {
                        const u32x4 x = reinterpret_cast<const u32x4*>(p)[j];
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (at + 4 * j + k < W) w[at + 4 * j + k] = x[k];
                    }
            }
        }
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int j = 0; j < W; ++j) w[j] = 0;
    }
    __device__ __forceinline__ float at(int e) const {
        if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, w[e]);
        else return word_f32<T>(w[e / 2], e & 1);
    }
    // eight values as a 16-bit MFMA operand (zeros past the end)
    __device__ __forceinline__ bf16x8 op8(int s) const {
        u32x4 r;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = 4 * s + j < W ? w[4 * s + j] : 0u;
        return __builtin_bit_cast(bf16x8, r);
    }
};

// a row as the products with a transposed state read it
template <typename T, int DT>
using WalkRow = GroupRow<T, DT, sizeof(T) == 2>;

// c += x . y^T over the columns
template <typename T, int DT, bool FLAT>
__device__ __forceinline__ f32x4 dot_groups(const GroupRow<T, DT, FLAT>& x, const GroupRow<T, DT, FLAT>& y, f32x4 c) {
    if constexpr (sizeof(T) == 4) {
        // (two sums over halves: fewer roundings in a row, and shorter chains)
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 2 * DT; ++e) {
            c = mma4(x.at(e), y.at(e), c);
            d = mma4(x.at(2 * DT + e), y.at(2 * DT + e), d);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] += d[i];
    } else {
        constexpr bool F16 = __is_same(T, __half);
#pragma unroll
        for (int s = 0; s < GroupRow<T, DT>::S; ++s) c = mfma::mma_in<F16>(x.op8(s), y.op8(s), c);
    }
    return c;
}

// ---------------------------------------------------------------------------
// Operands of products over 16 contraction indices 4g + i (tokens or latents of a tile).
// ---------------------------------------------------------------------------
struct F4 {          // fp32 products
    float v[4];
};
template <int P>
struct Split4 {      // fp32 values as P bf16 parts
    bf16x4 p[P];
};
struct Exact4 {      // bf16 values
    bf16x4 x;
};
__device__ __forceinline__ bf16x8 cat(bf16x4 a, bf16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

__device__ __forceinline__ f32x4 mm(const F4& a, const F4& b, f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = mma4(a.v[i], b.v[i], c);
    return c;
}
// A third part goes with zeros into the same instruction.  (The 16x16x16 one has room for just
// that part, but its sum must not continue one of 16x16x32: nothing waits for the longer
// instruction there, and sums came out without some of its terms.)
__device__ __forceinline__ bf16x8 third(bf16x4 x) { return cat(x, bf16x4{}); }
template <int P>
__device__ __forceinline__ f32x4 mm(const Split4<P>& a, const Exact4& b, f32x4 c) {
    c = mfma::mma(cat(a.p[0], a.p[1]), cat(b.x, b.x), c);
    if constexpr (P == 3) c = mfma::mma(third(a.p[2]), cat(b.x, b.x), c);
    return c;
}
template <int P>
__device__ __forceinline__ f32x4 mm(const Exact4& a, const Split4<P>& b, f32x4 c) {
    c = mfma::mma(cat(a.x, a.x), cat(b.p[0], b.p[1]), c);
    if constexpr (P == 3) c = mfma::mma(cat(a.x, a.x), third(b.p[2]), c);
    return c;
}
// (without the parts' products below 2^-26 of the whole)
template <int P, int R>
__device__ __forceinline__ f32x4 mm(const Split4<P>& a, const Split4<R>& b, f32x4 c) {
    const bf16x8 two = cat(a.p[0], a.p[1]);
    c = mfma::mma(two, cat(b.p[0], b.p[0]), c);
    c = mfma::mma(two, cat(b.p[1], b.p[1]), c);
    if constexpr (P == 3 && R == 3) c = mfma::mma(cat(a.p[0], a.p[2]), cat(b.p[2], b.p[0]), c);
    else if constexpr (P == 3) c = mfma::mma(third(a.p[2]), cat(b.p[0], b.p[0]), c);
    else if constexpr (R == 3) c = mfma::mma(cat(a.p[0], a.p[0]), third(b.p[2]), c);
    return c;
}

// c += a b for a c that collects many tiles: fp32 products are summed over the tile first, so
// that c is rounded once a tile and not once a product.
template <typename A, typename B>
__device__ __forceinline__ f32x4 collect(const A& a, const B& b, f32x4 c) {
    if constexpr (__is_same(A, F4)) {
        const f32x4 r = mm(a, b, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] += r[i];
        return c;
    } else {
        return mm(a, b, c);
    }
}

// nearest parts: what is left after two is within 2^-18 of x, after three within 2^-27
template <int P>
__device__ __forceinline__ Split4<P> split4(f32x4 x) {
    Split4<P> r;
#pragma unroll
    for (int n = 0; n < P; ++n) {
        r.p[n] = __builtin_convertvector(x, bf16x4);
        const u32x2 b = __builtin_bit_cast(u32x2, r.p[n]);
        if (n + 1 < P)
            x = f32x4{x[0] - __builtin_bit_cast(float, b[0] << 16), x[1] - __builtin_bit_cast(float, b[0] & 0xffff0000u),
                      x[2] - __builtin_bit_cast(float, b[1] << 16), x[3] - __builtin_bit_cast(float, b[1] & 0xffff0000u)};
    }
    return r;
}
// P: bf16 parts of an fp32 factor of 16-bit kernels
template <typename T, int P> struct ProdOf { typedef Split4<P> F; };     // type of an fp32 factor
template <int P> struct ProdOf<float, P> { typedef F4 F; };
template <typename F>
__device__ __forceinline__ F factor(float x0, float x1, float x2, float x3) {
    F r;
    if constexpr (__is_same(F, F4)) {
        r.v[0] = x0;
        r.v[1] = x1;
        r.v[2] = x2;
        r.v[3] = x3;
    } else {
        r = split4<sizeof(F) / sizeof(bf16x4)>(f32x4{x0, x1, x2, x3});
    }
    return r;
}

// Tokens 4g + i of a 16-token tile, value column col_of(dt, c): the factor of the products
// over tokens.
template <typename T, int DT>
struct TokCols {
    typedef typename std::conditional<sizeof(T) == 4, F4,
                                      typename std::conditional<__is_same(T, __half), Split4<2>, Exact4>::type>::type Op;
    ColRow<T, DT> r[4];
    __device__ __forceinline__ Op op(int dt) const {
        Op o;
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) o.v[i] = r[i].get(dt);
        } else if constexpr (__is_same(T, __half)) {
            o = split4<2>(f32x4{r[0].get(dt), r[1].get(dt), r[2].get(dt), r[3].get(dt)});     // (exact: 11 bits)
        } else {
            const unsigned sel = dt & 1 ? 0x07060302u : 0x05040100u;
            u32x2 p;
            p[0] = __builtin_amdgcn_perm(r[1].w[dt / 2], r[0].w[dt / 2], sel);
            p[1] = __builtin_amdgcn_perm(r[3].w[dt / 2], r[2].w[dt / 2], sel);
            o.x = __builtin_bit_cast(bf16x4, p);
        }
        return o;
    }
};

// the columns of one step (two column tiles) of the product below, u as P bf16 parts
template <typename T, int DT, int P>
__device__ __forceinline__ f32x4 dot_split(const WalkRow<T, DT>& x, int s, const bf16x8 (&u)[P], f32x4 c) {
    if constexpr (__is_same(T, __half)) {
        const f16x8 xf = __builtin_bit_cast(f16x8, x.op8(s));
        bf16x8 xh, xl;
#pragma unroll
        for (int e = 0; e < 8; ++e) SPLIT2(mfma::bf16, (float)xf[e], xh[e], xl[e]);
#pragma unroll
        for (int n = 0; n < P; ++n) {
            c = mfma::mma(xh, u[n], c);
            if (n + 1 < P) c = mfma::mma(xl, u[n], c);
        }
    } else {
#pragma unroll
        for (int n = 0; n < P; ++n) c = mfma::mma(x.op8(s), u[n], c);
    }
    return c;
}
// column tiles 2s and 2s + 1 of a transposed state as the parts above (zeros past the end)
template <int DT, int P>
__device__ __forceinline__ void split_step(const f32x4 (&u)[DT], int s, Split4<P> (&x)[2]) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        if (2 * s + q < DT) x[q] = split4<P>(u[2 * s + q < DT ? 2 * s + q : 0]);
        else x[q] = Split4<P>{};
    }
}
template <int P>
__device__ __forceinline__ void cat_step(const Split4<P> (&x)[2], bf16x8 (&r)[P]) {
#pragma unroll
    for (int n = 0; n < P; ++n) r[n] = cat(x[0].p[n], x[1].p[n]);
}

// c += x . u over the columns: rows of x (lane column = row) against a transposed state
// (rows = columns walk_col(dt, 4g + i), lane column = latent); C rows are x's rows.
template <typename T, int DT, int P>
__device__ __forceinline__ f32x4 dot_state(const WalkRow<T, DT>& x, const f32x4 (&u)[DT], f32x4 c) {
    if constexpr (sizeof(T) == 4) {
        f32x4 d[3] = {};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            c = mma4(x.at(list_at<DT, false>(dt, 0)), u[dt][0], c);
#pragma unroll
            for (int i = 1; i < 4; ++i) d[i - 1] = mma4(x.at(list_at<DT, false>(dt, i)), u[dt][i], d[i - 1]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = (c[i] + d[0][i]) + (d[1][i] + d[2][i]);
    } else {
#pragma unroll
        for (int s = 0; s < GroupRow<T, DT>::S; ++s) {
            Split4<P> y[2];
            bf16x8 parts[P];
            split_step<DT, P>(u, s, y);
            cat_step(y, parts);
            c = dot_split<T, DT, P>(x, s, parts, c);
        }
    }
    return c;
}

// ---------------------------------------------------------------------------
// 16-bit values of an LDS tile the other way round: lane (g, c) gets rows 4g + i of column c
// from a tile whose rows start at `tile`, `pitch` apart (ds_read_b64_tr_b16: lane c of a
// group points at four columns of row 4g + c / 4).
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
__device__ __forceinline__ u32x2 tile_tr(const void* tile, int pitch, int g, int c) {
    const short* p = (const short*)tile + (4 * g + (c >> 2)) * pitch + 4 * (c & 3);
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}
template <int P>
__device__ __forceinline__ Split4<P> split_tr(const bf16x4* first, int quads, int pitch, int g, int c) {   // parts `quads` apart
    Split4<P> r;
#pragma unroll
    for (int n = 0; n < P; ++n) r.p[n] = __builtin_bit_cast(bf16x4, tile_tr(first + n * quads, pitch, g, c));
    return r;
}

// Tokens 4g + i of the tile in LDS, value column walk_col(dt, c): the factor of the products
// over tokens.
template <typename T, int DT>
struct TileCols {
    typedef typename TokCols<T, DT>::Op Op;
    static constexpr bool FLAT = sizeof(T) == 2;
    typename std::conditional<FLAT, u32x2[DT], ColRow<T, DT>[4]>::type r;
    // the column tiles of the piece that starts at tile d0; rows from `tile`, `pitch` apart
    __device__ __forceinline__ void load_piece(const T* tile, int pitch, int g, int c, int d0) {
        if constexpr (FLAT) {
#pragma unroll
            for (int dt = d0; dt < d0 + step_most<T>(); ++dt)
                if (dt < d0 + step_of<T, DT>(d0)) r[dt] = tile_tr(tile + 16 * dt, pitch, g, c);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) r[i].load_piece(tile + (4 * g + i) * pitch, c, d0);
        }
    }
    // tokens that are off become zero, whatever they hold
    __device__ __forceinline__ void keep(const bool (&on)[4], int d0) {
        if constexpr (FLAT) {
            const unsigned m0 = (on[0] ? 0xffffu : 0u) | (on[1] ? 0xffff0000u : 0u);
            const unsigned m1 = (on[2] ? 0xffffu : 0u) | (on[3] ? 0xffff0000u : 0u);
#pragma unroll
            for (int dt = d0; dt < d0 + step_most<T>(); ++dt) {
                if (dt >= d0 + step_of<T, DT>(d0)) continue;
                r[dt][0] &= m0;
                r[dt][1] &= m1;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int k = d0; k < d0 + step_most<T>(); ++k)
                    if (k < d0 + step_of<T, DT>(d0)) r[i].w[k] = on[i] ? r[i].w[k] : 0u;
        }
    }
    __device__ __forceinline__ Op op(int dt) const {
        Op o;
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) o.v[i] = r[i].get(dt);
        } else if constexpr (__is_same(T, __half)) {
            const unsigned a = r[dt][0], b = r[dt][1];
            o = split4<2>(f32x4{word_f32<T>(a, false), word_f32<T>(a, true), word_f32<T>(b, false), word_f32<T>(b, true)});
        } else {
            o.x = __builtin_bit_cast(bf16x4, r[dt]);
        }
        return o;
    }
};

// A transposed state of 16 latents in wave-private LDS, a row a latent: fp32, or (FLAT) the rows
// of the first bf16 part and behind them those of the others, from where both products over it
// read their operands.
template <typename T, int DT, int P>
struct StateTile {
    static constexpr bool FLAT = sizeof(T) == 2;
    static constexpr int D = 16 * DT, PITCH = FLAT ? D + 8 : D + 4;
    static constexpr int FLOATS = FLAT ? 8 * PITCH * P : 16 * PITCH;
    static constexpr int QUADS = 16 * PITCH / 4;                     // of one part
    typedef bf16x4 __attribute__((may_alias)) quad_a;
    static __device__ __forceinline__ quad_a* quad(float* tile, int g, int c, int dt) {
        return reinterpret_cast<quad_a*>(tile) + (c * PITCH + 16 * dt + 4 * g) / 4;
    }
    static __device__ __forceinline__ void put_parts(float* tile, const Split4<P>& x, int g, int c, int dt) {
#pragma unroll
        for (int n = 0; n < P; ++n) quad(tile, g, c, dt)[n * QUADS] = x.p[n];
    }
    static __device__ __forceinline__ void put(float* tile, const f32x4 (&u)[DT], int g, int c) {
#pragma unroll
        for (int pc = 0, dt = 0; pc < walk_pieces<DT, FLAT>(); dt = walk_start<DT, FLAT>(++pc)) {
            if constexpr (FLAT) {
                put_parts(tile, split4<P>(u[dt]), g, c, dt);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k < piece_of<DT>(dt)) tile[c * PITCH + col_of<DT>(dt, 4 * g + i) + k] = u[dt + k < DT ? dt + k : 0][i];
            }
        }
    }
    // put, and c + x . u
    static __device__ __forceinline__ f32x4 put_dot(float* tile, const WalkRow<T, DT>& x, const f32x4 (&u)[DT], int g, int cl,
                                                    f32x4 c) {
        if constexpr (FLAT) {
#pragma unroll
            for (int s = 0; s < GroupRow<T, DT>::S; ++s) {
                Split4<P> y[2];
                bf16x8 parts[P];
                split_step<DT, P>(u, s, y);
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    if (2 * s + q < DT) put_parts(tile, y[q], g, cl, 2 * s + q);
                cat_step(y, parts);
                c = dot_split<T, DT, P>(x, s, parts, c);
            }
            return c;
        } else {
            put(tile, u, g, cl);
            return dot_state<T, DT, P>(x, u, c);
        }
    }
    // c + x . u for a u that was put before
    static __device__ __forceinline__ f32x4 dot(float* tile, const WalkRow<T, DT>& x, const f32x4 (&u)[DT], int g, int cl,
                                                f32x4 c) {
        if constexpr (FLAT) {
#pragma unroll
            for (int s = 0; s < GroupRow<T, DT>::S; ++s) {
                Split4<P> y[2] = {};
                bf16x8 parts[P];
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    if (2 * s + q < DT) {
#pragma unroll
                        for (int n = 0; n < P; ++n) y[q].p[n] = quad(tile, g, cl, 2 * s + q)[n * QUADS];
                    }
                cat_step(y, parts);
                c = dot_split<T, DT, P>(x, s, parts, c);
            }
            return c;
        } else {
            return dot_state<T, DT, P>(x, u, c);
        }
    }
    // latents 4g + i, value column walk_col(dt, c): the factor of the products over latents
    struct Cols {
        typename std::conditional<FLAT, Split4<P>[DT], ColRow<float, DT>[4]>::type r;
        __device__ __forceinline__ void load_piece(const float* tile, int g, int c, int d0) {
            if constexpr (FLAT) {
#pragma unroll
                for (int dt = d0; dt < d0 + step_most<T>(); ++dt)
                    if (dt < d0 + step_of<T, DT>(d0))
                        r[dt] = split_tr<P>((const bf16x4*)tile + 4 * dt, QUADS, PITCH, g, c);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) r[i].load_piece(tile + (4 * g + i) * PITCH, c, d0);
            }
        }
        __device__ __forceinline__ typename ProdOf<T, P>::F op(int dt) const {
            if constexpr (FLAT) return r[dt];
            else return factor<F4>(r[0].get(dt), r[1].get(dt), r[2].get(dt), r[3].get(dt));
        }
    };
};

// dv += X^T . e for the 16 latents whose state is in `tile` (dv starts at the first of them)
template <typename Tile, typename T, int DT, typename F>
__device__ __forceinline__ void add_state_product(f32x4 (&dv)[DT], const float* tile, const F& e, bool first, int g, int c) {
#pragma unroll
    for (int st = 0, d0 = 0; st < steps<T, DT>(); d0 = step_start<T, DT>(++st)) {
        typename Tile::Cols xc;
        xc.load_piece(tile, g, c, d0);
#pragma unroll
        for (int dt = d0; dt < d0 + step_most<T>(); ++dt)
            if (dt < d0 + step_of<T, DT>(d0))
                dv[dt] = mm(xc.op(dt), e, first ? f32x4{0.f, 0.f, 0.f, 0.f} : dv[dt]);
    }
}

// A C tile [token 4g + i][latent c] of factors in wave-private LDS, read back as the factor
// with lane column = token and contraction index = latent.
template <typename T, int P>
struct TurnTile {
    static constexpr bool FLAT = sizeof(T) == 2;
    static constexpr int PITCH = 20;                                 // fp32 rows a token, 16-bit rows a latent
    static constexpr int QUADS = 16 * PITCH / 4;                     // of one part
    static constexpr int FLOATS = FLAT ? 8 * PITCH * P : 16 * PITCH;
    typedef typename ProdOf<T, P>::F F;
    typedef bf16x4 __attribute__((may_alias)) quad_a;
    static __device__ __forceinline__ void put(float* tile, const F& f, int g, int c) {
        if constexpr (FLAT) {
            quad_a* q = reinterpret_cast<quad_a*>(tile) + (c * PITCH + 4 * g) / 4;
#pragma unroll
            for (int n = 0; n < P; ++n) q[n * QUADS] = f.p[n];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) tile[(4 * g + i) * PITCH + c] = f.v[i];
        }
    }
    static __device__ __forceinline__ F get(const float* tile, int g, int c) {
        if constexpr (FLAT) {
            return split_tr<P>((const bf16x4*)tile, QUADS, PITCH, g, c);
        } else {
            const f32x4 r = *reinterpret_cast<const f32x4_a*>(tile + c * PITCH + 4 * g);
            return factor<F>(r[0], r[1], r[2], r[3]);
        }
    }
};

// dv of a tile (rows = value columns, lane column = token) as rows a token
template <int DT, bool FLAT>
__device__ __forceinline__ void put_rows(float* rows, int pitch, const f32x4 (&dv)[DT], int g, int c) {
#pragma unroll
    for (int pc = 0, dt = 0; pc < walk_pieces<DT, FLAT>(); dt = walk_start<DT, FLAT>(++pc)) {
        if constexpr (FLAT) {
            *reinterpret_cast<f32x4_a*>(rows + c * pitch + 16 * dt + 4 * g) = dv[dt];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k < piece_of<DT>(dt)) rows[c * pitch + col_of<DT>(dt, 4 * g + i) + k] = dv[dt + k < DT ? dt + k : 0][i];
        }
    }
}

// Over the lane groups of a lane column: the sum of x over lower groups, over higher
// groups, and over all.
__device__ __forceinline__ void group_scan(float x, int g, float& below, float& above, float& all) {
    float even, odd, lo, hi;
    lane_pair<16>(x, even, odd);
    lane_pair<32>(even + odd, lo, hi);
    below = (g & 1 ? even : 0.0f) + (g & 2 ? lo : 0.0f);
    above = (g & 1 ? 0.0f : odd) + (g & 2 ? 0.0f : hi);
    all = lo + hi;
}
// value of register i (wave-uniform) of token j = 4 (j / 4) + i at every lane of its column
__device__ __forceinline__ float token_value(const float (&x)[4], int j, int c) {
    const int i = j & 3;
    const float v = i == 0 ? x[0] : i == 1 ? x[1] : i == 2 ? x[2] : x[3];
    return __shfl(v, (j >> 2) * 16 + c, 64);
}


// ---------------------------------------------------------------------------
// Value columns in which dY is not finite at this token or a later one.  Such a column of X, and of
// dV from there back, is that infinity (NaN for both signs), which products do not give by
// themselves: an infinity times the parts of a weight, or times the weight 0 of a latent past the
// bank, is NaN.  Bit 4 dt + i stands for column walk_col(dt, 4g + i).  The backward walks keep the
// bits in LDS, two words a lane group for the whole workgroup (a training step of N 16384, H 16, M
// 256, D 128 takes 1420 us, 1409 without any of this and 1446 with the bits in registers).
// ---------------------------------------------------------------------------
template <typename T, int DT>
struct WildCols {
    static constexpr bool FLAT = sizeof(T) == 2;
    unsigned pos = 0, neg = 0;
    __device__ __forceinline__ void take(float v, int dt, int i) {
        const unsigned bit = 1u << (4 * dt + i);
        pos |= !(v <= 3.4e38f) ? bit : 0u;          // (NaN: both)
        neg |= !(v >= -3.4e38f) ? bit : 0u;
    }
    __device__ __forceinline__ void take_row(const T* row, int g) {
        for (int dt = 0; dt < DT; ++dt)
            for (int i = 0; i < 4; ++i) {
                const T v = row[walk_col<DT, FLAT>(dt, 4 * g + i)];
                if constexpr (sizeof(T) == 4) take(v, dt, i);
                else take(word_f32<T>(__builtin_bit_cast(unsigned short, v), false), dt, i);
            }
    }
    __device__ __forceinline__ bool any() const { return __any((pos | neg) != 0); }
    __device__ __forceinline__ bool has(int dt, int i) const { return ((pos | neg) >> (4 * dt + i)) & 1; }
    __device__ __forceinline__ float value(int dt, int i) const {
        const unsigned n = 4 * dt + i;
        const float inf = __builtin_inff();
        return (pos >> n) & (neg >> n) & 1 ? __builtin_nanf("") : (pos >> n) & 1 ? inf : -inf;
    }
    // a column is wild whichever lane shows it
    __device__ __forceinline__ void add_to(unsigned* bits, int g) const {
        if (pos != 0) __hip_atomic_fetch_or(bits + 2 * g, pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (neg != 0) __hip_atomic_fetch_or(bits + 2 * g + 1, neg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void read(const unsigned* bits, int g) {
        pos = bits[2 * g];
        neg = bits[2 * g + 1];
    }
};
// NaN where a value of a state is not finite
template <int DT>
__device__ __forceinline__ float state_probe(const f32x4 (&x)[DT]) {
    float r = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) r = __builtin_fmaf(x[dt][i], 0.0f, r);
    return r;
}
// a chunk's terms of X: wild columns as they are to be
template <typename T, int MT, int DT>
__device__ __forceinline__ void set_wild(f32x4 (&x)[MT][DT], const T* rows, int stride, int t0, int t1, int g) {
    float probe = 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) probe += state_probe(x[mt]);
    if (!__any(probe != probe)) return;
    WildCols<T, DT> wild;
    for (int t = t0; t < t1; ++t) wild.take_row(rows + (size_t)t * stride, g);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[mt][dt][i] = wild.has(dt, i) ? wild.value(dt, i) : x[mt][dt][i];
}
// whether X after a chunk has wild columns, which go to `bits`
template <typename T, int MT, int DT>
__device__ __forceinline__ bool find_wild(const f32x4 (&x)[MT][DT], unsigned* bits, int g) {
    float probe = 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) probe += state_probe(x[mt]);
    if (!__any(probe != probe)) return false;
    WildCols<T, DT> wild;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) wild.take(x[mt][dt][i], dt, i);
    wild.add_to(bits, g);
    return true;
}
// a tile's dv rows in this wave's LDS: their wild columns
template <typename T, int DT>
__device__ __forceinline__ bool put_wild(float* rows, int pitch, const unsigned* bits, int g, int c) {
    wave_lds_sync();
    WildCols<T, DT> wild;
    wild.read(bits, g);
    if (!wild.any()) return false;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (wild.has(dt, i)) rows[c * pitch + walk_col<DT, sizeof(T) == 2>(dt, 4 * g + i)] = wild.value(dt, i);
    return true;
}

// Registers: the latents' rows stay there up to D = 64 (fp32: 32), else they are read again
// each tile, from cache.  Wide states spill all the same, and the spilled values come back once a
// tile.  Bytes a lane at D = 128: wave_gz 564 in fp32 (592 with decoder weights of its own; 220 and
// 300 at D = 96), 28 to 144 with three parts, at most 112 with two; wave_ds up to 140 in fp32, 104
// to 192 with three parts, 8 to 40 with two; wave_semi_gz 48 (280) in fp32, 20 to 108 in 16 bits;
// wave_semi_ds 124 in fp32, at most 64 in fp16.
template <typename T, int DT, bool SEP>
constexpr bool bwd_latents_in_regs() { return sizeof(T) == 2 ? DT <= 4 : DT <= (SEP ? 2 : 3); }

// Nothing is scheduled across: keeps a stage's operands from being loaded stages early, which
// is what the registers cannot hold.
template <int DT>
__device__ __forceinline__ void stage() {
    if constexpr (DT >= 4) __builtin_amdgcn_sched_barrier(0);
}

// fp32 array of one (b, h) through a buffer descriptor (see Bytes).
struct Floats {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Floats(const float* p, size_t n)
        : r(__builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(n * sizeof(float)), 0x00020000)) {}
    __device__ __forceinline__ float load(unsigned byte) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, byte, 0, 0));
    }
    __device__ __forceinline__ void store(unsigned byte, float x) const {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, byte, 0, 0);
    }
};

// One tile's token rows (K, V, g and, for separate decoder weights, Q_dec) in LDS, shared by
// the workgroup's waves: read from memory once, and held in no wave's registers.  Rows are
// padded by 16 bytes (the operand reads go down 16 rows).  The next tile travels in a few
// registers a thread while the current one is worked on.
template <typename T, int DT, bool SEP>
struct TileRows {
    static constexpr int D = 16 * DT;
    // (fp32 rows of 128: the backward walk's LDS has no room for Q_dec, read from cache there)
    static constexpr bool QD = SEP && !(sizeof(T) == 4 && DT == 8);
    static constexpr int R = QD ? 4 : 3;
    static constexpr int CPR = D * (int)sizeof(T) / 16;             // 16-byte pieces a row
    static constexpr int PITCH = D + 16 / (int)sizeof(T);           // elements
    static constexpr int CHUNKS = TT * CPR;                         // pieces of one array's tile
    static constexpr int PF = sizeof(T) == 2 ? 1 : 2;               // pieces of an array a thread can hold
    static constexpr size_t BYTES = (size_t)R * TT * PITCH * sizeof(T);
    u32x4 held[R][PF];
    static __device__ __forceinline__ u32x4 piece(const T* p, int stride, int x, int t, int t1) {
        return reinterpret_cast<const u32x4*>(p + (size_t)min(t + x / CPR, t1 - 1) * stride)[x % CPR];
    }
    static __device__ __forceinline__ void put(T* lds, int x, u32x4 val) {
        *reinterpret_cast<u32x4*>(lds + (x / CPR) * PITCH + (x % CPR) * (16 / (int)sizeof(T))) = val;
    }
    static __device__ __forceinline__ bool holds() { return CHUNKS <= PF * (int)blockDim.x; }
    __device__ __forceinline__ void fetch(const BwdPtrs& a, size_t tok, int stride, int t, int t1) {
        if (!holds()) return;
#pragma unroll
        for (int n = 0; n < PF; ++n) {
            const int x = min((int)(threadIdx.x + n * blockDim.x), CHUNKS - 1);
            held[0][n] = piece((const T*)a.K + tok, stride, x, t, t1);
            held[1][n] = piece((const T*)a.V + tok, stride, x, t, t1);
            held[2][n] = piece((const T*)a.dY + tok, stride, x, t, t1);
            if constexpr (QD) held[3][n] = piece((const T*)a.Qdec + tok, stride, x, t, t1);
        }
    }
    __device__ __forceinline__ void store(T* lds, const BwdPtrs& a, size_t tok, int stride, int t, int t1) {
        constexpr int A = TT * PITCH;                               // elements of one array's tile
        if (holds()) {
#pragma unroll
            for (int n = 0; n < PF; ++n) {
                const int x = threadIdx.x + n * blockDim.x;
                if (x < CHUNKS) {
#pragma unroll
                    for (int k = 0; k < R; ++k) put(lds + k * A, x, held[k][n]);
                }
            }
        } else {
            for (int x = threadIdx.x; x < CHUNKS; x += blockDim.x) {
                put(lds, x, piece((const T*)a.K + tok, stride, x, t, t1));
                put(lds + A, x, piece((const T*)a.V + tok, stride, x, t, t1));
                put(lds + 2 * A, x, piece((const T*)a.dY + tok, stride, x, t, t1));
                if constexpr (QD) put(lds + 3 * A, x, piece((const T*)a.Qdec + tok, stride, x, t, t1));
            }
        }
    }
    static __device__ __forceinline__ const T* row(const T* lds, int a, int r) { return lds + (a * TT + r) * PITCH; }
};

// ---------------------------------------------------------------------------
// Decoder log-sum-exp of every token.  One wave takes 64 tokens against all latents; the
// latents' rows come from cache.
// ---------------------------------------------------------------------------
constexpr int kLseTiles = 4;
template <typename T, int DT>
__global__ __launch_bounds__(256) void wave_lse_kernel(const T* __restrict__ Qd, const T* __restrict__ Kd, int N, int H,
                                                       int M, float scale, float* __restrict__ lse) {
    constexpr int D = 16 * DT;
    const int bh = blockIdx.y, b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int t0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * TT * kLseTiles;
    if (t0 >= N) return;
    GroupRow<T, DT> k[kLseTiles];
    float mx[kLseTiles], sum[kLseTiles];
#pragma unroll
    for (int j = 0; j < kLseTiles; ++j) {
        k[j].load(Qd + (((size_t)b * N + min(t0 + TT * j + c, N - 1)) * H + h) * D, g);
        mx[j] = kNegInf;
        sum[j] = 0.0f;
    }
    for (int m0 = 0; m0 < M; m0 += 16) {
        GroupRow<T, DT> q;
        q.load(Kd + ((size_t)h * M + min(m0 + c, M - 1)) * D, g);
#pragma unroll
        for (int j = 0; j < kLseTiles; ++j) {
            f32x4 s = dot_groups(q, k[j], f32x4{0.f, 0.f, 0.f, 0.f});
            float top = mx[j];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = m0 + 4 * g + i < M ? s[i] * scale : kNegInf;
                top = fmaxf(top, s[i]);
            }
            const float ref = safe_ref(top);
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = exp_nat(s[i] - ref);
            sum[j] = sum[j] * exp_nat(mx[j] - ref) + ((e[0] + e[1]) + (e[2] + e[3]));      // (one rounding of the sum)
            mx[j] = top;
        }
    }
#pragma unroll
    for (int j = 0; j < kLseTiles; ++j) {
        const float top = group_max(mx[j]), ref = safe_ref(top);
        const float all = group_sum(sum[j] * exp_nat(mx[j] - ref));
        const int t = t0 + TT * j + c;
        if (g == 0 && t < N) lse[(size_t)bh * N + t] = ref + __logf(all);
    }
}

template <typename T>
constexpr bool own_gy() { return sizeof(T) == 4; }
// g . y of a tile: each wave's sums over its latents meet in LDS at the tile's barrier.
// sums: [2][waves][16], the half of the tile's row buffer.
__device__ __forceinline__ void put_gy(float* sums, const float (&v)[4], int wv, int g, int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float r = mfma::row_sum16(v[i]);
        if (c == 0) sums[wv * TT + 4 * g + i] = r;
    }
}
__device__ __forceinline__ void store_gy(const float* sums, int NW, float* gy, int t, int t1) {
    const int i = threadIdx.x;
    if (i < TT && t + i < t1) {
        float r = 0.0f;
        for (int k = 0; k < NW; ++k) r += sums[k * TT + i];
        gy[t + i] = r;
    }
}

// ---------------------------------------------------------------------------
// Forward walk of a chunk: gz, tile states, the chunk's X and Y.  grid (NC, B*H), one wave
// per MT*16 latents; the waves share a tile's rows and exchange nothing else.
//
// j < 0: the whole tile.  j >= 0: the tile is being walked token by token (see kTileJump) and
// j is the token; the loop then comes back with the same tile.  (As an inner loop over
// tokens this took 45 to 60 registers more.)
// ---------------------------------------------------------------------------
template <typename T, int MT, int DT, bool SEP, int P>
__global__ __launch_bounds__(64 * (16 / MT)) void wave_gz_kernel(BwdPtrs a, int N, int H, int M, float scale, int chunk) {
    constexpr int D = 16 * DT;
    typedef typename ProdOf<T, P>::F F;
    typedef TileRows<T, DT, SEP> Rows;
    constexpr bool QREG = bwd_latents_in_regs<T, DT, SEP>(), OWN_GY = own_gy<T>(), FLAT = sizeof(T) == 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];
    const int ch = blockIdx.x, NC = gridDim.x, bh = blockIdx.y;
    const int b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, NW = blockDim.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = wv * 16 * MT;
    const int NT = (N + TT - 1) / TT;
    const int t0 = ch * chunk, t1 = min(N, t0 + chunk);
    const int stride = H * D;
    const size_t tok = ((size_t)b * N * H + h) * D;
    // this (b, h)'s rows of the per-token arrays, reached by 32-bit offsets
    const Floats gz_out(a.gz + (size_t)bh * N * M, (size_t)N * M), lse_in(a.lse + (size_t)bh * N, N);
    unsigned lat[MT];                             // byte offset of this lane's latent in a row
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) lat[mt] = mb + 16 * mt + c < M ? 4u * (mb + 16 * mt + c) : kNowhere;

    GroupRow<T, DT> q[QREG ? MT : 1], kd[SEP && QREG ? MT : 1];
    auto latent_row = [&](GroupRow<T, DT>& r, const void* base, int mt) {
        // (past the bank: its last row; such a latent has no decoder weight and is never stored)
        r.load((const T*)base + ((size_t)h * M + min(mb + 16 * mt + c, M - 1)) * D, g);
    };
    float mx[MT], den[MT], er[MT], ysum[MT];      // er = e^(max at the chunk's start - mx)
    f32x4 u[MT][DT], x[MT][DT];
    const size_t pbase = ((size_t)bh * NC + ch) * M;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mb + 16 * mt + c;
        const bool in = m < M;
        if constexpr (QREG) {
            latent_row(q[mt], a.Q, mt);
            if constexpr (SEP) latent_row(kd[mt], a.Kdec, mt);
        }
        mx[mt] = in ? a.pmax[pbase + m] : kNegInf;
        den[mt] = in ? a.pden[pbase + m] : 0.0f;
        er[mt] = mx[mt] == kNegInf ? 0.0f : 1.0f;
        ysum[mt] = 0.0f;
        GroupRow<float, DT, FLAT> r;
        if (in) r.load(a.pnum + (pbase + m) * D, g);
        else r.zero();
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) u[mt][dt][i] = r.at(list_at<DT, FLAT>(dt, i));
            x[mt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }

    Rows rows;
    rows.fetch(a, tok, stride, t0, t1);
    rows.store((T*)tile_lds, a, tok, stride, t0, t1);
    __syncthreads();
    int buf = 0, t = t0, j = -1;
    float* gsum = reinterpret_cast<float*>(tile_lds + 2 * Rows::BYTES);
    float* gy_out = a.gy + (size_t)bh * N;
    float gy[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    while (true) {
        const T* tl = (const T*)(tile_lds + buf * Rows::BYTES);
        if (j <= 0 && t + TT < t1) rows.fetch(a, tok, stride, t + TT, t1);
        float s[MT][4], al[MT][4], top[MT], lse[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) lse[i] = lse_in.load(4u * (t + 4 * g + i));
        bool slow = false;
        {
            GroupRow<T, DT> kr;
            kr.load(Rows::row(tl, 0, c), g);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if constexpr (!QREG) latent_row(q[0], a.Q, mt);
                const f32x4 r = dot_groups(kr, q[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
                top[mt] = kNegInf;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[mt][i] = t + 4 * g + i < t1 ? r[i] * scale : kNegInf;
                    top[mt] = fmaxf(top[mt], s[mt][i]);
                }
                top[mt] = group_max(top[mt]);
                const float low = mx[mt] == kNegInf ? __shfl(s[mt][0], c, 64) : mx[mt];
                slow |= !(top[mt] - low <= kTileJump) && mb + 16 * mt + c < M;
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            f32x4 z = {s[mt][0], s[mt][1], s[mt][2], s[mt][3]};
            if constexpr (SEP) {
                GroupRow<T, DT> qr;
                qr.load(Rows::QD ? Rows::row(tl, 3, c) : (const T*)a.Qdec + tok + (size_t)min(t + c, t1 - 1) * stride, g);
                if constexpr (!QREG) latent_row(kd[0], a.Kdec, mt);
                z = dot_groups(qr, kd[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int i = 0; i < 4; ++i) z[i] *= scale;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) al[mt][i] = t + 4 * g + i < t1 && lat[mt] != kNowhere ? exp_nat(z[i] - lse[i]) : 0.0f;
        }
        stage<DT>();
        // g_t . v_tau as the [t][tau] factor of sums over tau (C rows tau, lane column t)
        F gvf;
        float bad;
        WalkRow<T, DT> gr;
        gr.load(Rows::row(tl, 2, c), g);
        {
            WalkRow<T, DT> vr;
            vr.load(Rows::row(tl, 1, c), g);
            const f32x4 r = dot_groups(vr, gr, f32x4{0.f, 0.f, 0.f, 0.f});
            // a value of g that is not finite shows in its products with v (0 times it is NaN); the
            // backward walk then keeps it to its own token (see WildCols)
            bad = __builtin_fmaf(r[0], 0.0f, __builtin_fmaf(r[1], 0.0f, __builtin_fmaf(r[2], 0.0f, r[3] * 0.0f)));
            gvf = factor<F>(4 * g <= c ? r[0] : 0.0f, 4 * g + 1 <= c ? r[1] : 0.0f, 4 * g + 2 <= c ? r[2] : 0.0f,
                            4 * g + 3 <= c ? r[3] : 0.0f);
        }
        if (j <= 0) {
            const bool step = __any(slow || bad != bad);
            if (lane == 0) a.stepwise[((size_t)bh * NT + t / TT) * NW + wv] = step;
            j = __any(slow) ? 0 : -1;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                if (g == 0 && mb + 16 * mt + c < M) {
                    const size_t ti = ((size_t)bh * NT + t / TT) * M + mb + 16 * mt + c;
                    a.tmax[ti] = mx[mt];
                    a.tden[ti] = den[mt];
                }
        }
        F ef[MT], wf[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            stage<DT>();
            const float mnew = fmaxf(mx[mt], j >= 0 ? token_value(s[mt], j, c) : top[mt]);
            if (__any(mnew != mx[mt])) {
                const float r = mx[mt] == mnew ? 1.0f : mx[mt] == kNegInf ? 0.0f : exp_nat(mx[mt] - mnew);
                den[mt] *= r;
                er[mt] *= r;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) u[mt][dt][i] *= r;
                mx[mt] = mnew;
            }
            const float ref = safe_ref(mx[mt]);
            float e[4], d[4], run = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float ev = exp_nat(s[mt][i] - ref);
                e[i] = j < 0 || 4 * g + i == j ? ev : 0.0f;
                run += e[i];
                d[i] = run;
            }
            float below, above, all;
            group_scan(run, g, below, above, all);
            ef[mt] = factor<F>(e[0], e[1], e[2], e[3]);
            f32x4 p = dot_state<T, DT, P>(gr, u[mt], f32x4{0.f, 0.f, 0.f, 0.f});
            p = mm(gvf, ef[mt], p);
            float w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float dv = den[mt] + below + d[i];
                const float inv = __builtin_amdgcn_rcpf(dv > 0.0f ? dv : 1.0f);
                const bool on = j < 0 || 4 * g + i == j;
                const float gz = p[i] * inv;
                w[i] = on ? al[mt][i] * er[mt] * inv : 0.0f;      // (al is 0 past the sequence)
                ysum[mt] += w[i] == 0.0f ? 0.0f : w[i] * gz;
                if constexpr (OWN_GY) gy[i] += on && al[mt][i] != 0.0f ? al[mt][i] * gz : 0.0f;
                gz_out.store(on ? 4u * M * (t + 4 * g + i) + lat[mt] : kNowhere, gz);
            }
            den[mt] += all;
            wf[mt] = factor<F>(w[0], w[1], w[2], w[3]);
        }
        // U += E^T V, X += W^T g, a piece of value columns at a time
#pragma unroll
        for (int st = 0, d0 = 0; st < steps<T, DT>(); d0 = step_start<T, DT>(++st)) {
            stage<DT>();
            TileCols<T, DT> vc, gc;
            vc.load_piece(Rows::row(tl, 1, 0), Rows::PITCH, g, c, d0);
            gc.load_piece(Rows::row(tl, 2, 0), Rows::PITCH, g, c, d0);
#pragma unroll
            for (int dt = d0; dt < d0 + step_most<T>(); ++dt) {
                if (dt >= d0 + step_of<T, DT>(d0)) continue;
                const auto vo = vc.op(dt), go = gc.op(dt);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    u[mt][dt] = collect(vo, ef[mt], u[mt][dt]);
                    x[mt][dt] = collect(go, wf[mt], x[mt][dt]);
                }
            }
        }
        if (j >= 0 && ++j < min(TT, t1 - t)) continue;
        j = -1;
        float* sums = gsum + buf * NW * TT;
        if constexpr (OWN_GY) {
            put_gy(sums, gy, wv, g, c);
            gy[0] = gy[1] = gy[2] = gy[3] = 0.0f;
        }
        t += TT;
        buf ^= 1;
        if (t < t1) rows.store((T*)(tile_lds + buf * Rows::BYTES), a, tok, stride, t, t1);
        __syncthreads();
        if constexpr (OWN_GY) store_gy(sums, NW, gy_out, t - TT, t1);
        if (t >= t1) break;
    }
    set_wild<T, MT, DT>(x, (const T*)a.dY + tok, stride, t0, t1, g);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        ysum[mt] = group_sum(ysum[mt]);
        const int m = mb + 16 * mt + c;
        if (m < M) {
            if (g == 0) a.ysum[pbase + m] = ysum[mt];
            float* row = a.xsum + (pbase + m) * D;
#pragma unroll
            for (int pc = 0, dt = 0; pc < walk_pieces<DT, FLAT>(); dt = walk_start<DT, FLAT>(++pc))
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k < walk_piece<DT, FLAT>(dt))
                            row[walk_col<DT, FLAT>(dt, 4 * g + i) + k] = x[mt][dt + k < DT ? dt + k : 0][i];
        }
    }
}

// ---------------------------------------------------------------------------
// Reverse scan over chunks: the terms of chunk c (relative to the max at its start) become
// X, Y after chunk c (relative to the max at its end, the next chunk's start).  One thread
// per (b*h, latent, value column), and one more column for Y.
// ---------------------------------------------------------------------------
static __global__ __launch_bounds__(256) void wave_carry_kernel(float* __restrict__ xsum, float* __restrict__ ysum,
                                                         const float* __restrict__ pmax, int NC, int M, int D, int64_t rows) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;      // (65,535 (b, h) of 256 x 129 pass 2^31)
    if (gid >= rows * (D + 1)) return;
    const int64_t row = gid / (D + 1);
    const int col = (int)(gid % (D + 1)), bh = (int)(row / M), m = (int)(row % M);
    float run = 0.0f, mnext = 0.0f;       // X after chunk ch, relative to mnext = pmax of chunk ch + 1
    constexpr int BATCH = 8;
    for (int c1 = NC; c1 > 0; c1 -= BATCH) {
        float v[BATCH], mm[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const int ch = c1 - 1 - k;
            const size_t si = ((size_t)bh * NC + max(ch, 0)) * M + m;
            v[k] = col < D ? xsum[si * D + col] : ysum[si];
            mm[k] = pmax[si];
        }
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const int ch = c1 - 1 - k;
            if (ch < 0) break;
            const size_t si = ((size_t)bh * NC + ch) * M + m;
            if (col < D) xsum[si * D + col] = run;
            else ysum[si] = run;
            // relative to this chunk's start (a first chunk starts at -inf and has no reader)
            const float f = ch + 1 < NC && mm[k] != kNegInf ? exp_nat(mm[k] - mnext) : 0.0f;
            run = v[k] + (f > 0.0f ? run * f : 0.0f);
            mnext = mm[k];
        }
    }
}

// ---------------------------------------------------------------------------
// Backward walk of a chunk: ds and dv.  grid (NC, B*H), one wave per MT*16 latents.  Whether
// a tile is walked token by token is read from the forward walk's marks, for the whole
// workgroup alike (its waves add their dv rows at barriers).
// ---------------------------------------------------------------------------
constexpr int dv_pitch(int DT) { return 16 * DT + 4; }
// X tiles a wave has in LDS at a time: three parts of 96 or 128 columns leave room for one (eight
// waves of two took 160 and 209 KB)
template <typename T, int DT, int P>
__host__ __device__ constexpr bool one_x_tile() { return sizeof(T) == 2 && P == 3 && DT > 4; }
template <typename T, int MT, int DT, int P>
__host__ __device__ constexpr int ds_wave_floats() {      // wave-private LDS: X tiles, or the e / w tiles, or dv rows
    const int xt = (one_x_tile<T, DT, P>() ? 1 : MT) * StateTile<T, DT, P>::FLOATS;
    const int ew = 2 * MT * TurnTile<T, P>::FLOATS, dv = TT * dv_pitch(DT);
    const int a = xt > ew ? xt : ew;
    return a > dv ? a : dv;
}

template <typename T, int MT, int DT, bool SEP, int P>
__global__ __launch_bounds__(64 * (16 / MT)) void wave_ds_kernel(BwdPtrs a, int N, int H, int M, float scale, int chunk) {
    constexpr int D = 16 * DT, VP = dv_pitch(DT), WF = ds_wave_floats<T, MT, DT, P>();
    constexpr bool FLAT = sizeof(T) == 2, ONE = one_x_tile<T, DT, P>();
    typedef StateTile<T, DT, P> XTile;
    typedef TurnTile<T, P> Turn;
    constexpr int OD = sizeof(T) == 4 ? FLARE_F32 : __is_same(T, __half) ? FLARE_F16 : FLARE_BF16;
    typedef typename ProdOf<T, P>::F F;
    typedef TileRows<T, DT, SEP> Rows;
    constexpr bool QREG = bwd_latents_in_regs<T, DT, SEP>();
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int ch = blockIdx.x, NC = gridDim.x, bh = blockIdx.y;
    const int b = bh / H, h = bh % H;
    const int NW = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = wv * 16 * MT;
    const int NT = (N + TT - 1) / TT;
    const int t0 = ch * chunk, t1 = min(N, t0 + chunk);
    const int stride = H * D;
    const size_t tok = ((size_t)b * N * H + h) * D;
    T* tl = reinterpret_cast<T*>(smem + NW * WF);
    float* own = smem + wv * WF;
    float *etile = own, *wtile = own + MT * Turn::FLOATS, *xtile = own, *vtile = own;
    const size_t per = (size_t)N * M;
    const Floats gz_in(a.gz + bh * per, per), lse_in(a.lse + (size_t)bh * N, N), gy_in(a.gy + (size_t)bh * N, N);
    const Floats ds_out(a.ds + bh * per, per), al_out(SEP ? a.al + bh * per : a.ds, SEP ? per : 0);
    const Floats tmax_in(a.tmax + (size_t)bh * NT * M, (size_t)NT * M), tden_in(a.tden + (size_t)bh * NT * M, (size_t)NT * M);
    unsigned lat[MT];                             // byte offset of this lane's latent in a row
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) lat[mt] = mb + 16 * mt + c < M ? 4u * (mb + 16 * mt + c) : kNowhere;

    GroupRow<T, DT> q[QREG ? MT : 1], kd[SEP && QREG ? MT : 1];
    auto latent_row = [&](GroupRow<T, DT>& r, const void* base, int mt) {
        // (past the bank: its last row; such a latent has no decoder weight and is never stored)
        r.load((const T*)base + ((size_t)h * M + min(mb + 16 * mt + c, M - 1)) * D, g);
    };
    float mref[MT], ysum[MT];
    f32x4 x[MT][DT];
    const size_t pbase = ((size_t)bh * NC + ch) * M;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mb + 16 * mt + c;
        if constexpr (QREG) {
            latent_row(q[mt], a.Q, mt);
            if constexpr (SEP) latent_row(kd[mt], a.Kdec, mt);
        }
        const bool tail = m < M && ch + 1 < NC;
        mref[mt] = tail ? a.pmax[pbase + M + m] : 0.0f;
        ysum[mt] = tail ? a.ysum[pbase + m] : 0.0f;
        GroupRow<float, DT, FLAT> r;
        if (tail) r.load(a.xsum + (pbase + m) * D, g);
        else r.zero();
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[mt][dt][i] = r.at(list_at<DT, FLAT>(dt, i));
    }

    __shared__ unsigned wild_bits[8];
    if (threadIdx.x < 8) wild_bits[threadIdx.x] = 0;

    Rows rows;
    int t = t0 + (t1 - 1 - t0) / TT * TT, j = -1;
    rows.fetch(a, tok, stride, t, t1);
    rows.store(tl, a, tok, stride, t, t1);
    __syncthreads();
    bool some_wild = find_wild<T, MT, DT>(x, wild_bits, g);
    while (true) {
        const bool begin = j < 0;
        if (begin) {
            if (t > t0) rows.fetch(a, tok, stride, t - TT, t1);
            const int mark = a.stepwise[((size_t)bh * NT + t / TT) * NW + min(lane, NW - 1)];
            j = __any(mark) ? min(TT, t1 - t) - 1 : -1;
        }
        float s[MT][4], top[MT], m0[MT], d0[MT], gz[MT][4], lse[4], gy[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lse[i] = lse_in.load(4u * (t + 4 * g + i));
            gy[i] = SEP ? 0.0f : gy_in.load(4u * (t + 4 * g + i));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) gz[mt][i] = gz_in.load(4u * M * (t + 4 * g + i) + lat[mt]);
        }
        {
            GroupRow<T, DT> kr;
            kr.load(Rows::row(tl, 0, c), g);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                m0[mt] = tmax_in.load(4u * M * (t / TT) + lat[mt]);
                d0[mt] = tden_in.load(4u * M * (t / TT) + lat[mt]);
                if constexpr (!QREG) latent_row(q[0], a.Q, mt);
                const f32x4 r = dot_groups(kr, q[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
                top[mt] = kNegInf;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[mt][i] = t + 4 * g + i < t1 ? r[i] * scale : kNegInf;
                    top[mt] = fmaxf(top[mt], s[mt][i]);
                }
                top[mt] = group_max(top[mt]);
            }
        }
        stage<DT>();
        // g_t . v_tau as the [tau][t] factor of sums over t (C rows t, lane column tau)
        WalkRow<T, DT> vr;
        vr.load(Rows::row(tl, 1, c), g);
        F gvf;
        {
            WalkRow<T, DT> gr;
            gr.load(Rows::row(tl, 2, c), g);
            const f32x4 r = dot_groups(gr, vr, f32x4{0.f, 0.f, 0.f, 0.f});
            gvf = factor<F>(4 * g >= c ? r[0] : 0.0f, 4 * g + 1 >= c ? r[1] : 0.0f, 4 * g + 2 >= c ? r[2] : 0.0f,
                            4 * g + 3 >= c ? r[3] : 0.0f);
        }
        F wf[MT];
        float e[MT][4], ysuf[MT][4], dec[MT][4];          // Y at the token; the decoder's part of ds
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            stage<DT>();
            f32x4 z = {s[mt][0], s[mt][1], s[mt][2], s[mt][3]};
            if constexpr (SEP) {
                GroupRow<T, DT> qr;
                qr.load(Rows::QD ? Rows::row(tl, 3, c) : (const T*)a.Qdec + tok + (size_t)min(t + c, t1 - 1) * stride, g);
                if constexpr (!QREG) latent_row(kd[0], a.Kdec, mt);
                z = dot_groups(qr, kd[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int i = 0; i < 4; ++i) z[i] *= scale;
            }
            // the max after the tile; token by token, the max and the den at token j
            float mc = fmaxf(m0[mt], top[mt]), dj = 1.0f;
            if (j >= 0) {
                mc = m0[mt];
                dj = d0[mt];
                for (int k = 0; k <= j; ++k) {
                    const float sk = token_value(s[mt], k, c), mn = fmaxf(mc, sk), r = safe_ref(mn);
                    dj = (mc == kNegInf ? 0.0f : dj * exp_nat(mc - r)) + exp_nat(sk - r);
                    mc = mn;
                }
            }
            const float ref = safe_ref(mc);
            if (__any(ref != mref[mt])) {
                // (the max falls as the walk goes back; the bound keeps a last chunk's zeros zero)
                const float r = exp_nat(fminf(ref - mref[mt], 1.0f));
                ysum[mt] *= r;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[mt][dt][i] *= r;
                mref[mt] = ref;
            }
            float d[4], al[4], w[4], wg[4], run = 0.0f, wrun = 0.0f, below, above, all;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float ev = exp_nat(s[mt][i] - ref);
                e[mt][i] = j < 0 || 4 * g + i == j ? ev : 0.0f;
                run += e[mt][i];
                d[i] = run;
                al[i] = t + 4 * g + i < t1 && lat[mt] != kNowhere ? exp_nat(z[i] - lse[i]) : 0.0f;
                if constexpr (SEP) al_out.store(4u * M * (t + 4 * g + i) + lat[mt], al[i]);
            }
            group_scan(run, g, below, above, all);
            const float start = m0[mt] == kNegInf ? 0.0f : d0[mt] * exp_nat(m0[mt] - ref);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float dd = j >= 0 ? dj : start + below + d[i];
                w[i] = j < 0 || 4 * g + i == j ? al[i] * __builtin_amdgcn_rcpf(dd > 0.0f ? dd : 1.0f) : 0.0f;
                wg[i] = w[i] == 0.0f ? 0.0f : w[i] * gz[mt][i];
                wrun += wg[i];
            }
            group_scan(wrun, g, below, above, all);
            wf[mt] = factor<F>(w[0], w[1], w[2], w[3]);
            // Y at token 4g + i: later tokens and itself
            float suffix = ysum[mt] + above;
#pragma unroll
            for (int i = 3; i >= 0; --i) {
                suffix += wg[i];
                ysuf[mt][i] = suffix;
                dec[mt][i] = SEP ? 0.0f : al[i] * (gz[mt][i] - gy[i]);
            }
            ysum[mt] += all;
            Turn::put(etile + mt * Turn::FLOATS, factor<F>(e[mt][0], e[mt][1], e[mt][2], e[mt][3]), g, c);
            Turn::put(wtile + mt * Turn::FLOATS, wf[mt], g, c);
        }
        wave_lds_sync();
        F ef[MT];
        f32x4 G = {0.f, 0.f, 0.f, 0.f};       // [t][tau] summed over this wave's latents
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            ef[mt] = Turn::get(etile + mt * Turn::FLOATS, g, c);
            G = mm(Turn::get(wtile + mt * Turn::FLOATS, g, c), ef[mt], G);
        }
        wave_lds_sync();
        f32x4 dv[DT];                         // rows = value columns, lane column = token
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            stage<DT>();
            float* xt = xtile + (ONE ? 0 : mt * XTile::FLOATS);
            f32x4 xz = XTile::put_dot(xt, vr, x[mt], g, c, f32x4{0.f, 0.f, 0.f, 0.f});
            xz = mm(gvf, wf[mt], xz);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float r = SEP ? e[mt][i] * (xz[i] - ysuf[mt][i]) : e[mt][i] * (xz[i] - ysuf[mt][i]) + dec[mt][i];
                ds_out.store(j < 0 || 4 * g + i == j ? 4u * M * (t + 4 * g + i) + lat[mt] : kNowhere, r);
            }
            if constexpr (ONE) {
                wave_lds_sync();
                add_state_product<XTile, T, DT>(dv, xt, ef[mt], mt == 0, g, c);
                wave_lds_sync();
            }
        }
        wave_lds_sync();
        // (whole in every 16-bit instance: rounded to two parts it alone put dV of short sequences 5
        // to 40% further off where the states are two parts)
        typedef typename ProdOf<T, 3>::F Whole;
        const Whole gf = factor<Whole>(4 * g >= c ? G[0] : 0.0f, 4 * g + 1 >= c ? G[1] : 0.0f, 4 * g + 2 >= c ? G[2] : 0.0f,
                                       4 * g + 3 >= c ? G[3] : 0.0f);
        // dv and X += W^T g, a piece of value columns at a time.  Token by token the other tokens' g,
        // which may not be finite, are taken as zero.  (A select each time and no branch: after a
        // branch around it the compiler reads the product above too early on the skipped side.)
        bool on[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) on[i] = j < 0 || 4 * g + i == j;
#pragma unroll
        for (int st = 0, d1 = 0; st < steps<T, DT>(); d1 = step_start<T, DT>(++st)) {
            stage<DT>();
            typename XTile::Cols xc[ONE ? 1 : MT];
            TileCols<T, DT> gc;
            gc.load_piece(Rows::row(tl, 2, 0), Rows::PITCH, g, c, d1);
            if constexpr (!ONE) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) xc[mt].load_piece(xtile + mt * XTile::FLOATS, g, c, d1);
            }
            gc.keep(on, d1);
#pragma unroll
            for (int dt = d1; dt < d1 + step_most<T>(); ++dt) {
                if (dt >= d1 + step_of<T, DT>(d1)) continue;
                f32x4 r = {0.f, 0.f, 0.f, 0.f};
                if constexpr (ONE) {
                    r = dv[dt];
                } else {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) r = mm(xc[mt].op(dt), ef[mt], r);
                }
                const auto go = gc.op(dt);
                dv[dt] = mm(go, gf, r);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[mt][dt] = collect(go, wf[mt], x[mt][dt]);
            }
        }
        // rows of this pass; the tile's last pass brings the next tile in
        const bool last = j <= 0, more = last && t > t0;
        wave_lds_sync();
        put_rows<DT, FLAT>(vtile, VP, dv, g, c);
        if (j >= 0 || some_wild) {
            // (a token whose g is not finite is walked by itself)
            if (j >= 0) {
                WildCols<T, DT> wild;
                wild.take_row(Rows::row(tl, 2, j), g);
                wild.add_to(wild_bits, g);
            }
            some_wild = put_wild<T, DT>(vtile, VP, wild_bits, g, c);
        }
        if (NW == 1) {
            wave_lds_sync();
            if (more) rows.store(tl, a, tok, stride, t - TT, t1);
        } else {
            __syncthreads();
            if (more) rows.store(tl, a, tok, stride, t - TT, t1);      // every wave is done with this tile's rows
        }
        for (int e = threadIdx.x; e < TT * D / 4; e += blockDim.x) {
            const int ti = e / (D / 4), col = 4 * (e % (D / 4));
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            for (int k = 0; k < NW; ++k) {
                const f32x4 r = *reinterpret_cast<const f32x4_a*>(smem + k * WF + ti * VP + col);
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[n] += r[n];
            }
            const float o[4] = {acc[0], acc[1], acc[2], acc[3]};
            if (t + ti < t1 && (j < 0 || ti == j)) store_cols<4>(a.dV, tok + (size_t)(t + ti) * stride + col, o, OD);
        }
        if (NW == 1) wave_lds_sync();
        else __syncthreads();
        if (!last) {
            --j;
            continue;
        }
        if (!more) break;
        j = -1;
        t -= TT;
    }
}

}  // namespace wave
}  // namespace flare
