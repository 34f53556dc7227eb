// flare_wave.h -- chunked causal FLARE forward with wave-private latents and fp32 matrix
// products (phases 1 and 3; phase 2 is chunk_prefix_kernel).
//
// Serves fp32 inputs of every bank and 16-bit inputs of the banks that have no instance of
// the 16-bit kernels in flare_ar_prep.hip / flare_ar_out.hip: M <= 256, Dk = Dv = 16 DT.
// Everything the tokenwise kernels (flare_ar.hip) hold in fp32 stays in fp32: the weights
// E and W, the numerator U and every product of them run on the fp32 MFMA (16x16x4); the
// scores of 16-bit inputs run on the 16-bit MFMA, whose products are exact.
//
// Why waves own latents: a wave holds MT*16 latents over all D value columns, so scores,
// running max, den, numerator and the in-tile products need no other wave; the waves of a
// workgroup only add their partial outputs, one barrier per 16-token tile (none when one
// wave holds the bank).  The operand layouts of v_mfma_f32_16x16x4 then make every product
// of a tile a register-to-register chain.  With lane = (g, c), g = lane / 16, c = lane % 16:
//   C of a product        row 4g + i (i = register), column c
//   A / B of a product    row (column) c, contraction index g; register i of a C tile is
//                         therefore the operand for contraction indices 4g + i.
//   scores^T [m][t], U [m][d], G^T [tau][t], y [t][d] are all C tiles; W and E contract over
//   m straight from the scores' registers, G over tau straight from its own.  Only E of the
//   U update needs the other orientation; it crosses through a wave-private LDS tile.
//
// What bounds it: the fp32 MFMA and the vector instructions together, which two waves a SIMD
// hardly overlap.  A 64 x 32 bank issues 88 MFMAs a 16-token tile and wave in phase 3 (2,816
// cycles of its SIMD's matrix pipe, busy 40% of the kernel) and about 880 vector instructions
// (52%).  Measured on MI355X, whole forward, tokenwise kernels -> these:
//   bf16 B 8, N 4096, H 16, M 64, D 32     4937 -> 158 us (prepare 41, scan 7, output 124)
//   fp16 B 3, N 1531, H 8, M 96, D 64, cached state and mask   1135 ->  72 us
//   fp32 B 1, N 256, H 8, M 64, D 32        283 ->  30 us
// Errors against 64 bits: fp32 outputs 2.5e-7 -> 1.1e-7, 16-bit ones unchanged.
#pragma once

#include "flare_common.h"
#include "flare_mfma.h"

namespace flare {
namespace wave {

using mfma::bf16x8;
using mfma::f32x4;
using mfma::kLog2e;

// Words as they are loaded: rows of any element type are read and written through these.
typedef unsigned u32;
typedef u32 u32_a __attribute__((may_alias));
typedef u32 u32x2 __attribute__((ext_vector_type(2), may_alias));
typedef u32 u32x4 __attribute__((ext_vector_type(4), may_alias));
typedef unsigned short u16_a __attribute__((may_alias));
typedef float f32x4_a __attribute__((ext_vector_type(4), may_alias));

constexpr int TT = 16;              // tokens per tile

// An array through a buffer descriptor: loads past its end read 0 and stores there are
// dropped, so edge tokens need no branches and no clamped addresses, and a lane's address is
// one 32-bit offset.  (A branch per element split the tile into some 130 blocks that nothing
// could be scheduled across: 144 us for phase 3 of the narrow bank above.)
constexpr unsigned kNowhere = 0x80000000u;                          // byte offset past every array
struct Bytes {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Bytes(const void* p, size_t n)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)n, 0x00020000)) {}
    __device__ __forceinline__ u32x4 b128(unsigned at) const {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
    }
    __device__ __forceinline__ u32x2 b64(unsigned at) const {
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0));
    }
    __device__ __forceinline__ unsigned b32(unsigned at) const { return __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0); }
    __device__ __forceinline__ unsigned b16(unsigned at) const {
        return (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0);
    }
    __device__ __forceinline__ void put128(unsigned at, u32x4 x) const {
        __builtin_amdgcn_raw_buffer_store_b128(x, r, at, 0, 0);
    }
    __device__ __forceinline__ void put64(unsigned at, u32x2 x) const { __builtin_amdgcn_raw_buffer_store_b64(x, r, at, 0, 0); }
    __device__ __forceinline__ void put32(unsigned at, unsigned x) const { __builtin_amdgcn_raw_buffer_store_b32(x, r, at, 0, 0); }
    __device__ __forceinline__ void put16(unsigned at, unsigned x) const {
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)x, r, at, 0, 0);
    }
};
// A latent's max may rise by this much (nats) inside a tile before the tile runs token by
// token: below it every den and weight of the tile keeps full fp32 precision against the
// tile's max (e^-60 is far above the fp32 underflow).
constexpr float kTileJump = 60.0f;

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Rows of D contraction elements as an MFMA operand: lane (g, c) holds its share of row c.
// ---------------------------------------------------------------------------
template <typename T, int D>
struct RowOp {   // 16-bit: steps of 32 columns, 8 a lane group; a last step of 16 fills two groups
    static constexpr int S = (D + 31) / 32;
    bf16x8 a[S];
    // byte offset of this lane within a row, and the load from it
    static __device__ __forceinline__ unsigned lane(int g) { return 16 * g; }
    __device__ __forceinline__ void load(const Bytes& b, unsigned row, int g) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (32 * s + 32 <= D) {
                a[s] = __builtin_bit_cast(bf16x8, b.b128(row + 64 * s));
            } else {
                // the groups past the row read nowhere: zeros
                a[s] = __builtin_bit_cast(bf16x8, b.b128(g < 2 ? row + 64 * s : kNowhere));
            }
        }
    }
};
template <int D>
struct RowOp<float, D> {   // lane group g holds columns [g D/4, (g+1) D/4)
    f32x4 a[D / 16];
    static __device__ __forceinline__ unsigned lane(int g) { return g * D; }
    __device__ __forceinline__ void load(const Bytes& b, unsigned row, int) {
#pragma unroll
        for (int s = 0; s < D / 16; ++s) a[s] = __builtin_bit_cast(f32x4, b.b128(row + 16 * s));
    }
};

// c += x . y^T over D (rows of x become C rows, rows of y C columns)
template <typename T, int D>
__device__ __forceinline__ f32x4 dot_rows(const RowOp<T, D>& x, const RowOp<T, D>& y, f32x4 c) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int s = 0; s < D / 16; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) c = mma4(x.a[s][e], y.a[s][e], c);
    } else {
        constexpr bool F16 = __is_same(T, __half);
#pragma unroll
        for (int s = 0; s < RowOp<T, D>::S; ++s) c = mfma::mma_in<F16>(x.a[s], y.a[s], c);
    }
    return c;
}

// ---------------------------------------------------------------------------
// Column tiles of a row of D = 16 DT values.  Which 16 columns make tile dt is free (a
// product only needs both sides to agree), so lane c takes consecutive columns, in pieces
// of 4, 2 and 1 tiles: loads and stores are as wide as the pieces.
// ---------------------------------------------------------------------------
// (closed forms: they fold away for a tile index known after unrolling)
template <int DT>
__host__ __device__ constexpr int piece_off(int dt) {  // first tile of the piece that holds tile dt
    constexpr int full = DT / 4 * 4;
    return dt < full ? (dt & ~3) : (DT - full == 3 && dt - full == 2) ? full + 2 : full;
}
template <int DT>
__host__ __device__ constexpr int piece_of(int dt) {   // size of that piece
    constexpr int full = DT / 4 * 4;
    return dt < full ? 4 : DT - full == 3 ? (dt - full < 2 ? 2 : 1) : DT - full;
}
// The pieces by number: a loop that steps by piece_of does not unroll for DT = 3 and 6, and the
// register arrays that its body indexes then lie in memory (up to 592 bytes a lane; a training
// step of fp32 B 1, N 2048, H 8, M 128, D 96 took 329 us so and takes 256, block-causal in blocks of
// 64 408 and 271, fp16 B 2, M 256, D 96 428 and 387).
template <int DT>
__host__ __device__ constexpr int pieces() { return DT / 4 + (DT % 4 == 0 ? 0 : DT % 4 == 3 ? 2 : 1); }
template <int DT>
__host__ __device__ constexpr int piece_start(int p) { return p <= DT / 4 ? 4 * p : DT / 4 * 4 + 2; }
// column of tile dt at lane c
template <int DT>
__device__ __forceinline__ int col_of(int dt, int c) {
    return 16 * piece_off<DT>(dt) + c * piece_of<DT>(dt) + (dt - piece_off<DT>(dt));
}

template <typename T>
__device__ __forceinline__ float word_f32(unsigned w, bool hi) {
    if constexpr (__is_same(T, __half)) {
        return (float)__builtin_bit_cast(mfma::f16, (unsigned short)(hi ? w >> 16 : w & 0xffffu));
    } else {
        return __builtin_bit_cast(float, hi ? (w & 0xffff0000u) : (w << 16));
    }
}

// One row's columns of lane c, raw (16-bit types stay packed until they are used).
template <typename T, int DT>
struct ColRow {
    static constexpr int W = sizeof(T) == 4 ? DT : (DT + 1) / 2;
    unsigned w[W];
    __device__ __forceinline__ void load(const T* row, int c) {
#pragma unroll
        for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc)) load_piece(row, c, dt);
    }
    // the columns of the piece that starts at tile dt
    __device__ __forceinline__ void load_piece(const T* row, int c, int dt) {
        const T* p = row + col_of<DT>(dt, c);
        const int P = piece_of<DT>(dt);
        const int at = sizeof(T) == 4 ? dt : dt / 2, words = sizeof(T) == 4 ? P : P / 2;
        if (words == 4) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (at + j < W) w[at + j] = x[j];
        } else if (words == 2) {
            const u32x2 x = *reinterpret_cast<const u32x2*>(p);
            w[at] = x[0];
            if (at + 1 < W) w[at + 1] = x[1];
        } else if (words == 1) {
            w[at] = *reinterpret_cast<const u32_a*>(p);
        } else {
            w[at] = *reinterpret_cast<const u16_a*>(p);
        }
    }
    // the same from a buffer: `row` is the row's byte offset
    __device__ __forceinline__ void load(const Bytes& b, unsigned row, int c) {
#pragma unroll
        for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc)) {
            const int P = piece_of<DT>(dt), E = (int)sizeof(T);
            const unsigned at = row + c * (P * E) + 16 * dt * E;
            const int k = sizeof(T) == 4 ? dt : dt / 2;
            if (P * E == 16) {
                const u32x4 x = b.b128(at);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (k + j < W) w[k + j] = x[j];
            } else if (P * E == 8) {
                const u32x2 x = b.b64(at);
                w[k] = x[0];
                if (k + 1 < W) w[k + 1] = x[1];
            } else if (P * E == 4) {
                w[k] = b.b32(at);
            } else {
                w[k] = b.b16(at);
            }
        }
    }
    __device__ __forceinline__ float get(int dt) const {
        if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, w[dt]);
        else return word_f32<T>(w[dt / 2], dt & 1);
    }
};

// x and x of the lane SWAP away (in some order), in every lane.
template <int SWAP>
__device__ __forceinline__ void lane_pair(float x, float& a, float& b) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    unsigned lo, hi;    // (bit casts need scalars: of a vector's element they read element 0)
    if constexpr (SWAP == 32) {
        auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        lo = r[0];
        hi = r[1];
    } else {
        auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        lo = r[0];
        hi = r[1];
    }
    a = __builtin_bit_cast(float, lo);
    b = __builtin_bit_cast(float, hi);
}
// sum / max over the four lane groups (lanes c, c + 16, c + 32, c + 48), in every lane
__device__ __forceinline__ float group_max(float x) {
    float a, b;
    lane_pair<32>(x, a, b);
    lane_pair<16>(fmaxf(a, b), a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float group_sum(float x) {
    float a, b;
    lane_pair<32>(x, a, b);
    lane_pair<16>(a + b, a, b);
    return a + b;
}

__device__ __forceinline__ float exp_nat(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }
__device__ __forceinline__ float safe_ref(float m) { return m == kNegInf ? 0.0f : m; }
// A reference of -inf (no token yet, every score -inf) counts as this, so that -inf - ref is
// -inf and not NaN; and a den of 0 (then U is 0 as well) as this.
constexpr float kLowRef = -1e38f, kTinyDen = 1e-37f;

// Writes by other lanes of the wave to LDS are visible after this (a wave's LDS
// operations complete in order; the fence keeps the compiler from reordering them).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Registers decide what a wave keeps at hand.  The latents' rows stay in registers unless
// they are fp32 rows of 96 columns or more (64 registers at D = 128): those are read again
// each tile, from cache.  The next tile's tokens are fetched ahead up to D = 64; beyond, the
// second wave of a SIMD covers the latency (fetching ahead spilled 92 to 764 bytes a lane).
// Without it wave_output still spills 216 bytes in fp32 at D = 128 with decoder weights of its own
// (16 with shared ones), and 12 to 56 in fp16 at D 96 and 128.
template <typename T, int DT, bool SEP>
constexpr bool latents_in_regs() { return sizeof(T) == 2 ? (DT <= 6 || !SEP) : (DT <= 3 || (DT == 4 && !SEP)); }
template <int DT>
constexpr bool fetch_ahead() { return DT <= 4; }
// Largest workgroup: M <= 256, and waves of 16 latents only up to M = 128 (a workgroup of 16
// waves would halve their registers).
__host__ __device__ constexpr int wave_threads(int MT) { return MT == 4 ? 256 : 512; }

// ---------------------------------------------------------------------------
// Phase 1: the summary (max, den, num) of one chunk.  grid = (NC, B*H), one wave per
// MT*16 latents.  Scores are taken as [tau][m] (C rows = tokens), which is the A operand of
// U^T += V^T E directly, and U^T keeps a latent in one lane column, so a moved max rescales
// it with per-lane factors.
// ---------------------------------------------------------------------------
template <typename T, int MT, int DT>
__global__ __launch_bounds__(wave_threads(MT)) void wave_prepare_kernel(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, int N, int H, int M, float scale,
    int chunk, float* __restrict__ cmax, float* __restrict__ cden, float* __restrict__ cnum,
    const int32_t* __restrict__ tmask) {
    constexpr int D = 16 * DT;
    const int ch = blockIdx.x, NC = gridDim.x, bh = blockIdx.y;
    const int b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = w * 16 * MT;

    constexpr bool QREG = latents_in_regs<T, DT, false>(), AHEAD = fetch_ahead<DT>();
    RowOp<T, D> q[QREG ? MT : 1];
    const Bytes qb(Q + (size_t)h * M * D, (size_t)M * D * sizeof(T));
    auto load_q = [&](RowOp<T, D>& r, int mt) {                  // past the bank: zeros
        r.load(qb, (mb + 16 * mt + c) * (D * (int)sizeof(T)) + RowOp<T, D>::lane(g), g);
    };
    if constexpr (QREG) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) load_q(q[mt], mt);
    }
    float mx[MT], den[MT];
    f32x4 u[MT][DT];       // U^T: row 4g + i is the value column col_of(dt, 4g + i), lane c the latent
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        mx[mt] = kNegInf;
        den[mt] = 0.0f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) u[mt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // the chunk's rows of this head, by byte offset from its first token
    const int t0 = ch * chunk, t1 = min(N, t0 + chunk);
    const unsigned stride = (unsigned)(H * D) * sizeof(T);
    const size_t first = (((size_t)b * N + t0) * H + h) * D;
    const size_t span = (size_t)(t1 - t0 - 1) * stride + D * sizeof(T);
    const Bytes kb(K + first, span), vb(V + first, span);
    unsigned krow = c * stride + RowOp<T, D>::lane(g), vrow = 4 * g * stride;
    RowOp<T, D> kn;
    ColRow<T, DT> vn[4];
    auto fetch = [&]() {                                          // (past the chunk: zeros)
        kn.load(kb, krow, g);
#pragma unroll
        for (int i = 0; i < 4; ++i) vn[i].load(vb, vrow + i * stride, c);
        krow += TT * stride;
        vrow += TT * stride;
    };
    if constexpr (AHEAD) fetch();
    for (int t = t0; t < t1; t += TT) {
        if constexpr (!AHEAD) fetch();
        const RowOp<T, D> k = kn;
        float v[4][DT];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) v[i][dt] = vn[i].get(dt);
        if constexpr (AHEAD) fetch();
        bool ok[4];                                               // token t + 4g + i takes part
#pragma unroll
        for (int i = 0; i < 4; ++i) ok[i] = t + 4 * g + i < t1;
        if (tmask != nullptr) {
            // (a masked token's value may be anything: it must not meet a weight of zero)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ok[i] = ok[i] && tmask[(size_t)b * N + min(t + 4 * g + i, t1 - 1)] != 0;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) v[i][dt] = ok[i] ? v[i][dt] : 0.0f;
            }
        }
        f32x4 e[MT];
        float mnew[MT];
        bool moved = false;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if constexpr (!QREG) load_q(q[0], mt);
            f32x4 s = dot_rows<T, D>(k, q[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
            float top = kNegInf;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = ok[i] ? s[i] * scale : kNegInf;
                top = fmaxf(top, s[i]);
            }
            mnew[mt] = fmaxf(mx[mt], group_max(top));
            moved |= mnew[mt] != mx[mt];
            e[mt] = s;
        }
        if (__any(moved)) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const float r = mx[mt] == kNegInf ? 0.0f : exp_nat(mx[mt] - mnew[mt]);
                den[mt] *= r;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) u[mt][dt][i] *= r;
                mx[mt] = mnew[mt];
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const float ref = safe_ref(mx[mt]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[mt][i] = exp_nat(e[mt][i] - ref);
                den[mt] += e[mt][i];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) u[mt][dt] = mma4(v[i][dt], e[mt][i], u[mt][dt]);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        den[mt] = group_sum(den[mt]);
        const int m = mb + 16 * mt + c;
        if (m < M) {
            const size_t si = ((size_t)bh * NC + ch) * M + m;
            if (g == 0) {
                cmax[si] = mx[mt];
                cden[si] = den[mt];
            }
            float* row = cnum + si * D;
#pragma unroll
            for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc))
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float* p = row + col_of<DT>(dt, 4 * g + i);
                    const int P = piece_of<DT>(dt);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (j < P) p[j] = u[mt][dt + j < DT ? dt + j : 0][i];
                }
        }
    }
}

// n consecutive results to Y (out_dtype code), starting at element idx
template <int P>
__device__ __forceinline__ void store_cols(void* Y, size_t idx, const float* x, int out_dtype) {
    if (out_dtype == FLARE_F32) {
        float* p = reinterpret_cast<float*>(Y) + idx;
        if constexpr (P == 4) {
            *reinterpret_cast<f32x4_a*>(p) = f32x4{x[0], x[1], x[2], x[3]};
        } else {
#pragma unroll
            for (int j = 0; j < P; ++j) p[j] = x[j];
        }
    } else {
        unsigned short h[P];
#pragma unroll
        for (int j = 0; j < P; ++j)
            h[j] = out_dtype == FLARE_BF16 ? __builtin_bit_cast(unsigned short, (mfma::bf16)x[j])
                                           : __builtin_bit_cast(unsigned short, (mfma::f16)x[j]);
        unsigned short* p = reinterpret_cast<unsigned short*>(Y) + idx;
        if constexpr (P == 4) {
            *reinterpret_cast<u32x2*>(p) = u32x2{h[0] | (unsigned)h[1] << 16, h[2] | (unsigned)h[3] << 16};
        } else if constexpr (P == 2) {
            *reinterpret_cast<u32_a*>(p) = h[0] | (unsigned)h[1] << 16;
        } else {
            *p = h[0];
        }
    }
}

// the same to a buffer, at byte offset `at`
__device__ __forceinline__ void put_cols(const Bytes& y, unsigned at, const float (&x)[4], int P, int out_dtype) {
    if (out_dtype == FLARE_F32) {
        const u32x4 r = {__builtin_bit_cast(u32, x[0]), __builtin_bit_cast(u32, x[1]), __builtin_bit_cast(u32, x[2]),
                         __builtin_bit_cast(u32, x[3])};
        if (P == 4) y.put128(at, r);
        else if (P == 2) y.put64(at, u32x2{r[0], r[1]});
        else y.put32(at, r[0]);
    } else {
        u32 h[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            h[k] = out_dtype == FLARE_BF16 ? __builtin_bit_cast(unsigned short, (mfma::bf16)x[k])
                                           : __builtin_bit_cast(unsigned short, (mfma::f16)x[k]);
        if (P == 4) y.put64(at, u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16});
        else if (P == 2) y.put32(at, h[0] | h[1] << 16);
        else y.put16(at, h[0]);
    }
}

// ---------------------------------------------------------------------------
// Phase 3: replay of one chunk from its exclusive prefix, and the readout.
// grid = (NC, B*H), one wave per MT*16 latents (NW = blockDim.x / 64 waves).
//
// Per 16-token tile and wave, from scores^T [m][t]:
//   m' = max(m, tile max), E = e^(s - m'), d_t = d + cumulative E along the tokens,
//   W = p / d_t with p = e^(s_dec - wave max) the decoder weights before their sum,
//   G^T = E W^T (masked to tau <= t),  y = W U + G V,  U += E^T V.
// One wave: W takes the softmax sum at once.  Several: each wave writes its y, max and sum
// to LDS and the workgroup merges them (the token softmax over waves), double-buffered.
//
// j < 0: the whole tile.  A tile in which some latent's max rises by more than kTileJump, whose
// V holds a non-finite value, or whose first token has no finite reference near the tile's max,
// is walked token by token (j = the token, the loop comes back with the same tile): the same
// body with every other token masked, so that the reference moves exactly to each token, as in
// the tokenwise recurrence.
// ---------------------------------------------------------------------------
template <int MT, int DT>
__host__ __device__ constexpr int e_pitch() { return 16 * MT + 4; }

template <int MT, int DT>
inline size_t wave_output_lds(int NW) {
    return sizeof(float) * ((size_t)NW * TT * e_pitch<MT, DT>() + (NW > 1 ? 2 * (size_t)NW * TT * (16 * DT + 2) : 0));
}

template <typename T, int MT, int DT, bool SEP>
__global__ __launch_bounds__(wave_threads(MT)) void wave_output_kernel(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, const T* __restrict__ Qdec,
    const T* __restrict__ Kdec, int N, int H, int M, float scale, int chunk, const float* __restrict__ pmax,
    const float* __restrict__ pden, const float* __restrict__ pnum, void* __restrict__ Y, int out_dtype,
    const int32_t* __restrict__ tmask) {
    constexpr int D = 16 * DT;
    constexpr int EP = e_pitch<MT, DT>();
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int ch = blockIdx.x, NC = gridDim.x, bh = blockIdx.y;
    const int b = bh / H, h = bh % H;
    const int NW = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = w * 16 * MT;
    float* etile = smem + w * TT * EP;                 // this wave's E, [tau][m]
    float* ypart = smem + NW * TT * EP;                // [2][NW][TT][D]
    float* ystat = ypart + 2 * NW * TT * D;            // [2][NW][2][TT]: max, sum

    constexpr bool QREG = latents_in_regs<T, DT, SEP>(), AHEAD = fetch_ahead<DT>();
    RowOp<T, D> q[QREG ? MT : 1], kd[SEP && QREG ? MT : 1];
    const size_t bank = (size_t)M * D;
    const Bytes qbank(Q + h * bank, bank * sizeof(T)), kbank(SEP ? Kdec + h * bank : Q, SEP ? bank * sizeof(T) : 0);
    auto load_latent = [&](RowOp<T, D>& r, const Bytes& from, int mt) {          // past the bank: zeros
        r.load(from, (mb + 16 * mt + c) * (D * (int)sizeof(T)) + RowOp<T, D>::lane(g), g);
    };
    if constexpr (QREG) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            load_latent(q[mt], qbank, mt);
            if constexpr (SEP) load_latent(kd[mt], kbank, mt);
        }
    }
    // latent mb + 16 mt + 4g + i: max, den (the same in the 16 lanes of a row), U row
    float mx[MT][4], den[MT][4];
    f32x4 u[MT][DT];
    {
        const size_t pbase = ((size_t)bh * NC + ch) * M;
        const Bytes pm(pmax + pbase, 4 * (size_t)M), pd(pden + pbase, 4 * (size_t)M), pn(pnum + pbase * D, 4 * bank);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = mb + 16 * mt + 4 * g + i;
                const float x = __builtin_bit_cast(float, pm.b32(4 * m));
                mx[mt][i] = m < M ? x : kNegInf;
                den[mt][i] = __builtin_bit_cast(float, pd.b32(4 * m));
                ColRow<float, DT> r;
                r.load(pn, m * (4 * D), c);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) u[mt][dt][i] = r.get(dt);
            }
    }

    // the chunk's rows of this head, by byte offset from its first token
    const int t0 = ch * chunk, t1 = min(N, t0 + chunk);
    const unsigned stride = (unsigned)(H * D) * sizeof(T);
    const size_t first = (((size_t)b * N + t0) * H + h) * D;
    const size_t span = (size_t)(t1 - t0 - 1) * stride + D * sizeof(T);
    const Bytes kb(K + first, span), vb(V + first, span), qb(SEP ? Qdec + first : K, SEP ? span : 0);
    const int osize = out_dtype == FLARE_F32 ? 4 : 2;
    const unsigned ostride = (unsigned)(H * D) * osize;
    const Bytes yb((const char*)Y + first * osize, (size_t)(t1 - t0 - 1) * ostride + D * osize);
    unsigned krow = c * stride + RowOp<T, D>::lane(g), vrow = 4 * g * stride;
    RowOp<T, D> kn, qn;
    ColRow<T, DT> vn[4];
    auto fetch = [&]() {                                // (past the chunk: zeros)
        kn.load(kb, krow, g);
        if constexpr (SEP) qn.load(qb, krow, g);
#pragma unroll
        for (int i = 0; i < 4; ++i) vn[i].load(vb, vrow + i * stride, c);
    };
    fetch();
    int buf = 0, t = t0, j = -1;
    while (true) {
        // scores^T, then the next tile's loads
        f32x4 s[MT], p[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if constexpr (!QREG) load_latent(q[0], qbank, mt);
            s[mt] = dot_rows<T, D>(q[QREG ? mt : 0], kn, f32x4{0.f, 0.f, 0.f, 0.f});
            if constexpr (SEP) {
                if constexpr (!QREG) load_latent(kd[0], kbank, mt);
                p[mt] = dot_rows<T, D>(kd[QREG ? mt : 0], qn, f32x4{0.f, 0.f, 0.f, 0.f});
            }
        }
        float v[4][DT];
        float vbad = 0.0f;                             // NaN when a value is not finite
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                v[i][dt] = vn[i].get(dt);
                vbad = __builtin_fmaf(v[i][dt], 0.0f, vbad);
            }
        bool live = t + c < t1;                        // token t + c takes part
        if (tmask != nullptr) live = live && tmask[(size_t)b * N + min(t + c, t1 - 1)] != 0;
        const unsigned lmask = (unsigned)(__ballot(live) & 0xffffu);   // the 16 tokens, wave-uniform
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[mt][i] *= scale;
                if constexpr (SEP) p[mt][i] *= scale;
                else p[mt][i] = s[mt][i];
            }
        if (mb + 16 * MT > M) {                        // this wave's share ends past the bank
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool out = mb + 16 * mt + 4 * g + i >= M;
                    s[mt][i] = out ? kNegInf : s[mt][i];
                    p[mt][i] = out ? kNegInf : p[mt][i];
                }
        }
        // the tokens of this pass: the others score -inf and hold no value
        auto keep = [&](unsigned take) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[mt][i] = (take >> c) & 1 ? s[mt][i] : kNegInf;
                    p[mt][i] = (take >> c) & 1 ? p[mt][i] : kNegInf;
                }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) v[i][dt] = (take >> (4 * g + i)) & 1 ? v[i][dt] : 0.0f;
        };
        if (j < 0 && __any(vbad != vbad) && lmask != 0) j = __builtin_ctz(lmask);
        if (j >= 0) keep(1u << j);
        else if (lmask != 0xffffu) keep(lmask);

        bool moved = false;                            // a score passes its latent's max
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) moved |= s[mt][i] > mx[mt][i];
        if (__any(moved)) {
            float top[MT][4], rise = 0.0f;             // rise: the largest move of a reference in the tile
            const int first = lmask ? __builtin_ctz(lmask) : 0;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    top[mt][i] = mfma::row_max16(s[mt][i]);
                    // (no earlier token: from the tile's first live one)
                    const float low = mx[mt][i] == kNegInf ? __shfl(s[mt][i], (lane & 48) | first, 64) : mx[mt][i];
                    const float up = top[mt][i] == kNegInf ? 0.0f : top[mt][i] - low;
                    rise = fmaxf(rise, up == up ? up : 2.0f * kTileJump);
                }
            if (j < 0 && __any(rise > kTileJump)) {
                j = first;
                keep(1u << j);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) top[mt][i] = mfma::row_max16(s[mt][i]);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float mnew = fmaxf(mx[mt][i], top[mt][i]);
                    const float r = mx[mt][i] == mnew ? 1.0f : mx[mt][i] == kNegInf ? 0.0f : exp_nat(mx[mt][i] - mnew);
                    den[mt][i] *= r;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) u[mt][dt][i] *= r;
                    mx[mt][i] = mnew;
                }
        }
        // this pass's output rows (masked tokens come with the first one), and the tokens left
        const unsigned take = j < 0 ? lmask : 1u << j;
        const unsigned rows = j < 0 ? 0xffffu : j == __builtin_ctz(lmask) ? take | (~lmask & 0xffffu) : take;
        const unsigned after = j < 0 ? 0u : lmask & ~((2u << j) - 1u);

        // decoder weights of this wave's latents (a masked token's scores are -inf: weights 0)
        float wmax = kNegInf, psum = 0.0f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) wmax = fmaxf(fmaxf(wmax, fmaxf(p[mt][0], p[mt][1])), fmaxf(p[mt][2], p[mt][3]));
        wmax = group_max(wmax);
        {
            const float ref = fmaxf(wmax, kLowRef);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[mt][i] = exp_nat(p[mt][i] - ref);
                    psum += p[mt][i];
                }
        }
        psum = group_sum(psum);
        const float norm = NW > 1 ? 1.0f : psum > 0.0f ? 1.0f / psum : psum;       // (a NaN stays one)
        f32x4 e[MT], wt[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[mt][i] = exp_nat(s[mt][i] - fmaxf(mx[mt][i], kLowRef));
                const float d = den[mt][i] + mfma::row_scan16(e[mt][i]);
                wt[mt][i] = p[mt][i] * norm * __builtin_amdgcn_rcpf(fmaxf(d, kTinyDen));
                den[mt][i] = mfma::row_bcast15(d);
            }
            *reinterpret_cast<f32x4_a*>(etile + c * EP + 16 * mt + 4 * g) = e[mt];
        }
        wave_lds_sync();
        // the next tile's rows, once this one has no further pass
        if (AHEAD && after == 0) {
            krow += TT * stride;
            vrow += TT * stride;
            fetch();
        }
        // G^T [tau][t], masked to tau <= t
        f32x4 ga = {0.f, 0.f, 0.f, 0.f}, gb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            ga = mma4(e[mt][0], wt[mt][0], ga);
            gb = mma4(e[mt][1], wt[mt][1], gb);
            ga = mma4(e[mt][2], wt[mt][2], ga);
            gb = mma4(e[mt][3], wt[mt][3], gb);
        }
        f32x4 y[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) y[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) y[dt] = mma4(wt[mt][i], u[mt][dt][i], y[dt]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float gm = 4 * g + i <= c ? ga[i] + gb[i] : 0.0f;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) y[dt] = mma4(gm, v[i][dt], y[dt]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const float ea = etile[(4 * g + i) * EP + 16 * mt + c];
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) u[mt][dt] = mma4(ea, v[i][dt], u[mt][dt]);
            }
        }
        wave_lds_sync();
        if (NW == 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned row = (rows >> (4 * g + i)) & 1 ? (unsigned)(t - t0 + 4 * g + i) * ostride : kNowhere;
#pragma unroll
                for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc)) {
                    float o[4];
                    const int P = piece_of<DT>(dt);
#pragma unroll
                    for (int k = 0; k < 4; ++k) o[k] = k < P ? y[dt + k < DT ? dt + k : 0][i] : 0.0f;
                    put_cols(yb, row + col_of<DT>(dt, c) * osize, o, P, out_dtype);
                }
            }
        } else {
            float* yw = ypart + ((size_t)buf * NW + w) * TT * D;
            if (j < 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) yw[(4 * g + i) * D + col_of<DT>(dt, c)] = y[dt][i];
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if ((rows >> (4 * g + i)) & 1) {
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) yw[(4 * g + i) * D + col_of<DT>(dt, c)] = y[dt][i];
                    }
            }
        }
        if (NW > 1) {
            float* sw = ystat + ((size_t)buf * NW + w) * 2 * TT;
            if (g == 0 && ((rows >> c) & 1)) {
                sw[c] = wmax;
                sw[TT + c] = psum;
            }
        }
        if (after != 0) {                              // this tile's next token
            j = __builtin_ctz(after);
            continue;
        }
        j = -1;
        if (NW > 1) {
            __syncthreads();
            const float* yr = ypart + (size_t)buf * NW * TT * D;
            const float* sr = ystat + (size_t)buf * NW * 2 * TT;
            for (int x = threadIdx.x; x < TT * D / 4; x += blockDim.x) {
                const int ti = x / (D / 4), col = 4 * (x % (D / 4));
                float mm = kNegInf;
                for (int k = 0; k < NW; ++k) mm = fmaxf(mm, sr[k * 2 * TT + ti]);
                const float ref = safe_ref(mm);
                float sum = 0.0f;
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                for (int k = 0; k < NW; ++k) {
                    const float f = exp_nat(sr[k * 2 * TT + ti] - ref);
                    sum += f * sr[k * 2 * TT + TT + ti];
                    const f32x4 yk = *reinterpret_cast<const f32x4_a*>(yr + ((size_t)k * TT + ti) * D + col);
#pragma unroll
                    for (int n = 0; n < 4; ++n) acc[n] += f * yk[n];
                }
                const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
                float o[4];
#pragma unroll
                for (int n = 0; n < 4; ++n) o[n] = acc[n] * inv;
                put_cols(yb, (unsigned)(t - t0 + ti) * ostride + col * osize, o, 4, out_dtype);
            }
            buf ^= 1;
        }
        t += TT;
        if (t >= t1) break;
        if constexpr (!AHEAD) {
            krow += TT * stride;
            vrow += TT * stride;
            fetch();
        }
    }
}

}  // namespace wave
}  // namespace flare
