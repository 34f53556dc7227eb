// flare_wave_semi.h -- backward of the block-causal (semi-autoregressive) layer with
// wave-private latents, on the operands and products of flare_wave_bwd.h.
//
// Every token of block b reads the state after block b, so with D, U, z = U / D at the block's
// end and X, Y the reverse sums over blocks from b on,
//   gz_t = g_t . z        X += sum_{t in b} (alpha_t / D) g_t      Y += sum (alpha_t / D) gz_t
//   ds_tau = e^{s_tau} (v_tau . X - Y)      dv_tau = sum_m e^{s_tau} X
// and nothing inside a block depends on token order: no in-tile products, no token-by-token
// tiles.  Two walks over chunks of whole blocks, each passing over a block's 16-token tiles
// twice, take the place of one M x D state per block in memory:
//   wave_semi_gz   pass 0 adds the block to U, pass 1 forms gz and the chunk's X and Y terms;
//   wave_semi_ds   (last block first) pass 0 adds the block to X and Y, pass 1 forms ds and dv.
// X is fixed during pass 1, so its transposed copy for dv is written to LDS once a block
// (D <= 64; wider states leave no room beside the partial dv rows and are written per tile).
//
// Bound by the latency of a step's chain (load, scores, exponentials, products, barrier) at two
// to four waves a SIMD.  Measured, forward and backward, against one state per block in memory:
// bf16 B 2, N 8192, blocks of 64, H 16, M 128, D 64: 1449 -> 485 us (wave_semi_gz 101,
// wave_semi_ds 143 of it).
#pragma once

#include "flare_wave_bwd.h"

namespace flare {
namespace wave {

// Rows of a step's arrays in LDS (see TileRows); which arrays, and the tile, are the caller's.
template <typename T, int DT, int R>
struct StepRows {
    static constexpr int D = 16 * DT, CPR = D * (int)sizeof(T) / 16, PITCH = D + 16 / (int)sizeof(T);
    static constexpr int CHUNKS = TT * CPR, PF = sizeof(T) == 2 ? 1 : 2, A = TT * PITCH;
    static constexpr size_t BYTES = (size_t)R * A * sizeof(T);
    u32x4 held[R][PF];
    static __device__ __forceinline__ bool holds() { return CHUNKS <= PF * (int)blockDim.x; }
    static __device__ __forceinline__ u32x4 piece(const T* p, int stride, int x, int t) {
        return reinterpret_cast<const u32x4*>(p + (size_t)(t + x / CPR) * stride)[x % CPR];
    }
    static __device__ __forceinline__ void put(T* lds, int x, u32x4 val) {
        *reinterpret_cast<u32x4*>(lds + (x / CPR) * PITCH + (x % CPR) * (16 / (int)sizeof(T))) = val;
    }
    __device__ __forceinline__ void fetch(const T* p0, const T* p1, const T* p2, int stride, int t) {
        if (!holds()) return;
#pragma unroll
        for (int n = 0; n < PF; ++n) {
            const int x = min((int)(threadIdx.x + n * blockDim.x), CHUNKS - 1);
            held[0][n] = piece(p0, stride, x, t);
            held[1][n] = piece(p1, stride, x, t);
            if constexpr (R == 3) held[2][n] = piece(p2, stride, x, t);
        }
    }
    __device__ __forceinline__ void store(T* lds, const T* p0, const T* p1, const T* p2, int stride, int t) {
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
                put(lds, x, piece(p0, stride, x, t));
                put(lds + A, x, piece(p1, stride, x, t));
                if constexpr (R == 3) put(lds + 2 * A, x, piece(p2, stride, x, t));
            }
        }
    }
    static __device__ __forceinline__ const T* row(const T* lds, int a, int r) { return lds + a * A + r * PITCH; }
};

// ---------------------------------------------------------------------------
// Readout of the block-causal forward from the blocks' states z = U / den in memory
// ([B*H][N/block][M][D], fp32): y = sum over latents of the decoder's weight times z.  A wave
// takes NTK tiles of 16 tokens of one block against all latents, twice: the largest score, then the
// weights relative to it and their sum, the weights' C tiles being the factor of the fp32 products
// with z as they are.  (A running log-sum-exp and weights taken from it: lse up to 3.5% and y 60%
// further from 64 bits in fp32, in the same time.)  Bound by
// the latency of z's and the latents' rows from cache (a block's z serves its few waves).
// Measured: forward and backward of bf16 B 4, N 640, blocks of 32, H 16, M 192, D 64 take 333 us.
// ---------------------------------------------------------------------------
template <typename T, int DT, int NTK>
__global__ __launch_bounds__(256) void wave_semi_output_kernel(const T* __restrict__ Qd, const T* __restrict__ Kd,
                                                               const float* __restrict__ z, int N, int H, int M, float scale,
                                                               int block, void* __restrict__ Y, int out_dtype,
                                                               float* __restrict__ lse_out) {
    constexpr int D = 16 * DT;
    const int bh = blockIdx.y, b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int t0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * TT * NTK;
    if (t0 >= N) return;                          // (N and block are multiples of 16 NTK)
    const Bytes zb(z + ((size_t)bh * (N / block) + t0 / block) * M * D, (size_t)M * D * sizeof(float));
    GroupRow<T, DT> k[NTK];
    float ref[NTK], sum[NTK];
#pragma unroll
    for (int j = 0; j < NTK; ++j) {
        k[j].load(Qd + (((size_t)b * N + t0 + TT * j + c) * H + h) * D, g);
        ref[j] = kNegInf;
        sum[j] = 0.0f;
    }
    auto scores = [&](int m0, f32x4 (&s)[NTK]) {
        GroupRow<T, DT> q;
        q.load(Kd + ((size_t)h * M + min(m0 + c, M - 1)) * D, g);
#pragma unroll
        for (int j = 0; j < NTK; ++j) {
            s[j] = dot_groups(q, k[j], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int i = 0; i < 4; ++i) s[j][i] = m0 + 4 * g + i < M ? s[j][i] * scale : kNegInf;
        }
    };
    for (int m0 = 0; m0 < M; m0 += 16) {
        f32x4 s[NTK];
        scores(m0, s);
#pragma unroll
        for (int j = 0; j < NTK; ++j) ref[j] = fmaxf(ref[j], fmaxf(fmaxf(s[j][0], s[j][1]), fmaxf(s[j][2], s[j][3])));
    }
    f32x4 y[NTK][DT];
#pragma unroll
    for (int j = 0; j < NTK; ++j) {
        ref[j] = safe_ref(group_max(ref[j]));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) y[j][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int m0 = 0; m0 < M; m0 += 16) {
        ColRow<float, DT> r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i].load(zb, (m0 + 4 * g + i) * (4 * D), c);     // past the bank: zeros
        f32x4 s[NTK];
        scores(m0, s);
#pragma unroll
        for (int j = 0; j < NTK; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) s[j][i] = exp_nat(s[j][i] - ref[j]);          // 0 past the bank
            sum[j] += (s[j][0] + s[j][1]) + (s[j][2] + s[j][3]);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) y[j][dt] = mma4(r[i].get(dt), s[j][i], y[j][dt]);
        }
    }
#pragma unroll
    for (int j = 0; j < NTK; ++j) {
        const int t = t0 + TT * j + c;
        const float all = group_sum(sum[j]), norm = 1.0f / all;
        const size_t row = (((size_t)b * N + t) * H + h) * D;
#pragma unroll
        for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc))
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float o[4];
                const int P = piece_of<DT>(dt);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = e < P ? y[j][dt + e < DT ? dt + e : 0][i] * norm : 0.0f;
                const size_t at = row + col_of<DT>(dt, 4 * g + i);
                if (P == 4) store_cols<4>(Y, at, o, out_dtype);
                else if (P == 2) store_cols<2>(Y, at, o, out_dtype);
                else store_cols<1>(Y, at, o, out_dtype);
            }
        if (lse_out != nullptr && g == 0) lse_out[(size_t)bh * N + t] = ref[j] + __logf(all);
    }
}

// ---------------------------------------------------------------------------
// Forward walk: grid (NC, B*H), one wave per MT*16 latents.  chunk and N are multiples of
// block, block a multiple of 16.
// ---------------------------------------------------------------------------
template <typename T, int MT, int DT, bool SEP, int P>
__global__ __launch_bounds__(64 * (16 / MT)) void wave_semi_gz_kernel(BwdPtrs a, int N, int H, int M, float scale,
                                                                      int chunk, int block) {
    constexpr int D = 16 * DT, R = SEP ? 3 : 2;
    typedef typename ProdOf<T, P>::F F;
    typedef StepRows<T, DT, R> Rows;
    constexpr bool QREG = bwd_latents_in_regs<T, DT, SEP>(), FLAT = sizeof(T) == 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];
    const int ch = blockIdx.x, NC = gridDim.x, bh = blockIdx.y;
    const int b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, NW = blockDim.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = wv * 16 * MT;
    const int NB = N / block;
    const int t0 = ch * chunk, t1 = min(N, t0 + chunk);
    const int stride = H * D;
    const size_t tok = ((size_t)b * N * H + h) * D;
    const T *kb = (const T*)a.K + tok, *vb = (const T*)a.V + tok, *gb = (const T*)a.dY + tok, *qb = (const T*)a.Qdec + tok;
    const Floats gz_out(a.gz + (size_t)bh * N * M, (size_t)N * M), lse_in(a.lse + (size_t)bh * N, N);
    const Floats dmax(a.tmax + (size_t)bh * NB * M, (size_t)NB * M), dden(a.tden + (size_t)bh * NB * M, (size_t)NB * M);

    GroupRow<T, DT> q[QREG ? MT : 1], kd[SEP && QREG ? MT : 1];
    auto latent_row = [&](GroupRow<T, DT>& r, const void* base, int mt) {
        // (past the bank: its last row; such a latent is never stored)
        r.load((const T*)base + ((size_t)h * M + min(mb + 16 * mt + c, M - 1)) * D, g);
    };
    unsigned lat[MT];
    float mx[MT], den[MT], part[MT], er[MT], inv[MT], ysum[MT];
    f32x4 u[MT][DT], x[MT][DT];
    const size_t pbase = ((size_t)bh * NC + ch) * M;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mb + 16 * mt + c;
        const bool in = m < M;
        lat[mt] = in ? 4u * m : kNowhere;
        if constexpr (QREG) {
            latent_row(q[mt], a.Q, mt);
            if constexpr (SEP) latent_row(kd[mt], a.Kdec, mt);
        }
        mx[mt] = in ? a.pmax[pbase + m] : kNegInf;
        den[mt] = in ? a.pden[pbase + m] : 0.0f;
        er[mt] = mx[mt] == kNegInf ? 0.0f : 1.0f;
        part[mt] = ysum[mt] = 0.0f;
        inv[mt] = 0.0f;
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
    rows.fetch(kb, vb, vb, stride, t0);
    rows.store((T*)tile_lds, kb, vb, vb, stride, t0);
    __syncthreads();
    int buf = 0, t = t0, pass = 0;
    float* gsum = reinterpret_cast<float*>(tile_lds + 2 * Rows::BYTES);
    float* gy_out = a.gy + (size_t)bh * N;
    while (true) {
        const T* tl = (const T*)(tile_lds + buf * Rows::BYTES);
        // the next step: the block's next tile, its second pass, or the next block
        const bool end = (t + TT) % block == 0;
        const int np = end ? pass ^ 1 : pass;
        const int nt = !end ? t + TT : pass == 0 ? t + TT - block : t + TT;
        const bool more = nt < t1;
        if (more) rows.fetch(kb, np ? gb : vb, np ? qb : vb, stride, nt);

        GroupRow<T, DT> kr;
        kr.load(Rows::row(tl, 0, c), g);
        f32x4 s[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if constexpr (!QREG) latent_row(q[0], a.Q, mt);
            s[mt] = dot_groups(kr, q[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int i = 0; i < 4; ++i) s[mt][i] *= scale;
        }
        F f[MT];
        if (pass == 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const float top = group_max(fmaxf(fmaxf(s[mt][0], s[mt][1]), fmaxf(s[mt][2], s[mt][3])));
                const float mnew = fmaxf(mx[mt], top);
                const float r = mx[mt] == mnew ? 1.0f : mx[mt] == kNegInf ? 0.0f : exp_nat(mx[mt] - mnew);
                if (__any(r != 1.0f)) {
                    den[mt] *= r;
                    part[mt] *= r;
                    er[mt] *= r;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) u[mt][dt][i] *= r;
                }
                mx[mt] = mnew;
                const float ref = safe_ref(mnew);
                float e[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    e[i] = exp_nat(s[mt][i] - ref);
                    part[mt] += e[i];
                }
                f[mt] = factor<F>(e[0], e[1], e[2], e[3]);
            }
            if (end) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    den[mt] += group_sum(part[mt]);
                    part[mt] = 0.0f;
                    inv[mt] = 1.0f / (den[mt] > 0.0f ? den[mt] : 1.0f);
                    if (g == 0) {
                        dmax.store(4u * M * (t / block) + lat[mt], mx[mt]);
                        dden.store(4u * M * (t / block) + lat[mt], den[mt]);
                    }
                }
            }
#pragma unroll
            for (int st = 0, d0 = 0; st < steps<T, DT>(); d0 = step_start<T, DT>(++st)) {
                TileCols<T, DT> vc;
                vc.load_piece(Rows::row(tl, 1, 0), Rows::PITCH, g, c, d0);
#pragma unroll
                for (int dt = d0; dt < d0 + step_most<T>(); ++dt) {
                    if (dt >= d0 + step_of<T, DT>(d0)) continue;
                    const auto vo = vc.op(dt);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) u[mt][dt] = collect(vo, f[mt], u[mt][dt]);
                }
            }
        } else {
            WalkRow<T, DT> gr;
            gr.load(Rows::row(tl, 1, c), g);
            float lse[4], gy[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 4; ++i) lse[i] = lse_in.load(4u * (t + 4 * g + i));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                f32x4 z = s[mt];
                if constexpr (SEP) {
                    GroupRow<T, DT> qr;
                    qr.load(Rows::row(tl, R - 1, c), g);
                    if constexpr (!QREG) latent_row(kd[0], a.Kdec, mt);
                    z = dot_groups(qr, kd[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int i = 0; i < 4; ++i) z[i] *= scale;
                }
                const f32x4 p = dot_state<T, DT, P>(gr, u[mt], f32x4{0.f, 0.f, 0.f, 0.f});
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float gz = p[i] * inv[mt];
                    const float al = lat[mt] != kNowhere ? exp_nat(z[i] - lse[i]) : 0.0f;
                    w[i] = al * (er[mt] * inv[mt]);
                    if constexpr (own_gy<T>()) gy[i] += al != 0.0f ? al * gz : 0.0f;
                    ysum[mt] += w[i] == 0.0f ? 0.0f : w[i] * gz;
                    gz_out.store(4u * M * (t + 4 * g + i) + lat[mt], gz);
                }
                f[mt] = factor<F>(w[0], w[1], w[2], w[3]);
            }
            if constexpr (own_gy<T>()) put_gy(gsum + buf * NW * TT, gy, wv, g, c);
#pragma unroll
            for (int st = 0, d0 = 0; st < steps<T, DT>(); d0 = step_start<T, DT>(++st)) {
                TileCols<T, DT> gc;
                gc.load_piece(Rows::row(tl, 1, 0), Rows::PITCH, g, c, d0);
#pragma unroll
                for (int dt = d0; dt < d0 + step_most<T>(); ++dt) {
                    if (dt >= d0 + step_of<T, DT>(d0)) continue;
                    const auto go = gc.op(dt);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) x[mt][dt] = collect(go, f[mt], x[mt][dt]);
                }
            }
        }
        if (more) rows.store((T*)(tile_lds + (buf ^ 1) * Rows::BYTES), kb, np ? gb : vb, np ? qb : vb, stride, nt);
        __syncthreads();
        if (own_gy<T>() && pass == 1) store_gy(gsum + buf * NW * TT, NW, gy_out, t, t1);
        if (!more) break;
        buf ^= 1;
        t = nt;
        pass = np;
    }
    set_wild<T, MT, DT>(x, gb, stride, t0, t1, g);
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
// Backward walk: ds and dv.  grid (NC, B*H), one wave per MT*16 latents.
// ---------------------------------------------------------------------------
template <int DT>
__host__ __device__ constexpr bool semi_x_stays() { return DT <= 4; }
template <typename T, int MT, int DT, int P>
__host__ __device__ constexpr int semi_wave_floats() {
    const int xt = (one_x_tile<T, DT, P>() ? 1 : MT) * StateTile<T, DT, P>::FLOATS, dv = TT * dv_pitch(DT);
    return semi_x_stays<DT>() ? xt + dv : (xt > dv ? xt : dv);
}

template <typename T, int MT, int DT, bool SEP, int P>
__global__ __launch_bounds__(64 * (16 / MT)) void wave_semi_ds_kernel(BwdPtrs a, int N, int H, int M, float scale,
                                                                      int chunk, int block) {
    constexpr int D = 16 * DT, VP = dv_pitch(DT), R = SEP ? 3 : 2, WF = semi_wave_floats<T, MT, DT, P>();
    typedef StateTile<T, DT, P> XTile;
    constexpr bool STAYS = semi_x_stays<DT>(), ONE = one_x_tile<T, DT, P>();
    constexpr int OD = sizeof(T) == 4 ? FLARE_F32 : __is_same(T, __half) ? FLARE_F16 : FLARE_BF16;
    typedef typename ProdOf<T, P>::F F;
    typedef StepRows<T, DT, R> Rows;
    constexpr bool QREG = bwd_latents_in_regs<T, DT, SEP>(), FLAT = sizeof(T) == 2;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int ch = blockIdx.x, NC = gridDim.x, bh = blockIdx.y;
    const int b = bh / H, h = bh % H;
    const int NW = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = wv * 16 * MT;
    const int NB = N / block;
    const int t0 = ch * chunk, t1 = min(N, t0 + chunk);
    const int stride = H * D;
    const size_t tok = ((size_t)b * N * H + h) * D;
    const T *kb = (const T*)a.K + tok, *vb = (const T*)a.V + tok, *gb = (const T*)a.dY + tok, *qb = (const T*)a.Qdec + tok;
    constexpr int voff = STAYS ? MT * XTile::FLOATS : 0;
    float *xtile = smem + wv * WF, *vtile = xtile + voff;
    T* tl = reinterpret_cast<T*>(smem + NW * WF);
    const size_t per = (size_t)N * M;
    const Floats gz_in(a.gz + bh * per, per), lse_in(a.lse + (size_t)bh * N, N), gy_in(a.gy + (size_t)bh * N, N);
    const Floats ds_out(a.ds + bh * per, per), al_out(SEP ? a.al + bh * per : a.ds, SEP ? per : 0);
    const Floats dmax(a.tmax + (size_t)bh * NB * M, (size_t)NB * M), dden(a.tden + (size_t)bh * NB * M, (size_t)NB * M);

    GroupRow<T, DT> q[QREG ? MT : 1], kd[SEP && QREG ? MT : 1];
    auto latent_row = [&](GroupRow<T, DT>& r, const void* base, int mt) {
        r.load((const T*)base + ((size_t)h * M + min(mb + 16 * mt + c, M - 1)) * D, g);
    };
    unsigned lat[MT];
    float mref[MT], inv[MT], ysum[MT], part[MT], mrow[MT][4];      // mrow: the block's max of latent 4g + i
    f32x4 x[MT][DT];
    const size_t pbase = ((size_t)bh * NC + ch) * M;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mb + 16 * mt + c;
        lat[mt] = m < M ? 4u * m : kNowhere;
        if constexpr (QREG) {
            latent_row(q[mt], a.Q, mt);
            if constexpr (SEP) latent_row(kd[mt], a.Kdec, mt);
        }
        const bool tail = m < M && ch + 1 < NC;
        mref[mt] = tail ? a.pmax[pbase + M + m] : 0.0f;
        ysum[mt] = tail ? a.ysum[pbase + m] : 0.0f;
        part[mt] = inv[mt] = 0.0f;
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
    int t = t1 - TT, pass = 0;
    rows.fetch(kb, gb, qb, stride, t);
    rows.store(tl, kb, gb, qb, stride, t);
    __syncthreads();
    bool some_wild = find_wild<T, MT, DT>(x, wild_bits, g);
    while (true) {
        const bool begin = (t + TT) % block == 0, end = t % block == 0;     // first / last tile of a pass
        const int np = end ? pass ^ 1 : pass;
        const int nt = !end ? t - TT : pass == 0 ? t + block - TT : t - TT;
        const bool more = nt >= t0;
        if (more) rows.fetch(kb, np ? vb : gb, np ? vb : qb, stride, nt);
        if (begin && pass == 0) {
            // a new block: X and Y relative to its max
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const float ref = safe_ref(dmax.load(4u * M * (t / block) + lat[mt]));
                const float d = dden.load(4u * M * (t / block) + lat[mt]);
                inv[mt] = 1.0f / (d > 0.0f ? d : 1.0f);
                // (the max falls as the walk goes back; the bound keeps a last chunk's zeros zero)
                const float r = exp_nat(fminf(ref - mref[mt], 1.0f));
                ysum[mt] *= r;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[mt][dt][i] *= r;
                mref[mt] = ref;
#pragma unroll
                for (int i = 0; i < 4; ++i) mrow[mt][i] = __shfl(ref, 4 * g + i, 64);
            }
        }
        float gz[MT][4], lse[4], gy[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lse[i] = lse_in.load(4u * (t + 4 * g + i));
            gy[i] = SEP ? 0.0f : gy_in.load(4u * (t + 4 * g + i));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) gz[mt][i] = gz_in.load(4u * M * (t + 4 * g + i) + lat[mt]);
        }
        GroupRow<T, DT> kr;
        kr.load(Rows::row(tl, 0, c), g);
        if (pass == 0) {
            F wf[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                f32x4 z;
                if constexpr (SEP) {
                    GroupRow<T, DT> qr;
                    qr.load(Rows::row(tl, R - 1, c), g);
                    if constexpr (!QREG) latent_row(kd[0], a.Kdec, mt);
                    z = dot_groups(qr, kd[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
                } else {
                    if constexpr (!QREG) latent_row(q[0], a.Q, mt);
                    z = dot_groups(kr, q[QREG ? mt : 0], f32x4{0.f, 0.f, 0.f, 0.f});
                }
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float al = lat[mt] != kNowhere ? exp_nat(z[i] * scale - lse[i]) : 0.0f;
                    if constexpr (SEP) al_out.store(4u * M * (t + 4 * g + i) + lat[mt], al);
                    w[i] = al * inv[mt];
                    part[mt] += w[i] == 0.0f ? 0.0f : w[i] * gz[mt][i];
                }
                wf[mt] = factor<F>(w[0], w[1], w[2], w[3]);
            }
#pragma unroll
            for (int st = 0, d0 = 0; st < steps<T, DT>(); d0 = step_start<T, DT>(++st)) {
                TileCols<T, DT> gc;
                gc.load_piece(Rows::row(tl, 1, 0), Rows::PITCH, g, c, d0);
#pragma unroll
                for (int dt = d0; dt < d0 + step_most<T>(); ++dt) {
                    if (dt >= d0 + step_of<T, DT>(d0)) continue;
                    const auto go = gc.op(dt);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) x[mt][dt] = collect(go, wf[mt], x[mt][dt]);
                }
            }
            if (end) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    ysum[mt] += group_sum(part[mt]);
                    part[mt] = 0.0f;
                    if constexpr (STAYS) XTile::put(xtile + mt * XTile::FLOATS, x[mt], g, c);
                }
                const float probe = state_probe(x[0]);
                if (__any(probe != probe)) {          // (t is the block's first token)
                    WildCols<T, DT> wild;
                    for (int k = 0; k < block; ++k) wild.take_row(gb + (size_t)(t + k) * stride, g);
                    wild.add_to(wild_bits, g);
                    some_wild = true;
                }
            }
            __syncthreads();
            if (more) rows.store(tl, kb, np ? vb : gb, np ? vb : qb, stride, nt);
            __syncthreads();
        } else {
            WalkRow<T, DT> vr;
            vr.load(Rows::row(tl, 1, c), g);
            F ef[MT];
            f32x4 dv[DT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if constexpr (!QREG) latent_row(q[0], a.Q, mt);
                const GroupRow<T, DT>& qm = q[QREG ? mt : 0];
                const f32x4 s = dot_groups(kr, qm, f32x4{0.f, 0.f, 0.f, 0.f});       // [tau][m]
                const f32x4 st = dot_groups(qm, kr, f32x4{0.f, 0.f, 0.f, 0.f});      // [m][tau]
                const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                float* xt = xtile + (ONE ? 0 : mt * XTile::FLOATS);
                const f32x4 xz = STAYS ? XTile::dot(xt, vr, x[mt], g, c, zero) : XTile::put_dot(xt, vr, x[mt], g, c, zero);
                float et[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float r = exp_nat(s[i] * scale - mref[mt]) * (xz[i] - ysum[mt]);
                    if constexpr (!SEP) r += exp_nat(s[i] * scale - lse[i]) * (gz[mt][i] - gy[i]);
                    ds_out.store(4u * M * (t + 4 * g + i) + lat[mt], r);
                    et[i] = mb + 16 * mt + 4 * g + i < M ? exp_nat(st[i] * scale - mrow[mt][i]) : 0.0f;
                }
                ef[mt] = factor<F>(et[0], et[1], et[2], et[3]);
                if constexpr (ONE) {
                    wave_lds_sync();
                    add_state_product<XTile, T, DT>(dv, xt, ef[mt], mt == 0, g, c);
                    wave_lds_sync();
                }
            }
            if constexpr (!ONE) {
                wave_lds_sync();
#pragma unroll
                for (int st = 0, d1 = 0; st < steps<T, DT>(); d1 = step_start<T, DT>(++st)) {
                    typename XTile::Cols xc[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) xc[mt].load_piece(xtile + mt * XTile::FLOATS, g, c, d1);
#pragma unroll
                    for (int dt = d1; dt < d1 + step_most<T>(); ++dt) {
                        if (dt >= d1 + step_of<T, DT>(d1)) continue;
                        dv[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) dv[dt] = mm(xc[mt].op(dt), ef[mt], dv[dt]);
                    }
                }
            }
            wave_lds_sync();
            put_rows<DT, FLAT>(vtile, VP, dv, g, c);
            if (some_wild) put_wild<T, DT>(vtile, VP, wild_bits, g, c);
            __syncthreads();
            if (more) rows.store(tl, kb, np ? vb : gb, np ? vb : qb, stride, nt);     // every wave is done with this tile
            for (int e = threadIdx.x; e < TT * D / 4; e += blockDim.x) {
                const int ti = e / (D / 4), col = 4 * (e % (D / 4));
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                for (int k = 0; k < NW; ++k) {
                    const f32x4 r = *reinterpret_cast<const f32x4_a*>(smem + k * WF + voff + ti * VP + col);
#pragma unroll
                    for (int n = 0; n < 4; ++n) acc[n] += r[n];
                }
                const float o[4] = {acc[0], acc[1], acc[2], acc[3]};
                store_cols<4>(a.dV, tok + (size_t)(t + ti) * stride + col, o, OD);
            }
            __syncthreads();
        }
        if (!more) break;
        t = nt;
        pass = np;
    }
}

}  // namespace wave
}  // namespace flare
