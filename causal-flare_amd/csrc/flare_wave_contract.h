// flare_wave_contract.h -- the backward's contractions of the score gradients with the token
// and latent rows, on the products of flare_wave_bwd.h (fp32 MFMA for fp32 inputs, bf16
// parts for 16-bit ones):
//   rows   out[t][d] = scale sum_m G[t][m] R[m][d]            (dK, dQ_dec)
//   cols   P[group][m][d] = sum_{t in group} G[t][m] R[t][d]  (dQ, dK_dec, before the sum
//                                                              over groups and sequences)
// G is ds, or da = alpha (gz - gy) formed as it is read (score_grad_da), or both with rows of
// their own.  Serves the banks without an instance of bwd_dk_mfma / bwd_dq_mfma.
//
// Both are bound by reading G once (fp32, [B*H, N, M]).  rows: a wave takes 32 tokens against
// all latents, R's rows come from cache.  cols: the four waves of a workgroup take a quarter
// of a 512-token group each and add their tiles through LDS, so that a group's serial chain
// is 8 tiles and no result is split over the chip's workgroups further than the groups.
#pragma once

#include "flare_wave_bwd.h"

namespace flare {
namespace wave {

// One source of score gradients: DS, or da from C, AL and gy.
struct GradSrc {
    Floats ds, c, al, gy;
    bool own, cgz;
    __device__ __forceinline__ float at(unsigned byte, int t) const {
        if (own) return ds.load(byte);
        return score_grad_da(c.load(byte), al.load(byte), gy.load(4u * t), cgz);
    }
    // four latents of one token
    __device__ __forceinline__ f32x4 four(unsigned byte, int t) const {
        if (own) return load4(ds, byte);
        const f32x4 x = load4(c, byte), y = load4(al, byte);
        const float z = gy.load(4u * t);
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = score_grad_da(x[i], y[i], z, cgz);
        return r;
    }
    static __device__ __forceinline__ f32x4 load4(const Floats& f, unsigned byte) {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(f.r, byte, 0, 0));
    }
};
__device__ __forceinline__ GradSrc grad_src(const ContractPtrs& p, bool own, int bh, int N, int M) {
    const size_t per = (size_t)N * M, at = bh * per;
    return GradSrc{Floats(p.ds + at, per), Floats(own ? p.ds : p.c + at, own ? 0 : per),
                   Floats(own ? p.ds : p.al + at, own ? 0 : per), Floats(p.gy + (size_t)bh * N, N), own, p.cgz};
}

// grid (ceil(N / 128), B*H), four waves of 32 tokens.  r1 / r2: rows [H, M, D] that ds / da
// contract with (either may be null).
constexpr int kRowTiles = 2;
template <typename T, int DT, int P>
__global__ __launch_bounds__(256) void wave_rows_kernel(ContractPtrs p, const T* __restrict__ r1, const T* __restrict__ r2,
                                                        int N, int H, int M, float scale, T* __restrict__ out) {
    constexpr int D = 16 * DT;
    constexpr int OD = sizeof(T) == 4 ? FLARE_F32 : __is_same(T, __half) ? FLARE_F16 : FLARE_BF16;
    typedef typename ProdOf<T, P>::F F;
    const int bh = blockIdx.y, b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int t0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * TT * kRowTiles;
    if (t0 >= N) return;
    f32x4 acc[kRowTiles][DT];
#pragma unroll
    for (int k = 0; k < kRowTiles; ++k)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[k][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int term = 0; term < 2; ++term) {
        const T* r = term == 0 ? r1 : r2;
        if (r == nullptr) continue;
        const GradSrc src = grad_src(p, term == 0, bh, N, M);
        const T* rh = r + (size_t)h * M * D;
        for (int m0 = 0; m0 < M; m0 += 16) {
            TokCols<T, DT> q;
            f32x4 x[kRowTiles];
#pragma unroll
            for (int k = 0; k < kRowTiles; ++k) {
                const int t = t0 + TT * k + c;       // (past N: reads 0)
                x[k] = src.four(4u * (unsigned)(t * M + m0 + 4 * g), t);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) q.r[i].load(rh + (size_t)(m0 + 4 * g + i) * D, c);
            F f[kRowTiles];
#pragma unroll
            for (int k = 0; k < kRowTiles; ++k) f[k] = factor<F>(x[k][0], x[k][1], x[k][2], x[k][3]);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const auto op = q.op(dt);
#pragma unroll
                for (int k = 0; k < kRowTiles; ++k) acc[k][dt] = collect(f[k], op, acc[k][dt]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kRowTiles; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + TT * k + 4 * g + i;
            if (t >= N) continue;
            const size_t row = (((size_t)b * N + t) * H + h) * D;
#pragma unroll
            for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc)) {
                float o[4];
                const int cols = piece_of<DT>(dt);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = e < cols ? scale * acc[k][dt + e < DT ? dt + e : 0][i] : 0.0f;
                const size_t at = row + col_of<DT>(dt, c);
                if (cols == 4) store_cols<4>(out, at, o, OD);
                else if (cols == 2) store_cols<2>(out, at, o, OD);
                else store_cols<1>(out, at, o, OD);
            }
        }
}

// grid (groups, ceil(M / (16 MT)), B*H), four waves.  r1 / r2: rows [B, N, H, D].
template <typename T, int MT, int DT, int P>
__global__ __launch_bounds__(256) void wave_cols_kernel(ContractPtrs p, const T* __restrict__ r1, const T* __restrict__ r2,
                                                        int N, int H, int M, float* __restrict__ partial) {
    constexpr int D = 16 * DT, PITCH = D + 4;
    typedef typename ProdOf<T, P>::F F;
    __shared__ __attribute__((aligned(16))) float part[4][16 * MT][PITCH];
    const int bh = blockIdx.z, b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    const int mb = blockIdx.y * 16 * MT;
    const int t0 = blockIdx.x * kBwdGroup + w * (kBwdGroup / 4), t1 = min(N, t0 + kBwdGroup / 4);
    const size_t stride = (size_t)H * D;
    unsigned lat[MT];
    f32x4 acc[MT][DT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        lat[mt] = mb + 16 * mt + c < M ? 4u * (mb + 16 * mt + c) : kNowhere;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[mt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int term = 0; term < 2; ++term) {
        const T* r = term == 0 ? r1 : r2;
        if (r == nullptr) continue;
        const GradSrc src = grad_src(p, term == 0, bh, N, M);
        const T* rh = r + ((size_t)b * N * H + h) * D;
        for (int t = t0; t < t1; t += TT) {
            TokCols<T, DT> k;
            float x[MT][4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ti = t + 4 * g + i;
                k.r[i].load(rh + (size_t)min(ti, N - 1) * stride, c);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[mt][i] = src.at(4u * M * ti + lat[mt], ti);
            }
            F f[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) f[mt] = factor<F>(x[mt][0], x[mt][1], x[mt][2], x[mt][3]);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const auto op = k.op(dt);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt][dt] = collect(op, f[mt], acc[mt][dt]);
            }
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int pc = 0, dt = 0; pc < pieces<DT>(); dt = piece_start<DT>(++pc))
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e < piece_of<DT>(dt))
                        part[w][16 * mt + c][col_of<DT>(dt, 4 * g + i) + e] = acc[mt][dt + e < DT ? dt + e : 0][i];
    __syncthreads();
    for (int x = threadIdx.x; x < 16 * MT * D; x += 256) {
        const int m = x / D, d = x % D;
        if (mb + m < M)
            partial[(((size_t)bh * gridDim.x + blockIdx.x) * M + mb + m) * D + d] =
                (part[0][m][d] + part[1][m][d]) + (part[2][m][d] + part[3][m][d]);
    }
}

}  // namespace wave
}  // namespace flare
