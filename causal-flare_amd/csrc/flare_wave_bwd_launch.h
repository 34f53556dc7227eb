// flare_wave_bwd_launch.h -- instances and launchers of flare_wave_bwd.h for one input type
// (included by one translation unit per type).
#pragma once

#include "flare_internal.h"
#include "flare_wave_bwd.h"
#include "flare_wave_contract.h"
#include "flare_wave_semi.h"

namespace flare {
namespace wave {

// Latent tiles per wave of the walks: 32 latents.  With 16, four waves a SIMD fit up to D = 64,
// but each tile's rows, g v^T products and sums over latents serve half as many: B 4, N 4096,
// H 16, M 128, D 64 takes 122 + 228 us so and 124 + 166 us with 32; fp32 B 2, N 1024, H 8, M 64,
// D 64 takes 43 + 36 and 33 + 30 us.  At D = 128 a wave of 16 spills as well.
constexpr int kWalkTiles = 2;

// bf16 parts of the fp32 factors (flare_wave_bwd.h): two for the banks whose kernels hold states
// and score gradients as bf16 hi + lo (the 16-bit kernels in flare_ar_bwd.hip and
// flare_bwd_mfma.hip: M 128 and 256, D 64 and 128), three for the others, which were fp32
// throughout.  Three take 437 us where two take 400 (bf16 B 2, N 2048, H 8, M 192, D 128), 305
// and 295 (B 4, M 96, D 64, decoder weights of their own), 230 and 214 (B 4, N 2011, H 16, M 64,
// D 32); of a 256 x 128 bank's X tiles three parts of both would not fit the LDS.
template <typename T, int DT>
bool three_parts(int64_t M) { return sizeof(T) == 2 && !((DT == 4 || DT == 8) && (M == 128 || M == 256)); }
// CALL(P) with the bank's parts (no instance of two where there is no such bank)
#define FLARE_WAVE_PARTS(CALL)                                     \
    if constexpr (sizeof(T) == 2 && DT != 4 && DT != 8) {          \
        return CALL(3);                                            \
    } else {                                                       \
        if constexpr (sizeof(T) == 2)                              \
            if (three_parts<T, DT>(M)) return CALL(3);             \
        return CALL(2);                                            \
    }

template <typename T, int DT>
int launch_lse(const BwdPtrs& p, int64_t B, int64_t N, int64_t H, int64_t M, float scale, hipStream_t st) {
    const int64_t per = TT * kLseTiles * 4;
    hipLaunchKernelGGL((wave_lse_kernel<T, DT>), dim3((unsigned)((N + per - 1) / per), (unsigned)(B * H)), dim3(256), 0, st,
                       (const T*)p.Qdec, (const T*)p.Kdec, (int)N, (int)H, (int)M, scale, (float*)p.lse);
    return check_launch("wave_lse_kernel");
}
inline int launch_carry(const BwdPtrs& p, int64_t NC, int64_t M, int64_t D, int64_t rows, hipStream_t st) {
    const int64_t cols = rows * (D + 1);
    hipLaunchKernelGGL(wave_carry_kernel, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, st, p.xsum, p.ysum, p.pmax,
                       (int)NC, (int)M, (int)D, rows);
    return check_launch("wave_carry_kernel");
}
// Dynamic LDS above the default limit of 64 KB.
inline int allow_lds(const void* kernel, size_t lds, const char* name) {
    if (lds <= 64 * 1024) return FLARE_OK;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess) return FLARE_OK;
    const hipError_t e = hipGetLastError();
    set_error("%s: %zu bytes of LDS refused: %s", name, lds, hipGetErrorString(e));
    return FLARE_ERR_LAUNCH;
}

template <typename T, int MT, int DT, bool SEP, int P>
int bwd_at(const BwdPtrs& p, int64_t B, int64_t N, int64_t H, int64_t M, float scale, int64_t chunk, hipStream_t st) {
    typedef TileRows<T, DT, SEP> Rows;
    const int NW = (int)((M + 16 * MT - 1) / (16 * MT));
    const int64_t NC = (N + chunk - 1) / chunk;
    const dim3 grid((unsigned)NC, (unsigned)(B * H));
    int rc = launch_lse<T, DT>(p, B, N, H, M, scale, st);
    if (rc) return rc;
    const size_t walk_lds = 2 * Rows::BYTES + 2 * NW * TT * sizeof(float);     // row buffers, g . y sums
    hipLaunchKernelGGL((wave_gz_kernel<T, MT, DT, SEP, P>), grid, dim3(64 * NW), walk_lds, st, p, (int)N, (int)H, (int)M,
                       scale, (int)chunk);
    if ((rc = check_launch("wave_gz_kernel"))) return rc;
    if ((rc = launch_carry(p, NC, M, 16 * DT, B * H * M, st))) return rc;
    const size_t lds = sizeof(float) * (size_t)NW * ds_wave_floats<T, MT, DT, P>() + Rows::BYTES;
    if ((rc = allow_lds((const void*)wave_ds_kernel<T, MT, DT, SEP, P>, lds, "wave_ds_kernel"))) return rc;
    hipLaunchKernelGGL((wave_ds_kernel<T, MT, DT, SEP, P>), grid, dim3(64 * NW), lds, st, p, (int)N, (int)H, (int)M, scale,
                       (int)chunk);
    return check_launch("wave_ds_kernel");
}

template <typename T, int MT, int DT, bool SEP, int P>
int semi_at(const BwdPtrs& p, int64_t B, int64_t N, int64_t H, int64_t M, float scale, int64_t chunk, int64_t block,
            hipStream_t st) {
    typedef StepRows<T, DT, SEP ? 3 : 2> Rows;
    const int NW = (int)((M + 16 * MT - 1) / (16 * MT));
    const int64_t NC = (N + chunk - 1) / chunk;
    const dim3 grid((unsigned)NC, (unsigned)(B * H));
    int rc = launch_lse<T, DT>(p, B, N, H, M, scale, st);
    if (rc) return rc;
    const size_t walk_lds = 2 * Rows::BYTES + 2 * NW * TT * sizeof(float);
    hipLaunchKernelGGL((wave_semi_gz_kernel<T, MT, DT, SEP, P>), grid, dim3(64 * NW), walk_lds, st, p, (int)N, (int)H,
                       (int)M, scale, (int)chunk, (int)block);
    if ((rc = check_launch("wave_semi_gz_kernel"))) return rc;
    if ((rc = launch_carry(p, NC, M, 16 * DT, B * H * M, st))) return rc;
    const size_t lds = sizeof(float) * (size_t)NW * semi_wave_floats<T, MT, DT, P>() + Rows::BYTES;
    if ((rc = allow_lds((const void*)wave_semi_ds_kernel<T, MT, DT, SEP, P>, lds, "wave_semi_ds_kernel"))) return rc;
    hipLaunchKernelGGL((wave_semi_ds_kernel<T, MT, DT, SEP, P>), grid, dim3(64 * NW), lds, st, p, (int)N, (int)H, (int)M, scale,
                       (int)chunk, (int)block);
    return check_launch("wave_semi_ds_kernel");
}

template <typename T, int DT>
int bwd_dt(const BwdPtrs& p, bool sep, int64_t B, int64_t N, int64_t H, int64_t M, float scale, int64_t chunk,
           hipStream_t st) {
#define FLARE_CALL(P)                                                               \
    (sep ? bwd_at<T, kWalkTiles, DT, true, P>(p, B, N, H, M, scale, chunk, st)      \
         : bwd_at<T, kWalkTiles, DT, false, P>(p, B, N, H, M, scale, chunk, st))
    FLARE_WAVE_PARTS(FLARE_CALL)
#undef FLARE_CALL
}

template <typename T, int DT>
int semi_dt(const BwdPtrs& p, bool sep, int64_t B, int64_t N, int64_t H, int64_t M, float scale, int64_t chunk,
            int64_t block, hipStream_t st) {
#define FLARE_CALL(P)                                                                      \
    (sep ? semi_at<T, kWalkTiles, DT, true, P>(p, B, N, H, M, scale, chunk, block, st)     \
         : semi_at<T, kWalkTiles, DT, false, P>(p, B, N, H, M, scale, chunk, block, st))
    FLARE_WAVE_PARTS(FLARE_CALL)
#undef FLARE_CALL
}

template <typename T, int DT>
int semi_output_dt(const WaveArgs& a, int64_t block, const float* z, void* Y, int out_dtype, float* lse, hipStream_t st) {
    // (two tiles a wave share a block's z rows; blocks that are an odd number of tiles take one)
    const bool two = block % 32 == 0;
    const int64_t per = 4 * TT * (two ? 2 : 1);
    const dim3 grid((unsigned)((a.N + per - 1) / per), (unsigned)(a.B * a.H));
    if (two)
        hipLaunchKernelGGL((wave_semi_output_kernel<T, DT, 2>), grid, dim3(256), 0, st, (const T*)a.Qdec, (const T*)a.Kdec, z,
                           (int)a.N, (int)a.H, (int)a.M, a.scale, (int)block, Y, out_dtype, lse);
    else
        hipLaunchKernelGGL((wave_semi_output_kernel<T, DT, 1>), grid, dim3(256), 0, st, (const T*)a.Qdec, (const T*)a.Kdec, z,
                           (int)a.N, (int)a.H, (int)a.M, a.scale, (int)block, Y, out_dtype, lse);
    return check_launch("wave_semi_output_kernel");
}

template <typename T, int DT, int P>
int rows_at(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, float scale,
            void* out, hipStream_t st) {
    const int64_t per = 4 * TT * kRowTiles;
    hipLaunchKernelGGL((wave_rows_kernel<T, DT, P>), dim3((unsigned)((N + per - 1) / per), (unsigned)(B * H)), dim3(256), 0, st,
                       p, (const T*)r1, (const T*)r2, (int)N, (int)H, (int)M, scale, (T*)out);
    return check_launch("wave_rows_kernel");
}
template <typename T, int DT, int P>
int cols_at(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, float* partial,
            hipStream_t st) {
    constexpr int MT = DT <= 4 ? 2 : 1;
    hipLaunchKernelGGL((wave_cols_kernel<T, MT, DT, P>),
                       dim3((unsigned)((N + kBwdGroup - 1) / kBwdGroup), (unsigned)((M + 16 * MT - 1) / (16 * MT)),
                            (unsigned)(B * H)),
                       dim3(256), 0, st, p, (const T*)r1, (const T*)r2, (int)N, (int)H, (int)M, partial);
    return check_launch("wave_cols_kernel");
}
template <typename T, int DT>
int rows_dt(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, float scale,
            void* out, hipStream_t st) {
#define FLARE_CALL(P) (rows_at<T, DT, P>(p, r1, r2, B, N, H, M, scale, out, st))
    FLARE_WAVE_PARTS(FLARE_CALL)
#undef FLARE_CALL
}
template <typename T, int DT>
int cols_dt(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, float* partial,
            hipStream_t st) {
#define FLARE_CALL(P) (cols_at<T, DT, P>(p, r1, r2, B, N, H, M, partial, st))
    FLARE_WAVE_PARTS(FLARE_CALL)
#undef FLARE_CALL
}

#define FLARE_WAVE_DT_CASES(NAME, ...)                                                       \
    switch (D / 16) {                                                                        \
        case 1: return NAME<T, 1>(__VA_ARGS__);                                              \
        case 2: return NAME<T, 2>(__VA_ARGS__);                                              \
        case 3: return NAME<T, 3>(__VA_ARGS__);                                              \
        case 4: return NAME<T, 4>(__VA_ARGS__);                                              \
        case 6: return NAME<T, 6>(__VA_ARGS__);                                              \
        case 8: return NAME<T, 8>(__VA_ARGS__);                                              \
        default: break;                                                                      \
    }                                                                                        \
    set_error("wave backward: D=%lld has no instance", (long long)D);                        \
    return FLARE_ERR_INVALID;

template <typename T>
int rows_type(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D,
              float scale, void* out, hipStream_t st) {
    FLARE_WAVE_DT_CASES(rows_dt, p, r1, r2, B, N, H, M, scale, out, st)
}
template <typename T>
int cols_type(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D,
              float* P, hipStream_t st) {
    FLARE_WAVE_DT_CASES(cols_dt, p, r1, r2, B, N, H, M, P, st)
}

template <typename T>
int bwd_type(const BwdPtrs& p, bool sep, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D, float scale,
             int64_t chunk, hipStream_t st) {
    FLARE_WAVE_DT_CASES(bwd_dt, p, sep, B, N, H, M, scale, chunk, st)
}

template <typename T>
int semi_type(const BwdPtrs& p, bool sep, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D, float scale,
              int64_t chunk, int64_t block, hipStream_t st) {
    FLARE_WAVE_DT_CASES(semi_dt, p, sep, B, N, H, M, scale, chunk, block, st)
}

template <typename T>
int semi_output_type(const WaveArgs& a, int64_t block, const float* z, void* Y, int out_dtype, float* lse, hipStream_t st) {
    const int64_t D = a.D;
    FLARE_WAVE_DT_CASES(semi_output_dt, a, block, z, Y, out_dtype, lse, st)
}

}  // namespace wave
}  // namespace flare
