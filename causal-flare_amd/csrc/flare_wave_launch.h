// flare_wave_launch.h -- instances and launchers of flare_wave.h for one input type
// (included by one translation unit per type, so that they compile side by side).
#pragma once

#include "flare_internal.h"
#include "flare_wave.h"

namespace flare {
namespace wave {

// Latent tiles per wave, the chunk being set: the most that still leave a wave per SIMD (1024),
// since fewer, larger waves repeat less (V, the y rows, G V); below that, smaller waves for a
// shorter chain.  Narrow banks (D <= 32) go up to 64 latents, a 64-latent bank then needs no
// second wave and no barrier; wider ones to 32, for registers.  Phase 3, us, with 64 / 32 / 16
// latents a wave: bf16 B 8, N 4096, H 16, M 64, D 32 (2048 / 4096 / 8192 waves) 124 / 132 / 145;
// fp32 B 2, N 1024, H 8, M 64, D 64 in chunks of 128 (256 / 512 waves of 32 / 16) 46 / 36.
// 16 latents a wave only up to M = 128 (see wave_threads) and D = 64.
template <int DT>
int latent_tiles(const WaveArgs& a) {
    const int64_t wgs = a.B * a.H * ((a.N + a.chunk - 1) / a.chunk);
    for (int mt = DT <= 2 ? 4 : 2; mt > 1; mt >>= 1)
        if (wgs * ((a.M + 16 * mt - 1) / (16 * mt)) >= 1024) return mt;
    return a.M <= 128 && DT <= 4 ? 1 : 2;
}

template <typename T, int MT, int DT>
int prepare_at(const WaveArgs& a, float* cmax, float* cden, float* cnum, hipStream_t st) {
    const int NW = (int)((a.M + 16 * MT - 1) / (16 * MT));
    const int64_t NC = (a.N + a.chunk - 1) / a.chunk;
    hipLaunchKernelGGL((wave_prepare_kernel<T, MT, DT>), dim3((unsigned)NC, (unsigned)(a.B * a.H)), dim3(64 * NW), 0, st,
                       (const T*)a.Q, (const T*)a.K, (const T*)a.V, (int)a.N, (int)a.H, (int)a.M, a.scale, (int)a.chunk,
                       cmax, cden, cnum, a.tmask);
    return check_launch("wave_prepare_kernel");
}

template <typename T, int MT, int DT, bool SEP>
int output_at(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
              hipStream_t st) {
    const int NW = (int)((a.M + 16 * MT - 1) / (16 * MT));
    const int64_t NC = (a.N + a.chunk - 1) / a.chunk;
    const size_t lds = wave_output_lds<MT, DT>(NW);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)wave_output_kernel<T, MT, DT, SEP>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            set_error("wave_output_kernel: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
            return FLARE_ERR_LAUNCH;
        }
    }
    hipLaunchKernelGGL((wave_output_kernel<T, MT, DT, SEP>), dim3((unsigned)NC, (unsigned)(a.B * a.H)), dim3(64 * NW),
                       lds, st, (const T*)a.Q, (const T*)a.K, (const T*)a.V, (const T*)(a.Qdec ? a.Qdec : a.K),
                       (const T*)(a.Kdec ? a.Kdec : a.Q), (int)a.N, (int)a.H, (int)a.M, a.scale, (int)a.chunk, pmax,
                       pden, pnum, Y, out_dtype, a.tmask);
    return check_launch("wave_output_kernel");
}

template <typename T, int MT, int DT>
int output_sep(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
               hipStream_t st) {
    return a.Qdec || a.Kdec ? output_at<T, MT, DT, true>(a, pmax, pden, pnum, Y, out_dtype, st)
                            : output_at<T, MT, DT, false>(a, pmax, pden, pnum, Y, out_dtype, st);
}

template <typename T, int DT>
int prepare_dt(const WaveArgs& a, float* cmax, float* cden, float* cnum, hipStream_t st) {
    const int mt = latent_tiles<DT>(a);
    if constexpr (DT <= 2)
        if (mt == 4) return prepare_at<T, 4, DT>(a, cmax, cden, cnum, st);
    if constexpr (DT <= 4)
        if (mt == 1) return prepare_at<T, 1, DT>(a, cmax, cden, cnum, st);
    return prepare_at<T, 2, DT>(a, cmax, cden, cnum, st);
}
template <typename T, int DT>
int output_dt(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
              hipStream_t st) {
    const int mt = latent_tiles<DT>(a);
    if constexpr (DT <= 2)
        if (mt == 4) return output_sep<T, 4, DT>(a, pmax, pden, pnum, Y, out_dtype, st);
    if constexpr (DT <= 4)
        if (mt == 1) return output_sep<T, 1, DT>(a, pmax, pden, pnum, Y, out_dtype, st);
    return output_sep<T, 2, DT>(a, pmax, pden, pnum, Y, out_dtype, st);
}

#define FLARE_WAVE_DT(D, CALL)      \
    switch ((D) / 16) {             \
        case 1: return CALL(1);     \
        case 2: return CALL(2);     \
        case 3: return CALL(3);     \
        case 4: return CALL(4);     \
        case 6: return CALL(6);     \
        case 8: return CALL(8);     \
        default: break;             \
    }

template <typename T>
int prepare_type(const WaveArgs& a, float* cmax, float* cden, float* cnum, hipStream_t st) {
#define FLARE_CALL(DT) prepare_dt<T, DT>(a, cmax, cden, cnum, st)
    FLARE_WAVE_DT(a.D, FLARE_CALL)
#undef FLARE_CALL
    set_error("wave_prepare: D=%lld has no instance", (long long)a.D);
    return FLARE_ERR_INVALID;
}
template <typename T>
int output_type(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
                hipStream_t st) {
#define FLARE_CALL(DT) output_dt<T, DT>(a, pmax, pden, pnum, Y, out_dtype, st)
    FLARE_WAVE_DT(a.D, FLARE_CALL)
#undef FLARE_CALL
    set_error("wave_output: D=%lld has no instance", (long long)a.D);
    return FLARE_ERR_INVALID;
}

}  // namespace wave
}  // namespace flare
