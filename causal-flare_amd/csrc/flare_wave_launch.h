// flare_wave_launch.h -- instances and launchers of flare_wave.h for one input type
// (included by one translation unit per type, so that they compile side by side).
#pragma once

#include "flare_internal.h"
#include "flare_wave.h"

namespace flare {
namespace wave {

// Latent tiles per wave.  Narrow banks (D <= 32) take 64 latents in one wave: the numerator
// is then 32 registers or less, a 64-latent bank needs no second wave and no barrier, and V
// is read once.  Wider ones keep 32 latents, for occupancy.
template <int DT>
constexpr int latent_tiles(int64_t M) { return DT <= 2 && M > 32 ? 4 : 2; }

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
    if constexpr (DT <= 2)
        if (latent_tiles<DT>(a.M) == 4) return prepare_at<T, 4, DT>(a, cmax, cden, cnum, st);
    return prepare_at<T, 2, DT>(a, cmax, cden, cnum, st);
}
template <typename T, int DT>
int output_dt(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
              hipStream_t st) {
    if constexpr (DT <= 2)
        if (latent_tiles<DT>(a.M) == 4) return output_sep<T, 4, DT>(a, pmax, pden, pnum, Y, out_dtype, st);
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
