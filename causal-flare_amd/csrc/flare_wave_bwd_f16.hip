// flare_wave_bwd_f16.hip -- the f16 instances of flare_wave_bwd.h, flare_wave_semi.h and flare_wave_contract.h.
#include "flare_wave_bwd_launch.h"

namespace flare {
namespace wave {
int bwd_f16(const BwdPtrs& p, bool sep, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D, float scale,
           int64_t chunk, hipStream_t st) {
    return bwd_type<__half>(p, sep, B, N, H, M, D, scale, chunk, st);
}
int semi_f16(const BwdPtrs& p, bool sep, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D, float scale,
             int64_t chunk, int64_t block, hipStream_t st) {
    return semi_type<__half>(p, sep, B, N, H, M, D, scale, chunk, block, st);
}
int rows_f16(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D,
             float scale, void* out, hipStream_t st) {
    return rows_type<__half>(p, r1, r2, B, N, H, M, D, scale, out, st);
}
int cols_f16(const ContractPtrs& p, const void* r1, const void* r2, int64_t B, int64_t N, int64_t H, int64_t M, int64_t D,
             float* P, hipStream_t st) {
    return cols_type<__half>(p, r1, r2, B, N, H, M, D, P, st);
}
int semi_output_f16(const WaveArgs& a, int64_t block, const float* z, void* Y, int out_dtype, float* lse, hipStream_t st) {
    return semi_output_type<__half>(a, block, z, Y, out_dtype, lse, st);
}
}  // namespace wave
}  // namespace flare
