// flare_wave_bf16.hip -- the bf16 instances of flare_wave.h.
#include "flare_wave_launch.h"

namespace flare {
namespace wave {
int prepare_bf16(const WaveArgs& a, float* cmax, float* cden, float* cnum, hipStream_t st) {
    return prepare_type<__hip_bfloat16>(a, cmax, cden, cnum, st);
}
int output_bf16(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
              hipStream_t st) {
    return output_type<__hip_bfloat16>(a, pmax, pden, pnum, Y, out_dtype, st);
}
}  // namespace wave
}  // namespace flare
