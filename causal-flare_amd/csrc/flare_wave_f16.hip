// flare_wave_f16.hip -- the f16 instances of flare_wave.h.
#include "flare_wave_launch.h"

namespace flare {
namespace wave {
int prepare_f16(const WaveArgs& a, float* cmax, float* cden, float* cnum, hipStream_t st) {
    return prepare_type<__half>(a, cmax, cden, cnum, st);
}
int output_f16(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
              hipStream_t st) {
    return output_type<__half>(a, pmax, pden, pnum, Y, out_dtype, st);
}
}  // namespace wave
}  // namespace flare
