// flare_wave_f32.hip -- the f32 instances of flare_wave.h.
#include "flare_wave_launch.h"

namespace flare {
namespace wave {
int prepare_f32(const WaveArgs& a, float* cmax, float* cden, float* cnum, hipStream_t st) {
    return prepare_type<float>(a, cmax, cden, cnum, st);
}
int output_f32(const WaveArgs& a, const float* pmax, const float* pden, const float* pnum, void* Y, int out_dtype,
              hipStream_t st) {
    return output_type<float>(a, pmax, pden, pnum, Y, out_dtype, st);
}
}  // namespace wave
}  // namespace flare
