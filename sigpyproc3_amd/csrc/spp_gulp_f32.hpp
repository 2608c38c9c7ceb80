// One-DM dedispersion of a float32 gulp (gulp_f32.hip), called by spp_dedisperse.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace spp {

// True when blocks of 64 outputs (launch_ded_f32) suit a gulp of nout outputs whose largest delay is
// max_delay; blocks of 512 (k_gulp_f32) otherwise.
bool ded_f32_small_blocks(int64_t nchans, int64_t nout, int64_t max_delay);

// out[t] = float32(sum over c of in[t + delays[c]][c] in float64 and channel order), t < nout.
// Negative rows wrap by nsamps; rows outside the gulp after that read as 0.
int launch_ded_f32(const float* in, const int32_t* delays, float* out, int64_t nchans, int64_t nsamps, int64_t nout,
                   hipStream_t st);

}  // namespace spp
