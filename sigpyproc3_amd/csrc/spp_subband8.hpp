// Subbands of an 8-bit gulp with whole bands per block (subband8.hip), called by spp_subband.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace spp {

// True when the kernel takes this launch (nbits == 8).
bool subband8_applies(const void* in, int64_t nchans, int64_t nsamps, int64_t nout, int64_t nsubs);

// out[t * nsubs + chan_to_sub[c]] += in[t + delays[c]][c] over all channels, t < nout, on an `out`
// that is already zero; flat indices >= out_size are dropped.
int launch_subband8(const uint8_t* in, const int32_t* delays, const int32_t* chan_to_sub, float* out, int64_t nchans,
                    int64_t nsamps, int64_t nout, int64_t nsubs, int64_t out_size, hipStream_t st);

}  // namespace spp
