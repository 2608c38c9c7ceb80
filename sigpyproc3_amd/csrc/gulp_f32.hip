// One-DM dedispersion of a float32 gulp: the dedisperse form of kernels.dedisperse
// (core/kernels.py:340-362) for float32 samples, out[t] = float32(sum over c, in channel order
// and in float64, of in[t + d_c][c]).
//
// The sum of one output is a serial chain over the channels, so the parallelism is the outputs:
// a lane owns one output and a block only 64 of them, so that a gulp of 16384 samples
// still gives nearly every CU a block. What the kernel must hide is then latency. A block's first
// wave only sums; the others plan and load: chunks of FC_CC channels (one 128-byte line of
// each row), FC_DEPTH of them loading into registers and one in LDS, written there channel by
// channel and already shifted by each channel's delay, so that a sum is one LDS read at a
// constant offset, a conversion and an add. One barrier per chunk.
//
// Measured on 1024 channels x 16384 samples, maximum delay 1738 (67 MB): 659 -> 40 us against 512
// outputs and 16 channels per stage without loads in flight across stages (29 blocks); 65536
// samples 655 -> 85 us (3.2 TB/s). Bound by the loading waves' instructions per chunk (plan,
// addresses, LDS writes: about 1.2 us for 32 channels): four chunks in flight (44 us) or 16
// waves (49 us) are slower, and 128 outputs per block run the same 85 us at 65536 samples.
#include "spp_gulp_f32.hpp"

#include "spp_common.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace {

constexpr int FC_WAVES = 8;
constexpr int FC_T = 64;           // outputs per block, one per lane of the summing wave
constexpr int FC_CC = 32;          // channels per chunk: 128 bytes of a row
constexpr int FC_SPREAD = 96;      // delay spread of one pass over a chunk at most
constexpr int FC_LPR = FC_CC / 4;  // lanes loading one row (4 floats each)
constexpr int FC_DELAYS = 4096;    // channels whose delays are kept in LDS (more: read from memory)
constexpr int FC_DEPTH = 2;        // passes loading at a time (even: pass i goes to tile i % 2)

typedef float f32x4 __attribute__((ext_vector_type(4)));
// Word 3 of a raw buffer resource on gfx9-family GPUs: 32-bit data format, no swizzle.
constexpr int kBufferFlags = 0x00020000;

// Inclusive min / max scans over lanes 0..31 (rows 0 and 1 of 16 lanes).
__device__ __forceinline__ int scan_min32(int v) {
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x111, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x112, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x114, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x118, 0xf, 0xf, false));
    return min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x142, 0xa, 0xf, false));
}
__device__ __forceinline__ int scan_max32(int v) {
    v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x111, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x112, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x114, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x118, 0xf, 0xf, false));
    return max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, 0x142, 0xa, 0xf, false));
}

// A pass: channels [s, s + n) of the chunk at channel c0, whose delays span [dmin, dmax] (at
// most FC_SPREAD apart); dl holds the chunk's delays, lane k (and k + 32) channel c0 + k.
struct Pass {
    int64_t c0;
    int s, n, dmin, dmax, dl;
};

__global__ __launch_bounds__(64 * FC_WAVES) void k_ded_f32(const float* __restrict__ in,
                                                           const int32_t* __restrict__ delays,
                                                           float* __restrict__ out, int64_t nchans,
                                                           int64_t nsamps, int64_t nout, int64_t nblocks) {
    constexpr int T = FC_T;
    constexpr int PITCH = T + 2;  // floats per channel of a tile
    constexpr int RPI = 64 * (FC_WAVES - 1) / FC_LPR;     // rows per load instruction of the loading waves
    constexpr int NLD = (T + FC_SPREAD + RPI - 1) / RPI;  // row loads per thread and pass
    __shared__ float tile[2][FC_CC * PITCH];
    __shared__ int2 run[2];  // per tile: the first channel summed and how many
    __shared__ int32_t sdel[FC_DELAYS];
    // consecutive output ranges on one XCD: their row windows overlap in its L2
    const int64_t logical = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    if (logical >= nblocks) return;
    const int64_t t0 = logical * T;
    if (nchans <= FC_DELAYS) {
        for (int i = threadIdx.x; i < static_cast<int>(nchans); i += 64 * FC_WAVES) sdel[i] = delays[i];
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave == 0) {
        double acc = 0.0;
        auto sum_tile = [&](int b) {
            const int2 r = run[b];
            const float* __restrict__ mine = tile[b] + lane;
            if (r.y == FC_CC) {
                // the reads of 16 channels in flight, then the chain of adds
#pragma unroll
                for (int h = 0; h < FC_CC; h += 16) {
                    float x[16];
#pragma unroll
                    for (int k = 0; k < 16; ++k) x[k] = mine[(h + k) * PITCH];
#pragma unroll
                    for (int k = 0; k < 16; ++k) acc += static_cast<double>(x[k]);
                }
            } else {
                for (int k = r.x; k < r.x + r.y; ++k) acc += static_cast<double>(mine[k * PITCH]);
            }
            return r.y;
        };
        __syncthreads();
        for (;;) {
            if (sum_tile(0) == 0) break;
            __syncthreads();
            if (sum_tile(1) == 0) break;
            __syncthreads();
        }
        const int64_t t = t0 + lane;
        if (t < nout) out[t] = static_cast<float>(acc);
        return;
    }
    const int ptid = threadIdx.x - 64;
    const int q = ptid % FC_LPR, r0 = ptid / FC_LPR;

    // Passes in channel order, planned alike in every loading wave from the chunk's delays. They
    // come from LDS: loads return in order, so a wait for delays from memory would drain the rows
    // in flight. n == 0: no pass is left.
    int64_t pc = 0;
    int ps = 0;
    auto load_delay = [&](int64_t c) {
        const int64_t i = min<int64_t>(c + (lane & 31), nchans - 1);
        if (nchans <= FC_DELAYS) return sdel[i];
        const int d = delays[i];
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        return d;
    };
    int dcur = load_delay(0), dnext = load_delay(FC_CC);
    auto next_pass = [&]() {
        Pass p{pc, ps, 0, 0, 0, dcur};
        const int cnt = static_cast<int>(max<int64_t>(0, min<int64_t>(FC_CC, nchans - pc)));
        const bool in_run = lane >= ps && lane < cnt;
        const int mn = scan_min32(in_run ? dcur : INT_MAX), mx = scan_max32(in_run ? dcur : INT_MIN);
        // spreads only grow along the run, so the lanes that fit are its prefix
        const bool fits = in_run && static_cast<int64_t>(mx) - mn <= FC_SPREAD;
        p.n = __popcll(__ballot(fits));
        const int last = __builtin_amdgcn_readfirstlane(max(ps + p.n - 1, 0));
        p.dmin = __builtin_amdgcn_readlane(mn, last);
        p.dmax = __builtin_amdgcn_readlane(mx, last);
        ps += p.n;
        if (ps >= cnt) {
            ps = 0;
            pc += FC_CC;
            dcur = dnext;
        }
        dnext = load_delay(pc + FC_CC);
        return p;
    };
    // The pass's rows [t0 + dmin, t0 + dmax + T), 4 channels per lane; lanes whose channels the
    // pass does not sum load nothing. A lane at the end of a row whose 4 channels would cross it
    // takes the row's last 4 and keeps those that are its own.
    const bool wide = nchans >= 4;
    auto lane_chan = [&](const Pass& p) { return wide ? min<int64_t>(p.c0 + 4 * q, nchans - 4) : p.c0 + 4 * q; };
    auto load_pass = [&](const Pass& p, f32x4 (&v)[NLD]) {
        const int nrows = p.n > 0 ? T + (p.dmax - p.dmin) : 0;
        const int64_t rbase = t0 + p.dmin;
        const int64_t c = lane_chan(p);
        const bool mine = 4 * q < p.s + p.n && 4 * q + 4 > p.s;
        const int64_t span = 4 * nchans * nrows;
        if (wide && rbase >= 0 && rbase + nrows <= nsamps && span < (int64_t(1) << 31)) {
            // one buffer of the pass's rows: lanes and rows that load nothing read past its end (0)
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(in) + rbase * nchans, 0, static_cast<int>(span), kBufferFlags);
            const uint32_t step = static_cast<uint32_t>(4 * nchans) * RPI;
            const uint32_t off = static_cast<uint32_t>(4 * nchans) * r0 + static_cast<uint32_t>(4 * c);
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                uint32_t past = mine && r0 + RPI * i < nrows ? 0u : 0x80000000u;
                asm volatile("" : "+v"(past));  // a select, not a branch round the load
                v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (off + step * i) | past, 0, 0));
            }
        } else {
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int r = r0 + RPI * i;
                int64_t row = rbase + r;
                if (row < 0) row += nsamps;  // numba wraparound of a negative index
                v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (mine && r < nrows && row >= 0 && row < nsamps) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (c + j < nchans) v[i][j] = in[row * nchans + c + j];
                }
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        }
    };
    auto store_pass = [&](const Pass& p, const f32x4 (&v)[NLD], int b) {
        const int nrows = p.n > 0 ? T + (p.dmax - p.dmin) : 0;
        const int col = static_cast<int>(lane_chan(p) - p.c0);
        float* __restrict__ dst[4];
        int rel[4];  // of channel col + j; its sample r belongs to output r - rel
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = col + j;
            rel[j] = __shfl(p.dl, k & 31) - p.dmin;
            if (k < max(4 * q, p.s) || k >= p.s + p.n) rel[j] = nrows;  // not this lane's, or not summed: no output
            dst[j] = tile[b] + k * PITCH - rel[j];
        }
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int r = r0 + RPI * i;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (static_cast<unsigned>(r - rel[j]) < static_cast<unsigned>(T) && r < nrows) dst[j][r] = v[i][j];
        }
        if (ptid == 0) run[b] = make_int2(p.s, p.n);
    };

    // While pass i is summed from one tile, pass i + 1 goes from registers into the other and
    // the FC_DEPTH passes after it are loading. A tile is rewritten only after the barrier that
    // ended the pass that read it; both roles leave at the first empty pass, before its barrier.
    f32x4 v[FC_DEPTH][NLD];
    Pass p[FC_DEPTH];
#pragma unroll
    for (int j = 0; j < FC_DEPTH; ++j) {
        p[j] = next_pass();
        load_pass(p[j], v[j]);
    }
    // Pass j of the ring into its tile, the pass FC_DEPTH after it into its registers; false past
    // the last pass.
    auto advance = [&](auto ring) {
        constexpr int j = decltype(ring)::value;
        const bool more = p[j].n > 0;
        store_pass(p[j], v[j], j & 1);
        p[j] = next_pass();
        load_pass(p[j], v[j]);
        __syncthreads();
        return more;
    };
    static_assert(FC_DEPTH == 2, "one step of the ring per pass loading");
    using std::integral_constant;
    while (advance(integral_constant<int, 0>{}) && advance(integral_constant<int, 1>{})) {
    }
}

}  // namespace

namespace spp {

bool ded_f32_small_blocks(int64_t nchans, int64_t nout, int64_t max_delay) {
    // The 512-output blocks read half as much around their windows and sum up to 256 rows of delay
    // spread in one pass of 16 channels; this kernel's 64-output blocks fill the chip eight times
    // sooner and load passes ahead, but a pass spans 96 rows. So: passes of either kind (the mean
    // number of channels that fit one), times what a pass takes (us, measured over 1 to 1024 channels
    // x 16384 to 1000000 samples, per block on each CU). This kernel against the other: 1024 x 16384
    // 40 / 659, 256 x 131072 at a delay of 5000 221 / 300, 64 x 524288 at 32000 970 / 1440, but
    // 8 x 131072 14 / 8, 3 x 262144 45 / 21, 64 x 262144 at 1024 103 / 79, 512 x 393216 at 8192
    // 1024 / 810.
    auto passes = [&](int64_t spread, int64_t width) {
        const int64_t fit = max_delay > 0 ? std::min(width, 1 + spread * nchans / max_delay) : width;
        return static_cast<double>(ceil_div(nchans, fit));
    };
    const double cus = device_cu_count();
    const double here = passes(FC_SPREAD, FC_CC), blocks = ceil_div(nout, int64_t(FC_T)) / cus;
    const double there = passes(256, 16), blocks512 = ceil_div(nout, int64_t(512)) / cus;
    const double chain = nchans <= 16 ? 7.0 : 11.0;  // a pass of the other on an idle chip
    return std::max(6.0 + here, blocks * (1.6 + 0.4 * here)) <= 1.05 * there * std::max(chain, 5.0 * blocks512);
}

int launch_ded_f32(const float* in, const int32_t* delays, float* out, int64_t nchans, int64_t nsamps, int64_t nout,
                   hipStream_t st) {
    const int64_t nblocks = ceil_div(nout, int64_t(FC_T));
    SPP_REQUIRE(nblocks <= 0x7ffffff0LL, "gulp too long");
    hipLaunchKernelGGL(k_ded_f32, dim3(static_cast<unsigned>(ceil_div(nblocks, int64_t(8)) * 8)), dim3(64 * FC_WAVES),
                       0, st, in, delays, out, nchans, nsamps, nout, nblocks);
    SPP_LAUNCHED("k_ded_f32");
    return SPP_OK;
}

}  // namespace spp
