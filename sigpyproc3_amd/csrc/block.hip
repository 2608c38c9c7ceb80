// In-memory filterbank blocks (float32, [nchans][nsamps], channel-major): per-row rolls and
// the DM-time transform.
//
// Both read row r at column (t + off_r) mod ncols. The host turns the reference's shifts
// into offsets: a circular roll by s gives off = -s mod ncols (kernels.roll_block,
// core/kernels.py:1059-1099); the valid-columns form gives off = start - s with
// start = max(0, max s) (kernels.roll_block_valid, core/kernels.py:1102-1152), so the
// wrap never triggers there.
//
// The DM-time transform adds the rolled rows of every channel in channel order, starting
// from 0, in float32 (the per-column order of np.sum(..., axis=0) in kernels.dmt_block,
// core/kernels.py:1155-1193), so results are bit-exact to the reference's.
#include "spp_common.hpp"

#include <algorithm>

namespace {

constexpr int RB_THREADS = 256;

__global__ __launch_bounds__(RB_THREADS) void k_roll_rows(const float* __restrict__ in, int64_t ncols,
                                                          const int64_t* __restrict__ off,
                                                          int64_t out_cols, float* __restrict__ out) {
    const int64_t r = blockIdx.y;
    const int64_t o = off[r];
    const float* __restrict__ src = in + r * ncols;
    float* __restrict__ dst = out + r * out_cols;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * RB_THREADS + threadIdx.x; t < out_cols;
         t += static_cast<int64_t>(gridDim.x) * RB_THREADS) {
        int64_t j = t + o;
        if (j >= ncols) j -= ncols;
        dst[t] = src[j];
    }
}

// The same roll with 16-byte stores: a thread writes RV float4s of row blockIdx.y (out rows
// 16-byte aligned: out 16-byte aligned, out_cols % 4 == 0), reading the 4 sources of each as
// plain loads (the source offset is arbitrary; a float4 that straddles the wrap takes its
// elements one by one).
constexpr int RV = 4;
__global__ __launch_bounds__(RB_THREADS) void k_roll_rows4(const float* __restrict__ in, int64_t ncols,
                                                           const int64_t* __restrict__ off,
                                                           int64_t out_cols, float* __restrict__ out) {
    const int64_t r = blockIdx.y;
    const int64_t o = off[r];
    const float* __restrict__ src = in + r * ncols;
    float4* __restrict__ dst = reinterpret_cast<float4*>(out + r * out_cols);
    const int64_t nv = out_cols / 4;
    const int64_t v0 = static_cast<int64_t>(blockIdx.x) * RB_THREADS * RV + threadIdx.x;
    float4 q[RV];
#pragma unroll
    for (int i = 0; i < RV; ++i) {
        const int64_t v = v0 + static_cast<int64_t>(i) * RB_THREADS;
        if (v >= nv) break;
        int64_t j = 4 * v + o;
        if (j >= ncols) j -= ncols;
        if (j + 4 <= ncols) {
            q[i] = make_float4(src[j], src[j + 1], src[j + 2], src[j + 3]);
        } else {
            float e[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) e[k] = src[j + k >= ncols ? j + k - ncols : j + k];
            q[i] = make_float4(e[0], e[1], e[2], e[3]);
        }
    }
#pragma unroll
    for (int i = 0; i < RV; ++i) {
        const int64_t v = v0 + static_cast<int64_t>(i) * RB_THREADS;
        if (v < nv) dst[v] = q[i];
    }
}

// DM-time transform. A block sums DT_D DM rows over DT_K * 256 output samples. Per channel the
// rows read the same samples at offsets that differ by little, so the window that covers them
// is staged in LDS once (loads with the LDS flag, a stage of channels ahead of the sums) and each
// row reads it at its own offset: one LDS read and one add per (row, channel, sample), where a
// thread per output made one L2 read of it. A channel whose rows' offsets span more than the
// window holds is read from memory instead. Every output adds its channels in order.
//
// Measured on 1024 channels x 8192 samples, 512 DM rows: 2436 -> 618 us (4.3e9 adds; the LDS
// reads alone take 220 at 128 bytes per clock and CU, the rest is the wait of each 5-channel
// stage). Windows of 128 spare samples and 8 channels run 528 there but leave 2000 channels x
// 16384, 128 rows (offsets up to 450 apart) to memory. Where most channels are added from memory:
// 1024 x 65536, 32 rows spread over 30000 samples, 1230 us (1587 with a thread per output and one load
// in flight, 2380 in a tile with one in flight).
constexpr int DT_D = 8;         // DM rows per block
constexpr int DT_K = 4;         // samples per thread
constexpr int DT_CC = 5;        // channels per stage
constexpr int DT_SPREAD = 512;  // offset spread of a window's rows at most
constexpr int DT_PLAN = 480;    // channels whose windows are planned at a time (two blocks' LDS fit a CU)
// Word 3 of a raw buffer resource on gfx9-family GPUs: 32-bit data format, no swizzle.
constexpr int kBufferFlags = 0x00020000;
typedef __attribute__((address_space(3))) void lds_void_t;

__global__ __launch_bounds__(RB_THREADS) void k_dmt(const float* __restrict__ in, int64_t nchans,
                                                    int32_t ncols, const int64_t* __restrict__ off,
                                                    int64_t ndm, int32_t out_cols, float* __restrict__ out) {
    constexpr int K = DT_K, CC = DT_CC;
    constexpr int T = RB_THREADS * K;
    constexpr int W = T + DT_SPREAD;  // samples of a staged window
    static_assert(W % 64 == 0 && DT_PLAN % CC == 0, "whole waves of loads per window, whole stages per plan");
    __shared__ float win[2][CC * W];
    __shared__ int32_t wstart[DT_PLAN];  // column of a window's first sample; -1: not staged
    __shared__ uint4 wrel[DT_PLAN];      // the rows' offsets in the window, 16 bits each
    static_assert(DT_D == 8, "eight 16-bit offsets per channel");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t i0 = static_cast<int64_t>(blockIdx.y) * DT_D;
    const int t0 = blockIdx.x * T;

    // The window of channel c: rows' offsets relative to the first row's, the nearer way round
    // the block. Rows past the last repeat it.
    auto plan = [&](int64_t c, int slot) {
        int32_t o[DT_D];
#pragma unroll
        for (int r = 0; r < DT_D; ++r) o[r] = static_cast<int32_t>(off[min<int64_t>(i0 + r, ndm - 1) * nchans + c]);
        int rel[DT_D], mn = 0, mx = 0;
#pragma unroll
        for (int r = 0; r < DT_D; ++r) {
            rel[r] = o[r] - o[0];
            if (2 * static_cast<int64_t>(rel[r]) > ncols) rel[r] -= ncols;
            else if (2 * static_cast<int64_t>(rel[r]) < -static_cast<int64_t>(ncols)) rel[r] += ncols;
            mn = min(mn, rel[r]);
            mx = max(mx, rel[r]);
        }
        int col = o[0] + t0;  // both below ncols
        col = col >= ncols ? col - ncols : col;
        col += mn;
        col = col < 0 ? col + ncols : col;
        wstart[slot] = mx - mn <= DT_SPREAD ? col : -1;  // W <= ncols (dmt_in_tiles)
        auto pair = [&](int r) {
            return static_cast<uint32_t>((rel[r] - mn) & 0xffff) | static_cast<uint32_t>(rel[r + 1] - mn) << 16;
        };
        wrel[slot] = make_uint4(pair(0), pair(2), pair(4), pair(6));
    };
    // A stage's windows into LDS, a wave 64 samples at a time.
    auto stage = [&](int b, int64_t c, int slot) {
#pragma unroll
        for (int k = 0; k < CC; ++k) {
            const int start = __builtin_amdgcn_readfirstlane(wstart[slot + k]);
            if (c + k >= nchans || start < 0) continue;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(in) + (c + k) * ncols, 0, ncols * 4, kBufferFlags);
#pragma unroll
            for (int u = 0; u < (W + RB_THREADS - 1) / RB_THREADS; ++u) {
                const int x = RB_THREADS * u + 64 * wave;
                if (x >= W) break;
                int col = start + x + lane;  // < 2 * ncols
                col = col >= ncols ? col - ncols : col;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)(&win[b][k * W + x]), 4, 4 * col, 0, 0, 0);
            }
        }
    };

    float acc[DT_D][K];
#pragma unroll
    for (int r = 0; r < DT_D; ++r)
#pragma unroll
        for (int k = 0; k < K; ++k) acc[r][k] = 0.0f;
    auto add_staged = [&](int b, int k, int slot) {
        const float* __restrict__ w = &win[b][k * W + tid];
        const uint4 q = wrel[slot + k];
        const uint32_t rel2[4] = {static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(q.x)),
                                  static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(q.y)),
                                  static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(q.z)),
                                  static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(q.w))};
        float v[DT_D][K];
#pragma unroll
        for (int r = 0; r < DT_D; ++r) {
            const float* __restrict__ src = w + ((rel2[r / 2] >> (16 * (r & 1))) & 0xffffu);
#pragma unroll
            for (int j = 0; j < K; ++j) v[r][j] = src[RB_THREADS * j];
        }
#pragma unroll
        for (int r = 0; r < DT_D; ++r)
#pragma unroll
            for (int j = 0; j < K; ++j) acc[r][j] = acc[r][j] + v[r][j];
    };
    // A channel without a window: a row's loads at a time, the rows' waits at the end. (The empty asm
    // keeps the compiler from mixing the rows: with all 32 loads in one group the staged sums get fewer
    // registers, 630 us instead of 587 at 1024 x 8192, 512 rows, for 1002 instead of 1230 at the spread rows named above.)
    auto add_direct = [&](int64_t c) {
        const float* __restrict__ row = in + c * ncols;
        int td[K];  // the thread's samples; those past the last output repeat it
#pragma unroll
        for (int j = 0; j < K; ++j) td[j] = min(t0 + tid + RB_THREADS * j, out_cols - 1);
        float v[DT_D][K];
#pragma unroll
        for (int r = 0; r < DT_D; ++r) {
            const int o = static_cast<int>(off[min<int64_t>(i0 + r, ndm - 1) * nchans + c]);
#pragma unroll
            for (int j = 0; j < K; ++j) {
                const int col = o + td[j];
                v[r][j] = row[col >= ncols ? col - ncols : col];
            }
            asm volatile("");
        }
#pragma unroll
        for (int r = 0; r < DT_D; ++r)
#pragma unroll
            for (int j = 0; j < K; ++j) acc[r][j] = acc[r][j] + v[r][j];
        asm volatile("");
    };
    for (int64_t c0 = 0; c0 < nchans; c0 += DT_PLAN) {
        bool mine = true;
        for (int s = tid; s < DT_PLAN && c0 + s < nchans; s += RB_THREADS) {
            plan(c0 + s, s);
            mine = mine && wstart[s] >= 0;
        }
        const bool all_staged = __syncthreads_and(mine);
        const int64_t ce = min(nchans, c0 + DT_PLAN);
        stage(0, c0, 0);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the windows have landed
        __syncthreads();
        int b = 0;
        for (int64_t c = c0; c < ce; c += CC, b ^= 1) {
            const int slot = static_cast<int>(c - c0);
            if (c + CC < ce) stage(b ^ 1, c + CC, slot + CC);
            const int nk = static_cast<int>(min<int64_t>(CC, ce - c));
            if (all_staged && nk == CC) {
#pragma unroll
                for (int k = 0; k < CC; ++k) add_staged(b, k, slot);
            } else {
#pragma unroll 1
                for (int k = 0; k < nk; ++k) {
                    if (__builtin_amdgcn_readfirstlane(wstart[slot + k]) >= 0) add_staged(b, k, slot);
                    else add_direct(c + k);
                }
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the next windows have landed
            __syncthreads();
        }
    }
#pragma unroll
    for (int r = 0; r < DT_D; ++r) {
        if (i0 + r >= ndm) break;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int t = t0 + tid + RB_THREADS * j;
            if (t < out_cols) out[(i0 + r) * out_cols + t] = acc[r][j];
        }
    }
}

// One thread per output sample of one DM row, eight channels' loads in flight.
__global__ __launch_bounds__(RB_THREADS) void k_dmt_rows(const float* __restrict__ in, int64_t nchans,
                                                         int64_t ncols, const int64_t* __restrict__ off,
                                                         int64_t out_cols, float* __restrict__ out) {
    const int64_t i = blockIdx.y;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * RB_THREADS + threadIdx.x;
    if (t >= out_cols) return;
    const int64_t* __restrict__ oi = off + i * nchans;
    auto at = [&](int64_t c) {
        const int64_t j = t + oi[c];
        return in[c * ncols + (j >= ncols ? j - ncols : j)];
    };
    float acc = 0.0f;
    int64_t c = 0;
    for (; c + 8 <= nchans; c += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = at(c + k);
#pragma unroll
        for (int k = 0; k < 8; ++k) acc = acc + v[k];
    }
    for (; c < nchans; ++c) acc = acc + at(c);
    out[i * out_cols + t] = acc;
}

int check_offsets(const int64_t* off_host, int64_t n, int64_t ncols) {
    for (int64_t k = 0; k < n; ++k) {
        SPP_REQUIRE(off_host[k] >= 0 && off_host[k] < ncols, "offset %lld outside [0, %lld)",
                    static_cast<long long>(off_host[k]), static_cast<long long>(ncols));
    }
    return SPP_OK;
}

}  // namespace

extern "C" int spp_roll_rows(const float* in, int64_t nrows, int64_t ncols, const int64_t* off_host,
                             const int64_t* off, int64_t out_cols, float* out, void* stream) {
    spp::clear_error();
    SPP_REQUIRE(in != nullptr && off != nullptr && out != nullptr && off_host != nullptr, "null argument");
    SPP_REQUIRE(nrows > 0 && ncols > 0 && out_cols > 0 && out_cols <= ncols,
                "need nrows, ncols > 0 and 0 < out_cols <= ncols");
    SPP_REQUIRE(nrows <= 65535, "at most 65535 rows per call");
    if (check_offsets(off_host, nrows, ncols)) return SPP_EINVAL;
    for (int64_t r = 0; r < nrows; ++r) {
        if (off_host[r] + out_cols > ncols && out_cols < ncols) {
            // only a full-width (circular) output may wrap
            SPP_REQUIRE(false, "row %lld: offset %lld + out_cols %lld wraps in a valid-columns roll",
                        static_cast<long long>(r), static_cast<long long>(off_host[r]),
                        static_cast<long long>(out_cols));
        }
    }
    if (out_cols % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
        const int64_t bx4 = spp::ceil_div(out_cols / 4, int64_t(RB_THREADS) * RV);
        SPP_REQUIRE(bx4 <= 0x7fffffffLL, "too many columns");
        hipLaunchKernelGGL(k_roll_rows4, dim3(static_cast<unsigned>(bx4), static_cast<unsigned>(nrows)),
                           dim3(RB_THREADS), 0, spp::as_stream(stream), in, ncols, off, out_cols, out);
        SPP_LAUNCHED("k_roll_rows4");
        return SPP_OK;
    }
    const int64_t bx = std::min<int64_t>(spp::ceil_div(out_cols, int64_t(RB_THREADS)), 4096);
    hipLaunchKernelGGL(k_roll_rows, dim3(static_cast<unsigned>(bx), static_cast<unsigned>(nrows)),
                       dim3(RB_THREADS), 0, spp::as_stream(stream), in, ncols, off, out_cols, out);
    SPP_LAUNCHED("k_roll_rows");
    return SPP_OK;
}

namespace spp {

// True when the tiled transform (k_dmt) takes the call.
bool dmt_in_tiles(int64_t ncols, int64_t ndm, int64_t out_cols) {
    // A window must fit the row (with every channel added from memory, 1024 channels x 1024 samples,
    // 2048 rows take 917 us in tiles and 481 with a thread per output; 1500 samples 1217 and 721), its
    // byte offsets 32 bits, and a tile must hold four rows or more (it sums eight whatever it holds:
    // 256 x 300000, offsets far apart, 2 rows 315 and 100, 4 rows 327 and 195; near each other 3
    // rows 150 and 118, 4 rows 170 and 190). And a tile per CU: 256 rows of 1024 channels x 2048 samples
    // (64 tiles): 151 us with a thread per output, 402 in small tiles; 512 rows of 336 x 5001 (320
    // tiles): 203 tiled, 453 with a thread per output.
    const int64_t by = ceil_div(ndm, int64_t(DT_D)), bx = ceil_div(out_cols, int64_t(RB_THREADS) * DT_K);
    return ncols >= RB_THREADS * DT_K + DT_SPREAD && ncols < (int64_t(1) << 29) && ndm >= DT_D / 2 && bx * by >= device_cu_count();
}

}  // namespace spp

extern "C" int spp_dmt(const float* in, int64_t nchans, int64_t ncols, const int64_t* off_host,
                       const int64_t* off, int64_t ndm, int64_t out_cols, float* out, void* stream) {
    spp::clear_error();
    SPP_REQUIRE(in != nullptr && off != nullptr && out != nullptr && off_host != nullptr, "null argument");
    SPP_REQUIRE(nchans > 0 && ncols > 0 && ndm > 0 && out_cols > 0 && out_cols <= ncols,
                "need nchans, ncols, ndm > 0 and 0 < out_cols <= ncols");
    SPP_REQUIRE(ndm <= 65535, "at most 65535 DM rows per call");
    if (check_offsets(off_host, ndm * nchans, ncols)) return SPP_EINVAL;
    if (out_cols < ncols) {
        for (int64_t k = 0; k < ndm * nchans; ++k)
            SPP_REQUIRE(off_host[k] + out_cols <= ncols, "offset %lld + out_cols %lld wraps in a valid-columns transform",
                        static_cast<long long>(off_host[k]), static_cast<long long>(out_cols));
    }
    const int64_t by = spp::ceil_div(ndm, int64_t(DT_D)), bx = spp::ceil_div(out_cols, int64_t(RB_THREADS) * DT_K);
    if (!spp::dmt_in_tiles(ncols, ndm, out_cols)) {
        const int64_t bx1 = spp::ceil_div(out_cols, int64_t(RB_THREADS));
        SPP_REQUIRE(bx1 <= 0x7fffffffLL, "too many columns");
        hipLaunchKernelGGL(k_dmt_rows, dim3(static_cast<unsigned>(bx1), static_cast<unsigned>(ndm)), dim3(RB_THREADS), 0,
                           spp::as_stream(stream), in, nchans, ncols, off, out_cols, out);
        SPP_LAUNCHED("k_dmt_rows");
        return SPP_OK;
    }
    hipLaunchKernelGGL(k_dmt, dim3(static_cast<unsigned>(bx), static_cast<unsigned>(by)), dim3(RB_THREADS), 0,
                       spp::as_stream(stream), in, nchans, static_cast<int32_t>(ncols), off, ndm,
                       static_cast<int32_t>(out_cols), out);
    SPP_LAUNCHED("k_dmt");
    return SPP_OK;
}
