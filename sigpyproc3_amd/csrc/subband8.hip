// Subbands of an 8-bit gulp (kernels.subband, core/kernels.py:379-401) with whole bands per
// block: out[t * nsubs + band] = sum over the band's channels of in[t + d_c][c].
//
// The byte-staged kernel (k_gulp_int) combines channel groups with float atomics, one per
// (output, band), and runs at the rate the L2 takes those: 2e10 per second. Here a block owns
// SB_T outputs and every band whose first channel lies in its channel range, so each output is
// one plain store. That needs bands of consecutive channels (a map that only rises or only falls): a
// block reads the whole map once to find out, and keeps the atomics for any other map and
// for the bands that are too wide for one block.
//
// A stage takes SB_Q groups of 16 channels: SB_Q lanes read 16 bytes each of one row, side by
// side. A lane loads 4 rows, transposes them in registers (v_perm), and writes 4 consecutive
// samples of a channel per dword into that channel's series in LDS. Row blocks are common to the
// stage, so that a row's line is read by all lanes that need it at once, but a channel keeps only
// the blocks of its own SB_T outputs (the others go to a spare dword), so that a series has the
// same length whatever the delays. Summing, a thread owns 4 consecutive outputs: per
// channel two series dwords, a funnel shift, and adds of packed 16-bit lanes (the odd bytes by
// v_perm; the even ones as the raw 32-bit sum minus 256 times the odd sum).
//
// Measured on 1024 channels x 131072 samples, 64 bands, maximum delay 5077 (166 MB in and out):
// a whole call 407 -> 69 us, 7 of them zeroing the output. The loads alone take 48, the sums about 25
// (a block has two stages, so half of them overlap no load) and the stores 8. Narrower stages (32
// channels, four blocks per CU) ran 87 when this form ran 78, 2048 outputs per block 105. (The map
// is looked through by shuffles: LDS atomics on one address took 4 us more per block.)
#include "spp_subband8.hpp"

#include "spp_common.hpp"

#include <algorithm>
#include <climits>

namespace {

constexpr int SB_THREADS = 256;
constexpr int SB_T = 4 * SB_THREADS;       // outputs per block, 4 per thread
constexpr int SB_Q = 4;                    // 16-channel groups per stage
constexpr int SB_CH = 16 * SB_Q;           // channels per stage
constexpr int SB_NRB = SB_T / 4 + 1;       // series dwords of a channel: its outputs' and the funnel's upper one
constexpr int SB_PITCH = SB_NRB + 2;       // a spare dword, and odd: the groups a wave writes fall 16 banks apart
constexpr int SB_UNITS = 6;                // units of the next stage each thread loads ahead
// Word 3 of a raw buffer resource on gfx9-family GPUs: 32-bit data format, no swizzle.
constexpr int kBufferFlags = 0x00020000;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Bytes 1 and 3 of x into the low bytes of its two 16-bit lanes.
__device__ __forceinline__ uint32_t odd_bytes(uint32_t x) { return __builtin_amdgcn_perm(x, x, 0x0c030c01u); }

// 4x4 byte transpose: byte c of word r moves to byte r of word c.
__device__ __forceinline__ void transpose4(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    const uint32_t ab_lo = __builtin_amdgcn_perm(b, a, 0x05010400u);  // a0 b0 a1 b1
    const uint32_t ab_hi = __builtin_amdgcn_perm(b, a, 0x07030602u);  // a2 b2 a3 b3
    const uint32_t cd_lo = __builtin_amdgcn_perm(d, c, 0x05010400u);
    const uint32_t cd_hi = __builtin_amdgcn_perm(d, c, 0x07030602u);
    a = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100u);
    b = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302u);
    c = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100u);
    d = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302u);
}

__global__ __launch_bounds__(SB_THREADS) void k_subband8(const uint8_t* __restrict__ in,
                                                         const int32_t* __restrict__ delays,
                                                         const int32_t* __restrict__ chan_to_sub,
                                                         float* __restrict__ out, int64_t nchans, int64_t nsamps,
                                                         int64_t nout, int64_t nsubs, int64_t out_size,
                                                         int64_t chans_per_group, int64_t ngroups,
                                                         int64_t nblocks, int widest) {
    __shared__ uint32_t series[SB_CH * SB_PITCH];
    __shared__ int32_t sdel[2][SB_CH], ssub[2][SB_CH], sshift[2][SB_CH];
    __shared__ int32_t gmin[2][SB_Q], gmax[2][SB_Q];
    __shared__ int4 bound[SB_THREADS / 64];  // per wave: band starts about the block's range
    __shared__ int32_t order[SB_THREADS / 64];
    // consecutive blocks on one XCD: the channel groups of one time tile share row lines in its L2
    const int64_t logical = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    if (logical >= nblocks) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    static_assert(SB_CH == 64, "lane k of a wave holds channel k's band and shift");
    const int64_t t0 = (logical / ngroups) * SB_T;
    const int64_t cb = (logical % ngroups) * chans_per_group;
    const int64_t ce = min(nchans, cb + chans_per_group);

    // Bands of consecutive channels (a non-decreasing or non-increasing map)? Then this block's
    // channels are the bands that start in [cb, ce), to their ends. A band of more than `widest`
    // channels is not one block's chain of stages: the blocks whose ranges it covers each add
    // their part of it. 1024 channels x 131072, one band of 961 among 63 of one channel: 197 us in
    // one block, 175 shared; 4096 x 16384, one of 3969 among 127: 463 and 90.
    bool valid = true, up = true, down = true;
    int start_cb = 0, after_cb = static_cast<int>(nchans);  // band starts: last up to cb, first past it
    int start_ce = 0, after_ce = static_cast<int>(nchans);  // and about ce
    for (int64_t c4 = tid; c4 < nchans; c4 += 4 * SB_THREADS) {
        int s[4], prev[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t c = min(c4 + j * SB_THREADS, nchans - 1);
            s[j] = chan_to_sub[c];
            prev[j] = chan_to_sub[max<int64_t>(c - 1, int64_t(0))];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = static_cast<int>(min(c4 + j * SB_THREADS, nchans - 1));
            valid = valid && s[j] >= 0 && s[j] < nsubs;
            up = up && s[j] >= prev[j];
            down = down && s[j] <= prev[j];
            if (s[j] != prev[j]) {
                if (c <= cb) start_cb = max(start_cb, c);
                else after_cb = min(after_cb, c);
                if (c <= ce) start_ce = max(start_ce, c);
                else after_ce = min(after_ce, c);
            }
        }
    }
    up = __all(valid && up);
    down = __all(valid && down);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        start_cb = max(start_cb, __shfl_xor(start_cb, o));
        after_cb = min(after_cb, __shfl_xor(after_cb, o));
        start_ce = max(start_ce, __shfl_xor(start_ce, o));
        after_ce = min(after_ce, __shfl_xor(after_ce, o));
    }
    if (lane == 0) {
        bound[tid >> 6] = make_int4(start_cb, after_cb, start_ce, after_ce);
        order[tid >> 6] = (up ? 1 : 0) | (down ? 2 : 0);
    }
    __syncthreads();
    int4 bd = bound[0];
    int ord = order[0];
#pragma unroll
    for (int w = 1; w < SB_THREADS / 64; ++w) {
        const int4 b = bound[w];
        bd = make_int4(max(bd.x, b.x), min(bd.y, b.y), max(bd.z, b.z), min(bd.w, b.w));
        ord &= order[w];
    }
    const bool sorted = __builtin_amdgcn_readfirstlane(ord) != 0;
    const int head0 = __builtin_amdgcn_readfirstlane(bd.x), head1 = __builtin_amdgcn_readfirstlane(bd.y);
    const int tail0 = __builtin_amdgcn_readfirstlane(bd.z), tail1 = __builtin_amdgcn_readfirstlane(bd.w);
    const bool head = sorted && head0 < cb;                // the block's first channel is in a band before it,
    const bool tail = sorted && ce < nchans && tail0 < ce;  // its last one in a band that goes on
    bool shared_head = head && head1 - head0 > widest;
    const bool shared_tail = tail && tail1 - tail0 > widest;
    const int64_t lo = head && !shared_head ? head1 : cb;
    const int64_t hi = tail && !shared_tail ? tail1 : ce;
    if (lo >= ce) return;  // one band of another block

    uint32_t raw = 0, odd = 0, wide[4] = {0, 0, 0, 0};
    int packed = 0;  // channels in the 16-bit lanes
    const int64_t ta = t0 + 4 * tid;
    auto widen = [&]() {
        const uint32_t even = raw - (odd << 8);
        wide[0] += even & 0xffffu;
        wide[1] += odd & 0xffffu;
        wide[2] += even >> 16;
        wide[3] += odd >> 16;
        raw = odd = 0;
        packed = 0;
    };
    // Finished bands wait until four consecutive ones make one 16-byte store per output (a
    // store per band and output costs a quarter of the whole at 128 bands).
    typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
    float* __restrict__ orow = out + ta * nsubs;
    const int nvalid = static_cast<int>(max<int64_t>(0, min<int64_t>(4, nout - ta)));
    const int64_t room = out_size - ta * nsubs;  // floats from orow on that may be written
    f32x4_any held[4];                           // [output][band]
    int nheld = 0, held0 = 0;
    bool held_whole = sorted;  // the held bands are this block's alone: plain stores
    auto drain = [&]() {
        if (nheld == 4 && held_whole && room >= 3 * nsubs + held0 + 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j < nvalid) *reinterpret_cast<f32x4_any*>(orow + j * nsubs + held0) = held[j];
        } else {
#pragma unroll 1
            for (int b = 0; b < nheld; ++b) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int64_t i = j * nsubs + held0 + b;
                    if (j < nvalid && i < room) {
                        const float v = b == 0 ? held[j][0] : b == 1 ? held[j][1] : b == 2 ? held[j][2] : held[j][3];
                        if (held_whole) orow[i] = v;
                        else atomicAdd(orow + i, v);
                    }
                }
            }
        }
        nheld = 0;
    };
    auto flush = [&](int band, bool whole) {
        widen();
        if (band >= 0) {
            if (nheld == 4 || (nheld > 0 && (band != held0 + nheld || whole != held_whole))) drain();
            if (nheld == 0) {
                held0 = band;
                held_whole = whole;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = static_cast<float>(wide[j]);
                held[j][0] = nheld == 0 ? v : held[j][0];
                held[j][1] = nheld == 1 ? v : held[j][1];
                held[j][2] = nheld == 2 ? v : held[j][2];
                held[j][3] = nheld == 3 ? v : held[j][3];
            }
            ++nheld;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) wide[j] = 0;
    };

    // Tables of the stage at channel c (double-buffered: a stage's are written while the one
    // before is still summed), from the delay d and band s of channel c + tid (tid < SB_CH).
    auto load_tables = [&](int64_t c, int& d, int& s) {
        if (tid < SB_CH) {
            const int64_t ch = min(c + tid, nchans - 1);
            d = delays[ch];
            s = chan_to_sub[ch];
        }
    };
    auto write_tables = [&](int p, int d, int s) {
        if (tid < SB_CH) {
            sdel[p][tid] = d;
            sshift[p][tid] = 8 * (d & 3);
            ssub[p][tid] = s;
            int mn = d, mx = d;  // over the 16 lanes of the group
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                mn = min(mn, __shfl_xor(mn, o));
                mx = max(mx, __shfl_xor(mx, o));
            }
            if ((tid & 15) == 0) {
                gmin[p][tid >> 4] = mn;
                gmax[p][tid >> 4] = mx;
            }
        }
    };
    // Staging geometry: unit (group q, row block b) is rows t0 + dmin + 4 b + k of the lane's 16
    // channels; channel k's series starts at row block ((d_k & ~3) - dmin) / 4.
    const int q = tid & (SB_Q - 1);
    constexpr int BSTEP = SB_THREADS / SB_Q;
    int64_t rbase = 0, cq = 0;
    int dmin = 0, b0 = 0, b1 = 0, nb = 0;
    bool inside = false, fast = false;
    auto set_geometry = [&](int64_t c, int p) {
        dmin = gmin[p][0];
        int dmax = gmax[p][0];
#pragma unroll
        for (int i = 1; i < SB_Q; ++i) {
            dmin = min(dmin, gmin[p][i]);
            dmax = max(dmax, gmax[p][i]);
        }
        dmin = __builtin_amdgcn_readfirstlane(dmin & ~3);
        dmax = __builtin_amdgcn_readfirstlane(dmax);
        b0 = (gmin[p][q] - dmin) >> 2;
        b1 = ((gmax[p][q] - dmin) >> 2) + SB_NRB;
        nb = ((dmax - dmin) >> 2) + SB_NRB;
        rbase = t0 + dmin;
        cq = c + 16 * q;
        // 16-byte loads of whole groups; a stage at the end of rows of a partial group, or with
        // rows outside the gulp, goes dword by dword
        inside = rbase >= 0 && rbase + int64_t(4) * nb <= nsamps && (int64_t(4) * nb) * nchans < (int64_t(1) << 31);
        fast = inside && (nchans - c >= SB_CH || (nchans - c) % 16 == 0);
    };
    auto load_fast = [&](int b, u32x4 (&w)[4]) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(in) + rbase * nchans, 0, static_cast<int>(int64_t(4) * nb * nchans), kBufferFlags);
        // units no channel of the group keeps read past the buffer's end (0, no traffic)
        uint32_t off = b >= b0 && b < b1 && cq < nchans
                           ? static_cast<uint32_t>(4 * b) * static_cast<uint32_t>(nchans) + static_cast<uint32_t>(cq)
                           : 0x80000000u;
        asm volatile("" : "+v"(off));  // a select, not a branch round the loads
#pragma unroll
        for (int k = 0; k < 4; ++k)
            w[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, k * static_cast<int>(nchans), 0));
    };
    auto load_slow = [&](int b, u32x4 (&w)[4]) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int64_t row = rbase + 4 * b + k;
            if (row < 0) row += nsamps;  // numba wraparound of a negative index
            w[k] = u32x4{0, 0, 0, 0};
            if (row < 0 || row >= nsamps) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (cq + 4 * i < nchans)  // rows are whole dwords
                    w[k][i] = *reinterpret_cast<const uint32_t*>(in + row * nchans + cq + 4 * i);
        }
    };

    u32x4 ahead[SB_UNITS][4];  // the next stage's first units, loading while this one is summed
    auto load_ahead = [&]() {
        if (!fast) return;
#pragma unroll
        for (int i = 0; i < SB_UNITS; ++i) load_fast(tid / SB_Q + i * BSTEP, ahead[i]);
    };
    int64_t c = lo & ~int64_t(15);
    int dn = 0, sn = 0;
    load_tables(c, dn, sn);
    write_tables(0, dn, sn);
    load_tables(c + SB_CH, dn, sn);
    __syncthreads();
    if (c < hi) {
        set_geometry(c, 0);
        load_ahead();
    }
    for (int p = 0; c < hi; c += SB_CH, p ^= 1) {
        {
            int bk[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) bk[i] = (sdel[p][16 * q + i] - dmin) >> 2;
            uint32_t* __restrict__ dst = series + 16 * q * SB_PITCH;
            auto store_unit = [&](int b, u32x4 (&w)[4]) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint32_t x[4] = {w[0][i], w[1][i], w[2][i], w[3][i]};
                    transpose4(x[0], x[1], x[2], x[3]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int k = 4 * i + j;
                        dst[k * SB_PITCH + min(static_cast<uint32_t>(b - bk[k]), static_cast<uint32_t>(SB_NRB))] = x[j];
                    }
                }
            };
            if (fast) {
#pragma unroll
                for (int i = 0; i < SB_UNITS; ++i)
                    if (i * BSTEP < nb) store_unit(tid / SB_Q + i * BSTEP, ahead[i]);  // uniform
                for (int b = tid / SB_Q + SB_UNITS * BSTEP; b < nb; b += BSTEP) {
                    load_fast(b, ahead[0]);
                    store_unit(b, ahead[0]);
                }
            } else {
                for (int b = max(b0 - b0 % BSTEP, 0) + tid / SB_Q; b < b1; b += BSTEP) {
                    if (b < b0) continue;
                    load_slow(b, ahead[0]);
                    store_unit(b, ahead[0]);
                }
            }
        }
        write_tables(p ^ 1, dn, sn);
        __syncthreads();
        if (c + SB_CH < hi) {
            load_tables(c + 2 * SB_CH, dn, sn);
            set_geometry(c + SB_CH, p ^ 1);
            load_ahead();
        }
        // Summing, four channels at a time with the next four's dwords being read. Lane k holds
        // channel k's band and funnel shift, so no step waits for a table; bit k of `ends` says
        // that channel k is the last of its band's run.
        const int k0 = static_cast<int>(max<int64_t>(lo - c, int64_t(0)));
        const int k1 = static_cast<int>(min<int64_t>(hi - c, SB_CH));
        const int my_sub = ssub[p][lane], my_shift = sshift[p][lane];
        const int next_sub = lane < 63 ? ssub[p][lane + 1] : ssub[p ^ 1][0];
        const uint64_t ends = __ballot(next_sub != my_sub || c + lane + 1 >= hi);
        const uint32_t* __restrict__ x = series + tid;
        uint32_t dl[4], dh[4];
        auto read4 = [&](int k) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                dl[j] = x[(k + j) * SB_PITCH];
                dh[j] = x[(k + j) * SB_PITCH + 1];
            }
        };
        read4(0);
#pragma unroll 1
        for (int k = 0; k < k1; k += 4) {
            uint32_t v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = __builtin_amdgcn_alignbit(dh[j], dl[j], static_cast<uint32_t>(__builtin_amdgcn_readlane(my_shift, k + j)));
            read4(min(k + 4, SB_CH - 4));
            const uint32_t end4 = static_cast<uint32_t>(ends >> k) & 15u;
            const bool whole = (end4 & 7u) == 0 && k >= k0 && k + 4 <= k1;  // all four in one run
#pragma unroll 1
            for (int j = 0; j < 4; ++j) {
                if (whole) {
                    raw += v[0] + v[1];
                    raw += v[2] + v[3];
                    odd += odd_bytes(v[0]) + odd_bytes(v[1]);
                    odd += odd_bytes(v[2]) + odd_bytes(v[3]);
                    packed += 4;
                    j = 3;
                } else {
                    if (k + j < k0 || k + j >= k1) continue;
                    const uint32_t vj = j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3];
                    raw += vj;
                    odd += odd_bytes(vj);
                    ++packed;
                }
                if ((end4 >> j) & 1u) {
                    flush(__builtin_amdgcn_readlane(my_sub, k + j),
                          sorted && !shared_head && !(shared_tail && c + k + j + 1 >= hi));
                    shared_head = false;
                }
            }
            if (packed > 252) widen();  // 257 samples of 255 fit a 16-bit lane
        }
        __syncthreads();  // this stage's series and tables are no longer read
    }
    drain();
}

}  // namespace

namespace spp {

bool subband8_applies(const void* in, int64_t nchans, int64_t nsamps, int64_t nout, int64_t nsubs) {
    // Rows of whole dwords; exact float sums for the atomics.
    if (nchans % 4 != 0 || reinterpret_cast<uintptr_t>(in) % 4 != 0 || nchans * 255 >= (int64_t(1) << 24)) return false;
    // The byte-staged kernel pays an atomic per output and band (or channel group, of which a short
    // gulp gets more than bands), this one a block's chain of stages per band. Measured, this one
    // against that (us): 64-channel bands 63 / 143 (16 of 1024 channels x 131072), 17-channel 298 /
    // 1334 (128 of 2176 x 174534); 128-channel 116 / 152 (32 of 4096 x 65536) but 110 / 98 with
    // only 8 bands; 512-channel 292 / 112. A map that is not sorted costs both the same atomics.
    const int64_t width = ceil_div(nchans, nsubs);
    if (width > 64 && (width > 128 || nsubs < 32)) return false;
    // A block loads its 16-channel groups' rows over their whole delay spread, however few of them a
    // channel keeps, so the atomics must pay for the spread as well as for a block's latency. Without
    // spread, 8 bands x 32768 outputs: 23 / 12.5 (64 channels), 22.5 / 33 (512 channels, 32 groups);
    // 16 x 32768 25 / 31. With 8192 rows of spread: 8 x 98304 82 / 51, 32 x 98304 97 / 162, 8 x 458752
    // 117 / 236; with 16384: 8 x 131072 (32 channels) 105 / 46, 8 x 491520 119 / 121.
    // With fewer than 8 bands there are few atomics, and the other kernel is slow only where delays
    // spread (64 channels in one band x 524288 19 / 37 at 200 rows, 20 / 15 at none; 128 in two x 131072
    // 18 / 16 at none, 29 / 49 at 1500) or bands are narrow (64 in 4 x 524288 24 / 37, x 131072 20 / 13).
    const int64_t groups = std::min(ceil_div(int64_t(8) * device_cu_count(), ceil_div(nout, int64_t(512))), ceil_div(nchans, int64_t(16)));
    const int64_t spread = (nsamps - nout) * 16 / std::max<int64_t>(nchans, 16);
    if (nsubs < 8)
        return (spread >= 128 && nout * nchans >= 12000000) ||
               (nsubs >= 4 && nchans <= 64 && nout * nsubs >= 700000 + 110 * spread);
    return nout * std::max(nsubs, groups) >= 300000 + 110 * spread;
}

int launch_subband8(const uint8_t* in, const int32_t* delays, const int32_t* chan_to_sub, float* out, int64_t nchans,
                    int64_t nsamps, int64_t nout, int64_t nsubs, int64_t out_size, hipStream_t st) {
    const int64_t bx = ceil_div(nout, int64_t(SB_T));
    const int64_t want = ceil_div(int64_t(8) * device_cu_count(), bx);
    const int64_t most = ceil_div(nchans, int64_t(SB_CH));
    const int64_t cpg = ceil_div(ceil_div(nchans, std::max<int64_t>(1, std::min(want, most))), int64_t(SB_CH)) * SB_CH;
    const int64_t groups = ceil_div(nchans, cpg);
    const int64_t nblocks = bx * groups;
    SPP_REQUIRE(nblocks <= 0x7ffffff0LL, "gulp too long");
    // Few time tiles, or bands, leave CUs idle while one block sums a wide band: 512 channels with a band
    // of 250 x 40000 50 us in one block, 33 shared; four of 200 in 1024 channels 56 and 52, but x 131072
    // 101 and 136; one of 200 in 228 channels and four bands x 262144 110 and 83.
    const int widest = bx <= 40 || nsubs < 8 ? 128 : 256;
    hipLaunchKernelGGL(k_subband8, dim3(static_cast<unsigned>(ceil_div(nblocks, int64_t(8)) * 8)), dim3(SB_THREADS),
                       0, st, in, delays, chan_to_sub, out, nchans, nsamps, nout, nsubs, out_size, cpg, groups,
                       nblocks, widest);
    SPP_LAUNCHED("k_subband8");
    return SPP_OK;
}

}  // namespace spp
