// conv2d in one launch for 3 x 3 windows with any steps: a workgroup brings the part of the input that its output positions look at into
// LDS once and reads every filter tap from there.
//
// The repacking path (conv2d.hip) writes a channels-last copy of the input, and behind its launch boundary the main kernel reads that copy
// once per tap: of the 19.2 us of a layer of 64 x 56 x 56 pixels, 32 images, 128 filters, step 2, the first launch took 8.  Here nothing is
// repacked and no scratch memory is used.  Per block of 32 channels a workgroup
//   - loads its WINDOW, the input rows from the first to the last that its positions need, four pixels of 8 channels to
//     a thread, turns them into four runs of 8 channels in registers and stores these to LDS: [8-channel group][position];
//   - loads its filters' 32 * R * S consecutive values as they lie, stores them to LDS, takes out 8 channels x all taps to a
//     thread, turns them into runs of 8 channels per tap in registers and stores these in the same place: [tap][8-channel group][filter];
//   - multiplies, tap by tap: both operands of a 16x16x32 MFMA are 16 bytes per lane of these layouts.  Positions that a tap moves into
//     the padding read 16 bytes of zeros.
// The loads of the next block are in flight meanwhile.
#include <algorithm>

#include "conv2d.h"
#include "conv2d_store.h"
#include "gemm_fast.h"
#include "tune.h"

namespace nt {
namespace {

constexpr int kWindowBM = 224, kWindowBN = 64, kWindowWaveM = 112, kWindowThreads = 512;
constexpr int kWindowItems = 3;     // (run of four pixels, 8 channels) items per thread
constexpr int kWindowZeros = 256;                                   // bytes at the beginning of LDS, of which 16 are read as zeros

struct ConvWindowParams {
    const void *x, *w;
    void *y;
    int N, C, H, W, K, P, Q, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w;
    int64_t xs0, xs1, ws0;  // element strides of the input's image and channel and of the filter's output channel
    int dense_out;
    int64_t ys[4];
    int M;
    float one_by_pq, one_by_q, one_by_runs;  // for quick_quotient
    unsigned x_bytes, w_bytes;
    int window;  // positions of the largest window
    int plane;   // bytes of an 8-channel group of the window in LDS
};

// Tiles of 224 positions x 64 filters on eight waves of 112 x 32: two groups of four waves take turns with the taps and add up at the end.
// What bounds it where the chip holds all tiles at once: a chain per block of channels -- the loads' way from memory, the filters' twice
// through LDS, nine taps -- in which MFMAs are busy 15 % of the time, vector instructions 43 %, LDS 33 % (3 us a block of 32 channels, and 6 for the launch, the first loads and the output).  So: large tiles,
// that few workgroups load the same filters (112 positions 15 us where these take 13), 64 filters rather than 128, whose values would take twice as long
// through LDS (14), loads dealt out between the taps (all at once they held up the first tap by 1.2 us), quotients by reciprocals before the first loads
// (0.8 us).  Exchanging the filters' pieces inside quads of lanes instead of LDS costs more vector instructions than it saves (18 us).
// 32 images of 64 x 56 x 56, 128 filters, step 2, alone: 20.2 -> 13.2 us (among others 19.2 -> 12.1); 64 filters, step 1: 28.5 -> 21; 32 of 128 x 28 x 28, 128 filters: 22.8 -> 17.7;
// 8 of 64 x 112 x 112, 128 filters, step 2: 18.5 -> 12.6.
template <typename T, int R, int S>
__global__ __launch_bounds__(kWindowThreads, 2) void conv2d_window_kernel(ConvWindowParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef Elem<T> E;
    typedef typename E::vec8 vec8;
    typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
    typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
    constexpr int kTaps = R * S, BN = kWindowBN, kWaveN = 32, TM = kWindowWaveM / 16, TN = 2;
    constexpr unsigned kBehind = 0x80000000u;  // an offset behind every descriptor: reads zeros
    extern __shared__ __attribute__((aligned(1024))) unsigned char memory[];
    NT_LDS unsigned char *lds = (NT_LDS unsigned char *)memory;
    NT_LDS unsigned char *filters = lds + kWindowZeros + 4 * p.plane;

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int group = wave >> 2, wave_m = (wave >> 1) & 1, wave_n = wave & 1;
    const int i16 = lane & 15, kg = lane >> 4;
    const int m0 = blockIdx.x * kWindowBM, n0 = blockIdx.y * BN;
    const int PQ = p.P * p.Q, HW = p.H * p.W;

    // the filters' loads first: their addresses are at hand
    __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.w, 0, p.w_bytes, 0x00020000);
    // four threads to a filter: pieces f_group, f_group + 4, ... of its values on the way in, 8-channel group f_group on the way out
    const int f_row = t >> 2, f_group = t & 3;
    const unsigned w_src = (unsigned)(((int64_t)min(n0 + f_row, p.K - 1) * p.ws0 + f_group * 8) * 2);
    uint4_t w_regs[kTaps];
    const auto load_filters = [&](int i, int c0) {
        // (C % 8 == 0: what belongs to channels that are not there is whole pieces)
        const unsigned src = c0 + 32 <= p.C || (i * 4 + f_group) * 8 < (p.C - c0) * kTaps ? w_src : kBehind;
        w_regs[i] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, src + i * 64, c0 * kTaps * 2, 0));
    };
    const bool has_filter = wave < 4;
    if (has_filter) {
#pragma unroll
        for (int i = 0; i < kTaps; ++i) load_filters(i, 0);
    }

    // ---- the window: from row `top` of image0 to row `bottom` of image1 ----
    const int m_last = min(m0 + kWindowBM, p.M) - 1;
    const int image0 = quick_quotient(m0, PQ, p.one_by_pq), image1 = quick_quotient(m_last, PQ, p.one_by_pq);
    const int top = min(max(quick_quotient(m0 - image0 * PQ, p.Q, p.one_by_q) * p.stride_h - p.pad_h, 0), p.H - 1);
    const int bottom = min(quick_quotient(m_last - image1 * PQ, p.Q, p.one_by_q) * p.stride_h - p.pad_h + (R - 1) * p.dil_h, p.H - 1);
    const int first = image0 * HW + top * p.W;  // the window's first position, counted over all images
    // runs of four positions: of the first image, of each image between, of the last
    const int length0 = ((image1 > image0 ? p.H : bottom + 1) - top) * p.W, runs0 = (length0 + 3) / 4;
    const int runs_whole = (HW + 3) / 4, length1 = (bottom + 1) * p.W;
    const int runs = image1 > image0 ? runs0 + (image1 - image0 - 1) * runs_whole + (length1 + 3) / 4 : runs0;

    __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, p.x_bytes, 0x00020000);
    // this thread's items; one that is none loads zeros and stores nothing
    unsigned x_src[kWindowItems];
    int x_dst[kWindowItems];  // and, in the lowest bits, which group of 8 channels
#pragma unroll
    for (int i = 0; i < kWindowItems; ++i) {
        const int id = i * kWindowThreads + t;
        const int chunk = (id >= runs) + (id >= 2 * runs) + (id >= 3 * runs) + (id >= 4 * runs), run = id - chunk * runs;
        int image = image0, start;
        if (run < runs0) {
            start = top * p.W + min(4 * run, length0 - 4);  // (where the length is no multiple of four the last run begins earlier)
        } else {
            const int rest = run - runs0, skip = quick_quotient(rest, runs_whole, p.one_by_runs);
            image = image0 + 1 + skip;
            start = min(4 * (rest - skip * runs_whole), (image == image1 ? length1 : HW) - 4);
        }
        const int position = image * HW + start - first;
        const bool live = chunk < 4 && position + 4 <= p.window;
        x_src[i] = live ? (unsigned)((image * p.xs0 + (int64_t)chunk * 8 * p.xs1 + start) * 2) : kBehind;
        x_dst[i] = live ? (kWindowZeros + chunk * p.plane + position * 16) | chunk : -1;
    }
    // filters of a group are permuted in fours so that neither the four groups that a wave stores together nor the two that a
    // read of fragments serves together meet in a bank: group 0, 1, 2, 3 by 0, 3, 1, 2
    const auto permuted = [](int filter, int channels) { return filter ^ (((channels >> 1) + (channels & 1) * (3 - (channels >> 1) * 2)) << 2); };
    NT_LDS unsigned char *filter_dst = filters + (f_group * BN + permuted(f_row, f_group)) * 16;

    uint2_t x_regs[kWindowItems][8];
    const auto load_window = [&](int i, int c0) {
        if (i * kWindowThreads >= runs * 4) return;  // (uniform)
        const unsigned src = c0 + (x_dst[i] & 3) * 8 < p.C ? x_src[i] : kBehind;
#pragma unroll
        for (int j = 0; j < 8; ++j) x_regs[i][j] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(x_rsrc, src, (int)((c0 + j) * p.xs1 * 2), 0));
    };
#pragma unroll
    for (int i = 0; i < kWindowItems; ++i) load_window(i, 0);
    NT_LDS unsigned char *raw_in = filters + f_row * (kTaps * 64) + f_group * 16;
    NT_LDS unsigned char *raw_out = filters + f_row * (kTaps * 64) + f_group * (kTaps * 16);
    const auto stage_block = [&]() {
        if (has_filter) {
#pragma unroll
            for (int i = 0; i < kTaps; ++i) *(NT_LDS uint4_t *)(raw_in + i * 64) = w_regs[i];
        }
#pragma unroll
        for (int i = 0; i < kWindowItems; ++i) {
            if (x_dst[i] < 0) continue;
            NT_LDS unsigned char *to = lds + (x_dst[i] & ~15);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
            uint4_t even, odd;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                even[d] = __builtin_amdgcn_perm(x_regs[i][2 * d + 1][h], x_regs[i][2 * d][h], 0x05040100u);
                odd[d] = __builtin_amdgcn_perm(x_regs[i][2 * d + 1][h], x_regs[i][2 * d][h], 0x07060302u);
            }
            const bool flip = lane & 4;
            const uint4_t f0 = flip ? odd : even, f1 = flip ? even : odd;
            *(NT_LDS uint4_t *)(to + h * 32 + (flip ? 16 : 0)) = f0;
            *(NT_LDS uint4_t *)(to + h * 32 + (flip ? 0 : 16)) = f1;
            }
        }
        lds_barrier();
        unsigned values[kTaps * 4];
        if (has_filter) {
#pragma unroll
            for (int i = 0; i < kTaps; ++i) {
            const uint4_t v = *(const NT_LDS uint4_t *)(raw_out + i * 16);
#pragma unroll
            for (int d = 0; d < 4; ++d) values[i * 4 + d] = v[d];
            }
        }
        lds_barrier();  // (every wave has its values: their places are taken by the new layout)
        if (has_filter) static_for<0, kTaps>([&](auto tap_tag) {
            constexpr int tap = decltype(tap_tag)::value;
            uint4_t v;
            static_for<0, 4>([&](auto d_tag) {
                constexpr int d = decltype(d_tag)::value;
                constexpr int lo = 2 * d * kTaps + tap, hi = lo + kTaps;  // element numbers of channels 2 d and 2 d + 1
                constexpr unsigned selector = (lo & 1 ? 0x0302u : 0x0100u) | (hi & 1 ? 0x07060000u : 0x05040000u);
                v[d] = __builtin_amdgcn_perm(values[hi / 2], values[lo / 2], selector);
            });
            *(NT_LDS uint4_t *)(filter_dst + tap * (4 * BN * 16)) = v;
        });
    };

    // ---- operands of the MFMAs ----
    int a_addr[TM];
    unsigned a_taps[TM];  // the taps that stay inside the image
#pragma unroll
    for (int ti = 0; ti < TM; ++ti) {
        const int m = m0 + wave_m * kWindowWaveM + ti * 16 + i16;
        const int image = quick_quotient(m, PQ, p.one_by_pq), pq = m - image * PQ;
        const int oy = quick_quotient(pq, p.Q, p.one_by_q), y = oy * p.stride_h - p.pad_h, x = (pq - oy * p.Q) * p.stride_w - p.pad_w;
        a_addr[ti] = kWindowZeros + kg * p.plane + (image * HW + y * p.W + x - first) * 16;
        unsigned rows = 0, taps = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) rows |= (unsigned)(x + s * p.dil_w) < (unsigned)p.W ? 1u << s : 0u;
#pragma unroll
        for (int r = 0; r < R; ++r) taps |= m < p.M && (unsigned)(y + r * p.dil_h) < (unsigned)p.H ? rows << (r * S) : 0u;
        a_taps[ti] = taps;
    }
    const NT_LDS unsigned char *b_src = filters + (kg * BN + wave_n * kWaveN + permuted(i16, kg)) * 16;
    float4_t acc[TM][TN];
#pragma unroll
    for (int ti = 0; ti < TM; ++ti)
#pragma unroll
        for (int tj = 0; tj < TN; ++tj) acc[ti][tj] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // taps first, first + 2, ...  (the other group's wave on the SIMD covers the reads: fragments of a second tap would not fit the registers),
    // and between them the loads of the block of channels at `next`, if there is one: all at once they would hold up the first tap
    const auto multiply = [&](int first, int next) {
        static_for<0, (kTaps + 1) / 2>([&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value, kSteps = (kTaps + 1) / 2;
            const int tap = first + 2 * i;
            if (2 * i + 1 < kTaps || first == 0) {
                const int r = tap / S, s = tap - r * S;
                const int shift = (r * p.dil_h * p.W + s * p.dil_w) * 16;
                const NT_LDS unsigned char *b = b_src + tap * (4 * BN * 16);
                vec8 as[TM], bs[TN];
#pragma unroll
                for (int tj = 0; tj < TN; ++tj) bs[tj] = *(const NT_LDS vec8 *)(b + tj * 256);
#pragma unroll
                for (int ti = 0; ti < TM; ++ti) as[ti] = *(const NT_LDS vec8 *)(lds + ((a_addr[ti] + shift) & __builtin_amdgcn_sbfe((int)a_taps[ti], tap, 1)));
#pragma unroll
                for (int ti = 0; ti < TM; ++ti)
#pragma unroll
                    for (int tj = 0; tj < TN; ++tj) acc[ti][tj] = E::mfma16(as[ti], bs[tj], acc[ti][tj]);
            }
            if (next < p.C) {
                if (has_filter) static_for<i * kTaps / kSteps, (i + 1) * kTaps / kSteps>([&](auto j) { load_filters(decltype(j)::value, next); });
                static_for<i * kWindowItems / kSteps, (i + 1) * kWindowItems / kSteps>([&](auto j) { load_window(decltype(j)::value, next); });
            }
        });
    };

    if (t < kWindowZeros / 16) *(NT_LDS uint4_t *)(lds + t * 16) = uint4_t{0, 0, 0, 0};
    int turn = group;  // which group takes the even taps changes from block to block: an odd number of taps is dealt out evenly
    for (int c0 = 0; c0 < p.C; c0 += 32) {
        if (c0 > 0) lds_barrier();  // (the block before has been multiplied)
        stage_block();
        lds_barrier();
#pragma unroll
        for (int ti = 0; ti < TM; ++ti) asm volatile("" : "+v"(a_addr[ti]));  // (the taps' addresses are worked out where they are used: 36 of them would not fit the registers)
        multiply(turn, c0 + 32);
        turn ^= 1;
    }
    lds_barrier();

    // ---- the groups add up: each keeps half of its filters' accumulators and hands the other half over ----
    NT_LDS float4_t *mine = (NT_LDS float4_t *)lds + wave * (TM * 64) + lane, *theirs = (NT_LDS float4_t *)lds + (wave ^ 4) * (TM * 64) + lane;
    float4_t sum[TM][1];
#pragma unroll
    for (int ti = 0; ti < TM; ++ti) {
        mine[ti * 64] = group == 0 ? acc[ti][1] : acc[ti][0];
        sum[ti][0] = group == 0 ? acc[ti][0] : acc[ti][1];
    }
    lds_barrier();
#pragma unroll
    for (int ti = 0; ti < TM; ++ti) sum[ti][0] += theirs[ti * 64];
    lds_barrier();
    store_conv_tile<T, TM, 1, 1>(p, sum, lds + wave * 4096, m0 + wave_m * kWindowWaveM, n0 + wave_n * kWaveN + group * 16, lane);
#endif
}

// bytes from the first to the last element that the kernel reads
int64_t x_extent(const Conv2dRequest &q) { return ((int64_t)(q.N - 1) * q.xs[0] + (int64_t)(q.C - 1) * q.xs[1] + (int64_t)q.H * q.W) * 2; }
int64_t w_extent(const Conv2dRequest &q) { return ((int64_t)(q.K - 1) * q.ws[0] + (int64_t)q.C * q.R * q.S) * 2; }

// The positions of the largest window, 0 when the kernel does not take the problem.
int window_positions(const Conv2dRequest &q) {
    if (q.R != 3 || q.S != 3 || q.C % 8 || q.C < 32) return 0;
    if (q.xs[3] != 1 || q.xs[2] != q.W || q.W < 4 || q.xs[0] < 0 || q.xs[1] < 0) return 0;  // the pixels of a channel lie one after another
    if (q.ws[3] != 1 || q.ws[2] != q.S || q.ws[1] != (int64_t)q.R * q.S || q.ws[0] < 0) return 0;
    if (x_extent(q) >= (int64_t(1) << 31) || w_extent(q) >= (int64_t(1) << 31)) return 0;  // 32-bit buffer offsets
    if ((int64_t)q.N * q.H * q.W > 0x3fffffffll || (int64_t)q.N * q.P * q.Q > 0x3fffffffll) return 0;
    if (q.N > 1 << 20 || q.P > 1 << 20) return 0;  // (quick_quotient)
    // Every output row looks at the image at its top or below it, and at its bottom or above it, so that the first and the last row of a
    // window are those of its first and its last position, but for what lies in the padding.
    if (q.pad_h > (q.R - 1) * q.dil_h || (int64_t)(q.P - 1) * q.stride_h - q.pad_h > q.H - 1) return 0;
    const int PQ = q.P * q.Q;
    // the most rows that a tile of positions looks at: output rows of an image are stride_h input rows apart, the first of an image and the
    // last of the one before it H - P * stride_h more
    const int64_t images = std::min<int64_t>(q.N, (kWindowBM - 2) / PQ + 2), out_rows = std::min<int64_t>((kWindowBM + q.Q - 2) / q.Q + 1, (int64_t)q.N * q.P);
    const int64_t rows = std::min<int64_t>(images * q.H, (out_rows - 1) * q.stride_h + (images - 1) * std::max(0, q.H - q.P * q.stride_h) + (q.R - 1) * q.dil_h + 1);
    const int64_t window = rows * q.W;
    if (((window + 3 * images) / 4 + 1) * 4 > kWindowItems * kWindowThreads) return 0;
    return (int)window;
}

// Whether this kernel is expected to be faster than the repacking path, in microseconds, by both models fitted to 320 convolutions (1 to
// 32 images of 7 x 7 to 112 x 112, 32 to 256 channels, 16 to 512 filters, steps 1 and 2; 8 and 6 % off on average): it wins where its
// workgroups fill the chip about once -- fewer leave CUs idle that the other path's parts of the contraction use, more pay the long block.  Of
// the 320 the 44 it is taken for run in 0.84 of the other paths' time on average, 1.03 at worst.  With steps of 2 and more a block takes longer the fuller the chip is, and
// the data hardly counts beside it (379 others of up to 512 channels, steps 1 to 3): without the second estimate the longer contractions of such layers were taken too (us, repacked /
// here: 14 images of 240 x 112 x 115, 264 filters 139 / 168; 9 of 328 x 56 x 59, 352 44 / 53).  With it the 93 of 260 drawn ones that are taken run in 0.83 of the
// other path's time, three of them in more than 1.04 (480 channels of 112 x 115, 208 filters, step 2 65.3 / 75.5), two of 103 that were taken before in more than 1.02.
bool window_pays(const Conv2dRequest &q) {
    const int units = std::max(1, compute_units());
    const int64_t positions = (int64_t)q.N * q.P * q.Q, workgroups = (positions + kWindowBM - 1) / kWindowBM * ceil_div(q.K, kWindowBN);
    const float rounds = (float)((workgroups + units - 1) / units), blocks = (float)ceil_div(q.C, 32);
    const float megabytes = ((float)q.N * q.C * q.H * q.W + (float)positions * q.K + (float)q.K * q.C * q.R * q.S) * 2e-6f;
    const bool scattered = conv2d_dense_output(q) == 0 || (conv2d_dense_output(q) == 1 && q.P * q.Q % 8 != 0);
    float time = 2.8f + rounds * (2.2f + 2.85f * blocks + (scattered ? 5.3f : 0.0f)) + 0.153f * megabytes;
    if (q.stride_h > 1 || q.stride_w > 1)
        time = std::max(time, 2.7f + rounds * (2.1f + 3.39f * blocks + (scattered ? 3.9f : 0.0f)) + 0.47f * blocks * (float)workgroups / (float)units + 0.063f * megabytes);
    return time < 0.95f * conv2d_repacked_time(q);
}

template <typename T>
int run_window(const Conv2dRequest &q, int window, hipStream_t stream) {
    const int M = q.N * q.P * q.Q, PQ = q.P * q.Q;
    ConvWindowParams p;
    p.x = q.x; p.w = q.w; p.y = q.y;
    p.N = q.N; p.C = q.C; p.H = q.H; p.W = q.W; p.K = q.K; p.P = q.P; p.Q = q.Q;
    p.pad_h = q.pad_h; p.pad_w = q.pad_w; p.stride_h = q.stride_h; p.stride_w = q.stride_w; p.dil_h = q.dil_h; p.dil_w = q.dil_w;
    p.xs0 = q.xs[0]; p.xs1 = q.xs[1]; p.ws0 = q.ws[0];
    p.dense_out = conv2d_dense_output(q);
    for (int d = 0; d < 4; ++d) p.ys[d] = q.ys[d];
    p.M = M;
    p.one_by_pq = 1.0f / (float)PQ;
    p.one_by_q = 1.0f / (float)q.Q;
    p.one_by_runs = 1.0f / (float)((q.H * q.W + 3) / 4);
    p.x_bytes = (unsigned)x_extent(q);
    p.w_bytes = (unsigned)w_extent(q);
    p.window = window;
    // the rows that a read of fragments serves together are four positions of one group and four of the next: a step of 1 fills 16-byte slots one
    // after another in both, a step of 2 every other slot, so that the next group is moved by one
    p.plane = (window * 16 + 255) / 256 * 256 + (q.stride_w % 2 == 0 ? 16 : 0);
    // (the sums that the groups exchange take the same place, 7 KiB a wave)
    constexpr int kMostBytes = kWindowZeros + 4 * (kWindowItems * kWindowThreads * 16 + 16) + 9 * 4 * kWindowBN * 16;
    static_assert(kMostBytes <= 160 * 1024, "the largest window and its filters in LDS (132.3 KiB)");
    const size_t bytes = std::max(kWindowZeros + 4 * (size_t)p.plane + (size_t)q.R * q.S * 4 * kWindowBN * 16, (size_t)(kWindowThreads / 64) * (kWindowWaveM / 16) * 1024);
    const dim3 grid((unsigned)ceil_div(M, kWindowBM), (unsigned)ceil_div(q.K, kWindowBN));
    if (grid.y > 65535) return NINETOOTHED_NO_KERNEL;
    note_launch(kLaunchConv2d, kConvWindow, "conv2d_window_kernel, one launch, input windows in LDS");
    conv2d_window_kernel<T, 3, 3><<<grid, dim3(kWindowThreads), bytes, stream>>>(p);
    return (int)hipGetLastError();
}

}  // namespace

int conv2d_window(const Conv2dRequest &q, hipStream_t stream, bool if_it_pays) {
    if (q.dtype != NINETOOTHED_FLOAT16 && q.dtype != NINETOOTHED_BFLOAT16) return NINETOOTHED_NO_KERNEL;
    // (what the kernel takes comes first: the expected times go through all tiles and numbers of parts of the other path)
    const int window = window_positions(q);
    if (window == 0 || (if_it_pays && !window_pays(q))) return NINETOOTHED_NO_KERNEL;
    return q.dtype == NINETOOTHED_FLOAT16 ? run_window<half_t>(q, window, stream) : run_window<bf16_t>(q, window, stream);
}

}  // namespace nt
