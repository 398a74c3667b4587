// Row softmax for gfx950.  Bandwidth-bound: every element is read once and
// written once; a row (or row segment) lives in registers between the two.
//
// A "segment" is what one program of the arrange-and-apply softmax handles:
// columns [s * block, min((s + 1) * block, N)) of one row.  With block >= N
// (the usual call) a segment is a whole row.
#include "nt_common.h"
#include "tune.h"
#include "workspace.h"

#include <algorithm>
#include <cstdlib>

namespace nt {
namespace {

struct SoftmaxParams {
    const void *in;
    void *out;
    int64_t rows, cols;
    int64_t in_row_stride, in_col_stride, out_row_stride, out_col_stride;
    int64_t block;      // segment length
    int64_t segments;   // per row
};

constexpr float kLog2e = 1.4426950408889634f;

template <bool kIsMax>
NT_DEVICE float combine(float a, float b) {
    return kIsMax ? fmaxf(a, b) : a + b;
}

template <bool kIsMax, int kControl>
NT_DEVICE float combine_dpp(float v) {
    return combine<kIsMax>(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kControl, 0xf, 0xf, true)));
}

// Reduction over aligned groups of kLanes lanes of a wave, the result in every lane: lane permutations inside the vector
// unit (DPP within 16 lanes, then the two half-row swaps), where shuffles would take six dependent trips through LDS.
template <bool kIsMax, int kLanes = 64>
NT_DEVICE float wave_reduce(float v) {
    static_assert(kLanes >= 4, "whole quads");
    v = combine_dpp<kIsMax, 0xb1>(v);                            // quad_perm [1, 0, 3, 2]
    v = combine_dpp<kIsMax, 0x4e>(v);                            // quad_perm [2, 3, 0, 1]
    if constexpr (kLanes >= 8) v = combine_dpp<kIsMax, 0x141>(v);  // row_half_mirror: the other quad of 8 lanes
    if constexpr (kLanes >= 16) v = combine_dpp<kIsMax, 0x140>(v);  // row_mirror: the other 8 of 16 lanes
    if constexpr (kLanes >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
        v = combine<kIsMax>(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
    }
    if constexpr (kLanes >= 64) {
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
        v = combine<kIsMax>(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
    }
    return v;
}

// exp(x - m) is computed as exp2(x * log2e - shift) with shift = m * log2e, rounded.  That rounding is a factor of up to
// 1 + |m| 2^-24 on every exponential; where all of a segment's share one shift it cancels against their sum.
//
// A product that overflows (a mask of fp32's or bf16's lowest value fills a part, or the whole segment) would leave infinity minus
// infinity: there the factor is 1, since values of that size are equal or at least 2^100 apart.
struct Base {
    float scale, shift;
};

NT_DEVICE bool overflows(float m) { return fabsf(m) > 2.3e38f; }  // m * log2e does

NT_DEVICE Base base_of(float m) {
#pragma clang fp contract(off)  // (the difference of two shifts is that of the rounded products)
    const float scale = overflows(m) ? 1.0f : kLog2e;
    return {scale, m == -INFINITY ? 0.0f : m * scale};  // (without a finite element there is nothing to subtract: the exponentials are zeros)
}

NT_DEVICE float exponential(float x, Base base) { return __builtin_amdgcn_exp2f(fmaf(x, base.scale, -base.shift)); }

// The factor that takes exponentials relative to `part_max` to exponentials relative to `total_max`: from the difference of the two
// SHIFTS, so that the rounding of each cancels.  exp(part_max - total_max) leaves a rounding of its own on every part (fp32
// rows of 4096 values of spread 5, 2-norm of the error against 64 bits: 1.1e-5 around 1000, 1.2 % around 10^6; so 8e-8 at both).
NT_DEVICE float rescale(float part_max, float total_max) {
    const float apart = overflows(part_max) || overflows(total_max) ? part_max - total_max : base_of(part_max).shift - base_of(total_max).shift;
    return part_max == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(apart);
}

// Reduction over the kRowThreads threads that share a segment: waves, then partial results across waves through LDS.
template <int kRowThreads, bool kIsMax>
NT_DEVICE float group_reduce(float v, float *scratch) {
    constexpr int kLanes = kRowThreads < 64 ? kRowThreads : 64;
    v = wave_reduce<kIsMax, kLanes>(v);
    if constexpr (kRowThreads > 64) {
        constexpr int kWaves = kRowThreads / 64;
        const int wave = threadIdx.x >> 6;
        __syncthreads();  // scratch may still be read from a previous reduction
        if ((threadIdx.x & 63) == 0) scratch[wave] = v;
        __syncthreads();
        v = scratch[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) v = combine<kIsMax>(v, scratch[w]);
    }
    return v;
}

template <typename T>
struct Vec16 {  // 16 bytes of T
    static constexpr int kWidth = 16 / sizeof(T);
    typedef T type __attribute__((ext_vector_type(16 / sizeof(T))));
};

// Segments of unit column stride that fit the registers of the kRowThreads threads that share one: read once, written
// once, in one launch.  A segment is cut into one part per wave; a part has its own maximum and its own sum of
// exponentials relative to it, and the parts meet in ONE exchange (shared by all: two floats per wave in LDS, one
// barrier), so a wave computes as soon as its own loads are back.
//
// Thread t of a group owns vectors t, t + kRowThreads, ... (coalesced 16-byte accesses).  The segment may start at any
// element and have any length: vectors are counted from its first 16-byte boundary, and the up to 2 (W - 1) elements
// before the first and behind the last whole vector belong to the first threads, one each (two in groups of 8).
//
// 2-byte elements are kept as they were read where more than 64 fall to a thread (64 registers then hold 128 of them, so 1024
// threads hold a segment of 131072): the exponential is computed twice, once for the sum and once for the result, which only
// pays where floats would not fit (fp16 [64, 50257], 49 elements a thread: 6.5 us on floats, 7.4 computed twice).
//
// What bounds it: memory where there are segments for every CU (fp32 4096 x 4096 20.3 us = 6.6 TB/s; fp16 8192 x 4099 21.9 us =
// 6.1 TB/s, 190 us with element-wise loads; fp16 4096 x 50257 145 us = 5.7 TB/s, 230 us in two sweeps over memory), the
// arithmetic of the CUs that have a segment where there are few (fp16 [64, 50257] 6.2 us, 11.4 over two launches).  Launches of
// a few microseconds gain or lose a little against loads that were waited for one by one (bf16 9000 x 2000 13.1 -> 12.0 us, fp32
// 8192 x 2000 20.9 -> 20.1, but bf16 5274 x 1792 6.9 -> 7.3 and fp32 5274 x 1792 11.8 -> 12.0: 64 threads there, 256 are 13 % slower on bf16).
template <typename T, int kRowThreads, int kVecs>
__global__ __launch_bounds__(kRowThreads > 256 ? kRowThreads : 256) void softmax_split_in_registers_kernel(SoftmaxParams p) {
    typedef typename Vec16<T>::type vec_t;
    constexpr int W = Vec16<T>::kWidth;
    typedef vec_t access_t __attribute__((aligned(sizeof(T))));
    constexpr int kGroups = kRowThreads > 256 ? 1 : 256 / kRowThreads;  // segments per workgroup
    constexpr bool kRaw = sizeof(T) == 2 && kVecs * W > 64;
    constexpr int kHeld = kRaw ? 1 : kVecs;
    constexpr int kEdgeElems = (2 * (W - 1) + kRowThreads - 1) / kRowThreads;
    constexpr int kWaves = kRowThreads > 64 ? kRowThreads / 64 : 1;
    __shared__ float2_t parts[kWaves];

    const int group = threadIdx.x / kRowThreads;
    const int t = threadIdx.x % kRowThreads;
    const int64_t seg = (int64_t)blockIdx.x * kGroups + group;
    const int64_t total = p.rows * p.segments;
    const bool active = seg < total;  // (more than one segment per workgroup: no barriers below)
    const int64_t row = active ? seg / p.segments : 0;
    const int64_t start = active ? (seg % p.segments) * p.block : 0;
    const int len = active ? (int)min(p.block, p.cols - start) : 0;

    const T *src = (const T *)p.in + row * p.in_row_stride + start;
    T *dst = (T *)p.out + row * p.out_row_stride + start;
    const int head = min(len, (int)((0 - (uintptr_t)src) & 15) / (int)sizeof(T));
    const int nvec = (len - head) / W;
    const int tail_first = head + nvec * W;
    const auto edge_index = [&](int j) {  // -> element, len and beyond: none
        const int e = j * kRowThreads + t;
        return e < head ? e : tail_first + (e - head);
    };

    vec_t raw[kRaw ? kVecs : 1];
    float x[kHeld][W];
    float edge[kEdgeElems];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < kEdgeElems; ++j) {
        const int e = edge_index(j);
        edge[j] = e < len ? (float)src[e] : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < kVecs; ++j) {
        const int v = j * kRowThreads + t;
        vec_t in;
        if (v < nvec) {
            in = *(const access_t *)(src + head + (int64_t)v * W);  // (a non-temporal load here costs 7-20 % of the rate; the non-temporal store below gains)
        } else {
#pragma unroll
            for (int e = 0; e < W; ++e) in[e] = (T)-INFINITY;
        }
        if constexpr (kRaw) {
            raw[j] = in;
        } else {
#pragma unroll
            for (int e = 0; e < W; ++e) x[j][e] = (float)in[e];
        }
    }
#pragma unroll
    for (int j = 0; j < kEdgeElems; ++j) m = fmaxf(m, edge[j]);
#pragma unroll
    for (int j = 0; j < kVecs; ++j)
#pragma unroll
        for (int e = 0; e < W; ++e) m = fmaxf(m, kRaw ? (float)raw[kRaw ? j : 0][e] : x[kRaw ? 0 : j][e]);
    // the compiler must not keep the converted values from one sweep over the registers to the next (two floats per register)
    const auto forget_conversions = [&] {
        if constexpr (kRaw) {
#pragma unroll
            for (int j = 0; j < kVecs; ++j) {
                int4_t bits = __builtin_bit_cast(int4_t, raw[j]);
                asm("" : "+v"(bits));
                raw[j] = __builtin_bit_cast(vec_t, bits);
            }
        }
    };
    forget_conversions();
    m = wave_reduce<true, (kRowThreads < 64 ? kRowThreads : 64)>(m);
    const Base from = base_of(m);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < kVecs; ++j)
#pragma unroll
        for (int e = 0; e < W; ++e) {
            if constexpr (kRaw) {
                s += exponential((float)raw[j][e], from);
            } else {
                x[j][e] = exponential(x[j][e], from);
                s += x[j][e];
            }
        }
#pragma unroll
    for (int j = 0; j < kEdgeElems; ++j) {
        edge[j] = exponential(edge[j], from);
        s += edge[j];
    }
    forget_conversions();
    s = wave_reduce<false, (kRowThreads < 64 ? kRowThreads : 64)>(s);
    float factor;
    if constexpr (kWaves > 1) {
        if ((threadIdx.x & 63) == 0) parts[threadIdx.x >> 6] = float2_t{m, s};
        __syncthreads();
        const float2_t part = parts[threadIdx.x & (kWaves - 1)];  // (a part per lane, as often as they fit a wave)
        const float total_max = wave_reduce<true, kWaves>(part[0]);
        const float sum = wave_reduce<false, kWaves>(part[1] * rescale(part[0], total_max));
        factor = rescale(m, total_max) / sum;
    } else {
        factor = 1.0f / s;
    }
#pragma unroll
    for (int j = 0; j < kVecs; ++j) {
        const int v = j * kRowThreads + t;
        if (v < nvec) {
            vec_t o;
#pragma unroll
            for (int e = 0; e < W; ++e) o[e] = (T)((kRaw ? exponential((float)raw[kRaw ? j : 0][e], from) : x[kRaw ? 0 : j][e]) * factor);
            __builtin_nontemporal_store(o, (access_t *)(dst + head + (int64_t)v * W));
        }
    }
#pragma unroll
    for (int j = 0; j < kEdgeElems; ++j) {
        const int e = edge_index(j);
        if (e < len) dst[e] = (T)(edge[j] * factor);
    }
}

// Rows of up to 64 bytes (a softmax over 4 or 8 classes, for millions of rows): one THREAD per row.  A group of
// 8 lanes per row, the smallest the vector path has, leaves most lanes without a vector on such rows.  A thread
// fetches its row in pieces of kBytes (the largest power of two that divides the row's bytes and its pitch),
// consecutive threads consecutive rows.
template <typename T, int kBytes>
__global__ __launch_bounds__(256) void softmax_thread_per_row_kernel(SoftmaxParams p, int pieces) {
    constexpr int kWidth = kBytes / (int)sizeof(T);  // elements per piece
    constexpr int kMaxPieces = 64 / kBytes;
    typedef T piece_t __attribute__((ext_vector_type(kWidth)));
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= p.rows) return;
    const piece_t *src = (const piece_t *)((const T *)p.in + row * p.in_row_stride);
    piece_t *dst = (piece_t *)((T *)p.out + row * p.out_row_stride);
    float x[kMaxPieces][kWidth];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < kMaxPieces; ++j) {
        if (j < pieces) {
            const piece_t raw = src[j];
#pragma unroll
            for (int e = 0; e < kWidth; ++e) {
                x[j][e] = (float)raw[e];
                m = fmaxf(m, x[j][e]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < kWidth; ++e) x[j][e] = -INFINITY;
        }
    }
    const Base from = base_of(m);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < kMaxPieces; ++j)
#pragma unroll
        for (int e = 0; e < kWidth; ++e) {
            x[j][e] = exponential(x[j][e], from);
            s += x[j][e];
        }
    const float inv = 1.0f / s;
#pragma unroll
    for (int j = 0; j < kMaxPieces; ++j) {
        if (j < pieces) {
            piece_t o;
#pragma unroll
            for (int e = 0; e < kWidth; ++e) o[e] = (T)(x[j][e] * inv);
            dst[j] = o;
        }
    }
}

template <typename T, int kBytes>
hipError_t launch_thread_per_row(const SoftmaxParams &p, hipStream_t stream) {
    note_launch(kLaunchSoftmax, 1, "softmax_thread_per_row_kernel, rows of up to 64 bytes");
    softmax_thread_per_row_kernel<T, kBytes><<<dim3((unsigned)((p.rows + 255) / 256)), dim3(256), 0, stream>>>(p, (int)(p.cols * (int64_t)sizeof(T) / kBytes));
    return hipGetLastError();
}

// Element path: any strides, length up to kRowThreads * kElems (what the register kernel does not take: columns that are not one element apart).
template <typename T, int kRowThreads, int kElems>
__global__ __launch_bounds__(kRowThreads > 256 ? kRowThreads : 256) void softmax_elem_kernel(SoftmaxParams p) {
    constexpr int kGroups = kRowThreads > 256 ? 1 : 256 / kRowThreads;
    __shared__ float scratch[16];

    const int group = threadIdx.x / kRowThreads;
    const int t = threadIdx.x % kRowThreads;
    const int64_t seg = (int64_t)blockIdx.x * kGroups + group;
    const int64_t total = p.rows * p.segments;
    const bool active = seg < total;
    const int64_t row = active ? seg / p.segments : 0;
    const int64_t start = active ? (seg % p.segments) * p.block : 0;
    const int len = active ? (int)min(p.block, p.cols - start) : 0;

    const T *src = (const T *)p.in + row * p.in_row_stride + start * p.in_col_stride;
    T *dst = (T *)p.out + row * p.out_row_stride + start * p.out_col_stride;

    float x[kElems];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < kElems; ++j) {
        const int c = j * kRowThreads + t;
        x[j] = c < len ? (float)src[(int64_t)c * p.in_col_stride] : -INFINITY;
        m = fmaxf(m, x[j]);
    }
    m = group_reduce<kRowThreads, true>(m, scratch);
    const Base from = base_of(m);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < kElems; ++j) {
        x[j] = exponential(x[j], from);
        s += x[j];
    }
    s = group_reduce<kRowThreads, false>(s, scratch);
    const float inv = 1.0f / s;
#pragma unroll
    for (int j = 0; j < kElems; ++j) {
        const int c = j * kRowThreads + t;
        if (c < len) dst[(int64_t)c * p.out_col_stride] = (T)(x[j] * inv);
    }
}

// One access of the kernels for long segments: 16 bytes of a segment whose columns are one element apart (global
// accesses need the element's alignment only), else one element.
template <typename T, bool kVec>
struct WideAccess {
    static constexpr int kWidth = kVec ? Vec16<T>::kWidth : 1;
    typedef typename Vec16<T>::type aligned_type;
    typedef aligned_type type __attribute__((aligned(sizeof(T))));
};

template <typename T, bool kVec>
NT_DEVICE void wide_load(const T *src, int64_t col_stride, int64_t index, int64_t count, float (&x)[WideAccess<T, kVec>::kWidth]) {
    constexpr int W = WideAccess<T, kVec>::kWidth;
    if constexpr (kVec) {
        if ((index + 1) * W <= count) {
            const typename WideAccess<T, kVec>::type v = *(const typename WideAccess<T, kVec>::type *)(src + index * W);
#pragma unroll
            for (int e = 0; e < W; ++e) x[e] = (float)v[e];
        } else {
#pragma unroll
            for (int e = 0; e < W; ++e) x[e] = index * W + e < count ? (float)src[index * W + e] : -INFINITY;
        }
    } else {
        x[0] = index < count ? (float)src[index * col_stride] : -INFINITY;
    }
}

// exp(x - maximum) / sum of one access, stored
template <typename T, bool kVec>
NT_DEVICE void wide_store(T *dst, int64_t col_stride, int64_t index, int64_t count, const float (&x)[WideAccess<T, kVec>::kWidth], Base from, float inv) {
    constexpr int W = WideAccess<T, kVec>::kWidth;
    if constexpr (kVec) {
        if ((index + 1) * W <= count) {
            typename WideAccess<T, kVec>::type v;
#pragma unroll
            for (int e = 0; e < W; ++e) v[e] = (T)(exponential(x[e], from) * inv);
            *(typename WideAccess<T, kVec>::type *)(dst + index * W) = v;
        } else {
#pragma unroll
            for (int e = 0; e < W; ++e)
                if (index * W + e < count) dst[index * W + e] = (T)(exponential(x[e], from) * inv);
        }
    } else {
        if (index < count) dst[index * col_stride] = (T)(exponential(x[0], from) * inv);
    }
}

// Long segments: one workgroup of 1024 threads per segment, two sweeps over memory: running
// maximum and sum together (a thread rescales its sum once per round of independent loads),
// then the write; the second sweep hits L2 for segments that fit there.
constexpr int kLoopThreads = 1024;

template <typename T, bool kVec>
__global__ __launch_bounds__(kLoopThreads) void softmax_loop_kernel(SoftmaxParams p) {
    constexpr int W = WideAccess<T, kVec>::kWidth;
    constexpr int kLoopUnroll = kVec ? 2 : 8;
    __shared__ float scratch[kLoopThreads / 64];
    const int64_t seg = blockIdx.x;
    const int64_t row = seg / p.segments;
    const int64_t start = (seg % p.segments) * p.block;
    const int64_t len = min(p.block, p.cols - start);
    const T *src = (const T *)p.in + row * p.in_row_stride + start * p.in_col_stride;
    T *dst = (T *)p.out + row * p.out_row_stride + start * p.out_col_stride;
    const int64_t pieces = (len + W - 1) / W;

    float m = -INFINITY, s = 0.0f;
    for (int64_t base = threadIdx.x; base < pieces; base += kLoopThreads * kLoopUnroll) {
        float x[kLoopUnroll][W];
        float round_max = -INFINITY;
#pragma unroll
        for (int u = 0; u < kLoopUnroll; ++u) {
            wide_load<T, kVec>(src, p.in_col_stride, base + u * kLoopThreads, len, x[u]);
#pragma unroll
            for (int e = 0; e < W; ++e) round_max = fmaxf(round_max, x[u][e]);
        }
        if (round_max > m) {
            s *= rescale(m, round_max);
            m = round_max;
        }
        const Base from = base_of(m);
#pragma unroll
        for (int u = 0; u < kLoopUnroll; ++u)
#pragma unroll
            for (int e = 0; e < W; ++e) s += exponential(x[u][e], from);
    }
    const float total_max = group_reduce<kLoopThreads, true>(m, scratch);
    s = group_reduce<kLoopThreads, false>(s * rescale(m, total_max), scratch);  // (every thread's sum is relative to its own maximum)
    const float inv = 1.0f / s;
    const Base from = base_of(total_max);
    for (int64_t base = threadIdx.x; base < pieces; base += kLoopThreads * kLoopUnroll) {
        float x[kLoopUnroll][W];
#pragma unroll
        for (int u = 0; u < kLoopUnroll; ++u) wide_load<T, kVec>(src, p.in_col_stride, base + u * kLoopThreads, len, x[u]);
#pragma unroll
        for (int u = 0; u < kLoopUnroll; ++u) wide_store<T, kVec>(dst, p.out_col_stride, base + u * kLoopThreads, len, x[u], from, inv);
    }
}

// Few long segments: each is cut into parts, a workgroup of 256 threads per part, two launches.  The first leaves
// every part's maximum and its sum of exponentials relative to that maximum in `partials`; the second combines
// the parts of its segment and writes its own part (its input is the first launch's and comes from the caches).
// kVec: unit column strides, 16 bytes per access (global accesses need the element's alignment only).
constexpr int kSplitThreads = 256;
constexpr int kSplitUnroll = 4;

struct SplitPartial {
    float max, sum;
};

template <typename T, bool kVec>
__global__ __launch_bounds__(kSplitThreads) void softmax_split_partial_kernel(SoftmaxParams p, int64_t part_len, SplitPartial *partials) {
    constexpr int W = WideAccess<T, kVec>::kWidth;
    __shared__ float scratch[kSplitThreads / 64];
    const int64_t seg = blockIdx.y;
    const int64_t row = seg / p.segments;
    const int64_t start = (seg % p.segments) * p.block + (int64_t)blockIdx.x * part_len;
    const int64_t seg_end = min((seg % p.segments + 1) * p.block, p.cols);
    const int64_t count = max((int64_t)0, min(part_len, seg_end - start));
    const T *src = (const T *)p.in + row * p.in_row_stride + start * p.in_col_stride;
    const int64_t pieces = (count + W - 1) / W;
    float m = -INFINITY, s = 0.0f;
    for (int64_t base = threadIdx.x; base < pieces; base += kSplitThreads * kSplitUnroll) {
        float x[kSplitUnroll][W];
        float round_max = -INFINITY;
#pragma unroll
        for (int u = 0; u < kSplitUnroll; ++u) {
            wide_load<T, kVec>(src, p.in_col_stride, base + u * kSplitThreads, count, x[u]);
#pragma unroll
            for (int e = 0; e < W; ++e) round_max = fmaxf(round_max, x[u][e]);
        }
        if (round_max > m) {
            s *= rescale(m, round_max);
            m = round_max;
        }
        const Base from = base_of(m);
#pragma unroll
        for (int u = 0; u < kSplitUnroll; ++u)
#pragma unroll
            for (int e = 0; e < W; ++e) s += exponential(x[u][e], from);
    }
    const float part_max = group_reduce<kSplitThreads, true>(m, scratch);
    s = group_reduce<kSplitThreads, false>(s * rescale(m, part_max), scratch);
    if (threadIdx.x == 0) {
        SplitPartial r;
        r.max = part_max;
        r.sum = s;
        partials[seg * gridDim.x + blockIdx.x] = r;
    }
}

template <typename T, bool kVec>
__global__ __launch_bounds__(kSplitThreads) void softmax_split_finish_kernel(SoftmaxParams p, int64_t part_len, const SplitPartial *partials) {
    constexpr int W = WideAccess<T, kVec>::kWidth;
    __shared__ float scratch[kSplitThreads / 64];
    const int64_t seg = blockIdx.y;
    const int64_t row = seg / p.segments;
    const int64_t start = (seg % p.segments) * p.block + (int64_t)blockIdx.x * part_len;
    const int64_t seg_end = min((seg % p.segments + 1) * p.block, p.cols);
    const int64_t count = max((int64_t)0, min(part_len, seg_end - start));
    // the parts of this segment (at most one per thread)
    SplitPartial mine;
    mine.max = -INFINITY;
    mine.sum = 0.0f;
    if (threadIdx.x < gridDim.x) mine = partials[seg * gridDim.x + threadIdx.x];
    const float total_max = group_reduce<kSplitThreads, true>(mine.max, scratch);
    const float inv = 1.0f / group_reduce<kSplitThreads, false>(mine.sum * rescale(mine.max, total_max), scratch);
    const Base from = base_of(total_max);
    const T *src = (const T *)p.in + row * p.in_row_stride + start * p.in_col_stride;
    T *dst = (T *)p.out + row * p.out_row_stride + start * p.out_col_stride;
    const int64_t pieces = (count + W - 1) / W;
    for (int64_t base = threadIdx.x; base < pieces; base += kSplitThreads * kSplitUnroll) {
        float x[kSplitUnroll][W];
#pragma unroll
        for (int u = 0; u < kSplitUnroll; ++u) wide_load<T, kVec>(src, p.in_col_stride, base + u * kSplitThreads, count, x[u]);
#pragma unroll
        for (int u = 0; u < kSplitUnroll; ++u) wide_store<T, kVec>(dst, p.out_col_stride, base + u * kSplitThreads, count, x[u], from, inv);
    }
}

// true when the segments were served by the two launches over parts.  `in_registers`: the segments are short enough for
// the kernel that reads them once in one launch; that one wins unless a few segments of its longest leave most CUs
// with nothing to compute (fp16 [1, 131072] 12.0 us against 7.8 in parts, [16, 100000] 10.5 against 8.9, [64, 131072] 13.3 against
// 12.6; but [4, 65536] 6.2 against 7.0, [64, 50257] 6.5 against 11.4, fp32 [16, 50257] 6.4 against 7.4, [128, 50257] 11.0 against 15.7).
template <typename T>
bool run_split(const SoftmaxParams &p, int64_t len, bool in_registers, hipStream_t stream, hipError_t *status) {
    const int64_t total = p.rows * p.segments;
    const int64_t bytes = len * (int64_t)sizeof(T);
    if (total > 128) return false;
    if (in_registers ? (sizeof(T) == 4 || len <= 65536 || total > 64) : bytes < (1 << 16)) return false;
    const int64_t wanted = std::min<int64_t>(kSplitThreads, std::max<int64_t>(2, 1024 / total));  // (the finishing launch reads one part per thread)
    int64_t part_len = std::max<int64_t>(4096, (((len + wanted - 1) / wanted + 2047) / 2048) * 2048);
    const int64_t parts = (len + part_len - 1) / part_len;
    if (parts < 2 || parts > kSplitThreads) return false;
    WorkspaceLease lease(stream);
    SplitPartial *partials = (SplitPartial *)lease.get(kWorkspaceSoftmaxParts, (size_t)(total * parts) * sizeof(SplitPartial));
    if (partials == nullptr) return false;  // no scratch: one workgroup per segment
    const dim3 grid((unsigned)parts, (unsigned)total), block(kSplitThreads);
    note_launch(kLaunchSoftmax, kSplitThreads, "softmax_split_partial_kernel + softmax_split_finish_kernel, long segments cut into parts");
    if (p.in_col_stride == 1 && p.out_col_stride == 1) {
        softmax_split_partial_kernel<T, true><<<grid, block, 0, stream>>>(p, part_len, partials);
        softmax_split_finish_kernel<T, true><<<grid, block, 0, stream>>>(p, part_len, partials);
    } else {
        softmax_split_partial_kernel<T, false><<<grid, block, 0, stream>>>(p, part_len, partials);
        softmax_split_finish_kernel<T, false><<<grid, block, 0, stream>>>(p, part_len, partials);
    }
    *status = hipGetLastError();
    return true;
}

// Whole vectors of the longest segments that 256, 512 and 1024 threads hold (why there: at the choice in run_softmax).
template <typename T> constexpr int64_t kMostVecs256 = sizeof(T) == 4 ? 768 : 2048;
template <typename T> constexpr int64_t kMostVecs512 = sizeof(T) == 4 ? 2048 : 4096;
constexpr int64_t kMostVecs1024 = 1024 * 16;

// Segments of kFewest .. kMost whole vectors.
template <typename T, int kRowThreads, int64_t kFewest, int64_t kMost>
hipError_t launch_in_registers(const SoftmaxParams &p, int64_t len, hipStream_t stream) {
    const int64_t total = p.rows * p.segments;
    constexpr int kGroups = kRowThreads > 256 ? 1 : 256 / kRowThreads;
    const dim3 grid((unsigned)((total + kGroups - 1) / kGroups)), block(kRowThreads > 256 ? kRowThreads : 256);
    const int64_t vecs = (len / Vec16<T>::kWidth + kRowThreads - 1) / kRowThreads;  // per thread
    note_launch(kLaunchSoftmax, kRowThreads, "softmax_split_in_registers_kernel, one launch, this many threads per row segment, one part per wave");
    static_assert(kMost <= 16 * kRowThreads, "at most 16 vectors per thread");
    // kPrevious: the next smaller step
#define NT_SOFTMAX_VECS(N, kPrevious) \
    if constexpr (kFewest <= N * kRowThreads && kMost > kPrevious * kRowThreads) { \
        if (vecs <= N) { \
            softmax_split_in_registers_kernel<T, kRowThreads, N><<<grid, block, 0, stream>>>(p); \
            return hipGetLastError(); \
        } \
    }
    // (a thread computes all its vectors, also those behind the end of a segment: steps of one where a step is most of the work)
    NT_SOFTMAX_VECS(1, 0)
    NT_SOFTMAX_VECS(2, 1)
    NT_SOFTMAX_VECS(3, 2)
    NT_SOFTMAX_VECS(4, 3)
    NT_SOFTMAX_VECS(5, 4)
    NT_SOFTMAX_VECS(6, 5)
    NT_SOFTMAX_VECS(7, 6)
    NT_SOFTMAX_VECS(8, 7)
    NT_SOFTMAX_VECS(10, 8)
    NT_SOFTMAX_VECS(12, 10)
    NT_SOFTMAX_VECS(16, 12)
#undef NT_SOFTMAX_VECS
    return hipErrorInvalidValue;
}

template <typename T, int kRowThreads, int kElems>
hipError_t launch_elem(const SoftmaxParams &p, hipStream_t stream) {
    const int64_t total = p.rows * p.segments;
    constexpr int kGroups = kRowThreads > 256 ? 1 : 256 / kRowThreads;
    const dim3 grid((unsigned)((total + kGroups - 1) / kGroups)), block(kRowThreads > 256 ? kRowThreads : 256);
    note_launch(kLaunchSoftmax, kRowThreads, "softmax_elem_kernel, element by element, this many threads per row segment");
    softmax_elem_kernel<T, kRowThreads, kElems><<<grid, block, 0, stream>>>(p);
    return hipGetLastError();
}

// `variant`: 0 = library's choice, 1 = one wave per segment, 2 = one workgroup per segment
template <typename T>
int run_softmax(const SoftmaxParams &p, int variant, hipStream_t stream) {
    constexpr int W = Vec16<T>::kWidth;
    const int64_t total = p.rows * p.segments;
    if (total == 0 || p.cols == 0) return 0;
    if (total > 0x7fffffffll) return NINETOOTHED_NO_KERNEL;
    const int64_t len = p.block < p.cols ? p.block : p.cols;
    const bool unit_columns = p.in_col_stride == 1 && p.out_col_stride == 1;
    // rows of up to 64 bytes, many of them: a thread per row
    if (variant == 0 && p.segments == 1 && unit_columns && p.cols * (int64_t)sizeof(T) <= 64 && p.rows >= 4096 &&
        (p.rows + 255) / 256 <= 0x7fffffffll) {
        const uint64_t bits = (uint64_t)(p.cols * sizeof(T)) | (uint64_t)(p.in_row_stride * (int64_t)sizeof(T)) | (uint64_t)(p.out_row_stride * (int64_t)sizeof(T)) |
                              (uint64_t)(uintptr_t)p.in | (uint64_t)(uintptr_t)p.out;  // what every piece's address and size is a multiple of
        if (bits % 16 == 0) return (int)launch_thread_per_row<T, 16>(p, stream);
        if (bits % 8 == 0) return (int)launch_thread_per_row<T, 8>(p, stream);
        if (bits % 4 == 0) return (int)launch_thread_per_row<T, 4>(p, stream);
        if constexpr (sizeof(T) == 2) {
            if (p.cols <= 8) return (int)launch_thread_per_row<T, 2>(p, stream);  // (up to 32 pieces of one element would not stay in registers)
        }
    }
    // segments that 1024 threads hold in registers: 64 of them per thread (2-byte elements as they are, two per register)
    const bool in_registers = unit_columns && len <= kMostVecs1024 * W;
    if (variant == 0) {
        hipError_t status = hipSuccess;
        if (run_split<T>(p, len, in_registers, stream, &status)) return (int)status;
    }
    if (in_registers) {
        const int64_t nvec = len / W;
        // Threads per segment.  Few vectors each keep a wave's work short where a launch has many segments; many threads fetch a
        // segment sooner where it has few.  Measured (us, threads per segment: time): fp16 30000 x 131 16: 4.8, 32: 6.7; 30000 x 515
        // 32: 10.8, 64: 12.4; 20000 x 1000 32: 13.8, 64: 13.1, 256: 22; 8192 x 4096 64: 20.6, 256: 20.9, 512: 24; 300 x 4099 64: 3.9,
        // 256: 3.6; fp32 5000 x 3000 256: 19.0, 512: 19.9; 8192 x 4096 64: 47.4, 256: 45.2, 512: 44.0; 4000 x 8195 512: 48.0, 1024: 45.0; fp16
        // 11832 x 4152 256: 33.5, 512: 44.6; 4000 x 12289 256: 33.4, 512: 32.8, 1024: 39.4; 4000 x 32000 512: 86.6, 1024: 89.5; 4096 x 50257
        // 512: 149, 1024: 145
        if (variant == 0 && p.segments == 1) {
            if (nvec <= 8) return (int)launch_in_registers<T, 8, 0, 8>(p, len, stream);
            if (nvec <= 32) return (int)launch_in_registers<T, 16, 9, 32>(p, len, stream);
            if (nvec <= 96) return (int)launch_in_registers<T, 32, 33, 96>(p, len, stream);
        }
        const bool one_wave = nvec <= 512 && (variant == 1 || (variant == 0 && (total >= 4096 || nvec <= 64)));
        if (one_wave) return (int)launch_in_registers<T, 64, 0, 512>(p, len, stream);
        if (nvec <= kMostVecs256<T>) return (int)launch_in_registers<T, 256, 0, kMostVecs256<T>>(p, len, stream);
        if (nvec <= kMostVecs512<T>) return (int)launch_in_registers<T, 512, kMostVecs256<T> + 1, kMostVecs512<T>>(p, len, stream);
        return (int)launch_in_registers<T, 1024, kMostVecs512<T> + 1, kMostVecs1024>(p, len, stream);
    }
    // element by element (any strides): as many threads per segment as keep every thread at
    // 4 .. 16 elements, from 8 lanes of a wave to a workgroup of 1024
    if (len <= 8 * 4) return (int)launch_elem<T, 8, 4>(p, stream);
    if (len <= 16 * 4) return (int)launch_elem<T, 16, 4>(p, stream);
    if (len <= 32 * 4) return (int)launch_elem<T, 32, 4>(p, stream);
    if (len <= 64 * 4) return (int)launch_elem<T, 64, 4>(p, stream);
    if (len <= 64 * 16) return (int)launch_elem<T, 64, 16>(p, stream);
    if (len <= 256 * 16) return (int)launch_elem<T, 256, 16>(p, stream);
    // (us, 256 / 1024 threads / the loop kernel: stored by columns 4096 x 4099 fp32 227 / 233 / 327, fp16 163 / 161 / 221; 4096 x 8192
    // fp16 305 / 354 / 638; every second column 4096 x 8192 fp32 159 / 153 / 154, but fp16 113 / 65 / 76; 1024 threads / the loop
    // kernel: every second column 4096 x 12289 fp32 232 / 239, by columns 2048 x 16384 fp32 432 / 620, fp16 393 / 501)
    if (len <= 256 * 32) return (int)launch_elem<T, 256, 64>(p, stream);
    if (len <= 1024 * 16) return (int)launch_elem<T, 1024, 16>(p, stream);
    note_launch(kLaunchSoftmax, kLoopThreads, "softmax_loop_kernel, two sweeps over a long row segment");
    if (unit_columns)
        softmax_loop_kernel<T, true><<<dim3((unsigned)total), dim3(kLoopThreads), 0, stream>>>(p);
    else
        softmax_loop_kernel<T, false><<<dim3((unsigned)total), dim3(kLoopThreads), 0, stream>>>(p);
    return (int)hipGetLastError();
}

int softmax_entry(NineToothedStream stream, const NineToothedTensor &input, const NineToothedTensor &output, int dtype,
                  int block_size, int variant) {
    if (!input.shape || !output.shape || !input.strides || !output.strides) return hipErrorInvalidValue;
    if (input.shape[0] != output.shape[0] || input.shape[1] != output.shape[1]) return hipErrorInvalidValue;
    SoftmaxParams p;
    p.in = input.data;
    p.out = output.data;
    p.rows = (int64_t)input.shape[0];
    p.cols = (int64_t)input.shape[1];
    p.in_row_stride = input.strides[0];
    p.in_col_stride = input.strides[1];
    p.out_row_stride = output.strides[0];
    p.out_col_stride = output.strides[1];
    p.block = block_size > 0 ? block_size : (p.cols > 0 ? p.cols : 1);
    p.segments = p.cols > 0 ? (p.cols + p.block - 1) / p.block : 0;
    switch (dtype) {
        case NINETOOTHED_FLOAT32:
            return run_softmax<float>(p, variant, (hipStream_t)stream);
        case NINETOOTHED_FLOAT16:
            return run_softmax<half_t>(p, variant, (hipStream_t)stream);
        case NINETOOTHED_BFLOAT16:
            return run_softmax<bf16_t>(p, variant, (hipStream_t)stream);
        default:
            return NINETOOTHED_NO_KERNEL;
    }
}

}  // namespace
}  // namespace nt

extern "C" {

NineToothedResult launch_nt_softmax(NineToothedStream stream, NineToothedTensor input, NineToothedTensor output,
                                    int dtype, int block_size) {
    return nt::softmax_entry(stream, input, output, dtype, block_size, 0);
}

NineToothedResult launch_nt_softmax_config(NineToothedStream stream, int config, NineToothedTensor input,
                                           NineToothedTensor output, int dtype, int block_size) {
    if (config < 0 || config > 2) return NINETOOTHED_NO_KERNEL;
    return nt::softmax_entry(stream, input, output, dtype, block_size, config);
}

}  // extern "C"
