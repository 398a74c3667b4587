// The epilogue that the convolution kernels on 16x16x32 MFMAs share.
#pragma once

#include "gemm_fast.h"

namespace nt {

// n / d for 0 <= n < 2^31 and quotients below 2^22, one_by_d = 1.0f / d: three roundings of 2^-24 leave the product less than one off.
NT_DEVICE int quick_quotient(int n, int d, float one_by_d) {
    const int q = (int)((float)n * one_by_d), rest = n - q * d;
    return q + (rest >= d) - (rest < 0);
}

// Stores a wave's tile of TM x TN accumulator blocks of a convolution.  A lane holds, per block of 16 positions x 16 output channels,
// channel lane % 16 and the positions 4 * (lane / 16) + 0 .. 3.  The blocks pass through the wave's slab of LDS, [channel][position] with
// 16-byte chunks swizzled by channel, kSlabBlocks blocks of channels at a time: per output channel the positions of an image are
// contiguous, and 8 of them leave with one store.  `first_row` and `first_filter`: the tile's first position (over all images) and channel.
// Params: the output's y, K, P, Q, M, one_by_pq (1.0f / (P * Q)), dense_out (1: a contiguous NCHW tensor on a 16-byte boundary; 2: channels last; 0: any strides)
// and ys (element strides).
template <typename T, int TM, int TN, int kSlabBlocks, typename Params>
NT_DEVICE void store_conv_tile(const Params &p, const float4_t (&acc)[TM][TN], NT_LDS unsigned char *slab, int first_row, int first_filter, int lane) {
    typedef typename Elem<T>::vec8 vec8;
    constexpr int kWaveM = TM * 16, kSlabChannels = 16 * kSlabBlocks, kChunks = kWaveM / 8;
    constexpr int kSlots = kChunks <= 4 ? 4 : kChunks <= 8 ? 8 : 16, kRowBytes = kSlots * 16;  // (a power of two, for the swizzle)
    static_assert(TN % kSlabBlocks == 0 && kChunks <= 16, "whole slabs");
    const int i16 = lane & 15, kg = lane >> 4;
    const int PQ = p.P * p.Q;
    T *Y = (T *)p.y;
    const bool whole_chunks = PQ % 8 == 0 && p.dense_out == 1;
#pragma unroll
    for (int tg = 0; tg < TN / kSlabBlocks; ++tg) {
#pragma unroll
        for (int tb = 0; tb < kSlabBlocks; ++tb)
#pragma unroll
            for (int ti = 0; ti < TM; ++ti) {
                typedef T vec4 __attribute__((ext_vector_type(4)));
                vec4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = Elem<T>::from_float(acc[ti][tg * kSlabBlocks + tb][e]);
                const int channel = tb * 16 + i16;
                const int chunk = (ti * 2 + (kg >> 1)) ^ (channel & (kSlots - 1));
                *(NT_LDS vec4 *)(slab + channel * kRowBytes + chunk * 16 + 8 * (kg & 1)) = v;
            }
        const int first_channel = first_filter + tg * kSlabChannels;
        if (p.dense_out == 2) {
            // channels-last output: a lane gathers 8 channels of one row from the slab and stores them with one
            // instruction (the channels of the slab are 32 or 64 consecutive bytes of the tensor)
            constexpr int kGroups = kSlabChannels / 8;
#pragma unroll
            for (int it = 0; it < (kGroups * kWaveM + 63) / 64; ++it) {
                const int idx = it * 64 + lane;
                const int row = idx / kGroups, first = (idx % kGroups) * 8;
                if (row >= kWaveM) continue;
                vec8 v;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int channel = first + e;
                    v[e] = *(const NT_LDS T *)(slab + channel * kRowBytes + (((row >> 3) ^ (channel & (kSlots - 1))) * 16) + (row & 7) * 2);
                }
                const int m = first_row + row;
                const int out_channel = first_channel + first;
                if (m >= p.M || out_channel >= p.K) continue;
                const int image = quick_quotient(m, PQ, p.one_by_pq), pq = m - image * PQ;
                const int oy = pq / p.Q, ox = pq - oy * p.Q;
                T *to = Y + (int64_t)image * p.ys[0] + (int64_t)oy * p.ys[2] + (int64_t)ox * p.ys[3] + out_channel;
                if (out_channel + 8 <= p.K) {
                    typedef vec8 unaligned_vec8 __attribute__((aligned(2)));
                    *(unaligned_vec8 *)to = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (out_channel + e < p.K) to[e] = v[e];
                }
            }
            continue;
        }
#pragma unroll
        for (int it = 0; it < kSlabChannels * kSlots / 64; ++it) {
            const int idx = it * 64 + lane;
            const int channel = idx / kSlots;
            const int phys = idx % kSlots;
            const int chunk = phys ^ (channel & (kSlots - 1));
            vec8 v = *(const NT_LDS vec8 *)(slab + channel * kRowBytes + phys * 16);
            const int m = first_row + chunk * 8;
            if (chunk >= kChunks || m >= p.M) continue;
            const int out_channel = first_channel + channel;
            if (out_channel >= p.K) continue;  // a partial last tile of output channels
            int image = quick_quotient(m, PQ, p.one_by_pq), pq = m - image * PQ;
            if (whole_chunks) {  // the 8 rows lie in one image and start at a multiple of 8
                __builtin_nontemporal_store(v, (vec8 *)(Y + ((int64_t)image * p.K + out_channel) * PQ + pq));  // +2 % over a plain store
            } else if (p.dense_out == 1 && pq + 8 <= PQ && m + 8 <= p.M) {
                // the 8 rows lie in one image, only not on a 16-byte boundary (a 7 x 7 map): one store all the same
                // (global accesses need the element's alignment only)
                typedef vec8 unaligned_vec8 __attribute__((aligned(2)));
                *(unaligned_vec8 *)(Y + ((int64_t)image * p.K + out_channel) * PQ + pq) = v;
            } else {
                // (any output strides: a channels-last tensor, a slice of a wider one)
                int oy = pq / p.Q, ox = pq - oy * p.Q;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (m + e < p.M) Y[(int64_t)image * p.ys[0] + (int64_t)out_channel * p.ys[1] + (int64_t)oy * p.ys[2] + (int64_t)ox * p.ys[3]] = v[e];
                    if (++ox == p.Q) {
                        ox = 0;
                        if (++oy == p.P) {
                            oy = 0;
                            ++image;
                        }
                    }
                }
            }
        }
    }
}

}  // namespace nt
