// Skinny products for gfx950: C[M, N] = A[M, K] @ B[N, K]^T with few rows (`x @ w.T` of a decoding step), which are bound by
// reading B once.
//
// What the tile kernels spend on such a product: barriers that tie all waves to the slowest fill, every workgroup at the
// same position of K at the same time (the rows of B lie a power of two of bytes apart as a rule, so that all of these
// reads meet in the same memory channels: 4.5 TB/s where starts 2 KiB apart give 6.1), B kept in caches that it does not
// fit (non-temporal loads: 6.9 TB/s against 6.3), and a second launch where tiles do not fill the chip.
//
// Here every wave streams its own part of B through a ring in LDS that no other wave touches -- no barrier before the end --
// and the waves of a workgroup, all on the same columns of C and each on its own pieces of K in turn, add up their
// accumulators through LDS once, behind the loop.  The way through LDS is for the sake of the address unit: a load whose
// neighbouring lanes lie in different cache lines (the layout of an MFMA operand) passes at 16 bytes per cycle and CU (38
// GB/s whatever the level it hits), one whose lanes run along whole lines at 64 (149 GB/s from L2, 65-70 from memory).
//
// Measured (us, best tile instance -> this, bf16 / fp16 operands that no cache holds): 16 x 50256 x 4096 93.7 -> 71.0 (5.8 TB/s);
// 16 x 8192 x 8192 36.2 -> 24.3; 16 x 4096 x 4096 14.9 -> 8.5; 10 x 3960 x 4352 17.5 -> 8.4; 32 x 4096 x 4096 15.0 -> 10.4;
// 48 x 8192 x 2048 15.0 -> 11.5; 64 x 1024 x 8192 29.7 -> 22.6.
//
// Operands as in the tile kernels with tails and a transposed rhs: rows of A and B with k contiguous and on 16-byte
// boundaries, K a multiple of 8, any N.
#pragma once

#include <type_traits>

#include "gemm_fast.h"

namespace nt {

// MB: 16-row blocks of C (the product has at most 16 MB rows); NB: 16-column blocks per workgroup; kWaves: parts of K;
// kStages: depth of a wave's ring; kAuxB: cache policy of the fills of B (0, or 2: non-temporal).  A stage holds 64 positions of k: one cache line of every row of A and of B.
template <int MB, int NB>
struct SkinnyStage {
    static constexpr int kStep = 64;
    static constexpr int kFillsA = MB * 2, kFillsB = NB * 2;  // of 1 KiB, 8 rows each
    static constexpr int kBytesA = kFillsA * 1024;
    static constexpr int kFills = kFillsA + kFillsB, kBytes = kFills * 1024;
};

template <typename T, int MB, int NB, int kWaves, int kStages, int kAuxB>
__global__ __launch_bounds__(kWaves * 64) void gemm_skinny_kernel(GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef Elem<T> E;
    typedef typename E::vec8 vec8;
    typedef SkinnyStage<MB, NB> Stage;
    constexpr int kStep = Stage::kStep, BN = NB * 16;
    constexpr unsigned kBehind = 0x7fffffffu;  // behind every descriptor, whatever is added: such a fill writes zeros and reads nothing
    static_assert(kStages >= 2 && kStages <= 4, "2..4 stages");

    // an array per stage: the compiler then knows that a fill does not alias the reads of another stage
    __shared__ __attribute__((aligned(1024))) unsigned char lds0[kWaves * Stage::kBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char lds1[kWaves * Stage::kBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char lds2[kStages > 2 ? kWaves * Stage::kBytes : 16];
    __shared__ __attribute__((aligned(1024))) unsigned char lds3[kStages > 3 ? kWaves * Stage::kBytes : 16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.x * BN;
    auto stage = [&](auto tag) -> NT_LDS unsigned char * {
        constexpr int i = decltype(tag)::value;
        if constexpr (i == 0) return (NT_LDS unsigned char *)lds0 + wave * Stage::kBytes;
        else if constexpr (i == 1) return (NT_LDS unsigned char *)lds1 + wave * Stage::kBytes;
        else if constexpr (i == 2) return (NT_LDS unsigned char *)lds2 + wave * Stage::kBytes;
        else return (NT_LDS unsigned char *)lds3 + wave * Stage::kBytes;
    };

    // descriptors that end with the matrices; rows past M, columns past N and positions past K go behind them
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.a, 0, (unsigned)((((int64_t)p.m - 1) * p.lda + p.k) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.b + (int64_t)n0 * p.ldb), 0,
                                                                            (unsigned)((((int64_t)min(BN, p.n - n0) - 1) * p.ldb + p.k) * 2), 0x00020000);

    // what lane l fills: instruction j rows 8 j .. + 7, one cache line each, its 16-byte pieces exchanged by the tile kernels' swizzle
    // (which piece of a row a lane takes is the same for even and for odd instructions: the swizzle has a period of 16 rows)
    unsigned a_src[Stage::kFillsA], b_src[Stage::kFillsB];
    int piece_k[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) piece_k[j] = a_phys_chunk16<kStep>(j * 8 + lane / 8, lane % 8) * 8;
#pragma unroll
    for (int j = 0; j < Stage::kFillsA; ++j) {
        const int r = j * 8 + lane / 8;
        a_src[j] = r < p.m ? (unsigned)(r * (int)p.lda + piece_k[j & 1]) * 2u : kBehind;
    }
#pragma unroll
    for (int j = 0; j < Stage::kFillsB; ++j) {
        const int r = j * 8 + lane / 8;
        b_src[j] = n0 + r < p.n ? (unsigned)(r * (int)p.ldb + piece_k[j & 1]) * 2u : kBehind;
    }

    const int pieces = (p.k + kStep - 1) / kStep;  // dealt to the waves in turn
    const int steps = (pieces + kWaves - 1) / kWaves;
    const int first = (int)(blockIdx.x * (unsigned)(1024 / kStep) % (unsigned)pieces);  // starts 2 KiB apart
    auto fill = [&](auto tag, int step) {
        NT_LDS unsigned char *to = stage(tag);
        const int piece = step * kWaves + wave;
        const int at = piece + first < pieces ? piece + first : piece + first - pieces;
        const int k0 = piece < pieces ? at * kStep : p.k;  // (past the end: zeros)
        unsigned past[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) past[j] = k0 + piece_k[j] < p.k ? 0u : 0x80000000u;
#pragma unroll
        for (int j = 0; j < Stage::kFillsB; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, to + Stage::kBytesA + j * 1024, 16, (b_src[j] + (unsigned)k0 * 2u) | past[j & 1], 0, 0, kAuxB);
#pragma unroll
        for (int j = 0; j < Stage::kFillsA; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, to + j * 1024, 16, (a_src[j] + (unsigned)k0 * 2u) | past[j & 1], 0, 0, 0);
    };

    float4_t acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[mb][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    int frag[kStep / 32];  // operand fragments of the 16x16x32 MFMA, as in the tile kernels (16 rows further: the same swizzle)
#pragma unroll
    for (int ks = 0; ks < kStep / 32; ++ks) frag[ks] = i16 * (kStep * 2) + a_phys_chunk16<kStep>(i16, ks * 4 + kg) * 16;
    auto multiply = [&](auto tag) {
        const NT_LDS unsigned char *from = stage(tag);
#pragma unroll
        for (int ks = 0; ks < kStep / 32; ++ks) {
            vec8 a[MB], b[NB];
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) a[mb] = *(const NT_LDS vec8 *)(from + frag[ks] + mb * 2048);
#pragma unroll
            for (int j = 0; j < NB; ++j) b[j] = *(const NT_LDS vec8 *)(from + Stage::kBytesA + frag[ks] + j * 2048);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[mb][j] = E::mfma16(b[j], a[mb], acc[mb][j]);  // lane: row i16 of C, columns 4 kg .. + 3 of the block
        }
    };

    static_for<0, kStages - 1>([&](auto s) { fill(s, decltype(s)::value); });
    for (int step = 0; step < steps; step += kStages) {
        static_for<0, kStages>([&](auto s) {
            constexpr int kS = decltype(s)::value;
            // this step's stage has landed; the reads of the one before it are done, its stage is refilled
            // (steps past the end multiply zeros)
            wait_vmcnt<(kStages - 2) * Stage::kFills>();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            fill(std::integral_constant<int, (kS + kStages - 1) % kStages>(), step + kS + kStages - 1);
            multiply(s);
        });
    }

    // ---- sum over the waves, epilogue: a thread finishes four columns of a row ----
    wait_vmcnt<0>();
    __syncthreads();
    NT_LDS float4_t *sums = (NT_LDS float4_t *)lds0;  // (kWaves x NB KiB: no more than the stages' own)
    static_assert(Stage::kBytes >= NB * 1024, "the sums fit a stage");
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb > 0) __syncthreads();
#pragma unroll
        for (int j = 0; j < NB; ++j) sums[(wave * NB + j) * 64 + lane] = acc[mb][j];
        __syncthreads();
        for (int item = threadIdx.x; item < NB * 64; item += kWaves * 64) {
            float4_t sum = sums[item];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) sum += sums[w * NB * 64 + item];
            const int row = mb * 16 + (item & 15), col = n0 + (item >> 6) * 16 + 4 * ((item >> 4) & 3);
            if (row >= p.m || col >= p.n) continue;
            const bool whole = col + 4 <= p.n;
            if (p.out_float) {
                typedef float4_t unaligned_t __attribute__((aligned(4)));
                float *c = (float *)p.c + (int64_t)row * p.ldc + col;
                if (whole) *(unaligned_t *)c = sum;
                else
                    for (int e = 0; col + e < p.n; ++e) c[e] = sum[e];
                continue;
            }
            typedef T out_t __attribute__((ext_vector_type(4)));
            typedef out_t unaligned_t __attribute__((aligned(2)));
            out_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (p.linear) {
                    v[e] = E::from_float(linear_value(p, sum[e], col + e < p.n ? linear_bias<T>(p, col + e) : 0.0f));
                    continue;
                }
                v[e] = E::from_float(sum[e]);
                if (p.bias != nullptr && col + e < p.n) {  // the product is rounded to the element type, then combined in fp32
                    const T input = ((const T *)p.bias)[(int64_t)row * p.bias_stride_m + (int64_t)(col + e) * p.bias_stride_n];
                    v[e] = E::from_float(p.beta * E::to_float(input) + p.alpha * E::to_float(v[e]));
                }
            }
            T *c = (T *)p.c + (int64_t)row * p.ldc + col;
            if (whole) *(unaligned_t *)c = v;
            else
                for (int e = 0; col + e < p.n; ++e) c[e] = v[e];
        }
    }
#endif
}

}  // namespace nt
