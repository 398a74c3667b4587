// C ABI for the GEMM family: launch_nt_matmul, launch_nt_addmm,
// launch_nt_conv2d and the tile-selection entry points.
#include <algorithm>
#include <cmath>
#include <memory>
#include <mutex>
#include <type_traits>
#include <shared_mutex>
#include <unordered_map>
#include <vector>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "conv2d.h"
#include "gemm_fast.h"
#include "gemm_generic.h"
#include "gemm_skinny.h"
#include "tune.h"
#include "workspace.h"

namespace nt {
namespace {

struct GemmProblem {
    int dtype, out_dtype;
    int m, n, k;
    const void *a, *b, *bias;
    void *c;
    int64_t sam, sak, sbk, sbn, scm, scn, sim, sin;
    float alpha, beta;
    int batch = 1;  // independent products that share the shapes; operands move by these element strides
    int64_t a_batch = 0, b_batch = 0, c_batch = 0, bias_batch = 0;
    // set by the entry point that allocates nothing: split-K parts go here instead of the stream's workspace
    float *fixed_scratch = nullptr;
    size_t fixed_scratch_bytes = 0;
    bool hinted = false;  // the caller gave block sizes: the call stays on kernels without scratch memory
    // a linear epilogue: max(product * alpha + column_bias[n], lower) in fp32
    bool linear = false;
    const void *column_bias = nullptr;  // may be null; its stride is sin
    bool bias_float = false;
    float lower = -INFINITY;
    bool addmm() const { return bias != nullptr; }
};

int g_tile_order = 0;  // see GemmParams::order; changed only by measurement builds

typedef hipError_t (*LaunchFn)(const GemmProblem &, hipStream_t);
typedef bool (*AcceptFn)(const GemmProblem &);

struct GemmInstance {
    const char *name;
    int bm, bn, bk;
    AcceptFn accepts;
    LaunchFn launch;
};

// the fast instances take B row-major ([K, N], unit column stride) or transposed ([N, K] storage, unit k stride)
bool b_is_transposed(const GemmProblem &q) { return q.sbn != 1 && q.sbk == 1; }

template <int BM, int BN, int BK, int kStages, bool kTail = false>
bool fast_accepts(const GemmProblem &q) {
    if (q.dtype != NINETOOTHED_FLOAT16 && q.dtype != NINETOOTHED_BFLOAT16) return false;
    // the element type, or fp32 for a plain product (the accumulators as they are)
    if (q.out_dtype != q.dtype && !(q.out_dtype == NINETOOTHED_FLOAT32 && !q.addmm())) return false;
    if (q.m <= 0 || q.n <= 0 || q.k <= 0) return false;
    // any number of rows: rows past M read as zeros and are not stored; N and K must fit the tile,
    // or, for the instances with tails, be multiples of 8 (whole 16-byte chunks)
    // (K: whole 16-byte chunks of the k-contiguous rows; N: only where rows of B run along it.  With a
    // transposed B any N goes: C is then stored element by element when its rows are not 16-byte aligned)
    if (kTail ? (q.k % 8 || (q.n % 8 && !b_is_transposed(q))) : (q.n % BN || q.k % BK)) return false;
    if (q.sak != 1 || q.scn != 1) return false;
    if (q.sam % 8 || q.sam < q.k || q.scm < q.n) return false;
    if (((uintptr_t)q.a & 15) || ((uintptr_t)q.b & 15)) return false;
    if (!kTail && (((uintptr_t)q.c & 15) || q.scm % 8)) return false;
    // (a batch: the operands of every product on 16-byte boundaries; the outputs too, unless the instance stores element by element)
    if (q.batch > 1 && ((q.a_batch | q.b_batch) % 8 || (!kTail && q.c_batch % 8) || (int64_t)((q.m + BM - 1) / BM) * ((q.n + BN - 1) / BN) * q.batch > 0x7fffffffll)) return false;
    // per-lane 32-bit byte offsets inside one tile panel
    if ((int64_t)BM * q.sam * 2 >= (int64_t(1) << 31)) return false;
    if (b_is_transposed(q)) {  // B as [N, K] with K contiguous (`x @ w.T`)
        if (q.sbn % 8 || q.sbn < q.k) return false;
        if ((int64_t)BN * q.sbn * 2 >= (int64_t(1) << 31)) return false;
    } else {
        if (q.sbn != 1 || q.sbk % 8 || q.sbk < q.n) return false;
        if ((int64_t)q.k * q.sbk * 2 >= (int64_t(1) << 31)) return false;
    }
    return true;
}

// Whether a product's tiles are dealt to the XCDs one by one (bit 8 of GemmParams::order) instead of in contiguous ranges: a tall product -- at least 9 rows
// of tiles and three times as many as columns, with K in parts twice as many -- whose number of tiles is no multiple of 8.  One by one, a strip of 8 tile rows gives every XCD a row
// of its own, whose panel of the lhs it reads once for all the few columns; ranges read it into two or three L2s.  Us, ranges / one by one: 128 x 128
// tiles with K in parts 19 x 3 of them, K 12800 40.7 / 32.8, 17 x 3, 6400 24.2 / 20.5, 23 x 2, 6400 22.4 / 20.2, 12 x 7, 12800 44.4 / 41.9; 64 x 64 in parts 41 x 2,
// 12800 27.2 / 23.9; 128 x 256 39 x 7, 2368 53.1 / 47.8; 128 x 128 on a deep ring 17 x 3, 4672 29.0 / 27.6.  Less tall ones gain by ranges (11 x 7 of 128 x 128 in parts
// 0.9 of the time, 46 x 19 in one piece 0.91), and so do 256 x 256 tiles (44 x 9, K 4672 0.92) -- but for products with
// next to no contraction whose output's rows are no whole lines: one by one an XCD writes neighbouring tiles of a row at the same time, whose shared lines meet
// in its L2 (bf16, ranges / one by one: 7388 x 9416 x 88 73.4 / 61.3, 7341 x 7208 x 16 57.6 / 45.3, 6692 x 5960 x 88 52.2 / 45.5; a K of 192 no difference).
bool tiles_one_by_one(const GemmParams &p, int bm, bool in_parts, int64_t out_row_bytes) {
    if (p.tiles_m * (int64_t)p.tiles_n % 8 == 0) return false;
    if (bm > 128) return p.k <= 128 && out_row_bytes % 128 != 0;
    return p.tiles_n > 1 && p.tiles_m >= 9 && p.tiles_m / (in_parts ? 2 : 3) >= p.tiles_n;
}

void fill_params(GemmParams &p, const GemmProblem &q, int bm, int bn, bool in_parts = false) {
    p.a = q.a;
    p.b = q.b;
    p.c = q.c;
    p.bias = q.linear ? q.column_bias : q.bias;
    p.linear = q.linear;
    p.bias_float = q.bias_float;
    p.lower = q.lower;
    p.m = q.m;
    p.n = q.n;
    p.k = q.k;
    p.lda = q.sam;
    p.ldb = b_is_transposed(q) ? q.sbn : q.sbk;
    p.ldc = q.scm;
    p.bias_stride_m = q.sim;
    p.bias_stride_n = q.sin;
    p.alpha = q.alpha;
    p.beta = q.beta;
    p.tiles_m = (q.m + bm - 1) / bm;
    p.tiles_n = (q.n + bn - 1) / bn;
    p.order = g_tile_order | (tiles_one_by_one(p, bm, in_parts, q.scm * (q.out_dtype == NINETOOTHED_FLOAT32 ? 4 : 2)) ? 0x100 : 0);
    p.bias_vector = q.bias != nullptr && q.sin == 1 && q.sim % 8 == 0 && ((uintptr_t)q.bias & 15) == 0 && q.n % 8 == 0 && (q.batch == 1 || q.bias_batch % 8 == 0);
    p.c_vector = ((uintptr_t)q.c & 15) == 0 && q.scm % 8 == 0 && q.n % 8 == 0 && (q.batch == 1 || q.c_batch % 8 == 0);
    p.kt_per_split = 0;
    p.out_float = q.out_dtype == NINETOOTHED_FLOAT32;
    p.batch = q.batch;
    p.a_batch = q.a_batch;
    p.b_batch = q.b_batch;
    p.c_batch = q.c_batch;
    p.bias_batch = q.bias_batch;
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int kStages, int kOcc, int kAblate, int kLoad, int kAux, bool kTail, bool kLines>
hipError_t fast_launch_form(const GemmProblem &q, hipStream_t stream) {
    GemmParams p;
    fill_params(p, q, BM, BN);
    const dim3 grid(p.tiles_m * p.tiles_n * q.batch), block(WM * WN * 64);
    const bool f32 = q.out_dtype == NINETOOTHED_FLOAT32, addmm = q.addmm();
    if (b_is_transposed(q)) {
        if (f32) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kPlain, kAblate, kLoad, kAux, true, true, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
        else if (addmm) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kAddmm, kAblate, kLoad, kAux, false, true, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
        else if (q.linear) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kLinear, kAblate, kLoad, kAux, false, true, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
        else gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kPlain, kAblate, kLoad, kAux, false, true, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
    } else {
        if (f32) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kPlain, kAblate, kLoad, kAux, true, false, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
        else if (addmm) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kAddmm, kAblate, kLoad, kAux, false, false, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
        else if (q.linear) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kLinear, kAblate, kLoad, kAux, false, false, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
        else gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kStages, kOcc, kPlain, kAblate, kLoad, kAux, false, false, kTail, false, kLines><<<grid, block, 0, stream>>>(p);
    }
    return hipGetLastError();
}

// Whether rows of the k-contiguous operands are staged by whole cache lines, in a ring of five stages (kLines of the kernel): where some begin inside a
// 128-byte line; of a product with a row-major rhs only from 65 rows on, since its lhs is all that gains (17 x 768 x 11104 12.1 us without, 12.9 with).
// bf16, one k tile after another / by whole lines, us, rhs transposed and not: 128 x 128 tiles 4096 x 1024 x 4088 58.5 / 39.9, 47.1 / 39.5; 1394 x
// 2176 x 3080 41.3 / 30.1, 34.4 / 29.8; 64 x 64 4096 x 1024 x 4088 95.4 / 63.5, 79.5 / 64.3; 300 x 4096 x 1000 10.2 / 8.8, 9.2 / 8.5; 64 x 128 77 x 832 x
// 5576 36.9 / 26.6, 28.8 / 26.3.  Rows that begin with a line gain nothing and wait for a line more: 2048^3 on 64 x 128 23.7 / 27.0, on 64 x 64 27.8 /
// 28.4, fp16 863 x 2368 x 704 on 128 x 128 7.7 / 8.1, 283 x 1016 x 12224 there in parts 24.6 / 25.7.
bool rows_straddle_lines(const GemmProblem &q) {
    const auto inside = [&](const void *data, int64_t pitch, int64_t batch) { return ((uintptr_t)data | (uintptr_t)(pitch * 2) | (uintptr_t)(q.batch > 1 ? batch * 2 : 0)) % 128 != 0; };
    if (b_is_transposed(q)) return inside(q.a, q.sam, q.a_batch) || inside(q.b, q.sbn, q.b_batch);
    return q.m > 64 && inside(q.a, q.sam, q.a_batch);
}

constexpr const char *kLinesNote = "rows by whole lines";  // (of a launch)

// ... and whether that pays: another line has to land before the first step, which short contractions do not make up for.  In one piece from a K of
// 256 on with a transposed rhs and of 768 without, and 5e8 products, of batches, whose matrices begin anywhere in a line too, 1e8 (bf16, us, k tiles / lines:
// 64 x 64 tiles 4096 x 4096 x 72 18.5 / 21.1, 2048 x 1024 x 136 4.7 / 5.0, 1024 x 512 x 520 4.2 / 4.5, 4096 x 1024 x 264 8.8 / 8.4, 11 of 66 x 288 x 760 6.7 / 6.1; not transposed
// 4096 x 1024 x 264 7.9 / 8.3, x 776 15.7 / 14.6; 128 x 128 tiles 4096 x 4096 x 24 13.3 / 15.0, 2048 x 1024 x 392 6.7 / 6.4).  In parts, of a few k tiles each, on 128 x 128 tiles only
// with a transposed rhs, from 8 tiles on where K is at most 9000, from 32 on otherwise (416 x 832 x 3800 16.3 / 15.0, 1024 x 1024 x 16392 55.1 / 50.9, but 256 x
// 512 x 16392 19.3 / 20.9, 166 x 120 x 3488 9.6 / 10.5; not transposed 270 x 232 x 16392 16.5 / 19.3, 1024 x 512 x 8200 22.4 / 23.8), on 64 x 64 from 16 tiles on
// and 64 without (128 x 128 x 8200 9.4 / 10.1, 1024 x 1024 x 8200 38.3 / 34.4).
bool lines_pay(const GemmProblem &q, int bm, int bn, bool in_parts) {
    const bool transposed = b_is_transposed(q);
    if (!in_parts) return q.k >= (transposed ? 256 : 768) && (double)q.batch * q.m * q.n * q.k >= (q.batch > 1 ? 1e8 : 5e8);
    const int64_t tiles = (int64_t)ceil_div(q.m, bm) * ceil_div(q.n, bn);
    return bm == 128 ? transposed && tiles >= (q.k <= 9000 ? 8 : 32) : tiles >= (transposed ? 16 : 64);
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int kStages, int kOcc, int kAblate, int kLoad, int kAux, bool kTail, bool kLines>
hipError_t fast_launch_typed(const GemmProblem &q, hipStream_t stream) {
    if constexpr (kLines)
        if (rows_straddle_lines(q) && lines_pay(q, BM, BN, false)) {
            note_launch_detail(kLinesNote);
            return fast_launch_form<T, BM, BN, BK, WM, WN, 5, kOcc, kAblate, kLoad, kAux, kTail, true>(q, stream);
        }
    return fast_launch_form<T, BM, BN, BK, WM, WN, kStages, kOcc, kAblate, kLoad, kAux, kTail, false>(q, stream);
}

template <int BM, int BN, int BK, int WM, int WN, int kStages, int kOcc, int kAblate = 0, int kLoad = 1, int kAux = 0, bool kTail = false, bool kLines = false>
hipError_t fast_launch(const GemmProblem &q, hipStream_t stream) {
    if (q.dtype == NINETOOTHED_FLOAT16) return fast_launch_typed<half_t, BM, BN, BK, WM, WN, kStages, kOcc, kAblate, kLoad, kAux, kTail, kLines>(q, stream);
    return fast_launch_typed<bf16_t, BM, BN, BK, WM, WN, kStages, kOcc, kAblate, kLoad, kAux, kTail, kLines>(q, stream);
}

// ---- split-K: problems with too few output tiles for 256 CUs (a few rows, or small M x N with a long K) ----
// The k range is cut into parts, each (tile, part) is a workgroup that writes an fp32 tile to scratch
// memory of the stream, and a second kernel sums the parts and applies the epilogue.

// What a k tile costs a workgroup with a CU to itself (`alone`) and the CU per workgroup (`shared`), in microseconds, and the rate at which
// the partial products are written and read (bytes per microsecond), by the tile of the instance.
struct SplitCost {
    int area, resident;  // workgroups per CU
    float alone, shared, rate;
};
constexpr SplitCost kSplitCosts[] = {{64 * 64, 2, 0.234f, 0.214f, 0.8e6f}, {128 * 128, 1, 0.3f, 0.3f, 4.0e6f}, {128 * 256, 2, 0.39f, 0.28f, 5.1e6f}, {256 * 256, 1, 0.29f, 0.29f, 5.8e6f}};

constexpr const SplitCost *split_cost(int bm, int bn) {
    for (const SplitCost &cost : kSplitCosts)
        if (cost.area == bm * bn) return &cost;
    return nullptr;
}

// Number of parts for tiles of bm x bn x bk, 1 = do not split (`scratch_limit`: bytes the partial products may take).
// Of the numbers whose workgroups are all on the chip at once, the one of least expected time -- and two parts of any number of tiles below
// 320 (of 256 x 256 ones, whose parts are the largest, up to 128): more of them than the chip holds run in rounds, which the untuned choice
// leaves alone; the tuner, or a call by the instance's index, takes them.
// Fitted to 59 products of 1 to 3000 rows, 2 to 48 parts: 3 % (64 x 64), 1 % (others) slower than the best number on average; 512
// workgroups whatever the shape were 11 and 10 % slower.  (128 x 128: five products of 100 to 1024 rows, a step 0.22 to 0.46 us with
// the rhs in the caches and in memory; 222 x 2752 x 15040 34.5 us in five parts, 39 in four, 43 in eight, without the summing.)
int split_parts(const GemmProblem &q, int bm, int bn, int bk, int *kt_per_part, int64_t scratch_limit = int64_t(64) << 20) {
    const int64_t tiles = (int64_t)((q.m + bm - 1) / bm) * ((q.n + bn - 1) / bn);
    const int num_kt = (q.k + bk - 1) / bk;
    if (tiles >= 320) return 1;
    const SplitCost *cost = split_cost(bm, bn);
    const int64_t part_bytes = (int64_t)q.m * ((q.n + 7) / 8 * 8) * 4;
    int best = 1;
    float best_time = 0.0f;
    for (int parts = 2; parts <= std::min(256, num_kt / 2); parts += std::max(1, parts / 8)) {  // at least two k tiles each
        const int64_t workgroups = tiles * parts;
        if (parts * part_bytes > scratch_limit || ((parts > 2 || cost->area == 256 * 256) && workgroups > 256 * cost->resident)) break;
        const int per_part = (num_kt + parts - 1) / parts;
        const float time = (float)per_part * std::max(cost->alone, (float)((workgroups + 255) / 256) * cost->shared) + (float)(parts * part_bytes) / cost->rate;
        if (best == 1 || time < best_time) {
            best = parts;
            best_time = time;
        }
    }
    if (best == 1) return 1;
    const int per_part = (num_kt + best - 1) / best;
    if (kt_per_part) *kt_per_part = per_part;
    return (num_kt + per_part - 1) / per_part;                      // every part has at least one k tile
}

template <int BM, int BN, int BK, int kStages>
bool split_accepts(const GemmProblem &q) {
    // the operands, outputs and epilogues of the one-pass instances with tails (the second kernel writes four
    // consecutive elements of C at a time where N, the row pitch and the address of C allow it, else one)
    if (q.batch != 1) return false;
    return fast_accepts<BM, BN, BK, kStages, true>(q) && split_parts(q, BM, BN, BK, nullptr) >= 2;
}

// out[m][n] = epilogue(sum over parts): four consecutive columns per thread.  The parts are [m][pitch] tiles, pitch = N
// rounded up to 8; kVector: N is a multiple of 4 and the rows of C start on 16-byte (fp32) / 8-byte boundaries -- else
// the four values are stored one by one, those inside N.  Bound by the latency of a chain of loads where C is small and the parts are
// many: kGroups threads share the parts of a value (every kGroups-th each, met in LDS) and a thread keeps eight loads in flight.
// The parameters are those of the product (C of them is what is written here).
template <typename T, typename TOut, int kEpilogue, bool kVector, int kGroups>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(const float *parts, int num_parts, GemmParams p) {
    const int m = p.m, n = p.n;
    typedef float float4_t __attribute__((ext_vector_type(4)));
    typedef TOut out4_t __attribute__((ext_vector_type(4)));
    constexpr int kColumns = 256 / kGroups;  // values (of four columns) per workgroup
    __shared__ float4_t sums[kGroups > 1 ? kGroups - 1 : 1][kColumns];
    const int pitch = (n + 7) / 8 * 8;
    const int columns = pitch / 4;
    const int64_t total = (int64_t)m * columns;
    const int slot = threadIdx.x % kColumns, group = threadIdx.x / kColumns;
    const int64_t index = (int64_t)blockIdx.x * kColumns + slot;
    const int row = (int)(index / columns);
    const int col = (int)(index - (int64_t)row * columns) * 4;
    const bool inside = index < total && col < n;
    float4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
    if (inside) {
        const float *src = parts + (int64_t)row * pitch + col;
#pragma unroll 8
        for (int part = group; part < num_parts; part += kGroups) sum += *(const float4_t *)(src + (int64_t)part * m * pitch);
    }
    if constexpr (kGroups > 1) {
        if (group > 0) sums[group - 1][slot] = sum;
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int g = 0; g < kGroups - 1; ++g) sum += sums[g][slot];
    }
    if (!inside) return;
    TOut *c = (TOut *)p.c + (int64_t)row * p.ldc;
    out4_t out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (kEpilogue == kAddmm) {
            // as in the one-pass kernels: the product is rounded to the element type, then combined in fp32
            const float product = Elem<T>::to_float(Elem<T>::from_float(sum[e]));
            const float input = kVector || col + e < n ? Elem<T>::to_float(((const T *)p.bias)[(int64_t)row * p.bias_stride_m + (int64_t)(col + e) * p.bias_stride_n]) : 0.0f;
            out[e] = Elem<T>::from_float(p.beta * input + p.alpha * product);
        } else if constexpr (kEpilogue == kLinear) {
            out[e] = Elem<T>::from_float(linear_value(p, sum[e], kVector || col + e < n ? linear_bias<T>(p, col + e) : 0.0f));
        } else if constexpr (std::is_same<TOut, float>::value) {
            out[e] = sum[e];
        } else {
            out[e] = Elem<T>::from_float(sum[e]);
        }
    }
    if constexpr (kVector) {
        __builtin_nontemporal_store(out, (out4_t *)(c + col));
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col + e < n) c[col + e] = out[e];
    }
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int kStages, int kOcc, bool kLines>
hipError_t split_launch_typed(const GemmProblem &q, hipStream_t stream) {
    static_assert(split_cost(BM, BN) != nullptr, "a cost for the tile");
    int kt_per_part = 0;
    // with a fixed array the part count shrinks until the partial products fit; the call is refused when not even two parts do
    const int parts = q.fixed_scratch != nullptr ? split_parts(q, BM, BN, BK, &kt_per_part, (int64_t)q.fixed_scratch_bytes) : split_parts(q, BM, BN, BK, &kt_per_part);
    if (parts < 2) return (hipError_t)(q.fixed_scratch != nullptr && split_parts(q, BM, BN, BK, nullptr) >= 2 ? NINETOOTHED_SCRATCH_LIMIT : NINETOOTHED_NO_KERNEL);
    const int pitch = (q.n + 7) / 8 * 8;  // of the partial tiles: whole 16-byte chunks, whatever N is
    const size_t scratch_bytes = (size_t)parts * q.m * pitch * sizeof(float);
    // the lock of the workspace registry also serialises host threads that enqueue onto the fixed array
    WorkspaceLease lease(stream);
    float *scratch;
    if (q.fixed_scratch != nullptr) {
        if (scratch_bytes > q.fixed_scratch_bytes) return (hipError_t)NINETOOTHED_SCRATCH_LIMIT;
        scratch = q.fixed_scratch;
    } else {
        scratch = (float *)lease.get(kWorkspaceGemmParts, scratch_bytes);
        if (scratch == nullptr) return (hipError_t)NINETOOTHED_NO_KERNEL;  // no scratch (graph capture, out of memory): the caller takes a one-pass instance
    }
    GemmParams result;  // (the summing kernel's)
    fill_params(result, q, BM, BN, true);
    GemmParams p = result;
    p.c = scratch;
    p.ldc = pitch;
    p.c_vector = 1;  // (the scratch tensor is aligned and its rows hold whole chunks: a chunk that begins inside N is stored whole)
    p.bias = nullptr;
    p.kt_per_split = kt_per_part;
    const dim3 grid(p.tiles_m * p.tiles_n * parts), block(WM * WN * 64);
    const auto launch = [&](auto stages_tag, auto lines_tag) {
        constexpr int kRing = decltype(stages_tag)::value;
        constexpr bool kByLines = decltype(lines_tag)::value;
        if (b_is_transposed(q)) gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kRing, kOcc, kPlain, 0, 1, 0, true, true, true, true, kByLines><<<grid, block, 0, stream>>>(p);
        else gemm_nn_fast_kernel<T, BM, BN, BK, WM, WN, kRing, kOcc, kPlain, 0, 1, 0, true, false, true, true, kByLines><<<grid, block, 0, stream>>>(p);
    };
    const bool by_lines = kLines && rows_straddle_lines(q) && lines_pay(q, BM, BN, true);
    if (by_lines) note_launch_detail(kLinesNote);
    if (by_lines) launch(std::integral_constant<int, kLines ? 5 : kStages>(), std::integral_constant<bool, kLines>());
    else launch(std::integral_constant<int, kStages>(), std::false_type());
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int64_t values = (int64_t)q.m * (pitch / 4);
    const int64_t out_size = q.out_dtype == NINETOOTHED_FLOAT32 ? 4 : 2;
    const bool vector = q.n % 4 == 0 && (q.scm * out_size) % (4 * out_size) == 0 && ((uintptr_t)q.c & (4 * out_size - 1)) == 0;
    const auto reduce = [&](auto vector_tag, auto groups_tag) {
        constexpr bool kVector = decltype(vector_tag)::value;
        constexpr int kGroups = decltype(groups_tag)::value;
        const dim3 reduce_grid((unsigned)((values + 256 / kGroups - 1) / (256 / kGroups)));
        if (q.addmm()) gemm_split_reduce_kernel<T, T, kAddmm, kVector, kGroups><<<reduce_grid, dim3(256), 0, stream>>>(scratch, parts, result);
        else if (q.linear) gemm_split_reduce_kernel<T, T, kLinear, kVector, kGroups><<<reduce_grid, dim3(256), 0, stream>>>(scratch, parts, result);
        else if (q.out_dtype == NINETOOTHED_FLOAT32) gemm_split_reduce_kernel<T, float, kPlain, kVector, kGroups><<<reduce_grid, dim3(256), 0, stream>>>(scratch, parts, result);
        else gemm_split_reduce_kernel<T, T, kPlain, kVector, kGroups><<<reduce_grid, dim3(256), 0, stream>>>(scratch, parts, result);
    };
    const auto reduce_in_groups = [&](auto vector_tag) {
        // one thread per value where that fills the chip, or the parts are few; else a value's parts over four or sixteen threads
        if (parts < 8 || values >= 256 * 1024) reduce(vector_tag, std::integral_constant<int, 1>());
        else if (parts < 32 || values >= 64 * 1024) reduce(vector_tag, std::integral_constant<int, 4>());
        else reduce(vector_tag, std::integral_constant<int, 16>());
    };
    if (vector) reduce_in_groups(std::true_type());
    else reduce_in_groups(std::false_type());
    return hipGetLastError();
}

template <int BM, int BN, int BK, int WM, int WN, int kStages, int kOcc, bool kLines>
hipError_t split_launch(const GemmProblem &q, hipStream_t stream) {
    if (q.dtype == NINETOOTHED_FLOAT16) return split_launch_typed<half_t, BM, BN, BK, WM, WN, kStages, kOcc, kLines>(q, stream);
    return split_launch_typed<bf16_t, BM, BN, BK, WM, WN, kStages, kOcc, kLines>(q, stream);
}

// ---- skinny products: at most 64 rows against a k-contiguous rhs, the k range over the waves of a workgroup ----
bool skinny_accepts(const GemmProblem &q) { return q.m <= 64 && q.batch == 1 && b_is_transposed(q) && fast_accepts<64, 64, 64, 4, true>(q); }

template <typename T, int MB, int NB, int kWaves, int kStages>
hipError_t skinny_launch_rows(const GemmProblem &q, hipStream_t stream) {
    GemmParams p;
    fill_params(p, q, MB * 16, NB * 16);
    // a B that the 256 MiB Infinity Cache cannot hold beside a program's other tensors is streamed past the caches (16 x 50256 x
    // 4096 71 us, 79 otherwise); a smaller one may still lie there from its last use (16 x 4096 x 2048
    // 5.1 us, 5.6 past the caches; 24 x 8192 x 4096 12.8 against 15.9)
    if ((int64_t)q.n * q.sbn * 2 > (int64_t)128 << 20) gemm_skinny_kernel<T, MB, NB, kWaves, kStages, 2><<<dim3(p.tiles_n), dim3(kWaves * 64), 0, stream>>>(p);
    else gemm_skinny_kernel<T, MB, NB, kWaves, kStages, 0><<<dim3(p.tiles_n), dim3(kWaves * 64), 0, stream>>>(p);
    return hipGetLastError();
}

template <typename T, int NB>
hipError_t skinny_launch_typed(const GemmProblem &q, hipStream_t stream) {
    // (16 columns per workgroup: four waves with rings of four stages, 16-40 KiB each; 32 columns: with more rows than
    // 16 two waves, so that more than one workgroup fits the LDS of a CU -- 32 x 50256 x 4096 82 us with two, 95 with four)
    if constexpr (NB == 1) {
        if (q.m <= 16) return skinny_launch_rows<T, 1, NB, 4, 4>(q, stream);
        if (q.m <= 32) return skinny_launch_rows<T, 2, NB, 4, 4>(q, stream);
        if (q.m <= 48) return skinny_launch_rows<T, 3, NB, 4, 4>(q, stream);
        return skinny_launch_rows<T, 4, NB, 4, 4>(q, stream);
    } else {
        if (q.m <= 16) return skinny_launch_rows<T, 1, NB, 4, 3>(q, stream);
        if (q.m <= 32) return skinny_launch_rows<T, 2, NB, 2, 3>(q, stream);
        if (q.m <= 48) return skinny_launch_rows<T, 3, NB, 2, 3>(q, stream);
        return skinny_launch_rows<T, 4, NB, 2, 3>(q, stream);
    }
}

template <int NB>
hipError_t skinny_launch(const GemmProblem &q, hipStream_t stream) {
    return q.dtype == NINETOOTHED_FLOAT16 ? skinny_launch_typed<half_t, NB>(q, stream) : skinny_launch_typed<bf16_t, NB>(q, stream);
}

bool generic_accepts(const GemmProblem &q) {
    if (q.batch < 1 || q.batch > 65535) return false;  // (the batch is the grid's y extent)
    if (q.dtype == NINETOOTHED_FLOAT8_E5M2 && q.batch != 1) return false;
    if (q.dtype == NINETOOTHED_FLOAT8_E5M2)  // widened to fp16; addmm rounds its product to fp16, so it writes fp16
        return (q.out_dtype == NINETOOTHED_FLOAT16 || (q.out_dtype == NINETOOTHED_FLOAT32 && !q.addmm())) && q.m >= 0 && q.n >= 0 && q.k >= 0;
    if (q.dtype != NINETOOTHED_FLOAT16 && q.dtype != NINETOOTHED_BFLOAT16 && q.dtype != NINETOOTHED_FLOAT32) return false;
    if (q.out_dtype != q.dtype && q.out_dtype != NINETOOTHED_FLOAT32) return false;
    return q.m >= 0 && q.n >= 0 && q.k >= 0;
}

// out = epilogue(sum over the parts of the k range), any output strides; fp32 throughout (an fp32 addmm does not round its product)
__global__ __launch_bounds__(256) void gemm_generic_reduce_kernel(const float *parts, int num_parts, int m, int n, float *c, int64_t scm, int64_t scn, const float *bias,
                                                                 int64_t bias_stride_m, int64_t bias_stride_n, float alpha, float beta) {
    const int64_t total = (int64_t)m * n;
    for (int64_t index = (int64_t)blockIdx.x * 256 + threadIdx.x; index < total; index += (int64_t)gridDim.x * 256) {
        float sum = parts[index];
        for (int part = 1; part < num_parts; ++part) sum += parts[index + (int64_t)part * total];
        const int row = (int)(index / n), col = (int)(index - (int64_t)row * n);
        if (bias != nullptr) sum = beta * bias[(int64_t)row * bias_stride_m + (int64_t)col * bias_stride_n] + alpha * sum;
        c[(int64_t)row * scm + (int64_t)col * scn] = sum;
    }
}

// fp32 products with too few 128 x 128 tiles for the chip: parts of the k range as the grid's y extent, each writing an
// fp32 tile to scratch memory of the stream, then the sum (512^3 50 -> 23 us, 1024^3 96 -> 41, [128, 4096] x [4096, 128]
// 347 -> 28, [64, 8192] x [8192, 64] 776 -> 38).  NINETOOTHED_NO_KERNEL: not worth it, or no scratch -- the caller runs the product in one pass.
hipError_t generic_launch_in_parts(const GemmProblem &q, hipStream_t stream) {
    const int64_t tiles = (int64_t)ceil_div(q.m, kGenBM) * ceil_div(q.n, kGenBN);
    const int num_kt = ceil_div(q.k, kGenBK);
    if (q.batch != 1 || q.hinted || q.fixed_scratch != nullptr || tiles == 0 || tiles >= 192) return (hipError_t)NINETOOTHED_NO_KERNEL;
    int64_t parts = std::min<int64_t>({(512 + tiles - 1) / tiles, num_kt / 4, 256});
    while (parts >= 2 && parts * q.m * q.n * 4 > (int64_t(64) << 20)) --parts;
    if (parts < 2) return (hipError_t)NINETOOTHED_NO_KERNEL;
    const int kt_per_part = (int)((num_kt + parts - 1) / parts);
    parts = (num_kt + kt_per_part - 1) / kt_per_part;  // every part has at least one k tile
    WorkspaceLease lease(stream);
    float *scratch = (float *)lease.get(kWorkspaceGemmParts, (size_t)parts * q.m * q.n * sizeof(float));
    if (scratch == nullptr) return (hipError_t)NINETOOTHED_NO_KERNEL;
    StridedProblem<float, float> prob;
    prob.m = q.m;
    prob.n = q.n;
    prob.k = q.k;
    prob.a = (const float *)q.a;
    prob.b = (const float *)q.b;
    prob.c = scratch;
    prob.bias = nullptr;
    prob.sam = q.sam;
    prob.sak = q.sak;
    prob.sbk = q.sbk;
    prob.sbn = q.sbn;
    prob.scm = q.n;
    prob.scn = 1;
    prob.sbm_ = prob.sbn_ = 0;
    prob.alpha = 1.0f;
    prob.beta = 0.0f;
    prob.a_batch = prob.b_batch = prob.bias_batch = 0;
    prob.c_batch = (int64_t)q.m * q.n;
    prob.k_chunk = kt_per_part * kGenBK;
    note_launch(kLaunchGemm, 0, "128x128x32 waves 2x2 any-stride, k range in parts, then gemm_generic_reduce_kernel");
    gemm_generic_kernel<StridedProblem<float, float>><<<dim3((unsigned)tiles, (unsigned)parts), dim3(kGenThreads), 0, stream>>>(prob);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int64_t total = (int64_t)q.m * q.n;
    gemm_generic_reduce_kernel<<<dim3((unsigned)std::min<int64_t>((total + 255) / 256, 256 * 8)), dim3(256), 0, stream>>>(
        scratch, (int)parts, q.m, q.n, (float *)q.c, q.scm, q.scn, (const float *)q.bias, q.sim, q.sin, q.alpha, q.beta);
    return hipGetLastError();
}

template <typename T, typename TOut>
hipError_t generic_launch_typed(const GemmProblem &q, hipStream_t stream) {
    if constexpr (std::is_same<T, float>::value) {
        const hipError_t in_parts = generic_launch_in_parts(q, stream);
        if ((int)in_parts != NINETOOTHED_NO_KERNEL) return in_parts;
    }
    StridedProblem<T, TOut> prob;
    prob.k_chunk = 0;
    prob.m = q.m;
    prob.n = q.n;
    prob.k = q.k;
    prob.a = (const T *)q.a;
    prob.b = (const T *)q.b;
    prob.c = (TOut *)q.c;
    prob.bias = (const T *)q.bias;
    prob.sam = q.sam;
    prob.sak = q.sak;
    prob.sbk = q.sbk;
    prob.sbn = q.sbn;
    prob.scm = q.scm;
    prob.scn = q.scn;
    prob.sbm_ = q.sim;
    prob.sbn_ = q.sin;
    prob.alpha = q.alpha;
    prob.beta = q.beta;
    prob.a_batch = q.a_batch;
    prob.b_batch = q.b_batch;
    prob.c_batch = q.c_batch;
    prob.bias_batch = q.bias_batch;
    const int64_t tiles = (int64_t)ceil_div(q.m, kGenBM) * ceil_div(q.n, kGenBN);
    if (tiles == 0) return hipSuccess;  // empty launch is legal
    gemm_generic_kernel<StridedProblem<T, TOut>><<<dim3((unsigned)tiles, (unsigned)q.batch), dim3(kGenThreads), 0, stream>>>(prob);
    return hipGetLastError();
}

template <typename TOut>
hipError_t fp8_launch_typed(const GemmProblem &q, hipStream_t stream) {
    Fp8E5m2Problem<TOut> prob;
    prob.m = q.m;
    prob.n = q.n;
    prob.k = q.k;
    prob.a = (const uint8_t *)q.a;
    prob.b = (const uint8_t *)q.b;
    prob.c = (TOut *)q.c;
    prob.sam = q.sam;
    prob.sak = q.sak;
    prob.sbk = q.sbk;
    prob.sbn = q.sbn;
    prob.scm = q.scm;
    prob.scn = q.scn;
    prob.bias = (const uint8_t *)q.bias;
    prob.sbm_ = q.sim;
    prob.sbn_ = q.sin;
    prob.alpha = q.alpha;
    prob.beta = q.beta;
    const int64_t tiles = (int64_t)ceil_div(q.m, kGenBM) * ceil_div(q.n, kGenBN);
    if (tiles == 0) return hipSuccess;
    gemm_generic_kernel<Fp8E5m2Problem<TOut>><<<dim3((unsigned)tiles), dim3(kGenThreads), 0, stream>>>(prob);
    return hipGetLastError();
}

hipError_t generic_launch(const GemmProblem &q, hipStream_t stream) {
    const bool f32out = q.out_dtype == NINETOOTHED_FLOAT32;
    if (q.dtype == NINETOOTHED_FLOAT8_E5M2) return f32out ? fp8_launch_typed<float>(q, stream) : fp8_launch_typed<half_t>(q, stream);
    if (q.dtype == NINETOOTHED_FLOAT32) return generic_launch_typed<float, float>(q, stream);
    if (q.dtype == NINETOOTHED_FLOAT16)
        return f32out ? generic_launch_typed<half_t, float>(q, stream) : generic_launch_typed<half_t, half_t>(q, stream);
    return f32out ? generic_launch_typed<bf16_t, float>(q, stream) : generic_launch_typed<bf16_t, bf16_t>(q, stream);
}

int heuristic_choice(const GemmProblem &q, int bm, int bn, int bk);
template <bool kColumns> bool cut_accepts(const GemmProblem &q);
template <bool kColumns> hipError_t cut_launch(const GemmProblem &q, hipStream_t stream);

// BM, BN, BK, wave grid WM x WN, LDS stages, waves per SIMD the register budget allows
#define NT_FAST_INSTANCE(BM, BN, BK, WM, WN, ST, OCC) \
    {#BM "x" #BN "x" #BK " waves " #WM "x" #WN " stages " #ST " lds-direct", BM, BN, BK, fast_accepts<BM, BN, BK, ST>, fast_launch<BM, BN, BK, WM, WN, ST, OCC>}

// the same kernels with partial last tiles along N and K (both multiples of 8); LINES: with the form for rows that begin inside cache lines
#define NT_TAIL_INSTANCE(BM, BN, BK, WM, WN, ST, OCC, LINES) \
    {#BM "x" #BN "x" #BK " waves " #WM "x" #WN " stages " #ST " lds-direct tails", BM, BN, BK, fast_accepts<BM, BN, BK, ST, true>, fast_launch<BM, BN, BK, WM, WN, ST, OCC, 0, 1, 0, true, LINES>}

#define NT_SPLIT_INSTANCE(BM, BN, BK, WM, WN, ST, OCC, LINES) \
    {#BM "x" #BN "x" #BK " waves " #WM "x" #WN " stages " #ST " lds-direct tails split-k", BM, BN, BK, split_accepts<BM, BN, BK, ST>, split_launch<BM, BN, BK, WM, WN, ST, OCC, LINES>}

// positions in kInstances (the tuning cache and the heuristics refer to instances by position)
enum InstanceIndex {
    kAnyStride, k256x256x32, k256x256x64, k128x128x64, k64x64x64, k128x256x32,
    kTail256x256x32, kTail128x256x32, kTail128x128x64, kTail64x64x64, kSplit64x64x64, kSplit128x128x64,
    kSplit128x256x32, kSplit256x256x32, kSkinny16, kSkinny32, kDeep128x128x64, kDeep64x64x128, kDeep64x128x64,
    kCutColumns, kCutRows,
};

const GemmInstance kInstances[] = {
    {"128x128x32 waves 2x2 any-stride", kGenBM, kGenBN, kGenBK, generic_accepts, generic_launch},
    NT_FAST_INSTANCE(256, 256, 32, 2, 4, 5, 2),  // 5 x 32 KiB: the whole LDS of a CU
    NT_FAST_INSTANCE(256, 256, 64, 2, 4, 2, 2),
    NT_FAST_INSTANCE(128, 128, 64, 2, 2, 2, 2),
    NT_FAST_INSTANCE(64, 64, 64, 2, 2, 4, 2),  // small problems: more, smaller tiles to occupy the CUs
    NT_FAST_INSTANCE(128, 256, 32, 1, 4, 3, 2),  // two workgroups per CU: mid-size problems
    NT_TAIL_INSTANCE(256, 256, 32, 2, 4, 5, 2, false),
    NT_TAIL_INSTANCE(128, 256, 32, 1, 4, 3, 2, false),
    NT_TAIL_INSTANCE(128, 128, 64, 2, 2, 2, 2, false),
    NT_TAIL_INSTANCE(64, 64, 64, 2, 2, 4, 2, true),
    NT_SPLIT_INSTANCE(64, 64, 64, 2, 2, 4, 2, true),
    NT_SPLIT_INSTANCE(128, 128, 64, 2, 4, 4, 2, true),  // (two stages, two workgroups per CU: 222 x 2752 x 15040 43.3 us, here 39.4; 283 x 1016 x 12224 26.8, 23.3; 256 x 8192 x 8192 59.9, 52.2)
    NT_SPLIT_INSTANCE(128, 256, 32, 1, 4, 3, 2, false),  // a few hundred rows against a wide rhs: 64 to 160 large tiles
    NT_SPLIT_INSTANCE(256, 256, 32, 2, 4, 5, 2, false),
    {"64x16x64 skinny, split-k over the waves of a workgroup", 64, 16, 64, skinny_accepts, skinny_launch<1>},
    {"64x32x64 skinny, split-k over the waves of a workgroup", 64, 32, 64, skinny_accepts, skinny_launch<2>},
    // One workgroup per CU with most of its LDS: three or four fills of 16 to 32 KiB in flight instead of one, for products whose
    // tiles the chip holds all at once, so that nothing else covers the latency of a fill.
    NT_TAIL_INSTANCE(128, 128, 64, 2, 4, 4, 2, true),
    NT_TAIL_INSTANCE(64, 64, 128, 2, 2, 4, 1, false),
    NT_TAIL_INSTANCE(64, 128, 64, 2, 4, 5, 2, true),
    {"256x256x32 for whole rounds of the chip, the columns left on their own (smaller tiles or split-k)", 256, 256, 32, cut_accepts<true>, cut_launch<true>},
    {"256x256x32 for whole rounds of the chip, the rows left on their own (smaller tiles or split-k)", 256, 256, 32, cut_accepts<false>, cut_launch<false>},
#ifdef NT_GEMM_ABLATION
#define NT_LOAD_INSTANCE(BM, BN, BK, WM, WN, ST, OCC, LD, AUX) \
    {#BM "x" #BN "x" #BK " waves " #WM "x" #WN " stages " #ST " load " #LD " aux " #AUX, BM, BN, BK, fast_accepts<BM, BN, BK, ST>, fast_launch<BM, BN, BK, WM, WN, ST, OCC, 0, LD, AUX>}
#define NT_ABLATED_INSTANCE(BM, BN, BK, WM, WN, ST, OCC, AB) \
    {#BM "x" #BN "x" #BK " waves " #WM "x" #WN " stages " #ST " ABLATED " #AB " (wrong results)", BM, BN, BK, fast_accepts<BM, BN, BK, ST>, fast_launch<BM, BN, BK, WM, WN, ST, OCC, AB>}
    NT_LOAD_INSTANCE(256, 256, 32, 2, 4, 4, 2, 1, 0),
    NT_LOAD_INSTANCE(256, 256, 32, 2, 2, 4, 1, 1, 0),
    NT_LOAD_INSTANCE(256, 256, 32, 2, 2, 5, 1, 1, 0),
    NT_LOAD_INSTANCE(256, 256, 64, 2, 2, 2, 1, 1, 0),
    NT_LOAD_INSTANCE(128, 256, 32, 1, 4, 3, 2, 1, 0),
    NT_ABLATED_INSTANCE(256, 256, 32, 2, 4, 4, 2, 1),
    NT_ABLATED_INSTANCE(256, 256, 32, 2, 4, 4, 2, 2),
    NT_ABLATED_INSTANCE(256, 256, 32, 2, 4, 4, 2, 3),
#endif
};
constexpr int kNumInstances = sizeof(kInstances) / sizeof(kInstances[0]);
static_assert(kNumInstances > kCutRows, "InstanceIndex names the first instances of the table");

inline bool is_split(int instance) { return instance >= kSplit64x64x64 && instance <= kSplit256x256x32; }
inline bool is_cut(int instance) { return instance == kCutColumns || instance == kCutRows; }

// choices read from a tuning file: an instance index counts only together with the block sizes saved next to it
bool gemm_choice_known(int index, const int *extra, int extras) {
    return index >= 0 && index < kNumInstances && extras == 3 && extra[0] == kInstances[index].bm && extra[1] == kInstances[index].bn &&
           extra[2] == kInstances[index].bk;
}
const bool g_gemm_check_registered = tune_register_check(kTuneGemm, gemm_choice_known);

// ---- tuned choices: (dtype, output dtype, M, N, K, addmm, rhs layout) -> instance ----
void tune_values(const GemmProblem &q, int (&values)[7]) {
    int layout = b_is_transposed(q) ? 1 : (q.sbn == 1 ? 0 : 2);  // rhs row-major, transposed, other strides
    // + 4: operands that the direct-to-LDS instances cannot read in place (they run on dense copies, whose own
    // problem -- same sizes when K is a multiple of 8 -- must not share this one's entry)
    const bool in_place = q.sak == 1 && q.sam % 8 == 0 && q.k % 8 == 0 && (((uintptr_t)q.a | (uintptr_t)q.b) & 15) == 0 &&
                          (b_is_transposed(q) ? q.sbn % 8 == 0 : (q.sbn == 1 && q.sbk % 8 == 0 && q.n % 8 == 0));
    if (!in_place && (q.dtype == NINETOOTHED_FLOAT16 || q.dtype == NINETOOTHED_BFLOAT16)) layout += 4;
    const int v[7] = {q.dtype, q.out_dtype, q.m, q.n, q.k, q.addmm() ? 1 : 0, layout};
    for (int i = 0; i < 7; ++i) values[i] = v[i];
}

int lookup_tuned(const GemmProblem &q) {
    int values[7];
    tune_values(q, values);
    const int choice = tune_lookup(kTuneGemm, values, 7);
    return choice >= 0 && choice < kNumInstances ? choice : -1;
}

// The skinny instance that a product runs on if nothing is recorded for it, or -1.  The lines lie where the tile instances win
// with B in the Infinity Cache (us, tiles / 16 columns /
// 32 columns): m = 16: 4096 x 4096 13.3 / 8.0 / 10.8; 8192 x 4096 15.6 / 12.3 / 11.8; 8192 x 8192 32.5 / 24.1 / 43.5; 16384 x 4096 30.9 /
// 25.2 / 21.9; 12288 x 2048 10.5 / 11.3 / 11.4; m = 40: 2048 x 2048 6.3 / 5.8 / 8.0; 2048 x 512 3.9 / 4.4 / 4.5; 6144 x 4096 17.0 / 16.5 /
// 13.8; 12288 x 4096 25.9 / 34.3 / 28.0; m = 64: 4096 x 2048 9.8 / 8.8 / 9.3; 2048 x 1024 4.5 / 5.2 / 5.8; 4096 x 8192 19.4 / 24.0 / 38.1.
int skinny_choice(const GemmProblem &q) {
    if (!kInstances[kSkinny16].accepts(q)) return -1;
    const bool long_k = q.k > 4096;
    if (q.m <= 32) {
        if (q.n <= 4096 || long_k) return kSkinny16;
        return q.n <= 8192 || q.k >= 4096 ? (int)kSkinny32 : -1;
    }
    if (q.k < (q.m <= 48 ? 1024 : 2048)) return -1;
    if (q.n <= 4096) return q.m <= 48 || !long_k || q.n <= 1024 ? (int)kSkinny16 : -1;
    return q.n <= 8192 && q.k > 2048 && !long_k ? (int)kSkinny32 : -1;
}

// ---- tiles over whole rounds of the chip ----
// 336 tiles of 256 x 256 on 256 CUs take two rounds, the second with 80 CUs at work.  The columns (or rows) of tiles that fill whole
// rounds run in one launch, what is left as a product of its own before it: K in parts where it has few tiles, else 128 x 128 tiles on a deep ring,
// of which up to two rounds (half a round of 256 x 256 tiles left, 128) still take less time than another round of large ones.  Both launches read one operand whole: the
// smaller one (rows cut off 1500 x 14336 x 4096 read its rhs of 117 MB twice: 168 us with inputs that come from memory, 144 with them in the caches).
// One launch of 256 x 256 tiles / this, bf16, us, sustained with changing inputs: 1500 x 14336 x 4096 (84 tiles left) 169 / 156, 4608 x 4608 x 4096 (72) 153 /
// 148, 1314 x 15104 x 13688 (102) 815 / 667, 1571 x 12672 x 1128 (98) 59.2 / 59.4; single products: 2079 x 9088 x 3264 (72) 132 / 104, 1153 x
// 14208 x 12736 (25) 483 / 354, 4635 x 4736 x 12544 (114) 467 / 432, 2470 x 9536 x 1280 (130) 57.7 / 55.8; more left: 2311 x 11328 x 3136 (200) 130 / 139.
// Of a short K, 2967 x 7872 x 512 (120) 31.9 / 28.9, but 2058 x 7680 x 512 (18) has 19.3 on 128 x 256 tiles against 22, which only the tuner knows.
template <bool kColumns>
int64_t cut_whole(const GemmProblem &q, int64_t units) {  // columns (rows) of 256 x 256 tiles that fill whole rounds
    const int64_t along = ceil_div(kColumns ? q.n : q.m, 256), across = ceil_div(kColumns ? q.m : q.n, 256);
    return along * across / units * units / across;
}

template <bool kColumns>
void cut_problem(const GemmProblem &q, int64_t whole_tiles, GemmProblem &whole, GemmProblem &left) {
    const int64_t size = 2, out_size = q.out_dtype == NINETOOTHED_FLOAT32 ? 4 : 2;
    const int64_t at = whole_tiles * 256;
    whole = left = q;
    if (kColumns) {
        whole.n = (int)at;
        left.n = q.n - whole.n;
        left.b = (const char *)q.b + at * q.sbn * size;
        left.c = (char *)q.c + at * q.scn * out_size;
        if (q.bias != nullptr) left.bias = (const char *)q.bias + at * q.sin * size;
        if (q.column_bias != nullptr) left.column_bias = (const char *)q.column_bias + at * q.sin * (q.bias_float ? 4 : size);
    } else {
        whole.m = (int)at;
        left.m = q.m - whole.m;
        left.a = (const char *)q.a + at * q.sam * size;
        left.c = (char *)q.c + at * q.scm * out_size;
        if (q.bias != nullptr) left.bias = (const char *)q.bias + at * q.sim * size;
    }
}

template <bool kColumns>
bool cut_accepts(const GemmProblem &q) {
    if ((q.dtype != NINETOOTHED_FLOAT16 && q.dtype != NINETOOTHED_BFLOAT16) || q.batch != 1 || q.hinted || q.fixed_scratch != nullptr || q.m <= 0 || q.n <= 0) return false;
    const int64_t along = ceil_div(kColumns ? q.n : q.m, 256), across = ceil_div(kColumns ? q.m : q.n, 256), tiles = along * across;
    // (asking for the number of compute units takes longer than the rest of a small product's choice: no part has as few as 16)
    if (kColumns != (q.m <= q.n) || q.k < 512 || tiles <= 16) return false;
    const int64_t units = compute_units();
    if (units <= 0 || tiles <= units || tiles % units == 0 || tiles > 4 * units + units / 2) return false;  // (what a round costs shrinks to the spread between runs)
    const int64_t whole = cut_whole<kColumns>(q, units);
    if (whole < 1 || 2 * (along - whole) * across > units) return false;
    GemmProblem top, left;
    cut_problem<kColumns>(q, whole, top, left);
    return kInstances[kTail256x256x32].accepts(top) && kInstances[kDeep128x128x64].accepts(left);
}

template <bool kColumns>
hipError_t cut_launch(const GemmProblem &q, hipStream_t stream) {
    const int64_t units = std::max(1, compute_units());
    GemmProblem whole, left;
    cut_problem<kColumns>(q, cut_whole<kColumns>(q, units), whole, left);
    int rest = (int64_t)ceil_div(left.m, 128) * ceil_div(left.n, 128) <= units ? heuristic_choice(left, 0, 0, 0) : (int)kDeep128x128x64;
    if (rest <= kAnyStride || !kInstances[rest].accepts(left)) rest = kDeep128x128x64;
    hipError_t result = kInstances[rest].launch(left, stream);  // (first: a split-K instance may find no scratch memory)
    if ((int)result == NINETOOTHED_NO_KERNEL && is_split(rest)) {
        rest = kDeep128x128x64;
        result = kInstances[rest].launch(left, stream);
    }
    if (result != hipSuccess) return result;
    note_launch_detail(kInstances[rest].name);
    return kInstances[kInstances[k256x256x32].accepts(whole) ? k256x256x32 : kTail256x256x32].launch(whole, stream);
}

// Untuned choice: the largest direct-to-LDS tile that still gives every CU a
// tile (256 CUs), falling back to smaller tiles, then to the any-stride kernel.
int heuristic_choice(const GemmProblem &q, int bm, int bn, int bk) {
    if (bm > 0 && bn > 0) {  // caller fixed the blocks: nearest accepting instance
        int best = -1;
        long best_d = 0;
        for (int i = 0; i < kNumInstances; ++i) {
            if (!kInstances[i].accepts(q)) continue;
            long d = labs(kInstances[i].bm - bm) + labs(kInstances[i].bn - bn) + (bk > 0 ? labs(kInstances[i].bk - bk) : 0);
            if (best < 0 || d < best_d) {
                best = i;
                best_d = d;
            }
        }
        return best;
    }
    // untuned preference (measured on square problems): 256x256 tiles from 256 tiles up,
    // 128x256 from 128 tiles up, 128x128 from 256 tiles up, else the smallest tile that divides
    struct Rule { int instance; int64_t min_tiles; };
    // too few tiles for the chip: split K (64-row tiles for up to 64 rows, else 128 x 128)
    // (64 x 64 tiles of the product: where they fill the chip, a skinny product runs on them in one pass -- 256 x 4096 x 4096
    // 19 us against 27 with K in parts of 128 x 128 tiles, 128 x 4096 x 14336 33 against 42 -- and tiles that the product
    // fills to less than half along M or N are passed over: 64 x 4096 x 128256 259 us on 256 x 256 tiles, 220 on 64 x 64)
    if (const int skinny = skinny_choice(q); skinny >= 0) return skinny;
    const int64_t tiles_64 = (int64_t)((q.m + 63) / 64) * ((q.n + 63) / 64);
    const bool small_tiles_fill_the_chip = q.batch == 1 && tiles_64 >= 256 && kInstances[kTail64x64x64].accepts(q);
    const auto few_tiles = [&](int instance) {
        const GemmInstance &inst = kInstances[instance];
        // (with a short K the second kernel costs more than the idle CUs: 512^3 8 us split, 5 in one pass; of up to 64 rows 33 x 832 x 2088 9.1 and
        // 7.4, but 14 x 1688 x 2528 7.3 and 11.4, 9 x 136 x 2640 7.3 and 8.7)
        const int64_t tiles = (int64_t)((q.m + inst.bm - 1) / inst.bm) * ((q.n + inst.bn - 1) / inst.bn);
        return q.batch == 1 && !small_tiles_fill_the_chip && q.k >= (q.m <= 64 ? 2304 : 2048) && tiles < 192 && 2 * tiles <= 256 * split_cost(inst.bm, inst.bn)->resident &&
               inst.accepts(q);
    };
    if (q.m <= 64 && few_tiles(kSplit64x64x64)) return kSplit64x64x64;
    if (few_tiles(kSplit128x128x64)) return kSplit128x128x64;
    if (few_tiles(kSplit64x64x64)) return kSplit64x64x64;
    // All tiles on the chip at once, one per CU: the deep ring of the smallest tiles of which that holds (bf16, us on the GPU, the best of the other
    // instances / this): 64 x 64 x 128 512 x 512 x 2048 10.4 / 9.2, 130 x 4096 x 4096 19.2 / 15.8, 1000 x 1000 x 16384 80.5 / 58.2; 64 x 128 x 64
    // 1024 x 2048 x 2048 15.2 / 12.9, 70 x 14336 x 2048 16.6 / 15.3; 128 x 128 x 64 2048 x 2048 x 4096 47.2 / 32.1, 1500 x 2048 x 512 10.1 / 7.3.
    // Where the next smaller tiles fit too, or a ring of them would be filled but a few times, the larger ones only leave more CUs idle: 276 x 128
    // x 384 3.9 on 64 x 64 x 64, 4.7 on 64 x 128, 5.7 on 128 x 128; 720 x 448 x 832 4.8, 5.4 on 64 x 64 x 128, 6.1 on 64 x 128; 34 x 2944 x 1792 6.2,
    // 6.9; 361 x 776 x 1920 9.8, 8.6.  (660 products: where the limits are, 0.99 of the time of 64 x 64 x 64 below 257 tiles of that size.)
    // More tiles: 384 of 128 x 128, 700 x 8192 x 2048 35.7 / 34.4, but 1024 of them with a K of 256 17.3 / 18.0, so that the rules below keep those.
    struct DeepRule { int instance, min_k, min_tiles; };
    for (const DeepRule &rule : {DeepRule{kDeep64x64x128, 1920, 48}, DeepRule{kDeep64x128x64, 320, 1}, DeepRule{kDeep128x128x64, 256, 1}}) {
        const GemmInstance &inst = kInstances[rule.instance];
        const int64_t tiles = (int64_t)((q.m + inst.bm - 1) / inst.bm) * ((q.n + inst.bn - 1) / inst.bn) * q.batch;
        if (tiles > 256) continue;
        if (q.k >= rule.min_k && tiles >= rule.min_tiles && inst.accepts(q)) return rule.instance;
        break;
    }
    for (int cut : {(int)kCutColumns, (int)kCutRows})  // (the one of the longer dimension)
        if (kInstances[cut].accepts(q)) return cut;
    // (an instance with tails accepts what its plain form accepts, so it comes right after it: a partial
    // last tile costs less than a smaller tile everywhere)
    const Rule rules[] = {{k256x256x32, 256}, {k256x256x64, 256}, {kTail256x256x32, 256}, {k128x256x32, 128}, {kTail128x256x32, 128},
                          {k128x128x64, 256}, {kTail128x128x64, 256}, {k64x64x64, 1}, {kTail64x64x64, 1}, {k128x128x64, 1}, {kTail128x128x64, 1},
                          {k128x256x32, 1}, {kTail128x256x32, 1}, {k256x256x64, 1}, {k256x256x32, 1}, {kTail256x256x32, 1}};
    for (const Rule &rule : rules) {
        const GemmInstance &inst = kInstances[rule.instance];
        if (!inst.accepts(q)) continue;
        const int64_t per_matrix = (int64_t)((q.m + inst.bm - 1) / inst.bm) * ((q.n + inst.bn - 1) / inst.bn);
        // (a batch of small matrices reaches any number of tiles: a tile that such a matrix fills to less than
        // 60 % is left to the rules of the second pass, which start from the small tiles -- unless 64 x 64 tiles
        // would be as empty: 197 x 197 fills 59 % of one 256 x 256 tile and 59 % of sixteen 64 x 64 ones)
        if (small_tiles_fill_the_chip && (inst.bm > 64 || inst.bn > 64) &&
            ((int64_t)q.m * 2 < (int64_t)((q.m + inst.bm - 1) / inst.bm) * inst.bm || (int64_t)q.n * 2 < (int64_t)((q.n + inst.bn - 1) / inst.bn) * inst.bn))
            continue;
        const int64_t small_tiles = tiles_64 * 64 * 64;
        if (q.batch > 1 && rule.min_tiles > 1 && (int64_t)q.m * q.n * 5 < per_matrix * inst.bm * inst.bn * 3 && per_matrix * inst.bm * inst.bn * 9 > small_tiles * 10) continue;
        if (per_matrix * q.batch >= rule.min_tiles) return rule.instance;
    }
    return kInstances[kAnyStride].accepts(q) ? kAnyStride : -1;
}

bool read_matrix(const NineToothedTensor &t, uint64_t &d0, uint64_t &d1, int64_t &s0, int64_t &s1) {
    if (t.shape == nullptr || t.strides == nullptr) return false;
    d0 = t.shape[0];
    d1 = t.shape[1];
    s0 = t.strides[0];
    s1 = t.strides[1];
    return true;
}

int build_problem(GemmProblem &q, const NineToothedTensor *input, const NineToothedTensor &a, const NineToothedTensor &b,
                  const NineToothedTensor *beta, const NineToothedTensor *alpha, const NineToothedTensor &c, int dtype,
                  int out_dtype) {
    uint64_t am, ak, bk, bn, cm, cn;
    if (!read_matrix(a, am, ak, q.sam, q.sak) || !read_matrix(b, bk, bn, q.sbk, q.sbn) || !read_matrix(c, cm, cn, q.scm, q.scn))
        return hipErrorInvalidValue;
    if (ak != bk || am != cm || bn != cn) return hipErrorInvalidValue;
    if (am > 0x7fffffffull || bn > 0x7fffffffull || ak > 0x7fffffffull) return NINETOOTHED_NO_KERNEL;
    q.dtype = dtype;
    q.out_dtype = out_dtype;
    q.m = (int)am;
    q.n = (int)bn;
    q.k = (int)ak;
    q.a = a.data;
    q.b = b.data;
    q.c = c.data;
    q.bias = nullptr;
    q.sim = q.sin = 0;
    q.alpha = 1.0f;
    q.beta = 0.0f;
    if (input != nullptr && input->data != nullptr) {
        uint64_t im, in_;
        if (!read_matrix(*input, im, in_, q.sim, q.sin)) return hipErrorInvalidValue;
        if (im != cm || in_ != cn) return hipErrorInvalidValue;
        if (beta == nullptr || alpha == nullptr || beta->data == nullptr || alpha->data == nullptr) return hipErrorInvalidValue;
        q.bias = input->data;
        q.beta = (float)Scalar0d::as_double(*beta);
        q.alpha = (float)Scalar0d::as_double(*alpha);
    }
    if ((q.m > 0 && q.n > 0) && (q.a == nullptr && q.k > 0)) return hipErrorInvalidValue;
    return 0;
}

// ---- fp8 (e5m2) operands of large products: widened copies, then the fp16 instances ----
// An e5m2 value is the upper byte of the fp16 value it equals, so widening is exact and the fp16 kernels compute
// what the widening any-stride kernel computes (every product exact, fp32 sums).  One pass per operand writes a dense
// fp16 copy in the operand's own orientation -- rows contiguous or columns contiguous -- into the stream's scratch
// buffers; the direct-to-LDS instances then run the product several times faster than the any-stride kernel.
__global__ __launch_bounds__(256) void widen_e5m2_kernel(const uint8_t *src, int64_t outer, int64_t inner, int64_t outer_stride,
                                                         int64_t inner_stride, int64_t pitch, uint16_t *dst, int vectors) {
    typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
    const int64_t per_row = vectors ? inner / 16 : inner;
    const int64_t total = outer * per_row;
    for (int64_t index = (int64_t)blockIdx.x * 256 + threadIdx.x; index < total; index += (int64_t)gridDim.x * 256) {
        const int64_t row = index / per_row, piece = index - row * per_row;
        if (vectors) {  // 16 bytes in, 32 out: byte b of a dword becomes the upper byte of half b
            const uint4_t in = *(const uint4_t *)(src + row * outer_stride + piece * 16);
            uint4_t lo, hi;
            lo[0] = __builtin_amdgcn_perm(0u, in[0], 0x010c000cu);
            lo[1] = __builtin_amdgcn_perm(0u, in[0], 0x030c020cu);
            lo[2] = __builtin_amdgcn_perm(0u, in[1], 0x010c000cu);
            lo[3] = __builtin_amdgcn_perm(0u, in[1], 0x030c020cu);
            hi[0] = __builtin_amdgcn_perm(0u, in[2], 0x010c000cu);
            hi[1] = __builtin_amdgcn_perm(0u, in[2], 0x030c020cu);
            hi[2] = __builtin_amdgcn_perm(0u, in[3], 0x010c000cu);
            hi[3] = __builtin_amdgcn_perm(0u, in[3], 0x030c020cu);
            uint4_t *out = (uint4_t *)(dst + row * pitch + piece * 16);
            __builtin_nontemporal_store(lo, out);
            __builtin_nontemporal_store(hi, out + 1);
        } else {
            dst[row * pitch + piece] = (uint16_t)((unsigned)src[row * outer_stride + piece * inner_stride] << 8);
        }
    }
}

// writes the widened copy of a [d0, d1] matrix with element strides (s0, s1) and returns the copy's strides
hipError_t widen_e5m2(hipStream_t stream, const void *src, int64_t d0, int64_t d1, int64_t s0, int64_t s1, uint16_t *dst, int64_t &t0, int64_t &t1) {
    const bool by_columns = s0 == 1 && s1 != 1;  // columns contiguous: the copy keeps that orientation
    const int64_t outer = by_columns ? d1 : d0, inner = by_columns ? d0 : d1;
    const int64_t outer_stride = by_columns ? s1 : s0, inner_stride = by_columns ? s0 : s1;
    const int64_t pitch = (inner + 7) / 8 * 8;  // rows of the copy start on 16-byte boundaries
    t0 = by_columns ? 1 : pitch;
    t1 = by_columns ? pitch : 1;
    if (outer == 0 || inner == 0) return hipSuccess;
    const int vectors = inner_stride == 1 && inner % 16 == 0 && outer_stride % 16 == 0 && ((uintptr_t)src & 15) == 0;
    const int64_t work = outer * (vectors ? inner / 16 : inner);
    const unsigned blocks = (unsigned)std::min<int64_t>((work + 255) / 256, 256 * 32);
    widen_e5m2_kernel<<<dim3(blocks), dim3(256), 0, stream>>>((const uint8_t *)src, outer, inner, outer_stride, inner_stride, pitch, dst, vectors);
    return hipGetLastError();
}

int run_gemm(hipStream_t stream, const GemmProblem &q, int bm, int bn, int bk, bool may_copy = true);

// ---- fp16 / bf16 operands that the direct-to-LDS instances cannot read in place ----
// A K that is no multiple of 8, rows that do not start on 16-byte boundaries, an lhs stored by columns, operands with
// other strides: the any-stride kernel gathers such operands two bytes at a time and reaches a fifth of the fast
// instances' rate.  For products that are large enough, one pass per operand writes a dense copy with k contiguous --
// the lhs as [M][K8], the rhs as [N][K8], K8 = K rounded up to 8 with zeros in between, which add nothing to the sums --
// and the product runs on the instances with tails, which take a k-contiguous rhs with any N.
// dst[i][j] = j < d1 ? src[i * s0 + j * s1] : 0 for j < pitch; 64 x 64 tiles through LDS, so that the reads run along
// whichever dimension has the smaller stride and the writes along j, 16 bytes per lane on both sides where the
// source is contiguous along that dimension
__global__ __launch_bounds__(256) void repack_operand_kernel(const uint16_t *src, int64_t d0, int64_t d1, int64_t s0, int64_t s1, uint16_t *dst, int64_t pitch,
                                                            int64_t src_batch) {
    src += (int64_t)blockIdx.y * src_batch;  // a batch of matrices: the copies lie one after another
    dst += (int64_t)blockIdx.y * d0 * pitch;
    typedef uint16_t ushort8_t __attribute__((ext_vector_type(8)));
    typedef ushort8_t unaligned_ushort8_t __attribute__((aligned(2)));  // (global accesses need the element's alignment only)
    constexpr int kPitch = 72;  // rows of the tile start on 16-byte boundaries
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * kPitch];
    const int64_t tiles_j = (pitch + 63) / 64;
    const int64_t i0 = (int64_t)(blockIdx.x / tiles_j) * 64, j0 = (int64_t)(blockIdx.x % tiles_j) * 64;
    const int t = threadIdx.x;
    const bool along_i = s0 < s1;  // consecutive threads read consecutive i
    const int64_t fast_stride = along_i ? s0 : s1;
    if (fast_stride != 1) {  // (uniform) no dimension is contiguous: consecutive threads fetch consecutive elements
#pragma unroll 4
        for (int e = t; e < 64 * 64; e += 256) {
            const int fast = e & 63, slow = e >> 6;
            const int i = along_i ? fast : slow, j = along_i ? slow : fast;
            uint16_t value = 0;
            if (i0 + i < d0 && j0 + j < d1) value = src[(i0 + i) * s0 + (j0 + j) * s1];
            tile[i * kPitch + j] = value;
        }
    } else
    // eight consecutive elements of the source's contiguous dimension per thread, in one load
#pragma unroll
    for (int e = t; e < 64 * 8; e += 256) {
        const int fast = (e & 7) * 8, slow = e >> 3;
        const int i = along_i ? fast : slow, j = along_i ? slow : fast;
        const int64_t limit = along_i ? d0 - (i0 + i) : d1 - (j0 + j);  // elements left along the faster dimension
        const bool slow_inside = along_i ? j0 + j < d1 : i0 + i < d0;
        ushort8_t values = {0, 0, 0, 0, 0, 0, 0, 0};
        if (slow_inside && limit > 0) {
            const uint16_t *from = src + (i0 + i) * s0 + (j0 + j) * s1;
            if (fast_stride == 1 && limit >= 8) {
                values = *(const unaligned_ushort8_t *)from;
            } else {
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    if (c < limit) values[c] = from[c * fast_stride];
            }
        }
        if (along_i) {
#pragma unroll
            for (int c = 0; c < 8; ++c) tile[(i + c) * kPitch + j] = values[c];
        } else {
            *(ushort8_t *)&tile[i * kPitch + j] = values;
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = t; e < 64 * 8; e += 256) {
        const int j = (e & 7) * 8, i = e >> 3;
        if (i0 + i >= d0 || j0 + j >= pitch) continue;  // (pitch is a multiple of 8: whole vectors)
        *(ushort8_t *)(dst + (i0 + i) * pitch + j0 + j) = *(const ushort8_t *)&tile[i * kPitch + j];
    }
}

hipError_t repack_operand(hipStream_t stream, const void *src, int64_t d0, int64_t d1, int64_t s0, int64_t s1, uint16_t *dst, int64_t pitch, int batch = 1,
                          int64_t src_batch = 0) {
    const int64_t tiles = ((d0 + 63) / 64) * ((pitch + 63) / 64);
    if (tiles == 0 || batch == 0) return hipSuccess;
    if (tiles > 0x7fffffffll || batch > 65535) return hipErrorInvalidValue;
    repack_operand_kernel<<<dim3((unsigned)tiles, (unsigned)batch), dim3(256), 0, stream>>>((const uint16_t *)src, d0, d1, s0, s1, dst, pitch, src_batch);
    return hipGetLastError();
}

// Writes the dense copies of q's operands into the stream's buffers (`lease` must stay alive until everything that
// reads them is enqueued) and describes the product on them in `dense`.  0, an error, or NINETOOTHED_NO_KERNEL when
// this way does not apply.
int make_dense_copies(hipStream_t stream, const GemmProblem &q, int bm, int bn, int bk, WorkspaceLease &lease, GemmProblem &dense) {
    if ((q.dtype != NINETOOTHED_FLOAT16 && q.dtype != NINETOOTHED_BFLOAT16) || q.batch < 1 || q.batch > 65535) return NINETOOTHED_NO_KERNEL;
#ifndef NT_GEMM_COPY_LOG2
#define NT_GEMM_COPY_LOG2 21
#endif
    // (the any-stride kernel is slower from small sizes on: 512^3 36-45 us in place against 11-13 us on copies,
    // 256^3 22-25 against 12; below 128^3 everything is one launch's time)
    if ((int64_t)q.m * q.n * q.k * q.batch < ((int64_t)1 << NT_GEMM_COPY_LOG2) || q.fixed_scratch != nullptr) return NINETOOTHED_NO_KERNEL;
    const int64_t k8 = ((int64_t)q.k + 7) / 8 * 8;
    dense = q;
    dense.k = (int)k8;
    dense.sam = k8;
    dense.sak = 1;
    dense.sbk = 1;
    dense.sbn = k8;
    dense.a_batch = (int64_t)q.m * k8;  // (a batch: one copy per product, also of an operand that the products share)
    dense.b_batch = (int64_t)q.n * k8;
    // (alignment of the copies is a fact, not a property of these placeholder addresses)
    dense.a = dense.b = (const void *)(uintptr_t)256;
    const int choice = heuristic_choice(dense, bm, bn, bk);
    if (choice < 0 || choice == kAnyStride) return NINETOOTHED_NO_KERNEL;  // (the output's layout rules the fast instances out)
    // (buffers of their own: the sources may be the widened copies of fp8 operands)
    if (((int64_t)q.m + q.n) * k8 * 2 * q.batch > (int64_t(1) << 32)) return NINETOOTHED_NO_KERNEL;  // (a batch whose copies would take more than 4 GiB)
    uint16_t *a = (uint16_t *)lease.get(kWorkspaceGemmLhsDense, (size_t)q.m * k8 * 2 * q.batch);
    uint16_t *b = a != nullptr ? (uint16_t *)lease.get(kWorkspaceGemmRhsDense, (size_t)q.n * k8 * 2 * q.batch) : nullptr;
    if (a == nullptr || b == nullptr) return NINETOOTHED_NO_KERNEL;
    dense.a = a;
    dense.b = b;
    if (hipError_t err = repack_operand(stream, q.a, q.m, q.k, q.sam, q.sak, a, k8, q.batch, q.a_batch)) return (int)err;
    if (hipError_t err = repack_operand(stream, q.b, q.n, q.k, q.sbn, q.sbk, b, k8, q.batch, q.b_batch)) return (int)err;
    return 0;
}

// 0 / an error when the product ran on copies, NINETOOTHED_NO_KERNEL when this way does not apply
int run_gemm_on_repacked_copies(hipStream_t stream, const GemmProblem &q, int bm, int bn, int bk) {
    WorkspaceLease lease(stream);  // held until the product is enqueued: it reads the copies
    GemmProblem dense;
    if (const int status = make_dense_copies(stream, q, bm, bn, bk, lease, dense)) return status;
    return run_gemm(stream, dense, bm, bn, bk, false);
}

// 0 / an error when the product ran on widened copies, NINETOOTHED_NO_KERNEL when this way does not apply (tiny
// products; negative strides; no scratch memory, as under graph capture before a call of the same size outside one):
// the widening any-stride kernel, which reads its operands byte by byte, then serves the call (512^3: 70 us against
// 12 us this way, 8192^3: 16.8 ms against 0.83 ms)
int run_gemm_on_widened_copies(hipStream_t stream, const GemmProblem &q, int bm, int bn, int bk) {
    if (q.dtype != NINETOOTHED_FLOAT8_E5M2 || q.batch != 1) return NINETOOTHED_NO_KERNEL;
    if (q.fixed_scratch != nullptr) return NINETOOTHED_NO_KERNEL;  // (the entry point that allocates nothing: no buffers for copies)
    if (q.out_dtype != NINETOOTHED_FLOAT16 && (q.out_dtype != NINETOOTHED_FLOAT32 || q.addmm())) return NINETOOTHED_NO_KERNEL;
    if ((int64_t)q.m * q.n * q.k < ((int64_t)1 << 18)) return NINETOOTHED_NO_KERNEL;
    if (q.sam < 0 || q.sak < 0 || q.sbk < 0 || q.sbn < 0 || (q.addmm() && (q.sim < 0 || q.sin < 0))) return NINETOOTHED_NO_KERNEL;
    WorkspaceLease lease(stream);  // held until the product is enqueued: it reads the copies
    const auto bytes = [](int64_t d0, int64_t d1) { return (size_t)(std::max(d0, d1) + 8) * (size_t)(std::min(d0, d1) + 8) * 2; };  // (either orientation, padded rows)
    uint16_t *a = (uint16_t *)lease.get(kWorkspaceGemmLhsWidened, bytes(q.m, q.k));
    uint16_t *b = a != nullptr ? (uint16_t *)lease.get(kWorkspaceGemmRhsWidened, bytes(q.k, q.n)) : nullptr;
    uint16_t *bias = b != nullptr && q.addmm() ? (uint16_t *)lease.get(kWorkspaceGemmBiasWidened, bytes(q.m, q.n)) : nullptr;
    if (a == nullptr || b == nullptr || (q.addmm() && bias == nullptr)) return NINETOOTHED_NO_KERNEL;
    GemmProblem wide = q;
    wide.dtype = NINETOOTHED_FLOAT16;
    wide.a = a;
    wide.b = b;
    if (hipError_t err = widen_e5m2(stream, q.a, q.m, q.k, q.sam, q.sak, a, wide.sam, wide.sak)) return (int)err;
    if (hipError_t err = widen_e5m2(stream, q.b, q.k, q.n, q.sbk, q.sbn, b, wide.sbk, wide.sbn)) return (int)err;
    if (q.addmm()) {
        wide.bias = bias;
        if (hipError_t err = widen_e5m2(stream, q.bias, q.m, q.n, q.sim, q.sin, bias, wide.sim, wide.sin)) return (int)err;
    }
    return run_gemm(stream, wide, bm, bn, bk);
}

// an output stored by columns (`out.T`): C^T = B^T A^T is the same product with a row-major output, which the
// direct-to-LDS instances write (the any-stride kernel would store it two bytes at a time)
bool output_by_columns(const GemmProblem &q) { return q.scn != 1 && q.scm == 1 && q.n > 1; }

GemmProblem transposed_problem(const GemmProblem &q) {
    GemmProblem t = q;
    t.m = q.n;
    t.n = q.m;
    t.a = q.b;
    t.b = q.a;
    t.sam = q.sbn;
    t.sak = q.sbk;
    t.sbk = q.sak;
    t.sbn = q.sam;
    t.scm = q.scn;
    t.scn = q.scm;
    t.sim = q.sin;
    t.sin = q.sim;
    t.a_batch = q.b_batch;
    t.b_batch = q.a_batch;
    return t;
}

// A product whose 256 x 256 tiles are a few more than whole rounds of the chip's 256 CUs (17 x 17 = 289 of them for
// 4352^2) pays a whole round for the few: the tile rows that fill whole rounds run in one pass, the rows left over
// -- at most 51 tiles -- as a product of their own with the k range in parts, so that they occupy the chip once for
// a fraction of a round.  NINETOOTHED_NO_KERNEL when the shape is not of that kind or scratch memory is not to be had.
// (It comes before the cut instances, which also take up to half a round left, on smaller tiles, and a shorter K.  Where both apply they take 0.88 to 1.09 of
// this way's time, 0.97 on average: 4352 x 4352 x 4096 142 us here, 131 there, but 6598 x 2816 x 12872 396 and 433.)
int run_gemm_last_rows_in_parts(hipStream_t stream, const GemmProblem &q) {
    if ((q.dtype != NINETOOTHED_FLOAT16 && q.dtype != NINETOOTHED_BFLOAT16) || q.batch != 1 || q.fixed_scratch != nullptr) return NINETOOTHED_NO_KERNEL;
    static const bool enabled = getenv("NT_GEMM_NO_ROW_SPLIT") == nullptr;  // (set for A/B measurements: every product in one pass)
    if (!enabled) return NINETOOTHED_NO_KERNEL;
    const int64_t tiles_m = ceil_div(q.m, 256), tiles_n = ceil_div(q.n, 256), tiles = tiles_m * tiles_n;
    // (measured, one pass -> this way: 4352 x 4096 x 4352 160 -> 143 us, 4096 x 4096 x 4352 158 -> 135, 5120 x 4096 x 3584
    // 159 -> 139, 4104^3 172 -> 143; not for more than three rounds -- 8192 x 4096 x 8448 436 -> 447 --, for more than 51
    // tiles left over in parts of 256 x 256 tiles -- 4608^2 x 4096, 72 of them: 162 -> 173, 148 as a cut instance -- or a short k range -- 4352 x 1024 x 4352 49 -> 63)
    if (tiles <= 256 || tiles > 768 || tiles % 256 == 0 || q.k < 2048) return NINETOOTHED_NO_KERNEL;
    const int64_t top_rows = tiles / 256 * 256 / tiles_n;
    const int64_t bottom_tiles = (tiles_m - top_rows) * tiles_n;
    if (top_rows < 1 || top_rows >= tiles_m || bottom_tiles * 5 > 256) return NINETOOTHED_NO_KERNEL;
    if (ceil_div(top_rows * tiles_n, (int64_t)256) >= ceil_div(tiles, (int64_t)256)) return NINETOOTHED_NO_KERNEL;  // (no round saved)
    const int64_t size = q.dtype == NINETOOTHED_FLOAT16 || q.dtype == NINETOOTHED_BFLOAT16 ? 2 : 4;
    const int64_t out_size = q.out_dtype == NINETOOTHED_FLOAT32 ? 4 : size;
    GemmProblem top = q, bottom = q;
    top.m = (int)(top_rows * 256);
    bottom.m = q.m - top.m;
    bottom.a = (const char *)q.a + (int64_t)top.m * q.sam * size;
    bottom.c = (char *)q.c + (int64_t)top.m * q.scm * out_size;
    if (q.bias != nullptr) bottom.bias = (const char *)q.bias + (int64_t)top.m * q.sim * size;
    const int whole = kInstances[k256x256x32].accepts(top) ? (int)k256x256x32 : (int)kTail256x256x32;
    if (!kInstances[whole].accepts(top) || !kInstances[kSplit256x256x32].accepts(bottom)) return NINETOOTHED_NO_KERNEL;
    int result = (int)kInstances[kSplit256x256x32].launch(bottom, stream);  // (first: it is the one that may find no scratch memory)
    if (result != 0) return result;
    note_launch(kLaunchGemm, whole, "256x256x32 tiles: the tile rows that fill whole rounds in one pass, the last rows with the k range in parts");
    return (int)kInstances[whole].launch(top, stream);
}

int run_gemm(hipStream_t stream, const GemmProblem &q, int bm, int bn, int bk, bool may_copy) {
    if (q.m == 0 || q.n == 0) return 0;
    if (output_by_columns(q) && !q.linear) return run_gemm(stream, transposed_problem(q), bn, bm, bk, may_copy);
    if (bm <= 0 && bn <= 0 && bk <= 0) {
        const int rows_split = run_gemm_last_rows_in_parts(stream, q);
        if (rows_split != NINETOOTHED_NO_KERNEL) return rows_split;
    }
    if (q.dtype == NINETOOTHED_FLOAT8_E5M2) {
        const int widened = run_gemm_on_widened_copies(stream, q, bm, bn, bk);
        if (widened != NINETOOTHED_NO_KERNEL) return widened;
    }
    int choice = -1;
    if ((bm <= 0 || bn <= 0) && q.batch == 1) choice = lookup_tuned(q);  // (tuned choices are recorded for single products)
    // (choices are timed and recorded for the plain product, which the any-stride kernel may win; it has no linear epilogue)
    GemmProblem with_hints;
    const bool hinted = bm > 0 || bn > 0 || bk > 0;
    if (hinted) {
        with_hints = q;
        with_hints.hinted = true;
    }
    const GemmProblem &asked = hinted ? with_hints : q;
    if (choice < 0 || !kInstances[choice].accepts(asked) || (choice == kAnyStride && q.linear)) choice = heuristic_choice(asked, bm, bn, bk);
    if (choice < 0 || (choice == kAnyStride && q.linear)) return NINETOOTHED_NO_KERNEL;
    if (choice == kAnyStride && may_copy) {
        const int copied = run_gemm_on_repacked_copies(stream, q, bm, bn, bk);
        if (copied != NINETOOTHED_NO_KERNEL) return copied;
    }
    note_launch(kLaunchGemm, choice, kInstances[choice].name);
    int result = (int)kInstances[choice].launch(asked, stream);
    if (result == NINETOOTHED_NO_KERNEL && is_split(choice)) {  // a split-K instance without scratch memory
        for (int fallback : {(int)kTail64x64x64, (int)kTail128x128x64, (int)kTail256x256x32, (int)kAnyStride})
            if (kInstances[fallback].accepts(q) && !(fallback == kAnyStride && q.linear)) {
                note_launch(kLaunchGemm, fallback, kInstances[fallback].name);
                return (int)kInstances[fallback].launch(q, stream);
            }
    }
    return result;
}

}  // namespace
}  // namespace nt

using namespace nt;

extern "C" {

NineToothedResult launch_nt_matmul(NineToothedStream stream, NineToothedTensor lhs, NineToothedTensor rhs,
                                   NineToothedTensor output, int dtype, int output_dtype, int block_size_m,
                                   int block_size_n, int block_size_k) {
    GemmProblem q;
    if (int err = build_problem(q, nullptr, lhs, rhs, nullptr, nullptr, output, dtype, output_dtype)) return err;
    return run_gemm((hipStream_t)stream, q, block_size_m, block_size_n, block_size_k);
}

NineToothedResult launch_nt_batched_matmul(NineToothedStream stream, NineToothedTensor lhs, NineToothedTensor rhs,
                                           NineToothedTensor output, int dtype, int output_dtype, int block_size_m,
                                           int block_size_n, int block_size_k) {
    if (!lhs.shape || !rhs.shape || !output.shape || !lhs.strides || !rhs.strides || !output.strides) return hipErrorInvalidValue;
    const uint64_t batch = output.shape[0];
    // an operand with a single matrix is shared by all products
    if ((lhs.shape[0] != batch && lhs.shape[0] != 1) || (rhs.shape[0] != batch && rhs.shape[0] != 1)) return hipErrorInvalidValue;
    if (batch > 0x7fffffffull) return NINETOOTHED_NO_KERNEL;
    const NineToothedTensor a = {lhs.data, lhs.shape + 1, lhs.strides + 1}, b = {rhs.data, rhs.shape + 1, rhs.strides + 1},
                            c = {output.data, output.shape + 1, output.strides + 1};
    GemmProblem q;
    if (int err = build_problem(q, nullptr, a, b, nullptr, nullptr, c, dtype, output_dtype)) return err;
    if (batch == 0) return 0;
    q.batch = (int)batch;
    q.a_batch = lhs.shape[0] == 1 ? 0 : lhs.strides[0];
    q.b_batch = rhs.shape[0] == 1 ? 0 : rhs.strides[0];
    q.c_batch = output.strides[0];
    return run_gemm((hipStream_t)stream, q, block_size_m, block_size_n, block_size_k);
}

NineToothedResult launch_nt_addmm(NineToothedStream stream, NineToothedTensor input, NineToothedTensor mat1,
                                  NineToothedTensor mat2, NineToothedTensor beta, NineToothedTensor alpha,
                                  NineToothedTensor output, int dtype, int block_size_m, int block_size_n,
                                  int block_size_k) {
    if (input.data == nullptr) return hipErrorInvalidValue;
    GemmProblem q;
    const int output_dtype = dtype == NINETOOTHED_FLOAT8_E5M2 ? NINETOOTHED_FLOAT16 : dtype;  // fp8 operands: the rounded product is fp16
    if (int err = build_problem(q, &input, mat1, mat2, &beta, &alpha, output, dtype, output_dtype)) return err;
    return run_gemm((hipStream_t)stream, q, block_size_m, block_size_n, block_size_k);
}

// A bias per column, a scale and a lower bound ride on the product, whatever instance it runs on.  As a product into an fp32 tensor and
// a tile map over that: 1500 x 14336 x 4096 bf16 202 us, here 172; 28 x 3392 x 256 fp16 13.5 (two launches from the host and an allocation), here 6.7.
NineToothedResult launch_nt_linear(NineToothedStream stream, NineToothedTensor lhs, NineToothedTensor rhs, NineToothedTensor bias,
                                   int bias_dtype, double scale, double lower, NineToothedTensor output, int dtype,
                                   int block_size_m, int block_size_n, int block_size_k) {
    if (dtype != NINETOOTHED_FLOAT16 && dtype != NINETOOTHED_BFLOAT16) return NINETOOTHED_NO_KERNEL;
    GemmProblem q;
    if (int err = build_problem(q, nullptr, lhs, rhs, nullptr, nullptr, output, dtype, dtype)) return err;
    q.linear = true;
    q.alpha = (float)scale;
    q.lower = (float)lower;
    if (q.lower != q.lower) return NINETOOTHED_NO_KERNEL;  // (a bound that is no number makes every result none)
    if (q.m == 0 || q.n == 0) return 0;
    if (q.k == 0 || q.scn != 1 || q.scm < q.n || q.sam < 0 || q.sak < 0 || q.sbk < 0 || q.sbn < 0) return NINETOOTHED_NO_KERNEL;
    if (bias.data != nullptr) {
        if (bias_dtype != dtype && bias_dtype != NINETOOTHED_FLOAT32) return NINETOOTHED_NO_KERNEL;
        if (bias.shape == nullptr || bias.strides == nullptr || bias.shape[0] != (uint64_t)q.n) return hipErrorInvalidValue;
        if (bias.strides[0] < 0) return NINETOOTHED_NO_KERNEL;
        q.column_bias = bias.data;
        q.sin = bias.strides[0];
        q.bias_float = bias_dtype == NINETOOTHED_FLOAT32;
    }
    // an output that shares memory with an operand: tiles that are written while others still read it (a product into a tensor of
    // its own and a second pass have no such order to keep)
    const uintptr_t first = (uintptr_t)q.c, last = first + (((uintptr_t)q.m - 1) * q.scm + q.n) * 2;
    const auto shares = [&](const void *data, int64_t elements, int64_t size) { return (uintptr_t)data < last && first < (uintptr_t)data + (uintptr_t)(elements * size); };
    if (shares(q.a, (int64_t)(q.m - 1) * q.sam + (int64_t)(q.k - 1) * q.sak + 1, 2) || shares(q.b, (int64_t)(q.k - 1) * q.sbk + (int64_t)(q.n - 1) * q.sbn + 1, 2) ||
        (q.column_bias != nullptr && shares(q.column_bias, (int64_t)(q.n - 1) * q.sin + 1, q.bias_float ? 4 : 2)))
        return NINETOOTHED_NO_KERNEL;
    return run_gemm((hipStream_t)stream, q, block_size_m, block_size_n, block_size_k);
}

}  // extern "C"

namespace nt {
namespace {

// Scratch memory of launch_nt_matmul_static_scratch: part of the library's code object, so every GPU the
// library runs on holds its own copy from the first use until the process ends.  Host code never uses the
// array's name as an address (on the host it is a stand-in, not device memory): the device address is
// asked for once per device and only that pointer is handed to kernels.
constexpr size_t kStaticScratchBytes = size_t(NINETOOTHED_STATIC_SCRATCH_BYTES);
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_static_scratch_mutex;
void *g_static_scratch_address[kMaxDevices] = {};

// the array's address on the current device
int static_scratch_address(void **address) {
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return (int)err;
    if (device < 0 || device >= kMaxDevices) return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
    if (g_static_scratch_address[device] == nullptr) {
        void *found = nullptr;
        err = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
        if (err != hipSuccess) return (int)err;
        if (found == nullptr) return (int)hipErrorInvalidSymbol;
        g_static_scratch_address[device] = found;
    }
    *address = g_static_scratch_address[device];
    return 0;
}

}  // namespace
}  // namespace nt

extern "C" {

NineToothedResult launch_nt_matmul_static_scratch(NineToothedStream stream, NineToothedTensor lhs, NineToothedTensor rhs,
                                                  NineToothedTensor output, int dtype, int output_dtype, int block_size_m,
                                                  int block_size_n, int block_size_k) {
    GemmProblem q;
    if (int err = build_problem(q, nullptr, lhs, rhs, nullptr, nullptr, output, dtype, output_dtype)) return err;
    void *address = nullptr;
    if (int err = static_scratch_address(&address)) return err;
    q.fixed_scratch = (float *)address;
    q.fixed_scratch_bytes = kStaticScratchBytes;
    return run_gemm((hipStream_t)stream, q, block_size_m, block_size_n, block_size_k);
}

int nt_gemm_num_configs(void) { return kNumInstances; }

NineToothedResult nt_gemm_config_name(int config, char *buffer, int size) {
    if (config < 0 || config >= kNumInstances || buffer == nullptr || size <= 0) return NINETOOTHED_NO_KERNEL;
    snprintf(buffer, (size_t)size, "%s", kInstances[config].name);
    return 0;
}

NineToothedResult launch_nt_gemm_config(NineToothedStream stream, int config, NineToothedTensor input,
                                        NineToothedTensor mat1, NineToothedTensor mat2, NineToothedTensor beta,
                                        NineToothedTensor alpha, NineToothedTensor output, int dtype,
                                        int output_dtype) {
    if (config < 0 || config >= kNumInstances) return NINETOOTHED_NO_KERNEL;
    GemmProblem q;
    if (int err = build_problem(q, &input, mat1, mat2, &beta, &alpha, output, dtype, output_dtype)) return err;
    if (q.m == 0 || q.n == 0) return 0;
    if (!kInstances[config].accepts(q)) return NINETOOTHED_NO_KERNEL;
    note_launch(kLaunchGemm, config, kInstances[config].name);
    return (int)kInstances[config].launch(q, (hipStream_t)stream);
}

NineToothedResult nt_tune_gemm_for_caller(NineToothedStream stream_, NineToothedTensor input, NineToothedTensor mat1,
                                          NineToothedTensor mat2, NineToothedTensor beta, NineToothedTensor alpha,
                                          NineToothedTensor output, int dtype, int output_dtype, int iters, float call_ms,
                                          float split_call_ms, int *best_config, float *best_ms) {
    hipStream_t stream = (hipStream_t)stream_;
    GemmProblem given;
    if (int err = build_problem(given, &input, mat1, mat2, &beta, &alpha, output, dtype, output_dtype)) return err;
    // (what the launch functions do first: an output stored by columns is the transposed product)
    GemmProblem q = output_by_columns(given) ? transposed_problem(given) : given;
    int best = -1;
    float best_time = 0.0f;
    // A problem that a single instance accepts has nothing to time.  Operands that only the any-stride kernel reads
    // in place run on dense copies (launch_nt_matmul / launch_nt_addmm): then the product on the copies is what
    // gets timed and recorded, under its own key, where the launch functions look it up.
    int accepting = 0;
    for (int i = 0; i < kNumInstances; ++i) accepting += kInstances[i].accepts(q) ? 1 : 0;
    std::unique_ptr<WorkspaceLease> lease;  // (keeps the copies in place while they are timed)
    if (accepting <= 1) {
        GemmProblem dense;
        lease.reset(new WorkspaceLease(stream));
        const int copied = stream_is_capturing(stream) ? NINETOOTHED_NO_KERNEL : make_dense_copies(stream, q, 0, 0, 0, *lease, dense);
        if (copied != 0) {
            if (best_config) *best_config = accepting == 1 ? -2 : -1;
            if (best_ms) *best_ms = 0.0f;
            if (copied != NINETOOTHED_NO_KERNEL) return copied;
            return accepting == 1 ? 0 : NINETOOTHED_NO_KERNEL;
        }
        q = dense;
        const int known = lookup_tuned(q);
        if (known >= 0 && kInstances[known].accepts(q)) {  // (an earlier process has timed it: the file was loaded)
            if (best_config) *best_config = known;
            if (best_ms) *best_ms = 0.0f;
            return 0;
        }
    }
    // (inside a graph capture nothing is timed: the problem stays on the fixed preference order and nothing is recorded)
    // the untuned rule's instance is timed first and stays unless another one is more than 2 % faster: timings of a
    // few launches scatter by about that much, and the choice should not differ from process to process for nothing.
    // A skinny instance stays unless another one is more than 25 % faster: timing launches find B in the caches that
    // the launch before has left it in, a program that works through its layers finds it in memory, where the skinny
    // kernels lose less (32 x 14336 x 4096: 18.9 us on tiles with B in the caches, 29.0 without; 22.9 and 24.9 on 32
    // columns per workgroup).
    const int preferred = heuristic_choice(q, 0, 0, 0);
    const float margin = preferred == kSkinny16 || preferred == kSkinny32 ? 0.25f : 0.02f;
    auto instance_of = [&](int i) { return preferred < 0 ? i : (i == 0 ? preferred : (i - 1 < preferred ? i - 1 : i)); };
    const int result = tune_time(stream, kNumInstances, iters, [&](int i) -> int {
        const int instance = instance_of(i);
        if (!kInstances[instance].accepts(q)) return NINETOOTHED_NO_KERNEL;
        return (int)kInstances[instance].launch(q, stream);
    }, &best, &best_time, margin, [&](int i, float measured) { return std::max(measured, is_split(instance_of(i)) || is_cut(instance_of(i)) ? split_call_ms : call_ms); });
    if (best >= 0) best = instance_of(best);
    if (best_config) *best_config = best;
    if (best_ms) *best_ms = best_time;
    if (result != 0) return result;
    if (best < 0) return stream_is_capturing(stream) ? 0 : NINETOOTHED_NO_KERNEL;
    int values[7];
    tune_values(q, values);
    const int blocks[3] = {kInstances[best].bm, kInstances[best].bn, kInstances[best].bk};
    tune_record(kTuneGemm, values, 7, best, blocks, 3);
    return 0;
}

NineToothedResult nt_tune_gemm(NineToothedStream stream, NineToothedTensor input, NineToothedTensor mat1,
                               NineToothedTensor mat2, NineToothedTensor beta, NineToothedTensor alpha,
                               NineToothedTensor output, int dtype, int output_dtype, int iters, int *best_config,
                               float *best_ms) {
    return nt_tune_gemm_for_caller(stream, input, mat1, mat2, beta, alpha, output, dtype, output_dtype, iters, 0.0f, 0.0f, best_config, best_ms);
}

// The cached instance for a problem given by its sizes (row-major rhs), or -1.
int nt_tune_cache_lookup(int dtype, int output_dtype, int m, int n, int k, int addmm) {
    const int values[7] = {dtype, output_dtype, m, n, k, addmm ? 1 : 0, 0};
    const int choice = tune_lookup(kTuneGemm, values, 7);
    return choice >= 0 && choice < kNumInstances ? choice : -1;
}

}  // extern "C"

namespace nt {
namespace {

bool conv2d_choice_known(int index, const int *, int) { return index >= kConvGather && index <= kConvWindow; }
const bool g_conv2d_check_registered = tune_register_check(kTuneConv2d, conv2d_choice_known);

// validates the call and fills the request; returns 0, an error, or -1 when there is nothing to compute
int conv2d_request(Conv2dRequest &request, const NineToothedTensor &input, const NineToothedTensor &filter, const NineToothedTensor &output,
                   int dtype, int padding_h, int padding_w, int stride_h = 1, int stride_w = 1, int dilation_h = 1, int dilation_w = 1) {
    if (dtype != NINETOOTHED_FLOAT16 && dtype != NINETOOTHED_BFLOAT16 && dtype != NINETOOTHED_FLOAT32) return NINETOOTHED_NO_KERNEL;
    if (!input.shape || !filter.shape || !output.shape || !input.strides || !filter.strides || !output.strides)
        return hipErrorInvalidValue;
    if (padding_h < 0 || padding_w < 0 || stride_h < 1 || stride_w < 1 || dilation_h < 1 || dilation_w < 1) return hipErrorInvalidValue;
    const int64_t N = (int64_t)input.shape[0], C = (int64_t)input.shape[1], H = (int64_t)input.shape[2], W = (int64_t)input.shape[3];
    const int64_t K = (int64_t)filter.shape[0], R = (int64_t)filter.shape[2], S = (int64_t)filter.shape[3];
    if ((int64_t)filter.shape[1] != C) return hipErrorInvalidValue;
    // Windows start every `stride` positions of the padded input, as many as the output has rows / columns: either the
    // number that fit (floor, the usual convolution) or one more that hangs over the edge (the reference's
    // `Tensor.tile` without `floor_mode`, src/ninetoothed/tensor.py:237-248; what hangs over reads as padding).
    const int64_t span_h = H + 2 * padding_h - dilation_h * (R - 1) - 1, span_w = W + 2 * padding_w - dilation_w * (S - 1) - 1;
    const int64_t P = (int64_t)output.shape[2], Q = (int64_t)output.shape[3];
    if ((int64_t)output.shape[0] != N || (int64_t)output.shape[1] != K) return hipErrorInvalidValue;
    if (span_h < 0 || span_w < 0) {
        if (P > 0 && Q > 0) return hipErrorInvalidValue;  // the filter does not fit the padded input: no output positions
    } else {
        const int64_t fit_h = span_h / stride_h + 1, fit_w = span_w / stride_w + 1;
        const int64_t over_h = (span_h + stride_h - 1) / stride_h + 1, over_w = (span_w + stride_w - 1) / stride_w + 1;
        if ((P != fit_h && P != over_h) || (Q != fit_w && Q != over_w)) return hipErrorInvalidValue;
    }
    if (P <= 0 || Q <= 0 || N == 0 || K == 0) return -1;  // nothing to write
    if (N * P * Q > 0x7fffffffll || C * R * S > 0x7fffffffll || K > 0x7fffffffll || N > 0x7fffffffll) return NINETOOTHED_NO_KERNEL;
    request.dtype = dtype;
    request.x = input.data;
    request.w = filter.data;
    request.y = output.data;
    request.N = (int)N; request.C = (int)C; request.H = (int)H; request.W = (int)W;
    request.K = (int)K; request.R = (int)R; request.S = (int)S; request.P = (int)P; request.Q = (int)Q;
    request.pad_h = padding_h; request.pad_w = padding_w;
    request.stride_h = stride_h; request.stride_w = stride_w; request.dil_h = dilation_h; request.dil_w = dilation_w;
    for (int d = 0; d < 4; ++d) {
        request.xs[d] = input.strides[d];
        request.ws[d] = filter.strides[d];
        request.ys[d] = output.strides[d];
    }
    return 0;
}

template <typename T>
hipError_t conv2d_gather(const Conv2dRequest &r, hipStream_t stream) {
    Conv2dProblem<T> prob;
    prob.m = r.N * r.P * r.Q;
    prob.n = r.K;
    prob.k = r.C * r.R * r.S;
    prob.x = (const T *)r.x;
    prob.w = (const T *)r.w;
    prob.y = (T *)r.y;
    prob.C = r.C; prob.H = r.H; prob.W = r.W; prob.R = r.R; prob.S = r.S; prob.P = r.P; prob.Q = r.Q;
    prob.pad_h = r.pad_h;
    prob.pad_w = r.pad_w;
    prob.stride_h = r.stride_h; prob.stride_w = r.stride_w; prob.dil_h = r.dil_h; prob.dil_w = r.dil_w;
    for (int d = 0; d < 4; ++d) {
        prob.xs[d] = r.xs[d];
        prob.ws[d] = r.ws[d];
        prob.ys[d] = r.ys[d];
    }
    const int64_t tiles = (int64_t)ceil_div(prob.m, kGenBM) * ceil_div(prob.n, kGenBN);
    gemm_generic_kernel<Conv2dProblem<T>><<<dim3((unsigned)tiles), dim3(kGenThreads), 0, stream>>>(prob);
    return hipGetLastError();
}

// 1 x 1 filters without padding: per image Y[K, P*Q] = W[K, C] . X[C, P*Q], a batch of row-major products on
// the tensors as they lie (no repacking, no scratch memory).  NINETOOTHED_NO_KERNEL when the call is not that
// or no one-pass GEMM instance of the fast kind takes it.
int conv2d_pointwise(const Conv2dRequest &r, hipStream_t stream) {
    if (!(r.R == 1 && r.S == 1 && r.pad_h == 0 && r.pad_w == 0 && r.stride_h == 1 && r.stride_w == 1 && r.P == r.H && r.Q == r.W && r.xs[3] == 1 && r.xs[2] == r.W && r.ys[3] == 1 && r.ys[2] == r.Q && r.ws[1] == 1))
        return NINETOOTHED_NO_KERNEL;
    GemmProblem q;
    q.dtype = q.out_dtype = r.dtype;
    q.m = r.K;
    q.n = r.P * r.Q;
    q.k = r.C;
    q.a = r.w;
    q.b = r.x;
    q.c = r.y;
    q.bias = nullptr;
    q.sam = r.ws[0]; q.sak = 1;
    q.sbk = r.xs[1]; q.sbn = 1;
    q.scm = r.ys[1]; q.scn = 1;
    q.sim = q.sin = 0;
    q.alpha = 1.0f; q.beta = 0.0f;
    q.batch = r.N;
    q.a_batch = 0;
    q.b_batch = r.xs[0];
    q.c_batch = r.ys[0];
    q.hinted = true;  // (one launch, no scratch memory)
    const int choice = heuristic_choice(q, 0, 0, 0);
    if (choice <= kAnyStride || is_split(choice)) return NINETOOTHED_NO_KERNEL;
    note_launch(kLaunchConv2d, kConvPointwise, kInstances[choice].name);
    return (int)kInstances[choice].launch(q, stream);
}

int conv2d_run(const Conv2dRequest &r, int path, hipStream_t stream) {
    // fp32 tensors: the gathering kernel on fp32 MFMAs (the other paths move 16-bit elements)
    if (r.dtype == NINETOOTHED_FLOAT32) {
        if (path != kConvAuto && path != kConvGather) return NINETOOTHED_NO_KERNEL;
        note_launch(kLaunchConv2d, kConvGather, "gemm_generic_kernel with an im2col gather, fp32 MFMA");
        return (int)conv2d_gather<float>(r, stream);
    }
    if (path == kConvAuto || path == kConvPointwise) {
        const int pointwise = conv2d_pointwise(r, stream);
        if (pointwise != NINETOOTHED_NO_KERNEL || path == kConvPointwise) return pointwise;
    }
    if (path == kConvAuto || path == kConvDirect) {
        note_launch(kLaunchConv2d, kConvDirect, "conv2d_direct_kernel, one launch on the tensors as they lie");
        const int direct = conv2d_direct(r, stream);
        if (direct != NINETOOTHED_NO_KERNEL || path == kConvDirect) return direct;
    }
    if (path == kConvAuto || path == kConvWindow) {
        const int window = conv2d_window(r, stream, path == kConvAuto);
        if (window != NINETOOTHED_NO_KERNEL || path == kConvWindow) return window;
    }
    if (path == kConvAuto || path == kConvRepack) {
        const int fast = conv2d_fast(r, stream);
        if (fast != NINETOOTHED_NO_KERNEL || path == kConvRepack) return fast;
    }
    note_launch(kLaunchConv2d, kConvGather, "gemm_generic_kernel with an im2col gather");
    return r.dtype == NINETOOTHED_FLOAT16 ? (int)conv2d_gather<half_t>(r, stream) : (int)conv2d_gather<bf16_t>(r, stream);
}

void conv2d_tune_values(const Conv2dRequest &r, int (&values)[11]) {
    const int dense_x = r.xs[3] == 1 && r.xs[2] == r.W && r.xs[1] == (int64_t)r.H * r.W && r.xs[0] == (int64_t)r.C * r.H * r.W;
    const int v[11] = {r.dtype, r.N, r.C, r.H, r.W, r.K, r.R, r.S, r.pad_h, r.pad_w, dense_x};
    for (int i = 0; i < 11; ++i) values[i] = v[i];
}

}  // namespace
}  // namespace nt

extern "C" {

NineToothedResult launch_nt_conv2d(NineToothedStream stream, NineToothedTensor input, NineToothedTensor filter,
                                   NineToothedTensor output, int dtype, int padding_h, int padding_w, int block_size_m,
                                   int block_size_n, int block_size_k) {
    (void)block_size_n;
    (void)block_size_k;
    Conv2dRequest request;
    const int status = conv2d_request(request, input, filter, output, dtype, padding_h, padding_w);
    if (status != 0) return status < 0 ? 0 : status;
    // block_size_m: 1 = the gather kernel, 2 = the repacking path, 3 = the one-launch path, 4 = a 1 x 1 filter as a
    // batch of plain products, NINETOOTHED_CONV2D_WINDOWS = input windows in LDS; otherwise the tuned choice for this problem, else the library's order
    int path = block_size_m >= kConvGather && block_size_m <= kConvPointwise ? block_size_m : block_size_m == NINETOOTHED_CONV2D_WINDOWS ? kConvWindow : kConvAuto;
    if (block_size_m == 0) {
        int values[11];
        conv2d_tune_values(request, values);
        const int tuned = tune_lookup(kTuneConv2d, values, 11);
        if (tuned >= kConvGather && tuned <= kConvWindow) path = tuned;
    }
    int result = conv2d_run(request, path, (hipStream_t)stream);
    // (a tuned path that needs scratch memory it cannot get, e.g. under graph capture, or windows that do not take the problem: the library's order)
    if (result == NINETOOTHED_NO_KERNEL && path != kConvAuto && (block_size_m == 0 || path == kConvWindow)) result = conv2d_run(request, kConvAuto, (hipStream_t)stream);
    return result;
}

NineToothedResult launch_nt_conv2d_strided(NineToothedStream stream, NineToothedTensor input, NineToothedTensor filter,
                                           NineToothedTensor output, int dtype, int padding_h, int padding_w, int stride_h,
                                           int stride_w, int dilation_h, int dilation_w, int block_size_m, int block_size_n,
                                           int block_size_k) {
    if (stride_h == 1 && stride_w == 1 && dilation_h == 1 && dilation_w == 1) {
        Conv2dRequest plain;  // (an output with one more window than fits is not launch_nt_conv2d's problem)
        const int status = conv2d_request(plain, input, filter, output, dtype, padding_h, padding_w);
        if (status != 0) return status < 0 ? 0 : status;
        if (plain.P == plain.H + 2 * padding_h - plain.R + 1 && plain.Q == plain.W + 2 * padding_w - plain.S + 1)
            return launch_nt_conv2d(stream, input, filter, output, dtype, padding_h, padding_w, block_size_m, block_size_n, block_size_k);
    }
    (void)block_size_n;
    (void)block_size_k;
    Conv2dRequest request;
    const int status = conv2d_request(request, input, filter, output, dtype, padding_h, padding_w, stride_h, stride_w, dilation_h, dilation_w);
    if (status != 0) return status < 0 ? 0 : status;
    // the ways that take windows with steps: input windows in LDS, 2 = repacking pass plus GEMM loop, 1 = gather kernel (nothing is tuned here)
    const int path = block_size_m == kConvGather || block_size_m == kConvRepack ? block_size_m : block_size_m == NINETOOTHED_CONV2D_WINDOWS ? kConvWindow : kConvAuto;
    int result = conv2d_run(request, path, (hipStream_t)stream);
    if (result == NINETOOTHED_NO_KERNEL && path == kConvRepack) result = conv2d_run(request, kConvGather, (hipStream_t)stream);
    if (result == NINETOOTHED_NO_KERNEL && path == kConvWindow) result = conv2d_run(request, kConvAuto, (hipStream_t)stream);
    return result;
}

NineToothedResult nt_tune_conv2d(NineToothedStream stream, NineToothedTensor input, NineToothedTensor filter, NineToothedTensor output,
                                 int dtype, int padding_h, int padding_w, int iters, int *best_path, float *best_ms) {
    if (best_path) *best_path = -1;
    if (best_ms) *best_ms = 0.0f;
    Conv2dRequest request;
    const int status = conv2d_request(request, input, filter, output, dtype, padding_h, padding_w);
    if (status != 0) return status < 0 ? 0 : status;
    int values[11];
    conv2d_tune_values(request, values);
    const int paths[5] = {kConvPointwise, kConvDirect, kConvWindow, kConvRepack, kConvGather};
    int best = -1;
    float best_time = 0.0f;
    // an earlier way stays unless a later one is more than 3 % faster: the first three need no scratch memory and one launch
    const int result = tune_time((hipStream_t)stream, 5, iters, [&](int i) -> int { return conv2d_run(request, paths[i], (hipStream_t)stream); }, &best, &best_time, 0.03f);
    if (result != 0) return result;
    if (best < 0) return 0;  // (a stream under graph capture: nothing was timed)
    tune_record(kTuneConv2d, values, 11, paths[best]);
    if (best_path) *best_path = paths[best];
    if (best_ms) *best_ms = best_time;
    return 0;
}

#ifdef NT_GEMM_ABLATION
void nt_debug_set_tile_order(int order) { g_tile_order = order; }
#endif

const char *nt_version(void) { return "nt_hip 0.2 gfx950"; }

}  // extern "C"
