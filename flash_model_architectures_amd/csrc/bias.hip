// Per-expert bias of the expert projections: y[row, :] += bias[expert(row), :] after a projection, and
// its gradient d_bias[e, :] = sum of the grouped gradient rows of expert e.  The reference supports
// biases only on its torch path (F.linear(x, W[e], bias[e]), xma/layers/moe/__init__.py:103-106) and
// asserts them away on its kernel path (:54,79).  Both kernels are plain HBM streams.
#include "common.h"

namespace xma {

constexpr int kBiasRowsPerBlock = 8;

// Block = 8 rows x up to 32 column chunks per pass; row p is routed row p, written at out_index[p] (or p).
template <typename T, bool VEC, typename SeT>
__global__ __launch_bounds__(256) void add_expert_bias_kernel(T* __restrict__ y, int64_t ld_y,
                                                               const T* __restrict__ bias, int64_t ld_bias,
                                                               const SeT* __restrict__ expert_of_row,
                                                               const void* __restrict__ out_index, int idx_is_i64,
                                                               int64_t rows, int64_t cols) {
    constexpr int PV = VEC ? Elem<T>::kPerVec : 1;
    const int64_t chunks = cols / PV;
    const int cl = threadIdx.x % 32, rl = threadIdx.x / 32;
    for (int64_t p0 = (int64_t)blockIdx.x * kBiasRowsPerBlock; p0 < rows; p0 += (int64_t)gridDim.x * kBiasRowsPerBlock) {
        const int64_t p = p0 + rl;
        if (p >= rows) continue;
        const int64_t e = (int64_t)expert_of_row[p];
        const int64_t r = out_index ? load_index(out_index, idx_is_i64, p) : p;
        T* row = y + r * ld_y;
        const T* b = bias + e * ld_bias;
        for (int64_t c = cl; c < chunks; c += 32) {
            if constexpr (VEC) {
                float a[PV], v[PV];
                Elem<T>::unpack(load_stream(row + c * PV), a);
                Elem<T>::unpack(*reinterpret_cast<const uint4*>(b + c * PV), v);
#pragma unroll
                for (int q = 0; q < PV; ++q) a[q] += v[q];
                store_stream(row + c * PV, Elem<T>::pack(a));
            } else {
                Elem<T>::store(row + c, Elem<T>::load(row + c) + Elem<T>::load(b + c));
            }
        }
    }
}

// Block (x = column block of CL chunks, y = expert): 1024 / CL row lanes walk the expert's rows in order, IN_FLIGHT at a time, and
// keep fp32 partial sums of their chunk; the lanes are added through LDS in lane order.  The order of the additions is
// fixed, so the result is reproducible.
// Few experts are few blocks, and a block waits for memory: with 32 chunks, one row in flight and the 32 lanes added up by
// one of them, 12004 rows of 512 and 1024 columns over 6 experts in 16 bits took 13 and 39 us; so 5.5 and 12.6.
// ONE_FROM: from so many rows on they are read one at a time.
template <typename T, bool VEC, int CL, int IN_FLIGHT, int64_t ONE_FROM>
__global__ __launch_bounds__(1024) void expert_colsum_kernel(const T* __restrict__ src, int64_t ld,
                                                              const int32_t* __restrict__ offsets,
                                                              T* __restrict__ out, int64_t ld_out, int64_t cols) {
    constexpr int PV = VEC ? Elem<T>::kPerVec : 1;
    constexpr int RL = 1024 / CL, COLS = CL * PV;
    constexpr int GROUPS = 1024 / COLS < RL ? 1024 / COLS : RL, PER_GROUP = RL / GROUPS;
    __shared__ float part[RL][COLS + 1];
    const int cl = threadIdx.x % CL, rl = threadIdx.x / CL;
    const int e = blockIdx.y;
    const int64_t chunk = (int64_t)blockIdx.x * CL + cl;
    const int64_t chunks = cols / PV;
    const int64_t begin = offsets[e], end = offsets[e + 1];
    float acc[PV];
#pragma unroll
    for (int q = 0; q < PV; ++q) acc[q] = 0.0f;
    if (chunk < chunks) {
        const T* column = src + chunk * PV;
        int64_t r = begin + rl;
        const int64_t together = end - begin < ONE_FROM ? end : begin;
        for (; r + (IN_FLIGHT - 1) * RL < together; r += IN_FLIGHT * RL) {
            if constexpr (VEC) {
                uint4 v[IN_FLIGHT];
#pragma unroll
                for (int i = 0; i < IN_FLIGHT; ++i) v[i] = load_stream(column + (r + i * RL) * ld);
#pragma unroll
                for (int i = 0; i < IN_FLIGHT; ++i) {
                    float a[PV];
                    Elem<T>::unpack(v[i], a);
#pragma unroll
                    for (int q = 0; q < PV; ++q) acc[q] += a[q];
                }
            } else {
                float v[IN_FLIGHT];
#pragma unroll
                for (int i = 0; i < IN_FLIGHT; ++i) v[i] = Elem<T>::load(column + (r + i * RL) * ld);
#pragma unroll
                for (int i = 0; i < IN_FLIGHT; ++i) acc[0] += v[i];
            }
        }
        for (; r < end; r += RL) {
            if constexpr (VEC) {
                float a[PV];
                Elem<T>::unpack(load_stream(column + r * ld), a);
#pragma unroll
                for (int q = 0; q < PV; ++q) acc[q] += a[q];
            } else {
                acc[0] += Elem<T>::load(column + r * ld);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < PV; ++q) part[rl][cl * PV + q] = acc[q];
    __syncthreads();
    const int c = threadIdx.x % COLS, group = threadIdx.x / COLS;
    if (group < GROUPS) {
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < PER_GROUP; ++i) sum += part[group * PER_GROUP + i][c];
        part[group * PER_GROUP][c] = sum;
    }
    __syncthreads();
    const int64_t column = (int64_t)blockIdx.x * COLS + c;
    if (group == 0 && column < cols) {
        float total = 0.0f;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) total += part[g * PER_GROUP][c];
        Elem<T>::store(out + (int64_t)e * ld_out + column, total);
    }
}

// Few blocks wait for memory, many are bound by it.  By blocks of 32 chunks, us with 32 chunks and one row in flight / 32 and
// two / 32 and four / 8 and four:
//   128 blocks, 2048 rows (16384 x 4096 in 16 bits, 8 experts) 41 / 26 / 26 / 24
//   160, 16 rows (512 x 520 in fp32, 32 experts) 3.1 / 3.1 / 3.1 / 4.2
//   224, 16384 rows (16384 x 28672 in fp32, one expert) 316 / 273 / 282 / 369
//   1024, 4096 rows (131072 x 8192 in 16 bits, 32 experts) 322 / 334 / 374 / 349
// and times the fastest form of each call, from 1024 rows on: 128 blocks 1.59 / 1.05 / 1.09 / 1.01; 160 1.41 / 1.00 / 1.08 / 1.35; 256
// 1.09 / 1.00 / 1.05 / 1.13; 320 1.00 / 1.16 / 1.07 / 1.26; 512 1.00 / 1.09 / 1.05 / 1.10.  Experts of a hundred rows gain from four
// in flight there too (one takes 1.11 times as long at 128 rows of 16 bits, 1.05 at 256, 0.99 at 375; 1.03 and 0.99 at 128 and 256
// in fp32): below kManyRows.
constexpr int64_t kWideColsumBlocks = 160, kManyColsumBlocks = 320, kAnyRows = (int64_t)1 << 62;
template <typename T>
constexpr int64_t kManyRows = Elem<T>::kPerVec * 40;
// Without vectors a chunk is one element, and narrow blocks read few bytes of a row: 32 / 64 chunks, four rows in flight, times
// the fastest: 128 blocks 1.00 / 1.40, 256 1.09 / 1.04, 512 1.39 / 1.00 (8 chunks: 2.35, 2.50, 3.38); 32 blocks 1.5 / 2.8, and 16
// chunks 1.0.
constexpr int64_t kFewScalarColsumBlocks = 64, kManyScalarColsumBlocks = 256;

}  // namespace xma

using namespace xma;

extern "C" {

int xma_add_expert_bias(void* y, int64_t ld_y, const void* bias, int64_t ld_bias, const void* expert_of_row,
                        int se_is_i64, const void* out_index, int idx_is_i64, int64_t rows, int64_t cols, int dtype,
                        void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    XMA_REQUIRE(valid_dtype(dtype), "xma_add_expert_bias: bad dtype %d", dtype);
    XMA_REQUIRE(rows >= 0 && cols >= 0 && ld_y >= cols && ld_bias >= cols, "xma_add_expert_bias: bad shape");
    if (rows == 0 || cols == 0) return 0;
    XMA_REQUIRE(y && bias && expert_of_row, "xma_add_expert_bias: null pointer");
    const int64_t blocks = ceil_div(rows, kBiasRowsPerBlock);
    const dim3 grid((unsigned)(blocks < 256 * 16 ? blocks : 256 * 16)), block(256);
#define XMA_BIAS_LAUNCH(VEC, SeT)                                                                                     \
    hipLaunchKernelGGL((add_expert_bias_kernel<T_, VEC, SeT>), grid, block, 0, stream, (T_*)y, ld_y, (const T_*)bias, \
                       ld_bias, (const SeT*)expert_of_row, out_index, idx_is_i64, rows, cols)
    XMA_DISPATCH_DTYPE(
        dtype, T_,
        const bool vec = aligned16(y) && aligned16(bias) && ld_y % Elem<T_>::kPerVec == 0 &&
                         ld_bias % Elem<T_>::kPerVec == 0 && cols % Elem<T_>::kPerVec == 0;
        if (vec) {
            if (se_is_i64) XMA_BIAS_LAUNCH(true, int64_t);
            else XMA_BIAS_LAUNCH(true, int32_t);
        } else {
            if (se_is_i64) XMA_BIAS_LAUNCH(false, int64_t);
            else XMA_BIAS_LAUNCH(false, int32_t);
        })
#undef XMA_BIAS_LAUNCH
    return check_launch("xma_add_expert_bias");
}

int xma_expert_colsum(const void* src, int64_t ld, const int32_t* expert_offsets, int32_t num_experts, int64_t cols,
                      void* out, int64_t ld_out, int dtype, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    XMA_REQUIRE(valid_dtype(dtype), "xma_expert_colsum: bad dtype %d", dtype);
    XMA_REQUIRE(num_experts >= 1 && num_experts <= 65535 && cols >= 0 && ld >= cols && ld_out >= cols,
                "xma_expert_colsum: bad shape");
    if (cols == 0) return 0;
    XMA_REQUIRE(src && expert_offsets && out, "xma_expert_colsum: null pointer");
    XMA_DISPATCH_DTYPE(
        dtype, T_,
        const bool vec = aligned16(src) && aligned16(out) && ld % Elem<T_>::kPerVec == 0 &&
                         ld_out % Elem<T_>::kPerVec == 0 && cols % Elem<T_>::kPerVec == 0;
        const int64_t chunks = vec ? cols / Elem<T_>::kPerVec : cols;
        const int64_t blocks = ceil_div(chunks, 32) * num_experts;
#define XMA_COLSUM_LAUNCH(VEC, CL, IN_FLIGHT, ONE_FROM)                                                                     \
    hipLaunchKernelGGL((expert_colsum_kernel<T_, VEC, CL, IN_FLIGHT, ONE_FROM>),                                            \
                       dim3((unsigned)ceil_div(chunks, CL), (unsigned)num_experts), dim3(1024), 0, stream, (const T_*)src, ld, \
                       expert_offsets, (T_*)out, ld_out, cols)
        if (vec && blocks < kWideColsumBlocks) XMA_COLSUM_LAUNCH(true, 8, 4, kAnyRows);
        else if (vec && blocks < kManyColsumBlocks) XMA_COLSUM_LAUNCH(true, 32, 2, kAnyRows);
        else if (vec) XMA_COLSUM_LAUNCH(true, 32, 4, kManyRows<T_>);
        else if (blocks < kFewScalarColsumBlocks) XMA_COLSUM_LAUNCH(false, 16, 4, kAnyRows);
        else if (blocks < kManyScalarColsumBlocks) XMA_COLSUM_LAUNCH(false, 32, 4, kAnyRows);
        else XMA_COLSUM_LAUNCH(false, 64, 4, kAnyRows))
#undef XMA_COLSUM_LAUNCH
    return check_launch("xma_expert_colsum");
}

}  // extern "C"
