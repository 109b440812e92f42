// Forward projections (TN) over few routed rows per expert: a decoded token, a serving batch, a short prompt.
//
//   C[p, n] = sum_k A[row(p), k] * W[e][n, k] (+ bias[e][n])     plain, tanh-GELU or gated epilogue
//
// Bound by reading the weights of the experts that are hit, once, from HBM.  The tiled kernels give a compute unit
// 256 weight rows and one wave per SIMD, so a call with a few row tiles leaves most of the device idle and every
// tile waits for its own prologue.  Here a work-group owns 16 * NF weight rows and 16 * RF routed rows and its four
// waves SPLIT THE REDUCTION: each streams its quarter of the weight rows straight from memory into matrix-instruction
// operands (no LDS, no barrier, U * NF 16-byte loads of weights in flight per lane and several work-groups per compute
// unit), and the four partial tiles are added in wave order through LDS.  Many small work-groups keep HBM busy
// whatever the number of experts that are hit.
//
// A lane loads two adjacent 16-byte chunks, so that the four lanes of a weight row touch a whole 128-byte line with
// each of the two loads; one chunk per 64-byte half line (either half by a load of its own) held 5.0 TB/s where this
// holds 5.9.  A kernel that only reads reaches 6.2.
//
// Measured against the 256 x 256 kernel, up + down projection: H 2048, I 1024, E 64, k 6, one token (6 experts, 75 MB
// of weights) 21 us instead of 82; 16 tokens 117 us instead of 207 (5.6 TB/s of weights); H 4096, I 14336, E 8, k 2,
// 32 tokens 467 us instead of 653 (6.0 TB/s), 64 tokens 484 us instead of 666.  In fp32 (a 128 x 128 register-staged
// kernel before) one token 36 us instead of 248, 16 tokens 225 us with whole lines and 247 with half lines.
// What was chosen by measurement: four waves (eight: 2-5 % slower); U = 2 (4: no gain at 32 x 16 blocks of H 4096, 20 %
// slower at I 768); streaming loads of the weights 7-10 % slower; 64 x 16 blocks only for many columns (3 % there, 20-30 %
// slower for the smallest layers).
//
// Which rows a work-group has is found by each wave on its own from the expert offsets (RowTileScan), so there is
// no table to build in a launch of its own.
#include <type_traits>

#include "grouped_gemm_common.h"

namespace xma {
namespace skinny {

constexpr int THREADS = 256, WAVES = THREADS / kWaveSize;

// acc(16 x 16) += W(16 weight rows x 4 chunks) * X(16 routed rows x 4 chunks)^T where lane l supplies the 16-byte chunk
// l / 16 of row l % 16 of both operands; register r of lane l is [weight row 4 * (l / 16) + r][routed row l % 16].
// The order in which a chunk's elements meet the matrix instruction's reduction slots does not matter as long as it is
// the same for both operands.
template <typename T>
__device__ __forceinline__ void mma(const uint4& w, const uint4& x, f32x4_t& acc) {
    if constexpr (std::is_same<T, float>::value) {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.x), __uint_as_float(x.x), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.y), __uint_as_float(x.y), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.z), __uint_as_float(x.z), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.w), __uint_as_float(x.w), acc, 0, 0, 0);
    } else if constexpr (std::is_same<T, bf16_t>::value) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x),
                                                      acc, 0, 0, 0);
    } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, w), __builtin_bit_cast(f16x8_t, x), acc,
                                                     0, 0, 0);
    }
}

// value as the layer's type holds it
template <typename T>
__device__ __forceinline__ float rounded(float v) {
    if constexpr (std::is_same<T, float>::value) return v;
    T t;
    Elem<T>::store(&t, v);
    return Elem<T>::load(&t);
}

template <typename T>
__device__ __forceinline__ void store4(T* p, const float (&v)[4]) {
    if constexpr (std::is_same<T, float>::value)
        *reinterpret_cast<uint4*>(p) = Elem<float>::pack(v);
    else
        *reinterpret_cast<uint2*>(p) = make_uint2(Elem<T>::pack2(v[0], v[1]), Elem<T>::pack2(v[2], v[3]));
}
template <typename T>
__device__ __forceinline__ void load4(const T* p, float (&v)[4]) {
    if constexpr (std::is_same<T, float>::value) {
        Elem<float>::unpack(*reinterpret_cast<const uint4*>(p), v);
    } else {
        const uint2 raw = *reinterpret_cast<const uint2*>(p);
        float u[8];
        Elem<T>::unpack(make_uint4(raw.x, raw.y, 0u, 0u), u);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = u[q];
    }
}

// NF: 16-row blocks of weights per work-group; a gated tile (EPI_PAIRED) takes NF / 2 blocks of each half.
// RF: 16-row blocks of routed rows.  U: 64-byte steps of every row requested together.
template <typename T, int NF, int RF, int EPI, int U>
__global__ __launch_bounds__(THREADS) void skinny_gemm_kernel(const GemmParams P) {
    constexpr int PV = Elem<T>::kPerVec;
    constexpr int STEP = 4 * PV;  // reduction elements of one 64-byte step
    constexpr bool PAIRED = EPI == EPI_PAIRED;
    constexpr int NF_OUT = PAIRED ? NF / 2 : NF;  // blocks of output columns
    constexpr int BM = 16 * RF, BN_OUT = 16 * NF_OUT;
    static_assert(!PAIRED || NF % 2 == 0, "a gated tile pairs blocks");
    static_assert(U % 2 == 0, "a batch is whole 128-byte lines");
    __shared__ __attribute__((aligned(16))) f32x4_t partial[WAVES][NF * RF][kWaveSize];

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWaveSize);
    const int row_tile = blockIdx.x / P.col_tiles;
    const int col_tile = blockIdx.x - row_tile * P.col_tiles;

    int expert = 0;
    int32_t m_begin, m_end;
    const RowTileScan tiles(P.offsets, P.num_experts, BM, lane);
    if (row_tile >= tiles.total) return;  // (the same for every wave of the work-group)
    tiles.find(row_tile, expert, m_begin, m_end);

    const T* A = reinterpret_cast<const T*>(P.a);
    const T* W = reinterpret_cast<const T*>(P.b) + (int64_t)expert * P.b_expert_stride;
    const int64_t n_out = PAIRED ? P.n / 2 : P.n;
    const int64_t n0 = (int64_t)col_tile * BN_OUT;
    const int row16 = lane & 15, quarter = lane >> 4;

    // Rows past the end of the tile or of the weights read an existing row: their results are dropped.
    const T* xp[RF];  // rows' starts
    const T* wp[NF];
#pragma unroll
    for (int r = 0; r < RF; ++r) {
        int64_t p = m_begin + r * 16 + row16;
        p = p < m_end ? p : m_end - 1;
        const int64_t src = P.in_index ? source_row(P, p) : p;
        xp[r] = A + src * P.lda;
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        int64_t n = n0 + (f % NF_OUT) * 16 + row16;
        n = n < n_out ? n : n_out - 1;
        wp[f] = W + (n + (f >= NF_OUT ? n_out : 0)) * P.ldb;
    }

    f32x4_t acc[NF][RF];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < RF; ++r) acc[f][r] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // this wave's steps, in whole 128-byte lines
    const int steps = (int)((P.k + STEP - 1) / STEP);
    const int per_wave = ((steps + WAVES - 1) / WAVES + 1) / 2 * 2;
    const int first = wave * per_wave < steps ? wave * per_wave : steps;
    const int last = first + per_wave < steps ? first + per_wave : steps;
    const int whole = P.k % STEP == 0 ? last : (last < steps ? last : steps - 1);  // steps without missing elements
    const int batches = whole > first ? (whole - first) / U : 0;

    uint4 w[2][U][NF], x[2][U][RF];
    auto load_batch = [&](int set, int step) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // a lane takes two adjacent chunks of a 128-byte line, so either load touches the whole of it
            const int64_t k = (int64_t)(step + (u & ~1)) * STEP + (quarter * 2 + (u & 1)) * PV;
#pragma unroll
            for (int f = 0; f < NF; ++f) w[set][u][f] = *reinterpret_cast<const uint4*>(wp[f] + k);
#pragma unroll
            for (int r = 0; r < RF; ++r) x[set][u][r] = *reinterpret_cast<const uint4*>(xp[r] + k);
        }
    };
    auto multiply_batch = [&](int set) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int r = 0; r < RF; ++r) mma<T>(w[set][u][f], x[set][u][r], acc[f][r]);
    };
    if (batches > 0) load_batch(0, first);
    for (int b = 0; b < batches; b += 2) {
        if (b + 1 < batches) load_batch(1, first + (b + 1) * U);
        multiply_batch(0);
        if (b + 1 < batches) {
            if (b + 2 < batches) load_batch(0, first + (b + 2) * U);
            multiply_batch(1);
        }
    }
    // the remaining steps one by one; elements past the end of the reduction are zero in both operands
    for (int s = first + batches * U; s < last; ++s) {
        const int64_t k = (int64_t)s * STEP + quarter * PV;
        const bool exists = k < P.k;
        const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
        uint4 wv[NF], xv[RF];
#pragma unroll
        for (int f = 0; f < NF; ++f) wv[f] = exists ? *reinterpret_cast<const uint4*>(wp[f] + k) : zero;
#pragma unroll
        for (int r = 0; r < RF; ++r) xv[r] = exists ? *reinterpret_cast<const uint4*>(xp[r] + k) : zero;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < RF; ++r) mma<T>(wv[f], xv[r], acc[f][r]);
    }

#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < RF; ++r) partial[wave][f * RF + r][lane] = acc[f][r];
    __syncthreads();

    // epilogue: a thread owns four adjacent columns of one row (for a gated tile, of both halves)
    T* C = reinterpret_cast<T*>(P.c);
    T* H = reinterpret_cast<T*>(P.aux);
    for (int item = threadIdx.x; item < NF_OUT * RF * kWaveSize; item += THREADS) {
        const int block = item / kWaveSize, l = item % kWaveSize;
        const int f = block / RF, r = block % RF;
        const int64_t p = m_begin + r * 16 + (l & 15);
        const int64_t n = n0 + f * 16 + 4 * (l >> 4);
        if (p >= m_end || n >= n_out) continue;
        auto sum_of = [&](int frag, int64_t column, float (&v)[4]) {
            f32x4_t s = partial[0][frag * RF + r][l];
#pragma unroll
            for (int wv = 1; wv < WAVES; ++wv) s += partial[wv][frag * RF + r][l];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = s[q];
            if (P.bias != nullptr) {
                float b[4];
                load4(reinterpret_cast<const T*>(P.bias) + (int64_t)expert * P.ld_bias + column, b);
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] += b[q];
            }
        };
        const int64_t out_row = P.out_index ? load_index(P.out_index, P.idx_is_i64, p) : p;
        constexpr bool FAST = !std::is_same<T, float>::value;
        float v[4], o[4];
        sum_of(f, n, v);
        if constexpr (PAIRED) {
            float g[4];
            sum_of(f + NF_OUT, n_out + n, g);
            if (H) {
                store4(H + p * P.ld_aux + n, v);
                store4(H + p * P.ld_aux + n_out + n, g);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q] = gated_forward<FAST>(P.act, rounded<T>(v[q]), rounded<T>(g[q]));
            store4(C + out_row * P.ldc + n, o);
        } else if (P.act == ACT_GELU_TANH) {
            if (H) store4(H + p * P.ld_aux + n, v);
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q] = gelu_tanh_forward<FAST>(rounded<T>(v[q]));
            store4(C + out_row * P.ldc + n, o);
        } else {
            store4(C + out_row * P.ldc + n, v);
        }
    }
}

template <typename T, int NF, int RF, int EPI, int U>
static int launch(const GemmParams& params, int64_t rows, hipStream_t stream) {
    GemmParams P = params;
    const int64_t n_out = EPI == EPI_PAIRED ? P.n / 2 : P.n;
    P.col_tiles = (int32_t)ceil_div(n_out, EPI == EPI_PAIRED ? 8 * NF : 16 * NF);
    const int64_t row_tiles = rows / (16 * RF) + (rows < P.num_experts ? rows : P.num_experts);
    const int64_t grid = row_tiles * P.col_tiles;
    XMA_REQUIRE(grid < ((int64_t)1 << 31), "xma_grouped_gemm: %lld tiles exceed the grid limit", (long long)grid);
    hipLaunchKernelGGL((skinny_gemm_kernel<T, NF, RF, EPI, U>), dim3((unsigned)grid), dim3(THREADS), 0, stream, P);
    return check_launch("xma_grouped_gemm");
}

// work-groups of the 128 x 64 form when every expert has one row tile
static int64_t wide_tiles(const xma_grouped_gemm_args& a) { return a.n / 128 * a.num_experts; }

template <typename T>
static int dispatch(const xma_grouped_gemm_args& a, const GemmParams& P, hipStream_t stream) {
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    constexpr bool FP32 = std::is_same<T, float>::value;
#define XMA_SKINNY(NF, RF)                                                             \
    (shape == EPI_PAIRED ? launch<T, NF, RF, EPI_PAIRED, 2>(P, a.rows, stream)          \
                         : launch<T, NF, RF, EPI_PLAIN, 2>(P, a.rows, stream))
    if (a.rows <= kSkinnyOneBlock * (int64_t)a.num_experts) {
        if constexpr (!FP32)
            if (a.n >= kSkinnyWideColumns) return XMA_SKINNY(4, 1);
        return XMA_SKINNY(2, 1);
    }
    if constexpr (!FP32) {
        if (a.rows > kSkinnyTwoBlocks * (int64_t)a.num_experts)
            return wide_tiles(a) >= kSkinnyWideTiles ? XMA_SKINNY(8, 4) : XMA_SKINNY(4, 4);
    }
    return XMA_SKINNY(4, 2);
#undef XMA_SKINNY
}

}  // namespace skinny

bool skinny_gemm_supports(const xma_grouped_gemm_args& a) {
    if (a.kind != XMA_GEMM_TN || a.k <= 0 || a.num_experts > kMaxScannedExperts) return false;
    const int64_t experts = a.num_experts;
    if (a.dtype == XMA_F32) return a.rows <= kSkinnyRowsF32 * experts;
    if (a.rows <= kSkinnyTwoBlocks * experts) return true;
    if (a.rows > kSkinnyRows * experts) return false;
    if (a.k < kSkinnyLongReduction) return ceil_div(a.n, 256) * experts <= kSkinnyTiledRound;
    return a.n < 4096 || skinny::wide_tiles(a) >= kSkinnyWideTiles;
}

int launch_skinny_gemm(const xma_grouped_gemm_args& a, hipStream_t stream) {
    GemmParams P;
    fill_params(a, P);
    if (a.dtype == XMA_F32) return skinny::dispatch<float>(a, P, stream);
    return a.dtype == XMA_BF16 ? skinny::dispatch<bf16_t>(a, P, stream) : skinny::dispatch<f16_t>(a, P, stream);
}

}  // namespace xma
