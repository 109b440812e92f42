// Forward projections (TN) over few routed rows per expert: a decoded token, a serving batch, a short prompt.
//
//   C[p, n] = sum_k A[row(p), k] * W[e][n, k] (+ bias[e][n])     plain, tanh-GELU or gated epilogue
//
// Bound by reading the weights of the experts that are hit, once, from HBM.  The tiled kernels give a compute unit
// 256 weight rows and one wave per SIMD, so a call with a few row tiles leaves most of the device idle and every
// tile waits for its own prologue.  Here a work-group owns 16 * NF weight rows and up to 16 * RF routed rows and its four
// waves SPLIT THE REDUCTION: each streams its quarter of the weight rows straight from memory into matrix-instruction
// operands (no LDS, no barrier, U * NF 16-byte loads of weights in flight per lane and several work-groups per compute
// unit), and the four partial tiles are added in wave order through LDS.  Many small work-groups keep HBM busy
// whatever the number of experts that are hit.
//
// A tile is as tall as the registers allow, so that an expert with many rows has few tiles to stream its weights for, and
// does the work of the 16-row blocks that have a row in them (one, two or all of them): for evenly spread rows that is as
// fast as tiles of just that height, and a skewed call is up to 1.8 times as fast as with tiles of 16 and 32 rows
// (H 2048, I 768, E 128, k 8, 128 tokens, up projection: 82 us by 16 rows, 55 by 32, 45 by 64; even: 140, 137, 136).
//
// A lane loads two adjacent 16-byte chunks, so that the four lanes of a weight row touch a whole 128-byte line with
// each of the two loads; one chunk per 64-byte half line (either half by a load of its own) held 5.0 TB/s where this
// holds 5.9.  A kernel that only reads reaches 6.2.
//
// Measured against tiles of 256 x 256, up + down projection (the smaller tiles of that kernel: see skinny_gemm_supports): H 2048, I 1024, E 64, k 6, one token (6 experts, 75 MB
// of weights) 21 us instead of 82; 16 tokens 117 us instead of 207 (5.6 TB/s of weights); H 4096, I 14336, E 8, k 2,
// 32 tokens 467 us instead of 653 (6.0 TB/s), 64 tokens 484 us instead of 666.  In fp32 (a 128 x 128 register-staged
// kernel before) one token 36 us instead of 248, 16 tokens 225 us with whole lines and 247 with half lines.
// What was chosen by measurement: four waves (eight: 2-5 % slower); U = 2 (4: no gain at 32 x 16 blocks of H 4096, 20 %
// slower at I 768); streaming loads of the weights 7-10 % slower.
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
// RF: 16-row blocks of routed rows of the tallest tile.  U: 64-byte steps of every row requested together.
template <typename T, int NF, int RF, int EPI, int U>
__global__ __launch_bounds__(THREADS) void skinny_gemm_kernel(const GemmParams P) {
    constexpr int PV = Elem<T>::kPerVec;
    constexpr int STEP = 4 * PV;  // reduction elements of one 64-byte step
    constexpr bool PAIRED = EPI == EPI_PAIRED;
    constexpr int NF_OUT = PAIRED ? NF / 2 : NF;  // blocks of output columns
    constexpr int BM = 16 * RF, BN_OUT = 16 * NF_OUT;
    constexpr int PASS = RF < 2 ? RF : 2;  // blocks of routed rows whose partial tiles are in LDS at a time
    static_assert(!PAIRED || NF % 2 == 0, "a gated tile pairs blocks");
    static_assert(U % 2 == 0, "a batch is whole 128-byte lines");
    __shared__ __attribute__((aligned(16))) f32x4_t partial[WAVES][NF * PASS][kWaveSize];

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

    // epilogue of the blocks of routed rows [first_block, first_block + blocks) whose partial tiles are in LDS: a thread
    // owns four adjacent columns of one row (for a gated tile, of both halves)
    auto write_blocks = [&](int first_block, int blocks) {
        T* C = reinterpret_cast<T*>(P.c);
        T* H = reinterpret_cast<T*>(P.aux);
        for (int item = threadIdx.x; item < NF_OUT * blocks * kWaveSize; item += THREADS) {
            const int block = item / kWaveSize, l = item % kWaveSize;
            const int f = block / blocks, r = block % blocks;
            const int64_t p = m_begin + (first_block + r) * 16 + (l & 15);
            const int64_t n = n0 + f * 16 + 4 * (l >> 4);
            if (p >= m_end || n >= n_out) continue;
            auto sum_of = [&](int frag, int64_t column, float (&v)[4]) {
                f32x4_t s = partial[0][frag * PASS + r][l];
#pragma unroll
                for (int wv = 1; wv < WAVES; ++wv) s += partial[wv][frag * PASS + r][l];
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
    };

    // the whole of a tile with LIVE blocks of routed rows
    auto run = [&](auto live_tag) __attribute__((always_inline)) {
        constexpr int LIVE = decltype(live_tag)::value;
        // Rows past the end of the tile or of the weights read an existing row: their results are dropped.
        const T* xp[LIVE];  // rows' starts
        const T* wp[NF];
#pragma unroll
        for (int r = 0; r < LIVE; ++r) {
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

        f32x4_t acc[NF][LIVE];
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < LIVE; ++r) acc[f][r] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

        // this wave's steps, in whole 128-byte lines
        const int steps = (int)((P.k + STEP - 1) / STEP);
        const int per_wave = ((steps + WAVES - 1) / WAVES + 1) / 2 * 2;
        const int first = wave * per_wave < steps ? wave * per_wave : steps;
        const int last = first + per_wave < steps ? first + per_wave : steps;
        const int whole = P.k % STEP == 0 ? last : (last < steps ? last : steps - 1);  // steps without missing elements
        const int batches = whole > first ? (whole - first) / U : 0;

        uint4 w[2][U][NF], x[2][U][LIVE];
        auto load_batch = [&](int set, int step) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // a lane takes two adjacent chunks of a 128-byte line, so either load touches the whole of it
                const int64_t k = (int64_t)(step + (u & ~1)) * STEP + (quarter * 2 + (u & 1)) * PV;
#pragma unroll
                for (int f = 0; f < NF; ++f) w[set][u][f] = *reinterpret_cast<const uint4*>(wp[f] + k);
#pragma unroll
                for (int r = 0; r < LIVE; ++r) x[set][u][r] = *reinterpret_cast<const uint4*>(xp[r] + k);
            }
        };
        auto multiply_batch = [&](int set) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int r = 0; r < LIVE; ++r) mma<T>(w[set][u][f], x[set][u][r], acc[f][r]);
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
            uint4 wv[NF], xv[LIVE];
#pragma unroll
            for (int f = 0; f < NF; ++f) wv[f] = exists ? *reinterpret_cast<const uint4*>(wp[f] + k) : zero;
#pragma unroll
            for (int r = 0; r < LIVE; ++r) xv[r] = exists ? *reinterpret_cast<const uint4*>(xp[r] + k) : zero;
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int r = 0; r < LIVE; ++r) mma<T>(wv[f], xv[r], acc[f][r]);
        }

#pragma unroll
        for (int r0 = 0; r0 < LIVE; r0 += PASS) {
            constexpr int HERE = LIVE < PASS ? LIVE : PASS;
            if (r0 > 0) __syncthreads();  // the partial tiles of the blocks ahead are read
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int r = 0; r < HERE; ++r)
                    if (r0 + r < LIVE) partial[wave][f * PASS + r][lane] = acc[f][r0 + r];
            __syncthreads();
            write_blocks(r0, LIVE - r0 < PASS ? LIVE - r0 : PASS);
        }
    };
    const int live = (m_end - m_begin + 15) / 16;
    if constexpr (RF == 4) {
        if (live > 2) return run(std::integral_constant<int, 4>{});
    }
    if constexpr (RF >= 2) {
        if (live > 1) return run(std::integral_constant<int, 2>{});
    }
    run(std::integral_constant<int, 1>{});
}

template <typename T, int NF, int RF, int EPI>
static int launch(const xma_grouped_gemm_args& a, hipStream_t stream) {
    GemmParams P;
    fill_params(a, P);
    const int64_t n_out = EPI == EPI_PAIRED ? a.n / 2 : a.n;
    P.col_tiles = (int32_t)ceil_div(n_out, EPI == EPI_PAIRED ? 8 * NF : 16 * NF);
    const int64_t row_tiles = a.rows / (16 * RF) + (a.rows < a.num_experts ? a.rows : a.num_experts);
    const int64_t grid = row_tiles * P.col_tiles;
    XMA_REQUIRE(grid < ((int64_t)1 << 31), "xma_grouped_gemm: %lld tiles exceed the grid limit", (long long)grid);
    hipLaunchKernelGGL((skinny_gemm_kernel<T, NF, RF, EPI, 2>), dim3((unsigned)grid), dim3(THREADS), 0, stream, P);
    return check_launch("xma_grouped_gemm");
}

template <typename T>
static int dispatch(const xma_grouped_gemm_args& a, hipStream_t stream) {
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    const GemmForm form = skinny_gemm_form(a);
#define XMA_SKINNY(NF, RF)                              \
    if (form.tile_cols == 16 * NF && form.tile_rows == 16 * RF) \
    return shape == EPI_PAIRED ? launch<T, NF, RF, EPI_PAIRED>(a, stream) : launch<T, NF, RF, EPI_PLAIN>(a, stream)
    XMA_SKINNY(2, 1);
    XMA_SKINNY(2, 2);
    XMA_SKINNY(4, 2);
    if constexpr (!std::is_same<T, float>::value) {
        XMA_SKINNY(4, 1);
        XMA_SKINNY(4, 4);
        XMA_SKINNY(8, 4);
    }
#undef XMA_SKINNY
    set_error("xma_grouped_gemm: no streaming kernel of %d x %d", form.tile_cols, form.tile_rows);
    return 1;
}

// ---- which calls stream, by which tiles ------------------------------------------------------------------------
// An expert's weights are streamed once per row tile, so what a call costs depends on how its rows fall on the experts,
// which only the device knows; the rules here see the number of rows and of experts.  Both ways are measured: rows spread
// evenly, and skewed (logits falling like Zipf's law, s = 1.2: a quarter of 128 experts is hit, the first one by
// every token).  A skewed call may stream the weights of one expert many times.  bf16, us, up projection unless
// said otherwise, this kernel / the 256 x 256 kernel, by rows per expert on average:
//   H 4096, I 14336, E 8: 8 rows 306 / 429, skewed 201 / 341; 20 rows 319 / 431, 368 / 434; 40 rows 359 / 434, 451 / 440
//     down: 26 rows 176 / 223, skewed 216 / 217; 40 rows 203 / 218, skewed 265 / 217
//   H 4096, I 8192, E 8, down: 26 rows 123 / 171, skewed 112 / 147; 40 rows 129 / 166, skewed 145 / 149
//   H 2048, I 4096, E 32, down: 26 rows 112 / 133, skewed 81 / 91; 40 rows 123 / 133, skewed 110 / 94
//   H 2048, I 1024, E 64: 8 rows 95 / 153, skewed 48 / 53; 20 rows 99 / 153, 64 / 57; 40 rows 125 / 154, 102 / 102
//     down (k 1024): 26 rows 60 / 57
//   H 2048, I 768, E 128: 8 rows 137 / 189, skewed 55 / 54; 20 rows 148 / 193, 82 / 59; 40 rows 186 / 196, 137 / 103
//   H 512, I 1024, E 4, down (k 1024): 26 rows 10 / 26
// Up to kSkinnyTwoBlocks rows per expert every call streams.  Up to kSkinnyRows those do whose reductions are long but
// not longest (the tiled kernel pays its prologue per tile, and cuts the longest reductions until the device is
// full) or whose projection is wide, and of the short reductions those of too few tiles of 256 x 256 to fill the device.
// Beyond kSkinnyRows even calls gain nothing (128 experts at 64 rows: 255 / 223).
// These lines were drawn against tiles of 256 x 256.  A call that does not stream now takes tiles of up to 192 x 128 where they are
// faster, and against those it streams for too long.  This kernel / the fastest tiles, up projection, even calls, us by rows:
//   H 4096, I 14336, E 8: 8 rows 331 / 339, 20 rows 359 / 350, 40 rows 388 / 379; down 8 rows 168 / 173, 20 rows 173 / 167
//   H 2048, I 1024, E 64: 8 rows 100 / 129, 20 rows 110 / 128, 40 rows 132 / 131; down 44 / 43, 50 / 42
//   H 2048, I 768, E 128: 8 rows 149 / 156, 20 rows 168 / 192, 40 rows 195 / 162; down 79 / 78, 20 rows 95 / 81; skewed, 20 rows
//     180 / 213, down 106 / 96, 40 rows up 230 / 197
//   H 2048, I 8192, E 16: 8 rows 195 / 196, 20 rows 218 / 196, 40 rows 260 / 200; down 115 / 132, 127 / 132, 131 / 131
//   H 2048, I 1024, E 8: 8 rows 15 / 21, 20 rows 17 / 21, 40 rows 21 / 23
//   H 1024, I 4096, E 128, down: 8 rows 184 / 190, 20 rows 210 / 192, 40 rows 253 / 196
// Median over 1270 calls that stream: 0.93 of the fastest tiles at 8 rows, 1.05 at 14, 1.10 at 20, 1.16 at 30, 1.25 at 40.
constexpr int kSkinnyRows = 40;
constexpr int kSkinnyTwoBlocks = 20;
constexpr int kSkinnyOneBlock = 8;
constexpr int64_t kSkinnyLongReduction = 2048, kSkinnyLongestReduction = 8192;
constexpr int64_t kSkinnyWideTiles = 1024;  // work-groups of 128 weight rows
constexpr int64_t kSkinnyDevice = 256;      // compute units
// fp32, against the fp32 kernel with its tiles of 32 rows: H 2048, I 1024, E 64: 8 rows 184 / 191, down 102 / 131, skewed
// 116 / 93; 12 rows 201 / 193, skewed 152 / 123; H 2048, I 8192, E 8, down, whose tiles are half as many as there are
// compute units: 20 rows 126 / 245, 24 rows 240 / 245.
constexpr int kSkinnyRowsF32 = 24;

// work-groups of the tiled kernels when every expert has one row tile
static int64_t tiled_work_groups(const xma_grouped_gemm_args& a) {
    if (a.dtype != XMA_F32) return ceil_div(a.n, 256) * a.num_experts;
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    return (shape == EPI_PAIRED ? ceil_div(a.n / 2, 64) : ceil_div(a.n, 128)) * a.num_experts;
}

}  // namespace skinny

bool skinny_gemm_supports(const xma_grouped_gemm_args& a) {
    using namespace skinny;
    if (a.kind != XMA_GEMM_TN || a.k <= 0 || a.num_experts > kMaxScannedExperts) return false;
    const int64_t experts = a.num_experts;
    const bool fp32 = a.dtype == XMA_F32;
    if (a.rows <= (fp32 ? kSkinnyOneBlock : kSkinnyTwoBlocks) * experts) return true;
    if (a.rows > (fp32 ? kSkinnyRowsF32 : kSkinnyRows) * experts) return false;
    if (fp32) return tiled_work_groups(a) < kSkinnyDevice;
    if (a.k < kSkinnyLongReduction) return tiled_work_groups(a) <= kSkinnyDevice;
    return a.k <= kSkinnyLongestReduction || a.n / 128 * experts >= kSkinnyWideTiles;
}

// A tall tile costs what its blocks of 16 rows with a row in them cost, but for the registers it needs, which leave room for
// fewer work-groups.  us, up / down projection by weight rows x routed rows of the tile:
//   H 2048, I 768, E 128, 4 rows per expert: 32 x 16 135 / 74, 32 x 32 133 / 78, 64 x 32 134 / 72, 64 x 64 133 / 78; 8 rows,
//     skewed: 82 / 46, 63 / 38, 55 / 30, 45 / 29; 14 rows: 64 x 32 141 / 89, 64 x 64 140 / 92, skewed 80 / 45, 66 / 41
//   H 2048, I 1024, E 64, 4 rows, skewed: 32 x 16 38 / 21, 32 x 32 34 / 20; even: 92 / 43, 91 / 42
//   H 576, I 256, E 128, 1 row: 32 x 16 13.3 / 9.4, 32 x 32 14.5 / 10.6, 64 x 32 14.3 / 9.6
//   H 4096, I 14336, E 8, 8 rows: up 64 x 16 305, 64 x 32 306, skewed 259, 201; 26 / 40 rows: 64 x 64 337 / 384, 128 x 64 333 / 359
//   H 2048, I 4096, E 32, 26 / 40 rows: 64 x 64 201 / 238, 128 x 64 212 / 244
// (64 x 32 pays from kSkinnyManyRows rows on, where a skewed call has so many more row tiles that taller ones are worth
// their registers, or with kSkinnyManyColumns, which fill the device all the same)
constexpr int64_t kSkinnyManyColumns = 16384;
constexpr int64_t kSkinnyManyRows = 512;
GemmForm skinny_gemm_form(const xma_grouped_gemm_args& a) {
    using namespace skinny;
    const int64_t experts = a.num_experts;
    const bool fp32 = a.dtype == XMA_F32;
    const bool many_columns = !fp32 && a.n >= kSkinnyManyColumns;
    int nf, rf;
    if (a.rows <= 16) {  // one tile per expert
        nf = many_columns ? 4 : 2;
        rf = 1;
    } else if (a.rows <= kSkinnyOneBlock * experts) {
        nf = many_columns || (!fp32 && a.rows >= kSkinnyManyRows) ? 4 : 2;
        rf = nf == 2 && !fp32 && a.k < 1024 ? 1 : 2;
    } else if (fp32 || (a.rows <= kSkinnyTwoBlocks * experts && a.k < kSkinnyLongReduction)) {
        nf = 4;
        rf = 2;
    } else {
        nf = many_columns && a.rows > kSkinnyTwoBlocks * experts ? 8 : 4;
        rf = 4;
    }
    return {XMA_FORM_STREAMING, 16 * rf, 16 * nf};
}

int launch_skinny_gemm(const xma_grouped_gemm_args& a, hipStream_t stream) {
    if (a.dtype == XMA_F32) return skinny::dispatch<float>(a, stream);
    return a.dtype == XMA_BF16 ? skinny::dispatch<bf16_t>(a, stream) : skinny::dispatch<f16_t>(a, stream);
}

}  // namespace xma
