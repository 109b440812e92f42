// Ragged (per-expert) GEMM in true fp32 on gfx950 (v_mfma_f32_32x32x2_f32), all three operand layouts.
//
// Bound by the matrix cores: a 32 x 32 x 2 step takes 64 cycles, sixteen times the time per FLOP of the 16-bit kernels,
// so operands are a small stream next to it (32 FLOP per byte of L2 traffic in a 128 x 128 tile) and what is left to lose
// is (1) everything a wave does between matrix instructions and (2) rows of a tile that do not exist.
//   (1) Loads go L2 -> LDS without registers (global_load_lds_dwordx4), two stages of 32 reduction elements deep, one
//       barrier per stage, two or more work-groups per compute unit to fill each other's gaps.  The matrix instruction
//       takes one fp32 element per lane, so an operand whose reduction index is strided in HBM is used in its HBM
//       layout (32 lanes read 32 adjacent elements of a reduction row): nothing is transposed.
//   (2) The four waves split the COLUMNS of a tile, every wave has all of its rows: a tile with few rows leaves out
//       whole 32-row blocks in every wave alike, so an expert's last tile costs what its rows cost.
// The tile height (32 * MB rows) is chosen so that small calls still fill the device.
//
// Measured (157 TFLOP/s nominal, a large library product 0.153): 8 groups of 1024 rows, N 8192, K 2048, TFLOP/s TN / NN /
// MT 140 / 145 / 139 against 123 / 117 / 110 for the register-staged 128 x 128 kernel this one replaces and 145 for a loop
// of library products; 8 groups of about 256 rows, H 256, I 512, up + down projection 36 us instead of 93 us.  What made
// the difference beyond the loads: dealing them out between the matrix instructions (136 -> 146 TFLOP/s at K 4096),
// pinning the LDS reads ahead (129 -> 136).  With the loads left out altogether the loop reaches 151.
//
// Tile layouts in LDS, one stage of 32 reduction elements:
//   K-contiguous operand: [tile rows][32], 128-byte rows, 16-byte chunk c of row r at c ^ ((r >> 1) & 7): the sixteen
//     rows a quarter wave reads in one ds_read_b128 cover all 64 banks;
//   K-strided operand: [32][tile rows], read one element per lane.
// Lane l = (h = l / 32, i = l % 32) of matrix instruction j of group kk takes reduction element 8 kk + 4 h + j of both.
#include <type_traits>

#include "grouped_gemm_common.h"

namespace xma {
namespace f32 {

constexpr int BN = 128, BK = 32, THREADS = 256, WAVES = 4, KK = BK / 8;
constexpr int kRowBytes = BK * 4;
constexpr int64_t kFullDeviceTiles = 512;  // two work-groups on every compute unit

// Split of a partly filled last round (see locate_work).  A stage of a 128 x 128 tile takes 3.7 us with two work-groups on a
// compute unit, so a part of 16 stages (of flatter tiles, as many times more) is already worth an exchange of 64 KiB, and a
// last round matters up to many rounds.  A last round of more tiles than half the compute units is left alone: a work-group
// that has a compute unit to itself runs almost at the rate of two.  8192 rows, 8 experts, 2048 columns, us without / with:
// K 8192 (1088 tiles, 64 of them in the third round) 2412 / 2117, K 16384 5022 / 4366; last rounds of 256 tiles cut in two
// or three: 1713 / 1820 (K 4096), 314 / 334 (K 2048).
constexpr int kSplitStages = 16, kSplitParts = 8, kSplitRounds = 32, kSplitTiles = 128;
constexpr double kSplitFlops = 2e10;  // below that (0.14 ms) the launch that clears the counters costs what a split gains

__device__ __attribute__((aligned(16))) uint32_t zero_chunk[4];  // zero-initialised

__device__ __forceinline__ void wait_loads_and_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (0 << 8));  // vmcnt = 0, lgkmcnt = 0
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void block_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ int opaque(int v) {
    asm("" : "+v"(v));
    return v;
}

// The loads of one operand of R tile rows.  Load i of wave w fills the 1 KiB block (4 i + w) of the operand's tile.
// Whatever does not exist (rows and columns outside the operand, the end of the reduction) is fetched from a chunk of
// zeros, so every lane takes part in every load.  A load of a stage inside the reduction costs one 64-bit add: missing
// rows stand still on the chunk of zeros.
template <int R, bool STRIDED>
struct Loads {
    static constexpr int LOADS = R / 32;
    static constexpr int CHUNKS = STRIDED ? R / 4 : kRowBytes / 16;  // 16-byte chunks per LDS row
    static constexpr int ROWS = 64 / CHUNKS;                          // LDS rows per load
    const float* ptr[LOADS];                  // the lane's chunk in the stage that is requested next
    int64_t step[STRIDED ? 1 : LOADS];        // elements from stage to stage, 0 for what does not exist
    int32_t red0;                             // reduction index of load 0 in stage 0
    static constexpr int RED_STEP = STRIDED ? 4 * ROWS : 0;  // ... from load to load

    __device__ static __forceinline__ const float* zeros() { return reinterpret_cast<const float*>(zero_chunk); }

    // row_fn(tile row) returns the HBM row base or nullptr
    template <typename RowFn>
    __device__ __forceinline__ void setup_rows(int wave, int lane, RowFn row_fn) {
        static_assert(!STRIDED, "layout");
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int row = (4 * i + wave) * ROWS + lane / CHUNKS;
            const int chunk = (lane % CHUNKS) ^ ((row >> 1) & 7);  // the same for every i
            const float* base = row_fn(row);
            ptr[i] = base != nullptr ? base + chunk * 4 : zeros();
            step[i] = base != nullptr ? BK : 0;
            red0 = chunk * 4;
        }
    }
    // `base` points at (reduction row 0, first tile column); `left` columns exist from there
    __device__ __forceinline__ void setup_strided(int wave, int lane, const float* base, int64_t ld, int64_t left) {
        static_assert(STRIDED, "layout");
        const int chunk = lane % CHUNKS;
        const bool exists = chunk * 4 < left;
        red0 = wave * ROWS + lane / CHUNKS;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) ptr[i] = exists ? base + (int64_t)(red0 + i * RED_STEP) * ld + chunk * 4 : zeros();
        step[0] = exists ? BK * ld : 0;
    }
    // Make stage 0 the stage `first` of the reduction (the parts of a split tile start in the middle).
    __device__ __forceinline__ void skip_stages(int first) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) ptr[i] += first * step[STRIDED ? 0 : i];
    }
    // Load i of a stage of which the first `left` reduction elements exist (WHOLE: all BK).
    template <bool WHOLE>
    __device__ __forceinline__ void issue(int i, char* tile, int wave, int left) {
        send(tile, i, wave, WHOLE || red0 + i * RED_STEP < left ? ptr[i] : zeros());
        ptr[i] += step[STRIDED ? 0 : i];
    }
    // the same for a K-strided operand whose reduction rows are gathered: `row` is the source row
    __device__ __forceinline__ void issue_gathered(int i, char* tile, int wave, int left, const float* base, int64_t ld,
                                                   int lane, int32_t row) const {
        const bool ok = step[0] != 0 && red0 + i * RED_STEP < left;
        send(tile, i, wave, ok ? base + row * ld + (lane % CHUNKS) * 4 : zeros());
    }
    __device__ __forceinline__ static void send(char* tile, int i, int wave, const float* p) {
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t*>(p),
                                         (__attribute__((address_space(3))) void*)(tile + (i * 4096 + wave * 1024)), 16, 0, 0);
    }
};

// The four elements (reduction 8 kk + 4 h .. + 3) of tile row `row` of one operand.  `var` is the lane's part of the
// address: for the K-contiguous layout one per kk, for the K-strided one a single offset.
template <int R, bool STRIDED>
__device__ __forceinline__ f32x4_t read_fragment(const char* tile, const int (&var)[KK], int block, int kk) {
    if constexpr (STRIDED) {
        f32x4_t v;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = *reinterpret_cast<const float*>(tile + (var[0] + ((8 * kk + j) * R + 32 * block) * 4));
        return v;
    } else {
        return *reinterpret_cast<const f32x4_t*>(tile + (var[kk] + block * 32 * kRowBytes));
    }
}
template <int R, bool STRIDED>
__device__ __forceinline__ void fragment_offsets(int row0, int lane, int (&var)[KK]) {
    const int i = lane & 31, h = lane >> 5;
    if constexpr (STRIDED) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) var[kk] = 0;
        var[0] = opaque((4 * h * R + row0 + i) * 4);
    } else {
        const int row = row0 + i;  // row0 is a multiple of 32: the swizzle is the same for every block
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) var[kk] = opaque(row * kRowBytes + (((2 * kk + h) ^ ((row >> 1) & 7)) << 4));
    }
}

template <int MB, int KIND, int EPI>
__global__ __launch_bounds__(THREADS, 2) void gemm_kernel(const GemmParams P) {
    constexpr int BM = 32 * MB;
    constexpr bool A_STRIDED = KIND == XMA_GEMM_MT, B_STRIDED = KIND != XMA_GEMM_TN;
    constexpr int BN_OUT = EPI == EPI_PAIRED ? BN / 2 : BN;
    constexpr int A_BYTES = BM * kRowBytes, STAGE_BYTES = A_BYTES + BN * kRowBytes;
    // two arrays, so that the compiler sees that reads of one stage do not touch the loads in flight to the other
    __shared__ __attribute__((aligned(1024))) char even_stage[STAGE_BYTES];
    __shared__ __attribute__((aligned(1024))) char odd_stage[STAGE_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- which tile ----
    const bool table = KIND == XMA_GEMM_MT || P.tile_count != nullptr;
    const RowTileScan tiles(P.offsets, table ? 0 : P.num_experts, BM, lane);
    const int row_tiles =
        KIND == XMA_GEMM_MT ? P.row_tiles_max * P.num_experts : table ? P.tile_count[0] : tiles.total;
    int row_tile, col_tile;
    TileWork work;
    work.parts = 1;
    if constexpr (KIND == XMA_GEMM_MT) {
        if (!locate_tile<true>(row_tiles, P.col_tiles, row_tile, col_tile)) return;
    } else {
        if (!locate_work<false>(row_tiles, P.col_tiles, P.round_tiles, P.most_parts, kSplitRounds, kSplitTiles, work)) return;
        row_tile = work.row_tile;
        col_tile = work.col_tile;
    }

    const float* A = reinterpret_cast<const float*>(P.a);
    const float* B = reinterpret_cast<const float*>(P.b);
    int expert;
    int64_t m_begin, m_end, tile_i0 = 0, n0, red_len;
    if constexpr (KIND == XMA_GEMM_MT) {
        expert = row_tile / P.row_tiles_max;
        tile_i0 = (int64_t)(row_tile % P.row_tiles_max) * BM;
        m_begin = P.offsets[expert];
        m_end = P.offsets[expert + 1];
        red_len = m_end - m_begin;
        n0 = (int64_t)col_tile * BN;
    } else {
        if (table) {
            expert = P.tile_expert[row_tile];
            m_begin = P.tile_row0[row_tile];
            const int64_t e_end = P.offsets[expert + 1];
            m_end = m_begin + BM < e_end ? m_begin + BM : e_end;
        } else {
            int32_t row0, row_end;
            tiles.find(row_tile, expert, row0, row_end);
            m_begin = row0;
            m_end = row_end;
        }
        red_len = P.k;
        n0 = (int64_t)col_tile * BN_OUT;
    }
    const int64_t rows_here = KIND == XMA_GEMM_MT ? P.n - tile_i0 : m_end - m_begin;
    const int live = rows_here >= BM ? MB : (int)((rows_here + 31) / 32);  // 32-row blocks with a row in them

    // ---- operand loads ----
    Loads<BM, A_STRIDED> la;
    Loads<BN, B_STRIDED> lb;
    const bool gathered = KIND == XMA_GEMM_MT && P.in_index != nullptr;
    const float* gather_base = B + n0;
    if constexpr (KIND == XMA_GEMM_MT) {
        la.setup_strided(wave, lane, A + m_begin * P.lda + tile_i0, P.lda, P.n - tile_i0);
        lb.setup_strided(wave, lane, B + m_begin * P.ldb + n0, P.ldb, P.k - n0);
    } else {
        la.setup_rows(wave, lane, [&](int r) -> const float* {
            const int64_t p = m_begin + r;
            if (p >= m_end) return nullptr;
            return A + (P.in_index ? source_row(P, p) : p) * P.lda;
        });
        const float* W = B + (int64_t)expert * P.b_expert_stride;
        if constexpr (KIND == XMA_GEMM_TN) {
            lb.setup_rows(wave, lane, [&](int r) -> const float* {
                if constexpr (EPI == EPI_PAIRED) {
                    const int64_t half = P.n / 2, j = n0 + (r % BN_OUT);
                    return j < half ? W + (r < BN_OUT ? j : half + j) * P.ldb : nullptr;
                } else {
                    return n0 + r < P.n ? W + (n0 + r) * P.ldb : nullptr;
                }
            });
        } else {
            lb.setup_strided(wave, lane, W + n0, P.ldb, P.n - n0);
        }
    }
    if constexpr (KIND != XMA_GEMM_MT) {
        if (work.parts > 1) {
            const int64_t all = (red_len + BK - 1) / BK;
            const int first = (int)(work.part * all / work.parts), end = (int)((work.part + 1) * all / work.parts);
            la.skip_stages(first);
            lb.skip_stages(first);
            red_len = ((int64_t)end * BK < red_len ? (int64_t)end * BK : red_len) - (int64_t)first * BK;
        }
    }
    // MT with a row gather: the source rows of the next stage's loads, requested a stage ahead
    int32_t next_rows[Loads<BN, B_STRIDED>::LOADS];
    auto lookup_rows = [&](int stage) __attribute__((always_inline)) {
        if constexpr (KIND == XMA_GEMM_MT) {
#pragma unroll
            for (int i = 0; i < Loads<BN, B_STRIDED>::LOADS; ++i) {
                int64_t p = m_begin + (int64_t)stage * BK + lb.red0 + i * Loads<BN, B_STRIDED>::RED_STEP;
                p = p < m_end ? p : m_end - 1;
                next_rows[i] = (int32_t)source_row(P, p);
            }
        }
    };
    const int stages = (int)((red_len + BK - 1) / BK);
    constexpr int LA = Loads<BM, A_STRIDED>::LOADS, LB = Loads<BN, B_STRIDED>::LOADS;
    // load number i (0 <= i < LA + LB) of a stage
    auto issue = [&](auto whole_tag, int i, char* stage_lds, int left) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
        if (i < LA) la.template issue<WHOLE>(i, stage_lds, wave, left);
        else if (gathered) lb.issue_gathered(i - LA, stage_lds + A_BYTES, wave, left, gather_base, P.ldb, lane, next_rows[i - LA]);
        else lb.template issue<WHOLE>(i - LA, stage_lds + A_BYTES, wave, left);
    };

    f32x16_t acc[MB];
#pragma unroll
    for (int mi = 0; mi < MB; ++mi)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mi][r] = 0.0f;
    int a_var[KK], b_var[KK];
    fragment_offsets<BM, A_STRIDED>(0, lane, a_var);
    fragment_offsets<BN, B_STRIDED>(wave * 32, lane, b_var);

    if (stages > 0) {
        if (gathered) lookup_rows(0);
#pragma unroll
        for (int i = 0; i < LA + LB; ++i)
            issue(std::false_type{}, i, even_stage, red_len < BK ? (int)red_len : BK);
        if (gathered && stages > 1) lookup_rows(1);
        wait_loads_and_lds();
        block_barrier();
    }
    // One stage.  On entry the fragments of its first group of eight reduction elements are in registers (set 0).
    //   - The fragments of every group are requested before the group ahead of it is multiplied (pinned: left alone, the
    //     compiler sinks the reads to their use); the last group is multiplied after the barrier, behind the reads of the
    //     next stage's first group, so a wave never waits for LDS with nothing to multiply.
    //   - The loads of the next stage are dealt out one per four (LIVE) matrix instructions.  Issued together at the
    //     start of the stage they fill the load queue of the compute unit and both waves of a SIMD stand in front of it.
    // NEXT: 2 = the next stage is whole, 1 = only its first `left` reduction elements exist, 0 = there is none.
    auto step = [&](auto live_tag, auto next_tag, auto& fa, auto& fb, char* here, char* there,
                    int s) __attribute__((always_inline)) {
        constexpr int LIVE = decltype(live_tag)::value, NEXT = decltype(next_tag)::value;
        const int left = NEXT == 1 ? (int)(red_len - (int64_t)(s + 1) * BK) : BK;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const bool last = kk + 1 == KK;
            if (last) {
                wait_loads_and_lds();
                block_barrier();
            }
            const char* source = last ? there : here;
            const int set = (kk + 1) & 1, group = last ? 0 : kk + 1;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (!last || NEXT != 0) {
                    if (j == 0) fb[set] = read_fragment<BN, B_STRIDED>(source + A_BYTES, b_var, 0, group);
                    if (j < LIVE) fa[set][j] = read_fragment<BM, A_STRIDED>(source, a_var, j, group);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int mi = 0; mi < LIVE; ++mi)
                    acc[mi] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[kk & 1][j], fa[kk & 1][mi][j], acc[mi], 0, 0, 0);
                const int i = 4 * kk + j;
                if (NEXT != 0 && i < LA + LB) {
                    issue(std::integral_constant<bool, NEXT == 2>{}, i, there, left);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (NEXT != 0 && kk == KK - 2 && gathered && s + 2 < stages) lookup_rows(s + 2);
        }
    };
    auto run = [&](auto live_tag) __attribute__((always_inline)) {
        constexpr int LIVE = decltype(live_tag)::value;
        constexpr std::integral_constant<int, 2> whole{};
        f32x4_t fa[2][LIVE], fb[2];
        if (stages == 0) return;
        fb[0] = read_fragment<BN, B_STRIDED>(even_stage + A_BYTES, b_var, 0, 0);
#pragma unroll
        for (int mi = 0; mi < LIVE; ++mi) fa[0][mi] = read_fragment<BM, A_STRIDED>(even_stage, a_var, mi, 0);
        const int whole_stages = (int)(red_len / BK);
        int s = 0;
        for (; s + 3 <= whole_stages; s += 2) {
            step(live_tag, whole, fa, fb, even_stage, odd_stage, s);
            step(live_tag, whole, fa, fb, odd_stage, even_stage, s + 1);
        }
        // up to three stages remain
        constexpr std::integral_constant<int, 1> partial{};
        constexpr std::integral_constant<int, 0> none{};
        if (s + 3 == stages) {
            step(live_tag, partial, fa, fb, even_stage, odd_stage, s);
            step(live_tag, partial, fa, fb, odd_stage, even_stage, s + 1);
            s += 2;
        } else if (s + 2 == stages) {
            step(live_tag, partial, fa, fb, even_stage, odd_stage, s);
            step(live_tag, none, fa, fb, odd_stage, even_stage, s + 1);
            return;
        }
        step(live_tag, none, fa, fb, even_stage, odd_stage, s);
    };
    if constexpr (MB == 4) {
        if (live == 4) run(std::integral_constant<int, 4>{});
        else if (live == 3) run(std::integral_constant<int, 3>{});
        else if (live == 2) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 1>{});
    } else if constexpr (MB == 2) {
        if (live == 2) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 1>{});
    } else {
        run(std::integral_constant<int, 1>{});
    }

    // ---- a split tile: every part parks its sums, the part that arrives last adds them up in part order and goes on ----
    // (what the exchange between XCDs relies on is written at the same place of the 16-bit kernel)
    if constexpr (KIND != XMA_GEMM_MT) {
        if (work.parts > 1) {
            auto part_buffer = [&](int part) {
                return reinterpret_cast<uint64_t*>(P.split_partials +
                                                   (int64_t)(part * work.split_tiles + work.split_tile) * (BM * BN));
            };
            uint64_t* mine = part_buffer(work.part);
#pragma unroll
            for (int mi = 0; mi < MB; ++mi)
#pragma unroll
                for (int g = 0; g < 8; ++g) {
                    const float2 v{acc[mi][2 * g], acc[mi][2 * g + 1]};
                    __hip_atomic_store(mine + (mi * 8 + g) * THREADS + tid, __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                }
            wait_loads_and_lds();
            __syncthreads();
            int* arrivals = reinterpret_cast<int*>(even_stage);
            if (tid == 0)
                arrivals[0] = __hip_atomic_fetch_add(P.split_counters + work.split_tile, 1, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            const bool last = arrivals[0] == work.parts - 1;
            __syncthreads();
            if (!last) return;
#pragma unroll
            for (int mi = 0; mi < MB; ++mi)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[mi][r] = 0.0f;
            for (int part = 0; part < work.parts; ++part) {
                const uint64_t* src = part_buffer(part);
                uint64_t v[MB * 8];
#pragma unroll
                for (int i = 0; i < MB * 8; ++i)
                    v[i] = __hip_atomic_load(src + i * THREADS + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < MB * 8; ++i) {
                    const float2 f = __builtin_bit_cast(float2, v[i]);
                    acc[i / 8][2 * (i % 8)] += f.x;
                    acc[i / 8][2 * (i % 8) + 1] += f.y;
                }
            }
        }
    }

    // ---- epilogue: registers -> LDS [BM][128], 512-byte rows, chunk c of row r at c ^ (r & 31) -> HBM ----
    // Register r of lane (h, i): tile row i (+ 32 mi), tile column 32 wave + 8 (r / 4) + 4 h + r % 4.
    constexpr int HALF_BLOCKS = (MB + 1) / 2;
    auto c_block = [&](int mi) { return (mi < HALF_BLOCKS ? even_stage : odd_stage) + (mi % HALF_BLOCKS) * 32 * 512; };
    static_assert(HALF_BLOCKS * 32 * 512 <= STAGE_BYTES, "the tile is staged in the two stage buffers");
    {
        const int i = lane & 31, h = lane >> 5;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = wave * 32 + 8 * g + 4 * h;
            float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (KIND == XMA_GEMM_TN) {
                if (P.bias != nullptr) {  // tile column `col` is weight row n0 + col; see setup_rows for a gated tile
                    const int64_t n = EPI == EPI_PAIRED ? n0 + (col % BN_OUT) + (col >= BN_OUT ? P.n / 2 : 0) : n0 + col;
                    const bool there = EPI == EPI_PAIRED ? n0 + (col % BN_OUT) < P.n / 2 : n < P.n;
                    if (there)
                        Elem<float>::unpack(*reinterpret_cast<const uint4*>(reinterpret_cast<const float*>(P.bias) +
                                                                            (int64_t)expert * P.ld_bias + n), bias);
                }
            }
#pragma unroll
            for (int mi = 0; mi < MB; ++mi) {
                f32x4_t v;
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = acc[mi][4 * g + q] + bias[q];
                *reinterpret_cast<f32x4_t*>(c_block(mi) + i * 512 + (((col >> 2) ^ i) << 4)) = v;
            }
        }
    }
    __syncthreads();

    float* C = reinterpret_cast<float*>(P.c);
    float* H = reinterpret_cast<float*>(P.aux);
    const int cc = tid & 31, r0 = tid >> 5;  // the thread's chunk column and its row of every eight
    auto rows_of_block = [&](const char* block, int mi) {
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int br = r0 + 8 * it;
            const int64_t r = mi * 32 + br;
            if (r >= rows_here) continue;
            auto chunk = [&](int c) { return *reinterpret_cast<const uint4*>(block + br * 512 + ((c ^ br) << 4)); };
            if constexpr (KIND == XMA_GEMM_MT) {
                const int64_t j = n0 + cc * 4;
                if (j < P.k)
                    *reinterpret_cast<uint4*>(C + (int64_t)expert * P.c_expert_stride + (tile_i0 + r) * P.ldc + j) = chunk(cc);
            } else {
                const int64_t p = m_begin + r;
                const int64_t out_row = P.out_index ? load_index(P.out_index, P.idx_is_i64, p) : p;
                if constexpr (EPI == EPI_PLAIN) {
                    const int64_t n = n0 + cc * 4;
                    if (n >= P.n) continue;
                    const uint4 v = chunk(cc);
                    if (KIND == XMA_GEMM_TN && P.act == ACT_GELU_TANH) {
                        if (H) *reinterpret_cast<uint4*>(H + p * P.ld_aux + n) = v;
                        float h[4], o[4];
                        Elem<float>::unpack(v, h);
#pragma unroll
                        for (int q = 0; q < 4; ++q) o[q] = gelu_tanh_forward<false>(h[q]);
                        *reinterpret_cast<uint4*>(C + out_row * P.ldc + n) = Elem<float>::pack(o);
                    } else {
                        *reinterpret_cast<uint4*>(C + out_row * P.ldc + n) = v;
                    }
                } else if constexpr (EPI == EPI_PAIRED) {
                    const int64_t half = P.n / 2, j = n0 + (cc % 16) * 4;
                    if (j >= half) continue;
                    if (H) *reinterpret_cast<uint4*>(H + p * P.ld_aux + (cc < 16 ? j : half + j)) = chunk(cc);
                    if (cc < 16) {
                        float u[4], g[4], o[4];
                        Elem<float>::unpack(chunk(cc), u);
                        Elem<float>::unpack(chunk(cc + 16), g);
#pragma unroll
                        for (int q = 0; q < 4; ++q) o[q] = gated_forward<false>(P.act, u[q], g[q]);
                        *reinterpret_cast<uint4*>(C + out_row * P.ldc + j) = Elem<float>::pack(o);
                    }
                } else {  // EPI_BACKWARD: the product is the activation's upstream gradient
                    const int64_t n = n0 + cc * 4;
                    if (n >= P.n) continue;
                    const float* saved = reinterpret_cast<const float*>(P.aux) + p * P.ld_aux + n;
                    float u[4], g[4], d[4], du[4], dg[4];
                    Elem<float>::unpack(*reinterpret_cast<const uint4*>(saved), u);
                    Elem<float>::unpack(chunk(cc), d);
                    if (P.act == ACT_GELU_TANH) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) du[q] = gelu_tanh_backward<false>(u[q], d[q]);
                        *reinterpret_cast<uint4*>(C + out_row * P.ldc + n) = Elem<float>::pack(du);
                    } else {
                        Elem<float>::unpack(*reinterpret_cast<const uint4*>(saved + P.n), g);
#pragma unroll
                        for (int q = 0; q < 4; ++q) gated_backward<false>(P.act, u[q], g[q], d[q], du[q], dg[q]);
                        *reinterpret_cast<uint4*>(C + out_row * P.ldc + n) = Elem<float>::pack(du);
                        *reinterpret_cast<uint4*>(C + out_row * P.ldc + P.n + n) = Elem<float>::pack(dg);
                    }
                }
            }
        }
    };
#pragma unroll
    for (int mi = 0; mi < MB; ++mi)
        if (mi < live) rows_of_block(c_block(mi), mi);
}

template <int MB, int KIND, int EPI>
static int launch(const xma_grouped_gemm_args& a, hipStream_t stream) {
    constexpr int BM = 32 * MB;
    GemmParams P;
    fill_params(a, P);
    int64_t grid;
    if (KIND == XMA_GEMM_MT) {
        P.row_tiles_max = (int32_t)ceil_div(a.n, BM);
        P.col_tiles = (int32_t)ceil_div(a.k, BN);
        grid = grid_for_tiles((int64_t)P.row_tiles_max * a.num_experts, P.col_tiles);
    } else {
        const int64_t rt = max_row_tiles(a.rows, a.num_experts, BM);
        P.row_tiles_max = (int32_t)rt;
        P.col_tiles = (int32_t)(EPI == EPI_PAIRED ? ceil_div(a.n / 2, BN / 2) : ceil_div(a.n, BN));
        place_split_region(a, P);
        P.round_tiles = (MB == 4 ? 2 : MB == 2 ? 3 : 4) * compute_units();  // by their registers
        const int64_t parts = 2.0 * a.rows * a.n * a.k < kSplitFlops ? 1 : ceil_div(a.k, BK) / (kSplitStages * 4 / MB);
        P.most_parts = (int32_t)(parts < 1 ? 1 : parts > kSplitParts ? kSplitParts : parts);
        grid = grid_for_work(rt * P.col_tiles, P.round_tiles);
        if (a.num_experts > kMaxScannedExperts) launch_build_row_tiles(a, BM, rt, P, stream);
        else if (P.most_parts > 1) launch_clear_split_counters(P, stream);
    }
    XMA_REQUIRE(grid < ((int64_t)1 << 31), "xma_grouped_gemm: %lld tiles exceed the grid limit", (long long)grid);
    hipLaunchKernelGGL((gemm_kernel<MB, KIND, EPI>), dim3((unsigned)grid), dim3(THREADS), 0, stream, P);
    return check_launch("xma_grouped_gemm");
}

// The tallest tile that still gives every compute unit two work-groups to run side by side.  At half and a quarter of
// that bound, 2048 rows, K 256, 64 output columns per tile: 25 and 28 us instead of 21 us for the up projection; taller
// tiles move fewer operand bytes per FLOP (64-row tiles on a large call: 125 instead of 146 TFLOP/s).
static int row_blocks(const xma_grouped_gemm_args& a) {
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    const bool mt = a.kind == XMA_GEMM_MT;
    const int64_t cols = mt ? ceil_div(a.k, BN) : shape == EPI_PAIRED ? ceil_div(a.n / 2, BN / 2) : ceil_div(a.n, BN);
    const int64_t rows = mt ? a.n * a.num_experts : a.rows;
    return rows * cols >= kFullDeviceTiles * 128 ? 4 : rows * cols >= kFullDeviceTiles * 64 ? 2 : 1;
}
template <int KIND, int EPI>
static int launch_for_size(const xma_grouped_gemm_args& a, hipStream_t stream) {
    switch (row_blocks(a)) {
        case 4: return launch<4, KIND, EPI>(a, stream);
        case 2: return launch<2, KIND, EPI>(a, stream);
        default: return launch<1, KIND, EPI>(a, stream);
    }
}

}  // namespace f32

GemmForm f32_gemm_form(const xma_grouped_gemm_args& a) { return {XMA_FORM_TILED, 32 * f32::row_blocks(a), f32::BN}; }

int launch_f32_gemm(const xma_grouped_gemm_args& a, hipStream_t stream) {
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    switch (a.kind) {
        case XMA_GEMM_TN:
            if (shape == EPI_PAIRED) return f32::launch_for_size<XMA_GEMM_TN, EPI_PAIRED>(a, stream);
            return f32::launch_for_size<XMA_GEMM_TN, EPI_PLAIN>(a, stream);
        case XMA_GEMM_NN:
            if (shape == EPI_BACKWARD) return f32::launch_for_size<XMA_GEMM_NN, EPI_BACKWARD>(a, stream);
            return f32::launch_for_size<XMA_GEMM_NN, EPI_PLAIN>(a, stream);
        default:
            return f32::launch_for_size<XMA_GEMM_MT, EPI_PLAIN>(a, stream);
    }
}

}  // namespace xma
