// Pieces shared by the grouped-GEMM kernels: kernel arguments, the row-tile list that maps
// work-groups to (expert, rows) without host synchronisation, and the XCD-aware tile walk.
#pragma once

#include "common.h"

namespace xma {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;  // 16 bytes moved as ONE vector access

constexpr int kNumXcd = 8;     // accelerator complex dies, each with a private L2
constexpr int kBandTiles = 4;  // row tiles per band of the tile walk (2, 8 and 16 measured slower)

// ---- kernel arguments -----------------------------------------------------------------------------
struct GemmParams {
    const void* a;
    const void* b;
    void* c;
    void* aux;
    const int32_t* offsets;
    const void* in_index;
    const void* out_index;
    const int32_t* tile_expert;  // [row tiles] expert of each row tile (TN/NN; only beyond kMaxScannedExperts experts)
    const int32_t* tile_row0;    // [row tiles] first grouped row of each row tile
    const int32_t* tile_count;   // [1] number of row tiles actually present; nullptr: no table
    int64_t lda, ldb, ldc, ld_aux, b_expert_stride, c_expert_stride;
    int64_t n, k;
    int32_t num_experts, in_fan_out, idx_is_i64;
    int32_t row_tiles_max;  // upper bound used for the grid (TN/NN); MT: row tiles per expert
    int32_t col_tiles;
    // split-K of the last, partly filled round of tiles (TN/NN kernels of 16 and 32 bits)
    int32_t* split_counters;  // [kSplitSlots] arrivals per split tile, zero at launch
    float* split_partials;    // [kSplitSlots][tile] fp32 accumulators of the parts
    // MT with gathered rows (16 bits): byte offset of the source row of every routed row, kRowOffsetsPadding entries more
    const uint32_t* row_offsets;
    int32_t tile_rows;    // rows of the tallest tile (16-bit TN/NN)
    int32_t most_parts;   // parts of a split tile at most (fp32)
    int32_t round_tiles;  // tiles that run at a time on the whole device, a multiple of kNumXcd
    // MT: experts in descending order of their row counts, one record {expert, first row, end row, 0} per slot;
    // nullptr: slot e is expert e
    const int32_t* expert_order;
    // fused activation of the epilogue (enum Activation) and the optional per-expert bias of the forward kinds
    const void* bias;
    int64_t ld_bias;
    int32_t act;
};

// The kernels are instantiated for three epilogue shapes; the activation inside a shape is a run-time value
// (GemmParams::act), so SwiGLU and GLU, or the two backward forms, share one instantiation.
//   EPI_PLAIN     store the product (optionally through tanh-GELU, keeping the pre-activation)
//   EPI_PAIRED    TN: tile columns [0, 128) and [128, 256) are the two halves of a gated pre-activation
//   EPI_BACKWARD  NN: the product is the activation's upstream gradient; the saved pre-activation is read back
constexpr int EPI_PLAIN = 0, EPI_PAIRED = 1, EPI_BACKWARD = 2;
inline void split_epilogue(int epilogue, int& shape, int& act) {
    switch (epilogue) {
        case XMA_EPI_SWIGLU: shape = EPI_PAIRED; act = ACT_SWIGLU; break;
        case XMA_EPI_GLU: shape = EPI_PAIRED; act = ACT_GLU; break;
        case XMA_EPI_SWIGLU_BWD: shape = EPI_BACKWARD; act = ACT_SWIGLU; break;
        case XMA_EPI_GLU_BWD: shape = EPI_BACKWARD; act = ACT_GLU; break;
        case XMA_EPI_GELU_TANH: shape = EPI_PLAIN; act = ACT_GELU_TANH; break;
        case XMA_EPI_GELU_TANH_BWD: shape = EPI_BACKWARD; act = ACT_GELU_TANH; break;
        default: shape = EPI_PLAIN; act = ACT_NONE; break;
    }
}

// At most kSplitSlots tiles are split, those of one round of the device.  Their parts' sums take kSplitSlots tiles of 256 x 256 at
// most: as many pairs of a tile and a part exist as places of a round (512 of 192 x 128, or 1024 of 32 x 128).
constexpr int kSplitSlots = 256;
constexpr int kMaxSplit = 4;
constexpr int kSplitMaxRounds = 8;
constexpr int kSplitMinStages = 32;  // a part must keep this many 64-deep stages of the reduction
constexpr int64_t kSplitTileFloats = 256 * 256;
inline int64_t tile_table_bytes(int64_t row_tiles) { return ((4 + 2 * row_tiles) * (int64_t)sizeof(int32_t) + 255) / 256 * 256; }
inline int64_t split_region_bytes() {
    return kSplitSlots * (int64_t)sizeof(int32_t) + kSplitSlots * kSplitTileFloats * (int64_t)sizeof(float);
}

// The weight-gradient kind walks the experts in descending order of their row counts (ties: lower expert first), so
// that the cost of consecutive bands of tiles falls monotonically and dealing them to the XCDs forwards and backwards
// in turn (locate_tile<true>) gives every XCD about the same work however skewed the routing is.  One block;
// rank sort for up to kMaxOrderedExperts experts, natural order beyond.
constexpr int kMaxOrderedExperts = 1024;
inline int64_t expert_order_bytes(int64_t E) { return 4 * E * (int64_t)sizeof(int32_t); }

// routed row p -> source row of the gathered operand (indices are < 2^31, so divide in 32 bits)
__device__ __forceinline__ int64_t source_row(const GemmParams& P, int64_t p) {
    return (int64_t)((uint32_t)load_index(P.in_index, P.idx_is_i64, p) / (uint32_t)P.in_fan_out);
}

// Row-tile list for the row-grouped kinds beyond kMaxScannedExperts experts (grouped_gemm.hip): fills P.tile_count,
// tile_expert and tile_row0 in the workspace, for up to `row_tiles` tiles of BM rows, and clears P.split_counters if set.
void launch_build_row_tiles(const xma_grouped_gemm_args& a, int BM, int64_t row_tiles, GemmParams& P, hipStream_t stream);

// Work-group -> (row tile, column tile).  Tiles are numbered in bands of kBandTiles row tiles x all column
// tiles, row tile fastest, so that work-groups running at the same time share A row panels and B column
// panels.  The hardware deals work-groups round-robin to the XCDs (block b runs on XCD b % 8, as that XCD's
// b / 8-th block; checked on the device), and each XCD has a private L2, so neighbouring tiles must go to
// the same XCD.  Two ways to deal the tiles:
//   SPREAD = false: XCD x takes the x-th of eight equal contiguous ranges of the tile sequence (ranges may
//     cut a band).  Balanced to one tile when every tile costs the same (row-grouped kinds).
//   SPREAD = true: every group of eight consecutive bands is dealt one band per XCD, forwards and backwards in
//     turn; spreads a run of expensive bands (the weight-gradient tiles of an overloaded expert) over all XCDs and,
//     when band costs fall monotonically, balances them.
// `row_tiles` is the number of row tiles actually present.  Returns false when this work-group has no tile.
template <bool SPREAD, int BAND = kBandTiles>
__device__ __forceinline__ bool locate_tile(int row_tiles, int col_tiles, int& row_tile, int& col_tile) {
    const int xcd = blockIdx.x % kNumXcd;
    const int local = blockIdx.x / kNumXcd;
    const int per_band = BAND * col_tiles;
    int band, in_band;
    if constexpr (SPREAD) {
        // forwards over the XCDs for even groups of eight bands, backwards for odd ones
        const int group = local / per_band;
        band = group * kNumXcd + ((group & 1) ? kNumXcd - 1 - xcd : xcd);
        in_band = local % per_band;
    } else {
        const int total = row_tiles * col_tiles;
        const int per_xcd = (total + kNumXcd - 1) / kNumXcd;
        const int tile = xcd * per_xcd + local;
        if (local >= per_xcd || tile >= total) return false;
        band = tile / per_band;
        in_band = tile - band * per_band;
    }
    const int band_first = band * BAND;
    if (band_first >= row_tiles) return false;
    const int band_rows = row_tiles - band_first < BAND ? row_tiles - band_first : BAND;
    row_tile = band_first + in_band % band_rows;
    col_tile = in_band / band_rows;
    return col_tile < col_tiles;
}

// The small tiles of the row-grouped kinds differ in cost, and under a skewed routing the tall ones come first: an eighth of
// the sequence each leaves most of them to a few XCDs.  While the tiles are few they are therefore dealt in bands of two, where
// that gives every XCD about as many bands; beyond, the panels that neighbouring tiles share in an XCD's L2 are worth more.
// Four GEMMs of a layer, us, eighths / bands of two: 1531 tokens, 128 experts, 8 each, skewed (89 row tiles) 336 / 322; 1500, 64
// experts, 6 each, skewed (67) 353 / 316, even (64) 390 / 379; 3000, even (128) 628 / 652; 5000, 128 experts, skewed (248) 865
// / 894.
constexpr int kDealtBand = 2, kMostDealtTiles = 104;
__device__ __forceinline__ bool deal_row_tiles(int row_tiles) {
    const int bands = (row_tiles + kDealtBand - 1) / kDealtBand, even = (bands + kNumXcd - 1) / kNumXcd * kNumXcd;
    return row_tiles <= kMostDealtTiles && 4 * even <= 5 * bands;
}
inline int64_t grid_for_dealt_tiles(int64_t row_tiles, int64_t col_tiles) {
    const int64_t rows = row_tiles < kMostDealtTiles ? row_tiles : kMostDealtTiles;
    return ceil_div(ceil_div(rows, kDealtBand), kNumXcd) * kNumXcd * kDealtBand * col_tiles;
}

// Row-grouped kinds with split-K of the remainder.  With T tiles on a device that runs C of them at a time (round_tiles: one
// per compute unit of 256 x 256 tiles, two of the smaller ones) the first floor(T / C) * C tiles fill whole rounds; the
// R = T mod C tiles of the last round would leave C - R places idle for a whole tile time, so each of them is cut along the
// reduction into min(most_parts, C / R) parts that run side by side.  Only when the launch has fewer than most_rounds rounds
// (the idle places of a last round matter less the more rounds there are), only for up to most_tiles tiles, and only while a
// part is worth its exchange (most_parts, which the kernels derive from the reduction): every part parks its fp32 sums in memory
// and the last one reads them all back.  16-bit kernels: 40-50 k cycles for a 256 x 256 tile, or about 17 stages of the main loop (measured;
// reductions of 14336 and 28672 split in three gain 7 % and 5 % of their launches), so a part keeps kSplitMinStages stages.
// Work-groups are dealt per XCD as in locate_tile<false>: XCD x takes the x-th eighth of the whole tiles, then the x-th
// eighth of the parts (part-major, so neighbours share panels).
// HALVES: tiles of a last round that are not cut along the reduction, and leave half the places free, go to two work-groups
// by their rows.
struct TileWork {
    int row_tile, col_tile;
    int part, parts;  // this work-group reduces stages [part * n / parts, (part + 1) * n / parts)
    int split_tile;   // index of the tile among the split ones
    int split_tiles;
    int half, halves;  // this work-group has the rows of one half of the tile
};
template <bool HALVES>
__device__ __forceinline__ bool locate_work(int row_tiles, int col_tiles, int round_tiles, int most_parts, int most_rounds,
                                            int most_tiles, TileWork& w) {
    const int xcd = blockIdx.x % kNumXcd;
    const int local = blockIdx.x / kNumXcd;
    const int total = row_tiles * col_tiles;
    const int whole = total / round_tiles * round_tiles;
    const int rem = total - whole;
    int parts = rem > 0 && rem <= most_tiles && total < most_rounds * round_tiles ? round_tiles / rem : 1;
    parts = parts > most_parts ? most_parts : parts;
    parts = parts < 1 ? 1 : parts;
    const int halves = HALVES && parts == 1 && 2 * rem <= round_tiles ? 2 : 1;
    w.half = 0;
    w.halves = 1;
    const int whole_per_xcd = whole / kNumXcd;
    int tile;
    if (local < whole_per_xcd) {
        tile = xcd * whole_per_xcd + local;
        w.part = 0;
        w.parts = 1;
        w.split_tile = 0;
    } else {
        const int items = rem * parts * halves;
        const int per_xcd = (items + kNumXcd - 1) / kNumXcd;
        const int l = local - whole_per_xcd;
        const int q = xcd * per_xcd + l;
        if (l >= per_xcd || q >= items) return false;
        w.part = q / rem;
        w.split_tile = q - w.part * rem;
        w.parts = parts;
        if (halves > 1) {
            w.half = w.part;
            w.halves = 2;
            w.part = 0;
        }
        tile = whole + w.split_tile;
    }
    w.split_tiles = rem;
    const int per_band = kBandTiles * col_tiles;
    const int band = tile / per_band, in_band = tile - band * per_band;
    const int band_first = band * kBandTiles;
    const int band_rows = row_tiles - band_first < kBandTiles ? row_tiles - band_first : kBandTiles;
    w.row_tile = band_first + in_band % band_rows;
    w.col_tile = in_band / band_rows;
    return true;
}
// number of work-groups that covers every case of locate_work() for up to `tiles` tiles
inline int64_t grid_for_work(int64_t tiles, int round_tiles) { return (ceil_div(tiles, kNumXcd) + round_tiles / kNumXcd + 1) * kNumXcd; }

// number of work-groups that covers up to `row_tiles` x `col_tiles` under either dealing of locate_tile()
inline int64_t grid_for_tiles(int64_t row_tiles, int64_t col_tiles) {
    const int64_t bands = ceil_div(row_tiles, kBandTiles);
    return ceil_div(bands, kNumXcd) * kNumXcd * kBandTiles * col_tiles;
}

constexpr int kSmallestTileRows = 32;  // of any kernel that may use a table of tiles
inline int64_t max_row_tiles(int64_t rows, int E, int BM) { return rows / BM + E; }

// ---- row tiles without a table ---------------------------------------------------------------------------------
// Expert e owns ceil(count_e / bm) consecutive row tiles.  How many there are and which expert and rows a tile has, found
// by each wave on its own from the offsets: lane l adds up the tiles of the l-th run of consecutive experts, one prefix
// sum over the lanes.  Costs a load and some thirty instructions, against a launch of its own (3-6 us and the gap
// before the next) for a table of tiles.
constexpr int kMaxScannedExperts = 512;  // up to eight experts per lane
struct RowTileScan {
    const int32_t* offsets;
    int experts, per_lane, bm;
    int first_tile;  // of the lane's run
    int upto;        // first_tile + the run's tiles
    int total;

    // (up to 2^31 - 1 rows: no sum of a row and a tile's height is taken in signed 32 bits)
    __device__ __forceinline__ int tiles_of(int32_t begin, int32_t end) const {
        return (int)(((uint32_t)(end - begin) + (uint32_t)bm - 1u) / (uint32_t)bm);
    }
    __device__ __forceinline__ RowTileScan(const int32_t* __restrict__ expert_offsets, int E, int tile_rows, int lane)
        : offsets(expert_offsets), experts(E), per_lane((E + kWaveSize - 1) / kWaveSize), bm(tile_rows) {
        const int e0 = lane * per_lane;
        int32_t begin = offsets[e0 < E ? e0 : E];
        int mine = 0;
        for (int i = 1; i <= per_lane; ++i) {
            const int32_t end = offsets[e0 + i < E ? e0 + i : E];
            mine += tiles_of(begin, end);
            begin = end;
        }
        upto = wave_inclusive_sum(mine);
        first_tile = upto - mine;
        total = __builtin_amdgcn_readlane(upto, kWaveSize - 1);
    }
    // tile < total
    __device__ __forceinline__ void find(int tile, int& expert, int32_t& row0, int32_t& row_end) const {
        const int l = __ffsll((unsigned long long)__ballot(tile < upto)) - 1;
        int before = __builtin_amdgcn_readlane(first_tile, l);
        expert = l * per_lane;
        int32_t begin = offsets[expert], end = offsets[expert + 1];
        for (int i = 1; i < per_lane && tile >= before + tiles_of(begin, end); ++i) {
            before += tiles_of(begin, end);
            ++expert;
            begin = end;
            end = offsets[expert + 1];
        }
        // (the compiler does not see that these are the same in every lane)
        expert = __builtin_amdgcn_readfirstlane(expert);
        row0 = __builtin_amdgcn_readfirstlane(begin + (tile - before) * bm);
        row_end = __builtin_amdgcn_readfirstlane(end - row0 > bm ? row0 + bm : end);
    }
};

// The MFMA instruction of the register-staged kernel for 16-bit types: acc(32x32) += X(32 x 16) * Y(32 x 16)^T,
// lane l supplies row l%32 and the 8 reduction elements 8*(l/32)..8*(l/32)+7 of both operands.
template <typename T>
struct Mma;
template <>
struct Mma<bf16_t> {
    template <typename V>
    __device__ static __forceinline__ void run(const V& x, const V& y, f32x16_t& acc) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, x), __builtin_bit_cast(bf16x8_t, y),
                                                      acc, 0, 0, 0);
    }
};
// The 16x16x32 form, which the LDS-DMA kernel is built on: acc(16x16) += X(16 x 32) * Y(16 x 32)^T; lane l supplies row l%16 and the 8 reduction
// elements 8*(l/16)..+7 of both operands; result register r of lane l is D[4*(l/16) + r][l%16] (rows from X).  Half the
// accumulator traffic per FLOP of the 32x32x16 form: under the device's power cap it sustains a higher clock.  Written
// as inline assembly with the accumulator tied in place: the compiler's builtin has no tied form for a four-register
// result and copies accumulators once all 256 are live.
template <typename T>
struct Mma16;
template <>
struct Mma16<bf16_t> {
    template <typename V>
    __device__ static __forceinline__ void run(const V& x, const V& y, f32x4_t& acc) {
        asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(x), "v"(y));
    }
};
template <>
struct Mma16<f16_t> {
    template <typename V>
    __device__ static __forceinline__ void run(const V& x, const V& y, f32x4_t& acc) {
        asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(x), "v"(y));
    }
};
template <>
struct Mma<f16_t> {
    template <typename V>
    __device__ static __forceinline__ void run(const V& x, const V& y, f32x16_t& acc) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, x), __builtin_bit_cast(f16x8_t, y),
                                                     acc, 0, 0, 0);
    }
};
template <>
struct Mma<float> {
    // a 16-byte fragment holds 4 reduction steps per lane half; one 32x32x2 MFMA per component
    __device__ static __forceinline__ void run(const uint4& x, const uint4& y, f32x16_t& acc) {
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(x.x), __uint_as_float(y.x), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(x.y), __uint_as_float(y.y), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(x.z), __uint_as_float(y.z), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(x.w), __uint_as_float(y.w), acc, 0, 0, 0);
    }
};

// Clears P.split_counters, for a launch that may split.
void launch_clear_split_counters(const GemmParams& P, hipStream_t stream);
// Compute units of the current device, rounded down to a multiple of the XCD count and capped at the
// number of split slots (the split-K scheme treats that many tiles as one round).
int compute_units();
// The split-K region of the workspace.
inline void place_split_region(const xma_grouped_gemm_args& a, GemmParams& P) {
    char* split = reinterpret_cast<char*>(a.workspace) +
                  (xma_grouped_gemm_workspace_bytes(a.num_experts, a.rows) - split_region_bytes());
    P.split_counters = reinterpret_cast<int32_t*>(split);
    P.split_partials = reinterpret_cast<float*>(split + kSplitSlots * sizeof(int32_t));
}

// a 16-bit launch splits the tiles of its last round only when a part keeps kSplitMinStages stages
inline bool may_split(int64_t reduction) { return (reduction + 63) / 64 >= 2 * kSplitMinStages; }

// Fills the fields of GemmParams that do not depend on the tile shape.
void fill_params(const xma_grouped_gemm_args& a, GemmParams& P);

// Which kernel takes a call, and the rows and columns of its (tallest) tile.  The launch functions and
// xma_grouped_gemm_form() ask the same functions.
struct GemmForm {
    int kernel;  // enum xma_gemm_form
    int tile_rows, tile_cols;
};

// The LDS-DMA pipelined kernel for 16-bit element types (grouped_gemm_dma.hip).
bool dma_gemm_supports(const xma_grouped_gemm_args& a);
struct DmaTile {
    int rows, cols;  // the tallest tile of the launch
};
DmaTile dma_gemm_tile(const xma_grouped_gemm_args& a);
int launch_dma_gemm(const xma_grouped_gemm_args& a, hipStream_t stream);
// MT whose B rows are row_offsets[p] bytes behind a.b, for arguments that dma_gemm_supports() and whole vectors.  The table
// is read up to kRowOffsetsPadding entries past the last routed row; what is read there is not used.
constexpr int kRowOffsetsPadding = 256;
int launch_gathered_weight_gradient(const xma_grouped_gemm_args& a, const uint32_t* row_offsets, hipStream_t stream);

// The kernel for fp32 operands in whole, aligned vectors (grouped_gemm_f32.hip).
GemmForm f32_gemm_form(const xma_grouped_gemm_args& a);
int launch_f32_gemm(const xma_grouped_gemm_args& a, hipStream_t stream);

// The weight-streaming kernel for few routed rows per expert (grouped_gemm_skinny.hip).
bool skinny_gemm_supports(const xma_grouped_gemm_args& a);
GemmForm skinny_gemm_form(const xma_grouped_gemm_args& a);
int launch_skinny_gemm(const xma_grouped_gemm_args& a, hipStream_t stream);

}  // namespace xma
