// Ragged (per-expert) GEMM for 16-bit element types on gfx950, built around the LDS-DMA load path
// (global_load_lds_dwordx4): tiles travel L2 -> LDS without passing through registers, several
// stages are kept in LDS so that loads stay in flight while a stage is multiplied, and operands whose
// reduction index is strided in HBM are fetched in their HBM layout and transposed by the LDS read
// itself (ds_read_b64_tr_b16).
//
// Tile 256 x 256 per work-group, 4 waves as 2 x 2, one wave per SIMD with the whole 512-register budget:
// each wave owns 128 x 128 (8 x 8 blocks of the 16x16x32 matrix instruction, 256 accumulator registers).  A
// wave that is alone on its SIMD has nobody to hide its stalls, so the main loop is software-pipelined by hand:
// the fragments of the 32-deep reduction block k+1 are read from LDS while block k is multiplied, DMA loads are
// dealt out one every eight matrix instructions, and the order of the three streams is pinned slot by slot.
//
// What bounds the loop (measured): what the L2 has to fetch and deliver.  A compute unit pulls a 256 x 256
// tile's operands from L2 at 128 FLOP per byte, the L2 delivers whole 128-byte lines about 1.5 x faster than
// half lines (so K-contiguous operands are staged 64 reduction elements at a time, 128-byte rows; see
// Ring64x5), and the 32 tiles an XCD runs at a time share their operand panels in its L2 as long as they walk
// the reduction in step (see Kernel::phase).
//
// The same body runs tiles of 32, 64, 128 and 192 rows of 128 columns with half the LDS and half the registers, two
// work-groups on a compute unit, for calls whose experts have few rows or that have few tiles (see dma_gemm_tile).  They are
// bound by the L2 too: 15.5 TB/s of operand lines at the fine-grained layer (128 x 128, counted), where 256 x 256 asks for 9.8.
//
// LDS is a pool of five 32 KiB slabs (all 160 KiB of the compute unit), or of 80 KiB in slabs of 16 and 8 KiB.
// Tile layouts inside a slab:
//   K-contiguous operand (A in TN/NN, W in TN): [tile rows][BK k]; the 16-byte chunks of a row are
//     XOR-swizzled by the row number so that the 16 rows a quarter-wave reads in one ds_read_b128 cover all
//     64 banks.
//   K-strided operand (W in NN, both operands in MT): [BK k][tile rows], 512 or 256 bytes per k row; chunk c
//     of k row r sits at c ^ ((r & 3) << 2), so that the four k rows one transposing read touches fall
//     into different bank groups.
// A DMA load writes lane l's 16 bytes at (wave-uniform LDS base) + 16*l, so the swizzles are applied
// by choosing which HBM chunk each lane fetches.  Masked rows / reduction tails are fetched from a
// 16-byte page of zeros, which keeps every lane active and the outstanding-load count uniform.
#include <cmath>
#include <type_traits>

#include "grouped_gemm_common.h"

namespace xma {
namespace dma {

constexpr int THREADS = 256, NUM_WAVES = THREADS / 64, WAVES_N = 2;

__shared__ __attribute__((aligned(1024))) char slab0[32768];
__shared__ __attribute__((aligned(1024))) char slab1[32768];
__shared__ __attribute__((aligned(1024))) char slab2[32768];
__shared__ __attribute__((aligned(1024))) char slab3[32768];
__shared__ __attribute__((aligned(1024))) char slab4[32768];
__shared__ __attribute__((aligned(1024))) char half_slab0[16384];
__shared__ __attribute__((aligned(1024))) char half_slab1[16384];
__shared__ __attribute__((aligned(1024))) char half_slab2[16384];
__shared__ __attribute__((aligned(1024))) char half_slab3[16384];
__shared__ __attribute__((aligned(1024))) char half_slab4[16384];
__shared__ __attribute__((aligned(1024))) char extra_slab0[8192];
__shared__ __attribute__((aligned(1024))) char extra_slab1[8192];

// A tile of BM rows and BN columns, four waves as 2 x 2.  The tiles of 256 columns have the compute unit to themselves; those of 128
// columns take half its LDS, so that two work-groups share it.
template <int BM_, int BN_>
struct Tile {
    static constexpr int BM = BM_, BN = BN_, WM = BM / 2, WN = BN / 2;
    static constexpr int MI = WM / 16, NI = WN / 16;  // blocks of 16 x 16 per wave
    static_assert(((BM == 256 || BM == 128) && BN == 256) || ((BM == 192 || BM == 128 || BM == 64 || BM == 32) && BN == 128), "tile size");
    // The epilogue stages the tile through LDS, SLAB_BLOCKS blocks of 16 rows of each wave row at a time.
    static constexpr int SLAB_BLOCKS = MI < 2 ? 1 : 2;
    static constexpr int OUT_SLABS = MI / SLAB_BLOCKS;
    // A tile row of 192 rows does not fit one slab: rows 128..191 live in a slab of their own, and a wave row's blocks
    // 4 and 5 are theirs, so that the slab of a block is known at compile time.
    static constexpr bool EXTRA = BM == 192;
    static constexpr int MAIN_BLOCKS = EXTRA ? 4 : MI;
    // first tile row of block mi of wave row wr
    __device__ static __forceinline__ int block_row(int wr, int mi) {
        return mi < MAIN_BLOCKS ? wr * (MAIN_BLOCKS * 16) + mi * 16 : 128 + wr * 32 + (mi - MAIN_BLOCKS) * 16;
    }

    // The slabs are distinct arrays on purpose: the compiler can then prove that a fragment read of
    // one slab does not alias the DMA writes still in flight to the others, and does not drain them.
    template <int I>
    __device__ static __forceinline__ char* slab() {
        static_assert(I >= 0 && I < 7, "slab index");
        if constexpr (I == 5) return extra_slab0;
        if constexpr (I == 6) return extra_slab1;
        if constexpr (BN == 256) {
            if constexpr (I == 0) return slab0;
            if constexpr (I == 1) return slab1;
            if constexpr (I == 2) return slab2;
            if constexpr (I == 3) return slab3;
            return slab4;
        } else {
            if constexpr (I == 0) return half_slab0;
            if constexpr (I == 1) return half_slab1;
            if constexpr (I == 2) return half_slab2;
            if constexpr (I == 3) return half_slab3;
            return half_slab4;
        }
    }
};
constexpr int groups_per_cu(int BN) { return BN == 256 ? 1 : 2; }
// fp32 sums of the tallest tile of BN columns: what a part of a split tile parks in the workspace
constexpr int split_tile_floats(int BN) { return BN == 256 ? 256 * 256 : 192 * 128; }

__device__ __attribute__((aligned(16))) uint32_t g_zero_page[4];  // zero-initialised

typedef __attribute__((ext_vector_type(4))) short short4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
#define XMA_LDS(p) ((__attribute__((address_space(3))) void*)(p))
#define XMA_LDS_S4(p) ((__attribute__((address_space(3))) short4_t*)(p))

__device__ __forceinline__ void compiler_fence() { asm volatile("" ::: "memory"); }

// s_waitcnt with only the vector-memory counter constrained (lgkmcnt = 15, expcnt = 7)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    compiler_fence();
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (7 << 4) | (0xF << 8) | ((N >> 4) << 14));
    compiler_fence();
}

// s_waitcnt on the vector-memory counter and for every LDS read of this wave (lgkmcnt = 0)
template <int N>
__device__ __forceinline__ void wait_vmcnt_and_lds() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    compiler_fence();
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
    compiler_fence();
}

// s_waitcnt for every LDS read and scalar load of this wave alone (vmcnt = 63)
__device__ __forceinline__ void wait_lds() {
    compiler_fence();
    __builtin_amdgcn_s_waitcnt(0xF | (7 << 4) | (0 << 8) | (3 << 14));
    compiler_fence();
}

__device__ __forceinline__ void block_barrier() {
    compiler_fence();
    __builtin_amdgcn_s_barrier();
    compiler_fence();
}

// LDS accesses add ONE integer byte offset to a slab, and the variable part of the offset is passed
// through opaque() so that the optimiser cannot split it into a chain of partial sums: the compiler
// attaches the "this access belongs to slab X" information it needs to keep DMA loads to the other
// slabs in flight only to accesses whose address is a short derivation from the array.
__device__ __forceinline__ int opaque(int v) {
    asm("" : "+v"(v));
    return v;
}

// The epilogue requests what it needs from HBM and LDS in batches and uses the values afterwards.  Left alone,
// the compiler sinks each load into the conditional block that uses it and then waits for them one by one;
// pin() makes the value live where it is called, and batch_fence() keeps the scheduler from moving the uses
// up between the requests.
template <typename V>
__device__ __forceinline__ void pin(V& v) {
    asm volatile("" : "+v"(v));
}
__device__ __forceinline__ void batch_fence() { __builtin_amdgcn_sched_barrier(0); }

// ---- tile geometry for a stage depth of BK reduction elements ---------------------------------------
// (of an operand tile of ROWS rows)
template <int ROWS, int BK>
struct Geometry {
    static constexpr int CPR = BK / 8;            // 16-byte chunks per K-contiguous row
    static constexpr int ROW_BYTES = BK * 2;
    static constexpr int ROWS_PER_LOAD = 64 / CPR;  // tile rows one DMA instruction covers
    static constexpr int LOADS = ROWS * BK * 2 / 1024 / NUM_WAVES;  // DMA instructions per wave, operand and stage
    static constexpr int KROW_CHUNKS = ROWS / 8;             // 16-byte chunks per K-strided row
    static constexpr int KROWS_PER_LOAD = 64 / KROW_CHUNKS;  // reduction rows one DMA instruction covers
    static_assert(BK == 32 || BK == 64, "stage depth");

    __device__ static __forceinline__ int swizzle(int row) { return BK == 32 ? (row >> 2) & 3 : (row >> 1) & 7; }

    // K-contiguous tile: byte offset of the fragment (row, reduction elements kb*32 + 8*quarter .. +7)
    __device__ static __forceinline__ int kcontig_offset(int row, int kb, int quarter) {
        return row * ROW_BYTES + (((4 * kb + quarter) ^ swizzle(row)) << 4);
    }
    // K-strided tile: byte offset of the first of the two transposing reads of the fragment
    // (tile rows col0..col0+15, reduction elements kb*32 .. +31).  Within each 16-lane group the
    // instruction hands lane i the i-th 16-bit element of four 16-element rows, where row j is assembled
    // from the 8-byte pieces addressed by lanes 4j..4j+3.  So lane i of group g addresses (k row 8g + i/4,
    // columns 4*(i%4)..+3) and receives four consecutive k of column i; a second read four k rows further
    // down completes the eight reduction elements 8g .. 8g+7 of the MFMA operand.
    __device__ static __forceinline__ int kstrided_offset(int col0, int kb, int lane) {
        const int i = lane & 15, group = lane >> 4;
        const int col = col0 + 4 * (i & 3);
        const int krow0 = kb * 32 + 8 * group + (i >> 2);
        const int chunk = (col >> 3) ^ ((krow0 & 3) << 2);  // (krow0 + 4) & 3 == krow0 & 3
        return krow0 * (ROWS * 2) + (chunk << 4) + ((col & 4) << 1);
    }
};

template <bool STRIDED, int ROWS>
__device__ __forceinline__ u32x4_t read_fragment(const char* slab_base, int offset) {
    if constexpr (STRIDED) {
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(XMA_LDS_S4(slab_base + offset));
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(XMA_LDS_S4(slab_base + (offset + 4 * (ROWS * 2))));
        const u32x2_t a = __builtin_bit_cast(u32x2_t, lo), b = __builtin_bit_cast(u32x2_t, hi);
        return u32x4_t{a.x, a.y, b.x, b.y};
    } else {
        return *reinterpret_cast<const u32x4_t*>(slab_base + offset);
    }
}

// ---- per-thread DMA plan of one operand ---------------------------------------------------------------
// DMA instruction i of wave w fills the 1 KiB block (i * NUM_WAVES + w) of the operand's LDS tile:
//   K-contiguous tile: tile rows [R * (i * NUM_WAVES + w), +R), R = ROWS_PER_LOAD; lane l -> row + l / CPR,
//     physical chunk l % CPR (the logical chunk it fetches is the XOR-swizzled one, and because R * NUM_WAVES
//     is a multiple of the swizzle period it is the same for every i);
//   K-strided tile: k rows [K * (i * NUM_WAVES + w), +K), K = KROWS_PER_LOAD; lane l -> k row + l / KROW_CHUNKS, physical
//     chunk l % KROW_CHUNKS.
// Three address plans:
//   ROWS     one pointer per instruction (rows that are gathered through an index table or end anywhere),
//   UNIFORM  K-contiguous rows at a constant stride, with one extra jump in the middle of the tile
//            (the up|gate halves of a fused SwiGLU weight tile): one pointer, the rest is scalar arithmetic,
//   STRIDED  K-strided tile: one pointer, constant stride between instructions.
//   GATHERED K-strided tile whose reduction rows lie anywhere: byte offsets of the rows, which are the same for the lanes that
//            fetch one row, are read from a table by scalar loads a phase ahead.  (A vector load would do it per lane, but
//            the compiler waits for vector loads and for the LDS-DMA loads in flight together.)
enum LoadPlan { PLAN_ROWS, PLAN_UNIFORM, PLAN_STRIDED, PLAN_GATHERED };

typedef __attribute__((address_space(4))) const uint32_t scalar_u32_t;  // read by scalar loads where the address is uniform

template <typename T, int ROWS, int BK, LoadPlan PLAN>
struct OperandLoads {
    using G = Geometry<ROWS, BK>;
    static constexpr int LOADS = G::LOADS;
    static constexpr bool KSTRIDED = PLAN == PLAN_STRIDED || PLAN == PLAN_GATHERED;
    static constexpr int RED_STRIDE = KSTRIDED ? G::KROWS_PER_LOAD * NUM_WAVES : 0;  // reduction rows between i and i+1
    const T* ptr[PLAN == PLAN_ROWS ? LOADS : 1];  // HBM address of this lane's chunk in stage 0
    bool valid[KSTRIDED ? 1 : LOADS];  // false: always the zero page (row / column outside the operand)
    int64_t load_stride, mid_jump;  // UNIFORM / STRIDED: elements from instruction i to i+1; UNIFORM: extra at LOADS/2
    int64_t step;                   // elements to advance per stage
    int32_t red0;                   // reduction index covered by the lane in stage 0, instruction 0
    // GATHERED: column offset of the lane's chunk, a mask for each of the rows of a load (all ones in the lanes that fetch
    // it), the table at the wave's first row, and the offsets of the rows of the stage that is requested next
    static constexpr bool GATHERED = PLAN == PLAN_GATHERED;
    uint32_t column, row_mask[GATHERED ? G::KROWS_PER_LOAD : 1];
    scalar_u32_t* table;
    uint32_t row[GATHERED ? LOADS * G::KROWS_PER_LOAD : 1];
    int wave_lds;                   // byte offset of the wave's first 1 KiB block inside the operand's LDS tile

    __device__ static __forceinline__ const T* zero_page() { return reinterpret_cast<const T*>(g_zero_page); }

    // ROWS: row_fn(tile row) returns the HBM row base or nullptr.
    template <typename RowFn>
    __device__ __forceinline__ void setup_rows(int wave, int lane, RowFn row_fn) {
        static_assert(PLAN == PLAN_ROWS, "plan");
        const int chunk = (lane % G::CPR) ^ G::swizzle(wave * G::ROWS_PER_LOAD + lane / G::CPR);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const T* base = row_fn((i * NUM_WAVES + wave) * G::ROWS_PER_LOAD + lane / G::CPR);
            valid[i] = base != nullptr;
            ptr[i] = valid[i] ? base + chunk * 8 : zero_page();
        }
        red0 = chunk * 8;
        step = BK;
        wave_lds = wave * 1024;
    }

    // UNIFORM: tile row r lives at base + r * ld (+ jump in the lower half of the tile); rows_fn(tile row) says whether it exists.
    template <typename ValidFn>
    __device__ __forceinline__ void setup_uniform(int wave, int lane, const T* base, int64_t ld, int64_t jump,
                                                  ValidFn valid_fn) {
        static_assert(PLAN == PLAN_UNIFORM, "plan");
        const int row = wave * G::ROWS_PER_LOAD + lane / G::CPR;
        const int chunk = (lane % G::CPR) ^ G::swizzle(row);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) valid[i] = valid_fn(i * NUM_WAVES * G::ROWS_PER_LOAD + row);
        ptr[0] = base + row * ld + chunk * 8;
        load_stride = NUM_WAVES * G::ROWS_PER_LOAD * ld;
        mid_jump = jump;
        red0 = chunk * 8;
        step = BK;
        wave_lds = wave * 1024;
    }

    // STRIDED: `base` points at (reduction row 0, first tile column); `cols_left` = number of valid columns
    // from there; ld = row stride.
    __device__ __forceinline__ void setup_strided(int wave, int lane, const T* base, int64_t ld, int64_t cols_left) {
        static_assert(PLAN == PLAN_STRIDED, "plan");
        const int krow = wave * G::KROWS_PER_LOAD + lane / G::KROW_CHUNKS;
        const int chunk = (lane % G::KROW_CHUNKS) ^ ((krow & 3) << 2);  // RED_STRIDE is a multiple of 4: same for every i
        valid[0] = chunk * 8 < cols_left;
        ptr[0] = valid[0] ? base + (int64_t)krow * ld + chunk * 8 : zero_page();
        load_stride = RED_STRIDE * ld;
        mid_jump = 0;
        red0 = krow;
        step = (int64_t)BK * ld;
        wave_lds = wave * 1024;
    }

    // GATHERED: `base` points at the first tile column of source row 0, table[r] is the byte offset of reduction row r.
    __device__ __forceinline__ void setup_gathered(int wave, int lane, const T* base, const uint32_t* offsets, int64_t cols_left) {
        static_assert(PLAN == PLAN_GATHERED, "plan");
        const int krow = wave * G::KROWS_PER_LOAD + lane / G::KROW_CHUNKS;
        const int chunk = (lane % G::KROW_CHUNKS) ^ ((krow & 3) << 2);
        valid[0] = chunk * 8 < cols_left;
        ptr[0] = base;
        column = chunk * 16;
#pragma unroll
        for (int j = 0; j < G::KROWS_PER_LOAD; ++j) row_mask[j] = lane / G::KROW_CHUNKS == j ? ~0u : 0u;
        table = (scalar_u32_t*)offsets + wave * G::KROWS_PER_LOAD;
        load_stride = mid_jump = 0;
        red0 = krow;
        step = 0;
        wave_lds = wave * 1024;
    }
    // Requests the row offsets of a stage; up to a load's rows past the end of the reduction are read from the table.
    __device__ __forceinline__ void look_up(int64_t stage) {
        scalar_u32_t* at = table + stage * BK;
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
#pragma unroll
            for (int j = 0; j < G::KROWS_PER_LOAD; ++j) row[i * G::KROWS_PER_LOAD + j] = at[i * RED_STRIDE + j];
    }

    // Make stage 0 the stage `first` of the reduction (split-K parts start in the middle).
    __device__ __forceinline__ void skip_stages(int64_t first) {
#pragma unroll
        for (int i = 0; i < (PLAN == PLAN_ROWS ? LOADS : 1); ++i) ptr[i] += first * step;
    }

    // Issue this wave's loads I0 <= i < I1 of the stage `stage` into the tile at slab_base + tile_off.
    // MASKED = false is for a stage that lies wholly inside the reduction, of a tile none of whose rows and columns
    // is missing (all_valid): the address is the lane's pointer plus a wave-uniform offset and nothing is compared
    // or selected.  A wave that is alone on its SIMD pays an issue slot for every instruction, and the masked form
    // spends five on each load (a 64-bit compare, a mask and, two selects), the plain one none.
    template <int I0, int I1, bool MASKED>
    __device__ __forceinline__ void issue(char* slab_base, int tile_off, int64_t stage, int64_t red_len) const {
        const int64_t red_left = red_len - stage * BK;  // wave-uniform
        const int64_t stage_off = stage * step;
#pragma unroll
        for (int i = I0; i < I1; ++i) {
            const T* p;
            if constexpr (PLAN == PLAN_ROWS) {
                p = ptr[i] + stage_off;
            } else if constexpr (GATHERED) {
                uint32_t off = column;
#pragma unroll
                for (int j = 0; j < G::KROWS_PER_LOAD; ++j) off += row[i * G::KROWS_PER_LOAD + j] & row_mask[j];
                p = reinterpret_cast<const T*>(reinterpret_cast<const char*>(ptr[0]) + off);
            } else p = ptr[0] + (stage_off + i * load_stride + (i >= LOADS / 2 ? mid_jump : 0));
            if constexpr (MASKED) {
                const bool ok = valid[KSTRIDED ? 0 : i] && (red0 + i * RED_STRIDE < red_left);
                // computed for every lane and then selected: a branch around the load would make the number of
                // loads in flight differ between waves
                asm("" : "+v"(p));
                p = ok ? p : zero_page();
            }
            // The wave's share of the LDS address goes through an empty asm that also names the stage, so that the
            // address of every load is ONE scalar add on the spot; left alone, the compiler forms all eighty
            // addresses of a trip round the ring ahead of the loop, runs out of scalar registers and reads them
            // back from vector lanes.  (Not volatile: a volatile asm fences the instruction scheduler, which
            // then cannot spread the loads and LDS reads between the matrix instructions.)
            int w = wave_lds;
            asm("" : "+s"(w) : "s"((int)stage));
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t*>(p),
                                             XMA_LDS(slab_base + (tile_off + i * NUM_WAVES * 1024 + w)), 16, 0, 0);
        }
    }

    // true when no row or column of this wave's share of the operand tile is missing
    __device__ __forceinline__ bool all_valid() const {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < (KSTRIDED ? 1 : LOADS); ++i) ok = ok && valid[i];
        return ok;
    }
};

// ---- pipeline policies --------------------------------------------------------------------------------------
// A policy says where the tiles of stage j live, which loads the step at cycle position P issues in
// each of its phases (one phase = 32 reduction elements), and how many loads may still be in flight when
// the step reaches its barrier.  Loads are spread evenly over the phases: the texture path of a compute
// unit takes about sixteen cycles per DMA instruction and a wave that issues into a full queue stalls,
// matrix instructions included.
//
// Ring64x5: stage j of 64 reduction elements (two phases of 32) keeps its A tile in slab (2j) % 5 and its B tile
// in slab (2j + 1) % 5, so every DMA instruction of a K-contiguous operand asks for whole 128-byte lines.  At a
// step's barrier the next stage has landed and the A tile of the one after is in flight.  The step's own slabs then
// take the B tile of stage s+2 (during the rest of the step) and the A tile of stage s+3 (during the first phase of
// the next step): every load is issued between one and a half and two and a half phases before the barrier that
// needs it.
template <typename TL_>
struct Ring64x5 {
    using TL = TL_;
    static constexpr int BK = 64, CYCLE = 5, KK = 2;
    static constexpr int LA = Geometry<TL::BM, BK>::LOADS, LB = Geometry<TL::BN, BK>::LOADS;
    static constexpr int WAIT = LA;                // loads that may stay in flight at a step's barrier
    static constexpr int PROLOGUE_WAIT = LA + LB;  // ... and when the first stage is needed
    static constexpr int phase_loads(int phase) { return phase == 0 ? LA : LB; }
    template <int P> struct At {
        static constexpr int A_SLAB = (2 * P) % 5, A_OFF = 0, B_SLAB = (2 * P + 1) % 5, B_OFF = 0;
    };
    static constexpr int LOOKAHEAD = 2;  // a step at stage s issues loads of stages up to s + LOOKAHEAD
    template <typename K> __device__ static __forceinline__ void prologue(K& k) {
        k.look_up(0);
        k.template issue_a<0, 0, LA, true>(0); k.template issue_b<0, 0, LB, true>(0);
        k.look_up(1);
        k.template issue_a<1, 0, LA, true>(1); k.template issue_b<1, 0, LB, true>(1);
    }
    // load number I (0 <= I < phase_loads(PH)) of phase PH of the step at ring position P on stage s
    template <int P, int PH, int I, bool MASKED, typename K> __device__ static __forceinline__ void issue_one(K& k, int64_t s) {
        if constexpr (PH == 0) k.template issue_a<(P + 2) % CYCLE, I, I + 1, MASKED>(s + 2);
        else k.template issue_b<(P + 2) % CYCLE, I, I + 1, MASKED>(s + 2);
    }
};

// Ring64x2: two whole stages, for tiles of 128 columns: 192 rows need 40 KiB a stage.  All loads of stage s+2 go out in the
// second phase of step s, one to two phases before the barrier that needs them.
template <typename TL_>
struct Ring64x2 {
    using TL = TL_;
    static constexpr int BK = 64, CYCLE = 2, KK = 2;
    static constexpr int LA = Geometry<TL::BM, BK>::LOADS, LB = Geometry<TL::BN, BK>::LOADS;
    static constexpr int WAIT = 0, PROLOGUE_WAIT = LA + LB;
    static constexpr int phase_loads(int phase) { return phase == 0 ? 0 : LA + LB; }
    template <int P> struct At {
        static constexpr int A_SLAB = 2 * P, A_OFF = 0, B_SLAB = 2 * P + 1, B_OFF = 0;
        static constexpr int EXTRA_SLAB = 5 + P;
    };
    static constexpr int LOOKAHEAD = 2;
    template <typename K> __device__ static __forceinline__ void prologue(K& k) {
        k.template issue_a<0, 0, LA, true>(0); k.template issue_b<0, 0, LB, true>(0);
        k.template issue_a<1, 0, LA, true>(1); k.template issue_b<1, 0, LB, true>(1);
    }
    template <int P, int PH, int I, bool MASKED, typename K> __device__ static __forceinline__ void issue_one(K& k, int64_t s) {
        static_assert(PH == 1, "no loads in the first phase");
        if constexpr (I < LA) k.template issue_a<P, I, I + 1, MASKED>(s + 2);
        else k.template issue_b<P, I - LA, I - LA + 1, MASKED>(s + 2);
    }
};

template <typename T, int KIND, int EPI, typename Pipe, bool GATHER>
struct Kernel {
    static constexpr int BK = Pipe::BK;
    using TL = typename Pipe::TL;
    static constexpr int BM = TL::BM, BN = TL::BN, WM = TL::WM, WN = TL::WN, MI = TL::MI, NI = TL::NI;
    static constexpr bool A_STRIDED = KIND == XMA_GEMM_MT;
    static constexpr bool B_STRIDED = KIND != XMA_GEMM_TN;
    static constexpr int BN_OUT = EPI == EPI_PAIRED ? BN / 2 : BN;

    OperandLoads<T, BM, BK, A_STRIDED ? PLAN_STRIDED : PLAN_ROWS> la;
    OperandLoads<T, BN, BK, GATHER ? PLAN_GATHERED : B_STRIDED ? PLAN_STRIDED : PLAN_UNIFORM> lb;
    int64_t red_len;
    int wave, lane;
    int a_off[4], b_off[4], extra_off[4];  // variable parts of the fragment offsets (see fragment_offsets)
    u32x4_t fa[2][MI], fb[2][NI];  // fragments: the 32-deep block being multiplied and the one being read

    template <int P, int I0, int I1, bool MASKED> __device__ __forceinline__ void issue_a(int64_t stage) {
        using At = typename Pipe::template At<P>;
        constexpr int MAIN = TL::EXTRA ? 4 : I1, M1 = I1 < MAIN ? I1 : MAIN;  // a load covers 32 tile rows over the waves
        if constexpr (I0 < M1) la.template issue<I0, M1, MASKED>(TL::template slab<At::A_SLAB>(), At::A_OFF, stage, red_len);
        if constexpr (TL::EXTRA && I1 > 4)
            la.template issue<(I0 < 4 ? 4 : I0), I1, MASKED>(TL::template slab<At::EXTRA_SLAB>(), -4 * NUM_WAVES * 1024, stage, red_len);
    }
    template <int P, int I0, int I1, bool MASKED> __device__ __forceinline__ void issue_b(int64_t stage) {
        lb.template issue<I0, I1, MASKED>(TL::template slab<Pipe::template At<P>::B_SLAB>(), Pipe::template At<P>::B_OFF, stage, red_len);
    }

    // the gathered rows of the B tile of a stage, ahead of its loads
    __device__ __forceinline__ void look_up(int64_t stage) {
        if constexpr (GATHER) lb.look_up(stage);
    }

    // Byte offsets of this lane's fragments inside an operand tile.  Only the part that is not a
    // compile-time constant goes through opaque(): for the K-contiguous layout the 16-row block adds a
    // constant (the swizzle repeats every 16 rows); for the K-strided layout the 32-deep block adds 64 * ROWS bytes and
    // the odd 16-column block of a 32-column pair adds 32 bytes (two chunks; the swizzle leaves that bit alone).
    template <bool STRIDED, int ROWS>
    __device__ __forceinline__ void fragment_offsets(int row0, int (&var)[4]) const {
        using G = Geometry<ROWS, BK>;
        if constexpr (STRIDED) {
#pragma unroll
            for (int b = 0; b < ROWS / 64; ++b) var[b] = opaque(G::kstrided_offset(row0 + b * 32, 0, lane));
        } else {
#pragma unroll
            for (int kb = 0; kb < BK / 32; ++kb) var[kb] = opaque(G::kcontig_offset(row0 + (lane & 15), kb, lane >> 4));
        }
    }
    template <bool STRIDED, int ROWS>
    __device__ static __forceinline__ int fragment_offset(const int (&var)[4], int block, int kb) {
        return STRIDED ? var[block >> 1] + (block & 1) * 32 + kb * (32 * ROWS * 2) : var[kb] + block * (16 * Geometry<ROWS, BK>::ROW_BYTES);
    }
    __device__ __forceinline__ void init_fragments() {
        fragment_offsets<A_STRIDED, BM>(TL::block_row(wave / WAVES_N, 0), a_off);
        if constexpr (TL::EXTRA) fragment_offsets<A_STRIDED, BM>(TL::block_row(wave / WAVES_N, TL::MAIN_BLOCKS) - 128, extra_off);
        fragment_offsets<B_STRIDED, BN>((wave % WAVES_N) * WN, b_off);
    }

    // One fragment of the 32-deep block kb of the stage held at ring position P: A block mi / B block ni.
    template <int P>
    __device__ __forceinline__ u32x4_t read_a(int kb, int mi) const {
        using At = typename Pipe::template At<P>;
        if constexpr (TL::EXTRA) {
            static_assert(!A_STRIDED, "rows that do not fit one slab");
            if (mi >= TL::MAIN_BLOCKS)
                return read_fragment<false, BM>(TL::template slab<At::EXTRA_SLAB>(),
                                                fragment_offset<false, BM>(extra_off, mi - TL::MAIN_BLOCKS, kb));
        }
        return read_fragment<A_STRIDED, BM>(TL::template slab<At::A_SLAB>(), At::A_OFF + fragment_offset<A_STRIDED, BM>(a_off, mi, kb));
    }
    template <int P>
    __device__ __forceinline__ u32x4_t read_b(int kb, int ni) const {
        using At = typename Pipe::template At<P>;
        return read_fragment<B_STRIDED, BN>(TL::template slab<At::B_SLAB>(), At::B_OFF + fragment_offset<B_STRIDED, BN>(b_off, ni, kb));
    }
    // All fragments of a block.
    template <int P>
    __device__ __forceinline__ void read_fragments(int kb, u32x4_t (&af)[MI], u32x4_t (&bf)[NI]) const {
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) bf[ni] = read_b<P>(kb, ni);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) af[mi] = read_a<P>(kb, mi);
    }

    // One phase = one 32-deep block = MI * NI matrix instructions of 16 cycles.  A wave that is alone on its SIMD
    // has nobody to hide its stalls, so the three instruction streams are interleaved by hand: the phase is cut into
    // slots of two matrix instructions (one B block against two A blocks; of one, where the wave has one A block), 32 of them for
    // a 256 x 256 tile.  The MI + NI reads of the NEXT phase's fragments and the phase's DMA loads are spread evenly over the
    // slots: for 256 x 256 every odd slot reads one block and every fourth issues one load.  The matrix instructions are inline
    // assembly, which the instruction scheduler cannot classify, so the order is pinned with a scheduling fence
    // after each slot.  RP / RKB: ring position and block of the fragments being read; LP / LPH: the step and phase
    // whose loads go out.
    //
    // The granularity and the placement are measured choices (benchmark layer, all launches of a pass, same
    // session): against 16 slots of four instructions with the B blocks read two per slot in the first four slots
    // and the loads in the odd slots, this schedule is 3.3 % faster; with the loads in slot 1 instead of slot 0 of
    // every four 2.6 %; 16 slots with the reads spread out and the loads in even slots 1.4 %.  The kinds differ in
    // the best order of the reads: all A blocks, then all B blocks where both operands cost the same number of LDS
    // instructions (TN, MT), alternating where the transposed operand costs twice as many (NN).  One instruction
    // per slot makes no difference where it compiles (NN: +-0.5 %); for TN and MT the compiler runs out of scalar
    // registers ("illegal VGPR to SGPR copy"), and with the scalar operands of the loads forced through
    // v_readfirstlane it spills thousands of vector registers.
    //
    // The tail tile of an expert's rows runs exactly the same instruction stream on zeros for the rows that do not
    // exist.  Skipping the missing 16-row blocks was measured and is a LOSS: the 32 work-groups an XCD runs at a
    // time share their operand panels through the L2 only while they walk the reduction in step; a tile that
    // finishes early puts its compute unit out of step for the rest of the launch, its requests stop hitting lines
    // its neighbours brought in, and the launch, which is bound by what the L2 has to fetch, gets 13-16 % slower
    // (8 tail tiles among 67 at the benchmark shape).
    // Tail tiles of up to 128 rows as tiles of 128 x 256, which cost half: the input gradients gain where the reductions are
    // short, the forward kinds win here and lose there (us, without / with, up, down, dact, dX: 16384 tokens, 64 experts, 6
    // each, H 2048, I 1024 772 / 762, 431 / 435, 469 / 467, 760 / 737; 128 experts, 8 each, skewed 744 / 734, 470 / 491, 478 /
    // 467, 797 / 755; 12000 tokens of the first 567 / 584, 314 / 325, 346 / 343, 557 / 554; 8192 tokens, 8 experts, 4 each, I
    // 8192 1999 / 1990, 819 / 819, 1217 / 1155, 1623 / 1621).  So the input gradients have them.
    template <int RP, int LP, int LPH, bool MASKED>
    __device__ __forceinline__ void phase(int rkb, int cur, int64_t s, f32x4_t (&acc)[MI][NI]) {
        constexpr int IN_SLOT = MI < 2 ? 1 : 2, SLOTS = MI * NI / IN_SLOT, PER_B = MI / IN_SLOT;
        constexpr int READ_SLOTS = GATHER && LPH == 1 ? SLOTS - SLOTS / 8 : SLOTS;  // (see step)
        constexpr int READS = MI + NI, LOADS = Pipe::phase_loads(LPH);
        const int nxt = cur ^ 1;
#pragma unroll
        for (int slot = 0; slot < SLOTS; ++slot) {
            const int ni = slot / PER_B, m0 = (slot % PER_B) * IN_SLOT;
#pragma unroll
            for (int i = 0; i < IN_SLOT; ++i) Mma16<T>::run(fb[cur][ni], fa[cur][m0 + i], acc[m0 + i][ni]);
#pragma unroll
            for (int r = 0; r < READS; ++r) {  // the r-th fragment block of the next phase
                const int last = (r + 1) * READ_SLOTS / READS - 1;
                if (slot != (last < 0 ? 0 : last)) continue;
                if constexpr (KIND == XMA_GEMM_NN && MI == NI) {
                    if (r % 2 == 0) fa[nxt][r / 2] = read_a<RP>(rkb, r / 2);
                    else fb[nxt][r / 2] = read_b<RP>(rkb, r / 2);
                } else {
                    if (r < MI) fa[nxt][r] = read_a<RP>(rkb, r);
                    else fb[nxt][r - MI] = read_b<RP>(rkb, r - MI);
                }
            }
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                if (slot == i * SLOTS / LOADS) issue_slot<LP, LPH, MASKED>(i, s);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    template <int LP, int LPH, bool MASKED>
    __device__ __forceinline__ void issue_slot(int i, int64_t s) {
        // i is a constant after unrolling
        auto one = [&](auto tag) {
            constexpr int I = decltype(tag)::value;
            if constexpr (I < Pipe::phase_loads(LPH)) Pipe::template issue_one<LP, LPH, I, MASKED>(*this, s);
        };
        switch (i) {
            case 0: one(std::integral_constant<int, 0>{}); break;
            case 1: one(std::integral_constant<int, 1>{}); break;
            case 2: one(std::integral_constant<int, 2>{}); break;
            case 3: one(std::integral_constant<int, 3>{}); break;
            case 4: one(std::integral_constant<int, 4>{}); break;
            case 5: one(std::integral_constant<int, 5>{}); break;
            case 6: one(std::integral_constant<int, 6>{}); break;
            case 7: one(std::integral_constant<int, 7>{}); break;
            case 8: one(std::integral_constant<int, 8>{}); break;
            default: one(std::integral_constant<int, 9>{}); break;
        }
    }
    // One pipeline step at ring position P on stage s.  On entry the fragments of the stage's first block are in
    // registers (set 0).  Phase 0 multiplies block 0 while block 1 is read and the A tile of stage s+2 is requested.
    // Then the step waits until its own LDS reads are done and the loads of stage s+1 have landed, and meets the
    // other waves: stage s+1 is then complete for everybody and nobody reads stage s any more, so its slabs can be
    // refilled while block 1 is multiplied from registers and the first fragments of stage s+1 are read.  A step is
    // branch-free: stages past the end of the reduction fetch the zero page, which keeps the count of loads in
    // flight the same at every step and lets the compiler see that the loop needs no other wait on vector memory.
    template <int P, bool MASKED>
    __device__ __forceinline__ void step(int64_t s, f32x4_t (&acc)[MI][NI]) {
        static_assert(Pipe::KK == 2 && Pipe::phase_loads(0) <= 10 && Pipe::phase_loads(1) <= 10, "two phases of up to ten loads");
        // Gathered rows: the offsets of the B tile that is requested in the second phase.  Scalar loads share a counter with
        // the fragment reads and return in any order, so the compiler waits for all of both wherever a fragment is used
        // while they are on their way.  Hence the reads of a stage's first block are done a few slots early and waited for
        // here, and nothing else is until the step's barrier.
        if constexpr (GATHER) {
            wait_lds();
            look_up(s + 2);
        }
        phase<P, P, 0, MASKED>(1, 0, s, acc);
        wait_vmcnt_and_lds<Pipe::WAIT>();
        block_barrier();
        phase<(P + 1) % Pipe::CYCLE, P, 1, MASKED>(0, 1, s, acc);
    }

    template <int P>
    __device__ __forceinline__ void steps_from(int64_t s, int64_t count, f32x4_t (&acc)[MI][NI]) {
        if constexpr (P < Pipe::CYCLE) {
            if (P < count) {
                step<P, true>(s + P, acc);
                steps_from<P + 1>(s, count, acc);
            }
        }
    }
    template <int P, bool MASKED>
    __device__ __forceinline__ void full_cycle(int64_t s, f32x4_t (&acc)[MI][NI]) {
        if constexpr (P < Pipe::CYCLE) {
            step<P, MASKED>(s + P, acc);
            full_cycle<P + 1, MASKED>(s, acc);
        }
    }

    // `plain_steps`: the first that many steps only issue loads of stages that lie wholly inside the reduction, in a
    // tile without missing rows or columns; they take the unmasked form of the loads.
    __device__ __forceinline__ void run_stages(int64_t num_stages, int64_t plain_steps, f32x4_t (&acc)[MI][NI]) {
        read_fragments<0>(0, fa[0], fb[0]);
        int64_t s = 0;
        for (; s + Pipe::CYCLE <= plain_steps; s += Pipe::CYCLE) full_cycle<0, false>(s, acc);
        for (; s + Pipe::CYCLE <= num_stages; s += Pipe::CYCLE) full_cycle<0, true>(s, acc);
        steps_from<0>(s, num_stages - s, acc);  // fewer than CYCLE steps remain
    }

    __device__ __forceinline__ void run(f32x4_t (&acc)[MI][NI]) {
        const int64_t num_stages = (red_len + BK - 1) / BK;
        if (num_stages > 0) {
            Pipe::prologue(*this);
            wait_vmcnt<Pipe::PROLOGUE_WAIT>();
            block_barrier();
            // wave-uniform: validity is a property of rows and columns of the tile, combined over the lanes; the
            // plain and the masked loops issue the same loads and meet at the same barriers, so the waves of a
            // work-group may disagree
            const bool whole = __builtin_amdgcn_readfirstlane(__all((int)(la.all_valid() && lb.all_valid()))) != 0;
            const int64_t plain = whole ? red_len / BK - Pipe::LOOKAHEAD : 0;
            run_stages(num_stages, plain, acc);
            wait_vmcnt<0>();  // the trailing zero-page loads
            // The matrix instructions are inline assembly, so the compiler does not know that the accumulators are
            // still being written when the loop ends and would not keep the distance the hardware needs between a
            // matrix instruction and a read of its result: 32 idle cycles cover it.
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        }
        block_barrier();  // every wave is done reading the slabs; no load is in flight any more
    }
};

// What a work-group multiplies.
struct TilePlace {
    int expert;
    int64_t m_begin, m_end;  // the tile's routed rows; MT: the expert's, which are reduced over
    int64_t i0, n0;          // first row (MT) and column of the result
    TileWork work;
};

template <typename T, int KIND, int EPI, typename Pipe, bool GATHER = false>
__device__ __forceinline__ void multiply_tile(const GemmParams& P, const TilePlace& place) {
    using K = Kernel<T, KIND, EPI, Pipe, GATHER>;
    using TL = typename Pipe::TL;
    constexpr int BM = TL::BM, BN = TL::BN, WM = TL::WM, WN = TL::WN, MI = TL::MI, NI = TL::NI;
    constexpr int OUT_SLABS = TL::OUT_SLABS, SLAB_BLOCKS = TL::SLAB_BLOCKS;
    constexpr int PV = 8;
    constexpr int BN_OUT = K::BN_OUT;

    const int tid = threadIdx.x;
    K k;
    k.lane = tid & 63;
    k.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int expert = place.expert;
    const int64_t m_begin = place.m_begin, m_end = place.m_end, tile_i0 = place.i0, n0 = place.n0;
    const TileWork& work = place.work;
    k.red_len = KIND == XMA_GEMM_MT ? m_end - m_begin : P.k;
    const T* A = reinterpret_cast<const T*>(P.a);
    const T* B = reinterpret_cast<const T*>(P.b);

    // ---- operand load plans ----
    if constexpr (KIND == XMA_GEMM_MT) {
        k.la.setup_strided(k.wave, k.lane, A + m_begin * P.lda + tile_i0, P.lda, P.n - tile_i0);
        if constexpr (GATHER) k.lb.setup_gathered(k.wave, k.lane, B + n0, P.row_offsets + m_begin, P.k - n0);
        else k.lb.setup_strided(k.wave, k.lane, B + m_begin * P.ldb + n0, P.ldb, P.k - n0);
    } else {
        // The three ways of finding a row's source are told apart once, outside the per-row code, and rows past
        // the end look up the tile's first row (which always exists) and are then dropped: with a branch per
        // row the eight index loads of a lane would wait for each other.
        auto plan_rows = [&](auto source_of) {
            k.la.setup_rows(k.wave, k.lane, [&](int r) -> const T* {
                const int64_t p = m_begin + r;
                const bool exists = p < m_end;
                const T* row = A + source_of(exists ? p : m_begin) * P.lda;
                return exists ? row : nullptr;
            });
        };
        const uint32_t fan_out = (uint32_t)P.in_fan_out;
        if (P.in_index == nullptr)
            plan_rows([&](int64_t p) { return p; });
        else if (P.idx_is_i64)
            plan_rows([&](int64_t p) {
                return (int64_t)((uint32_t)reinterpret_cast<const int64_t*>(P.in_index)[p] / fan_out);
            });
        else
            plan_rows([&](int64_t p) {
                return (int64_t)((uint32_t)reinterpret_cast<const int32_t*>(P.in_index)[p] / fan_out);
            });
        const T* W = B + (int64_t)expert * P.b_expert_stride;
        if constexpr (KIND == XMA_GEMM_TN) {
            if constexpr (EPI == EPI_PAIRED) {
                // tile row r < BN_OUT: weight row n0 + r (up half); others: P.n / 2 + n0 + r - BN_OUT (gate half)
                const int64_t half = P.n / 2;
                k.lb.setup_uniform(k.wave, k.lane, W + n0 * P.ldb, P.ldb, (half - BN_OUT) * P.ldb,
                                   [&](int r) { return n0 + (r % BN_OUT) < half; });
            } else {
                k.lb.setup_uniform(k.wave, k.lane, W + n0 * P.ldb, P.ldb, 0, [&](int r) { return n0 + r < P.n; });
            }
        } else {
            k.lb.setup_strided(k.wave, k.lane, W + n0, P.ldb, P.n - n0);
        }
    }
    if constexpr (KIND != XMA_GEMM_MT) {
        if (work.parts > 1) {
            const int64_t stages = (k.red_len + K::BK - 1) / K::BK;
            const int64_t first = work.part * stages / work.parts, end = (work.part + 1) * stages / work.parts;
            k.la.skip_stages(first);
            k.lb.skip_stages(first);
            k.red_len = (end * K::BK < k.red_len ? end * K::BK : k.red_len) - first * K::BK;
        }
    }
    k.init_fragments();
    f32x4_t acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    k.run(acc);

    // ---- split-K: every part parks its accumulators; the part that arrives last adds them up in part order
    // (so the result does not depend on the arrival order) and goes on to the epilogue ----
    if constexpr (KIND != XMA_GEMM_MT) {
        if (work.parts > 1) {
            // The parts of a tile run on different XCDs, whose L2 caches are not kept coherent with each other.  Fences
            // at device scope would do (each writes back and invalidates the XCD's whole L2, once per wave, under
            // every other work-group of the XCD: 150-200 k cycles per exchange, measured).  Instead the partial sums
            // and the arrival counter are accessed with relaxed DEVICE-SCOPE ATOMIC stores, loads and one
            // read-modify-write.  What the exchange relies on, and where each piece comes from:
            //   (1) a device-scope atomic access is performed at the level of the memory hierarchy that all XCDs
            //       share, never out of an XCD's private L2: the gfx942/gfx950 memory model of the compiler gives such
            //       accesses the sc1 bit for exactly that reason (atomicity across the XCDs of one device);
            //   (2) `s_waitcnt vmcnt(0)` returns when every earlier vector-memory access of the wave, stores
            //       included, has been acknowledged by the level that performs it;
            //   (3) the work-group barrier (with its release / acquire fences at work-group scope, which also stop
            //       the compiler from moving memory accesses across it) orders the four waves: when thread 0 counts
            //       the arrival, all partial sums of the work-group have been performed;
            //   (4) the read-modify-write on the counter is performed at the same shared level, so the part that
            //       reads parts - 1 comes after every other part's sums; its loads, device-scope atomics again, are
            //       issued after a further work-group barrier and cannot be satisfied from a stale line of its L2.
            // The compiler cannot reorder any of this: the waits carry memory clobbers, the barriers are fences, and
            // atomics are never merged, widened or hoisted across them.
            auto part_buffer = [&](int part) {
                return reinterpret_cast<uint64_t*>(P.split_partials +
                                                   (int64_t)(part * work.split_tiles + work.split_tile) * split_tile_floats(BN));
            };
            uint64_t* mine = part_buffer(work.part);
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        const float2 v{acc[mi][ni][2 * g], acc[mi][ni][2 * g + 1]};
                        __hip_atomic_store(mine + ((mi * NI + ni) * 2 + g) * THREADS + tid, __builtin_bit_cast(uint64_t, v),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
            wait_vmcnt<0>();  // this wave's partial sums have reached memory ...
            __syncthreads();  // ... and so have everybody else's, before the arrival is counted
            int* arrivals = reinterpret_cast<int*>(TL::template slab<0>());
            if (tid == 0)
                arrivals[0] = __hip_atomic_fetch_add(P.split_counters + work.split_tile, 1, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            const bool last = arrivals[0] == work.parts - 1;
            __syncthreads();  // the slab is reused below
            if (!last) return;
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            // The sums are requested 32 loads at a time and added afterwards: with all 256 accumulators live the
            // compiler otherwise fetches them one by one, a full memory latency each.
            for (int part = 0; part < work.parts; ++part) {
                const uint64_t* src = part_buffer(part);
#pragma unroll
                for (int m2 = 0; m2 < OUT_SLABS; ++m2) {
                    uint64_t v[SLAB_BLOCKS][NI][2];
#pragma unroll
                    for (int h = 0; h < SLAB_BLOCKS; ++h)
#pragma unroll
                        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                            for (int g = 0; g < 2; ++g)
                                v[h][ni][g] = __hip_atomic_load(src + (((SLAB_BLOCKS * m2 + h) * NI + ni) * 2 + g) * THREADS + tid,
                                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    batch_fence();
#pragma unroll
                    for (int h = 0; h < SLAB_BLOCKS; ++h)
#pragma unroll
                        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                            for (int g = 0; g < 2; ++g) pin(v[h][ni][g]);
#pragma unroll
                    for (int h = 0; h < SLAB_BLOCKS; ++h)
#pragma unroll
                        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                            for (int g = 0; g < 2; ++g) {
                                const float2 f = __builtin_bit_cast(float2, v[h][ni][g]);
                                acc[SLAB_BLOCKS * m2 + h][ni][2 * g] += f.x;
                                acc[SLAB_BLOCKS * m2 + h][ni][2 * g + 1] += f.y;
                            }
                    batch_fence();
                }
            }
        }
    }

    // ---- epilogue: accumulators -> LDS (slab mi holds SLAB_ROWS / 2 tile rows of each wave row, see row_base) -> HBM ----
    // Store phase: each thread owns one 16-byte chunk column (cc) and, per slab, the IT buffer rows
    // tid / C_CHUNKS + ROW_STEP * it.  What the rows need from HBM (scatter indices, the saved pre-activation of the
    // activation backward) is requested in batches before it is used: the indices of all slabs before the
    // accumulators are packed (and waited for after that), a slab's pre-activations one slab ahead.
    T* C = reinterpret_cast<T*>(P.c);
    constexpr int C_CHUNKS = BN / PV;             // 32 or 16
    constexpr int ROW_STEP = THREADS / C_CHUNKS;  // 8 or 16
    constexpr int SLAB_ROWS = 32 * SLAB_BLOCKS;   // buffer rows of a slab, half of them of each wave row
    constexpr int IT = SLAB_ROWS / ROW_STEP;      // 8, 4 or 2
    // Per-lane coordinates are derived from a fresh, opaque copy of the thread index: derived from `tid` they
    // would be the values computed before the main loop, which the compiler then keeps in scratch memory
    // across the loop and reloads in the middle of the epilogue's batched requests.
    // A wave that is alone on its SIMD issues one vector instruction every 4-5 cycles, so this part of the kernel
    // is bound by its instruction count: row arithmetic is 32-bit and relative to the tile (the thread's first
    // buffer row r0 plus a compile-time constant), and whether a row exists is one compare against a scalar where
    // the row is used, not a mark kept per row.
    const int etid = opaque(tid);
    const int cc = etid & (C_CHUNKS - 1);
    const int r0 = (etid / C_CHUNKS) & (ROW_STEP - 1);
    auto buffer_row = [&](int it) { return r0 + it * ROW_STEP; };
    // tile row of buffer row r0 + ROW_STEP * it of slab mi, less r0: the upper half of the buffer rows are tile
    // rows from mi * SLAB_ROWS / 2, the lower half the same rows of the lower wave row (+WM)
    auto row_base = [](int mi, int it) { return TL::block_row(it / (IT / 2), mi * SLAB_BLOCKS) + (it % (IT / 2)) * ROW_STEP; };
    const int rows_here = (int)(m_end - m_begin);  // 1..BM
    auto row_exists = [&](int mi, int it) { return r0 < rows_here - row_base(mi, it); };
    // a row of the tile that exists: the wanted one or, past the end, the last one
    auto safe_row = [&](int mi, int it) {
        const int r = r0 + row_base(mi, it);
        return (uint32_t)(r < rows_here ? r : rows_here - 1);
    };

    int32_t orow[OUT_SLABS][IT];  // output row of each owned row (of the last existing row for rows past the end)
    if constexpr (KIND != XMA_GEMM_MT) {
        auto fill = [&](auto index_of) {
#pragma unroll
            for (int mi = 0; mi < OUT_SLABS; ++mi)
#pragma unroll
                for (int it = 0; it < IT; ++it) orow[mi][it] = index_of(safe_row(mi, it));
            batch_fence();  // the loads stay in flight while the accumulators are packed; they are waited for after that
        };
        if (EPI == EPI_BACKWARD || P.out_index == nullptr) {  // that epilogue only writes grouped rows
            const int32_t first = (int32_t)m_begin;
            fill([&](uint32_t r) { return first + (int32_t)r; });
        } else if (P.idx_is_i64) {
            const int64_t* index = reinterpret_cast<const int64_t*>(P.out_index) + m_begin;
            fill([&](uint32_t r) { return (int32_t)index[r]; });
        } else {
            const int32_t* index = reinterpret_cast<const int32_t*>(P.out_index) + m_begin;
            fill([&](uint32_t r) { return index[r]; });
        }
    }

    // Activation backward: the saved pre-activation chunks (the two halves of a gated one; tanh-GELU has a single
    // half, fetched twice) of the rows of slab mi, double-buffered so that slab mi+1 is on its way from HBM while
    // slab mi is processed
    constexpr bool SWBWD = EPI == EPI_BACKWARD;
    u32x4_t hu[SWBWD ? 2 : 1][IT], hg[SWBWD ? 2 : 1][IT];
    auto load_saved = [&](int mi, u32x4_t (&up)[IT], u32x4_t (&gate)[IT]) {
        // branch-free: rows / columns outside the tile's part of the operand re-read a valid chunk
        const int64_t n = n0 + cc * PV < P.n ? n0 + cc * PV : 0;
        const int64_t second_half = P.act == ACT_GELU_TANH ? 0 : P.n;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const T* h = reinterpret_cast<const T*>(P.aux) + (m_begin + safe_row(mi, it)) * P.ld_aux;
            up[it] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(h + n));
            gate[it] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(h + second_half + n));
        }
    };
    if constexpr (SWBWD) load_saved(0, hu[0], hg[0]);

    // MFMA result register r of lane l in block (mi, ni): tile row 16*mi + l%16, tile column 16*ni + 4*(l/16) + r.
    // Slab s holds the blocks mi = SLAB_BLOCKS * s + h of both wave rows wr as buffer rows wr * SLAB_ROWS / 2 + 16 * h + 0..15.
    // An LDS row holds C_CHUNKS chunks of 8 columns; chunk c of buffer row br sits at c ^ (br % C_CHUNKS).
    {
        const int wn0 = (k.wave % WAVES_N) * WN;
        const int br0 = (k.wave / WAVES_N) * (SLAB_ROWS / 2) + (etid & 15);  // buffer row of the first block of a slab
        const int quarter = (etid >> 4) & 3;
        // Forward kinds: the expert's bias row, added to the fp32 sums before they are rounded.  Tile column c is
        // weight row n0 + c, or for a gated tile n0 + c (c < BN/2) and N/2 + n0 + c - BN/2 (c >= BN/2).
        float bias[KIND == XMA_GEMM_TN ? NI : 1][KIND == XMA_GEMM_TN ? 4 : 1];
        bool with_bias = false;
        if constexpr (KIND == XMA_GEMM_TN) {
            with_bias = P.bias != nullptr;
            if (with_bias) {
                const T* row = reinterpret_cast<const T*>(P.bias) + (int64_t)expert * P.ld_bias;
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
                    const int c = wn0 + ni * 16 + 4 * quarter;
                    int64_t n;
                    bool exists;
                    if constexpr (EPI == EPI_PAIRED) {
                        const int64_t half_n = P.n / 2;
                        n = n0 + (c % BN_OUT) + (c >= BN_OUT ? half_n : 0);
                        exists = n0 + (c % BN_OUT) < half_n;
                    } else {
                        n = n0 + c;
                        exists = n < P.n;
                    }
                    const uint2 raw = *reinterpret_cast<const uint2*>(row + (exists ? n : 0));
                    float v[8];
                    Elem<T>::unpack(make_uint4(raw.x, raw.y, 0u, 0u), v);
#pragma unroll
                    for (int q = 0; q < 4; ++q) bias[ni][q] = exists ? v[q] : 0.0f;
                }
            }
        }
        // (the bias is a copy of the code of its own: a wave alone on its SIMD pays for every instruction, and as
        // one copy the compiler adds a selected zero to every sum of a launch that has no bias)
        auto write_rows = [&](char* buf, const f32x4_t (&even)[NI], const f32x4_t (&odd)[NI], auto bias_tag) {
            // (a slab of one block has no odd one)
            constexpr bool BIAS = decltype(bias_tag)::value;
#pragma unroll
            for (int h = 0; h < SLAB_BLOCKS; ++h) {
                const int br = br0 + 16 * h;
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
                    const f32x4_t& a = h == 0 ? even[ni] : odd[ni];
                    const int c = wn0 + ni * 16 + 4 * quarter;
                    const int chunk = (c >> 3) ^ (br & (C_CHUNKS - 1));
                    float v[4] = {a[0], a[1], a[2], a[3]};
                    if constexpr (BIAS) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[q] += bias[KIND == XMA_GEMM_TN ? ni : 0][KIND == XMA_GEMM_TN ? q : 0];
                    }
                    *reinterpret_cast<uint2*>(buf + br * (BN * 2) + (chunk << 4) + (quarter & 1) * 8) =
                        make_uint2(Elem<T>::pack2(v[0], v[1]), Elem<T>::pack2(v[2], v[3]));
                }
            }
        };
        auto write_all = [&](auto bias_tag) {
            write_rows(TL::template slab<0>(), acc[0], acc[SLAB_BLOCKS - 1], bias_tag);
            if constexpr (OUT_SLABS >= 2) write_rows(TL::template slab<1>(), acc[2], acc[3], bias_tag);
            if constexpr (OUT_SLABS >= 3) write_rows(TL::template slab<2>(), acc[4], acc[5], bias_tag);
            if constexpr (OUT_SLABS >= 4) write_rows(TL::template slab<3>(), acc[6], acc[7], bias_tag);
        };
        if (KIND == XMA_GEMM_TN && with_bias) write_all(std::true_type{});
        else write_all(std::false_type{});
    }
    if constexpr (KIND != XMA_GEMM_MT) {
        batch_fence();
#pragma unroll
        for (int mi = 0; mi < OUT_SLABS; ++mi)
#pragma unroll
            for (int it = 0; it < IT; ++it) pin(orow[mi][it]);
    }
    __syncthreads();

    auto store_rows = [&](const char* buf, auto mi_tag, const int32_t (&out_row)[IT]) {
        constexpr int mi = decltype(mi_tag)::value;
        auto chunk_at = [&](int br, int c) {
            return *reinterpret_cast<const u32x4_t*>(buf + br * (BN * 2) + ((c ^ (br & (C_CHUNKS - 1))) << 4));
        };
        auto to_uint4 = [](const u32x4_t& v) { return make_uint4(v[0], v[1], v[2], v[3]); };
        // the thread's chunk of each of its IT rows of the slab, requested together
        auto read_own_chunks = [&](u32x4_t (&v)[IT]) {
#pragma unroll
            for (int it = 0; it < IT; ++it) v[it] = chunk_at(buffer_row(it), cc);
            batch_fence();
#pragma unroll
            for (int it = 0; it < IT; ++it) pin(v[it]);
        };
        if constexpr (KIND == XMA_GEMM_MT) {
            const int64_t j = n0 + cc * PV;
            T* out = C + (int64_t)expert * P.c_expert_stride + j;
            u32x4_t v[IT];
            read_own_chunks(v);
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int64_t i = tile_i0 + r0 + row_base(mi, it);
                // streaming store: a weight gradient is read again only by the optimizer, so it should not push the
                // operand panels of the running tiles out of the caches (1-2 % on this kind)
                if (i < P.n && j < P.k) __builtin_nontemporal_store(v[it], reinterpret_cast<u32x4_t*>(out + i * P.ldc));
            }
        } else if constexpr (EPI == EPI_PLAIN) {
            const int64_t n = n0 + cc * PV;
            u32x4_t v[IT];
            read_own_chunks(v);
            if (KIND == XMA_GEMM_TN && P.act == ACT_GELU_TANH) {
                // tanh-GELU of the product; the rounded product itself is kept as the pre-activation
#pragma unroll
                for (int it = 0; it < IT; ++it) {
                    if (!row_exists(mi, it) || n >= P.n) continue;
                    const int64_t p = m_begin + r0 + row_base(mi, it);
                    if (P.aux) *reinterpret_cast<u32x4_t*>(reinterpret_cast<T*>(P.aux) + p * P.ld_aux + n) = v[it];
                    float h[PV], o[PV];
                    Elem<T>::unpack(to_uint4(v[it]), h);
#pragma unroll
                    for (int q = 0; q < PV; ++q) o[q] = gelu_tanh_forward<true>(h[q]);
                    *reinterpret_cast<uint4*>(C + (int64_t)out_row[it] * P.ldc + n) = Elem<T>::pack(o);
                }
            } else {
#pragma unroll
                for (int it = 0; it < IT; ++it)
                    if (row_exists(mi, it) && n < P.n)
                        __builtin_nontemporal_store(v[it], reinterpret_cast<u32x4_t*>(C + (int64_t)out_row[it] * P.ldc + n));
            }
        } else if constexpr (EPI == EPI_PAIRED) {
            // The slab row holds the chunks of the up half, then the matching chunks of the gate half.  Thread cc
            // handles chunk pair cc % HALF_CHUNKS on every other owned row (even `it` for cc < HALF_CHUNKS, odd
            // otherwise), so that every lane computes.
            constexpr int HALF_CHUNKS = C_CHUNKS / 2;
            const int64_t half_n = P.n / 2;
            const int pair = cc % HALF_CHUNKS;
            const int64_t j = n0 + pair * PV;
            const bool odd = cc >= HALF_CHUNKS;
            const int r1 = r0 + (odd ? ROW_STEP : 0);  // the thread's first buffer row among those it computes
            u32x4_t ups[IT / 2], gates[IT / 2];
#pragma unroll
            for (int it2 = 0; it2 < IT / 2; ++it2) {
                const int br = r1 + 2 * it2 * ROW_STEP;
                ups[it2] = chunk_at(br, pair);
                gates[it2] = chunk_at(br, pair + HALF_CHUNKS);
            }
            batch_fence();
#pragma unroll
            for (int it2 = 0; it2 < IT / 2; ++it2) {
                pin(ups[it2]);
                pin(gates[it2]);
            }
            // one copy of the loop per activation, chosen once: inside it the activation is a constant
            auto rows = [&](auto act_tag) {
                constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
                for (int it2 = 0; it2 < IT / 2; ++it2) {
                    const int32_t row_out = odd ? out_row[2 * it2 + 1] : out_row[2 * it2];
                    if (r1 >= rows_here - row_base(mi, 2 * it2) || j >= half_n) continue;
                    const int64_t p = m_begin + r1 + row_base(mi, 2 * it2);
                    const u32x4_t up = ups[it2], gate = gates[it2];
                    if (P.aux) {
                        T* h = reinterpret_cast<T*>(P.aux) + p * P.ld_aux;
                        __builtin_nontemporal_store(up, reinterpret_cast<u32x4_t*>(h + j));
                        __builtin_nontemporal_store(gate, reinterpret_cast<u32x4_t*>(h + half_n + j));
                    }
                    float u[PV], g[PV], o[PV];
                    Elem<T>::unpack(to_uint4(up), u);
                    Elem<T>::unpack(to_uint4(gate), g);
#pragma unroll
                    for (int q = 0; q < PV; ++q) o[q] = gated_forward<true>(ACT, u[q], g[q]);
                    { const uint4 pk = Elem<T>::pack(o); __builtin_nontemporal_store(u32x4_t{pk.x, pk.y, pk.z, pk.w}, reinterpret_cast<u32x4_t*>(C + (int64_t)row_out * P.ldc + j)); }
                }
            };
            if (P.act == ACT_SWIGLU) rows(std::integral_constant<int, ACT_SWIGLU>{});
            else rows(std::integral_constant<int, ACT_GLU>{});
        } else {  // EPI_BACKWARD
            const int64_t n = n0 + cc * PV;
            if constexpr (mi + 1 < OUT_SLABS) load_saved(mi + 1, hu[(mi + 1) & 1], hg[(mi + 1) & 1]);
            u32x4_t dv[IT];
            read_own_chunks(dv);
            auto rows = [&](auto act_tag) {
                constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
                for (int it = 0; it < IT; ++it) {
                    if (!row_exists(mi, it) || n >= P.n) continue;
                    float u[PV], g[PV], d[PV], du[PV], dg[PV];
                    Elem<T>::unpack(to_uint4(hu[mi & 1][it]), u);
                    Elem<T>::unpack(to_uint4(hg[mi & 1][it]), g);
                    Elem<T>::unpack(to_uint4(dv[it]), d);
                    T* out = C + (int64_t)out_row[it] * P.ldc;
                    if constexpr (ACT == ACT_GELU_TANH) {
#pragma unroll
                        for (int q = 0; q < PV; ++q) du[q] = gelu_tanh_backward<true>(u[q], d[q]);
                        *reinterpret_cast<uint4*>(out + n) = Elem<T>::pack(du);
                    } else {
#pragma unroll
                        for (int q = 0; q < PV; ++q) gated_backward<true>(ACT, u[q], g[q], d[q], du[q], dg[q]);
                        { const uint4 a = Elem<T>::pack(du), b = Elem<T>::pack(dg); __builtin_nontemporal_store(u32x4_t{a.x, a.y, a.z, a.w}, reinterpret_cast<u32x4_t*>(out + n)); __builtin_nontemporal_store(u32x4_t{b.x, b.y, b.z, b.w}, reinterpret_cast<u32x4_t*>(out + P.n + n)); }
                    }
                }
            };
            if (P.act == ACT_SWIGLU) rows(std::integral_constant<int, ACT_SWIGLU>{});
            else if (P.act == ACT_GLU) rows(std::integral_constant<int, ACT_GLU>{});
            else rows(std::integral_constant<int, ACT_GELU_TANH>{});
        }
    };
    store_rows(TL::template slab<0>(), std::integral_constant<int, 0>{}, orow[0]);
    if constexpr (OUT_SLABS >= 2) store_rows(TL::template slab<1>(), std::integral_constant<int, 1>{}, orow[1]);
    if constexpr (OUT_SLABS >= 3) store_rows(TL::template slab<2>(), std::integral_constant<int, 2>{}, orow[2]);
    if constexpr (OUT_SLABS >= 4) store_rows(TL::template slab<3>(), std::integral_constant<int, 3>{}, orow[3]);
}

template <typename T, int KIND, int EPI, int BM, int BN, bool GATHER = false>
__global__ __launch_bounds__(THREADS, groups_per_cu(BN)) void grouped_gemm_dma_kernel(const GemmParams P) {
    TilePlace place;
    place.i0 = 0;
    place.work.parts = 1;
    if constexpr (KIND == XMA_GEMM_MT) {
        int row_tile, col_tile;
        if (!locate_tile<true>(P.row_tiles_max * P.num_experts, P.col_tiles, row_tile, col_tile)) return;
        const int slot = row_tile / P.row_tiles_max;
        place.i0 = (int64_t)(row_tile % P.row_tiles_max) * BM;
        if (P.expert_order != nullptr) {  // experts in descending order of their row counts
            const int32_t* record = P.expert_order + 4 * slot;
            place.expert = record[0];
            place.m_begin = record[1];
            place.m_end = record[2];
        } else {
            place.expert = slot;
            place.m_begin = P.offsets[slot];
            place.m_end = P.offsets[slot + 1];
        }
        place.n0 = (int64_t)col_tile * BN;
    } else {
        // the row tiles present and this one's rows: from the table, or from the offsets when there is none
        const bool table = P.tile_count != nullptr;
        const RowTileScan tiles(P.offsets, table ? 0 : P.num_experts, P.tile_rows, threadIdx.x & 63);
        const int most_parts = (int)((P.k + 63) / 64 / kSplitMinStages);
        TileWork& work = place.work;
        const int row_tiles = table ? P.tile_count[0] : tiles.total;
        if (BN == 128 && most_parts < 2 && deal_row_tiles(row_tiles)) {
            if (!locate_tile<true, kDealtBand>(row_tiles, P.col_tiles, work.row_tile, work.col_tile)) return;
        } else if (!locate_work<BN == 256 && KIND == XMA_GEMM_NN>(row_tiles, P.col_tiles, P.round_tiles, most_parts < kMaxSplit ? most_parts : kMaxSplit,
                                kSplitMaxRounds, kSplitSlots, work)) {
            return;
        }
        int32_t row0, row_end;
        if (table) {
            place.expert = P.tile_expert[work.row_tile];
            row0 = P.tile_row0[work.row_tile];
            const int32_t last = P.offsets[place.expert + 1];
            row_end = last - row0 > P.tile_rows ? row0 + P.tile_rows : last;
        } else {
            tiles.find(work.row_tile, place.expert, row0, row_end);
        }
        place.m_begin = row0;
        place.m_end = row_end;
        place.n0 = (int64_t)work.col_tile * (EPI == EPI_PAIRED ? BN / 2 : BN);
    }
    if constexpr (KIND == XMA_GEMM_MT) {
        multiply_tile<T, KIND, EPI, Ring64x5<Tile<BM, BN>>, GATHER>(P, place);
    } else if constexpr (BN == 256 && KIND == XMA_GEMM_NN) {
        // Flat tiles: halves of the tiles of a last round, and an expert's last rows.  (The forward kinds gain nothing from them
        // on balance, see phase().)
        if (place.work.halves > 1) {
            place.m_begin += 128 * place.work.half;
            if (place.m_begin >= place.m_end) return;
            place.m_end = place.m_end - place.m_begin > 128 ? place.m_begin + 128 : place.m_end;
        }
        if (place.m_end - place.m_begin <= 128) multiply_tile<T, KIND, EPI, Ring64x5<Tile<128, BN>>>(P, place);
        else multiply_tile<T, KIND, EPI, Ring64x5<Tile<BM, BN>>>(P, place);
    } else if constexpr (BN == 256) {
        multiply_tile<T, KIND, EPI, Ring64x5<Tile<BM, BN>>>(P, place);
    } else {
        const int64_t rows = place.m_end - place.m_begin;
        if (rows > 128) multiply_tile<T, KIND, EPI, Ring64x2<Tile<BM, BN>>>(P, place);
        else if (rows > 64) multiply_tile<T, KIND, EPI, Ring64x2<Tile<128, BN>>>(P, place);
        else if (rows > 32) multiply_tile<T, KIND, EPI, Ring64x2<Tile<64, BN>>>(P, place);
        else multiply_tile<T, KIND, EPI, Ring64x2<Tile<32, BN>>>(P, place);
    }
}

static __global__ __launch_bounds__(1024) void build_expert_order_kernel(const int32_t* __restrict__ offsets, int E,
                                                                         int32_t* __restrict__ records) {
    __shared__ int32_t count[kMaxOrderedExperts];
    if (E > kMaxOrderedExperts) {
        for (int e = threadIdx.x; e < E; e += blockDim.x) {
            records[4 * e] = e;
            records[4 * e + 1] = offsets[e];
            records[4 * e + 2] = offsets[e + 1];
            records[4 * e + 3] = 0;
        }
        return;
    }
    const int e = threadIdx.x;
    int32_t begin = 0, end = 0;
    if (e < E) {
        begin = offsets[e];
        end = offsets[e + 1];
        count[e] = end - begin;
    }
    __syncthreads();
    if (e < E) {
        const int32_t mine = end - begin;
        int slot = 0;
        for (int o = 0; o < E; ++o) slot += (count[o] > mine || (count[o] == mine && o < e)) ? 1 : 0;
        records[4 * slot] = e;
        records[4 * slot + 1] = begin;
        records[4 * slot + 2] = end;
        records[4 * slot + 3] = 0;
    }
}

template <typename T, int KIND, int EPI, int BM, int BN, bool GATHER = false>
static int launch(const xma_grouped_gemm_args& a, int tile_rows, hipStream_t stream, const uint32_t* row_offsets = nullptr) {
    GemmParams P;
    fill_params(a, P);
    P.tile_rows = tile_rows;
    P.row_offsets = row_offsets;
    int64_t grid;
    if (KIND == XMA_GEMM_MT) {
        P.row_tiles_max = (int32_t)ceil_div(a.n, BM);
        P.col_tiles = (int32_t)ceil_div(a.k, BN);
        grid = grid_for_tiles((int64_t)P.row_tiles_max * a.num_experts, P.col_tiles);
        if (a.workspace != nullptr) {  // size checked by the caller
            int32_t* records = reinterpret_cast<int32_t*>(a.workspace);
            hipLaunchKernelGGL(build_expert_order_kernel, dim3(1), dim3(1024), 0, stream, a.expert_offsets,
                               a.num_experts, records);
            P.expert_order = records;
        }
    } else {
        const int64_t rt = max_row_tiles(a.rows, a.num_experts, tile_rows);
        P.row_tiles_max = (int32_t)rt;
        place_split_region(a, P);
        P.round_tiles = compute_units() * groups_per_cu(BN);
        const int bn_out = EPI == EPI_PAIRED ? BN / 2 : BN;
        const int64_t n_out = EPI == EPI_PAIRED ? a.n / 2 : a.n;
        P.col_tiles = (int32_t)ceil_div(n_out, bn_out);
        grid = grid_for_work(rt * P.col_tiles, P.round_tiles);
        if (BN == 128 && !may_split(a.k)) {
            const int64_t dealt = grid_for_dealt_tiles(rt, P.col_tiles);
            grid = grid > dealt ? grid : dealt;
        }
        if (a.num_experts > kMaxScannedExperts) {
            launch_build_row_tiles(a, tile_rows, rt, P, stream);
        } else if (may_split(a.k)) {
            launch_clear_split_counters(P, stream);
        }
    }
    XMA_REQUIRE(grid < ((int64_t)1 << 31), "xma_grouped_gemm: %lld tiles exceed the grid limit", (long long)grid);
    hipLaunchKernelGGL((grouped_gemm_dma_kernel<T, KIND, EPI, BM, BN, GATHER>), dim3((unsigned)grid), dim3(THREADS), 0, stream, P);
    return check_launch("xma_grouped_gemm");
}

template <typename T, int BM, int BN>
static int dispatch(const xma_grouped_gemm_args& a, int tile_rows, hipStream_t stream) {
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    switch (a.kind) {
        case XMA_GEMM_TN:
            if (shape == EPI_PAIRED) return launch<T, XMA_GEMM_TN, EPI_PAIRED, BM, BN>(a, tile_rows, stream);
            return launch<T, XMA_GEMM_TN, EPI_PLAIN, BM, BN>(a, tile_rows, stream);
        case XMA_GEMM_NN:
            if (shape == EPI_BACKWARD) return launch<T, XMA_GEMM_NN, EPI_BACKWARD, BM, BN>(a, tile_rows, stream);
            return launch<T, XMA_GEMM_NN, EPI_PLAIN, BM, BN>(a, tile_rows, stream);
        default:
            return launch<T, XMA_GEMM_MT, EPI_PLAIN, BN, BN>(a, tile_rows, stream);
    }
}

}  // namespace dma

// Token rows of the up-projection's weight gradient, read where they are instead of from a grouped copy.  us, copy + kernel /
// kernel that gathers: fine-grained layer (16384 tokens, H 2048, 64 experts, 6 each) 88 + 705 / 775, skewed (128 experts, 8
// each) 111 + 765 / 825, Mixtral-shaped (8192 tokens, H 4096) 42 + 3160 / 3160; and a buffer of the routed rows less.  The loop
// has the same instructions but for four vector ones a load; at the fine-grained sizes it waits longer for its rows.
template <typename T>
static int launch_gathered(const xma_grouped_gemm_args& a, const uint32_t* row_offsets, hipStream_t stream) {
    const DmaTile tile = dma_gemm_tile(a);
    return tile.cols == 256 ? dma::launch<T, XMA_GEMM_MT, EPI_PLAIN, 256, 256, true>(a, tile.rows, stream, row_offsets)
                            : dma::launch<T, XMA_GEMM_MT, EPI_PLAIN, 128, 128, true>(a, tile.rows, stream, row_offsets);
}

int launch_gathered_weight_gradient(const xma_grouped_gemm_args& a, const uint32_t* row_offsets, hipStream_t stream) {
    return a.dtype == XMA_BF16 ? launch_gathered<bf16_t>(a, row_offsets, stream)
                               : launch_gathered<f16_t>(a, row_offsets, stream);
}

// 16-bit element types; the weight-gradient layout only without a row index.  (Rows that are looked up take a table of byte
// offsets and sizes that fit it: launch_gathered_weight_gradient, which a layer's native backward pass calls.)
bool dma_gemm_supports(const xma_grouped_gemm_args& a) {
    if (a.dtype != XMA_BF16 && a.dtype != XMA_F16) return false;
    if (a.kind == XMA_GEMM_MT && a.in_index != nullptr) return false;
    return true;
}

// ---- which tile a call takes ----------------------------------------------------------------------------------------
//
// 256 x 256 tiles have a compute unit each: the fewest bytes of operands per operation, but nothing overlaps what a tile
// does outside its main loop, an expert's last rows cost a whole tile, and a launch with few tiles leaves compute units
// idle.  Tiles of up to 192 x 128 run two on a compute unit, so that one's set-up and stores run under the other's main
// loop, and an expert's last rows take a tile of 32, 64, 128 or 192 rows; per operation they ask the L2 for two thirds more.
//
// Row-grouped kinds: the cost of each form is estimated from the tiles that experts have whose numbers of rows spread as
// randomly chosen ones do, and two per cent more, in rounds of the device (K: the reduction in units of 1024):
//   256 x 256: 20 + 24 K a round (34 where the epilogue has an activation of two halves or its backward); a partly filled last
//     round costs a whole one, or is split along the reduction for 40 more;
//   192, 128, 64, 32 x 128, two per compute unit: 7 (10) + 33, 24, 20, 24 K, 1.45 times that where rows do not start at whole
//     lines of 128 bytes; a last round of half the places or less two thirds of a whole one.
// These are not times: small tiles take about 0.75 of it, and a remainder of 32 rows costs its neighbour more than itself.  They
// are the constants whose choice cost least over 10302 calls (1 to 256 experts, 20 to 20000 rows each, 12 layers) timed in all
// three forms: 1.2 % more than the fastest on average where rows are spread evenly, 4 % under a skewed routing.  95 % of the
// former are within 3 % of 256 x 256 everywhere or faster, on average they take 0.74 of its time.  The worst are experts whose
// rows lie just above a multiple of 192 or 256, which a few rows more or less decide.
// us, 256 x 256 / up to 192 / up to 128 rows, evenly spread unless said otherwise:
//   64 experts, H 2048, I 1024: 1536 rows each, up 784 / 857 / 902, dX 755 / 819 / 858; 281, 228 / 205 / 244 and 217 / 186 / 228;
//     75, 143 / 133 / 132 and 114 / 110 / 112
//   128 experts, H 2048, I 768, 96 rows, skewed: up 107 / 102 / 99, down 71 / 58 / 57, dX 127 / 106 / 104
//   6 experts, H 512, I 1024, 2000 rows: up 49 / 42 / 37, down 28 / 23 / 20, dact 41 / 38 / 34, dX 48 / 38 / 30
//   16 experts, H 1024, I 4096, 125 rows: up 68 / 60 / 71, down 61 / 40 / 43, dX 98 / 83 / 91
//   8 experts, H 4096, I 14336, 2048 rows: up 3082 / 3832 / 4256, down 1427 / 1876 / 2146
//   one round of 256 x 256, two of the others: 4 experts, H 4096, I 14336, 187 rows, up 231 / 362 / 306, dact 119 / 185 / 162; 8
//     experts, H 6144, I 2048, 200 rows, down 48 / 74 / 54
//   rows of 1040 and 15056 bytes: 32 experts, H 520, I 7528, 200 rows, down 140 / 235 / 191, up 299 / 391 / 339
//
// Weight gradients: tiles of 128 x 128 where 256 x 256 leave much of the device idle, or where the reductions (the rows of an
// expert) are short.  us, 256 x 256 / 128 x 128 (one launch back to back with itself, evenly spread rows):
//   one round of large tiles, 16 experts, 1024 x 1024: 500 rows 26 / 28, 1000 37 / 39, 2000 59 / 65, 4000 101 / 124, 8000
//     199 / 267; 8 experts, 2048 x 1024, 16000 rows 375 / 542
//   a second round of three quarters, 8 experts, 2048 x 1792: 2000 rows 100 / 110, 4000 175 / 204, 16000 696 / 1050
//   fewer than four bands of row tiles, which leave half the XCDs without work: 4 experts, 768 x 3072: 1500 rows 73 / 43, 4000
//     165 / 102, 9000 353 / 229; 6 experts, 2048 x 1024, 9000 rows, skewed (an expert's tiles are one band): 411 / 275
//   two rounds and more: 64 experts, 2048 x 1024, 281 rows 133 / 125, 375 149 / 147; 64 experts, 2048 x 2048, 281 253 / 241, 375
//     284 / 286, 562 346 / 392; 128 experts, 1536 x 2048, 375 444 / 500
// Long launches of many tiles turn earlier: with 4096 tiles 1.05 times as long in small ones at 390 rows, with 8192 at 300, with
// 16384 at 220, hence rows^2 * tiles.  Over 4310 calls of 1 to 256 experts, 20 to 20000 evenly spread rows each, the choice costs
// 0.8 % more than the faster of the two on average, and is within 3 % of 256 x 256 or faster in 97 %.  Under a skewed routing
// small tiles win for longer (one expert's reductions bound the launch), which the host cannot see.
namespace {

constexpr int kSpreadPoints = 5;
// the i-th of a few numbers of rows that stand for those of the experts
int64_t rows_at(double mean, int i) {
    constexpr double kDeviations[kSpreadPoints] = {-1.4, -0.7, 0, 0.7, 1.4};
    const double rows = mean + kDeviations[i] * sqrt(mean + 4e-4 * mean * mean);
    return rows < 0 ? 0 : (int64_t)(rows + 0.5);
}

constexpr int kHeights = 4;
constexpr int kSmallRows[kHeights] = {32, 64, 128, 192};
constexpr double kSmallLoop[kHeights] = {24, 20, 24, 33};
int height_for(int64_t rows) {
    int i = 0;
    while (i < kHeights - 1 && rows > kSmallRows[i]) ++i;
    return i;
}

double estimate_256(double rows, int64_t experts, int64_t col_tiles, double k1024, int shape) {
    double tiles = 0;
    for (int i = 0; i < kSpreadPoints; ++i) tiles += (double)ceil_div(rows_at(rows, i), 256) / kSpreadPoints;
    const double set_up = shape == EPI_PLAIN ? 20 : 34, loop = 24 * k1024;
    const double rounds = tiles * (double)experts * (double)col_tiles / 256;
    const int64_t full = (int64_t)(rounds + 1e-6);
    const double rest = rounds - (double)full;
    if (full > 0 && rest < 1e-5) return full * (set_up + loop);
    int parts = 1;
    if (rounds < kSplitMaxRounds) {
        parts = rest * kMaxSplit < 1 ? kMaxSplit : (int)(1 / rest);
        if (parts > k1024 * 16 / kSplitMinStages) parts = (int)(k1024 * 16 / kSplitMinStages);
    }
    return full * (set_up + loop) + set_up + (parts > 1 ? loop / parts + 40 : loop);
}

double estimate_small(double rows, int64_t experts, int64_t col_tiles, double k1024, int shape, bool whole_lines, int tallest) {
    double count[kHeights] = {};
    for (int i = 0; i < kSpreadPoints; ++i) {
        const int64_t r = rows_at(rows, i);
        count[tallest] += (double)(r / kSmallRows[tallest]) / kSpreadPoints;
        if (r % kSmallRows[tallest] > 0) count[height_for(r % kSmallRows[tallest])] += 1.0 / kSpreadPoints;
    }
    double tiles = 0, work = 0, longest = 0;
    for (int h = 0; h < kHeights; ++h) {
        const double cost = ((shape == EPI_PLAIN ? 7 : 10) + kSmallLoop[h] * k1024) * (whole_lines ? 1 : 1.45);
        tiles += count[h];
        work += count[h] * cost;
        if (count[h] > 0) longest = cost;
    }
    if (tiles == 0) return 0;
    const double mean = work / tiles;
    constexpr double kHalfRound = 0.66;
    tiles *= (double)experts * (double)col_tiles;
    if (tiles <= 256) {  // fewer than one per compute unit, or split along the reduction
        double parts = (int)(512 / (tiles < 1 ? 1 : tiles));
        if (parts > kMaxSplit) parts = kMaxSplit;
        if (parts > k1024 * 16 / kSplitMinStages) parts = (int)(k1024 * 16 / kSplitMinStages);
        if (parts < 2) parts = 1;
        return (tiles * parts > 256 ? 1 : kHalfRound) * longest / parts;
    }
    const double rounds = tiles / 512;
    const int64_t full = (int64_t)(rounds + 1e-6);
    const double rest = rounds - (double)full;
    if (rest < 1e-5) return full * mean;
    const double part = rest <= 0.5 ? kHalfRound : 1;
    if (full == 0) return part * longest;
    const double mixed = part * mean + 0.5 * (longest - mean);
    return full * mean + (mixed < part * longest ? mixed : part * longest);
}

// Tiles of the XCD that has most of them: bands of kBandTiles row tiles are dealt in turn (locate_tile<true>).
int64_t busiest_xcd(int64_t row_tiles, int64_t col_tiles) {
    const int64_t bands = ceil_div(ceil_div(row_tiles, kBandTiles), kNumXcd);
    return (row_tiles < kBandTiles ? row_tiles : bands * kBandTiles) * col_tiles;
}

// Rounds of `places` tiles, the last of which takes `part` of a whole one, and more the fuller it is.
double rounds_of(int64_t tiles, int places, double part) {
    const int64_t full = tiles / places;
    const double rest = (double)(tiles % places) / places;
    const double rounds = rest > 0 ? (double)full + part + (1 - part) * rest : (double)full;
    return rounds < 1 ? 1 : rounds;
}

bool small_weight_gradient_tiles(const xma_grouped_gemm_args& a, double rows) {
    const double tiles = (double)a.num_experts * ceil_div(a.n, 256) * ceil_div(a.k, 256);
    if (tiles >= 512) return rows < 330 && rows * rows * tiles < 5e8;
    // 32 compute units of an XCD, two places each for small tiles; us of a round, least squares over the calls of few tiles
    const int64_t large = busiest_xcd(a.num_experts * ceil_div(a.n, 256), ceil_div(a.k, 256));
    const int64_t small = busiest_xcd(a.num_experts * ceil_div(a.n, 128), ceil_div(a.k, 128));
    const double x = rows / 1024;
    const double time_large = rounds_of(large, 32, 0.8) * (14.4 + 24 * x);
    const double time_small = rounds_of(small, 64, 0.7) * (6.6 + 13.6 * x * (1 + 0.1 * log2(1 + x)));
    // (with at most one large tile per compute unit a skewed call takes up to twice as long in large tiles; an even one loses a
    // seventh at most to the other mistake)
    return time_small < (large <= 32 ? 1.2 : 1.03) * time_large;
}

}  // namespace

DmaTile dma_gemm_tile(const xma_grouped_gemm_args& a) {
    const double rows = (double)a.rows / a.num_experts;
    if (a.kind == XMA_GEMM_MT) return small_weight_gradient_tiles(a, rows) ? DmaTile{128, 128} : DmaTile{256, 256};
    int shape = EPI_PLAIN, act = ACT_NONE;
    split_epilogue(a.epilogue, shape, act);
    const double k1024 = (double)a.k / 1024;
    const bool whole_lines = a.n % 64 == 0 && a.k % 64 == 0;
    auto estimate = [&](int tallest) {
        return estimate_small(rows, a.num_experts, ceil_div(a.n, 128), k1024, shape, whole_lines, tallest);
    };
    const double big = estimate_256(rows, a.num_experts, ceil_div(a.n, 256), k1024, shape);
    const double tall = estimate(kHeights - 1), flat = estimate(kHeights - 2);
    if (big < tall && big < flat) return DmaTile{256, 256};
    return tall <= flat ? DmaTile{192, 128} : DmaTile{128, 128};
}

template <typename T>
static int launch_tiles(const xma_grouped_gemm_args& a, hipStream_t stream) {
    const DmaTile tile = dma_gemm_tile(a);
    return tile.cols == 256 ? dma::dispatch<T, 256, 256>(a, tile.rows, stream)
                            : dma::dispatch<T, 192, 128>(a, tile.rows, stream);
}

int launch_dma_gemm(const xma_grouped_gemm_args& a, hipStream_t stream) {
    return a.dtype == XMA_BF16 ? launch_tiles<bf16_t>(a, stream) : launch_tiles<f16_t>(a, stream);
}

}  // namespace xma
