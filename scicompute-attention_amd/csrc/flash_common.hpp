// Shared pieces of the flash prefill kernels (flash_reg.hip, flash_pair.hip, flash_wide.hpp) and of
// their dispatch (flash_fwd.hip): MFMA wrappers, the workgroup order, the LDS-DMA pipeline's
// helpers, the online-softmax row state, the tile geometries and the launchers' declarations.
//
// Formulation (every kernel): S^T = K Q^T with v_mfma_f32_32x32x16_{f16,bf16} (A = K rows from LDS,
// B = Q^T in registers for the whole tile). In the S^T accumulator every lane holds 16 keys of ONE
// query row, so the row max/sum need a single exchange between the two 32-lane halves and the
// online-softmax state (m, l) is one register per lane. The P^T accumulator, converted to
// fp16/bf16, is directly the B operand of O^T = V^T P^T (the key order inside an MFMA k-step
// matches the accumulator layout), so P never leaves registers. The O rescale is lazy (only when
// the running max grows by more than kRescaleSlack, decided per wave).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "sca_device.hpp"

namespace sca_hip {

constexpr int kRowsPerWave = 32;
constexpr int kRowGroups = 4;
constexpr int kBlockM = kRowGroups * kRowsPerWave;  // 128 query rows per workgroup
constexpr int kKPad = 8;        // K rows padded by 16 B
constexpr int kVPad = 4;        // V^T rows padded by 8 B
constexpr float kRescaleSlack = 8.0f;  // log2 units the running max may lag behind

// Geometry per head_dim. Every wave owns 32 query rows and 32 keys of each KV tile:
// KSPLIT waves share a row group and split the tile's keys between them (their softmax states
// are merged once at the end), so a SIMD holds KSPLIT waves whose MFMA and VALU phases overlap.
template <int D>
struct FlashGeom {
    static constexpr int KSPLIT = D <= 128 ? 2 : 1;
    static constexpr int WAVES = kRowGroups * KSPLIT;
    static constexpr int THREADS = WAVES * kWave;
    static constexpr int BN = 32 * KSPLIT;               // keys per tile
    static constexpr int STAGES = 3;                     // LDS ring depth
    static constexpr int KS = D / 16;                    // QK k-steps
    static constexpr int DT = D / 32;                    // 32-row tiles of O^T
    static constexpr int KSTR = D + kKPad;               // K row stride (elements)
    static constexpr int VSTR = BN + kVPad;              // V^T row stride (elements)
    static constexpr int K_CHUNKS = BN * D / 8;          // 16 B chunks per K tile
    static constexpr int K_PER_THREAD = (K_CHUNKS + THREADS - 1) / THREADS;
    static constexpr int V_UNITS = (BN / 4) * (D / 8);   // 4 keys x 8 dims per unit
    static constexpr int V_PER_THREAD = (V_UNITS + THREADS - 1) / THREADS;
    static constexpr int K_STAGE = BN * KSTR;
    static constexpr int V_STAGE = D * VSTR;
    static constexpr int STAGE_BYTES = STAGES * (K_STAGE + V_STAGE) * 2;
    static constexpr int MERGE_FLOATS = DT * 16 + 2;     // per lane: O^T + m + l
    static constexpr int MERGE_BYTES = KSPLIT > 1 ? kRowGroups * kWave * MERGE_FLOATS * 4 : 0;
    static constexpr int LDS_BYTES = STAGE_BYTES > MERGE_BYTES ? STAGE_BYTES : MERGE_BYTES;
};

// ---- Two-group causal pair kernel ---------------------------------------------------------------
// Small causal grids: each workgroup owns the complementary 64-row tiles A = T-1-t (long) and
// B = t (short) and runs them concurrently in two groups of four waves (one wave of each group
// per SIMD), each group with its own K/V ring. Group 0 takes A's key tiles [0, x); group 1
// takes all of B, finishes B (a two-way merge and the stores), then takes A's key tiles
// [x, n_A). The two groups' A states are merged once at the end, so the short tile's setup,
// merge and stores run beside the long tile's key loop instead of after it. x balances the
// two groups' barrier intervals.
// Within a group: 2 row groups of 32 rows x 2 waves of 32 keys per 64-key tile; the pipeline
// step j computes QK of tile j+1 under the softmax of tile j, then PV of tile j.
template <int D>
struct PairGeom {
    static constexpr int GW = 4;                      // waves per group
    static constexpr int THREADS = 2 * GW * kWave;
    static constexpr int BM = 64;                     // rows per row tile
    static constexpr int BN = 64;                     // keys per key tile
    static constexpr int KS = D / 16;
    static constexpr int DT = D / 32;
    static constexpr int CPR = D / 8;
    static constexpr int ROW_BYTES = D * 2;
    static constexpr int TILE_BYTES = BN * D * 2;
    static constexpr int IPW = BN * CPR / (kWave * GW);  // DMA instructions per wave per tile
    static constexpr int RING_BYTES = 4 * TILE_BYTES;    // K slots 0, 1, then V slots 0, 1
    // Final merge: per row group, three partial states (16-byte quads) and their (m, l).
    static constexpr int MERGE_QUADS = 2 * 3 * 4 * DT * kWave;
    static constexpr int MERGE_BYTES = MERGE_QUADS * 16 + 2 * 3 * kWave * 8;
    static constexpr int LDS_BYTES = 2 * RING_BYTES > MERGE_BYTES ? 2 * RING_BYTES : MERGE_BYTES;
    static_assert(IPW >= 1 && BN * CPR == IPW * kWave * GW, "tile must split evenly into DMAs");
    static_assert(2 * 4 * DT * kWave * 16 + 2 * kWave * 8 <= RING_BYTES,
                  "the B merge fits group 1's ring");
    static_assert(TILE_BYTES < 65536, "slot offsets are DS immediates");
};

template <int D>
struct WideGeom {
    static constexpr int WAVES = 4;
    static constexpr int THREADS = WAVES * kWave;
    static constexpr int RT = 2;                      // 32-row subtiles per wave
    static constexpr int BM = 128;                    // rows per workgroup
    static constexpr int BN = 64;                     // keys per tile
    static constexpr int KS = D / 16;                 // QK k-steps
    static constexpr int DT = D / 32;                 // O^T tiles of 32 dims
    static constexpr int CPR = D / 8;                 // 16-byte chunks per row
    static constexpr int ROW_BYTES = 2 * D;
    static constexpr int TILE_BYTES = BN * ROW_BYTES;
    static constexpr int IPW = BN * CPR / (kWave * WAVES);  // DMA instructions per wave per tile
    static constexpr int SLOTS = 4;
    static constexpr int V_BASE = SLOTS * TILE_BYTES;
    static constexpr int RING_BYTES = 2 * SLOTS * TILE_BYTES;
    // Merge: every wave hands one subtile's O (DT*16 floats per lane), m and up to two denominators to
    // its partner.
    static constexpr int MERGE_FLOATS = DT * 16 + 3;
    static constexpr int MERGE_BYTES = WAVES * kWave * MERGE_FLOATS * 4;
    static constexpr int LDS_BYTES = RING_BYTES > MERGE_BYTES ? RING_BYTES : MERGE_BYTES;
    static_assert(IPW >= 1 && BN * CPR == IPW * kWave * WAVES, "tile must split evenly");
    // V reads of the two upper slots go through a second address (slot offsets are DS immediates
    // below 64 KB).
    static constexpr bool V_SPLIT = (SLOTS - 1) * TILE_BYTES + 25 * ROW_BYTES > 65536;
    static_assert((SLOTS - 1) * TILE_BYTES + ROW_BYTES <= 65536 && TILE_BYTES + 25 * ROW_BYTES <= 65536,
                  "slot offsets are DS immediates");
};

template <int D>
struct DsplitGeom {
    static constexpr int WAVES = 4;
    static constexpr int THREADS = WAVES * kWave;
    static constexpr int BM = 128;                    // rows per workgroup
    static constexpr int BN = 32;                     // keys per tile
    static constexpr int KS = D / 16;                 // QK k-steps
    static constexpr int DT = D / 64;                 // O^T tiles of 32 dims per wave (half of D)
    static constexpr int CPR = D / 8;                 // 16-byte chunks per row
    static constexpr int ROW_BYTES = 2 * D;
    static constexpr int TILE_BYTES = BN * ROW_BYTES;
    static constexpr int IPW = BN * CPR / (kWave * WAVES);  // DMA instructions per wave per tile
    static constexpr int SLOTS = 4;
    static constexpr int V_BASE = SLOTS * TILE_BYTES;
    static constexpr int P_BASE = 2 * V_BASE;            // 2 parities x 4 waves x 2 KB
    static constexpr int ALPHA_BASE = P_BASE + 16384;    // 2 parities x 4 waves x 32 floats
    static constexpr int FLAG_BASE = ALPHA_BASE + 1024;  // 2 parities x 4 ints
    static constexpr int LDS_BYTES = FLAG_BASE + 32;
    static_assert(D % 64 == 0 && BN * CPR == IPW * kWave * WAVES, "tile must split evenly");
    static_assert((SLOTS - 1) * TILE_BYTES + 25 * ROW_BYTES <= 65536, "slot offsets are DS immediates");
};

// Packed variable-length launch: cumulative token offsets and the work list (2 int32 per row
// tile: sequence, tile), device-resident.
struct VarlenArgs {
    const int32_t* cu_q;
    const int32_t* cu_kv;
    const int32_t* tiles;
};

// How the rows and keys of a launch are cut (wide and split-dims kernels).
//   pack   query heads of one KV head whose rows share row tiles (1, or the whole GQA group): packed
//          row R is query R / pack of head R % pack of the group;
//   splits key ranges per row tile, each in a workgroup of its own. With more than one, workgroup
//          (tile, split) writes the unnormalised fp32 state of its rows - O, m (log2 units), l - to
//          part_o [split][row][D] and part_ml [split][row][2] (row = (b*H_q + h)*S_q + q), and
//          flash_combine_kernel merges them.
struct SplitArgs {
    int pack;
    int splits;
    float* part_o;
    float* part_ml;
};

// The key tiles [first, first + count) of `n_tiles` that split `split` of `splits` takes.
__device__ __forceinline__ void SplitRange(int n_tiles, int splits, int split, int* first, int* count) {
    const int chunk = (n_tiles + splits - 1) / splits;
    *first = split * chunk;
    *count = max(0, min(n_tiles - *first, chunk));
}

// Launchers, instantiated in the file of their kernel. Every one validates its grid and returns 0
// or a status.
template <typename E, int D, bool kCausal>
int LaunchFlashReg(const sca_flash_params& p, hipStream_t s);   // flash_reg.hip
template <typename E, int D>
int LaunchFlashPair(const sca_flash_params& p, hipStream_t s);  // flash_pair.hip (causal)
template <typename E, int D, bool kCausal>
int LaunchFlashWide(const sca_flash_params& p, const SplitArgs& sp, hipStream_t s);  // flash_wide.hpp
template <typename E, int D, bool kCausal>
int LaunchFlashDsplit(const sca_flash_params& p, const SplitArgs& sp, hipStream_t s);  // flash_dsplit.hip
template <typename E, int D, bool kCausal>
int LaunchFlashVarlen(const sca_flash_varlen_params& v, hipStream_t s);  // flash_wide.hpp

namespace {

template <typename E>
struct Mfma;

template <>
struct Mfma<F16> {
    typedef _Float16 pair_t __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ floatx16 mma(const half8& a, const half8& b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    // Two floats -> packed pair (round to nearest even), as the raw 32-bit word.
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, pair_t));
    }
    // acc + a.x + a.y in fp32 (v_dot2 with (1, 1)).
    static __device__ __forceinline__ float sum2(uint32_t w, float acc) {
        const pair_t ones = {static_cast<_Float16>(1.0f), static_cast<_Float16>(1.0f)};
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(pair_t, w), ones, acc, false);
    }
};

template <>
struct Mfma<BF16> {
    typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ floatx16 mma(const bf16x8& a, const bf16x8& b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, pair_t));
    }
    static __device__ __forceinline__ float sum2(uint32_t w, float acc) {
        const pair_t ones = {static_cast<__bf16>(1.0f), static_cast<__bf16>(1.0f)};
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(pair_t, w), ones, acc, false);
    }
};

// Workgroup -> (row tile index, batch*head). The dispatcher deals workgroups to the eight XCDs
// round robin (workgroup w on XCD w % 8), and each XCD has its own L2. When the (batch, KV head)
// groups divide by eight, XCD x takes groups x, x + 8, ...: the query heads that read one KV head
// run on one XCD and share its L2 (C3, 4 x 8 groups of 4 heads: +5%). Otherwise w runs row tile
// w / bh_count of head w % bh_count. Either way row tile t starts before t + 1 (so longest-first
// orders survive), and the mapping is a bijection on [0, tiles * bh_count).
// In 32 bits (the launchers bound the grid, and with it every factor, below 2^31): a 64-bit division
// takes about 130 instructions on this chip, and eight of them cost each workgroup 0.4 us.
// `heads` is the number of head units per batch entry: H_q, or H_kv when a unit packs a whole group.
__device__ __forceinline__ void XcdOrder(const sca_flash_params& p, uint32_t heads, int* tile_linear,
                                         int* b, int* h) {
    const uint32_t w = blockIdx.x;
    const uint32_t kv_heads = static_cast<uint32_t>(p.num_kv_heads);
    const uint32_t groups = static_cast<uint32_t>(p.batch) * kv_heads;
    const uint32_t gsz = heads / kv_heads;
    const uint32_t bh_count = groups * gsz;
    uint32_t bh;
    if (groups % 8 != 0) {
        *tile_linear = static_cast<int>(w / bh_count);
        bh = w % bh_count;
    } else {
        const uint32_t per_tile = bh_count / 8;  // workgroups of one row tile on one XCD
        const uint32_t pos = w / 8;
        const uint32_t rem = pos % per_tile;
        *tile_linear = static_cast<int>(pos / per_tile);
        bh = ((rem / gsz) * 8 + w % 8) * gsz + rem % gsz;
    }
    *b = static_cast<int>(bh / heads);
    *h = static_cast<int>(bh % heads);
}

// Scheduling-group masks of __builtin_amdgcn_sched_group_barrier.
constexpr int kSchedValu = 0x002;
constexpr int kSchedMfma = 0x008;
constexpr int kSchedDsRead = 0x100;


// ============================================================================================
// The DMA pipeline of the pair, wide and split-dims kernels.
//
// K and V tiles go straight from global memory to LDS with buffer loads to LDS (16 bytes per
// lane, no VGPR staging, no transposition) through a buffer resource bounded at the sequence's
// last row, so rows past seq_kv read as zero. Loads are issued ahead of their use and retired
// with explicit vmcnt waits plus one barrier per tile. LDS rows are unpadded; 16-byte chunks are
// XOR-swizzled per row (SwzK / SwzV) so that both the K reads and the V transpose reads are
// bank-conflict free. The PV A operand (V^T fragments) comes from ds_read_b64_tr_b16: within each
// 16-lane group, lane j receives element j % 4 of the 8 bytes read by lane 4*i + j/4 (i = 0..3),
// i.e. one head-dim column over 4 consecutive keys.
// ============================================================================================

// 16-byte-chunk swizzles for 64 LDS banks (a 256-byte bank window of 16 chunks). A row of D
// elements is D/8 chunks, so row r starts at chunk (D/8 * r) mod 16 of the window, and XOR with a
// value below the power of two that divides D/8 stays inside the row:
//   K: the 32 rows a wave reads in one ds_read_b128 land on 16 distinct 4-bank groups;
//   V: the 8 keys x 4 chunks of one transpose read land on 16 distinct groups.
// D/8 = 0 mod 16 (128, 256): every row starts at the same chunk, the swizzle does all the work;
// 8 mod 16 (64, 192): odd rows start half a window on; 4 or 12 mod 16 (32, 96, 160): four rows
// already cover the window, so V needs none.
template <int D>
__device__ __forceinline__ int SwzK(int row) {
    constexpr int kStart = (D / 8) % 16;
    static_assert(kStart % 4 == 0, "head_dim is a multiple of 32");
    return kStart == 0 ? (row & 15) : kStart == 8 ? ((row >> 1) & 7) : ((row >> 2) & 3);
}
template <int D>
__device__ __forceinline__ int SwzV(int row) {
    constexpr int kStart = (D / 8) % 16;
    return kStart == 0 ? ((row & 3) << 2) : kStart == 8 ? (((row >> 1) & 1) << 2) : 0;
}

// Fragment addresses: the swizzle permutes chunks only inside aligned groups, so the addresses of
// k-step ks and ks + KPeriod (and of O tile dt and dt + VPeriod) differ by a constant, which goes
// into the read's immediate offset.
template <int D>
constexpr int KPeriod() {
    constexpr int kStart = (D / 8) % 16;
    return kStart == 0 ? (D / 16 < 8 ? D / 16 : 8) : kStart == 8 ? 4 : 2;
}
template <int D>
constexpr int VPeriod() {
    constexpr int kStart = (D / 8) % 16;
    return kStart == 0 ? (D / 32 < 4 ? D / 32 : 4) : kStart == 8 ? 2 : 1;
}

// (lower-half value, upper-half value) of v for lanes l and l ^ 32, on every lane, from one
// v_permlane32_swap: it exchanges the upper 32 lanes of its first operand with the lower 32 lanes
// of its second, so with both operands holding v the first ends as (v_lo, v_lo) and the second as
// (v_hi, v_hi). Issued from inline asm with both registers as in/out operands (the builtin's
// second result is not reliably kept apart from the first), after the two wait states a VALU
// write needs before the permlane reads it.
__device__ __forceinline__ void HalfPair(float v, float* lo, float* hi) {
    uint32_t a = __builtin_bit_cast(uint32_t, v);
    uint32_t b = a;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    *lo = __builtin_bit_cast(float, a);
    *hi = __builtin_bit_cast(float, b);
}
__device__ __forceinline__ float HalfMax(float v) {
    float lo, hi;
    HalfPair(v, &lo, &hi);
    return fmaxf(lo, hi);
}
__device__ __forceinline__ float HalfSum(float v) {
    float lo, hi;
    HalfPair(v, &lo, &hi);
    return lo + hi;
}

// Stores one 32-dim O^T tile of a row (16 values per lane, two lanes per row: lane half hh holds dims
// 8g + 4hh + 0..3 of each group g) scaled by inv, as 16-byte chunks: the two halves of a row swap
// words so that hh = 0 holds all of groups 0 and 2 and hh = 1 all of 1 and 3. `dst` is the row's first
// dim of the tile (8-byte aligned); every lane of the wave takes part in the swap.
template <typename M>
__device__ __forceinline__ void StoreTile(uint16_t* dst, int hh, bool row_ok, const float (&v)[16]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
        uint32_t a0 = M::pack(v[4 * g], v[4 * g + 1]), a1 = M::pack(v[4 * g + 2], v[4 * g + 3]);
        uint32_t b0 = M::pack(v[4 * g + 4], v[4 * g + 5]), b1 = M::pack(v[4 * g + 6], v[4 * g + 7]);
        // (a, b) -> lower half: a of both halves; upper half: b of both (see HalfPair for the waits).
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1"
                     : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
        if (row_ok) *reinterpret_cast<u32x4*>(dst + 8 * (g + hh)) = u32x4{a0, a1, b0, b1};
    }
}

// The same tile unnormalised and in fp32, for a merge over key splits.
__device__ __forceinline__ void StorePartialTile(float* dst, int hh, bool row_ok, const float (&v)[16]) {
    if (!row_ok) return;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        *reinterpret_cast<float4*>(dst + 8 * g + 4 * hh) =
            make_float4(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
    }
}

// ---- Online softmax of one 32-key x 32-row S^T tile (lane: 16 keys of one row; lanes l and
// l ^ 32 hold the other 16 keys of the same row) -----------------------------------------------
// Per-lane row state: the running max used for the exponentials (m, log2 units), the raw-score
// threshold above which it must move (thr = (m + kRescaleSlack) / scale2), the exponent bias
// (-m, or 0 while no key of the row was visible) and this lane's share of the denominator.
struct RowState {
    float m;
    float thr;
    float neg_mu;
    float l;
};

__device__ __forceinline__ void ResetRow(RowState& r) {
    r.m = neg_inf();
    r.thr = neg_inf();
    r.neg_mu = 0.0f;
    r.l = 0.0f;
}

// What the softmax denominator sums. P is rounded to the input type for the PV product, so at head dims
// other than 64 and 128 the output is divided by the sum of the rounded weights: the rounding cancels
// (equal values give exactly that value), as in the register-staged kernel. The LSE is made of the
// unrounded sum, which those kernels add up only when it is asked for. At 64 and 128 one unrounded
// sum serves both. Against the unrounded sum for all (2 x 16 heads x 4096 causal): D 32 58.8 -> 55.5
// us, D 96 119.7 -> 121.7, D 160 177 -> 184, D 192 225 -> 218; with LSE, 16/8 heads, D 256 134.7 -> 136.4.
enum Denominator { kUnrounded, kRounded, kRoundedAndUnrounded };
template <int D>
constexpr Denominator DenominatorFor(bool lse) {
    return D == 64 || D == 128 ? kUnrounded : lse ? kRoundedAndUnrounded : kRounded;
}

// The VALU operations that turn a lane's 16 scores into P, as codes: 16 exponent arguments
// s * scale2 - m (0-15), 16 exponentials (16-31), 8 packs to the input type (32-39), 16 additions of
// the unrounded weights (40-55), 8 pair sums of the rounded ones (56-63). SoftmaxOp gives the n-th of
// the SoftmaxOps operations of a kernel, in an order that keeps each result at least two operations
// from its first use (one, for the last pair sum).
constexpr int SoftmaxOps(Denominator den) {
    return den == kUnrounded ? 56 : den == kRounded ? 48 : 64;
}
__host__ __device__ constexpr int SoftmaxOp(Denominator den, int n) {
    constexpr int kUn[56] = {0,  1,  2,  3,  16, 17, 4,  5,  18, 19, 6,  7,  20, 21,
                             32, 33, 8,  9,  22, 23, 34, 10, 11, 24, 25, 35, 40, 41,
                             12, 13, 26, 27, 36, 42, 43, 14, 15, 28, 29, 37, 44, 45,
                             30, 31, 46, 47, 38, 39, 48, 49, 50, 51, 52, 53, 54, 55};
    constexpr int kRo[48] = {0,  1,  2,  3,  16, 17, 4,  5,  18, 19, 6,  7,  20, 21, 32, 33,
                             8,  9,  22, 23, 34, 56, 10, 11, 24, 25, 35, 57, 12, 13, 26, 27,
                             36, 58, 14, 15, 28, 29, 37, 59, 30, 31, 38, 60, 39, 61, 62, 63};
    constexpr int kBo[64] = {0,  1,  2,  3,  16, 17, 4,  5,  18, 19, 6,  7,  20, 21, 32, 33,
                             8,  9,  22, 23, 34, 56, 10, 11, 24, 25, 35, 57, 40, 41, 12, 13,
                             26, 27, 36, 58, 42, 43, 14, 15, 28, 29, 37, 59, 44, 45, 30, 31,
                             60, 46, 47, 38, 39, 61, 48, 49, 50, 51, 62, 52, 53, 63, 54, 55};
    return den == kUnrounded ? kUn[n < 56 ? n : 0] : den == kRounded ? kRo[n < 48 ? n : 0] : kBo[n];
}

__device__ __forceinline__ float Max16(const floatx16& s) {
    const float a = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    const float b = fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7]));
    const float c = fmaxf(fmaxf(s[8], s[9]), fmaxf(s[10], s[11]));
    const float d = fmaxf(fmaxf(s[12], s[13]), fmaxf(s[14], s[15]));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// Transposed 8-byte LDS read at byte address addr + OFF. Issued from inline asm so that the
// compiler's conservative LDS-DMA tracking adds no wait for DMAs still in flight; the caller
// retires the reads with WaitLdsTied before the registers are used.
template <int OFF>
__device__ __forceinline__ uint2 TrReadAsm(uint32_t addr) {
    uint2 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
    return r;
}

// lgkmcnt(0), tied to the registers it guards so that no use of them is scheduled above it,
// and to the P operands (a, b) so that it is not hoisted above the exponentials either.
template <typename V, int N>
__device__ __forceinline__ void WaitLdsTied(V (&regs)[N], V& a, V& b) {
    if constexpr (N == 8) {
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(regs[0]), "+v"(regs[1]), "+v"(regs[2]), "+v"(regs[3]), "+v"(regs[4]),
                       "+v"(regs[5]), "+v"(regs[6]), "+v"(regs[7]), "+v"(a), "+v"(b));
    } else if constexpr (N == 4) {
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(regs[0]), "+v"(regs[1]), "+v"(regs[2]), "+v"(regs[3]), "+v"(a),
                       "+v"(b));
    } else {
        static_assert(N == 8 || N == 4, "tied wait covers 4 or 8 registers");
    }
}

__device__ __forceinline__ uint32_t LdsAddr(const void* p) {
    return static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t*)(p)));
}

// V^T fragments of one key tile for the PV MFMAs: for O tile dt, k-step ps, the transposed
// reads at rows 16*ps and 16*ps + 8 of the lane's V position (v_addr[dt], LDS byte address of
// the slot-0 copy); SLOT_OFF selects the slot.
template <int SLOT_OFF, int ROW_BYTES, int DT, typename vec8>
__device__ __forceinline__ void ReadVFrags(const uint32_t (&v_addr)[DT], vec8 (&va)[2 * DT]) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const uint2 l0 = TrReadAsm<SLOT_OFF>(v_addr[dt]);
        const uint2 h0 = TrReadAsm<SLOT_OFF + 8 * ROW_BYTES>(v_addr[dt]);
        const uint2 l1 = TrReadAsm<SLOT_OFF + 16 * ROW_BYTES>(v_addr[dt]);
        const uint2 h1 = TrReadAsm<SLOT_OFF + 24 * ROW_BYTES>(v_addr[dt]);
        va[2 * dt] = __builtin_bit_cast(vec8, make_uint4(l0.x, l0.y, h0.x, h0.y));
        va[2 * dt + 1] = __builtin_bit_cast(vec8, make_uint4(l1.x, l1.y, h1.x, h1.y));
    }
}

constexpr int kSchedValuTrans = 0x402;  // VALU and transcendental

// 16-byte DMA of lane data from a raw buffer (base, num_records) at voffset + soffset into LDS
// at lds + 16 * lane. Bytes at or beyond num_records read as zero. (The buffer resource is
// built here rather than in the kernel body: a buffer-resource local in a kernel body makes the
// host pass drop the kernel's launch stub.)
__device__ __forceinline__ void DmaToLds(const uint8_t* base, int num_records, uint8_t* lds,
                                         uint32_t voffset, uint32_t soffset) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(base), 0, num_records, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(lds), 16,
                                             voffset, soffset, 0, 0);
}

// MFMAs issued from inline asm: S^T accumulators in VGPRs, O^T accumulators in AGPRs.
template <typename E>
struct MfmaAsm;

template <>
struct MfmaAsm<F16> {
    // S^T: A (K fragment) in VGPRs, B (Q fragment) in AGPRs, accumulator in VGPRs.
    template <typename V>
    static __device__ __forceinline__ void first_v(floatx16& c, const V& a, const V& b) {
        asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
    }
    template <typename V>
    static __device__ __forceinline__ void acc_v(floatx16& c, const V& a, const V& b) {
        asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
    }
    template <typename V>
    static __device__ __forceinline__ void acc_a(floatx16& c, const V& a, const V& b) {
        asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
};

template <>
struct MfmaAsm<BF16> {
    // S^T: A (K fragment) in VGPRs, B (Q fragment) in AGPRs, accumulator in VGPRs.
    template <typename V>
    static __device__ __forceinline__ void first_v(floatx16& c, const V& a, const V& b) {
        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
    }
    template <typename V>
    static __device__ __forceinline__ void acc_v(floatx16& c, const V& a, const V& b) {
        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
    }
    template <typename V>
    static __device__ __forceinline__ void acc_a(floatx16& c, const V& a, const V& b) {
        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
};

template <int OFF, typename V>
__device__ __forceinline__ void ReadB128Asm(V& dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}

template <int OFF>
__device__ __forceinline__ void ReadB64Asm(uint2& dst, uint32_t addr) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}

template <int OFF, typename V>
__device__ __forceinline__ void WriteB128Asm(uint32_t addr, const V& src) {
    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(src), "i"(OFF) : "memory");
}

// lgkmcnt(N) tied to the register it guards (the asm uses below it cannot move above it).
template <int N, typename V>
__device__ __forceinline__ void WaitLgkmTied(V& reg) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(reg) : "i"(N));
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): for asm immediates.
template <int N, typename F>
__device__ __forceinline__ void StaticFor(F&& f) {
    [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
        (f(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ void Fence() { __builtin_amdgcn_sched_barrier(0); }

// Gives a value the AGPR register class (an empty asm with an AGPR in/out operand), so that the
// loop-carried accumulators and Q fragments stay in AGPRs instead of being copied in and out.
template <typename V>
__device__ __forceinline__ void PinAgpr(V& x) {
    asm volatile("" : "+a"(x));
}

// 32 wait states ahead of VALU access to the O accumulators (AGPRs), tied to them: the compiler
// does not track the inline-asm MFMAs that last wrote O.
template <int DT>
__device__ __forceinline__ void SettleO(floatx16 (&o)[2][DT]) {
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) PinAgpr(o[r][dt]);
    }
}

}  // namespace
}  // namespace sca_hip
