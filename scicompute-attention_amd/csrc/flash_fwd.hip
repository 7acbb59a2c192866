// Flash prefill forward for gfx950: O = softmax(scale * Q K^T + mask) V, fp16/bf16 in, fp32
// accumulation, optional natural-log LSE. No score matrix is ever written to memory.
//
// Semantics follow the reference kernel (src/backends/flash/flash_fwd_impl.cuh:45-279,
// flash_online_softmax.cuh:34-99, flash_causal_mask.cuh:14-28): bottom-right causal mask
// (key j visible from row i iff j <= i + diagonal), masked logits are exactly -inf, GQA maps
// q head h to kv head h / (H_q / H_kv), P is rounded to the input dtype before the PV product,
// out = O / l (0 when l == 0), LSE = m + ln(l) (-inf when l == 0).
//
// Four kernels share one formulation (flash_common.hpp); this file validates and picks:
//   * flash_wide.hpp (head_dim 32 to 160: every non-causal grid, large causal grids and, at 64 and
//     128, packed variable-length batches in one launch): 4 waves of 64 query rows, K/V tiles
//     DMA'd into LDS;
//   * flash_pair.hip (head_dim 64 and 128, causal grids too small to balance 128-row tiles);
//   * flash_dsplit.hip (head_dim 192 and 256): the same with the dims of O split over two waves;
//   * flash_reg.hip (any head_dim whose K/V extent passes the 32-bit buffer offsets of the DMA
//     kernels, or with negative K/V row strides; small calls of one or two key tiles at head dims other
//     than 64 and 128): K/V staged through registers.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "flash_common.hpp"

namespace sca_hip {
namespace {

// Whether the DMA kernels' unsigned 32-bit buffer offsets reach every row (plus the rings' overrun).
bool DmaReach(const sca_flash_params& p) {
    constexpr int64_t kOverrun = 8 * 64;
    return p.k_ss >= 0 && p.v_ss >= 0 && (p.seq_kv + kOverrun) * p.k_ss * 2 < (1LL << 31) &&
           (p.seq_kv + kOverrun) * p.v_ss * 2 < (1LL << 31);
}

// One or two key tiles and a grid that leaves CUs idle: latency is all there is, and the register-staged
// kernel's shorter prologue wins at the head dims that also have it. Microseconds, register-staged
// against the kernel that serves longer calls:
//   one tile, up to one row tile per CU: D 96, 8 x 24 x 44 6.1 / 6.8; D 160, 16 x 16 x 64 8.9 / 9.5;
//   D 256, 4 x 16 x 30 7.6 / 8.7, from 44 keys on 10.7 / 9.9;
//   two, up to half the CUs (16 to 128 workgroups alike; at 192 the order turns): causal D 96 x 70 keys
//   7.35 / 7.73, x 96 7.58 / 7.82, x 104 7.80 / 7.85, x 120 7.98 / 7.91, D 32 x 80 5.56 / 5.61, D 96 20
//   rows x 110 keys 7.05 / 7.35 and 5 x 126 7.14 / 7.33; non-causal D 96 x 95 7.62 / 7.39; D 160 x 70 9.55
//   / 9.81, x 96 9.87 / 9.99, x 128 11.9 / 10.2, non-causal x 96 9.22 / 9.83. With LSE they stay with
//   the kernels whose LSE sums unrounded weights.
bool FewTilesCall(const sca_flash_params& p) {
    if (p.head_dim == 64 || p.head_dim == 128) return false;
    const int64_t row_tiles = (p.seq_q + 127) / 128 * p.batch * p.num_heads;
    if (p.seq_kv <= (p.head_dim > 160 ? 32 : 64)) return row_tiles <= CuCount();
    if (p.head_dim > 160 || p.lse != nullptr || 2 * row_tiles > CuCount()) return false;
    if (p.head_dim == 160) return p.seq_kv <= 96;
    return p.causal && p.seq_kv <= (p.head_dim == 96 && p.seq_q <= 32 ? 128 : 100);
}

// ---- Which kernel, and how its rows and keys are cut -------------------------------------------
struct FlashPlan {
    bool pair;
    int pack;
    int splits;
};

constexpr int64_t kMaxSplitBytes = int64_t{64} << 20;
constexpr int64_t kMinSplitKeys = 4 * 64;  // of each key range

int64_t SplitBytes(const sca_flash_params& p, int splits) {
    return splits <= 1 ? 0 : p.batch * p.num_heads * p.seq_q * splits * (p.head_dim + 2) * 4;
}

// Causal grids with at most one 128-row tile per CU run the pair kernel at head_dim 64 and 128 (64-row
// tiles in complementary pairs, so every workgroup holds the same share of the triangle); larger
// causal grids and every non-causal grid run the wide kernel (longest tiles first when causal).
// Measured warm: at 320-448 tiles on 256 CUs the longest-first 128-row grid is 20-30% faster than a
// second partial wave of pairs; at 256 tiles the pairs are 30% faster.
//
// Packing (a GQA group's rows share row tiles) is taken where it leaves fewer row tiles: with few
// query rows a tile per head is mostly empty and K/V are streamed once per query head. Unsplit only
// past one row tile per CU: below that the tiles run side by side and fewer of them save nothing.
//
// Splitting the keys (allow_split: the caller has scratch for the partial states) pays where the row
// tiles do not fill the CUs and the keys are many. The estimate below, in microseconds, weighs it
// against the unsplit kernel: a wide or split-dims workgroup takes about 0.1 + 0.0068 D per 64 keys and
// 4 + 0.022 D beside them (modelled one to a CU; at D 32 and 64 two or three share one, so there the
// rounds are overstated and no split goes past one workgroup per CU), a pair workgroup 1.19 times the step per 64 keys of two
// groups and 5 beside them (both fitted to measurements at D = 32 .. 256), and the merge's launch 8 plus
// its partials' write and read at 4.5 TB/s (with 5 for the launch 24 x 256 over 1,354 keys split, 28.1 us
// against 26.5 for the pairs).
FlashPlan PlanFlash(const sca_flash_params& p, bool allow_split) {
    const int64_t cus = CuCount();
    const int64_t group = p.num_heads / p.num_kv_heads;
    const int64_t tiles = (p.seq_q + 127) / 128;
    FlashPlan plan{false, 1, 1};
    plan.pair = p.causal && (p.head_dim == 64 || p.head_dim == 128) &&
                tiles * p.batch * p.num_heads <= cus;
    const int64_t packed_tiles = (p.seq_q * group + 127) / 128;
    const int pack = packed_tiles < tiles * group && p.seq_q * group < (1LL << 30)
                         ? static_cast<int>(group) : 1;
    if (!plan.pair && tiles * p.batch * p.num_heads > cus) plan.pack = pack;
    if (!allow_split) return plan;

    const double step = 0.1 + 0.0068 * static_cast<double>(p.head_dim);
    const double fixed = 4.0 + 0.022 * static_cast<double>(p.head_dim);
    const int64_t keys_max = p.seq_kv;
    const double keys_avg = p.causal ? static_cast<double>(p.diagonal) + 0.5 * static_cast<double>(p.seq_q)
                                     : static_cast<double>(p.seq_kv);
    auto wide_us = [&](int64_t units, int64_t splits) {
        const double longest = static_cast<double>((keys_max + 64 * splits - 1) / (64 * splits)) * step + fixed;
        const double rounds = static_cast<double>((units * splits + cus - 1) / cus);
        const double all = rounds * (keys_avg / 64.0 / static_cast<double>(splits) * step + fixed);
        return longest > all ? longest : all;
    };
    double best;
    const int64_t units_pack = (pack > 1 ? packed_tiles : tiles) * p.batch * p.num_heads / pack;
    if (plan.pair) {
        const int64_t t64 = (p.seq_q + 63) / 64;
        const int64_t n_a = (p.seq_kv + 63) / 64;
        const int64_t n_b = t64 > 1 ? (p.diagonal + 64 + 63) / 64 + 4 : 0;
        const int64_t wgs = (t64 + 1) / 2 * p.batch * p.num_heads;
        // With half the CUs idle the clock is a quarter higher.
        const double pair_step = (2 * wgs <= cus ? 0.8 : 1.0) * 1.19 * step;
        best = static_cast<double>((wgs + cus - 1) / cus) *
               (0.5 * static_cast<double>(n_a + n_b) * pair_step + 5.0);
    } else {
        best = wide_us(units_pack, 1);
    }
    best *= 0.93;  // a split has to promise more than the estimate's error
    for (int64_t splits = 2; splits <= 16 && splits * kMinSplitKeys <= p.seq_kv; ++splits) {
        const int64_t bytes = SplitBytes(p, static_cast<int>(splits));
        if (bytes > kMaxSplitBytes) break;
        const double us = wide_us(units_pack, splits) + 8.0 + 2.0 * static_cast<double>(bytes) / 4.5e6;
        if (us < best) {
            best = us;
            plan = FlashPlan{false, pack, static_cast<int>(splits)};
        }
    }
    return plan;
}

// Merges the partial states of `splits` key ranges: out = sum_s O_s 2^(m_s - m*) / sum_s l_s 2^(m_s - m*)
// with m* = max_s m_s (log2 units), states with l_s = 0 (no visible key) skipped and out = 0 when the
// denominator is 0; LSE = m* + log2 of the denominator, in natural units. A state of NaN scores has
// l_s = NaN and m_s = NaN or -inf and makes the row NaN, as in the unsplit kernels; this file is
// therefore compiled with NaN semantics, unlike theirs. One thread per row and 4 dims; bound by the
// partials' bytes.
constexpr int kCombineThreads = 256;

template <typename E>
__global__ __launch_bounds__(kCombineThreads) void flash_combine_kernel(const sca_flash_params p,
                                                                        const SplitArgs sp) {
    using M = Mfma<E>;
    const uint32_t quads = static_cast<uint32_t>(p.head_dim) / 4;
    const uint32_t rows = static_cast<uint32_t>(p.batch * p.num_heads * p.seq_q);
    const uint32_t idx = blockIdx.x * kCombineThreads + threadIdx.x;
    const uint32_t row = idx / quads;
    if (row >= rows) return;
    const uint32_t d0 = (idx % quads) * 4;
    const float2* ml = reinterpret_cast<const float2*>(sp.part_ml) + row;
    const float* po = sp.part_o + static_cast<int64_t>(row) * p.head_dim + d0;
    float m = neg_inf();
#pragma unroll 4
    for (int s = 0; s < sp.splits; ++s) m = fmaxf(m, ml[static_cast<int64_t>(s) * rows].x);
    float l = 0.0f;
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int s = 0; s < sp.splits; ++s) {
        const float2 st = ml[static_cast<int64_t>(s) * rows];
        if (st.y == 0.0f) continue;  // empty: its O may not have been written
        const float w = fast_exp2(st.x - m);
        l = fmaf(st.y, w, l);
        const float4 v = *reinterpret_cast<const float4*>(po + static_cast<int64_t>(s) * rows * p.head_dim);
        a[0] = fmaf(v.x, w, a[0]);
        a[1] = fmaf(v.y, w, a[1]);
        a[2] = fmaf(v.z, w, a[2]);
        a[3] = fmaf(v.w, w, a[3]);
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const uint32_t seq_q = static_cast<uint32_t>(p.seq_q), heads = static_cast<uint32_t>(p.num_heads);
    const uint32_t bh = row / seq_q;
    uint16_t* out = static_cast<uint16_t*>(p.out) + static_cast<int64_t>(bh / heads) * p.o_sb +
                    static_cast<int64_t>(bh % heads) * p.o_sh +
                    static_cast<int64_t>(row % seq_q) * p.o_ss + d0;
    *reinterpret_cast<uint2*>(out) =
        make_uint2(M::pack(a[0] * inv, a[1] * inv), M::pack(a[2] * inv, a[3] * inv));
    if (p.lse != nullptr && d0 == 0) {
        p.lse[row] = l > 0.0f ? (m + __log2f(l)) * kLn2 : neg_inf();
    }
}

template <typename E, bool kCausal>
int LaunchForDim(const sca_flash_params& p, const FlashPlan& plan, const SplitArgs& sp, hipStream_t s) {
    const bool reach = DmaReach(p) && !FewTilesCall(p);
    switch (p.head_dim) {
        case 32:
            return reach ? LaunchFlashWide<E, 32, kCausal>(p, sp, s) : LaunchFlashReg<E, 32, kCausal>(p, s);
        case 64:
            if (!reach) return LaunchFlashReg<E, 64, kCausal>(p, s);
            if (kCausal && plan.pair) return LaunchFlashPair<E, 64>(p, s);
            return LaunchFlashWide<E, 64, kCausal>(p, sp, s);
        case 96:
            return reach ? LaunchFlashWide<E, 96, kCausal>(p, sp, s) : LaunchFlashReg<E, 96, kCausal>(p, s);
        case 128:
            if (!reach) return LaunchFlashReg<E, 128, kCausal>(p, s);
            if (kCausal && plan.pair) return LaunchFlashPair<E, 128>(p, s);
            return LaunchFlashWide<E, 128, kCausal>(p, sp, s);
        case 160:
            return reach ? LaunchFlashWide<E, 160, kCausal>(p, sp, s) : LaunchFlashReg<E, 160, kCausal>(p, s);
        case 192:
            return reach ? LaunchFlashDsplit<E, 192, kCausal>(p, sp, s) : LaunchFlashReg<E, 192, kCausal>(p, s);
        case 256:
            return reach ? LaunchFlashDsplit<E, 256, kCausal>(p, sp, s) : LaunchFlashReg<E, 256, kCausal>(p, s);
        default: break;
    }
    return SetError(SCA_E_UNSUPPORTED_HEAD_DIM,
                    "flash: head_dim=" + std::to_string(p.head_dim) + " is not instantiated");
}

template <typename E>
int LaunchTyped(const sca_flash_params& p, void* scratch, int64_t scratch_bytes, hipStream_t s) {
    FlashPlan plan = PlanFlash(p, scratch != nullptr && DmaReach(p));
    if (SplitBytes(p, plan.splits) > scratch_bytes) plan = PlanFlash(p, false);
    SplitArgs sp{plan.pack, plan.splits, nullptr, nullptr};
    const int64_t rows = p.batch * p.num_heads * p.seq_q;
    if (plan.splits > 1) {
        sp.part_o = static_cast<float*>(scratch);
        sp.part_ml = sp.part_o + rows * plan.splits * p.head_dim;
    }
    const int rc = p.causal ? LaunchForDim<E, true>(p, plan, sp, s) : LaunchForDim<E, false>(p, plan, sp, s);
    if (rc != 0 || plan.splits == 1) return rc;
    const int64_t threads = rows * (p.head_dim / 4);
    hipLaunchKernelGGL((flash_combine_kernel<E>),
                       dim3(static_cast<unsigned>((threads + kCombineThreads - 1) / kCombineThreads)),
                       dim3(kCombineThreads), 0, s, p, sp);
    return CheckLaunch("flash_combine_kernel", s);
}

bool Aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }


template <typename E>
int LaunchVarlenTyped(const sca_flash_varlen_params& v, hipStream_t s) {
    if (v.head_dim == 64) {
        return v.causal ? LaunchFlashVarlen<E, 64, true>(v, s) : LaunchFlashVarlen<E, 64, false>(v, s);
    }
    return v.causal ? LaunchFlashVarlen<E, 128, true>(v, s) : LaunchFlashVarlen<E, 128, false>(v, s);
}



int LdsBytesFor(int64_t head_dim) {
    switch (head_dim) {
        case 32: return WideGeom<32>::LDS_BYTES;
        case 64: return std::max(WideGeom<64>::LDS_BYTES, PairGeom<64>::LDS_BYTES);
        case 96: return WideGeom<96>::LDS_BYTES;
        case 128: return std::max(WideGeom<128>::LDS_BYTES, PairGeom<128>::LDS_BYTES);
        case 160: return WideGeom<160>::LDS_BYTES;
        case 192: return DsplitGeom<192>::LDS_BYTES;
        case 256: return DsplitGeom<256>::LDS_BYTES;
        default: return -1;
    }
}

}  // namespace
}  // namespace sca_hip

using sca_hip::SetError;

extern "C" {

int64_t sca_hip_flash_lds_bytes(int32_t head_dim, int64_t elem_bytes) {
    if (elem_bytes != 2) return -1;
    return sca_hip::LdsBytesFor(head_dim);
}

int sca_hip_flash_tile(int32_t head_dim, int32_t* block_m, int32_t* block_n, int32_t* waves,
                       int32_t* stages) {
    if (sca_hip::LdsBytesFor(head_dim) < 0) {
        return SetError(SCA_E_UNSUPPORTED_HEAD_DIM,
                        "flash: no tile for head_dim=" + std::to_string(head_dim));
    }
    // The wide kernel's tile (at head_dim 64 and 128: every non-causal and every large causal
    // grid); head_dim 192 and 256 the split-dims kernel's.
    int32_t bn = sca_hip::WideGeom<128>::BN, nw = sca_hip::WideGeom<128>::WAVES,
            ns = sca_hip::WideGeom<128>::SLOTS;
    if (head_dim > 160) {
        using G = sca_hip::DsplitGeom<256>;
        bn = G::BN, nw = G::WAVES, ns = G::SLOTS;
    }
    if (block_m != nullptr) *block_m = sca_hip::kBlockM;
    if (block_n != nullptr) *block_n = bn;
    if (waves != nullptr) *waves = nw;
    if (stages != nullptr) *stages = ns;
    return 0;
}

int sca_hip_flash_varlen_supported(int32_t head_dim) { return head_dim == 64 || head_dim == 128; }

int64_t sca_hip_flash_varlen_tiles(const int32_t* cu_q, const int32_t* cu_kv, int64_t num_seqs,
                                   int32_t causal, int32_t* tiles_out) {
    if (cu_q == nullptr || cu_kv == nullptr || num_seqs < 1) {
        return -SetError(SCA_E_SHAPE_MISMATCH, "flash varlen: null cu_seqlens or no sequences");
    }
    constexpr int64_t kRows = 128;  // rows per workgroup of the varlen launch
    struct Tile {
        int64_t keys;
        int32_t seq;
        int32_t tile;
    };
    std::vector<Tile> tiles;
    for (int64_t s = 0; s < num_seqs; ++s) {
        const int64_t sq = static_cast<int64_t>(cu_q[s + 1]) - cu_q[s];
        const int64_t skv = static_cast<int64_t>(cu_kv[s + 1]) - cu_kv[s];
        if (sq < 0 || skv < 0 || (causal && skv < sq) || (sq > 0 && skv == 0)) {
            return -SetError(SCA_E_SHAPE_MISMATCH,
                             "flash varlen: sequence " + std::to_string(s) + " has S_q=" +
                                 std::to_string(sq) + ", S_kv=" + std::to_string(skv));
        }
        for (int64_t t = 0; t * kRows < sq; ++t) {
            const int64_t last = std::min(sq, (t + 1) * kRows) - 1 + (skv - sq);
            const int64_t keys = causal ? std::min(skv, last + 1) : skv;
            tiles.push_back({keys, static_cast<int32_t>(s), static_cast<int32_t>(t)});
        }
    }
    std::stable_sort(tiles.begin(), tiles.end(),
                     [](const Tile& a, const Tile& b) { return a.keys > b.keys; });
    if (tiles_out != nullptr) {
        for (size_t i = 0; i < tiles.size(); ++i) {
            tiles_out[2 * i] = tiles[i].seq;
            tiles_out[2 * i + 1] = tiles[i].tile;
        }
    }
    return static_cast<int64_t>(tiles.size());
}

int sca_hip_flash_fwd_varlen(const sca_flash_varlen_params* v, void* stream) {
    if (v == nullptr || v->q == nullptr || v->k == nullptr || v->v == nullptr ||
        v->out == nullptr || v->cu_seqlens_q == nullptr || v->cu_seqlens_kv == nullptr ||
        (v->num_tiles > 0 && v->tiles == nullptr)) {
        return SetError(SCA_E_SHAPE_MISMATCH, "flash varlen: null pointer");
    }
    if (!sca_hip_flash_varlen_supported(static_cast<int32_t>(v->head_dim))) {
        return SetError(SCA_E_UNSUPPORTED_HEAD_DIM,
                        "flash varlen: head_dim=" + std::to_string(v->head_dim) +
                            " has no one-launch kernel (64 and 128 do)");
    }
    if (v->dtype != SCA_DTYPE_F16 && v->dtype != SCA_DTYPE_BF16) {
        return SetError(SCA_E_UNSUPPORTED_DTYPE, "flash varlen: fp16/bf16 only");
    }
    if (v->num_heads < 1 || v->num_kv_heads < 1 || v->num_heads % v->num_kv_heads != 0 ||
        v->num_tiles < 0 || v->max_seq_kv < 0 || v->num_seqs < 1) {
        return SetError(SCA_E_SHAPE_MISMATCH, "flash varlen: invalid heads or counts");
    }
    if (!sca_hip::Aligned16(v->q) || !sca_hip::Aligned16(v->k) || !sca_hip::Aligned16(v->v) ||
        !sca_hip::Aligned16(v->out) || v->q_ss % 8 || v->q_sh % 8 || v->k_ss % 8 ||
        v->k_sh % 8 || v->v_ss % 8 || v->v_sh % 8 || v->o_ss % 8 || v->o_sh % 8) {
        return SetError(SCA_E_LAYOUT_MISMATCH,
                        "flash varlen: pointers must be 16 B aligned and strides multiples of 8");
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    return v->dtype == SCA_DTYPE_F16 ? sca_hip::LaunchVarlenTyped<sca_hip::F16>(*v, s)
                                     : sca_hip::LaunchVarlenTyped<sca_hip::BF16>(*v, s);
}

}  // extern "C"

namespace sca_hip {
namespace {
int ValidateFlash(const sca_flash_params* p) {
    if (p == nullptr) return SetError(SCA_E_SHAPE_MISMATCH, "flash: null params");
    if (p->q == nullptr || p->k == nullptr || p->v == nullptr || p->out == nullptr) {
        return SetError(SCA_E_SHAPE_MISMATCH, "flash: null pointer");
    }
    if (p->dtype != SCA_DTYPE_F16 && p->dtype != SCA_DTYPE_BF16) {
        return SetError(SCA_E_UNSUPPORTED_DTYPE,
                        "flash: dtype id " + std::to_string(p->dtype) +
                            " (the MFMA kernel computes in fp16/bf16 only)");
    }
    if (p->batch < 1 || p->num_heads < 1 || p->num_kv_heads < 1 || p->seq_q < 1 ||
        p->seq_kv < 1 || p->num_heads % p->num_kv_heads != 0) {
        return SetError(SCA_E_SHAPE_MISMATCH,
                        "flash: invalid geometry B=" + std::to_string(p->batch) +
                            " Hq=" + std::to_string(p->num_heads) +
                            " Hkv=" + std::to_string(p->num_kv_heads) +
                            " Sq=" + std::to_string(p->seq_q) + " Skv=" + std::to_string(p->seq_kv));
    }
    if (p->seq_q > (1LL << 30) || p->seq_kv > (1LL << 30) || p->k_ss > (1LL << 24) ||
        p->v_ss > (1LL << 24)) {
        return SetError(SCA_E_SEQ_TOO_LONG,
                        "flash: seq_q/seq_kv must be <= 2^30 and K/V row strides <= 2^24 elements");
    }
    if (p->causal && p->diagonal < 0) {
        return SetError(SCA_E_SHAPE_MISMATCH,
                        "flash: causal needs diagonal >= 0 (seq_kv >= seq_q); diagonal=" +
                            std::to_string(p->diagonal));
    }
    if (!(p->scale > 0.0f)) {
        return SetError(SCA_E_SHAPE_MISMATCH, "flash: scale must be > 0");
    }
    if (!sca_hip::Aligned16(p->q) || !sca_hip::Aligned16(p->k) || !sca_hip::Aligned16(p->v) ||
        !sca_hip::Aligned16(p->out) || p->q_ss % 8 || p->q_sh % 8 || p->q_sb % 8 ||
        p->k_ss % 8 || p->k_sh % 8 || p->k_sb % 8 || p->v_ss % 8 || p->v_sh % 8 ||
        p->v_sb % 8 || p->o_ss % 4 || p->o_sh % 4 || p->o_sb % 4) {
        return SetError(SCA_E_LAYOUT_MISMATCH,
                        "flash: q/k/v/out must be 16 B aligned with 16 B-multiple row strides");
    }
    return 0;
}
}  // namespace
}  // namespace sca_hip

extern "C" {

int64_t sca_hip_flash_split_bytes(const sca_flash_params* p) {
    // Short calls, which the host's own work bounds, are answered first.
    if (p != nullptr && p->seq_kv < 2 * sca_hip::kMinSplitKeys) return 0;
    if (sca_hip::ValidateFlash(p) != 0 || !sca_hip::DmaReach(*p)) return 0;
    return sca_hip::SplitBytes(*p, sca_hip::PlanFlash(*p, true).splits);
}

int sca_hip_flash_fwd_split(const sca_flash_params* p, void* scratch, int64_t scratch_bytes,
                            void* stream) {
    const int rc = sca_hip::ValidateFlash(p);
    if (rc != 0) return rc;
    if (!sca_hip::Aligned16(scratch)) {
        return SetError(SCA_E_LAYOUT_MISMATCH, "flash: scratch must be 16 B aligned");
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    return p->dtype == SCA_DTYPE_F16
               ? sca_hip::LaunchTyped<sca_hip::F16>(*p, scratch, scratch_bytes, s)
               : sca_hip::LaunchTyped<sca_hip::BF16>(*p, scratch, scratch_bytes, s);
}

int sca_hip_flash_fwd(const sca_flash_params* p, void* stream) {
    return sca_hip_flash_fwd_split(p, nullptr, 0, stream);
}

}  // extern "C"
