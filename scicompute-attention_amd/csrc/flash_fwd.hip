// Flash prefill forward for gfx950: O = softmax(scale * Q K^T + mask) V, fp16/bf16 in, fp32
// accumulation, optional natural-log LSE. No score matrix is ever written to memory.
//
// Semantics follow the reference kernel (src/backends/flash/flash_fwd_impl.cuh:45-279,
// flash_online_softmax.cuh:34-99, flash_causal_mask.cuh:14-28): bottom-right causal mask
// (key j visible from row i iff j <= i + diagonal), masked logits are exactly -inf, GQA maps
// q head h to kv head h / (H_q / H_kv), P is rounded to the input dtype before the PV product,
// out = O / l (0 when l == 0), LSE = m + ln(l) (-inf when l == 0).
//
// Three kernels share one formulation (flash_common.hpp); this file validates and picks:
//   * flash_wide.hip (head_dim 32 to 160: every non-causal grid, large causal grids and, at 64 and
//     128, packed variable-length batches in one launch): 4 waves of 64 query rows, K/V tiles
//     DMA'd into LDS;
//   * flash_pair.hip (head_dim 64 and 128, causal grids too small to balance 128-row tiles);
//   * flash_dsplit.hip (head_dim 192 and 256): the same with the dims of O split over two waves;
//   * flash_reg.hip (any head_dim whose K/V extent passes the 32-bit buffer offsets of the DMA
//     kernels, or with negative K/V row strides): K/V staged through registers.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "flash_common.hpp"

namespace sca_hip {
namespace {

// Causal grids with at most one 128-row tile per CU run the pair kernel (64-row tiles in
// complementary pairs, so every workgroup holds the same share of the triangle); larger causal
// grids and every non-causal grid run the wide kernel (longest tiles first when causal). Measured
// warm: at 320-448 tiles on 256 CUs the longest-first 128-row grid is 20-30% faster than a
// second partial wave of pairs; at 256 tiles the pairs are 30% faster.
bool UsePairs(const sca_flash_params& p) {
    static int cu_count = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
            (void)hipGetLastError();
            n = 256;
        }
        return n > 0 ? n : 256;
    }();
    const int64_t tiles128 = (p.seq_q + 127) / 128 * p.batch * p.num_heads;
    return tiles128 <= static_cast<int64_t>(cu_count);
}

template <typename E, bool kCausal>
int LaunchForDim(const sca_flash_params& p, hipStream_t s) {
    switch (p.head_dim) {
        case 32: return LaunchFlashWide<E, 32, kCausal>(p, s);
        case 64:
            if (kCausal && UsePairs(p)) return LaunchFlashPair<E, 64>(p, s);
            return LaunchFlashWide<E, 64, kCausal>(p, s);
        case 96: return LaunchFlashWide<E, 96, kCausal>(p, s);
        case 128:
            if (kCausal && UsePairs(p)) return LaunchFlashPair<E, 128>(p, s);
            return LaunchFlashWide<E, 128, kCausal>(p, s);
        case 160: return LaunchFlashWide<E, 160, kCausal>(p, s);
        case 192: return LaunchFlashDsplit<E, 192, kCausal>(p, s);
        case 256: return LaunchFlashDsplit<E, 256, kCausal>(p, s);
        default: break;
    }
    return SetError(SCA_E_UNSUPPORTED_HEAD_DIM,
                    "flash: head_dim=" + std::to_string(p.head_dim) + " is not instantiated");
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

int sca_hip_flash_fwd(const sca_flash_params* p, void* stream) {
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
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (p->dtype == SCA_DTYPE_F16) {
        return p->causal ? sca_hip::LaunchForDim<sca_hip::F16, true>(*p, s)
                         : sca_hip::LaunchForDim<sca_hip::F16, false>(*p, s);
    }
    return p->causal ? sca_hip::LaunchForDim<sca_hip::BF16, true>(*p, s)
                     : sca_hip::LaunchForDim<sca_hip::BF16, false>(*p, s);
}

}  // extern "C"
