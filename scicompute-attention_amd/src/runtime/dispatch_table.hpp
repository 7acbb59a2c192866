// Compiled-in dispatch thresholds of the MI355X build.
//
// The routing rules are the reference's (src/runtime/dispatch_table.inc:30-37, r0) except one:
// short sequences (seq_kv <= 128) go to the flash kernel, which serves every length without a
// score workspace, instead of the reference's score-materialising tiled kernel (not built here).
// Split counts are derived from the compute-unit count: enough workgroups for every CU to hold
// several, each split still covering at least `min_tokens_per_split` keys.
#pragma once

#include <cstdint>

namespace sca {
namespace detail {

struct DispatchThresholds {
    int64_t decode_max_seq_q;      // seq_q <= this and seq_kv >= decode_min_seq_kv => decode
    int64_t decode_min_seq_kv;
    int64_t short_max_seq_kv;      // seq_kv <= this => "short sequence" rule (flash here)
    int64_t min_tokens_per_split;  // lower bound on keys per split
    int64_t workgroups_per_cu;     // split-K target occupancy
    int64_t max_splits;            // cap on the split count (explicit and automatic)
    const char* revision;          // reported by Explain()
};

inline constexpr DispatchThresholds kDispatchThresholds{
    /* decode_max_seq_q     */ 1,
    /* decode_min_seq_kv    */ 256,
    /* short_max_seq_kv     */ 128,
    /* min_tokens_per_split */ 512,
    /* workgroups_per_cu    */ 6,
    /* max_splits           */ 64,
    /* revision             */ "r0-mi355x",
};

// Split count of the decode kernels for `batch` sequences of up to `seq_kv` keys. A head slot is
// one KV head and up to 16 of its query heads; the MFMA kernel runs a workgroup per (sequence,
// split, slot) with four waves per slot (slot_waves = 4, the contiguous default) or per (sequence,
// split, four slots) with one wave per slot (slot_waves = 1, the paged default).
//  - Four waves per slot: a batch with at least one slot per CU runs unsplit, which also skips
//    the combine kernel (measured on MI355X, fp16, H_q 32, H_kv 8, D 128: 64 x 4096 keys 6.07 TB/s
//    against 5.65 at 8 splits; 128 x 2048 6.02 against 5.64; 32 x 4096 5.74 against 5.42);
//    smaller batches take splits until every CU holds 4 workgroups, but no more than 8 unless
//    fewer would leave CUs without a workgroup (C4, 16 x 4096: 8 splits, 5.97 TB/s; 8 x 32768:
//    8 splits, 5.95 against 5.47 at 64; 4 x 16384: 8, 5.84 against 5.66 at 32; 1 x 65536: 32,
//    5.60 against 5.22 at 64).
//  - One wave per slot: splits are added until every CU holds `workgroups_per_cu` workgroups.
//  - head_dim outside {64, 128}: unsplit once the batch gives every CU a workgroup, else splits
//    until every CU holds four, with no cap at 8 (made for the VALU kernel, a workgroup per
//    (sequence, split, 1-8 heads): fp16, H_q 32, H_kv 8, D 96: 4 x 16384 keys 32 splits, 4.34 TB/s
//    against 3.37 at 8; 16 x 4096 8 splits, 4.63, the best of 1..32; 64 x 4096 unsplit 5.05 against
//    5.10 at 4; the MFMA kernel at D 96 and 32 is within 6% of its best there: 16 x 4096 4.80 TB/s
//    against 4.88 at 4). fp32 with D 64 or 128 runs the VALU kernel under the MFMA rule (16 x 4096,
//    D 128: 5.21 TB/s at 8 splits against 5.52 at 4);
//  - 16-bit types (`half`) with head_dim >= 160 and groups above 2, where the MFMA kernel's rings
//    leave room for one workgroup per CU: one workgroup per CU (bf16, H_q 32, H_kv 8: D 192, 16 x
//    4096 2 splits 5.23 TB/s against 4.45 at 8; D 160, 4 x 8192 8 splits 4.77 against 4.10 at 16;
//    D 256, 2 x 16384 16 splits 4.82 against 4.25 at 32).
// Each split keeps at least `min_tokens_per_split` keys.
inline int64_t DecodeSplits(int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                            int64_t seq_kv, int64_t cu_count, int slot_waves = 4,
                            int64_t head_dim = 128, bool half = false) {
    const auto& th = kDispatchThresholds;
    if (batch < 1 || num_kv_heads < 1 || seq_kv < 1) return 1;
    const int64_t group = num_heads / num_kv_heads;
    const int64_t slots = num_kv_heads * ((group + 15) / 16);
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    int64_t splits;
    const bool mfma = head_dim == 64 || head_dim == 128;
    if (!mfma) {
        const int64_t jobs = batch * slots;
        const bool one_per_cu = half && head_dim >= 160 && group > 2;
        splits = jobs >= cus ? 1 : one_per_cu ? cus / jobs : (4 * cus + jobs - 1) / jobs;
    } else if (slot_waves == 1) {
        const int64_t wgs_per_split = batch * ((slots + 3) / 4);
        splits = (th.workgroups_per_cu * cus + wgs_per_split - 1) / wgs_per_split;
    } else {
        const int64_t jobs = batch * slots;
        if (jobs >= cus) {
            splits = 1;
        } else {
            const int64_t fill = (cus + jobs - 1) / jobs;  // one workgroup per CU
            const int64_t four = (4 * cus + jobs - 1) / jobs;
            splits = four < 8 ? four : (fill > 8 ? fill : 8);
        }
    }
    const int64_t by_length = (seq_kv + th.min_tokens_per_split - 1) / th.min_tokens_per_split;
    if (splits > by_length) splits = by_length;
    if (splits > th.max_splits) splits = th.max_splits;
    return splits < 1 ? 1 : splits;
}

// What the contiguous backend runs for fp32 and for head_dim >= 160: the count above, except that a
// batch whose workgroups would leave half the CUs idle (few sequences, splits at their minimum length)
// takes shorter splits, down to 128 keys, until every CU has a workgroup: one CU streams about 60 GB/s,
// and 500 such keys take it 8 us and more (fp32 D 128, 1 x 3000 30.3 -> 14.8 us, 4 x 16/4 x 2000 29.6 ->
// 14.8; bf16 D 256, 2 x 1000 34 -> 13). Up to head_dim 128 in 16 bits the two launches bound the call
// and the longer merge costs 3% (4 x 700, D 128: 12.4 -> 12.8), so the count stays.
// An unsplit call stays unsplit while a slot's K and V (`key_bytes` per key) are below 256 KiB: it saves
// the merge's launch (unsplit / split, us: fp32 D 128, 2 sequences of 130 keys 9.7 / 12.3, of 256 13.7 /
// 12.5; fp32 D 64 x 511 9.6 / 12.6; bf16 D 256 x 256 12.7 / 12.8, x 300 15.2 / 13.0; paged bf16 D 128,
// 3 x 130 13.9 / 15.7, x 511 15.3 / 17.6, D 192 x 300 17.3 / 17.2, x 400 19.9 / 17.3).
inline int64_t FillSplits(int64_t splits, int64_t jobs, int64_t longest, int64_t cu_count,
                          int64_t key_bytes) {
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    if (2 * splits * jobs > cus || (splits == 1 && longest * key_bytes < (256 << 10))) return splits;
    int64_t fill = cus / jobs;
    const int64_t by_length = (longest + 127) / 128;
    fill = fill < by_length ? fill : by_length;
    fill = fill < kDispatchThresholds.max_splits ? fill : kDispatchThresholds.max_splits;
    return fill > splits ? fill : splits;
}

// The contiguous backend's split count (four waves per slot); `half`: 16-bit types.
inline int64_t ContiguousDecodeSplits(int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                                      int64_t seq_kv, int64_t cu_count, int64_t head_dim, bool half) {
    const int64_t splits =
        DecodeSplits(batch, num_heads, num_kv_heads, seq_kv, cu_count, 4, head_dim, half);
    if (batch < 1 || num_kv_heads < 1 || (half && head_dim < 160)) return splits;
    const int64_t slots = num_kv_heads * ((num_heads / num_kv_heads + 15) / 16);
    return FillSplits(splits, batch * slots, seq_kv, cu_count, 2 * head_dim * (half ? 2 : 4));
}

struct LengthSummary {
    int64_t longest;
    bool uniform;  // longest <= 11/10 of the mean
};
inline LengthSummary SummarizeLengths(const int64_t* lengths, int64_t batch) {
    int64_t longest = 0;
    int64_t total = 0;
    for (int64_t b = 0; b < batch; ++b) {
        const int64_t len = lengths[b] > 0 ? lengths[b] : 0;
        longest = len > longest ? len : longest;
        total += len;
    }
    return {longest, 10 * longest * batch <= 11 * total};
}

// Paged 16-bit calls whose group is too small for the MFMA kernel (the launcher's rule) run the VALU
// kernel, a workgroup per (sequence, KV head, split), four to a CU.
inline bool PagedValuGroup(int64_t head_dim, int64_t group) {
    return head_dim != 64 && head_dim != 128 &&
           ((group == 1 && head_dim != 32) || (group == 2 && head_dim >= 160));
}
// Its splits for known lengths: unsplit from two workgroups per CU on (four, below head_dim 192 from 512
// keys on), else until every CU holds four; and eight where the batch is ragged (the launch ends with its
// longest sequences) or, with one head per KV head, below head_dim 192 from 512 keys on; 128 keys each at
// least (bf16, unsplit / 8, us: 16/16 heads, D 96: 64 x 1000 85 / 72, 128 x
// 128..4000 405 / 274; D 256: 64 x 1000 180 / 186, 128 x 128..4000 765 / 712; 16/8, D 160: 128 x 600 77 / 98,
// 32 x 2000 119 / 64, 64 x 512..8192 524 / 280; unsplit / 2: D 96 40 x 300 20 / 22, D 192 16/8 64 x 1000 78 / 80,
// D 160 75 / 68).
inline int64_t PagedValuSplits(int64_t head_dim, const int64_t* lengths, int64_t batch, int64_t num_heads,
                               int64_t num_kv_heads, int64_t cu_count) {
    const LengthSummary len = SummarizeLengths(lengths, batch);
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    const int64_t jobs = batch * num_kv_heads;
    const bool split_pays = head_dim < 192 && len.longest >= 512;
    int64_t splits = jobs >= (split_pays ? 4 : 2) * cus ? 1 : (4 * cus + jobs - 1) / jobs;
    if ((!len.uniform || (split_pays && num_heads == num_kv_heads)) && splits < 8) splits = 8;
    if (splits > len.longest / 128) splits = len.longest / 128;
    if (splits > kDispatchThresholds.max_splits) splits = kDispatchThresholds.max_splits;
    return splits < 1 ? 1 : splits;
}

// Work split of the paged MFMA decode kernel for a batch whose host-side lengths are known.
// slot_waves = 1: one wave per head slot, a workgroup serves four slots; 4: four waves share one
// slot's key tiles. Measured on MI355X over 48-step decode loops (bf16, H_q 32, H_kv 8, D 128):
//  - near-uniform batches (longest <= 11/10 of the mean) that leave some CUs free with one split:
//    one wave per slot, one workgroup per CU (uniform 64 x 8448 keys: 5.89 TB/s vs 5.58);
//  - ragged batches with at most two slots per CU: four waves per slot, `workgroups_per_cu`
//    workgroups per CU (C5, 64 x 512..16384: 5.74 TB/s vs 5.61; 16 sequences: 4.98 vs 4.26;
//    64 x 6000..10000: 5.55 vs 5.41 for one wave per slot at one workgroup per CU);
//  - otherwise (many sequences): one wave per slot, `workgroups_per_cu` workgroups per CU
//    (256 x 512..4096: 5.56 TB/s vs 5.54).
// Each split keeps at least `min_tokens_per_split` keys of the longest sequence.
struct PagedDecodePlanResult {
    int64_t splits;
    int32_t slot_waves;
};

inline PagedDecodePlanResult PagedDecodePlan(const int64_t* lengths, int64_t batch,
                                             int64_t num_heads, int64_t num_kv_heads,
                                             int64_t cu_count) {
    const auto& th = kDispatchThresholds;
    if (lengths == nullptr || batch < 1 || num_kv_heads < 1 || num_heads < num_kv_heads) {
        return {1, 0};
    }
    const LengthSummary len = SummarizeLengths(lengths, batch);
    const int64_t longest = len.longest;
    if (longest < 1) return {1, 0};
    const int64_t group = num_heads / num_kv_heads;
    const int64_t slots = num_kv_heads * ((group + 15) / 16);
    const int64_t quads = (slots + 3) / 4;
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    const bool uniform = len.uniform;
    int64_t splits;
    int32_t slot_waves;
    if (uniform && batch * quads <= cus) {
        slot_waves = 1;
        splits = cus / (batch * quads);
    } else if (batch * slots <= 2 * cus) {
        slot_waves = 4;
        splits = (th.workgroups_per_cu * cus + batch * slots - 1) / (batch * slots);
    } else {
        slot_waves = 1;
        splits = (th.workgroups_per_cu * cus + batch * quads - 1) / (batch * quads);
    }
    const int64_t by_length = (longest + th.min_tokens_per_split - 1) / th.min_tokens_per_split;
    if (splits > by_length) splits = by_length;
    if (splits > th.max_splits) splits = th.max_splits;
    return {splits < 1 ? 1 : splits, slot_waves};
}

// What the paged backend runs: the plan above, except
//  - one wave per slot that would leave half the CUs without a workgroup (few sequences, splits at
//    their minimum length) becomes four waves per slot at the same splits: four times the
//    workgroups, each with a quarter of the tiles per wave, and shorter splits where that still
//    leaves CUs idle (FillSplits);
//  - head_dim >= 160, where the kernel's rings leave room for one workgroup per CU. Near-uniform or short
//    (up to 512 keys) batches that reach a quarter of the CUs with one wave per slot: that, split until
//    every CU has a workgroup, 128 keys each at least (us, one wave / four: bf16 32/8, D 160: 153 x 108
//    keys 38 / 62, 40 x 300 23 / 31, 128 x 600 73 / 107, 64 x 1000 62 / 72, 150 x 16..200 30 / 64). Others
//    four waves per slot, unsplit from two slots per CU on, two workgroups per CU down to half a slot per
//    CU and one below (bf16, H_kv 8: D 256, 16 x 512..16384 4 splits 5.52 TB/s against 5.00 at 12; D 256,
//    4 x 4000..9000 x 16 heads 4 splits 4.73 against 3.95 at 12).
inline PagedDecodePlanResult PagedDecodePlanFor(int64_t head_dim, const int64_t* lengths,
                                                int64_t batch, int64_t num_heads,
                                                int64_t num_kv_heads, int64_t cu_count) {
    PagedDecodePlanResult plan = PagedDecodePlan(lengths, batch, num_heads, num_kv_heads, cu_count);
    if (plan.slot_waves == 0) return plan;
    const int64_t slots = num_kv_heads * ((num_heads / num_kv_heads + 15) / 16);
    const int64_t jobs = batch * slots;
    const int64_t cus = cu_count > 0 ? cu_count : 256;
    const LengthSummary len = SummarizeLengths(lengths, batch);
    const int64_t longest = len.longest;
    if (head_dim >= 160) {
        const auto& th = kDispatchThresholds;
        const int64_t wgs = batch * ((slots + 3) / 4);  // of one wave per slot
        if ((len.uniform || longest <= 512) && 4 * wgs >= cus) {
            int64_t splits = cus / wgs;
            splits = splits < longest / 128 ? splits : longest / 128;
            return {splits < 1 ? 1 : splits, 1};
        }
        const int64_t by_length = (longest + th.min_tokens_per_split - 1) / th.min_tokens_per_split;
        int64_t splits = jobs >= 2 * cus ? 1 : 2 * jobs >= cus ? 2 * cus / jobs : cus / jobs;
        splits = splits < by_length ? splits : by_length;
        splits = splits < th.max_splits ? splits : th.max_splits;
        return {FillSplits(splits < 1 ? 1 : splits, jobs, longest, cus, 4 * head_dim), 4};
    }
    if (plan.slot_waves == 1 && 2 * plan.splits * batch * ((slots + 3) / 4) <= cus) {
        plan.slot_waves = 4;
        plan.splits = FillSplits(plan.splits, jobs, longest, cus, 4 * head_dim);
    }
    return plan;
}

}  // namespace detail
}  // namespace sca
