// The pure split rules of decode (runtime/dispatch_table.hpp) at the edges of their clamps, on 256 CUs.
// Compiled by tests/test_decode_plan.py.

#include <cstdint>
#include <cstdio>
#include <vector>

#include "runtime/dispatch_table.hpp"

using namespace sca::detail;

namespace {
int failures = 0;

void Check(const char* what, int64_t got, int64_t want) {
    if (got == want) return;
    std::printf("%s: %lld, expected %lld\n", what, static_cast<long long>(got), static_cast<long long>(want));
    ++failures;
}

void CheckPlan(const char* what, int64_t head_dim, const std::vector<int64_t>& lengths, int64_t heads,
               int64_t kv_heads, int64_t splits, int32_t waves) {
    const auto p = PagedDecodePlanFor(head_dim, lengths.data(), static_cast<int64_t>(lengths.size()), heads,
                                      kv_heads, 256);
    Check(what, p.splits, splits);
    Check(what, p.slot_waves, waves);
}
}  // namespace

int main() {
    // Splits for idle CUs: not when half of them have a workgroup, at most 128 keys each and the table's
    // cap, never fewer than before, and the default CU count when it is unknown.
    Check("half busy", FillSplits(8, 17, 100000, 256, 1024), 8);
    Check("half idle", FillSplits(8, 16, 100000, 256, 1024), 16);
    Check("short keys", FillSplits(2, 1, 257, 256, 1024), 3);
    Check("the table's cap", FillSplits(1, 1, 1 << 20, 256, 512), 64);
    Check("never fewer", FillSplits(3, 4, 130, 256, 1024), 3);
    Check("unknown CU count", FillSplits(1, 8, 1 << 20, 0, 512), 32);
    // Unsplit calls stay unsplit below 256 KiB of K and V a slot.
    Check("below 256 KiB", FillSplits(1, 16, 255, 256, 1024), 1);
    Check("from 256 KiB", FillSplits(1, 16, 256, 256, 1024), 2);
    Check("no keys", FillSplits(1, 1, 0, 256, 1024), 1);

    // Contiguous KV: the fill is for fp32 and for head_dim >= 160.
    Check("fp32 1 x 3000", ContiguousDecodeSplits(1, 32, 8, 3000, 256, 128, false), 24);
    Check("16 bits 1 x 3000", ContiguousDecodeSplits(1, 32, 8, 3000, 256, 128, true), 6);
    Check("fp32 4 x 2000", ContiguousDecodeSplits(4, 16, 4, 2000, 256, 128, false), 16);
    Check("16 bits 4 x 2000", ContiguousDecodeSplits(4, 16, 4, 2000, 256, 128, true), 4);
    Check("fp32 2 x 1000, D 256", ContiguousDecodeSplits(2, 32, 8, 1000, 256, 256, false), 8);
    Check("16 bits 2 x 1000, D 256", ContiguousDecodeSplits(2, 32, 8, 1000, 256, 256, true), 8);
    Check("D 160: one workgroup per CU", ContiguousDecodeSplits(4, 32, 8, 8192, 256, 160, true), 8);
    Check("D 160, fp32: four", ContiguousDecodeSplits(4, 32, 8, 8192, 256, 160, false), 16);
    Check("D 192, a group of two: four", ContiguousDecodeSplits(4, 16, 8, 8192, 256, 192, true), 16);
    Check("D 256, a slot per CU", ContiguousDecodeSplits(32, 32, 8, 4096, 256, 256, true), 1);
    Check("fp32 2 x 255", ContiguousDecodeSplits(2, 32, 8, 255, 256, 128, false), 1);
    Check("fp32 2 x 256", ContiguousDecodeSplits(2, 32, 8, 256, 256, 128, false), 2);
    Check("fp32 1 x 511, D 64", ContiguousDecodeSplits(1, 8, 8, 511, 256, 64, false), 1);
    Check("16 bits 2 x 300, D 256", ContiguousDecodeSplits(2, 32, 8, 300, 256, 256, true), 3);
    Check("no keys at all", ContiguousDecodeSplits(1, 32, 8, 0, 256, 256, true), 1);
    Check("no batch", ContiguousDecodeSplits(0, 32, 8, 100, 256, 256, true), 1);

    // Paged KV: four waves per slot where one leaves half the CUs idle, and from head_dim 160 on.
    CheckPlan("all lengths 0", 160, std::vector<int64_t>(8, 0), 32, 8, 1, 0);
    CheckPlan("4 x 3000", 128, std::vector<int64_t>(4, 3000), 32, 8, 6, 4);
    CheckPlan("1 x 8000", 128, {8000}, 32, 8, 32, 4);
    CheckPlan("1 x 100", 96, {100}, 32, 8, 1, 4);
    CheckPlan("64 x 8448 keeps its plan", 128, std::vector<int64_t>(64, 8448), 32, 8, 2, 1);
    CheckPlan("D 160, 64 x 4000", 160, std::vector<int64_t>(64, 4000), 32, 8, 2, 1);
    CheckPlan("D 256, half a slot per CU", 256, std::vector<int64_t>(16, 16384), 32, 8, 4, 4);
    CheckPlan("D 160, two slots per CU, ragged", 160, [] {
        std::vector<int64_t> v(64, 1000);
        v[5] = 4000;
        return v;
    }(), 32, 8, 1, 4);
    CheckPlan("D 256, below", 256, std::vector<int64_t>(4, 9000), 64, 16, 4, 4);
    CheckPlan("3 x 511", 128, std::vector<int64_t>(3, 511), 16, 16, 1, 4);
    CheckPlan("D 192, 300 keys", 192, {300, 5}, 32, 8, 1, 4);
    CheckPlan("D 192, 400 keys", 192, {400, 5}, 32, 8, 4, 4);
    CheckPlan("D 160, 153 x 108: one wave", 160, std::vector<int64_t>(153, 108), 32, 8, 1, 1);
    CheckPlan("D 160, 40 x 300", 160, std::vector<int64_t>(40, 300), 32, 8, 2, 1);
    CheckPlan("D 192, 150 short ragged", 192, [] {
        std::vector<int64_t> v(150, 60);
        v[3] = 512;
        return v;
    }(), 32, 8, 1, 1);
    CheckPlan("D 192, one past", 192, [] {
        std::vector<int64_t> v(150, 60);
        v[3] = 513;
        return v;
    }(), 32, 8, 1, 4);
    CheckPlan("D 160, 31 x 300: too few", 160, std::vector<int64_t>(31, 300), 32, 8, 1, 4);

    // Small groups over paged KV: the VALU kernel's own splits.
    const auto valu = [](int64_t d, int64_t n, int64_t len, int64_t heads, int64_t kv, int64_t first) {
        std::vector<int64_t> v(static_cast<size_t>(n), len);
        v[0] = first;
        return PagedValuSplits(d, v.data(), n, heads, kv, 256);
    };
    Check("group 1, D 96", PagedValuGroup(96, 1), 1);
    Check("group 1, D 32", PagedValuGroup(32, 1), 0);
    Check("group 1, D 128", PagedValuGroup(128, 1), 0);
    Check("group 2, D 96", PagedValuGroup(96, 2), 0);
    Check("group 2, D 160", PagedValuGroup(160, 2), 1);
    Check("group 3, D 256", PagedValuGroup(256, 3), 0);
    Check("153 x 108", valu(96, 153, 108, 16, 16, 108), 1);
    Check("64 x 1000, D 96", valu(96, 64, 1000, 16, 16, 1000), 7);
    Check("64 x 1000, D 192", valu(192, 64, 1000, 16, 16, 1000), 1);
    Check("64 x 511", valu(96, 64, 511, 16, 16, 511), 1);
    Check("40 x 300", valu(96, 40, 300, 16, 16, 300), 1);
    Check("two heads, 64 x 1000, D 160", valu(160, 64, 1000, 16, 8, 1000), 2);
    Check("two heads, 64 x 1000, D 192", valu(192, 64, 1000, 16, 8, 1000), 1);
    Check("two heads, 63 x 1000, D 192", valu(192, 63, 1000, 16, 8, 1000), 3);
    Check("ragged", valu(256, 64, 500, 16, 16, 4000), 8);
    Check("four workgroups per CU", valu(160, 32, 2000, 16, 8, 2000), 4);
    Check("one short sequence", valu(256, 1, 100, 8, 8, 100), 1);
    Check("no keys", valu(256, 4, 0, 8, 8, 0), 1);
    if (failures == 0) std::printf("decode rules: ok\n");
    return failures == 0 ? 0 : 1;
}
