// ============================================================================================
// Wide-row kernel (head_dim 32, 64, 96, 128 and 160): one wave per SIMD and 64 query rows per wave.
//
// Why: the fragment reads from LDS are what bounds the 32-row kernels. Every K fragment (32 keys x
// 16 dims) and every V^T fragment feeds one MFMA per 32 query rows a wave holds, and the
// transposed V reads stream at about half the rate of ds_read_b128. With 64 rows per wave each
// fragment feeds two MFMAs, which halves the LDS bytes per FLOP. 64 rows need about 220 VGPRs
// plus 64 (D = 64) to 160 (D = 160) accumulator registers for O and half as many for Q, which only
// one wave per SIMD has (two up to D = 64); that wave then has to overlap its own VALU work with
// its MFMAs. It does when O lives in AGPRs and the instruction stream alternates one MFMA with a
// few VALU instructions, so the step below is written in an explicit order: every MFMA, fragment
// read and wait is an inline asm statement, the C++ VALU code between them is fenced with
// sched_barrier, and the data hazards the compiler cannot see are covered by waits stated at each
// use (see the step). D = 160 fills the register file (240 AGPRs) and the LDS (160 KB).
//
// Workgroup: 4 waves = 2 row groups (64 rows each, two 32-row subtiles) x 2 key halves (32 keys
// of every 64-key tile); K and V tiles come by buffer->LDS DMA into rings of four slots each,
// three tiles ahead. The two key halves of a row group are merged through LDS at the end.
//
// Measured (MI355X, 2 x 16 heads x 4096 keys) against the register-staged kernel that served these
// head dims before: D = 160 causal 398 -> 173 us (432 -> 996 TF/s), non-causal 723 -> 333 us (1,032);
// D = 96 causal 175 -> 122 us (847), non-causal 315 -> 221 us (932); D = 32 causal 78 -> 57 us,
// non-causal 141 -> 102 us (672: the softmax VALU bounds it, at 4 MFMAs per 48 VALU operations).
//
// With one workgroup per CU (from D = 96 on) its fixed part is not hidden: 8,192 workgroups of one key tile (D = 128)
// took 322 us, 9.2 us each beside the step; with the K/V DMAs ahead of the wait for Q, 32-bit index
// arithmetic, no rescale of the zero O and both key halves sharing the merge and the stores 246 us.
// ============================================================================================

#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "flash_common.hpp"

namespace sca_hip {
namespace {

// kMode: plain, packed varlen, or cut (rows packed and / or keys split: SplitArgs).
enum WideMode { kPlain, kPackedVarlen, kCut };

template <typename E, int D, bool kCausal, WideMode kMode, Denominator kDen>
__global__ __launch_bounds__(WideGeom<D>::THREADS, 1) void flash_fwd_wide_kernel(
    const sca_flash_params p, int num_q_tiles, const VarlenArgs vl, const SplitArgs sp) {
    using G = WideGeom<D>;
    using M = Mfma<E>;
    using A = MfmaAsm<E>;
    using vec8 = typename E::vec8;
    constexpr int BN = G::BN;
    constexpr int BM = G::BM;
    constexpr int RB = G::ROW_BYTES;
    constexpr bool kVarlen = kMode == kPackedVarlen;

    extern __shared__ __align__(16) uint8_t lds8[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid % kWave;
    const int lr = lane & 31;
    const int hh = lane >> 5;
    const int rg = wave & 1;   // row group: rows 64*rg .. +64 of the row tile
    const int kq = wave >> 1;  // key half: keys 32*kq .. +32 of every key tile

    const int pack = kMode == kCut ? sp.pack : 1;
    const int splits = kMode == kCut ? sp.splits : 1;
    int tile_linear, b_, unit;
    XcdOrder(p, static_cast<uint32_t>(p.num_heads) / static_cast<uint32_t>(pack), &tile_linear, &b_,
             &unit);
    int split = 0;
    if (splits > 1) {
        split = tile_linear % splits;
        tile_linear /= splits;
    }
    const int64_t b = b_;
    const int64_t h0 = static_cast<int64_t>(unit) * pack;  // first query head
    const int64_t h_kv =
        static_cast<int>(h0) / (static_cast<int>(p.num_heads) / static_cast<int>(p.num_kv_heads));
    // Causal: longest row tiles first. A packed varlen launch takes the sequence and row tile of
    // work entry tile_linear (the list is longest first); tok_*: the sequence's first token.
    int qt = kCausal ? (num_q_tiles - 1 - tile_linear) : tile_linear;
    int seq_q = static_cast<int>(p.seq_q);
    int seq_kv = static_cast<int>(p.seq_kv);
    int diag = static_cast<int>(p.diagonal);
    int64_t tok_q = 0, tok_kv = 0;
    if constexpr (kVarlen) {
        const int seq = vl.tiles[2 * tile_linear];
        qt = vl.tiles[2 * tile_linear + 1];
        tok_q = vl.cu_q[seq];
        tok_kv = vl.cu_kv[seq];
        seq_q = vl.cu_q[seq + 1] - static_cast<int>(tok_q);
        seq_kv = vl.cu_kv[seq + 1] - static_cast<int>(tok_kv);
        diag = kCausal ? seq_kv - seq_q : 0;
    }
    const float scale2 = p.scale * kLog2e;
    const float inv_scale2 = 1.0f / scale2;
    const int q0 = qt * BM;
    // This lane's rows (subtile 0, subtile 1): query position and head offset within the unit.
    int qi[G::RT], hl[G::RT];
#pragma unroll
    for (int r = 0; r < G::RT; ++r) {
        qi[r] = q0 + 64 * rg + 32 * r + lr;
        hl[r] = 0;
        if (pack > 1) {
            const int row = qi[r];
            qi[r] = static_cast<int>(static_cast<uint32_t>(row) / static_cast<uint32_t>(pack));
            hl[r] = row - qi[r] * pack;
        }
    }

    int n_tiles = (seq_kv + BN - 1) / BN;
    int n_plain = seq_kv / BN;
    if (kCausal) {
        const int q_first = pack > 1 ? q0 / pack : q0;
        const int q_last = pack > 1 ? (q0 + BM - 1) / pack : q0 + BM - 1;
        const int last_key = q_last + diag;
        const int causal_tiles = last_key < 0 ? 0 : last_key / BN + 1;
        if (causal_tiles < n_tiles) n_tiles = causal_tiles;
        const int plain = (q_first + diag + 1) / BN;
        if (plain < n_plain) n_plain = plain;
    }
    if (n_plain > n_tiles) n_plain = n_tiles;
    if (splits > 1) {
        // Key tiles [first, first + count): the keys, the causal diagonal and K/V start there.
        int first, count;
        SplitRange(n_tiles, splits, split, &first, &count);
        if (count == 0) {  // fewer key tiles than splits: a state that the merge skips
            if (hh == 0) {
                const int r = kq;  // each of the two waves of a row group covers one subtile
                const int q = r == 0 ? qi[0] : qi[1];
                const int64_t row = (b * p.num_heads + h0 + (r == 0 ? hl[0] : hl[1])) * seq_q + q;
                if (q < seq_q) {
                    float* ml = sp.part_ml + 2 * (split * p.batch * p.num_heads * seq_q + row);
                    ml[0] = neg_inf();
                    ml[1] = 0.0f;
                }
            }
            return;
        }
        tok_kv = static_cast<int64_t>(first) * BN;
        seq_kv = min(seq_kv - first * BN, count * BN);
        diag -= first * BN;
        n_tiles = count;
        n_plain = max(0, min(n_plain - first, count));
    }

    // ---- DMA (buffer resources bounded at the sequence's last row) ----
    const uint8_t* k_bytes = reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.k) + b * p.k_sb + h_kv * p.k_sh + tok_kv * p.k_ss);
    const uint8_t* v_bytes = reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.v) + b * p.v_sb + h_kv * p.v_sh + tok_kv * p.v_ss);
    const int k_row_bytes = static_cast<int>(p.k_ss) * 2;
    const int v_row_bytes = static_cast<int>(p.v_ss) * 2;
    const int k_records = (seq_kv - 1) * k_row_bytes + RB;
    const int v_records = (seq_kv - 1) * v_row_bytes + RB;
    uint32_t dma_koff[G::IPW], dma_voff[G::IPW];
#pragma unroll
    for (int i = 0; i < G::IPW; ++i) {
        const int P = (wave * G::IPW + i) * kWave + lane;
        const int row = P / G::CPR;
        const int pos = P % G::CPR;
        dma_koff[i] = row * k_row_bytes + (pos ^ SwzK<D>(row)) * 16;
        dma_voff[i] = row * v_row_bytes + (pos ^ SwzV<D>(row)) * 16;
    }
    auto issue_k = [&](int slot, int t) __attribute__((always_inline)) {
        uint8_t* dst = lds8 + slot * G::TILE_BYTES + wave * G::IPW * 1024;
        const uint32_t off = static_cast<uint32_t>(t * BN * k_row_bytes);
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) DmaToLds(k_bytes, k_records, dst + i * 1024, dma_koff[i], off);
    };
    auto issue_v = [&](int slot, int t) __attribute__((always_inline)) {
        uint8_t* dst = lds8 + G::V_BASE + slot * G::TILE_BYTES + wave * G::IPW * 1024;
        const uint32_t off = static_cast<uint32_t>(t * BN * v_row_bytes);
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) DmaToLds(v_bytes, v_records, dst + i * 1024, dma_voff[i], off);
    };
    // DMA instruction n (of 2*IPW: K's then V's) of the step that fetches K(t + 1) and V(t).
    auto issue_one = [&](int n, int k_slot, int v_slot, int t_k, int t_v) __attribute__((always_inline)) {
        if (n < G::IPW) {
            uint8_t* dst = lds8 + k_slot * G::TILE_BYTES + wave * G::IPW * 1024;
            DmaToLds(k_bytes, k_records, dst + n * 1024, dma_koff[n],
                     static_cast<uint32_t>(t_k * BN * k_row_bytes));
        } else {
            const int i = n - G::IPW;
            uint8_t* dst = lds8 + G::V_BASE + v_slot * G::TILE_BYTES + wave * G::IPW * 1024;
            DmaToLds(v_bytes, v_records, dst + i * 1024, dma_voff[i],
                     static_cast<uint32_t>(t_v * BN * v_row_bytes));
        }
    };

    // ---- fragment addresses (LDS byte addresses of slot 0; slots are immediate offsets) ----
    const uint32_t lds_base = LdsAddr(lds8);
    const int k_row = 32 * kq + lr;
    constexpr int KP = KPeriod<D>(), VP = VPeriod<D>();
    uint32_t k_addr[KP];
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) {
        k_addr[ks] = lds_base + k_row * RB + (((2 * ks) ^ hh ^ SwzK<D>(k_row)) * 16);
    }
    const int grp = lane >> 4;
    const int sl = lane & 15;
    const int v_key = 32 * kq + 4 * hh + (sl >> 2);
    const int v_chunk = 2 * (grp & 1) + ((sl & 3) >> 1);
    const int v_half = (sl & 1) * 8;
    uint32_t v_addr[VP];
#pragma unroll
    for (int dt = 0; dt < VP; ++dt) {
        v_addr[dt] = lds_base + G::V_BASE + v_key * RB +
                     (((4 * dt + v_chunk) ^ SwzV<D>(v_key)) * 16) + v_half;
    }
    uint32_t v_addr_hi[G::V_SPLIT ? VP : 1];  // slots 2 and 3
    if constexpr (G::V_SPLIT) {
#pragma unroll
        for (int dt = 0; dt < VP; ++dt) v_addr_hi[dt] = v_addr[dt] + 2 * G::TILE_BYTES;
    }

    floatx16 o[G::RT][G::DT];
#pragma unroll
    for (int r = 0; r < G::RT; ++r) {
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[r][dt][i] = 0.0f;
            PinAgpr(o[r][dt]);
        }
    }
    // Row state (RowState); the denominator is summed in two halves (rs.l and l2), which keeps
    // the two dependency chains of its additions apart. lw: the rounded weights' sum beside the
    // unrounded one (kRoundedAndUnrounded).
    RowState rs[G::RT];
    float l2[G::RT];
    float lw[G::RT];
#pragma unroll
    for (int r = 0; r < G::RT; ++r) {
        ResetRow(rs[r]);
        l2[r] = 0.0f;
        lw[r] = 0.0f;
    }

    // K fragments of the next key tile, and two V^T fragment buffers (tile parity).
    vec8 kf[G::KS];
    vec8 va[2][2 * G::DT];
    auto read_k1 = [&]<int SLOT, int ks>() __attribute__((always_inline)) {
        ReadB128Asm<SLOT * G::TILE_BYTES + (ks / KP) * KP * 32>(kf[ks], k_addr[ks % KP]);
    };
    // Transposed V read i (of 4*DT) of the V tile in slot SLOT into buffer VB.
    auto read_v1 = [&]<int SLOT, int VB, int i>() __attribute__((always_inline)) {
        constexpr int dt = i / 4;
        constexpr int part = i % 4;
        constexpr bool kHi = G::V_SPLIT && SLOT >= 2;
        constexpr int kOff = (kHi ? SLOT - 2 : SLOT) * G::TILE_BYTES + (dt / VP) * VP * 64 + part * 8 * RB;
        const uint2 r = TrReadAsm<kOff>(kHi ? v_addr_hi[kHi ? dt % VP : 0] : v_addr[dt % VP]);
        // fragment 2*dt + ps holds (rows 16*ps, 16*ps + 8) of the lane's V column
        uint4 w = __builtin_bit_cast(uint4, va[VB][2 * dt + part / 2]);
        if constexpr (part % 2 == 0) {
            w.x = r.x;
            w.y = r.y;
        } else {
            w.z = r.x;
            w.w = r.y;
        }
        va[VB][2 * dt + part / 2] = __builtin_bit_cast(vec8, w);
    };

    // Masking of S^T subtile r of key tile t (uniform `masked`), and the lane's local maximum.
    auto mask_max = [&](floatx16& sr, int r, int t, bool masked) __attribute__((always_inline)) -> float {
        if (masked) {
            const int kbase = t * BN + 32 * kq + 4 * hh;
            const int lim = kCausal ? min(seq_kv - 1, qi[r] + diag) : seq_kv - 1;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = kbase + 8 * (i / 4) + (i % 4);
                sr[i] = key > lim ? neg_inf() : sr[i];
            }
        }
        return Max16(sr);
    };
    // The rare rescale of both subtiles for a new key tile with raw lane maxima lm (RowState).
    auto rescale_if_grown = [&](float lm0, float lm1) __attribute__((always_inline)) {
        if (__builtin_amdgcn_ballot_w64((lm0 > rs[0].thr) || (lm1 > rs[1].thr)) == 0) return;
        SettleO(o);
        const float lmv[2] = {lm0, lm1};
#pragma unroll
        for (int r = 0; r < G::RT; ++r) {
            const float cmax = HalfMax(lmv[r]) * scale2;  // row maximum, log2 units
            const bool grow = cmax > rs[r].m + kRescaleSlack;
            const float m_new = grow ? cmax : rs[r].m;
            const float alpha = grow ? fast_exp2(rs[r].m - m_new) : 1.0f;  // 0 when m was -inf
            rs[r].m = m_new;
            rs[r].l *= alpha;
            l2[r] *= alpha;
            if constexpr (kDen == kRoundedAndUnrounded) lw[r] *= alpha;
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
                Fence();  // one O tile at a time through VGPRs
#pragma unroll
                for (int i = 0; i < 16; ++i) o[r][dt][i] *= alpha;
                PinAgpr(o[r][dt]);
            }
            Fence();
            rs[r].thr = (m_new + kRescaleSlack) * inv_scale2;
            rs[r].neg_mu = (m_new == neg_inf()) ? 0.0f : -m_new;
        }
        asm volatile("s_nop 4");
    };

    // ---- prologue: K(0..3), V(0..2) in flight; S(0), its maxima and rescale; K(1) and V(0)
    //      fragments read for step 0; K(2) and V(1) landed before step 0 ----
    issue_k(0, 0);
    // Q fragments (B operand of S^T = K Q^T): subtile r, k-step ks. Rows past seq_q repeat the last
    // one (their results are not stored). Requested behind K(0) and pinned only after the other
    // tiles' DMAs are issued, so that nothing waits for them but the first QK.
    vec8 qf[G::RT][G::KS];
#pragma unroll
    for (int r = 0; r < G::RT; ++r) {
        const int row = min(qi[r], seq_q - 1);
        const uint16_t* q_row = static_cast<const uint16_t*>(p.q) + b * p.q_sb +
                                (h0 + hl[r]) * p.q_sh + (tok_q + row) * p.q_ss + 8 * hh;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            qf[r][ks] = __builtin_bit_cast(vec8, *reinterpret_cast<const uint4*>(q_row + 16 * ks));
        }
    }
    issue_k(1, 1);
    issue_v(0, 0);
    issue_k(2, 2);
    issue_v(1, 1);
    issue_k(3, 3);
    issue_v(2, 2);
#pragma unroll
    for (int r = 0; r < G::RT; ++r) {
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) PinAgpr(qf[r][ks]);
    }
    WaitVm<4 * G::IPW>();  // K(0), K(1), V(0)
    __builtin_amdgcn_s_barrier();
    floatx16 s0[G::RT], s1[G::RT];
    StaticFor<G::KS>([&](auto ks) { read_k1.template operator()<0, ks>(); });
    WaitLgkmTied<0>(kf[0]);
#pragma unroll
    for (int ks = 1; ks < G::KS; ++ks) WaitLgkmTied<0>(kf[ks]);
#pragma unroll
    for (int r = 0; r < G::RT; ++r) {
        A::first_v(s0[r], kf[0], qf[r][0]);
#pragma unroll
        for (int ks = 1; ks < G::KS; ++ks) A::acc_v(s0[r], kf[ks], qf[r][ks]);
    }
    asm volatile("s_nop 15\n\ts_nop 15");  // the QK results are complete; kf has been read
    {
        // The first maxima; O and l are zero, so nothing is rescaled.
#pragma unroll
        for (int r = 0; r < G::RT; ++r) {
            rs[r].m = HalfMax(mask_max(s0[r], r, 0, n_plain == 0)) * scale2;
            rs[r].thr = (rs[r].m + kRescaleSlack) * inv_scale2;
            rs[r].neg_mu = (rs[r].m == neg_inf()) ? 0.0f : -rs[r].m;
        }
    }
    StaticFor<G::KS>([&](auto ks) { read_k1.template operator()<1, ks>(); });
    StaticFor<4 * G::DT>([&](auto i) { read_v1.template operator()<0, 0, i>(); });
    WaitVm<2 * G::IPW>();  // K(2), V(1)
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();

    // One step for key tile j (S = j & 3, VB = j & 1). On entry S(j) is masked and the rescale
    // for tile j is done, kf holds K(j+1)'s fragments and va[VB] V(j)'s. Four regions, each one
    // MFMA stream with VALU and LDS work placed between its MFMAs:
    //   A  QK(j+1) of subtile 0          | the 8 exponential pairs of S(j) subtile 0
    //   B  PV(j) of subtile 0            | exponential pairs 0-3 of subtile 1, V(j+1)'s reads
    //   C  QK(j+1) of subtile 1          | exponential pairs 4-7 of subtile 1, S(j+1) subtile 0's
    //                                      masking and maximum
    //   D  PV(j) of subtile 1            | S(j+1) subtile 1's masking and maximum, K(j+2)'s
    //                                      fragment reads, the DMAs of K(j+4) and V(j+3)
    // then the rare rescale for tile j+1, the DMA wait (K(j+3) and V(j+2) must land: only the
    // two groups issued in this step stay in flight) and the barrier. Hazards the compiler
    // does not see (inline-asm MFMAs): a QK result is read by VALU only after at least two
    // later MFMAs and 5 wait states; kf is rewritten only after two later MFMAs; the O
    // accumulators are read by VALU only through SettleO; P operands are written by VALU at
    // least a region before their MFMAs.
    auto step = [&]<bool kMaskable, int S>(int j, floatx16 (&s_in)[G::RT],
                                           floatx16 (&s_out)[G::RT]) __attribute__((always_inline)) {
        constexpr int VB = S & 1;
        constexpr int NPV = 2 * G::DT;  // PV MFMAs per subtile
        constexpr int kOps = SoftmaxOps(kDen);  // of each subtile
        // S(j+1) is a real tile. With little register room (D = 160) the QK of a tile past the
        // end runs too (its scores are all masked): merging "computed" and "not computed" scores
        // would make the compiler copy MFMA results it does not know to be in flight.
        const bool next_ok = !kMaskable || D > 128 || j + 1 < n_tiles;
        const bool next_masked = kMaskable && j + 1 >= n_plain;
        uint32_t pw[G::RT][8];
        // The VALU operations that turn S(j) subtile r into P, in place (SoftmaxOp); op(r, n) runs
        // the n-th. (Unrounded sums use v_add: a v_dot2 issued between MFMAs does not overlap with
        // them.)
        auto op = [&](int r, int n) __attribute__((always_inline)) {
            const int c = SoftmaxOp(kDen, n);
            if (c < 16) {
                s_in[r][c] = fmaf(s_in[r][c], scale2, rs[r].neg_mu);
            } else if (c < 32) {
                s_in[r][c - 16] = fast_exp2(s_in[r][c - 16]);
            } else if (c < 40) {
                pw[r][c - 32] = M::pack(s_in[r][2 * (c - 32)], s_in[r][2 * (c - 32) + 1]);
            } else if (c >= 56) {
                float& sum = kDen == kRoundedAndUnrounded ? lw[r] : c % 2 == 0 ? rs[r].l : l2[r];
                sum = M::sum2(pw[r][c - 56], sum);
            } else if (c % 2 == 0) {
                rs[r].l += s_in[r][c - 40];
            } else {
                l2[r] += s_in[r][c - 40];
            }
        };
        auto qk = [&](int r, int ks) __attribute__((always_inline)) {
            if (!next_ok) return;  // the last tile has no S(j+1)
            if (ks == 0) {
                A::first_v(s_out[r], kf[0], qf[r][0]);
            } else {
                A::acc_v(s_out[r], kf[ks], qf[r][ks]);
            }
        };
        vec8 pb[G::RT][2];
        auto pack_p = [&](int r) __attribute__((always_inline)) {
            pb[r][0] = __builtin_bit_cast(vec8, make_uint4(pw[r][0], pw[r][1], pw[r][2], pw[r][3]));
            pb[r][1] = __builtin_bit_cast(vec8, make_uint4(pw[r][4], pw[r][5], pw[r][6], pw[r][7]));
        };
        auto pv = [&](int r, int i) __attribute__((always_inline)) {
            A::acc_a(o[r][i / 2], va[VB][i], pb[r][i % 2]);
        };
        // The step's 2*IPW DMA instructions (K(j+4) into K slot S, V(j+3) into V slot S-1),
        // spread over the four regions: in region g, after MFMA i, instruction number
        // g*kDmaPerRegion + i / kDmaSpacing when i is a multiple of kDmaSpacing.
        constexpr int kDmaPerRegion = (2 * G::IPW + 3) / 4;
        auto dma = [&](int g, int i) __attribute__((always_inline)) {
            constexpr int kSpacing = 8 / kDmaPerRegion > 0 ? 8 / kDmaPerRegion : 1;
            if (i % kSpacing != 0) return;
            const int n = g * kDmaPerRegion + i / kSpacing;
            if (n >= 2 * G::IPW || i / kSpacing >= kDmaPerRegion) return;
            const bool is_k = n < G::IPW;
            if (kMaskable && (is_k ? j + 4 >= n_tiles : j + 3 >= n_tiles)) return;
            issue_one(n, S, (S + 3) & 3, j + 4, j + 3);
        };

        // ---- A ----
        constexpr int kOpsA = (kOps + G::KS - 1) / G::KS;  // VALU operations per QK MFMA
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            qk(0, ks);
            Fence();
#pragma unroll
            for (int q = 0; q < kOpsA; ++q) {
                if (ks * kOpsA + q < kOps) op(0, ks * kOpsA + q);
            }
            dma(0, ks);
            Fence();
        }
        pack_p(0);
        // P operands: 2 wait states after their VALU writes (the compiler does not see the
        // inline-asm MFMA that reads them).
        asm volatile("s_nop 1" : "+v"(pb[0][0]), "+v"(pb[0][1]));
        // ---- B ----
        constexpr int kVReadsB = 4 * G::DT / NPV;  // V reads per PV MFMA
        constexpr int kOpsB = (kOps / 2 + NPV - 1) / NPV;  // subtile 1's operations, first half
        StaticFor<NPV>([&](auto i) __attribute__((always_inline)) {
            pv(0, i);
            Fence();
#pragma unroll
            for (int q = 0; q < kOpsB; ++q) {
                if (i * kOpsB + q < kOps / 2) op(1, i * kOpsB + q);
            }
            dma(1, i);
            StaticFor<kVReadsB>([&](auto q) __attribute__((always_inline)) {
                read_v1.template operator()<(S + 1) & 3, VB ^ 1, i * kVReadsB + q>();
            });
            Fence();
        });
        // ---- C ----
        float lm0 = neg_inf(), lm1 = neg_inf();
        constexpr int kOpsC = (kOps / 2 + G::KS - 1) / G::KS;  // and second half
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            qk(1, ks);
            Fence();
#pragma unroll
            for (int q = 0; q < kOpsC; ++q) {
                if (ks * kOpsC + q < kOps / 2) op(1, kOps / 2 + ks * kOpsC + q);
            }
            dma(2, ks);
            if (ks == G::KS / 2) {
                if (next_ok) lm0 = mask_max(s_out[0], 0, j + 1, next_masked);
            }
            Fence();
        }
        pack_p(1);
        // P operands: 2 wait states after their VALU writes.
        asm volatile("s_nop 1" : "+v"(pb[1][0]), "+v"(pb[1][1]));
        // ---- D ----
        StaticFor<NPV>([&](auto i) __attribute__((always_inline)) {
            pv(1, i);
            Fence();
            if constexpr (i == 1) {
                asm volatile("s_nop 4");
                if (next_ok) lm1 = mask_max(s_out[1], 1, j + 1, next_masked);
            }
            if constexpr (i >= 1) {
                // KS K reads over the MFMAs 1 .. NPV-1 (kf was last read two MFMAs ago).
                constexpr int kPer = (G::KS + NPV - 2) / (NPV - 1);
                StaticFor<kPer>([&](auto q) __attribute__((always_inline)) {
                    constexpr int ks = (i - 1) * kPer + q;
                    if constexpr (ks < G::KS) read_k1.template operator()<(S + 2) & 3, ks>();
                });
            }
            dma(3, i);
            Fence();
        });
        // ---- rare rescale for tile j+1 ----
        if (next_ok) rescale_if_grown(lm0, lm1);
        Fence();
        // ---- K(j+3) and V(j+2) landed (at the tail, everything); fragment reads retired ----
        if (!kMaskable || j + 4 < n_tiles) {
            WaitVm<2 * G::IPW>();
        } else {
            WaitVm<0>();
        }
        WaitLgkmTied<0>(kf[G::KS - 1]);
        __builtin_amdgcn_s_barrier();
    };

    int j = 0;
    // Steady state: plain tiles with the full ring ahead, four steps per trip.
    for (; j + 5 <= n_plain && j + 8 <= n_tiles; j += 4) {
        step.template operator()<false, 0>(j, s0, s1);
        step.template operator()<false, 1>(j + 1, s1, s0);
        step.template operator()<false, 2>(j + 2, s0, s1);
        step.template operator()<false, 3>(j + 3, s1, s0);
    }
    // Tail (j is a multiple of 4 here): masked steps, same slot rotation.
    for (; j < n_tiles; j += 4) {
        step.template operator()<true, 0>(j, s0, s1);
        if (j + 1 >= n_tiles) break;
        step.template operator()<true, 1>(j + 1, s1, s0);
        if (j + 2 >= n_tiles) break;
        step.template operator()<true, 2>(j + 2, s0, s1);
        if (j + 3 >= n_tiles) break;
        step.template operator()<true, 3>(j + 3, s1, s0);
    }

    // ---- epilogue: merge the key halves of each row group, normalise, store ----
    WaitVm<0>();
    SettleO(o);
    __builtin_amdgcn_s_barrier();
    // Wave kq finishes subtile kq: it hands its O and (m, denominators) of the other subtile to its
    // partner, as quads (quad k of lane L at k*64 + L: conflict-free 16-byte accesses).
    constexpr bool kBoth = kDen == kRoundedAndUnrounded;
    auto region = [&](int w) { return reinterpret_cast<float*>(lds8) + w * kWave * G::MERGE_FLOATS; };
    auto hand_over = [&]<int R>() __attribute__((always_inline)) {
        float4* q4 = reinterpret_cast<float4*>(region(wave)) + lane;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                q4[(dt * 4 + g) * kWave] = make_float4(o[R][dt][4 * g], o[R][dt][4 * g + 1],
                                                       o[R][dt][4 * g + 2], o[R][dt][4 * g + 3]);
            }
        }
        const float l = rs[R].l + l2[R];
        float* st = region(wave) + G::DT * 16 * kWave;
        reinterpret_cast<float2*>(st)[lane] = make_float2(rs[R].m, kBoth ? lw[R] : l);
        if constexpr (kBoth) st[2 * kWave + lane] = l;
    };
    auto finish = [&]<int R>() __attribute__((always_inline)) {
        const float* from = region(wave ^ 2);
        const float4* q4 = reinterpret_cast<const float4*>(from) + lane;
        const float2 other = reinterpret_cast<const float2*>(from + G::DT * 16 * kWave)[lane];
        const float mm = fmaxf(rs[R].m, other.x);
        float w0 = (rs[R].m == neg_inf()) ? 0.0f : fast_exp2(rs[R].m - mm);
        float w1 = (other.x == neg_inf()) ? 0.0f : fast_exp2(other.x - mm);
        const float l = rs[R].l + l2[R];
        const float l_tot = HalfSum((kBoth ? lw[R] : l) * w0) + HalfSum(other.y * w1);
        float l_lse = l_tot;
        if constexpr (kBoth) {
            l_lse = HalfSum(l * w0) + HalfSum(from[(G::DT * 16 + 2) * kWave + lane] * w1);
        }
        const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        const int row = qi[R];
        const bool row_ok = row < seq_q;
        const int64_t h = h0 + hl[R];
        const int64_t flat = (b * p.num_heads + h) * seq_q + row;  // not used by varlen launches
        if (splits > 1) {
            if constexpr (kBoth) {  // one denominator for the merge: O to the scale of the unrounded one
                const float c = l_tot > 0.0f ? l_lse / l_tot : 0.0f;
                w0 *= c;
                w1 *= c;
            }
            const int64_t at = split * p.batch * p.num_heads * seq_q + flat;
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
                float a[16];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 v = q4[(dt * 4 + g) * kWave];
                    a[4 * g] = o[R][dt][4 * g] * w0 + v.x * w1;
                    a[4 * g + 1] = o[R][dt][4 * g + 1] * w0 + v.y * w1;
                    a[4 * g + 2] = o[R][dt][4 * g + 2] * w0 + v.z * w1;
                    a[4 * g + 3] = o[R][dt][4 * g + 3] * w0 + v.w * w1;
                }
                StorePartialTile(sp.part_o + at * D + 32 * dt, hh, row_ok, a);
            }
            if (row_ok && hh == 0) {
                *reinterpret_cast<float2*>(sp.part_ml + 2 * at) = make_float2(mm, l_lse);
            }
            return;
        }
        uint16_t* out_row = static_cast<uint16_t*>(p.out) + b * p.o_sb + h * p.o_sh +
                            (tok_q + row) * p.o_ss;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
            float a[16];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 v = q4[(dt * 4 + g) * kWave];
                a[4 * g] = (o[R][dt][4 * g] * w0 + v.x * w1) * inv;
                a[4 * g + 1] = (o[R][dt][4 * g + 1] * w0 + v.y * w1) * inv;
                a[4 * g + 2] = (o[R][dt][4 * g + 2] * w0 + v.z * w1) * inv;
                a[4 * g + 3] = (o[R][dt][4 * g + 3] * w0 + v.w * w1) * inv;
            }
            StoreTile<M>(out_row + 32 * dt, hh, row_ok, a);
        }
        if (row_ok && p.lse != nullptr && hh == 0) {
            p.lse[flat] = l_lse > 0.0f ? (mm + __log2f(l_lse)) * kLn2 : neg_inf();
        }
    };
    if (kq == 0) {
        hand_over.template operator()<1>();
    } else {
        hand_over.template operator()<0>();
    }
    __syncthreads();
    if (kq == 0) {
        finish.template operator()<0>();
    } else {
        finish.template operator()<1>();
    }
}

}  // namespace

template <typename E, int D, bool kCausal>
int LaunchFlashWide(const sca_flash_params& p, const SplitArgs& sp, hipStream_t s) {
    using G = WideGeom<D>;
    const int64_t num_q_tiles = (p.seq_q * sp.pack + G::BM - 1) / G::BM;
    const int64_t blocks = num_q_tiles * p.batch * (p.num_heads / sp.pack) * sp.splits;
    if (blocks <= 0) return 0;
    if (blocks > 0x7fffffffLL) {
        return SetError(SCA_E_SEQ_TOO_LONG, "flash: grid of " + std::to_string(blocks) +
                                                " workgroups exceeds the launch limit");
    }
    auto launch = [&]<WideMode kMode, Denominator kDen>() -> int {
        if (const int rc = EnsureLdsLimit<&flash_fwd_wide_kernel<E, D, kCausal, kMode, kDen>>(
                G::LDS_BYTES, "flash LDS limit")) {
            return rc;
        }
        hipLaunchKernelGGL((flash_fwd_wide_kernel<E, D, kCausal, kMode, kDen>),
                           dim3(static_cast<unsigned>(blocks)), dim3(G::THREADS), G::LDS_BYTES, s, p,
                           static_cast<int>(num_q_tiles), VarlenArgs{nullptr, nullptr, nullptr}, sp);
        return CheckLaunch("flash_fwd_wide_kernel", s);
    };
    const bool cut = sp.pack != 1 || sp.splits != 1;
    if (p.lse != nullptr) {
        constexpr Denominator kDen = DenominatorFor<D>(true);
        return cut ? launch.template operator()<kCut, kDen>() : launch.template operator()<kPlain, kDen>();
    }
    constexpr Denominator kDen = DenominatorFor<D>(false);
    return cut ? launch.template operator()<kCut, kDen>() : launch.template operator()<kPlain, kDen>();
}

// One launch over a packed batch: the wide kernel, one workgroup per (work entry, head).
template <typename E, int D, bool kCausal>
int LaunchFlashVarlen(const sca_flash_varlen_params& v, hipStream_t s) {
    using G = WideGeom<D>;
    static_assert(G::BM == 128, "the work list's row tiles are 128 rows");
    static_assert(DenominatorFor<D>(false) == kUnrounded);
    // 32-bit buffer offsets: a sequence's rows plus the wide kernel's ring overrun must fit.
    const int64_t rows_k = v.max_seq_kv + 8 * G::BN;
    if (rows_k * v.k_ss * 2 >= (1LL << 31) || rows_k * v.v_ss * 2 >= (1LL << 31)) {
        return SetError(SCA_E_SEQ_TOO_LONG, "flash varlen: a sequence of " +
                                                std::to_string(v.max_seq_kv) +
                                                " keys exceeds the 32-bit tile offsets");
    }
    const int64_t blocks = v.num_tiles * v.num_heads;
    if (blocks <= 0) return 0;
    if (blocks > 0x7fffffffLL) {
        return SetError(SCA_E_SEQ_TOO_LONG, "flash varlen: grid too large");
    }
    sca_flash_params p{};
    p.q = v.q;
    p.k = v.k;
    p.v = v.v;
    p.out = v.out;
    p.lse = nullptr;
    p.batch = 1;
    p.num_heads = v.num_heads;
    p.num_kv_heads = v.num_kv_heads;
    p.head_dim = v.head_dim;
    p.q_sh = v.q_sh, p.q_ss = v.q_ss;
    p.k_sh = v.k_sh, p.k_ss = v.k_ss;
    p.v_sh = v.v_sh, p.v_ss = v.v_ss;
    p.o_sh = v.o_sh, p.o_ss = v.o_ss;
    p.scale = v.scale;
    p.causal = v.causal;
    p.dtype = v.dtype;
    if (const int rc = EnsureLdsLimit<&flash_fwd_wide_kernel<E, D, kCausal, kPackedVarlen, kUnrounded>>(
            G::LDS_BYTES, "flash LDS limit")) {
        return rc;
    }
    hipLaunchKernelGGL((flash_fwd_wide_kernel<E, D, kCausal, kPackedVarlen, kUnrounded>),
                       dim3(static_cast<unsigned>(blocks)), dim3(G::THREADS), G::LDS_BYTES, s, p,
                       0, VarlenArgs{v.cu_seqlens_q, v.cu_seqlens_kv, v.tiles},
                       SplitArgs{1, 1, nullptr, nullptr});
    return CheckLaunch("flash_fwd_wide_kernel (varlen)", s);
}

}  // namespace sca_hip
