// ============================================================================================
// Split-dims kernel (head_dim 192 and 256): one wave per SIMD, 64 query rows per wave pair.
//
// Why: 64 rows x 256 dims of O and Q are 384 registers a lane, so the wide kernel's wave (64 rows,
// all dims) does not fit, and a wave of 32 rows reads every fragment from LDS for one MFMA, which
// bounds it. Here the two waves of a 64-row group share the rows differently in the two products:
//   QK, softmax: wave dh owns subtile dh (32 rows) and computes its scores for all 32 keys of a
//                tile, so the row state (m, l) stays in one wave;
//   PV:          wave dh owns dims [dh*D/2, +D/2) of all 64 rows, so every transposed V fragment
//                (the slow LDS reads) feeds two MFMAs. Its own subtile's P comes from registers,
//                the partner's through LDS (2 KB per wave and tile).
// O (64 rows x D/2) and Q (32 rows x D) take 192 AGPRs at D = 256.
//
// Pipeline, step t: QK of tile t+2, softmax of tile t+1, PV of tile t, one barrier. A move of the
// running max for tile u is decided by the owner at the end of step u-2, published as 32 factors
// and a flag that holds u, and applied by both waves to O at the end of step u-1 (after PV(u-1)).
// K and V tiles (32 keys) come by buffer->LDS DMA into rings of four slots each; loads past the
// last tile are out of the resource's range and cost no traffic, so every step issues the same
// number and waits on the same count. As in the wide kernel the order inside a step is explicit and
// hazards the compiler cannot see (inline-asm MFMAs and LDS reads) are covered where they arise.
//
// Measured (MI355X) against the register-staged kernel that served these head dims before: D = 256,
// 16 heads x 4096 keys causal 325 -> 139 us (423 -> 992 TF/s), 2 x 16 heads non-causal 1,279 ->
// 504 us (1,090); D = 192, 2 x 16 heads causal 454 -> 220 us (939), non-causal 849 -> 422 (976);
// short sequences too (8 heads x 300 keys, D = 256: 27 -> 16 us).
// ============================================================================================

#include <hip/hip_runtime.h>

#include <string>

#include "flash_common.hpp"

namespace sca_hip {
namespace {

// kCut: rows packed and / or keys split (SplitArgs).
template <typename E, int D, bool kCausal, bool kCut, Denominator kDen>
__global__ __launch_bounds__(DsplitGeom<D>::THREADS, 1) void flash_fwd_dsplit_kernel(
    const sca_flash_params p, int num_q_tiles, const SplitArgs sp) {
    using G = DsplitGeom<D>;
    using M = Mfma<E>;
    using A = MfmaAsm<E>;
    using vec8 = typename E::vec8;
    constexpr int BN = G::BN;
    constexpr int BM = G::BM;
    constexpr int RB = G::ROW_BYTES;

    extern __shared__ __align__(16) uint8_t lds8[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid % kWave;
    const int lr = lane & 31;
    const int hh = lane >> 5;
    const int rg = wave & 1;   // rows 64*rg .. +64 of the row tile
    const int dh = wave >> 1;  // QK: rows 32*dh of those; PV: dims D/2*dh .. +D/2

    const int pack = kCut ? sp.pack : 1;
    const int splits = kCut ? sp.splits : 1;
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
    const int qt = kCausal ? (num_q_tiles - 1 - tile_linear) : tile_linear;
    const int seq_q = static_cast<int>(p.seq_q);
    int seq_kv = static_cast<int>(p.seq_kv);
    int diag = static_cast<int>(p.diagonal);
    const float scale2 = p.scale * kLog2e;
    const float inv_scale2 = 1.0f / scale2;
    const int q0 = qt * BM;
    // This lane's rows, of the owned subtile and of the partner's: query position and head offset
    // within the unit.
    int qi[2], hl[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        qi[r] = q0 + 64 * rg + 32 * (dh ^ r) + lr;
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
    int64_t key0 = 0;
    const int64_t rows_all = p.batch * p.num_heads * seq_q;
    const int64_t flat_own = (b * p.num_heads + h0 + hl[0]) * seq_q + qi[0];
    if (splits > 1) {
        // Key tiles [first, first + count): the keys, the causal diagonal and K/V start there.
        int first, count;
        SplitRange(n_tiles, splits, split, &first, &count);
        if (count == 0) {  // fewer key tiles than splits: a state that the merge skips
            if (hh == 0 && qi[0] < seq_q) {
                float* ml = sp.part_ml + 2 * (split * rows_all + flat_own);
                ml[0] = neg_inf();
                ml[1] = 0.0f;
            }
            return;
        }
        key0 = static_cast<int64_t>(first) * BN;
        seq_kv = min(seq_kv - first * BN, count * BN);
        diag -= first * BN;
        n_tiles = count;
        n_plain = max(0, min(n_plain - first, count));
    }

    // ---- DMA (buffer resources bounded at the last row any row of this tile attends) ----
    const uint8_t* k_bytes = reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.k) + b * p.k_sb + h_kv * p.k_sh + key0 * p.k_ss);
    const uint8_t* v_bytes = reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.v) + b * p.v_sb + h_kv * p.v_sh + key0 * p.v_ss);
    const int k_row_bytes = static_cast<int>(p.k_ss) * 2;
    const int v_row_bytes = static_cast<int>(p.v_ss) * 2;
    const int rows = min(seq_kv, n_tiles * BN);
    const int k_records = (rows - 1) * k_row_bytes + RB;
    const int v_records = (rows - 1) * v_row_bytes + RB;
    uint32_t dma_koff[G::IPW], dma_voff[G::IPW];
#pragma unroll
    for (int i = 0; i < G::IPW; ++i) {
        const int P = (wave * G::IPW + i) * kWave + lane;
        const int row = P / G::CPR;
        const int pos = P % G::CPR;
        dma_koff[i] = row * k_row_bytes + (pos ^ SwzK<D>(row)) * 16;
        dma_voff[i] = row * v_row_bytes + (pos ^ SwzV<D>(row)) * 16;
    }
    // DMA instruction i of this wave's share of K tile t (into K slot t & 3) or V tile t.
    auto dma_k = [&](int i, int slot, int t) __attribute__((always_inline)) {
        DmaToLds(k_bytes, k_records, lds8 + slot * G::TILE_BYTES + (wave * G::IPW + i) * 1024,
                 dma_koff[i], static_cast<uint32_t>(t * BN * k_row_bytes));
    };
    auto dma_v = [&](int i, int slot, int t) __attribute__((always_inline)) {
        DmaToLds(v_bytes, v_records,
                 lds8 + G::V_BASE + slot * G::TILE_BYTES + (wave * G::IPW + i) * 1024, dma_voff[i],
                 static_cast<uint32_t>(t * BN * v_row_bytes));
    };

    // ---- fragment addresses (LDS byte addresses of slot 0; slots are immediate offsets) ----
    const uint32_t lds_base = LdsAddr(lds8);
    constexpr int KP = KPeriod<D>();
    uint32_t k_addr[KP];
#pragma unroll
    for (int ks = 0; ks < KP; ++ks) {
        k_addr[ks] = lds_base + lr * RB + (((2 * ks) ^ hh ^ SwzK<D>(lr)) * 16);
    }
    const int grp = lane >> 4;
    const int sl = lane & 15;
    const int v_key = 4 * hh + (sl >> 2);
    const int v_chunk = 2 * (grp & 1) + ((sl & 3) >> 1);
    const int v_half = (sl & 1) * 8;
    uint32_t v_addr[G::DT];
#pragma unroll
    for (int dt = 0; dt < G::DT; ++dt) {
        v_addr[dt] = lds_base + G::V_BASE + v_key * RB +
                     (((4 * (dh * G::DT + dt) + v_chunk) ^ SwzV<D>(v_key)) * 16) + v_half;
    }
    // P fragments: [parity][wave][k-step][lane] of 16 bytes; own slot to write, partner's to read.
    const uint32_t p_own = lds_base + G::P_BASE + wave * 2048 + lane * 16;
    const uint32_t p_partner = lds_base + G::P_BASE + (wave ^ 2) * 2048 + lane * 16;
    // Rescale factors [parity][wave][32] and flags [parity][row group][dh] (the tile they are for).
    float* const s_alpha = reinterpret_cast<float*>(lds8 + G::ALPHA_BASE);
    int* const s_flag = reinterpret_cast<int*>(lds8 + G::FLAG_BASE);
    const uint32_t flag_addr = lds_base + G::FLAG_BASE + rg * 8;

    floatx16 o[2][G::DT];  // the owned subtile's rows, then the partner's
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[r][dt][i] = 0.0f;
            PinAgpr(o[r][dt]);
        }
    }
    RowState rs;
    float l2 = 0.0f;  // second half of the denominator (two addition chains)
    float lw = 0.0f;  // the rounded weights' sum beside the unrounded one (kRoundedAndUnrounded)
    ResetRow(rs);

    vec8 kf[G::KS];           // K fragments of the next QK
    vec8 va[2][2 * G::DT];    // V^T fragments by tile parity
    auto read_k1 = [&]<int SLOT, int ks>() __attribute__((always_inline)) {
        ReadB128Asm<SLOT * G::TILE_BYTES + (ks / KP) * KP * 32>(kf[ks], k_addr[ks % KP]);
    };
    // Transposed V read i (of 4*DT) of the V tile in slot SLOT into buffer VB.
    auto read_v1 = [&]<int SLOT, int VB, int i>() __attribute__((always_inline)) {
        constexpr int dt = i / 4;
        constexpr int part = i % 4;
        const uint2 r = TrReadAsm<SLOT * G::TILE_BYTES + part * 8 * RB>(v_addr[dt]);
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

    // Masking of the owned scores of key tile t (uniform `masked`), and the lane's maximum.
    auto mask_max = [&](floatx16& sr, int t, bool masked) __attribute__((always_inline)) -> float {
        if (masked) {
            const int kbase = t * BN + 4 * hh;
            const int lim = kCausal ? min(seq_kv - 1, qi[0] + diag) : seq_kv - 1;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = kbase + 8 * (i / 4) + (i % 4);
                sr[i] = key > lim ? neg_inf() : sr[i];
            }
        }
        return Max16(sr);
    };
    // The owner's decision for tile t with raw lane maximum lm; publishes the factors of O.
    auto decide = [&](float lm, int t, int par) __attribute__((always_inline)) {
        if (__builtin_amdgcn_ballot_w64(lm > rs.thr) == 0) return;
        const float cmax = HalfMax(lm) * scale2;  // row maximum, log2 units
        const bool grow = cmax > rs.m + kRescaleSlack;
        const float m_new = grow ? cmax : rs.m;
        const float alpha = grow ? fast_exp2(rs.m - m_new) : 1.0f;  // 0 when m was -inf
        rs.m = m_new;
        rs.l *= alpha;
        l2 *= alpha;
        lw *= alpha;
        rs.thr = (m_new + kRescaleSlack) * inv_scale2;
        rs.neg_mu = (m_new == neg_inf()) ? 0.0f : -m_new;
        if (hh == 0) s_alpha[(par * 4 + rg * 2 + dh) * 32 + lr] = alpha;
        if (lane == 0) s_flag[par * 4 + rg * 2 + dh] = t;
    };
    // O of both subtiles by the factors published for tile t (flags f of subtiles 0 and 1).
    auto apply = [&](uint2 f, int t, int par) __attribute__((always_inline)) {
        const int f0 = __builtin_amdgcn_readfirstlane(static_cast<int>(f.x));
        const int f1 = __builtin_amdgcn_readfirstlane(static_cast<int>(f.y));
        if (f0 != t && f1 != t) return;
        SettleO(o);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int sub = dh ^ r;
            const float published = s_alpha[(par * 4 + rg * 2 + sub) * 32 + lr];
            const float alpha = (sub == 0 ? f0 : f1) == t ? published : 1.0f;
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
                Fence();  // one O tile at a time through VGPRs
#pragma unroll
                for (int i = 0; i < 16; ++i) o[r][dt][i] *= alpha;
                PinAgpr(o[r][dt]);
            }
            Fence();
        }
        asm volatile("s_nop 4");
    };
    // The VALU operations that turn the owned scores into P (SoftmaxOp); op(n, ...) runs the n-th.
    constexpr int kOps = SoftmaxOps(kDen);
    auto op = [&](int n, floatx16& s, uint32_t (&pw)[8]) __attribute__((always_inline)) {
        const int c = SoftmaxOp(kDen, n);
        if (c < 16) {
            s[c] = fmaf(s[c], scale2, rs.neg_mu);
        } else if (c < 32) {
            s[c - 16] = fast_exp2(s[c - 16]);
        } else if (c < 40) {
            pw[c - 32] = M::pack(s[2 * (c - 32)], s[2 * (c - 32) + 1]);
        } else if (c >= 56) {
            float& sum = kDen == kRoundedAndUnrounded ? lw : c % 2 == 0 ? rs.l : l2;
            sum = M::sum2(pw[c - 56], sum);
        } else if (c % 2 == 0) {
            rs.l += s[c - 40];
        } else {
            l2 += s[c - 40];
        }
    };
    auto pack_p = [&](const uint32_t (&pw)[8], vec8 (&pb)[2]) __attribute__((always_inline)) {
        pb[0] = __builtin_bit_cast(vec8, make_uint4(pw[0], pw[1], pw[2], pw[3]));
        pb[1] = __builtin_bit_cast(vec8, make_uint4(pw[4], pw[5], pw[6], pw[7]));
    };
    auto write_p = [&]<int PAR>(const vec8 (&pb)[2]) __attribute__((always_inline)) {
        WriteB128Asm<PAR * 8192>(p_own, pb[0]);
        WriteB128Asm<PAR * 8192 + 1024>(p_own, pb[1]);
    };

    // ---- prologue: S(0) -> P(0), S(1); K(2) and V(0) fragments. Issue order: K(0), K(1), then
    //      (K(t+2), V(t)) as in the steps ----
    auto issue = [&](int t_k, int t_v) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) dma_k(i, t_k & 3, t_k);
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) dma_v(i, t_v & 3, t_v);
    };
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) dma_k(i, t, t);
    }
    // Q fragments of the owned subtile (B operand of S^T = K Q^T). Rows past seq_q repeat the last
    // one (their results are not stored); pinned only after the other tiles' DMAs are issued, so that
    // nothing waits for them but the first QK.
    vec8 qf[G::KS];
    {
        const uint16_t* q_row = static_cast<const uint16_t*>(p.q) + b * p.q_sb +
                                (h0 + hl[0]) * p.q_sh +
                                static_cast<int64_t>(min(qi[0], seq_q - 1)) * p.q_ss + 8 * hh;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            qf[ks] = __builtin_bit_cast(vec8, *reinterpret_cast<const uint4*>(q_row + 16 * ks));
        }
    }
    issue(2, 0);
    issue(3, 1);
#pragma unroll
    for (int ks = 0; ks < G::KS; ++ks) PinAgpr(qf[ks]);
    if (tid < 8) s_flag[tid] = 0;  // tile 0 is never rescaled for
    WaitVm<4 * G::IPW>();          // K(0), K(1)
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    floatx16 s0, s1;
    vec8 pb0[2], pb1[2];
    auto qk_all = [&](floatx16& s) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) WaitLgkmTied<0>(kf[ks]);
        A::first_v(s, kf[0], qf[0]);
#pragma unroll
        for (int ks = 1; ks < G::KS; ++ks) A::acc_v(s, kf[ks], qf[ks]);
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s));  // complete, and kf has been read
    };
    StaticFor<G::KS>([&](auto ks) __attribute__((always_inline)) { read_k1.template operator()<0, ks>(); });
    qk_all(s0);
    StaticFor<G::KS>([&](auto ks) __attribute__((always_inline)) { read_k1.template operator()<1, ks>(); });
    {
        const float lm = mask_max(s0, 0, n_plain == 0);
        decide(lm, 0, 0);  // O is zero: the factors published for tile 0 are never read
    }
    qk_all(s1);
    {
        uint32_t pw[8];
#pragma unroll
        for (int n = 0; n < kOps; ++n) op(n, s0, pw);
        pack_p(pw, pb0);
        write_p.template operator()<0>(pb0);
        const float lm = mask_max(s1, 1, n_plain <= 1);
        decide(lm, 1, 1);
    }
    WaitVm<2 * G::IPW>();  // K(2), V(0)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    issue(4, 2);  // K slots 0 and 1 were read before the barrier
    issue(5, 3);
    StaticFor<G::KS>([&](auto ks) __attribute__((always_inline)) { read_k1.template operator()<2, ks>(); });
    StaticFor<4 * G::DT>([&](auto i) __attribute__((always_inline)) { read_v1.template operator()<0, 0, i>(); });
    WaitVm<4 * G::IPW>();  // K(3), V(1)
    WaitLgkmTied<0>(kf[G::KS - 1]);
    __builtin_amdgcn_s_barrier();

    // One step for key tile t (S = t & 3). On entry kf holds K(t+2)'s fragments, va[t & 1] V(t)'s,
    // s_in the masked scores of tile t+1 (its decision made), pb_in the owned P(t); the partner's
    // P(t) and the flags of tile t+1 are in LDS; K(t+3) and V(t+1) have landed.
    //   A  QK(t+2) | partner's P(t), flags(t+1), V(t+1)'s fragments; exponentials of tile t+1
    //   B  PV(t), own subtile first | write P(t+1), mask and maximum of tile t+2, K(t+3)'s fragments
    //   then the factors of tile t+1 to O, the decision for tile t+2, the waits and the barrier.
    auto step = [&]<bool kMaskable, int S>(int t, floatx16& s_in, floatx16& s_out, vec8 (&pb_in)[2],
                                           vec8 (&pb_out)[2]) __attribute__((always_inline)) {
        constexpr int VB = S & 1;
        constexpr int NPV = 4 * G::DT;  // PV MFMAs: 2 subtiles x DT x 2 k-steps
        vec8 pbx[2];
        uint2 flags;
        uint32_t pw[8];
        // ---- A ----
        constexpr int kOpsA = (kOps + G::KS - 1) / G::KS;
        constexpr int kVReads = (4 * G::DT + G::KS - 4) / (G::KS - 3);
        StaticFor<G::KS>([&](auto ks) __attribute__((always_inline)) {
            if constexpr (ks == 0) {
                A::first_v(s_out, kf[0], qf[0]);
            } else {
                A::acc_v(s_out, kf[ks], qf[ks]);
            }
            Fence();
            if constexpr (ks == 0) {
                ReadB128Asm<VB * 8192>(pbx[0], p_partner);
                ReadB128Asm<VB * 8192 + 1024>(pbx[1], p_partner);
                ReadB64Asm<(VB ^ 1) * 16>(flags, flag_addr);
            }
            StaticFor<kVReads>([&](auto q) __attribute__((always_inline)) {
                constexpr int i = (ks - 1) * kVReads + q;
                if constexpr (ks >= 1 && i < 4 * G::DT) {
                    read_v1.template operator()<(S + 1) & 3, VB ^ 1, i>();
                }
            });
#pragma unroll
            for (int q = 0; q < kOpsA; ++q) {
                if (ks * kOpsA + q < kOps) op(ks * kOpsA + q, s_in, pw);
            }
            if constexpr (ks % 4 == 2 && ks / 4 < G::IPW) dma_k(ks / 4, (S + 2) & 3, t + 6);
            Fence();
        });
        pack_p(pw, pb_out);
        // The partner's P and the flags have arrived (every read of region A, in order).
        WaitLgkmTied<0>(pbx[0]);
        WaitLgkmTied<0>(pbx[1]);
        WaitLgkmTied<0>(flags);
        // ---- B ----
        float lm = neg_inf();
        StaticFor<NPV>([&](auto i) __attribute__((always_inline)) {
            constexpr bool kOwn = i < NPV / 2;
            constexpr int f = i % (NPV / 2);  // fragment 2*dt + k-step
            if constexpr (kOwn) {
                A::acc_a(o[0][f / 2], va[VB][f], pb_in[f % 2]);
            } else {
                A::acc_a(o[1][f / 2], va[VB][f], pbx[f % 2]);
            }
            Fence();
            if constexpr (i == 0) write_p.template operator()<VB ^ 1>(pb_out);
            if constexpr (i == 2) {
                asm volatile("s_nop 4");
                lm = mask_max(s_out, t + 2, kMaskable && t + 2 >= n_plain);
            }
            if constexpr (i >= 2) {
                // KS K reads over the MFMAs 2 .. (kf was last read three MFMAs ago).
                constexpr int kPer = (G::KS + NPV - 4) / (NPV - 3);
                StaticFor<kPer>([&](auto q) __attribute__((always_inline)) {
                    constexpr int ks = (i - 2) * kPer + q;
                    if constexpr (ks < G::KS) read_k1.template operator()<(S + 3) & 3, ks>();
                });
            }
            if constexpr (i % 4 == 1 && i / 4 < G::IPW) dma_v(i / 4, S, t + 4);
            Fence();
        });
        apply(flags, t + 1, VB ^ 1);
        decide(lm, t + 2, VB);
        Fence();
        // K(t+4) and V(t+2) landed (the groups of this step and the one before stay in flight);
        // fragment reads and LDS writes retired.
        WaitVm<4 * G::IPW>();
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(kf[G::KS - 1])::"memory");
        __builtin_amdgcn_s_barrier();
    };

    int t = 0;
    for (; t + 6 <= n_plain; t += 4) {
        step.template operator()<false, 0>(t, s1, s0, pb0, pb1);
        step.template operator()<false, 1>(t + 1, s0, s1, pb1, pb0);
        step.template operator()<false, 2>(t + 2, s1, s0, pb0, pb1);
        step.template operator()<false, 3>(t + 3, s0, s1, pb1, pb0);
    }
    for (; t < n_tiles; t += 4) {
        step.template operator()<true, 0>(t, s1, s0, pb0, pb1);
        if (t + 1 >= n_tiles) break;
        step.template operator()<true, 1>(t + 1, s0, s1, pb1, pb0);
        if (t + 2 >= n_tiles) break;
        step.template operator()<true, 2>(t + 2, s1, s0, pb0, pb1);
        if (t + 3 >= n_tiles) break;
        step.template operator()<true, 3>(t + 3, s0, s1, pb1, pb0);
    }

    // ---- epilogue: share 1/l, normalise, store ----
    WaitVm<0>();
    SettleO(o);
    constexpr bool kBoth = kDen == kRoundedAndUnrounded;
    const float l_lse = HalfSum(rs.l + l2);
    const float l_tot = kBoth ? HalfSum(lw) : l_lse;
    if (splits > 1) {
        // The unnormalised state: both subtiles' O at the scale of their owner's m (and, with two
        // denominators, to the scale of the unrounded one, which the merge takes).
        if (hh == 0) {
            if (kBoth) s_alpha[(rg * 2 + dh) * 32 + lr] = l_tot > 0.0f ? l_lse / l_tot : 0.0f;
            if (qi[0] < seq_q) {
                *reinterpret_cast<float2*>(sp.part_ml + 2 * (split * rows_all + flat_own)) =
                    make_float2(rs.m, l_lse);
            }
        }
        if (kBoth) __syncthreads();
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int64_t flat = (b * p.num_heads + h0 + hl[r]) * seq_q + qi[r];
            float* dst = sp.part_o + (split * rows_all + flat) * D + dh * (D / 2);
            const float to_l = kBoth ? s_alpha[(rg * 2 + (dh ^ r)) * 32 + lr] : 1.0f;
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
                float a[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) a[i] = o[r][dt][i] * to_l;
                StorePartialTile(dst + 32 * dt, hh, qi[r] < seq_q, a);
            }
        }
        return;
    }
    if (hh == 0) {
        s_alpha[(rg * 2 + dh) * 32 + lr] = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        if (qi[0] < seq_q && p.lse != nullptr) {
            p.lse[flat_own] = l_lse > 0.0f ? (rs.m + __log2f(l_lse)) * kLn2 : neg_inf();
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float inv = s_alpha[(rg * 2 + (dh ^ r)) * 32 + lr];
        uint16_t* out_row = static_cast<uint16_t*>(p.out) + b * p.o_sb + (h0 + hl[r]) * p.o_sh +
                            static_cast<int64_t>(qi[r]) * p.o_ss + dh * (D / 2);
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
            float a[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) a[i] = o[r][dt][i] * inv;
            StoreTile<M>(out_row + 32 * dt, hh, qi[r] < seq_q, a);
        }
    }
}

}  // namespace

template <typename E, int D, bool kCausal>
int LaunchFlashDsplit(const sca_flash_params& p, const SplitArgs& sp, hipStream_t s) {
    using G = DsplitGeom<D>;
    const int64_t num_q_tiles = (p.seq_q * sp.pack + G::BM - 1) / G::BM;
    const int64_t blocks = num_q_tiles * p.batch * (p.num_heads / sp.pack) * sp.splits;
    if (blocks <= 0) return 0;
    if (blocks > 0x7fffffffLL) {
        return SetError(SCA_E_SEQ_TOO_LONG, "flash: grid of " + std::to_string(blocks) +
                                                " workgroups exceeds the launch limit");
    }
    auto launch = [&]<bool kCut, Denominator kDen>() -> int {
        if (const int rc = EnsureLdsLimit<&flash_fwd_dsplit_kernel<E, D, kCausal, kCut, kDen>>(
                G::LDS_BYTES, "flash LDS limit")) {
            return rc;
        }
        hipLaunchKernelGGL((flash_fwd_dsplit_kernel<E, D, kCausal, kCut, kDen>),
                           dim3(static_cast<unsigned>(blocks)), dim3(G::THREADS), G::LDS_BYTES, s, p,
                           static_cast<int>(num_q_tiles), sp);
        return CheckLaunch("flash_fwd_dsplit_kernel", s);
    };
    const bool cut = sp.pack != 1 || sp.splits != 1;
    if (p.lse != nullptr) {
        constexpr Denominator kDen = DenominatorFor<D>(true);
        return cut ? launch.template operator()<true, kDen>() : launch.template operator()<false, kDen>();
    }
    constexpr Denominator kDen = DenominatorFor<D>(false);
    return cut ? launch.template operator()<true, kDen>() : launch.template operator()<false, kDen>();
}

#define SCA_INSTANTIATE(E, D)                                                     \
    template int LaunchFlashDsplit<E, D, false>(const sca_flash_params&, const SplitArgs&, hipStream_t); \
    template int LaunchFlashDsplit<E, D, true>(const sca_flash_params&, const SplitArgs&, hipStream_t);
SCA_INSTANTIATE(F16, 192)
SCA_INSTANTIATE(F16, 256)
SCA_INSTANTIATE(BF16, 192)
SCA_INSTANTIATE(BF16, 256)

}  // namespace sca_hip
