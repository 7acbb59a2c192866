// Causal pair kernel (head_dim 64 and 128, causal grids too small to balance 128-row tiles): two
// 4-wave groups that run a complementary pair of 64-row tiles side by side; described at its
// geometry (flash_common.hpp).

#include <hip/hip_runtime.h>

#include <string>

#include "flash_common.hpp"

namespace sca_hip {
namespace {

template <typename E, int D>
__global__ __launch_bounds__(PairGeom<D>::THREADS, 1) void flash_fwd_pair_kernel(
    const sca_flash_params p, int num_q_tiles) {
    using G = PairGeom<D>;
    using M = Mfma<E>;
    using vec8 = typename E::vec8;
    constexpr int BN = G::BN;
    constexpr int BM = G::BM;
    constexpr int ROW_BYTES = G::ROW_BYTES;

    extern __shared__ __align__(16) uint8_t lds8[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid % kWave;
    const int lr = lane & 31;
    const int hh = lane >> 5;
    const int g = wave / G::GW;        // group
    const int w4 = wave % G::GW;       // wave within the group
    const int rg = w4 % 2;             // row group: rows 32*rg .. of the row tile
    const int kq = w4 / 2;             // keys 32*kq .. of every key tile

    // The groups share the workgroup barrier: every interval between two barriers is one
    // pipeline step (or setup / merge phase) of each group. The group with fewer intervals
    // pads with empty ones before the final merge, so both groups reach the same count.
    int syncs = 0;
    auto gsync = [&]() {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        ++syncs;
    };

    int tile_linear, b_, h_;
    XcdOrder(p, static_cast<uint32_t>(p.num_heads), &tile_linear, &b_, &h_);
    const int64_t b = b_, h = h_;
    const int64_t h_kv = h_ / (static_cast<int>(p.num_heads) / static_cast<int>(p.num_kv_heads));
    const int seq_q = static_cast<int>(p.seq_q);
    const int seq_kv = static_cast<int>(p.seq_kv);
    const int diag = static_cast<int>(p.diagonal);
    const float scale2 = p.scale * kLog2e;
    const float inv_scale2 = 1.0f / scale2;

    const uint8_t* k_bytes = reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.k) + b * p.k_sb + h_kv * p.k_sh);
    const uint8_t* v_bytes = reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.v) + b * p.v_sb + h_kv * p.v_sh);
    const int k_row_bytes = static_cast<int>(p.k_ss) * 2;
    const int v_row_bytes = static_cast<int>(p.v_ss) * 2;
    const int k_records = (seq_kv - 1) * k_row_bytes + ROW_BYTES;
    const int v_records = (seq_kv - 1) * v_row_bytes + ROW_BYTES;
    uint32_t dma_koff[G::IPW], dma_voff[G::IPW];
#pragma unroll
    for (int i = 0; i < G::IPW; ++i) {
        const int P = (w4 * G::IPW + i) * kWave + lane;
        const int row = P / G::CPR;
        const int pos = P % G::CPR;
        dma_koff[i] = row * k_row_bytes + (pos ^ SwzK<D>(row)) * 16;
        dma_voff[i] = row * v_row_bytes + (pos ^ SwzV<D>(row)) * 16;
    }
    uint8_t* const ring = lds8 + g * G::RING_BYTES;
    // K tile t -> K slot t & 1, V tile t -> V slot t & 1 of this group's ring.
    auto issue_k = [&](int t) {
        uint8_t* dst = ring + (t & 1) * G::TILE_BYTES + w4 * G::IPW * 1024;
        const uint32_t off = static_cast<uint32_t>(t * BN * k_row_bytes);
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) DmaToLds(k_bytes, k_records, dst + i * 1024, dma_koff[i], off);
    };
    auto issue_v = [&](int t) {
        uint8_t* dst = ring + (2 + (t & 1)) * G::TILE_BYTES + w4 * G::IPW * 1024;
        const uint32_t off = static_cast<uint32_t>(t * BN * v_row_bytes);
#pragma unroll
        for (int i = 0; i < G::IPW; ++i) DmaToLds(v_bytes, v_records, dst + i * 1024, dma_voff[i], off);
    };
    // Fragment offsets, with the group's ring base folded in so slot offsets stay immediates.
    const int wkey_base = 32 * kq;
    const int k_row = wkey_base + lr;
    uint32_t k_frag[G::KS];
#pragma unroll
    for (int ks = 0; ks < G::KS; ++ks) {
        k_frag[ks] = g * G::RING_BYTES + k_row * ROW_BYTES + (((2 * ks) ^ hh ^ SwzK<D>(k_row)) * 16);
    }
    const int grp = lane >> 4;
    const int sl = lane & 15;
    const int v_key = wkey_base + 4 * hh + (sl >> 2);
    const int v_chunk = 2 * (grp & 1) + ((sl & 3) >> 1);
    const int v_half = (sl & 1) * 8;
    uint32_t v_frag[G::DT], v_addr[G::DT];
#pragma unroll
    for (int dt = 0; dt < G::DT; ++dt) {
        v_frag[dt] = g * G::RING_BYTES + v_key * ROW_BYTES +
                     (((4 * dt + v_chunk) ^ SwzV<D>(v_key)) * 16) + v_half;
        v_addr[dt] = LdsAddr(lds8) + v_frag[dt];
    }

    // Row tiles: A = T-1-t (long), B = t (short; none when they coincide).
    const int qa = num_q_tiles - 1 - static_cast<int>(tile_linear);
    const int qb = static_cast<int>(tile_linear);
    const bool has_b = qb < qa;
    auto key_tiles = [&](int qt, int& n, int& n_plain) {
        const int q0 = qt * BM;
        n = (seq_kv + BN - 1) / BN;
        n_plain = seq_kv / BN;
        const int last_key = q0 + BM - 1 + diag;
        const int causal_tiles = last_key < 0 ? 0 : last_key / BN + 1;
        if (causal_tiles < n) n = causal_tiles;
        const int plain = (q0 + diag + 1) / BN;
        if (plain < n_plain) n_plain = plain;
        if (n_plain > n) n_plain = n;
    };
    int n_a, plain_a, n_b = 0, plain_b = 0;
    key_tiles(qa, n_a, plain_a);
    if (has_b) key_tiles(qb, n_b, plain_b);
    // Group 0: A tiles [0, x). Group 1: B, its merge, then A tiles [x, n_a). A key range
    // [kb, ke) takes ke - kb + 2 barrier intervals (two for its prologue), B's merge two, so
    // x + 2 = (n_b + 2) + 2 + (n_a - x + 2) balances the groups.
    int x = (n_a + n_b + (has_b ? 4 : 0) + 1) / 2;
    if (x > n_a) x = n_a;
    if (x < 1) x = 1;
    const int syncs_g0 = x + 2;
    const int syncs_g1 = (has_b ? n_b + 4 : 0) + (x < n_a ? n_a - x + 2 : 0);
    const int syncs_all = syncs_g0 > syncs_g1 ? syncs_g0 : syncs_g1;

    vec8 qf[G::KS];
    auto load_q = [&](int qt) {
        // Rows past seq_q repeat the last one (their results are not stored).
        const int row = min(qt * BM + rg * 32 + lr, seq_q - 1);
        const uint16_t* q_row = static_cast<const uint16_t*>(p.q) + b * p.q_sb + h * p.q_sh +
                                static_cast<int64_t>(row) * p.q_ss + 8 * hh;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            qf[ks] = __builtin_bit_cast(vec8, *reinterpret_cast<const uint4*>(q_row + 16 * ks));
        }
    };

    floatx16 o[G::DT];
    RowState rs;
    auto reset_state = [&]() {
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
        }
        ResetRow(rs);
    };

    auto qk_slot = [&](int slot) {
        const uint8_t* base = lds8 + slot * G::TILE_BYTES;
        vec8 a[G::KS];
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) a[ks] = *reinterpret_cast<const vec8*>(base + k_frag[ks]);
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) acc = M::mma(a[ks], qf[ks], acc);
        return acc;
    };

    // Key tiles [kb, ke) of row tile qt into the running state (o, rs.m, rs.l).
    auto run_keys = [&](int qt, int kb, int ke, int n_plain) {
        if (kb >= ke) return;
        const int my_q = qt * BM + rg * 32 + lr;
        const int lim = min(seq_kv - 1, my_q + diag);
        // Keys above lim_j read as -inf.
        auto mask = [&](int jt, int lim_j, floatx16& sv) {
            const int kbase = jt * BN + wkey_base + 4 * hh;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = kbase + 8 * (i / 4) + (i % 4);
                sv[i] = key > lim_j ? neg_inf() : sv[i];
            }
        };
        // Scores of one tile -> exponent arguments in place (t = s * scale2 - m), the first
        // half's weights (keys of pw[0..3]) and their sum. Returns the lane's raw maximum.
        auto prep = [&](floatx16& sv, uint32_t (&ph)[4], float& sh) {
            const float lm = Max16(sv);
#pragma unroll
            for (int i = 0; i < 16; ++i) sv[i] = fmaf(sv[i], scale2, rs.neg_mu);
            float a = 0.0f, c = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p0 = fast_exp2(sv[2 * i]);
                const float p1 = fast_exp2(sv[2 * i + 1]);
                ph[i] = M::pack(p0, p1);
                a += p0;
                c += p1;
            }
            sh = a + c;
            // Pinned here: otherwise they sink below the rare rescale branch, out of PV's shadow.
#pragma unroll
            for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(ph[i]));
            asm volatile("" : "+v"(sh));
            return lm;
        };
        // Lazy rescale, decided after prep ran with the current maximum: only when some lane of
        // the wave sees a raw score above its threshold does the wave exchange the two half-row
        // maxima and move m (to the row maximum, when it exceeds m by more than kRescaleSlack),
        // scaling O and l by 2^(m_old - m_new); the tile's exponent arguments and first-half
        // weights are then redone. The exponentials stay bounded by 2^kRescaleSlack.
        auto fix = [&](float lm, floatx16& sv, uint32_t (&ph)[4], float& sh) {
            if (__builtin_amdgcn_ballot_w64(lm > rs.thr) == 0) return;
            const float tmax = HalfMax(lm) * scale2;
            const bool grow = tmax > rs.m + kRescaleSlack;
            const float m_new = grow ? tmax : rs.m;
            const float alpha = grow ? fast_exp2(rs.m - m_new) : 1.0f;
            const float neg_mu_new = (m_new == neg_inf()) ? 0.0f : -m_new;
            const float delta = neg_mu_new - rs.neg_mu;
            rs.m = m_new;
            rs.l *= alpha;
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
                for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
            }
            rs.thr = (rs.m + kRescaleSlack) * inv_scale2;
            rs.neg_mu = neg_mu_new;
#pragma unroll
            for (int i = 0; i < 16; ++i) sv[i] += delta;
            float a = 0.0f, c = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p0 = fast_exp2(sv[2 * i]);
                const float p1 = fast_exp2(sv[2 * i + 1]);
                ph[i] = M::pack(p0, p1);
                a += p0;
                c += p1;
            }
            sh = a + c;
        };
        // Prologue: K(kb), K(kb+1), V(kb); QK(kb) once K(kb) has landed.
        issue_k(kb);
        if (kb + 1 < ke) issue_k(kb + 1);
        issue_v(kb);
        if (kb + 1 < ke) {
            WaitVm<2 * G::IPW>();
        } else {
            WaitVm<G::IPW>();
        }
        gsync();
        floatx16 s_cur = qk_slot(kb & 1);
        uint32_t ph_cur[4];
        float sh_cur;
        if (kb >= n_plain) mask(kb, lim, s_cur);
        // The first maxima; O and l are zero, so nothing is rescaled.
        rs.m = HalfMax(Max16(s_cur)) * scale2;
        rs.thr = (rs.m + kRescaleSlack) * inv_scale2;
        rs.neg_mu = (rs.m == neg_inf()) ? 0.0f : -rs.m;
        prep(s_cur, ph_cur, sh_cur);
        WaitVm<0>();
        gsync();  // K(kb) read by every wave before step kb refills its slot
        // Step j (S = j & 1): K(j+2) into K slot S and V(j+1) into V slot S^1 (both read in
        // step j-1), QK(j+1) from K slot S^1, PV(j) from V slot S. The softmax work is split
        // between the two MFMA runs of the step so that each has VALU and transcendental work
        // to hide: under QK(j+1) the second half of tile j's weights; under PV(j) tile j+1's
        // maximum, exponent arguments and first-half weights (with the current maximum; the
        // rare move of the maximum redoes them after PV). The range's last step (LAST) has no
        // next tile: it only finishes tile j's weights and runs PV(j).
        auto step = [&]<int S, bool MASK, bool LAST = false>(
                        int j, floatx16& s_in, uint32_t (&ph_in)[4], float sh_in, floatx16& s_out,
                        uint32_t (&ph_out)[4], float& sh_out) {
            vec8 kf[G::KS];
            if constexpr (!LAST) {
                const uint8_t* base = lds8 + (S ^ 1) * G::TILE_BYTES;
#pragma unroll
                for (int ks = 0; ks < G::KS; ++ks) {
                    kf[ks] = *reinterpret_cast<const vec8*>(base + k_frag[ks]);
                }
            }
            vec8 va[2 * G::DT];
            ReadVFrags<(2 + S) * G::TILE_BYTES, ROW_BYTES>(v_addr, va);
            if (j + 2 < ke) issue_k(j + 2);
            if (j + 1 < ke) issue_v(j + 1);
            uint32_t pw[8];
            {
                float a = 0.0f, c = 0.0f;
#pragma unroll
                for (int i = 4; i < 8; ++i) {
                    const float p0 = fast_exp2(s_in[2 * i]);
                    const float p1 = fast_exp2(s_in[2 * i + 1]);
                    pw[i] = M::pack(p0, p1);
                    a += p0;
                    c += p1;
                }
                rs.l += sh_in + (a + c);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) pw[i] = ph_in[i];
            if constexpr (!LAST) {
                floatx16 acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
                for (int ks = 0; ks < G::KS; ++ks) acc = M::mma(kf[ks], qf[ks], acc);
                s_out = acc;
#pragma unroll
                for (int i = 0; i < G::KS; ++i) {
                    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(kSchedValuTrans, 3, 0);
                }
                if constexpr (MASK) mask(j + 1, lim, s_out);
            }
            vec8 pb0 = __builtin_bit_cast(vec8, make_uint4(pw[0], pw[1], pw[2], pw[3]));
            vec8 pb1 = __builtin_bit_cast(vec8, make_uint4(pw[4], pw[5], pw[6], pw[7]));
            WaitLdsTied(va, pb0, pb1);
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
                o[dt] = M::mma(va[2 * dt], pb0, o[dt]);
                o[dt] = M::mma(va[2 * dt + 1], pb1, o[dt]);
            }
            if constexpr (!LAST) {
                const float lm = prep(s_out, ph_out, sh_out);
#pragma unroll
                for (int i = 0; i < 2 * G::DT; ++i) {
                    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(kSchedValuTrans, 6, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                fix(lm, s_out, ph_out, sh_out);
            }
            WaitVm<0>();
            gsync();
        };
        floatx16 s_next;
        uint32_t ph_next[4];
        float sh_next;
        int j = kb;
        // Steps whose next tile needs no mask, then the rest up to the range's last step; each
        // run alternates the two register sets and slots by the step's parity.
        auto run = [&]<bool MASK>(int j_end) {
            if (j < j_end && (j & 1)) {
                step.template operator()<1, MASK>(j, s_cur, ph_cur, sh_cur, s_next, ph_next, sh_next);
                s_cur = s_next;
#pragma unroll
                for (int i = 0; i < 4; ++i) ph_cur[i] = ph_next[i];
                sh_cur = sh_next;
                ++j;
            }
            for (; j + 2 <= j_end; j += 2) {
                step.template operator()<0, MASK>(j, s_cur, ph_cur, sh_cur, s_next, ph_next, sh_next);
                step.template operator()<1, MASK>(j + 1, s_next, ph_next, sh_next, s_cur, ph_cur, sh_cur);
            }
            if (j < j_end) {
                step.template operator()<0, MASK>(j, s_cur, ph_cur, sh_cur, s_next, ph_next, sh_next);
                s_cur = s_next;
#pragma unroll
                for (int i = 0; i < 4; ++i) ph_cur[i] = ph_next[i];
                sh_cur = sh_next;
                ++j;
            }
        };
        run.template operator()<false>(min(ke, n_plain) - 1);
        run.template operator()<true>(ke - 1);
        if (j & 1) {
            step.template operator()<1, true, true>(j, s_cur, ph_cur, sh_cur, s_next, ph_next, sh_next);
        } else {
            step.template operator()<0, true, true>(j, s_cur, ph_cur, sh_cur, s_next, ph_next, sh_next);
        }
    };
    float4* const mquad = reinterpret_cast<float4*>(lds8);
    if (g == 0) {
        load_q(qa);
        reset_state();
        run_keys(qa, 0, x, plain_a);
    } else {
        if (has_b) {
            load_q(qb);
            reset_state();
            run_keys(qb, 0, n_b, plain_b);
            // B's two key halves meet here: the kq = 1 waves hand their state to kq = 0
            // through group 1's ring (idle now: the last step's barrier retired every read).
            float4* const bq = reinterpret_cast<float4*>(ring);
            float2* const bst = reinterpret_cast<float2*>(bq + 2 * 4 * G::DT * kWave);
            if (kq == 1) {
#pragma unroll
                for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        bq[(rg * 4 * G::DT + 4 * dt + q4) * kWave + lane] =
                            make_float4(o[dt][4 * q4], o[dt][4 * q4 + 1], o[dt][4 * q4 + 2],
                                        o[dt][4 * q4 + 3]);
                    }
                }
                bst[rg * kWave + lane] = make_float2(rs.m, rs.l);
            }
            gsync();
            if (kq == 0) {
                const float2 st = bst[rg * kWave + lane];
                const float mm = fmaxf(rs.m, st.x);
                const float w0 = (rs.m == neg_inf()) ? 0.0f : fast_exp2(rs.m - mm);
                const float w1 = (st.x == neg_inf()) ? 0.0f : fast_exp2(st.x - mm);
                const float l_tot = HalfSum(rs.l * w0 + st.y * w1);
                const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
                const int row = qb * BM + rg * 32 + lr;
                const bool row_ok = row < seq_q;
                uint16_t* out_row = static_cast<uint16_t*>(p.out) + b * p.o_sb + h * p.o_sh +
                                    static_cast<int64_t>(row) * p.o_ss;
#pragma unroll
                for (int dt = 0; dt < G::DT; ++dt) {
                    float acc[16];
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        const float4 v = bq[(rg * 4 * G::DT + 4 * dt + q4) * kWave + lane];
                        acc[4 * q4] = o[dt][4 * q4] * w0 + v.x * w1;
                        acc[4 * q4 + 1] = o[dt][4 * q4 + 1] * w0 + v.y * w1;
                        acc[4 * q4 + 2] = o[dt][4 * q4 + 2] * w0 + v.z * w1;
                        acc[4 * q4 + 3] = o[dt][4 * q4 + 3] * w0 + v.w * w1;
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[i] *= inv;
                    StoreTile<M>(out_row + 32 * dt, hh, row_ok, acc);
                }
                if (row_ok && p.lse != nullptr && hh == 0) {
                    p.lse[(b * p.num_heads + h) * p.seq_q + row] =
                        l_tot > 0.0f ? (mm + __log2f(l_tot)) * kLn2 : neg_inf();
                }
            }
            gsync();  // the merge buffer is the ring of the next key range
        }
        load_q(qa);
        reset_state();
        run_keys(qa, x, n_a, plain_a);
    }

    // Both groups reach the same barrier count (the counts are uniform per group).
    while (syncs < syncs_all) gsync();

    // A's four states per row group (groups 0 and 1, key halves 0 and 1) merge into the
    // (g = 0, kq = 0) wave of the row group; the other three hand theirs over through LDS.
    __syncthreads();
    float2* const mstat = reinterpret_cast<float2*>(mquad + G::MERGE_QUADS);
    const int src = g * 2 + kq;  // 0 = the merging wave
    if (src != 0) {
        float4* mbuf = mquad + ((rg * 3 + src - 1) * 4 * G::DT) * kWave + lane;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                mbuf[(4 * dt + q4) * kWave] = make_float4(o[dt][4 * q4], o[dt][4 * q4 + 1],
                                                          o[dt][4 * q4 + 2], o[dt][4 * q4 + 3]);
            }
        }
        mstat[(rg * 3 + src - 1) * kWave + lane] = make_float2(rs.m, rs.l);
    }
    __syncthreads();
    if (src == 0) {
        float2 st[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) st[q] = mstat[(rg * 3 + q) * kWave + lane];
        float mm = rs.m;
#pragma unroll
        for (int q = 0; q < 3; ++q) mm = fmaxf(mm, st[q].x);
        float wq[4];
        wq[0] = (rs.m == neg_inf()) ? 0.0f : fast_exp2(rs.m - mm);
        float l = rs.l * wq[0];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            wq[q + 1] = (st[q].x == neg_inf()) ? 0.0f : fast_exp2(st[q].x - mm);
            l += st[q].y * wq[q + 1];
        }
        const float l_tot = HalfSum(l);
        const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        const int row = qa * BM + rg * 32 + lr;
        const bool row_ok = row < seq_q;
        uint16_t* out_row = static_cast<uint16_t*>(p.out) + b * p.o_sb + h * p.o_sh +
                            static_cast<int64_t>(row) * p.o_ss;
        const float4* mb = mquad + (rg * 3 * 4 * G::DT) * kWave + lane;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
            float acc[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = o[dt][i] * wq[0];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const float4 v = mb[(q * 4 * G::DT + 4 * dt + q4) * kWave];
                    acc[4 * q4] += v.x * wq[q + 1];
                    acc[4 * q4 + 1] += v.y * wq[q + 1];
                    acc[4 * q4 + 2] += v.z * wq[q + 1];
                    acc[4 * q4 + 3] += v.w * wq[q + 1];
                }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] *= inv;
            StoreTile<M>(out_row + 32 * dt, hh, row_ok, acc);
        }
        if (row_ok && p.lse != nullptr && hh == 0) {
            p.lse[(b * p.num_heads + h) * p.seq_q + row] =
                l_tot > 0.0f ? (mm + __log2f(l_tot)) * kLn2 : neg_inf();
        }
    }
}

}  // namespace

template <typename E, int D>
int LaunchFlashPair(const sca_flash_params& p, hipStream_t s) {
    using G = PairGeom<D>;
    const int64_t num_q_tiles = (p.seq_q + G::BM - 1) / G::BM;
    const int64_t blocks = (num_q_tiles + 1) / 2 * p.batch * p.num_heads;
    if (blocks <= 0) return 0;
    if (blocks > 0x7fffffffLL) {
        return SetError(SCA_E_SEQ_TOO_LONG, "flash: grid of " + std::to_string(blocks) +
                                                " workgroups exceeds the launch limit");
    }
    if (const int rc =
            EnsureLdsLimit<&flash_fwd_pair_kernel<E, D>>(G::LDS_BYTES, "flash LDS limit")) {
        return rc;
    }
    hipLaunchKernelGGL((flash_fwd_pair_kernel<E, D>), dim3(static_cast<unsigned>(blocks)),
                       dim3(G::THREADS), G::LDS_BYTES, s, p, static_cast<int>(num_q_tiles));
    return CheckLaunch("flash_fwd_pair_kernel", s);
}

template int LaunchFlashPair<F16, 64>(const sca_flash_params&, hipStream_t);
template int LaunchFlashPair<F16, 128>(const sca_flash_params&, hipStream_t);
template int LaunchFlashPair<BF16, 64>(const sca_flash_params&, hipStream_t);
template int LaunchFlashPair<BF16, 128>(const sca_flash_params&, hipStream_t);

}  // namespace sca_hip
