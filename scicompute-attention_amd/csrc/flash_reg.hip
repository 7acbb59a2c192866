// Register-staged flash kernel: 4 row groups of 32 query rows, K/V staged through registers into an
// LDS ring with V transposed on the way in. It addresses K and V with 64-bit pointers per tile, so
// it serves the calls that the DMA kernels' 32-bit buffer offsets cannot reach (K/V extents of 2 GiB
// and more, negative row strides), at any head_dim; and, with the shorter prologue, small calls of one
// or two key tiles at head dims other than 64 and 128 (FewTilesCall). The DMA kernels are 1.4-2.5x
// faster on long calls.

#include <hip/hip_runtime.h>

#include <string>

#include "flash_common.hpp"

namespace sca_hip {
namespace {

__device__ __forceinline__ uint32_t Half16(const uint4& v, int t) {
    const uint32_t w = (t < 2) ? v.x : (t < 4) ? v.y : (t < 6) ? v.z : v.w;
    return (t & 1) ? (w >> 16) : (w & 0xffffu);
}

template <typename E, int D, bool kCausal>
__global__ __launch_bounds__(FlashGeom<D>::THREADS, 1) void flash_fwd_kernel(
    const sca_flash_params p, int num_q_tiles) {
    using G = FlashGeom<D>;
    using M = Mfma<E>;
    using vec8 = typename E::vec8;
    constexpr int BN = G::BN;

    extern __shared__ __align__(16) uint16_t lds[];
    uint16_t* sK = lds;                           // [STAGES][BN][KSTR]
    uint16_t* sV = lds + G::STAGES * G::K_STAGE;  // [STAGES][D][VSTR]  (V^T)

    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int lane = tid % kWave;
    const int lr = lane & 31;
    const int hh = lane >> 5;
    const int rg = wave % kRowGroups;  // row group
    const int kh = wave / kRowGroups;  // which 32 keys of every tile this wave owns

    // Block -> (tile, batch*head). Causal: longest row tiles are dispatched first.
    int tile_linear, b_, h_;
    XcdOrder(p, static_cast<uint32_t>(p.num_heads), &tile_linear, &b_, &h_);
    const int qt = kCausal ? (num_q_tiles - 1 - tile_linear) : tile_linear;
    const int64_t b = b_, h = h_;
    const int64_t h_kv = h_ / (static_cast<int>(p.num_heads) / static_cast<int>(p.num_kv_heads));
    const int q0 = qt * kBlockM;
    const int wave_q0 = q0 + rg * kRowsPerWave;
    const int my_q = wave_q0 + lr;
    const int seq_q = static_cast<int>(p.seq_q);
    const int seq_kv = static_cast<int>(p.seq_kv);
    const int diag = static_cast<int>(p.diagonal);

    const uint16_t* q_ptr = static_cast<const uint16_t*>(p.q) + b * p.q_sb + h * p.q_sh;
    const uint16_t* k_ptr = static_cast<const uint16_t*>(p.k) + b * p.k_sb + h_kv * p.k_sh;
    const uint16_t* v_ptr = static_cast<const uint16_t*>(p.v) + b * p.v_sb + h_kv * p.v_sh;

    // Q^T fragments (B operand of S^T = K Q^T): lane holds Q[my_q][16*ks + 8*hh + 0..7].
    vec8 qf[G::KS];
    {
        const uint16_t* q_row = q_ptr + static_cast<int64_t>(my_q) * p.q_ss + 8 * hh;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) {
            uint4 raw = make_uint4(0, 0, 0, 0);
            if (my_q < seq_q) raw = *reinterpret_cast<const uint4*>(q_row + 16 * ks);
            qf[ks] = __builtin_bit_cast(vec8, raw);
        }
        // Retire the Q loads here on every path. Otherwise the waitcnt pass, which merges the
        // loop-entry state conservatively, waits for *all* outstanding loads (including the
        // next tile's prefetch) before the first MFMA of every tile.
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), expcnt/lgkmcnt unconstrained
    }

    int n_tiles = (seq_kv + BN - 1) / BN;
    // Tiles [0, n_plain) are inside seq_kv and fully visible to every row of the workgroup.
    int n_plain = seq_kv / BN;
    if (kCausal) {
        const int last_key = q0 + kBlockM - 1 + diag;
        const int causal_tiles = last_key < 0 ? 0 : last_key / BN + 1;
        if (causal_tiles < n_tiles) n_tiles = causal_tiles;
        const int plain = (q0 + diag + 1) / BN;
        if (plain < n_plain) n_plain = plain;
    }
    if (n_plain > n_tiles) n_plain = n_tiles;

    floatx16 o[G::DT];
#pragma unroll
    for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
    }
    float m_used = neg_inf();  // running max used for the exponentials (log2 units)
    float l_run = 0.0f;        // sum of this lane's rounded weights
    const float scale2 = p.scale * kLog2e;

    // ---- staging: global -> registers -> LDS ------------------------------------------------
    // Per-thread 32-bit element offsets inside one tile, fixed for the whole kernel.
    int k_off[G::K_PER_THREAD], k_row[G::K_PER_THREAD], k_lds[G::K_PER_THREAD];
#pragma unroll
    for (int i = 0; i < G::K_PER_THREAD; ++i) {
        const int c = tid + i * G::THREADS;
        const int row = c / (D / 8);
        const int col = (c % (D / 8)) * 8;
        k_row[i] = c < G::K_CHUNKS ? row : (1 << 30);
        k_off[i] = row * static_cast<int>(p.k_ss) + col;
        k_lds[i] = row * G::KSTR + col;
    }
    int v_off[G::V_PER_THREAD], v_key[G::V_PER_THREAD], v_lds[G::V_PER_THREAD];
#pragma unroll
    for (int i = 0; i < G::V_PER_THREAD; ++i) {
        const int u = tid + i * G::THREADS;
        const int kg = u / (D / 8);
        const int dc = u % (D / 8);
        v_key[i] = u < G::V_UNITS ? 4 * kg : (1 << 30);
        v_off[i] = 4 * kg * static_cast<int>(p.v_ss) + 8 * dc;
        v_lds[i] = 8 * dc * G::VSTR + 4 * kg;
    }
    const int v_ss = static_cast<int>(p.v_ss);

    uint4 k_stage[G::K_PER_THREAD];
    uint4 v_stage[G::V_PER_THREAD][4];

    auto load_tile = [&](int t) {
        const int key0 = t * BN;
        const uint16_t* kt = k_ptr + static_cast<int64_t>(key0) * p.k_ss;
        const uint16_t* vt = v_ptr + static_cast<int64_t>(key0) * p.v_ss;
        const int limit = seq_kv - key0;  // keys of this tile that exist
#pragma unroll
        for (int i = 0; i < G::K_PER_THREAD; ++i) {
            k_stage[i] = make_uint4(0, 0, 0, 0);
            if (k_row[i] < limit) k_stage[i] = *reinterpret_cast<const uint4*>(kt + k_off[i]);
        }
#pragma unroll
        for (int i = 0; i < G::V_PER_THREAD; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v_stage[i][j] = make_uint4(0, 0, 0, 0);
                if (v_key[i] + j < limit) {
                    v_stage[i][j] = *reinterpret_cast<const uint4*>(vt + v_off[i] + j * v_ss);
                }
            }
        }
    };

    auto store_tile = [&](int stage) {
        uint16_t* k_dst = sK + stage * G::K_STAGE;
        uint16_t* v_dst = sV + stage * G::V_STAGE;
#pragma unroll
        for (int i = 0; i < G::K_PER_THREAD; ++i) {
            if (k_row[i] < BN) *reinterpret_cast<uint4*>(k_dst + k_lds[i]) = k_stage[i];
        }
#pragma unroll
        for (int i = 0; i < G::V_PER_THREAD; ++i) {
            if (v_key[i] < BN) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const uint32_t lo = Half16(v_stage[i][0], t) | (Half16(v_stage[i][1], t) << 16);
                    const uint32_t hi = Half16(v_stage[i][2], t) | (Half16(v_stage[i][3], t) << 16);
                    *reinterpret_cast<uint2*>(v_dst + v_lds[i] + t * G::VSTR) = make_uint2(lo, hi);
                }
            }
        }
    };

    const int wkey_base = 32 * kh;  // this wave's first key inside a tile
    const uint16_t* k_frag_base = sK + (wkey_base + lr) * G::KSTR + 8 * hh;
    const uint16_t* v_frag_base = sV + lr * G::VSTR + wkey_base + 4 * hh;

    // S^T[key][q] for this wave's 32 keys x 32 rows of the tile in `stage`.
    auto qk = [&](int stage) {
        const uint16_t* k_tile = k_frag_base + stage * G::K_STAGE;
        vec8 a[G::KS];
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) a[ks] = *reinterpret_cast<const vec8*>(k_tile + 16 * ks);
        floatx16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < G::KS; ++ks) s = M::mma(a[ks], qf[ks], s);
        return s;
    };

    if (n_tiles > 0) {
        load_tile(0);
        store_tile(0);
        if (n_tiles > 1) {
            load_tile(1);
            store_tile(1);
        }
    }
    __syncthreads();
    floatx16 s_cur = qk(0);

    // One pipeline step. Tiles j and j+1 are resident in LDS, tile j+2 is being fetched:
    //   region A: QK MFMAs of tile j+1 interleaved with the softmax VALU work of tile j;
    //   O rescale (only when some lane's running max moved);
    //   region C: PV MFMAs of tile j; then tile j+2 goes to LDS and the workgroup syncs.
    auto step = [&]<bool kMask>(int j) {
        if (j + 2 < n_tiles) load_tile(j + 2);
        const int stage = j % G::STAGES;
        const int next_stage = (j + 1) % G::STAGES;

        // ---- region A (straight-line code) ----
        floatx16 s_nxt = qk(next_stage);  // for the last tile this reads a stale stage; unused
        floatx16 s = s_cur;
        if constexpr (kMask) {
            const int lim = kCausal ? min(seq_kv - 1, my_q + diag) : seq_kv - 1;
            const int kbase = j * BN + wkey_base + 4 * hh;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = kbase + 8 * (i / 4) + (i % 4);
                s[i] = key > lim ? neg_inf() : s[i];
            }
        }
        float tmax = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])),
                           fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
        tmax = fmaxf(tmax, fmaxf(fmaxf(fmaxf(s[8], s[9]), fmaxf(s[10], s[11])),
                                 fmaxf(fmaxf(s[12], s[13]), fmaxf(s[14], s[15]))));
        tmax = fmaxf(tmax, xor32(tmax)) * scale2;
        // Lazy rescale: the max used for the exponentials only moves when the row max grew by
        // more than kRescaleSlack (weights stay <= 2^slack).
        const bool grow = tmax > m_used + kRescaleSlack;
        const float m_new = grow ? tmax : m_used;
        const float alpha = grow ? fast_exp2(m_used - m_new) : 1.0f;
        m_used = m_new;
        l_run *= alpha;
        const float mu = (m_used == neg_inf()) ? 0.0f : m_used;
        uint32_t pw[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float p0 = fast_exp2(fmaf(s[2 * i], scale2, -mu));
            const float p1 = fast_exp2(fmaf(s[2 * i + 1], scale2, -mu));
            pw[i] = M::pack(p0, p1);
            l_run = M::sum2(pw[i], l_run);
        }
        // Materialise P here: without this use the exponentials are sunk into region C, past
        // the rescale branch, and no longer overlap the QK MFMAs.
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(pw[i]));
        // interleave: K-fragment reads first, then one MFMA per ~12 VALU instructions
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, G::KS, 0);
#pragma unroll
        for (int i = 0; i < G::KS; ++i) {
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedValu, 12, 0);
        }

        // ---- O rescale (rare) ----
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
                for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
            }
        }

        // ---- region C: O^T[d][q] += V^T[d][key] P^T[key][q] ----
        // k-step ps covers keys 16*ps + {0..3, 8..11} (hh = 0) or 16*ps + {4..7, 12..15} (hh = 1).
        const vec8 pb0 = __builtin_bit_cast(vec8, make_uint4(pw[0], pw[1], pw[2], pw[3]));
        const vec8 pb1 = __builtin_bit_cast(vec8, make_uint4(pw[4], pw[5], pw[6], pw[7]));
        const uint16_t* v_tile = v_frag_base + stage * G::V_STAGE;
        vec8 va[G::DT][2];
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int ps = 0; ps < 2; ++ps) {
                const uint16_t* vrow = v_tile + 32 * dt * G::VSTR + 16 * ps;
                const uint2 lo = *reinterpret_cast<const uint2*>(vrow);
                const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 8);
                va[dt][ps] = __builtin_bit_cast(vec8, make_uint4(lo.x, lo.y, hi.x, hi.y));
            }
        }
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
            o[dt] = M::mma(va[dt][0], pb0, o[dt]);
            o[dt] = M::mma(va[dt][1], pb1, o[dt]);
        }
        // all V^T fragment reads in flight before the first PV MFMA
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 2 * G::DT, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 2 * G::DT, 0);

        if (j + 2 < n_tiles) store_tile((j + 2) % G::STAGES);
        __syncthreads();
        s_cur = s_nxt;
    };

    int j = 0;
    for (; j < n_plain; ++j) step.template operator()<false>(j);
    for (; j < n_tiles; ++j) step.template operator()<true>(j);

    // Merge the KSPLIT partial states of each row group through LDS.
    if constexpr (G::KSPLIT > 1) {
        float* mbuf = reinterpret_cast<float*>(lds) + (rg * kWave + lane) * G::MERGE_FLOATS;
        if (kh == 1) {
#pragma unroll
            for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
                for (int i = 0; i < 16; ++i) mbuf[dt * 16 + i] = o[dt][i];
            }
            mbuf[G::DT * 16] = m_used;
            mbuf[G::DT * 16 + 1] = l_run;
        }
        __syncthreads();
        if (kh == 1) return;
        const float m_o = mbuf[G::DT * 16];
        const float l_o = mbuf[G::DT * 16 + 1];
        const float mm = fmaxf(m_used, m_o);
        const float wa = (m_used == neg_inf()) ? 0.0f : fast_exp2(m_used - mm);
        const float wb = (m_o == neg_inf()) ? 0.0f : fast_exp2(m_o - mm);
        m_used = mm;
        l_run = l_run * wa + l_o * wb;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = o[dt][i] * wa + mbuf[dt * 16 + i] * wb;
        }
    }

    // Epilogue: merge the two lane halves' sums, normalise, store.
    const float l_tot = l_run + xor32(l_run);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (my_q < seq_q) {
        uint16_t* out_row = static_cast<uint16_t*>(p.out) + b * p.o_sb + h * p.o_sh +
                            static_cast<int64_t>(my_q) * p.o_ss;
#pragma unroll
        for (int dt = 0; dt < G::DT; ++dt) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d0 = 32 * dt + 8 * g + 4 * hh;
                const uint32_t lo = M::pack(o[dt][4 * g + 0] * inv, o[dt][4 * g + 1] * inv);
                const uint32_t hi = M::pack(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv);
                *reinterpret_cast<uint2*>(out_row + d0) = make_uint2(lo, hi);
            }
        }
        if (p.lse != nullptr && hh == 0) {
            p.lse[(b * p.num_heads + h) * p.seq_q + my_q] =
                l_tot > 0.0f ? (m_used + __log2f(l_tot)) * kLn2 : neg_inf();
        }
    }
}

}  // namespace

template <typename E, int D, bool kCausal>
int LaunchFlashReg(const sca_flash_params& p, hipStream_t s) {
    using G = FlashGeom<D>;
    const int64_t num_q_tiles = (p.seq_q + kBlockM - 1) / kBlockM;
    const int64_t blocks = num_q_tiles * p.batch * p.num_heads;
    if (blocks <= 0) return 0;
    if (blocks > 0x7fffffffLL) {
        return SetError(SCA_E_SEQ_TOO_LONG, "flash: grid of " + std::to_string(blocks) +
                                                " workgroups exceeds the launch limit");
    }
    if (const int rc =
            EnsureLdsLimit<&flash_fwd_kernel<E, D, kCausal>>(G::LDS_BYTES, "flash LDS limit")) {
        return rc;
    }
    hipLaunchKernelGGL((flash_fwd_kernel<E, D, kCausal>), dim3(static_cast<unsigned>(blocks)),
                       dim3(G::THREADS), G::LDS_BYTES, s, p, static_cast<int>(num_q_tiles));
    return CheckLaunch("flash_fwd_kernel", s);
}

#define SCA_INSTANTIATE(E, D)                                                    \
    template int LaunchFlashReg<E, D, false>(const sca_flash_params&, hipStream_t); \
    template int LaunchFlashReg<E, D, true>(const sca_flash_params&, hipStream_t);
#define SCA_INSTANTIATE_DIMS(E) \
    SCA_INSTANTIATE(E, 32) SCA_INSTANTIATE(E, 64) SCA_INSTANTIATE(E, 96) SCA_INSTANTIATE(E, 128) \
    SCA_INSTANTIATE(E, 160) SCA_INSTANTIATE(E, 192) SCA_INSTANTIATE(E, 256)
SCA_INSTANTIATE_DIMS(F16)
SCA_INSTANTIATE_DIMS(BF16)

}  // namespace sca_hip
