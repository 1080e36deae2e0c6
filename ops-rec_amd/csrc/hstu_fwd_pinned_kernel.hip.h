// HSTU jagged attention forward at the head-dim slots 256 and 128: two (at 128 three) wavefronts per SIMD, the output sums in pinned accumulators.
//
// hstu_fwd_kernel needs 400 registers and more at this slot, so one wavefront per SIMD, which copies every score out of the accumulators
// (195 copies beside 32 MFMAs a step) and has nothing to run while it waits: 35 % of the time in MFMAs.  Here a wavefront (32 query
// rows) has 128 accumulators, all of them output sums, and 128 vector registers: 64 for Q, 16 for the scores of one 32-key block, which
// become P where they stand, 8 for the packed P of the block before.  One step is S^T(t) = K(t) Q^T, 16 MFMAs, then the 16 of
// O^T += V^T(t - 1) P^T(t - 1) with the vector work of silu(S(t)) between them; the second wavefront of the SIMD fills the first half.
// The sums are added in the order of hstu_fwd_kernel.
//
// LDS, 80 KiB, so that two workgroups share a CU: K in a ring of three slots, V of two.  At the start of a step the slots of the step
// before are free: V(t) is requested (a step ahead of its use), then K(t + 2) (two steps ahead).  The slot 128 has half of everything
// and with it room for three workgroups, and for a third V slot: V(t + 1) is requested.
//
// One workgroup per (query tile, K/V pair, query head of the pair) slot: no list, no counters, no workspace.  Slots go level after level
// (heaviest tiles of all pairs first), or pair after pair (a.pair_major): see the host's rule.
//
// Measured, f16, 96 x 2 heads, 512 rows on 3072 keys 412 -> 318 us; bf16, 32 x 8 heads of 1024 rows 243 -> 202 us, 200 x 4 of 65 .. 128 rows
// 57.8 -> 36.5, 24 x 8 of 1000 .. 4000 rows 1007 -> 855 (0.90 PFLOP/s).  Bound by power from there on: the clock falls to 1.9 GHz.
#pragma once
#include "hstu_fwd_short_kernel.hip.h"
#include "hstu_pinned_acc.hip.h"

namespace hstu {

template <typename Tag, int D>
__global__ __launch_bounds__(256, D == 256 ? 2 : 3) void hstu_fwd_pinned_kernel(const FwdArgs a)
{
    constexpr int CPR = D / 8;                  // 16-byte chunks per row
    constexpr int SUB_BYTES = 32 * D * 2;       // a 32-key sub-tile
    constexpr int LPW = SUB_BYTES / 4096;       // 1 KiB load instructions per sub-tile and wavefront
    constexpr int KSTEPS = D / 16, MTILES = D / 32, NCH = 2 * MTILES;
    constexpr int KS = 3, VS = D == 256 ? 2 : 3;               // ring slots
    // what may be under way when a step starts: behind V(t - 1), VS - 1 steps ago, and K(t), two steps ago
    constexpr int kOpen = VS == 2 ? LPW : 2 * LPW;
    constexpr int kAccRegs = MTILES * 16;
    constexpr uint32_t kPastEnd = 0x40000000u;
    constexpr int kV0 = 0, kK0 = VS * SUB_BYTES;
    __shared__ __attribute__((aligned(1024))) uint8_t s_ring[(VS + KS) * SUB_BYTES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int ln = lane & 31;
    const int lh = lane >> 5;

    // ---- rows past the last offset ----
    uint16_t* const out16 = static_cast<uint16_t*>(a.out);
    {
        const int64_t last_offset = load_index_uniform(a.offs_q, a.n_batch, a.idx64);
        const int64_t first_tail = last_offset < 0 ? 0 : (last_offset < a.total_q ? last_offset : a.total_q);
        const int64_t row_elems = static_cast<int64_t>(a.n_heads_q) * a.d_v;
        const int64_t n_tail = (a.total_q - first_tail) * row_elems;
        for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + tid; e < n_tail; e += static_cast<int64_t>(gridDim.x) * 256) {
            out16[first_tail * row_elems + e] = 0;
        }
    }

    // ---- the item of this workgroup ----
    const int n_levels = a.n_qtiles, ratio = a.head_ratio, n_pairs = a.n_batch * a.n_heads_k;
    ShortSlot slot = short_slot(static_cast<int>(blockIdx.x), n_pairs, ratio);
    if (a.pair_major != 0) {
        const int j = static_cast<int>(blockIdx.x) >> 3;
        const int per_pair = n_levels * ratio;
        const int turn = div_small(j, per_pair);
        const int rem = j - turn * per_pair;
        slot.level = div_small(rem, ratio);
        slot.r = rem - slot.level * ratio;
        // The workgroups of an XCD go to its four shader engines in turn, whether or not they find work: with a multiple of four slots a pair
        // would meet the same engines at every level, and those of a level that few sequences have would stand idle -- so the levels move on
        // by one place per pair.  d 128, 175 x 4 heads, 300..400 rows on 1500 keys 236 -> 212 us; d 256, 146 x 8, 200..400 on 900 469 -> 409;
        // other counts of slots per pair level.
        if ((per_pair & 3) == 0) {
            slot.level += turn - div_small(turn, n_levels) * n_levels;
            slot.level -= slot.level >= n_levels ? n_levels : 0;
        }
        slot.pair = turn * 8 + (static_cast<int>(blockIdx.x) & 7);
    }
    if (slot.pair >= n_pairs || slot.level >= n_levels) {
        return;
    }
    const int b = div_small(slot.pair, a.n_heads_k);
    const int hk = slot.pair - b * a.n_heads_k;
    const int h = hk * ratio + slot.r;
    const bool ctx_first = a.mask_type == 0 && a.num_ctx != nullptr;
    const int qt = ctx_first ? (slot.level == 0 ? 0 : n_levels - slot.level) : n_levels - 1 - slot.level;
    int64_t q0 = load_index_uniform(a.offs_q, b, a.idx64), q1 = load_index_uniform(a.offs_q, b + 1, a.idx64);
    int64_t k0 = load_index_uniform(a.offs_k, b, a.idx64), k1 = load_index_uniform(a.offs_k, b + 1, a.idx64);
    int n_ctx = 0, n_tgt = 0;
    if (a.mask_type == 0) {
        if (a.num_ctx) {
            n_ctx = static_cast<int>(load_index_uniform(a.num_ctx, b, a.idx64));
        }
        if (a.num_tgt) {
            n_tgt = static_cast<int>(load_index_uniform(a.num_tgt, b, a.idx64));
        }
    }
    // defensive clamps: malformed offsets must not turn into out-of-bounds addresses
    q1 = q1 < a.total_q ? q1 : a.total_q;
    k1 = k1 < a.total_k ? k1 : a.total_k;
    q0 = q0 < 0 ? 0 : q0;
    k0 = k0 < 0 ? 0 : k0;
    int sq = static_cast<int>(q1 > q0 ? q1 - q0 : 0);
    int sk = static_cast<int>(k1 > k0 ? k1 - k0 : 0);
    sq = sq < a.max_q ? sq : a.max_q;
    sk = sk < a.max_k ? sk : a.max_k;
    const int r0 = qt * kBlockM;
    if (r0 >= sq) {
        return;
    }
    n_ctx = n_ctx < 0 ? 0 : n_ctx;
    n_tgt = n_tgt < 0 ? 0 : (n_tgt > sk ? sk : n_tgt);
    const int delta = sk - sq;
    const int hist_k = sk - n_tgt;
    const int wr0 = r0 + wave * kWaveM;
    const bool wave_active = wr0 < sq;  // inactive wavefronts still take part in loads and barriers

    const uint32_t q_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_qk * 2u;  // bytes per row
    const uint32_t k_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_qk * 2u;
    const uint32_t v_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_v * 2u;
    const uint32_t o_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_v * 2u;
    const __amdgpu_buffer_rsrc_t q_rsrc =
        make_rsrc(static_cast<const uint8_t*>(a.q) + (q0 * a.n_heads_q + h) * static_cast<int64_t>(a.d_qk) * 2,
                  static_cast<uint32_t>(sq - 1) * q_stride + a.d_qk * 2u);
    const u32x4_t k_rsrc = make_rsrc_words(static_cast<const uint8_t*>(a.k) + (k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_qk) * 2,
                                           sk > 0 ? static_cast<uint32_t>(sk - 1) * k_stride + a.d_qk * 2u : 0u);
    const u32x4_t v_rsrc = make_rsrc_words(static_cast<const uint8_t*>(a.v) + (k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_v) * 2,
                                           sk > 0 ? static_cast<uint32_t>(sk - 1) * v_stride + a.d_v * 2u : 0u);

    // ---- keys needed by this item ----
    int kmax;
    if (a.mask_type == 0) {
        const int r1 = (r0 + kBlockM < sq) ? r0 + kBlockM : sq;
        kmax = r1 + delta;
        if (r0 < n_ctx) {
            kmax = kmax > hist_k ? kmax : hist_k;
        }
        kmax = kmax < 0 ? 0 : (kmax > sk ? sk : kmax);
    } else {
        kmax = sk;
    }
    const int n_sub = (kmax + 31) / 32;
    const WaveBounds wb = wave_bounds(a.mask_type, wr0, sq, sk, n_ctx, n_tgt, a.target_group, wave_active);
    const int nx_w = (wb.lim_max + 31) / 32;  // sub-tiles this wavefront's rows can see (<= n_sub)
    // The lane's number, worked out anew: for what is needed in few steps, or at the end, and not worth a register throughout.
    auto fresh_lane = []() -> int {
        int n = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
        asm volatile("" : "+v"(n));
        return n;
    };
    // the keys from c0 on that row wr0 + ln sees, of 32: visible(j) = j < lim  &&  !(hole_lo <= j < hole_hi)
    auto visible_keys = [&](int ln, int c0) -> uint32_t {
        int lim = sk, hole_lo = 0, hole_hi = 0;
        if (a.mask_type == 0) {
            const int row = wr0 + ln < sq - 1 ? wr0 + ln : sq - 1;
            lim = row + delta + 1;
            if (row < n_ctx) {
                lim = lim > hist_k ? lim : hist_k;
            }
            lim = lim < 0 ? 0 : (lim > sk ? sk : lim);
            if (n_tgt > 0 && a.target_group > 0) {
                const int ti = row - (sq - n_tgt);
                if (ti >= 0) {
                    hole_lo = hist_k;
                    hole_hi = hist_k + (ti / a.target_group) * a.target_group;
                }
            }
        }
        auto bits = [](int n) { return n >= 32 ? 0xffffffffu : (n <= 0 ? 0u : (1u << n) - 1u); };
        return bits(lim - c0) & ~(bits(hole_hi - c0) & ~bits(hole_lo - c0));
    };

    // ---- requests ----
    uint32_t k_src[LPW], v_src[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const int piece = (wave * LPW + i) * 64 + lane;  // 16-byte piece within the sub-tile
        const int r = piece / CPR;
        const int kc = k_chunk_swizzle<D>(r, piece % CPR);  // XOR swizzles are their own inverse
        const int vc = v_chunk_swizzle<D>(r, piece % CPR);
        k_src[i] = (kc * 8 < a.d_qk) ? static_cast<uint32_t>(r) * k_stride + kc * 16u : kOutOfRange;
        v_src[i] = (vc * 8 < a.d_v) ? static_cast<uint32_t>(r) * v_stride + vc * 16u : kOutOfRange;
    }
    const uint32_t ring_lds = lds_address(reinterpret_cast<uint16_t*>(s_ring));
    const uint32_t wave_at = static_cast<uint32_t>(wave) * (LPW * 1024u);
    auto request_k = [&](int ks, int x) {
        const uint32_t add = x < n_sub ? static_cast<uint32_t>(x * 32) * k_stride : kPastEnd;
        const uint32_t at = ring_lds + kK0 + static_cast<uint32_t>(ks) * SUB_BYTES + wave_at;
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            request_to_lds_b128(k_rsrc, at + i * 1024u, k_src[i] + add);
        }
    };
    auto request_v = [&](int vs, int x) {
        const uint32_t add = x < n_sub ? static_cast<uint32_t>(x * 32) * v_stride : kPastEnd;
        const uint32_t at = ring_lds + kV0 + static_cast<uint32_t>(vs) * SUB_BYTES + wave_at;
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            request_to_lds_b128(v_rsrc, at + i * 1024u, v_src[i] + add);
        }
    };

    // LDS read offsets in a sub-tile (bytes).  K operand of MFMA step js: row ln, chunk 2 js + lh; V^T operand of output tile mt: the
    // transposing read of hstu_fwd_kernel.  The swizzles are XORs, so step js and tile mt flip the bits of 32 js and of 64 mt.
    const int k_first_off = (ln * D + k_chunk_swizzle<D>(ln, lh) * 8) * 2;
    int v_first_off;
    {
        const int vr0 = 4 * lh + ((lane & 15) >> 2);
        const int col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        v_first_off = (vr0 * D + v_chunk_swizzle<D>(vr0, col >> 3) * 8 + (col & 7)) * 2;
    }

    acc_fence<kAccRegs>();
    acc_zero_all(std::make_integer_sequence<int, kAccRegs>{});
    u32x4_t qf[KSTEPS];
    if (n_sub > 0) {
        request_k(0, 0);
        const uint32_t row_off = static_cast<uint32_t>(wr0 + ln) * q_stride;
#pragma unroll
        for (int js = 0; js < KSTEPS; ++js) {
            const int d0 = 16 * js + 8 * lh;
            qf[js] = __builtin_amdgcn_raw_buffer_load_b128(q_rsrc, static_cast<int>(d0 < a.d_qk ? row_off + d0 * 2u : kOutOfRange), 0, 0);
        }
#pragma unroll
        for (int x = 0; x < VS - 2; ++x) {
            request_v(x, x);
        }
#pragma unroll
        for (int x = 1; x < KS - 1; ++x) {
            request_k(x, x);
        }
        __builtin_amdgcn_s_waitcnt(0);  // (everything, once: the compiler does not know of the requests in assembly)
    }

    const float c_exp = a.c_exp;
    uint32_t pk[8];
    f32x16_t s;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        pk[i] = 0;
    }
#define HSTU_FENCE() __builtin_amdgcn_sched_barrier(0)
    // one sub-tile: S^T(t) = K Q^T then PV(t - 1) with silu(t) between its products, P^T(t) packed behind it
    auto block = [&](auto masked, auto with_pv, auto with_qk, int k_at, int v_at, int t) {
        constexpr bool kMasked = decltype(masked)::value, kPv = decltype(with_pv)::value, kQk = decltype(with_qk)::value;
        constexpr int kAhead = 2;
        u32x4_t op[kAhead + 1];
        acc_fence<kAccRegs>();
        int k_off = k_first_off + k_at, v_off = v_first_off + v_at;
        asm volatile("" : "+v"(k_off), "+v"(v_off));  // (not to be worked out ahead of the sweep, eight registers each)
        auto fetch = [&](int k) {  // operand of slot k: K, then V^T
            if (k < KSTEPS) {
                if constexpr (kQk) {
                    op[k % (kAhead + 1)] = *reinterpret_cast<const u32x4_t*>(s_ring + (k_off ^ (k * 32)));
                }
            } else if (k < KSTEPS + NCH) {
                if constexpr (kPv) {
                    const int c = k - KSTEPS, j2 = c / MTILES, mt = c % MTILES;
                    const uint16_t* const p = reinterpret_cast<const uint16_t*>(s_ring + (v_off ^ (mt * 64))) + 16 * j2 * D;
                    const u32x2_t lo = lds_read_tr16_b64(p);
                    const u32x2_t hi = lds_read_tr16_b64(p + 8 * D);
                    op[k % (kAhead + 1)] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
                }
            }
        };
        if constexpr (kQk) {
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                fetch(k);
            }
            HSTU_FENCE();
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = 0.f;
            }
#pragma unroll
            for (int js = 0; js < KSTEPS; ++js) {
                fetch(js + kAhead);
                HSTU_FENCE();
                s = mfma32<Tag>(op[js % (kAhead + 1)], qf[js], s);
                asm volatile("" : "+v"(s));
                HSTU_FENCE();
            }
        } else {
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                fetch(KSTEPS + k);
            }
        }
        uint32_t vis = 0;
        if constexpr (kMasked && kQk) {
            const int l = fresh_lane();
            vis = visible_keys(l & 31, t * 32) >> (4 * (l >> 5));
        }
        // S becomes P two elements at a time, in two parts, in place
        float tt[2];
        auto part = [&](int k) {
            const int i = k / 2;
            if (k % 2 == 0) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    tt[e] = 1.0f + __builtin_amdgcn_exp2f(s[2 * i + e] * c_exp);
                }
                asm volatile("" : "+v"(tt[0]), "+v"(tt[1]));
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    tt[e] = s[2 * i + e] * __builtin_amdgcn_rcpf(tt[e]);
                }
                // (rounded to fp32 here, as in the other forward kernels: left to itself the compiler takes the product and the rounding to fp16
                // as one instruction in unmasked blocks, and the last bit of a row would depend on the kernel that its batch takes)
                asm volatile("" : "+v"(tt[0]), "+v"(tt[1]));
                s[2 * i] = tt[0];
                s[2 * i + 1] = tt[1];
                if constexpr (kMasked) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int el = 2 * i + e;
                        s[el] = (vis >> (8 * (el / 4) + el % 4)) & 1u ? s[el] : 0.f;
                    }
                }
            }
        };
        auto pack = [&](int i) {
            pk[i] = pack2<Tag>(s[2 * i], s[2 * i + 1]);
            asm volatile("" : "+v"(pk[i]));
        };
        acc_fence<kAccRegs>();
        constexpr int kFirst = NCH >= 16 ? 2 : 1;  // (the last score product has to end first)
        auto parts_done = [](int g) constexpr { return g < kFirst ? 0 : ((g - kFirst + 1) * 16 + NCH - kFirst - 1) / (NCH - kFirst); };
        static_for<NCH>([&](auto ci) {
            constexpr int c = ci;
            if constexpr (kPv) {
                fetch(KSTEPS + c + kAhead);
                HSTU_FENCE();
                acc_mfma<Tag, c % MTILES>(op[(KSTEPS + c) % (kAhead + 1)], u32x4_t{pk[4 * (c / MTILES)], pk[4 * (c / MTILES) + 1],
                                                                                 pk[4 * (c / MTILES) + 2], pk[4 * (c / MTILES) + 3]});
                HSTU_FENCE();
            }
            if constexpr (kQk) {
#pragma unroll
                for (int k = c > 0 ? parts_done(c - 1) : 0; k < parts_done(c); ++k) {
                    part(k);
                }
                HSTU_FENCE();
            }
        });
        if constexpr (kQk) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                pack(i);
            }
        }
        HSTU_FENCE();
    };
#undef HSTU_FENCE

    typedef std::true_type yes_t;
    typedef std::false_type no_t;
    // sub-tiles before this one are wholly visible to all rows of the wavefront
    int full_tiles = wb.lim_min >> 5;
    if (wb.any_hole) {
        const int before_targets = hist_k > 0 ? hist_k >> 5 : 0;
        full_tiles = full_tiles < before_targets ? full_tiles : before_targets;
    }
    if (n_sub > 0) {
        int ks = 0, vs = VS - 1;  // slots of K(t), V(t - 1)
        for (int t = 0; t <= n_sub; ++t) {
            // K(t) and V(t - 1) have landed, for everybody; the slots of the step before are free
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kOpen) : "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            const int k_free = ks == 0 ? KS - 1 : ks - 1, v_free = vs == 0 ? VS - 1 : vs - 1;
            request_v(v_free, t + VS - 2);
            request_k(k_free, t + KS - 1);
            __builtin_amdgcn_sched_barrier(0);
            const int k_at = kK0 + ks * SUB_BYTES, v_at = kV0 + vs * SUB_BYTES;
            if (t > 0 && t < full_tiles && t < nx_w) {
                block(no_t{}, yes_t{}, yes_t{}, k_at, v_at, t);
            } else if (t > 0 && t < nx_w) {
                block(yes_t{}, yes_t{}, yes_t{}, k_at, v_at, t);
            } else if (t < nx_w) {
                block(yes_t{}, no_t{}, yes_t{}, k_at, v_at, t);
            } else if (t == nx_w && t > 0) {
                block(no_t{}, yes_t{}, no_t{}, k_at, v_at, t);
            }
            ks = ks == KS - 1 ? 0 : ks + 1;
            vs = vs == VS - 1 ? 0 : vs + 1;
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // the ring is free
    }

    // ---- store O: lane holds query row (wr0 + ln), dims 32*mt + 8*g + 4*lh + 0..3 (see hstu_fwd_kernel) ----
    acc_settle();
    const float c_out = a.c_out;
    const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(out16 + (q0 * a.n_heads_q + h) * static_cast<int64_t>(a.d_v),
                                                    static_cast<uint32_t>(sq - 1) * o_stride + a.d_v * 2u);
    const int lane_e = fresh_lane(), ln_e = lane_e & 31, lh_e = lane_e >> 5;
    uint16_t* const stage = reinterpret_cast<uint16_t*>(s_ring) + wave * 32 * D;
    const uint32_t o_row = static_cast<uint32_t>(wr0 + ln_e) * o_stride;
    const bool staged = a.out_vec_ok != 0;
    static_for<MTILES>([&](auto mt) {
        const f32x16_t o = acc_block<decltype(mt)::value>(std::make_integer_sequence<int, 16>{});
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const u32x2_t w = {pack2<Tag>(o[4 * g + 0] * c_out, o[4 * g + 1] * c_out), pack2<Tag>(o[4 * g + 2] * c_out, o[4 * g + 3] * c_out)};
            if (staged) {
                *reinterpret_cast<u32x2_t*>(stage + ln_e * D + (((4 * mt + g) ^ (ln_e & (CPR - 1))) * 8 + 4 * lh_e)) = w;
            } else {
                const int d0 = 32 * mt + 8 * g + 4 * lh_e;
                __builtin_amdgcn_raw_buffer_store_b64(w, o_rsrc, static_cast<int>(d0 < a.d_v ? o_row + d0 * 2u : kOutOfRange), 0, 0);
            }
        }
    });
    if (staged) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        constexpr int RPI = 64 / CPR;    // rows per store instruction
        constexpr int kNonTemporal = 2;  // cache policy bit nt: the rows are not read again by this kernel
        const int cc = lane_e % CPR;
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i) {
            const int r = i * RPI + lane_e / CPR;
            const u32x4_t piece = *reinterpret_cast<const u32x4_t*>(stage + r * D + (cc ^ (r & (CPR - 1))) * 8);
            const uint32_t off = (cc * 8 < a.d_v) ? static_cast<uint32_t>(wr0 + r) * o_stride + cc * 16u : kOutOfRange;
            __builtin_amdgcn_raw_buffer_store_b128(piece, o_rsrc, static_cast<int>(off), 0, kNonTemporal);
        }
    }
}

}  // namespace hstu
