// HSTU jagged attention forward for gfx950: fp32 inputs, fp32 output.
//
// A wavefront owns 16 query rows and works alone: both products run on v_mfma_f32_16x16x4_f32, whose operand layouts let it
// read K and V from memory straight into the registers the instruction takes, 16 keys a block, the next block on its way
// while the products of this one run; no LDS and no barrier in the sweep.  The fp32 matrix instruction is slow (32 cycles for
// 2048 flops, 154 TFLOP/s of the card), so the sweep is bound by the matrix pipe, and a small launch by how long ONE
// wavefront sweeps: a workgroup's wavefronts therefore stand for row groups x key shares, a.f32_splits of them dealing the
// key blocks of one row group and adding their outputs through LDS in a fixed order.  The host takes as many shares as
// it needs to fill the machine (f32_splits() there).
//
// Layouts (lane l, i = l % 16, g = l / 16): A[i][g], B[g][i], accumulator rows 4 g + r, column i.  The contraction order of
// S^T = K Q^T is free: step (j, e) contracts the head dims 16 j + 4 g + e, so a lane holds 16-byte pieces of its row.
// S^T leaves a lane with keys 4 g + r of query i, which is the B operand of step r of O^T += V^T P^T; there the M index of
// tile (h, t) is mapped to head dim 64 h + 4 i + t, so that a lane's A operands of four tiles are 16 bytes of one V row
// and its outputs 16-byte pieces of one output row.
//
// Measured (MI355X), the kernel this one replaced (one 128-row tile per workgroup, K and V through one LDS buffer without
// overlap) against it: see the dispatch rule in hstu_mi355.hip.
#pragma once
#include "hstu_fwd_kernel.hip.h"

namespace hstu {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// one 16-byte piece at off + base (base uniform and inside the descriptor); outside the descriptor it reads zeros
__device__ __forceinline__ f32x4_t buffer_f32x4(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, uint32_t base = 0)
{
    return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(off), static_cast<int>(base), 0));
}

template <int D, bool HAS_RAB, bool HAS_MASK>
__global__ __launch_bounds__(f32_waves(D) * 64) void hstu_fwd_f32_kernel(const FwdArgs a)
{
    constexpr int W = f32_waves(D);
    constexpr int KCH = D / 16;                 // 16-byte pieces of a Q or K row per lane
    constexpr int H = D >= 64 ? D / 64 : 1;     // spans of 64 output dims
    constexpr int T = D >= 64 ? 4 : D / 16;     // tiles per span; a lane's V piece holds one element of each
    constexpr bool kTurns = D <= 64 && !(D == 64 && (HAS_RAB || HAS_MASK));  // registers for two blocks side by side
    static_assert(D == 32 || D % 64 == 0, "head-dim slots 32, 64, 128, 256");

    __shared__ __attribute__((aligned(16))) float s_part[W * H * T * 4 * 64];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int i = lane & 15;
    const int g = lane >> 4;
    const int splits = a.f32_splits;
    const int group = wave / splits;
    const int share = wave - group * splits;
    const int rows_per_wg = 16 * (W / splits);

    // slots: tile levels from the last (longest key ranges) down, pairs padded to a multiple of 8 so that the tiles of a
    // pair run on one XCD
    const int bh_pad = (a.bh + 7) & ~7;
    const int lvl = blockIdx.x / bh_pad;
    const int bhid = blockIdx.x - lvl * bh_pad;
    if (bhid >= a.bh) {
        return;
    }
    const int qt = (a.max_q + rows_per_wg - 1) / rows_per_wg - 1 - lvl;
    const int b = bhid / a.n_heads_q;
    const int h = bhid - b * a.n_heads_q;
    const int hk = h / a.head_ratio;

    int64_t q0 = load_index(a.offs_q, b, a.idx64);
    int64_t q1 = load_index(a.offs_q, b + 1, a.idx64);
    int64_t k0 = load_index(a.offs_k, b, a.idx64);
    int64_t k1 = load_index(a.offs_k, b + 1, a.idx64);
    int n_ctx = (a.mask_type == 0 && a.num_ctx) ? static_cast<int>(load_index(a.num_ctx, b, a.idx64)) : 0;
    int n_tgt = (a.mask_type == 0 && a.num_tgt) ? static_cast<int>(load_index(a.num_tgt, b, a.idx64)) : 0;
    q1 = q1 < a.total_q ? q1 : a.total_q;
    k1 = k1 < a.total_k ? k1 : a.total_k;
    q0 = q0 < 0 ? 0 : q0;
    k0 = k0 < 0 ? 0 : k0;
    int sq = static_cast<int>(q1 > q0 ? q1 - q0 : 0);
    int sk = static_cast<int>(k1 > k0 ? k1 - k0 : 0);
    sq = uniform(sq < a.max_q ? sq : a.max_q);
    sk = uniform(sk < a.max_k ? sk : a.max_k);

    float* const out32 = static_cast<float*>(a.out);
    if (qt == 0) {  // rows past the last offset belong to no sequence: zero-fill them
        const int64_t last = load_index(a.offs_q, a.n_batch, a.idx64);
        const int64_t first_tail = last < 0 ? 0 : last;
        const int64_t row_elems = static_cast<int64_t>(a.n_heads_q) * a.d_v;
        const int64_t n_tail = (a.total_q > first_tail ? a.total_q - first_tail : 0) * row_elems;
        float* tail = out32 + first_tail * row_elems;
        for (int64_t e = static_cast<int64_t>(bhid) * (W * 64) + tid; e < n_tail; e += static_cast<int64_t>(a.bh) * (W * 64)) {
            tail[e] = 0.f;
        }
    }
    if (qt * rows_per_wg >= sq) {
        return;
    }
    const int wr0 = qt * rows_per_wg + group * 16;
    const bool wave_active = wr0 < sq;
    n_ctx = uniform(n_ctx < 0 ? 0 : n_ctx);
    n_tgt = uniform(n_tgt < 0 ? 0 : (n_tgt > sk ? sk : n_tgt));
    const int hist_k = sk - n_tgt;

    // visibility of the lane's row: visible(j) = j < lim && !(hist_k <= j < hole_hi)
    int row = wr0 + i;
    row = row < sq - 1 ? row : sq - 1;
    int lim = sk;
    int hole_hi = 0;
    if (a.mask_type == 0) {
        lim = row + (sk - sq) + 1;
        if (row < n_ctx) {
            lim = lim > hist_k ? lim : hist_k;
        }
        lim = lim < 0 ? 0 : (lim > sk ? sk : lim);
        const int ti = row - (sq - n_tgt);
        if (n_tgt > 0 && a.target_group > 0 && ti >= 0) {
            hole_hi = hist_k + (ti / a.target_group) * a.target_group;
        }
    }
    const WaveBounds wb = wave_bounds(a.mask_type, wr0, sq, sk, n_ctx, n_tgt, a.target_group, wave_active, 16);
    const int n_blocks = uniform((wb.lim_max + 15) / 16);

    const uint32_t q_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_qk * 4u;
    const uint32_t k_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_qk * 4u;
    const uint32_t v_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_v * 4u;
    const uint32_t o_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_v * 4u;
    const __amdgpu_buffer_rsrc_t q_rsrc =
        make_rsrc(static_cast<const float*>(a.q) + (q0 * a.n_heads_q + h) * static_cast<int64_t>(a.d_qk),
                  static_cast<uint32_t>(sq - 1) * q_stride + a.d_qk * 4u);
    const __amdgpu_buffer_rsrc_t k_rsrc =
        make_rsrc(static_cast<const float*>(a.k) + (k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_qk),
                  sk > 0 ? static_cast<uint32_t>(sk - 1) * k_stride + a.d_qk * 4u : 0u);
    const __amdgpu_buffer_rsrc_t v_rsrc =
        make_rsrc(static_cast<const float*>(a.v) + (k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_v),
                  sk > 0 ? static_cast<uint32_t>(sk - 1) * v_stride + a.d_v * 4u : 0u);
    const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(out32 + (q0 * a.n_heads_q + h) * static_cast<int64_t>(a.d_v),
                                                    static_cast<uint32_t>(sq - 1) * o_stride + a.d_v * 4u);
    const uint32_t bias_bytes = static_cast<uint32_t>(a.max_q) * static_cast<uint32_t>(a.max_k) * 4u;
    const int64_t bias_plane = (static_cast<int64_t>(b) * a.n_heads_q + h) * a.max_q * static_cast<int64_t>(a.max_k);
    const __amdgpu_buffer_rsrc_t rab_rsrc =
        make_rsrc(HAS_RAB ? static_cast<const float*>(a.rab) + bias_plane : nullptr, HAS_RAB ? bias_bytes : 0u);
    const __amdgpu_buffer_rsrc_t mask_rsrc =
        make_rsrc(HAS_MASK ? static_cast<const float*>(a.mask) + bias_plane : nullptr, HAS_MASK ? bias_bytes : 0u);
    const uint32_t bias_row_off = static_cast<uint32_t>(wr0 + i) * static_cast<uint32_t>(a.max_k) * 4u;

    uint32_t k_off[KCH];  // of the lane's pieces of key i of a block
#pragma unroll
    for (int j = 0; j < KCH; ++j) {
        const int d0 = 16 * j + 4 * g;
        k_off[j] = d0 < a.d_qk ? static_cast<uint32_t>(i) * k_stride + d0 * 4u : kOutOfRange;
    }
    // of the lane's pieces of keys 4 g + r of a block (one offset and three additions where registers are short)
    constexpr int VR = kTurns ? 4 : 1;
    uint32_t v_off[H][VR];
#pragma unroll
    for (int s = 0; s < H; ++s) {
        const int d0 = 64 * s + T * i;
#pragma unroll
        for (int r = 0; r < VR; ++r) {
            v_off[s][r] = d0 < a.d_v ? static_cast<uint32_t>(4 * g + r) * v_stride + d0 * 4u : kOutOfRange;
        }
    }

    struct Block {
        f32x4_t k[KCH];
        f32x4_t v[H][4];
        f32x4_t rab;
        f32x4_t mask;
    };
    // four values of a [max_q][max_k] row at keys c0 + 4 g ..; rows that are not 16-byte aligned element by element
    auto load_plane = [&](__amdgpu_buffer_rsrc_t rsrc, int c0) {
        const uint32_t off = bias_row_off + static_cast<uint32_t>(c0 + 4 * g) * 4u;
        if (a.bias_vec_ok != 0) {
            return buffer_f32x4(rsrc, off);
        }
        // (laundered so that the optimiser does not fold these loads with the vector load of the other branch)
        uint32_t eoff = off;
        asm volatile("" : "+v"(eoff));
        f32x4_t w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, static_cast<int>(eoff + 4u * e), 0, 0));
            w[e] = x;
        }
        return w;
    };
    // (a block past the last, which is asked for and never used, is the last one again: the bases stay inside the sequence)
    auto load_block = [&](int block, Block& x) {
        const int c0 = uniform((block < n_blocks ? block : n_blocks - 1) * 16);
        const uint32_t kb = static_cast<uint32_t>(c0) * k_stride;
        const uint32_t vb = static_cast<uint32_t>(c0) * v_stride;
#pragma unroll
        for (int j = 0; j < KCH; ++j) {
            x.k[j] = buffer_f32x4(k_rsrc, k_off[j], kb);
        }
        if constexpr (HAS_RAB) {
            x.rab = load_plane(rab_rsrc, c0);
        }
        if constexpr (HAS_MASK) {
            x.mask = load_plane(mask_rsrc, c0);
        }
#pragma unroll
        for (int s = 0; s < H; ++s) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t off = VR == 4 ? v_off[s][r % VR] : v_off[s][0] + static_cast<uint32_t>(r) * v_stride;
                if constexpr (T == 4) {
                    x.v[s][r] = buffer_f32x4(v_rsrc, off, vb);
                } else {
                    typedef __attribute__((ext_vector_type(2))) float f32x2_t;
                    const f32x2_t w = __builtin_bit_cast(f32x2_t, __builtin_amdgcn_raw_buffer_load_b64(v_rsrc, static_cast<int>(off), static_cast<int>(vb), 0));
                    x.v[s][r] = f32x4_t{w[0], w[1], 0.f, 0.f};
                }
            }
        }
    };

    f32x4_t acc[H][T];
#pragma unroll
    for (int s = 0; s < H; ++s) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            acc[s][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (share < n_blocks) {
        f32x4_t qf[KCH];
#pragma unroll
        for (int j = 0; j < KCH; ++j) {
            const int d0 = 16 * j + 4 * g;
            qf[j] = buffer_f32x4(q_rsrc, d0 < a.d_qk ? static_cast<uint32_t>(wr0 + i) * q_stride + d0 * 4u : kOutOfRange);
        }
        const float c_exp = a.c_exp;
        auto products = [&](int block, const Block& cur) {
            const int c0 = block * 16;
            f32x4_t s = HAS_RAB ? cur.rab : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < KCH; ++j) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[j][e], qf[j][e], s, 0, 0, 0);
                }
            }
            // P^T = S^T * sigmoid(alpha * S^T), masked
            // (the conditions are combined without branches: the products and the first use of S stay one basic block, in which the
            // element-wise stage can be scheduled; the compiler's wait states are right either way)
            const bool hole = wb.any_hole & (c0 + 16 > hist_k) & (c0 < wb.hole_hi_max);
            const bool full = !HAS_MASK & (c0 + 16 <= wb.lim_min) & !hole;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[r] *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(s[r] * c_exp));
            }
            if (!full) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = c0 + 4 * g + r;
                    const bool visible = key < lim && !(key >= hist_k && key < hole_hi);
                    const float p = HAS_MASK ? s[r] * cur.mask[r] : s[r];
                    s[r] = visible ? p : 0.f;
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int sp = 0; sp < H; ++sp) {
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        acc[sp][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.v[sp][r][t], s[r], acc[sp][t], 0, 0, 0);
                    }
                }
            }
        };
        // two blocks in turn, each asked for while the products of the other run (with wide heads through copies, which
        // the compiler keeps without spilling)
        Block even;
        Block odd;
        load_block(share, even);
        if constexpr (kTurns) {
            for (int block = share; block < n_blocks; block += 2 * splits) {
                load_block(block + splits, odd);
                products(block, even);
                if (block + splits >= n_blocks) {
                    break;
                }
                load_block(block + 2 * splits, even);
                products(block + splits, odd);
            }
        } else {
            for (int block = share; block < n_blocks; block += splits) {
                load_block(block + splits, odd);
                products(block, even);
                even = odd;
            }
        }
    }

    // a lane's accumulators are dims 64 sp + T (4 g + r) + t of row wr0 + i: units (sp, r) of T values each
    const float c_out = a.c_out;
    const uint32_t row_off = static_cast<uint32_t>(wr0 + i) * o_stride;
    auto store_unit = [&](int sp, int r, const float* value) {
        const int d0 = 64 * sp + T * (4 * g + r);
        const uint32_t off = (wave_active && d0 < a.d_v) ? row_off + d0 * 4u : kOutOfRange;
        if constexpr (T == 4) {
            const f32x4_t w = {value[0] * c_out, value[1] * c_out, value[2] * c_out, value[3] * c_out};
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, w), o_rsrc, static_cast<int>(off), 0, 0);
        } else {
            typedef __attribute__((ext_vector_type(2))) float f32x2_t;
            const f32x2_t w = {value[0] * c_out, value[1] * c_out};
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, w), o_rsrc, static_cast<int>(off), 0, 0);
        }
    };
    if (splits == 1) {
#pragma unroll
        for (int sp = 0; sp < H; ++sp) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float value[T];
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    value[t] = acc[sp][t][r];
                }
                store_unit(sp, r, value);
            }
        }
        return;
    }
    float* const mine = s_part + wave * (H * T * 4 * 64);
#pragma unroll
    for (int sp = 0; sp < H; ++sp) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                mine[((sp * 4 + r) * T + t) * 64 + lane] = acc[sp][t][r];
            }
        }
    }
    __syncthreads();
    const float* const parts = s_part + (wave - share) * (H * T * 4 * 64);
    for (int u = share; u < H * 4; u += splits) {
        float value[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            value[t] = parts[(u * T + t) * 64 + lane];
        }
        for (int p = 1; p < splits; ++p) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                value[t] += parts[p * (H * T * 4 * 64) + (u * T + t) * 64 + lane];
            }
        }
        store_unit(u / 4, u % 4, value);
    }
}

}  // namespace hstu
