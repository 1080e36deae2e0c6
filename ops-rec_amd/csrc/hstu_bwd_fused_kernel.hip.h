// HSTU jagged attention backward for gfx950 (MI355X): the five products in two launches, dS handed from the first to the second.
//
//   hstu_bwd_kv_fused_kernel    a workgroup per 128-key tile of one (sequence, K/V head), 32 keys per wavefront:
//                                 S = Q . K^T,  P,  dV^T += dO^T . P,   dP = dO . V^T,  dS,  dK^T += Q^T . dS
//                               and dS, rounded, into a workspace
//   hstu_bwd_dq_from_ds_kernel  a workgroup per 128-row query tile: dQ^T += K^T . dS^T
//                                                        (formulas and conventions: hstu_bwd_kernel.hip.h)
//
// The key-tile kernel keeps both output sums in accumulator registers it names itself (hstu_pinned_acc.hip.h: 128 at the head-dim slot
// 128), K in vector registers and V in LDS, so that what is left fits 128 vector registers and two wavefronts share a SIMD: left to the
// compiler, a wavefront with both sums needs 328 registers, and dV and dK came from two workgroups that each formed S.  Its blocks are
// written out in slots of one matrix instruction: the score algebra of the 16 elements of a lane is dealt over the products behind S,
// and operands come from LDS two slots ahead; volatile empty assembly pins both, because the compiler otherwise gathers the score
// algebra in one place.  All products of a block use operands that the block has at hand, so exp and reciprocal are taken once per
// pair (three times where the kernels recompute).
//
// What bounds it, bf16: large launches the power the card may draw -- 8 x 8 heads, d 128, 4096..8000 rows: 1.22 ms = 1.02 PFLOP/s at 1.8
// GHz with 47 % of the matrix cycles busy, where a large library product reaches 1.22 PFLOP/s; the pair of launches 2.9 -> 2.0 ms against
// 2.0 + 0.9 ms of the kernels that recompute.  Ordinary ones the vector unit and the longest workgroup: 32 x 4 heads, d 128, 256..1024
// rows 62 + 21 us, where the query-tile kernel with dS and P took 61 and the kernels that read them 41.  A wavefront with 64 keys and
// all 512 registers, one per SIMD, took as long as this one (1.39 ms at the large shape) and has half as many workgroups.
// With attn_bias a step also clears what its rows do not see and moves the bias to its keys, and the registers are what it is built around: a loop of
// steps with a mask and one of steps without (under one loop the compiler keeps the scores of the block with a mask, 16 registers, through the one
// without), offsets of the transposed reads worked out where they are used (8 registers).  With both in one loop the slot 128 kept four of the eight K
// fragments in scratch memory, and a wait for such a load, whose count is in order, is one for everything asked for before it, the bias and the tiles of
// the next two steps: 16 x 4 heads, d 128, 512..2048 rows 245 us, now 177, the training call 415 -> 340.  (Slots 64 and 256, which did not spill: 0.98 ..
// 1.00 of the time.  Without a bias the unrolled loop of both is the faster one by 1 to 3 %.)
// The query-tile kernel moves dS once: at the large shape 3.8 GB fetched, 2.6 of them dS, in 0.65 ms = 5.8 TB/s.
#pragma once
#include "hstu_bias_requests.h"
#include "hstu_bwd_kernel.hip.h"
#include "hstu_fwd_short_kernel.hip.h"
#include "hstu_pinned_acc.hip.h"

namespace hstu {

// The dS workspace: 2 KiB tiles of 32 query rows x 32 keys, those of a (head, sequence, 32-row group) side by side in key order.
// For a causal mask over equal offsets and bounds of queries and keys without context rows (ds_tri) group g holds the tiles 0 .. g, otherwise all
// ceil(max_k / 32).  Sequences are placed by their first row, 32 rows of slack each, so that the host knows the size without the
// lengths: floor(q0 / 32) + b groups lie ahead of sequence b at most.
// In a tile, row half h2 (16 rows) is 1 KiB: key k's 16 rows (32 bytes) at ((k ^ 4 h2) * 32): the key-tile kernel, which has 8 rows of
// a key in a lane, writes a half with one instruction, and the query-tile kernel reads its operand transposed from a copy in LDS
// without bank conflicts.
constexpr int kDsTileBytes = 2048;
__device__ __forceinline__ int64_t ds_tiles_ahead(const BwdArgs& a, int64_t q0, int b)
{
    const int64_t n_blk = (a.max_k + 31) / 32;
    const int64_t groups = q0 / 32 + b;
    return a.ds_tri ? (groups * (n_blk + 1) + 1) / 2 : groups * n_blk;
}
__device__ __forceinline__ uint8_t* ds_tiles_of(const BwdArgs& a, int64_t q0, int b, int h)
{
    return static_cast<uint8_t*>(a.ds_tiles) + ((h - a.head_first) * a.ds_head_tiles + ds_tiles_ahead(a, q0, b)) * kDsTileBytes;
}
__device__ __forceinline__ uint32_t ds_seq_bytes(const BwdArgs& a, int sq)
{
    const uint32_t groups = static_cast<uint32_t>(sq + 31) >> 5;
    return ((groups * (a.ds_tri ? groups + 1u : 2u * (static_cast<uint32_t>(a.max_k + 31) >> 5))) >> 1) * kDsTileBytes;
}
__device__ __forceinline__ uint32_t ds_group_offset(const BwdArgs& a, int g)
{
    const uint32_t u = static_cast<uint32_t>(g);
    return ((u * (a.ds_tri ? u + 1u : 2u * (static_cast<uint32_t>(a.max_k + 31) >> 5))) >> 1) * kDsTileBytes;
}

// In a masked block, whether element e of a lane (row 8 (e / 4) + e % 4 of the block, 4 more in the upper half-wave) is visible to the
// lane's key, from the rows' bit masks over keys that the lanes 0 .. 31 hold: a row's mask is that of its half-wave's lanes.
__device__ __forceinline__ bool row_sees(uint32_t visible, int e)
{
    const int r = 8 * (e / 4) + e % 4;
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(visible), r));
    const uint32_t up = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(visible), r + 4));
    return __builtin_amdgcn_inverse_ballot_w64((static_cast<uint64_t>(up) << 32) | lo);
}

// 16 bytes of attn_bias per lane straight into registers, as assembly for the reason the tile requests are: the kernel waits for them by
// count.  The registers pass through, so that whatever read them before has been issued, and hold the values once the wait is over.
template <int OFFSET>
__device__ __forceinline__ void request_bias(u32x4_t& dst, u32x4_t rsrc, uint32_t voffset)
{
    asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen offset:%3" : "+v"(dst) : "v"(voffset), "s"(rsrc), "n"(OFFSET));
}

// Clears what hstu_bwd_dq_from_ds_kernel does not write of the attn_bias gradient: in the rows of a 32-row group, the keys past the blocks
// that the group's tiles cover; rows past their sequence whole.  Workgroup `wg` of `n_wgs` takes its share of the groups, a wavefront a
// row at a time.  (max_k a multiple of 8, the gradient on a 16-byte boundary.)
__device__ __forceinline__ void clear_unswept(const BwdArgs& a, int wg, int n_wgs, int wave, int lane)
{
    typedef uint32_t piece_t __attribute__((ext_vector_type(4)));
    const piece_t zero = {0u, 0u, 0u, 0u};
    const int groups = (a.max_q + 31) / 32;
    const int64_t n_items = static_cast<int64_t>(a.n_batch) * a.n_heads_q * groups;
    const int row_pieces = a.max_k / 8;
    for (int64_t item = static_cast<int64_t>(wg) * 4 + wave; item < n_items; item += static_cast<int64_t>(n_wgs) * 4) {
        const int64_t plane = item / groups;
        const int r0 = static_cast<int>(item - plane * groups) * 32;
        const SeqInfo si = load_seq(a, uniform(static_cast<int>(plane / a.n_heads_q)));
        int limit = r0 < si.sq ? (swept_key_limit(a, si, r0) + 31) & ~31 : 0;
        limit = limit < si.sk ? limit : si.sk;
        piece_t* const first = reinterpret_cast<piece_t*>(static_cast<uint16_t*>(a.drab) + (plane * a.max_q + r0) * a.max_k);
        const int rows = a.max_q - r0 < 32 ? a.max_q - r0 : 32;
        if (limit == 0) {  // whole rows: one run
            for (int i = lane; i < rows * row_pieces; i += 64) {
                __builtin_nontemporal_store(zero, first + i);
            }
            continue;
        }
        for (int r = 0; r < rows; ++r) {
            for (int i = (r0 + r < si.sq ? limit / 8 : 0) + lane; i < row_pieces; i += 64) {
                __builtin_nontemporal_store(zero, first + static_cast<int64_t>(r) * row_pieces + i);
            }
        }
    }
}

template <typename Tag, int D, bool HAS_RAB = false>
__global__ __launch_bounds__(kDkvThreads, bwd_kv_fused_wgs_per_cu(D)) void hstu_bwd_kv_fused_kernel(const BwdArgs a)
{
    typedef SubTile<D> T;
    constexpr int LPW = T::LPW, KSTEPS = T::KSTEPS, MTILES = T::MTILES, NCH = 2 * T::MTILES;
    constexpr int kStageElems = 2 * T::ELEMS;  // a Q sub-tile, then a dO sub-tile
    constexpr int kAccRegs = 2 * MTILES * 16;  // dV blocks, then dK blocks
    __shared__ __attribute__((aligned(1024))) uint16_t s_ring[3 * kStageElems];
    __shared__ __attribute__((aligned(1024))) uint16_t s_v[4 * T::ELEMS];  // V rows, a sub-tile per wavefront
    constexpr uint32_t kPastEnd = 0x40000000u;
    constexpr bool kTwoLoops = HAS_RAB;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int ln = lane & 31;
    const int lh = lane >> 5;

    // key tile 0 is seen by the most query rows: heaviest first
    const int grid_heads = a.head_count / a.head_ratio;
    const int per_level = a.n_batch * grid_heads;
    int kt_idx, rem;
    slot_of(a, static_cast<int>(blockIdx.x) - (HAS_RAB ? a.clear_wgs : 0), a.n_ktiles, per_level, kt_idx, rem);
    const int b = rem / grid_heads;
    const int hk = a.head_first / a.head_ratio + rem - b * grid_heads;
    zero_tail_rows(a.dk, a.offs_k, a.n_batch, a.idx64, a.total_k, static_cast<int64_t>(a.n_heads_k) * a.d_qk, kDkvThreads);
    zero_tail_rows(a.dv, a.offs_k, a.n_batch, a.idx64, a.total_k, static_cast<int64_t>(a.n_heads_k) * a.d_v, kDkvThreads);
    if constexpr (HAS_RAB) {
        if (static_cast<int>(blockIdx.x) < a.clear_wgs) {
            if (a.bias_vec_ok == 2) {
                clear_unswept(a, static_cast<int>(blockIdx.x), a.clear_wgs, wave, lane);
            } else {
                clear_share(a.drab, a.drab_clear_bytes, blockIdx.x, static_cast<unsigned>(a.clear_wgs), tid, kDkvThreads);
            }
            return;
        }
    }
    if (rem >= per_level) {
        return;
    }
    const SeqInfo si = load_seq(a, b);
    const int sq = si.sq, sk = si.sk;
    const int c0 = kt_idx * kBlockM;
    if (c0 >= sk) {
        return;
    }
    const int cw0 = c0 + wave * 32;

    const uint32_t q_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_qk * 2u;
    const uint32_t g_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_v * 2u;
    const uint32_t k_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_qk * 2u;
    const uint32_t v_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_v * 2u;
    const uint32_t k_bytes = static_cast<uint32_t>(sk - 1) * k_stride + a.d_qk * 2u;
    const uint32_t v_bytes = static_cast<uint32_t>(sk - 1) * v_stride + a.d_v * 2u;
    const int64_t k_first = (si.k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_qk) * 2;
    const int64_t v_first = (si.k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_v) * 2;

    uint32_t q_src[LPW], g_src[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const int slot = (wave * LPW + i) * 64 + lane;
        const int r = (slot / T::CPR) & 31;
        const int cs = both_ways_swizzle<D>(r, slot % T::CPR);
        q_src[i] = (cs * 8 < a.d_qk) ? static_cast<uint32_t>(r) * q_stride + cs * 16u : kOutOfRange;
        g_src[i] = (cs * 8 < a.d_v) ? static_cast<uint32_t>(r) * g_stride + cs * 16u : kOutOfRange;
    }
    // plain read of row ln: the chunk of MFMA step js is that of step 0 with the bits of 2 js flipped (the swizzle is an XOR), so one
    // register serves all steps; the offsets are worked out where they are used, because KSTEPS more registers are not to be had
    const int n_first_off = (ln * D + both_ways_swizzle<D>(ln, lh) * 8) * 2;  // (in bytes)
    int t_lane_off[MTILES][2];
    {
        const int vr0 = 4 * lh + ((lane & 15) >> 2);
#pragma unroll
        for (int mt = 0; mt < MTILES; ++mt) {
            const int col = 32 * mt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
            t_lane_off[mt][0] = vr0 * D + both_ways_swizzle<D>(vr0, col >> 3) * 8 + (col & 7);
            t_lane_off[mt][1] = (vr0 + 8) * D + both_ways_swizzle<D>(vr0 + 8, col >> 3) * 8 + (col & 7);
        }
    }

    // query sub-tiles that can see a key of this tile (as in hstu_bwd_dkv_kernel)
    const int n_qsub = (sq + 31) / 32;
    int x_first = 0;
    int x_skip_from = -1, x_skip_to = -1;
    if (a.mask_type == 0) {
        const int first_row = c0 - si.delta;
        const int x_causal = first_row > 0 ? first_row / 32 : 0;
        if (si.n_ctx > 0 && c0 < si.hist_k) {
            const int ctx_end = ((si.n_ctx < sq ? si.n_ctx : sq) + 31) / 32;
            if (x_causal > ctx_end) {
                x_skip_from = ctx_end;
                x_skip_to = x_causal < n_qsub ? x_causal : n_qsub;
            }
        } else {
            x_first = x_causal;
        }
    }
    const int nx = (n_qsub > x_first ? n_qsub - x_first : 0) - (x_skip_to - x_skip_from);
    const int n_iter = nx * a.head_ratio;

    // The next request and the current step: query head, its descriptors, query sub-tile.  Nothing is worked out per step that
    // changes with the head only.
    const int first_h = hk * a.head_ratio;
    const uint32_t q_bytes = static_cast<uint32_t>(sq - 1) * q_stride + a.d_qk * 2u;
    const uint32_t g_bytes = static_cast<uint32_t>(sq - 1) * g_stride + a.d_v * 2u;
    const uint8_t* q_head = static_cast<const uint8_t*>(a.q) + (si.q0 * a.n_heads_q + first_h) * static_cast<int64_t>(a.d_qk) * 2;
    const uint8_t* g_head = static_cast<const uint8_t*>(a.grad) + (si.q0 * a.n_heads_q + first_h) * static_cast<int64_t>(a.d_v) * 2;
    const uint8_t* ds_head = ds_tiles_of(a, si.q0, b, first_h);
    const uint32_t ds_bytes = ds_seq_bytes(a, sq);
    int req_left = n_iter, req_x = x_first;
    int cur_x = x_first;
    const uint32_t ring_lds = lds_address(s_ring) + static_cast<uint32_t>(wave) * (LPW * 1024u);
    auto request = [&](int stage) {
        // (past the last one: sent out of range -- moves no data, keeps the count per step constant)
        const u32x4_t q_rsrc = make_rsrc_words(q_head, q_bytes);
        const u32x4_t g_rsrc = make_rsrc_words(g_head, g_bytes);
        const uint32_t qb = req_left > 0 ? static_cast<uint32_t>(req_x * 32) * q_stride : kPastEnd;
        const uint32_t gb = req_left > 0 ? static_cast<uint32_t>(req_x * 32) * g_stride : kPastEnd;
        const uint32_t base = ring_lds + static_cast<uint32_t>(stage) * (kStageElems * 2u);
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            request_to_lds_b128(q_rsrc, base + i * 1024u, q_src[i] + qb);
            request_to_lds_b128(g_rsrc, base + T::ELEMS * 2u + i * 1024u, g_src[i] + gb);
        }
        --req_left;
        if (++req_x == x_skip_from) {
            req_x = x_skip_to;
        }
        if (req_x >= n_qsub) {
            req_x = x_first;
            if (req_left > 0) {
                q_head += a.d_qk * 2;
                g_head += a.d_v * 2;
            }
        }
    };
    // attn_bias of the next step's block: lane (ln, lh) has row ln, keys 8 lh .. + 7 and 16 + 8 lh .. + 7 (past the row's end the next row's:
    // a step drops what the row does not see)
    u32x4_t bias[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
    BiasRequests wanted;
    wanted.plane = reinterpret_cast<uint64_t>(a.rab) + (HAS_RAB ? bias_plane_of(a, b, first_h) * 2 : 0);
    wanted.pitch = static_cast<uint32_t>(a.max_k) * 2u;
    wanted.size = static_cast<uint32_t>(a.max_q) * wanted.pitch;
    wanted.x = wanted.first = x_first;
    wanted.skip_from = x_skip_from;
    wanted.skip_to = x_skip_to;
    wanted.end = n_qsub;
    wanted.left = n_iter;
    wanted.set_lane(a.max_k, cw0, ln, lh);
    auto next_bias = [&]() {
        const u32x4_t rsrc = make_rsrc_words(reinterpret_cast<const uint8_t*>(wanted.plane), wanted.bytes());
        const uint32_t off = wanted.offset();
        request_bias<0>(bias[0], rsrc, off);
        request_bias<32>(bias[1], rsrc, off);
        wanted.advance();
    };
    // The product with a 0/1 matrix that moves a lane's pieces to its keys (see hstu_bwd_dkv_kernel): the element of k-slot (lh, e) of
    // product j that is 1 is e = ln - 16 j - 8 lh.  Eight registers for the whole sweep are not to be had: a block works it out.
    const uint32_t one = (std::is_same<Tag, bf16_tag>::value ? 0x3f80u : 0x3c00u) << (16 * (ln & 1));  // 1.0 in the input type, in its half
    const int one_word = (ln - 8 * lh) >> 1;  // (8 lh is even; words 0 .. 3 of product 0, 8 .. 11 of product 1)
    // The sub-tiles all of whose rows see all keys of this wavefront: from the first whose first row does, past the context rows, up to
    // those with target rows or without 32 rows.  The others take the general path.
    int full_from = n_qsub, full_to = 0;
    if (cw0 + 32 <= sk) {
        full_from = 0;
        full_to = sq >> 5;
        if (a.mask_type == 0) {
            const int row = cw0 + 31 - si.delta;  // the first row that sees the last of these keys
            full_from = row > 0 ? (row + 31) >> 5 : 0;
            const int past_ctx = (si.n_ctx + 31) >> 5;
            full_from = full_from > past_ctx ? full_from : past_ctx;
            if (si.n_tgt > 0) {
                const int rows = sq > si.n_tgt ? sq - si.n_tgt : 0;
                full_to = rows >> 5;
            }
        }
    }

    acc_fence<kAccRegs>();
    acc_zero_all(std::make_integer_sequence<int, kAccRegs>{});
    const ScoreConsts sconst = score_consts(a.alpha, a.scale);
    u32x4_t kf[KSTEPS];
    if (n_iter > 0) {
        if constexpr (HAS_RAB) {
            next_bias();
        }
        request(0);
        request(1);
        const u32x4_t v_rsrc = make_rsrc_words(static_cast<const uint8_t*>(a.v) + v_first, v_bytes);
        const uint32_t v_lds = lds_address(s_v) + static_cast<uint32_t>(wave) * (T::ELEMS * 2u);
#pragma unroll
        for (int i = 0; i < T::KIB; ++i) {
            const int slot = i * 64 + lane;
            const int r = slot / T::CPR;
            const int cs = both_ways_swizzle<D>(r, slot % T::CPR);
            request_to_lds_b128(v_rsrc, v_lds + i * 1024u, (cs * 8 < a.d_v) ? static_cast<uint32_t>(cw0 + r) * v_stride + cs * 16u : kOutOfRange);
        }
        const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(static_cast<const uint8_t*>(a.k) + k_first, k_bytes);
        const uint32_t k_off = static_cast<uint32_t>(cw0 + ln) * k_stride;
#pragma unroll
        for (int js = 0; js < KSTEPS; ++js) {
            const int d0 = 16 * js + 8 * lh;
            kf[js] = __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, static_cast<int>(d0 < a.d_qk ? k_off + d0 * 2u : kOutOfRange), 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0);  // (everything, once: the compiler does not know of the requests in assembly)
        if constexpr (HAS_RAB) {
            asm volatile("" : "+v"(bias[0]), "+v"(bias[1]));
        }
    }

    auto read_n = [&](const uint16_t* tile, int first_off, int js) -> u32x4_t {
        return *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint8_t*>(tile) + (first_off ^ (js * 32)));
    };
    uint32_t t_off[2] = {0, 0};  // (kTwoLoops) bytes from the ring's first stage
    auto read_t = [&](const uint16_t* tile, int c) -> u32x4_t {
        const int j2 = c / MTILES, mt = c % MTILES;
        u32x2_t lo, hi;
        if constexpr (kTwoLoops) {
            // (the output tile's bits flipped where it is read: offsets worked out ahead are registers that are not to be had)
            uint32_t o[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                asm volatile("v_xor_b32 %0, %2, %1" : "=v"(o[i]) : "v"(t_off[i]), "n"(64 * mt));
                o[i] += 32u * j2 * D;
            }
            lo = lds_read_tr16_b64(reinterpret_cast<const uint16_t*>(reinterpret_cast<const uint8_t*>(tile) + o[0]));
            hi = lds_read_tr16_b64(reinterpret_cast<const uint16_t*>(reinterpret_cast<const uint8_t*>(tile) + o[1]));
        } else {
            lo = lds_read_tr16_b64(tile + t_lane_off[mt][0] + 16 * j2 * D);
            hi = lds_read_tr16_b64(tile + t_lane_off[mt][1] + 16 * j2 * D);
        }
        const u32x4_t r = {lo[0], lo[1], hi[0], hi[1]};
        return r;
    };
    auto quad = [](const uint32_t (&w)[8], int j2) -> u32x4_t {
        const u32x4_t r = {w[4 * j2], w[4 * j2 + 1], w[4 * j2 + 2], w[4 * j2 + 3]};
        return r;
    };
    int cur_stage = 0;  // (kTwoLoops) the current step's
    const uint32_t ds_lane = static_cast<uint32_t>(ln * 32 + lh * 16);
#define HSTU_FENCE() __builtin_amdgcn_sched_barrier(0)

    // (masked blocks) lane = row: its visible keys
    auto rows_see = [&](int rq0) -> uint32_t { return row_sees_keys(si, a.mask_type, a.target_group, rq0 + ln, cw0); };

    auto block = [&](auto masked, const uint16_t* q_tile, int rq0, const f32x16_t& s_first) {
        constexpr bool kMasked = decltype(masked)::value;
        const uint16_t* const g_tile = q_tile + T::ELEMS;
        uint32_t pk[8], ds[8];
        f32x16_t s, dp;
        // The operands that come from LDS, kAhead slots of one MFMA ahead of their use across the phases: Q plain, dO plain, dO and Q
        // transposed; V, which only dP reads, kAheadV slots ahead.
        constexpr int kAhead = HAS_RAB ? 1 : 2, kAheadV = HAS_RAB ? 1 : 2;
        u32x4_t op[kAhead + 1], vo[kAheadV + 1];
        acc_fence<kAccRegs>();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = 0.f;
            dp[i] = 0.f;
        }
        if constexpr (HAS_RAB) {
            s = s_first;
        }
        uint32_t visible = 0;
        if constexpr (kMasked) {
            visible = rows_see(rq0);
        }
        int n_off = n_first_off;
        asm volatile("" : "+v"(n_off));  // (not to be worked out ahead of the sweep)
        if constexpr (kTwoLoops) {
            const uint32_t at = static_cast<uint32_t>(cur_stage) * (kStageElems * 2u);
            t_off[0] = 2u * t_lane_off[0][0] + at;
            t_off[1] = 2u * t_lane_off[0][1] + at;
            asm volatile("" : "+v"(t_off[0]), "+v"(t_off[1]));
            n_off += static_cast<int>(at);
            asm volatile("" : "+v"(n_off));
        }
        int v_off = wave * T::ELEMS * 2 + n_first_off;
        asm volatile("" : "+v"(v_off));
        auto fetch = [&](int k) {  // operand of slot k
            if (k < KSTEPS) {
                op[k % (kAhead + 1)] = read_n(q_tile, n_off, k);
            } else if (k < 2 * KSTEPS) {
                op[k % (kAhead + 1)] = read_n(g_tile, n_off, k - KSTEPS);
            } else if (k < 2 * KSTEPS + NCH) {
                op[k % (kAhead + 1)] = read_t(g_tile, k - 2 * KSTEPS);
            } else if (k < 2 * KSTEPS + 2 * NCH) {
                op[k % (kAhead + 1)] = read_t(q_tile, k - 2 * KSTEPS - NCH);
            }
        };
        auto fetch_v = [&](int js) {
            if (js >= 0 && js < KSTEPS) {
                vo[js % (kAheadV + 1)] = read_n(s_v, v_off, js);
            }
        };
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            fetch(k);
        }
        HSTU_FENCE();
#pragma unroll
        for (int js = 0; js < KSTEPS; ++js) {
            fetch(js + kAhead);
            fetch_v(js + kAheadV - KSTEPS);
            HSTU_FENCE();
            s = mfma32<Tag>(op[js % (kAhead + 1)], kf[js], s);
            asm volatile("" : "+v"(s));
            HSTU_FENCE();
        }
        // scores: two elements at a time from S to P and f (dS = f dP; f takes S's place), in two parts
        float t[2];
        auto part = [&](int k) {
            const int i = k / 2;
            if (k % 2 == 0) {
#pragma unroll
                for (int e2 = 0; e2 < 2; ++e2) {
                    t[e2] = __builtin_amdgcn_exp2f(s[2 * i + e2] * sconst.c_exp);
                }
#pragma unroll
                for (int e2 = 0; e2 < 2; ++e2) {
                    t[e2] = __builtin_fmaf(t[e2], sconst.ci, sconst.ci);
                }
                asm volatile("" : "+v"(t[0]), "+v"(t[1]));  // (keeps the part in its slot)
            } else {
                float p[2];
#pragma unroll
                for (int e2 = 0; e2 < 2; ++e2) {
                    t[e2] = __builtin_amdgcn_rcpf(t[e2]);
                }
#pragma unroll
                for (int e2 = 0; e2 < 2; ++e2) {
                    p[e2] = s[2 * i + e2] * t[e2];
                    s[2 * i + e2] = __builtin_fmaf(p[e2], __builtin_fmaf(-t[e2], sconst.inv_scale, sconst.alpha), t[e2]);
                }
                if constexpr (kMasked) {
#pragma unroll
                    for (int e2 = 0; e2 < 2; ++e2) {
                        p[e2] = row_sees(visible, 2 * i + e2) ? p[e2] : 0.f;
                    }
                }
                pk[i] = pack2<Tag>(p[0], p[1]);
                asm volatile("" : "+v"(pk[i]));
            }
        };
        // slot g of the 2 NCH behind S: how many of the 16 parts are done at its end
        constexpr int kSlots = KSTEPS + NCH / 2;  // (the last words of P are read by the second half of dV's chunks)
        auto parts_done = [](int g) constexpr {
            const int n = g < 1 ? 0 : (g * 16 + kSlots - 3) / (kSlots - 2);
            return n < 16 ? n : 16;
        };
        auto scores_of_slot = [&](int g) {
#pragma unroll
            for (int k = g > 0 ? parts_done(g - 1) : 0; k < parts_done(g); ++k) {
                part(k);
            }
        };
#pragma unroll
        for (int js = 0; js < KSTEPS; ++js) {
            fetch(KSTEPS + js + kAhead);
            fetch_v(js + kAheadV);
            HSTU_FENCE();
            dp = mfma32<Tag>(op[(KSTEPS + js) % (kAhead + 1)], vo[js % (kAheadV + 1)], dp);
            asm volatile("" : "+v"(dp));
            HSTU_FENCE();
            scores_of_slot(js);
            HSTU_FENCE();
        }
        acc_fence<kAccRegs>();
        HSTU_FENCE();
        static_for<NCH>([&](auto ci) {
            constexpr int c = ci;
            fetch(2 * KSTEPS + c + kAhead);
            HSTU_FENCE();
            acc_mfma<Tag, c % MTILES>(op[(2 * KSTEPS + c) % (kAhead + 1)], quad(pk, c / MTILES));
            HSTU_FENCE();
            scores_of_slot(KSTEPS + c);
            if constexpr (c >= NCH / 2) {
                constexpr int slot = c - NCH / 2;
#pragma unroll
                for (int i = slot * 16 / NCH; i < (slot + 1) * 16 / NCH; ++i) {
                    float v[2];
#pragma unroll
                    for (int e2 = 0; e2 < 2; ++e2) {
                        v[e2] = s[2 * i + e2] * dp[2 * i + e2];
                        if constexpr (kMasked) {
                            v[e2] = row_sees(visible, 2 * i + e2) ? v[e2] : 0.f;
                        }
                    }
                    ds[i] = pack2<Tag>(v[0], v[1]);
                    asm volatile("" : "+v"(ds[i]));
                }
            }
            HSTU_FENCE();
        });
        acc_fence<kAccRegs>();
        // dS to the workspace: the two lanes of a key trade halves, 8 rows each
        {
            typedef __attribute__((ext_vector_type(2))) unsigned u2_t;
            const __amdgpu_buffer_rsrc_t ds_rsrc = make_rsrc(ds_head, ds_bytes);
            const uint32_t tile = ds_group_offset(a, rq0 >> 5) + static_cast<uint32_t>(cw0 >> 5) * kDsTileBytes;
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                const u2_t d0 = __builtin_amdgcn_permlane32_swap(ds[4 * h2 + 0], ds[4 * h2 + 2], false, false);
                const u2_t d1 = __builtin_amdgcn_permlane32_swap(ds[4 * h2 + 1], ds[4 * h2 + 3], false, false);
                const u32x4_t w = {d0[0], d1[0], d0[1], d1[1]};
                // (the tile's offset in the vector offset: with a scalar register as the scalar offset the compiler leaves no wait state
                // between the store and the next write of its data registers, and such stores were seen to take the later values)
                __builtin_amdgcn_raw_buffer_store_b128(w, ds_rsrc, static_cast<int>((ds_lane ^ (128u * h2)) + 1024u * h2 + tile), 0, 0);
            }
        }
        acc_fence<kAccRegs>();
        HSTU_FENCE();
        static_for<NCH>([&](auto ci) {
            constexpr int c = ci;
            fetch(2 * KSTEPS + NCH + c + kAhead);
            HSTU_FENCE();
            acc_mfma<Tag, MTILES + c % MTILES>(op[(2 * KSTEPS + NCH + c) % (kAhead + 1)], quad(ds, c / MTILES));
            HSTU_FENCE();
        });
    };

    auto step = [&](auto kind, const uint16_t* q_tile, int stage_o) {
        constexpr int kKind = decltype(kind)::value;  // 0: masked or not by the sub-tile; 1: no block of it masked; 2: all
        // this step's sub-tile has landed for everybody; the stage of the previous step is free
        acc_fence<kAccRegs>();
        HSTU_FENCE();
        if constexpr (HAS_RAB) {
            asm volatile("s_waitcnt vmcnt(%2)" : "+v"(bias[0]), "+v"(bias[1]) : "n"(2 * LPW) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LPW) : "memory");
        }
        __builtin_amdgcn_s_barrier();
        HSTU_FENCE();
        f32x16_t s;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = 0.f;
        }
        const int x = cur_x;
        const bool masked = kKind == 2 || (kKind == 0 && (x < full_from || x >= full_to));
        if constexpr (HAS_RAB) {
            // the matrix pipe transposes the bias into the scores' accumulators; its registers take the next block's at once
            int word = one_word;
            asm volatile("" : "+v"(word));
            u32x4_t route[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    route[j][i] = word == 8 * j + i ? one : 0u;
                }
            }
            if (masked) {
                // (A lane holds its row's bias, so the row's bit mask is at hand.  This side of next_bias(): behind it, where branches meet, the
                // compiler would copy registers that the request still fills.)
                clear_unseen(bias, static_cast<int>(rows_see(x * 32) >> (8 * lh)));
            }
            s = mfma32<Tag>(bias[0], route[0], s);
            s = mfma32<Tag>(bias[1], route[1], s);
            asm volatile("" : "+v"(s));
            HSTU_FENCE();
            next_bias();
        }
        request(stage_o);
        HSTU_FENCE();
        if (!masked) {
            block(std::false_type{}, q_tile, x * 32, s);
        } else if (cw0 < swept_key_limit(a, si, x * 32)) {  // (otherwise nothing is visible: the query-tile kernel does not read this tile)
            block(std::true_type{}, q_tile, x * 32, s);
        }
        if (++cur_x == x_skip_from) {
            cur_x = x_skip_to;
        }
        if (cur_x >= n_qsub) {
            cur_x = x_first;
            ds_head += a.ds_head_tiles * kDsTileBytes;
        }
    };

    if (n_iter > 0) {
        [[maybe_unused]] constexpr std::integral_constant<int, 0> any{};
        int it = 0;
        if constexpr (kTwoLoops) {
            auto next = [&]() {
                cur_stage = cur_stage == 2 ? 0 : cur_stage + 1;
                ++it;
            };
            while (it < n_iter) {
                while (it < n_iter && cur_x >= full_from && cur_x < full_to) {
                    step(std::integral_constant<int, 1>{}, s_ring, cur_stage == 0 ? 2 : cur_stage - 1);
                    next();
                }
                while (it < n_iter && (cur_x < full_from || cur_x >= full_to)) {
                    step(std::integral_constant<int, 2>{}, s_ring, cur_stage == 0 ? 2 : cur_stage - 1);
                    next();
                }
            }
        }
        while (!kTwoLoops) {  // (step it reads stage it mod 3 and has stage (it + 2) mod 3 filled)
            step(any, s_ring, 2);
            if (++it >= n_iter) {
                break;
            }
            step(any, s_ring + kStageElems, 0);
            if (++it >= n_iter) {
                break;
            }
            step(any, s_ring + 2 * kStageElems, 1);
            if (++it >= n_iter) {
                break;
            }
        }
    }

    if constexpr (HAS_RAB) {
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(bias[0]), "+v"(bias[1]) : : "memory");  // (the last request lands before its registers are used again)
    }
    acc_settle();
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    typedef std::make_integer_sequence<int, 16> Regs;
    uint16_t* const stage = s_ring + wave * T::ELEMS;
    auto store = [&](auto first, const void* out, int64_t first_byte, uint32_t bytes, uint32_t stride, int dims) {
        f32x16_t acc[MTILES];
        static_for<MTILES>([&](auto mt) { acc[mt] = acc_block<decltype(first)::value + mt>(Regs{}); });
        const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(static_cast<const uint8_t*>(out) + first_byte, bytes);
        if (a.grad_vec_ok == 0) {
            store_tile_pieces<Tag, D>(acc, rsrc, static_cast<uint32_t>(cw0) * stride, stride, dims, lane);
            return;
        }
        store_tile_rows<Tag, D>(stage, acc, rsrc, static_cast<uint32_t>(cw0) * stride, stride, dims, lane);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    store(std::integral_constant<int, 0>{}, a.dv, v_first, v_bytes, v_stride, a.d_v);
    store(std::integral_constant<int, MTILES>{}, a.dk, k_first, k_bytes, k_stride, a.d_qk);
}

#undef HSTU_FENCE

// WANT_DRAB: the dS values are written to the attn_bias gradient as well (cleared by the key-tile kernel of the launch before)
template <typename Tag, int D, bool WANT_DRAB>
__global__ __launch_bounds__(256, bwd_dq_from_ds_wgs_per_cu(D)) void hstu_bwd_dq_from_ds_kernel(const BwdArgs a)
{
    typedef SubTile<D> T;
    constexpr int LPW = T::LPW, MTILES = T::MTILES, NCH = 2 * T::MTILES;
    constexpr int kStageElems = T::ELEMS + 4 * (kDsTileBytes / 2);  // a K sub-tile, then the wavefronts' dS tiles
    __shared__ __attribute__((aligned(1024))) uint16_t s_ring[3 * kStageElems];
    constexpr uint32_t kPastEnd = 0x40000000u;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int ln = lane & 31;
    const int lh = lane >> 5;

    // heaviest (last) query tiles first; with context rows the first tile of a sequence, which sweeps all of its history keys, ahead
    const int per_level = a.n_batch * a.head_count;
    int lvl, rem;
    slot_of(a, static_cast<int>(blockIdx.x), a.n_qtiles, per_level, lvl, rem);
    const int n_levels = live_levels(a, lane, kBlockM, a.n_qtiles);
    const int qt = (a.mask_type == 0 && a.num_ctx != nullptr) ? (lvl == 0 ? 0 : n_levels - lvl) : n_levels - 1 - lvl;
    const int b = rem / a.head_count;
    const int h = a.head_first + rem - b * a.head_count;
    const int hk = h / a.head_ratio;
    zero_tail_rows(a.dq, a.offs_q, a.n_batch, a.idx64, a.total_q, static_cast<int64_t>(a.n_heads_q) * a.d_qk, 256);
    if (lvl >= n_levels || rem >= per_level) {
        return;  // a level that no sequence of the batch has, or a slot past the last pair
    }
    const SeqInfo si = load_seq(a, b);
    const int sq = si.sq, sk = si.sk;
    const int r0 = qt * kBlockM;
    if (r0 >= sq) {
        return;
    }
    const int wr0 = r0 + wave * kWaveM;

    const uint32_t q_stride = static_cast<uint32_t>(a.n_heads_q) * a.d_qk * 2u;
    const uint32_t k_stride = static_cast<uint32_t>(a.n_heads_k) * a.d_qk * 2u;
    const u32x4_t k_rsrc = make_rsrc_words(static_cast<const uint8_t*>(a.k) + (si.k0 * a.n_heads_k + hk) * static_cast<int64_t>(a.d_qk) * 2,
                                           sk > 0 ? static_cast<uint32_t>(sk - 1) * k_stride + a.d_qk * 2u : 0u);
    const u32x4_t ds_rsrc = make_rsrc_words(ds_tiles_of(a, si.q0, b, h), ds_seq_bytes(a, sq));
    uint32_t k_src[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const int slot = (wave * LPW + i) * 64 + lane;
        const int r = (slot / T::CPR) & 31;
        const int cs = both_ways_swizzle<D>(r, slot % T::CPR);
        k_src[i] = (cs * 8 < a.d_qk) ? static_cast<uint32_t>(r) * k_stride + cs * 16u : kOutOfRange;
    }
    int t_lane_off[MTILES][2];
    const int vr0 = 4 * lh + ((lane & 15) >> 2);
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt) {
        const int col = 32 * mt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        t_lane_off[mt][0] = vr0 * D + both_ways_swizzle<D>(vr0, col >> 3) * 8 + (col & 7);
        t_lane_off[mt][1] = (vr0 + 8) * D + both_ways_swizzle<D>(vr0 + 8, col >> 3) * 8 + (col & 7);
    }
    // transposed read of the dS tile: lane = row (half (lane >> 4) & 1 of 16), keys vr0 (+ 8) (+ 16 j2)
    const int ds_half = (lane >> 4) & 1;
    const int ds_lane_off = ds_half * 512 + (vr0 ^ (4 * ds_half)) * 16 + 4 * (lane & 3);

    // keys needed by this tile
    int kmax;
    if (a.mask_type == 0) {
        const int r1 = (r0 + kBlockM < sq) ? r0 + kBlockM : sq;
        kmax = r1 + si.delta;
        if (r0 < si.n_ctx) {
            kmax = kmax > si.hist_k ? kmax : si.hist_k;
        }
        kmax = kmax < 0 ? 0 : (kmax > sk ? sk : kmax);
    } else {
        kmax = sk;
    }
    const int n_sub = (kmax + 31) / 32;
    const int nx_w = (swept_key_limit(a, si, wr0) + 31) / 32;
    const uint32_t ds_first = ds_group_offset(a, wr0 >> 5) + lane * 16u;

    const uint32_t bias_bytes = static_cast<uint32_t>(a.max_q) * static_cast<uint32_t>(a.max_k) * 2u;
    const __amdgpu_buffer_rsrc_t drab_rsrc =
        make_rsrc(WANT_DRAB ? static_cast<uint16_t*>(a.drab) + bias_plane_of(a, b, h) : nullptr, WANT_DRAB ? bias_bytes : 0u);
    // 8 keys of a row of the gradient, up to the sequence's last; `end`: the first key past those that the wavefront writes now
    auto store_piece = [&](const u32x4_t& w, int row, int key, int end) {
        const uint32_t off = (static_cast<uint32_t>(row) * static_cast<uint32_t>(a.max_k) + static_cast<uint32_t>(key)) * 2u;
        const bool write = row < sq && key < sk;
        __builtin_amdgcn_raw_buffer_store_b128(w, drab_rsrc, static_cast<int>(write && key + 8 <= a.max_k ? off : kOutOfRange), 0, 0);
        if (end > a.max_k) {  // (a piece that would reach into the next row: its keys one by one)
            const bool part = write && key + 8 > a.max_k;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint16_t value = static_cast<uint16_t>(e % 2 ? w[e / 2] >> 16 : w[e / 2] & 0xffffu);
                __builtin_amdgcn_raw_buffer_store_b16(value, drab_rsrc, static_cast<int>(part && key + e < sk ? off + 2u * e : kOutOfRange), 0, 0);
            }
        }
    };

    f32x16_t acc[MTILES];
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc[mt][i] = 0.f;
        }
    }
    u32x4_t even[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};  // (WANT_DRAB) the pieces of an even step, until the odd one's are there
    const uint32_t ring_lds = lds_address(s_ring);
    auto request = [&](int stage, int x) {
        const uint32_t base = ring_lds + static_cast<uint32_t>(stage) * (kStageElems * 2u);
        const uint32_t kb = x < n_sub ? static_cast<uint32_t>(x * 32) * k_stride : kPastEnd;
        const uint32_t db = x < nx_w ? ds_first + static_cast<uint32_t>(x) * kDsTileBytes : kOutOfRange;
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            request_to_lds_b128(k_rsrc, base + (static_cast<uint32_t>(wave) * LPW + i) * 1024u, k_src[i] + kb);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            request_to_lds_b128(ds_rsrc, base + T::ELEMS * 2u + static_cast<uint32_t>(wave) * kDsTileBytes + i * 1024u, db + i * 1024u);
        }
    };
    auto step = [&](const uint16_t* k_tile, int stage_o, int x) {
        // sub-tile x has landed for everybody, the stage of step x - 1 is free
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW + 2) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        request(stage_o, x + 2);
        __builtin_amdgcn_sched_barrier(0);
        if (x >= nx_w) {
            return;  // nothing of this sub-tile is visible to the rows of this wavefront
        }
        const uint16_t* const ds_tile = k_tile + T::ELEMS + wave * (kDsTileBytes / 2);
        uint32_t pk[8];
#pragma unroll
        for (int j2 = 0; j2 < 2; ++j2) {
            const u32x2_t lo = lds_read_tr16_b64(ds_tile + ds_lane_off + 16 * j2 * 16);
            const u32x2_t hi = lds_read_tr16_b64(ds_tile + ds_lane_off + (16 * j2 + 8) * 16);
            pk[4 * j2 + 0] = lo[0];
            pk[4 * j2 + 1] = lo[1];
            pk[4 * j2 + 2] = hi[0];
            pk[4 * j2 + 3] = hi[1];
        }
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int j2 = c / MTILES, mt = c % MTILES;
            const u32x2_t lo = lds_read_tr16_b64(k_tile + t_lane_off[mt][0] + 16 * j2 * D);
            const u32x2_t hi = lds_read_tr16_b64(k_tile + t_lane_off[mt][1] + 16 * j2 * D);
            const u32x4_t kt = {lo[0], lo[1], hi[0], hi[1]};
            const u32x4_t pb = {pk[4 * j2 + 0], pk[4 * j2 + 1], pk[4 * j2 + 2], pk[4 * j2 + 3]};
            acc[mt] = mfma32<Tag>(kt, pb, acc[mt]);
        }
        if constexpr (WANT_DRAB) {
            // The two lanes of a row trade halves (see store_bias_row_values): 8 keys of a row per lane and piece.  Rows start at multiples
            // of four bytes, which is what a 16-byte store needs.
            typedef __attribute__((ext_vector_type(2))) unsigned u2_t;
            u32x4_t now[2];
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                const u2_t d0 = __builtin_amdgcn_permlane32_swap(pk[4 * h2 + 0], pk[4 * h2 + 2], false, false);
                const u2_t d1 = __builtin_amdgcn_permlane32_swap(pk[4 * h2 + 1], pk[4 * h2 + 3], false, false);
                now[h2] = u32x4_t{d0[0], d1[0], d0[1], d1[1]};
            }
            if (a.drab_lines == 0 || ((x & 1) == 0 && x + 1 >= nx_w)) {
#pragma unroll
                for (int h2 = 0; h2 < 2; ++h2) {
                    store_piece(now[h2], wr0 + ln, x * 32 + 16 * h2 + 8 * lh, x * 32 + 32);
                }
            } else {
                // Whole lines: the blocks of an even step and the odd one behind it leave together, 64 keys = 128 bytes of a row, eight
                // rows an instruction.  The pieces go through the wavefront's own dS tile of this step, whose values are in registers
                // by now, 16 rows at a time.
                if ((x & 1) == 0) {
                    even[0] = now[0];
                    even[1] = now[1];
                    return;
                }
                uint8_t* const stage = reinterpret_cast<uint8_t*>(const_cast<uint16_t*>(ds_tile));
                const int c0 = (x - 1) * 32;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    if ((ln >> 4) == half) {
                        const int r = ln & 15;
#pragma unroll
                        for (int h2 = 0; h2 < 2; ++h2) {
                            *reinterpret_cast<u32x4_t*>(stage + r * 128 + (((2 * h2 + lh) ^ (r & 7)) * 16)) = even[h2];
                            *reinterpret_cast<u32x4_t*>(stage + r * 128 + (((4 + 2 * h2 + lh) ^ (r & 7)) * 16)) = now[h2];
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const int r = i * 8 + (lane >> 3);
                        const u32x4_t piece = *reinterpret_cast<const u32x4_t*>(stage + r * 128 + (((lane & 7) ^ (r & 7)) * 16));
                        store_piece(piece, wr0 + 16 * half + r, c0 + 8 * (lane & 7), c0 + 64);
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
            }
        }
    };
    if (n_sub > 0) {
        request(0, 0);
        request(1, 1);
        int x = 0;
        while (true) {  // (step x reads stage x mod 3 and has stage (x + 2) mod 3 filled)
            step(s_ring, 2, x);
            if (++x >= n_sub) {
                break;
            }
            step(s_ring + kStageElems, 0, x);
            if (++x >= n_sub) {
                break;
            }
            step(s_ring + 2 * kStageElems, 1, x);
            if (++x >= n_sub) {
                break;
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const __amdgpu_buffer_rsrc_t dq_rsrc =
        make_rsrc(static_cast<uint8_t*>(a.dq) + (si.q0 * a.n_heads_q + h) * static_cast<int64_t>(a.d_qk) * 2,
                  static_cast<uint32_t>(sq - 1) * q_stride + a.d_qk * 2u);
    if (a.grad_vec_ok == 0) {
        store_tile_pieces<Tag, D>(acc, dq_rsrc, static_cast<uint32_t>(wr0) * q_stride, q_stride, a.d_qk, lane);
        return;
    }
    store_tile_rows<Tag, D>(s_ring + wave * T::ELEMS, acc, dq_rsrc, static_cast<uint32_t>(wr0) * q_stride, q_stride, a.d_qk, lane);
}

}  // namespace hstu
