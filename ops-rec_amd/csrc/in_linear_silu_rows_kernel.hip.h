// in_linear_silu forward for gfx950 with the weights in registers: the kernel for many rows and k of 129 to 512.
//
// Same outputs and rounding points as in_linear_silu_kernel (in_linear_silu_kernel.hip.h), the same permuted placement of weight
// rows as MFMA rows.  What bounds that kernel is neither its bytes nor its products but that the two take turns: a workgroup's tile
// is short k steps with a barrier each and then an epilogue, 1280 tiles of the layer shape (20480 x 512 -> 2048) over 768
// resident workgroups are 1.7 rounds, and a round's products are over when its stores begin.  Here a workgroup stays on one block
// of 256 output columns for all its rows: each of its eight wavefronts (two per SIMD) holds the weights of 32 columns over the
// whole of k as MFMA operands (4 registers per k step, 128 accumulators at k = 512), x rows stream through a ring of three 32-row
// tiles in LDS, and a tile is KS MFMAs per wavefront behind ONE barrier.  The products of a tile are a chain on one sum, the
// rounding, SiLU and staging of the tile before fill it, and the tile before that leaves as whole 128-byte lines.
//
// Measured (us, bf16; the other kernel -> this one): 20480 x 512 -> 2048 70.3 -> 52.6 (3.6 TB/s, 817 TFLOP/s), 131072 rows 472 -> 373 (against
// the power limit: 1.8 GHz, matrix pipe 38 % and LDS 26 % busy), 40000 x 384 -> 3072 167 -> 128, 20480 x 256 -> 4096 86.9 -> 69.9 (5.0 TB/s).
// Not kept: four wavefronts of 64 columns, one per SIMD (half the LDS reads; one wavefront issues a vector instruction every 6.4
// cycles and no faster: 69.8); the epilogue behind its own tile's products (68.4); weights straight from memory (60.7, see there).
#pragma once
#include "hstu_fwd_short_kernel.hip.h"
#include "in_linear_silu_kernel.hip.h"
#include "in_linear_silu_rows_kernel.h"

namespace hstu {

constexpr int kIlsRowsStages = 3;

// KS = k steps of 16 (k <= 16 KS; what is past k is zero in both operands)
template <typename Tag, int KS>
__global__ __launch_bounds__(kIlsRowsThreads, 2) void in_linear_silu_rows_kernel(const InLinearSiluArgs a)
{
    constexpr int kPitch = KS <= 16 ? 256 : 512;  // 16-bit elements per x row in LDS
    static_assert(KS * 16 <= kPitch && KS % 8 == 0, "a row is whole groups of 16 chunks");
    constexpr int kStageElems = kIlsRowsTile * kPitch;
    constexpr int kEpiElems = kIlsRowsTile * 64;  // one result of 32 rows x 64 columns
    constexpr int kWaves = kIlsRowsThreads / 64;
    constexpr int kStagedElems = 2 * (kWaves / 2) * 2 * kEpiElems;  // [parity of the tile][pair][result]
    constexpr int kPieceElems = 32 * 256;  // of the weights on their way in
    constexpr int kLdsElems = kIlsRowsStages * kStageElems + kStagedElems;
    constexpr int kLdsElemsIn = kStageElems + kWaves * kPieceElems;
    __shared__ __attribute__((aligned(1024))) uint16_t s_all[kLdsElems > kLdsElemsIn ? kLdsElems : kLdsElemsIn];
    uint16_t* const s_x = s_all;
    uint16_t* const s_epi = s_all + kIlsRowsStages * kStageElems;

    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int pair = wave >> 1, side = wave & 1;  // two wavefronts share 64 columns = 128-byte lines of the outputs
    const int r = lane & 31, half = lane >> 5;
    // workgroup b runs on XCD b % 8: an XCD takes consecutive (row group, column block) places, column blocks fastest, so that the
    // column blocks of a row group read its x rows through one L2
    const int n_cols = (a.n + kIlsRowsCols - 1) / kIlsRowsCols;
    const int places = n_cols * a.row_groups;
    const int per_xcd = (places + kIlsXcds - 1) / kIlsXcds;
    const int place = (blockIdx.x % kIlsXcds) * per_xcd + blockIdx.x / kIlsXcds;
    if (static_cast<int>(blockIdx.x / kIlsXcds) >= per_xcd || place >= places) {
        return;
    }
    const int row_group = uniform(place / n_cols);
    const int pair_col0 = uniform((place - row_group * n_cols) * kIlsRowsCols) + 64 * pair;
    const int col0 = pair_col0 + 32 * side;  // the wavefront's first column
    const int tile0 = row_group * a.group_tiles + min(row_group, a.longer_groups);
    const int tiles = a.group_tiles + (row_group < a.longer_groups ? 1 : 0);
    const uint32_t row_bytes = static_cast<uint32_t>(a.k) * 2u;

    // ---- x requests: one instruction fills 1 KiB, kRowsPerReq rows (a row's 16-byte chunk c stands at place c ^ (row % 16)).
    // A request past the last tile reads nothing and keeps the count of requests per tile.
    constexpr int kChunks = kPitch / 8;
    constexpr int kRowsPerReq = 64 / kChunks;
    constexpr int kReqs = kIlsRowsTile / kRowsPerReq / kWaves;
    uint32_t req_off[kReqs];
#pragma unroll
    for (int i = 0; i < kReqs; ++i) {
        const int row = (wave + kWaves * i) * kRowsPerReq + lane / kChunks;
        const int chunk = (lane % kChunks) ^ (row & 15);
        req_off[i] = 8 * chunk < a.k ? static_cast<uint32_t>(row) * row_bytes + chunk * 16u : kOutOfRange;
    }
    auto request = [&](int t) {
        const int64_t row0 = static_cast<int64_t>(tile0 + (t < tiles ? t : 0)) * kIlsRowsTile;
        const int64_t left = t < tiles ? a.m - row0 : 0;
        const uint32_t rows = left < kIlsRowsTile ? static_cast<uint32_t>(left) : kIlsRowsTile;
        const u32x4_t rsrc = make_rsrc_words(static_cast<const uint8_t*>(a.x) + row0 * row_bytes, rows * row_bytes);
        const uint32_t base = lds_address(s_x + (t % kIlsRowsStages) * kStageElems);
#pragma unroll
        for (int i = 0; i < kReqs; ++i) {
            request_to_lds_b128(rsrc, base + (wave + kWaves * i) * 1024, req_off[i]);
        }
    };

    // ---- weights: lane (r, half) holds k values 16 s + 8 half .. + 7 of the row that MFMA row r stands for.  They come through LDS,
    // 256 k values of a wavefront's 32 rows at a time in a piece of its own behind the first x tile: as registers straight from
    // memory a load is 32 rows x 32 bytes, and the eight wavefronts' lines are as large as the L1 (4096 rows of the layer shape
    // 21.6 -> 16.6 us)
    const int rows_w = max(min(32, a.n - col0), 0);  // 0: no column of this wavefront exists
    u32x4_t w_rsrc = make_rsrc_words(static_cast<const uint8_t*>(a.weight) + static_cast<int64_t>(rows_w > 0 ? col0 : 0) * row_bytes,
                                     static_cast<uint32_t>(rows_w) * row_bytes);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        w_rsrc[i] = static_cast<uint32_t>(uniform(static_cast<int>(w_rsrc[i])));  // (worked out by the vector unit)
    }
    uint16_t* const piece = s_all + kStageElems + wave * kPieceElems;
    u32x4_t w[KS];
#pragma unroll
    for (int h = 0; h < (KS + 15) / 16; ++h) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = 2 * i + half;
            const int chunk = 32 * h + (r ^ (row & 15));
            const uint32_t off = 8 * chunk < a.k ? static_cast<uint32_t>(ils_column_of_mfma_row(row)) * row_bytes + chunk * 16u : kOutOfRange;
            request_to_lds_b128(w_rsrc, lds_address(piece + i * 512), off);
        }
        if (h == 0) {
            request(0);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int s = 16 * h; s < KS && s < 16 * (h + 1); ++s) {
            w[s] = *reinterpret_cast<const u32x4_t*>(piece + r * 256 + ((2 * (s & 15) + half) ^ (r & 15)) * 8);
            // the accumulator half of the register file: left to itself the compiler copies them from there tile by tile
            asm volatile("" : "+a"(w[s])::"memory");
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    f32x16_t bias;  // of the lane's accumulator elements: column 16 (e / 8) + 8 half + e % 8
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int col = col0 + 16 * (q >> 1) + 8 * half + 4 * (q & 1);
        const float4 v = a.bias != nullptr && col < a.n ? *reinterpret_cast<const float4*>(a.bias + col) : make_float4(0.f, 0.f, 0.f, 0.f);
        bias[4 * q] = v.x, bias[4 * q + 1] = v.y, bias[4 * q + 2] = v.z, bias[4 * q + 3] = v.w;
    }

    // ---- where the pair's results go: 8 lanes per row, 8 columns each (split sizes are multiples of 16: one split per lane), rows
    // 16 side + 8 q + lane / 8 of a tile by this wavefront
    const int out_row = 16 * side + (lane >> 3), out_chunk = lane & 7;
    const int out_col = pair_col0 + 8 * out_chunk;
    const bool have_col = out_col < a.n;
    const int split1 = a.split_end[0], split2 = a.split_end[1], split3 = a.split_end[2];
    uint16_t* split_base;
    int split_cols, split_col;
    if (out_col < split1) {
        split_base = static_cast<uint16_t*>(a.user), split_cols = split1, split_col = out_col;
    } else if (out_col < split2) {
        split_base = static_cast<uint16_t*>(a.value), split_cols = split2 - split1, split_col = out_col - split1;
    } else if (out_col < split3) {
        split_base = static_cast<uint16_t*>(a.query), split_cols = split3 - split2, split_col = out_col - split2;
    } else {
        split_base = static_cast<uint16_t*>(a.key), split_cols = a.n - split3, split_col = out_col - split3;
    }
    int out_at = tile0 * kIlsRowsTile + out_row;  // the lane's first row of the tile that is stored next
    const int out_end = have_col ? static_cast<int>(a.m) : 0;
    uint16_t* lin_at = static_cast<uint16_t*>(a.linear_output) + static_cast<int64_t>(out_at) * a.n + out_col;
    uint16_t* split_at = split_base + static_cast<int64_t>(out_at) * split_cols + split_col;

    // staged rows of 128 bytes, 16-byte chunks XOR-ed with the row: a chunk column written by 32 rows and rows read whole both spread
    // over the banks
    auto staged_at = [&](int t, int row, int chunk) {
        return s_epi + ((t & 1) * (kWaves / 2) + pair) * 2 * kEpiElems + row * 64 + ((chunk ^ row) & 7) * 8;
    };
    auto store = [&](int t) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint16_t* from = staged_at(t, out_row + 8 * q, out_chunk);
            const u32x4_t lin = *reinterpret_cast<const u32x4_t*>(from);
            const u32x4_t out = *reinterpret_cast<const u32x4_t*>(from + kEpiElems);
            if (out_at + 8 * q < out_end) {
                __builtin_nontemporal_store(lin, reinterpret_cast<u32x4_t*>(lin_at + static_cast<int64_t>(8 * q) * a.n));
                __builtin_nontemporal_store(out, reinterpret_cast<u32x4_t*>(split_at + static_cast<int64_t>(8 * q) * split_cols));
            }
        }
        out_at += kIlsRowsTile;
        lin_at += static_cast<int64_t>(kIlsRowsTile) * a.n;
        split_at += static_cast<int64_t>(kIlsRowsTile) * split_cols;
    };

    // ---- step t: the products of tile t, and between them the results of tile t - 1 rounded and staged; the stores of tile t - 2, whose
    // lines both wavefronts of the pair have staged by then, come first.  Before tile t is read every wavefront waits for its own
    // requests of that tile: by count, everything issued behind them may be open.  Per step a wavefront issues kReqs requests and,
    // from step 2 on, 4 stores (none where no column of its pair exists; the rows of all tiles but the last are whole).
    const bool stores = pair_col0 < a.n;
    // byte offset of the lane's row and first chunk: that of k step s differs in three bits (s % 8) and by whole groups (s / 8)
    const uint32_t x_at = r * kPitch * 2u + ((half ^ (r & 15)) * 16u);
    auto round_pair = [&](const f32x16_t& sum, int i, u32x4_t& lin, u32x4_t& out) {  // elements 2 i, 2 i + 1
        // linear_output = the sum rounded once; SiLU is taken of the rounded value, as in the reference
        lin[i & 3] = pack2<Tag>(sum[2 * i], sum[2 * i + 1]);
        float lo, hi;
        ils_unpack2<Tag>(lin[i & 3], lo, hi);
        out[i & 3] = pack2<Tag>(ils_silu(lo), ils_silu(hi));
    };
    auto stage = [&](int t, int run, u32x4_t lin, u32x4_t out) {
        uint16_t* at = staged_at(t, r, 4 * side + 2 * run + half);
        *reinterpret_cast<u32x4_t*>(at) = lin;
        *reinterpret_cast<u32x4_t*>(at + kEpiElems) = out;
    };
    f32x16_t prev = bias;  // the sums of the tile before, bias added (last, as in the other kernel: a row's bits do not depend on m)
    for (int t = 0; t < tiles; ++t) {
        __builtin_amdgcn_sched_barrier(0);
        if (t == 0) {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        } else if (t <= 2 || !stores) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kReqs) : "memory");
        } else if (t == 3) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kReqs + 4) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kReqs + 8) : "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (t == 0) {
            request(1);  // (the weights passed through its place)
        }
        request(t + 2);  // into the place of tile t - 1, which every wavefront is past
        const uint32_t at = x_at + (t % kIlsRowsStages) * (kStageElems * 2);
        auto read_x = [&](int s) {
            return *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint8_t*>(s_x) + (at ^ (32u * (s & 7))) + (s >> 3) * 256);
        };
        constexpr int kAhead = 3;
        u32x4_t x[kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            x[s] = read_x(s);
        }
        if (t > 1) {
            store(t - 2);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16_t acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            acc[e] = 0.0f;
        }
        u32x4_t lin, out;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            acc = mfma32<Tag>(w[s], x[s % kAhead], acc);
            if (s + kAhead < KS) {
                x[s % kAhead] = read_x(s + kAhead);
            }
            if (s % (KS / 8) == KS / 8 - 1) {  // (in step 0 these are no results yet: nothing reads what they stage)
                const int i = s / (KS / 8);
                round_pair(prev, i, lin, out);
                if (i % 4 == 3) {
                    stage(t - 1, i / 4, lin, out);
                }
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product,
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an operand read
            __builtin_amdgcn_sched_group_barrier(0x002, 128 / KS, 0);  // and vector work of the epilogue
        }
        __builtin_amdgcn_sched_barrier(0);
        prev = acc + bias;
    }
    __syncthreads();
    u32x4_t lin, out;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        round_pair(prev, i, lin, out);
        if (i % 4 == 3) {
            stage(tiles - 1, i / 4, lin, out);
        }
    }
    if (tiles > 1) {
        store(tiles - 2);
    }
    __syncthreads();
    store(tiles - 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // requests past the last tile still write LDS
}

}  // namespace hstu
