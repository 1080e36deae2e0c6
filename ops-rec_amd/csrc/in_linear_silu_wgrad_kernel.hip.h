// The weight gradient of in_linear_silu for gfx950, with the element-wise stage in front of it:
//
//   d_mixed = cat(user_grad, value_grad, query_grad, key_grad) * silu'(linear_output)      (stored: d x needs it)
//   d weight [n, k] = d_mixed^T @ x,   bias_grad [n] = column sums of d_mixed
//
// The contraction runs over the m rows of the batch -- tens of thousands -- into an output of a few hundred tiles at most, so
// the rows are cut into chunks and every (chunk, tile) has a workgroup; the fp32 partial outputs go through the workspace and
// a second kernel adds them in a fixed order (the same bits every launch).  As a library product with one workgroup per output
// tile this took 134 us at m = 20480, n = 2048, k = 512 (104 workgroups), behind 48 us for the element-wise stage and 5 us for
// the column sums; here the three together: see the dispatch rule in in_linear_silu_mi355.hip.
//
// Workgroup: eight wavefronts, 128 columns of d_mixed by KB columns of x (128, 256 or 512: one tile spans k where it can, so
// that the element-wise stage runs once), 32 rows a step.  Each thread turns 8 elements of linear_output and of the gradients
// into d_mixed, stores them, and puts them into LDS beside the 32 rows of x; both operands of the 32x32x16 MFMA contract over
// rows, so both are read back with the transposing LDS read.  Two LDS stages, the next step's rows on their way in registers:
// one barrier a step.  Bound by the bytes of the element-wise stage up to k of a few hundred, by the products above.
#pragma once
#include "in_linear_silu_bwd_kernel.hip.h"

namespace hstu {

constexpr int kWgradThreads = 512;
constexpr int kWgradCols = 128;  // columns of d_mixed (rows of the weight) per workgroup
constexpr int kWgradRows = 32;   // rows per step

// KB = columns of x per workgroup
template <typename Tag, int KB>
__global__ __launch_bounds__(kWgradThreads, KB >= 256 ? 2 : 4) void in_linear_silu_wgrad_kernel(const InLinearSiluWgradArgs a)
{
    constexpr int NB = kWgradCols;
    constexpr int R = kWgradRows;
    constexpr int WK = KB == 128 ? 2 : 4;      // wavefronts along x's columns
    constexpr int WN = 8 / WK;                 // and along d_mixed's
    constexpr int AB = NB / WN / 32;           // 32-column blocks of a wavefront
    constexpr int BB = KB / WK / 32;
    constexpr int XCH = R * KB / 8 / kWgradThreads;  // 16-byte pieces of x per thread and step
    constexpr int kStage = R * (NB + KB);            // 16-bit elements of an LDS stage
    static_assert(XCH >= 1 && R * NB / 8 == kWgradThreads, "a step is dealt evenly over the threads");
    __shared__ __attribute__((aligned(1024))) uint16_t s_tiles[2 * kStage];
    __shared__ __attribute__((aligned(16))) float s_sums[R * NB];  // [32 rows of a step][128 columns]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);

    // tiles of a chunk share its rows: with whole groups of 8 chunks, a chunk's workgroups run on one XCD (b mod 8)
    const int tiles_k = (a.k + KB - 1) / KB;
    const int tiles = ((a.n + NB - 1) / NB) * tiles_k;
    int chunk, tile;
    if (a.chunks % 8 == 0) {
        const int j = blockIdx.x >> 3;
        chunk = (j / tiles) * 8 + (blockIdx.x & 7);
        tile = j % tiles;
    } else {
        chunk = blockIdx.x / tiles;
        tile = blockIdx.x - chunk * tiles;
    }
    const int tile_n = tile / tiles_k, tile_k = tile - tile_n * tiles_k;
    const int n0 = tile_n * NB, k0 = tile_k * KB;
    const bool first_k = tile_k == 0;  // this tile stores d_mixed and takes the column sums
    const int64_t row_begin = static_cast<int64_t>(chunk) * a.chunk_rows;
    const int64_t row_end = row_begin + a.chunk_rows < a.m ? row_begin + a.chunk_rows : a.m;

    // ---- the thread's 8 elements of a step: row tid / 16, columns 8 (tid % 16) ..
    const int erow = tid >> 4;
    const int col = n0 + 8 * (tid & 15);
    const bool in_cols = col < a.n;
    const uint16_t* grad = nullptr;
    int grad_cols = 0, grad_col = 0;
    if (in_cols) {
        if (col < a.split_end[0]) {
            grad = static_cast<const uint16_t*>(a.user_grad), grad_cols = a.split_end[0], grad_col = col;
        } else if (col < a.split_end[1]) {
            grad = static_cast<const uint16_t*>(a.value_grad), grad_cols = a.split_end[1] - a.split_end[0], grad_col = col - a.split_end[0];
        } else if (col < a.split_end[2]) {
            grad = static_cast<const uint16_t*>(a.query_grad), grad_cols = a.split_end[2] - a.split_end[1], grad_col = col - a.split_end[1];
        } else {
            grad = static_cast<const uint16_t*>(a.key_grad), grad_cols = a.n - a.split_end[2], grad_col = col - a.split_end[2];
        }
    }
    // the chunk's rows behind descriptors: rows past its end and columns past the matrices read as zeros and are not stored (the
    // host keeps a chunk under 2 GiB); a step's base is uniform and inside the chunk
    const int rows = row_end > row_begin ? static_cast<int>(row_end - row_begin) : 0;  // (the last chunks may be empty)
    const uint32_t lin_bytes = static_cast<uint32_t>(a.n) * 2u, x_bytes = static_cast<uint32_t>(a.k) * 2u;
    const __amdgpu_buffer_rsrc_t lin_rsrc =
        make_rsrc(static_cast<const uint8_t*>(a.linear_output) + row_begin * lin_bytes, static_cast<uint32_t>(rows) * lin_bytes);
    const __amdgpu_buffer_rsrc_t d_rsrc = make_rsrc(static_cast<const uint8_t*>(a.d_mixed) + row_begin * lin_bytes,
                                                    first_k ? static_cast<uint32_t>(rows) * lin_bytes : 0u);
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(static_cast<const uint8_t*>(a.x) + row_begin * x_bytes, static_cast<uint32_t>(rows) * x_bytes);
    const uint32_t lin_off = in_cols ? static_cast<uint32_t>(erow) * lin_bytes + static_cast<uint32_t>(col) * 2u : kOutOfRange;
    const uint16_t* gp = grad + (row_begin + erow) * grad_cols + grad_col;  // (a block of columns may take two gradients: no descriptor)
    const int64_t g_step = static_cast<int64_t>(R) * grad_cols;
    uint32_t x_off[XCH];
#pragma unroll
    for (int i = 0; i < XCH; ++i) {
        const int slot = tid + i * kWgradThreads;
        const int xcol = k0 + 8 * (slot % (KB / 8));
        x_off[i] = xcol < a.k ? static_cast<uint32_t>(slot / (KB / 8)) * x_bytes + static_cast<uint32_t>(xcol) * 2u : kOutOfRange;
    }

    u32x4_t z4, g4, x4[XCH];
    const u32x4_t zero = {0u, 0u, 0u, 0u};
    auto load_step = [&](int row0) {
        z4 = __builtin_amdgcn_raw_buffer_load_b128(lin_rsrc, static_cast<int>(lin_off), static_cast<int>(static_cast<uint32_t>(row0) * lin_bytes), 0);
        g4 = zero;
        if (in_cols && row0 + erow < rows) {
            g4 = *reinterpret_cast<const u32x4_t*>(gp);
        }
        gp += g_step;
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            x4[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, static_cast<int>(x_off[i]), static_cast<int>(static_cast<uint32_t>(row0) * x_bytes), 0);
        }
    };

    // Column sums in two levels: a thread's sums of eight steps, then of the chunk, in LDS places of its own.  (In one chain of hundreds
    // of additions the bias gradient came out twice as far from its 64-bit value as with the element-wise kernel's blocks of 64 rows,
    // 3.5e-7 against 1.4e-7 at 20000 rows; in two levels 1.6e-7, at the same time per call.)
    const bool want_sums = a.partial_sums != nullptr && first_k;
    float* const my_sums = s_sums + erow * NB + 8 * (tid & 15);
    float sums[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        sums[e] = 0.0f;
        my_sums[e] = 0.0f;
    }
    auto flush_sums = [&]() {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            my_sums[e] += sums[e];
            sums[e] = 0.0f;
        }
    };
    f32x16_t acc[AB][BB];
#pragma unroll
    for (int i = 0; i < AB; ++i) {
#pragma unroll
        for (int j = 0; j < BB; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0f;
            }
        }
    }
    // operand reads: the lane's address of a 4-row piece of each 32-column block (the mapping of the V tiles of the forward
    // kernel); rows + 8 and + 16 keep the swizzle, which is by row mod 4
    const int wn = wave / WK, wk = wave - wn * WK;
    const int tr_row = 4 * (lane >> 5) + ((lane & 15) >> 2);
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    int a_off[AB], b_off[BB];
#pragma unroll
    for (int i = 0; i < AB; ++i) {
        const int c = 32 * (AB * wn + i) + tr_col;
        a_off[i] = tr_row * NB + v_chunk_swizzle<NB>(tr_row, c >> 3) * 8 + (c & 7);
    }
#pragma unroll
    for (int j = 0; j < BB; ++j) {
        const int c = 32 * (BB * wk + j) + tr_col;
        b_off[j] = R * NB + tr_row * KB + v_chunk_swizzle<KB>(tr_row, c >> 3) * 8 + (c & 7);
    }
    auto read_tr = [&](const uint16_t* p, int row_elems) -> u32x4_t {
        const u32x2_t lo = lds_read_tr16_b64(p);
        const u32x2_t hi = lds_read_tr16_b64(p + 8 * row_elems);
        const u32x4_t r = {lo[0], lo[1], hi[0], hi[1]};
        return r;
    };

    // d_mixed, two elements (pair e of four): into d4, and into the column sums
    u32x4_t d4;
    auto stage_pair = [&](int e) {
        float z[2], g[2], d[2];
        ils_unpack2<Tag>(z4[e], z[0], z[1]);
        ils_unpack2<Tag>(g4[e], g[0], g[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z[h] * -1.4426950408889634f));
            d[h] = g[h] * (s * (1.0f + z[h] * (1.0f - s)));
            sums[2 * e + h] += d[h];
        }
        d4[e] = pack2<Tag>(d[0], d[1]);
    };
    auto put_x = [&](uint16_t* st) {
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            const int slot = tid + i * kWgradThreads;
            const int xrow = slot / (KB / 8);
            *reinterpret_cast<u32x4_t*>(st + R * NB + xrow * KB + v_chunk_swizzle<KB>(xrow, slot % (KB / 8)) * 8) = x4[i];
        }
    };
    auto put_d = [&](uint16_t* st, int row0, bool inside) {
        *reinterpret_cast<u32x4_t*>(st + erow * NB + v_chunk_swizzle<NB>(erow, tid & 15) * 8) = d4;
        __builtin_amdgcn_raw_buffer_store_b128(d4, d_rsrc, static_cast<int>(inside ? lin_off : kOutOfRange),
                                               static_cast<int>(inside && first_k ? static_cast<uint32_t>(row0) * lin_bytes : 0u),
                                               2);  // (non-temporal)
    };

    // A step's products run with the element-wise stage of the next step between them (the wavefronts of a SIMD meet at every
    // barrier, so that one after the other the vector unit and the matrix pipe would idle in turn); the rows of the step after
    // that are on their way meanwhile.  (Past the chunk the stage works on zeros, which change no column sum.)
    if (rows > 0) {
        load_step(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            stage_pair(e);
        }
        put_x(s_tiles);
        put_d(s_tiles, 0, true);
        if (R < rows) {
            load_step(R);
        }
        __syncthreads();
    }
    int stage = 0;
    for (int row0 = 0; row0 < rows; row0 += R) {
        const uint16_t* const st = s_tiles + stage * kStage;
        uint16_t* const next = s_tiles + (stage ^ 1) * kStage;
        const bool more = row0 + R < rows;
        put_x(next);
        if (!more) {
            z4 = zero;
            g4 = zero;
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            u32x4_t da[AB], xb[BB];
#pragma unroll
            for (int i = 0; i < AB; ++i) {
                da[i] = read_tr(st + a_off[i] + 16 * kk * NB, NB);
            }
#pragma unroll
            for (int j = 0; j < BB; ++j) {
                xb[j] = read_tr(st + b_off[j] + 16 * kk * KB, KB);
            }
#pragma unroll
            for (int i = 0; i < AB; ++i) {
#pragma unroll
                for (int j = 0; j < BB; ++j) {
                    acc[i][j] = mfma32<Tag>(da[i], xb[j], acc[i][j]);
                    if ((i * BB + j) % (AB * BB / 2) == 0) {
                        stage_pair(2 * kk + (i * BB + j) / (AB * BB / 2));
                    }
                }
            }
        }
        // (the order asked of the scheduler, which would put the stage behind all the products: a share of it behind each)
#pragma unroll
        for (int u = 0; u < 2 * AB * BB; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                     // an MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 128 / (2 * AB * BB), 0);  // vector instructions
        }
        put_d(next, row0 + R, more);  // (without a branch around it: the stage would move into that)
        if (row0 + 2 * R < rows) {
            load_step(row0 + 2 * R);
        }
        if (want_sums && (row0 & (7 * R)) == 7 * R) {
            flush_sums();
        }
        __syncthreads();
        stage ^= 1;
    }

    // ---- partial outputs: accumulator element 4 g + e of a lane is row 8 g + 4 (lane / 32) + e of its block, column lane % 32
    float* const part = a.partial + static_cast<int64_t>(chunk) * a.n * a.k;
#pragma unroll
    for (int i = 0; i < AB; ++i) {
#pragma unroll
        for (int j = 0; j < BB; ++j) {
            const int c = k0 + 32 * (BB * wk + j) + (lane & 31);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = n0 + 32 * (AB * wn + i) + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (r < a.n && c < a.k) {
                    part[static_cast<int64_t>(r) * a.k + c] = acc[i][j][e];
                }
            }
        }
    }
    if (!want_sums) {
        return;
    }
    flush_sums();
    __syncthreads();
    if (tid < NB && n0 + tid < a.n) {
        float total[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < R; ++r) {
            total[r & 3] += s_sums[r * NB + tid];
        }
        a.partial_sums[static_cast<int64_t>(chunk) * a.n + n0 + tid] = (total[0] + total[1]) + (total[2] + total[3]);
    }
}

// weight_grad and bias_grad = the partial outputs, added in one order whatever finished first: eight chunks pairwise at a time.  A thread owns four consecutive elements (k is a
// multiple of 16); its loads of eight chunks are in flight together.
template <typename Tag>
__global__ __launch_bounds__(256) void in_linear_silu_wgrad_sum_kernel(const InLinearSiluWgradArgs a)
{
    typedef __attribute__((ext_vector_type(4))) float f32x4;
    const int64_t quads = static_cast<int64_t>(a.n) * a.k / 4;
    const int64_t bias_quads = a.bias_grad != nullptr ? a.n / 4 : 0;
    for (int64_t q = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; q < quads + bias_quads; q += static_cast<int64_t>(gridDim.x) * 256) {
        const bool is_bias = q >= quads;
        const int64_t stride = is_bias ? a.n / 4 : quads;
        const f32x4* const from = reinterpret_cast<const f32x4*>(is_bias ? a.partial_sums : a.partial) + (is_bias ? q - quads : q);
        f32x4 total = {0.0f, 0.0f, 0.0f, 0.0f};
        int c = 0;
        for (; c + 8 <= a.chunks; c += 8) {
            f32x4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                v[u] = from[(c + u) * stride];
            }
            total += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        }
        for (; c < a.chunks; ++c) {
            total += from[c * stride];
        }
        if (is_bias) {
            reinterpret_cast<f32x4*>(a.bias_grad)[q - quads] = total;
        } else {
            const u32x2_t w = {pack2<Tag>(total[0], total[1]), pack2<Tag>(total[2], total[3])};
            reinterpret_cast<u32x2_t*>(a.weight_grad)[q] = w;
        }
    }
}

}  // namespace hstu
