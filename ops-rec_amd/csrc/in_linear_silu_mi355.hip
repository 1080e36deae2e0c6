// C ABI of in_linear_silu forward: argument checks, choice of the kernel variant, launch.  Host-side counterpart of
// the reference's adapter checks (ascendc/activation/in_linear_silu/torch_extension/in_linear_silu_plugin.cpp:36-66)
// and of its host tiling (ascendc/activation/in_linear_silu/in_linear_silu_forward/op_host/in_linear_silu.cpp).
#include "../../include/ops_rec_activation_mi355.h"

#include <hip/hip_runtime.h>

#include "hstu_error.h"
#include "in_linear_silu_bwd_kernel.hip.h"
#include "in_linear_silu_kernel.hip.h"
#include "in_linear_silu_rows_kernel.h"
#include "in_linear_silu_wgrad_kernel.hip.h"

namespace {

using hstu::InLinearSiluArgs;

struct IlsVariant {
    const char* name;
    void (*kernel)(const InLinearSiluArgs);
    int tile_n;  // output columns per workgroup
};

// [type: bf16, fp16][ring of 2 stages; 3 stages; 4 stages; 2 stages with 128 x 256 tiles].  Measured on MI355X over
// k = 64 .. 8192: for 128 x 128 tiles, workgroups per CU count for more than prefetch depth (4 stages, two workgroups
// per CU, slowest everywhere up to k = 2048); 3 stages win by 3-7 % for k = 128 .. 512, 2 stages by 2-4 % at k <= 64
// and k = 768.  From k = 1024 on the products dominate and the 128 x 256 tile (twice the MFMAs per k step and per byte
// staged, two workgroups per CU) wins: 633 -> 549 us at k = 2048, 607 -> 484 us at m = n = 8192, k = 4096
// (1.14 PFLOP/s).
#define ILS_VARIANT(tag, tagname, S, W) \
    {"in_linear_silu_" tagname "_stages" #S "_tile" #W, hstu::in_linear_silu_kernel<hstu::tag, S, (W) / 64>, W}
const IlsVariant kVariants[2][4] = {
    {ILS_VARIANT(bf16_tag, "bf16", 2, 128), ILS_VARIANT(bf16_tag, "bf16", 3, 128), ILS_VARIANT(bf16_tag, "bf16", 4, 128),
     ILS_VARIANT(bf16_tag, "bf16", 2, 256)},
    {ILS_VARIANT(f16_tag, "f16", 2, 128), ILS_VARIANT(f16_tag, "f16", 3, 128), ILS_VARIANT(f16_tag, "f16", 4, 128),
     ILS_VARIANT(f16_tag, "f16", 2, 256)},
};

int compute_units_or_256()  // (a size asked for where there is no device)
{
    int cus = 0;
    return hstu::compute_units(&cus) == HSTU_OK ? cus : 256;
}

// groups of rows of the kernel with the weights in registers: one workgroup per CU in all
int rows_groups(const in_linear_silu_params* p)
{
    const int cus = compute_units_or_256();
    const int64_t tiles = (p->m + hstu::kIlsRowsTile - 1) / hstu::kIlsRowsTile;
    const int64_t cols = (p->n + hstu::kIlsRowsCols - 1) / hstu::kIlsRowsCols;
    const int64_t groups = cus / cols > 1 ? cus / cols : 1;
    return static_cast<int>(groups < tiles ? groups : tiles);
}

// The kernel with the weights in registers, where it is taken (us, bf16, the other kernel -> this one; 1600 calls with k of 144 to 512 and n up to
// 32768 measured on both):
//   k of 129 to 512: the registers hold no more, and at k = 128 the kernels are level, 20480 x 4096 65.3 -> 66.2: both write at 5 TB/s;
//   splits that begin at 128-byte lines: elsewhere neighbouring wavefronts write parts of a line (100000 rows of 240 -> 960 132 -> 147, 40000
//     of 272 -> 1088 65 -> 70);
//   six 32-row tiles per workgroup at least, to pay for the weights on their way in: 4 tiles 2048 x 512 16.4 -> 16.6, 1024 x 256 12.0 -> 12.8; 6 tiles
//     1536 x 384 18.9 -> 18.5, 1536 x 192 15.7 -> 15.5; 8 tiles 2048 x 512 27.5 -> 24.7, 4096 x 256 20.2 -> 19.4; 20 tiles 2048 x 512 70.3 -> 52.6;
//     131072 rows, 128 tiles, 472 -> 373;
//   past 24 blocks of columns, where few groups of rows are left, leave compute units idle and bring in all of the weights each, 20 tiles: below that
//     7680 x 384, 2064 rows 24.3 -> 26.6, 7680 x 320, 3122 rows 29.7 -> 33.7, 8192 x 512, 1791 rows 27.1 -> 29.2, 13824 x 288, 1444 rows 26.1 -> 28.6,
//     22528 x 512, 474 rows 22.3 -> 26.2, at 13 to 14 tiles 22528 x 352, 17920 x 320, 11264 x 352 0.86 to 0.88 x, others up to 1.2 x; from 20 tiles on
//     442 of 468 calls faster, up to 1.53 x (23552 x 256, 30 tiles, 0.91 x, 24576 x 192, 4201 rows, 86.7 -> 103.5).  Still six where the last of the
//     other kernel's k steps of 32 is half empty (20800 x 400, 637 rows 30.2 -> 25.8, 10304 x 368, 2155 rows 41.0 -> 31.0; 8704 x 272, 1744 rows
//     21.8 -> 23.5), and where 64 blocks and more leave no compute unit idle, which goes either way: 16384 x 256, 903 rows 1.12 x, 1000 rows
//     level, 16384 x 512, 801 rows 28.2 -> 29.1, 768 rows, exactly one round of the other kernel, 22.7 -> 27.4;
//   up to k = 160, of which the instance for 256 spends 16 steps, less than eight tiles, a round and a bit of the other kernel: 2304 x 144, 5911 rows 1.10
//     x, 16128 x 144, 777 rows 17.6 -> 16.5; more tiles 576 x 144, 130972 rows 65.3 -> 79.7, 1920 x 160, 49364 rows 76.9 -> 81.9, 6912 x 144, 20951 rows
//     level (k = 176: 1408 x 176, 30462 rows 40.2 -> 39.6).
const hstu::IlsRowsVariant* select_rows(const in_linear_silu_params* p)
{
    if (p->k <= 128 || p->k > 512 || p->m > 0x7fffffff - hstu::kIlsRowsTile) {
        return nullptr;
    }
    for (int i = 0; i < 4; ++i) {
        if (p->split[i] % 64 != 0) {
            return nullptr;
        }
    }
    const int64_t tiles = p->m / hstu::kIlsRowsTile, groups = rows_groups(p), cols = (p->n + hstu::kIlsRowsCols - 1) / hstu::kIlsRowsCols;
    const bool six_pay = cols <= 24 || p->k % 32 != 0 || (cols >= 64 && cols * groups == compute_units_or_256());
    if (tiles < (six_pay ? 6 : 20) * groups || (p->k <= 160 && tiles >= 8 * groups)) {
        return nullptr;
    }
    const hstu::IlsRowsVariant* v = hstu::ils_rows_variants(p->dtype == HSTU_DT_BF16);
    while (p->k > 16 * v->steps) {
        ++v;
    }
    return v;
}

const IlsVariant* select(const in_linear_silu_params* p)
{
    int ring;
    if (p->k >= 1024) {
        ring = 3;
    } else {
        ring = (p->k <= 64 || p->k > 512) ? 0 : 1;
    }
    return &kVariants[p->dtype == HSTU_DT_BF16 ? 0 : 1][ring];
}

constexpr int64_t kMinDim = 16;
constexpr int64_t kMaxDim = 512 * 16;

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

// x tiles kept to one XCD each (see the kernel): for a weight matrix of at most 2 MiB -- half an L2 -- with at most 16 n
// tiles per m tile, rows long enough for the x tiles to weigh against the outputs, and at least four groups of m tiles
bool xcd_groups(const in_linear_silu_params* p)
{
    return p->n * p->k * 2 <= (int64_t{2} << 20) && p->n <= 2048 && p->k >= 128 && p->m >= 4096;
}

// workgroups of a launch: m tiles (rounded up to whole groups of one per XCD in the grouped order) times n tiles
int64_t grid_size(const in_linear_silu_params* p)
{
    if (select_rows(p) != nullptr) {  // (the kernel deals places to the XCDs in equal runs)
        const int64_t places = rows_groups(p) * ((p->n + hstu::kIlsRowsCols - 1) / hstu::kIlsRowsCols);
        return (places + hstu::kIlsXcds - 1) / hstu::kIlsXcds * hstu::kIlsXcds;
    }
    const int tile_n = select(p)->tile_n;
    int64_t tiles_m = (p->m + hstu::kIlsTileM - 1) / hstu::kIlsTileM;
    const int64_t tiles_n = (p->n + tile_n - 1) / tile_n;
    if (xcd_groups(p)) {
        tiles_m = (tiles_m + hstu::kIlsXcds - 1) / hstu::kIlsXcds * hstu::kIlsXcds;
    }
    return tiles_m * tiles_n;
}

int validate(const in_linear_silu_params* p)
{
    if (p == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "params is NULL");
    }
    if (p->struct_size != sizeof(in_linear_silu_params)) {
        return hstu::set_error(HSTU_ERR_INVALID, "struct_size %u does not match this library (%zu)", p->struct_size,
                               sizeof(in_linear_silu_params));
    }
    if (p->x == nullptr || p->weight == nullptr || p->user == nullptr || p->value == nullptr || p->query == nullptr ||
        p->key == nullptr || p->linear_output == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "x, weight and the five outputs must all be given");
    }
    if (p->dtype != HSTU_DT_BF16 && p->dtype != HSTU_DT_FP16) {
        return hstu::set_error(HSTU_ERR_INVALID, "dtype %d is not bf16 or fp16", p->dtype);
    }
    if (p->m < 1) {
        return hstu::set_error(HSTU_ERR_INVALID, "x tensor must be non-empty");
    }
    int64_t total = 0;
    for (int i = 0; i < 4; ++i) {
        if (p->split[i] < kMinDim || p->split[i] > kMaxDim || p->split[i] % kMinDim != 0) {
            return hstu::set_error(HSTU_ERR_INVALID, "uvqk dim must in range[16, 8192] and multiples of 16.");
        }
        total += p->split[i];
    }
    if (p->k < kMinDim || p->k > kMaxDim || p->k % kMinDim != 0) {
        return hstu::set_error(HSTU_ERR_INVALID, "x dim[1] must in range[16, 8192] and multiples of 16.");
    }
    if (p->n < 4 * kMinDim || p->n > 4 * kMaxDim || p->n % kMinDim != 0) {
        return hstu::set_error(HSTU_ERR_INVALID, "weight dim[0] must in range[64, 32768] and multiples of 16.");
    }
    if (total != p->n) {
        return hstu::set_error(HSTU_ERR_INVALID, "weight_dim[0] must equal to sum(splitList).");
    }
    if (p->n % (4 * p->k) != 0) {
        return hstu::set_error(HSTU_ERR_INVALID, "weight dim[0] must be a multiple of 4 x dim[1]");
    }
    const void* ptrs[] = {p->x, p->weight, p->bias, p->user, p->value, p->query, p->key, p->linear_output};
    for (const void* ptr : ptrs) {
        if (!aligned16(ptr)) {
            return hstu::set_error(HSTU_ERR_INVALID, "every tensor must start at a multiple of 16 bytes");
        }
    }
    const int64_t tiles = grid_size(p);
    if (tiles > 0x7fffffff) {
        return hstu::set_error(HSTU_ERR_INVALID, "too many rows: %lld tiles of %d rows", static_cast<long long>(tiles),
                               hstu::kIlsTileM);
    }
    return HSTU_OK;
}

int validate_bwd(const in_linear_silu_bwd_params* p)
{
    if (p == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "params is NULL");
    }
    if (p->struct_size != sizeof(in_linear_silu_bwd_params)) {
        return hstu::set_error(HSTU_ERR_INVALID, "struct_size %u does not match this library (%zu)", p->struct_size,
                               sizeof(in_linear_silu_bwd_params));
    }
    if (p->linear_output == nullptr || p->user_grad == nullptr || p->value_grad == nullptr || p->query_grad == nullptr ||
        p->key_grad == nullptr || p->d_mixed == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "linear_output, the four gradients and d_mixed must all be given");
    }
    if (p->dtype != HSTU_DT_BF16 && p->dtype != HSTU_DT_FP16) {
        return hstu::set_error(HSTU_ERR_INVALID, "dtype %d is not bf16 or fp16", p->dtype);
    }
    if (p->m < 1) {
        return hstu::set_error(HSTU_ERR_INVALID, "linear_output tensor must be non-empty");
    }
    int64_t total = 0;
    for (int i = 0; i < 4; ++i) {
        if (p->split[i] < kMinDim || p->split[i] > kMaxDim || p->split[i] % kMinDim != 0) {
            return hstu::set_error(HSTU_ERR_INVALID, "uvqk dim must in range[16, 8192] and multiples of 16.");
        }
        total += p->split[i];
    }
    if (p->n < 4 * kMinDim || p->n > 4 * kMaxDim || p->n % kMinDim != 0) {
        return hstu::set_error(HSTU_ERR_INVALID, "weight dim[0] must in range[64, 32768] and multiples of 16.");
    }
    if (total != p->n) {
        return hstu::set_error(HSTU_ERR_INVALID, "linear_output dim[1] must equal to sum(split_list).");
    }
    const void* ptrs[] = {p->linear_output, p->user_grad, p->value_grad, p->query_grad, p->key_grad, p->d_mixed};
    for (const void* ptr : ptrs) {
        if (!aligned16(ptr)) {
            return hstu::set_error(HSTU_ERR_INVALID, "every tensor must start at a multiple of 16 bytes");
        }
    }
    if ((p->m + hstu::kIlsBwdRows - 1) / hstu::kIlsBwdRows * ((p->n + hstu::kIlsBwdCols - 1) / hstu::kIlsBwdCols) > 0x7fffffff) {
        return hstu::set_error(HSTU_ERR_INVALID, "too many rows");
    }
    return HSTU_OK;
}

int64_t bwd_row_blocks(const in_linear_silu_bwd_params* p) { return (p->m + hstu::kIlsBwdRows - 1) / hstu::kIlsBwdRows; }

uint64_t bwd_workspace_bytes(const in_linear_silu_bwd_params* p)
{
    return p->bias_grad == nullptr ? 0 : static_cast<uint64_t>(bwd_row_blocks(p)) * static_cast<uint64_t>(p->n) * sizeof(float);
}

int validate_weight(const in_linear_silu_bwd_weight_params* p)
{
    if (p == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "params is NULL");
    }
    if (p->struct_size != sizeof(in_linear_silu_bwd_weight_params)) {
        return hstu::set_error(HSTU_ERR_INVALID, "struct_size %u does not match this library (%zu)", p->struct_size,
                               sizeof(in_linear_silu_bwd_weight_params));
    }
    const int rc = validate_bwd(&p->stage);
    if (rc != HSTU_OK) {
        return rc;
    }
    if (p->x == nullptr || p->weight_grad == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "x and weight_grad must be given");
    }
    if (p->k < kMinDim || p->k > kMaxDim || p->k % kMinDim != 0) {
        return hstu::set_error(HSTU_ERR_INVALID, "x dim[1] must in range[16, 8192] and multiples of 16.");
    }
    if (!aligned16(p->x) || !aligned16(p->weight_grad) || !aligned16(p->stage.bias_grad)) {
        return hstu::set_error(HSTU_ERR_INVALID, "every tensor must start at a multiple of 16 bytes");
    }
    return HSTU_OK;
}

// How the weight gradient is cut: tiles of 128 x tile_k (the narrowest of the three widths that spans k, 512 above), and the
// number of chunks of rows, each of eight 32-row steps at least, that an estimate of the time puts first -- rounds of
// workgroups over the CUs (two of the narrowest tile each, one of the others) times a chunk's steps, and the partial outputs, which
// are written and read back once.  Chunks beyond eight come in whole groups of 8, one per XCD.  The estimate only has to rank
// chunk counts: over 14 shapes of 1000 .. 300000 rows, n 256 .. 8192, k 64 .. 1024 its choice took 0.97 .. 1.12 of the best of thirteen
// counts (worst 20000 x 1024 x 128: 33.2 against 29.7 us); below 1000 rows the eight steps bind (700 x 512 x 128: 14.3 against 9.4 us).
// Measured, element-wise stage + column sums + library product -> the two kernels: m 20480, n 2048, k 512 187 -> 92 us (by the
// counters 340 MB moved by the first kernel, 69 MB by the second, which adds the partial outputs: 84 + 14 us in a trace, 4.2 TB/s);
// m 95697, n 512, k 128 338 -> 76 us.
struct WeightPlan {
    int tile_k;
    int tiles;
    int chunks;
    int64_t chunk_rows;
};
WeightPlan plan_weight(const in_linear_silu_bwd_weight_params* p)
{
    WeightPlan w;
    w.tile_k = p->k <= 128 ? 128 : (p->k <= 256 ? 256 : 512);
    w.tiles = static_cast<int>((p->stage.n + hstu::kWgradCols - 1) / hstu::kWgradCols * ((p->k + w.tile_k - 1) / w.tile_k));
    int cus = 0;
    if (hstu::compute_units(&cus) != HSTU_OK) {
        cus = 256;  // (a size asked for where there is no device)
    }
    const int64_t slots = w.tile_k == 128 ? 2 * cus : cus;  // resident workgroups
    const int64_t steps = (p->stage.m + hstu::kWgradRows - 1) / hstu::kWgradRows;
    // (a chunk stays behind 32-bit descriptors)
    const int64_t widest = p->stage.n > p->k ? p->stage.n : p->k;
    const int64_t least = (steps * hstu::kWgradRows * widest * 2) / (int64_t{1} << 30) + 1;
    const int64_t most = steps / 8 < 64 ? steps / 8 : 64;
    const double step_us = w.tile_k == 512 ? 1.2 : 0.8;
    const double partial_us = static_cast<double>(p->stage.n) * static_cast<double>(p->k) * 8.0 / 6e6;  // written and read back once
    int64_t chunks = least;
    double best = 0.0;
    for (int64_t c = least; c <= most || c == least; ++c) {
        if (c > 8 && c % 8 != 0) {
            continue;
        }
        const double rounds = static_cast<double>((w.tiles * c + slots - 1) / slots);
        const double cost = rounds * (static_cast<double>((steps + c - 1) / c) * step_us + 3.0) + static_cast<double>(c) * partial_us;
        if (c == least || cost < best) {
            best = cost;
            chunks = c;
        }
    }
    w.chunk_rows = (steps + chunks - 1) / chunks * hstu::kWgradRows;
    w.chunks = static_cast<int>(chunks);
    return w;
}

uint64_t weight_workspace_bytes(const in_linear_silu_bwd_weight_params* p)
{
    const WeightPlan w = plan_weight(p);
    const uint64_t per_chunk = static_cast<uint64_t>(p->stage.n) * static_cast<uint64_t>(p->k + (p->stage.bias_grad != nullptr ? 1 : 0));
    return static_cast<uint64_t>(w.chunks) * per_chunk * sizeof(float);
}

}  // namespace

extern "C" {

// Up to two tiles of 512 columns span k.  From the third on the element-wise stage, which each of them runs for itself, and the
// narrower tiles of a plain product decide: stage + library product against the kernels of in_linear_silu_bwd_weight (GPU time, bf16),
// k 256 .. 768: 1.05 .. 4.3 of their time from m = 512 on; k 1024: 0.93 .. 1.31 (n 4096 .. 28672; level from n 8192 on); k 1152: 0.85 ..
// 1.04; 1280: 0.91 .. 1.04; 1408: 0.68 .. 1.04 (1.31 at m 100000); 1536: 0.70 .. 1.04 (1.18 at n 12288, m 100000); 2048: 0.81 .. 0.91;
// 3072: 0.59 .. 0.80.  (n and m hardly matter: 32768 x 512, as large a weight as 8192 x 2048, 1.14 .. 1.21.)
HSTU_API int in_linear_silu_bwd_weight_pays(const in_linear_silu_bwd_weight_params* p) { return p != nullptr && p->k <= 1024 ? 1 : 0; }

HSTU_API int in_linear_silu_bwd_weight_workspace_size(const in_linear_silu_bwd_weight_params* p, uint64_t* workspace_bytes)
{
    if (workspace_bytes == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "workspace_bytes is NULL");
    }
    *workspace_bytes = 0;
    const int rc = validate_weight(p);
    if (rc != HSTU_OK) {
        return rc;
    }
    *workspace_bytes = weight_workspace_bytes(p);
    return HSTU_OK;
}

HSTU_API int in_linear_silu_bwd_weight(const in_linear_silu_bwd_weight_params* p, void* workspace, uint64_t workspace_bytes, void* stream)
{
    const int rc = validate_weight(p);
    if (rc != HSTU_OK) {
        return rc;
    }
    const uint64_t need = weight_workspace_bytes(p);
    if (workspace == nullptr || workspace_bytes < need || !aligned16(workspace)) {
        return hstu::set_error(HSTU_ERR_WORKSPACE, "workspace of %llu bytes (16-byte aligned) needed for the weight gradient, got %llu",
                               static_cast<unsigned long long>(need), static_cast<unsigned long long>(workspace_bytes));
    }
    const WeightPlan w = plan_weight(p);
    const in_linear_silu_bwd_params& s = p->stage;
    hstu::InLinearSiluWgradArgs a;
    a.linear_output = s.linear_output;
    a.user_grad = s.user_grad;
    a.value_grad = s.value_grad;
    a.query_grad = s.query_grad;
    a.key_grad = s.key_grad;
    a.x = p->x;
    a.d_mixed = s.d_mixed;
    a.weight_grad = p->weight_grad;
    a.bias_grad = s.bias_grad;
    a.m = s.m;
    a.n = static_cast<int>(s.n);
    a.k = static_cast<int>(p->k);
    a.chunks = w.chunks;
    a.chunk_rows = w.chunk_rows;
    a.partial = static_cast<float*>(workspace);
    a.partial_sums = s.bias_grad != nullptr ? a.partial + static_cast<int64_t>(w.chunks) * a.n * a.k : nullptr;
    a.split_end[0] = static_cast<int>(s.split[0]);
    a.split_end[1] = a.split_end[0] + static_cast<int>(s.split[1]);
    a.split_end[2] = a.split_end[1] + static_cast<int>(s.split[2]);
    const bool bf16 = s.dtype == HSTU_DT_BF16;
    void (*const kernel)(const hstu::InLinearSiluWgradArgs) =
        w.tile_k == 128   ? (bf16 ? hstu::in_linear_silu_wgrad_kernel<hstu::bf16_tag, 128> : hstu::in_linear_silu_wgrad_kernel<hstu::f16_tag, 128>)
        : w.tile_k == 256 ? (bf16 ? hstu::in_linear_silu_wgrad_kernel<hstu::bf16_tag, 256> : hstu::in_linear_silu_wgrad_kernel<hstu::f16_tag, 256>)
                          : (bf16 ? hstu::in_linear_silu_wgrad_kernel<hstu::bf16_tag, 512> : hstu::in_linear_silu_wgrad_kernel<hstu::f16_tag, 512>);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(w.tiles * w.chunks)), dim3(hstu::kWgradThreads), 0, static_cast<hipStream_t>(stream), a);
    const int64_t quads = (static_cast<int64_t>(a.n) * a.k + a.n) / 4;
    const unsigned sum_grid = static_cast<unsigned>((quads + 255) / 256 < 8192 ? (quads + 255) / 256 : 8192);
    hipLaunchKernelGGL(bf16 ? hstu::in_linear_silu_wgrad_sum_kernel<hstu::bf16_tag> : hstu::in_linear_silu_wgrad_sum_kernel<hstu::f16_tag>,
                       dim3(sum_grid), dim3(256), 0, static_cast<hipStream_t>(stream), a);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        return hstu::set_error(HSTU_ERR_RUNTIME, "launch of in_linear_silu_wgrad failed: %s", hipGetErrorString(err));
    }
    return HSTU_OK;
}

HSTU_API int in_linear_silu_bwd_dmixed_workspace_size(const in_linear_silu_bwd_params* p, uint64_t* workspace_bytes)
{
    if (workspace_bytes == nullptr) {
        return hstu::set_error(HSTU_ERR_NULLPTR, "workspace_bytes is NULL");
    }
    *workspace_bytes = 0;
    const int rc = validate_bwd(p);
    if (rc != HSTU_OK) {
        return rc;
    }
    *workspace_bytes = bwd_workspace_bytes(p);
    return HSTU_OK;
}

HSTU_API int in_linear_silu_bwd_dmixed(const in_linear_silu_bwd_params* p, void* workspace, uint64_t workspace_bytes,
                                       void* stream)
{
    const int rc = validate_bwd(p);
    if (rc != HSTU_OK) {
        return rc;
    }
    const uint64_t need = bwd_workspace_bytes(p);
    if (need > 0 && (workspace == nullptr || workspace_bytes < need || !aligned16(workspace))) {
        return hstu::set_error(HSTU_ERR_WORKSPACE, "workspace of %llu bytes (16-byte aligned) needed for the bias gradient, got %llu",
                               static_cast<unsigned long long>(need), static_cast<unsigned long long>(workspace_bytes));
    }
    hstu::InLinearSiluBwdArgs a;
    a.linear_output = p->linear_output;
    a.user_grad = p->user_grad;
    a.value_grad = p->value_grad;
    a.query_grad = p->query_grad;
    a.key_grad = p->key_grad;
    a.d_mixed = p->d_mixed;
    a.partial_sums = need > 0 ? static_cast<float*>(workspace) : nullptr;
    a.m = p->m;
    a.n = static_cast<int>(p->n);
    a.split_end[0] = static_cast<int>(p->split[0]);
    a.split_end[1] = a.split_end[0] + static_cast<int>(p->split[1]);
    a.split_end[2] = a.split_end[1] + static_cast<int>(p->split[2]);
    const unsigned col_blocks = static_cast<unsigned>((p->n + hstu::kIlsBwdCols - 1) / hstu::kIlsBwdCols);
    const unsigned row_blocks = static_cast<unsigned>(bwd_row_blocks(p));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (p->dtype == HSTU_DT_BF16) {
        hipLaunchKernelGGL(hstu::in_linear_silu_dmixed_kernel<hstu::bf16_tag>, dim3(row_blocks * col_blocks),
                           dim3(hstu::kIlsBwdThreads), 0, s, a);
    } else {
        hipLaunchKernelGGL(hstu::in_linear_silu_dmixed_kernel<hstu::f16_tag>, dim3(row_blocks * col_blocks),
                           dim3(hstu::kIlsBwdThreads), 0, s, a);
    }
    if (need > 0) {
        hipLaunchKernelGGL(hstu::in_linear_silu_bias_grad_kernel,
                           dim3(static_cast<unsigned>((p->n + hstu::kIlsBiasCols - 1) / hstu::kIlsBiasCols)),
                           dim3(hstu::kIlsBiasCols * hstu::kIlsBiasLanes), 0, s, a.partial_sums, p->bias_grad,
                           static_cast<int>(row_blocks), a.n);
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        return hstu::set_error(HSTU_ERR_RUNTIME, "launch of in_linear_silu_dmixed failed: %s", hipGetErrorString(err));
    }
    return HSTU_OK;
}

HSTU_API const char* in_linear_silu_fwd_kernel_name(const in_linear_silu_params* params)
{
    if (validate(params) != HSTU_OK) {
        return nullptr;
    }
    const hstu::IlsRowsVariant* rows = select_rows(params);
    return rows != nullptr ? rows->name : select(params)->name;
}

HSTU_API int in_linear_silu_fwd(const in_linear_silu_params* p, void* stream)
{
    const int rc = validate(p);
    if (rc != HSTU_OK) {
        return rc;
    }
    InLinearSiluArgs a;
    a.x = p->x;
    a.weight = p->weight;
    a.bias = p->bias;
    a.user = p->user;
    a.value = p->value;
    a.query = p->query;
    a.key = p->key;
    a.linear_output = p->linear_output;
    a.m = p->m;
    a.n = static_cast<int>(p->n);
    a.k = static_cast<int>(p->k);
    a.split_end[0] = static_cast<int>(p->split[0]);
    a.split_end[1] = a.split_end[0] + static_cast<int>(p->split[1]);
    a.split_end[2] = a.split_end[1] + static_cast<int>(p->split[2]);
    a.xcd_groups = xcd_groups(p) ? 1 : 0;
    a.row_groups = a.group_tiles = a.longer_groups = 0;
    const hstu::IlsRowsVariant* rows = select_rows(p);
    if (rows != nullptr) {
        const int row_tiles = static_cast<int>((p->m + hstu::kIlsRowsTile - 1) / hstu::kIlsRowsTile);
        a.row_groups = rows_groups(p);
        a.group_tiles = row_tiles / a.row_groups;
        a.longer_groups = row_tiles % a.row_groups;
    }
    const unsigned grid = static_cast<unsigned>(grid_size(p));
    hipLaunchKernelGGL(rows != nullptr ? rows->kernel : select(p)->kernel, dim3(grid),
                       dim3(rows != nullptr ? hstu::kIlsRowsThreads : hstu::kIlsThreads), 0, static_cast<hipStream_t>(stream), a);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        return hstu::set_error(HSTU_ERR_RUNTIME, "launch of %s failed: %s", in_linear_silu_fwd_kernel_name(p), hipGetErrorString(err));
    }
    return HSTU_OK;
}

}  // extern "C"
