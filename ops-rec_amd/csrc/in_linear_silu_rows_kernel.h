// The kernel of in_linear_silu with the weights in registers (in_linear_silu_rows_kernel.hip.h), for the host: its tile sizes and its
// instances, which a source of their own compiles (in_linear_silu_kernels_rows.hip).
#pragma once
#include "hstu_args.h"

namespace hstu {

constexpr int kIlsRowsTile = 32;   // x rows per step
constexpr int kIlsRowsCols = 256;  // output columns per workgroup: eight wavefronts of 32
constexpr int kIlsRowsThreads = 512;

// for k of at most 16 * steps
struct IlsRowsVariant {
    const char* name;
    void (*kernel)(const InLinearSiluArgs);
    int steps;
};
// [k up to 256; up to 384; up to 512]
const IlsRowsVariant* ils_rows_variants(bool bf16);

}  // namespace hstu
