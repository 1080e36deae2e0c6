// in_linear_silu with the weights in registers
#include "in_linear_silu_rows_kernel.hip.h"

namespace hstu {
namespace {
#define HSTU_ILS_ROWS(tag, tagname)                                                            \
    {{"in_linear_silu_" tagname "_rows256", in_linear_silu_rows_kernel<tag, 16>, 16},          \
     {"in_linear_silu_" tagname "_rows384", in_linear_silu_rows_kernel<tag, 24>, 24},          \
     {"in_linear_silu_" tagname "_rows512", in_linear_silu_rows_kernel<tag, 32>, 32}}
const IlsRowsVariant kRows[2][3] = {HSTU_ILS_ROWS(bf16_tag, "bf16"), HSTU_ILS_ROWS(f16_tag, "f16")};
}  // namespace
const IlsRowsVariant* ils_rows_variants(bool bf16) { return kRows[bf16 ? 0 : 1]; }
}  // namespace hstu
