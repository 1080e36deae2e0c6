// forward kernels with the output sums in pinned accumulators
#include "hstu_fwd_pinned_kernel.hip.h"
#include "hstu_variants.h"

namespace hstu {
namespace {
const ShortVariant kPinned[2] = {{"hstu_fwd_bf16_d256_rabfalse_maskfalse_pinned", hstu_fwd_pinned_kernel<bf16_tag, 256>},
                                 {"hstu_fwd_f16_d256_rabfalse_maskfalse_pinned", hstu_fwd_pinned_kernel<f16_tag, 256>}};
}  // namespace
const ShortVariant* fwd_variants_pinned() { return kPinned; }
}  // namespace hstu
