// forward kernels with the output sums in pinned accumulators
#include "hstu_fwd_pinned_kernel.hip.h"
#include "hstu_variants.h"

namespace hstu {
namespace {
#define HSTU_PINNED(tag, tagname)                                                                    \
    {{"hstu_fwd_" tagname "_d128_rabfalse_maskfalse_pinned", hstu_fwd_pinned_kernel<tag, 128>},      \
     {"hstu_fwd_" tagname "_d256_rabfalse_maskfalse_pinned", hstu_fwd_pinned_kernel<tag, 256>}}
const ShortVariant kPinned[2][2] = {HSTU_PINNED(bf16_tag, "bf16"), HSTU_PINNED(f16_tag, "f16")};
}  // namespace
const ShortVariant (*fwd_variants_pinned())[2] { return kPinned; }
}  // namespace hstu
