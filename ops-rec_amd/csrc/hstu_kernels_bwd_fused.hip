// backward kernels of the order that hands dS alone from one launch to the next
#include "hstu_bwd_fused_kernel.hip.h"
#include "hstu_variants.h"

namespace hstu {
namespace {
#define HSTU_BWD_FUSED(tag, tagname, D) \
    {"hstu_bwd_" tagname "_d" #D "_fused", hstu_bwd_kv_fused_kernel<tag, D>, hstu_bwd_kv_fused_kernel<tag, D, true>, \
     hstu_bwd_dq_from_ds_kernel<tag, D, false>, hstu_bwd_dq_from_ds_kernel<tag, D, true>}
const BwdFusedVariant kFused[2][3] = {
    {HSTU_BWD_FUSED(bf16_tag, "bf16", 64), HSTU_BWD_FUSED(bf16_tag, "bf16", 128), HSTU_BWD_FUSED(bf16_tag, "bf16", 256)},
    {HSTU_BWD_FUSED(f16_tag, "f16", 64), HSTU_BWD_FUSED(f16_tag, "f16", 128), HSTU_BWD_FUSED(f16_tag, "f16", 256)}};
}  // namespace
const BwdFusedVariant (*bwd_variants_fused())[3] { return kFused; }
}  // namespace hstu
