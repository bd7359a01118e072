// The tracked bf16 flash-attention kernel of head dim 128 (device code: attention_bf16_kernels.h).  A translation unit of
// its own because it is compiled without the VGPR-form MFMA option: with 128 output accumulator registers per lane the P.V
// accumulators have to live in the AGPR half.
#include "attention_bf16_kernels.h"

namespace hdit_attn {
HDIT_ATTN_LAUNCH(launch_tracked_d128, 128, attn_fwd_kernel, attn_fwd_multi_kernel, Lds)
}  // namespace hdit_attn
