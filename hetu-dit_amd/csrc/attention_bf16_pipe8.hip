// The bf16 flash-attention kernels with workgroups of eight waves, 256 query rows, one per CU: two waves per SIMD that share
// their K and V tiles.  The pipelined ones, and the tracked one of head dim 128 (device code and its description:
// attention_bf16_kernels.h).
#define HDIT_ATTN_WAVES 8
#include "attention_bf16_kernels.h"

namespace hdit_attn {
HDIT_ATTN_LAUNCH(launch_tracked8_d128, 128, attn_fwd_kernel, attn_fwd_multi_kernel, Lds)
HDIT_ATTN_LAUNCH(launch_pipe8_d64, 64, attn_fwd_pipe_kernel, attn_fwd_pipe_multi_kernel, PipeLds)
HDIT_ATTN_LAUNCH(launch_pipe8_d128, 128, attn_fwd_pipe_kernel, attn_fwd_pipe_multi_kernel, PipeLds)
}  // namespace hdit_attn
