// The bf16 flash-attention kernels of head dim 64 with workgroups of four waves, 128 query rows: the tracked one, three per
// CU, and the pipelined one, two per CU (device code and its description: attention_bf16_kernels.h).  Which launches they
// serve: `is_pipelined` and `pipe_rows` in attention_bf16.hip.
#define HDIT_ATTN_WAVES 4
#include "attention_bf16_kernels.h"

namespace hdit_attn {
HDIT_ATTN_LAUNCH(launch_tracked4_d64, 64, attn_fwd_kernel, attn_fwd_multi_kernel, Lds)
HDIT_ATTN_LAUNCH(launch_pipe4_d64, 64, attn_fwd_pipe_kernel, attn_fwd_pipe_multi_kernel, PipeLds)
}  // namespace hdit_attn
