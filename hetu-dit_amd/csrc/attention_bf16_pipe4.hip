// The pipelined bf16 flash-attention kernel with workgroups of four waves, 128 query rows, two per CU (device code and its
// description: attention_bf16_kernels.h).  Which launches it serves: `pipe_rows` in attention_bf16.hip.
#define HDIT_ATTN_QUERY_BLOCKS 1
#define HDIT_ATTN_WAVES 4
#include "attention_bf16_kernels.h"

namespace hdit_attn {
HDIT_ATTN_LAUNCH(launch_pipe4_d64, 64, attn_fwd_pipe_kernel, attn_fwd_pipe_multi_kernel, PipeLds)
}  // namespace hdit_attn
