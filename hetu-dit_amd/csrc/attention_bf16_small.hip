// Joint flash attention, head dim 64, with one 32-row query block per wave: workgroups of 128 query rows, three per CU
// (device code and its description: attention_bf16_kernels.h).  Which launches it serves: `small_tiles_serve` in attention_bf16.hip.
// A wave does half the MFMAs and softmax of a 64-row wave on the same fragment reads (LDS busy for about half of the
// time, no longer a quarter), which costs 8 % per row on a full chip, and needs 168 registers instead of 256.
#define HDIT_ATTN_QUERY_BLOCKS 1
#include "attention_bf16_kernels.h"

namespace hdit_attn {
int launch_d64_small(const AttnParams& P, int q_tiles, unsigned grid, hipStream_t stream) {
  hipLaunchKernelGGL(attn_fwd_kernel<64>, dim3(grid), dim3(256), Lds<64>::TOTAL, stream, P, q_tiles);
  return HDIT_OK;
}

int launch_multi_d64_small(const AttnParams* P, const int* q_tiles, const int* nblocks, int count, hipStream_t stream) {
  AttnMulti M;
  const int grid = fill_multi(M, P, q_tiles, nblocks, count);
  hipLaunchKernelGGL(attn_fwd_multi_kernel<64>, dim3((unsigned)grid), dim3(256), Lds<64>::TOTAL, stream, M);
  return HDIT_OK;
}
}  // namespace hdit_attn
