// Joint (image + text) flash attention forward for gfx950, bf16 in/out: the C entry point and the head-dim-64
// kernels (device code and its description: attention_bf16_kernels.h).
#include "attention_bf16_kernels.h"

namespace {

bool seg_ok(const hdit_seq_segment& s, bool need_ptr) {
  if (s.len < 0) return false;
  if (s.len == 0) return true;
  if (need_ptr && !s.ptr) return false;
  if (((uintptr_t)s.ptr) & 15) return false;
  if (s.stride_b % 8 || s.stride_s % 8 || s.stride_h % 8) return false;
  return true;
}

Seg2 make_seg(const hdit_seq_segment* s) {
  Seg2 r;
  r.p0 = (const __bf16*)s[0].ptr;
  r.sb0 = s[0].stride_b;
  r.ss0 = s[0].stride_s;
  r.sh0 = s[0].stride_h;
  r.len0 = s[0].len;
  r.p1 = (const __bf16*)s[1].ptr;
  r.sb1 = s[1].stride_b;
  r.ss1 = s[1].stride_s;
  r.sh1 = s[1].stride_h;
  r.len1 = s[1].len;
  return r;
}

}  // namespace

namespace hdit_attn {
int launch_d64(const AttnParams& P, int q_tiles, unsigned grid, bool pipelined, hipStream_t stream) {
  if (pipelined) {
    static std::atomic<bool> attr{false};  // setting the attribute twice from two threads is harmless
    if (!attr.load(std::memory_order_acquire)) {
      if (hipFuncSetAttribute((const void*)attn_fwd_pipe_kernel<64>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              PipeLds<64>::TOTAL) != hipSuccess)
        return HDIT_ELAUNCH;
      attr.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL(attn_fwd_pipe_kernel<64>, dim3(grid), dim3(256), PipeLds<64>::TOTAL, stream, P, q_tiles);
  } else {
    hipLaunchKernelGGL(attn_fwd_kernel<64>, dim3(grid), dim3(256), Lds<64>::TOTAL, stream, P, q_tiles);
  }
  return HDIT_OK;
}

int launch_multi_d64(const AttnParams* P, const int* q_tiles, const int* nblocks, int count, bool pipelined, hipStream_t stream) {
  AttnMulti M;
  const int grid = fill_multi(M, P, q_tiles, nblocks, count);
  static std::atomic<bool> attr{false};  // setting the attributes twice from two threads is harmless
  if (!attr.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute((const void*)attn_fwd_pipe_multi_kernel<64>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            PipeLds<64>::TOTAL) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_fwd_multi_kernel<64>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            Lds<64>::TOTAL) != hipSuccess)
      return HDIT_ELAUNCH;
    attr.store(true, std::memory_order_release);
  }
  if (pipelined)
    hipLaunchKernelGGL(attn_fwd_pipe_multi_kernel<64>, dim3((unsigned)grid), dim3(256), PipeLds<64>::TOTAL, stream, M);
  else
    hipLaunchKernelGGL(attn_fwd_multi_kernel<64>, dim3((unsigned)grid), dim3(256), Lds<64>::TOTAL, stream, M);
  return HDIT_OK;
}
}  // namespace hdit_attn

namespace hdit_host {
int attn_validate(const hdit_attn_args* a) {
  if (!a) return HDIT_EINVAL;
  if (a->batch <= 0 || a->heads <= 0) return HDIT_EINVAL;
  if (a->head_dim != 64 && a->head_dim != 128) return HDIT_EUNSUPPORTED;
  for (int i = 0; i < 2; i++)
    if (!seg_ok(a->q[i], true) || !seg_ok(a->k[i], true) || !seg_ok(a->v[i], true) || !seg_ok(a->o[i], true))
      return HDIT_EINVAL;
  if (a->k[0].len != a->v[0].len || a->k[1].len != a->v[1].len) return HDIT_EINVAL;
  if (a->q[0].len != a->o[0].len || a->q[1].len != a->o[1].len) return HDIT_EINVAL;
  if (a->q[0].len + a->q[1].len > 0 && a->k[0].len + a->k[1].len == 0) return HDIT_EINVAL;
  return HDIT_OK;
}
}  // namespace hdit_host

namespace {
// validated arguments -> kernel parameters; false: no query rows, nothing to do
bool to_params(const hdit_attn_args* a, AttnParams& P, int& q_tiles, unsigned& grid) {
  P.q = make_seg(a->q);
  P.k = make_seg(a->k);
  P.v = make_seg(a->v);
  P.o = make_seg(a->o);
  P.heads = a->heads;
  P.sq = a->q[0].len + a->q[1].len;
  P.skv = a->k[0].len + a->k[1].len;
  if (P.sq == 0) return false;
  const float scale = a->scale > 0.f ? a->scale : 1.0f / sqrtf((float)a->head_dim);
  P.scale_log2 = scale * 1.4426950408889634f;
  q_tiles = (P.sq + BQ - 1) / BQ;
  grid = (unsigned)(q_tiles * a->batch * a->heads);
  return true;
}
}  // namespace

namespace {
// Which kernel serves a problem.
// d = 128: the tracked kernel runs one wave per SIMD as well, so the pipelined one serves every grid.
// d = 64: the small and the tracked kernel give the same bits; the pipelined one, whose softmax reference is fixed, does
// not.  So whether a problem gets the pipelined kernel is decided from the problem alone (launched on its own or merged
// with others, it keeps its bits), and in the same way with and without the text queries of a joint sequence, whose
// image rows keep their bits: a query segment that is left out counts as if it were there (`rows_with_text`), and query
// patches of joint sequences never get that kernel.  (Exception: image rows in a workgroup of the pipelined kernel that
// also holds text rows.  If a text row outgrows the fixed reference by 2^64, the tracked kernel computes the workgroup.)
// What decides is how the workgroups fill the CUs, in microseconds per tile of 64 keys (measured on MI355X for one and
// two batch elements of 24 heads and 333 - 4470 rows, less a fixed 4.5 us):
//   small      (128 query rows, three workgroups per CU)   0.75 with one per CU, 1.10 with two, 1.60 with three
//   tracked    (256 rows, two per CU)                       1.16, 1.95
//   pipelined  (256 rows, one per CU)                       1.05 a round
// So the small tiles serve grids that would leave CUs idle (333 rows 12.8 -> 9.2 us, 1117 rows 23.5 -> 18.0, 1024 of
// 4429 rows 68 -> 54) or half idle in the last round (2 x 1357 rows 45 -> 39, 4000 rows 118 -> 108), the pipelined
// kernel one full round (2445 rows 49.6 -> 43.4), the tracked kernel everything larger: per row it does the least.
// A problem with fewer query than key rows is a patch of a pipeline, which shares its launch with the other patches of
// the step or runs alone: it is decided by the whole sequence.  Small tiles serve both uses well (24 heads, 1024 of
// 4429 rows: alone 54 us, pipelined 68, tracked 78; four in one launch, one with 333 text queries, 164, pipelined 170) until
// the patches of a step make more than two full rounds of the tracked kernel's.  The pipelined kernel serves patches of
// longer sequences only where the keys are one segment, so that no text queries can be left out (648 of 5517 rows, two
// batch elements: 84 us, tracked 96).
// HDIT_ATTN_PIPE=0 keeps every launch on the tracked-reference kernel with 256 rows, =1 puts every eligible launch on the
// pipelined ones (for A/B timing).
enum Kind { TRACKED, PIPELINED, SMALL, KINDS };
constexpr int SMALL_BQ = 128;

double fill_cost(Kind kind, int64_t workgroups, int cus) {
  const int64_t per_cu = (workgroups + cus - 1) / cus;
  if (kind == PIPELINED) return 1.05 * (double)per_cu;
  if (kind == TRACKED) return 1.95 * (double)(per_cu / 2) + (per_cu % 2 ? 1.16 : 0.0);
  const int rest = (int)(per_cu % 3);
  if (per_cu < 3) return rest == 1 ? 0.75 : 1.10;
  return 1.60 * (double)(per_cu / 3) + 0.55 * rest;
}

// The query rows of a problem, a segment counted with its key rows where its queries were left out: one that is empty
// while the other one lies within the key segment of its own.
int rows_with_text(const hdit_attn_args* a) {
  int rows = a->q[0].len + a->q[1].len;
  for (int s = 0; s < 2; s++)
    if (a->q[s].len == 0 && a->q[1 - s].len <= a->k[1 - s].len) rows += a->k[s].len;
  return rows;
}

// the kernel of a problem, with its grid in that kernel's tiles
Kind choose(const hdit_attn_args* a, const AttnParams& P, int& q_tiles, unsigned& grid) {
  static const char* pipe_env = getenv("HDIT_ATTN_PIPE");
  const bool pipe_off = pipe_env && pipe_env[0] == '0', pipe_force = pipe_env && pipe_env[0] == '1';
  const bool strides_ok = a->k[0].stride_s < (1 << 22) && a->k[1].stride_s < (1 << 22) && a->v[0].stride_s < (1 << 22) &&
                          a->v[1].stride_s < (1 << 22);  // a tile step (64 rows, in bytes) fits 32 bits
  const bool can_pipe = !pipe_off && strides_ok && (P.skv + BKV - 1) / BKV >= PIPE_MIN_TILES;
  if (a->head_dim == 128 || pipe_off || pipe_force) return can_pipe ? PIPELINED : TRACKED;
  const int cus = hdit_host::num_cus(), tiles_small = (P.sq + SMALL_BQ - 1) / SMALL_BQ;
  if (cus <= 0) return TRACKED;  // no device to ask: the launch reports it
  const int64_t bh = (int64_t)a->batch * a->heads;
  const int rows = rows_with_text(a);
  bool small;
  Kind large;
  if (rows < P.skv) {
    small = bh * ((P.skv + BQ - 1) / BQ) <= 4 * (int64_t)cus;
    const bool joint = a->k[0].len > 0 && a->k[1].len > 0;
    large = can_pipe && !joint && bh * q_tiles * 8 <= (int64_t)cus * 5 ? PIPELINED : TRACKED;
  } else {
    const int64_t grid_large = bh * ((rows + BQ - 1) / BQ), grid_small = bh * ((rows + SMALL_BQ - 1) / SMALL_BQ);
    const double tracked = fill_cost(TRACKED, grid_large, cus), cost = fill_cost(SMALL, grid_small, cus);
    const double piped = can_pipe ? fill_cost(PIPELINED, grid_large, cus) : 1e30;
    // (a few per cent are less than the model resolves: 2 x 4429 rows 264.7 us on small tiles, 264.1 tracked)
    small = cost < 0.93 * tracked && cost < piped;
    large = piped < tracked ? PIPELINED : TRACKED;
  }
  if (small) {
    q_tiles = tiles_small;
    grid = (unsigned)(bh * tiles_small);
    return SMALL;
  }
  return large;
}

int launch_one(int head_dim, const AttnParams& P, int q_tiles, unsigned grid, Kind kind, hipStream_t s) {
  if (kind == SMALL) return hdit_attn::launch_d64_small(P, q_tiles, grid, s);
  return head_dim == 64 ? hdit_attn::launch_d64(P, q_tiles, grid, kind == PIPELINED, s)
                        : hdit_attn::launch_d128(P, q_tiles, grid, kind == PIPELINED, s);
}
}  // namespace

extern "C" __attribute__((visibility("default"))) int hdit_attn_fwd_bf16(const hdit_attn_args* a, void* stream) {
  int rc = hdit_host::attn_validate(a);
  if (rc != HDIT_OK) return rc;
  AttnParams P;
  int q_tiles;
  unsigned grid;
  if (!to_params(a, P, q_tiles, grid)) return HDIT_OK;
  const Kind kind = choose(a, P, q_tiles, grid);
  rc = launch_one(a->head_dim, P, q_tiles, grid, kind, (hipStream_t)stream);
  if (rc != HDIT_OK) return rc;
  return hdit_host::check_launch("hdit_attn_fwd_bf16");
}

extern "C" __attribute__((visibility("default"))) int hdit_attn_fwd_bf16_multi(const hdit_attn_args* args, int count, void* stream) {
  if (!args || count <= 0 || count > HDIT_ATTN_MAX_MULTI) return HDIT_EINVAL;
  if (count == 1) return hdit_attn_fwd_bf16(args, stream);
  for (int i = 0; i < count; i++) {
    const int rc = hdit_host::attn_validate(&args[i]);
    if (rc != HDIT_OK) return rc;
    if (args[i].head_dim != args[0].head_dim) return HDIT_EINVAL;
  }
  // one merged launch per kind of kernel the problems want
  for (int kind = 0; kind < KINDS; kind++) {
    AttnParams P[HDIT_ATTN_MAX_MULTI];
    int q_tiles[HDIT_ATTN_MAX_MULTI], nblocks[HDIT_ATTN_MAX_MULTI], n = 0;
    for (int i = 0; i < count; i++) {
      unsigned grid;
      if (!to_params(&args[i], P[n], q_tiles[n], grid)) continue;
      if ((int)choose(&args[i], P[n], q_tiles[n], grid) != kind) continue;
      nblocks[n++] = (int)grid;
    }
    if (n == 0) continue;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if (n == 1) rc = launch_one(args[0].head_dim, P[0], q_tiles[0], (unsigned)nblocks[0], (Kind)kind, s);
    else if (kind == SMALL) rc = hdit_attn::launch_multi_d64_small(P, q_tiles, nblocks, n, s);
    else
      rc = args[0].head_dim == 64 ? hdit_attn::launch_multi_d64(P, q_tiles, nblocks, n, kind == PIPELINED, s)
                                  : hdit_attn::launch_multi_d128(P, q_tiles, nblocks, n, kind == PIPELINED, s);
    if (rc != HDIT_OK) return rc;
    if ((rc = hdit_host::check_launch("hdit_attn_fwd_bf16_multi")) != HDIT_OK) return rc;
  }
  return HDIT_OK;
}
