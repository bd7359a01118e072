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
// Between small and tracked the whole launch decides (`small_tiles_serve`), with all problems that are merged in it: the
// same model holds for the patches of a step.  24 heads, image rows + 333 of text, us on tracked / small tiles:
//   4096 in two patches 137 / 159, in four 149 / 164; two batch elements of 4600 in two 307 / 335, of 2304 + 154 in two
//   116 / 92, of 5184 in eight (four per launch) 263 / 234; one patch of 1024 alone 79 / 58, with the text queries 82 / 79
// Patches of sequences up to 4 * CUs workgroups are never pipelined (1024 of 4429 rows alone 54 us small, 68 pipelined),
// those of longer ones only where the keys are one segment, so that no text queries can be left out (648 of 5517 rows,
// two batch elements: 84 us, small 92, tracked 96).
// HDIT_ATTN_PIPE=0 keeps every launch on the tracked-reference kernel with 256 rows, =1 puts every eligible launch on the
// pipelined ones (for A/B timing).
enum Kind { TRACKED, PIPELINED, SMALL };
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

int64_t workgroups(const hdit_attn_args* a, int rows, int rows_per_workgroup) {
  return (int64_t)a->batch * a->heads * ((rows + rows_per_workgroup - 1) / rows_per_workgroup);
}

bool pipe_off() {
  static const char* pipe_env = getenv("HDIT_ATTN_PIPE");
  return pipe_env && pipe_env[0] == '0';
}

bool wants_pipelined(const hdit_attn_args* a, const AttnParams& P) {
  static const char* pipe_env = getenv("HDIT_ATTN_PIPE");
  const bool pipe_force = pipe_env && pipe_env[0] == '1';
  const bool strides_ok = a->k[0].stride_s < (1 << 22) && a->k[1].stride_s < (1 << 22) && a->v[0].stride_s < (1 << 22) &&
                          a->v[1].stride_s < (1 << 22);  // a tile step (64 rows, in bytes) fits 32 bits
  if (pipe_off() || !strides_ok || (P.skv + BKV - 1) / BKV < PIPE_MIN_TILES) return false;
  if (a->head_dim == 128 || pipe_force) return true;
  const int cus = hdit_host::num_cus();
  if (cus <= 0) return false;  // no device to ask: the launch reports it
  const int rows = rows_with_text(a);
  if (rows < P.skv) {
    const bool joint = a->k[0].len > 0 && a->k[1].len > 0;
    return !joint && workgroups(a, P.skv, BQ) > 4 * (int64_t)cus && workgroups(a, rows, BQ) * 8 <= (int64_t)cus * 5;
  }
  const double tracked = fill_cost(TRACKED, workgroups(a, rows, BQ), cus), small = fill_cost(SMALL, workgroups(a, rows, SMALL_BQ), cus);
  const double piped = fill_cost(PIPELINED, workgroups(a, rows, BQ), cus);
  return piped < tracked && !(small < 0.93 * tracked && small < piped);
}

// Whether a launch of these many workgroups is better off with small tiles.  Where every workgroup of 256 rows has a CU
// to itself it is (no more than two small ones then share a CU); above, the fill decides, by more than the few per cent
// that the model resolves (2 x 4429 rows: 264.7 us on small tiles, 264.1 tracked).
bool small_tiles_serve(int64_t grid_tracked, int64_t grid_small) {
  const int cus = hdit_host::num_cus();
  if (pipe_off() || cus <= 0) return false;
  return grid_tracked <= cus || fill_cost(SMALL, grid_small, cus) < 0.93 * fill_cost(TRACKED, grid_tracked, cus);
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
  Kind kind = wants_pipelined(a, P) ? PIPELINED : TRACKED;
  if (kind == TRACKED && a->head_dim == 64 && small_tiles_serve(grid, workgroups(a, P.sq, SMALL_BQ))) {
    kind = SMALL;
    q_tiles = (P.sq + SMALL_BQ - 1) / SMALL_BQ;
    grid = (unsigned)workgroups(a, P.sq, SMALL_BQ);
  }
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
  // one merged launch of the problems for the pipelined kernel, one of the others
  for (int pass = 0; pass < 2; pass++) {
    AttnParams P[HDIT_ATTN_MAX_MULTI];
    const hdit_attn_args* of[HDIT_ATTN_MAX_MULTI];
    int q_tiles[HDIT_ATTN_MAX_MULTI], nblocks[HDIT_ATTN_MAX_MULTI], n = 0;
    int64_t grid_tracked = 0, grid_small = 0;
    for (int i = 0; i < count; i++) {
      unsigned grid;
      if (!to_params(&args[i], P[n], q_tiles[n], grid)) continue;
      if (wants_pipelined(&args[i], P[n]) != (pass == 0)) continue;
      grid_tracked += grid;
      grid_small += workgroups(&args[i], P[n].sq, SMALL_BQ);
      of[n] = &args[i];
      nblocks[n++] = (int)grid;
    }
    Kind kind = pass == 0 ? PIPELINED : TRACKED;
    if (kind == TRACKED && args[0].head_dim == 64 && n > 0 && small_tiles_serve(grid_tracked, grid_small)) {
      kind = SMALL;
      for (int i = 0; i < n; i++) {
        q_tiles[i] = (P[i].sq + SMALL_BQ - 1) / SMALL_BQ;
        nblocks[i] = (int)workgroups(of[i], P[i].sq, SMALL_BQ);
      }
    }
    if (n == 0) continue;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if (n == 1) rc = launch_one(args[0].head_dim, P[0], q_tiles[0], (unsigned)nblocks[0], kind, s);
    else if (kind == SMALL) rc = hdit_attn::launch_multi_d64_small(P, q_tiles, nblocks, n, s);
    else
      rc = args[0].head_dim == 64 ? hdit_attn::launch_multi_d64(P, q_tiles, nblocks, n, kind == PIPELINED, s)
                                  : hdit_attn::launch_multi_d128(P, q_tiles, nblocks, n, kind == PIPELINED, s);
    if (rc != HDIT_OK) return rc;
    if ((rc = hdit_host::check_launch("hdit_attn_fwd_bf16_multi")) != HDIT_OK) return rc;
  }
  return HDIT_OK;
}
