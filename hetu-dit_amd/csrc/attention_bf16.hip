// Joint (image + text) flash attention forward for gfx950, bf16 in/out: the C entry points and the choice of the kernel
// (device code and its description: attention_bf16_kernels.h).
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
bool to_params(const hdit_attn_args* a, AttnParams& P) {
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
  return true;
}

// Which kernel serves a problem.  The pipelined ones where there are enough tiles of keys (pipe_min_tiles) and a tile's step
// fits 32 bits; the tracked one otherwise.  That is decided from keys and strides alone, and a row's result depends on the row
// and the keys alone: neither rows that are left out (the text queries of a joint sequence) nor other problems of the
// launch change a bit.
// HDIT_ATTN_PIPE=0 keeps every launch on the tracked kernel, =4 and =8 every other one of head dim 64 on workgroups of four
// or eight waves (for A/B timing).
char pipe_env() {
  static const char* env = getenv("HDIT_ATTN_PIPE");
  return env ? env[0] : 0;
}

bool is_pipelined(const hdit_attn_args* a, const AttnParams& P) {
  const bool strides_ok = a->k[0].stride_s < (1 << 22) && a->k[1].stride_s < (1 << 22) && a->v[0].stride_s < (1 << 22) &&
                          a->v[1].stride_s < (1 << 22);  // a tile step (64 rows, in bytes) fits 32 bits
  return pipe_env() != '0' && strides_ok && (P.skv + BKV - 1) / BKV >= hdit_attn::pipe_min_tiles(a->head_dim);
}

int64_t rows_of(const hdit_attn_args* a) { return a->q[0].len + a->q[1].len; }

int64_t workgroups(const hdit_attn_args* a, int rows_per_workgroup) {
  return (int64_t)a->batch * a->heads * ((rows_of(a) + rows_per_workgroup - 1) / rows_per_workgroup);
}

// A launch of workgroups of eight waves, one per CU: `full` of them with 256 rows and, dealt out behind those, `half` with
// 128, which take HALF_COST of the time.  Returns the rounds it takes.
constexpr double HALF_COST = 0.62;
double rounds(int64_t full, int64_t half, int64_t cus) {
  const int64_t whole = full / cus, late = full % cus, early = cus - late;  // CUs that are free at `whole`, at `whole` + 1
  if (half == 0) return (double)(whole + (late > 0));
  for (int64_t n = 1;; n++) {  // n half tiles one after the other on the early CUs, and what fits beside them on the late ones
    const double end = n * HALF_COST;
    const int64_t on_late = end > 1.0 ? (int64_t)((end - 1.0) / HALF_COST + 1e-9) : 0;
    if (early * n + late * on_late >= half) return (double)whole + (late && end < 1.0 ? 1.0 : end);
  }
}

// How many 256-row tiles a (batch, head) of a problem has; the rows behind them go to half tiles.  A launch that ends with
// a round of few workgroups is over sooner if those are twice as many of half the rows: as many whole tiles as fill whole
// rounds, or all of them (a last one with more than 128 rows counts as whole), whichever ends first.  24 heads of 16896
// rows at d = 128 are 1584 workgroups, six rounds and 48: 2845 -> 2725 us, 2854 -> 2789 in another run; 12000 rows (1128) 1439 ->
// 1360; 512 rows (48) 20.9 -> 15.4.
struct Tiling {
  int full;
  double rounds;
};
Tiling tiling(const hdit_attn_args* a, int64_t cus) {
  const int64_t bh = (int64_t)a->batch * a->heads, rows = rows_of(a), most = rows / 256 + (rows % 256 > 128);
  auto end = [&](int64_t f) { return rounds(bh * f, rows > 256 * f ? bh * ((rows - 256 * f + 127) / 128) : 0, cus); };
  Tiling best = {(int)most, end(most)};
  for (int64_t whole = bh * most / cus; whole >= 0 && whole + 2 > bh * most / cus; whole--) {
    const int64_t f = whole * cus / bh;
    if (end(f) < best.rounds - 0.05) best = {(int)f, end(f)};
  }
  return best;
}

// Query rows per workgroup of a pipelined launch at head dim 64, by how the workgroups fill the CUs.  Measured on MI355X,
// 24 heads and more, microseconds per tile of 64 keys:
//   128 rows, four waves, two workgroups per CU   0.55 where a CU has one, 0.90 where it has two
//   256 rows, eight waves, one per CU             0.86, and 1 us more until it has begun (five tiles ahead, no neighbour)
// Per row the same, so the last round decides, and small workgroups where CUs would be idle.  128 / 256 rows: 333 rows
// 8.6 / 11.4 us, 2 x 666 15.0 / 16.1, 2 x 1357 37.1 / 39.3, 1024 of 4429 rows 41.0 / 57.5, two of them 63.3 / 60.1, 4470
// rows 127.9 / 122.4, 2 x 4429 227 / 247, 17776 rows with 48 heads 3443 / 3378.
int pipe_rows(const hdit_attn_args* const* of, int count, int cus) {
  if (pipe_env() == '4') return 128;
  if (pipe_env() == '8') return 256;
  int64_t small = 0, large = 0, tiles = 0;
  for (int i = 0; i < count; i++) {
    small += workgroups(of[i], 128), large += workgroups(of[i], 256);
    const int64_t t = (of[i]->k[0].len + of[i]->k[1].len + BKV - 1) / BKV;
    if (t > tiles) tiles = t;
  }
  if (cus <= 0) return 256;  // no device to ask: the launch reports it
  small = (small + cus - 1) / cus;
  const double cost_small = tiles * (0.90 * (double)(small / 2) + 0.55 * (double)(small % 2));
  const double cost_large = tiles * 0.86 * (count == 1 ? tiling(of[0], cus).rounds : (double)((large + cus - 1) / cus)) + 1.0;
  return cost_small <= 1.05 * cost_large ? 128 : 256;  // (2 x 4429 rows: modelled 228 / 219, measured 242 / 244)
}

// Query rows per workgroup of a launch.  The tracked kernel serves few keys: d = 64 small workgroups, ahead at every fill
// (attention_bf16_kernels.h), d = 128 large ones.
int launch_rows(const hdit_attn_args* const* of, int count, bool pipelined, int cus) {
  if (of[0]->head_dim == 128) return 256;
  return pipelined ? pipe_rows(of, count, cus) : 128;
}

// The problems of one call that one kernel serves, as one launch.
int launch_some(const hdit_attn_args* const* of, const AttnParams* P, int count, bool pipelined, hipStream_t s) {
  const int hd = of[0]->head_dim, cus = hdit_host::num_cus();
  const int rows = launch_rows(of, count, pipelined, cus), part = rows == 256 ? rows / 2 : rows;
  int q_tiles[HDIT_ATTN_MAX_MULTI], q_full[HDIT_ATTN_MAX_MULTI], nblocks[HDIT_ATTN_MAX_MULTI];
  for (int i = 0; i < count; i++) {
    const bool tiled = pipelined && rows == 256 && count == 1 && cus > 0;
    q_full[i] = tiled ? tiling(of[i], cus).full : P[i].sq / rows + (P[i].sq % rows > part);
    const int left = P[i].sq - q_full[i] * rows;
    q_tiles[i] = q_full[i] + (left > 0 ? (left + part - 1) / part : 0);
    nblocks[i] = of[i]->batch * of[i]->heads * q_tiles[i];
  }
  if (!pipelined)
    return hd == 64 ? hdit_attn::launch_tracked4_d64(P, q_tiles, q_full, nblocks, count, s)
                    : hdit_attn::launch_tracked8_d128(P, q_tiles, q_full, nblocks, count, s);
  if (hd == 128) return hdit_attn::launch_pipe8_d128(P, q_tiles, q_full, nblocks, count, s);
  return rows == 128 ? hdit_attn::launch_pipe4_d64(P, q_tiles, q_full, nblocks, count, s)
                     : hdit_attn::launch_pipe8_d64(P, q_tiles, q_full, nblocks, count, s);
}
}  // namespace

extern "C" __attribute__((visibility("default"))) int hdit_attn_rows(const hdit_attn_args* args, int count, int cus) {
  if (!args || count <= 0 || count > HDIT_ATTN_MAX_MULTI || cus <= 0) return HDIT_EINVAL;
  const hdit_attn_args* of[HDIT_ATTN_MAX_MULTI];
  AttnParams P[HDIT_ATTN_MAX_MULTI];
  for (int i = 0; i < count; i++) {
    const int rc = hdit_host::attn_validate(&args[i]);
    if (rc != HDIT_OK) return rc;
    if (!to_params(&args[i], P[i]) || args[i].head_dim != args[0].head_dim) return HDIT_EINVAL;
    if (is_pipelined(&args[i], P[i]) != is_pipelined(&args[0], P[0])) return HDIT_EINVAL;
    of[i] = &args[i];
  }
  return launch_rows(of, count, is_pipelined(args, P[0]), cus);
}

extern "C" __attribute__((visibility("default"))) int hdit_attn_fwd_bf16(const hdit_attn_args* a, void* stream) {
  int rc = hdit_host::attn_validate(a);
  if (rc != HDIT_OK) return rc;
  AttnParams P;
  if (!to_params(a, P)) return HDIT_OK;
  rc = launch_some(&a, &P, 1, is_pipelined(a, P), (hipStream_t)stream);
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
  // one merged launch of the problems for the pipelined kernels, one of the others
  for (int pass = 0; pass < 2; pass++) {
    AttnParams P[HDIT_ATTN_MAX_MULTI];
    const hdit_attn_args* of[HDIT_ATTN_MAX_MULTI];
    int n = 0;
    for (int i = 0; i < count; i++) {
      if (!to_params(&args[i], P[n]) || is_pipelined(&args[i], P[n]) != (pass == 0)) continue;
      of[n++] = &args[i];
    }
    if (n == 0) continue;
    int rc = launch_some(of, P, n, pass == 0, (hipStream_t)stream);
    if (rc != HDIT_OK) return rc;
    if ((rc = hdit_host::check_launch("hdit_attn_fwd_bf16_multi")) != HDIT_OK) return rc;
  }
  return HDIT_OK;
}
