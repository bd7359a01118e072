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

// A launch of workgroups of eight waves, one per CU: `full` of them with 256 rows and, dealt out behind those, `half` with
// 128, which take HALF_COST of the time.  Returns the rounds it takes.
//
// Workgroups go to the XCDs in turn, and there, in order, to four shader engines of eight CUs in turn.  One whose engine
// has no CU free waits, and everything behind it does, also where another engine has one: with 30 full tiles on an XCD the
// third half tile runs behind a full one, not on one of the two CUs that are free.  24 heads of 2654 rows in full / half
// tiles per head, us (rounds by this model): d = 64 10 / 1 68.0 (1.65), 8 / 5 56.7 (1.3), 0 / 21 55.0 (1.3); d = 128
// 10 / 1 108 (1.65), 0 / 21 88 (1.3); 4000 rows, d = 64, 10 / 12 127.8 (2.3), 16 / 0 109.5 (2).  Over 180 such launches the
// model's times are off by 4 % rms.  HALF_COST is fitted to them: 0.66 at d = 64, 0.64 at d = 128.
constexpr double HALF_COST = 0.65;
constexpr int XCD_CUS = 32, ENGINES = 4;
double rounds(int64_t full, int64_t half, int64_t cus) {
  const int64_t xcds = cus > XCD_CUS ? cus / XCD_CUS : 1;
  const int64_t f = (full + xcds - 1) / xcds, n = (full + half + xcds - 1) / xcds;  // on the first XCD, which has most
  const int64_t whole = f / XCD_CUS;
  const int late = (int)(f % XCD_CUS);  // CUs that are free at `whole` + 1, the others at `whole`
  constexpr int SLOTS = XCD_CUS / ENGINES;
  // Per engine: CUs that have begun a half tile, those ended and followed by another, and the ends of all, in order (a ring).
  int taken[ENGINES] = {}, ended[ENGINES] = {};
  double ends[ENGINES][SLOTS];
  double start = 0.0, end = late > 0;
  for (int64_t w = f; w < n; w++) {
    const int e = (int)(w % ENGINES), first_late = SLOTS - (late / ENGINES + (e < late % ENGINES));
    const double fresh = taken[e] < first_late ? 0.0 : taken[e] < SLOTS ? 1.0 : 1e30;
    const bool again = taken[e] > 0 && ends[e][ended[e] % SLOTS] < fresh;
    const double at = again ? ends[e][ended[e] % SLOTS] : fresh;
    if (at > start) start = at;
    (again ? ended : taken)[e]++;
    ends[e][(taken[e] + ended[e] - 1) % SLOTS] = start + HALF_COST;
    if (start + HALF_COST > end) end = start + HALF_COST;
  }
  return (double)whole + end;
}

// How many 256-row tiles a (batch, head) of a problem has; the rows behind them go to half tiles.  A launch that ends with
// a round of few workgroups is over sooner if those are twice as many of half the rows: as many whole tiles as fill whole
// rounds, or all of them (a last one with more than 128 rows counts as whole), whichever ends first.  24 heads at d = 128,
// us: 16896 rows are 1584 workgroups, six rounds and 48: 2823 with all of them whole, 2668 with 64 whole tiles per head;
// 3830 rows 181.5 -> 153.4; 2654 rows 108 -> 88.
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
    if (f == most) continue;
    const double e = end(f);
    if (e < best.rounds - 0.05) best = {(int)f, e};
  }
  return best;
}

// Query rows per workgroup of a pipelined launch at head dim 64, by how the workgroups fill the CUs.  A CU takes a round of
// two workgroups of 128 rows (four waves each) or of one with 256 (eight) in about the same time, 0.9 us per tile of 64 keys
// and 5 us for beginning and end, the eight waves in a little less; one workgroup of 128 alone in 0.56 of it, a half tile of
// 128 in a workgroup of eight waves in HALF_COST.  So the last round decides, and where it is the same the large workgroups,
// unless more than half of their waves have no rows (2 x 666 rows 15.1 / 15.7).
// Measured on MI355X, 128 / 256 rows, us: 24 heads 1357 rows 23.5 / 23.1, 2445 41.9 / 39.1, 2654 45.2 / 52.1, 4470 131.9 /
// 123.7, 2 x 1357 37.9 / 39.2, 2 x 1024 of 4429 65.6 / 59.9, 2 x 1357 of 4429 99.7 / 102.1, 2 x 4429 235 / 235, 4 x 2637 169 / 178;
// 48 heads 8000 rows 703 / 676, 13226 1906 / 1826, 17776 3444 / 3428.
// Over 143 launches of 400 - 13000 keys the choice is 0.5 % slower than the better one on average (always 128: 1.8 %, always 256:
// 1.7 %), 11 % at most.  Merged launches deal out problem by problem, half tiles in between, and large workgroups lose step with
// more rounds: of more than two rounds they were level or behind in most launches, up to 15 %; of one or two ahead by 2 - 6 %
// with the patches of SD3 steps (1357 + 1024 rows of 4429 69.0 / 65.8).
int pipe_rows(const hdit_attn_args* const* of, int count, int cus, Tiling& tiles) {
  if (pipe_env() == '4') return 128;
  if (pipe_env() == '8') return 256;
  if (cus <= 0) return 256;  // no device to ask: the launch reports it
  int64_t waves = 0, small = 0, full = 0, half = 0;
  for (int i = 0; i < count; i++) {
    const int64_t bh = (int64_t)of[i]->batch * of[i]->heads, rows = rows_of(of[i]), rest = rows % 256;
    waves += bh * ((rows + 31) / 32), small += bh * ((rows + 127) / 128), full += bh * (rows / 256 + (rest > 128)), half += bh * (rest > 0 && rest <= 128);
  }
  const int64_t rest = small % (2 * cus);
  const double rounds_small = (double)(small / (2 * cus)) + (rest == 0 ? 0.0 : rest <= cus ? 0.56 : 1.0);
  if (count == 1) tiles = tiling(of[0], cus);
  const double rounds_large = count == 1 ? tiles.rounds : rounds(full, half, cus);
  if ((count > 1 && rounds_large > 2.0) || (double)waves < 0.5 * rounds_large * 8 * cus) return 128;
  return rounds_small <= 0.99 * rounds_large ? 128 : 256;
}

// Query rows per workgroup of a launch.  The tracked kernel serves few keys: d = 64 small workgroups, ahead at every fill
// (attention_bf16_kernels.h), d = 128 large ones.  `tiles`: of a single problem, where the choice needed it.
int launch_rows(const hdit_attn_args* const* of, int count, bool pipelined, int cus, Tiling& tiles) {
  if (of[0]->head_dim == 128) return 256;
  return pipelined ? pipe_rows(of, count, cus, tiles) : 128;
}

// The problems of one call that one kernel serves, as one launch; `pinned` rows per workgroup where there is a choice and
// it is not 0.
int launch_some(const hdit_attn_args* const* of, const AttnParams* P, int count, bool pipelined, int pinned, hipStream_t s) {
  const int hd = of[0]->head_dim, cus = hdit_host::num_cus();
  Tiling tiles = {-1, 0.0};
  const int rows = pinned && pipelined && hd == 64 ? pinned : launch_rows(of, count, pipelined, cus, tiles);
  const int part = rows == 256 ? rows / 2 : rows;
  int q_tiles[HDIT_ATTN_MAX_MULTI], q_full[HDIT_ATTN_MAX_MULTI], nblocks[HDIT_ATTN_MAX_MULTI];
  for (int i = 0; i < count; i++) {
    const bool tiled = pipelined && rows == 256 && count == 1 && cus > 0;
    if (tiled && tiles.full < 0) tiles = tiling(of[i], cus);
    q_full[i] = tiled ? tiles.full : P[i].sq / rows + (P[i].sq % rows > part);
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
  Tiling tiles;
  return launch_rows(of, count, is_pipelined(args, P[0]), cus, tiles);
}

namespace {
int attn_fwd(const hdit_attn_args* args, int count, int pinned, hipStream_t stream, const char* what) {
  if (!args || count <= 0 || count > HDIT_ATTN_MAX_MULTI) return HDIT_EINVAL;
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
    int rc = launch_some(of, P, n, pass == 0, pinned, stream);
    if (rc != HDIT_OK) return rc;
    if ((rc = hdit_host::check_launch(what)) != HDIT_OK) return rc;
  }
  return HDIT_OK;
}
}  // namespace

extern "C" __attribute__((visibility("default"))) int hdit_attn_fwd_bf16(const hdit_attn_args* a, void* stream) {
  return attn_fwd(a, 1, 0, (hipStream_t)stream, "hdit_attn_fwd_bf16");
}

extern "C" __attribute__((visibility("default"))) int hdit_attn_fwd_bf16_multi(const hdit_attn_args* args, int count, void* stream) {
  return attn_fwd(args, count, 0, (hipStream_t)stream, "hdit_attn_fwd_bf16_multi");
}

extern "C" __attribute__((visibility("default"))) int hdit_attn_fwd_bf16_rows(const hdit_attn_args* args, int count, int rows, void* stream) {
  if (rows != 128 && rows != 256) return HDIT_EINVAL;
  return attn_fwd(args, count, rows, (hipStream_t)stream, "hdit_attn_fwd_bf16_rows");
}
