// Device code of the bf16 flash-attention kernels, shared by the translation units that instantiate them
// (attention_bf16_pipe4.hip, _pipe8.hip: workgroups of four and of eight waves; the C entry points and the choice between
// them: attention_bf16.hip).
//
// Joint (image + text) flash attention forward for gfx950, bf16 in/out.
//
// Two kernels: the pipelined one further down serves everything that has enough
// keys (pipe_min_tiles); the one described here ("tracked") the rest, and the rows
// for which the pipelined kernel's fixed softmax reference does not hold.
//
// Work split: one workgroup = 4 or 8 waves = 128 or 256 query rows of one (batch,
// head); each wave owns 32 query rows (one MFMA column block) and walks the keys in
// tiles of 64.  (Waves of 64 rows read half the K and V fragments per row, but with
// few keys what counts is how soon a workgroup is done: 48 heads, d = 64, four waves,
// 64 / 32 rows per wave: 333 x 128 9.8 / 5.8 us, 4096 x 77 24.0 / 21.9; 192 heads,
// 1024 x 192 29.6 / 21.9.  d = 128, 24 heads, four waves of 64 / eight of 32 rows:
// 128 x 128 11.2 / 8.5, 4096 x 77 29.5 / 27.5.)  K and V tiles go straight from global memory into two
// LDS buffers (direct-to-LDS loads, one barrier per tile).
//
// The scores are produced transposed, S^T = K . Q^T, with K rows as the MFMA
// "A" operand and the wave's Q rows (held in registers for the whole kernel)
// as the "B" operand.  In the 32x32 accumulator layout a lane then owns ONE
// query column and 16 keys per block, so the online-softmax row max / row sum
// are in-lane reductions plus a single exchange between lane l and l^32, and
// the rescale factor is a per-lane scalar.  The same accumulator registers,
// rounded to bf16, are directly the "B" operand (P^T, 16 keys per step) of
// O^T = V^T . P^T; the matching V^T "A" fragments are fetched from the
// row-major V tile with the LDS transpose read (ds_read_b64_tr_b16), choosing
// key rows in the order the accumulator layout dictates.
//
// Q, K, V, O are each up to two sequence segments in different buffers, so the
// joint [image, text] / [text, image] sequences and the "fresh text + stale
// image buffer" K/V of a PipeFusion patch need no concatenation copy.
#pragma once
#include <atomic>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "hdit_common.h"

namespace hdit_attn {

struct Seg2 {
  const __bf16* p0;
  const __bf16* p1;
  int64_t sb0, ss0, sh0, sb1, ss1, sh1;
  int len0, len1;
};

__device__ __forceinline__ const __bf16* row_ptr(const Seg2& s, int b, int h, int r) {
  // r must be < len0 + len1.  Every field is read and the values are selected: with a branch the compiler may
  // merge the two sides into one load through a selected address, which forces the kernel's parameter block
  // out of the scalar registers into private memory.
  const bool a = r < s.len0;
  const __bf16* p = a ? s.p0 : s.p1;
  const int64_t sb = a ? s.sb0 : s.sb1, ss = a ? s.ss0 : s.ss1, sh = a ? s.sh0 : s.sh1;
  return p + b * sb + (int64_t)(a ? r : r - s.len0) * ss + h * sh;
}

struct AttnParams {
  Seg2 q, k, v, o;
  int heads, sq, skv;
  float scale_log2;
};

constexpr int BKV = 64;  // keys per tile

// From how many key tiles on the pipelined kernels serve a problem; their loop needs three.  At d = 64 they begin later
// than the tracked one and are ahead where the loop is long enough.  Tracked / pipelined, 128 rows per workgroup, us:
//   48 heads   256 x 256 7.0 / 7.4, 2048 x 256 14.0 / 16.2, 384 x 384 8.6 / 8.5, 1024 x 384 12.1 / 12.1, 448 x 448 9.3 / 9.0
//   192 heads  320 x 320 13.3 / 15.8, 384 x 384 16.2 / 18.7, 1024 x 384 30.8 / 32.6, 448 x 448 18.6 / 19.5
// At d = 128 they are ahead at once: 24 heads, 192 x 192 14.5 / 10.5.
constexpr int pipe_min_tiles(int head_dim) { return head_dim == 64 ? 7 : 3; }

// Launch of `count` problems of one head dim, on argument blocks the entry point has validated and converted, as one grid:
// the tracked and the pipelined kernels, with 128 (four waves) and with 256 query rows per workgroup (eight).  A (batch,
// head) is q_tiles workgroups, the first q_full of them with all their rows; nblocks is their number for the whole problem.
int launch_tracked4_d64(const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count, hipStream_t stream);
int launch_tracked8_d128(const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count, hipStream_t stream);
int launch_pipe4_d64(const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count, hipStream_t stream);
int launch_pipe8_d64(const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count, hipStream_t stream);
int launch_pipe8_d128(const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count, hipStream_t stream);

}  // namespace hdit_attn

namespace {

using hdit_attn::AttnParams;
using hdit_attn::Seg2;

using hdit_attn::BKV;
constexpr int QB = 1;        // 32-row query blocks per wave of the tracked kernel
constexpr int WQ = 32 * QB;  // query rows per wave
#ifndef HDIT_ATTN_WAVES
#define HDIT_ATTN_WAVES 4  // waves per workgroup (attention_bf16_pipe8.hip: 8)
#endif
constexpr int NWAVE = HDIT_ATTN_WAVES;
constexpr int NTHR = 64 * NWAVE;
constexpr int BQ = WQ * NWAVE;

template <int HD>
struct Lds {
  // K and V tiles come straight from global memory (global_load_lds_dwordx4: no staging registers, no
  // ds_write), which lands a wave's 64 x 16 bytes contiguously -- eight (d = 64) or four (d = 128) unpadded
  // rows.  The spread over the 64-bank (256-byte) LDS window therefore comes from XOR swizzles applied on the
  // source side.  A ds_read_b128 pass covers 16 consecutive K rows, which must land on 16 distinct 16-byte
  // slots; a transpose-read pass covers 4 consecutive V rows x 64 bytes, which must land on 4 distinct 64-byte
  // slots.  d = 64 (rows of 128 bytes): slot p of K row r holds chunk p ^ ((r>>1)&7), slot p of V row r holds
  // chunk p ^ 4*((r>>1)&1).  d = 128 (rows of 256 bytes, a whole bank window): K chunk p ^ (r&15), V chunk
  // p ^ 4*(r&3).
  static constexpr int K_ROW = HD * 2;
  static constexpr int V_ROW = HD * 2;
  static constexpr int K_BYTES = BKV * K_ROW;
  static constexpr int V_BYTES = BKV * V_ROW;
  static constexpr int STAGE = K_BYTES + V_BYTES;
  // d = 128: the Q fragments (32 registers) live in LDS instead, one private region per wave, rows strided like
  // the K rows, and are read per k-step next to the K fragments: the registers they would occupy are what the
  // loop otherwise spills (and reloads from scratch on every tile, with few waves per SIMD to hide that).
  static constexpr bool Q_IN_LDS = HD == 128;
  static constexpr int Q_ROW = HD * 2 + 16;
  static constexpr int Q_OFF = 2 * STAGE;
  static constexpr int Q_WAVE_BYTES = WQ * Q_ROW;
  static constexpr int TOTAL = 2 * STAGE + (Q_IN_LDS ? NWAVE * Q_WAVE_BYTES : 0);
  static_assert(TOTAL <= 160 * 1024, "attention tiles do not fit the LDS");
};

// One wave-wide direct-to-LDS copy: lane l's 16 bytes land at LDS byte address lds_addr + 16*l.  Inline
// assembly, so the compiler's wait-count bookkeeping does not see it; the tile loop waits for it explicitly.
// AGENT: issued at agent scope (sc1), which the CU's L1 never serves.  The pipelined kernel waits for "all but the
// newest n" requests and relies on completion in issue order, and a request that hits in L1 -- the rows of a clamped
// tile, a tile requested again past the end, a short sequence the previous workgroup on the CU has just read --
// completes ahead of older misses; from L2, hits and misses complete in issue order.  The kernels that wait for
// everything (vmcnt(0)) do not care about the order and keep the L1 (2 % faster where two workgroups of a CU read
// the same keys).
template <bool AGENT>
__device__ __forceinline__ void lds_dma16(const unsigned char* base_uniform, unsigned voff, unsigned lds_addr_uniform) {
  // the base is wave-uniform by construction; say so, or a base the compiler keeps in vector registers ends up in
  // the scalar-address operand
  const uint64_t bu = (uint64_t)base_uniform;
  const uint64_t base = ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(bu >> 32)) << 32) |
                        (unsigned)__builtin_amdgcn_readfirstlane((int)bu);
  if constexpr (AGENT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 sc1"
                 :
                 : "s"(lds_addr_uniform), "v"(voff), "s"(base)
                 : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_addr_uniform), "v"(voff), "s"(base)
                 : "m0", "memory");
}
template <bool AGENT>
__device__ __forceinline__ void lds_dma16_ptr(const unsigned char* ptr_per_lane, unsigned lds_addr_uniform) {
  if constexpr (AGENT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off sc1"
                 :
                 : "s"(lds_addr_uniform), "v"(ptr_per_lane)
                 : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds_addr_uniform), "v"(ptr_per_lane)
                 : "m0", "memory");
}
__device__ __forceinline__ unsigned lds_address(const unsigned char* p) {
  return (unsigned)(uintptr_t)((const __attribute__((address_space(3))) unsigned char*)p);
}

// s_waitcnt immediate: all but the newest n vector-memory operations have completed, and every LDS operation
constexpr int waitcnt_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0070; }

// The running row maximum is only raised when some row's maximum grew by more than this many powers of
// two; until then exp2(s - m) may reach 2^8, harmless for the bf16 P operand and the fp32 row sums, and the
// accumulator rescale (the most expensive VALU block after the exponentials) is skipped for most tiles.
constexpr float RESCALE_THRESHOLD = 8.0f;

// Where a workgroup works.  A (batch, head) has q_full tiles of BQ query rows and q_tiles - q_full of HALF rows behind them:
// in workgroups of eight waves a half tile leaves half of the waves without rows, so that what is over after the full
// rounds of a launch is spread over twice as many CUs; elsewhere it is the partly filled last tile.
// Workgroups go to the 8 XCDs round-robin by id, and each XCD has its own L2: all query tiles of one
// (batch, head) run on one XCD, so that its K and V are fetched into one L2 instead of eight.  Within that,
// the half tiles come after all full ones: workgroups are placed in id order, one per CU first, so when a launch has a few
// more workgroups than CUs it is the light ones that share a CU with a full one.
constexpr int HALF = NWAVE == 8 ? BQ / 2 : BQ;
struct Place {
  int b, h, q0, rows;
};
__device__ __forceinline__ Place place(const AttnParams& P, int q_tiles, int q_full, int block_id, int nblocks) {
  // The arguments that are needed next are requested together with those of the divisions, not behind them: 0.2 us.
  asm volatile("" : "+s"(q_tiles) : "s"(P.q.p0), "s"(P.q.len0), "s"(P.k.p0), "s"(P.k.len0), "s"(P.v.p0), "s"(P.skv));
  const int nbh = nblocks / q_tiles;
  const bool by_xcd = nbh % 8 == 0;
  const int slot = by_xcd ? (block_id >> 3) : block_id;
  const int full = (by_xcd ? nbh / 8 : nbh) * q_full;
  const bool half = slot >= full;
  const int of_bh = half ? q_tiles - q_full : q_full, s = half ? slot - full : slot;
  const int qt = s % of_bh, bhl = s / of_bh;
  const int bh = by_xcd ? bhl * 8 + (block_id & 7) : bhl;
  Place at;
  at.b = bh / P.heads, at.h = bh % P.heads;
  at.q0 = half ? q_full * BQ + qt * HALF : qt * BQ;
  at.rows = half ? HALF : BQ;
  return at;
}

// The whole kernel for one workgroup: the online softmax with a running reference that follows the column
// maxima.  Also the second pass of the pipelined kernels, for the rows whose fixed reference did not hold: bit l of
// `rows` stands for the wave's row l, the others have been written.
template <int HD>
__device__ __forceinline__ void attn_tracked_body(const AttnParams& P, int q_tiles, int q_full, unsigned char* lds,
                                                  int block_id, int nblocks, unsigned rows = ~0u) {
  using L = Lds<HD>;
  constexpr int KS = HD / 16;       // k-steps of the S^T MFMA (over head dim)
  constexpr int DB = HD / 32;       // 32-wide d blocks of O^T
  constexpr int CPR = HD / 8;       // 16-byte chunks per row
  constexpr int NCH = BKV * CPR / NTHR;  // chunks per thread per tile (K and V each)
  // FOLD: the softmax scale is multiplied into Q once and the running reference m is subtracted inside the
  // score MFMA (its first k-step accumulates onto -m), so the accumulators feed exp2 directly: one FMA less
  // per score in a loop that is bound by the VALU.  Costs 32 registers; the d = 128 kernel has none to spare.
  constexpr bool FOLD = HD == 64;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, lh = lane >> 5;
  const Place at = place(P, q_tiles, q_full, block_id, nblocks);
  const int b = at.b, h = at.h, q0 = at.q0 + wave * WQ;
  // a wave past the last query row, or past the rows of a half tile, or with no row to do over, still stages K/V tiles and
  // meets the barriers, but does no arithmetic
  const bool active = __builtin_amdgcn_readfirstlane(q0 < P.sq && wave * WQ < at.rows && rows != 0);

  // ---- Q fragments: lane holds q row (qb*32 + l32), d = 16*ks + 8*lh .. +7
  bf16x8 qf[QB][L::Q_IN_LDS ? 1 : KS];
  unsigned char* qlds = lds + L::Q_OFF + wave * L::Q_WAVE_BYTES;
  if constexpr (L::Q_IN_LDS) {
    // the wave's query rows, 16 lanes per row (coalesced 256-byte rows), into its private LDS region;
    // only this wave reads them back, so its own wait for the writes is all the synchronisation needed
    constexpr int RPI = 64 / CPR;  // rows per wave-wide load
#pragma unroll
    for (int i = 0; i < WQ / RPI; i++) {
      const int row = i * RPI + lane / CPR, cc = lane % CPR;
      const int r = min(q0 + row, P.sq - 1);
      const i32x4 raw = *(const i32x4*)(row_ptr(P.q, b, h, r) + cc * 8);
      *(i32x4*)(qlds + row * L::Q_ROW + cc * 16) = raw;
    }
  } else
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    int r = min(q0 + qb * 32 + l32, P.sq - 1);
    const __bf16* rp = row_ptr(P.q, b, h, r);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const i32x4 raw = *(const i32x4*)(rp + ks * 16 + lh * 8);
      if constexpr (FOLD) {
        float f[8];
        hdit::unpack8(raw, f);
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] *= P.scale_log2;
        qf[qb][ks] = __builtin_bit_cast(bf16x8, hdit::pack8(f));
      } else {
        qf[qb][ks] = __builtin_bit_cast(bf16x8, raw);
      }
    }
  }

  // ---- K/V tile staging: global -> registers -> LDS.  A tile that lies inside one segment is addressed as
  // (wave-uniform base) + (loop-invariant per-thread offset); the tile that straddles the segment boundary
  // and the last, clamped tile take the per-row path.
  unsigned koff[2][NCH], voff[2][NCH];
  // direct-to-LDS (d = 64): request i of a wave covers rows 8*(wave + NWAVE*i) .. +7, lane -> (row, slot lane%8);
  // the chunk fetched for a slot is the slot index XORed with the row's swizzle (the same for every i)
  constexpr int RPI = 64 / CPR;  // rows per request
  const int dma_row = wave * RPI + lane / CPR;
  const int dma_kc = (lane % CPR) ^ (HD == 64 ? ((dma_row >> 1) & 7) : (dma_row & 15));
  const int dma_vc = (lane % CPR) ^ (4 * (HD == 64 ? ((dma_row >> 1) & 1) : (dma_row & 3)));
  const unsigned lds_base_addr = __builtin_amdgcn_readfirstlane(lds_address(lds));
#pragma unroll
  for (int i = 0; i < NCH; i++) {
    const int row = dma_row + NWAVE * RPI * i;
    koff[0][i] = (unsigned)((row * P.k.ss0 + dma_kc * 8) * 2);
    koff[1][i] = (unsigned)((row * P.k.ss1 + dma_kc * 8) * 2);
    voff[0][i] = (unsigned)((row * P.v.ss0 + dma_vc * 8) * 2);
    voff[1][i] = (unsigned)((row * P.v.ss1 + dma_vc * 8) * 2);
  }
  const unsigned char* kb0 = (const unsigned char*)(P.k.p0 + b * P.k.sb0 + h * P.k.sh0);
  const unsigned char* kb1 = (const unsigned char*)(P.k.p1 + b * P.k.sb1 + h * P.k.sh1);
  const unsigned char* vb0 = (const unsigned char*)(P.v.p0 + b * P.v.sb0 + h * P.v.sh0);
  const unsigned char* vb1 = (const unsigned char*)(P.v.p1 + b * P.v.sb1 + h * P.v.sh1);
  const int len0 = P.k.len0;
  // tile t straight into LDS stage `stage`
  auto dma_tile = [&](int t, int stage) {
    const int r0 = t * BKV;
    const unsigned kdst = lds_base_addr + stage * L::STAGE + __builtin_amdgcn_readfirstlane(wave) * 1024;
    const unsigned vdst = kdst + L::K_BYTES;
    if (r0 + BKV <= len0) {
      const unsigned char* kb = kb0 + (int64_t)r0 * P.k.ss0 * 2;
      const unsigned char* vb = vb0 + (int64_t)r0 * P.v.ss0 * 2;
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        lds_dma16<false>(kb, koff[0][i], kdst + i * (NWAVE * 1024));
        lds_dma16<false>(vb, voff[0][i], vdst + i * (NWAVE * 1024));
      }
    } else if (r0 >= len0 && r0 + BKV <= P.skv) {
      const unsigned char* kb = kb1 + (int64_t)(r0 - len0) * P.k.ss1 * 2;
      const unsigned char* vb = vb1 + (int64_t)(r0 - len0) * P.v.ss1 * 2;
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        lds_dma16<false>(kb, koff[1][i], kdst + i * (NWAVE * 1024));
        lds_dma16<false>(vb, voff[1][i], vdst + i * (NWAVE * 1024));
      }
    } else {
#pragma unroll
      for (int i = 0; i < NCH; i++) {
        const int r = min(r0 + dma_row + NWAVE * RPI * i, P.skv - 1);
        lds_dma16_ptr<false>((const unsigned char*)(row_ptr(P.k, b, h, r) + dma_kc * 8), kdst + i * (NWAVE * 1024));
        lds_dma16_ptr<false>((const unsigned char*)(row_ptr(P.v, b, h, r) + dma_vc * 8), vdst + i * (NWAVE * 1024));
      }
    }
  };
  f32x16 oacc[DB][QB];
#pragma unroll
  for (int i = 0; i < DB; i++)
#pragma unroll
    for (int j = 0; j < QB; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) oacc[i][j][v] = 0.f;
  // running reference m of the online softmax (log2 units) and running sum per query column.  With FOLD the
  // accumulators of a score block start from negm = -m (the same value in all 16 entries: a lane owns one
  // query column per qb) and m starts at 0 until the first tile sets it to that tile's column maxima.
  float m_run[QB], l_run[QB];
  f32x16 negm[QB];
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    m_run[qb] = FOLD ? 0.f : -INFINITY, l_run[qb] = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v++) negm[qb][v] = 0.f;
  }
  bool first = true;

  // lane-constant part of the V^T transpose-read address:
  // 16-lane group G = lane/16, x = lane%16: key row 4*(G/2) + x/4, column 16*(G%2) + 4*(x%4)
  const int vt_row = 4 * (lane >> 5) + ((lane & 15) >> 2);
  const int vt_off = vt_row * L::V_ROW + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  const int vt_swz = HD == 64 ? ((vt_row >> 1) & 1) : (vt_row & 3);  // XORed into the 64-byte piece index
  const int k_off = l32 * L::K_ROW;
  const int k_swz = HD == 64 ? ((l32 >> 1) & 7) : (l32 & 15);  // direct-to-LDS layout: chunk c of K row r sits in slot c ^ this
  const bf16x2 ones2 = {(__bf16)1.0f, (__bf16)1.0f};

  // one K/V tile: scores, online softmax, PV.  MASK: keys >= valid do not exist (last tile only).
  auto tile_compute = [&](const unsigned char* sk, auto mask_tag, int valid) {
    constexpr bool MASK = decltype(mask_tag)::value;
    const unsigned char* sv = sk + L::K_BYTES;
    // ---- S^T[kb][qb] = K_tile . Q^T (first k-step starts from a zero accumulator operand)
    f32x16 sacc[2][QB];
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (L::Q_IN_LDS) {
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        bf16x8 qk[QB], kf[2];
#pragma unroll
        for (int qb = 0; qb < QB; qb++) qk[qb] = *(const bf16x8*)(qlds + (qb * 32 + l32) * L::Q_ROW + lh * 16 + ks * 32);
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
          kf[kb] = *(const bf16x8*)(sk + k_off + kb * 32 * L::K_ROW + (((ks * 2 + lh) ^ k_swz) << 4));
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
          for (int qb = 0; qb < QB; qb++)
            sacc[kb][qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kb], qk[qb], ks == 0 ? zero16 : sacc[kb][qb], 0, 0, 0);
      }
    }
    auto mask_scores = [&]() {
      if (MASK) {
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
          for (int v = 0; v < 16; v++) {
            int key = kb * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
            if (key >= valid) {
#pragma unroll
              for (int qb = 0; qb < QB; qb++) sacc[kb][qb][v] = -INFINITY;
            }
          }
      }
    };
    auto scores_from_registers = [&]() {
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          bf16x8 kf = *(const bf16x8*)(sk + k_off + kb * 32 * L::K_ROW +
                                       (((ks * 2 + lh) ^ k_swz) << 4));
#pragma unroll
          for (int qb = 0; qb < QB; qb++)
            sacc[kb][qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[qb][L::Q_IN_LDS ? 0 : ks], ks == 0 ? (FOLD ? negm[qb] : zero16) : sacc[kb][qb], 0, 0, 0);
        }
      }
      mask_scores();
    };
    if constexpr (L::Q_IN_LDS) mask_scores();
    else scores_from_registers();
    if constexpr (FOLD) {
      // Both key blocks start from the reference vectors.  Reading them once more here keeps them alive past the
      // second block's first MFMA, which the compiler otherwise ties to a copy of them (16 v_mov_b64 per tile)
      // instead of naming them as its addend the way the first block's does.
      asm volatile("" : : "v"(negm[0]), "v"(negm[QB - 1]));
    }

    // ---- online softmax in the log2 domain.  A lane owns one query column per qb and 32 of its 64 keys;
    // the other 32 live in lane^32.
    bf16x8 pf[QB][4];  // [qb][u], u = 2*kb + half: the 16 keys of PV k-step u
    if constexpr (FOLD) {
      float mrel[QB];  // column maxima relative to the running reference
#pragma unroll
      for (int qb = 0; qb < QB; qb++) {
        float mx = fmaxf(sacc[0][qb][0], sacc[1][qb][0]);
#pragma unroll
        for (int v = 1; v < 16; v++) mx = fmaxf(fmaxf(mx, sacc[0][qb][v]), sacc[1][qb][v]);  // one v_max3 per step
        auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(mx), __float_as_int(mx), false, false);
        mrel[qb] = fmaxf(__int_as_float(sw[0]), __int_as_float(sw[1]));
      }
      // Move the reference (and rescale) where a column outgrew the threshold; the branch is wave-uniform, the decision
      // every column's own (the others move by 0, which changes no bit): a query row's result does not depend on the
      // rows it shares a wave with, so workgroups of 128 and of 256 rows give the same bits.
      const bool grow = first || mrel[0] > RESCALE_THRESHOLD || mrel[QB - 1] > RESCALE_THRESHOLD;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
        for (int qb = 0; qb < QB; qb++) {
          const float d = first || mrel[qb] > RESCALE_THRESHOLD ? mrel[qb] : 0.f;
          m_run[qb] += d;
          if (!first) {
            const float alpha = __builtin_amdgcn_exp2f(-d);
            l_run[qb] *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
              for (int v = 0; v < 16; v++) oacc[db][qb][v] *= alpha;
          }
#pragma unroll
          for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int v = 0; v < 16; v++) sacc[kb][qb][v] -= d;
#pragma unroll
          for (int v = 0; v < 16; v++) negm[qb][v] = -m_run[qb];
        }
        first = false;
      }
    } else {
      float mcand[QB];
#pragma unroll
      for (int qb = 0; qb < QB; qb++) {
        float mx = fmaxf(sacc[0][qb][0], sacc[1][qb][0]);
#pragma unroll
        for (int v = 1; v < 16; v++) mx = fmaxf(fmaxf(mx, sacc[0][qb][v]), sacc[1][qb][v]);  // one v_max3 per step
        auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(mx), __float_as_int(mx), false, false);
        mx = fmaxf(__int_as_float(sw[0]), __int_as_float(sw[1]));
        mcand[qb] = fmaxf(m_run[qb], mx * P.scale_log2);
      }
      // raise the running maxima (and rescale) only if some row outgrew the threshold: wave-uniform branch, every column's
      // own decision, as above (the others are multiplied by 1)
      const bool grow = (mcand[0] - m_run[0] > RESCALE_THRESHOLD) || (mcand[QB - 1] - m_run[QB - 1] > RESCALE_THRESHOLD);
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
        for (int qb = 0; qb < QB; qb++) {
          const bool move = mcand[qb] - m_run[qb] > RESCALE_THRESHOLD;  // always at the first tile, from -inf
          const float alpha = move ? __builtin_amdgcn_exp2f(m_run[qb] - mcand[qb]) : 1.0f;
          m_run[qb] = move ? mcand[qb] : m_run[qb];
          l_run[qb] *= alpha;
#pragma unroll
          for (int db = 0; db < DB; db++)
#pragma unroll
            for (int v = 0; v < 16; v++) oacc[db][qb][v] *= alpha;
        }
      }
    }
#pragma unroll
    for (int qb = 0; qb < QB; qb++) {
      const float m = m_run[qb];
      float rs = l_run[qb];
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
          i32x4 pk;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float s0 = sacc[kb][qb][hh * 8 + 2 * e], s1 = sacc[kb][qb][hh * 8 + 2 * e + 1];
            const float p0 = __builtin_amdgcn_exp2f(FOLD ? s0 : __builtin_fmaf(s0, P.scale_log2, -m));
            const float p1 = __builtin_amdgcn_exp2f(FOLD ? s1 : __builtin_fmaf(s1, P.scale_log2, -m));
            const uint32_t pp = hdit::pack2(p0, p1);
            pk[e] = (int)pp;
            // row sum of exactly the bf16 values that enter the PV product
            rs = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pp), ones2, rs, false);
          }
          pf[qb][kb * 2 + hh] = __builtin_bit_cast(bf16x8, pk);
        }
      }
      l_run[qb] = rs;
    }

    // ---- O^T[db][qb] += V^T . P^T
#pragma unroll
    for (int u = 0; u < 4; u++) {
#pragma unroll
      for (int db = 0; db < DB; db++) {
        const unsigned char* va = sv + vt_off + (u * 16) * L::V_ROW + ((db ^ vt_swz) << 6);
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(va));
        s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (s16x4 __attribute__((address_space(3)))*)(va + 8 * L::V_ROW));
        typedef __attribute__((ext_vector_type(8))) short s16x8;
        s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        bf16x8 vf = __builtin_bit_cast(bf16x8, both);
#pragma unroll
        for (int qb = 0; qb < QB; qb++)
          oacc[db][qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[qb][u], oacc[db][qb], 0, 0, 0);
      }
    }
  };

  const int NT = (P.skv + BKV - 1) / BKV;
  // Tile t+1 is fetched while tile t is worked on: its requests are issued behind the barrier that published
  // tile t, into the stage tile t-1 vacated; every wave waits for its own requests before the next barrier.
  dma_tile(0, 0);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
  if (NT > 1) dma_tile(1, 1);
  auto next_tile = [&](int t) {  // end of iteration t: publish tile t+1, start fetching tile t+2
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's share of tile t+1 has landed
    __syncthreads();
    if (t + 2 < NT) dma_tile(t + 2, t & 1);
  };

  if (!active) {
    // no query rows: stage this wave's share of every K/V tile and meet the same barriers, nothing else
    for (int t = 0; t < NT - 1; t++) next_tile(t);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    return;
  }
  for (int t = 0; t < NT - 1; t++) {
    tile_compute(lds + (t & 1) * L::STAGE, std::false_type{}, BKV);
    next_tile(t);
  }
  {
    const int t = NT - 1;
    const int valid = P.skv - t * BKV;
    if (valid < BKV) tile_compute(lds + (t & 1) * L::STAGE, std::true_type{}, valid);
    else tile_compute(lds + (t & 1) * L::STAGE, std::false_type{}, BKV);
  }

  // ---- normalise and write O[q][d]: lane owns q = qb*32 + l32, d = 32*db + 8*(v/4) + 4*lh + v%4
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(l_run[qb]), __float_as_int(l_run[qb]), false, false);
    const float inv = 1.0f / (__int_as_float(sw[0]) + __int_as_float(sw[1]));
    const int r = q0 + qb * 32 + l32;
    if (r >= P.sq || !((rows >> l32) & 1)) continue;
    __bf16* op = (__bf16*)row_ptr(P.o, b, h, r);
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        i32x2 out;
        out[0] = (int)hdit::pack2(oacc[db][qb][g * 4 + 0] * inv, oacc[db][qb][g * 4 + 1] * inv);
        out[1] = (int)hdit::pack2(oacc[db][qb][g * 4 + 2] * inv, oacc[db][qb][g * 4 + 3] * inv);
        *(i32x2*)(op + db * 32 + g * 8 + lh * 4) = out;
      }
  }
}

template <int HD>
__global__ void __launch_bounds__(NTHR, HD == 64 ? 3 : 2) attn_fwd_kernel(const AttnParams P, int q_tiles, int q_full) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  attn_tracked_body<HD>(P, q_tiles, q_full, lds, (int)blockIdx.x, (int)gridDim.x);
}

// Several independent attention problems of one head dim in one grid (the blocks of neighbouring pipeline patches
// that run side by side): problem i owns the workgroups [start[i], start[i + 1]), each range a multiple of 8 long so
// that a workgroup's position modulo 8 -- the XCD it lands on -- is the same inside its problem as in the launch.
constexpr int ATTN_MAX_MULTI = HDIT_ATTN_MAX_MULTI;
struct AttnMulti {
  AttnParams p[ATTN_MAX_MULTI];
  int q_tiles[ATTN_MAX_MULTI], q_full[ATTN_MAX_MULTI];
  int nblocks[ATTN_MAX_MULTI];   // workgroups that have work (the range may be padded beyond them)
  int start[ATTN_MAX_MULTI + 1];
  int count;
};

template <int HD>
__global__ void __launch_bounds__(NTHR, HD == 64 ? 3 : 2) attn_fwd_multi_kernel(const AttnMulti M) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int i = 0;
#pragma unroll 1
  while (i + 1 < M.count && (int)blockIdx.x >= M.start[i + 1]) i++;
  const int local = (int)blockIdx.x - M.start[i];
  if (local >= M.nblocks[i]) return;
  attn_tracked_body<HD>(M.p[i], M.q_tiles[i], M.q_full[i], lds, local, M.nblocks[i]);
}

// ---------------------------------------------------------------------------------------------------------
// The pipelined kernels.
//
// What bounds a tile is the sum of what the vector ALU has to issue (the exponentials, packs, and about 8 cycles for
// every MFMA) and, beside it, the matrix pipe -- and where the whole chip works, the board's power.  An MFMA runs beside
// vector instructions of its own wave and of the SIMD's other waves (measured: 32 MFMAs of 32 cycles in one wave, 256
// additions, exponentials, maxima or packs in the other: the longer of the two plus 8 cycles per MFMA).  The exceptions
// are the dot products (v_dot2*): they wait for the matrix pipe, 256 of them beside those MFMAs take the sum of both.  The
// row sums of the kernel above are dot products; here they are 4x4x4 MFMAs, which add four of a lane's own values.
//
// So a wave's instruction stream is laid out so that both always have work: between two barriers it is one basic block in
// which every MFMA is followed by its share of everything else, pinned there (`sched_barrier`):
//
//   slots [0, F)        P.V of keys 32-63 of tile t-1, scores of keys 32-63 of tile t     | softmax of keys  0-31 of tile t
//   slots [F, 2F)       P.V of keys  0-31 of tile t,   scores of keys  0-31 of tile t+1   | softmax of keys 32-63 of tile t
//
// F = HD / 4.  A wave owns 32 query rows in 256 registers, so that a SIMD has two waves: one alone issues an instruction
// every 4.5 cycles at best (165 of them per tile at d = 64).  The MFMAs are 16x16x32: less energy per flop (see
// gemm_bf16.hip).  A lane owns one query column of each of two 16-row blocks and 4 of every 16 keys.
// Operands: fragment f (two MFMAs) is read FRAG_LEAD fragments ahead, across the barrier too; the tile requests are
// dealt over the slots and have a pointer per lane that moves on from tile to tile.
//
// Measured on one box, former kernels (64 rows per wave: tracked as above, or pipelined with one wave per SIMD, dot products,
// 32x32x16 MFMAs, requests in one piece; the better of them) -> this one, us.  d = 64, 24 heads: 2 x 666 rows 17.7 -> 15.2, 1357
// 27.1 -> 23.0, 4470 131 -> 122, 1024 of 4429 rows 53.0 -> 40.7, two of them 74.7 -> 58.5, 2 x 4429 258 -> 231; 17776 rows with 48
// heads 3544 -> 3309 (1.17 PFLOP/s).  d = 128, 24 heads: 333 rows 21.1 -> 12.3, 1536 50.2 -> 41.2, 4608 261 -> 217, 9728 1078 -> 911
// (1.28 PFLOP/s), 16896 3316 -> 2660 (1.32).  Of the steps, at 2 x 4429 rows: this layout 244, the loop unrolled over the ring 241 (a
// fragment's address needs no addition), one exponential per MFMA in place of two in turn with none 235, the query rows
// requested in front of the tiles 1 us.  With 32x32x16 MFMAs a SIMD's tile takes fewer cycles (each MFMA holds the issue
// port) but the clock falls by more: 2 x 4429 rows 244 us at 1.92 GHz against 244 at 2.15.
//
// For the block to have no branch the reference of the online softmax is fixed after the first tile (its column
// maxima plus a margin: p = 2^(s - m) may then grow to PIPE_LIMIT and shrink to nothing without any loss
// of relative precision in fp32 / bf16): no maxima, no rescale in the loop.  (The key that holds the maximum has a p that
// bf16 represents exactly.  With the maxima of 32 keys instead of the tile's 64, as the kernel above has them, results with
// peaked logits were up to 1.2 % further from 64 bits.)  Rows whose sum ends at or above
// the limit (infinity and NaN included) are left to the body of the kernel above, which the workgroup then runs for them,
// in those of its waves that have such a row: logits that rise by 44 (in base e) over the largest of the first 64 keys.
// What that costs, us, with no such row / one in 1000 / in 256 / in 128 / in 32 / for comparison the kernel above alone: d = 64
// 2 x 4429 rows of 24 heads 235 / 328 / 423 / 424 / 494 / 258, 17776 rows of 48 heads 3390 / 4988 / 5562 / 6416 / 7429 / 3782; d = 128
// 4608 rows of 24 heads 225 / 369 / 375 / 423 / 472 / 262.
// (A limit near the end of fp32 would leave rows that rise by up to 104 in the first pass, but their error against 64 bits
// grows: 0.1 - 2.5 % at d = 64, and at d = 128, where this kernel rounds scaled queries to bf16 and the tracked one does not,
// 2 - 70 %.)
// So a row's result depends on that row and the keys alone, whatever rows it shares a wave or workgroup with.
template <int HD>
struct PipeLds {
  // tiles between two barriers: eight waves wait for each other half as often where twice the slots fit (17776 keys,
  // 48 heads, d = 64: 3800 us with one, 3658 with two)
  static constexpr int SYNC = HD == 64 && NWAVE == 8 ? 2 : 1;
  static constexpr int RING = SYNC == 2 ? 8 : 4;  // LDS slots per operand
  // Iteration t requests K tile t + LEAD and V tile t + LEAD - 1.  It reads K tiles t and t + 1 and V tiles t - 1 and t: a
  // slot is requested again at the earliest when every wave has passed a barrier behind its last use.
  static constexpr int LEAD = SYNC == 2 ? 5 : 3;
  static constexpr int MASK = RING - 1;
  static constexpr int ROW = HD * 2;      // bytes of a K or V row
  static constexpr int TILE = BKV * ROW;  // bytes of one K or V tile
  static constexpr int V_OFF = RING * TILE;
  static constexpr int FLAG_OFF = 2 * RING * TILE;
  // Eight waves: where the query rows of wave w (half a tile) are while the loop has not begun.  In the slots of K tiles
  // LEAD .. and of V tile LEAD - 1, which iteration 0 and later ones request; where these are not enough (d = 128), behind
  // the rings, over the flag.
  static constexpr int K_FREE = RING - LEAD;
  __device__ static constexpr int q_slot(int w) {
    const int pair = w / 2;
    return (pair < K_FREE ? (LEAD + pair) * TILE : pair == K_FREE ? V_OFF + (LEAD - 1) * TILE : FLAG_OFF + (pair - K_FREE - 1) * TILE) +
           (w % 2) * (TILE / 2);
  }
  static constexpr int BEHIND = NWAVE == 8 ? (NWAVE / 2 - K_FREE - 1) * TILE : 0;
  static constexpr int END = FLAG_OFF + (BEHIND > 16 ? BEHIND : 16);
  // the launch also covers the tracked kernel's layout, which a workgroup falls back to
  static constexpr int TOTAL = END > Lds<HD>::TOTAL ? END : Lds<HD>::TOTAL;
  static_assert(TOTAL <= 160 * 1024, "rings do not fit the LDS");
  static_assert(NWAVE != 4 || HD != 64 || TOTAL <= 80 * 1024, "two workgroups per CU");
};
constexpr float PIPE_MARGIN = 24.0f;  // an integer: the exact p's stay exact
constexpr float PIPE_LIMIT = 0x1p40f;
constexpr int FRAG_LEAD = 3;

template <int... I, class F>
__device__ __forceinline__ void static_for_seq(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(std::make_integer_sequence<int, N>{}, f);
}

constexpr int waitcnt_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0f70; }

// true: the fixed reference did not hold for some row of the workgroup; those of this wave are set in `rows`
template <int HD>
__device__ __forceinline__ bool attn_pipe_body(const AttnParams& P, int q_tiles, int q_full, unsigned char* lds, int block_id,
                                               int nblocks, unsigned& rows) {
  using PL = PipeLds<HD>;
  constexpr int KS = HD / 32, DB = HD / 16, CPR = HD / 8, NCH = BKV * CPR / NTHR, RPI = 64 / CPR, ROW = PL::ROW;
  constexpr int TILE = PL::TILE, V_OFF = PL::V_OFF, LEAD = PL::LEAD, MASK = PL::MASK, SYNC = PL::SYNC;
  constexpr int F = 2 * DB + 4 * KS;  // fragments per iteration, two MFMAs each
  constexpr int PER = F / 8;          // MFMAs per pair of scores (16 pairs)
  static_assert(WQ == 32, "written for 32 query rows per wave");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, lg = lane >> 4;
  const Place at = place(P, q_tiles, q_full, block_id, nblocks);
  const int b = at.b, h = at.h, q0 = at.q0 + wave * 32;
  const bool active = __builtin_amdgcn_readfirstlane(q0 < P.sq && wave * 32 < at.rows);
  const int NT = (P.skv + BKV - 1) / BKV;  // >= pipe_min_tiles (host)
  rows = 0;

  typedef __attribute__((address_space(3))) int lds_int;
  lds_int* const flag = (lds_int*)(uintptr_t)(lds_address(lds) + PL::FLAG_OFF);

  // ---- K / V tile requests, straight into LDS.  Slot p of K row r holds chunk p ^ ((r>>1)&7) (d = 64) or p ^ (r&15), as
  // in the kernel above: a fragment read covers 16 rows.  A transpose read takes 32 bytes of each of 16 V rows: slot p of
  // V row r holds chunk p ^ 2*((r>>1)&3) (d = 64) or p ^ 2*(r&7), which spreads eight rows over the banks.
  const int dma_row = wave * RPI + lane / CPR;
  const int dma_kc = (lane % CPR) ^ (HD == 64 ? ((dma_row >> 1) & 7) : (dma_row & 15));
  const int dma_vc = (lane % CPR) ^ (2 * (HD == 64 ? ((dma_row >> 1) & 3) : (dma_row & 7)));
  const unsigned lds_base_addr = __builtin_amdgcn_readfirstlane(lds_address(lds));
  const int len0 = P.k.len0;
  const int full0 = len0 / BKV;               // tiles [0, full0) lie in segment 0
  const int first1 = (len0 + BKV - 1) / BKV;  // tiles [first1, full_all) lie in segment 1
  const int full_all = P.skv / BKV;
  const uint64_t kb0 = (uint64_t)(P.k.p0 + b * P.k.sb0 + h * P.k.sh0);
  const uint64_t vb0 = (uint64_t)(P.v.p0 + b * P.v.sb0 + h * P.v.sh0);
  // segment 1 bases moved back by the rows of segment 0, so that they too are indexed by the row number
  const uint64_t kb1 = (uint64_t)(P.k.p1 + b * P.k.sb1 + h * P.k.sh1) - (uint64_t)((int64_t)len0 * P.k.ss1 * 2);
  const uint64_t vb1 = (uint64_t)(P.v.p1 + b * P.v.sb1 + h * P.v.sh1) - (uint64_t)((int64_t)len0 * P.v.ss1 * 2);
  const unsigned krow0 = (unsigned)(P.k.ss0 * 2), krow1 = (unsigned)(P.k.ss1 * 2);  // bytes per row
  const unsigned vrow0 = (unsigned)(P.v.ss0 * 2), vrow1 = (unsigned)(P.v.ss1 * 2);
  const unsigned wave_dst = lds_base_addr + __builtin_amdgcn_readfirstlane(wave) * 1024;
  // A pointer per lane and request.  It moves on by one tile (a uniform step that fits 32 bits: host) while the tiles lie
  // inside one segment; where one straddles the boundary, begins a segment or is the clamped last one, the pointers are
  // formed row by row, outside of the block that holds the arithmetic.  Past the end the last tile is requested again
  // (into a slot nobody reads any more): every iteration issues the same number of requests.
  uint64_t kp[NCH], vp[NCH];
  auto k_ptrs = [&](int t) __attribute__((always_inline)) {
    const int r0 = min(t, NT - 1) * BKV;
#pragma unroll
    for (int i = 0; i < NCH; i++) {
      const int r = min(r0 + dma_row + NWAVE * RPI * i, P.skv - 1);
      const bool in0 = r < len0;
      kp[i] = (in0 ? kb0 : kb1) + (uint64_t)(unsigned)r * (in0 ? krow0 : krow1) + dma_kc * 16;
    }
  };
  auto v_ptrs = [&](int t) __attribute__((always_inline)) {
    const int r0 = min(t, NT - 1) * BKV;
#pragma unroll
    for (int i = 0; i < NCH; i++) {
      const int r = min(r0 + dma_row + NWAVE * RPI * i, P.skv - 1);
      const bool in0 = r < len0;
      vp[i] = (in0 ? vb0 : vb1) + (uint64_t)(unsigned)r * (in0 ? vrow0 : vrow1) + dma_vc * 16;
    }
  };
  // request i of the tile the pointers stand at, into the slot at dst (this wave's share of it)
  auto dma_k = [&](int i, unsigned dst) __attribute__((always_inline)) {
    lds_dma16_ptr<true>((const unsigned char*)kp[i], dst + i * (NWAVE * 1024));
  };
  auto dma_v = [&](int i, unsigned dst) __attribute__((always_inline)) {
    lds_dma16_ptr<true>((const unsigned char*)vp[i], dst + i * (NWAVE * 1024));
  };
  auto tile_k = [&](int t) __attribute__((always_inline)) {
    k_ptrs(t);
#pragma unroll
    for (int i = 0; i < NCH; i++) dma_k(i, wave_dst + (unsigned)(t & MASK) * TILE);
  };
  auto tile_v = [&](int t) __attribute__((always_inline)) {
    v_ptrs(t);
#pragma unroll
    for (int i = 0; i < NCH; i++) dma_v(i, wave_dst + V_OFF + (unsigned)(t & MASK) * TILE);
  };
  // The end of SYNC iterations: everything older than the requests of the newest LEAD - 1 - SYNC iterations has landed (a
  // wave's requests complete in order), which the barrier publishes.  Fragment reads may be in flight over it.
  auto stage_end = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * NCH * (LEAD - 1 - SYNC)));
    asm volatile("" : : : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };

  // ---- prologue: a zero V tile in the last slot (the lagged P.V of iteration 0 multiplies it by P = 0), the query rows,
  // tiles K0 | K1 V0 | K2 V1 .. in request order
  {
    const i32x4 z = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < TILE / (16 * NTHR); i++) *(i32x4*)(lds + V_OFF + MASK * TILE + i * (16 * NTHR) + tid * 16) = z;
  }
  // The query rows, requested in front of the tiles.  Eight waves: the way K comes, into slots that the first iterations
  // request -- as loads into registers their first use waits for every tile requested behind them, because the compiler's
  // count of requests in flight leaves out those of the inline assembly (256 keys, 48 heads: 7.9 us, 7.4 this way; d = 128
  // 11.9, 10.8).  Four waves have half the tiles in flight and a neighbour on the CU, and lose more by the requests'
  // addresses than they gain (7.4 us, 7.6 this way).
  constexpr bool Q_LDS = NWAVE == 8;
  const unsigned qbase = lds_base_addr + (Q_LDS ? PL::q_slot(__builtin_amdgcn_readfirstlane(wave)) : 0);
  i32x4 qraw[2][KS];
  if constexpr (!Q_LDS) {
#pragma unroll
    for (int qb = 0; qb < 2; qb++) {
      const __bf16* rp = row_ptr(P.q, b, h, min(q0 + qb * 16 + l16, P.sq - 1));
#pragma unroll
      for (int ks = 0; ks < KS; ks++) qraw[qb][ks] = *(const i32x4*)(rp + ks * 32 + lg * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
  } else if (active) {
    auto chunk = [&](int row) __attribute__((always_inline)) { return (lane % CPR) ^ (HD == 64 ? ((row >> 1) & 7) : (row & 15)); };
    const int uq0 = __builtin_amdgcn_readfirstlane(q0);
    const uint64_t qb0 = (uint64_t)(P.q.p0 + b * P.q.sb0 + h * P.q.sh0), qb1 = (uint64_t)(P.q.p1 + b * P.q.sb1 + h * P.q.sh1);
    int64_t ss0 = P.q.ss0 * 2, ss1 = P.q.ss1 * 2;
    int qlen0 = P.q.len0;
    asm volatile("" : "+s"(ss0), "+s"(ss1), "+s"(qlen0));  // values: selected below, not loaded from a selected address
    const bool in0 = uq0 < qlen0;
    const int64_t ss = in0 ? ss0 : ss1;
    if (uq0 + 32 <= (in0 ? qlen0 : P.sq) && ss >= 0 && ss < (1 << 26)) {  // 32 rows of one segment: a base and 32-bit offsets
      const uint64_t base = (in0 ? qb0 : qb1) + (in0 ? uq0 : uq0 - qlen0) * ss;
#pragma unroll
      for (int j = 0; j < 32 / RPI; j++) {
        const int row = j * RPI + lane / CPR;
        lds_dma16<true>((const unsigned char*)base, (unsigned)(row * (int)ss + chunk(row) * 16), qbase + j * 1024);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 32 / RPI; j++) {
        const int row = j * RPI + lane / CPR, r = min(q0 + row, P.sq - 1);
        const bool first = r < qlen0;
        const uint64_t rp = (first ? qb0 : qb1) + (uint64_t)((first ? r : r - qlen0) * (first ? ss0 : ss1));
        lds_dma16_ptr<true>((const unsigned char*)rp + chunk(row) * 16, qbase + j * 1024);
      }
    }
  }
  tile_k(0);
#pragma unroll
  for (int j = 1; j < LEAD; j++) {
    tile_k(j);
    tile_v(j - 1);
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(2 * NCH * (LEAD - 1)));  // the query rows and K0 have landed
  __syncthreads();

  const int nb = NT - 1;  // pipelined iterations
  if (!active) {
    // no query rows: this wave's share of every tile and the same barriers, nothing else
    stage_end();
    for (int t = 0; t < nb; t++) {
      tile_k(t + LEAD);
      tile_v(t + LEAD - 1);
      if (SYNC == 1 || (t & 1)) stage_end();
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
    if (SYNC == 2) __syncthreads();  // the last tile is published
    __syncthreads();                 // the flag barrier
    return *(volatile lds_int*)flag != 0;
  }

  // ---- Q fragments, softmax scale folded in: lane holds q row (qb*16 + l16), d = 32*ks + 8*lg .. +7
  const int k_swz = HD == 64 ? ((l16 >> 1) & 7) : l16;
  bf16x8 qf[2][KS];
#pragma unroll
  for (int qb = 0; qb < 2; qb++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      typedef const __attribute__((address_space(3))) i32x4 lds_chunk;
      float f[8];
      if constexpr (Q_LDS) qraw[qb][ks] = *(lds_chunk*)(uintptr_t)(qbase + (qb * 16 + l16) * ROW + (((ks * 4 + lg) ^ k_swz) << 4));
      hdit::unpack8(qraw[qb][ks], f);
#pragma unroll
      for (int e = 0; e < 8; e++) f[e] *= P.scale_log2;
      qf[qb][ks] = __builtin_bit_cast(bf16x8, hdit::pack8(f));
    }

  // ---- fragments: the lane part of the LDS addresses, the slot of the tile (a scalar), an immediate
  typedef __attribute__((address_space(3))) unsigned char lds_byte;
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  const int vt_row = 4 * lg + (l16 >> 2);  // transpose read: key row of this lane's 8 bytes, columns 4*(l16&3)
  const int vt_swz = HD == 64 ? ((vt_row >> 1) & 3) : (vt_row & 7);
  unsigned kaddr[KS], vaddr[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) kaddr[ks] = lds_address(lds) + l16 * ROW + (((ks * 4 + lg) ^ k_swz) << 4);
#pragma unroll
  for (int db = 0; db < DB; db++) vaddr[db] = lds_address(lds) + V_OFF + vt_row * ROW + ((db ^ vt_swz) << 5) + (l16 & 3) * 8;
  // keys 16*kb .. +15 of a tile, d = 32*ks .. +31
  auto k_frag = [&](unsigned slot_off, int kb, int ks) __attribute__((always_inline)) -> bf16x8 {
    return *(const __attribute__((address_space(3))) bf16x8*)((lds_byte*)(uintptr_t)(kaddr[ks] + slot_off) + kb * 16 * ROW);
  };
  // d = 16*db .. +15 of keys 32*half .. +31, in the order of the score accumulators: k-slot 8*lg + j is key 4*lg + j of the
  // first 16 keys (j < 4) or of the second
  auto v_frag = [&](unsigned slot_off, int half, int db) __attribute__((always_inline)) -> bf16x8 {
    lds_byte* va = (lds_byte*)(uintptr_t)(vaddr[db] + slot_off) + half * 32 * ROW;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(va));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(va + 16 * ROW));
    return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  f32x4 oacc[DB][2], negm[2], lsum[2];
  // scores of the two halves of a tile, [16 keys][query block]; a half's registers take the next tile's scores as
  // soon as its probabilities are packed
  f32x4 s0[2][2], s1[2][2];
  i32x4 pk[2][2];  // probabilities [half][query block], the P^T operand: [2*kb], [2*kb + 1] hold the lane's keys of block kb
#pragma unroll
  for (int qb = 0; qb < 2; qb++) {
#pragma unroll
    for (int db = 0; db < DB; db++) oacc[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
    negm[qb] = lsum[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
    pk[0][qb] = pk[1][qb] = i32x4{0, 0, 0, 0};
  }
  auto score = [&](f32x4 (&sn)[2][2], const bf16x8& kf, int kb, int ks, int qb) __attribute__((always_inline)) {
    sn[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qb][ks], ks == 0 ? negm[qb] : sn[kb][qb], 0, 0, 0);
  };
  auto pv = [&](const bf16x8& vf, int half, int db, int qb) __attribute__((always_inline)) {
    oacc[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8, pk[half][qb]), oacc[db][qb], 0, 0, 0);
  };
  // pair n: half n / 8, 16 keys (n % 8) / 4, query block (n % 4) / 2, accumulator entries 2 * (n % 2) and the next
  float pe[2];
  auto pair_exp = [&](int n, int e) __attribute__((always_inline)) {
    pe[e] = __builtin_amdgcn_exp2f((n < 8 ? s0 : s1)[(n % 8) / 4][(n % 4) / 2][2 * (n % 2) + e]);
  };
  auto pair_pack = [&](int n) __attribute__((always_inline)) {
    pk[n / 8][(n % 4) / 2][2 * ((n % 8) / 4) + n % 2] = (int)hdit::pack2(pe[0], pe[1]);
  };
  // row sums of exactly the bf16 values that enter the P.V product: a lane's own four of pairs n - 1 and n (n odd)
  auto pair_sum = [&](int n) __attribute__((always_inline)) {
    const s16x4 ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
    const int qb = (n % 4) / 2, e = 2 * ((n % 8) / 4);
    const i32x2 p4 = {pk[n / 8][qb][e], pk[n / 8][qb][e + 1]};
    lsum[qb] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_bit_cast(s16x4, p4), lsum[qb], 0, 0, 0);
  };
  auto all_scores = [&](f32x4 (&sn)[2][2], unsigned slot_off, int half) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const bf16x8 kf = k_frag(slot_off, 2 * half + kb, ks);
#pragma unroll
        for (int qb = 0; qb < 2; qb++) score(sn, kf, kb, ks, qb);
      }
  };
  auto all_pv = [&](unsigned slot_off, int half) __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < DB; db++) {
      const bf16x8 vf = v_frag(slot_off, half, db);
#pragma unroll
      for (int qb = 0; qb < 2; qb++) pv(vf, half, db, qb);
    }
  };

  // ---- the first tile sets the reference: raw scores, column maxima plus the margin, then the scores of its first 32 keys
  // again on top of -m
  {
    all_scores(s0, 0, 0);
    all_scores(s1, 0, 1);
#pragma unroll
    for (int qb = 0; qb < 2; qb++) {
      float mx = s0[0][qb][0];
#pragma unroll
      for (int e = 0; e < 4; e++) mx = fmaxf(fmaxf(fmaxf(fmaxf(mx, s0[0][qb][e]), s0[1][qb][e]), s1[0][qb][e]), s1[1][qb][e]);
      auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_int(mx), __float_as_int(mx), false, false);
      mx = fmaxf(__int_as_float(s16[0]), __int_as_float(s16[1]));
      auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_int(mx), __float_as_int(mx), false, false);
      mx = fmaxf(__int_as_float(s32[0]), __int_as_float(s32[1]));
      const float m = mx + PIPE_MARGIN;
      negm[qb] = f32x4{-m, -m, -m, -m};
    }
    all_scores(s0, 0, 0);
  }
  stage_end();
  if (tid == 0) *flag = 0;  // (two barriers and more in front of its next use)

  // fragment f of iteration t, in the order of use
  auto read_frag = [&](int f, unsigned vprev, unsigned cur, unsigned next) __attribute__((always_inline)) -> bf16x8 {
    if (f < DB) return v_frag(vprev, 1, f);
    f -= DB;
    if (f < 2 * KS) return k_frag(cur, 2 + f / KS, f % KS);
    f -= 2 * KS;
    if (f < DB) return v_frag(cur, 0, f);
    f -= DB;
    return k_frag(next, f / KS, f % KS);
  };
  bf16x8 ahead[FRAG_LEAD];  // the first fragments of the next iteration
#pragma unroll
  for (int f = 0; f < FRAG_LEAD; f++) ahead[f] = v_frag(MASK * TILE, 1, f);
  k_ptrs(LEAD);
  v_ptrs(LEAD - 1);
  // One iteration; the slots of its tiles are constants (the loop is unrolled over the ring), so that a fragment's address
  // is a register and an immediate.
  auto iteration = [&](auto Slot, int t) __attribute__((always_inline)) {
    constexpr int slot = decltype(Slot)::value;
    constexpr unsigned prev = ((slot + MASK) & MASK) * TILE, cur = slot * TILE, next = ((slot + 1) & MASK) * TILE;
    const unsigned kdst = wave_dst + ((slot + LEAD) & MASK) * TILE, vdst = wave_dst + V_OFF + ((slot + LEAD - 1) & MASK) * TILE;
    // whether the tiles requested next follow these inside one segment
    const bool next0 = t + LEAD + 1 < full0, next1 = t + LEAD - 1 >= first1 && t + LEAD + 1 < full_all;
    const unsigned kstep = (next0 ? krow0 : krow1) * BKV, vstep = (next0 ? vrow0 : vrow1) * BKV;
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 fr[F];
#pragma unroll
    for (int f = 0; f < FRAG_LEAD; f++) fr[f] = ahead[f];
    static_for<2 * F>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      constexpr int f = i / 2, qb = (i ^ f) & 1;  // the query block changes with every second MFMA
      if constexpr (f < DB) pv(fr[f], 1, f, qb);
      else if constexpr (f < DB + 2 * KS) score(s1, fr[f], (f - DB) / KS, (f - DB) % KS, qb);
      else if constexpr (f < 2 * DB + 2 * KS) pv(fr[f], 0, f - DB - 2 * KS, qb);
      else score(s0, fr[f], (f - 2 * DB - 2 * KS) / KS, (f - 2 * DB - 2 * KS) % KS, qb);
      if constexpr (i % 2 == 0) {
        if constexpr (f + FRAG_LEAD < F) fr[f + FRAG_LEAD] = read_frag(f + FRAG_LEAD, prev, cur, next);
        else ahead[f + FRAG_LEAD - F] = v_frag(cur, 1, f + FRAG_LEAD - F);
      }
      // softmax: a pair's exponentials in the first and the middle one of its PER slots, its pack in the next (the last of
      // a half at once: P.V begins)
      constexpr int n = i / PER;
      if constexpr (i % PER == 0 && n > 0 && n != 8) pair_pack(n - 1);
      if constexpr (i % PER == 0) pair_exp(n, 0);
      if constexpr (i % PER == PER / 2) pair_exp(n, 1);
      if constexpr (i % PER == PER - 1 && (n == 7 || n == 15)) pair_pack(n);
      // tile requests
      constexpr int RSTEP = F / NCH;
      if constexpr (i % RSTEP == RSTEP / 2) {
        constexpr int r = i / RSTEP;
        if constexpr (r < NCH) {
          dma_k(r, kdst);
          kp[r] += kstep;
        } else {
          dma_v(r - NCH, vdst);
          vp[r - NCH] += vstep;
        }
      }
      // the row sums last: they wait for the matrix pipe
      if constexpr (i % PER == 0 && n >= 2 && n % 2 == 0) pair_sum(n - 1);
      if constexpr (i == 2 * F - 1) pair_sum(15);
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (SYNC == 1 || slot % 2 == 1) stage_end();
    if (!(next0 || next1)) {
      k_ptrs(t + LEAD + 1);
      v_ptrs(t + LEAD);
    }
  };
  for (int t = 0; t < nb;) {
    bool more = true;
    static_for<PL::RING>([&](auto Slot) __attribute__((always_inline)) {
      if (more) {
        iteration(Slot, t);
        more = ++t < nb;
      }
    });
  }
  if (SYNC == 2) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
    __syncthreads();
  }

  // ---- the last tile: nothing to run ahead for
  {
    const int t = NT - 1;
    const unsigned prev = (unsigned)((t + MASK) & MASK) * TILE, cur = (unsigned)(t & MASK) * TILE;
    const int valid = P.skv - t * BKV;
    all_pv(prev, 1);
    all_scores(s1, cur, 1);
    if (valid < BKV) {
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int key = kb * 16 + 4 * lg + e;
#pragma unroll
          for (int qb = 0; qb < 2; qb++) {
            if (key >= valid) s0[kb][qb][e] = -INFINITY;
            if (key + 32 >= valid) s1[kb][qb][e] = -INFINITY;
          }
        }
    }
#pragma unroll
    for (int n = 0; n < 16; n++) {
      pair_exp(n, 0);
      pair_exp(n, 1);
      pair_pack(n);
      if (n % 2) pair_sum(n);
    }
    all_pv(cur, 0);
    all_pv(cur, 1);
  }

  // ---- the row sums: four lanes hold the parts of a row's
  float total[2];
  bool held[2];  // compared as bits: not above the limit, infinite or not a number
#pragma unroll
  for (int qb = 0; qb < 2; qb++) {
    auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_int(lsum[qb][0]), __float_as_int(lsum[qb][0]), false, false);
    total[qb] = __int_as_float(s16[0]) + __int_as_float(s16[1]);
    auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_int(total[qb]), __float_as_int(total[qb]), false, false);
    total[qb] = __int_as_float(s32[0]) + __int_as_float(s32[1]);
    held[qb] = __float_as_uint(total[qb]) < __float_as_uint(PIPE_LIMIT);
    rows |= (unsigned)(__builtin_amdgcn_ballot_w64(!held[qb]) & 0xffffull) << (16 * qb);
  }
  if (rows != 0 && lane == 0) *flag = 1;

  // ---- normalise and write O[q][d]: lane owns q = qb*16 + l16, d = 16*db + 4*lg + e
#pragma unroll
  for (int qb = 0; qb < 2; qb++) {
    const float inv = 1.0f / total[qb];
    const int r = q0 + qb * 16 + l16;
    if (r >= P.sq || !held[qb]) continue;
    __bf16* op = (__bf16*)row_ptr(P.o, b, h, r);
#pragma unroll
    for (int db = 0; db < DB; db++) {
      i32x2 out;
      out[0] = (int)hdit::pack2(oacc[db][qb][0] * inv, oacc[db][qb][1] * inv);
      out[1] = (int)hdit::pack2(oacc[db][qb][2] * inv, oacc[db][qb][3] * inv);
      *(i32x2*)(op + db * 16 + lg * 4) = out;
    }
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));  // nothing may land in LDS after this
  __syncthreads();
  return *(volatile lds_int*)flag != 0;
}

// The second pass.  It takes its arguments from the kernel's parameter block again, through an address the compiler
// cannot connect with the first pass: whatever the two passes would share -- segment addresses, strides, positions --
// would otherwise be held in scalar registers, or spilled, all through the first pass (83 of them), and its loop is
// scheduled around that.  A second pass inlined twice (waves with and without query rows), arguments shared -> this
// form: d = 128, 24 heads, 16896 x 16896 3444 -> 3336 us (1.02 -> 1.05 PFLOP/s), 4608 x 4608 274 -> 267, 1536 x 1536
// 55.3 -> 52.2; d = 64, 1357 x 1357 28.9 -> 27.9, 333 x 333 13.4 -> 12.8.  Without any second pass the same d = 128
// times, 26.5 and 12.6.
template <int HD>
__device__ __forceinline__ void attn_second_pass(size_t params_at, int q_tiles, int q_full, unsigned char* lds, int block_id, int nblocks,
                                                 unsigned rows) {
  typedef const __attribute__((address_space(4))) int64_t* const_ptr;
  uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr() + params_at;
  asm volatile("" : "+s"(at), "+s"(q_tiles), "+s"(q_full), "+s"(block_id), "+s"(nblocks));
  static_assert(sizeof(AttnParams) % 8 == 0, "copied in 8-byte pieces");
  struct Raw {
    int64_t v[sizeof(AttnParams) / 8];
  } raw;
#pragma unroll
  for (unsigned i = 0; i < sizeof(AttnParams) / 8; i++) raw.v[i] = ((const_ptr)at)[i];
  const AttnParams P = __builtin_bit_cast(AttnParams, raw);
  __syncthreads();  // every wave has read the flag, whose bytes this pass may overwrite
  attn_tracked_body<HD>(P, q_tiles, q_full, lds, block_id, nblocks, rows);
}

template <int HD>
__global__ void __launch_bounds__(NTHR, 2) attn_fwd_pipe_kernel(const AttnParams P, int q_tiles, int q_full) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  unsigned rows;
  if (attn_pipe_body<HD>(P, q_tiles, q_full, lds, (int)blockIdx.x, (int)gridDim.x, rows))
    attn_second_pass<HD>(0, q_tiles, q_full, lds, (int)blockIdx.x, (int)gridDim.x, rows);
}

template <int HD>
__global__ void __launch_bounds__(NTHR, 2) attn_fwd_pipe_multi_kernel(const AttnMulti M) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int i = 0;
#pragma unroll 1
  while (i + 1 < M.count && (int)blockIdx.x >= M.start[i + 1]) i++;
  const int local = (int)blockIdx.x - M.start[i];
  if (local >= M.nblocks[i]) return;
  unsigned rows;
  if (attn_pipe_body<HD>(M.p[i], M.q_tiles[i], M.q_full[i], lds, local, M.nblocks[i], rows))
    attn_second_pass<HD>(offsetof(AttnMulti, p) + i * sizeof(AttnParams), M.q_tiles[i], M.q_full[i], lds, local, M.nblocks[i],
                         rows);
}

// Host side of a multi launch: the table of `count` problems, ranges padded to multiples of 8 workgroups.
inline int fill_multi(AttnMulti& M, const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count) {
  M.count = count;
  int at = 0;
  for (int i = 0; i < ATTN_MAX_MULTI; i++) {
    M.start[i] = at;
    if (i < count) {
      M.p[i] = P[i], M.q_tiles[i] = q_tiles[i], M.q_full[i] = q_full[i], M.nblocks[i] = nblocks[i];
      at += (nblocks[i] + 7) / 8 * 8;
    } else {
      M.p[i] = P[0], M.q_tiles[i] = 1, M.q_full[i] = 1, M.nblocks[i] = 0;
    }
  }
  M.start[ATTN_MAX_MULTI] = at;
  return at;
}

// One grid of `count` problems: a kernel that takes one, or one that takes a table.
template <class One, class Multi>
int launch_grid(One one, Multi multi, int lds_bytes, std::atomic<bool>& attr_set, const AttnParams* P, const int* q_tiles,
                const int* q_full, const int* nblocks, int count, hipStream_t stream) {
  if (lds_bytes > 64 * 1024 && !attr_set.load(std::memory_order_acquire)) {  // setting them twice from two threads is harmless
    if (hipFuncSetAttribute((const void*)one, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess ||
        hipFuncSetAttribute((const void*)multi, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
      return HDIT_ELAUNCH;
    attr_set.store(true, std::memory_order_release);
  }
  if (count == 1) {
    hipLaunchKernelGGL(one, dim3((unsigned)nblocks[0]), dim3(NTHR), lds_bytes, stream, P[0], q_tiles[0], q_full[0]);
    return HDIT_OK;
  }
  AttnMulti M;
  const int grid = fill_multi(M, P, q_tiles, q_full, nblocks, count);
  hipLaunchKernelGGL(multi, dim3((unsigned)grid), dim3(NTHR), lds_bytes, stream, M);
  return HDIT_OK;
}

}  // namespace

#define HDIT_ATTN_LAUNCH(name, HD, kernel, multi_kernel, lds)                                                              \
  int name(const AttnParams* P, const int* q_tiles, const int* q_full, const int* nblocks, int count, hipStream_t stream) {                   \
    static std::atomic<bool> attr_set{false};                                                                              \
    return launch_grid(kernel<HD>, multi_kernel<HD>, lds<HD>::TOTAL, attr_set, P, q_tiles, q_full, nblocks, count, stream); \
  }
