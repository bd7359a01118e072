// Grouped bf16 GEMM for gfx950:  C[m, n] = epilogue(A[m, k] . B[n, k]^T + bias)
//
// Persistent kernel, one 256-thread workgroup (2x2 waves) per CU, walking a
// static list of output tiles of (64*TM) x (64*TN) elements; a wave owns a
// (32*TM) x (32*TN) sub-tile in accumulators (v_mfma_f32_16x16x32_bf16).
//
// What bounds the large shapes is the board's power: the main loop holds 1.9 - 2.0 of 2.4 GHz.  The 16x16x32 MFMA moves
// half the accumulator bytes per flop of the 32x32x16 one and costs less energy: bare loops of either on random operands,
// all CUs, run at 2.00 and 1.73 PFLOP/s (1.89 where no operand is shared by consecutive MFMAs, 2.00 where one is).  Bias
// epilogue, 32x32x16 -> 16x16x32 on one box: 8192 x 2048 x 6144 149.9 -> 138.3 us, 8192 x 1536 x 6144 116.7 -> 109.0,
// 8192 x 4608 x 1536 99.2 -> 94.2, 4608 x 3072 x 15360 327 -> 312, 8192^3 762 -> 709 (1.55 PFLOP/s); with GELU 8192 x 6144 x
// 1536 140.6 -> 131.6.  The shapes that do not fill the chip are bound otherwise (below) and stay level.  Both
// instructions give the same bits.
//
// Staging.  Both operands are k-contiguous, so A and B tiles are staged the
// same way, in slabs of 64 k (128 bytes per row).  A wave-wide request fetches
// 8 rows x 128 bytes, eight lanes per row: every request covers whole 128-byte
// cache lines (64-byte row pieces were measured at half the L2->CU rate,
// 29 B/clk/CU against 58).  LDS rows are 128 bytes whose 16-byte chunks are
// XOR-swizzled with (row>>1)&7: the 16 lanes of a ds_read_b128 pass (16 rows,
// one chunk) land on 16 distinct 16-byte slots of the 256-byte bank window.
//
// Pipeline.  The k slabs of all tiles of a workgroup form one flat stream; tile
// boundaries are invisible to it, so a tile's first slabs arrive during the
// previous tile's last slab and epilogue.  A slab is worked on in eight quarters
// (two k-steps of 32 times four quarters of the wave's tile), whose fragments are
// read two quarters ahead; the workgroup barrier sits before the last two
// quarters of a slab, whose fragments are already in registers, so that the first
// fragments of the next slab are read under their MFMAs.
//  * 256-row shapes, 192x192: direct to LDS (global_load_lds_dwordx4, swizzle applied on
//    the source side), three A slots and two B slots.  During slab g the A rows
//    of slab g+2 are requested (quarters 0..5) into the slot slab g-1 vacated;
//    behind the barrier that ends slab g, the B rows of slab g+2 go into the B
//    slot just vacated.  Requests retire in order, so the wait in front of the
//    barrier leaves exactly the newest A requests in flight.
//  * 128x256: two LDS stages, register-staged.  While slab h is
//    multiplied out of stage h&1, the registers holding slab h+1 are written
//    to the other stage and immediately refilled with the global loads of slab
//    h+2, one write+load pair every few MFMAs.
//  * ring shapes (64x64 to 128x192), for the launches that do not fill the chip: a slab is 8 to 48 MFMAs per wave,
//    and what bounds it is the operands' way to the CU: time per slab is proportional to its bytes, 25 - 40 B/clk/CU,
//    whatever its MFMAs.  (The requests alone, no arithmetic, take the same time: 85 - 90 GB/s per CU whether 64 or 248 CUs
//    of the chip work, whatever the stages, the waves, the row pitch or the order of the rows; 135 only where everything
//    is in the XCD's L2 already.)  Direct to LDS through a ring of 3 to 8 stages; the fragments of a whole slab are
//    double-buffered in registers, so a slab has one barrier and no wait for LDS inside, and its stage is free for
//    the request of the slab NS ahead as soon as it begins.  Measured (warm weights, microseconds per slab): 128x128
//    0.36 - 0.39, 0.54 before with four stages and fragments one k-step ahead; 128x192 0.45, 0.67 before
//    (register-staged); 64x128 0.27; 64x64 0.19.  Small tiles are what short problems need: 333 x 1536 x 6144 is 36
//    tiles of 128x128 (61 us at first), 144 of 64x64 (27 us).
//
// Epilogue.  A lane's accumulator holds one output row m and 4 consecutive n of
// a 16-column block; lanes l and l^16 swap runs of two neighbouring blocks
// (v_permlane16_swap) to own 8 consecutive n.  bias / GELU-tanh are applied there, the bf16 result is staged
// through a wave-private 8 KiB window inside the LDS stage (the A slot) the last
// slab just vacated (ring shapes: behind the stages) and written back with 16 lanes covering 256 contiguous bytes of a row
// (gate and residual are applied in that coalesced layout, in fp32).
//
// One launch covers up to HDIT_GEMM_MAX_PROBLEMS problems.  Tiles are dealt to
// workgroups so that the workgroups of one XCD (workgroup id mod 8; each XCD
// has a private L2) own a contiguous, 8-tile-row-grouped range.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "hdit_common.h"

namespace {

constexpr int BK = 64;           // k elements per LDS stage
constexpr int ROW_BYTES = 128;   // BK * sizeof(bf16)
constexpr int NUM_XCD = 8;
constexpr int GROUP_M = 8;
constexpr int NW = 4;
constexpr int NT = 256;
constexpr int EPI_WAVE_BYTES = 8192;  // 32 rows x 128 columns of bf16

struct GemmTable {
  int count;
  int tile_start[HDIT_GEMM_MAX_PROBLEMS + 1];
  hdit_gemm_problem p[HDIT_GEMM_MAX_PROBLEMS];
};

constexpr int RING_MAX_MMA = 6;  // TM * TN of the shapes that take their slabs through a ring

template <int TM_, int TN_>
struct Cfg {
  static constexpr int TM = TM_, TN = TN_;
  static constexpr int BM = 64 * TM, BN = 64 * TN;
  static constexpr int WM = 32 * TM, WN = 32 * TN;
  static constexpr int A_LOADS = BM / 8 / NW;  // wave-wide loads (8 rows x 128 bytes) per wave per slab
  static constexpr int B_LOADS = BN / 8 / NW;
  static constexpr int LOADS = A_LOADS + B_LOADS;
  static constexpr int A_BYTES = BM * ROW_BYTES;
  static constexpr int B_BYTES = BN * ROW_BYTES;
  static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
  // DMA: the 256-row shapes and 192x192 take their operand slabs straight from global memory into LDS
  // (global_load_lds_dwordx4: no staging registers, no ds_write).  A has three slots (requested two slabs
  // ahead), B two (requested one slab ahead, first in the queue); the epilogue windows alias the A slot the
  // tile's last slab vacated, which is exactly as large (192x192: they lie behind the slots).
  static constexpr bool DMA = TM == 4 || (TM == 3 && TN == 3);
  static constexpr int A_SLOTS = 3, B_SLOTS = 2;
  static constexpr int B_OFF = A_SLOTS * A_BYTES;
  static constexpr bool EPI_ALIAS = NW * EPI_WAVE_BYTES <= A_BYTES;
  static constexpr int DMA_BYTES = A_SLOTS * A_BYTES + B_SLOTS * B_BYTES + (EPI_ALIAS ? 0 : NW * EPI_WAVE_BYTES);
  // RING: the shapes with short slabs (8 to 48 MFMAs per wave) take them the same way into a ring of NS stages
  // (A then B), as many as fit beside the epilogue windows: only a lead of several slabs covers the latency of
  // operands that come from HBM.
  static constexpr bool RING = TM * TN <= RING_MAX_MMA;
  // windows of their own, behind the stages or slots
  static constexpr int EPI_OFF = DMA ? DMA_BYTES - NW * EPI_WAVE_BYTES : 160 * 1024 - NW * EPI_WAVE_BYTES;
  static constexpr int NS = RING ? (EPI_OFF / STAGE_BYTES < 8 ? EPI_OFF / STAGE_BYTES : 8) : 2;
  static constexpr bool DIRECT = DMA || RING;
  static constexpr int LDS_BYTES = DMA ? DMA_BYTES : RING ? 160 * 1024 : NS * STAGE_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "tile does not fit the LDS");
  static_assert(RING || DMA || NW * EPI_WAVE_BYTES <= STAGE_BYTES, "the epilogue windows live inside one stage");
  static_assert(!RING || NS >= 3, "a ring holds the slab being read and at least one on its way");
  static_assert(TN <= 4, "epilogue staging window is 128 columns wide");
};

struct TileCoord {
  int pi, m0, n0;
};

template <class C>
__device__ __forceinline__ TileCoord locate(const GemmTable& tab, int lid) {
  int pi = 0;
#pragma unroll 1
  while (pi + 1 < tab.count && lid >= tab.tile_start[pi + 1]) pi++;
  const int tiles_m = (tab.p[pi].m + C::BM - 1) / C::BM;
  const int tiles_n = (tab.p[pi].n + C::BN - 1) / C::BN;
  const int t = lid - tab.tile_start[pi];
  const int in_group = GROUP_M * tiles_n;
  const int first_m = (t / in_group) * GROUP_M;
  const int gsz = min(tiles_m - first_m, GROUP_M);
  TileCoord tc;
  tc.pi = pi;
  tc.m0 = (first_m + (t % in_group) % gsz) * C::BM;
  tc.n0 = ((t % in_group) / gsz) * C::BN;
  return tc;
}

// One wave-wide direct-to-LDS copy: lane l's 16 bytes at base + voff land at LDS byte address
// lds_addr + lds_off + 16*l; the sum is formed in M0 itself (one scalar instruction less per request than adding
// first and moving the result: a slab is 16 requests per wave).  Inline assembly, so the compiler's wait-count
// insertion does not see it: an extra operation in flight only makes the waits it computes for its own
// loads stricter than needed.
// Every direct-to-LDS request is issued at agent scope (sc1), which the CU's L1 never serves.  The kernels wait
// for "all but the newest n" requests and rely on completion in issue order; a request that hits in L1 completes
// ahead of older misses (measured: a ragged tile, whose out-of-range lanes all read the problem's last row, then
// multiplied a slab that had not landed).  From L2, hits and misses complete in issue order.
__device__ __forceinline__ void lds_dma16_sum(const unsigned char* base_uniform, unsigned voff, unsigned lds_addr_uniform,
                                              unsigned lds_off_uniform) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 sc1"
               :
               : "s"(lds_addr_uniform), "v"(voff), "s"(base_uniform), "s"(lds_off_uniform)
               : "m0", "scc");
}

__device__ __forceinline__ unsigned lds_address(const unsigned char* p) {
  return (unsigned)(uintptr_t)((const __attribute__((address_space(3))) unsigned char*)p);
}

#define SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

// s_waitcnt immediate that waits for all but the newest n vector-memory operations (and for nothing else)
constexpr int waitcnt_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0f70; }

// All tiles of one shape that this workgroup owns.
template <class C>
__device__ __forceinline__ void run_tiles(const GemmTable& tab, int total_tiles, int tiles_per_xcd, int wgs_per_xcd,
                                          int wg_in_xcd, unsigned char* lds) {
  constexpr int TM = C::TM, TN = C::TN;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int wm0 = (wave >> 1) * C::WM;
  const int wn0 = (wave & 1) * C::WN;

  // tiles of this workgroup: XCD x owns logical tiles [x*tiles_per_xcd, (x+1)*tiles_per_xcd),
  // dealt round-robin to that XCD's workgroups
  const int xcd = blockIdx.x % NUM_XCD;
  const int xcd_begin = xcd * tiles_per_xcd;
  const int xcd_end = min(xcd_begin + tiles_per_xcd, total_tiles);
  int lid = xcd_begin + wg_in_xcd;
  if (lid >= xcd_end) return;

  // ---- producer: the slab stream, two slabs ahead of the MFMAs ------------------
  // A wave-wide load covers rows 8*(wave + NW*i) + lane/8 of the A (or B) tile, chunk lane%8 of the row's
  // 128-byte slab.  Its LDS destination is row*128 + ((chunk ^ ((row>>1)&7)) << 4); (row>>1)&7 does not
  // depend on i, so the destinations of one lane differ by the constant NW*8*128 bytes.
  const int ld_row = lane >> 3;
  const int ld_chunk = lane & 7;
  const int st_row = wave * 8 + ld_row;
  const int st_off = st_row * ROW_BYTES + ((ld_chunk ^ ((st_row >> 1) & 7)) << 4);
  // A direct-to-LDS request lands lane l at byte 16*l of the wave's 1 KiB (row l/8, position l%8), so the
  // swizzle is applied on the source side: position c' of row r receives chunk c' ^ ((r>>1)&7).
  const int src_chunk = C::DIRECT ? (ld_chunk ^ ((st_row >> 1) & 7)) : ld_chunk;
  const unsigned lds_base_addr = __builtin_amdgcn_readfirstlane(lds_address(lds));
  int p_lid = lid;
  bool p_valid = true;
  int p_kt = 0, p_KT = 0;
  const unsigned char* p_abase = nullptr;
  const unsigned char* p_bbase = nullptr;
  unsigned p_off[C::LOADS];
  i32x4 G[C::DIRECT ? 1 : C::LOADS];  // the slab in flight between global memory and LDS (register-staged shapes)
  auto p_setup = [&]() {
    const TileCoord tc = locate<C>(tab, p_lid);
    const hdit_gemm_problem& pr = tab.p[tc.pi];
    p_abase = (const unsigned char*)pr.a;
    p_bbase = (const unsigned char*)pr.b;
    p_KT = pr.k / BK;
    p_kt = 0;
#pragma unroll
    for (int i = 0; i < C::A_LOADS; i++) {
      const int gr = min(tc.m0 + (wave + i * NW) * 8 + ld_row, pr.m - 1);
      unsigned row_off = (unsigned)gr * (unsigned)pr.lda;  // byte offsets stay below 2^32: checked on the host
      asm volatile("" : "+v"(row_off));  // a product of its own: fused with the addition it is a 64-bit multiply-add,
                                         // and the offsets then occupy register pairs for the whole kernel
      p_off[i] = (row_off + (unsigned)(src_chunk * 8)) * 2u;
    }
#pragma unroll
    for (int i = 0; i < C::B_LOADS; i++) {
      const int gr = min(tc.n0 + (wave + i * NW) * 8 + ld_row, pr.n - 1);
      unsigned row_off = (unsigned)gr * (unsigned)pr.ldb;
      asm volatile("" : "+v"(row_off));
      p_off[C::A_LOADS + i] = (row_off + (unsigned)(src_chunk * 8)) * 2u;
    }
  };
  // Once the stream is exhausted the last slab is simply loaded again and written to a stage nobody
  // reads: no branch may split the MFMA stream the loads are interleaved with.
  auto g_load = [&](int i) {
    const unsigned char* base = (i < C::A_LOADS ? p_abase : p_bbase) + (size_t)p_kt * ROW_BYTES;
    G[i] = *(const i32x4*)(base + p_off[i]);
  };
  // direct-to-LDS request i of the slab at the cursor: A rows into A slot `slot`, B rows into B slot `slot`
  const unsigned wave_lds = lds_base_addr + wave * 8 * ROW_BYTES;
  auto dma_a = [&](int slot, int i) {
    lds_dma16_sum(p_abase + (size_t)p_kt * ROW_BYTES, p_off[i], wave_lds + slot * C::A_BYTES, i * (NW * 8 * ROW_BYTES));
  };
  auto dma_b = [&](int slot, int i) {
    lds_dma16_sum(p_bbase + (size_t)p_kt * ROW_BYTES, p_off[C::A_LOADS + i], wave_lds + C::B_OFF + slot * C::B_BYTES,
                  i * (NW * 8 * ROW_BYTES));
  };
  // ring shapes: request i (A rows, then B rows) of the slab at the cursor into stage `slot`
  auto dma_ring = [&](int slot, int i) {
    if (i < C::A_LOADS)
      lds_dma16_sum(p_abase + (size_t)p_kt * ROW_BYTES, p_off[i], wave_lds + slot * C::STAGE_BYTES, i * (NW * 8 * ROW_BYTES));
    else
      lds_dma16_sum(p_bbase + (size_t)p_kt * ROW_BYTES, p_off[i], wave_lds + slot * C::STAGE_BYTES,
                    C::A_BYTES + (i - C::A_LOADS) * (NW * 8 * ROW_BYTES));
  };
  auto l_store = [&](int stage, int i) {
    const int tile_off = i < C::A_LOADS ? i * (NW * 8 * ROW_BYTES) : C::A_BYTES + (i - C::A_LOADS) * (NW * 8 * ROW_BYTES);
    *(i32x4*)(lds + stage * C::STAGE_BYTES + tile_off + st_off) = G[i];
  };
  auto p_advance = [&]() {
    if (!p_valid) return;
    if (++p_kt == p_KT) {
      p_lid += wgs_per_xcd;
      p_valid = p_lid < xcd_end;
      if (p_valid) p_setup();
      else p_kt = p_KT - 1;
    }
  };

  // ---- consumer ------------------------------------------------------------
  // fragment read offsets: row r, logical chunk c -> r*128 + ((c ^ ((r>>1)&7)) << 4); fragment rows are
  // l16 plus a multiple of 16, so (r>>1)&7 == (l16>>1)&7.  k-step ks (32 k) uses chunk 4*ks + lg.
  const int swz = (l16 >> 1) & 7;
  const int a_row = (wm0 + l16) * ROW_BYTES;
  const int b_row = (wn0 + l16) * ROW_BYTES;
  // fragments of half of the wave's rows and half of its columns, two slots each
  bf16x8 fa[2][TM], fb[4][TN];
  // ring shapes: the fragments of whole slabs, the one being multiplied and the next
  constexpr int SK = C::RING ? BK / 32 : 1;
  bf16x8 sfa[2][SK][2 * TM], sfb[2][SK][2 * TN];
  auto read_slab_frag = [&](const unsigned char* sbase, int buf, int r) {  // r-th fragment in the order of use
    const int ks = r / (2 * TM + 2 * TN), f = r % (2 * TM + 2 * TN);
    const int ch = ((ks * 4 + lg) ^ swz) << 4;
    if (f < 2 * TN) sfb[buf][ks][f] = *(const bf16x8*)(sbase + C::A_BYTES + b_row + ch + f * 16 * ROW_BYTES);
    else sfa[buf][ks][f - 2 * TN] = *(const bf16x8*)(sbase + a_row + ch + (f - 2 * TN) * 16 * ROW_BYTES);
  };
  auto read_a = [&](const unsigned char* abase, int ks, int half, int slot, int i) {
    fa[slot][i] = *(const bf16x8*)(abase + a_row + (((ks * 4 + lg) ^ swz) << 4) + (half * TM + i) * 16 * ROW_BYTES);
  };
  auto read_b = [&](const unsigned char* bbase, int ks, int half, int slot, int j) {
    fb[slot][j] = *(const bf16x8*)(bbase + b_row + (((ks * 4 + lg) ^ swz) << 4) + (half * TN + j) * 16 * ROW_BYTES);
  };
  auto read_first = [&](const unsigned char* abase, const unsigned char* bbase) {  // rows and columns of a slab's first quarter
#pragma unroll
    for (int i = 0; i < TM; i++) read_a(abase, 0, 0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; j++) read_b(bbase, 0, 0, 0, j);
#pragma unroll
    for (int j = 0; j < TN; j++) read_b(bbase, 0, 1, 1, j);
  };

  // The bias enters through the accumulators: a tile's accumulators start as bias (x) ones -- one MFMA per 16-column
  // block, whose A operand holds bias[n] at k = 0 and whose B operand holds 1 at k = 0 -- instead of zero.  The
  // epilogue then needs neither bias registers (the 256 x 256 shape could only find its 32 by spilling accumulators)
  // nor an LDS slot, and every shape forms bias + sum of products in the same order, so results do not depend on the
  // shape a problem is given.  Lane l < 16 fetches the bias of column l of each of the wave's column blocks; the
  // values of the next tile are requested at the start of the current tile's epilogue, in front of its stores.
  unsigned short bnext[2 * TN];
  auto fetch_bias = [&](const TileCoord& tc) {
    const hdit_gemm_problem& pr = tab.p[tc.pi];
    const unsigned short* bsrc = (const unsigned short*)pr.bias;
#pragma unroll
    for (int j = 0; j < 2 * TN; j++) {
      bnext[j] = 0;
      if (bsrc) bnext[j] = bsrc[min(tc.n0 + wn0 + j * 16 + l16, pr.n - 1)];
    }
  };
  fetch_bias(locate<C>(tab, lid));

  // prologue: the first slabs of the stream -- two into the slots of the 256-row shapes, NS into the stages of the ring
  // shapes; register-staged: slab 0 into stage 0, slab 1 into the registers
  p_setup();
  int stage = 0;
  int sa = 0, sb = 0;  // DMA: the A and B slots of the slab being multiplied
  if constexpr (C::DMA) {
    // slab 0 into slots (0, 0), slab 1 into slots (1, 1); slab 0 has landed before the first fragment read
#pragma unroll
    for (int i = 0; i < C::A_LOADS; i++) dma_a(0, i);
#pragma unroll
    for (int i = 0; i < C::B_LOADS; i++) dma_b(0, i);
    p_advance();
#pragma unroll
    for (int i = 0; i < C::A_LOADS; i++) dma_a(1, i);
#pragma unroll
    for (int i = 0; i < C::B_LOADS; i++) dma_b(1, i);
    p_advance();
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(C::LOADS));
    __syncthreads();
    read_first(lds, lds + C::B_OFF);
  } else if constexpr (C::RING) {
    // slabs 0 .. NS-1 into stages 0 .. NS-1; slab 0 has landed before the first fragment read
#pragma unroll
    for (int s = 0; s < C::NS; s++) {
#pragma unroll
      for (int i = 0; i < C::LOADS; i++) dma_ring(s, i);
      p_advance();
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_vm((C::NS - 1) * C::LOADS));
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SK * 2 * (TM + TN); r++) read_slab_frag(lds, 0, r);
  } else {
#pragma unroll
    for (int i = 0; i < C::LOADS; i++) g_load(i);
    p_advance();
#pragma unroll
    for (int i = 0; i < C::LOADS; i++) l_store(0, i);
#pragma unroll
    for (int i = 0; i < C::LOADS; i++) g_load(i);
    p_advance();
    __syncthreads();
    read_first(lds, lds + C::A_BYTES);
  }

  constexpr int NQ = TM * TN;  // MFMAs of a quarter of the wave's tile

  bool first_tile = true;
  while (true) {
    const TileCoord tc = locate<C>(tab, lid);
    const hdit_gemm_problem& pr = tab.p[tc.pi];
    const int KT = pr.k / BK;
    if (!first_tile) {
      __syncthreads();  // every wave has left the previous epilogue, whose staging windows the next writes reuse
    }
    first_tile = false;

    f32x4 acc[2 * TM][2 * TN];
    {
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      i32x4 ones_bits = {lg == 0 ? 0x3f80 : 0, 0, 0, 0};  // bf16 1.0 at k = 0 (lanes < 16 hold k = 0..7)
      bf16x8 ones;
      __builtin_memcpy(&ones, &ones_bits, 16);
#pragma unroll
      for (int j = 0; j < 2 * TN; j++) {
        i32x4 bb = {lg == 0 ? (int)bnext[j] : 0, 0, 0, 0};
        bf16x8 bfr;
        __builtin_memcpy(&bfr, &bb, 16);
#pragma unroll
        for (int i = 0; i < 2 * TM; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr, ones, zero, 0, 0, 0);
      }
    }

    // A slab is two k-steps of 32 k, a k-step four quarters of the wave's tile -- rows half a0 or a1, columns half b0 or
    // b1 -- in the order (a0,b0) (a0,b1) (a1,b1) (a1,b0): each needs one half that the one before did not.  A half is
    // read two quarters ahead, behind the first MFMAs of a quarter: a1 in quarter 0, b0 of the second k-step in 1, its
    // a0 in 2, its b1 in 3, its a1 in 4; behind the barrier (after 5) the next slab's a0 and b0 in 6 and b1 in 7.
    // The rows have two slots, the columns four (k-step, half).  Consecutive MFMAs share an operand.
    // `carry(t)`: what else is issued behind MFMA t.
    auto quarter = [&](int h, const unsigned char* rd_a, const unsigned char* rd_b, auto&& carry) {
      const int q = h & 3, ks = h >> 2, ah = q >> 1, bh = (q == 1 || q == 2) ? 1 : 0;
#pragma unroll
      for (int t = 0; t < NQ; t++) {
        const int j = t / TM, i = (j & 1) ? TM - 1 - t % TM : t % TM;
        f32x4& c = acc[ah * TM + i][bh * TN + j];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[2 * ks + bh][j], fa[ah][i], c, 0, 0, 0);
        if (h == 0 && t < TM) read_a(rd_a, 0, 1, 1, t);
        if (h == 1 && t < TN) read_b(rd_b, 1, 0, 2, t);
        if (h == 2 && t < TM) read_a(rd_a, 1, 0, 0, t);
        if (h == 3 && t < TN) read_b(rd_b, 1, 1, 3, t);
        if (h == 4 && t < TM) read_a(rd_a, 1, 1, 1, t);
        if (h == 6 && t < TM) read_a(rd_a, 0, 0, 0, t);
        if (h == 6 && t < TN) read_b(rd_b, 0, 0, 0, t);
        if (h == 7 && t < TN) read_b(rd_b, 0, 1, 1, t);
        carry(t);
        SCHED_FENCE();
      }
    };

    if constexpr (C::DMA) {
      for (int kt = 0; kt < KT; kt++) {
        const unsigned char* ab = lds + sa * C::A_BYTES;
        const unsigned char* bb = lds + C::B_OFF + sb * C::B_BYTES;
        // A rows of the slab after next go to the slot the previous slab vacated
        const int sa_req = sa == 0 ? C::A_SLOTS - 1 : sa - 1;
        constexpr int APQ = (C::A_LOADS + 5) / 6;  // A requests per quarter
#pragma unroll
        for (int h = 0; h < 6; h++) {
          quarter(h, ab, bb, [&](int t) {
#pragma unroll
            for (int r = 0; r < APQ; r++)
              if (h * APQ + r < C::A_LOADS && t == NQ - 1 - 3 * (APQ - 1 - r)) dma_a(sa_req, h * APQ + r);
          });
        }
        // ---- turn over: everything but the A requests just issued has landed (the next slab is complete),
        // and the last fragments of this slab are in registers
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(C::A_LOADS) & 0xf0ff);  // and lgkmcnt(0)
        __syncthreads();
        const int sb_req = sb;  // the B slot this slab vacates takes the B rows of the slab after next
        sa = sa == C::A_SLOTS - 1 ? 0 : sa + 1;
        sb ^= 1;
        constexpr int BPQ = (C::B_LOADS + 1) / 2;
#pragma unroll
        for (int h = 0; h < 2; h++)
          quarter(6 + h, lds + sa * C::A_BYTES, lds + C::B_OFF + sb * C::B_BYTES, [&](int t) {
#pragma unroll
            for (int r = 0; r < BPQ; r++)
              if (h * BPQ + r < C::B_LOADS && t == NQ - 1 - 2 * (BPQ - 1 - r)) dma_b(sb_req, h * BPQ + r);
          });
        p_advance();
      }
    } else if constexpr (C::RING) {
      // One slab: its MFMAs, on fragments that are in registers; under the first of them, the reads of the next
      // slab's fragments, under the others the requests of the slab NS ahead, into the stage this slab's fragments
      // have been read from.  One barrier per slab: every wave holds this slab's fragments, and the next slab has
      // landed (everything but the NS-2 slabs behind it).
      constexpr int NM = SK * 4 * NQ, NR = SK * 2 * (TM + TN);
      constexpr int RPM = (NR + (NM + 1) / 2 - 1) / ((NM + 1) / 2);  // reads behind each of the first MFMAs
      constexpr int RM = (NR + RPM - 1) / RPM;                       // MFMAs that carry them
      auto ring_slab = [&](int buf) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm((C::NS - 2) * C::LOADS) & 0xf0ff);  // and lgkmcnt(0)
        __syncthreads();
        const int rq = stage;
        stage = stage == C::NS - 1 ? 0 : stage + 1;
        const unsigned char* nbase = lds + stage * C::STAGE_BYTES;
#pragma unroll
        for (int t = 0; t < NM; t++) {
          const int ks = t / (4 * NQ), j = (t % (4 * NQ)) / (2 * TM), i0 = t % (2 * TM), i = (j & 1) ? 2 * TM - 1 - i0 : i0;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sfb[buf][ks][j], sfa[buf][ks][i], acc[i][j], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < RPM; r++)
            if (t < RM && t * RPM + r < NR) read_slab_frag(nbase, buf ^ 1, t * RPM + r);
#pragma unroll
          for (int q = 0; q < C::LOADS; q++)
            if (t >= RM && RM + q * (NM - RM) / C::LOADS == t) dma_ring(rq, q);
          SCHED_FENCE();
        }
        p_advance();
      };
      int kt = 0;
#pragma unroll 1
      for (; kt + 1 < KT; kt += 2) {
        ring_slab(0);
        ring_slab(1);
      }
      if (kt < KT) {
        ring_slab(0);
#pragma unroll
        for (int ks = 0; ks < SK; ks++) {
#pragma unroll
          for (int i = 0; i < 2 * TM; i++) sfa[0][ks][i] = sfa[1][ks][i];
#pragma unroll
          for (int j = 0; j < 2 * TN; j++) sfb[0][ks][j] = sfb[1][ks][j];
        }
      }
    } else
    for (int kt = 0; kt < KT; kt++) {
      const unsigned char* sbase = lds + stage * C::STAGE_BYTES;
      const int wstage = stage ^ 1;  // held slab h-1; every wave passed the barrier of that slab
      // registers of slab h+1 to LDS stage `wstage`, then the same registers refilled with slab h+2
      constexpr int LPQ = (C::LOADS + 5) / 6;
#pragma unroll
      for (int h = 0; h < 6; h++) {
        quarter(h, sbase, sbase + C::A_BYTES, [&](int t) {
#pragma unroll
          for (int r = 0; r < LPQ; r++)
            if (h * LPQ + r < C::LOADS && t == NQ - 1 - 2 * (LPQ - 1 - r)) {
              l_store(wstage, h * LPQ + r);
              g_load(h * LPQ + r);
            }
        });
      }
      p_advance();
      // ---- turn the stages over: the last fragments of this slab are in registers, slab h+1 is written
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __syncthreads();
      stage ^= 1;
      const unsigned char* nbase = lds + stage * C::STAGE_BYTES;
#pragma unroll
      for (int h = 0; h < 2; h++) quarter(6 + h, nbase, nbase + C::A_BYTES, [](int) {});
    }
    // staging window of this wave: inside the stage (the A slot) the tile's last slab vacated
    unsigned char* epi = lds + wave * EPI_WAVE_BYTES +
                         (C::RING || (C::DMA && !C::EPI_ALIAS) ? C::EPI_OFF
                          : C::DMA                             ? (sa == 0 ? C::A_SLOTS - 1 : sa - 1) * C::A_BYTES
                                                               : (stage ^ 1) * C::STAGE_BYTES);

    // ---- epilogue ---------------------------------------------------------
    auto epilogue = [&](auto mode_tag) {
      constexpr int MODE = decltype(mode_tag)::value;
      constexpr bool GATED = MODE == HDIT_EPI_GATE_RESIDUAL;
      // The lane-dependent addresses of the epilogue are recomputed per tile from an opaque copy of the lane id:
      // otherwise the compiler hoists some fifty of them out of the tile loop and, the main loop having no registers
      // to spare, spills them around it -- reloads that wait for every operand request in flight.
      int lane_e = lane;
      asm volatile("" : "+v"(lane_e));
      const int l16 = lane_e & 15, lg = lane_e >> 4;
      // all addressing below is a uniform base plus a 32-bit byte offset per lane (checked on the host)
      unsigned char* __restrict__ Cb = (unsigned char*)pr.c;
      const unsigned char* __restrict__ Rb = (const unsigned char*)pr.resid;
      const float* __restrict__ gate = pr.gate;
      const int M = pr.m, N = pr.n;
      const int ldc = (int)pr.ldc, ldr = (int)pr.ldr;
      const int ncol0 = tc.n0 + wn0;

      // Write-back layout: 16 lanes cover one 256-byte row segment, a wave covers 4 rows per pass, 8 passes
      // per 32-row block, done as two halves of 4.  The residual rows and the gate columns are requested one
      // block ahead, before the stores in front of them: vector memory operations retire in order, so a load
      // placed behind stores would wait for the stores' round trip.
      const int rchunk = lane_e & 15;
      const int wr_row = lane_e >> 4;
      const int wr_n = ncol0 + rchunk * 8;
      const int wr_nc = min(wr_n, N - 8);
      const bool wr_ok = rchunk < 4 * TN && wr_n < N;
      // The residual stream may be carried in fp32 (HDIT_EPI_RESID_F32 / HDIT_EPI_OUT_F32): a lane's 8 columns
      // are then 32 bytes, moved as two 16-byte accesses.
      const bool rf32 = GATED && (pr.epilogue & HDIT_EPI_RESID_F32) != 0;
      const bool of32 = GATED && (pr.epilogue & HDIT_EPI_OUT_F32) != 0;
      i32x4 rres[8], rres_hi[GATED ? 8 : 1];
      f32x4 gte0, gte1;
      bool straddle = false;
      auto prefetch_rows = [&](int i, int half) {
        const int mrow0 = tc.m0 + wm0 + i * 32;
#pragma unroll
        for (int it = half * 4; it < half * 4 + 4; it++) {
          const int mm = min(mrow0 + it * 4 + wr_row, M - 1);
          if (rf32) {
            const unsigned char* rp = Rb + (unsigned)((mm * ldr + wr_nc) * 4);
            rres[it] = *(const i32x4*)rp;
            rres_hi[GATED ? it : 0] = *(const i32x4*)(rp + 16);
          } else {
            rres[it] = *(const i32x4*)(Rb + (unsigned)((mm * ldr + wr_nc) * 2));
          }
        }
      };
      auto prefetch_gate = [&](int i) {
        const int mrow0 = tc.m0 + wm0 + i * 32;
        const int b_lo = min(mrow0, M - 1) / pr.rows_per_batch;
        straddle = min(mrow0 + 31, M - 1) >= (b_lo + 1) * pr.rows_per_batch;
        const float* g = gate + (int64_t)b_lo * pr.gate_stride + wr_nc;
        gte0 = *(const f32x4*)g;
        gte1 = *(const f32x4*)(g + 4);
      };
      {
        // bias of the next tile of this workgroup (this tile's is inside its accumulators: see the tile start)
        const int next_lid = lid + wgs_per_xcd;
        if (next_lid < xcd_end) fetch_bias(locate<C>(tab, next_lid));
      }
      if (GATED) {
        prefetch_rows(0, 0);
        prefetch_rows(0, 1);
        prefetch_gate(0);
      }

      typedef __attribute__((address_space(3))) i32x4 lds_i32x4;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const int mrow0 = tc.m0 + wm0 + i * 32;
        // Staging addresses: the XOR swizzle only touches bits 4-7, which are zero in the 256-byte aligned row
        // base, so slot (chunk ^ (row & 15)) of a row is (row base + ((row & 15) << 4)) ^ (chunk << 4): one register
        // and one v_xor per access, made opaque per block so that the sixteen write and eight read addresses are not
        // computed ahead and spilled.
        unsigned wa = lds_address(epi) + l16 * 256 + (l16 << 4);
        unsigned ra = lds_address(epi) + wr_row * 256 + ((rchunk ^ wr_row) << 4);
        asm volatile("" : "+v"(wa), "+v"(ra));
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
          for (int mi = 0; mi < 2; mi++) {
            // The accumulators of column blocks 2j (even) and 2j+1 (odd) hold columns 4*lg + e.  The swap exchanges
            // the odd 16-lane rows of the first with the even ones of the second: lanes of group 0 and 2 then own
            // columns 0..7 and 8..15 of the even block, those of group 1 and 3 the same columns of the odd one.
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; e++) {
              auto sw = __builtin_amdgcn_permlane16_swap(__float_as_int(acc[2 * i + mi][2 * j][e]),
                                                         __float_as_int(acc[2 * i + mi][2 * j + 1][e]), false, false);
              v[e] = __int_as_float(sw[0]);
              v[4 + e] = __int_as_float(sw[1]);
            }
            const int chunk = j * 4 + ((lg & 1) << 1) + (lg >> 1);  // 16-byte chunk inside the wave's 256-byte row
            if (MODE == HDIT_EPI_BIAS_GELU) {
#pragma unroll
              for (int e = 0; e < 8; e++) v[e] = hdit::gelu_tanh_f(v[e]);
            }
            *(lds_i32x4*)(uintptr_t)((wa ^ (unsigned)(chunk << 4)) + mi * 16 * 256) = hdit::pack8(v);
          }
          SCHED_FENCE();  // keeps the scheduler from pulling whole accumulator tiles into VGPRs at once
        }
        // coalesced write-back of this 32 x (32*TN) block
#pragma unroll
        for (int half = 0; half < 2; half++) {
          i32x4 outv[4], outv_hi[GATED ? 4 : 1];
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int it = half * 4 + q;
            const int r = it * 4 + wr_row;
            // row r = 4 it + wr_row: slot rchunk ^ (r & 15) = (rchunk ^ wr_row) ^ 4 (it & 3)
            i32x4 val = *(const lds_i32x4*)(uintptr_t)((ra ^ (unsigned)(((it & 3) * 4) << 4)) + it * 1024);
            if (GATED) {
              f32x4 g0 = gte0, g1 = gte1;
              if (straddle) {  // rows of this block belong to different batch elements: fetch the gate per row
                const int mm = min(mrow0 + r, M - 1);
                const float* g = gate + (int64_t)(mm / pr.rows_per_batch) * pr.gate_stride + wr_nc;
                g0 = *(const f32x4*)g;
                g1 = *(const f32x4*)(g + 4);
              }
              float u[8], rf[8];
              hdit::unpack8(val, u);
              if (rf32) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                  rf[e] = __int_as_float(rres[it][e]);
                  rf[4 + e] = __int_as_float(rres_hi[GATED ? it : 0][e]);
                }
              } else {
                hdit::unpack8(rres[it], rf);
              }
#pragma unroll
              for (int e = 0; e < 4; e++) {
                u[e] = __builtin_fmaf(g0[e], u[e], rf[e]);
                u[4 + e] = __builtin_fmaf(g1[e], u[4 + e], rf[4 + e]);
              }
              if (of32) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                  val[e] = __float_as_int(u[e]);
                  outv_hi[GATED ? q : 0][e] = __float_as_int(u[4 + e]);
                }
              } else {
                val = hdit::pack8(u);
              }
            }
            outv[q] = val;
          }
          SCHED_FENCE();
          if (GATED && i + 1 < TM) {
            prefetch_rows(i + 1, half);
            if (half == 1) prefetch_gate(i + 1);
          }
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int mm = mrow0 + (half * 4 + q) * 4 + wr_row;
            if (wr_ok && mm < M) {
              if (of32) {
                unsigned char* cp = Cb + (unsigned)((mm * ldc + wr_n) * 4);
                *(i32x4*)cp = outv[q];
                *(i32x4*)(cp + 16) = outv_hi[GATED ? q : 0];
              } else {
                *(i32x4*)(Cb + (unsigned)((mm * ldc + wr_n) * 2)) = outv[q];
              }
            }
          }
          SCHED_FENCE();
        }
      }
    };
    if ((pr.epilogue & HDIT_EPI_MODE_MASK) == HDIT_EPI_BIAS) epilogue(std::integral_constant<int, HDIT_EPI_BIAS>{});
    else if ((pr.epilogue & HDIT_EPI_MODE_MASK) == HDIT_EPI_BIAS_GELU) epilogue(std::integral_constant<int, HDIT_EPI_BIAS_GELU>{});
    else epilogue(std::integral_constant<int, HDIT_EPI_GATE_RESIDUAL>{});

    // Leave nothing of the epilogue in flight.  The compiler's bookkeeping of pending loads is path-insensitive:
    // one epilogue load it believes may still be pending makes it place a small vmcnt wait where the main loop
    // first reuses that register, and that wait drains the operand stream on every slab (the direct-to-LDS
    // requests are invisible to it, and the register-staged loads of the slab after next are younger).
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    lid += wgs_per_xcd;
    if (lid >= xcd_end) break;
  }
  // requests past the end of the stream are still in flight: nothing may land in LDS after this returns
  if constexpr (C::DIRECT) __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
}

// A launch with fewer tiles than CUs is bound by the latency of its weights, which come from HBM (every layer's are read
// once per pass): a CU has at most its LDS in flight, 128 KiB / 2 us.  So CUs without a tile -- up to four per XCD, which
// is enough to keep HBM busy and leaves room for another stream's launch -- run ahead and bring the weights into the
// last-level cache.  Measured, weights cold: 1357 x 1536 x 6144 on 132 tiles of 128 x 128 59.3 us without helpers, 47.5
// with two per XCD, 43.9 with four, 43.9 with eight; 1536 x 3072 x 15360 on 192 tiles of 128 x 192 170, 149, 148, 152;
// 333 x 1536 x 6144 on 144 tiles of 64 x 64 31.9, 31.9, 26.6, 24.4.  Only where they are done before the tiles
// (`build_and_launch`).
constexpr int HELPERS_PER_XCD = 4;

// A workgroup without tiles: helper `id` of `helpers` reads one word of every 128-byte line of a weight matrix, four
// slabs of all its rows at a time, so that the slabs behind the first few come from the last-level cache.
__device__ __forceinline__ void fetch_weights(const GemmTable& tab, int id, int helpers) {
  // the helpers are dealt to the problems, whose tiles run side by side
  const int pi = id % tab.count;
  const int of_problem = (helpers - pi + tab.count - 1) / tab.count;
  const hdit_gemm_problem& pr = tab.p[pi];
  const unsigned char* base = (const unsigned char*)pr.b;
  const unsigned KT = (unsigned)pr.k / BK, n = (unsigned)pr.n, pitch = (unsigned)pr.ldb * 2u;
  const unsigned per_chunk = 4u * n, total = (KT + 3) / 4 * per_chunk, step = (unsigned)of_problem * NT;
  constexpr int U = 8;
  for (unsigned u0 = (unsigned)(id / tab.count) * NT + threadIdx.x; u0 < total; u0 += U * step) {
    unsigned v[U];
#pragma unroll
    for (int i = 0; i < U; i++) {
      const unsigned u = min(u0 + i * step, total - 1);
      const unsigned chunk = u / per_chunk, r = u - chunk * per_chunk;
      const unsigned line = min(chunk * 4 + (r & 3), KT - 1);
      v[i] = *(const unsigned*)(base + (uint64_t)((r >> 2) * pitch) + line * ROW_BYTES);
    }
#pragma unroll
    for (int i = 0; i < U; i++) asm volatile("" : : "v"(v[i]));
  }
}

template <class C>
__global__ void __launch_bounds__(NT) gemm_kernel(const GemmTable tab, int total_tiles, int tiles_per_xcd,
                                                  int wgs_per_xcd) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int wg = blockIdx.x / NUM_XCD;
  if (wg >= wgs_per_xcd) {  // uniform over the workgroup
    fetch_weights(tab, blockIdx.x - wgs_per_xcd * NUM_XCD, gridDim.x - wgs_per_xcd * NUM_XCD);
    return;
  }
  run_tiles<C>(tab, total_tiles, tiles_per_xcd, wgs_per_xcd, wg, lds);
}

// Two tile shapes in one launch: the large tiles of the tall problems first, then the small tiles of the
// short ones (the text stream of a joint block), which a workgroup starts as soon as its large tiles are
// done: no second launch, and the small tiles fill the tail of the large ones.
template <class C1, class C2>
__global__ void __launch_bounds__(NT) gemm_kernel2(const GemmTable tab1, int total1, int per_xcd1, const GemmTable tab2,
                                                   int total2, int per_xcd2, int wgs_per_xcd) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int wg = blockIdx.x / NUM_XCD;
  run_tiles<C1>(tab1, total1, per_xcd1, wgs_per_xcd, wg, lds);
  __syncthreads();  // the second phase reuses the LDS of the first
  // the small tiles are dealt from the first workgroup on that has no tile in the last round of large ones
  const int xcd = blockIdx.x % NUM_XCD;
  const int own1 = max(min(per_xcd1, total1 - xcd * per_xcd1), 0);
  const int first = own1 % wgs_per_xcd;
  run_tiles<C2>(tab2, total2, per_xcd2, wgs_per_xcd, wg >= first ? wg - first : wg - first + wgs_per_xcd, lds);
}

std::atomic<int> g_num_cus{0};

int max_workgroups() {
  if (g_num_cus.load(std::memory_order_acquire) == 0) {
    int dev = 0, n = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) {
      hdit_host::set_error(hipGetErrorString(e));
      return -1;
    }
    g_num_cus.store(n, std::memory_order_release);
  }
  int max_wgs = g_num_cus.load(std::memory_order_relaxed) / NUM_XCD * NUM_XCD;  // one workgroup per CU: a wave may use the whole register file
  return max_wgs < NUM_XCD ? NUM_XCD : max_wgs;
}

// helper_us: how long each helper of an XCD's `n` works, n = 1 .. HELPERS_PER_XCD; tiles_us: how long the tiles take
template <class C>
int launch(const GemmTable& tab, int total_tiles, const double* helper_us, double tiles_us, hipStream_t stream) {
  static std::atomic<bool> attr_set{false};  // setting the attribute twice from two threads is harmless
  if (!attr_set.load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_kernel<C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    if (e != hipSuccess) {
      hdit_host::set_error(hipGetErrorString(e));
      return HDIT_ELAUNCH;
    }
    attr_set.store(true, std::memory_order_release);
  }
  const int max_wgs = max_workgroups();
  if (max_wgs < 0) return HDIT_ELAUNCH;
  const int tiles_per_xcd = (total_tiles + NUM_XCD - 1) / NUM_XCD;
  int wgs_per_xcd = max_wgs / NUM_XCD;
  // workgroups without a tile beside those with one, if they are done before the tiles
  int helpers = wgs_per_xcd - tiles_per_xcd;
  if (helpers > HELPERS_PER_XCD) helpers = HELPERS_PER_XCD;
  if (helpers <= 0 || helper_us[helpers - 1] > tiles_us) helpers = 0;
  if (wgs_per_xcd > tiles_per_xcd) wgs_per_xcd = tiles_per_xcd;
  hipLaunchKernelGGL(gemm_kernel<C>, dim3((wgs_per_xcd + helpers) * NUM_XCD), dim3(NT), C::LDS_BYTES, stream, tab, total_tiles,
                     tiles_per_xcd, wgs_per_xcd);
  return hdit_host::check_launch("hdit_gemm_bf16");
}

template <class C>
int fill_table(GemmTable& tab, const hdit_gemm_problem* problems, int count) {
  tab.count = count;
  int total = 0;
  for (int i = 0; i < count; i++) {
    tab.p[i] = problems[i];
    tab.tile_start[i] = total;
    total += ((problems[i].m + C::BM - 1) / C::BM) * ((problems[i].n + C::BN - 1) / C::BN);
  }
  for (int i = count; i <= HDIT_GEMM_MAX_PROBLEMS; i++) tab.tile_start[i] = total;
  return total;
}

template <class C1, class C2>
int launch2(const hdit_gemm_problem* p1, int n1, const hdit_gemm_problem* p2, int n2, hipStream_t stream) {
  constexpr int LDS = C1::LDS_BYTES > C2::LDS_BYTES ? C1::LDS_BYTES : C2::LDS_BYTES;
  static std::atomic<bool> attr_set{false};  // setting the attribute twice from two threads is harmless
  if (!attr_set.load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_kernel2<C1, C2>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) {
      hdit_host::set_error(hipGetErrorString(e));
      return HDIT_ELAUNCH;
    }
    attr_set.store(true, std::memory_order_release);
  }
  const int max_wgs = max_workgroups();
  if (max_wgs < 0) return HDIT_ELAUNCH;
  GemmTable t1, t2;
  const int total1 = fill_table<C1>(t1, p1, n1), total2 = fill_table<C2>(t2, p2, n2);
  const int per1 = (total1 + NUM_XCD - 1) / NUM_XCD, per2 = (total2 + NUM_XCD - 1) / NUM_XCD;
  int wgs_per_xcd = max_wgs / NUM_XCD;
  const int need = per1 + per2;  // a workgroup of its own for every tile, while there are CUs
  if (wgs_per_xcd > need) wgs_per_xcd = need;
  hipLaunchKernelGGL((gemm_kernel2<C1, C2>), dim3(wgs_per_xcd * NUM_XCD), dim3(NT), LDS, stream, t1, total1, per1, t2,
                     total2, per2, wgs_per_xcd);
  return hdit_host::check_launch("hdit_gemm_bf16");
}

using Cfg256x256 = Cfg<4, 4>;
using Cfg256x192 = Cfg<4, 3>;
using Cfg128x256 = Cfg<2, 4>;
using Cfg128x128 = Cfg<2, 2>;
using Cfg128x192 = Cfg<2, 3>;
using Cfg64x128 = Cfg<1, 2>;
using Cfg64x64 = Cfg<1, 1>;
using Cfg192x192 = Cfg<3, 3>;

std::atomic<int> g_force_cfg{-1};

// ---- launch planning ---------------------------------------------------------
// A launch deals its tiles to 256 workgroups (one per CU) in rounds; a tile costs (k / 64) slab times plus an epilogue
// with the fill of the pipeline.  Both depend on how many CUs work: a slab takes `lo` microseconds while at most half of
// them do (what the CU's requests take to come from the last-level cache) and `hi` while all do (the chip's power budget
// is shared), in between in between.  All figures fitted to MI355X times with weights that come from HBM: 300 random launches
// of the models' sizes (one or two problems, 64 - 17000 rows, N = 1536 - 21504, K = 1536 - 15360) under every shape; the
// model reproduces those launches within 4 - 10 % and its choice among the shapes is on average 0.1 % slower than the best
// of them (at most 4 %).  192 x 192 is there for what lies between the others: an eighth of those launches take it and are
// 5 % faster by it (2333+333 x 6144 x 1536 and 5523+333 x 1536 x 6144 11 %).
//
// What a plan has to get right is the last round.  One tile shape for everything wastes most of it: the 666-row text
// stream of a joint block on the image stream's 256-row tiles adds a nearly empty round, and 17 550 rows x 3072 columns
// are 828 tiles of 256 x 256, three rounds and 60 tiles (K = 12288: 1249 us on the 128 x 256 tiles that a model without
// `lo` preferred, 1076 us on 256 x 256, 1004 us on 768 tiles of 256 x 256 and 240 of 128 x 128).  So besides every single shape the planner prices launches of two shapes, the large tiles
// first: problems dealt to the shape that suits them, and the whole call on large tiles except the rows at the end of
// its tallest problem that would open another round; those take the small shape.
// Results do not depend on any of this (every shape forms the same sums in the same order).
struct Shape {
  int bm, bn;
  double lo, hi, epi_lo, epi_hi;
};
constexpr int NCFG = 8;
constexpr Shape kShape[NCFG] = {
    {256, 192, 0.763, 1.086, 4.7, 5.4}, {128, 256, 0.649, 0.840, 3.5, 4.6}, {128, 128, 0.358, 0.480, 2.9, 3.3},
    {256, 256, 0.979, 1.369, 5.4, 6.8}, {128, 192, 0.453, 0.638, 3.7, 3.8}, {64, 128, 0.270, 0.329, 1.6, 2.2},
    {64, 64, 0.211, 0.219, 0.4, 1.3},   {192, 192, 0.625, 0.904, 3.9, 4.5},
};
constexpr double kLaunchUs = 4.0;
constexpr int kSlots = 256;

int tiles_of(const hdit_gemm_problem& p, int c) {
  return ((p.m + kShape[c].bm - 1) / kShape[c].bm) * ((p.n + kShape[c].bn - 1) / kShape[c].bn);
}

struct Load {  // the tiles of some problems under one shape
  int tiles = 0;
  double slabs = 0;    // per tile, on average
  double cold_us = 0;  // per tile, on average: what its slabs take longer because few tiles share the weights
};

// Weights that one or two rows of tiles read come from HBM for a single CU or two, and every slab waits for that where no
// helper has fetched them: measured 0.2 - 0.3 us and 0.1 us more per slab, whatever the shape.  Merged patches of few rows,
// 4 x 146 rows x 6144 x 1536 with weights of their own: 128 tiles of 192 x 192, priced at 22.9 us, take 30.7, 256 tiles of 128 x
// 192 26.1; 2 x 162 x 12288 x 3072 53.0 and 44.0.
constexpr double kColdUs[2] = {0.20, 0.08};
constexpr int kHelpedTiles = 240;  // ring shapes, up to this many tiles: helpers fetch the weights (fetch_weights)

bool is_ring(int c) { return kShape[c].bm * kShape[c].bn <= RING_MAX_MMA * 64 * 64; }

Load load_of(const hdit_gemm_problem* ps, int count, int c) {
  Load l;
  for (int i = 0; i < count; i++) {
    const int t = tiles_of(ps[i], c);
    l.tiles += t;
    l.slabs += (double)t * (ps[i].k / BK);
    int sharing = 0;  // rows of tiles that read these weights
    for (int j = 0; j < count; j++)
      if (ps[j].b == ps[i].b) sharing += (ps[j].m + kShape[c].bm - 1) / kShape[c].bm;
    if (sharing > 0 && sharing <= 2) l.cold_us += (double)t * (ps[i].k / BK) * kColdUs[sharing - 1];
  }
  if (l.tiles) l.slabs /= l.tiles, l.cold_us /= l.tiles;
  if (is_ring(c) && l.tiles <= kHelpedTiles) l.cold_us = 0;
  return l;
}

// one tile of shape c while `busy` of the 256 CUs work on such tiles
double tile_us(int c, double slabs, int busy) {
  const double f = busy >= kSlots ? 1.0 : busy > kSlots / 2 ? 2.0 * busy / kSlots - 1.0 : 0.0;
  const Shape& s = kShape[c];
  return slabs * (s.lo + (s.hi - s.lo) * f) + s.epi_lo + (s.epi_hi - s.epi_lo) * f;
}
double tile_us(int c, const Load& l, int busy) { return tile_us(c, l.slabs, busy) + l.cold_us; }

// A partial round behind full ones has no helpers beside it, and without them the slabs of the ring shapes take as long as
// on a full chip (274 + 295 rows x 12288 x 3072: 384 tiles of 128 x 192 76 us, priced at 66 with `lo`; 256 of 256 x 192 61).
double single_us(const Load& l, int c) {
  const int full = l.tiles / kSlots, rem = l.tiles % kSlots;
  return full * tile_us(c, l, kSlots) + (rem ? tile_us(c, l, full && is_ring(c) ? kSlots : rem) : 0.0);
}

// Tiles of c1, then tiles of c2 in the same launch: the small tiles go first to the workgroups that have one large tile
// fewer (see gemm_kernel2).
double two_us(const Load& l1, int c1, const Load& l2, int c2) {
  if (l1.tiles == 0) return single_us(l2, c2);
  if (l2.tiles == 0) return single_us(l1, c1);
  const int full = l1.tiles / kSlots, rem = l1.tiles % kSlots;
  const int idle = rem ? kSlots - rem : 0;  // workgroups without a tile of the last large round
  const int base = l2.tiles / kSlots, extra = l2.tiles % kSlots;
  const int busy = rem + l2.tiles;  // CUs at work in the last round
  const double t1 = full * tile_us(c1, l1, kSlots), t1_last = rem ? tile_us(c1, l1, busy) : 0.0;
  const double t2 = tile_us(c2, l2, busy);
  const double of_idle = t1 + (base + (extra > 0 ? 1 : 0)) * t2;
  const double of_rest = t1 + t1_last + (base + (extra > idle ? 1 : 0)) * t2;
  return idle && of_idle > of_rest ? of_idle : of_rest;
}

// One shape for all problems.  A helper that is still fetching when the last tile is done holds the launch up: on 240
// tiles two per XCD are left, which bring in 80 GB/s each (75 - 98 measured).  649 + 430 rows x 12288 x 3072, 151 MB of
// weights: 126 us with them, 76 without; 883 + 183 x 9216 x 3072 86 and 60; 250 + 292 x 6144 x 1536 28 and 22.
constexpr double kHelperBytesPerUs = 80e3;

template <class C>
int build_and_launch(int cfg, const hdit_gemm_problem* problems, int count, hipStream_t stream) {
  GemmTable tab;
  const int total = fill_table<C>(tab, problems, count);
  if (total == 0) return HDIT_OK;
  double helper_us[HELPERS_PER_XCD] = {}, slabs = 0;
  for (int i = 0; i < count; i++) {
    if (problems[i].k / BK > slabs) slabs = problems[i].k / BK;
    for (int h = 1; h <= HELPERS_PER_XCD; h++) {
      const int of_problem = (h * NUM_XCD - i + count - 1) / count;  // as fetch_weights deals them
      const double us = of_problem > 0 ? 2.0 * problems[i].n * problems[i].k / (of_problem * kHelperBytesPerUs) : 0.0;
      if (us > helper_us[h - 1]) helper_us[h - 1] = us;
    }
  }
  return launch<C>(tab, total, helper_us, tile_us(cfg, slabs, total), stream);
}

int launch_cfg(int cfg, const hdit_gemm_problem* problems, int count, hipStream_t s) {
  switch (cfg) {
    case 0: return build_and_launch<Cfg256x192>(cfg, problems, count, s);
    case 1: return build_and_launch<Cfg128x256>(cfg, problems, count, s);
    case 4: return build_and_launch<Cfg128x192>(cfg, problems, count, s);
    case 3: return build_and_launch<Cfg256x256>(cfg, problems, count, s);
    case 5: return build_and_launch<Cfg64x128>(cfg, problems, count, s);
    case 6: return build_and_launch<Cfg64x64>(cfg, problems, count, s);
    case 7: return build_and_launch<Cfg192x192>(cfg, problems, count, s);
    default: return build_and_launch<Cfg128x128>(2, problems, count, s);
  }
}

// The problems of a call that have rows, checked.
int live_problems(const hdit_gemm_problem* problems, int count, hdit_gemm_problem* live, int& nlive) {
  if (!problems || count < 0 || count > HDIT_GEMM_MAX_PROBLEMS) return HDIT_EINVAL;
  nlive = 0;
  for (int i = 0; i < count; i++) {
    const hdit_gemm_problem& p = problems[i];
    if (p.m < 0 || p.n <= 0 || p.k <= 0) return HDIT_EINVAL;
    if (p.m == 0) continue;
    if (!p.a || !p.b || !p.c) return HDIT_EINVAL;
    if (p.k % BK != 0 || p.n % 8 != 0) return HDIT_EUNSUPPORTED;
    if (p.lda % 8 || p.ldb % 8 || p.ldc % 8) return HDIT_EINVAL;
    if (((uintptr_t)p.a | (uintptr_t)p.b | (uintptr_t)p.c | (uintptr_t)p.bias) & 15) return HDIT_EINVAL;
    // rows are addressed with 32-bit byte offsets from the operand base
    if ((int64_t)p.m * p.lda * 2 >= (1ll << 32) || (int64_t)p.n * p.ldb * 2 >= (1ll << 32)) return HDIT_EUNSUPPORTED;
    const int mode = p.epilogue & HDIT_EPI_MODE_MASK;
    const int c_bytes = (p.epilogue & HDIT_EPI_OUT_F32) ? 4 : 2, r_bytes = (p.epilogue & HDIT_EPI_RESID_F32) ? 4 : 2;
    if (p.epilogue & ~(HDIT_EPI_MODE_MASK | HDIT_EPI_RESID_F32 | HDIT_EPI_OUT_F32)) return HDIT_EINVAL;
    if (mode > HDIT_EPI_GATE_RESIDUAL) return HDIT_EINVAL;
    // the fp32 residual stream only exists in the gated-residual epilogue
    if (mode != HDIT_EPI_GATE_RESIDUAL && (p.epilogue & (HDIT_EPI_RESID_F32 | HDIT_EPI_OUT_F32))) return HDIT_EINVAL;
    if ((int64_t)p.m * p.ldc * c_bytes >= (1ll << 31)) return HDIT_EUNSUPPORTED;
    if (mode == HDIT_EPI_GATE_RESIDUAL) {
      if (!p.resid || !p.gate || p.rows_per_batch <= 0 || p.ldr % 8) return HDIT_EINVAL;
      if ((int64_t)p.m * p.ldr * r_bytes >= (1ll << 31)) return HDIT_EUNSUPPORTED;
      if (((uintptr_t)p.resid & 15) || ((uintptr_t)p.gate & 15) || p.gate_stride % 4) return HDIT_EINVAL;
    }
    live[nlive++] = p;
  }
  return HDIT_OK;
}

struct Plan {  // one shape for everything, or (two_cost < single_cost) two: large tiles and small ones
  int single = 0, big_cfg = 3, small_cfg = 2, nb = 0, ns = 0;
  double single_cost = 1e30, two_cost = 1e30;
  hdit_gemm_problem big[HDIT_GEMM_MAX_PROBLEMS + 1], small[HDIT_GEMM_MAX_PROBLEMS + 1];
};

void make_plan(const hdit_gemm_problem* live, int nlive, Plan& plan) {
  int &single = plan.single, &big_cfg = plan.big_cfg, &small_cfg = plan.small_cfg, &nb = plan.nb, &ns = plan.ns;
  double &single_cost = plan.single_cost, &two_cost = plan.two_cost;
  hdit_gemm_problem *const big = plan.big, *const small = plan.small;
  for (int c = 0; c < NCFG; c++) {
    const double t = single_us(load_of(live, nlive, c), c);
    if (t < single_cost) single_cost = t, single = c;
  }
  // two shapes, large tiles of 256 rows (c1) and small ones of 128 (c2)
  for (const int c1 : {3, 0}) {
    for (const int c2 : {2, 1}) {
      // (a) every problem where it is cheaper on its own
      hdit_gemm_problem b[HDIT_GEMM_MAX_PROBLEMS + 1], m[HDIT_GEMM_MAX_PROBLEMS + 1];
      int kb = 0, km = 0;
      for (int i = 0; i < nlive; i++) {
        const bool large = single_us(load_of(&live[i], 1, c1), c1) <= single_us(load_of(&live[i], 1, c2), c2);
        (large ? b[kb++] : m[km++]) = live[i];
      }
      // (large tiles that do not fill one round are better off alone, on whichever shape: 4316+154 x 1536 x 6144 as 136
      // tiles of 256 x 192 and 24 of 128 x 128 takes 97 us, all on 256 x 192 88, all on 128 x 256 83; 8192+666 x 1536 x
      // 6144 136 us against 130 on 256 x 256)
      const bool round = load_of(b, kb, c1).tiles >= kSlots;
      double t = two_us(load_of(b, kb, c1), c1, load_of(m, km, c2), c2);
      if (round && km && t < two_cost) {
        two_cost = t, big_cfg = c1, small_cfg = c2, nb = kb, ns = km;
        memcpy(big, b, kb * sizeof(*b));
        memcpy(small, m, km * sizeof(*m));
      }
      // (b) and (c): the problems that (a) gives large tiles, or all of them, except the rows that open another round
      for (int all = 0; all < 2; all++) {
        if (all) {
          for (int i = 0; i < km; i++) b[kb++] = m[i];
          km = 0;
        }
        const int excess = load_of(b, kb, c1).tiles % kSlots;
        int tall = 0;
        for (int i = 1; i < kb; i++)
          if (b[i].m > b[tall].m) tall = i;
        if (kb == 0 || excess == 0 || load_of(b, kb, c1).tiles < kSlots) continue;
        if (km >= HDIT_GEMM_MAX_PROBLEMS) continue;  // the table of the small tiles is full
        const int tiles_n = (b[tall].n + kShape[c1].bn - 1) / kShape[c1].bn;
        const int blocks = (b[tall].m + kShape[c1].bm - 1) / kShape[c1].bm;
        const int keep = blocks - (excess + tiles_n - 1) / tiles_n;
        // a gate per batch element is looked up by the row within the problem: only one batch element can be split
        const bool gated = (b[tall].epilogue & HDIT_EPI_MODE_MASK) == HDIT_EPI_GATE_RESIDUAL;
        if (keep <= 0 || (gated && b[tall].m > b[tall].rows_per_batch)) continue;
        const hdit_gemm_problem whole = b[tall];
        const int64_t r0 = (int64_t)keep * kShape[c1].bm;
        hdit_gemm_problem rest = whole;
        rest.m = whole.m - (int)r0;
        rest.a = (const char*)whole.a + r0 * whole.lda * 2;
        rest.c = (char*)whole.c + r0 * whole.ldc * ((whole.epilogue & HDIT_EPI_OUT_F32) ? 4 : 2);
        if (gated) rest.resid = (const char*)whole.resid + r0 * whole.ldr * ((whole.epilogue & HDIT_EPI_RESID_F32) ? 4 : 2);
        b[tall].m = (int)r0;
        m[km] = rest;
        t = two_us(load_of(b, kb, c1), c1, load_of(m, km + 1, c2), c2);
        if (t < two_cost) {
          two_cost = t, big_cfg = c1, small_cfg = c2, nb = kb, ns = km + 1;
          memcpy(big, b, kb * sizeof(*b));
          memcpy(small, m, (km + 1) * sizeof(*m));
        }
        b[tall] = whole;
      }
    }
  }
  static const bool debug = getenv("HDIT_GEMM_DEBUG") != nullptr;
  if (debug) {
    fprintf(stderr, "hdit_gemm_bf16 plan:");
    for (int i = 0; i < nlive; i++) fprintf(stderr, " [%dx%dx%d epi%d]", live[i].m, live[i].n, live[i].k, live[i].epilogue);
    fprintf(stderr, " single cfg%d %.1f us, two-shape(big cfg%d %d tiles, small cfg%d %d tiles) %.1f us\n", single,
            single_cost + kLaunchUs, big_cfg, load_of(big, nb, big_cfg).tiles, small_cfg, load_of(small, ns, small_cfg).tiles,
            two_cost + kLaunchUs);
  }
}

}  // namespace

extern "C" __attribute__((visibility("default"))) void hdit_gemm_force_config(int cfg) { g_force_cfg.store(cfg, std::memory_order_relaxed); }

extern "C" __attribute__((visibility("default"))) int hdit_gemm_plan(const hdit_gemm_problem* problems, int count) {
  hdit_gemm_problem live[HDIT_GEMM_MAX_PROBLEMS];
  int nlive = 0;
  const int rc = live_problems(problems, count, live, nlive);
  if (rc != HDIT_OK) return rc;
  if (nlive == 0) return HDIT_EINVAL;
  Plan plan;
  make_plan(live, nlive, plan);
  return plan.two_cost < plan.single_cost ? 16 * (1 + plan.big_cfg) + plan.small_cfg : plan.single;
}

extern "C" __attribute__((visibility("default"))) int hdit_gemm_bf16(const hdit_gemm_problem* problems, int count, void* stream) {
  hdit_gemm_problem live[HDIT_GEMM_MAX_PROBLEMS];
  int nlive = 0;
  const int rc = live_problems(problems, count, live, nlive);
  if (rc != HDIT_OK || nlive == 0) return rc;
  hipStream_t s = (hipStream_t)stream;
  const int forced = g_force_cfg.load(std::memory_order_relaxed);
  if (forced >= 0) return launch_cfg(forced, live, nlive, s);
  Plan plan;
  make_plan(live, nlive, plan);
  if (plan.two_cost < plan.single_cost) {
    const hdit_gemm_problem *big = plan.big, *small = plan.small;
    const int nb = plan.nb, ns = plan.ns;
    if (plan.big_cfg == 0 && plan.small_cfg == 2) return launch2<Cfg256x192, Cfg128x128>(big, nb, small, ns, s);
    if (plan.big_cfg == 0) return launch2<Cfg256x192, Cfg128x256>(big, nb, small, ns, s);
    if (plan.small_cfg == 2) return launch2<Cfg256x256, Cfg128x128>(big, nb, small, ns, s);
    return launch2<Cfg256x256, Cfg128x256>(big, nb, small, ns, s);
  }
  return launch_cfg(plan.single, live, nlive, s);
}
