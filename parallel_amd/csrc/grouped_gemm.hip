// Grouped bf16 GEMMs for the MoE expert path on gfx950 (MI355X).
//
// One kernel template covers the three contraction shapes of an expert layer:
//   MG / B K-contiguous   forward      c[r,n]   = sum_k a[r,k] w[g][n,k]
//   MG / B N-contiguous   input grad   da[r,n]  = sum_k dc[r,k] w[g][k,n]
//   KG                    weight grad  dw[g][m,n] = sum_{r in g} dc[r,m] a[r,n]
// MG = groups partition the rows of the activation operand (variable M per
// expert), KG = groups partition the reduction (variable K per expert).
//
// Tiling: WM x WN waves; each wave owns (BM/WM) x (BN/WN) of 32x32 sub-tiles,
// its row sub-tiles interleaved with the other wave rows'.  The products are
// v_mfma_f32_16x16x32_bf16 (four per sub-tile and 32 k, fp32 accumulators), but
// the weight gradients' v_mfma_f32_32x32x16_bf16 (the same bits).  On random
// data the others run against the card's power limit, and the 16x16x32
// shape reads and writes each accumulator once per 32 k where 32x32x16 does
// once per 16 (65536 x 3072 x 4096 over 128 experts 1387 us on random data, 1108
// on zeros; 1528 on random data with 32x32x16).  The expert GEMMs use
// 256-column tiles of 64 to 320 rows, by the mean rows per expert and by how
// many tiles run at once, on 8 waves (two waves per SIMD, one workgroup per CU);
// the small router GEMMs use 128x128 on 4 waves.  Operands move from HBM to LDS
// by DMA (buffer_load_dwordx4 ... lds, no register staging) into a ring of 32-
// or 64-deep k-tiles that fills the 160 KiB of LDS, so that 64 to 96 KiB of
// loads are in flight while one k-tile is multiplied; each wave fires its share
// of a k-tile's DMA between its MFMA groups.  At the roughly 256 rows per expert
// of a training step the expert GEMMs sit near the ridge of the roofline (about
// 256 flop per weight byte), and the weights stream from HBM only as fast as the
// bytes in flight per CU allow, so the ring takes all of the LDS: the epilogue
// stages its output through the ring stage it has just multiplied.  Each operand
// keeps its HBM layout in LDS (XOR swizzled): K-contiguous fragments are
// ds_read_b128, M/N-contiguous ones (weights in the input gradient, both
// operands of the weight gradient) are ds_read_b64_tr_b16 transpose reads.
// Buffer loads read zero past the resource size, so ragged rows and the K
// tail need no branches.  Row sub-tiles that lie wholly outside the valid
// rows skip their MFMAs (an expert's rows are split evenly over its m-tiles,
// so most m-tiles are partly filled).
//
// Tiles are mapped to groups on the device from the `offs` cumsum (no host
// sync).  The logical tile order is group-major, then n-tile, then m-tile, so
// consecutive tiles share an expert's weight tile and its activation rows;
// the launch index is remapped so that each XCD (blocks are dealt round-robin
// over the 8 XCDs) gets a contiguous run of logical tiles and the sharing
// happens in that XCD's L2.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "dma.h"
#include "gemm.h"

namespace moe {

enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_SWIGLU_FWD = 2, EPI_WGRAD = 4 };
enum { MODE_MG = 0, MODE_KG = 1 };

constexpr int kNumXcd = 8;

struct GemmParams {
  const bf16_t* A;  // MG: [rows, K] (lda);  KG: [rows, M] (lda)
  const bf16_t* B;  // MG: per group (stride_bg) [N, K] or [K, N] (ldb);  KG: [rows, N] (ldb)
  void* C;          // MG: [rows, ldc];  KG: per group (stride_cg) [M, N] (ldc)
  void* C2;         // SWIGLU_FWD: pre-activation [rows, 2N] (may be null)
  const int32_t* offs;
  int G;
  int rows;     // total activation rows (M for MG; sum of K for KG)
  int M, N, K;  // GEMM-internal sizes: MG: M = rows, N out cols, K reduction; KG: M x N output per group
  int64_t lda, ldb, ldc, ldp;
  int64_t stride_bg, stride_cg;
  uint32_t a_bytes;  // bytes addressable through the A buffer resource
  uint32_t b_bytes;  // bytes of one group's B (MG) or of all of B (KG)
  uint32_t c_bytes;  // bytes of the output: all of C (MG), one group's (KG) or one split's (split-K)
  uint32_t c2_bytes;  // SWIGLU_FWD: bytes of the pre-activation output (0 if none)
  int swiglu_I;      // SWIGLU_FWD: intermediate size I (weight rows gate: [0,I), up: [I,2I))
  int accumulate;
  int n_tiles, m_tiles_max;
  int total_tiles;     // exact tile count (grouped MG: worst case; the kernel counts the real ones)
  int k_splits, k_chunk;  // MG without groups: split the reduction, partial outputs stacked
  int64_t split_stride;   // elements between split partials of C
  int chunk_rows;         // KG without offs and G > 1: group g = rows [g*chunk_rows, ...)
  // KG into a rank-major bucket (0 = plain): group g's output starts
  // (g / bucket_rows) * bucket_stride + (g % bucket_rows) * stride_cg
  // elements into C instead of g * stride_cg.
  int bucket_rows;
  int64_t bucket_stride;
  // KG with groups: split the tiles over the XCDs by cost (k-steps plus an
  // epilogue allowance per tile) instead of by count (set by the host when
  // the costs fit in 30 bits).
  int cost_split;
};

// ---------------------------------------------------------------- helpers

// Total tiles over all groups, sum_g n_mult * ceil(cnt_g / BM) (wave-uniform).
template <int BM>
__device__ __forceinline__ int count_tiles(const int32_t* offs, int G, int rows, int n_mult) {
  const int lane = threadIdx.x & (kWave - 1);
  int total = 0;
  for (int c0 = 0; c0 < G; c0 += kWave) {
    int g = c0 + lane;
    int nt = 0;
    if (g < G) {
      int hi = min(max(offs[g], 0), rows);
      int lo = g ? min(max(offs[g - 1], 0), hi) : 0;
      nt = n_mult * ((hi - lo + BM - 1) / BM);
    }
    total += __builtin_amdgcn_readlane(wave_inclusive_scan(nt), kWave - 1);
  }
  return __builtin_amdgcn_readfirstlane(total);
}

// Weight gradients (KG): a tile of group g costs its k-steps, ceil(rows_g /
// BK), plus kEpiSteps for its epilogue.  Returns (split(part),
// split(part + 1)), split(x) being the first tile, in group-major order, whose
// cost start is at least x / kNumXcd of the total (wave-uniform): XCD x takes
// tiles [split(x), split(x + 1)).  Under skewed routing the tiles of the
// heavy experts are many times longer than the rest, and a split by count
// leaves some XCDs long tails.  Returns (-1, -1) when the costs are near
// uniform: the split by count is then as balanced and keeps whole rounds of
// tiles per block.
constexpr int kEpiSteps = 2;
template <int BK>
__device__ int2 kg_cost_split(const int32_t* offs, int G, int rows, int per_group, int part) {
  const int lane = threadIdx.x & (kWave - 1);
  auto tile_cost = [&](int g) {
    if (g >= G) return 0;
    const int hi = min(max(offs[g], 0), rows);
    const int lo = g ? min(max(offs[g - 1], 0), hi) : 0;
    return (hi - lo + BK - 1) / BK + kEpiSteps;
  };
  // Up to kCostChunks x 64 groups, every chunk's offsets are loaded at once
  // (one memory round trip at kernel start instead of one per chunk).
  constexpr int kCostChunks = 4;
  const bool cached = G <= kCostChunks * kWave;
  int tcr[kCostChunks];
#pragma unroll
  for (int c = 0; c < kCostChunks; ++c) tcr[c] = cached ? tile_cost(c * kWave + lane) : 0;
  auto chunk_cost = [&](int c0) {
    int v = 0;
#pragma unroll
    for (int c = 0; c < kCostChunks; ++c)
      if (cached && c0 == c * kWave) v = tcr[c];
    return cached ? v : tile_cost(c0 + lane);
  };
  int total = 0;
  float mx = 0.0f;  // largest tile cost
  for (int c0 = 0; c0 < G; c0 += kWave) {
    const int tc = chunk_cost(c0);
    total += __builtin_amdgcn_readlane(wave_inclusive_scan(per_group * tc), kWave - 1);
    mx = fmaxf(mx, wave_max(static_cast<float>(tc)));
  }
  // Near-uniform costs (the largest within a quarter of the mean): the split
  // by count is as balanced and keeps whole rounds of tiles per block.
  if (4.0f * mx * static_cast<float>(G) * per_group <= 5.0f * static_cast<float>(total)) return make_int2(-1, -1);
  // Both boundaries in one more pass (its loads hit the cache the first filled).
  int t_lo = static_cast<int>(static_cast<int64_t>(total) * part / kNumXcd);
  int t_hi = static_cast<int>(static_cast<int64_t>(total) * (part + 1) / kNumXcd);
  int b_lo = part <= 0 ? 0 : -1, b_hi = part + 1 >= kNumXcd ? G * per_group : -1;
  int base = 0;  // cost of the groups before this chunk
  for (int c0 = 0; c0 < G && (b_lo < 0 || b_hi < 0); c0 += kWave) {
    const int tc = chunk_cost(c0);
    const int incl = wave_inclusive_scan(per_group * tc);
    const int tot = __builtin_amdgcn_readlane(incl, kWave - 1);
    auto locate = [&](int target) {
      const int t = target - base;  // wave-uniform, and t < tot = incl[63]
      const int q = __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(incl > t)));  // first lane past t
      const int before = __builtin_amdgcn_readlane(incl - per_group * tc, q);
      const int cq = __builtin_amdgcn_readlane(tc, q);
      return (c0 + q) * per_group + min((t - before + cq - 1) / cq, per_group);
    };
    if (b_lo < 0 && t_lo - base < tot) b_lo = locate(t_lo);
    if (b_hi < 0 && t_hi - base < tot) b_hi = locate(t_hi);
    base += tot;
  }
  if (b_lo < 0) b_lo = G * per_group;
  if (b_hi < 0) b_hi = G * per_group;
  return make_int2(__builtin_amdgcn_readfirstlane(b_lo), __builtin_amdgcn_readfirstlane(b_hi));
}

// Tile configurations: BK-deep k-tiles staged through a STAGES-deep LDS ring.
// PIPE selects the k-loop:
//   0  every wave reads its fragments, multiplies and fires its share of the
//      DMA in each k-step (5-deep rings: block barrier every second k-step);
//   1  ping-pong: the two waves of a SIMD take turns, one multiplying half a
//      k-step from registers while the other reads the next half's fragments
//      and fires DMA into a ring of single operand tiles.
template <int BM_, int BN_, int BK_, int WM_, int WN_, int STAGES_, int PIPE_ = 0>
struct TileCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, STAGES = STAGES_, PIPE = PIPE_;
  static constexpr int kThreads = 64 * WM * WN;
};
// Weight gradients, and input gradients of one round of tiles: 160 KiB ring, 8 waves.
using BigTile = TileCfg<256, 256, 32, 2, 4, 5>;
// Expert GEMMs of few rows, bound by the weights' stream from HBM: 64-deep
// k-tiles (a K-contiguous weight row's 128 bytes, a whole cache line, per
// k-step) and as many weight bytes in flight as the LDS holds beside few rows:
// 96 KiB with 64-row tiles (4-deep ring of 40 KiB stages), 64 KiB with 128-row
// tiles (3-deep ring of 48 KiB), against 48 KiB with 320-row tiles.
using SlimTile = TileCfg<64, 256, 64, 2, 4, 4>;
using MidTile = TileCfg<128, 256, 64, 2, 4, 3>;
// Router GEMMs (N = E = 128): 80 KiB ring, 4 waves (two workgroups per CU).
using SmallTile = TileCfg<128, 128, 32, 2, 2, 5>;
// Experts of up to 320 rows in one m-tile: 320x256 tiles (five 32-row
// sub-tiles per wave, 160 accumulator registers per lane), A staged as 384
// rows, 4-deep ring of 40 KiB stages.
using WideTile = TileCfg<320, 256, 32, 2, 4, 4>;
// Ping-pong on 256x256 tiles, 64-deep k-steps: waves 0-3 (one per SIMD) own
// output columns 0-127, waves 4-7 columns 128-255; wave w and wave w + 4 share
// a SIMD.  The ring holds five 32 KiB operand tiles.
using PingTile = TileCfg<256, 256, 64, 2, 4, 5, 1>;

// A wave-uniform pointer moved to scalar registers (buffer resources must be).
template <class T>
__device__ __forceinline__ T* uniform_ptr(T* ptr) {
  const uint64_t v = reinterpret_cast<uint64_t>(ptr);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<T*>((static_cast<uint64_t>(hi) << 32) | lo);
}

__device__ __forceinline__ void store16(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, uint4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{v.x, v.y, v.z, v.w}, rsrc, off, 0, 0);
}
// The same store marked non-temporal (cache policy nt): for outputs no kernel
// of the step reads back (the weight gradients), so that their bytes do not
// push the operands still being streamed out of L2 and the last-level cache.
__device__ __forceinline__ void store16_nt(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, uint4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{v.x, v.y, v.z, v.w}, rsrc, off, 0, 2);
}
__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t off) {
  const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// ------------------------------------------------------------------ kernel
//
// Persistent blocks.  Block b runs on XCD b % 8 (launch indices are dealt
// round-robin over the XCDs) and takes the tiles xidx, xidx + nbx, ... of its
// XCD's contiguous share of the logical tiles, so the blocks of one XCD work
// on neighbouring tiles (an expert's weight slab and its activation rows stay
// in that XCD's L2).  With groups the real tile count is computed on the
// device from `offs` (the grid is sized without a host sync).
//
// Each block runs one continuous stream of k-steps over all its tiles: a DMA
// cursor fills the LDS ring LEAD k-steps ahead of the compute cursor (3 of 5
// stages with a block barrier every second k-step, else STAGES-1 with one per
// k-step) and runs straight across tile boundaries, so the ring never drains
// between tiles.  When the compute cursor finishes a tile, the wave writes it
// out (epilogue) while the DMA of the next tile is already in flight; the
// tile waits that follow leave that epilogue's stores outstanding, so they
// drain in the background.  Every epilogue issues the
// same number of store instructions per wave (out-of-range stores go to an
// offset past the buffer resource and are dropped), which keeps those waits
// exact.
//
// LDS layouts (per stage, per operand; 16-byte chunks, XOR-swizzled so that
// the MFMA fragment reads are free of bank conflicts: gfx950 LDS has 64 banks
// of 4 bytes, so the 16 lanes of a ds_read_b128 pass, or the 32 lanes of a
// ds_read_b64_tr_b16 pass, must touch 64 distinct banks):
//   K-contiguous operand  [R rows][BK k]:  chunk c of row r at slot c ^ kc_swizzle<BK>(r)
//   M/N-contiguous operand [BK k][R cols]: chunk c of k-row kk at slot c ^ mc_swizzle(kk)
// Each DMA instruction fills one contiguous 1 KiB block lane by lane (lane l
// -> bytes 16l..16l+15), so a lane loads whichever global chunk belongs at
// its slot.  K-contiguous fragments are one ds_read_b128; M/N-contiguous
// fragments are two ds_read_b64_tr_b16, which turn a 4 (k) x 16 (n) patch read
// by 16 lanes into 4 consecutive k per lane.

// A ds_read_b128 pass reads one chunk of 16 consecutive rows.  32-deep
// k-tiles (64-byte rows, 4 rows per 256 bytes): rows r and r + 4k differ in
// bits 2-3, which move the chunk to another 16-byte bank group.  64-deep
// k-tiles (128-byte rows, 2 rows per 256 bytes): bits 1-3 do.
template <int BK>
__device__ __forceinline__ constexpr int kc_swizzle(int r) {
  return BK == 32 ? (r >> 2) & 3 : (r >> 1) & 7;
}
// A transpose-read pass reads 16 columns (2 chunks) of k-rows kk .. kk + 3 and
// kk + 8 .. kk + 11: k-row kk & 3 selects the 64-byte bank quarter, bit 3 of kk
// the half of it (needs >= 16 chunks per k-row).  (32-column fragments: 4
// chunks of kk .. kk + 3.)
__device__ __forceinline__ constexpr int mc_swizzle(int kk) { return 4 * (kk & 3) | 2 * ((kk >> 3) & 1); }
// Epilogue staging of a wave's 32 x 64 bf16 pass (128-byte rows): chunk cc of
// row r at slot cc ^ stg_swizzle(r); the 8-byte writes (16 rows, both halves of
// a chunk; from 32x32x16, 32 rows of one half, with the halves of rows 16 .. 31
// exchanged), the row reads and the SwiGLU gate/up reads are each on distinct
// banks.
__device__ __forceinline__ constexpr int stg_swizzle(int r) { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }

// Store instructions per wave per epilogue (all issued unconditionally).
template <int EPI, int WTM, int SM, int SN>
constexpr int epilogue_stores() {
  // bf16 outputs are staged one 32-row x 64-column pass at a time
  return EPI == EPI_F32            ? SM * SN * 4
         : EPI == EPI_SWIGLU_FWD  ? (WTM / 16) * 3 * (SN / 2)
                                  : (WTM / 8) * (SN / 2);  // EPI_BF16; EPI_WGRAD (its fp32 variant issues more)
}

template <int MODE, bool B_KCONTIG, int EPI, class CFG>
__global__ __launch_bounds__(CFG::kThreads) void grouped_gemm_kernel(const GemmParams p) {
  constexpr int BM = CFG::BM, BN = CFG::BN, BK = CFG::BK, WM = CFG::WM, WN = CFG::WN, STAGES = CFG::STAGES;
  constexpr int NWAVES = WM * WN;
  constexpr int WTM = BM / WM;  // wave tile rows
  constexpr int WTN = BN / WN;  // wave tile cols
  constexpr int SM = WTM / 32;  // 32x32 sub-tiles per wave along M
  constexpr int SN = WTN / 32;  // ... along N
  // The MFMA: 16x16x32, but 32x32x16 for the weight gradients, whose operands
  // are both read by transposes.  16x16x32 takes 1.054 of their time (geometric
  // mean over 104 sizes, routings and outputs: 485 against 465 us at 65536 x
  // 1536 x 2048 over 128 experts, 235 against 208 at 32768 x 1024 x 1024 over 32
  // with Zipf routing) and was never the faster by more than 1%.
  constexpr bool M32 = MODE == MODE_KG;
  constexpr int FR = M32 ? 32 : 16, FK = M32 ? 16 : 32;  // rows (columns) and depth of an operand fragment
  constexpr int FPS = 32 / FR;                           // fragments per 32-row sub-tile and k-slice
  constexpr int AM = SM * FPS, AN = SN * FPS;            // a wave's fragments of A and of B per k-slice
  constexpr bool A_KC = (MODE == MODE_MG);
  constexpr bool B_KC = (MODE == MODE_MG) && B_KCONTIG;
  // A K-contiguous A tile occupies whole rounds of DMA instructions in LDS
  // (512 / BK rows per instruction, one instruction per wave per round): rows
  // past BM are never read and their DMA is out of range (zeros, no traffic).
  constexpr int A_ROWS = (MODE == MODE_MG) ? (BM + (512 / BK) * NWAVES - 1) / ((512 / BK) * NWAVES) * ((512 / BK) * NWAVES)
                                           : BM;
  constexpr int A_BYTES = A_ROWS * BK * 2, B_BYTES = BN * BK * 2;
  constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  constexpr int NI_A = A_BYTES / 1024, NI_B = B_BYTES / 1024;  // DMA instructions per k-tile
  // Ping-pong: the DMA of a k-tile is split by operand between the wave
  // groups (waves 0-3 fire A, waves 4-7 fire B), LPW instructions per wave.
  constexpr bool PING = CFG::PIPE == 1;
  constexpr int LPW_A = PING ? 0 : NI_A / NWAVES, LPW_B = PING ? 0 : NI_B / NWAVES;  // ... per wave and operand
  constexpr int LPW = PING ? NI_A / 4 : LPW_A + LPW_B;
  // Barrier cadence.  With a 5-deep ring the DMA runs LEAD = 3 k-steps ahead
  // and the block synchronises on even k-steps only: an even step waits for
  // its own k-tile and the next one, and the DMA of any step targets the
  // stage read three steps earlier, which every wave had left by the last
  // barrier.  Shallower rings synchronise every step with the DMA
  // STAGES - 1 steps ahead.
  //
  // (The ping-pong loop's schedule is written down at the loop.)
  constexpr bool PAIR = STAGES == 5 && !PING;
  constexpr int LEAD = PAIR ? STAGES - 2 : STAGES - 1;
  constexpr int WAIT = PAIR ? LPW : (STAGES - 2) * LPW;  // DMA younger than the k-tile waited for
  constexpr int RELAX = PING ? 1 : PAIR ? 2 : STAGES - 1;  // waits that an epilogue's stores precede
  constexpr int NST = epilogue_stores<EPI, WTM, SM, SN>();
  constexpr int SLOT = 32 * 64 * 2;  // staging bytes per wave (one 32-row x 64-column pass)
  static_assert(BK == 32 || BK == 64, "swizzles and DMA mapping cover 32- and 64-deep k-tiles");
  constexpr int RB = BK * 2;      // bytes per K-contiguous row of a k-tile
  constexpr int CPR = BK / 8;     // 16-byte chunks per K-contiguous row
  constexpr int RPI = 64 / CPR;   // K-contiguous rows per DMA instruction
  static_assert(WTM % 32 == 0 && WTN == 64, "wave tiles are whole 32x32 sub-tiles, 64 columns wide");
  // (The weight gradients keep the paired-barrier loop: their tiles are a few
  // k-steps each, and their operands' rows are whole lines already.  On the
  // ping-pong loop the up projection's took 631 against 494 us at 512 rows per
  // expert, 373 against 290 at 256.)
  static_assert(!PING || (MODE == MODE_MG && STAGES == 5 && BK == 64 && NWAVES == 8 && WM == 2 && WN == 4 && NI_A == NI_B &&
                          NI_A % 8 == 0),
                "the ping-pong loop's wave groups, ring and DMA schedule");
  static_assert(PING || (NI_A % NWAVES == 0 && NI_B % NWAVES == 0), "DMA instructions of each operand split evenly over waves");
  static_assert(EPI != EPI_SWIGLU_FWD || (SN % 2 == 0), "SwiGLU forward pairs gate/up sub-tiles");
  static_assert(STAGES >= 2 && STAGES <= 5, "ring depth");
  static_assert(NWAVES * SLOT <= STAGE_BYTES, "the epilogue stages every wave's pass in one ring stage");
  static_assert(WAIT + NST < 64, "vmcnt range");
  static_assert(A_KC || BM >= 128, "transpose-read swizzle needs >= 16 chunks per k-row");
  static_assert(B_KC || BN >= 128, "transpose-read swizzle needs >= 16 chunks per k-row");

  __shared__ __attribute__((aligned(1024))) char ring[STAGES * (PING ? A_BYTES : STAGE_BYTES)];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  // Wave-uniform values live in scalar registers: buffer resources and the
  // DMA LDS base (M0) must be uniform.
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Ping-pong wave groups: group grp = wave / 4 holds wave columns 2 grp and
  // 2 grp + 1; its four waves sit on the four SIMDs.
  const int grp = wave >> 2, w4 = wave & 3;
  const int wm = PING ? (w4 >> 1) : wave / WN, wn = PING ? grp * 2 + (w4 & 1) : wave % WN;
  const int i16 = lane & 15, q16 = lane >> 4;  // the lane's row (column) and k-group in a 16x16x32 MFMA operand
  const int l32 = lane & 31, khalf = lane >> 5;  // ... in a 32x32x16 one

  // ------------------------------------------------------ this block's tiles
  const int nbx = gridDim.x / kNumXcd;  // the grid is a multiple of kNumXcd
  const int xcd = blockIdx.x % kNumXcd, xidx = blockIdx.x / kNumXcd;
  const int real = (MODE == MODE_MG && p.offs) ? count_tiles<BM>(p.offs, p.G, p.rows, p.n_tiles) : p.total_tiles;
  int first, span;
  const int2 range = (MODE == MODE_KG && p.cost_split)
                         ? kg_cost_split<BK>(p.offs, p.G, p.rows, p.n_tiles * p.m_tiles_max, xcd)
                         : make_int2(-1, -1);
  if (range.x >= 0) {
    first = range.x;
    span = range.y - range.x;
  } else {
    const int share = (real + kNumXcd - 1) / kNumXcd;
    first = xcd * share;
    span = min(share, real - first);
  }
  // Weight gradients under skewed routing (the cost split above): the XCD's
  // tiles are dealt to its blocks in cost order, the heaviest group's first,
  // snaking (round r gives block xidx the tile at position r nbx + xidx on
  // even rounds, r nbx + nbx - 1 - xidx on odd ones), so that every block
  // gets about one tile of each cost level instead of every nbx-th tile of
  // the group-major order.  Consecutive positions are still mostly one
  // group's tiles, which the XCD's blocks take at about the same time (its
  // operand panels are shared through L2).  Lane m holds the m-th group
  // touching the range (up to 64 of them; more keep the plain deal): its
  // tiles in the range (sn_cnt, the first at sn_t0 from `first`) and the
  // tiles of the groups ranked before it (sn_pc); rank: larger k-steps
  // first, then the lower group.  Busiest block's k-steps against the mean
  // at C4's routing (simulated): up_wgrad 1.12 -> 1.09, down_wgrad 1.29 ->
  // 1.10.
  bool snake = false;
  int sn_cnt = 0, sn_t0 = 0, sn_pc = 0;
  if constexpr (MODE == MODE_KG) {
    if (range.x >= 0 && span > 0) {
      const int per_group = p.n_tiles * p.m_tiles_max;
      const int g0 = first / per_group, g1 = (first + span - 1) / per_group;
      if (g1 - g0 < kWave) {
        snake = true;
        const int g = g0 + lane;
        int cost = -1;
        if (g <= g1) {
          const int lo_t = max(first, g * per_group), hi_t = min(first + span, (g + 1) * per_group);
          sn_cnt = hi_t - lo_t;
          sn_t0 = lo_t - first;
          const int hi = min(max(p.offs[g], 0), p.rows);
          const int lo = g ? min(max(p.offs[g - 1], 0), hi) : 0;
          cost = (hi - lo + BK - 1) / BK;
        }
        int rank = 0;
        for (int m = 0; m < kWave; ++m) {
          const int cm = __builtin_amdgcn_readlane(cost, m);
          rank += (cm > cost || (cm == cost && m < lane)) ? 1 : 0;
        }
        for (int m = 0; m < kWave; ++m) {
          const int rm = __builtin_amdgcn_readlane(rank, m), cm = __builtin_amdgcn_readlane(sn_cnt, m);
          sn_pc += rm < rank ? cm : 0;
        }
      }
    }
  }
  int nt_blk;
  if (snake) {  // full rounds, plus the last partial round's slot of this block
    const int rounds = span / nbx, rem = span - rounds * nbx;
    nt_blk = rounds + (((rounds & 1) ? nbx - 1 - xidx : xidx) < rem ? 1 : 0);
  } else {
    nt_blk = span > xidx ? (span - xidx + nbx - 1) / nbx : 0;
  }
  const int ntiles = __builtin_amdgcn_readfirstlane(nt_blk);
  if (ntiles <= 0) return;

  // Lane l of a descriptor chunk describes block tile 64 * chunk + l:
  // group, first output row (absolute for MG, within the group for KG),
  // first output column, reduction rows [rb, re) (KG) or the tile's valid
  // rows end (MG), split-K index.
  struct Desc {
    int g, m0, n0, rb, re, split;
  };
  auto describe = [&](int chunk) __attribute__((always_inline)) {
    Desc d{0, 0, 0, 0, 0, 0};
    const int j = chunk * kWave + lane;
    const bool valid = j < ntiles;
    int L = first + xidx + j * nbx;
    if (MODE == MODE_KG && snake) {
      // position j nbx + slot in cost order -> the tile: the group (lane m)
      // whose positions [sn_pc, sn_pc + sn_cnt) hold it
      const int pos = j * nbx + ((j & 1) ? nbx - 1 - xidx : xidx);
      L = first;
      for (int m = 0; m < kWave; ++m) {
        const int pm = __builtin_amdgcn_readlane(sn_pc, m), cm = __builtin_amdgcn_readlane(sn_cnt, m);
        if (pos >= pm && pos < pm + cm) L = first + __builtin_amdgcn_readlane(sn_t0, m) + (pos - pm);
      }
    }
    if constexpr (MODE == MODE_MG) {
      if (p.offs) {
        // Per-lane search of the group holding tile L over the cumulative
        // per-group tile counts, one 64-group chunk at a time.
        const int target = valid ? L : 0x7fffffff;
        int found = 0, tg = 0, t0 = 0, r0 = 0, cn = 0, base = 0;
        for (int c0 = 0; c0 < p.G; c0 += kWave) {
          const int gg = c0 + lane;
          int lo = 0, hi = 0;
          if (gg < p.G) {
            hi = min(max(p.offs[gg], 0), p.rows);  // clamped: malformed offsets never address outside [0, rows)
            lo = gg ? min(max(p.offs[gg - 1], 0), hi) : 0;
          }
          const int cnt = hi - lo;
          const int nt = p.n_tiles * ((cnt + BM - 1) / BM);
          const int incl = wave_inclusive_scan(nt);
          const int tot = __builtin_amdgcn_readlane(incl, kWave - 1);
          const int t = target - base;
          int q = 0;  // smallest q with incl[q] > t
#pragma unroll
          for (int s = kWave / 2; s >= 1; s >>= 1)
            if (__shfl(incl, q + s - 1, kWave) <= t) q += s;
          const int exq = __shfl(incl - nt, q, kWave), loq = __shfl(lo, q, kWave), cq = __shfl(cnt, q, kWave);
          if (!found && t >= 0 && t < tot) {
            found = 1;
            tg = c0 + q;
            t0 = base + exq;
            r0 = loq;
            cn = cq;
          }
          base += tot;
        }
        if (valid && found) {
          const int local = L - t0;
          const int mt_g = (cn + BM - 1) / BM;
          const int nt = local / mt_g, mt = local - (local / mt_g) * mt_g;
          // The group's rows split evenly over its m-tiles (whole 32-row
          // sub-tiles): the m-tiles of one weight tile then run at the same
          // pace on neighbouring CUs and read each weight k-slice once from
          // HBM between them, where a full tile plus a short one would drift
          // apart and read it twice.  Every m-tile holds rows, since
          // (mt_g - 1) * rpt <= (mt_g - 1) * BM < cn.
          const int rpt = min(BM, ((cn + mt_g - 1) / mt_g + 31) & ~31);
          const int m0 = r0 + mt * rpt;
          d = Desc{tg, m0, nt * BN, r0, min(m0 + rpt, r0 + cn), 0};
        }
      } else {
        const int mtiles = (p.M + BM - 1) / BM;
        const int per_split = mtiles * p.n_tiles;
        const int split = L / per_split, local = L - split * per_split;
        const int nt = local / mtiles, mt = local - nt * mtiles;
        if (valid) d = Desc{0, mt * BM, nt * BN, 0, p.M, split};
      }
    } else {
      const int per_group = p.n_tiles * p.m_tiles_max;
      const int g = L / per_group, local = L - g * per_group;
      const int nt = local / p.m_tiles_max, mt = local - nt * p.m_tiles_max;
      if (valid) {
        int rb, re;
        if (p.offs) {
          re = min(max(p.offs[g], 0), p.rows);
          rb = g ? min(max(p.offs[g - 1], 0), re) : 0;
        } else {
          rb = min(g * p.chunk_rows, p.rows);
          re = min(rb + p.chunk_rows, p.rows);
        }
        d = Desc{g, mt * BM, nt * BN, rb, re, 0};
      }
    }
    return d;
  };
  auto pick = [](int v, int j) { return __builtin_amdgcn_readlane(v, j & (kWave - 1)); };

  // Per-tile scalars shared by both cursors.
  struct Tile {
    int g, m0, n0, rb, re, split, k_begin, kred, nk;
  };
  auto tile_of = [&](const Desc& d, int j) __attribute__((always_inline)) {
    Tile t;
    t.g = pick(d.g, j);
    t.m0 = pick(d.m0, j);
    t.n0 = pick(d.n0, j);
    t.rb = pick(d.rb, j);
    t.re = pick(d.re, j);
    t.split = pick(d.split, j);
    t.k_begin = (MODE == MODE_MG) ? t.split * p.k_chunk : 0;
    t.kred = (MODE == MODE_MG) ? min(p.K - t.k_begin, p.k_chunk) : (t.re - t.rb);
    t.nk = t.kred > 0 ? (t.kred + BK - 1) / BK : 0;
    return t;
  };

  // ------------------------------------------------------ DMA cursor
  // Each k-tile is NI_A + NI_B DMA instructions of 1 KiB; wave w issues A
  // instructions w*LPW_A .. w*LPW_A+LPW_A-1 (its slots j < LPW_A) and B
  // instructions w*LPW_B .. w*LPW_B+LPW_B-1 (slots j >= LPW_A).  Per lane and
  // slot: the LDS byte offset within a stage (wave-uniform), the k
  // (K-contiguous: the chunk's k; M/N-contiguous: the k-row) it adds per
  // k-tile, and a per-tile base offset (kOOB if the row or column is outside
  // the tile's valid range).
  const u32x4_t rsA = rsrc_words(p.A, p.a_bytes);
  // Row strides in bytes, in scalar registers (a ping-pong wave selects its
  // operand's at run time).
  const uint32_t lda2 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p.lda) * 2u);
  const uint32_t ldb2 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p.ldb) * 2u);
  // Slot j's operand (wave-uniform) and instruction index within the operand's k-tile.
  auto slot_is_a = [&](int j) { return PING ? grp == 0 : j < LPW_A; };
  auto slot_inst = [&](int j, bool& is_a) {
    is_a = slot_is_a(j);
    if constexpr (PING) return w4 * LPW + j;
    return is_a ? wave * LPW_A + j : wave * LPW_B + (j - LPW_A);
  };
  int dma_lds[LPW], dma_k[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    bool is_a;
    const int li = slot_inst(j, is_a);
    dma_lds[j] = __builtin_amdgcn_readfirstlane((is_a || PING ? 0 : A_BYTES) + li * 1024);
    if (is_a ? A_KC : B_KC) {
      const int r = li * RPI + lane / CPR;
      dma_k[j] = ((lane % CPR) ^ kc_swizzle<BK>(r)) * 8;
    } else {
      const int cpk = (is_a ? BM : BN) / 8;  // 16-byte chunks per k-row
      dma_k[j] = li * (64 / cpk) + lane / cpk;
    }
  }

  Desc dd = describe(0);
  int dchunk = 0;
  int dj = 0, dk = 0;  // DMA cursor: block tile and k-step
  Tile dt;
  u32x4_t rsB = rsrc_words(p.B, p.b_bytes);
  // Per slot: the lane's byte offset at the tile's first k-step (kOOB if the
  // row or column lies outside the tile, or past the last tile); a k-step
  // adds a uniform amount to it.
  uint32_t dma_pre[LPW];
  // Sets the DMA cursor on block tile j (skipping tiles without k-steps);
  // past the last tile the cursor issues out-of-range loads (zeros).
  auto dma_seek = [&](int j) __attribute__((always_inline)) {
    for (;; ++j) {
      if (j >= ntiles) {
        dj = ntiles;
#pragma unroll
        for (int j2 = 0; j2 < LPW; ++j2) dma_pre[j2] = kOOB;
        return;
      }
      if ((j >> 6) != dchunk) {
        dchunk = j >> 6;
        dd = describe(dchunk);
      }
      dt = tile_of(dd, j);
      if (dt.nk > 0) break;
    }
    dj = j;
    dk = 0;
    if (MODE == MODE_MG) rsB = rsrc_words(p.B + static_cast<int64_t>(dt.g) * p.stride_bg, p.b_bytes);
    const int mc_row0 = (MODE == MODE_KG) ? dt.rb : dt.k_begin;
#pragma unroll
    for (int j2 = 0; j2 < LPW; ++j2) {
      bool is_a;
      const int li = slot_inst(j2, is_a);
      if (is_a ? A_KC : B_KC) {
        const int r = li * RPI + lane / CPR;
        const int c = (lane % CPR) ^ kc_swizzle<BK>(r);
        bool ok;
        uint32_t row_bytes;
        if (is_a) {
          const int grow = dt.m0 + r;
          ok = grow < dt.re;
          row_bytes = static_cast<uint32_t>(grow) * lda2;
        } else {
          int wrow;
          if constexpr (EPI == EPI_SWIGLU_FWD) {
            // Tile row r -> (wave column, 64-column group, half): each
            // 64-column group of a wave tile holds 32 gate rows, then the
            // 32 matching up rows, so that one 64-column epilogue pass sees
            // both halves of its act columns.
            const int wcol = r / WTN;
            const int within = r % WTN;
            const int group = within / 64;
            const int half = (within % 64) / 32;
            const int act_col = (dt.n0 / 2) + wcol * (WTN / 2) + group * 32 + (within % 32);
            ok = act_col < p.swiglu_I;
            wrow = half * p.swiglu_I + act_col;
          } else {
            wrow = dt.n0 + r;
            ok = wrow < p.N;
          }
          row_bytes = static_cast<uint32_t>(wrow) * ldb2;
        }
        dma_pre[j2] = ok ? row_bytes + static_cast<uint32_t>(c) * 16u + static_cast<uint32_t>(dt.k_begin) * 2u : kOOB;
      } else {
        // first of the chunk's 8 columns
        const int col = (is_a ? dt.m0 : dt.n0) + ((lane % ((is_a ? BM : BN) / 8)) ^ mc_swizzle(dma_k[j2])) * 8;
        const uint32_t ld = is_a ? lda2 : ldb2;
        dma_pre[j2] = col < (is_a ? p.M : p.N)
                          ? static_cast<uint32_t>(mc_row0 + dma_k[j2]) * ld + static_cast<uint32_t>(col) * 2u
                          : kOOB;
      }
    }
  };
  // The DMA of the cursor's next k-step into the ring, in three parts:
  // dma_prepare fixes the stage and the k-step, dma_fire(j) computes slot j's
  // offset and issues it, dma_advance moves the cursor.  The compute loop
  // fires the slots between its MFMA groups (ping-pong: its fragment reads),
  // so that the texture unit works through the k-step's DMA while the matrix
  // cores run instead of taking every wave's burst at once.  The offsets live
  // in registers only around their own load, except in the weight gradients,
  // which keep the k-step's (1% of their time; the other GEMMs lose that much
  // by it).  Every k-step fires exactly LPW instructions per wave.
  uint32_t dma_at = 0;
  int dma_k0 = 0, dma_left = 0;  // the k-step's first k (or k-row) in the tile, and how many are left from there
  u32x4_t ra, rb;
  uint32_t doff[LPW], dlds[LPW];
  auto dma_offset = [&](int j) __attribute__((always_inline)) {
    const bool is_a = slot_is_a(j);
    const uint32_t step = (is_a ? A_KC : B_KC) ? 2u : (is_a ? lda2 : ldb2);
    // Past the last tile dma_pre is kOOB and stays out of range (the added
    // offset is below the 2 GiB operand limit).
    return dma_k[j] < dma_left ? dma_pre[j] + static_cast<uint32_t>(dma_k0) * step : kOOB;
  };
  // `at`: LDS byte offset of the stage (ping-pong: of the operand tile's slot).
  auto dma_prepare = [&](int at) __attribute__((always_inline)) {
    dma_k0 = dk * BK;
    dma_left = dt.kred - dma_k0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if constexpr (PING) {
        // every slot of a ping-pong wave is of its group's operand
        ra[w] = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(grp == 0 ? rsA[w] : rsB[w]));
        rb[w] = ra[w];
      } else {
        ra[w] = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(rsA[w]));
        rb[w] = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(rsB[w]));
      }
    }
    dma_at = lds_address(ring) + at;
    if constexpr (M32) {
#pragma unroll
      for (int j = 0; j < LPW; ++j) {
        doff[j] = dma_offset(j);
        dlds[j] = __builtin_amdgcn_readfirstlane(dma_at + dma_lds[j]);
      }
    }
  };
  auto dma_fire = [&](int j) __attribute__((always_inline)) {
    if constexpr (M32) {
      dma16(j < LPW_A ? ra : rb, doff[j], dlds[j]);
    } else {
      dma16(PING || j < LPW_A ? ra : rb, dma_offset(j), __builtin_amdgcn_readfirstlane(dma_at + dma_lds[j]));
    }
  };
  auto dma_advance = [&]() __attribute__((always_inline)) {
    if (dj < ntiles && ++dk == dt.nk) dma_seek(dj + 1);
  };
  auto dma_issue = [&](int at) __attribute__((always_inline)) {
    dma_prepare(at);
#pragma unroll
    for (int j = 0; j < LPW; ++j) dma_fire(j);
    dma_advance();
  };

  // ------------------------------------------------------ fragment reads
  // A wave's SM row sub-tiles are interleaved with the other wave rows':
  // sub-tile i covers tile rows sub_row(i) .. +31, so that the sub-tiles of a
  // partly filled tile spread over all waves (and SIMDs).  Its SN column
  // sub-tiles are contiguous: columns wn*WTN + 32 j.
  //
  // A fragment is FR rows (columns) x FK k, lane l holding row l % FR, k
  // 8 (l / FR) .. + 7; a 32-row sub-tile is FPS of them.  Each lane's byte
  // offset within a stage is precomputed per fragment class; a fragment
  // address is the stage base plus a lane offset plus a constant.
  // K-contiguous [R rows][CPR chunks] (16-row fragments): lane reads row
  // (tile_row + i16), chunk 4 ks + q16; fragment rows start on 16-row
  // boundaries, so the swizzle of row tile_row + i16 is that of i16.
  static_assert(!M32 || (!A_KC && !B_KC), "K-contiguous fragments are 16 rows x 32 k");
  constexpr int KS = BK / FK;
  auto sub_row = [&](int i) { return (wm + WM * i) * 32; };
  constexpr int B_OFF = PING ? 0 : A_BYTES;  // B's offset from the base its fragments are read with
  int a_kc[KS], b_kc[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int lane_off = i16 * RB + (((4 * ks + q16) ^ kc_swizzle<BK>(i16)) << 4);
    a_kc[ks] = sub_row(0) * RB + lane_off;
    b_kc[ks] = B_OFF + wn * WTN * RB + lane_off;
  }
  // M/N-contiguous [BK k-rows][R cols] (transpose reads): lane reads k-rows
  // FK ks + 4 h + i16 / 4, + 8 q16 (16-column fragments) or + 8 (q16 / 2), and
  // columns tile_col + 4 (i16 % 4), of 32-column fragments + 16 (q16 % 2).  The
  // swizzle depends only on bits 0, 1 and 3 of the k-row (16-deep slices change
  // bit 4 only), so each fragment has one lane offset; ks and h add constants.
  const int tr_krow = 8 * (q16 >> M32) + (i16 >> 2);
  const int tr_col = 4 * (i16 & 3) + 16 * (M32 & q16 & 1);
  const int half8 = (i16 & 1) << 3;
  int a_mc[AM], b_mc[AN];
#pragma unroll
  for (int t = 0; t < AM; ++t)
    a_mc[t] = tr_krow * BM * 2 + ((((sub_row(t / FPS) + FR * (t % FPS) + tr_col) >> 3) ^ mc_swizzle(tr_krow)) << 4) + half8;
#pragma unroll
  for (int t = 0; t < AN; ++t)
    b_mc[t] = B_OFF + tr_krow * BN * 2 + ((((wn * WTN + FR * t + tr_col) >> 3) ^ mc_swizzle(tr_krow)) << 4) + half8;
  auto tr_read = [](const char* at, int row_bytes) __attribute__((always_inline)) {
    const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)at);
    const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(at + 4 * row_bytes));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // Fragment t of A (sub-tile t / FPS's rows FR (t % FPS) ..) or of B (columns
  // FR t .. of the wave's) for k's FK ks .. of the k-tile at `base`.
  auto read_a = [&](const char* base, int ks, int t) __attribute__((always_inline)) {
    if constexpr (A_KC) {
      return *reinterpret_cast<const bf16x8_t*>(base + a_kc[ks] + ((t / 2) * WM * 32 + (t % 2) * 16) * RB);
    } else {
      return tr_read(base + a_mc[t] + FK * ks * BM * 2, BM * 2);
    }
  };
  auto read_b = [&](const char* base, int ks, int t) __attribute__((always_inline)) {
    if constexpr (B_KC) {
      return *reinterpret_cast<const bf16x8_t*>(base + b_kc[ks] + t * 16 * RB);
    } else {
      return tr_read(base + b_mc[t] + FK * ks * BN * 2, BN * 2);
    }
  };

  // acc[FPS i + h][t]: rows FR h .. of row sub-tile i, columns FR t .. of the wave's.
  using Acc = std::conditional_t<M32, f32x16_t, f32x4_t>;
  Acc acc[AM][AN];
  auto zero_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AM; ++i)
#pragma unroll
      for (int j = 0; j < AN; ++j)
#pragma unroll
        for (int r = 0; r < (M32 ? 16 : 4); ++r) acc[i][j][r] = 0.0f;
  };
  // Operands swapped: the result holds C^T fragments, so each lane owns one
  // output row and runs of 4 consecutive output columns.
  auto mfma_row = [&](int i, const bf16x8_t& a, const bf16x8_t (&b)[AN]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < AN; ++j) {
      if constexpr (M32) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], a, acc[i][j], 0, 0, 0);
      } else {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a, acc[i][j], 0, 0, 0);
      }
    }
  };
  // Run e (of 8) of 4 consecutive columns that the lane holds of row sub-tile
  // i's columns 64 h ..: its values, and its row and first column in there.
  struct Run {
    float4 v;
    int row, col;
  };
  auto acc_run = [&](int i, int h, int e) __attribute__((always_inline)) {
    if constexpr (M32) {
      const f32x16_t& c = acc[i][2 * h + e / 4];
      const int q = e % 4;
      return Run{make_float4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]), l32, 8 * e + 4 * khalf};
    } else {
      const f32x4_t& c = acc[2 * i + e / 4][4 * h + e % 4];
      return Run{make_float4(c[0], c[1], c[2], c[3]), 16 * (e / 4) + i16, 16 * (e % 4) + 4 * q16};
    }
  };

  // One k-tile of MFMAs over the first `na` row sub-tiles (the others hold no
  // rows of this tile; `na` is wave-uniform, so the guards are scalar
  // branches), with the prepared DMA slots fired between the MFMA groups:
  // slot s after group (ks, i) = s * KS SM / LPW.  The fragments of AHEAD row
  // sub-tiles are read before the first one's MFMAs, each further one's before
  // those of the sub-tile AHEAD before it.
  auto compute = [&](int na, const char* stage) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      constexpr int AHEAD = M32 ? 2 : 1;
      bf16x8_t af[AHEAD + 1][FPS], bfr[AN];
#pragma unroll
      for (int i = 0; i < AHEAD; ++i)
#pragma unroll
        for (int h = 0; h < FPS; ++h) af[i][h] = read_a(stage, ks, FPS * i + h);
#pragma unroll
      for (int j = 0; j < AN; ++j) bfr[j] = read_b(stage, ks, j);
#pragma unroll
      for (int i = 0; i < SM; ++i) {
        if (i + AHEAD < SM) {
#pragma unroll
          for (int h = 0; h < FPS; ++h) af[(i + AHEAD) % (AHEAD + 1)][h] = read_a(stage, ks, FPS * (i + AHEAD) + h);
        }
        if (i == 0 || i < na) {
#pragma unroll
          for (int h = 0; h < FPS; ++h) mfma_row(FPS * i + h, af[i % (AHEAD + 1)][h], bfr);
        }
#pragma unroll
        for (int s2 = 0; s2 < LPW; ++s2) {
          if ((s2 * KS * SM) / LPW == ks * SM + i) {
            __builtin_amdgcn_sched_barrier(0);
            dma_fire(s2);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
  };

  // Workgroup barrier without a memory fence (a fenced barrier would drain
  // every outstanding DMA); the empty asm statements keep LDS accesses from
  // moving across it.
  auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ------------------------------------------------------ epilogue
  // Lane owns the runs acc_run(i, h, e) of output rows m0 + sub_row(i) + row and
  // columns wcol0 + 64 h + col + {0..3}.
  // This wave's staging slot (no other wave touches it) in the ring stage
  // that the compute cursor has just finished: no DMA targets that stage
  // before the next block barrier, and a barrier before the epilogue
  // retires every wave's fragment reads of it.  Tiles written out before the
  // stream starts (empty weight-gradient groups) use the last stage, which
  // the prologue DMA leaves alone and no k-step fills before the first
  // barrier.
  char* slot = ring + (STAGES - 1) * (PING ? A_BYTES : STAGE_BYTES) + wave * SLOT;
  auto to_f32x8 = [](uint4 v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[2 * e] = lo_bf16(w[e]);
      f[2 * e + 1] = hi_bf16(w[e]);
    }
  };
  auto to_bf16x8 = [](const float* f) {
    return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]),
                      pack_bf16x2(f[6], f[7]));
  };
  auto round_bf16 = [](float x) { return bf16_to_f32(f32_to_bf16(x)); };
  const __amdgpu_buffer_rsrc_t rsC2 = make_rsrc(p.C2, p.c2_bytes);  // SwiGLU pre-activation (0 bytes if absent)

  auto epilogue = [&](const Tile& t) __attribute__((always_inline)) {
    const int wcol0 = t.n0 + wn * WTN;
    const int row_limit = (MODE == MODE_MG) ? t.re : p.M;
    // Output resource: MG writes [rows, ldc]; KG one group's [M, ldc]; split-K one split's partial.
    const int esize = (EPI == EPI_F32 || (EPI == EPI_WGRAD && p.ldp)) ? 4 : 2;
    const int64_t g_off = p.bucket_rows ? static_cast<int64_t>(t.g / p.bucket_rows) * p.bucket_stride +
                                              static_cast<int64_t>(t.g % p.bucket_rows) * p.stride_cg
                                        : static_cast<int64_t>(t.g) * p.stride_cg;
    const int64_t c_base = (MODE == MODE_KG)  ? g_off
                           : (EPI == EPI_F32) ? static_cast<int64_t>(t.split) * p.split_stride
                                              : 0;
    const __amdgpu_buffer_rsrc_t rsC = make_rsrc(uniform_ptr(static_cast<char*>(p.C) + c_base * esize), p.c_bytes);
    if (EPI == EPI_F32 || (EPI == EPI_WGRAD && p.ldp)) {
      // fp32 outputs (split-K partials, fp32 weight gradients): direct 16-byte stores.
#pragma unroll
      for (int ih = 0; ih < SM * (SN / 2); ++ih) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int i = ih / (SN / 2), h = ih % (SN / 2);
          const Run run = acc_run(i, h, e);
          const int row = t.m0 + sub_row(i) + run.row, col = wcol0 + 64 * h + run.col;
          const uint32_t off = (row < row_limit && col < p.N)
                                   ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(p.ldc) +
                                      static_cast<uint32_t>(col)) * 4u
                                   : kOOB;
          float4 v = run.v;
          if (EPI == EPI_WGRAD && p.accumulate) {
            const uint4 o = load16(rsC, off);
            v.x += __uint_as_float(o.x);
            v.y += __uint_as_float(o.y);
            v.z += __uint_as_float(o.z);
            v.w += __uint_as_float(o.w);
          }
          const uint4 o4 = make_uint4(__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z),
                                      __float_as_uint(v.w));
          if constexpr (EPI == EPI_WGRAD) {
            store16_nt(rsC, off, o4);
          } else {
            store16(rsC, off, o4);
          }
        }
      }
      return;
    }
    // bf16 outputs go through this wave's LDS slot one 32-row pass at a time,
    // so that every store is 16 bytes per lane over whole 128-byte row segments.
    // The 8-byte halves of a chunk are exchanged in rows 16 .. 31 where a
    // write's lanes hold 32 rows of one half (32x32x16).
    auto stg_at = [&](int row, int col) __attribute__((always_inline)) {
      return row * 128 + (((col >> 3) ^ stg_swizzle(row)) << 4) + ((((col >> 2) & 1) ^ (M32 & (row >> 4))) << 3);
    };
    auto stg_row = [&](int r, int chunk) __attribute__((always_inline)) {
      const uint4 v = *reinterpret_cast<const uint4*>(slot + r * 128 + ((chunk ^ stg_swizzle(r)) << 4));
      return M32 && (r & 16) ? make_uint4(v.z, v.w, v.x, v.y) : v;
    };
    const int rr8 = lane >> 3, c8 = lane & 7;  // row-read lane mapping: row 8n + rr8, chunk c8
    // One pass per 32 rows (row sub-tile i) and 64 columns (column group h:
    // sub-tiles 2h and 2h + 1).
#pragma unroll
    for (int ih = 0; ih < SM * (SN / 2); ++ih) {
      const int i = ih / (SN / 2), h = ih % (SN / 2);
      const int pcol0 = wcol0 + 64 * h;     // first output column of this pass
      const int prow0 = t.m0 + sub_row(i);  // first output row of this pass
      // Output offsets of this pass's row reads and, when accumulating, the
      // existing gradient, loaded before the staging so that their latency
      // overlaps it.
      uint32_t out_off[4];
      uint4 in0[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int row = prow0 + 8 * n + rr8, col = pcol0 + c8 * 8;
        const bool ok = row < row_limit && col < p.N;
        out_off[n] = ok ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(p.ldc) + static_cast<uint32_t>(col)) * 2u
                        : kOOB;
        if constexpr (EPI == EPI_WGRAD) {
          if (p.accumulate) in0[n] = load16(rsC, out_off[n]);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const Run run = acc_run(i, h, e);
        *reinterpret_cast<uint2*>(slot + stg_at(run.row, run.col)) =
            make_uint2(pack_bf16x2(run.v.x, run.v.y), pack_bf16x2(run.v.z, run.v.w));
      }
      if constexpr (EPI == EPI_SWIGLU_FWD) {
        // Slot columns 0-31 are gate, 32-63 the matching up columns.  A lane
        // takes one 8-column gate chunk and its up chunk: act = silu(gate) * up
        // with the reference's bf16 roundings (bf16 GEMM output, silu output,
        // product); gate | up go to the saved pre-activation.
        const int rr = lane >> 2, c4 = lane & 3;
        const int act_col = (t.n0 / 2) + wn * (WTN / 2) + 32 * h + c4 * 8;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const int r = 16 * n + rr;
          const uint4 gv = stg_row(r, c4), uv = stg_row(r, c4 + 4);
          const int row = prow0 + r;
          const bool ok = row < row_limit && act_col < p.swiglu_I;
          float gf[8], uf[8], af[8];
          to_f32x8(gv, gf);
          to_f32x8(uv, uf);
#pragma unroll
          for (int e = 0; e < 8; ++e) af[e] = round_bf16(silu_f(gf[e])) * uf[e];
          const uint32_t act_off = ok ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(p.ldc) +
                                         static_cast<uint32_t>(act_col)) * 2u
                                      : kOOB;
          const uint32_t pre_off = ok ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(p.ldp) +
                                         static_cast<uint32_t>(act_col)) * 2u
                                      : kOOB;
          store16(rsC, act_off, to_bf16x8(af));
          store16(rsC2, pre_off, gv);
          store16(rsC2, ok ? pre_off + static_cast<uint32_t>(p.swiglu_I) * 2u : kOOB, uv);
        }
      } else {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const int r = 8 * n + rr8;
          uint4 v = stg_row(r, c8);
          if constexpr (EPI == EPI_BF16) {
            store16(rsC, out_off[n], v);
          } else if constexpr (EPI == EPI_WGRAD) {
            if (p.accumulate) {
              // The fp32 accumulator rounded to bf16 plus the existing bf16
              // gradient, rounded once more (torch's bf16 add of the two).
              float a[8], o[8];
              to_f32x8(v, a);
              to_f32x8(in0[n], o);
#pragma unroll
              for (int e = 0; e < 8; ++e) a[e] += o[e];
              v = to_bf16x8(a);
            }
            store16_nt(rsC, out_off[n], v);
          }
        }
      }
    }
  };

  // ------------------------------------------------------ compute cursor
  Desc cd = dd;
  int cchunk = 0;
  int cj = 0, ck = 0;
  Tile ct;
  int n_act = 0;  // row sub-tiles of this wave that hold rows of the current tile (0: no MFMAs)
  // Sets the compute cursor on block tile j.  Tiles without k-steps (empty
  // groups of a weight gradient) are written out here directly: zeros, or
  // nothing when accumulating.  Returns false past the last tile.
  int relax = 0;  // steps whose tile wait still leaves the last epilogue's stores in flight
  auto compute_seek = [&](int j) __attribute__((always_inline)) -> bool {
    for (;; ++j) {
      if (j >= ntiles) return false;
      if ((j >> 6) != cchunk) {
        cchunk = j >> 6;
        cd = describe(cchunk);
      }
      ct = tile_of(cd, j);
      zero_acc();
      if (ct.nk > 0) break;
      if constexpr (MODE == MODE_KG) {  // (MG tiles always have k-steps)
        if (!p.accumulate) {
          epilogue(ct);
          relax = RELAX;
        }
      }
    }
    cj = j;
    ck = 0;
    const int row_limit = (MODE == MODE_MG) ? ct.re : p.M;
    const int wcol0 = ct.n0 + wn * WTN;
    // Sub-tiles (and waves) whose rows or columns all lie outside the tile
    // skip the MFMAs; every wave still takes part in the DMA and the barriers.
    // Sub-tile i starts at tile row 32 (wm + WM i): i < n_act exactly when
    // it starts below the tile's last row.
    const int subs = (min(row_limit - ct.m0, BM) + 31) / 32;  // 32-row sub-tiles holding rows
    int na = subs > wm ? (subs - wm + WM - 1) / WM : 0;
    if (!(EPI == EPI_SWIGLU_FWD || wcol0 < p.N)) na = 0;
    n_act = __builtin_amdgcn_readfirstlane(min(na, SM));
    return true;
  };

  // ------------------------------------------------------ the k-step stream
  dma_seek(0);
  const bool any = compute_seek(0);
  // Stores of tiles written out above precede every DMA, so the plain tile
  // wait already covers them.
  relax = 0;
#pragma unroll
  for (int s = 0; s < (PING ? 0 : LEAD); ++s) dma_issue(s * STAGE_BYTES);
  if constexpr (PING) {
    // Ping-pong over a ring of operand tiles.  A k-step is 64 deep, so that the
    // DMA of a K-contiguous operand moves whole 128-byte lines (with 32-deep
    // k-tiles the DMA of 65536 x 3072 x 4096 over 128 experts alone takes 1344
    // us, the loop 1630; with 64-deep ones 1059, and 1386 the loop).  k-step
    // c's B tile sits in ring slot 2c % 5, its A tile in slot (2c + 1) % 5.
    //
    // A k-step is two halves of 32 k.  In phase 4c + 2h (h = 0, 1) group 0
    // (waves 0-3) reads the fragments of half h, in phase 4c + 2h + 1 it
    // multiplies them; group 1 (waves 4-7) runs one phase later.  Each phase
    // ends with a block barrier, so on every SIMD one wave issues MFMAs from
    // registers while its partner reads fragments and fires DMA.
    //
    // DMA: group 0 fires all of A tile c + 1 in phase 4c.  Its slot held B
    // tile c - 1, read last in phase 4c - 1.  Group 1 fires B tile c + 2 in
    // phases 4c + 1 and 4c + 3, half in each; its slot held A tile c - 1.
    // Before group 0 reads k-step c + 1, the barrier ending phase 4c + 3
    // follows group 0's wait for A tile c + 1 (all its DMA) and group 1's for B
    // tile c + 1 (fired in phases 4c - 3 and 4c - 1: the LPW instructions of B
    // tile c + 2 may be in flight).  The weights, which come from HBM, are thus
    // fired 7 to 11 phases ahead, the activation rows, mostly in L2, 4.
    //
    // A tile ending with k-step c is written out by group 0 in phase 4c + 4 and
    // by group 1 in phase 4c + 5, after the phase's DMA, so that the next waits
    // leave the stores in flight.  Both stage through A tile c's slot: group 1
    // refills it from phase 4c + 5 on, each wave 8 KiB of it, the first half of
    // that in phase 4c + 5 and the second, where the wave stages, in phase
    // 4c + 7.
    constexpr int NF = 2 * (SM + SN);  // fragments of a half k-step
    static_assert(LPW == 8 && SLOT == 4096, "group 1 stages in the half of its DMA share fired last");
    bf16x8_t fa[AM], fb[AN];
    auto read_frag = [&](const char* sa, const char* sb, int h, int n) __attribute__((always_inline)) {
      if (n < AM) {
        fa[n] = read_a(sa, h, n);
      } else {
        fb[n - AM] = read_b(sb, h, n - AM);
      }
    };
    auto fire_range = [&](int lo, int hi) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < LPW; ++j)
        if (j >= lo && j < hi) dma_fire(j);
    };
    auto next2 = [](int slot5) { return slot5 >= 3 ? slot5 - 3 : slot5 + 2; };
    // Row sub-tiles without rows of the tile skip their MFMAs (wave-uniform branches).
    auto multiply = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < SM; ++i)
        if (i < n_act) {
          mfma_row(2 * i, fa[2 * i], fb);
          mfma_row(2 * i + 1, fa[2 * i + 1], fb);
        }
      __builtin_amdgcn_s_setprio(0);
    };
    // Prologue: A tile 0, B tiles 0 and 1.
    int dslot = grp == 0 ? 1 : 0;
    dma_issue(dslot * A_BYTES);
    dslot = next2(dslot);
    if (grp == 0) {
      wait_vmcnt<0>();
    } else {
      dma_issue(dslot * A_BYTES);
      dslot = next2(dslot);
      wait_vmcnt<LPW>();
    }
    barrier();
    if (grp == 1) barrier();
    bool pending = false;  // a finished tile waits for its epilogue
    int pslot = 0;         // ... and stages through this slot
    Tile pt = ct;
    int cb = 0;  // slot of the current B tile; A's is the next one
    for (;;) {
      const int ca = cb == 4 ? 0 : cb + 1;
      const char* sa = ring + ca * A_BYTES;
      const char* sb = ring + cb * A_BYTES;
      // ---- memory phase of the first half
      dma_prepare(dslot * A_BYTES);
      dslot = next2(dslot);
      if (pending) {
        pending = false;
        fire_range(0, LPW / 2);
        if (grp == 0) fire_range(LPW / 2, LPW);
        slot = ring + pslot * A_BYTES + (grp == 0 ? w4 * SLOT : w4 * 2 * SLOT + SLOT);
        epilogue(pt);
        relax = RELAX;
        if (!compute_seek(cj + 1)) break;
#pragma unroll
        for (int n = 0; n < NF; ++n) read_frag(sa, sb, 0, n);
      } else {
#pragma unroll
        for (int n = 0; n < NF; ++n) {
          read_frag(sa, sb, 0, n);
#pragma unroll
          for (int f = 0; f < LPW / 2; ++f)
            if (n == (f + 1) * NF / (LPW / 2) - 1) {
              __builtin_amdgcn_sched_barrier(0);
              dma_fire(f);
              if (grp == 0) dma_fire(LPW / 2 + f);
              __builtin_amdgcn_sched_barrier(0);
            }
        }
      }
      wait_lgkmcnt0();  // the fragments are in registers
      barrier();
      multiply();
      barrier();
      // ---- memory phase of the second half
#pragma unroll
      for (int n = 0; n < NF; ++n) {
        read_frag(sa, sb, 1, n);
        if (grp == 1) {
#pragma unroll
          for (int f = 0; f < LPW / 2; ++f)
            if (n == (f + 1) * NF / (LPW / 2) - 1) {
              __builtin_amdgcn_sched_barrier(0);
              dma_fire(LPW / 2 + f);
              __builtin_amdgcn_sched_barrier(0);
            }
        }
      }
      dma_advance();
      wait_lgkmcnt0();  // ... before the slots can be refilled
      const bool drain = relax > 0;
      relax = 0;
      if (grp == 1) {
        if (drain) {
          wait_vmcnt<LPW + NST>();
        } else {
          wait_vmcnt<LPW>();
        }
      }
      barrier();
      multiply();
      if (grp == 0) {
        if (drain) {
          wait_vmcnt<NST>();
        } else {
          wait_vmcnt<0>();
        }
      }
      barrier();
      if (++ck == ct.nk) {
        pending = true;
        pt = ct;
        pslot = ca;
      }
      cb = next2(cb);
    }
    if (grp == 0) barrier();
  } else if (any) {
    int cstage = 0, dstage = LEAD;
    int parity = 0;  // k-step count of the stream, mod 2
    for (;;) {
      // k-tiles of this step (and, pairwise, the next) landed: this wave's
      // DMA (all but the WAIT younger instructions, plus the last epilogue's
      // stores while they drain), then every wave's, via the barrier; the
      // barrier also retires the reads of the stages the next DMA overwrites.
      const bool drain = relax > 0;
      if (relax > 0) --relax;
      if (!PAIR || parity == 0) {
        if (drain) {
          wait_vmcnt<WAIT + NST>();
        } else {
          wait_vmcnt<WAIT>();
        }
        barrier();
      }
      parity ^= 1;
      dma_prepare(dstage * STAGE_BYTES);
      if (n_act > 0) {
        // Issue priority while the wave feeds its MFMAs, so that on a shared
        // SIMD the wave with matrix work ready goes before the other wave's
        // address arithmetic and epilogue (0.4-0.6% on the expert GEMMs).
        __builtin_amdgcn_s_setprio(1);
        compute(n_act, ring + cstage * STAGE_BYTES);
        __builtin_amdgcn_s_setprio(0);
      } else {
#pragma unroll
        for (int j = 0; j < LPW; ++j) dma_fire(j);
      }
      dma_advance();
      dstage = dstage + 1 == STAGES ? 0 : dstage + 1;
      cstage = cstage + 1 == STAGES ? 0 : cstage + 1;
      if (++ck == ct.nk) {
        slot = ring + (cstage == 0 ? STAGES - 1 : cstage - 1) * STAGE_BYTES + wave * SLOT;
        barrier();
        epilogue(ct);
        relax = RELAX;
        if (!compute_seek(cj + 1)) break;
      }
    }
  }
  wait_vmcnt<0>();  // retire the trailing DMA (zeros) before the LDS is released
}

// ------------------------------------------------------------ host side

namespace {

int round_up(int x, int m) { return (x + m - 1) / m * m; }

constexpr int64_t kMaxRsrcBytes = (1ll << 31) - 64;

int set_bytes(GemmParams& p, int64_t a_bytes, int64_t b_bytes, int64_t c_bytes, const char* name) {
  MOE_REQUIRE(a_bytes < kMaxRsrcBytes && b_bytes < kMaxRsrcBytes && c_bytes < kMaxRsrcBytes, MOE_ERR_UNSUPPORTED,
              "%s: operand of %lld / %lld / %lld bytes exceeds the 2 GiB buffer-resource range", name,
              (long long)a_bytes, (long long)b_bytes, (long long)c_bytes);
  p.a_bytes = static_cast<uint32_t>(a_bytes);
  p.b_bytes = static_cast<uint32_t>(b_bytes);
  p.c_bytes = static_cast<uint32_t>(c_bytes);
  return MOE_OK;
}

template <int MODE, bool B_KCONTIG, int EPI, class CFG>
int launch(GemmParams& p, hipStream_t stream, const char* name) {
  if (p.k_splits < 1) {
    p.k_splits = 1;
    p.k_chunk = p.K;
  }
  // Output column tiles; a SwiGLU tile covers BN/2 act columns (gate + up rows).
  p.n_tiles = (EPI == EPI_SWIGLU_FWD) ? (p.swiglu_I + CFG::BN / 2 - 1) / (CFG::BN / 2)
                                      : (p.N + CFG::BN - 1) / CFG::BN;
  int64_t tiles;  // exact, or (grouped MG) the worst case; the kernel counts the real tiles itself
  if (MODE == MODE_MG) {
    p.m_tiles_max = (p.M + CFG::BM - 1) / CFG::BM + (p.offs ? p.G : 0);
    tiles = static_cast<int64_t>(p.m_tiles_max) * p.n_tiles * (p.offs ? 1 : p.k_splits);
  } else {
    p.m_tiles_max = (p.M + CFG::BM - 1) / CFG::BM;
    tiles = static_cast<int64_t>(p.G) * p.m_tiles_max * p.n_tiles;
  }
  if (tiles <= 0) return MOE_OK;
  MOE_REQUIRE(tiles < (1ll << 30), MOE_ERR_UNSUPPORTED, "%s: too many tiles", name);
  if (MODE == MODE_KG) {  // cost split when every group cost and their sum fit in 30 bits
    const int64_t per_group = static_cast<int64_t>(p.n_tiles) * p.m_tiles_max;
    const int64_t bound = per_group * (p.rows / CFG::BK + p.G * (1 + kEpiSteps));
    p.cost_split = (p.offs && p.G > 1 && bound < (1ll << 30)) ? 1 : 0;
  }
  p.total_tiles = static_cast<int>(tiles);
  // Persistent grid: as many blocks as fit at once (capped by the tile
  // count), a multiple of the XCD count.
  const int dev = current_device();
  const int occ = cached_blocks_per_cu(dev, reinterpret_cast<const void*>(&grouped_gemm_kernel<MODE, B_KCONTIG, EPI, CFG>),
                                       CFG::kThreads, 0);
  const int64_t resident = static_cast<int64_t>(device_cus(dev)) * occ / kNumXcd * kNumXcd;
  const int grid = static_cast<int>(std::max<int64_t>(kNumXcd, std::min<int64_t>(round_up(static_cast<int>(tiles),
                                                                                          kNumXcd),
                                                                                 resident)));
  hipLaunchKernelGGL((grouped_gemm_kernel<MODE, B_KCONTIG, EPI, CFG>), dim3(grid), dim3(CFG::kThreads), 0, stream,
                     p);
  return launch_status(name);
}

// Bounds of launch_expert's rule, in mean rows per expert.
constexpr int64_t kFewMaxMeanRows = 2;
constexpr int64_t kSlimMaxMeanRows = 32;
constexpr int64_t kMidMaxMeanRows = 112;
constexpr int64_t kBigMaxMeanRows = 224;
constexpr int64_t kWideMaxMeanRows = 288;
constexpr int64_t kMidAgainMaxMeanRows = 352;
// Weight rows of at least this many elements (8 KiB) keep the larger tiles
// down to the fewest rows, up to kLongRowMaxMeanRows mean rows.
constexpr int kLongRow = 4096;
constexpr int64_t kLongRowMaxMeanRows = 64;

// Expert GEMM over grouped rows; the tile by the mean rows per expert (the
// real counts stay on the device).  An expert that fits one m-tile streams its
// weights through one CU's LDS per n-tile, so the tile is the smallest that
// holds nearly every expert under uniform routing, which leaves the most LDS
// for weights in flight; experts above it take further m-tiles.  Every tile
// adds an output's products in the same order: the results are the same bits.
// Kernel times in us at H 2048, I 768, 128 experts, top-8 (up_fwd / down_fwd /
// down_dgrad with its SwiGLU pass / up_dgrad; 64-, 128-, 320-row tiles and the
// 256-row ping-pong one, timed in turn):
//   mean rows      64-row             128-row            320-row            256-row
//     3 (T 48)     154/ 70/ 78/130    156/ 71/ 79/130    173/ 89/ 89/129    172/ 87/103/153
//    19 (T 301)    168/ 78/ 86/139    168/ 79/ 86/140    186/ 93/ 96/137    182/ 93/108/160
//    48 (T 768)    198/ 95/ 97/160    182/ 88/ 98/147    197/103/110/154    188/101/117/173
//    96 (T 1531)   216/109/118/182    197/ 98/117/157    214/113/130/173    204/108/132/186
//   131 (T 2100)   242/127/145/217    218/117/147/194    232/122/148/185    217/114/146/197
//   162 (T 2600)   267/138/169/240    240/123/146/203    243/126/163/206    226/117/156/199
//   200 (T 3200)   309/164/193/279    253/129/156/215    260/134/178/232    235/122/168/212
//   256 (T 4096)   363/202/229/338    289/152/191/259    281/148/205/256    297/151/222/283
//   312 (T 5000)   407/227/259/395    322/170/219/299    353/201/222/336    333/180/217/338
// Narrow outputs (at most 1024 columns: down_dgrad at I 768) have few n-tiles,
// and the 128-row tile's finer grid keeps winning up to kWideMaxMeanRows.
// Past that, up to kMidAgainMaxMeanRows, an expert is two m-tiles of the
// larger tiles, little more than half filled, and three nearly full ones of
// the 128-row tile.  Weight rows of 8 KiB (H 4096) are faster on the larger
// tiles while they are streamed for few rows: at 19 mean rows up_fwd takes 574
// on the 256-row tile against 592 to 594, up_dgrad 501 on the 320-row tile
// against 548 to 554.
//
// Calls of few tiles (small layers, a rank's share of the experts): a tile that
// leaves CUs idle costs its whole time, so the smallest that runs all of them
// at once is taken whatever the mean.  The input gradients' 256-row tiles, when
// one round of them is all, leave the ping-pong loop, which pays for its longer
// start from the second tile on.  us, the mean-row rule's choice -> now:
//   H 512, I 256, 8 experts, mean 400: the four GEMMs 21/14/23/20 (256-row)
//     -> 11/8/13/10 (64-row)
//   H 1024, I 512, 32 experts, mean 400: down_dgrad 44 (256-row) -> 33 (128-row),
//     up_dgrad 34 -> 32 (256-row, paired barriers)
//   H 1536, I 640, 16 experts, mean 288: up_fwd 56 (320-row) -> 28 (128-row)
//   H 2048, I 768, 32 experts, mean 352: down_dgrad 76 (128-row) -> 63 (256-row)
//   H 4096, I 1536, 16 experts, mean 320: down_dgrad 123 (128-row) -> 103 (256-row)
// Skewed routing: with few rows per expert on average a heavy expert takes
// several of the small tiles.  Zipf(1) counts still prefer them (H 2048, I 768,
// 128 experts, 32 mean rows: 64-row 169/84/88/148, 320-row 207/115/122/178; 96
// mean rows: 128-row 209/101/131/173, 320-row 266/132/157/214).  Where a
// sixteenth of the experts takes every row the larger tiles are up to 1.4
// times faster (H 4096, I 1536, 32 mean rows: down_fwd 83 on 64-row, 56 on
// 320-row tiles; 96 mean rows at H 2048: 90/51/76/91 on 128-row, 79/60/85/105).
// Large outputs at few rows are a few percent faster on the 320-row tile in the
// input gradients (H 2048, I 1408, 64 experts, 16 mean rows: up_dgrad 124 on
// 64-row, 118 on 320-row tiles), which under Zipf counts costs a third (32 mean
// rows: 192 against 142).
//
// The forward GEMMs of a few decoded tokens go to few_rows, which times both
// sides.
template <bool B_KCONTIG, int EPI>
int launch_expert(GemmParams& p, hipStream_t stream, const char* name) {
  const int out_cols = (EPI == EPI_SWIGLU_FWD) ? 2 * p.swiglu_I : p.N;
  const int64_t rows = p.rows, G = p.G;
  if constexpr (B_KCONTIG) {
    if (p.offs && rows <= kFewMaxMeanRows * G) {  // (a single group without offsets: the tiles)
      constexpr bool swiglu = EPI == EPI_SWIGLU_FWD;
      return few_rows(FewRows{p.A, p.B, static_cast<bf16_t*>(p.C), static_cast<bf16_t*>(p.C2), p.offs, p.G, p.rows,
                              swiglu ? p.swiglu_I : p.N, p.K},
                      swiglu, stream, name);
    }
  }
  const bool long_rows = p.ldb >= kLongRow && rows <= kLongRowMaxMeanRows * G;
  // Whether tiles of bm rows, at `per` rows per expert, all run at once.
  const int64_t n_tiles = (out_cols + 255) / 256, cus = device_cus(current_device());
  auto one_round = [&](int bm, double per) {
    return G * n_tiles * std::max<int64_t>(1, static_cast<int64_t>(std::ceil(per / bm))) <= cus;
  };
  const double mean = static_cast<double>(rows) / static_cast<double>(G);
  const double high = mean + 3.0 * std::sqrt(mean);  // few experts have more, under uniform routing
  if (!long_rows && (rows <= kSlimMaxMeanRows * G || one_round(SlimTile::BM, high)))
    return launch<MODE_MG, B_KCONTIG, EPI, SlimTile>(p, stream, name);
  if ((!long_rows && (rows <= (out_cols <= 1024 ? kWideMaxMeanRows : kMidMaxMeanRows) * G || one_round(MidTile::BM, high))) ||
      (rows > kWideMaxMeanRows * G && rows <= kMidAgainMaxMeanRows * G &&
       (one_round(MidTile::BM, mean) || !one_round(PingTile::BM, mean))))
    return launch<MODE_MG, B_KCONTIG, EPI, MidTile>(p, stream, name);
  // Up to 320 rows per expert in one m-tile, and the input gradients of long
  // weight rows.
  if (rows <= kWideMaxMeanRows * G && (rows > kBigMaxMeanRows * G || (long_rows && !B_KCONTIG)))
    return launch<MODE_MG, B_KCONTIG, EPI, WideTile>(p, stream, name);
  if constexpr (!B_KCONTIG) {
    if (one_round(BigTile::BM, mean)) return launch<MODE_MG, B_KCONTIG, EPI, BigTile>(p, stream, name);
  }
  return launch<MODE_MG, B_KCONTIG, EPI, PingTile>(p, stream, name);
}

// Operand checks.  `a` holds M rows, as does `b` when b_rows (the weight
// gradient's second operand); an operand of zero rows may be NULL.
int check_common(const void* a, const void* b, const int32_t* offs, int64_t G, int64_t M, int64_t N, int64_t K,
                 bool b_rows = false) {
  MOE_REQUIRE((a || M == 0) && (b || (b_rows && M == 0)), MOE_ERR_INVALID, "grouped gemm: null operand");
  MOE_REQUIRE(G >= 1 && G <= 4096, MOE_ERR_UNSUPPORTED, "grouped gemm: G=%lld outside [1,4096]", (long long)G);
  MOE_REQUIRE(offs || G == 1, MOE_ERR_INVALID, "grouped gemm: offs may be NULL only for G == 1");
  MOE_REQUIRE(M >= 0 && N > 0 && K > 0, MOE_ERR_INVALID, "grouped gemm: bad sizes M=%lld N=%lld K=%lld",
              (long long)M, (long long)N, (long long)K);
  MOE_REQUIRE(M < (1ll << 31) && N < (1 << 30) && K < (1 << 30), MOE_ERR_UNSUPPORTED, "grouped gemm: size overflow");
  MOE_REQUIRE(N % 8 == 0 && K % 8 == 0, MOE_ERR_UNSUPPORTED,
              "grouped gemm: N (%lld) and K (%lld) must be multiples of 8", (long long)N, (long long)K);
  MOE_REQUIRE(aligned16(a) && aligned16(b), MOE_ERR_INVALID, "grouped gemm: operands must be 16-byte aligned");
  return MOE_OK;
}

}  // namespace

// Router logits as split-K partials: partials[s][T][E] (f32), s < splits, each
// over the reduction range [s*k_chunk, (s+1)*k_chunk) of H.
int router_logits_partials(const bf16_t* x, const bf16_t* wr, float* partials, int T, int H, int E, int splits,
                           int k_chunk, hipStream_t stream) {
  GemmParams p{};
  p.A = x;
  p.B = wr;
  p.C = partials;
  p.G = 1;
  p.rows = p.M = T;
  p.N = E;
  p.K = H;
  p.lda = H;
  p.ldb = H;
  p.ldc = E;
  p.k_splits = splits;
  p.k_chunk = k_chunk;
  p.split_stride = static_cast<int64_t>(T) * E;
  int rc = set_bytes(p, static_cast<int64_t>(T) * H * 2, static_cast<int64_t>(E) * H * 2,
                     static_cast<int64_t>(T) * E * 4, "router logits");
  if (rc) return rc;
  return launch<MODE_MG, true, EPI_F32, SmallTile>(p, stream, "router logits (split-K)");
}

// Router weight gradient as row-chunk partials: partials[c][E][H] (f32) over
// rows [c*chunk_rows, (c+1)*chunk_rows) of T.
int router_wgrad_partials(const bf16_t* dl, const bf16_t* x, float* partials, int T, int H, int E, int chunks,
                          int chunk_rows, hipStream_t stream) {
  GemmParams p{};
  p.A = dl;
  p.B = x;
  p.C = partials;
  p.offs = nullptr;
  p.G = chunks;
  p.chunk_rows = chunk_rows;
  p.rows = T;
  p.M = E;
  p.N = H;
  p.lda = E;
  p.ldb = H;
  p.ldc = H;
  p.ldp = 1;  // f32 destination
  p.stride_cg = static_cast<int64_t>(E) * H;
  int rc = set_bytes(p, static_cast<int64_t>(T) * E * 2, static_cast<int64_t>(T) * H * 2,
                     static_cast<int64_t>(E) * H * 4, "router wgrad");
  if (rc) return rc;
  return launch<MODE_KG, false, EPI_WGRAD, SmallTile>(p, stream, "router wgrad (row chunks)");
}

// Router input gradient dx[T,H] = dl[T,E] . wr[E,H] (single group, reduction E).
int router_dgrad(const bf16_t* dl, const bf16_t* wr, bf16_t* dx, int T, int H, int E, hipStream_t stream) {
  GemmParams p{};
  p.A = dl;
  p.B = wr;
  p.C = dx;
  p.G = 1;
  p.rows = p.M = T;
  p.N = H;
  p.K = E;
  p.lda = E;
  p.ldb = H;
  p.ldc = H;
  int rc = set_bytes(p, static_cast<int64_t>(T) * E * 2, static_cast<int64_t>(E) * H * 2,
                     static_cast<int64_t>(T) * H * 2, "router dgrad");
  if (rc) return rc;
  return launch<MODE_MG, false, EPI_BF16, SmallTile>(p, stream, "router dgrad");
}

// SwiGLU backward, elementwise and in place over d_pre [rows, 2I]: the up
// half holds d_act (the bf16 input-gradient GEMM output) on entry; on exit
// d_pre = (d_gate | d_up) with the reference's bf16 roundings:
//   d_up = d * silu(gate),  d_silu = d * up,  d_gate = d_silu * s (1 + gate (1 - s)).
// One lane per 8 columns (16-byte loads and stores).  Only the rows of the
// groups, [0, offs[G-1]), are touched (read on the device, no host sync): the
// sentinel tail past them holds no pre-activations and stays as it is.
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(bf16_t* __restrict__ d_pre, const bf16_t* __restrict__ pre,
                                                         const int32_t* __restrict__ offs, int G, unsigned rows,
                                                         unsigned I) {
  const unsigned cpr = I / 8;  // 8-column chunks per half row
  const unsigned valid = offs ? static_cast<unsigned>(min(max(offs[G - 1], 0), static_cast<int>(rows))) : rows;
  const unsigned total = valid * cpr;
  for (unsigned c = blockIdx.x * blockDim.x + threadIdx.x; c < total; c += gridDim.x * blockDim.x) {
    const unsigned r = c / cpr, k = (c - r * cpr) * 8;
    bf16_t* dr = d_pre + static_cast<size_t>(r) * 2 * I;
    const bf16_t* pr = pre + static_cast<size_t>(r) * 2 * I;
    const uint4 dv = ntload16(dr + I + k);  // the last reads of d_act and of the saved pre-activations
    const uint4 gv = ntload16(pr + k);
    const uint4 uv = ntload16(pr + I + k);
    const uint32_t dw[4] = {dv.x, dv.y, dv.z, dv.w}, gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
    uint32_t og[4], ou[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float dg2[2], du2[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float d = h ? hi_bf16(dw[e]) : lo_bf16(dw[e]);
        const float g = h ? hi_bf16(gw[e]) : lo_bf16(gw[e]);
        const float u = h ? hi_bf16(uw[e]) : lo_bf16(uw[e]);
        const float sg = sigmoid_f(g);
        du2[h] = d * bf16_to_f32(f32_to_bf16(g * sg));
        dg2[h] = bf16_to_f32(f32_to_bf16(d * u)) * sg * (1.0f + g * (1.0f - sg));
      }
      og[e] = pack_bf16x2(dg2[0], dg2[1]);
      ou[e] = pack_bf16x2(du2[0], du2[1]);
    }
    *reinterpret_cast<uint4*>(dr + k) = make_uint4(og[0], og[1], og[2], og[3]);
    *reinterpret_cast<uint4*>(dr + I + k) = make_uint4(ou[0], ou[1], ou[2], ou[3]);
  }
}

}  // namespace moe

using namespace moe;

extern "C" int moe_grouped_gemm_swiglu_fwd(const void* xp, const void* w_gate_up, const int32_t* offs, int64_t G,
                                           int64_t M, int64_t H, int64_t I, void* act, void* pre, void* stream) {
  int rc = check_common(xp, w_gate_up, offs, G, M, 2 * I, H);
  if (rc) return rc;
  if (M == 0) return MOE_OK;  // no rows: empty outputs may be NULL
  MOE_REQUIRE(act && aligned16(act) && (!pre || aligned16(pre)), MOE_ERR_INVALID, "swiglu fwd: bad output pointer");
  GemmParams p{};
  p.A = static_cast<const bf16_t*>(xp);
  p.B = static_cast<const bf16_t*>(w_gate_up);
  p.C = act;
  p.C2 = pre;
  p.offs = offs;
  p.G = static_cast<int>(G);
  p.rows = p.M = static_cast<int>(M);
  p.N = static_cast<int>(2 * I);
  p.K = static_cast<int>(H);
  p.lda = H;
  p.ldb = H;
  p.ldc = I;
  p.ldp = 2 * I;
  p.stride_bg = 2 * I * H;
  p.swiglu_I = static_cast<int>(I);
  if ((rc = set_bytes(p, M * H * 2, 2 * I * H * 2, M * I * 2, "moe_grouped_gemm_swiglu_fwd"))) return rc;
  p.c2_bytes = pre ? static_cast<uint32_t>(M * 2 * I * 2) : 0u;  // < a_bytes-range: checked below
  MOE_REQUIRE(M * 2 * I * 2 < kMaxRsrcBytes, MOE_ERR_UNSUPPORTED, "swiglu fwd: pre-activation exceeds 2 GiB");
  return launch_expert<true, EPI_SWIGLU_FWD>(p, as_stream(stream), "moe_grouped_gemm_swiglu_fwd");
}

extern "C" int moe_grouped_gemm_fwd(const void* a, const void* w, const int32_t* offs, int64_t G, int64_t M, int64_t N,
                                    int64_t K, void* c, void* stream) {
  int rc = check_common(a, w, offs, G, M, N, K);
  if (rc) return rc;
  if (M == 0) return MOE_OK;
  MOE_REQUIRE(c && aligned16(c), MOE_ERR_INVALID, "grouped gemm fwd: bad output pointer");
  GemmParams p{};
  p.A = static_cast<const bf16_t*>(a);
  p.B = static_cast<const bf16_t*>(w);
  p.C = c;
  p.offs = offs;
  p.G = static_cast<int>(G);
  p.rows = p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.lda = K;
  p.ldb = K;
  p.ldc = N;
  p.stride_bg = N * K;
  if ((rc = set_bytes(p, M * K * 2, N * K * 2, M * N * 2, "moe_grouped_gemm_fwd"))) return rc;
  return launch_expert<true, EPI_BF16>(p, as_stream(stream), "moe_grouped_gemm_fwd");
}

// Router logits: f32 output, single group, no split.
extern "C" int moe_router_logits_fwd(const void* x, const void* wr, float* logits, int64_t T, int64_t H, int64_t E,
                                     void* stream) {
  int rc = check_common(x, wr, nullptr, 1, T, E, H);
  if (rc) return rc;
  if (T == 0) return MOE_OK;
  MOE_REQUIRE(logits && aligned16(logits), MOE_ERR_INVALID, "router logits: bad output pointer");
  return router_logits_partials(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(wr), logits,
                                static_cast<int>(T), static_cast<int>(H), static_cast<int>(E), 1,
                                static_cast<int>(H), as_stream(stream));
}

extern "C" int moe_grouped_gemm_dgrad(const void* dc, const void* w, const int32_t* offs, int64_t G, int64_t M,
                                      int64_t N, int64_t K, void* da, void* stream) {
  // da[M,K] = dc[M,N] . w[g] (w [G,N,K]): GEMM-internal reduction over N, output width K.
  int rc = check_common(dc, w, offs, G, M, K, N);
  if (rc) return rc;
  if (M == 0) return MOE_OK;
  MOE_REQUIRE(da && aligned16(da), MOE_ERR_INVALID, "grouped gemm dgrad: bad output pointer");
  GemmParams p{};
  p.A = static_cast<const bf16_t*>(dc);
  p.B = static_cast<const bf16_t*>(w);
  p.C = da;
  p.offs = offs;
  p.G = static_cast<int>(G);
  p.rows = p.M = static_cast<int>(M);
  p.N = static_cast<int>(K);
  p.K = static_cast<int>(N);
  p.lda = N;
  p.ldb = K;
  p.ldc = K;
  p.stride_bg = N * K;
  if ((rc = set_bytes(p, M * N * 2, N * K * 2, M * K * 2, "moe_grouped_gemm_dgrad"))) return rc;
  return launch_expert<false, EPI_BF16>(p, as_stream(stream), "moe_grouped_gemm_dgrad");
}

extern "C" int moe_grouped_gemm_dgrad_swiglu_bwd(const void* dy, const void* w_down, const void* pre,
                                                 const int32_t* offs, int64_t G, int64_t M, int64_t H, int64_t I,
                                                 void* d_pre, void* stream) {
  // d_act[M,I] = dy[M,H] . w_down[g] (w_down [G,H,I]) into the up half of
  // d_pre, then the SwiGLU backward in place.
  int rc = check_common(dy, w_down, offs, G, M, I, H);
  if (rc) return rc;
  if (M == 0) return MOE_OK;
  MOE_REQUIRE(pre && d_pre && aligned16(pre) && aligned16(d_pre), MOE_ERR_INVALID,
              "dgrad swiglu: bad pre/d_pre pointer");
  MOE_REQUIRE(M * I / 8 < (1ll << 31), MOE_ERR_UNSUPPORTED, "dgrad swiglu: too many rows");
  GemmParams p{};
  p.A = static_cast<const bf16_t*>(dy);
  p.B = static_cast<const bf16_t*>(w_down);
  p.C = static_cast<bf16_t*>(d_pre) + I;
  p.offs = offs;
  p.G = static_cast<int>(G);
  p.rows = p.M = static_cast<int>(M);
  p.N = static_cast<int>(I);
  p.K = static_cast<int>(H);
  p.lda = H;
  p.ldb = I;
  p.ldc = 2 * I;
  p.stride_bg = H * I;
  if ((rc = set_bytes(p, M * H * 2, H * I * 2, (M * 2 * I - I) * 2, "moe_grouped_gemm_dgrad_swiglu_bwd"))) return rc;
  hipStream_t st = as_stream(stream);
  if ((rc = launch_expert<false, EPI_BF16>(p, st, "moe_grouped_gemm_dgrad_swiglu_bwd"))) return rc;
  const int64_t chunks = M * I / 8;
  const int grid = static_cast<int>(std::min<int64_t>((chunks + 255) / 256, 4096));
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3(grid), dim3(256), 0, st, static_cast<bf16_t*>(d_pre),
                     static_cast<const bf16_t*>(pre), offs, static_cast<int>(G), static_cast<unsigned>(M),
                     static_cast<unsigned>(I));
  return launch_status("moe_grouped_gemm_dgrad_swiglu_bwd (swiglu)");
}

namespace {
int wgrad(const void* dc, const void* a, const int32_t* offs, int64_t G, int64_t M, int64_t N, int64_t K, void* dw,
          int dw_is_f32, int accumulate, int64_t bucket_rows, int64_t bucket_stride, void* stream, const char* name) {
  // dw[g][N,K] = dc[rows g, N]^T . a[rows g, K]: GEMM-internal output N x K, reduction over rows.
  // With no rows at all dW is still written (zeros) or left as it is (accumulate).
  int rc = check_common(dc, a, offs, G, M, N, K, /*b_rows=*/true);
  if (rc) return rc;
  MOE_REQUIRE(dw && aligned16(dw), MOE_ERR_INVALID, "%s: bad output pointer", name);
  if (M == 0) dc = a = dw;  // zero-byte operand resources: never read, but on a valid base
  GemmParams p{};
  p.A = static_cast<const bf16_t*>(dc);
  p.B = static_cast<const bf16_t*>(a);
  p.C = dw;
  p.offs = offs;
  p.G = static_cast<int>(G);
  p.rows = static_cast<int>(M);
  p.M = static_cast<int>(N);
  p.N = static_cast<int>(K);
  p.K = 0;
  p.lda = N;
  p.ldb = K;
  p.ldc = K;
  p.ldp = dw_is_f32 ? 1 : 0;
  p.stride_cg = N * K;
  p.accumulate = accumulate ? 1 : 0;
  p.chunk_rows = static_cast<int>(M);
  p.bucket_rows = static_cast<int>(bucket_rows);
  p.bucket_stride = bucket_stride;
  if ((rc = set_bytes(p, M * N * 2, M * K * 2, N * K * (dw_is_f32 ? 4 : 2), name))) return rc;
  return launch<MODE_KG, false, EPI_WGRAD, BigTile>(p, as_stream(stream), name);
}
}  // namespace

extern "C" int moe_grouped_gemm_wgrad(const void* dc, const void* a, const int32_t* offs, int64_t G, int64_t M,
                                      int64_t N, int64_t K, void* dw, int dw_is_f32, int accumulate, void* stream) {
  return wgrad(dc, a, offs, G, M, N, K, dw, dw_is_f32, accumulate, 0, 0, stream, "moe_grouped_gemm_wgrad");
}

extern "C" int moe_grouped_gemm_wgrad_bucket(const void* dc, const void* a, const int32_t* offs, int64_t G, int64_t M,
                                             int64_t N, int64_t K, void* bucket, int64_t bucket_rows,
                                             int64_t bucket_stride, int dw_is_f32, int accumulate, void* stream) {
  const char* name = "moe_grouped_gemm_wgrad_bucket";
  MOE_REQUIRE(bucket_rows >= 1 && bucket_rows <= G, MOE_ERR_INVALID, "%s: bucket_rows=%lld outside [1, G=%lld]", name,
              (long long)bucket_rows, (long long)G);
  MOE_REQUIRE(bucket_stride >= bucket_rows * N * K, MOE_ERR_INVALID,
              "%s: bucket_stride=%lld smaller than one rank's %lld x %lld x %lld shard", name,
              (long long)bucket_stride, (long long)bucket_rows, (long long)N, (long long)K);
  MOE_REQUIRE((bucket_stride * (dw_is_f32 ? 4 : 2)) % 16 == 0, MOE_ERR_UNSUPPORTED,
              "%s: rank chunks of %lld elements are not 16-byte aligned", name, (long long)bucket_stride);
  return wgrad(dc, a, offs, G, M, N, K, bucket, dw_is_f32, accumulate, bucket_rows, bucket_stride, stream, name);
}
