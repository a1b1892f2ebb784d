// The forward expert GEMMs of a decoding batch: experts of a few rows, whose
// weights are streamed from HBM once for almost no arithmetic.
//
// The tiled kernel (grouped_gemm.hip) gives such an expert ceil(N / 256) blocks
// that each walk all of K, so one decoded token keeps 48 of 256 CUs busy, and
// it stages the weights through LDS behind a block barrier per k-tile.  Here
// every wave is a block of its own and takes 16 weight rows (SwiGLU: 16 gate
// rows and the matching 16 up rows) of one expert for 16 of its rows: 384 waves
// for the same token.  A wave walks all of K in order, so that an output's
// products are added exactly as the tiled kernel adds them: a token's results
// are the same bits in a batch of any size.  Weights and rows go straight into
// the MFMA operand registers, D k-steps of loads in flight; there is no LDS and
// no barrier.  Bound by the weights' bytes from a few tokens on, by latency and
// the launch for one token.
//
// Up / down projection in us, weights out of the caches, against the 64-row
// tile: H 2048, I 768, 128 experts, 8 rows of 8 experts 25/16 against 38/22,
// one row in each of 64 134/80 against 140/85, 256 rows 193/126 against 194/126;
// H 4096, I 1536: 81/43 against 91/47 and 553/298 against 582/315 (8 and 256
// rows).  Reductions that are no multiple of anything: K 2304 / 1000 (H 2304,
// I 1000, 64 experts, 64 rows) 161/109 against 165/123, K 2560 (32 experts, 8
// rows) 85/44 against 87/55, K 14336 (8 experts, 8 rows) 231 against 257.
// Skewed (a sixteenth of the experts holds all rows, 16 rows each) 31/20 against
// 40/22.  In flight: 12 k-steps of the up projection (8: 1.00 of the time, 4:
// 1.05, 24: 1.04, over sizes), 16 of the down projection (8: 1.02, 24: 1.00).
#include "dma.h"
#include "gemm.h"

namespace moe {
namespace {

constexpr int kFewXcd = 8;

// D: k-steps (32 deep) of loads in flight.
template <int D, bool SWIGLU>
__global__ __launch_bounds__(kWave) void few_rows_kernel(const FewRows p, int n_tiles, uint32_t a_bytes,
                                                         uint32_t w_bytes) {
  constexpr int NT = SWIGLU ? 2 : 1;  // 16-row weight tiles: the gate rows and the matching up rows
  const int lane = threadIdx.x;
  const int i16 = lane & 15, q = lane >> 4;

  // Tasks in group-major order, then weight tile, then 16-row chunk (whose
  // waves read the same weights); an XCD's blocks take neighbouring tasks.
  auto rows_of = [&](int g, int& lo) {
    int hi = 0;
    lo = 0;
    if (g < p.G) {
      hi = min(max(p.offs[g], 0), p.rows);  // clamped: malformed offsets never address outside [0, rows)
      lo = g ? min(max(p.offs[g - 1], 0), hi) : 0;
    }
    return hi - lo;
  };
  int chunks = 0;  // 16-row chunks over all groups
  for (int c0 = 0; c0 < p.G; c0 += kWave) {
    int lo;
    const int cnt = rows_of(c0 + lane, lo);
    chunks += __builtin_amdgcn_readlane(wave_inclusive_scan((cnt + 15) / 16), kWave - 1);
  }
  const int total = __builtin_amdgcn_readfirstlane(chunks) * n_tiles;
  const int share = (total + kFewXcd - 1) / kFewXcd;
  const int idx = blockIdx.x / kFewXcd, task = (blockIdx.x % kFewXcd) * share + idx;
  if (idx >= share || task >= total) return;
  int g = 0, r0 = 0, rows = 0, tile = 0;
  for (int c0 = 0, base = 0; c0 < p.G; c0 += kWave) {
    int lo;
    const int cnt = rows_of(c0 + lane, lo);
    const int n = n_tiles * ((cnt + 15) / 16);
    const int incl = wave_inclusive_scan(n);
    const int tot = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (task < base + tot) {
      const int w = __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(base + incl > task)));
      const int local = task - base - __builtin_amdgcn_readlane(incl - n, w);
      const int gc = __builtin_amdgcn_readlane(cnt, w), nc = (gc + 15) / 16;
      tile = local / nc;
      const int chunk = local - tile * nc;
      g = c0 + w;
      r0 = __builtin_amdgcn_readlane(lo, w) + 16 * chunk;
      rows = min(16, gc - 16 * chunk);
      break;
    }
    base += tot;
  }

  // Lane (i16, q): row i16 of each operand, k 8 q .. 8 q + 7 of a k-step.
  const __amdgpu_buffer_rsrc_t rsA = make_rsrc(p.A, a_bytes);
  const __amdgpu_buffer_rsrc_t rsW = make_rsrc(p.W + static_cast<int64_t>(g) * (SWIGLU ? 2 : 1) * p.N * p.K, w_bytes);
  const uint32_t k2 = static_cast<uint32_t>(p.K) * 2u, lane_k = 16u * q;
  const uint32_t x_row = i16 < rows ? static_cast<uint32_t>(r0 + i16) * k2 + lane_k : kOOB;
  uint32_t w_row[NT];
#pragma unroll
  for (int s = 0; s < NT; ++s) {
    const int n = tile * 16 + i16;
    w_row[s] = n < p.N ? static_cast<uint32_t>(s * p.N + n) * k2 + lane_k : kOOB;
  }
  u32x4_t xf[D], wf[D][NT];
  auto load = [&](int u, int ks) __attribute__((always_inline)) {
    const uint32_t off = 64u * ks;
    const bool in = lane_k + off < k2;
    // (Not non-temporal: an operand load takes 64 bytes of each row, and the
    // line has to stay for the next one.)
#pragma unroll
    for (int s = 0; s < NT; ++s) wf[u][s] = __builtin_amdgcn_raw_buffer_load_b128(rsW, in ? w_row[s] + off : kOOB, 0, 0);
    xf[u] = __builtin_amdgcn_raw_buffer_load_b128(rsA, in ? x_row + off : kOOB, 0, 0);
  };
  f32x4_t acc[NT];
#pragma unroll
  for (int s = 0; s < NT; ++s) acc[s] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](int u) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < NT; ++s)
      acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[u][s]),
                                                       __builtin_bit_cast(bf16x8_t, xf[u]), acc[s], 0, 0, 0);
  };
  const int nks = (p.K + 31) / 32;
#pragma unroll
  for (int u = 0; u < D; ++u) load(u, u);
  int k0 = 0;
  for (; k0 + D < nks; k0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      multiply(u);
      load(u, k0 + D + u);
    }
  }
#pragma unroll
  for (int u = 0; u < D; ++u) multiply(u);  // (past K: zeros)

  // The operands are swapped, so the lane holds columns 4 q .. 4 q + 3 of row i16.
  const int n = tile * 16 + 4 * q;
  if (i16 >= rows || n >= p.N) return;
  const int64_t r = r0 + i16;
  bf16_t* c = p.C + r * p.N + n;
  if constexpr (SWIGLU) {
    float a[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      a[e] = bf16_to_f32(f32_to_bf16(silu_f(bf16_to_f32(f32_to_bf16(acc[0][e]))))) *
             bf16_to_f32(f32_to_bf16(acc[1][e]));
    *reinterpret_cast<uint2*>(c) = make_uint2(pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]));
    if (p.pre) {
      bf16_t* pre = p.pre + r * 2 * p.N + n;
#pragma unroll
      for (int s = 0; s < 2; ++s)
        *reinterpret_cast<uint2*>(pre + s * p.N) =
            make_uint2(pack_bf16x2(acc[s][0], acc[s][1]), pack_bf16x2(acc[s][2], acc[s][3]));
    }
  } else {
    *reinterpret_cast<uint2*>(c) = make_uint2(pack_bf16x2(acc[0][0], acc[0][1]), pack_bf16x2(acc[0][2], acc[0][3]));
  }
}

}  // namespace

int few_rows(const FewRows& p, bool swiglu, hipStream_t stream, const char* name) {
  const int n_tiles = (p.N + 15) / 16;
  // At most one 16-row chunk per nonempty group and one more per 16 further rows.
  const int64_t groups = p.G < p.rows ? p.G : p.rows;
  const int64_t most = (groups + (p.rows - groups) / 16) * n_tiles;
  MOE_REQUIRE(most < (1ll << 30), MOE_ERR_UNSUPPORTED, "%s: too many tiles", name);
  const dim3 grid(static_cast<unsigned>((most + kFewXcd - 1) / kFewXcd * kFewXcd));
  const uint32_t a_bytes = static_cast<uint32_t>(static_cast<int64_t>(p.rows) * p.K * 2);
  const uint32_t w_bytes = static_cast<uint32_t>(static_cast<int64_t>(swiglu ? 2 : 1) * p.N * p.K * 2);
  if (swiglu) {
    hipLaunchKernelGGL((few_rows_kernel<12, true>), grid, dim3(kWave), 0, stream, p, n_tiles, a_bytes, w_bytes);
  } else {
    hipLaunchKernelGGL((few_rows_kernel<16, false>), grid, dim3(kWave), 0, stream, p, n_tiles, a_bytes, w_bytes);
  }
  return launch_status(name);
}

}  // namespace moe
