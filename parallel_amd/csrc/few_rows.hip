// The forward expert GEMMs of a decoding batch: experts of a few rows, whose
// weights are streamed from HBM once for almost no arithmetic.
//
// The tiled kernel (grouped_gemm.hip) gives such an expert ceil(N / 256) blocks
// that each walk all of K, so one decoded token keeps 48 of 256 CUs busy, and
// it stages the weights through LDS behind a block barrier per k-tile.  Here a
// block takes 16 or more weight rows of one expert and splits K over its eight
// waves, so that the same token gives 384 blocks; a wave loads its weights
// straight into the MFMA operand registers, up to 16 loads of 1 KiB in flight,
// with the next tile's loads issued as the current tile's operands are used.
// The rows of the expert (16 at a time) stay in registers while the block
// walks its run of tiles.  The waves' partial sums meet in LDS, one barrier
// per tile.  Bound by the weights' bytes from a few tokens on (16 tokens at
// H 2048, I 768, 128 experts, top-8: 5.1 TB/s; the tiled kernel 4.4), by
// latency and the launch for one token.
#include <algorithm>

#include "dma.h"
#include "gemm.h"

namespace moe {
namespace {

constexpr int kFewWaves = 8;
constexpr int kFewXcd = 8;
constexpr int kPartRow = 20;  // floats per row of a 16 x 16 partial: the four row groups of a write hit distinct banks

// KS: 32-deep k-steps per wave; NT: 16-row weight sub-tiles per tile (SWIGLU:
// NT 2, the gate rows and the matching up rows).
template <int KS, int NT, bool SWIGLU>
__global__ __launch_bounds__(kFewWaves * kWave) void few_rows_kernel(const FewRows p, int n_tiles, uint32_t a_bytes,
                                                                     uint32_t w_bytes) {
  constexpr int L = KS * NT;             // loads per tile and wave
  constexpr int R = L <= 16 ? L : 16;    // ... in flight
  static_assert(L % R == 0 && (!SWIGLU || NT == 2), "a load's register is the same in every tile");
  __shared__ float part[2][kFewWaves][NT][16][kPartRow];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, q = lane >> 4;

  // Tiles in group-major order, then 16-row chunk, then weight rows; an XCD's
  // blocks take neighbouring runs.
  auto chunks_of = [&](int g, int& lo) {
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
    const int cnt = chunks_of(c0 + lane, lo);
    chunks += __builtin_amdgcn_readlane(wave_inclusive_scan((cnt + 15) / 16), kWave - 1);
  }
  const int64_t total = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(chunks)) * n_tiles;
  const int nb = gridDim.x, lb = (blockIdx.x % kFewXcd) * (nb / kFewXcd) + blockIdx.x / kFewXcd;
  const int64_t t_begin = total * lb / nb, t_end = total * (lb + 1) / nb;
  if (t_begin >= t_end) return;

  struct Tile {
    int g, r0, rows, nt;  // group, first row, rows (at most 16), weight tile
  };
  auto locate = [&](int64_t t) {
    const int chunk = static_cast<int>(t / n_tiles);
    Tile d{0, 0, 0, static_cast<int>(t - static_cast<int64_t>(chunk) * n_tiles)};
    int base = 0;
    for (int c0 = 0; c0 < p.G; c0 += kWave) {
      int lo;
      const int cnt = chunks_of(c0 + lane, lo);
      const int n = (cnt + 15) / 16;
      const int incl = wave_inclusive_scan(n);
      const int tot = __builtin_amdgcn_readlane(incl, kWave - 1);
      if (chunk < base + tot) {
        const int w = __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(base + incl > chunk)));
        const int local = chunk - base - __builtin_amdgcn_readlane(incl - n, w);
        d.g = c0 + w;
        d.r0 = __builtin_amdgcn_readlane(lo, w) + 16 * local;
        d.rows = min(16, __builtin_amdgcn_readlane(cnt, w) - 16 * local);
        break;
      }
      base += tot;
    }
    return d;
  };

  const int kb = wave * KS * 32 + 8 * q;  // this lane's first k
  const __amdgpu_buffer_rsrc_t rsA = make_rsrc(p.A, a_bytes);
  bf16x8_t xf[KS];
  auto load_x = [&](const Tile& d) __attribute__((always_inline)) {
    const uint32_t off = i16 < d.rows ? (static_cast<uint32_t>(d.r0 + i16) * static_cast<uint32_t>(p.K) +
                                         static_cast<uint32_t>(kb)) * 2u
                                      : kOOB;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      xf[ks] = __builtin_bit_cast(
          bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsA, kb + 32 * ks < p.K ? off + 64u * ks : kOOB, 0, 0));
  };
  // Byte offset of the lane's weight row and first k, per sub-tile.
  auto w_off = [&](const Tile& d, int s) __attribute__((always_inline)) {
    const int n = SWIGLU ? d.nt * 16 + i16 : (d.nt * NT + s) * 16 + i16;
    const int row = SWIGLU ? s * p.N + n : n;
    return n < p.N ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(p.K) + static_cast<uint32_t>(kb)) * 2u : kOOB;
  };
  auto w_rsrc = [&](const Tile& d) __attribute__((always_inline)) {
    return make_rsrc(p.W + static_cast<int64_t>(d.g) * (SWIGLU ? 2 : 1) * p.N * p.K, w_bytes);
  };
  u32x4_t wf[R];
  auto load_w = [&](__amdgpu_buffer_rsrc_t rs, const uint32_t (&off)[NT], int i) __attribute__((always_inline)) {
    const int s = i / KS, ks = i % KS;
    // (Not non-temporal: an operand load takes 64 bytes of each row, and the
    // line has to stay for the next one: up and down projection of 16 tokens
    // 109 + 58 us non-temporal against 105 + 52, H 2048, I 768, 128 experts.)
    wf[i % R] = __builtin_amdgcn_raw_buffer_load_b128(rs, kb + 32 * ks < p.K ? off[s] + 64u * ks : kOOB, 0, 0);
  };

  Tile cur = locate(t_begin);
  __amdgpu_buffer_rsrc_t rs_cur = w_rsrc(cur);
  uint32_t off_cur[NT];
#pragma unroll
  for (int s = 0; s < NT; ++s) off_cur[s] = w_off(cur, s);
  load_x(cur);
#pragma unroll
  for (int i = 0; i < R; ++i) load_w(rs_cur, off_cur, i);
  int buf = 0;
  for (int64_t t = t_begin; t < t_end; ++t) {
    const bool more = t + 1 < t_end;
    Tile nxt = cur;
    ++nxt.nt;
    if (more && nxt.nt == n_tiles) nxt = locate(t + 1);
    const __amdgpu_buffer_rsrc_t rs_nxt = w_rsrc(nxt);
    uint32_t off_nxt[NT];
#pragma unroll
    for (int s = 0; s < NT; ++s) off_nxt[s] = more ? w_off(nxt, s) : kOOB;
    f32x4_t acc[NT];
#pragma unroll
    for (int s = 0; s < NT; ++s) acc[s] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < L; ++i) {
      acc[i / KS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i % KS], __builtin_bit_cast(bf16x8_t, wf[i % R]),
                                                            acc[i / KS], 0, 0, 0);
      if (i + R < L) {
        load_w(rs_cur, off_cur, i + R);
      } else {
        load_w(rs_nxt, off_nxt, i + R - L);
      }
    }
    if (more && (nxt.g != cur.g || nxt.r0 != cur.r0)) load_x(nxt);
    // Lane (i16, q) holds rows 4 q + i, weight row i16 of each sub-tile.
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[buf][wave][s][4 * q + i][i16] = acc[s][i];
    // (The other buffer is read before the next tile's barrier and written after it.)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    auto sum = [&](int s, int m, int n) __attribute__((always_inline)) {
      float v = part[buf][0][s][m][n];
#pragma unroll
      for (int w = 1; w < kFewWaves; ++w) v += part[buf][w][s][m][n];
      return v;
    };
    if constexpr (SWIGLU) {
      const int m = tid >> 4, n = cur.nt * 16 + (tid & 15);
      if (tid < 256 && m < cur.rows && n < p.N) {
        const bf16_t g = f32_to_bf16(sum(0, m, tid & 15)), u = f32_to_bf16(sum(1, m, tid & 15));
        const int64_t r = cur.r0 + m;
        p.C[r * p.N + n] = f32_to_bf16(bf16_to_f32(f32_to_bf16(silu_f(bf16_to_f32(g)))) * bf16_to_f32(u));
        if (p.pre) {
          p.pre[r * 2 * p.N + n] = g;
          p.pre[r * 2 * p.N + p.N + n] = u;
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < (NT + 1) / 2; ++e) {
        const int id = e * kFewWaves * kWave + tid;  // (m, column of the tile)
        const int m = id / (16 * NT), col = id % (16 * NT), n = cur.nt * 16 * NT + col;
        if (m < cur.rows && n < p.N)
          p.C[static_cast<int64_t>(cur.r0 + m) * p.N + n] = f32_to_bf16(sum(col / 16, m, col % 16));
      }
    }
    buf ^= 1;
    cur = nxt;
    rs_cur = rs_nxt;
#pragma unroll
    for (int s = 0; s < NT; ++s) off_cur[s] = off_nxt[s];
  }
}

template <int KS, int NT, bool SWIGLU>
int few_launch(const FewRows& p, hipStream_t stream, const char* name) {
  const int n_tiles = (p.N + (SWIGLU ? 16 : 16 * NT) - 1) / (SWIGLU ? 16 : 16 * NT);
  const int dev = current_device();
  const int occ = cached_blocks_per_cu(dev, reinterpret_cast<const void*>(&few_rows_kernel<KS, NT, SWIGLU>),
                                       kFewWaves * kWave, 0);
  const int64_t most = static_cast<int64_t>((p.rows + 15) / 16 + std::min(p.G, p.rows)) * n_tiles;  // tiles at worst
  const int64_t resident = static_cast<int64_t>(device_cus(dev)) * occ;
  const int grid = static_cast<int>((std::min(most, resident) + kFewXcd - 1) / kFewXcd * kFewXcd);
  hipLaunchKernelGGL((few_rows_kernel<KS, NT, SWIGLU>), dim3(grid), dim3(kFewWaves * kWave), 0, stream, p, n_tiles,
                     static_cast<uint32_t>(static_cast<int64_t>(p.rows) * p.K * 2),
                     static_cast<uint32_t>(static_cast<int64_t>(SWIGLU ? 2 : 1) * p.N * p.K * 2));
  return launch_status(name);
}

}  // namespace

// k-steps per wave of 2, 3, 4, 6, 8 and 16: K up to 4096, within a quarter of
// the split (other reductions keep the tiled kernel).
bool few_rows_takes(int64_t K) { return K > 256 && K <= 4096; }

int few_rows(const FewRows& p, bool swiglu, hipStream_t stream, const char* name) {
  const int ks = (p.K + 255) / 256;
#define FEW(KS_, NT_)                                                   \
  return swiglu ? few_launch<KS_, 2, true>(p, stream, name) : few_launch<KS_, NT_, false>(p, stream, name)
  if (ks <= 2) FEW(2, 4);
  if (ks <= 3) FEW(3, 4);
  if (ks <= 4) FEW(4, 4);
  if (ks <= 6) FEW(6, 2);
  if (ks <= 8) FEW(8, 2);
  FEW(16, 1);
#undef FEW
}

}  // namespace moe
