// The fp32 expert path.
//
// The reference's grouped experts run in the modules' dtype, fp32 included
// (TF/integrations/moe.py:377-478: F.grouped_mm over the permuted rows,
// act_fn(gate) * up, the weighted sum over the k routes).  These kernels run
// that path on gfx950 with fp32 operands and fp32 arithmetic throughout:
//   - one grouped GEMM, C(i, j) (+)= sum_r A(i, r) B(r, j) with arbitrary
//     strides, on v_mfma_f32_32x32x2_f32 over LDS tiles,
//     grouped over the output rows (the projections and their input
//     gradients: rows of group g use weight g) or over the reduction rows
//     (the weight gradients: group g's rows give weight g's gradient);
//   - one wave per row for SwiGLU, its backward, the weighted combine, its
//     backward and the permute backward.
// It serves fp32 modules (the C1 configuration); the bf16 path is the tuned
// one.  The row permutation itself is moe_permute_fwd over the rows' bytes.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace moe {
namespace {

constexpr int kNumXcd = 8;

struct F32Gemm {
  const float* A;
  const float* B;
  float* C;
  const int32_t* offs;
  int G, mode, M, N, K;  // mode 0: groups over i (M rows in all), 1: groups over r (K rows in all)
  int64_t sAi, sAr, sBr, sBj, sCi, sCj, sBg, sCg;
  int accumulate;
};

// Group g's rows [lo, hi) from the inclusive offsets, clamped to [0, n).
__device__ __forceinline__ void f32_group_rows(const int32_t* offs, int g, int n, int& lo, int& hi) {
  lo = g ? min(max(offs[g - 1], 0), n) : 0;
  hi = min(max(offs[g], lo), n);
}

// How an operand reaches LDS: 16-byte loads along the reduction (its rows are
// contiguous in r), 16-byte loads along the output dimension, or 4-byte loads
// with any strides.
enum F32Load { kAlongR = 0, kAlongOut = 1, kScalar = 2 };

// Tile of C.  KSPLIT 1: WM x WN waves of SM x SN MFMA tiles of 32x32 each;
// KSPLIT 4: one 32x32 tile whose four waves take a quarter of each k-tile and
// are added at the end.  KW: k's per wave and k-tile.
template <int SM_, int SN_, int WM_, int WN_, int KSPLIT_, int KW_>
struct F32Tile {
  static constexpr int SM = SM_, SN = SN_, WM = WM_, WN = WN_, KSPLIT = KSPLIT_, KW = KW_;
  static constexpr int kThreads = kWave * WM * WN * KSPLIT;
  static constexpr int BM = 32 * SM * WM, BN = 32 * SN * WN, BK = KW * KSPLIT;
  // LDS rows (one k each) of 4 mod 16 floats: the lanes of a wave that write
  // pieces of 4 k's, and the two half-waves that read k and k + 1, mostly fall
  // on different banks.
  static constexpr int LDA = BM + 36, LDB = BN + 36;
};

// One C tile per block.  The MFMA is v_mfma_f32_32x32x2_f32 (64 cycles), so a
// 16-deep k-tile of a 64x64 block is 512 matrix cycles on every SIMD against
// 8 KiB of operands: the matrix pipe is the bound as long as the operands
// arrive, which they do from a double-buffered LDS tile filled through
// registers, the next k-tile's loads in flight during the current one's
// products and six blocks resident per CU (88 TFLOP/s on 8192 x 1024 x 1024
// over 32 experts, padding of the experts' rows left out; the same products
// loaded straight from memory into the MFMA operands, 4 strided bytes per
// lane, ran at 17).  Each output's products are added in increasing r
// (KSPLIT 4: in four interleaved quarters).  Lane l of an MFMA supplies
// A(l % 32, r + l / 32) and B(r + l / 32, l % 32), and holds D rows
// 8 (q / 4) + 4 (l / 32) + q % 4 (q = 0..15) of column l % 32.
template <int LA, int LB, class T>
__global__ __launch_bounds__(T::kThreads) void f32_grouped_gemm_kernel(const F32Gemm p, int tiles_j, int part) {
  constexpr int BM = T::BM, BN = T::BN, BK = T::BK, SM = T::SM, SN = T::SN;
  constexpr int NVA = BM * BK / 4 / T::kThreads, NVB = BN * BK / 4 / T::kThreads;
  static_assert(NVA >= 1 && NVB >= 1 && NVA * T::kThreads * 4 == BM * BK && NVB * T::kThreads * 4 == BN * BK,
                "every thread stages whole 16-byte pieces of both operands");
  constexpr int A_FLOATS = BK * T::LDA, STAGE = A_FLOATS + BK * T::LDB;
  static_assert(T::KSPLIT == 1 || 4 * 32 * 32 <= 2 * STAGE, "the wave partials fit in the ring");
  __shared__ __attribute__((aligned(16))) float lds[2 * STAGE];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;

  // The tile: block b is the (b / 8)-th of XCD b % 8's contiguous share of
  // the real tiles (group-major, then m-tile, then n-tile), or with `part` of
  // part tiles of every group.
  const int xcd = blockIdx.x % kNumXcd;
  const int64_t idx = blockIdx.x / kNumXcd;
  int mtiles = 0;  // m-tiles over all groups
  if (p.mode == 0) {
    for (int c0 = 0; c0 < p.G; c0 += kWave) {
      int lo = 0, hi = 0;
      if (c0 + lane < p.G) f32_group_rows(p.offs, c0 + lane, p.M, lo, hi);
      mtiles += __builtin_amdgcn_readlane(wave_inclusive_scan((hi - lo + BM - 1) / BM), kWave - 1);
    }
  } else {
    mtiles = p.G * ((p.M + BM - 1) / BM);
  }
  const int64_t real = static_cast<int64_t>(mtiles) * tiles_j, share = (real + kNumXcd - 1) / kNumXcd;
  int64_t tile = xcd * share + idx;
  if (part > 0) {
    const int per_group = static_cast<int>(real / p.G), gi = static_cast<int>(idx) / part;
    const int local = xcd * part + static_cast<int>(idx) - gi * part;
    if (gi >= p.G || local >= per_group) return;
    tile = static_cast<int64_t>(gi) * per_group + local;
  } else if (idx >= share || tile >= real) {
    return;
  }
  const int tj = static_cast<int>(tile % tiles_j);
  const int mt = static_cast<int>(tile / tiles_j);
  int g = 0, i0 = 0, i_end = p.M, r_begin = 0, r_end = p.K;
  if (p.mode == 0) {
    int base = 0;
    for (int c0 = 0; c0 < p.G; c0 += kWave) {
      int lo = 0, hi = 0;
      if (c0 + lane < p.G) f32_group_rows(p.offs, c0 + lane, p.M, lo, hi);
      const int nt = (hi - lo + BM - 1) / BM;
      const int incl = wave_inclusive_scan(nt);
      const int tot = __builtin_amdgcn_readlane(incl, kWave - 1);
      if (mt < base + tot) {
        const int q = __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(base + incl > mt)));
        const int local = mt - base - __builtin_amdgcn_readlane(incl - nt, q);
        const int n = __builtin_amdgcn_readlane(nt, q);
        const int rows_lo = __builtin_amdgcn_readlane(lo, q), rows_hi = __builtin_amdgcn_readlane(hi, q);
        // the group's rows split evenly over its m-tiles, in whole 32-row MFMA tiles
        const int rpt = min(BM, ((rows_hi - rows_lo + n - 1) / n + 31) & ~31);
        g = c0 + q;
        i0 = rows_lo + local * rpt;
        i_end = min(i0 + rpt, rows_hi);
        break;
      }
      base += tot;
    }
  } else {
    const int tiles_i = (p.M + BM - 1) / BM;
    g = mt / tiles_i;
    i0 = BM * (mt - g * tiles_i);
    i_end = min(i0 + BM, p.M);
    if (p.K > 0) f32_group_rows(p.offs, g, p.K, r_begin, r_end);  // no reduction rows: every group is empty
  }
  const int j0 = BN * tj;
  const float* B = p.B + (p.mode == 0 ? static_cast<int64_t>(g) * p.sBg : 0);
  float* C = p.C + (p.mode == 1 ? static_cast<int64_t>(g) * p.sCg : 0);

  // 16-byte piece v of this thread: its k and output index within the tile.
  // Along r: BK / 4 lanes take one row; along the output: whole k-rows.
  auto piece = [&](int v, int layout, int extent, int& k, int& o) __attribute__((always_inline)) {
    const int id = v * T::kThreads + tid;
    if (layout == kAlongR) {
      k = (id % (BK / 4)) * 4;
      o = id / (BK / 4);
    } else {
      k = id / (extent / 4);
      o = (id % (extent / 4)) * 4;
    }
  };
  // One piece from memory: elements (o + e, r) or (o, r + e), zeros outside
  // [0, o_end) and past r_end.
  auto fetch = [&](const float* P, int layout, int64_t so, int64_t sr, int o, int o_end, int r)
                   __attribute__((always_inline)) {
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (layout == kScalar) {
      if (r < r_end) {
        const float* q = P + static_cast<int64_t>(r) * sr + static_cast<int64_t>(o) * so;
        if (o < o_end) v.x = q[0];
        if (o + 1 < o_end) v.y = q[so];
        if (o + 2 < o_end) v.z = q[2 * so];
        if (o + 3 < o_end) v.w = q[3 * so];
      }
    } else if (o < o_end && r < r_end) {  // (sizes are multiples of 4 along the piece: all in or all out)
      v = *reinterpret_cast<const float4*>(P + (layout == kAlongR ? static_cast<int64_t>(o) * so + r
                                                                  : static_cast<int64_t>(r) * sr + o));
    }
    return v;
  };
  float4 ra[NVA], rb[NVB];
  auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < NVA; ++v) {
      int k, o;
      piece(v, LA, BM, k, o);
      ra[v] = fetch(p.A, LA, p.sAi, p.sAr, i0 + o, i_end, r_begin + t * BK + k);
    }
#pragma unroll
    for (int v = 0; v < NVB; ++v) {
      int k, o;
      piece(v, LB, BN, k, o);
      rb[v] = fetch(B, LB, p.sBj, p.sBr, j0 + o, p.N, r_begin + t * BK + k);
    }
  };
  auto put = [&](float* s, int layout, int ld, int k, int o, const float4& v) __attribute__((always_inline)) {
    if (layout == kAlongR) {
      s[k * ld + o] = v.x;
      s[(k + 1) * ld + o] = v.y;
      s[(k + 2) * ld + o] = v.z;
      s[(k + 3) * ld + o] = v.w;
    } else {
      *reinterpret_cast<float4*>(s + k * ld + o) = v;
    }
  };
  auto stage = [&](int t) __attribute__((always_inline)) {
    float* s = lds + (t & 1) * STAGE;
#pragma unroll
    for (int v = 0; v < NVA; ++v) {
      int k, o;
      piece(v, LA, BM, k, o);
      put(s, LA, T::LDA, k, o, ra[v]);
    }
#pragma unroll
    for (int v = 0; v < NVB; ++v) {
      int k, o;
      piece(v, LB, BN, k, o);
      put(s + A_FLOATS, LB, T::LDB, k, o, rb[v]);
    }
  };

  // A wave's 32-row tiles are interleaved with the other wave row's, so that
  // the rows of a partly filled tile spread over the waves; tiles without
  // rows skip their products.
  const int wm = T::KSPLIT == 1 ? wave / T::WN : 0, wn = T::KSPLIT == 1 ? wave % T::WN : 0;
  const int kw = T::KSPLIT == 1 ? 0 : wave * T::KW;  // this wave's k's within a k-tile
  const int subs = (i_end - i0 + 31) / 32;
  const int na = __builtin_amdgcn_readfirstlane(subs > wm ? (subs - wm + T::WM - 1) / T::WM : 0);
  f32x16_t acc[SM][SN];
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;
  static_assert(SM <= 2, "a wave has all its row tiles live, one or none");
  const int nk = (r_end - r_begin + BK - 1) / BK;  // 0: an empty group's zeros
  if (nk > 0) {
    load(0);
    stage(0);
    __syncthreads();
  }
  // One copy of the loop per count of live 32-row tiles: guards inside the
  // unrolled products made the compiler move the accumulators around and kept
  // it from spreading the LDS reads.
  auto loop = [&](auto live) __attribute__((always_inline)) {
    constexpr int NA = decltype(live)::value;
    for (int t = 0; t < nk; ++t) {
      if (t + 1 < nk) load(t + 1);
      const float* sa = lds + (t & 1) * STAGE + kw * T::LDA + wm * 32 + l32;
      const float* sb = lds + (t & 1) * STAGE + A_FLOATS + kw * T::LDB + wn * 32 * SN + l32;
#pragma unroll
      for (int u = 0; u < T::KW / 2; ++u) {
        float a[SM], b[SN];
#pragma unroll
        for (int i = 0; i < NA; ++i) a[i] = sa[(2 * u + half) * T::LDA + i * T::WM * 32];
#pragma unroll
        for (int j = 0; j < (NA ? SN : 0); ++j) b[j] = sb[(2 * u + half) * T::LDB + j * 32];
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int j = 0; j < SN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      // The other buffer was last read in step t - 1, before that step's barrier.
      if (t + 1 < nk) stage(t + 1);
      __syncthreads();
    }
  };
  if (na == SM) {
    loop(std::integral_constant<int, SM>{});
  } else if (na > 0) {
    loop(std::integral_constant<int, 1>{});
  } else {
    loop(std::integral_constant<int, 0>{});
  }
  if constexpr (T::KSPLIT > 1) {
    float* part = lds;  // [4][32][32], after the loop's last barrier
#pragma unroll
    for (int q = 0; q < 16; ++q) part[(wave * 32 + 8 * (q / 4) + 4 * half + (q % 4)) * 32 + l32] = acc[0][0][q];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 32 * 32 / T::kThreads; ++e) {
      const int id = e * T::kThreads + tid, row = id / 32, col = id % 32;
      const int i = i0 + row, j = j0 + col;
      if (i < i_end && j < p.N) {
        const float v = ((part[id] + part[1024 + id]) + part[2048 + id]) + part[3072 + id];
        float* c = C + static_cast<int64_t>(i) * p.sCi + static_cast<int64_t>(j) * p.sCj;
        *c = p.accumulate ? *c + v : v;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SN; ++j) {
        const int jc = j0 + (wn * SN + j) * 32 + l32;
        if (jc >= p.N) continue;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int ir = i0 + (wm + T::WM * i) * 32 + 8 * (q / 4) + 4 * half + (q % 4);
          if (ir < i_end) {
            float* c = C + static_cast<int64_t>(ir) * p.sCi + static_cast<int64_t>(jc) * p.sCj;
            *c = p.accumulate ? *c + acc[i][j][q] : acc[i][j][q];
          }
        }
      }
  }
}

template <int LA, int LB, class T>
int f32_launch_tile(const F32Gemm& p, hipStream_t stream) {
  const int tiles_j = (p.N + T::BN - 1) / T::BN;
  // mode 0: every group's rows in BM-row tiles, at most M / BM + G of them
  const int64_t tiles_i = p.mode == 0 ? (p.M + T::BM - 1) / T::BM + p.G
                                      : static_cast<int64_t>(p.G) * ((p.M + T::BM - 1) / T::BM);
  // A weight gradient's tile costs its group's rows.  Where the tiles take
  // several rounds, every XCD takes an eighth of each group's, so that skewed
  // rows load all of them alike; in one round contiguous shares, which read a
  // group's operands into one L2.  us, contiguous -> eighths, up / down
  // projection: H 1536, I 640, 64 experts, 4096 rows, Zipf(1) 352/209 -> 231/139,
  // uniform 210/102 -> 206/106; H 2048, I 768, 128 experts, 8192 rows, Zipf(1)
  // 982/513 -> 670/362, uniform 641/334 -> 639/327; H 1024, I 512, 32 experts,
  // 2048 rows, two experts with all of them 221/93 -> 152/85, Zipf(1) 99/56 ->
  // 94/66.  H 256, I 128, 8 experts, 512 rows (one round) stays: 7.0/6.9, 7.6/7.8
  // in eighths.
  const int64_t per_group = static_cast<int64_t>((p.M + T::BM - 1) / T::BM) * tiles_j;
  const int64_t part =
      p.mode == 1 && p.G * per_group > device_cus(current_device()) ? (per_group + kNumXcd - 1) / kNumXcd : 0;
  const int64_t blocks = part ? p.G * part * kNumXcd : (tiles_i * tiles_j + kNumXcd - 1) / kNumXcd * kNumXcd;
  MOE_REQUIRE(blocks < (1ll << 31) && tiles_i < (1ll << 31), MOE_ERR_UNSUPPORTED, "f32 grouped gemm: too many tiles");
  hipLaunchKernelGGL((f32_grouped_gemm_kernel<LA, LB, T>), dim3(static_cast<unsigned>(blocks)), dim3(T::kThreads), 0,
                     stream, p, tiles_j, static_cast<int>(part));
  return launch_status("moe_f32_grouped_gemm");
}

// The tile.  At 8192 rows over 32 experts, H 1024, I 512 (us; the straight
// 32x32-per-wave kernel this replaced in brackets): row-grouped GEMMs on 64x64
// up 193, down 103, their input gradients 108 and 198 (1020, 506, 310, 564);
// on 128x128 with 8 waves 194, 102, 150, 199, and at smaller calls (H 256,
// I 128, 128 rows per expert) 24 against 12: a 64x64 tile everywhere.  Weight
// gradients, whose reduction is an expert's rows: 157 and 83 on 128x128 with 8
// waves against 177 and 93 on 64x64 (290, 149), as long as those tiles fill
// the chip.  A weight gradient of few tiles and a long reduction (a router's:
// 32 x 1024 outputs over 2048 rows) is a serial chain on 16 blocks: 26 with
// its k-tiles split over the waves of 32x32 tiles against 76 (112); the row-
// grouped GEMMs keep one chain per output, whose sums are the router's logits.
template <int LA, int LB>
int f32_launch(const F32Gemm& p, hipStream_t stream) {
  const int cus = device_cus(current_device());
  auto tiles = [&](int bm, int bn) {  // of a weight gradient
    return static_cast<int64_t>(p.G) * ((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
  };
  if (p.mode == 1) {
    if (tiles(128, 128) >= cus) return f32_launch_tile<LA, LB, F32Tile<2, 1, 2, 4, 1, 16>>(p, stream);
    if (tiles(64, 64) < cus / 2 && p.K / p.G >= 512) return f32_launch_tile<LA, LB, F32Tile<1, 1, 1, 1, 4, 16>>(p, stream);
  }
  return f32_launch_tile<LA, LB, F32Tile<1, 1, 2, 2, 1, 16>>(p, stream);
}

// act[r, c] = silu(pre[r, c]) * pre[r, I + c] for the rows below n_valid.
__global__ void f32_swiglu_fwd_kernel(const float* __restrict__ pre, float* __restrict__ act, int S, int I,
                                      const int32_t* __restrict__ n_valid_ptr) {
  const int n_valid = min(*n_valid_ptr, S);
  for (int r = blockIdx.x; r < n_valid; r += gridDim.x) {
    const float* row = pre + static_cast<int64_t>(r) * 2 * I;
    for (int c = threadIdx.x; c < I; c += blockDim.x) {
      const float gt = row[c];
      act[static_cast<int64_t>(r) * I + c] = gt / (1.0f + expf(-gt)) * row[I + c];
    }
  }
}

// d_pre[r] = (d_act * up * silu'(gate), d_act * silu(gate)) for the rows below n_valid.
__global__ void f32_swiglu_bwd_kernel(const float* __restrict__ d_act, const float* __restrict__ pre,
                                      float* __restrict__ d_pre, int S, int I,
                                      const int32_t* __restrict__ n_valid_ptr) {
  const int n_valid = min(*n_valid_ptr, S);
  for (int r = blockIdx.x; r < n_valid; r += gridDim.x) {
    const float* row = pre + static_cast<int64_t>(r) * 2 * I;
    float* drow = d_pre + static_cast<int64_t>(r) * 2 * I;
    for (int c = threadIdx.x; c < I; c += blockDim.x) {
      const float gt = row[c], up = row[I + c], da = d_act[static_cast<int64_t>(r) * I + c];
      const float s = 1.0f / (1.0f + expf(-gt));
      drow[c] = da * up * (s * (1.0f + gt * (1.0f - s)));
      drow[I + c] = da * gt * s;
    }
  }
}

// out[t] = sum_j w[t, j] y[pos(t, j)] over the token's slots below n_valid.
__global__ void f32_combine_fwd_kernel(const float* __restrict__ y, const int32_t* __restrict__ pos_of_slot,
                                       const int32_t* __restrict__ n_valid_ptr, const float* __restrict__ w, int T,
                                       int H, int k, float* __restrict__ out) {
  const int n_valid = *n_valid_ptr;
  for (int t = blockIdx.x; t < T; t += gridDim.x) {
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
      float acc = 0.0f;
      for (int j = 0; j < k; ++j) {
        const int p = pos_of_slot[static_cast<int64_t>(t) * k + j];
        if (p < n_valid) acc += w[static_cast<int64_t>(t) * k + j] * y[static_cast<int64_t>(p) * H + c];
      }
      out[static_cast<int64_t>(t) * H + c] = acc;
    }
  }
}

// d_y[pos(t, j)] = w[t, j] d_out[t] (zeros for sentinel slots); d_w[t, j] =
// <y[pos(t, j)], d_out[t]> (zero for sentinel slots).  One block per token.
__global__ void f32_combine_bwd_kernel(const float* __restrict__ d_out, const float* __restrict__ y,
                                       const int32_t* __restrict__ pos_of_slot,
                                       const int32_t* __restrict__ n_valid_ptr, const float* __restrict__ w, int T,
                                       int H, int k, float* __restrict__ d_y, float* __restrict__ d_w) {
  __shared__ float part[kMaxSlots][4];
  const int n_valid = *n_valid_ptr;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  for (int t = blockIdx.x; t < T; t += gridDim.x) {
    float dot[kMaxSlots];
    for (int j = 0; j < kMaxSlots; ++j) dot[j] = 0.0f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
      const float g = d_out[static_cast<int64_t>(t) * H + c];
      for (int j = 0; j < k; ++j) {
        const int p = pos_of_slot[static_cast<int64_t>(t) * k + j];
        const bool ok = p < n_valid;
        d_y[static_cast<int64_t>(p) * H + c] = ok ? w[static_cast<int64_t>(t) * k + j] * g : 0.0f;
        if (ok) dot[j] += y[static_cast<int64_t>(p) * H + c] * g;
      }
    }
    for (int j = 0; j < k; ++j) {
      const float s = wave_sum(dot[j]);
      if (lane == 0) part[j][wave] = s;
    }
    __syncthreads();
    if (threadIdx.x < k) {
      const int j = threadIdx.x;
      const int p = pos_of_slot[static_cast<int64_t>(t) * k + j];
      d_w[static_cast<int64_t>(t) * k + j] = p < n_valid ? ((part[j][0] + part[j][1]) + part[j][2]) + part[j][3] : 0.0f;
    }
    __syncthreads();
  }
}

// d_x[t] = sum_j d_xp[pos(t, j)] over the token's slots below n_valid, then
// + d_add[t] when given (the router's input gradient, added as autograd
// would add it to the experts' sum).
__global__ void f32_permute_bwd_kernel(const float* __restrict__ d_xp, const int32_t* __restrict__ pos_of_slot,
                                       const int32_t* __restrict__ n_valid_ptr, int T, int H, int k,
                                       const float* __restrict__ d_add, float* __restrict__ d_x) {
  const int n_valid = *n_valid_ptr;
  for (int t = blockIdx.x; t < T; t += gridDim.x) {
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
      float acc = 0.0f;
      for (int j = 0; j < k; ++j) {
        const int p = pos_of_slot[static_cast<int64_t>(t) * k + j];
        if (p < n_valid) acc += d_xp[static_cast<int64_t>(p) * H + c];
      }
      if (d_add) acc += d_add[static_cast<int64_t>(t) * H + c];
      d_x[static_cast<int64_t>(t) * H + c] = acc;
    }
  }
}

int rows_grid(int64_t rows) { return static_cast<int>(std::min<int64_t>(std::max<int64_t>(rows, 1), 65535)); }

}  // namespace
}  // namespace moe

using namespace moe;

extern "C" int moe_f32_grouped_gemm(const float* A, const float* B, const int32_t* offs, int64_t G, int mode,
                                    int64_t M, int64_t N, int64_t K, int64_t sAi, int64_t sAr, int64_t sBr,
                                    int64_t sBj, int64_t sBg, float* C, int64_t sCi, int64_t sCj, int64_t sCg,
                                    int accumulate, void* stream) {
  MOE_REQUIRE(mode == 0 || mode == 1, MOE_ERR_INVALID, "f32 grouped gemm: mode must be 0 or 1");
  MOE_REQUIRE(G >= 1 && G <= 4096 && M >= 0 && N >= 0 && K >= 0 && M < (1ll << 31) && N < (1ll << 31) &&
                  K < (1ll << 31),
              MOE_ERR_INVALID, "f32 grouped gemm: bad sizes G=%lld M=%lld N=%lld K=%lld", (long long)G,
              (long long)M, (long long)N, (long long)K);
  if (N == 0 || M == 0) return MOE_OK;  // nothing to write: empty buffers may be NULL
  // A and B are read only when K > 0, offs always in mode 0 and only when K > 0 in mode 1
  MOE_REQUIRE(C && (K == 0 || (A && B)) && (offs || (mode == 1 && K == 0)), MOE_ERR_INVALID,
              "f32 grouped gemm: null pointer");
  F32Gemm p{A, B, C, offs, static_cast<int>(G), mode, static_cast<int>(M), static_cast<int>(N), static_cast<int>(K),
            sAi, sAr, sBr, sBj, sCi, sCj, sBg, sCg, accumulate ? 1 : 0};
  const bool a16 = aligned16(A), b16 = aligned16(B);
  const bool b_out = b16 && sBj == 1 && sBr % 4 == 0 && N % 4 == 0 && (mode == 1 || sBg % 4 == 0);
  hipStream_t st = as_stream(stream);
  if (mode == 0) {
    const bool a_r = a16 && sAr == 1 && sAi % 4 == 0 && K % 4 == 0;
    if (a_r && b16 && sBr == 1 && sBj % 4 == 0 && sBg % 4 == 0) return f32_launch<kAlongR, kAlongR>(p, st);
    if (a_r && b_out) return f32_launch<kAlongR, kAlongOut>(p, st);
  } else if (a16 && sAi == 1 && sAr % 4 == 0 && M % 4 == 0 && b_out) {
    return f32_launch<kAlongOut, kAlongOut>(p, st);
  }
  return f32_launch<kScalar, kScalar>(p, st);
}

extern "C" int moe_f32_swiglu_fwd(const float* pre, float* act, const int32_t* offsets, int64_t num_buckets,
                                  int64_t S, int64_t I, void* stream) {
  MOE_REQUIRE(S >= 0 && S < (1ll << 31) && I > 0 && num_buckets >= 1, MOE_ERR_INVALID, "f32 swiglu: bad sizes");
  if (S == 0) return MOE_OK;
  MOE_REQUIRE(pre && act && offsets, MOE_ERR_INVALID, "f32 swiglu: null pointer");
  hipLaunchKernelGGL(f32_swiglu_fwd_kernel, dim3(rows_grid(S)), dim3(256), 0, as_stream(stream), pre, act,
                     static_cast<int>(S), static_cast<int>(I), offsets + (num_buckets - 1));
  return launch_status("moe_f32_swiglu_fwd");
}

extern "C" int moe_f32_swiglu_bwd(const float* d_act, const float* pre, float* d_pre, const int32_t* offsets,
                                  int64_t num_buckets, int64_t S, int64_t I, void* stream) {
  MOE_REQUIRE(S >= 0 && S < (1ll << 31) && I > 0 && num_buckets >= 1, MOE_ERR_INVALID,
              "f32 swiglu bwd: bad sizes");
  if (S == 0) return MOE_OK;
  MOE_REQUIRE(d_act && pre && d_pre && offsets, MOE_ERR_INVALID, "f32 swiglu bwd: null pointer");
  hipLaunchKernelGGL(f32_swiglu_bwd_kernel, dim3(rows_grid(S)), dim3(256), 0, as_stream(stream), d_act, pre, d_pre,
                     static_cast<int>(S), static_cast<int>(I), offsets + (num_buckets - 1));
  return launch_status("moe_f32_swiglu_bwd");
}

extern "C" int moe_f32_combine_fwd(const float* y, const int32_t* pos_of_slot, const int32_t* offsets,
                                   int64_t num_buckets, const float* scores, int64_t T, int64_t H, int64_t k,
                                   float* out, void* stream) {
  MOE_REQUIRE(T >= 0 && H > 0 && k >= 1 && k <= kMaxSlots && num_buckets >= 1, MOE_ERR_INVALID,
              "f32 combine: bad sizes");
  if (T == 0) return MOE_OK;
  MOE_REQUIRE(y && pos_of_slot && offsets && scores && out, MOE_ERR_INVALID, "f32 combine: null pointer");
  hipLaunchKernelGGL(f32_combine_fwd_kernel, dim3(rows_grid(T)), dim3(256), 0, as_stream(stream), y, pos_of_slot,
                     offsets + (num_buckets - 1), scores, static_cast<int>(T), static_cast<int>(H),
                     static_cast<int>(k), out);
  return launch_status("moe_f32_combine_fwd");
}

extern "C" int moe_f32_combine_bwd(const float* d_out, const float* y, const int32_t* pos_of_slot,
                                   const int32_t* offsets, int64_t num_buckets, const float* scores, int64_t T,
                                   int64_t H, int64_t k, float* d_y, float* d_scores, void* stream) {
  MOE_REQUIRE(T >= 0 && H > 0 && k >= 1 && k <= kMaxSlots && num_buckets >= 1, MOE_ERR_INVALID,
              "f32 combine bwd: bad sizes");
  if (T == 0) return MOE_OK;
  MOE_REQUIRE(d_out && y && pos_of_slot && offsets && scores && d_y && d_scores, MOE_ERR_INVALID,
              "f32 combine bwd: null pointer");
  hipLaunchKernelGGL(f32_combine_bwd_kernel, dim3(rows_grid(T)), dim3(256), 0, as_stream(stream), d_out, y,
                     pos_of_slot, offsets + (num_buckets - 1), scores, static_cast<int>(T), static_cast<int>(H),
                     static_cast<int>(k), d_y, d_scores);
  return launch_status("moe_f32_combine_bwd");
}

extern "C" int moe_f32_permute_bwd(const float* d_xp, const int32_t* pos_of_slot, const int32_t* offsets,
                                   int64_t num_buckets, int64_t T, int64_t H, int64_t k, const float* d_add,
                                   float* d_x, void* stream) {
  MOE_REQUIRE(T >= 0 && H > 0 && k >= 1 && k <= kMaxSlots && num_buckets >= 1, MOE_ERR_INVALID,
              "f32 permute bwd: bad sizes");
  if (T == 0) return MOE_OK;
  MOE_REQUIRE(d_xp && pos_of_slot && offsets && d_x, MOE_ERR_INVALID, "f32 permute bwd: null pointer");
  hipLaunchKernelGGL(f32_permute_bwd_kernel, dim3(rows_grid(T)), dim3(256), 0, as_stream(stream), d_xp, pos_of_slot,
                     offsets + (num_buckets - 1), static_cast<int>(T), static_cast<int>(H), static_cast<int>(k),
                     d_add, d_x);
  return launch_status("moe_f32_permute_bwd");
}
