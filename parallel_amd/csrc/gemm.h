// Internal launchers shared between the GEMM and router translation units.
#pragma once

#include "common.h"

namespace moe {

// Raw buffer loads: offsets at or past the resource's byte size read as zero
// in hardware, so out-of-range rows and the K tail need no branches.
constexpr uint32_t kOOB = 0x80000000u;  // >= every resource size (host checks < 2 GiB)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// silu(g) = g * sigmoid(g), with the hardware exp and reciprocal (1 ulp).
__device__ __forceinline__ float sigmoid_f(float g) { return __builtin_amdgcn_rcpf(1.0f + __expf(-g)); }
__device__ __forceinline__ float silu_f(float g) { return g * sigmoid_f(g); }

// Forward expert GEMM for experts of a few rows (few_rows.hip): C[r, n] (bf16)
// = sum_k A[r, k] W[g][n, k] over the rows of every group, or with swiglu
// (W = [gate; up], N act columns) act and, if pre is given, gate | up.
// Operands as checked by the entry points; every byte count below 2 GiB.
struct FewRows {
  const bf16_t* A;     // [rows, K]
  const bf16_t* W;     // [G][N, K], or [G][2 N, K] with swiglu
  bf16_t* C;           // [rows, N]
  bf16_t* pre;         // swiglu: [rows, 2 N] or null
  const int32_t* offs;
  int G, rows, N, K;
};
int few_rows(const FewRows& p, bool swiglu, hipStream_t stream, const char* name);

// partials[s][T][E] (f32) = x[T, s-th K range] . wr[E, s-th K range]^T.
int router_logits_partials(const bf16_t* x, const bf16_t* wr, float* partials, int T, int H, int E, int splits,
                           int k_chunk, hipStream_t stream);

// partials[c][E][H] (f32) = dl[rows of chunk c, E]^T . x[rows of chunk c, H].
int router_wgrad_partials(const bf16_t* dl, const bf16_t* x, float* partials, int T, int H, int E, int chunks,
                          int chunk_rows, hipStream_t stream);

// dx[T,H] (bf16) = dl[T,E] . wr[E,H].
int router_dgrad(const bf16_t* dl, const bf16_t* wr, bf16_t* dx, int T, int H, int E, hipStream_t stream);

}  // namespace moe
