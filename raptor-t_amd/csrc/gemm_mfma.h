// The library's own dense products (gemm_mfma.hip, gemm_f32.hip), called by the entry points in gemm.cpp.
#pragma once
#include <cstdint>

namespace rt {

// Whether gemm_mfma_bt computes this product: 16-bit types, K a multiple of 64, N a multiple of 8, 16-byte aligned
// operands whose byte offsets fit 31 bits.
bool gemm_mfma_takes(const void* a, const void* bt, const void* bias, const void* c, int64_t m, int64_t n, int64_t k, int dtype);
// Whether it is also the faster way: not for a long reduction with few outputs, which hipBLASLt cuts.
bool gemm_mfma_pays(int64_t m, int64_t n, int64_t k);
// C[M,N] = A[M,K] . Bt[N,K]^T (+ bias, + tanh GELU)
int gemm_mfma_bt(const void* a, const void* bt, const void* bias, void* c, int64_t m, int64_t n, int64_t k, bool gelu, int dtype,
                 void* stream);
// QKV projection with the head split: the Q columns go to rows[M, 3 * heads * 64], K and V to the packed tiles.
int gemm_mfma_qkv(const void* a, const void* bt, const void* bias, void* rows, void* kt, void* vt, const int* seq_blocks_dev,
                  int batch, int64_t m, int heads, int64_t k, int dtype, void* stream);

// Into how many slices of the reduction this product should be cut if the caller can take fp32 slices [slices][M][N] of
// up to max_bytes and add them up itself (1: uncut, but in fp32; 0: uncut and in 16 bits, use gemm_mfma_bt).
int gemm_mfma_slices(int64_t m, int64_t n, int64_t k, int64_t max_bytes);
// The slices; `slices` >= 1 as gemm_mfma_slices gave it.
int gemm_mfma_part(const void* a, const void* bt, float* parts, int64_t m, int64_t n, int64_t k, int slices, int dtype, void* stream);
// The tile [rows, columns, slices] that the three above take; max_slices as gemm_mfma_slices gives it, 0 for the other two.
void gemm_mfma_tile(int64_t m, int64_t n, int64_t k, bool gelu, bool qkv, int max_slices, int* tile);

// gemm_f32.hip: the same product of fp32 operands on bf16 parts; K a multiple of 32, N of 4, 16-byte aligned operands whose
// byte offsets fit 31 bits.
bool gemm_f32_takes(const void* a, const void* bt, const void* bias, const void* c, int64_t m, int64_t n, int64_t k);
// Whether it is also the faster way: not for few outputs, which hipBLASLt cuts.
bool gemm_f32_pays(int64_t m, int64_t n, int64_t k);
int gemm_f32_bt(const void* a, const void* bt, const void* bias, void* c, int64_t m, int64_t n, int64_t k, bool gelu, void* stream);

}  // namespace rt
