// What the kernels of the dense products share: loads from memory straight to LDS, leave to use much of it, the GELU.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include "rt_common.h"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// 64 lanes x 16 bytes from srd[voff + soff] to LDS bytes [lds, lds + 1024).  Hidden from the compiler's wait
// counting on purpose (it would wait for every load before any LDS read); the waits stand in the kernels.
__device__ inline void load_to_lds(i32x4 srd, int voff, int soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :: "v"(voff), "s"(srd), "s"(soff), "s"(lds) : "memory");
}

__device__ inline i32x4 make_srd(const void* p, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return i32x4{int(uint32_t(a)), int(uint32_t(a >> 32) & 0xffffu), int(bytes), 0x00020000};
}

__device__ inline float gelu_tanh(float x) {   // x / (1 + 2^(x (k0 + k1 x^2))), as bias_gelu_kernel
  constexpr float K0 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  constexpr float K1 = K0 * 0.044715f;
  const float t = x * fmaf(K1, x * x, K0);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}

// More dynamic LDS than the default has to be asked for once per kernel and device.
inline int allow_lds(const void* kernel, int bytes, std::atomic<uint64_t>& done) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return rt::fail(RT_EIO, "hipGetDevice failed: no usable GPU");
  const uint64_t bit = uint64_t(1) << (dev & 63);
  if (done.load(std::memory_order_relaxed) & bit) return RT_OK;
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return rt::fail(RT_EIO, "gemm: %d bytes of LDS refused: %s", bytes, hipGetErrorString(e));
  done.fetch_or(bit, std::memory_order_relaxed);
  return RT_OK;
}

}  // namespace
