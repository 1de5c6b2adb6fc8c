// Dense products of the fp32 layers: C[M,N] = A[M,K] . Bt[N,K]^T (+ bias, + tanh GELU), all operands fp32, on the bf16 matrix
// instruction.  An operand is cut, exactly, into three bf16 parts, each rounded to nearest, and the six largest of the nine
// products of parts are added up in fp32; what is left out (second by third part twice, third by third) is at most 2^-24 of a
// product, of either sign.  A 16x16x32 bf16 instruction takes 16 cycles where fp32 instructions take 256 for the same 32
// reduction steps: six of them are 2.7 times as fast.
//
// A workgroup owns 64 x 64 outputs; each of its 4 or 8 waves takes every fourth or eighth run of 32 reduction steps of all of
// them, and the waves' sums meet in LDS at the end.  So a wave needs its operands for itself: loads straight to its own
// 16 KB of LDS (whole 128-byte rows; 16-byte pieces of 64 rows in the instruction's own layout would take four times as
// long), from there to registers, where they are cut; the next run's loads follow at once and have the cutting and the
// products ahead of them.  No barrier in the loop.  Two waves to a SIMD: one cuts (six vector instructions an element,
// 384 a run) while the other multiplies (96 matrix instructions a run).
//
// Bound by what a SIMD issues, the products of parts and the cutting (what-if builds: without two of the six products
// -36 %, without the loads -10 %; counters: 2440-2650 cycles a run, 1536 of them matrix instructions), and, up to 256 tiles, by
// one workgroup's chain.  Measured (us, operands in rotation, hipBLASLt tuned for the shape, the same on a solution picked for
// another row count, as a batch of a new length meets it / this kernel): 1024 x 2304 x 768 33.5, 47.9 / 33.0, 1024 x 3072 x 768 +
// GELU 40.6, 43.4 / 36.0, 1024 x 768 x 3072 39.5, 47.8 / 36.5, 4096 x 3072 x 768 + GELU 142, 158 / 124, 8192 x 2304 x 768 207,
// 215 / 178; relative error against 64 bits 4.0-9.9e-7 / 1.3-4.3e-7 (K = 768 to 3072).  A priority for one of a SIMD's two
// waves: no gain.
//
// Values that bf16 parts cannot hold: a part that overflows or is not finite makes a result that is not finite; a part below
// 2^-126 counts as zero, which moves a result by at most 2^-125 * K * (max |a| + max |b|) (products and sums of parts below it
// count: the instruction keeps those).  A workgroup with results that are not finite, or so small that this could show in their
// last bits, does its tile again on the fp32 instruction and takes those results from there.  Which ones is told by the largest
// magnitudes of a result's own row and column, so its bits depend on no other row or column.  Rows and columns of zeros have
// nothing to lose: 8192 x 2304 x 768 with one in every tile takes 400 us if each makes its tile run again, now 190 (the
// library 207).  A zero that terms cancel to, or that is left where a row and a column have no step in common, does run
// again: the tile takes 2.1 times as long.
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "gemm_mfma.h"
#include "lds_load.h"
#include "rt_launch.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 64, RUN = 32, BLOCKS = 4;                 // outputs of a tile each way, reduction steps of a run, blocks of 16
constexpr int WAVE_BYTES = 2 * TILE * RUN * 4;

struct Params {
  const float *a, *bt, *bias;
  float* c;
  int m, n, k, tiles_m, tiles_n;
};

// A lane's eight consecutive steps of one row.
struct Raw {
  f32x4 lo, hi;
};
struct Parts {
  bf16x8 p0, p1, p2;
};

__device__ inline uint32_t two(float x, float y) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2)); }

// The three parts of a pair; peak collects the largest magnitude.  For a number in [1, 2) the first rest is at most 2^-8, the
// second at most 2^-17 and a multiple of 2^-23, so the third part is exact without a conversion, the upper half of the rest.
// With the second part truncated, its rest is up to 2^-16 and what is left out 2^-23 of a product, always towards zero: a
// single product of 1 + 2^-8 + 2^-7 - d 2^-23 and 1 + 2^-8 - e 2^-23 was up to 1.95 * 2^-23 off, now 1.47 (2^-23 of it the
// instruction's sums, which are cut off), a sum of 768 such terms of either sign 1.6e-7, now 1.4e-7 (on the fp32 instruction
// 5.0e-7).  The conversion takes 1.5 % of a launch.
__device__ inline uint32_t upper(float x, float y) { return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u); }
__device__ inline void cut(float x, float y, uint32_t (&w)[3], float& peak) {
  peak = fmaxf(fmaxf(peak, fabsf(x)), fabsf(y));
  w[0] = two(x, y);
  x -= __uint_as_float(w[0] << 16);
  y -= __uint_as_float(w[0] & 0xffff0000u);
  w[1] = two(x, y);
  x -= __uint_as_float(w[1] << 16);
  y -= __uint_as_float(w[1] & 0xffff0000u);
  w[2] = upper(x, y);
}
__device__ inline Parts cut(const Raw& r, float& peak) {
  uint32_t w[4][3];
  cut(r.lo[0], r.lo[1], w[0], peak);
  cut(r.lo[2], r.lo[3], w[1], peak);
  cut(r.hi[0], r.hi[1], w[2], peak);
  cut(r.hi[2], r.hi[3], w[3], peak);
  return Parts{__builtin_bit_cast(bf16x8, u32x4{w[0][0], w[1][0], w[2][0], w[3][0]}),
               __builtin_bit_cast(bf16x8, u32x4{w[0][1], w[1][1], w[2][1], w[3][1]}),
               __builtin_bit_cast(bf16x8, u32x4{w[0][2], w[1][2], w[2][2], w[3][2]})};
}

template <int NW, bool GELU>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_f32_kernel(Params p) {
  // a run's operands of every wave, 128-byte rows, chunk c of row r at c ^ ((r >> 1) & 7); after the loop four waves' sums,
  // [row block][wave][column block][lane]
  extern __shared__ __align__(16) char smem[];
  f32x4 (*const room)[4][BLOCKS][64] = reinterpret_cast<f32x4 (*)[4][BLOCKS][64]>(smem);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  // XCD x takes the x-th eighth of the tiles, in groups of 8 row panels, the panel fastest
  const int total = p.tiles_m * p.tiles_n, per = gridDim.x >> 3, id = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
  if (id >= total) return;
  constexpr int G = 8;
  const int grp = id / (G * p.tiles_n), in = id - grp * G * p.tiles_n, h = min(G, p.tiles_m - grp * G);
  const int tn = in / h, tm = grp * G + (in - tn * h);

  const i32x4 sa = make_srd(p.a, uint32_t(p.m) * uint32_t(p.k) * 4u), sb = make_srd(p.bt, uint32_t(p.n) * uint32_t(p.k) * 4u);
  const uint32_t own = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)smem)) + w * WAVE_BYTES;
  int va[8], vb[8];                                            // rows past the end repeat the last one: nothing of them is stored
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 8 * i + (lane >> 3), chunk = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    va[i] = min(tm * TILE + r, p.m - 1) * p.k * 4 + chunk;
    vb[i] = min(tn * TILE + r, p.n - 1) * p.k * 4 + chunk;
  }
  const int runs = p.k / RUN;
  auto request = [&](int run) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) load_to_lds(sb, vb[i], run * (RUN * 4), own + 8192 + i * 1024);
#pragma unroll
    for (int i = 0; i < 8; ++i) load_to_lds(sa, va[i], run * (RUN * 4), own + i * 1024);
  };
  // rows 16 * i + l16 of an operand, steps 8 * g4 .. + 8
  const int row_lo = l16 * 128 + (((2 * g4) ^ (l16 >> 1)) << 4), row_hi = l16 * 128 + (((2 * g4 + 1) ^ (l16 >> 1)) << 4);
  auto read = [&](int at, int i) __attribute__((always_inline)) {
    const char* const b = smem + w * WAVE_BYTES + at + i * 2048;
    return Raw{*reinterpret_cast<const f32x4*>(b + row_lo), *reinterpret_cast<const f32x4*>(b + row_hi)};
  };

  f32x4 acc[BLOCKS][BLOCKS];
  // largest magnitudes of the tile's rows and columns (as bits, which order alike), the lane's share of those it reads
  __shared__ __align__(16) uint32_t peaks[2][TILE];
  if (threadIdx.x < 2 * TILE) peaks[0][threadIdx.x] = 0u;
  float peak_a[BLOCKS] = {}, peak_b[BLOCKS] = {};
  // the wave's runs; a run's rows are requested when the last run's have been cut
  auto products = [&](auto plain) __attribute__((always_inline)) {
    constexpr bool PLAIN = decltype(plain)::value;
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int j = 0; j < BLOCKS; ++j) acc[i][j] = f32x4(0.f);
    if (w >= runs) return;
    request(w);
#pragma clang loop unroll(disable)
    for (int r = w; r < runs; r += NW) {
      Raw ra[BLOCKS], rb[BLOCKS];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < BLOCKS; ++j) rb[j] = read(8192, j);
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i) ra[i] = read(0, i);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (r + NW < runs) request(r + NW);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (PLAIN) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
            for (int j = 0; j < BLOCKS; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(e < 4 ? rb[j].lo[e & 3] : rb[j].hi[e & 3],
                                                               e < 4 ? ra[i].lo[e & 3] : ra[i].hi[e & 3], acc[i][j], 0, 0, 0);
      } else {
        Parts b[BLOCKS], a[BLOCKS];
#pragma unroll
        for (int j = 0; j < BLOCKS; ++j) b[j] = cut(rb[j], peak_b[j]);
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) a[i] = cut(ra[i], peak_a[i]);
        auto row = [&](int i, bf16x8 Parts::*pb, bf16x8 Parts::*pa) __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < BLOCKS; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j].*pb, a[i].*pa, acc[i][j], 0, 0, 0);
        };
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) {
          row(i, &Parts::p0, &Parts::p2);                      // the smallest first
          row(i, &Parts::p2, &Parts::p0);
          row(i, &Parts::p1, &Parts::p1);
          row(i, &Parts::p0, &Parts::p1);
          row(i, &Parts::p1, &Parts::p0);
          row(i, &Parts::p0, &Parts::p0);
        }
      }
    }
  };
  // waves 0-3: all waves' sums of row block w
  f32x4 sum[BLOCKS];
  auto meet = [&]() __attribute__((always_inline)) {
    __syncthreads();                                           // the operands of all waves are read
    if (NW == 8) {                                             // a wave and its partner four further on first
      if (w >= 4) {
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
          for (int j = 0; j < BLOCKS; ++j) room[i][w - 4][j][lane] = acc[i][j];
      }
      __syncthreads();
      if (w < 4) {
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
          for (int j = 0; j < BLOCKS; ++j) acc[i][j] += room[i][w][j][lane];
      }
      __syncthreads();
    }
    if (w < 4) {
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
        for (int j = 0; j < BLOCKS; ++j) room[i][w][j][lane] = acc[i][j];
    }
    __syncthreads();
    if (w < 4) {
#pragma unroll
      for (int j = 0; j < BLOCKS; ++j) sum[j] = (room[w][0][j][lane] + room[w][1][j][lane]) + (room[w][2][j][lane] + room[w][3][j][lane]);
    }
  };
  products(std::false_type());
  meet();
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i) {
#pragma unroll
    for (int d = 16; d <= 32; d *= 2) {
      peak_a[i] = fmaxf(peak_a[i], __shfl_xor(peak_a[i], d));
      peak_b[i] = fmaxf(peak_b[i], __shfl_xor(peak_b[i], d));
    }
    if (g4 == 0) {
      atomicMax(&peaks[0][16 * i + l16], __float_as_uint(peak_a[i]));
      atomicMax(&peaks[1][16 * i + l16], __float_as_uint(peak_b[i]));
    }
  }
  __syncthreads();
  uint32_t bad = 0;                                            // a bit per result of the lane
  if (w < 4) {
    const float big_a = __uint_as_float(peaks[0][16 * w + l16]);
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      const f32x4 big_b = *reinterpret_cast<const f32x4*>(&peaks[1][16 * j + 4 * g4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // 2^-125 * K * (..) is less than a 2^-24th of what is at least `least`; products of zeros are zero either way
        const float least = big_a == 0.f || big_b[e] == 0.f ? 0.f : 0x1p-100f * float(p.k) * (big_a + big_b[e]);
        const float size = fabsf(sum[j][e]);
        if (!(size >= least && size < __builtin_inff())) bad |= 1u << (4 * j + e);
      }
    }
  }
  if (__syncthreads_or(bad)) {                                 // also: the sums are read
    f32x4 keep[BLOCKS];
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) keep[j] = sum[j];
    products(std::true_type());
    meet();
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[j][e] = bad >> (4 * j + e) & 1u ? sum[j][e] : keep[j][e];
  }

  if (w >= 4) return;
  const int row = tm * TILE + 16 * w + l16;
  const __amdgpu_buffer_rsrc_t sc = __builtin_amdgcn_make_buffer_rsrc(p.c, 0, uint32_t(p.m) * uint32_t(p.n) * 4u, 0x00020000);
#pragma unroll
  for (int j = 0; j < BLOCKS; ++j) {
    const int col = tn * TILE + 16 * j + 4 * g4;
    f32x4 v = sum[j];
    if (p.bias) v += *reinterpret_cast<const f32x4*>(p.bias + min(col, p.n - 4));
    if (GELU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
    }
    const uint32_t voff = col < p.n && row < p.m ? (uint32_t(row) * uint32_t(p.n) + uint32_t(col)) * 4u : 0xfffffff0u;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), sc, int(voff), 0, 0);
  }
}

}  // namespace

namespace rt {

bool gemm_f32_takes(const void* a, const void* bt, const void* bias, const void* c, int64_t m, int64_t n, int64_t k) {
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return k % RUN == 0 && n % 4 == 0 && m * k < (int64_t(1) << 29) && n * k < (int64_t(1) << 29) && m * n < (int64_t(1) << 29) &&
         aligned(a) && aligned(bt) && aligned(bias) && aligned(c);
}

// Where this kernel is faster than the library on a solution that was tuned for the very shape (the first M of a context), or at
// most 7 % slower: on one picked for another M, or where the library's timing errs, the library takes 1.2 to 2 times as long.
// The library: 5.35 us and 137 TFLOP/s, which it meets or stays behind.  This kernel: a workgroup's chain on eight waves (up to
// 256 tiles), slower when nearly every CU has one, or rounds of two workgroups of four waves per CU, a round that leaves half of
// them out at 0.55.  Fitted to 372 products (hidden 512, 768 and 1024, 31 row counts from 64 to 8192).  Both sides (us, library
// tuned for the shape, on a solution for another M / own): here 1024 x 2304 x 768 33.0, 48.4 / 34.2, 2048 x 768 x 768 22.2, 22-28 /
// 24.1, 704 x 2304 x 768 25.8, 26-48 / 23.5, 1024 x 768 x 3072 39.5, 47.8 / 36.5; there 512 x 2304 x 768 19.6, 25.9 / 23.6,
// 1024 x 768 x 768 13.6, 18.7 / 16.8, 640 x 768 x 3072 31.0, 47.5 / 37.2, 2048 x 2304 x 256 25.3, 32-37 / 26.9, 2113 x 3076 x 96
// 22.8 / 28.1.
bool gemm_f32_pays(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((m + TILE - 1) / TILE) * ((n + TILE - 1) / TILE), full = tiles / 512, rest = tiles % 512;
  const float steps = float(k), round = 2.9f + 0.0211f * steps;
  const float own = tiles <= 256 ? 8.5f + steps * (0.0088f + 0.0019f * float(tiles > 192 ? tiles - 192 : 0) / 64.f)
                                 : 4.4f + round * (float(full) + (rest == 0 ? 0.f : rest <= 256 ? 0.55f : 1.f));
  return own < 1.07f * (5.35f + 2e-6f / 136.8f * float(m) * float(n) * steps);
}

int gemm_f32_bt(const void* a, const void* bt, const void* bias, void* c, int64_t m, int64_t n, int64_t k, bool gelu, void* stream) {
  Params p{static_cast<const float*>(a), static_cast<const float*>(bt), static_cast<const float*>(bias), static_cast<float*>(c),
           int(m), int(n), int(k), int((m + TILE - 1) / TILE), int((n + TILE - 1) / TILE)};
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t tiles = int64_t(p.tiles_m) * p.tiles_n;
  const dim3 grid(unsigned((tiles + 7) / 8 * 8));
  auto go = [&](auto waves, auto act) {
    constexpr int NW = decltype(waves)::value, LDS = NW * WAVE_BYTES;
    constexpr bool GELU = decltype(act)::value;
    static std::atomic<uint64_t> done{0};
    if (int rc = allow_lds(reinterpret_cast<const void*>(&gemm_f32_kernel<NW, GELU>), LDS, done)) return rc;
    RT_LAUNCH((gemm_f32_kernel<NW, GELU>), grid, dim3(64 * NW), LDS, st, p);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? int(RT_OK) : rt::fail(RT_EIO, "fp32 gemm launch failed: %s", hipGetErrorString(e));
  };
  const std::integral_constant<int, 4> four;
  const std::integral_constant<int, 8> eight;
  if (tiles <= 256) return gelu ? go(eight, std::true_type()) : go(eight, std::false_type());
  return gelu ? go(four, std::true_type()) : go(four, std::false_type());
}

}  // namespace rt
