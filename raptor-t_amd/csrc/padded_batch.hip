// Between a padded batch [sequences, width] and the packed one the encoder takes: token counts from the mask, packed ids,
// and packed rows back to their padded places.  One launch each instead of one per sequence and tensor.
//
// All three are bound by their launch: a batch of 8 x 1700 ids is 0.1 MB, and the rows of one (8 x 1700 x 768 fp16, 41 MB
// moved) take 9 us.  What they replace, the same steps as tensor operators, took 0.48 ms of host time and launches
// around a model call of 1.75 ms (8 sequences of 150-1700 tokens).
#include <hip/hip_runtime.h>

#include <climits>

#include "rt_launch.h"

namespace {

constexpr int PACK_THREADS = 256;

// One workgroup per sequence: its token count, or -1 where the mask is not ones on a prefix of the row and zeros behind it.  A row
// qualifies if no entry is another number and its ones are as many as the place of the last of them.
template <typename T>
__global__ __launch_bounds__(PACK_THREADS) void padded_tokens_kernel(const T* __restrict__ mask, int64_t row_stride, int64_t width,
                                                                    int* __restrict__ tokens) {
  __shared__ int counts[PACK_THREADS / 64], ends[PACK_THREADS / 64];
  const T* const row = mask + blockIdx.x * row_stride;
  int count = 0, end = 0;
  for (int64_t i = threadIdx.x; i < width; i += PACK_THREADS) {
    const T v = row[i];
    if (v == 1) {
      ++count;
      end = max(end, int(i) + 1);
    } else if (v != 0) {
      end = INT_MAX;                                   // no row has as many ones
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    count += __shfl_xor(count, d, 64);
    end = max(end, __shfl_xor(end, d, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    counts[threadIdx.x >> 6] = count;
    ends[threadIdx.x >> 6] = end;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < PACK_THREADS / 64; ++w) {
      count += counts[w];
      end = max(end, ends[w]);
    }
    tokens[blockIdx.x] = end == count ? count : -1;
  }
}

struct PackArgs {
  const void* ids;
  const void* types;              // or NULL: zeros
  int64_t ids_stride, types_stride, width;
  const int* tokens;              // per sequence
  int block, fixed;               // a sequence takes its tokens rounded up to `block`, or `fixed` places where that is not 0
  int64_t total;
  int *out_ids, *out_pos, *out_types;
};

// Workgroup (c, s): places c * 256 .. + 256 of sequence s, whose first place is the sum of the lengths before it.
template <typename I, typename Y>
__global__ __launch_bounds__(PACK_THREADS) void pack_tokens_kernel(PackArgs a) {
  __shared__ long long part[PACK_THREADS / 64];
  const int s = blockIdx.y;
  auto length = [&](int t) { return a.fixed ? int64_t(a.fixed) : (int64_t(a.tokens[t]) + a.block - 1) / a.block * a.block; };
  const int64_t n = length(s), j = int64_t(blockIdx.x) * PACK_THREADS + threadIdx.x;
  if (int64_t(blockIdx.x) * PACK_THREADS >= n) return;
  long long before = 0;
  for (int t = threadIdx.x; t < s; t += PACK_THREADS) before += length(t);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) before += __shfl_xor(before, d, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = before;
  __syncthreads();
  before = 0;
  for (int w = 0; w < PACK_THREADS / 64; ++w) before += part[w];
  const int64_t to = before + j;
  if (j >= n || to >= a.total) return;
  const bool inside = j < a.width;                // past the padded width (a last block that reaches beyond it): zeros
  a.out_ids[to] = inside ? int(static_cast<const I*>(a.ids)[s * a.ids_stride + j]) : 0;
  a.out_pos[to] = int(j);
  a.out_types[to] = inside && a.types ? int(static_cast<const Y*>(a.types)[s * a.types_stride + j]) : 0;
}

// The sequences' places travel as kernel arguments: no copy to the device, nothing whose lifetime outlasts the launch.
constexpr int UNPACK_SEQUENCES = 128;
struct UnpackArgs {
  const uint4* packed;
  uint4* out;
  int64_t width;                  // rows of a padded sequence
  int vectors;                    // 16-byte vectors of a row
  int first;                      // sequence of the first workgroup row
  int64_t start[UNPACK_SEQUENCES];
  int real[UNPACK_SEQUENCES];
};
__global__ __launch_bounds__(PACK_THREADS) void unpack_rows_kernel(UnpackArgs a) {
  const int s = blockIdx.y;
  const int64_t per = a.width * a.vectors, filled = int64_t(a.real[s]) * a.vectors, base = a.start[s] * a.vectors;
  uint4* const out = a.out + (a.first + s) * per;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t i = (int64_t(blockIdx.x) * 4 + k) * PACK_THREADS + threadIdx.x;
    if (i < per) out[i] = i < filled ? a.packed[base + i] : uint4{0, 0, 0, 0};
  }
}

int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? RT_OK : rt::fail(RT_EIO, "%s launch failed: %s", what, hipGetErrorString(e));
}

}  // namespace

extern "C" {

int rt_padded_tokens(const void* mask, int elem_bytes, int64_t row_stride, int batch, int64_t width, int* tokens_dev,
                     void* stream) {
  RT_REQUIRE(mask && tokens_dev, RT_EINVAL, "NULL pointer");
  RT_REQUIRE(batch >= 1 && width >= 1 && width < (int64_t(1) << 31), RT_EINVAL, "bad shape: batch=%d width=%lld", batch, (long long)width);
  RT_REQUIRE(elem_bytes == 1 || elem_bytes == 4 || elem_bytes == 8, RT_EINVAL, "mask entries of %d bytes: must be 1, 4 or 8", elem_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto launch = [&](auto tag) {
    typedef decltype(tag) T;
    RT_LAUNCH(padded_tokens_kernel<T>, dim3(batch), dim3(PACK_THREADS), 0, st, (const T*)mask, row_stride, width, tokens_dev);
  };
  if (elem_bytes == 1) launch(uint8_t());
  else if (elem_bytes == 4) launch(int32_t());
  else launch(int64_t());
  return launched("padded_tokens");
}

int rt_pack_tokens(const void* ids, int ids_bytes, int64_t ids_stride, const void* types, int types_bytes, int64_t types_stride,
                   int batch, int64_t width, const int* tokens_dev, int block, int fixed_length, int64_t longest, int64_t total,
                   int* out_ids, int* out_positions, int* out_types, void* stream) {
  RT_REQUIRE(ids && tokens_dev && out_ids && out_positions && out_types, RT_EINVAL, "NULL pointer");
  RT_REQUIRE(batch >= 1 && batch <= 65535 && width >= 1 && block >= 1 && fixed_length >= 0 && longest >= 1 && total >= 1, RT_EINVAL,
             "bad shape: batch=%d width=%lld block=%d fixed_length=%d longest=%lld total=%lld", batch, (long long)width, block,
             fixed_length, (long long)longest, (long long)total);
  RT_REQUIRE((ids_bytes == 4 || ids_bytes == 8) && (!types || types_bytes == 4 || types_bytes == 8), RT_EINVAL,
             "ids and types must have 4 or 8 bytes");
  PackArgs a{ids, types, ids_stride, types_stride, width, tokens_dev, block, fixed_length, total, out_ids, out_positions, out_types};
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto launch = [&](auto i, auto y) {
    RT_LAUNCH((pack_tokens_kernel<decltype(i), decltype(y)>), dim3(unsigned((longest + PACK_THREADS - 1) / PACK_THREADS), batch),
              dim3(PACK_THREADS), 0, st, a);
  };
  if (ids_bytes == 4 && types_bytes == 8) launch(int32_t(), int64_t());
  else if (ids_bytes == 4) launch(int32_t(), int32_t());
  else if (types_bytes == 8) launch(int64_t(), int64_t());
  else launch(int64_t(), int32_t());
  return launched("pack_tokens");
}

int rt_unpack_rows(const void* packed, int64_t packed_rows, int64_t row_bytes, const int64_t* starts, const int64_t* tokens, int batch,
                   int64_t width, void* out, void* stream) {
  RT_REQUIRE(packed && starts && tokens && out, RT_EINVAL, "NULL pointer");
  RT_REQUIRE(batch >= 1 && width >= 1 && width < (int64_t(1) << 31) && row_bytes >= 16 && row_bytes % 16 == 0 && row_bytes < (1 << 24),
             RT_EINVAL, "bad shape: batch=%d width=%lld row_bytes=%lld", batch, (long long)width, (long long)row_bytes);
  RT_REQUIRE(((reinterpret_cast<uintptr_t>(packed) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0, RT_EINVAL, "rows must be 16-byte aligned");
  for (int s = 0; s < batch; ++s)
    RT_REQUIRE(starts[s] >= 0 && tokens[s] >= 0 && tokens[s] <= width && starts[s] + tokens[s] <= packed_rows, RT_EINVAL,
               "sequence %d: rows %lld .. + %lld outside of %lld packed ones or the width %lld", s, (long long)starts[s],
               (long long)tokens[s], (long long)packed_rows, (long long)width);
  const int64_t per = width * (row_bytes / 16), groups = (per + 4 * PACK_THREADS - 1) / (4 * PACK_THREADS);
  RT_REQUIRE(groups < (int64_t(1) << 24), RT_EINVAL, "a padded sequence of %lld bytes is too large", (long long)(per * 16));
  for (int first = 0; first < batch; first += UNPACK_SEQUENCES) {
    UnpackArgs a;
    a.packed = static_cast<const uint4*>(packed);
    a.out = static_cast<uint4*>(out);
    a.width = width;
    a.vectors = int(row_bytes / 16);
    a.first = first;
    const int n = batch - first < UNPACK_SEQUENCES ? batch - first : UNPACK_SEQUENCES;
    for (int s = 0; s < UNPACK_SEQUENCES; ++s) {
      a.start[s] = s < n ? starts[first + s] : 0;
      a.real[s] = s < n ? int(tokens[first + s]) : 0;
    }
    RT_LAUNCH(unpack_rows_kernel, dim3(unsigned(groups), n), dim3(PACK_THREADS), 0, static_cast<hipStream_t>(stream), a);
    if (int rc = launched("unpack_rows")) return rc;
  }
  return RT_OK;
}

}  // extern "C"
