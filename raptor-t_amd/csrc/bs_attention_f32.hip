// Block-sparse attention in fp32: the accuracy mode of the layer (the reference dispatches an
// fp32-output kernel when the attention buffer is fp32, layers/multi_headed_attention.cpp:198-199,
// layers/kernels/sparse_attention.cu:785-1120, :1582-1599).  Same inputs, plans and outputs as the
// fp16 / bf16 kernel of bs_attention.hip, with every tensor in fp32.
//
// The products run on the bf16 matrix instructions without losing fp32's digits: an operand is cut, exactly, into
// three bf16 parts (hi + mid + lo), and of the nine products of parts the six largest are added up in fp32.  The parts are
// rounded, not truncated, so what is left out (mid * lo twice, lo * lo) is at most 2^-24 of a product, of either sign: less
// than the roundings of an fp32 sum.  (Truncated parts leave out up to 2^-21, always towards zero: operands whose low bits
// are all ones were then twice as far from 64 bits as on the fp32 instruction, 8.8e-7 against 4.4e-7; now 2.2e-7.)  Six
// products of 16x16x32 take 96 cycles of a SIMD's matrix pipe where v_mfma_f32_16x16x4_f32 takes 256.
//
// One workgroup of eight waves per unit (64 queries of one head against the unit's list of key blocks).  A key
// block's K and V^T tiles are cut once for the whole workgroup, 8 + 8 numbers per thread, on their way into LDS, in
// the matrix instruction's fragment order (every operand read is 1 KiB in a row); two buffers, so the next tile
// is cut while the matrix pipe works on this one and the one after it is on its way from memory; one barrier per
// tile.  Wave w owns queries 16 (w & 3) .. + 16 and of every tile the keys 32 (w >> 2) .. + 32:
//   S^T[key][q] = sum_d K[key][d] Q[q][d]         2 tiles of 16 keys x 2 steps of 32 d x 6
//   online softmax per query (a lane's column), moving maximum, base 2 (the scale log2(e)/sqrt(d)
//   is folded into Q)
//   O^T[d][q] += sum_key V^T[d][key] P^T[key][q]  4 tiles of 16 d x 6
// and the two halves' states merge through LDS at the end.  A lane of an S^T accumulator holds keys
// 16 kt + 4 (lane >> 4) + i of query lane & 15: with a step's 32 keys taken in the order that makes these a lane's 8,
// P never leaves its registers; V^T is laid out in LDS in the same order.
//
// A unit is run again by the plain kernel below on v_mfma_f32_16x16x4_f32, which gives what fp32 arithmetic gives,
//   if its result is not finite: the parts of an infinity are no numbers (inf - inf);
//   if an output is below 2^-100 (values below 2^-109 lose digits: the bf16 instructions take a subnormal part for zero) or
//   a query lies outside 2^-109 .. 2^80, where digits that it or a key loses could reach a score.
// Values and weights below 2^-126 count as zero otherwise (exp2 is the hardware's instruction).
//
// Bound by the matrix pipe at 1 540 cycles per tile and SIMD (with the cutting, 700 vector cycles, beside it) and, with
// few units, by the longest row on one CU.  Measured (us, before: one tile at a time on v_mfma_f32_16x16x4_f32, units in flat
// order): 12 heads x 1024 tokens 82 -> 32, x 4 x 2048 493 -> 136, x 128 + 832 + 1984 178 -> 60 (the rounding of the parts
// is 4 % of it); the error against 64 bits 5.0e-7 -> 3.0e-7 of the result (the longer steps of the matrix instruction add up fewer
// partial sums), 0.4 to 0.65 of the fp32 instruction's over scores of size 0.1 to 10 and the mantissas above.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "rt_launch.h"

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int THREADS = 512;
constexpr int PITCH = 68;            // plain kernel, floats per LDS row: 16-byte aligned rows, rows 4 banks apart
constexpr int PLANE = 8192;          // bytes of one part of a tile
constexpr int BUFFER = 6 * PLANE;    // K and V^T, three parts each

struct ArgsF32 {
  const float* q; const float* k; const float* vt; float* out;
  const int* seq_blocks; int batch; int heads; int nb_total;
  const int* to_idx; const int* to_pos; int plan_heads;
  const int* from_idx; const int* from_pos;
  const int* seq_tokens;
  const float* q_rows; const float* q_bias; float q_scale;
};

// element (row, col) of a 64 x 64 tile in fragment order
__device__ __forceinline__ int frag_index(int row, int col) {
  return ((4 * (row >> 5) + (col >> 4)) * 64 + (row & 31) + 32 * ((col >> 3) & 1)) * 8 + (col & 7);
}

// token whose V column sits in slot p of a V^T tile (tokens 4-7 and 8-11 of every 16 swap places)
__device__ __forceinline__ int slot_token(int p) {
  const int e = p & 15;
  return (p & ~15) | ((e & 3) | ((e & 4) << 1) | ((e & 8) >> 1));
}

// Copies one tile from fragment order into LDS as dst[row][col].  Thread t of 256 takes 16 floats: four
// runs of 4 consecutive columns.  `V`: the tile is V^T[d][slot]; it is stored as dst[d][token].
template <bool V>
__device__ __forceinline__ void stage_tile(const float* __restrict__ src, float (*dst)[PITCH]) {
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int e = (threadIdx.x + it * 256) * 4;       // first element of the run, fragment order
    const f32x4 x = *reinterpret_cast<const f32x4*>(src + e);
    const int frag = e >> 9, lane = (e >> 3) & 63, sub = e & 7;
    const int row = 32 * (frag >> 2) + (lane & 31);
    const int col = 16 * (frag & 3) + 8 * (lane >> 5) + sub;
    if (V) {
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[row][slot_token(col + i)] = x[i];
    } else {
      *reinterpret_cast<f32x4*>(&dst[row][col]) = x;
    }
  }
}

__device__ __forceinline__ float group_max(float v) {     // over the four lanes that share lane & 15
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float group_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// Where a unit stands.
struct Unit {
  int g0, n, nbv, tail, block, h, p0, p1;        // its sequence's first block and blocks; see unit_of; its entries of the index
  int64_t head_base;                             // its head's tiles
};

// Row `i` of head h of sequence s, which has n blocks from g0 on.
template <bool MASKED> __device__ __forceinline__ Unit unit_of(const ArgsF32& a, int s, int g0, int n, int h, int i) {
  Unit u;
  u.g0 = g0;
  u.n = n;
  u.h = h;
  u.block = g0 + i;
  // blocks that hold real tokens and the real tokens of the last of them; at least one (a tile with every key
  // masked has no finite maximum); blocks from nbv on are padding as a whole and are left out
  const int tokens = MASKED ? min(max(a.seq_tokens[s], 1), 64 * n) : 64 * n;
  u.nbv = (tokens + 63) >> 6;
  u.tail = tokens - 64 * (u.nbv - 1);
  const int row = (a.plan_heads > 1 ? h : 0) * a.nb_total + u.block;
  u.p0 = a.to_pos[row];
  u.p1 = a.to_pos[row + 1];
  u.head_base = (int64_t(g0) * a.heads + int64_t(h) * n) * 4096;
  return u;
}

// flat unit id = block + head * n_s + first block of the sequence * heads
template <bool MASKED> __device__ __forceinline__ Unit unit_at(const ArgsF32& a, int unit) {
  int lo = 0, hi = a.batch;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.seq_blocks[mid] * a.heads <= unit) lo = mid; else hi = mid;
  }
  const int g0 = a.seq_blocks[lo], n = a.seq_blocks[lo + 1] - g0, rem = unit - g0 * a.heads, h = rem / n;
  return unit_of<MASKED>(a, lo, g0, n, h, rem - h * n);
}

// The unit on fp32 matrix instructions, four waves, no overlap: the arithmetic of fp32 itself.
template <bool MASKED>
__device__ void run_plain(const ArgsF32& a, const Unit& u, float (*ks)[PITCH], float (*vs)[PITCH]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool works = wave < 4;                         // the workgroup's other waves only keep its barriers
  const int qcol = lane & 15, grp = lane >> 4;
  const int dm = a.heads * 64;

  // Q^T operand: lane holds Q[16 wave + qcol][4 step + grp] for step = 0..15
  float qreg[16];
  if (works) {
    const int qrow = 16 * wave + qcol;
    if (a.q_rows) {
      const float* src = a.q_rows + (int64_t(u.block) * 64 + qrow) * (3 * dm) + u.h * 64;
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int d = 4 * s + grp;
        qreg[s] = (src[d] + (a.q_bias ? a.q_bias[u.h * 64 + d] : 0.f)) * a.q_scale;
      }
    } else {
      const float* src = a.q + u.head_base + int64_t(u.block - u.g0) * 4096;
#pragma unroll
      for (int s = 0; s < 16; ++s) qreg[s] = src[frag_index(qrow, 4 * s + grp)];
    }
  }

  f32x4 o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  for (int p = u.p0; p < u.p1; ++p) {
    const int blk = min(max(a.to_idx[p], 0), u.n - 1); // a malformed index must not lead outside the (sequence, head)
    if (MASKED && blk >= u.nbv) continue;                // the same in every thread of the workgroup
    __syncthreads();                                   // the previous tile's readers are done
    if (works) {
      stage_tile<false>(a.k + u.head_base + int64_t(blk) * 4096, ks);
      stage_tile<true>(a.vt + u.head_base + int64_t(blk) * 4096, vs);
    }
    __syncthreads();
    if (!works) continue;
    f32x4 s[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < 16; ++st)
        s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[16 * kt + qcol][4 * st + grp], qreg[st], s[kt], 0, 0, 0);
    }
    if (MASKED && blk == u.nbv - 1 && u.tail < 64) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (16 * kt + 4 * grp + e >= u.tail) s[kt][e] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[kt][e]);
    mx = group_max(mx);
    const float m_new = fmaxf(m, mx);                  // finite: key 0 of a block is never padding
    const float c = exp2f(m - m_new);
    float part = 0.f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[kt][e] = exp2f(s[kt][e] - m_new);
        part += s[kt][e];
      }
    l = l * c + group_sum(part);
    m = m_new;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      o[dt] *= c;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[16 * dt + qcol][16 * kt + 4 * grp + e], s[kt][e], o[dt], 0, 0, 0);
    }
  }
  if (!works) return;
  // O^T accumulator dt: lane holds d = 16 dt + 4 grp + e for query qcol
  const float inv = 1.0f / fmaxf(l, 1e-30f);          // a row that lists nothing but padding writes zeros
  float* dst = a.out + (int64_t(u.block) * 64 + 16 * wave + qcol) * dm + u.h * 64;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) *reinterpret_cast<f32x4*>(dst + 16 * dt + 4 * grp) = o[dt] * inv;
}

// Eight numbers as three bf16 parts; p[0] + p[1] + p[2] is the number.  Each part is what is left, rounded to nearest: the
// second is at most 2^-8 of the number and the third 2^-17, with either sign, and the third is exact.
__device__ __forceinline__ void cut8(const f32x4& x, const f32x4& y, u32x4 (&p)[3]) {
  float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
#pragma unroll
  for (int part = 0; part < 3; ++part) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2 * i], v[2 * i + 1]}, bf16x2));
      p[part][i] = w;
      if (part < 2) {
        v[2 * i] -= __uint_as_float(w << 16);
        v[2 * i + 1] -= __uint_as_float(w & 0xffff0000u);
      }
    }
  }
}

// The largest value of the four lanes that share lane & 15.
__device__ __forceinline__ float lanes_max(float v) {
  const uint32_t x = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  const uint32_t y = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
  const auto t = __builtin_amdgcn_permlane16_swap(y, y, false, false);
  return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}

__device__ __forceinline__ f32x4 mma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The six products of parts, the smallest first.
constexpr int PART_A[6] = {2, 1, 0, 1, 0, 0}, PART_B[6] = {0, 1, 2, 0, 1, 0};

template <bool MASKED>
__device__ void run_unit(const ArgsF32& a, const Unit& u, char* smem) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qcol = lane & 15, grp = lane >> 4, half = wave >> 2, dm = a.heads * 64;

  // Q operand: step s, lane: Q[16 (wave & 3) + qcol][32 s + 8 grp .. + 8]
  u32x4 q[2][3];
  bool bad = false;                                    // the unit has to be run again by the plain kernel
  {
    const int qrow = 16 * (wave & 3) + qcol;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int d = 32 * s + 8 * grp;
      f32x4 x, y;
      if (a.q_rows) {
        const float* src = a.q_rows + (int64_t(u.block) * 64 + qrow) * (3 * dm) + u.h * 64 + d;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (src[e] + (a.q_bias ? a.q_bias[u.h * 64 + d + e] : 0.f)) * a.q_scale;
        x = f32x4{v[0], v[1], v[2], v[3]};
        y = f32x4{v[4], v[5], v[6], v[7]};
      } else {
        const float* src = a.q + u.head_base + int64_t(u.block - u.g0) * 4096 + frag_index(qrow, d);
        x = *reinterpret_cast<const f32x4*>(src);
        y = *reinterpret_cast<const f32x4*>(src + 4);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = fabsf(e < 4 ? x[e & 3] : y[e & 3]);
        bad = bad | ((v != 0.f) & !((v >= 0x1p-109f) & (v <= 0x1p80f)));
      }
      cut8(x, y, q[s]);
    }
  }

  // A thread's part of a tile: lane's eight numbers of fragment `wave`, for K eight d of one key, for V^T keys
  // 16 j + 4 x .. + 4 and 16 j + 8 + 4 x .. + 4 of one d (j = wave & 3, x = lane >> 5).
  f32x4 kr[2], vr[2];
  auto block_of = [&](int p) { return min(max(a.to_idx[p], 0), u.n - 1); };   // a malformed index must not lead outside the (sequence, head)
  auto fetch = [&](int blk) __attribute__((always_inline)) {
    const int64_t at = u.head_base + int64_t(blk) * 4096 + threadIdx.x * 8;
    kr[0] = *reinterpret_cast<const f32x4*>(a.k + at);
    kr[1] = *reinterpret_cast<const f32x4*>(a.k + at + 4);
    vr[0] = *reinterpret_cast<const f32x4*>(a.vt + at);
    vr[1] = *reinterpret_cast<const f32x4*>(a.vt + at + 4);
  };
  const int row = 2 * (wave >> 2) + ((lane >> 4) & 1);             // the 16-row tile it belongs to
  const int k_at = row * 2048 + ((wave >> 1) & 1) * 1024 + (2 * (wave & 1) + (lane >> 5)) * 256 + qcol * 16;
  const int v_at = 3 * PLANE + row * 2048 + ((wave >> 1) & 1) * 1024 + (lane >> 5) * 256 + qcol * 16 + 8 * (wave & 1);
  auto store = [&](char* buf) __attribute__((always_inline)) {
    u32x4 p[3];
    cut8(kr[0], kr[1], p);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(buf + i * PLANE + k_at) = p[i];
    cut8(vr[0], vr[1], p);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      *reinterpret_cast<u32x2*>(buf + i * PLANE + v_at) = u32x2{p[i][0], p[i][1]};
      *reinterpret_cast<u32x2*>(buf + i * PLANE + v_at + 512) = u32x2{p[i][2], p[i][3]};
    }
  };

  f32x4 o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  int blk = 0, next = 0;                          // of the tile in LDS and of the one in registers
  if (u.p0 < u.p1) {
    blk = block_of(u.p0);
    fetch(blk);
    store(smem);
    if (u.p0 + 1 < u.p1) fetch(next = block_of(u.p0 + 1));
  }
  __syncthreads();
  for (int p = u.p0; p < u.p1; ++p) {
    const char* buf = smem + ((p - u.p0) & 1) * BUFFER;
    int after = 0;
    if (p + 1 < u.p1) {
      store(smem + ((p + 1 - u.p0) & 1) * BUFFER);     // its readers finished before the last barrier
      if (p + 2 < u.p1) fetch(after = block_of(p + 2));
    }
    // padding as a whole, or (the last tile with real tokens) in all the keys of this half: nothing to add
    const bool last_real = MASKED && blk == u.nbv - 1 && u.tail < 64;
    if (!MASKED || (blk < u.nbv && !(last_real && u.tail <= 32 * half))) {
      f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        u32x4 kf[2][3];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 3; ++i)
            kf[t][i] = *reinterpret_cast<const u32x4*>(buf + i * PLANE + (2 * half + t) * 2048 + st * 1024 + lane * 16);
#pragma unroll
        for (int c = 0; c < 6; ++c)
#pragma unroll
          for (int t = 0; t < 2; ++t) s[t] = mma(kf[t][PART_A[c]], q[st][PART_B[c]], s[t]);
      }
      if (last_real) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (32 * half + 16 * t + 4 * grp + e >= u.tail) s[t][e] = -INFINITY;
      }
      float mx = s[0][0];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[t][e]);
      const float m_new = fmaxf(m, lanes_max(mx));     // finite: the first key of this half is not padding
      if (__any(m_new != m)) {
        const float c = __builtin_amdgcn_exp2f(m - m_new);
        l *= c;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= c;
        m = m_new;
      }
      float part = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[t][e] = __builtin_amdgcn_exp2f(s[t][e] - m);
          part += s[t][e];
        }
      l += part;                                       // the lane's own keys; added up over the lanes at the end
      u32x4 pp[3];
      cut8(s[0], s[1], pp);
#pragma unroll
      for (int dt = 0; dt < 4; dt += 2) {
        u32x4 vf[2][3];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 3; ++i)
            vf[t][i] = *reinterpret_cast<const u32x4*>(buf + (3 + i) * PLANE + (dt + t) * 2048 + half * 1024 + lane * 16);
#pragma unroll
        for (int c6 = 0; c6 < 6; ++c6)
#pragma unroll
          for (int t = 0; t < 2; ++t) o[dt + t] = mma(vf[t][PART_A[c6]], pp[PART_B[c6]], o[dt + t]);
      }
    }
    blk = next;
    next = after;
    __syncthreads();
  }
  l = group_sum(l);

  // The upper half's state joins the lower half's (a half that has seen no key has m = -inf, l = 0).
  float* const room = reinterpret_cast<float*>(smem) + ((wave & 3) * 64 + lane) * 4;
  if (half) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) *reinterpret_cast<f32x4*>(room + dt * 1024) = o[dt];
    *reinterpret_cast<f32x4*>(room + 4096) = f32x4{m, l, 0.f, 0.f};
  }
  __syncthreads();
  if (!half) {
    const f32x4 ml = *reinterpret_cast<const f32x4*>(room + 4096);
    const float mm = fmaxf(m, ml[0]);
    const float c0 = m == -INFINITY ? 0.f : exp2f(m - mm), c1 = ml[0] == -INFINITY ? 0.f : exp2f(ml[0] - mm);
    l = l * c0 + ml[1] * c1;
    bad = bad | !(l < INFINITY);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      o[dt] = o[dt] * c0 + *reinterpret_cast<const f32x4*>(room + dt * 1024) * c1;
#pragma unroll
      for (int e = 0; e < 4; ++e) bad = bad | !(fabsf(o[dt][e]) < INFINITY);
    }
    // O^T accumulator dt: lane holds d = 16 dt + 4 grp + e for query qcol
    const float inv = 1.0f / fmaxf(l, 1e-30f);        // a row that lists nothing but padding writes zeros
    float* dst = a.out + (int64_t(u.block) * 64 + 16 * wave + qcol) * dm + u.h * 64;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const f32x4 r = o[dt] * inv;
#pragma unroll
      for (int e = 0; e < 4; ++e) bad = bad | ((r[e] != 0.f) & (fabsf(r[e]) < 0x1p-100f));
      *reinterpret_cast<f32x4*>(dst + 16 * dt + 4 * grp) = r;
    }
  }
  // (its barrier also lets the next unit have the LDS)
  if (__syncthreads_or(bad)) {
    float (*tiles)[PITCH] = reinterpret_cast<float (*)[PITCH]>(smem);
    run_plain<MASKED>(a, u, tiles, tiles + 64);
    __syncthreads();
  }
}

template <bool MASKED>
__global__ __launch_bounds__(THREADS) void bs_attention_f32_kernel(ArgsF32 a) {
  __shared__ __attribute__((aligned(16))) char smem[2 * BUFFER];
  const int n_units = a.nb_total * a.heads;
  if (a.from_pos) {
    // a plan the host has not checked must not lead outside from_idx: clamp the slice, skip bad ids
    const int begin = min(max(a.from_pos[blockIdx.x], 0), n_units);
    const int end = min(max(a.from_pos[blockIdx.x + 1], begin), n_units);
    for (int p = begin; p < end; ++p) {
      const int unit = a.from_idx[p];
      if (unit >= 0 && unit < n_units) run_unit<MASKED>(a, unit_at<MASKED>(a, unit), smem);
    }
    return;
  }
  // Without a plan one unit per workgroup, the rows that list every block (the first and the last of a sequence) first:
  // they take up to ten times as long as the others.  Two lists, the two ends of every (sequence, head) and the rows
  // between them.  Workgroups go to the XCDs round-robin: XCD x takes the x-th eighth of either list, so a head's tiles are
  // read into one L2.  Measured at 12 heads x 4 x 2048: 346 us in flat order, 136 in this one.  Every workgroup has a unit: with
  // a second list of all rows, whose ends returned at once, the workgroups at work came in a pattern that left a part
  // of every XCD idle (12 heads x 60 x 256 tokens 188, 60 x 320 195, 60 x 64 37; now 133, 183, 20).
  const int lane = threadIdx.x & 63, x = blockIdx.x & 7;
  const unsigned long long upto = (2ull << lane) - 1ull;            // the lanes up to this one
  int before = 0;                                                   // ends of earlier sequences
  for (int s0 = 0; s0 < a.batch; s0 += 64) {
    const int n = a.seq_blocks[min(s0 + lane + 1, a.batch)] - a.seq_blocks[min(s0 + lane, a.batch)];
    before += __popcll(__ballot(n >= 1)) + __popcll(__ballot(n >= 2));
  }
  const int64_t ends = int64_t(before) * a.heads, rows = n_units - ends;
  const int end_lo = int(ends * x / 8), end_hi = int(ends * (x + 1) / 8), row_lo = int(rows * x / 8), row_hi = int(rows * (x + 1) / 8);
  int j = int(blockIdx.x >> 3);
  const bool is_end = j < end_hi - end_lo;
  j = is_end ? j + end_lo : j - (end_hi - end_lo) + row_lo;
  if (!is_end && j >= row_hi) return;
  before = 0;
  for (int s0 = 0; s0 < a.batch; s0 += 64) {
    const int g0 = a.seq_blocks[min(s0 + lane, a.batch)], g1 = a.seq_blocks[min(s0 + lane + 1, a.batch)], n = g1 - g0;
    const unsigned long long one = __ballot(n >= 1), two = __ballot(n >= 2);
    const int ends_upto = before + __popcll(one & upto) + __popcll(two & upto);
    const int count = is_end ? min(n, 2) : max(n - 2, 0), last = (is_end ? ends_upto : g1 - ends_upto) * a.heads;
    const unsigned long long there = __ballot(last > j);
    if (there) {
      const int l = __builtin_ctzll(there), c = __builtin_amdgcn_readlane(count, l);
      const int k = j - (__builtin_amdgcn_readlane(last, l) - c * a.heads), h = k / c, i = k - h * c;
      const int first = __builtin_amdgcn_readlane(g0, l), blocks = __builtin_amdgcn_readlane(n, l);
      if (first + blocks > a.nb_total) return;
      run_unit<MASKED>(a, unit_of<MASKED>(a, s0 + l, first, blocks, h, !is_end ? i + 1 : i == 0 ? 0 : blocks - 1), smem);
      return;
    }
    before += __popcll(one) + __popcll(two);
  }
}

}  // namespace

namespace rt {

int launch_attention_f32(const void* q, const void* q_rows, const void* q_bias, float q_scale, const void* k,
                         const void* vt, void* out, const int* seq_blocks_dev, const int* seq_tokens_dev, int batch,
                         int total_blocks, int heads, const int* to_idx, const int* to_pos, int plan_heads,
                         const int* from_idx, const int* from_pos, int n_wg, void* stream) {
  const ArgsF32 a{(const float*)q, (const float*)k, (const float*)vt, (float*)out, seq_blocks_dev, batch, heads,
                  total_blocks, to_idx, to_pos, plan_heads, from_idx, from_pos, seq_tokens_dev,
                  (const float*)q_rows, (const float*)q_bias, q_scale};
  // an XCD's eighths of the two lists together: at most an eighth of the units and two more
  const unsigned units = unsigned(total_blocks) * unsigned(heads), grid = from_idx ? unsigned(n_wg) : 8u * ((units + 14) / 8);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (seq_tokens_dev) RT_LAUNCH(bs_attention_f32_kernel<true>, dim3(grid), dim3(THREADS), 0, st, a);
  else RT_LAUNCH(bs_attention_f32_kernel<false>, dim3(grid), dim3(THREADS), 0, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return rt::fail(RT_EIO, "fp32 bs_attention launch failed: %s", hipGetErrorString(e));
  return RT_OK;
}

}  // namespace rt
