// Block-sparse (BigBird-pattern) attention forward for gfx950, d = 64, 64-token blocks.
//
// Work unit = (sequence, head, from-block): 64 queries against the key blocks its CSR row
// lists (7/8 blocks for a sparse row, all n blocks for the two global rows).
//
// One wave owns all 64 queries of a unit and streams K / V^T tiles straight from global
// memory into MFMA operand registers: the QKV split kernel stores every 64x64 tile in
// "fragment order" (8 fragments of 64 lanes x 16 bytes), so each operand request is one fully
// coalesced 1 KiB buffer load and the tile loop needs no LDS and no barrier.
//
// MFMA formulation (v_mfma_f32_32x32x16_{f16,bf16}, fp32 accumulators):
//   S^T[key][query] = K[key][:] . Q[query][:]       A = K fragment,   B = Q fragment
//   O^T[d][query]  += V^T[d][key] . P^T[key][query]  A = V^T fragment, B = P (registers)
// Both products put the query on the accumulator column (lane & 31): max, sum and rescale
// factors are per-lane scalars and the S^T accumulators, after exp2, are the B operand of
// the second product, so P never leaves registers.  Softmax is evaluated in base 2 (q arrives
// pre-multiplied by log2(e)/sqrt(d)).
//
// Two tile loops:
//   pipelined (common path)  a (64 query x 64 key) tile is four 32x32 accumulator tiles
//       a = (key half, query half); step j issues, one matrix instruction per handful of
//       vector instructions, S^T(a[j+1]) and O^T += V^T P^T(a[j-1]) on the matrix pipe while
//       the vector pipe turns S^T(a[j]) into P^T(a[j]).  The reference maximum is fixed per row
//       (maximum over the row's first 32 keys, shared by a lane's two queries) and enters the
//       score product as the MFMA's C operand.  Nothing is tested inside the loop: a row whose
//       scores outgrow the reference shows up as a row sum that is not finite.
//   moving maximum (fallback) such rows and rows of more than 64 entries per wave are run by the loop that tracks the
//       maximum tile by tile.  The two loops never share a loop nest: the register allocator treats them apart, and the
//       pipelined one stays free of scratch-memory traffic.
//
// Schedule: one workgroup of four waves per global row (the first and the last block of a sparse sequence), whose tiles the waves
// share and whose results meet in LDS, then one per four other rows, a wave each; two workgroups to a CU, started by the
// hardware as earlier ones end.  Workgroups are dealt round-robin to the 8 XCDs, each of which has its own L2: XCD x owns the x-th
// eighth of the rows, head-major.  Few rows are cut finer (cut_rows).  With an LPT plan (from_idx / from_pos) n_wg
// workgroups walk their unit lists instead.
//
// Bound by the tile loop, where a wave alone on its SIMD takes 0.97 us a tile and two together 0.77 (matrix and vector
// pipe at the clock they leave each other, K / V^T requests on the CU's path from the L2), and by 4 us ahead of a row's first tile
// (geometry, block list, queries, tile: four dependent round trips), in which the SIMD's other wave runs alone.
// 8 x 4096 tokens, 12 heads, fp16, 62.6 GFLOP: 74 us.
//
// Replaces, from the reference: layers/kernels/sparse_attention.cu:2953-3190 (balanced,
// persistent workgroups over the LPT plan), :2111-2403 (one workgroup per unit) and the
// dispatcher :3192-3228.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rt_launch.h"


namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const int __attribute__((address_space(4))) const_int;   // loads through it are scalar loads

template <typename T> struct Mma;
template <> struct Mma<_Float16> {
  typedef f16x8 v8;
  typedef f16x4 v4;
  __device__ static f32x16 run(v8 a, v8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
  // a[0..7] = p[0..7] rounded to T; returns the fp32 sum of the ROUNDED values (what PV multiplies)
  __device__ static float pack(const float* p, v8& out) {
    float s = 0.f;
    u32x4 w;                                  // whole dwords: each pair stays one v_cvt_pk_f16_f32
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f16x2 h = __builtin_convertvector(f32x2{p[2 * i], p[2 * i + 1]}, f16x2);
      w[i] = __builtin_bit_cast(uint32_t, h);
      s = __builtin_amdgcn_fdot2(h, f16x2{1, 1}, s, false);
    }
    out = __builtin_bit_cast(v8, w);
    return s;
  }
  // pipelined loop: two values of P rounded to nearest (a value beyond fp16's range must become
  // infinite: that is how the loop's caller learns that the row outgrew its reference), their sums
  // kept in packed halves
  static constexpr bool kPackedSum = true;
  __device__ static uint32_t two(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
  }
  __device__ static uint32_t add(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, a) + __builtin_bit_cast(f16x2, b));
  }
  __device__ static float fold(uint32_t a, float acc) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), f16x2{1, 1}, acc, false);
  }
};
template <> struct Mma<__bf16> {
  typedef bf16x8 v8;
  typedef bf16x4 v4;
  __device__ static f32x16 run(v8 a, v8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
  // a[0..7] = p[0..7] rounded to bf16; returns the fp32 sum of the UNROUNDED values: converting the
  // rounded ones back would cost as many instructions again, and the rounding errors of a row's
  // sum (relative 2^-9 each, random sign) are far below what bf16 outputs resolve
  __device__ static float pack(const float* p, v8& out) {
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = static_cast<__bf16>(p[e]);
    return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
  }
  static constexpr bool kPackedSum = false;
  __device__ static uint32_t two(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
  }
  __device__ static uint32_t add(uint32_t a, uint32_t) { return a; }
  __device__ static float fold(uint32_t, float acc) { return acc; }
};

// Moving-maximum loop: a row's reference maximum only moves when the 32 values P = 2^(score -
// reference) a lane holds for one key tile add up to more than 2^11 (no single P can then exceed
// 2^11, far inside fp16's range, and P keeps its full relative precision at any magnitude): the row
// sum the kernel needs anyway doubles as the overflow test.
constexpr float SUM_LIMIT = 2048.0f;
// Pipelined loop: the lane's two queries share one reference; if their own maxima over the first 32
// keys lie further apart than this (log2 units), the smaller row's P would sink towards fp16's
// denormals and the unit takes the moving-maximum loop instead.
constexpr float MAX_REFERENCE_GAP = 8.0f;

// Online-softmax state of one wave for its 64 queries: O^T as [d tile][query tile].
struct State {
  f32x16 o[2][2];
  float m[2], l[2];      // per query tile: reference maximum (log2 units), partial row sum
};

// Reference of a query that has met keys, all of them with a score of minus infinity; -INFINITY: it has met none.  No
// finite score lies below it, so it gives way to any, and a share of a row's tiles that holds nothing but such keys adds
// nothing to the other shares.
constexpr float LOWEST = -3.402823466e+38f;

__device__ inline void state_init(State& st) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int e = 0; e < 16; ++e) st.o[t][nt][e] = 0.f;
  st.m[0] = st.m[1] = -INFINITY;
  st.l[0] = st.l[1] = 0.f;
}

// Scores of padded keys become minus infinity: no weight.  The others gain log2(times), as if the tile were listed that
// often.  s = 32 x 32 accumulator tile of key half kt; the key of element e in this lane is
// 32 kt + 8 (e >> 2) + (e & 3) + 4 (lane >> 5), padding from `tail` on.
__device__ inline void mask_padded(f32x16& s, int kt, int tail, int lane, int times = 1) {
  int lim = tail - 4 * (lane >> 5);
  asm volatile("" : "+v"(lim));       // the 16 comparisons are made here, not once per kernel and kept in 32 scalar pairs
#pragma unroll
  for (int e = 0; e < 16; ++e) s[e] = (32 * kt + 8 * (e >> 2) + (e & 3) >= lim) ? -INFINITY : s[e];
  if (times > 1) {
    const float gain = __builtin_amdgcn_logf(float(times));
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] += gain;
  }
}

template <typename T>
__device__ inline void load_tile(const T* __restrict__ tile, int lane, typename Mma<T>::v8 (&f)[8]) {
  typedef typename Mma<T>::v8 v8;
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = *reinterpret_cast<const v8*>(tile + i * 512 + lane * 8);
}

// Moving-maximum loop.  Streams key blocks row[first], row[first + step], ... of one (sequence,
// head) through the state.  kbase / vbase point at block 0 of that (sequence, head); n = blocks in
// the sequence.  The row's block ids are fetched 64 at a time into one register (lane j holds
// entry j) and handed out with v_readlane: one memory round trip per unit instead of one per key block.
template <typename T, bool MASKED>
__device__ inline void stream_tiles(const T* __restrict__ kbase, const T* __restrict__ vbase,
                                    const int* __restrict__ row, int first, int step, int cnt, int n, int tail, int nbv,
                                    int lane, const typename Mma<T>::v8 (&qf)[2][4], State& st) {
  typedef typename Mma<T>::v8 v8;
  v8 kf[8], vf[8];
  bool fresh = true;                                  // no reference maximum yet
  // Rows longer than 64 entries are walked in chunks of 64: the ids are only (re)loaded between
  // chunks, so inside the tile loop the only outstanding memory operations are the tile
  // prefetches and the waits on them can be exact.
  for (int j = first; j < cnt;) {
  const int chunk = j >> 6;
  const int hi = min(cnt, (chunk + 1) * 64);
  const int ids = (chunk * 64 + lane < cnt) ? row[chunk * 64 + lane] : 0;
  auto block_of = [&](int e) {                        // e is wave-uniform and inside the chunk
    const int b = __builtin_amdgcn_readlane(ids, e & 63);
    return b < 0 ? 0 : (b >= n ? n - 1 : b);
  };
  int bcur = block_of(j);
  load_tile<T>(kbase + int64_t(bcur) * 4096, lane, kf);
  load_tile<T>(vbase + int64_t(bcur) * 4096, lane, vf);
  for (; j < hi; j += step) {
    const int jn = j + step;
    const bool more = jn < hi;
    // keys beyond the sequence's true length are padding and get no weight: the tail of block nbv - 1 is masked, a
    // block from nbv on is left out as a whole (its tile has been requested like any other and is dropped)
    const bool padded = MASKED && tail < 64 && bcur == nbv - 1;
    const bool skipped = MASKED && bcur >= nbv;
    // the last iteration re-requests its own tile: loads stay unconditional, so they keep
    // their place in the instruction stream (a branch would sink them next to their use)
    const int bn = block_of(more ? jn : j);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      f32x16 sc[2];
      v8 pb[4];
      float psum;
      auto scores = [&](float init) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int e = 0; e < 16; ++e) sc[t][e] = init;
#pragma unroll
          for (int c = 0; c < 4; ++c) sc[t] = Mma<T>::run(kf[t * 4 + c], qf[nt][c], sc[t]);
        }
        if (MASKED && padded) {                         // wave-uniform, at most one tile of a row
          mask_padded(sc[0], 0, tail, lane);
          mask_padded(sc[1], 1, tail, lane);
        }
      };
      // exp2 of the (already shifted) scores -> P as the B operand of the second product:
      // step s takes accumulator registers 8*(s&1)..+7 of key tile s>>1.  Returns true when the
      // lane's 32 values of P add up to more than SUM_LIMIT (or to something not finite).
      auto exponentiate = [&]() {
        float part[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float p8[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) p8[e] = __builtin_amdgcn_exp2f(sc[s >> 1][8 * (s & 1) + e]);
          part[s] = Mma<T>::pack(p8, pb[s]);
        }
        psum = (part[0] + part[1]) + (part[2] + part[3]);
        return !(psum <= SUM_LIMIT);                    // also true for an infinite or undefined sum
      };
      bool redo = fresh && !skipped;
      if (!fresh && !skipped) {
        scores(-st.m[nt]);
        redo = __any(exponentiate());
      }
      if (redo) {
        // rare (always on the first tile): find the true maximum and move the reference there
        scores(0.f);
        float mx = sc[0][0];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[t][e]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(mx, fresh ? LOWEST : st.m[nt]);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) sc[t][e] -= m_new;
        if (!fresh) {
          const float alpha = __builtin_amdgcn_exp2f(st.m[nt] - m_new);
          st.l[nt] *= alpha;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) st.o[t][nt][e] *= alpha;
        }
        st.m[nt] = m_new;
        (void)exponentiate();
      }
      // the K fragments are dead once the second query tile's scores are final
      if (nt == 1) {
        __builtin_amdgcn_sched_barrier(0);
        load_tile<T>(kbase + int64_t(bn) * 4096, lane, kf);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (!skipped) {
        st.l[nt] += psum;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int s = 0; s < 4; ++s) st.o[t][nt] = Mma<T>::run(vf[t * 4 + s], pb[s], st.o[t][nt]);
      }
    }
    fresh = fresh && skipped;
    bcur = bn;
    __builtin_amdgcn_sched_barrier(0);
    load_tile<T>(vbase + int64_t(bn) * 4096, lane, vf);
    __builtin_amdgcn_sched_barrier(0);
  }
  }
}

// v_permlane32_swap: the upper 32 lanes of a change places with the lower 32 lanes of b.  Written as
// assembly, which says itself that a and b are two registers: an earlier compiler gave the builtin one where both operands hold the
// same value.  (The one in use copies the operand first; the LayerNorms' row sums rely on it.  s_nop: a vector instruction
// may just have written the operands.)
__device__ inline void swap_halves(unsigned& a, unsigned& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
// maximum / sum over lane l and lane l ^ 32, in both lanes
__device__ inline float pair_max(float x) {
  unsigned a = __builtin_bit_cast(unsigned, x), b = a;
  swap_halves(a, b);
  return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
__device__ inline float pair_sum(float x) {
  unsigned a = __builtin_bit_cast(unsigned, x), b = a;
  swap_halves(a, b);
  return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}

// the 64 rows of a unit's outputs
template <typename T> __device__ __forceinline__ __amdgpu_buffer_rsrc_t unit_rows(T* out_unit, int64_t row_stride) {
  return __builtin_amdgcn_make_buffer_rsrc(out_unit, 0, uint32_t(row_stride) * 128u, 0x00020000);
}

// Writes the wave's 64x64 output tile, O^T[d = 32t + 8*(e>>2) + 4*(lane>>5) + (e&3)]
// [query 32nt + (lane&31)] * w, to out[token][h*64 + d], through the wave's own LDS room (64 rows, OUT_PITCH bytes
// apart; no other wave touches it, and the LDS operations of one wave execute in order).  A lane holds 4
// consecutive d of its query per accumulator quad: every lane parks its 16 quads, then lane L takes the 16-byte
// chunk (L & 7) of tokens 8k + (L >> 3), so that a store instruction writes eight whole 128-byte lines.  Stores
// straight from the accumulators (lane pairs swapping quads) write 32 bytes to each of 32 lines per instruction,
// four pieces per line: same bits, 2-3 % more kernel time.
constexpr int OUT_PITCH = 144;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <typename T>
__device__ inline void store_output(T* __restrict__ out_unit, int64_t row_stride, int lane, const State& st,
                                    const float (&w)[2], char* stage) {
  const int l32 = lane & 31, hi = lane >> 5;
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    char* row = stage + (32 * nt + l32) * OUT_PITCH + 8 * hi;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t x0 = Mma<T>::two(st.o[t][nt][4 * q] * w[nt], st.o[t][nt][4 * q + 1] * w[nt]);
        const uint32_t x1 = Mma<T>::two(st.o[t][nt][4 * q + 2] * w[nt], st.o[t][nt][4 * q + 3] * w[nt]);
        *reinterpret_cast<u32x2*>(row + 64 * t + 16 * q) = u32x2{x0, x1};
      }
  }
  const char* rd = stage + (lane >> 3) * OUT_PITCH + (lane & 7) * 16;
  const __amdgpu_buffer_rsrc_t dst = unit_rows(out_unit, row_stride);
  const uint32_t at = uint32_t(lane >> 3) * uint32_t(row_stride) * 2u + uint32_t(lane & 7) * 16u;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(rd + k * 8 * OUT_PITCH);
    __builtin_amdgcn_raw_buffer_store_b128(v, dst, int(at + uint32_t(8 * k) * uint32_t(row_stride) * 2u), 0, rt::WRITE_THROUGH);
  }
}

struct Unit {
  int h, i, n, g0;
  int tail;               // real tokens in the sequence's last block that holds any (64: none padded)
  int nbv;                // blocks of the sequence that hold real tokens (n without padding): blocks from nbv on are
                          // padding as a whole and get no weight as keys
};

// One unit's row of the to-block CSR, for the wave that runs it (all fields wave-uniform).
struct Row {
  Unit u;
  int p0, cnt;            // the row is to_idx[p0 .. p0 + cnt)
  int goff;               // byte offset of the unit's (sequence, head) group inside K and V^T
};

template <typename T> struct Args {
  const T* q; const T* k; const T* vt; T* out;
  const int* seq_blocks; int batch, heads, nb_total;
  const int* to_idx; const int* to_pos; int plan_heads;
  const int* from_idx; const int* from_pos;
  const int* seq_tokens;                 // optional: true token count per sequence (padded tail in its last block)
  // optional: Q taken from the QKV projection's own output rows [tokens, 3 * heads * 64] (columns
  // 0 .. heads*64-1), bias added and scale applied while loading; q is then unused
  const T* q_rows; const T* q_bias; float q_scale;
};

constexpr int MAX_BATCH = 1024;         // sequences per launch (16 to a lane)
constexpr int MAX_BLOCKS = 4096;        // 64-token blocks per launch
constexpr int MAX_HEADS_QROWS = 64;     // heads whose query bias fits the LDS copy

__device__ inline bool is_global_row(const Unit& u) { return u.n >= RT_MIN_SPARSE_BLOCKS && (u.i == 0 || u.i == u.n - 1); }

// ---------------------------------------------------------------------------------------------
// memory requests of the pipelined loop: raw buffer loads, one resource per array, the tile's
// byte offset in a scalar register and the fragment's in the instruction's immediate field
// ---------------------------------------------------------------------------------------------
template <typename T> struct Buffers {
  __amdgpu_buffer_rsrc_t k, v, q;
};

template <typename T>
__device__ inline typename Mma<T>::v8 fetch(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(typename Mma<T>::v8, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// Where a unit's 64x64 query tile lies, as MFMA B fragments: fragment (nt, c) is a buffer load at
// vector offset voff, scalar offset soff + nt * nt_step + c * c_step.
struct QPlan { int voff, soff, nt_step, c_step; };
template <typename T>
__device__ inline QPlan q_plan(const Args<T>& a, const Unit& u, int lane) {
  QPlan q;
  if (a.q_rows) {
    // raw projection rows: request k = 4 nt + c takes the 128-byte head slices of queries 8k .. 8k + 7 whole,
    // eight lanes per query (eight cache lines per request; taking MFMA fragments straight from the rows
    // would touch 32 lines per request and return four times as slowly).  finish_q turns the eight
    // requests' registers into fragments through LDS.
    const int ld = a.heads * 384;                                   // bytes per token row of [T, 3 * heads * 64]
    q.voff = (lane >> 3) * ld + (lane & 7) * 16;
    q.soff = (u.g0 + u.i) * 64 * ld + u.h * 128;
    q.nt_step = 32 * ld;
    q.c_step = 8 * ld;
  } else {
    q.voff = lane * 16;
    q.soff = (u.g0 * a.heads + u.h * u.n + u.i) * 8192;
    q.nt_step = 4096;
    q.c_step = 1024;
  }
  return q;
}
template <typename T>
__device__ inline typename Mma<T>::v8 fetch_q(const Buffers<T>& b, const QPlan& q, int k) {   // k = 4 nt + c
  return fetch<T>(b.q, q.voff, q.soff + (k >> 2) * q.nt_step + (k & 3) * q.c_step);
}
template <typename T>
__device__ inline void request_q(const Args<T>& a, const Buffers<T>& b, const Unit& u, int lane,
                                 typename Mma<T>::v8 (&qf)[2][4]) {
  const QPlan q = q_plan<T>(a, u, lane);
#pragma unroll
  for (int k = 0; k < 8; ++k) qf[k >> 2][k & 3] = fetch_q<T>(b, q, k);
}

// What the queries-from-rows route keeps in LDS: a copy of the query bias and, per wave, room for one 64 x 64
// query tile in row order (rows Q_STAGE_PITCH bytes apart).
constexpr int Q_STAGE_PITCH = 144;
constexpr int Q_STAGE_BYTES = 64 * Q_STAGE_PITCH;
static_assert(OUT_PITCH == Q_STAGE_PITCH, "the output tile is parked in the room of the query tile");
template <typename T> struct QSide { const T* bias; char* stage; };

// Rows -> fragments through the wave's own LDS room (no other wave touches it: LDS operations of one wave
// execute in order), then (x + bias) * scale in fp32, rounded once: the arithmetic of the split kernel.
template <typename T>
__device__ inline void scale_q(const Args<T>& a, const T* qbias, const Unit& u, int lane, typename Mma<T>::v8 (&qf)[2][4]) {
  typedef typename Mma<T>::v8 v8;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const v8 bb = *reinterpret_cast<const v8*>(qbias + u.h * 64 + c * 16 + (lane >> 5) * 8);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        // pinned in fp32 before the rounding, as in the split kernel: multiply and rounding must not fuse
        float y = (float(qf[nt][c][e]) + float(bb[e])) * a.q_scale;
        asm volatile("" : "+v"(y));
        qf[nt][c][e] = static_cast<T>(y);
      }
  }
}
template <typename T>
__device__ inline void finish_q(const Args<T>& a, const QSide<T>& qs, const Unit& u, int lane,
                                typename Mma<T>::v8 (&qf)[2][4]) {
  typedef typename Mma<T>::v8 v8;
  if (!a.q_rows) return;
  {
    char* wr = qs.stage + (lane >> 3) * Q_STAGE_PITCH + (lane & 7) * 16;
#pragma unroll
    for (int k = 0; k < 8; ++k) *reinterpret_cast<v8*>(wr + k * 8 * Q_STAGE_PITCH) = qf[k >> 2][k & 3];
    const char* rd = qs.stage + (lane & 31) * Q_STAGE_PITCH + (lane >> 5) * 16;
#pragma unroll
    for (int k = 0; k < 8; ++k) qf[k >> 2][k & 3] = *reinterpret_cast<const v8*>(rd + (k >> 2) * 32 * Q_STAGE_PITCH + (k & 3) * 32);
  }
  scale_q<T>(a, qs.bias, u, lane, qf);
}

// lane j: byte offset inside K / V^T of the tile of the row's entry first + j * step (the first 64 of them)
template <typename T>
__device__ inline int row_offsets(const Args<T>& a, const Row& r, int first, int step, int lane) {
  const int e = first + lane * step;
  int blk = e < r.cnt ? a.to_idx[r.p0 + e] : 0;
  blk = blk < 0 ? 0 : (blk >= r.u.n ? r.u.n - 1 : blk);
  return r.goff + blk * 8192;
}

// CSR row bounds through scalar loads
template <typename T>
__device__ inline void describe(const Args<T>& a, const Unit& u, Row& r) {
  r.u = u;
  const int row = __builtin_amdgcn_readfirstlane((a.plan_heads > 1 ? u.h : 0) * a.nb_total + u.g0 + u.i);
  const_int* pos = (const_int*)(uintptr_t)(a.to_pos);
  r.p0 = pos[row];
  r.cnt = pos[row + 1] - r.p0;
  r.goff = (u.g0 * a.heads + u.h * u.n) * 8192;
}

#define SB() __builtin_amdgcn_sched_barrier(0)

// The pipelined loop's registers.
template <typename T> struct Tiles {
  typename Mma<T>::v8 qf[2][4], kf[8], vf[8];
};

// first tile of a row, requested in the loop's own order: K's first key half, then the halves the
// loop's first step does not request itself (so the loop's waits, which count requests still in
// flight, come out the same on its first trip as on any other)
template <typename T>
__device__ inline void request_first(const Buffers<T>& b, int so, int lane, Tiles<T>& t) {
  const int vo = lane * 16;
#pragma unroll
  for (int f = 0; f < 4; ++f) t.kf[f] = fetch<T>(b.k, vo + f * 1024, so);
  SB();
#pragma unroll
  for (int f = 4; f < 8; ++f) t.kf[f] = fetch<T>(b.k, vo + f * 1024, so);
#pragma unroll
  for (int f = 0; f < 4; ++f) t.vf[(f & 1) + 4 * (f >> 1)] = fetch<T>(b.v, vo + ((f & 1) + 4 * (f >> 1)) * 1024, so);
  SB();
  // the loop's first step multiplies an all-zero P with V^T's second key half, which is only
  // requested after it: whatever those registers hold must be finite
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int e = 0; e < 8; ++e) t.vf[(f & 1) + 2 + 4 * (f >> 1)][e] = static_cast<T>(0.f);
}

// Padding of a sequence, for the pipelined loop (MASKED kernels).  drop_off = byte offset (inside K / V^T) of the
// sequence's first block that is padding as a whole: tiles from there on are taken off the wave's tile list.
// pad_off = offset of the tile whose keys from `tail` on are padding, -1 if there is none.  The loop masks in its
// last tile only, so a row's padded tile is moved to the end of the list (the order of a row's tiles does not matter
// to the result beyond rounding; the reference comes from the first tile).  A row that lists it several times (the plan of
// 1024 tokens draws the last block once more for some rows) meets it once, with the binary logarithm of the number added to
// its scores: such a row took the moving-maximum loop before.  Sequences 17 tokens short, f16, before / now in us: 6 of 8512 in
// all 37.0 / 24.5, 10 x 1024 (16 heads) 64 / 42, 32 x 1024 168 / 109.  Where no row lists it twice: 30 x 1193-1483 123.1 / 123.2,
// 24 x 1563-2483 139.7 / 139.7, 14 x 77-376 13.15 / 13.22.
struct Padding { int pad_off, drop_off, tail, last; };
__device__ inline Padding padding_of(const Unit& u, int goff) {
  Padding pd;
  pd.pad_off = u.tail < 64 ? goff + (u.nbv - 1) * 8192 : -1;
  pd.drop_off = goff + u.nbv * 8192;
  pd.tail = u.tail;
  pd.last = 0;
  return pd;
}
// Lanes 0 .. my-1 of ids hold the tile offsets of the wave's entries.  Takes the tiles that are padding as a whole
// off the list (my shrinks), moves the padded tile to the last lane in use, further entries of it behind that, and sets
// pd.last to their number.
__device__ inline void pad_to_end(int& ids, int& my, int lane, Padding& pd) {
  pd.last = 0;
  const unsigned long long listed = __ballot(lane < my), dropped = __ballot(lane < my && ids >= pd.drop_off);
  const unsigned long long pads = pd.pad_off < 0 ? 0 : __ballot(lane < my && ids == pd.pad_off) & ~dropped;
  const unsigned long long front = listed & ~dropped & ~pads;
  if ((dropped | pads) == 0) return;
  if (dropped == 0 && (pads & (pads - 1)) == 0) {            // one: it and the last entry change places
    const int jp = __builtin_ctzll(pads);
    if (jp != my - 1) {
      const int moved = __builtin_amdgcn_readlane(ids, my - 1);
      ids = lane == jp ? moved : (lane == my - 1 ? pd.pad_off : ids);
    }
    pd.last = 1;
    return;
  }
  // a permutation: the others in order, the padded tiles, the dropped ones; lanes beyond the list stay
  auto below = [](unsigned long long m) { return int(__builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0))); };
  const int n_front = __popcll(front), n_pads = __popcll(pads);
  int dest = below(front);
  if (!(front >> lane & 1ull)) dest = (pads >> lane & 1ull) ? n_front + below(pads) : n_front + n_pads + below(dropped);
  if (lane >= my) dest = lane;
  ids = __builtin_amdgcn_ds_permute(dest * 4, ids);
  my = n_front + (n_pads > 0);
  pd.last = n_pads;
}

// reference of the pipelined loop: maximum over the row's first 32 keys, shared by the lane's two
// queries.  False if the two queries' maxima lie too far apart.  pad_first (MASKED only): the row's first tile
// is the padded one, so keys from the tail on do not count (there is always at least one that does).
template <typename T, bool MASKED>
__device__ inline bool fast_reference(const Tiles<T>& t, float& mref, bool pad_first, int tail, int lane) {
  typedef Mma<T> P;
  f32x16 s0 = {}, s1 = {};
  if (MASKED && pad_first) {
    mask_padded(s0, 0, tail, lane);
    s1 = s0;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    s0 = P::run(t.kf[c], t.qf[0][c], s0);
    s1 = P::run(t.kf[c], t.qf[1][c], s1);
  }
  float m0 = s0[0], m1 = s1[0];
#pragma unroll
  for (int e = 1; e < 16; ++e) { m0 = fmaxf(m0, s0[e]); m1 = fmaxf(m1, s1[e]); }
  m0 = pair_max(m0);
  m1 = pair_max(m1);
  mref = fmaxf(m0, m1);
  return !__any(!(fabsf(m0 - m1) <= MAX_REFERENCE_GAP));           // false also for NaN / infinite scores
}

// The pipelined tile loop over `my` (1..64) tiles whose byte offsets sit in the lanes of `ids`; the first tile is in flight
// or there (request_first).
template <typename T, bool MASKED>
__device__ inline void fast_loop(const Buffers<T>& b, int ids, int my, int lane, float mref, Tiles<T>& t, State& st, const Padding& pd) {
  typedef typename Mma<T>::v8 v8;
  typedef Mma<T> P;
  state_init(st);
  st.m[0] = st.m[1] = mref;
  f32x16 negm;                                        // the score products' C operand
#pragma unroll
  for (int e = 0; e < 16; ++e) negm[e] = -mref;
  int vo = lane * 16;
  auto ldk = [&](int f, int so) { t.kf[f] = fetch<T>(b.k, vo + f * 1024, so); };
  auto ldv = [&](int f, int so) { t.vf[f] = fetch<T>(b.v, vo + f * 1024, so); };
  f32x16 sc[2];
  v8 pb[2][2];
  float l0 = 0.f, l1 = 0.f;
  int so_cur = __builtin_amdgcn_readlane(ids, 0);
  // Everything requested so far must have arrived before the loop is entered (its first step needs
  // most of it anyway).  The waits inside the loop count the requests in flight; the compiler
  // derives them from the state at the loop's entry as well as from the loop's own requests, and
  // anything still pending there turns them into waits for all requests.
  __builtin_amdgcn_s_waitcnt(0x0F70);                 // vmcnt(0)
  // Inside the loop a wave yields to the other wave of its SIMD whenever that one is between two loops (queries,
  // reference, output): that code is a chain of short latencies, the loop always has matrix work in flight.
  __builtin_amdgcn_s_setprio(0);
  SB();
  // pipeline prologue: scores of the first accumulator tile; an all-zero P for the first step's PV slot
  sc[0] = negm;
#pragma unroll
  for (int c = 0; c < 4; ++c) sc[0] = P::run(t.kf[c], t.qf[0][c], sc[0]);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) pb[1][s][e] = static_cast<T>(0.f);

  // one tile: four steps; `last` (a std::bool_constant): the row's last tile
  auto tile = [&](int so_next, auto last) {
    constexpr bool LAST = decltype(last)::value;
    // keeps the fragment offsets inside the loop body, where they fold into the requests' immediate fields
    asm volatile("" : "+v"(vo));
#pragma unroll
    for (int S = 0; S < 4; ++S) {
      // consume sc[S & 1] (tile a[S]), produce sc[(S + 1) & 1] (a[S + 1]), multiply pb[(S + 1) & 1] (a[S - 1])
      const int nt = S & 1;
      const int ktn = ((S + 1) & 3) >> 1, ntn = (S + 1) & 1;          // a[S + 1]
      const int ktp = ((S + 3) & 3) >> 1, ntp = (S + 3) & 1;          // a[S - 1]
      f32x16& cur = sc[S & 1];
      f32x16& nxt = sc[(S + 1) & 1];
      v8 (&pprev)[2] = pb[(S + 1) & 1];
      float p[16];
      uint32_t w[8];
      uint32_t t01 = 0, t23 = 0, t45 = 0, t67 = 0;
      float lacc = 0.f;
      // a row's padded tile is its last one (pad_to_end): its scores lose the padded keys before they are exponentiated
      if (MASKED && LAST && pd.last) mask_padded(cur, S >> 1, pd.tail, lane, pd.last);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        SB();
        // matrix slot
        if ((i & 1) == 0) {
          const int c = i >> 1;
          // the last tile's last step has no following scores to start
          if (!(LAST && S == 3)) nxt = P::run(t.kf[ktn * 4 + c], t.qf[ntn][c], c == 0 ? negm : nxt);
        } else {
          const int tt = (i >> 1) & 1, s = i >> 2;
          st.o[tt][ntp] = P::run(t.vf[tt * 4 + 2 * ktp + s], pprev[s], st.o[tt][ntp]);
        }
        // tile requests: one per slot in the steps whose registers are free
        if (S == 1 && i >= 4) { const int f = (i & 1) + 2 + 4 * ((i >> 1) & 1); ldv(f, so_cur); }
        if (S == 1 && i < 4 && !LAST) ldk(i, so_next);
        if (S == 3 && !LAST) { if (i < 4) ldk(4 + i, so_next); else { const int f = (i & 1) + 4 * ((i >> 1) & 1); ldv(f, so_next); } }
        SB();
        // vector slot: two exponentials, rounding and sums of the previous slot's pair
        p[2 * i] = __builtin_amdgcn_exp2f(cur[2 * i]);
        p[2 * i + 1] = __builtin_amdgcn_exp2f(cur[2 * i + 1]);
        if (i > 0) {
          w[i - 1] = P::two(p[2 * i - 2], p[2 * i - 1]);
          if (!P::kPackedSum) lacc += p[2 * i - 2] + p[2 * i - 1];
        }
        if (P::kPackedSum) {
          if (i == 2) t01 = P::add(w[0], w[1]);
          if (i == 4) t23 = P::add(w[2], w[3]);
          if (i == 5) t01 = P::add(t01, t23);
          if (i == 6) t45 = P::add(w[4], w[5]);
          if (i == 7) t01 = P::add(t01, t45);
        }
      }
      SB();
      w[7] = P::two(p[14], p[15]);
      if (P::kPackedSum) {
        t67 = P::add(w[6], w[7]);
        t01 = P::add(t01, t67);
        if (nt == 0) l0 = P::fold(t01, l0); else l1 = P::fold(t01, l1);
      } else {
        lacc += p[14] + p[15];
        if (nt == 0) l0 += lacc; else l1 += lacc;
      }
      u32x4 lo = {w[0], w[1], w[2], w[3]}, up = {w[4], w[5], w[6], w[7]};
      pb[S & 1][0] = __builtin_bit_cast(v8, lo);
      pb[S & 1][1] = __builtin_bit_cast(v8, up);
      SB();
    }
  };

  for (int e = 0; e + 1 < my; ++e) {
    const int so_next = __builtin_amdgcn_readlane(ids, (e + 1) & 63);
    tile(so_next, std::false_type{});
    so_cur = so_next;
  }
  tile(so_cur, std::true_type{});
  // pipeline epilogue: the last tile's a[3] (second key half, second query half)
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int s = 0; s < 2; ++s) st.o[tt][1] = P::run(t.vf[tt * 4 + 2 + s], pb[1][s], st.o[tt][1]);
  st.l[0] = l0;
  st.l[1] = l1;
  __builtin_amdgcn_s_setprio(1);
}

__device__ inline bool sums_finite(const State& st) { return !__any(!(st.l[0] < INFINITY) || !(st.l[1] < INFINITY)); }

// moving-maximum loop on entries first, first + step, ... of row r
template <typename T, bool MASKED>
__device__ inline void slow_row(const Args<T>& a, const Buffers<T>& b, const QSide<T>& qbias, const Row& r, int first, int step,
                                int lane, bool have_q, typename Mma<T>::v8 (&qf)[2][4], State& st) {
  if (!have_q) {
    request_q<T>(a, b, r.u, lane, qf);
    finish_q<T>(a, qbias, r.u, lane, qf);
  }
  state_init(st);
  const int64_t gbase = int64_t(r.goff >> 1);
  stream_tiles<T, MASKED>(a.k + gbase, a.vt + gbase, a.to_idx + r.p0, first, step, r.cnt, r.u.n, r.u.tail, r.u.nbv, lane, qf, st);
}

// Entries first, first + step, ... of row r for the pipelined loop: the tiles the wave has (ids, my, pd), the first of them
// requested.
enum { SHARE_SLOW, SHARE_EMPTY, SHARE_RUNS };      // for the moving-maximum loop (more than 64 entries); no tile that counts
template <typename T, bool MASKED>
__device__ inline int begin_share(const Args<T>& a, const Buffers<T>& b, const Row& r, int first, int step, int lane, Tiles<T>& t,
                                  int& ids, int& my, Padding& pd) {
  first = __builtin_amdgcn_readfirstlane(first);
  my = __builtin_amdgcn_readfirstlane((r.cnt - first + step - 1) / step);           // this wave's entries
  if (my <= 0) return SHARE_EMPTY;
  if (my > 64) return SHARE_SLOW;
  ids = row_offsets<T>(a, r, first, step, lane);
  pd = padding_of(r.u, r.goff);
  if (MASKED) {
    pad_to_end(ids, my, lane, pd);
    if (my == 0) return SHARE_EMPTY;                   // every tile of this wave's share is padding
  }
  request_first<T>(b, __builtin_amdgcn_readlane(ids, 0), lane, t);
  return SHARE_RUNS;
}
// The share through the state, its queries in t.qf (they are there afterwards too).  False: the row has to be run with the
// moving-maximum loop instead (scores that outgrew the reference); the state is then undefined.
template <typename T, bool MASKED>
__device__ inline bool end_share(const Buffers<T>& b, int ids, int my, const Padding& pd, int lane, Tiles<T>& t, State& st) {
  float mref;
  if (!fast_reference<T, MASKED>(t, mref, pd.last > 0 && my == 1, pd.tail, lane)) return false;
  fast_loop<T, MASKED>(b, ids, my, lane, mref, t, st, pd);
  return sums_finite(st);
}

// One over a row's whole sum.  A row that has met nothing but padding writes zeros; one whose keys all have a score
// of minus infinity has no softmax (only the moving-maximum loop meets such rows).
__device__ inline float row_weight(float l, float m) {
  return l == 0.f && m == LOWEST ? __builtin_nanf("") : __builtin_amdgcn_rcpf(fmaxf(l, 1e-30f));
}

// ---- rows of a workgroup ----------------------------------------------------------------------------------------------
// A share's outputs in LDS: 64 queries x 64 fp32 in rows 272 bytes apart, which puts the 16 lanes of an access on different
// banks both for the writes (16 rows, 16 bytes of each) and for the reads (2 rows, every second 16 bytes).
constexpr int SLOT_PITCH = 68, SLOT_FLOATS = 64 * SLOT_PITCH;
template <typename T, int NW> struct Room {
  // a slot per wave; ahead of the merge, query tiles (wave w's own at stage(w), a shared row's at that of its number)
  __attribute__((aligned(16))) float slots[NW][SLOT_FLOATS];
  float m[8][64], l[8][64];                            // per share and query: reference and sum
  __attribute__((aligned(16))) T qbias[MAX_HEADS_QROWS * 64];
  __device__ __forceinline__ char* stage(int w) { return reinterpret_cast<char*>(slots) + w * Q_STAGE_BYTES; }
  // Per row: a wave's pipelined loop handed it back.  Between the rows of the last slot, behind the query tiles.  (With four
  // waves the room is half of a CU's LDS to the byte.)
  static_assert(NW * Q_STAGE_BYTES <= (NW - 1) * SLOT_FLOATS * 4, "the flags lie behind the query tiles");
  __device__ __forceinline__ int& failed(int row) { return reinterpret_cast<int&>(slots[NW - 1][row * SLOT_PITCH + 64]); }
};

// The bias copy and cleared flags; the caller's barrier follows.
template <typename T, int NW> __device__ __forceinline__ void ready_room(const Args<T>& a, Room<T, NW>& room) {
  if (a.q_rows)
    for (int i = threadIdx.x; i < a.heads * 64; i += 64 * NW) room.qbias[i] = a.q_bias ? a.q_bias[i] : static_cast<T>(0.f);
  if (threadIdx.x < 8) room.failed(threadIdx.x) = 0;
}

// Padding of sequence s, which has u.n blocks
template <typename T, bool MASKED> __device__ __forceinline__ void set_padding(const Args<T>& a, int s, Unit& u) {
  u.tail = 64;
  u.nbv = u.n;
  if (MASKED) {
    const int tokens = min(max(__builtin_amdgcn_readfirstlane(a.seq_tokens[s]), 1), 64 * u.n);
    u.nbv = (tokens + 63) >> 6;
    u.tail = tokens - 64 * (u.nbv - 1);
  }
}

// Lane l: where sequences l, l + 64, ... of the batch begin and end (CHUNKS of them).
template <typename T, int CHUNKS> struct Batch {
  int lane, sb0[CHUNKS], sb1[CHUNKS];
  __device__ __forceinline__ explicit Batch(const Args<T>& a) {
    lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      sb0[c] = a.seq_blocks[min(64 * c + lane, a.batch)];
      sb1[c] = a.seq_blocks[min(64 * c + lane + 1, a.batch)];
    }
  }
  // which sequences of chunk c there are, and which have global rows
  __device__ __forceinline__ unsigned long long there(const Args<T>& a, int c) const { return __ballot(64 * c + lane < a.batch); }
  __device__ __forceinline__ unsigned long long sparse(const Args<T>& a, int c) const {
    return __ballot(64 * c + lane < a.batch && sb1[c] - sb0[c] >= RT_MIN_SPARSE_BLOCKS);
  }
  __device__ __forceinline__ int sparse_count(const Args<T>& a) const {
    int n = 0;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) n += __popcll(sparse(a, c));
    return n;
  }
  // row i of sequence l of chunk c
  template <bool MASKED> __device__ __forceinline__ Unit unit_at(const Args<T>& a, int c, int l, int h, int i) const {
    Unit u;
    u.g0 = __builtin_amdgcn_readlane(sb0[c], l);
    u.n = __builtin_amdgcn_readlane(sb1[c], l) - u.g0;
    u.h = h;
    u.i = i;
    set_padding<T, MASKED>(a, 64 * c + l, u);
    return u;
  }
  // the first row of the k-th sequence that has global rows
  template <bool MASKED> __device__ __forceinline__ Unit global_row(const Args<T>& a, int h, int k) const {
    Unit u{};
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const unsigned long long mask = sparse(a, c);
      const int here = __popcll(mask);
      if (k >= 0 && k < here)
        u = unit_at<MASKED>(a, c, __builtin_ctzll(__ballot((mask >> lane & 1ull) && __popcll(mask & ((1ull << lane) - 1ull)) == k)), h, 0);
      k -= here;
    }
    return u;
  }
  // the j-th of the rows that are not global ones
  template <bool MASKED> __device__ __forceinline__ Unit other_row(const Args<T>& a, int h, int j) const {
    Unit u{};
    int before = 0;                                    // sequences with global rows in earlier chunks
    bool found = false;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const unsigned long long mask = sparse(a, c);
      const int listed = sb0[c] - 2 * (before + __popcll(mask & ((1ull << lane) - 1ull)));       // rows of earlier sequences
      before += __popcll(mask);
      if (!found && j < __builtin_amdgcn_readlane(sb1[c], 63) - 2 * before) {
        const int l = __popcll(there(a, c) & __ballot(listed <= j)) - 1;
        u = unit_at<MASKED>(a, c, l, h, j - __builtin_amdgcn_readlane(listed, l) + int(mask >> l & 1ull));
        found = true;
      }
    }
    return u;
  }
};

// The units of a caller's plan, whose ids are blk + head * n + first block * heads, in a batch of up to 64 sequences: lane l
// knows where sequence l begins and ends.
template <typename T> struct UnitsOfFew {
  struct Place {};
  Batch<T, 1> batch;
  __device__ __forceinline__ explicit UnitsOfFew(const Args<T>& a) : batch(a) {}
  __device__ __forceinline__ Place place(const Args<T>&, int) const { return {}; }
  template <bool MASKED> __device__ __forceinline__ Unit unit(const Args<T>& a, const Place&, int id) const {
    Unit u{};
    if (id >= __builtin_amdgcn_readlane(batch.sb1[0], 63) * a.heads) return u;
    const int l = __popcll(batch.there(a, 0) & __ballot(batch.sb0[0] * a.heads <= id)) - 1;
    const int g0 = __builtin_amdgcn_readlane(batch.sb0[0], l), n = __builtin_amdgcn_readlane(batch.sb1[0], l) - g0;
    const int rem = id - g0 * a.heads, h = rem / n;
    return batch.template unit_at<MASKED>(a, 0, l, h, rem - h * n);
  }
};
// The same in a batch of up to 1024: lane l knows where sequence 16 l begins, and the 16 that a unit may be of are looked up
// (place requests them, unit waits).  All 1024 in the lanes are 32 registers that the pipelined loop does not have: it
// spilled 47-66 (12 heads into 512, us, before / now: 65 sequences of 1-20 blocks f16 130 / 120, bf16 padded 144 / 122; 100 of 3 blocks 37.9 / 29.3).
template <typename T> struct UnitsOfMany {
  struct Place { int first, begins; };                 // lane l: where sequence first + l begins
  static_assert(MAX_BATCH <= 64 * 16, "a lane for every 16 sequences");
  int lane, begins16, total;
  __device__ __forceinline__ explicit UnitsOfMany(const Args<T>& a) {
    lane = threadIdx.x & 63;
    begins16 = a.seq_blocks[min(16 * lane, a.batch)];
    total = __builtin_amdgcn_readfirstlane(a.seq_blocks[a.batch]);
  }
  __device__ __forceinline__ Place place(const Args<T>& a, int id) const {
    const int first = max(16 * __popcll(__ballot(16 * lane < a.batch && begins16 * a.heads <= id)) - 16, 0);
    return {first, a.seq_blocks[min(first + lane, a.batch)]};
  }
  template <bool MASKED> __device__ __forceinline__ Unit unit(const Args<T>& a, const Place& p, int id) const {
    Unit u{};
    if (id >= total * a.heads) return u;
    const int l = __popcll(__ballot(lane < 16 && p.first + lane < a.batch && p.begins * a.heads <= id)) - 1;
    u.g0 = __builtin_amdgcn_readlane(p.begins, l);
    u.n = __builtin_amdgcn_readlane(p.begins, l + 1) - u.g0;
    const int rem = id - u.g0 * a.heads;
    u.h = rem / u.n;
    u.i = rem - u.h * u.n;
    set_padding<T, MASKED>(a, p.first + l, u);
    return u;
  }
};

template <typename T> __device__ __forceinline__ Buffers<T> buffers_of(const Args<T>& a) {
  Buffers<T> b;
  const uint32_t kv_bytes = uint32_t(a.nb_total) * uint32_t(a.heads) * 8192u;
  b.k = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.k), 0, kv_bytes, 0x00020000);
  b.v = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.vt), 0, kv_bytes, 0x00020000);
  b.q = a.q_rows ? __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.q_rows), 0, kv_bytes * 3u, 0x00020000)
                 : __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.q), 0, kv_bytes, 0x00020000);
  return b;
}

// The queries of a row in t.qf of all its WAVES waves: wave `part` fetches its part of the eight requests, all read the tile
// from LDS.  fetch_queries requests, share_queries ends behind the workgroup's barrier (none if a row has one wave).
template <int WAVES, typename T>
__device__ __forceinline__ void fetch_queries(const Args<T>& a, const Buffers<T>& b, const Unit& u, int part, int lane, Tiles<T>& t) {
  const QPlan q = q_plan<T>(a, u, lane);
#pragma unroll
  for (int j = 0; j < 8 / WAVES; ++j) t.qf[j >> 2][j & 3] = fetch_q<T>(b, q, part + j * WAVES);
}
template <int WAVES, typename T>
__device__ __forceinline__ void share_queries(const Args<T>& a, const T* qbias, const Unit& u, bool valid, char* stage, int part, int lane, Tiles<T>& t) {
  typedef typename Mma<T>::v8 v8;
  // rows, read as fragments; or the fragments as they are
  const int wr = a.q_rows ? (lane >> 3) * Q_STAGE_PITCH + (lane & 7) * 16 : lane * 16, wr_k = a.q_rows ? 8 * Q_STAGE_PITCH : 1024;
  const int rd = a.q_rows ? (lane & 31) * Q_STAGE_PITCH + (lane >> 5) * 16 : lane * 16;
  const int rd_nt = a.q_rows ? 32 * Q_STAGE_PITCH : 4096, rd_c = a.q_rows ? 32 : 1024;
  if (valid) {
#pragma unroll
    for (int j = 0; j < 8 / WAVES; ++j) *reinterpret_cast<v8*>(stage + wr + (part + j * WAVES) * wr_k) = t.qf[j >> 2][j & 3];
  }
  if (WAVES > 1) __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int k = 0; k < 8; ++k) t.qf[k >> 2][k & 3] = *reinterpret_cast<const v8*>(stage + rd + (k >> 2) * rd_nt + (k & 3) * rd_c);
  if (a.q_rows) scale_q<T>(a, qbias, u, lane, t.qf);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
// The state's outputs times w in the wave's slot, 16 runs of 4 per lane; ADD: plus what stands there times w4.
template <bool ADD> __device__ __forceinline__ void to_slot(float* slot, const State& st, const float (&w)[2], const float (&w4)[2], int lane) {
#pragma clang fp contract(off)
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4* const at = reinterpret_cast<f32x4*>(slot + (32 * nt + (lane & 31)) * SLOT_PITCH + 32 * t + 8 * q + 4 * (lane >> 5));
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = st.o[t][nt][4 * q + e] * w[nt];
        if (ADD) {
          const f32x4 kept = *at;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = x[e] + kept[e] * w4[nt];
        }
        *at = x;
      }
}

// The SHARES shares of a row, one or two per wave, to its output, in two steps: every wave scales its outputs to the largest of
// the shares' references and leaves them in its slot; then every wave adds up its part of the queries, over all of the row's
// slots, and stores it.  Sums are formed in the order ((0 + 4) + (2 + 6)) + ((1 + 5) + (3 + 7)), or its part for fewer shares,
// whoever forms them.
template <typename T, int NW, int SHARES>
__device__ __forceinline__ void merge_shares(Room<T, NW>& room, const State& st, T* out_unit, int64_t stride, bool valid, int row,
                                             int part, int lane, int wave) {
#pragma clang fp contract(off)
  constexpr int WAVES = SHARES < NW ? SHARES : NW;
  constexpr bool TWO = SHARES > NW;
  const int base = row * WAVES;                        // the row's first share
  auto reference = [&](int query) {                    // of the whole row; finite even if no share has met a key
    float m[SHARES];
#pragma unroll
    for (int s = 0; s < SHARES; ++s) m[s] = room.m[base + s][query];
#pragma unroll
    for (int s = 1; s < SHARES; ++s) m[0] = fmaxf(m[0], m[s]);
    return m[0];
  };
  {
    float w[2], w4[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int query = 32 * nt + (lane & 31);
      const float m = fmaxf(reference(query), LOWEST);
      w[nt] = __builtin_amdgcn_exp2f(st.m[nt] - m);
      w4[nt] = TWO ? __builtin_amdgcn_exp2f(room.m[part + 4][query] - m) : 0.f;
      if (lane < 32) {
        room.l[base + part][query] = st.l[nt] * w[nt];
        if (TWO) room.l[part + 4][query] *= w4[nt];
      }
    }
    to_slot<TWO>(room.slots[wave], st, w, w4, lane);
  }
  __syncthreads();
  if (!valid) return;
  // eight queries at a time, eight outputs per lane
  constexpr int TIMES = 8 / WAVES;
  const int first = part * (64 / WAVES) + (lane >> 3);
  float l[TIMES][SHARES];
  f32x4 x[TIMES][WAVES][2];
#pragma unroll
  for (int i = 0; i < TIMES; ++i) {
#pragma unroll
    for (int s = 0; s < SHARES; ++s) l[i][s] = room.l[base + s][first + 8 * i];
#pragma unroll
    for (int s = 0; s < WAVES; ++s) {
      const f32x4* const from = reinterpret_cast<const f32x4*>(room.slots[base + s] + (first + 8 * i) * SLOT_PITCH + (lane & 7) * 8);
      x[i][s][0] = from[0];
      x[i][s][1] = from[1];
    }
  }
#pragma unroll
  for (int i = 0; i < TIMES; ++i) {
#pragma unroll
    for (int half = SHARES / 2; half >= 1; half /= 2)
#pragma unroll
      for (int s = 0; s < half; ++s) {
        l[i][s] = l[i][s] + l[i][s + half];
        if (half < WAVES) {
          x[i][s][0] = x[i][s][0] + x[i][s + half][0];
          x[i][s][1] = x[i][s][1] + x[i][s + half][1];
        }
      }
    float w = __builtin_amdgcn_rcpf(fmaxf(l[i][0], 1e-30f));
    if (__any(l[i][0] == 0.f)) w = row_weight(l[i][0], reference(first + 8 * i));       // no key, or none with a finite score
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = Mma<T>::two(x[i][0][e >> 1][2 * (e & 1)] * w, x[i][0][e >> 1][2 * (e & 1) + 1] * w);
    __builtin_amdgcn_raw_buffer_store_b128(o, unit_rows(out_unit, stride), int((uint32_t(first + 8 * i) * uint32_t(stride) + uint32_t(lane & 7) * 8u) * 2u),
                                           0, rt::WRITE_THROUGH);
  }
}

// The workgroup's NW waves on their rows, from the first tile to the output: a row's tiles in SHARES shares, taken by that many
// waves side by side, or by all NW, two each, if there are fewer.  u: the wave's row; `valid`: it has one.
template <typename T, bool MASKED, int SHARES, int NW>
__device__ __forceinline__ void share_rows(const Args<T>& a, const Buffers<T>& b, Room<T, NW>& room, const QSide<T>& qbias,
                                           const Unit& u, bool valid, int lane, int wave) {
  constexpr int WAVES = SHARES < NW ? SHARES : NW;
  constexpr bool TWO = SHARES > NW;                    // part and part + 4 (u is valid in all waves)
  static_assert(SHARES <= 2 * NW && (!TWO || NW == 4), "one or two shares per wave");
  const int row = wave / WAVES, part = wave % WAVES;
  float* const slot = room.slots[wave];
  const float ones[2] = {1.f, 1.f};
  const int64_t stride = int64_t(a.heads) * 64;
  T* const out_unit = a.out + int64_t(u.g0 + u.i) * 64 * stride + u.h * 64;
  State st;
  Row r;
  bool redo;                                           // by the moving-maximum loop
  describe<T>(a, u, r);
  auto publish = [&](int s) {                          // what the row's other waves have to know of share s
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      st.l[nt] = pair_sum(st.l[nt]);
      if (lane < 32) {
        room.m[s][32 * nt + lane] = st.m[nt];
        room.l[s][32 * nt + lane] = st.l[nt];
      }
    }
  };
  {
    Tiles<T> t;
    int ids = 0, my = 0, what = SHARE_EMPTY;
    Padding pd;
    if (valid) {
      fetch_queries<WAVES, T>(a, b, u, part, lane, t);
      what = begin_share<T, MASKED>(a, b, r, TWO ? part + 4 : part, SHARES, lane, t, ids, my, pd);
    }
    share_queries<WAVES, T>(a, room.qbias, u, valid, room.stage(row), part, lane, t);
    if (TWO) __syncthreads();                          // the query tile is read: its place is a slot's
    state_init(st);
    bool ok = what == SHARE_RUNS ? end_share<T, MASKED>(b, ids, my, pd, lane, t, st) : what == SHARE_EMPTY;
    if (TWO) {
      publish(part + 4);
      to_slot<false>(slot, st, ones, ones, lane);
      state_init(st);
      what = begin_share<T, MASKED>(a, b, r, part, SHARES, lane, t, ids, my, pd);
      ok = (what == SHARE_RUNS ? end_share<T, MASKED>(b, ids, my, pd, lane, t, st) : what == SHARE_EMPTY) && ok;
    }
    redo = !ok;
    if (SHARES > 1 && redo && lane == 0) room.failed(row) = 1;
  }
  int any_failed = 0;                                  // the same in all waves
  if (SHARES > 1) {
    publish(row * WAVES + part);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW / WAVES; ++i) any_failed |= room.failed(i);
    any_failed = __builtin_amdgcn_readfirstlane(any_failed);
    redo = any_failed && __builtin_amdgcn_readfirstlane(room.failed(row)) != 0;
  }
  if (valid && redo) {
    typename Mma<T>::v8 qf[2][4];
    if (TWO) {                                         // (one row: all waves are here)
      slow_row<T, MASKED>(a, b, qbias, r, part + 4, SHARES, lane, false, qf, st);
      __syncthreads();                                 // the query tiles are read
      publish(part + 4);
      to_slot<false>(slot, st, ones, ones, lane);
    }
    slow_row<T, MASKED>(a, b, qbias, r, part, SHARES, lane, TWO, qf, st);
    if (SHARES > 1) publish(row * WAVES + part);
  }
  if constexpr (SHARES == 1) {
    if (!valid) return;
    float w[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) w[nt] = row_weight(pair_sum(st.l[nt]), st.m[nt]);
    store_output<T>(out_unit, stride, lane, st, w, qbias.stage);
  } else {
    if (any_failed) __syncthreads();
    merge_shares<T, NW, SHARES>(room, st, out_unit, stride, valid, row, part, lane, wave);
  }
}

// share_rows as the launch's cut has it.  Four shares of a row of more than 256 tiles would be longer than the pipelined loop
// takes: such a global row has eight, two to a wave (f16, us, moving-maximum loop / so: 16 heads 1 x 20480 tokens 114.5 / 88.3, 4 heads
// 19200 + 30 x 640 98.0 / 72.0, 1 head 16448 + 8 x 640 116.8 / 52.8).  Beyond 512 tiles the moving-maximum loop has them still.
constexpr int FOUR_SHARES = 4 * 64;
template <typename T, bool MASKED, int OTHERS, int GLOBAL, int NW>
__device__ __forceinline__ void cut_rows_of(const Args<T>& a, const Buffers<T>& b, Room<T, NW>& room, const QSide<T>& qbias, const Unit& u,
                                            bool global, bool valid, int lane, int wave) {
  if constexpr (OTHERS < GLOBAL) {
    if (!global) return share_rows<T, MASKED, OTHERS, NW>(a, b, room, qbias, u, valid, lane, wave);
    if constexpr (GLOBAL == 4)
      if (u.n > FOUR_SHARES) return share_rows<T, MASKED, 8, NW>(a, b, room, qbias, u, true, lane, wave);
  }
  static_assert(GLOBAL >= NW, "one row to the workgroup: it is there");
  share_rows<T, MASKED, GLOBAL, NW>(a, b, room, qbias, u, true, lane, wave);
}

// Workgroup b looks its rows up from the batch's prefix, XCD x taking the x-th eighth of the global rows and then of the rest, both
// head-major: the K / V^T tiles of a (sequence, head) are fetched into one L2.  A global row is a workgroup's, its tiles in
// GLOBAL shares; of the others it takes NW / OTHERS, each in OTHERS shares.  Nothing persists and nothing is drawn: as its waves
// end, the CU starts the next workgroup.  The rows of a workgroup are neighbours and run in step, so they ask for
// the window's tiles within a short time: 8 x 4096 tokens, 12 heads, 295 MB from beyond the L2 where persistent workgroups had 408
// (201 would do), 283 cycles a request and not 358; the CU's own cache meets a sixth of the requests.
// (Persistent workgroups whose waves drew single rows from ticket counters and requested the next row's queries and first tile
// inside the last one's steps took 85-90 us where this takes 74 at 8 x 4096 tokens, 12 heads; 92 / 84 at 16 x 512-4096, 28.6 /
// 24.9 at 5 x 320-3000, 14.7 / 10.9 at 20 x 100-300, 16 heads 139 / 127 at 13120 + 5184 + 10240 + 12224.)
template <typename T, bool MASKED, int OTHERS, int GLOBAL, int NW, int CHUNKS>
__global__ __launch_bounds__(64 * NW, 2) void bs_attention_kernel(Args<T> a) {
  constexpr int ROWS = NW / OTHERS;
  __shared__ Room<T, NW> room;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Batch<T, CHUNKS> batch(a);
  ready_room<T, NW>(a, room);
  const QSide<T> qbias{room.qbias, room.stage(wave)};
  const int n_sparse = batch.sparse_count(a), n_rows = a.nb_total - 2 * n_sparse;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;

  const int n_pairs = n_sparse * a.heads;
  const int p_lo = int(int64_t(n_pairs) * xcd / 8), p_hi = int(int64_t(n_pairs) * (xcd + 1) / 8), n_glob = 2 * (p_hi - p_lo);
  const bool global = slot < n_glob;
  Unit u;
  bool valid = true;
  if (global) {
    const int pair = p_lo + (slot >> 1), h = pair / n_sparse;
    u = batch.template global_row<MASKED>(a, h, pair - h * n_sparse);
    if (slot & 1) u.i = u.n - 1;
  } else {
    const int total = n_rows * a.heads;
    const int lo = int(int64_t(total) * xcd / 8), hi = int(int64_t(total) * (xcd + 1) / 8);
    const int first = lo + (slot - n_glob) * ROWS;
    if (first >= hi) return;
    const int item = first + wave / OTHERS;
    valid = item < hi;
    const int it = valid ? item : first, h = it / n_rows;
    u = batch.template other_row<MASKED>(a, h, it - h * n_rows);
  }
  __syncthreads();
  const Buffers<T> b = buffers_of(a);
  cut_rows_of<T, MASKED, OTHERS, GLOBAL, NW>(a, b, room, qbias, u, global, valid, batch.lane, wave);
}

// With a caller's plan workgroup c walks its slice: four waves, two workgroups per CU, a global row by all of them, other
// entries side by side as far as there are waves for them.  A unit's tiles are cut into as many shares as without a plan, so
// the bits are the same; a wave takes two of a global row's eight, or one of its four.  The slice is clamped to the list, ids
// outside it are skipped.  An LPT plan spreads each (sequence, head) over many XCDs: 8 x 4096 tokens into 512 95 us, without a plan
// 74; 16 x 512-4096 into 1024 116 / 84.
template <typename T, bool MASKED, int OTHERS, int GLOBAL, bool MANY>
__global__ __launch_bounds__(256, 2) void bs_attention_plan_kernel(Args<T> a) {
  constexpr int SIDE = OTHERS < 4 ? 4 / OTHERS : 1;    // rows side by side
  __shared__ Room<T, 4> room;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_units = a.nb_total * a.heads;
  const int begin = min(max(a.from_pos[blockIdx.x], 0), n_units);
  const int end = min(max(a.from_pos[blockIdx.x + 1], begin), n_units);
  if (begin == end) return;
  const std::conditional_t<MANY, UnitsOfMany<T>, UnitsOfFew<T>> units(a);
  ready_room<T, 4>(a, room);
  const QSide<T> qbias{room.qbias, room.stage(wave)};
  const Buffers<T> b = buffers_of(a);
  for (int p = begin; p < end;) {
    int ids[SIDE];                                     // the next entries in one round trip
#pragma unroll
    for (int w = 0; w < SIDE; ++w) {
      ids[w] = __builtin_amdgcn_readfirstlane(p + w < end ? a.from_idx[p + w] : -1);
      if (ids[w] >= n_units) ids[w] = -1;
    }
    if (ids[0] < 0) { ++p; continue; }
    decltype(units.place(a, 0)) at[SIDE];
#pragma unroll
    for (int w = 0; w < SIDE; ++w) at[w] = units.place(a, max(ids[w], 0));
    Unit u = units.template unit<MASKED>(a, at[0], ids[0]);
    const bool whole = is_global_row(u);
    int run = 1;
    if (!whole) {
      const int mine = SIDE * wave / 4;
      bool more = true;
#pragma unroll
      for (int w = 1; w < SIDE; ++w) {
        more = more && ids[w] >= 0;
        if (more) {
          const Unit v = units.template unit<MASKED>(a, at[w], ids[w]);
          more = !is_global_row(v);
          if (more) ++run;
          if (more && w == mine) u = v;
        }
      }
    }
    // what the code below derives from the lane number is derived again for every unit, not kept in registers
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    if (threadIdx.x < 8) room.failed(threadIdx.x) = 0;           // (the last rows' flags were read several barriers ago)
    __syncthreads();
    cut_rows_of<T, MASKED, OTHERS, GLOBAL, 4>(a, b, room, qbias, u, whole, SIDE * wave / 4 < run, lane, wave);
    p += run;
  }
}

// Pairs of global rows the batch can have at most: the host knows the block count, not the sequences' lengths.
int64_t most_pairs(int batch, int total_blocks, int heads) {
  const int sparse = total_blocks / RT_MIN_SPARSE_BLOCKS;
  return int64_t(sparse < batch ? sparse : batch) * heads;
}

// How a launch cuts its rows: shares of a row that is not global and of one that is, waves of a workgroup.  With few rows a
// row's chain of tiles is the time of the launch, so its tiles are spread over 4 or 2 waves while the workgroups, two to a CU
// at most, leave every wave a SIMD mostly to itself.  A global row's chain, a quarter of the sequence's blocks, is halved
// by workgroups of 8 waves where it would outlast the others' work; they fill a CU one at a time, which costs up to 15 % where
// there is work enough.  The longest sequence is not known here: half as long again as the average is taken for it.
// Measured (us in a graph, 12 heads, bf16; others, global, waves 4 4 4 / 2 4 4 / 1 4 4 / 1 8 8): 1 x 64 tokens 5.8 / 6.1 / 5.2 / 5.4,
// 1 x 192 6.0 / 7.0 / 6.9 / 9.1, 1 x 512 6.9 / 8.5 / 10.3 / 15.4, 1 x 1024 8.4 / 8.6 / 10.4 / 15.7, 1 x 1536 11.5 / 9.8 / 10.8 / 16.1,
// 2 x 1024 10.7 / 9.3 / 11.0 / 16.0, 1 x 2048 13.1 / 11.5 / 11.7 / 16.3, 1 x 2560 14.6 / 15.3 / 13.6 / 16.8, 2 x 2048 17.8 / 15.5 / 13.0 /
// 17.3, 1 x 4096 19.4 / 19.8 / 18.8 / 17.9, 2 x 4096 31.7 / 26.4 / 25.2 / 22.4, 4 x 4096 55.0 / 45.8 / 41.4 / 44.8, 16 heads 1 x 8192 39.1 /
// 37.2 / 37.6 / 37.6, 1 x 12288 55.7 / 50.8 / 52.0 / 48.0.
struct Cut { int others, global, waves; };
Cut cut_rows(int batch, int total_blocks, int heads) {
  const Cut four{1, 4, 4}, eight{1, 8, 8};
  if (batch > 64) return four;
  const int64_t units = int64_t(total_blocks) * heads, pairs = most_pairs(batch, total_blocks, heads), global = 2 * pairs;
  const int longest = total_blocks - batch + 1;         // tiles that a row can have at most
  const int likely = batch == 1 ? total_blocks : 3 * total_blocks / (2 * batch);
  const bool one_round = global + (units - global) / 8 <= 256;                        // of workgroups of 8 waves
  // Few units of long sequences: the global rows' chain is all of the time (f16, 4 4 4 / 2 4 4 / 1 8 8: 1 head 1 x 14080 tokens 38.3 / 38.0 /
  // 33.5, 2 heads 9920 + 64 29.6 / 28.3 / 25.6, 1 x 8192 25.4 / 23.9 / 22.1; 1 head 1 x 3840 13.2 / 13.3 / 13.4, 2 x 3200 12.8 / 12.7 / 13.5).
  if (likely > 75 && one_round) return eight;
  if (longest >= 3 && units <= 256) return {4, 4, 4};
  if (longest >= 2 && global + (units - global) / 2 <= 220) return {2, 4, 4};
  if (likely >= 60 && one_round) return eight;
  // From about 1050 units on a round of workgroups of 8 waves takes as long as the same work by 4 if the sequences are not short, and a
  // sequence much longer than the others is done earlier (f16, 1 4 4 / 1 8 8: 12 heads 3 x 1920 tokens 16.8 / 17.2, 3 x 2432 19.4 / 19.2, 640 + 2560 +
  // 2880 18.6 / 19.2, 3200 + 1920 + 1600 20.2 / 17.9, 4096 + 2 x 896 21.9 / 18.2, 4 heads 10 x 1728 14.9 / 15.4, 16000 + 9 x 128 50.1 / 42.4, 9600 + 11 x
  // 896 33.6 / 27.5; below the line 16 heads 3 x 1408 15.7 / 16.8, 640 + 2 x 1920 17.9 / 19.1).  32 CUs to an XCD, as launch_rows deals them.
  if (likely >= 38 && units >= 1056 && 2 * ((pairs + 7) / 8) + ((units + 7) / 8 + 7) / 8 <= 32) return eight;
  // more rounds, and a chain, 5 us and 0.25 a tile, that outlasts the units' 17 ns each (f16, 1 4 4 / 1 8 8: 12 heads 12800 + 1280 tokens 50.0 /
  // 41.0, 8 heads 2 x 11520 48.8 / 39.4, 4 heads 5 x 8192 38.7 / 35.3, 12 heads 2 x 7040 36.4 / 36.6; on the line 12 heads 2 x 8960 46.3 / 49.0; 4 heads
  // 5 x 5760 29.3 / 32.0, whose second round is nearly empty)
  if (likely >= 60 && 5 + 0.25 * likely > (batch == 1 ? 0.0167 : 0.0174) * double(units)) return eight;
  return four;
}

template <typename T> int launch_rows(const Args<T>& a, int n_wg, hipStream_t st) {
  const Cut cut = cut_rows(a.batch, a.nb_total, a.heads);
  auto go = [&](auto masked, auto others, auto global, auto waves, auto chunks) {
    constexpr bool MASKED = decltype(masked)::value;
    constexpr int OTHERS = decltype(others)::value, GLOBAL = decltype(global)::value, NW = decltype(waves)::value, CHUNKS = decltype(chunks)::value;
    if (a.from_pos) {
      RT_LAUNCH((bs_attention_plan_kernel<T, MASKED, OTHERS, GLOBAL, (CHUNKS > 1)>), dim3(unsigned(n_wg)), dim3(256), 0, st, a);
      return;
    }
    // every XCD's share of the global rows (two per head of each sequence that may have them) and of the others
    const int64_t units = int64_t(a.nb_total) * a.heads, pairs = most_pairs(a.batch, a.nb_total, a.heads);
    const int64_t per_xcd = 2 * ((pairs + 7) / 8) + ((units + 7) / 8 + NW / OTHERS - 1) / (NW / OTHERS);
    RT_LAUNCH((bs_attention_kernel<T, MASKED, OTHERS, GLOBAL, NW, CHUNKS>), dim3(unsigned(8 * per_xcd)), dim3(64 * NW), 0, st, a);
  };
  auto pick = [&](auto masked) {
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    const std::integral_constant<int, 4> four;
    const std::integral_constant<int, 8> eight;
    if (a.batch > 64) go(masked, one, four, four, std::integral_constant<int, MAX_BATCH / 64>());
    else if (cut.others == 4) go(masked, four, four, four, one);
    else if (cut.others == 2) go(masked, two, four, four, one);
    else if (cut.global == 8) go(masked, one, eight, eight, one);
    else go(masked, one, four, four, one);
  };
  if (a.seq_tokens) pick(std::true_type());
  else pick(std::false_type());
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? RT_OK : rt::fail(RT_EIO, "bs_attention launch failed: %s", hipGetErrorString(e));
}

int launch_attention(const void* q, const void* q_rows, const void* q_bias, float q_scale, const void* k, const void* vt,
                     void* out, const int* seq_blocks_dev, const int* seq_tokens_dev, int batch, int total_blocks,
                     int heads, const int* to_idx, const int* to_pos, int plan_heads, const int* from_idx,
                     const int* from_pos, int n_wg, int dtype, void* stream) {
  RT_REQUIRE((q || q_rows) && k && vt && out && seq_blocks_dev && to_idx && to_pos, RT_EINVAL, "NULL pointer");
  RT_REQUIRE(batch >= 1 && total_blocks >= batch && heads >= 1, RT_EINVAL, "bad geometry: batch=%d total_blocks=%d heads=%d",
             batch, total_blocks, heads);
  RT_REQUIRE(plan_heads == 1 || plan_heads == heads, RT_EINVAL, "plan_heads=%d must be 1 or heads=%d", plan_heads, heads);
  RT_REQUIRE((from_idx == nullptr) == (from_pos == nullptr), RT_EINVAL, "from_idx and from_pos go together");
  RT_REQUIRE(int64_t(total_blocks) * heads * 8192 * 3 < (int64_t(1) << 31), RT_EINVAL,
             "batch too large: %d blocks x %d heads (byte offsets are 32-bit)", total_blocks, heads);
  RT_REQUIRE(batch <= MAX_BATCH, RT_EINVAL, "at most %d sequences per launch, got %d", MAX_BATCH, batch);
  RT_REQUIRE(total_blocks <= MAX_BLOCKS, RT_EINVAL, "at most %d blocks (%d tokens) per launch, got %d blocks", MAX_BLOCKS,
             MAX_BLOCKS * 64, total_blocks);
  RT_REQUIRE(!q_rows || heads <= MAX_HEADS_QROWS, RT_EINVAL, "queries from the projection rows: at most %d heads, got %d",
             MAX_HEADS_QROWS, heads);
  RT_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(q_rows) | reinterpret_cast<uintptr_t>(q_bias) |
               reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(vt) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0,
             RT_EINVAL, "q (or qkv and its bias), k, vt, out must be 16-byte aligned");
  RT_REQUIRE(dtype == RT_F16 || dtype == RT_BF16 || dtype == RT_F32, RT_EINVAL, "unknown dtype %d", dtype);
  if (dtype == RT_F32) {
    RT_REQUIRE(!from_idx || n_wg >= 1, RT_EINVAL, "balanced launch needs n_wg >= 1, got %d", n_wg);
    return rt::launch_attention_f32(q, q_rows, q_bias, q_scale, k, vt, out, seq_blocks_dev, seq_tokens_dev, batch,
                                    total_blocks, heads, to_idx, to_pos, plan_heads, from_idx, from_pos, n_wg, stream);
  }
  RT_REQUIRE(!from_idx || n_wg >= 1, RT_EINVAL, "balanced launch needs n_wg >= 1, got %d", n_wg);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto rows = [&](auto tag) {
    typedef decltype(tag) T;
    return launch_rows(Args<T>{(const T*)q, (const T*)k, (const T*)vt, (T*)out, seq_blocks_dev, batch, heads, total_blocks, to_idx,
                               to_pos, plan_heads, from_idx, from_pos, seq_tokens_dev, (const T*)q_rows, (const T*)q_bias, q_scale},
                       n_wg, st);
  };
  return dtype == RT_F16 ? rows(_Float16()) : rows(__bf16());
}

}  // namespace

extern "C" int rt_bs_attention_fwd_masked(const void* q, const void* k, const void* vt, void* out,
                                          const int* seq_blocks_dev, const int* seq_tokens_dev, int batch,
                                          int total_blocks, int heads, const int* to_idx, const int* to_pos,
                                          int plan_heads, const int* from_idx, const int* from_pos, int n_wg,
                                          int dtype, void* stream) {
  RT_REQUIRE(q, RT_EINVAL, "NULL pointer");
  return launch_attention(q, nullptr, nullptr, 1.0f, k, vt, out, seq_blocks_dev, seq_tokens_dev, batch, total_blocks, heads,
                          to_idx, to_pos, plan_heads, from_idx, from_pos, n_wg, dtype, stream);
}

extern "C" int rt_bs_attention_fwd_qrows(const void* qkv, const void* qkv_bias, float q_scale, const void* k,
                                         const void* vt, void* out, const int* seq_blocks_dev,
                                         const int* seq_tokens_dev, int batch, int total_blocks, int heads,
                                         const int* to_idx, const int* to_pos, int plan_heads, const int* from_idx,
                                         const int* from_pos, int n_wg, int dtype, void* stream) {
  RT_REQUIRE(qkv, RT_EINVAL, "NULL pointer");             // qkv_bias may be NULL: the rows carry the bias already
  return launch_attention(nullptr, qkv, qkv_bias, q_scale, k, vt, out, seq_blocks_dev, seq_tokens_dev, batch, total_blocks,
                          heads, to_idx, to_pos, plan_heads, from_idx, from_pos, n_wg, dtype, stream);
}

extern "C" int rt_bs_attention_fwd(const void* q, const void* k, const void* vt, void* out, const int* seq_blocks_dev,
                                   int batch, int total_blocks, int heads, const int* to_idx, const int* to_pos,
                                   int plan_heads, const int* from_idx, const int* from_pos, int n_wg, int dtype,
                                   void* stream) {
  return rt_bs_attention_fwd_masked(q, k, vt, out, seq_blocks_dev, nullptr, batch, total_blocks, heads, to_idx, to_pos,
                                    plan_heads, from_idx, from_pos, n_wg, dtype, stream);
}

extern "C" int rt_bs_attention_cut(int batch, int total_blocks, int heads, int* others, int* global, int* waves) {
  RT_REQUIRE(others && global && waves, RT_EINVAL, "NULL pointer");
  RT_REQUIRE(batch >= 1 && total_blocks >= batch && heads >= 1, RT_EINVAL, "bad geometry: batch=%d total_blocks=%d heads=%d",
             batch, total_blocks, heads);
  const Cut cut = cut_rows(batch, total_blocks, heads);
  *others = cut.others;
  *global = cut.global;
  *waves = cut.waves;
  return RT_OK;
}

static_assert(RT_NO_ALLOC_MAX_BATCH <= MAX_BATCH && RT_NO_ALLOC_MAX_BLOCKS <= MAX_BLOCKS, "header limits exceed the kernel's");
extern "C" int rt_bs_attention_fwd_no_alloc(const void* q, const void* k, const void* vt, void* out,
                                            const int* seq_blocks_dev, const int* seq_tokens_dev, int batch,
                                            int total_blocks, int heads, const int* to_idx, const int* to_pos,
                                            int plan_heads, int dtype, void* stream) {
  RT_REQUIRE(q, RT_EINVAL, "NULL pointer");
  RT_REQUIRE(batch >= 1 && batch <= RT_NO_ALLOC_MAX_BATCH && total_blocks >= batch && total_blocks <= RT_NO_ALLOC_MAX_BLOCKS,
             RT_EINVAL, "rt_bs_attention_fwd_no_alloc takes at most %d sequences and %d blocks (%d tokens), got %d and %d",
             RT_NO_ALLOC_MAX_BATCH, RT_NO_ALLOC_MAX_BLOCKS, RT_NO_ALLOC_MAX_BLOCKS * 64, batch, total_blocks);
  return launch_attention(q, nullptr, nullptr, 1.0f, k, vt, out, seq_blocks_dev, seq_tokens_dev, batch, total_blocks, heads,
                          to_idx, to_pos, plan_heads, nullptr, nullptr, 0, dtype, stream);
}
