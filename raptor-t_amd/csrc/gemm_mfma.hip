// Dense products of the encoder layer on the matrix cores: C[M,N] = A[M,K] . Bt[N,K]^T for fp16 / bf16 with fp32
// accumulation, and what follows each product in its epilogue (bias; bias + tanh GELU; bias + the head split of
// the QKV projection into the packed K / V^T tiles the attention kernel reads).
//
// One persistent workgroup of 8 waves per CU computes tiles of TM x 256 outputs.  Operand tiles of 64 reduction
// steps go straight from memory to LDS (buffer_load ... lds, 16 bytes per lane); a wave owns a quarter of the columns
// (64) and one of the two row halves of the tile, 16x16x32 matrix instructions with fp32 accumulators.  (With random
// operands this part is power limited: a loop of nothing but matrix instructions runs at 1.96 GHz = 1.88 PFLOP/s
// with 16x16x32 in this order and at 1.68 GHz = 1.65 PFLOP/s with 32x32x16.)  The two waves of a SIMD are the two
// row halves of the same columns, so halves of different height (TM = 224: 128 + 96 rows) still load every SIMD alike.
//
//   LDS row of a stage: 64 elements = 128 bytes = 8 chunks of 16; chunk c of row r lies at c ^ ((r >> 1) & 7), which
//   puts the 16 rows a 16-lane group of ds_read_b128 touches on 16 different bank groups.  The loads write LDS
//   linearly, so the permutation is made in the global address: a lane fetches the chunk that belongs to its slot
//   (the eight lanes of a row still cover one whole 128-byte line).
//
//   LDS holds three stages of A and two of B (160 KB for a 256-row tile), so A, which comes from memory, is requested
//   two steps and a half ahead and B, the weights, which the L2 holds, one and a half.
//
//   Step s of the pipeline (64 reduction steps of one tile; the steps of a workgroup's tiles form one sequence) is two
//   halves of 32 reduction steps, each MT rows of four matrix instructions:
//     half 0         behind row i of products the fragment a[i] of half 1 is read (its register has just become free)
//     half 1, rows 0 and 1
//     wait for the own loads of step s+1 and the own reads of step s, barrier: every wave's part of s+1 has landed
//     and nobody reads step s any more
//     half 1, rest   between its products the first fragment reads of step s+1 and the loads of B(s+2) and A(s+3) into
//                    the stages just freed
//   so the matrix pipe has work across the barrier, and the loads of the next tile's first steps are requested before the
//   epilogue of the present one.  A tile's last step leaves its A stage empty: the epilogue turns its
//   outputs into whole rows there, and the load that belongs there follows in the next tile's first step.
//   (The compiler waits for the bias, and so for every load and store before it, at the head of a tile: the first bias is
//   requested outside the tile loop.  A tile therefore begins when the last one's outputs are stored.)
//
// Bound by the boundaries of tiles and by power.  Within a tile a step takes 2 600 cycles where its matrix instructions
// alone take 2 240, at 1.7-1.85 GHz with random operands; over a launch the matrix pipe is busy for 49 % (37184 x 2304 x 768
// with the head split), 54 % (x 3072 x 768), 50 % (the same with GELU), 39 % (x 768 x 768) and 62 % (x 768 x 3072) of the
// cycles at 1.9-2.3 GHz: the shorter the reduction, the more of it is first loads, epilogue and the last round.  Measured
// against hipBLASLt's best of 64 suggestions for the
// shape, in turn on one box (us): 37184 x 2304 x 768 113 against 127, 37184 x 3072 x 768 147 against 165 and with bias +
// GELU 165 against 225, 37184 x 768 x 3072 130 against 132, 37184 x 768 x 768 41 against 44, 40768 x 1024 x 4096 268
// against 340, 40768 x 4096 x 1024 274 against 282; the projection with the head split 141 against 114 + 38.
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "gemm_mfma.h"
#include "lds_load.h"
#include "rt_launch.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The matrix instruction as assembly, so that its accumulators stay where they are: given the choice the compiler
// writes them to other registers and runs out of them.  It cannot see the instruction's hazards then; the two that
// occur here (vector writes of an operand just before, vector reads of a result just after) are covered by the waits
// at both ends of main_loop and at the head of its loop.
template <typename T> struct Mma;
template <> struct Mma<_Float16> {
  typedef f16x8 v8;
  __device__ static void run(v8 a, v8 b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  __device__ static void zero(v8 a, v8 b, f32x4& d) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b)); }
  __device__ static void first(v8 a, v8 b, f32x4& d, f32x4 c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "v"(b), "v"(c)); }
  __device__ static uint32_t two(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2)); }
  __device__ static float lo(uint32_t w) { return float(__builtin_bit_cast(f16x2, w).x); }
  __device__ static float hi(uint32_t w) { return float(__builtin_bit_cast(f16x2, w).y); }
};
template <> struct Mma<__bf16> {
  typedef bf16x8 v8;
  __device__ static void run(v8 a, v8 b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  __device__ static void zero(v8 a, v8 b, f32x4& d) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b)); }
  __device__ static void first(v8 a, v8 b, f32x4& d, f32x4 c) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "v"(b), "v"(c)); }
  __device__ static uint32_t two(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2)); }
  __device__ static float lo(uint32_t w) { return __uint_as_float(w << 16); }
  __device__ static float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};

constexpr int TN = 256;                       // columns of a tile
constexpr int BK = 64;                        // reduction steps of a stage
constexpr int ROW = BK * 2;                   // bytes of an LDS row
constexpr int EPI_BYTES = 32 * 64 * 2;        // a wave's room for turning a 32 x 64 block of outputs into whole rows
constexpr int WAVES = 8;
constexpr int NON_TEMPORAL = 2;               // cache policy of a store
constexpr int B_STAGE = TN * ROW;

// An A stage also has to hold the epilogue's blocks of all waves.
template <int TM> constexpr int a_stage() { return TM * ROW > WAVES * EPI_BYTES ? TM * ROW : WAVES * EPI_BYTES; }
template <int TM> constexpr int lds_bytes() { return 3 * a_stage<TM>() + 2 * B_STAGE; }

#define SB() __builtin_amdgcn_sched_barrier(0)

// v_permlane32_swap: the upper 32 lanes of a change places with the lower 32 of b; v_permlane16_swap: lanes 16-31 and
// 48-63 of a with lanes 0-15 and 32-47 of b.
__device__ inline void permlane32_swap(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ inline void permlane16_swap(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// The value, worked out where it stands: what the compiler derives from the lane number alone it would otherwise keep
// in registers across the whole tile loop, which has none to spare.
__device__ __forceinline__ int again(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

struct Params {
  const void* a;          // [M, K]
  const void* bt;         // [N, K]
  const void* bias;       // [N] or NULL
  void* c;                // [M, N]
  int m, n, k;
  int tiles_m, tiles_n;
  int slices;             // parts the reduction is cut into (EPI_PART)
  // QKV split: N = 3 * heads * 64
  void* kt;
  void* vt;
  const int* seq_blocks;
  int batch, heads;
};

// Tiles in groups of 4 row panels, the panel fastest: the 32 tiles an XCD works on at a time share 4 panels of A and
// 8 of B instead of (columns fastest) 1 to 3 and up to 32.
__device__ __forceinline__ void tile_at(const Params& p, int tile, int& tm, int& tn) {
  constexpr int G = 4;
  const int per = G * p.tiles_n, grp = tile / per, in = tile - grp * per, h = min(G, p.tiles_m - grp * G);
  tn = in / h;
  tm = grp * G + (in - tn * h);
}

// Where the loads of one operand stand in the sequence of steps: tile, step inside it and the lanes' row offsets.
template <int ROWS, bool IS_A> struct Loader {
  static constexpr int GROUPS = ROWS / 8;     // groups of 8 rows, one load instruction each
  int v[4];
  int tile, last, stride, step, steps;
  __device__ __forceinline__ void rows(const Params& p, int w, int lane) {
    int tm, tn;
    tile_at(p, tile, tm, tn);
    const int r = w * 8 + (lane >> 3);
    const int chunk = ((lane & 7) ^ ((r >> 1) & 7)) * 16;     // rows j * 64 + r share it
    const int first = (IS_A ? tm : tn) * ROWS, end = (IS_A ? p.m : p.n) - 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = min(first + j * 64 + r, end) * p.k * 2 + chunk;
  }
  // Behind the workgroup's last tile the loads run on into that tile's first steps again: nobody uses them, and the
  // loop needs no test for the end.
  __device__ __forceinline__ void advance(const Params& p, int w, int lane) {
    if (++step == steps) {
      step = 0;
      if (tile + stride < last) {
        tile += stride;
        rows(p, w, lane);
      }
    }
  }
  // load J of 4: rows J * 64 + w * 8 .. + 8 of the tile
  template <int J> __device__ __forceinline__ void issue(i32x4 srd, uint32_t stage, int w) const {
    if (J * 8 + 8 <= GROUPS || J * 8 + w < GROUPS) load_to_lds(srd, v[J], step * ROW, stage + (J * 8 + w) * 1024);
  }
  __device__ __forceinline__ void issue_all(i32x4 srd, uint32_t stage, int w) const {
    issue<0>(srd, stage, w);
    issue<1>(srd, stage, w);
    issue<2>(srd, stage, w);
    issue<3>(srd, stage, w);
  }
};

// The stages that the present step reads (byte offsets in LDS); A's lie first.
template <int TM> struct Stages {
  static constexpr uint32_t B0 = 3 * a_stage<TM>();
  uint32_t a = 0, b = B0;
  __device__ __forceinline__ uint32_t next_a() const { return a == 2u * a_stage<TM>() ? 0u : a + a_stage<TM>(); }
  __device__ __forceinline__ uint32_t next_b() const { return b == B0 ? B0 + B_STAGE : B0; }
};

enum { EPI_NONE = 0, EPI_GELU = 1, EPI_QKV = 2, EPI_PART = 3 };

// ---- epilogues of a wave's MT x 4 blocks of 16 x 16 outputs, rows from m0, columns from n0 --------------------------
// Rows of C: 16 x 64 outputs at a time through the wave's LDS room (4 KB at `room`), stored as eight whole 128-byte rows
// per instruction.  A block's rows are read back while the next one is written, and the stores pass no test:
// offsets past the end of C are dropped by the range check.
template <typename T, int MT, int EPI, int POLICY>
__device__ __forceinline__ void store_rows(const f32x4 (&acc)[MT][4], __amdgpu_buffer_rsrc_t sc, int n, int m0, int n0, char* room) {
  const int lane = again(threadIdx.x & 63), l16 = lane & 15, g4 = lane >> 4;
  const bool col_ok = n0 + (lane & 7) * 8 < n;
  uint32_t voff = col_ok ? (uint32_t(m0 + (lane >> 3)) * uint32_t(n) + uint32_t(n0 + (lane & 7) * 8)) * 2u : 0xfffffff0u;
  const uint32_t ld8 = col_ok ? uint32_t(n) * 16u : 0u;         // eight rows
  const int wr = l16 * 128 + 8 * (g4 & 1), wx = l16 >> 1, rr = (lane >> 3) * 128;
#pragma unroll
  for (int i = 0; i <= MT; ++i) {
    u32x4 o[2];
    if (i > 0) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        o[j] = *reinterpret_cast<const u32x4*>(room + ((i - 1) & 1) * 2048 + j * 1024 + rr + (((lane & 7) ^ (((lane >> 4) + 4 * j) & 7)) << 4));
    }
    if (i < MT) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 v = acc[i][j];
        if (EPI == EPI_GELU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
        }
        *reinterpret_cast<u32x2*>(room + (i & 1) * 2048 + wr + (((2 * j + (g4 >> 1)) ^ wx) << 4)) =
            u32x2{Mma<T>::two(v[0], v[1]), Mma<T>::two(v[2], v[3])};
      }
    }
    if (i > 0) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        __builtin_amdgcn_raw_buffer_store_b128(o[j], sc, int(voff), 0, POLICY);
        voff += ld8;
      }
    }
    SB();
  }
}

// K and V^T tiles: the byte at which the tile of token `row` begins (lane's part), for head h; past the tensors' end where
// there is no such row or head, so the stores' range check drops what is written there.  seq_end: lane l holds the end of
// sequence l (batches of up to 64 sequences).
__device__ __forceinline__ uint32_t tile_offset(const Params& p, int seq_end, int row, int h) {
  if (row >= p.m || h >= p.heads) return 0xfffc0000u;
  const int g = row >> 6, lane = again(threadIdx.x & 63);
  int s, g0, end;                                          // the sequence block g belongs to
  if (p.batch <= 64) {
    s = __popcll(__ballot(lane < p.batch && seq_end <= g));
    g0 = s == 0 ? 0 : __builtin_amdgcn_readlane(seq_end, s - 1);
    end = __builtin_amdgcn_readlane(seq_end, s);
  } else {
    s = 0;
    for (int b0 = 0; b0 < p.batch; b0 += 64)
      s += __popcll(__ballot(b0 + lane < p.batch && p.seq_blocks[min(b0 + lane + 1, p.batch)] <= g));
    g0 = p.seq_blocks[s];
    end = p.seq_blocks[s + 1];
  }
  return uint32_t(g0 * p.heads + h * (end - g0) + (g - g0)) * 8192u + uint32_t(lane) * 16u;
}

// V^T tiles of head h from its column d0 (a multiple of 32) on (products taken with the tokens as rows): a lane's accumulators are 4 consecutive tokens of one
// column; fragment 4 * (d >> 5) + (token >> 4) wants, in lane (d & 31) + 32 * x, the tokens 4 x .. + 4 and 8 + 4 x .. + 4
// of its 16.
template <typename T, int MT, int NT>
__device__ __forceinline__ void store_v(const f32x4 (&acc)[MT][NT], const Params& p, int seq_end, int m0, int h, int d0 = 0) {
  const __amdgpu_buffer_rsrc_t sv = __builtin_amdgcn_make_buffer_rsrc(p.vt, 0, uint32_t(p.m) * uint32_t(p.heads) * 128u, 0x00020000);
#pragma unroll
  for (int i = 0; i < MT; i += 2) {
    const int row = m0 + 16 * i;
    const uint32_t t = tile_offset(p, seq_end, row, h) + uint32_t(((row >> 5) & 1) * 2048 + d0 * 128);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int j = 0; j < NT; j += 2) {
        const f32x4 &c = acc[i + q][j], &d = acc[i + q][j + 1];
        uint32_t x0 = Mma<T>::two(c[0], c[1]), x1 = Mma<T>::two(c[2], c[3]);
        uint32_t y0 = Mma<T>::two(d[0], d[1]), y1 = Mma<T>::two(d[2], d[3]);
        permlane16_swap(x0, y0);
        permlane16_swap(x1, y1);
        permlane32_swap(x0, y0);
        permlane32_swap(x1, y1);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{x0, x1, y0, y1}, sv, int(t + (2 * j + q) * 1024), 0, rt::WRITE_THROUGH);
      }
  }
}

// K tiles of head h from its column d0 (a multiple of 16) on (products taken with the columns as rows): a lane's accumulators are 4 consecutive columns of one
// token; fragment 4 * (token >> 5) + (d >> 4) wants, in lane (token & 31) + 32 * x, the columns 8 x .. + 8 of its 16.
template <typename T, int MT, int NT>
__device__ __forceinline__ void store_k(const f32x4 (&acc)[MT][NT], const Params& p, int seq_end, int m0, int h, int d0 = 0) {
  const __amdgpu_buffer_rsrc_t sk = __builtin_amdgcn_make_buffer_rsrc(p.kt, 0, uint32_t(p.m) * uint32_t(p.heads) * 128u, 0x00020000);
#pragma unroll
  for (int i = 0; i < MT; i += 2) {
    const int row = m0 + 16 * i;
    const uint32_t t = tile_offset(p, seq_end, row, h) + uint32_t(((row >> 5) & 1) * 4096 + d0 * 64);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const f32x4 &c = acc[i][j], &d = acc[i + 1][j];
      uint32_t x0 = Mma<T>::two(c[0], c[1]), x1 = Mma<T>::two(c[2], c[3]);
      uint32_t y0 = Mma<T>::two(d[0], d[1]), y1 = Mma<T>::two(d[2], d[3]);
      permlane16_swap(x0, y0);
      permlane16_swap(x1, y1);
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{x0, x1, y0, y1}, sk, int(t + j * 1024), 0, rt::WRITE_THROUGH);
    }
  }
}

// What the epilogue needs from memory, requested a step ahead: the bias of a wave's columns (of column block j the 4
// consecutive ones of a lane's accumulators, or (V) the one) for the tile after it, and where the batch's first 64
// sequences end.
struct Bias {
  u32x2 w[4];
  int seq_end;
};

// The steps of one tile: MT row blocks of 16 and four column blocks of 16 per wave.  Its first step
// lies in LDS on entry, and the following tile's on return.  The accumulators
// start from c0 (the bias of their columns): the first products take it as their C operand.  `load_bias` requests the
// next tile's bias at the head of the last step; it has arrived when main_loop returns.
template <typename T, int TM, int MT, int EPI, bool V_TILE, typename F>
__device__ __forceinline__ void main_loop(f32x4 (&acc)[MT][4], const f32x4 (&c0)[4], Bias& bias, F&& load_bias,
                                          Loader<TM, true>& lda, Loader<TN, false>& ldb, Stages<TM>& st, const Params& p,
                                          i32x4 sa, i32x4 sb, char* smem, uint32_t lds0, int w, int lane,
                                          const int (&offa)[2], const int (&offb)[2]) {
  typedef typename Mma<T>::v8 v8;
  v8 a[MT], b[2][4];
  // What may still be on its way at a step's barrier: the loads of A(s+2), which every wave has issued behind those of
  // s+1, or in a tile's first step, behind its loads of B(s+1), the stores of the last tile's outputs.  store_rows issues
  // 2 * MT of them whatever it stores (past the ends of C the range check drops them), and so do store_v and store_k; but behind
  // a V tile a wave whose columns lie past the end issues none, so with the head split nothing may be left: B(s+1) could be what is.
  constexpr int LEFT = TM / 64, STORES = EPI == EPI_QKV ? 0 : 2 * MT;
  enum { FIRST, INNER, LAST };
  // row i of a half: its four products, the columns in alternating direction (a row's last weights fragment is the
  // next row's first: fewer operand bits toggle)
  auto products = [&](int i, const v8 (&bb)[4], auto with_c0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = i & 1 ? 3 - j : j;
      if (decltype(with_c0)::value) {
        if (V_TILE) Mma<T>::first(a[i], bb[c], acc[i][c], c0[c]);
        else Mma<T>::first(bb[c], a[i], acc[i][c], c0[c]);
      } else {
        if (V_TILE) Mma<T>::run(a[i], bb[c], acc[i][c]);
        else Mma<T>::run(bb[c], a[i], acc[i][c]);
      }
    }
  };
  const std::false_type no;
  auto step = [&](auto which) __attribute__((always_inline)) {
    constexpr int W = decltype(which)::value;
    asm volatile("s_nop 1");
    const uint32_t na = st.next_a(), nb = st.next_b();
    {
      const char* la = smem + st.a + offa[1];
      const char* lb = smem + st.b + offb[1];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        products(i, b[0], std::integral_constant<bool, W == FIRST>());
        a[i] = *reinterpret_cast<const v8*>(la + i * 16 * ROW);
        if (i < 4) b[1][i] = *reinterpret_cast<const v8*>(lb + i * 16 * ROW);
        if (W == LAST && i == 0) load_bias();
        SB();
      }
    }
    products(0, b[1], no);
    SB();
    products(1, b[1], no);
    SB();
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(W == LAST ? 0 : W == FIRST ? STORES : LEFT) : "memory");
    // The compiler's own wait for these comes here, where everything has arrived already.  (With the head split it has
    // waited before: load_bias' two ways to load share registers, so each load waits for the one before it.)
    if (W == LAST) {
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(bias.w[j]));
      if (EPI == EPI_QKV) asm volatile("" : "+v"(bias.seq_end));
    }
    __builtin_amdgcn_s_barrier();
    SB();
    {
      const char* la = smem + na + offa[0];
      const char* lb = smem + nb + offb[0];
      if (W != LAST) {
        a[0] = *reinterpret_cast<const v8*>(la);
        b[0][0] = *reinterpret_cast<const v8*>(lb);
      }
#pragma unroll
      for (int i = 2; i < MT; ++i) {
        products(i, b[1], no);
        if (W != LAST) {
          if (i < 5) b[0][i - 1] = *reinterpret_cast<const v8*>(lb + (i - 1) * 16 * ROW);
          if (i == 2) a[1] = *reinterpret_cast<const v8*>(la + 16 * ROW);
          a[i] = *reinterpret_cast<const v8*>(la + i * 16 * ROW);
        }
        if (i == 2) ldb.template issue<0>(sb, lds0 + st.b, w);
        if (i == 3) ldb.template issue<1>(sb, lds0 + st.b, w);
        if (i == 4) ldb.template issue<2>(sb, lds0 + st.b, w);
        if (i == 5) ldb.template issue<3>(sb, lds0 + st.b, w);
        SB();
      }
    }
    ldb.advance(p, w, lane);
    if (W == FIRST) {                                // the load that the last tile's epilogue was in the way of
      lda.issue_all(sa, lds0 + (na == 2u * a_stage<TM>() ? 0u : na + a_stage<TM>()), w);
      lda.advance(p, w, lane);
    }
    if (W != LAST) {
      lda.issue_all(sa, lds0 + st.a, w);
      lda.advance(p, w, lane);
    }
    st.a = na;
    st.b = nb;
    SB();
  };
  {
    const char* la = smem + st.a + offa[0];
    const char* lb = smem + st.b + offb[0];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[0][j] = *reinterpret_cast<const v8*>(lb + j * 16 * ROW);
#pragma unroll
    for (int i = 0; i < MT; ++i) a[i] = *reinterpret_cast<const v8*>(la + i * 16 * ROW);
  }
  step(std::integral_constant<int, FIRST>());
  const int inner = lda.steps - 2;
#pragma clang loop unroll(disable)
  for (int s = 0; s < inner; ++s) step(std::integral_constant<int, INNER>());
  step(std::integral_constant<int, LAST>());
  asm volatile("s_nop 15\n\ts_nop 7");
  SB();
}

template <typename T, int TM, int MT0, int MT1, int EPI>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_bt_kernel(Params p) {
  extern __shared__ __align__(16) char smem[];
  static_assert(TM == 16 * (MT0 + MT1) && MT0 % 2 == 0 && MT1 % 2 == 0, "two halves");
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)smem));
  const __amdgpu_buffer_rsrc_t sc = __builtin_amdgcn_make_buffer_rsrc(p.c, 0, uint32_t(p.m) * uint32_t(p.n) * 2u, 0x00020000);
  const i32x4 sa = make_srd(p.a, uint32_t(p.m) * uint32_t(p.k) * 2u), sb = make_srd(p.bt, uint32_t(p.n) * uint32_t(p.k) * 2u);
  // Workgroups go to the 8 XCDs round-robin: XCD x takes the x-th eighth of the tiles (in tile_at's order), its
  // workgroups take neighbouring tiles, so the rows of A are fetched into one L2.
  const int total = p.tiles_m * p.tiles_n, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  int tile = int(int64_t(total) * xcd / 8) + slot;
  const int last = int(int64_t(total) * (xcd + 1) / 8);
  if (tile >= last) return;
  Loader<TM, true> lda;
  Loader<TN, false> ldb;
  lda.tile = ldb.tile = tile;
  lda.last = ldb.last = last;
  lda.stride = ldb.stride = slots;
  lda.step = ldb.step = 0;
  lda.steps = ldb.steps = p.k / BK;
  lda.rows(p, w, lane);
  ldb.rows(p, w, lane);
  Stages<TM> st;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    ldb.issue_all(sb, lds0 + Stages<TM>::B0 + q * B_STAGE, w);
    ldb.advance(p, w, lane);
    lda.issue_all(sa, lds0 + q * a_stage<TM>(), w);
    lda.advance(p, w, lane);
  }
  auto run = [&](auto mt_tag) {
    constexpr int MT = decltype(mt_tag)::value;
    const int a_row = w < 4 ? 0 : 16 * MT0;
    const int l16 = lane & 15, g4 = lane >> 4;         // a fragment's lane: row l16, reduction steps 8 * g4 .. + 8
    int offa[2], offb[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = ((4 * kk + g4) ^ (l16 >> 1)) << 4;
      offa[kk] = (a_row + l16) * ROW + c;
      offb[kk] = ((w & 3) * 64 + l16) * ROW + c;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    SB();
    Bias bias;
    auto load_bias = [&](int t) __attribute__((always_inline)) {
      const int lane = again(threadIdx.x & 63), l16 = lane & 15, g4 = lane >> 4;
      int tm, tn;
      tile_at(p, t, tm, tn);
      const int n0 = tn * TN + (w & 3) * 64;
      const bool v_tile = EPI == EPI_QKV && n0 >= 2 * p.heads * 64;
      const T* bp = static_cast<const T*>(p.bias);
      if (EPI == EPI_QKV) bias.seq_end = p.seq_blocks[min(lane + 1, p.batch)];
#pragma unroll
      for (int j = 0; j < 4; ++j) bias.w[j] = u32x2{0, 0};
      if (p.bias) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // columns past the end repeat the last ones: their products are not stored
          if (v_tile) bias.w[j].x = reinterpret_cast<const uint16_t*>(bp)[min(n0 + 16 * j + l16, p.n - 1)];
          else bias.w[j] = *reinterpret_cast<const u32x2*>(bp + min(n0 + 16 * j + 4 * g4, p.n - 4));
        }
      }
    };
    load_bias(tile);
    for (; tile < last; tile += slots) {
      int tm, tn;
      tile_at(p, tile, tm, tn);
      const int m0 = tm * TM + a_row, n0 = tn * TN + (w & 3) * 64;
      const int dm = p.heads * 64;
      const bool v_tile = EPI == EPI_QKV && n0 >= 2 * dm;
      f32x4 c0[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x2 x = bias.w[j];
        c0[j] = f32x4{Mma<T>::lo(x.x), Mma<T>::hi(x.x), Mma<T>::lo(x.y), Mma<T>::hi(x.y)};
        if (v_tile) c0[j] = f32x4(Mma<T>::lo(x.x));
      }
      const int following = tile + slots < last ? tile + slots : tile;
      auto next_bias = [&]() __attribute__((always_inline)) { load_bias(following); };
      f32x4 acc[MT][4];
      // (The assembly comments keep the compiler from merging equal code of the branches, which costs it registers.)
      if (EPI == EPI_QKV && v_tile) {
        asm volatile("; V tile");
        main_loop<T, TM, MT, EPI, true>(acc, c0, bias, next_bias, lda, ldb, st, p, sa, sb, smem, lds0, w, lane, offa, offb);
        if (n0 < p.n) store_v<T>(acc, p, bias.seq_end, m0, (n0 - 2 * dm) >> 6);
        asm volatile("; V tile done");
        continue;
      }
      main_loop<T, TM, MT, EPI, false>(acc, c0, bias, next_bias, lda, ldb, st, p, sa, sb, smem, lds0, w, lane, offa, offb);
      if (EPI == EPI_QKV && n0 >= dm) {
        store_k<T>(acc, p, bias.seq_end, m0, (n0 - dm) >> 6);
        asm volatile("; K tile done");
        continue;
      }
      // through the A stage of the tile's last step (st has moved on by one)
      store_rows<T, MT, EPI, NON_TEMPORAL>(acc, sc, p.n, m0, n0,
                                           smem + (st.a == 0 ? 2u * a_stage<TM>() : st.a - a_stage<TM>()) + w * EPI_BYTES);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the trailing loads write LDS of this workgroup
  };
  if (MT0 == MT1 || w < 4) run(std::integral_constant<int, MT0>());
  else run(std::integral_constant<int, MT1>());
}

// ---- smaller products ------------------------------------------------------------------------------------------------
// One workgroup per tile of TM x TC outputs and per slice of the reduction, WM x WN waves of MT x NT blocks of 16 x 16.
// Where the kernel above would give too few CUs a tile each, what bounds a product is the latency of a workgroup's chain
// of steps, and a wave issues in order: a memory instruction that has to wait for its unit holds up the matrix
// instructions behind it.  So every step is laid out by hand, one product, then at most two fragment reads and a load:
//   DEEP (small tiles)   both halves' fragments of step s+1 are read, into a second set of registers, between the products
//                        of step s: one barrier per step, no LDS latency in the chain
//   otherwise            fragments of half 1 are read between the products of half 0 (a row's in place, when its last product
//                        has been issued), and those of the next step's half 0 behind the barrier in half 1
// Between a step's barrier and the next the loads of the step STAGES ahead go to the stage that the barrier has freed.
// The bias and the ends of the batch's sequences come to LDS ahead of the first stage, so the epilogue waits for no memory.
// Slices (EPI_PART): the fp32 sums of slice s go to c[s][M][N] and the kernel that reads them, the layer's LayerNorm, adds
// them.
// Measured (us, one launch among others, fp16; before: the fragments of a half read in one burst, the loads in another, bias
// and sequence ends loaded behind the loop): 512 x 2304 x 768 7.6 -> 5.1, 512 x 768 x 3072 15.1 -> 9.4, 2048 x 768 x 768
// 7.9 -> 5.7, 4096 x 768 x 3072 25.4 -> 21.5, 5568 x 768 x 3072 33.9 -> 27.5, 8192 x 768 x 3072 42.6 -> 35.9.  Counters over
// two lengths of the reduction: a 64 x 64 step takes 365 cycles (its SIMD's matrix instructions 128), a 128 x 128 one 663 (512), a
// 192 x 192 one 1414 (1152).
template <typename T> struct Product;        // the instruction as a builtin: these accumulators leave registers to spare
template <> struct Product<_Float16> {
  __device__ static f32x4 run(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct Product<__bf16> {
  __device__ static f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

// 64 lanes x 4 bytes from srd[voff] to LDS bytes [lds, lds + 256), as load_to_lds
__device__ inline void load_words_to_lds(i32x4 srd, int voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" :: "v"(voff), "s"(srd), "s"(lds) : "memory");
}

// Rows of C (EPI_PART: of a slice, in fp32) as store_rows writes them, for any even NT: rows of the room lie 16 bytes further
// apart than they are long, which puts the 16 rows of a write on different banks.
template <int NT, int EPI> constexpr int block_pitch() { return NT * (EPI == EPI_PART ? 64 : 32) + 16; }
template <typename T, int MT, int NT, int EPI>
__device__ __forceinline__ void store_block(const f32x4 (&acc)[MT][NT], __amdgpu_buffer_rsrc_t sc, int n, int m0, int n0, char* room) {
  static_assert(NT % 2 == 0, "whole stores");
  constexpr int SIZE = EPI == EPI_PART ? 4 : 2, PER = 16 / SIZE;
  constexpr int CH = NT * SIZE, PITCH = block_pitch<NT, EPI>(), ST = CH / 4;      // 16-byte chunks of a row, stores per 16 rows
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  uint32_t voff[ST], rows16[ST];
  int rd[ST];
#pragma unroll
  for (int k = 0; k < ST; ++k) {
    const int c = k * 64 + lane, row = c / CH, ch = c - row * CH;
    const bool ok = n0 + ch * PER < n;
    voff[k] = ok ? (uint32_t(m0 + row) * uint32_t(n) + uint32_t(n0 + ch * PER)) * uint32_t(SIZE) : 0xfffffff0u;
    rows16[k] = ok ? uint32_t(n) * uint32_t(16 * SIZE) : 0u;
    rd[k] = row * PITCH + ch * 16;
  }
  const int wr = l16 * PITCH + g4 * 4 * SIZE;
#pragma unroll
  for (int i = 0; i <= MT; ++i) {
    u32x4 o[ST];
    if (i > 0) {
#pragma unroll
      for (int k = 0; k < ST; ++k) o[k] = *reinterpret_cast<const u32x4*>(room + ((i - 1) & 1) * 16 * PITCH + rd[k]);
    }
    if (i < MT) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        f32x4 v = acc[i][j];
        char* const to = room + (i & 1) * 16 * PITCH + wr + j * 16 * SIZE;
        if constexpr (EPI == EPI_PART) {
          *reinterpret_cast<f32x4*>(to) = v;
        } else {
          if (EPI == EPI_GELU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
          }
          *reinterpret_cast<u32x2*>(to) = u32x2{Mma<T>::two(v[0], v[1]), Mma<T>::two(v[2], v[3])};
        }
      }
    }
    if (i > 0) {
#pragma unroll
      for (int k = 0; k < ST; ++k) {
        __builtin_amdgcn_raw_buffer_store_b128(o[k], sc, int(voff[k]), 0, rt::WRITE_THROUGH);
        voff[k] += rows16[k];
      }
    }
    SB();
  }
}

constexpr int SMALL_EXTRA = 1024 + 256;       // LDS behind the stages: the tile's bias, the ends of the first 64 sequences

template <typename T, int MT, int NT, int WM, int WN, int STAGES, int EPI>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_bt_small_kernel(Params p) {
  typedef typename Mma<T>::v8 v8;
  extern __shared__ __align__(16) char smem[];
  constexpr int NW = WM * WN, TM = 16 * MT * WM, TC = 16 * NT * WN;
  constexpr int NA = TM / 8 / NW, NB = TC / 8 / NW, LOADS = NA + NB;      // load instructions of a wave and step
  constexpr uint32_t STAGE = (TM + TC) * ROW, BIAS = STAGES * STAGE, ENDS = BIAS + 1024;
  constexpr bool DEEP = MT * NT <= 8;
  static_assert(TM % (8 * NW) == 0 && TC % (8 * NW) == 0 && STAGES >= 2 && STAGES <= 4, "tile");
  static_assert(NW * 32 * block_pitch<NT, EPI>() <= BIAS && TC * 2 <= 1024, "room");
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  // XCD x takes the x-th eighth of the list: slice, groups of 8 row panels, column, panel
  const int tiles = p.tiles_m * p.tiles_n, total = tiles * p.slices, per = gridDim.x >> 3;
  const int id = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
  if (id >= total) return;
  const int slice = EPI == EPI_PART ? id / tiles : 0, tile = id - slice * tiles;
  constexpr int G = 8;
  const int grp = tile / (G * p.tiles_n), in = tile - grp * G * p.tiles_n, h = min(G, p.tiles_m - grp * G);
  const int tn = in / h, tm = grp * G + (in - tn * h);
  const int all = p.k / BK, first = EPI == EPI_PART ? all * slice / p.slices : 0;
  const int steps = (EPI == EPI_PART ? all * (slice + 1) / p.slices : all) - first;       // at least 2

  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)smem));
  const i32x4 sa = make_srd(p.a, uint32_t(p.m) * uint32_t(p.k) * 2u), sb = make_srd(p.bt, uint32_t(p.n) * uint32_t(p.k) * 2u);
  if (EPI != EPI_PART && w == 0) {             // past the end of the bias, and where there is none, the range check gives zeros
    load_to_lds(make_srd(p.bias, p.bias ? uint32_t(p.n) * 2u : 0u), tn * TC * 2 + lane * 16, 0, lds0 + BIAS);
    if (EPI == EPI_QKV) load_words_to_lds(make_srd(p.seq_blocks, uint32_t(p.batch + 1) * 4u), min(lane + 1, p.batch) * 4, lds0 + ENDS);
  }
  int va[NA], vb[NB];
  {
    const int r = w * 8 + (lane >> 3), chunk = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
#pragma unroll
    for (int j = 0; j < NA; ++j) va[j] = min(tm * TM + j * 8 * NW + r, p.m - 1) * p.k * 2 + chunk;
#pragma unroll
    for (int j = 0; j < NB; ++j) vb[j] = min(tn * TC + j * 8 * NW + r, p.n - 1) * p.k * 2 + chunk;
  }
  // loads [from, to) of a step: B's rows first
  auto issue = [&](int s, uint32_t stage, int from, int to) __attribute__((always_inline)) {
    const int soff = (first + s) * ROW;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      if (j < from || j >= to) continue;
      if (j < NB) load_to_lds(sb, vb[j % NB], soff, lds0 + stage + TM * ROW + (j * NW + w) * 1024);
      else load_to_lds(sa, va[(j - NB) % NA], soff, lds0 + stage + ((j - NB) * NW + w) * 1024);
    }
  };
#pragma unroll
  for (int q = 0; q < STAGES; ++q)
    if (q < steps) issue(q, q * STAGE, 0, LOADS);

  const int wm = w / WN, wn = w % WN;
  const int m0 = tm * TM + wm * 16 * MT, n0 = tn * TC + wn * 16 * NT, dm = p.heads * 64;
  const bool v_tile = EPI == EPI_QKV && n0 >= 2 * dm;
  int offa[2], offb[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int c = ((4 * kk + g4) ^ (l16 >> 1)) << 4;
    offa[kk] = (wm * 16 * MT + l16) * ROW + c;
    offb[kk] = (TM + wn * 16 * NT + l16) * ROW + c;
  }
  // all loads but those of the last `left` steps have landed, and the own reads
  auto wait = [&](int left) __attribute__((always_inline)) {
    if (STAGES > 3 && left == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(3 * LOADS) : "memory");
    else if (STAGES > 2 && left == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(2 * LOADS) : "memory");
    else if (left == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  };
  constexpr int SETS = DEEP ? 2 : 1, HALVES = DEEP ? 2 : 1;
  v8 a[SETS][HALVES][MT], b[SETS][2][NT];         // DEEP: [parity of the step][half]; else the row fragments in place
  f32x4 acc[MT][NT], c0[NT];
  auto loop = [&](auto v_tag) __attribute__((always_inline)) {
    constexpr bool V_TILE = decltype(v_tag)::value;
    uint32_t cur = 0;
    // product t of a half, the columns in alternating direction (fewer operand bits toggle); the first half's start from c0
    auto product = [&](int set, int kk, int t, auto init) __attribute__((always_inline)) {
      const int i = t / NT, j = t % NT, c = i & 1 ? NT - 1 - j : j;
      const v8 &fa = a[set][DEEP ? kk : 0][i], &fb = b[set][kk][c];
      acc[i][c] = Product<T>::run(V_TILE ? fa : fb, V_TILE ? fb : fa, decltype(init)::value && kk == 0 ? c0[c] : acc[i][c]);
      SB();
    };
    auto read_a = [&](int set, int kk, int i, uint32_t stage) __attribute__((always_inline)) {
      a[set][DEEP ? kk : 0][i] = *reinterpret_cast<const v8*>(smem + stage + offa[kk] + i * 16 * ROW);
      SB();
    };
    auto read_b = [&](int set, int kk, int j, uint32_t stage) __attribute__((always_inline)) {
      b[set][kk][j] = *reinterpret_cast<const v8*>(smem + stage + offb[kk] + j * 16 * ROW);
      SB();
    };
    // MORE: the step STAGES ahead exists; else it is looked at.  LAST: nothing follows
    auto deep_step = [&](int s, auto set_tag, auto init, auto more_tag, auto last_tag) __attribute__((always_inline)) {
      constexpr int SET = decltype(set_tag)::value, PROD = MT * NT, READS = 2 * (MT + NT);
      constexpr bool MORE = decltype(more_tag)::value, LAST = decltype(last_tag)::value;
      constexpr int AHEAD = 2 * PROD >= 16 ? 4 : 0, REST = 2 * PROD - AHEAD;      // products ahead of the barrier, behind it
      constexpr int EACH = READS > REST || PROD <= 4 ? 2 : 1;                     // reads behind a product
      const uint32_t nxt = cur == (STAGES - 1) * STAGE ? 0u : cur + STAGE;
#pragma unroll
      for (int t = 0; t < AHEAD; ++t) product(SET, 0, t, init);
      if (LAST) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                // the epilogue's room lies in the stages
      else if (MORE) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((STAGES - 2) * LOADS) : "memory");
      else wait(min(STAGES - 2, steps - 2 - s));
      __builtin_amdgcn_s_barrier();
      SB();
      const bool more = MORE || (!LAST && s + STAGES < steps);
#pragma unroll
      for (int t = AHEAD; t < 2 * PROD; ++t) {
        product(SET, t / PROD, t % PROD, init);
        if (LAST) continue;
        const int u = t - AHEAD;
#pragma unroll
        for (int r = u * EACH; r < min(READS, (u + 1) * EACH); ++r) {
          const int kk = r / (MT + NT), q = r % (MT + NT);
          if (q < NT) read_b(SET ^ 1, kk, q, nxt);
          else read_a(SET ^ 1, kk, q - NT, nxt);
        }
        const int from = (u * LOADS + REST - 1) / REST, to = ((u + 1) * LOADS + REST - 1) / REST;
        if (from < to && more) issue(s + STAGES, cur, from, to);
        SB();
      }
      cur = nxt;
    };
    auto step = [&](int s, auto init, auto more_tag, auto last_tag) __attribute__((always_inline)) {
      constexpr bool MORE = decltype(more_tag)::value, LAST = decltype(last_tag)::value;
      constexpr int AHEAD = MT >= 4 ? 1 : 0, REST = (MT - AHEAD) * NT, EVERY = REST >= 2 * NT ? 2 : 1;     // rows, products, reads of b
      const uint32_t nxt = cur == (STAGES - 1) * STAGE ? 0u : cur + STAGE;
#pragma unroll
      for (int t = 0; t < MT * NT; ++t) {
        product(0, 0, t, init);
        if (t % 2 == 0 && t / 2 < NT) read_b(0, 1, t / 2, cur);
        if (t % NT == NT - 1) read_a(0, 1, t / NT, cur);
      }
#pragma unroll
      for (int t = 0; t < AHEAD * NT; ++t) product(0, 1, t, std::false_type());
      if (MORE) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((STAGES - 2) * LOADS) : "memory");
      else wait(LAST ? 0 : min(STAGES - 2, steps - 2 - s));
      __builtin_amdgcn_s_barrier();
      SB();
      const bool more = MORE || (!LAST && s + STAGES < steps);
#pragma unroll
      for (int t = 0; t < REST; ++t) {
        const int i = AHEAD + t / NT;
        product(0, 1, AHEAD * NT + t, std::false_type());
        if (LAST) continue;
        if (t % EVERY == 0 && t / EVERY < NT) read_b(0, 0, t / EVERY, nxt);
        if (t % NT == 0 && t / NT < AHEAD) read_a(0, 0, t / NT, nxt);
        if (t % NT == NT - 1) read_a(0, 0, i, nxt);
        const int from = (t * LOADS + REST - 1) / REST, to = ((t + 1) * LOADS + REST - 1) / REST;
        if (from < to && more) issue(s + STAGES, cur, from, to);
        SB();
      }
      cur = nxt;
    };
    wait(min(STAGES, steps) - 1);
    __builtin_amdgcn_s_barrier();
    SB();
#pragma unroll
    for (int kk = 0; kk < HALVES; ++kk) {
#pragma unroll
      for (int j = 0; j < NT; ++j) read_b(0, kk, j, 0);
#pragma unroll
      for (int i = 0; i < MT; ++i) read_a(0, kk, i, 0);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const char* const bl = smem + BIAS + (wn * 16 * NT + 16 * j) * 2;
      if (EPI == EPI_PART) {
        c0[j] = f32x4(0.f);
      } else if (V_TILE) {
        c0[j] = f32x4(Mma<T>::lo(*reinterpret_cast<const uint16_t*>(bl + l16 * 2)));
      } else {
        const u32x2 x = *reinterpret_cast<const u32x2*>(bl + g4 * 8);
        c0[j] = f32x4{Mma<T>::lo(x.x), Mma<T>::hi(x.x), Mma<T>::lo(x.y), Mma<T>::hi(x.y)};
      }
    }
    SB();
    const std::true_type yes;
    const std::false_type no;
    int s = 1;
    if constexpr (DEEP) {
      const std::integral_constant<int, 0> even;
      const std::integral_constant<int, 1> odd;
      deep_step(0, even, yes, no, no);
#pragma clang loop unroll(disable)
      for (; s + 1 < steps - STAGES; s += 2) {
        deep_step(s, odd, no, yes, no);
        deep_step(s + 1, even, no, yes, no);
      }
#pragma clang loop unroll(disable)
      for (; s + 1 < steps - 1; s += 2) {
        deep_step(s, odd, no, no, no);
        deep_step(s + 1, even, no, no, no);
      }
      if (s + 1 < steps) {
        deep_step(s, odd, no, no, no);
        deep_step(s + 1, even, no, no, yes);
      } else {
        deep_step(s, odd, no, no, yes);
      }
    } else {
      step(0, yes, no, no);
#pragma clang loop unroll(disable)
      for (; s < steps - STAGES; ++s) step(s, no, yes, no);
#pragma clang loop unroll(disable)
      for (; s < steps - 1; ++s) step(s, no, no, no);
      step(s, no, no, yes);
    }
  };
  if (v_tile) loop(std::true_type());
  else loop(std::false_type());
  if (n0 >= p.n) return;

  char* const room = smem + w * 32 * block_pitch<NT, EPI>();
  if constexpr (EPI == EPI_PART) {
    const __amdgpu_buffer_rsrc_t sc =
        __builtin_amdgcn_make_buffer_rsrc(static_cast<float*>(p.c) + int64_t(slice) * p.m * p.n, 0, uint32_t(p.m) * uint32_t(p.n) * 4u, 0x00020000);
    store_block<T, MT, NT, EPI>(acc, sc, p.n, m0, n0, room);
    return;
  }
  if constexpr (EPI == EPI_QKV) {
    static_assert(MT % 2 == 0 && (NT == 2 || NT == 4), "a wave's columns lie in one head");
    if (n0 >= dm) {
      const int seq_end = *reinterpret_cast<const int*>(smem + ENDS + lane * 4), col = n0 - (v_tile ? 2 : 1) * dm;
      if (v_tile) store_v<T>(acc, p, seq_end, m0, col >> 6, col & 63);
      else store_k<T>(acc, p, seq_end, m0, col >> 6, col & 63);
      return;
    }
  }
  const __amdgpu_buffer_rsrc_t sc = __builtin_amdgcn_make_buffer_rsrc(p.c, 0, uint32_t(p.m) * uint32_t(p.n) * 2u, 0x00020000);
  store_block<T, MT, NT, EPI>(acc, sc, p.n, m0, n0, room);
}

int launched() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? RT_OK : rt::fail(RT_EIO, "gemm launch failed: %s", hipGetErrorString(e));
}

template <typename T, int TM, int MT0, int MT1, int EPI> int launch(const Params& base, hipStream_t st) {
  Params p = base;
  p.tiles_m = (p.m + TM - 1) / TM;
  p.tiles_n = (p.n + TN - 1) / TN;
  static std::atomic<uint64_t> done{0};
  if (int rc = allow_lds(reinterpret_cast<const void*>(&gemm_bt_kernel<T, TM, MT0, MT1, EPI>), lds_bytes<TM>(), done)) return rc;
  const int total = p.tiles_m * p.tiles_n;
  const int grid = total >= 256 ? 256 : (total + 7) / 8 * 8;
  RT_LAUNCH((gemm_bt_kernel<T, TM, MT0, MT1, EPI>), dim3(grid), dim3(512), lds_bytes<TM>(), st, p);
  return launched();
}

template <typename T, int MT, int NT, int WM, int WN, int STAGES, int EPI> int launch_small(const Params& base, hipStream_t st) {
  constexpr int TM = 16 * MT * WM, TC = 16 * NT * WN, LDS = STAGES * (TM + TC) * ROW + SMALL_EXTRA;
  Params p = base;
  p.tiles_m = (p.m + TM - 1) / TM;
  p.tiles_n = (p.n + TC - 1) / TC;
  static std::atomic<uint64_t> done{0};
  if (int rc = allow_lds(reinterpret_cast<const void*>(&gemm_bt_small_kernel<T, MT, NT, WM, WN, STAGES, EPI>), LDS, done)) return rc;
  const int total = p.tiles_m * p.tiles_n * p.slices;
  RT_LAUNCH((gemm_bt_small_kernel<T, MT, NT, WM, WN, STAGES, EPI>), dim3((total + 7) / 8 * 8), dim3(64 * WM * WN), LDS, st, p);
  return launched();
}

// ---- which kernel ----------------------------------------------------------------------------------------------------
// A product's time is estimated for every kernel and number of slices from a model with measured figures for each
// (microseconds, random fp16 operands, weights and activations in rotation through 180 MB and up to 340 MB, as a stack of
// layers finds them: with one set of operands in the caches the long reductions run a quarter faster and slices do not pay):
// one step of a workgroup that has its CU to itself, how much longer it takes when every CU has one, a step of two workgroups
// that share a CU, the launch, and what each round of workgroups spends on its first loads and its epilogue; plus the GELU
// by the outputs of a round, and the slices' way to memory and back.  The figures are a least-squares fit to 940 launches
// (15 row counts from 64 to 37184 at hidden 768, five from 128 to 40768 at 1024, all four products of a layer, up to six
// slices; root mean square of the error 7 %; all with plain stores, where those below 192 x 256 are written through now), over which the kernel that the model picks is 0.6 % slower than the fastest on
// average; with the LayerNorm behind it (20 row counts, up to eight slices) 1.3 %.  Where the lines fall, both sides (us):
//   512 x 3072 x 768 + GELU   128 x 64: 6.9, 64 x 64: 7.2, 128 x 128: 8.5    1024 x 2304 x 768 split   128 x 128: 8.3, 128 x 64: 9.1
//   2816 x 2304 x 768 split   128 x 256: 14.6, 128 x 128: 16.1, 192 x 256: 18.2    4096 x 2304 x 768 split   192 x 256: 21.2, 128 x 256: 23.9
//   2816 x 3072 x 768 + GELU  192 x 192: 17.5, 192 x 256: 18.0    8192 x 768 x 3072   128 x 192: 39.2, 192 x 192: 44.9, 192 x 256: 61.5
//   with the LayerNorm: 512 x 768 x 3072   2 slices of 64 x 64: 11.7, uncut 14.3    2816 x 768 x 3072   2 slices of 192 x 128: 28.8,
//   uncut 32.5    4096 x 768 x 3072   uncut 35.2, 2 slices 42.4
struct Choice {
  int tm, tc, slices;
};
struct Kernel {
  Choice c;
  float step, crowd, pair;      // pair 0: one workgroup per CU
  float launch, round;
  bool qkv, part;               // has the head split (32 rows and half a head per wave); writes slices
};
const Kernel kKernels[] = {
    {{256, 256, 1}, 1.072f, 0.467f, 0.f, 2.75f, 2.55f, true, false},
    {{224, 256, 1}, 0.927f, 0.544f, 0.f, 3.55f, 1.30f, true, false},
    {{192, 256, 1}, 0.830f, 0.559f, 0.f, 4.10f, 0.40f, true, false},
    {{192, 192, 1}, 0.594f, 0.416f, 0.f, 1.75f, 2.30f, false, false},
    {{128, 256, 1}, 0.605f, 0.394f, 0.f, 1.90f, 1.30f, true, false},
    {{192, 128, 1}, 0.475f, 0.301f, 0.f, 1.95f, 1.20f, false, true},
    {{128, 192, 1}, 0.463f, 0.328f, 0.f, 2.05f, 1.15f, false, false},
    {{128, 128, 1}, 0.328f, 0.265f, 0.f, 2.45f, 0.85f, true, true},
    {{128, 64, 1}, 0.267f, 0.150f, 0.631f, 1.60f, 0.90f, true, true},
    {{96, 64, 1}, 0.243f, 0.104f, 0.532f, 1.70f, 0.65f, false, true},
    {{64, 64, 1}, 0.162f, 0.081f, 0.404f, 2.05f, 0.55f, true, true},
};

// Products of few outputs hand their sums to the LayerNorm behind them in fp32, cut or not: rounded to 16 bits on the way they
// add 12 % (K = 768) to 18 % (K = 3072) to the error of its output against 64 bits (fp16 2.07e-4 -> 2.31e-4 and 2.48e-4, bf16
// 1.65e-3 -> 1.85e-3 and 1.96e-3), and one fp32 slice takes 0.2-0.4 us more than 16 bits (512 x 768 x 768 with the LayerNorm
// 8.6 -> 8.8).  The range is that of the products which pay for slices on operands in the caches; with more outputs
// the fp32 rows' way to memory and back would cost up to 6 us.
bool keeps_sums(int64_t m, int64_t n, int64_t k) {
  const int64_t rows = k <= 3072 ? 192 : 256;      // tiles of rows x 128 whose two slices are one round of workgroups
  return k >= 768 && m * n <= (k < 1344 ? 684 : k < 2048 ? 768 : 1160) * k && ((m + rows - 1) / rows) * ((n + 127) / 128) <= 128;
}

// max_slices 0: the caller takes the product itself; more: fp32 slices will do, which the caller's next kernel reads, and one
// slice is an uncut product in 16 bits, or in fp32 where keeps_sums.
Choice choose(int64_t m, int64_t n, int64_t k, int epi, int max_slices) {
  const int steps = int(k / BK);
  const bool sums = max_slices > 0 && keeps_sums(m, n, k);
  Choice best = kKernels[0].c;
  float best_us = 0.f;
  for (const Kernel& kn : kKernels) {
    if ((epi == EPI_QKV && !kn.qkv) || (sums && !kn.part)) continue;
    for (int s = 1; s <= (kn.part && max_slices > 1 ? max_slices : 1); ++s) {
      if (s > 1 && steps / s < 6) break;
      const int64_t wgs = ((m + kn.c.tm - 1) / kn.c.tm) * ((n + kn.c.tc - 1) / kn.c.tc) * s;
      const int64_t slots = kn.pair > 0.f ? 512 : 256, full = wgs / slots, rest = wgs % slots, rounds = full + (rest ? 1 : 0);
      const float alone = kn.step + kn.crowd * float(rest < 256 ? rest : 256) / 256.f, both = kn.pair > 0.f ? kn.pair : kn.step + kn.crowd;
      const float stepping = float(full) * both + (rest == 0 ? 0.f : rest <= 256 ? alone : both);
      float us = kn.launch + kn.round * float(rounds) + stepping * float((steps + s - 1) / s);
      if (epi == EPI_GELU) us += 2.9e-5f * float(kn.c.tm * kn.c.tc) * float(rounds) * (kn.pair > 0.f && full ? 2.f : 1.f);
      if (s > 1 || sums) us += 0.6f + float(m) * float(n) * (1.7e-6f * float(s) - 1.4e-6f);       // against 16 bits to the LayerNorm
      if (best_us == 0.f || us < best_us) { best_us = us; best = kn.c; best.slices = s; }
    }
  }
  return best;
}

template <typename T, int EPI> int dispatch(Params& p, const Choice& c, hipStream_t st) {
  p.slices = c.slices;
  if constexpr (EPI != EPI_PART) {
    if (c.tc == TN && c.tm >= 192) {
      if (c.tm == 256) return launch<T, 256, 8, 8, EPI>(p, st);
      if (c.tm == 224) return launch<T, 224, 8, 6, EPI>(p, st);
      return launch<T, 192, 6, 6, EPI>(p, st);
    }
    if (c.tc == 256) return launch_small<T, 4, 4, 2, 4, 3, EPI>(p, st);
  }
  if constexpr (EPI == EPI_NONE || EPI == EPI_GELU) {
    if (c.tc == 192 && c.tm == 192) return launch_small<T, 3, 6, 4, 2, 3, EPI>(p, st);
    if (c.tc == 192) return launch_small<T, 2, 6, 4, 2, 3, EPI>(p, st);
  }
  if constexpr (EPI != EPI_QKV) {
    if (c.tm == 192) return launch_small<T, 6, 2, 2, 4, 3, EPI>(p, st);
    if (c.tm == 96) return launch_small<T, 3, 2, 2, 2, 3, EPI>(p, st);
  }
  if (c.tc == 128) return launch_small<T, 2, 4, 4, 2, 4, EPI>(p, st);
  if (c.tm == 128) return launch_small<T, 4, 2, 2, 2, 3, EPI>(p, st);
  return launch_small<T, 2, 2, 2, 2, 4, EPI>(p, st);
}

}  // namespace

namespace rt {

bool gemm_mfma_takes(const void* a, const void* bt, const void* bias, const void* c, int64_t m, int64_t n, int64_t k, int dtype) {
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return (dtype == RT_F16 || dtype == RT_BF16) && k % BK == 0 && k >= 2 * BK && n % 8 == 0 && m * k < (int64_t(1) << 29) &&
         n * k < (int64_t(1) << 29) && (m + 256) * n < (int64_t(1) << 31) && aligned(a) && aligned(bt) && aligned(bias) && aligned(c);
}

// An uncut product is one chain of steps, 0.16 us each; with at most 64 of the smallest tiles most CUs have none and a
// library that cuts the reduction is ahead on long ones.  Measured (us in a graph, operands in rotation, hipBLASLt tuned for the
// shape / here): 64 x 768 x 1280 6.3 / 6.3, x 1536 7.0 / 6.7, x 2048 5.5-8.3 / 7.8, x 3072 7.4-10.7 / 10.7, x 8192 10.3 / 23.0;
// 256 x 1024 (64 tiles) x 1280 7.0 / 6.5, x 1536 7.6 / 7.0, x 2560 8.4-10.1 / 10.2, x 4096 11.1 / 13.5; 1 x 4096 x 1536
// 7.8 / 6.8, x 3072 8.8-10.7 / 11.1.  Between 1536 and 2560 it depends on which solution the library's timing has found.  More
// outputs, here: 512 x 768 (96 tiles) x 2048 8.6, 512 x 1024 x 4096 13.9.
bool gemm_mfma_pays(int64_t m, int64_t n, int64_t k) {
  return k <= 24 * BK || ((m + 63) / 64) * ((n + 63) / 64) > 64;
}

int gemm_mfma_bt(const void* a, const void* bt, const void* bias, void* c, int64_t m, int64_t n, int64_t k, bool gelu, int dtype,
                 void* stream) {
  Params p{};
  p.a = a; p.bt = bt; p.bias = bias; p.c = c;
  p.m = int(m); p.n = int(n); p.k = int(k);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Choice ch = choose(m, n, k, gelu ? EPI_GELU : EPI_NONE, 0);
  if (dtype == RT_F16) return gelu ? dispatch<_Float16, EPI_GELU>(p, ch, st) : dispatch<_Float16, EPI_NONE>(p, ch, st);
  return gelu ? dispatch<__bf16, EPI_GELU>(p, ch, st) : dispatch<__bf16, EPI_NONE>(p, ch, st);
}

int gemm_mfma_qkv(const void* a, const void* bt, const void* bias, void* rows, void* kt, void* vt, const int* seq_blocks_dev,
                  int batch, int64_t m, int heads, int64_t k, int dtype, void* stream) {
  Params p{};
  p.a = a; p.bt = bt; p.bias = bias; p.c = rows;
  p.m = int(m); p.n = 3 * heads * 64; p.k = int(k);
  p.kt = kt; p.vt = vt; p.seq_blocks = seq_blocks_dev; p.batch = batch; p.heads = heads;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Choice ch = choose(m, p.n, k, EPI_QKV, 0);
  return dtype == RT_F16 ? dispatch<_Float16, EPI_QKV>(p, ch, st) : dispatch<__bf16, EPI_QKV>(p, ch, st);
}

int gemm_mfma_slices(int64_t m, int64_t n, int64_t k, int64_t max_bytes) {
  if ((m + 256) * n * 4 >= (int64_t(1) << 32)) return 0;
  const int64_t fit = max_bytes / (m * n * 4);
  if (fit < 1) return 0;
  const int slices = choose(m, n, k, EPI_PART, int(fit > 8 ? 8 : fit)).slices;
  return slices > 1 || keeps_sums(m, n, k) ? slices : 0;
}

int gemm_mfma_part(const void* a, const void* bt, float* parts, int64_t m, int64_t n, int64_t k, int slices, int dtype, void* stream) {
  Params p{};
  p.a = a; p.bt = bt; p.c = parts;
  p.m = int(m); p.n = int(n); p.k = int(k);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Choice ch = choose(m, n, k, EPI_PART, slices);
  if (ch.slices != slices) return rt::fail(RT_EINVAL, "gemm: %d slices asked for, %d chosen", slices, ch.slices);
  return dtype == RT_F16 ? dispatch<_Float16, EPI_PART>(p, ch, st) : dispatch<__bf16, EPI_PART>(p, ch, st);
}

void gemm_mfma_tile(int64_t m, int64_t n, int64_t k, bool gelu, bool qkv, int max_slices, int* tile) {
  const Choice ch = choose(m, n, k, max_slices ? EPI_PART : qkv ? EPI_QKV : gelu ? EPI_GELU : EPI_NONE, max_slices);
  tile[0] = ch.tm;
  tile[1] = ch.tc;
  tile[2] = ch.slices;
}

}  // namespace rt
