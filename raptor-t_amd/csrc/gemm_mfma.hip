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
//   so the matrix pipe has work across the barrier, and the loads of the next tile's first steps are in flight
//   while the epilogue of the present one runs.  A tile's last step leaves its A stage empty: the epilogue turns its
//   outputs into whole rows there, and the load that belongs there follows in the next tile's first step.
//
// Bound by the power the part may draw: with random operands it holds 1.7-1.85 GHz in these loops, at 2 600 cycles a
// step where the matrix instructions alone take 2 240.  Measured against hipBLASLt's best of 64 suggestions for the
// shape, in turn on one box (us): 37184 x 2304 x 768 113 against 127, 37184 x 3072 x 768 147 against 165 and with bias +
// GELU 165 against 225, 37184 x 768 x 3072 130 against 132, 37184 x 768 x 768 41 against 44, 40768 x 1024 x 4096 268
// against 340, 40768 x 4096 x 1024 274 against 282; the projection with the head split 141 against 114 + 38.
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "gemm_mfma.h"
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
typedef int i32x4 __attribute__((ext_vector_type(4)));

// The matrix instruction as assembly, so that its accumulators stay where they are: given the choice the compiler
// writes them to other registers and runs out of them.  It cannot see the instruction's hazards then; the two that
// occur here (vector writes of an operand just before, vector reads of a result just after) are covered by the waits
// at both ends of main_loop and at the head of its loop.
template <typename T> struct Mma;
template <> struct Mma<_Float16> {
  typedef f16x8 v8;
  __device__ static void run(v8 a, v8 b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  __device__ static void first(v8 a, v8 b, f32x4& d, f32x4 c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c)); }
  __device__ static uint32_t two(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2)); }
  __device__ static float lo(uint32_t w) { return float(__builtin_bit_cast(f16x2, w).x); }
  __device__ static float hi(uint32_t w) { return float(__builtin_bit_cast(f16x2, w).y); }
};
template <> struct Mma<__bf16> {
  typedef bf16x8 v8;
  __device__ static void run(v8 a, v8 b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  __device__ static void first(v8 a, v8 b, f32x4& d, f32x4 c) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c)); }
  __device__ static uint32_t two(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2)); }
  __device__ static float lo(uint32_t w) { return __uint_as_float(w << 16); }
  __device__ static float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};

constexpr int TN = 256;                       // columns of a tile
constexpr int BK = 64;                        // reduction steps of a stage
constexpr int ROW = BK * 2;                   // bytes of an LDS row
constexpr int EPI_BYTES = 32 * 64 * 2;        // a wave's room for turning a 32 x 64 block of outputs into whole rows
constexpr int WAVES = 8;
constexpr int NT = 2;                         // cache policy of the stores of C: non-temporal
constexpr int B_STAGE = TN * ROW;

// An A stage also has to hold the epilogue's blocks of all waves.
template <int TM> constexpr int a_stage() { return TM * ROW > WAVES * EPI_BYTES ? TM * ROW : WAVES * EPI_BYTES; }
template <int TM> constexpr int lds_bytes() { return 3 * a_stage<TM>() + 2 * B_STAGE; }

#define SB() __builtin_amdgcn_sched_barrier(0)

// 64 lanes x 16 bytes from srd[voff + soff] to LDS bytes [lds, lds + 1024).  Hidden from the compiler's wait
// counting on purpose (it would wait for every load before any LDS read); the waits stand in the loop.
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

enum { EPI_NONE = 0, EPI_GELU = 1, EPI_QKV = 2 };

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
  // s+1, or in a tile's first step the stores of the last tile's outputs, which are as young.
  constexpr int LEFT = TM / 64, STORES = EPI == EPI_QKV ? LEFT : 2 * MT;
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
    if (W == LAST) {                                 // the compiler's own wait for these comes here, where it costs nothing
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
  // Workgroups go to the 8 XCDs round-robin: XCD x takes the x-th eighth of the tiles (columns vary fastest), its
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
      // K and V^T tiles: where the half tile of the 32 tokens from `row` on begins (lane's part), for the wave's first head
      auto half_tile = [&](void* base, int row, int h) __attribute__((always_inline)) {
        const int g = row >> 6, lane = again(threadIdx.x & 63);
        int s, g0, end;                                    // the sequence block g belongs to
        if (p.batch <= 64) {
          s = __popcll(__ballot(lane < p.batch && bias.seq_end <= g));
          g0 = s == 0 ? 0 : __builtin_amdgcn_readlane(bias.seq_end, s - 1);
          end = __builtin_amdgcn_readlane(bias.seq_end, s);
        } else {
          s = 0;
          for (int b0 = 0; b0 < p.batch; b0 += 64)
            s += __popcll(__ballot(b0 + lane < p.batch && p.seq_blocks[min(b0 + lane + 1, p.batch)] <= g));
          g0 = p.seq_blocks[s];
          end = p.seq_blocks[s + 1];
        }
        const int nb = end - g0;
        return static_cast<T*>(base) + (int64_t(g0) * p.heads + int64_t(h) * nb + (g - g0)) * 4096 + lane * 8;
      };
      // (The assembly comments keep the compiler from merging equal code of the branches, which costs it registers.)
      if (EPI == EPI_QKV && v_tile) {
        asm volatile("; V tile");
        main_loop<T, TM, MT, EPI, true>(acc, c0, bias, next_bias, lda, ldb, st, p, sa, sb, smem, lds0, w, lane, offa, offb);
        if (n0 >= p.n) continue;
        // A lane's accumulators are 4 consecutive tokens of one column; fragment 4 * (d >> 5) + (token >> 4) of the tile
        // wants, in lane (d & 31) + 32 * x, the tokens 4 x .. + 4 and 8 + 4 x .. + 4 of its 16.
#pragma unroll
        for (int i = 0; i < MT; i += 2) {
          const int row = m0 + 16 * i;
          if (row >= p.m) break;
          T* const t = half_tile(p.vt, row, (n0 - 2 * dm) >> 6) + ((row >> 5) & 1) * 1024;
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
              const f32x4 &c = acc[i + q][j], &d = acc[i + q][j + 1];
              uint32_t x0 = Mma<T>::two(c[0], c[1]), x1 = Mma<T>::two(c[2], c[3]);
              uint32_t y0 = Mma<T>::two(d[0], d[1]), y1 = Mma<T>::two(d[2], d[3]);
              permlane16_swap(x0, y0);
              permlane16_swap(x1, y1);
              permlane32_swap(x0, y0);
              permlane32_swap(x1, y1);
              *reinterpret_cast<u32x4*>(t + (2 * j + q) * 512) = u32x4{x0, x1, y0, y1};
            }
        }
        asm volatile("; V tile done");
        continue;
      }
      main_loop<T, TM, MT, EPI, false>(acc, c0, bias, next_bias, lda, ldb, st, p, sa, sb, smem, lds0, w, lane, offa, offb);
      if (EPI == EPI_QKV && n0 >= dm) {
        // A lane's accumulators are 4 consecutive columns of one token; fragment 4 * (token >> 5) + (d >> 4) of the tile
        // wants, in lane (token & 31) + 32 * x, the columns 8 x .. + 8 of its 16.
#pragma unroll
        for (int i = 0; i < MT; i += 2) {
          const int row = m0 + 16 * i;
          if (row >= p.m) break;
          T* const t = half_tile(p.kt, row, (n0 - dm) >> 6) + ((row >> 5) & 1) * 2048;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4 &c = acc[i][j], &d = acc[i + 1][j];
            uint32_t x0 = Mma<T>::two(c[0], c[1]), x1 = Mma<T>::two(c[2], c[3]);
            uint32_t y0 = Mma<T>::two(d[0], d[1]), y1 = Mma<T>::two(d[2], d[3]);
            permlane16_swap(x0, y0);
            permlane16_swap(x1, y1);
            *reinterpret_cast<u32x4*>(t + j * 512) = u32x4{x0, x1, y0, y1};
          }
        }
        asm volatile("; K tile done");
        continue;
      }
      // rows of C: 16 x 64 outputs at a time through the wave's LDS room (the A stage of the tile's last step; st has
      // moved on by one), stored as eight whole 128-byte rows per instruction.  A block's rows are read back while the
      // next one is written, and the stores pass no test: offsets past the end of C are dropped by the range check.
      const int lane = again(threadIdx.x & 63), l16 = lane & 15, g4 = lane >> 4;
      char* const epi = smem + (st.a == 0 ? 2u * a_stage<TM>() : st.a - a_stage<TM>()) + w * EPI_BYTES;
      const bool col_ok = n0 + (lane & 7) * 8 < p.n;
      uint32_t voff = col_ok ? (uint32_t(m0 + (lane >> 3)) * uint32_t(p.n) + uint32_t(n0 + (lane & 7) * 8)) * 2u : 0xfffffff0u;
      const uint32_t ld8 = col_ok ? uint32_t(p.n) * 16u : 0u;       // eight rows
      const int wr = l16 * 128 + 8 * (g4 & 1), wx = l16 >> 1, rr = (lane >> 3) * 128;
#pragma unroll
      for (int i = 0; i <= MT; ++i) {
        u32x4 o[2];
        if (i > 0) {
#pragma unroll
          for (int j = 0; j < 2; ++j)
            o[j] = *reinterpret_cast<const u32x4*>(epi + ((i - 1) & 1) * 2048 + j * 1024 + rr + (((lane & 7) ^ (((lane >> 4) + 4 * j) & 7)) << 4));
        }
        if (i < MT) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            f32x4 v = acc[i][j];
            if (EPI == EPI_GELU) {
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
            }
            *reinterpret_cast<u32x2*>(epi + (i & 1) * 2048 + wr + (((2 * j + (g4 >> 1)) ^ wx) << 4)) =
                u32x2{Mma<T>::two(v[0], v[1]), Mma<T>::two(v[2], v[3])};
          }
        }
        if (i > 0) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            __builtin_amdgcn_raw_buffer_store_b128(o[j], sc, int(voff), 0, NT);
            voff += ld8;
          }
        }
        SB();
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the trailing loads write LDS of this workgroup
  };
  if (MT0 == MT1 || w < 4) run(std::integral_constant<int, MT0>());
  else run(std::integral_constant<int, MT1>());
}

template <typename T, int TM, int MT0, int MT1, int EPI>
int launch(const Params& base, hipStream_t st) {
  Params p = base;
  p.tiles_m = (p.m + TM - 1) / TM;
  p.tiles_n = (p.n + TN - 1) / TN;
  static std::once_flag once;
  static hipError_t attr = hipSuccess;
  std::call_once(once, [] {
    attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_bt_kernel<T, TM, MT0, MT1, EPI>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes<TM>());
  });
  if (attr != hipSuccess) return rt::fail(RT_EIO, "gemm: %d bytes of LDS refused: %s", lds_bytes<TM>(), hipGetErrorString(attr));
  const int total = p.tiles_m * p.tiles_n;
  const int grid = total >= 256 ? 256 : (total + 7) / 8 * 8;
  RT_LAUNCH((gemm_bt_kernel<T, TM, MT0, MT1, EPI>), dim3(grid), dim3(512), lds_bytes<TM>(), st, p);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? RT_OK : rt::fail(RT_EIO, "gemm launch failed: %s", hipGetErrorString(e));
}

template <typename T, int EPI> int dispatch(const Params& p, hipStream_t st) {
  // rounds of 256 workgroups x height of a tile: the shortest schedule
  const int64_t tn = (p.n + TN - 1) / TN;
  auto cost = [&](int tm) { return (((p.m + tm - 1) / tm) * tn + 255) / 256 * (tm + 24); };
  const int heights[3] = {256, 224, 192};
  int best = 0;
  for (int i = 1; i < 3; ++i)
    if (cost(heights[i]) < cost(heights[best])) best = i;
  if (best == 0) return launch<T, 256, 8, 8, EPI>(p, st);
  if (best == 1) return launch<T, 224, 8, 6, EPI>(p, st);
  return launch<T, 192, 6, 6, EPI>(p, st);
}

}  // namespace

namespace rt {

// At least 64 tiles (a quarter of the CUs): with fewer, one CU's share of a long reduction is longer than what the
// library's smaller tiles take (2816 x 768 x 3072, 45 tiles: 40 us against 22).
bool gemm_mfma_takes(const void* a, const void* bt, const void* bias, const void* c, int64_t m, int64_t n, int64_t k, int dtype) {
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if ((m + 191) / 192 * ((n + TN - 1) / TN) < 64) return false;
  return (dtype == RT_F16 || dtype == RT_BF16) && k % BK == 0 && k >= 2 * BK && n % 8 == 0 && m * k < (int64_t(1) << 29) &&
         n * k < (int64_t(1) << 29) && (m + 256) * n < (int64_t(1) << 31) && aligned(a) && aligned(bt) && aligned(bias) && aligned(c);
}

int gemm_mfma_bt(const void* a, const void* bt, const void* bias, void* c, int64_t m, int64_t n, int64_t k, bool gelu, int dtype,
                 void* stream) {
  Params p{};
  p.a = a; p.bt = bt; p.bias = bias; p.c = c;
  p.m = int(m); p.n = int(n); p.k = int(k);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == RT_F16) return gelu ? dispatch<_Float16, EPI_GELU>(p, st) : dispatch<_Float16, EPI_NONE>(p, st);
  return gelu ? dispatch<__bf16, EPI_GELU>(p, st) : dispatch<__bf16, EPI_NONE>(p, st);
}

int gemm_mfma_qkv(const void* a, const void* bt, const void* bias, void* rows, void* kt, void* vt, const int* seq_blocks_dev,
                  int batch, int64_t m, int heads, int64_t k, int dtype, void* stream) {
  Params p{};
  p.a = a; p.bt = bt; p.bias = bias; p.c = rows;
  p.m = int(m); p.n = 3 * heads * 64; p.k = int(k);
  p.kt = kt; p.vt = vt; p.seq_blocks = seq_blocks_dev; p.batch = batch; p.heads = heads;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == RT_F16 ? dispatch<_Float16, EPI_QKV>(p, st) : dispatch<__bf16, EPI_QKV>(p, st);
}

}  // namespace rt
