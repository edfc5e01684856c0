// kernel_wave.hip -- matrix-core register simplex kernel for gfx950 (FP32).
//
// One workgroup of NW wavefronts per LP, persistent over a work queue.  The constraint rows
// of the condensed tableau live in matrix-core accumulators for the whole solve: a tile is
// 16 rows x 64 columns, the 16 accumulator registers of one v_mfma_f32_16x16x1_4b, so the
// rank-1 update of a pivot is one such instruction per tile,
//     T[16 rows][64 columns] += a[16 rows] (x) prow[64 columns],
// 1024 FMAs in 32 cycles of the matrix pipe, against 64 cycles of v_fma_f32.  With K = 1
// the instruction is a plain IEEE FMA per element (subnormals and signed zeros included;
// bit-compared with fmaf over 16M operand triples), so results stay bit-identical to the
// oracle and to the other kernels.
//
// Layout.  Wavefront w owns G column groups of 64 columns, every row.  Lane l of a group
// holds that group's column l in "column form": objective rows, nonbasic ids, the scaled
// pivot row -- exactly the instruction's B operand.  The pivot column, the right-hand side
// and the basic ids are in "row form": lane l holds row l + 64 p, which is the A operand of
// rows 64 p .. 64 p + 63 (the cbsz/abid modifiers broadcast one block of 16 rows to all four
// column blocks, so one register serves four tiles).  Neither operand is ever broadcast
// through LDS.  Objective rows, right-hand side, ids and reductions are replicated in every
// wavefront, so a pivot needs two barriers (pivot column, pivot row) when NW > 1 and none
// when NW = 1.
//
// Per pivot:
//   column  the four lanes that hold column s write it to LDS (16 rows per 128-bit store)
//           and zero it in place; every lane reads its rows back (row form)
//   ratio   theta and 1/a for all rows at once, DPP minimum, ballot: the pivot row r is
//           wave-uniform, its reciprocal is read from its lane
//   row     a scalar branch on r reads the registers of row r (16 lanes hold it), lane
//           permutes spread it to column form; the row itself is set to -0.0, so that the
//           update with a[r] = 1 leaves exactly the scaled row
//   update  the objective rows and the right-hand side in vector ALU, the tiles in the
//           matrix pipe; the next pricing (objective rows only) runs between the matrix
//           instructions
// What bounds it is the chain of one pivot (LDS round trip of the column, division, two
// reductions, the jumps into the register tables), about 0.75 us; the matrix pipe adds 13 ns
// per tile.  Measured against the column-per-lane kernel it replaced (every lane whole columns,
// update by v_fma_f32 with the pivot column read from LDS as broadcasts): one 105x103 LP
// 0.133 ms against 0.259, 1024 of them in the mixed batch 0.50 ms against 1.16, 8192 of a
// parametric family 0.45 ms against 0.88; and against the 2-D block kernel, 205x203 x 1024
// 7.3 ms against 14.5, and 16 LPs of 250x249, formerly streamed from HBM, 2.9 ms against 60.
// Replaces the reference's mykernel (simplex.cu:35-385), whose tableau lives in global
// memory and whose pivot takes ~4 log2(blockDim) barriers.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "kernels.hpp"
#include "simplex_device.hpp"

namespace blpg {


namespace {

__device__ __forceinline__ float rdlane(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// LDS byte address
__device__ __forceinline__ unsigned lds_addr(const float* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const float*)p;
}

// One step of the minimum over the 64 lanes: v_min_f32 with a DPP source (the IEEE minimum
// on the finite / infinite keys that reach it, without fminf's NaN canonicalisation); rows
// outside the step's row mask keep their value.  s_nop 1: the two wait states a DPP read of
// a VGPR needs after the VALU write.  After six steps lane 63 holds the minimum.
template <int STEP>
__device__ __forceinline__ void min_step(float& x) {
  if constexpr (STEP == 0)
    asm volatile("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf" : "+v"(x));
  else if constexpr (STEP == 1)
    asm volatile("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf" : "+v"(x));
  else if constexpr (STEP == 2)
    asm volatile("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf" : "+v"(x));
  else if constexpr (STEP == 3)
    asm volatile("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf" : "+v"(x));
  else if constexpr (STEP == 4)
    asm volatile("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf" : "+v"(x));
  else
    asm volatile("s_nop 1\n\tv_min_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\ts_nop 1" : "+v"(x));
}
__device__ __forceinline__ float wave_fmin(float x) {
  min_step<0>(x); min_step<1>(x); min_step<2>(x); min_step<3>(x); min_step<4>(x); min_step<5>(x);
  return rdlane(x, 63);
}

// compile-time loop: f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <class F, int... I>
__device__ __forceinline__ void unroll_seq(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unroll(F&& f) {
  unroll_seq(f, std::make_integer_sequence<int, N>{});
}

// Calls f(integral_constant<u>) for the u in [LO, LO + N) equal to the wave-uniform k: a
// binary tree of scalar branches, so that register indices inside f stay static.
template <int LO, int N, class F>
__device__ __forceinline__ void dispatch(int k, F&& f) {
  if constexpr (N == 1) {
    f(std::integral_constant<int, LO>{});
  } else {
    constexpr int H = N / 2;
    if (k < LO + H) dispatch<LO, H>(k, f);
    else dispatch<LO + H, N - H>(k, f);
  }
}

// ---- the tiles' accumulation registers ----
// Tile (ch, g) is a[16 (ch G + g) .. + 15], named in inline assembly: as C++ values the
// tiles would be live through every branch of the state machine, and the compiler copies
// or spills them there.  Nothing else in the kernels uses accumulation registers
// (acc_reserve makes the kernel own them).  The compiler does not see these instructions'
// hazards; the waits are here:
//   acc_settle  before an access that may follow a matrix instruction (8 passes: 11 wait
//               states until its result may be read or written)
//   acc_ready   before matrix instructions (2 wait states after a vector write of an
//               operand, 4 after a vector write of the execution mask); that no write of an
//               operand moved behind it is read from the listing by the build
template <int A>
__device__ __forceinline__ float acc_get() {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(A));
  return x;
}
template <int A>
__device__ __forceinline__ void acc_set(float x) {
  asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x), "n"(A));
}
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 11"); }
__device__ __forceinline__ void acc_ready() { asm volatile("s_nop 4"); }
// a[A .. A+15] += x (x) y: block ABID of x (16 rows) against all 64 columns of y
template <int A, int ABID>
__device__ __forceinline__ void acc_rank1(float x, float y) {
  asm volatile("v_mfma_f32_16x16x1_4b_f32 a[%2:%3], %0, %1, a[%2:%3] cbsz:2 abid:%4" ::"v"(x), "v"(y), "n"(A),
               "n"(A + 15), "n"(ABID));
}
// The indexed accesses jump into a table of equal-sized cases (a register number cannot be
// dynamic): one computed jump, where a tree of branches over the index costs ten.  The index
// is clamped to the table, so the jump stays inside it for any value.
//
// Registers 4b + I of tiles (CHUNK, 0 .. G-1), u = 4 CHUNK + I wave-uniform, to y; with
// CLEAR the lanes of `mask` then hold `z` there.
template <int CH, int G, bool CLEAR>
__device__ __forceinline__ void acc_row(int u, unsigned long long mask, float z, float (&y)[4 * G]) {
#define BLPG_ACC_HEAD                      \
  "s_nop 11\n\t"                           \
  "s_min_u32 %[t], %[u], %[cases] - 1\n\t" \
  "s_mul_i32 %[t], %[t], %[size]\n\t"      \
  "s_add_u32 %[t], %[t], 12\n\t"           \
  "s_getpc_b64 vcc\n\t"                    \
  "s_add_u32 vcc_lo, vcc_lo, %[t]\n\t"     \
  "s_addc_u32 vcc_hi, vcc_hi, 0\n\t"       \
  "s_setpc_b64 vcc\n\t"                    \
  ".set blpg_u, 0\n\t"                     \
  ".rept %[cases]\n\t"                     \
  ".set blpg_a, (blpg_u / 4) * 16 * %[g] + (blpg_u & 3)\n\t"
#define BLPG_ACC_TAIL                      \
  "s_branch Lacc%=\n\t"                    \
  ".set blpg_u, blpg_u + 1\n\t"            \
  ".endr\n"                                \
  "Lacc%=:\n\t"
  int t;
  if constexpr (G == 2) {
#define BLPG_RD8                                                                        \
  "v_accvgpr_read_b32 %[y0], a[blpg_a]\n\tv_accvgpr_read_b32 %[y1], a[blpg_a + 4]\n\t"      \
  "v_accvgpr_read_b32 %[y2], a[blpg_a + 8]\n\tv_accvgpr_read_b32 %[y3], a[blpg_a + 12]\n\t" \
  "v_accvgpr_read_b32 %[y4], a[blpg_a + 16]\n\tv_accvgpr_read_b32 %[y5], a[blpg_a + 20]\n\t" \
  "v_accvgpr_read_b32 %[y6], a[blpg_a + 24]\n\tv_accvgpr_read_b32 %[y7], a[blpg_a + 28]\n\t"
#define BLPG_Y8 [y0] "=&v"(y[0]), [y1] "=&v"(y[1]), [y2] "=&v"(y[2]), [y3] "=&v"(y[3]), \
                [y4] "=&v"(y[4]), [y5] "=&v"(y[5]), [y6] "=&v"(y[6]), [y7] "=&v"(y[7]), [t] "=&s"(t)
    if constexpr (CLEAR)
      asm volatile(BLPG_ACC_HEAD BLPG_RD8 "s_mov_b64 exec, %[mask]\n\t"
                   "v_accvgpr_write_b32 a[blpg_a], %[z]\n\tv_accvgpr_write_b32 a[blpg_a + 4], %[z]\n\t"
                   "v_accvgpr_write_b32 a[blpg_a + 8], %[z]\n\tv_accvgpr_write_b32 a[blpg_a + 12], %[z]\n\t"
                   "v_accvgpr_write_b32 a[blpg_a + 16], %[z]\n\tv_accvgpr_write_b32 a[blpg_a + 20], %[z]\n\t"
                   "v_accvgpr_write_b32 a[blpg_a + 24], %[z]\n\tv_accvgpr_write_b32 a[blpg_a + 28], %[z]\n\t"
                   BLPG_ACC_TAIL "s_mov_b64 exec, -1"
                   : BLPG_Y8
                   : [u] "s"(u), [mask] "s"(mask), [z] "v"(z), [size] "n"(136), [cases] "n"(4 * CH), [g] "n"(G)
                   : "vcc", "scc");
    else
      asm volatile(BLPG_ACC_HEAD BLPG_RD8 BLPG_ACC_TAIL
                   : BLPG_Y8
                   : [u] "s"(u), [size] "n"(68), [cases] "n"(4 * CH), [g] "n"(G)
                   : "vcc", "scc");
#undef BLPG_RD8
#undef BLPG_Y8
  } else {
    static_assert(G == 1 || G == 2);
#define BLPG_RD4                                                                        \
  "v_accvgpr_read_b32 %[y0], a[blpg_a]\n\tv_accvgpr_read_b32 %[y1], a[blpg_a + 4]\n\t"      \
  "v_accvgpr_read_b32 %[y2], a[blpg_a + 8]\n\tv_accvgpr_read_b32 %[y3], a[blpg_a + 12]\n\t"
#define BLPG_Y4 [y0] "=&v"(y[0]), [y1] "=&v"(y[1]), [y2] "=&v"(y[2]), [y3] "=&v"(y[3]), [t] "=&s"(t)
    if constexpr (CLEAR)
      asm volatile(BLPG_ACC_HEAD BLPG_RD4 "s_mov_b64 exec, %[mask]\n\t"
                   "v_accvgpr_write_b32 a[blpg_a], %[z]\n\tv_accvgpr_write_b32 a[blpg_a + 4], %[z]\n\t"
                   "v_accvgpr_write_b32 a[blpg_a + 8], %[z]\n\tv_accvgpr_write_b32 a[blpg_a + 12], %[z]\n\t"
                   BLPG_ACC_TAIL "s_mov_b64 exec, -1"
                   : BLPG_Y4
                   : [u] "s"(u), [mask] "s"(mask), [z] "v"(z), [size] "n"(72), [cases] "n"(4 * CH), [g] "n"(G)
                   : "vcc", "scc");
    else
      asm volatile(BLPG_ACC_HEAD BLPG_RD4 BLPG_ACC_TAIL
                   : BLPG_Y4
                   : [u] "s"(u), [size] "n"(36), [cases] "n"(4 * CH), [g] "n"(G)
                   : "vcc", "scc");
#undef BLPG_RD4
#undef BLPG_Y4
  }
}
// Column block u = 4 g + b (wave-uniform) of the lanes in `mask` to LDS: rows 16 ch + 4 q ..
// of every chunk at `at` + 64 ch bytes; with ZERO it is then zeroed in place.
template <int CH, int G, bool ZERO>
__device__ __forceinline__ void acc_col(int u, unsigned long long mask, unsigned at) {
  int t;
#define BLPG_COL_STORE                                                      \
  ".set blpg_a, blpg_u * 4\n\t"                                             \
  ".set blpg_c, 0\n\t"                                                      \
  ".rept %[ch]\n\t"                                                         \
  "ds_write_b128 %[at], a[blpg_a + blpg_c * 16 * %[g] : blpg_a + blpg_c * 16 * %[g] + 3] offset:blpg_c * 64\n\t" \
  ".set blpg_c, blpg_c + 1\n\t"                                             \
  ".endr\n\t"
  if constexpr (ZERO)
    asm volatile("s_mov_b64 exec, %[mask]\n\t" BLPG_ACC_HEAD BLPG_COL_STORE
                 ".set blpg_c, 0\n\t"
                 ".rept %[ch]\n\t"
                 "v_accvgpr_write_b32 a[blpg_a + blpg_c * 16 * %[g]], 0\n\t"
                 "v_accvgpr_write_b32 a[blpg_a + blpg_c * 16 * %[g] + 1], 0\n\t"
                 "v_accvgpr_write_b32 a[blpg_a + blpg_c * 16 * %[g] + 2], 0\n\t"
                 "v_accvgpr_write_b32 a[blpg_a + blpg_c * 16 * %[g] + 3], 0\n\t"
                 ".set blpg_c, blpg_c + 1\n\t"
                 ".endr\n\t" BLPG_ACC_TAIL "s_mov_b64 exec, -1\n\ts_waitcnt lgkmcnt(0)"
                 : [t] "=&s"(t)
                 : [u] "s"(u), [mask] "s"(mask), [at] "v"(at), [size] "n"(40 * CH + 4), [cases] "n"(4 * G),
                   [g] "n"(G), [ch] "n"(CH)
                 : "vcc", "scc", "memory");
  else
    asm volatile("s_mov_b64 exec, %[mask]\n\t" BLPG_ACC_HEAD BLPG_COL_STORE BLPG_ACC_TAIL
                 "s_mov_b64 exec, -1\n\ts_waitcnt lgkmcnt(0)"
                 : [t] "=&s"(t)
                 : [u] "s"(u), [mask] "s"(mask), [at] "v"(at), [size] "n"(8 * CH + 4), [cases] "n"(4 * G),
                   [g] "n"(G), [ch] "n"(CH)
                 : "vcc", "scc", "memory");
#undef BLPG_COL_STORE
#undef BLPG_ACC_HEAD
#undef BLPG_ACC_TAIL
}
// the kernel owns a[0 .. N)
template <int N>
__device__ __forceinline__ void acc_reserve() {
  static_assert(N == 32 || N == 64 || N == 128 || N == 160 || N == 176 || N == 208 || N == 224 || N == 256);
  if constexpr (N == 32) asm volatile("" ::: "a31");
  if constexpr (N == 64) asm volatile("" ::: "a63");
  if constexpr (N == 128) asm volatile("" ::: "a127");
  if constexpr (N == 160) asm volatile("" ::: "a159");
  if constexpr (N == 176) asm volatile("" ::: "a175");
  if constexpr (N == 208) asm volatile("" ::: "a207");
  if constexpr (N == 224) asm volatile("" ::: "a223");
  if constexpr (N == 256) asm volatile("" ::: "a255");
}

}  // namespace

enum : int { kEngDone = 0, kEngNoRow = 1 };

// IT: half tiles whose input loads are in flight together
template <int NW, int G, int CH, int IT>
struct WaveTab {
  using T = float;
  using KO = KeyOps<float>;
  static constexpr int NT = NW * 64;
  static constexpr int NG = NW * G;              // column groups of the LP
  static constexpr int RP = (CH + 3) / 4;        // row slots per lane (row form)
  static constexpr int RCAP = 16 * CH;           // constraint rows
  static constexpr int RB = 64 * RP;             // column buffer (row form reads)
  static constexpr int CB = 64 * NG;             // nonbasic columns
  static constexpr bool kBlockCrash = false;
  static constexpr bool kEngine = true;
  static constexpr int KB = 1;

  // Tile (ch, g): register 4b + i holds row 16 ch + 4 (lane / 16) + i, column
  // 64 (wv G + g) + 16 b + lane % 16 (both counted from 0).
  static constexpr int reg(int ch, int g, int b, int i) { return 16 * (ch * G + g) + 4 * b + i; }

  float row0[NG], row1[NG];  // objective rows, column form (every group, every wavefront)
  float lim[NG];   // a column may enter when its reduced cost is below lim: -eps_d, or
                   // -inf for a dead (or absent) column
  int nbv[NG];     // nonbasic variable of column 64 g + lane
  float rhs[RP];   // right-hand side, row form
  float acol[RP];  // the published column, row form
  float rcp[RP];   // 1 / acol
  int bsr[RP];     // basic variable, row form
  int redm;        // bit p: row lane + 64 p is redundant
  float z0, z1;    // right-hand sides of the objective rows
  float c0, c1;    // the published column's objective row entries
  int tid, lane, wv;
  int R, C, m, n;
  float neg_eps;
  int col_ready;   // column in acol, zeroed in the tiles (-1: none)
  int cph, rph;    // buffer phases
  float* colbuf;   // 2 x RB
  float* rowbuf;   // 2 x CB (NW > 1)
  uint8_t* target; // RCAP + CB + 2: warm-start targets
  int* wl;         // the warm-start list
  double* s_am;
  int blk;

  // Called once per state-machine step: per-thread indices and sizes become opaque values,
  // so the compiler does not hoist every stage's predicates out of the loop and hold them
  // in registers for the whole kernel.
  __device__ __forceinline__ void loop_fence() {
    asm volatile("" : "+v"(tid), "+v"(lane), "+s"(R), "+s"(C), "+s"(m), "+s"(n));
  }

  // ---- wave-uniform reads of distributed values ----
  template <typename U>
  __device__ __forceinline__ U slot(const U* a, int p, int cnt) const {
    // (the empty asm keeps the selection from becoming an indexed load, which would put
    // the array in scratch)
    U x = a[0];
    asm("" : "+v"(x));
#pragma unroll
    for (int u = 1; u < cnt; ++u) {
      U y = a[u];
      asm("" : "+v"(y));
      x = (u == p) ? y : x;
    }
    return x;
  }
  __device__ __forceinline__ float rowval(const float* a, int k) const { return rdlane(slot(a, k >> 6, RP), k & 63); }
  __device__ __forceinline__ int rowval(const int* a, int k) const {
    return __builtin_amdgcn_readlane(slot(a, k >> 6, RP), k & 63);
  }
  __device__ __forceinline__ float colval(const float* a, int c) const { return rdlane(slot(a, c >> 6, NG), c & 63); }
  __device__ __forceinline__ int colval(const int* a, int c) const {
    return __builtin_amdgcn_readlane(slot(a, c >> 6, NG), c & 63);
  }
  // index of the first set bit over the slots' ballots (slot first, then lane); -1: none
  template <int CNT, class P>
  __device__ __forceinline__ int first_of(P&& pred) const {
    int best = -1;
#pragma unroll
    for (int u = CNT - 1; u >= 0; --u) {
      const unsigned long long b = __ballot(pred(u));
      best = b != 0ull ? 64 * u + (__ffsll((long long)b) - 1) : best;
    }
    return uniform(best);
  }

  __device__ __forceinline__ void init(const double* A, const double* b, const double* c, const int8_t* sense) {
    double am = 0.0;
    const int q = lane >> 4, j = lane & 15;
    // IT half tiles' loads (16 rows x 32 columns each) go out together; entries outside the
    // LP are masked to +0.0 without branches: the loads are from clamped addresses
    constexpr int NH = 2 * CH * G;
    unroll<(NH + IT - 1) / IT>([&](auto uu) {
      constexpr int u0 = uu * IT, un = NH - u0 < IT ? NH - u0 : IT;
      __builtin_amdgcn_sched_barrier(0);
      double v[un][8];
      unroll<un>([&](auto w) {
        constexpr int h = u0 + w, ch = h / (2 * G), g = h / 2 % G, b0 = 2 * (h % 2);
        const int cb = 64 * (wv * G + g) + j;
        unroll<8>([&](auto e) {
          const int k = 16 * ch + 4 * q + e % 4, cj = cb + 16 * (b0 + e / 4);
          const unsigned off = (unsigned)((k < m ? k : m - 1) * n + (cj < n ? cj : n - 1));
          v[w][e] = A[off];
        });
      });
      unroll<un>([&](auto w) {
        constexpr int h = u0 + w, ch = h / (2 * G), g = h / 2 % G, b0 = 2 * (h % 2);
        const int cb = 64 * (wv * G + g) + j;
        unsigned rm[4], sg[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = 16 * ch + 4 * q + i, kc = k < m ? k : m - 1;
          rm[i] = (unsigned)((k - m) >> 31);
          sg[i] = sense != nullptr ? (sense[kc] == 2 ? 0x80000000u : 0u) : 0u;
        }
        unroll<8>([&](auto e) {
          constexpr int bb = b0 + e / 4, i = e % 4;
          const unsigned mk = rm[i] & (unsigned)((cb + 16 * bb - n) >> 31);
          const long long bits = __double_as_longlong(v[w][e]);
          const double x = __longlong_as_double(((long long)((unsigned)(bits >> 32) & mk) << 32) | ((unsigned)bits & mk));
          asm("v_max_f64 %0, %0, |%1|" : "+v"(am) : "v"(x));
          acc_set<reg(ch, g, bb, i)>(__uint_as_float(__float_as_uint((float)x) ^ (sg[i] & mk)));
        });
      });
    });
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int cj = 64 * g + lane;
      const float v = (float)(-c[cj < n ? cj : n - 1]);
      row0[g] = cj < n ? v : 0.0f;
      row1[g] = 0.0f;
      nbv[g] = cj < n ? cj : (cj == n ? n + m : -1);
      lim[g] = cj < n ? neg_eps : -inf_of<float>();
    }
    redm = 0;
    z0 = z1 = 0.0f;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int k = lane + 64 * p, kc = k < m ? k : m - 1;
      const double v = b[kc];
      const bool neg = sense != nullptr && sense[kc] == 2;
      rhs[p] = k < m ? (float)(neg ? -v : v) : 0.0f;
      bsr[p] = k < m ? n + k : -1;
      acol[p] = rcp[p] = 0.0f;
    }
    c0 = c1 = 0.0f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) am = fmax(am, __shfl_xor(am, off));
    if (lane == 0) s_am[wv] = am;
    col_ready = -1;
    if constexpr (NW > 1) __syncthreads();
  }

  __device__ __forceinline__ bool set_target(const int32_t* warm) {
    if (!warm) return false;
    for (int x = tid; x < RCAP + CB + 2; x += NT) target[x] = 0;
    __syncthreads();
    int any = 0;
    for (int i = tid; i < m; i += NT) {
      const int x = warm[i];
      wl[i] = x;
      if (x >= 0 && x < n + m) { target[x] = 1; any = 1; }
    }
    return __syncthreads_or(any) != 0;
  }

  __device__ __forceinline__ int warm_at(const int32_t*, int ci) const { return uniform(wl[ci]); }
  __device__ __forceinline__ int bs_now(int i) const { return rowval(bsr, i - 2); }
  __device__ __forceinline__ int bs_of(int i) const { return rowval(bsr, i - 2); }
  __device__ __forceinline__ int nb_of(int j) const { return colval(nbv, j - 1); }
  // tableau column of a nonbasic variable, -1 while it is basic
  __device__ __forceinline__ int find_nonbasic(int var) const {
    const int c = first_of<NG>([&](int g) { return nbv[g] == var; });
    return c < 0 ? -1 : c + 1;
  }
  __device__ __forceinline__ int find_basic(int var) const {
    const int k = first_of<RP>([&](int p) { return bsr[p] == var; });
    return k < 0 ? -1 : k + 2;
  }

  // The owner wavefront writes column s (tableau index) to LDS and, with ZERO, clears it in
  // the tiles; then every wavefront holds it in row form, with its reciprocals and its
  // objective row entries.  Two buffers: a wavefront writes one only after the barrier
  // behind every wavefront's reads of it.
  template <bool ZERO>
  __device__ __forceinline__ void publish_col(int s) {
    const int c = s - 1, go = c >> 6, ln = c & 63;
    cph ^= 1;
    float* cb = colbuf + cph * RB;
    if (NW == 1 || wv == go / G) {
      acc_col<CH, G, ZERO>(4 * (go - (NW == 1 ? 0 : wv * G)) + (ln >> 4), 0x0001000100010001ull << (ln & 15),
                           lds_addr(cb + 4 * (lane >> 4)));
    }
    c0 = colval(row0, c);
    c1 = colval(row1, c);
    if constexpr (NW > 1) __syncthreads();
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      // (the buffer holds 16 CH rows; beyond the LP's rows lanes hold 0, which no test takes)
      const float a = cb[lane + 64 * p];
      acol[p] = lane + 64 * p < m ? a : 0.0f;
    }
#pragma unroll
    for (int p = 0; p < RP; ++p) rcp[p] = 1.0f / acol[p];
    col_ready = ZERO ? s : -1;
  }

  // column s of the tiles from the column buffer (the column published last, or x0's)
  __device__ __forceinline__ void load_col(int s) {
    const int c = s - 1, go = c >> 6, ln = c & 63;
    const int q = lane >> 4;
    const float* cb = colbuf + cph * RB;
    const bool mine = (lane & 15) == (ln & 15);
    if (NW == 1 || wv == go / G) {
      acc_settle();
      dispatch<0, 4 * G>(4 * (go - (NW == 1 ? 0 : wv * G)) + (ln >> 4), [&](auto u) {
        constexpr int g = u / 4, bb = u % 4;
        if (mine)
          unroll<4 * CH>([&](auto e) { acc_set<reg(e / 4, g, bb, e % 4)>(cb[16 * (e / 4) + 4 * q + e % 4]); });
      });
    }
    col_ready = -1;
  }

  // Row k (constraint index) in column form: x = this wavefront's own groups.  With CLEAR
  // the row is set to -0.0 in the tiles.
  template <bool CLEAR>
  __device__ __forceinline__ void own_row(int k, float (&x)[G]) {
    const int q = (k >> 2) & 3;
    float y[4 * G];
    acc_row<CH, G, CLEAR>(4 * (k >> 4) + (k & 3), 0xFFFFull << (16 * q), -0.0f, y);
    // lanes 16q .. 16q+15 hold columns 16 bb + lane % 16 in y[bb]; group of lanes bb wants
    // its own block: a 4 x 4 exchange of 16-lane groups of which only block q is needed
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const auto e = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[4 * g + 0]), __float_as_uint(y[4 * g + 2]), false, false);
      const auto o = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[4 * g + 1]), __float_as_uint(y[4 * g + 3]), false, false);
      const unsigned ex = (q & 2) ? e[1] : e[0], ox = (q & 2) ? o[1] : o[0];
      const auto w = __builtin_amdgcn_permlane16_swap(ex, ox, false, false);
      x[g] = __uint_as_float((q & 1) ? w[1] : w[0]);
    }
  }
  // every group's part of row k: own groups in registers (NW = 1), else through LDS
  __device__ __forceinline__ void share_row(const float (&own)[G], float (&x)[NG]) {
    if constexpr (NW == 1) {
#pragma unroll
      for (int g = 0; g < G; ++g) x[g] = own[g];
    } else {
      rph ^= 1;
      float* rb = rowbuf + rph * CB;
#pragma unroll
      for (int g = 0; g < G; ++g) rb[64 * (wv * G + g) + lane] = own[g];
      __syncthreads();
#pragma unroll
      for (int g = 0; g < NG; ++g) x[g] = rb[64 * g + lane];
    }
  }

  // row of largest |T[i][s]| among constraint rows whose basic variable is not a target
  __device__ __forceinline__ int absmax_row(int s, float eps_p) {
    publish_col<false>(s);
    ArgMin<float> am;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int k = lane + 64 * p, x = bsr[p];
      const bool ok = k < m && !((redm >> p) & 1) && x >= 0 && !target[x < 0 ? 0 : x];
      am.add(ok, -tabs(acol[p]), k + 2, k + 2);
    }
    float bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    bp = uniform(bp);
    return (bp < 0 || !(uniform(-bv) > eps_p)) ? -1 : bp;
  }

  // Dantzig pricing on objective row orow: the most negative entry, lowest column on ties;
  // Bland: the smallest nonbasic id.
  __device__ __forceinline__ int price_end(const float (&d)[NG], float lv, float wmin) const {
    // (lv is this lane's minimum over its slots: a lane whose slot equals wmin holds it)
    (void)lv;
    const int c = first_of<NG>([&](int g) { return d[g] < lim[g] && d[g] == wmin; });
    return c < 0 ? -1 : c + 1;
  }
  __device__ __forceinline__ float price_key(const float (&d)[NG]) const {
    float lv = inf_of<float>();
#pragma unroll
    for (int g = 0; g < NG; ++g) lv = (d[g] < lim[g] && d[g] < lv) ? d[g] : lv;
    return lv;
  }
  __device__ __forceinline__ int pricing(int orow, bool bland, float) {
    float d[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) d[g] = orow == 0 ? row0[g] : row1[g];
    if (bland) {
#pragma unroll
      for (int g = 0; g < NG; ++g) d[g] = d[g] < lim[g] ? (float)nbv[g] : inf_of<float>();
      float lv = d[0];
#pragma unroll
      for (int g = 1; g < NG; ++g) lv = d[g] < lv ? d[g] : lv;
      const float wmin = wave_fmin(lv);
      if (!(wmin < inf_of<float>())) return -1;
      const int c = first_of<NG>([&](int g) { return d[g] == wmin; });
      return c + 1;
    }
    const float lv = price_key(d);
    return price_end(d, lv, wave_fmin(lv));
  }

  // Ratio test over the published column: smallest theta = max(beta, 0) / a over a > eps_p,
  // degenerate rows by the largest a; ties to the lowest row (Bland: smallest basic id).
  __device__ __forceinline__ int ratio(bool bland, float eps_p, float& theta) const {
    float key[RP];
    float lv = inf_of<float>();
    bool any[RP];
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const float a = acol[p];
      const bool ok = a > eps_p;
      const float th = (rhs[p] > 0.0f ? rhs[p] : 0.0f) / (ok ? a : 1.0f);
      key[p] = th > 0.0f ? th : -a;
      any[p] = ok;
      lv = (ok && key[p] < lv) ? key[p] : lv;
    }
    const float wmin = wave_fmin(lv);
    int k;
    if (bland) {
      ArgMin<float> am;
#pragma unroll
      for (int p = 0; p < RP; ++p) am.add(any[p], key[p], bsr[p], lane + 64 * p);
      float bv;
      int bk;
      wave_finish(am, bv, bk, k);
      k = uniform(k);
    } else {
      k = first_of<RP>([&](int p) { return any[p] && key[p] == wmin; });
    }
    theta = (k >= 0 && wmin > 0.0f) ? wmin : 0.0f;
    return k < 0 ? -1 : k + 2;
  }

  // Pivots.  Starts with the pivot (r, s), or with the ratio test of column s when r < 0;
  // with `fast` goes on -- pricing on objective row orow, ratio test, pivot -- until no
  // column prices out, the limit is reached, or Bland's rule sets in (kEngDone: the state
  // machine looks again), or no row passes the ratio test (kEngNoRow, column s unchanged).
  __device__ __forceinline__ int engine(int& r, int& s, bool fast, int orow, const Opt<float>& o,
                                        int maxit, bool keep_last, int& it, int& deg, int& last) {
    for (;;) {
      if (col_ready != s) publish_col<true>(s);
      if (r < 0) {
        float th;
        r = ratio(deg >= o.bland_after, o.eps_p, th);
        if (r < 0) {
          load_col(s);
          return kEngNoRow;
        }
        deg = (th == 0.0f) ? deg + 1 : 0;
      }
      const int k = r - 2, c = s - 1;
      // pivot row, scaled: prow (all groups), own (this wavefront's groups)
      float own[G], prow[NG];
      const float rp = rowval(rcp, k);
      own_row<true>(k, own);
      const int e = colval(nbv, c), lv = rowval(bsr, k);  // entering, leaving variable
      const float prow0 = rowval(rhs, k) * rp;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int gg = (NW == 1 ? 0 : wv * G) + g;
        own[g] = (64 * gg + lane == c) ? rp : own[g] * rp;
      }
      share_row(own, prow);
      // the column's multipliers: -T[i][s], and 1 for the pivot row (whose old entries are
      // -0.0, so the update leaves fma(1, prow, -0.0) = prow)
      float na[RP];
#pragma unroll
      for (int p = 0; p < RP; ++p) {
        const bool pr = lane + 64 * p == k;
        na[p] = pr ? 1.0f : -acol[p];
        rhs[p] = fma_t(na[p], prow0, pr ? -0.0f : rhs[p]);
        bsr[p] = pr ? e : bsr[p];
      }
      float d[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const bool pc = 64 * g + lane == c;
        row0[g] = fma_t(-c0, prow[g], pc ? 0.0f : row0[g]);
        row1[g] = fma_t(-c1, prow[g], pc ? 0.0f : row1[g]);
        nbv[g] = pc ? lv : nbv[g];
        d[g] = orow == 0 ? row0[g] : row1[g];
      }
      z0 = fma_t(-c0, prow0, z0);
      z1 = fma_t(-c1, prow0, z1);
      // tiles in the matrix pipe, the next column's pricing between them (a step of the
      // minimum after every few matrix instructions, which it would otherwise wait for).
      // Instructions issue in order, so what stands behind the last matrix instruction waits
      // for all of them.  With several wavefronts the bookkeeping and the end of the pricing
      // go in between: 205x203 per pivot 1.86 -> 1.83 us, 174x142 and 250x249 2% less too (with
      // one wavefront it changed nothing at 105x103 and cost 1% at 74x83).
      float pk = price_key(d);
      constexpr int NM = CH * G;
      static_assert(NW == 1 || NM >= 8);
      int sn = -1;
      acc_ready();
      unroll<NM>([&](auto u) {
        constexpr int ch = u / G, g = u % G;
        acc_rank1<reg(ch, g, 0, 0), ch % 4>(na[ch / 4], own[g]);
        // steps 0..5 spread over the first matrix instructions
        if constexpr (u < 6) {
          __builtin_amdgcn_sched_barrier(0);
          min_step<u < 6 ? (int)u : 0>(pk);
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NW > 1 && u == 6) {
#pragma unroll
          for (int p = 0; p < RP; ++p) asm volatile("" : "+v"(rhs[p]), "+v"(bsr[p]));
#pragma unroll
          for (int j = 0; j < NG; ++j) asm volatile("" : "+v"(row0[j]), "+v"(row1[j]), "+v"(nbv[j]));
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NW > 1 && u == 7) {
          sn = price_end(d, pk, rdlane(pk, 63));
          asm volatile("" ::"s"(sn));
          __builtin_amdgcn_sched_barrier(0);
        }
      });
      if constexpr (NM < 6) unroll<6>([&](auto u) { if constexpr (u >= NM) min_step<(int)u>(pk); });
      last = keep_last ? r | (s << 16) : -1;
      col_ready = -1;
      ++it;
      if (!fast || it >= maxit || deg >= o.bland_after) return kEngDone;
      if constexpr (NW == 1) sn = price_end(d, pk, rdlane(pk, 63));
      if (sn < 0) return kEngDone;
      s = sn;
      r = -1;
    }
  }

  // column of largest |T[r][j]| among live columns; -1 if all <= eps_p
  __device__ __forceinline__ int absmax_col(int r, float eps_p) {
    float own[G], x[NG];
    own_row<false>(r - 2, own);
    share_row(own, x);
    float lv = inf_of<float>();
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      x[g] = lim[g] > -inf_of<float>() ? -tabs(x[g]) : inf_of<float>();
      lv = x[g] < lv ? x[g] : lv;
    }
    const float wmin = wave_fmin(lv);
    if (!(-wmin > eps_p)) return -1;
    return first_of<NG>([&](int g) { return x[g] == wmin; }) + 1;
  }

  // dual simplex leaving row: most negative rhs below -tol (Bland: smallest basic id)
  __device__ __forceinline__ int dual_row(bool bland, float tol) {
    ArgMin<float> am;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int k = lane + 64 * p;
      am.add(k < m && !((redm >> p) & 1) && rhs[p] < -tol, bland ? (float)bsr[p] : rhs[p], k + 2, k + 2);
    }
    float bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    return uniform(bp);
  }

  // dual simplex entering column for leaving row r: smallest max(T[0][j],0)/-T[r][j] over
  // T[r][j] < -eps_p (dual-degenerate columns by the largest |T[r][j]|)
  __device__ __forceinline__ int dual_ratio(int r, bool bland, float eps_p, float& theta) {
    float own[G], x[NG];
    own_row<false>(r - 2, own);
    share_row(own, x);
    ArgMin<float> am;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = 1 + 64 * g + lane;
      const float a = x[g], d = row0[g];
      const bool ok = lim[g] > -inf_of<float>() && a < -eps_p;
      const float th = (d > 0.0f ? d : 0.0f) / (ok ? -a : 1.0f);
      const float key = th > 0.0f ? th : a;
      am.add(ok, key, bland ? nbv[g] : j, j);
    }
    float bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    bv = uniform(bv);
    theta = bv > 0.0f ? bv : 0.0f;
    return uniform(bp);
  }

  __device__ __forceinline__ void kill_col(int j) {
#pragma unroll
    for (int g = 0; g < NG; ++g) lim[g] = (64 * g + lane == j - 1) ? -inf_of<float>() : lim[g];
  }

  // only the right-hand side (column 0) is read and written this way by the driver
  __device__ __forceinline__ float get(int i, int) const { return i == 1 ? z1 : rowval(rhs, i - 2); }
  __device__ __forceinline__ void set(int i, int, float val) {
#pragma unroll
    for (int p = 0; p < RP; ++p) rhs[p] = (lane + 64 * p == i - 2) ? val : rhs[p];
  }
  __device__ __forceinline__ void mark_redund(int r) {
#pragma unroll
    for (int p = 0; p < RP; ++p) redm |= (lane + 64 * p == r - 2) ? 1 << p : 0;
    set(r, 0, 0.0f);
  }

  __device__ __forceinline__ int min_rhs_row() {
    float lv = inf_of<float>();
    bool in[RP];
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      in[p] = lane + 64 * p < m && !((redm >> p) & 1);
      lv = (in[p] && rhs[p] < lv) ? rhs[p] : lv;
    }
    const float wmin = wave_fmin(lv);
    const int k = first_of<RP>([&](int p) { return in[p] && rhs[p] == wmin; });
    return k < 0 ? -1 : k + 2;
  }

  // auxiliary column x0 (column C-1): -1 on live constraint rows, 1 on the phase-I row;
  // the phase-I row is 0 elsewhere (its rhs included)
  __device__ __forceinline__ void setup_x0() {
    const int x0 = C - 2;  // counted from 0
    if constexpr (NW > 1) __syncthreads();
    float* cb = colbuf + cph * RB;
    if (wv == 0) {
#pragma unroll
      for (int p = 0; p < RP; ++p) {
        const int k = lane + 64 * p;
        cb[k] = (k < m && !((redm >> p) & 1)) ? -1.0f : 0.0f;
      }
    }
    if constexpr (NW > 1) __syncthreads();
    load_col(x0 + 1);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const bool is = 64 * g + lane == x0;
      row0[g] = is ? 0.0f : row0[g];
      row1[g] = is ? 1.0f : 0.0f;
      lim[g] = is ? neg_eps : lim[g];
    }
    z1 = 0.0f;
  }

  // block crash entry points (unused: kBlockCrash is false)
  __device__ __forceinline__ int blk_word(int) const { return 0; }
  __device__ __forceinline__ int crash_prepare(int&, const int8_t*, float) { return -1; }
  __device__ __forceinline__ void pivot(int, int) {}

  __device__ __forceinline__ void write_outputs(int lp, const LpDesc& d, const Out& out, int status, int it,
                                                int p1, int unb, float wfin, int last) {
    double* x = out.x + d.x;
    int32_t* basis = out.basis + d.basis;
    for (int j = tid; j < n; j += NT) x[j] = 0.0;
    if (tid == 0) {
      double am = s_am[0];
      for (int w = 1; w < NW; ++w) am = fmax(am, s_am[w]);
      out.amax[lp] = am;
      out.status[lp] = status;
      out.pivots[lp] = it;
      out.p1[lp] = p1;
      out.unb[lp] = unb;
      if (out.lastpiv) out.lastpiv[lp] = last;
      out.obj[lp] = (double)z0;
      out.wfin[lp] = (double)wfin;
    }
    __syncthreads();
    if (wv == 0) {
#pragma unroll
      for (int p = 0; p < RP; ++p) {
        const int k = lane + 64 * p;
        if (k < m) {
          basis[k] = bsr[p];
          if (bsr[p] >= 0 && bsr[p] < n) x[bsr[p]] = (double)rhs[p];
        }
      }
    }
    // final tableau and nonbasic ids for the FP64 check (B^-1 is in the slack columns)
    if (out.tab) {
      float* tp = (float*)(out.tab + 8 * d.t);
      int32_t* np = (int32_t*)(out.tab + 8 * (d.t + (int64_t)R * C));
      if (wv == 0) {
        if (lane == 0) {
          tp[0] = z0;
          tp[C] = z1;
          np[0] = -1;
        }
#pragma unroll
        for (int p = 0; p < RP; ++p) {
          const int k = lane + 64 * p;
          if (k < m) tp[(int64_t)(k + 2) * C] = rhs[p];
        }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          const int j = 1 + 64 * g + lane;
          if (j < C) {
            tp[j] = row0[g];
            tp[C + j] = row1[g];
            np[j] = nbv[g];
          }
        }
      }
      const int q = lane >> 4;
      acc_settle();
      unroll<CH * G>([&](auto u) {
        constexpr int ch = u / G, g = u % G;
        const int j = 1 + 64 * (wv * G + g) + (lane & 15);
        unroll<4>([&](auto i) {
          const int k = 16 * ch + 4 * q + i;
          float* tk = tp + (int64_t)(k + 2) * C + j;
          unroll<4>([&](auto bb) {
            const float v = acc_get<reg(ch, g, bb, i)>();
            if (k < m && j + 16 * bb < C) tk[16 * bb] = v;
          });
        });
      });
    }
  }
};

template <int NW, int G, int CH, int IT>
__device__ __forceinline__ void wave_body(const LpDesc* __restrict__ desc, const double* __restrict__ pool,
                                          const int8_t* __restrict__ spool, const int32_t* __restrict__ idx,
                                          int32_t count, const int32_t* count_dev, int32_t* queue,
                                          const Out& out, const Opt<float>& o,
                                          const int32_t* __restrict__ warm_pool) {
  using Tab = WaveTab<NW, G, CH, IT>;
  __shared__ __align__(64) float colbuf[2 * Tab::RB];
  __shared__ float rowbuf[NW > 1 ? 2 * Tab::CB : 1];
  __shared__ uint8_t target[Tab::RCAP + Tab::CB + 2];
  __shared__ int wl[Tab::RCAP];
  __shared__ double s_am[NW];
  __shared__ int s_q;
  Tab t;
  t.s_am = s_am;
  t.tid = threadIdx.x;
  t.lane = threadIdx.x & 63;
  t.wv = uniform((int)(threadIdx.x >> 6));
  t.cph = t.rph = 0;
  t.colbuf = colbuf;
  t.rowbuf = rowbuf;
  t.target = target;
  t.wl = wl;
  t.blk = -1;
  t.neg_eps = -o.eps_d;
  acc_reserve<16 * CH * G>();
  if (count_dev) count = *count_dev;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_q = atomicAdd(queue, 1);
    __syncthreads();
    const int q = uniform(s_q);
    if (q >= count) break;
    const int lp = idx ? idx[q] : q;
    const LpDesc d = desc[lp];
    t.m = d.m; t.n = d.n; t.R = d.m + 2; t.C = d.n + 2;
    const int8_t* sense = d.s >= 0 ? spool + d.s : nullptr;
    t.init(pool + d.a, pool + d.b, pool + d.c, sense);
    const int32_t* warm = warm_pool ? warm_pool + d.basis : nullptr;
    if (!t.set_target(warm)) warm = nullptr;
    int status, it, p1, unb, last;
    float wfin;
    run_simplex<float>(t, d.m, d.n, sense, o, status, it, p1, unb, wfin, last, warm);
    t.write_outputs(lp, d, out, status, it, p1, unb, wfin, last);
  }
}

// ---------------------------------------------------------------------------------
// variant table: (waves per LP, column groups per wave, row chunks of 16, half tiles loaded
// together, vector registers left to the compiler); holds 16 ch constraint rows and 64 nw g
// nonbasic columns (the auxiliary x0 among them).  FP32 only.  vr + 16 ch g registers per lane
// set the residency: 128 for four waves per SIMD, 256 for two.
//   id nw g  ch it vr
#define BLPG_WAVE_VARIANTS(X) \
  X(0, 1, 1, 2, 2, 84)        \
  X(1, 1, 1, 4, 1, 64)        \
  X(2, 1, 2, 4, 3, 128)       \
  X(3, 1, 2, 5, 2, 96)        \
  X(4, 1, 2, 7, 8, 248)       \
  X(5, 3, 1, 11, 2, 80)       \
  X(6, 4, 1, 13, 7, 248)      \
  X(7, 4, 1, 16, 7, 248)

// (the attribute takes literals only; with accumulation registers in use the compiler takes
// the number it is given for its vector registers)
#define X(id, nw, g, ch, it, vr)                                                                \
  __global__ __launch_bounds__(nw * 64) __attribute__((amdgpu_num_vgpr(vr))) void k_wave_##id(  \
      const LpDesc* __restrict__ desc, const double* __restrict__ pool,                         \
      const int8_t* __restrict__ spool, const int32_t* __restrict__ idx, int32_t count,         \
      const int32_t* count_dev, int32_t* queue, Out out, Opt<float> o,                          \
      const int32_t* __restrict__ warm_pool) {                                                  \
    wave_body<nw, g, ch, it>(desc, pool, spool, idx, count, count_dev, queue, out, o, warm_pool); \
  }
BLPG_WAVE_VARIANTS(X)
#undef X

constexpr int kWaveVariants = 8;
// Variant 0 is accepted in FP64 too (32 rows x 65 columns): the smallest 2-D block that holds
// it runs it, faster than columns per lane did (27x32 x 1024: 0.109 ms against 0.113).
constexpr int kWave64Tile = 2;

int wave_variant_count() { return kWaveVariants; }

WaveVariant wave_variant(int precision, int v) {
  if (precision == 0) return v == 0 ? WaveVariant{1, 1, 32, true} : WaveVariant{1, 1, 0, false};
  switch (v) {
#define X(id, nw, g, ch, it, vr) \
  case id: return WaveVariant{nw, g, 16 * ch + 2, true};
    BLPG_WAVE_VARIANTS(X)
#undef X
    default: return WaveVariant{1, 1, 0, false};
  }
}

static const void* wave_fn(int v) {
  switch (v) {
#define X(id, nw, g, ch, it, vr) \
  case id: return reinterpret_cast<const void*>(&k_wave_##id);
    BLPG_WAVE_VARIANTS(X)
#undef X
    default: return nullptr;
  }
}

int wave_max_blocks_per_cu(int precision, int v) {
  if (precision == 0) return v == 0 ? tile_max_blocks_per_cu(0, kWave64Tile) : 0;
  const void* fn = wave_fn(v);
  if (!fn) return 0;
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, wave_variant(precision, v).nw * 64, 0) !=
      hipSuccess)
    return 0;
  return nb;
}

hipError_t launch_wave(const TileLaunch& L, hipStream_t st) {
  if (L.precision == 0) {
    if (L.variant != 0) return hipErrorInvalidValue;
    TileLaunch T = L;
    T.variant = kWave64Tile;
    return launch_tile(T, st);
  }
  const void* fn = wave_fn(L.variant);
  if (!fn) return hipErrorInvalidValue;
  const int nt = wave_variant(L.precision, L.variant).nw * 64;
  Opt<float> o{(float)L.eps_d, (float)L.eps_p, (float)L.tol, L.max_iter, L.bland_after};
  void* args[] = {(void*)&L.desc, (void*)&L.pool, (void*)&L.spool, (void*)&L.idx,
                  (void*)&L.count, (void*)&L.count_dev, (void*)&L.queue, (void*)&L.out,
                  (void*)&o, (void*)&L.warm};
  return hipLaunchKernel(fn, dim3(L.grid), dim3(nt), args, 0, st);
}

}  // namespace blpg
