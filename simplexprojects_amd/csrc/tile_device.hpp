// tile_device.hpp -- register-resident simplex kernel for gfx950, 2-D blocks per thread
// (instantiated by kernel_tile.hip in FP32 and kernel_tile64.hip in FP64).
//
// One workgroup (NW wavefronts) per LP, persistent over a work queue.  The condensed
// tableau never leaves the vector register file: thread t = gc + TC*gr owns rows
// gr + TR*k (k < RPT) and columns gc + TC*l (l < CPT), an RPT x CPT block.  A CU's 512 KB of
// VGPRs is 3.2x its LDS, so tableaux up to ~207x205 FP64 stay on-chip, and the rank-1 update
// is RPT*CPT register FMAs per thread with no memory traffic at all.
//
// The block lives in registers that only inline assembly names, v[NV ..): the kernel's
// amdgpu_num_vgpr attribute keeps the compiler to v[0 .. NV).  As a C++ array the block was
// live through every branch of the state machine, and the compiler held two copies of it
// (242 VGPRs for 98 of block, 552 bytes of scratch per lane for the 7 x 13 FP64 block).
// What the compiler still spills of its own values, FP64: 45 registers with the 7 x 13 block,
// 22 with 14 x 7, 62 with 11 x 9 (of the scratch accesses 1, 1 and 15 stand in the pivot loop,
// the others in the stages around it), at most 10 elsewhere; FP32: 6 with 7 x 13.
//
// What the decisions need is replicated in every wavefront, in two forms: row form (lane l
// holds rows l + 64 p: basic ids, the published column) and column form (lane l holds
// columns l + 64 g: nonbasic ids, the objective row in use).  Every wavefront makes the same
// pricing and ratio test, so a pivot has two barriers and no broadcast:
//   column  the TR owners of column s write it to LDS and zero it in their blocks -- barrier
//   ratio   theta over the rows, minimum by DPP, ballot: r is wave-uniform
//   row     the TC owners of row r write it to LDS and set it to -0.0 -- barrier
//   update  block += column (x) (row / -p) with multiplier -1 for row r, whose -0.0 entries
//           become the scaled row exactly; the objective row is updated in column form
//           too, so the next pricing runs beside the FMAs instead of after them
// The pivot row's entry at column s is published as 1, which scales to the reciprocal; the
// column is published twice, the second time with -1 at row r.  So neither the scaling nor
// the update selects anything per element.
//
// What bounds it is the chain of one pivot (two LDS round trips and barriers, an FP64
// division, two reductions).  FP64, one LP alone, per pivot: 0.97 us at 27x32, 1.53 at
// 105x103, 2.13 at 174x142, 2.61 at 205x203; with every reduction on one wavefront and its
// result broadcast (four barriers), and the block as a C++ array, 105x103 took 3.26, 174x142
// 3.83 and 205x203 24.3 (spilled).  1024 LPs of 105x103 took 2.27 ms, now 1.05 on four
// wavefronts each and 0.80 on two (the instance for many LPs).  Of 4000
// cycles at 105x103 the column's way through LDS takes 880, the ratio test 970, the row 140,
// the reciprocal and the second barrier 650, pricing 670 and the update 700.
//
// Arithmetic and rule are those of kernel_stream.hip and the oracle, operation for
// operation: results are bit-identical across kernels.  Replaces the reference's
// mykernel (simplex.cu:35-385), whose tableau lives in global memory.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "kernels.hpp"
#include "simplex_device.hpp"

namespace blpg {

// ---- the block's registers: element E (32-bit words: 1 or 2 per element) is in
//      v[NV + words E], or, for blocks beyond the 256 vector registers, in a[NV ..): with
//      accumulation registers in use the attribute keeps the compiler to a[0 .. NV) too ----
template <typename T, int NV, int E>
struct Reg {
  static constexpr int W = (int)sizeof(T) / 4;
  static constexpr int FIT = (256 - NV) / W;  // elements in vector registers
  static constexpr bool acc = E >= FIT;
  static constexpr int N = NV + W * (acc ? E - FIT : E);
};
template <typename T, int NV, int E>
__device__ __forceinline__ T blk_get() {
  using G = Reg<T, NV, E>;
  T x;
  if constexpr (G::W == 1) {
    if constexpr (G::acc) asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(G::N));
    else asm volatile("v_mov_b32 %0, v[%1]" : "=v"(x) : "n"(G::N));
  } else if constexpr (G::acc) {
    unsigned lo, hi;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(lo) : "n"(G::N));
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(hi) : "n"(G::N + 1));
    x = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
  } else {
    asm volatile("v_mov_b64 %0, v[%1:%2]" : "=v"(x) : "n"(G::N), "n"(G::N + 1));
  }
  return x;
}
template <typename T, int NV, int E>
__device__ __forceinline__ void blk_set(T x) {
  using G = Reg<T, NV, E>;
  if constexpr (G::W == 1) {
    if constexpr (G::acc) asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x), "n"(G::N));
    else asm volatile("v_mov_b32 v[%1], %0" ::"v"(x), "n"(G::N));
  } else if constexpr (G::acc) {
    const unsigned long long w = (unsigned long long)__double_as_longlong(x);
    asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"((unsigned)w), "n"(G::N));
    asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"((unsigned)(w >> 32)), "n"(G::N + 1));
  } else {
    asm volatile("v_mov_b64 v[%1:%2], %0" ::"v"(x), "n"(G::N), "n"(G::N + 1));
  }
}
// element += a * b, one rounding
template <typename T, int NV, int E>
__device__ __forceinline__ void blk_fma(T a, T b) {
  using G = Reg<T, NV, E>;
  if constexpr (G::acc) blk_set<T, NV, E>(fma_t(a, b, blk_get<T, NV, E>()));
  else if constexpr (G::W == 1) asm volatile("v_fmac_f32 v[%2], %0, %1" ::"v"(a), "v"(b), "n"(G::N));
  else asm volatile("v_fmac_f64 v[%2:%3], %0, %1" ::"v"(a), "v"(b), "n"(G::N), "n"(G::N + 1));
}

// Column l (row k) of a thread's block, CNT elements STEP apart in the registers, straight
// to LDS at a0 (and a1, with TWO), OFF elements apart there; then the registers are set to z.
// A register number cannot be dynamic, so the wave-uniform index x jumps into a table of
// CASES equal-sized entries (clamped, so that it stays inside for any value), the first
// elements NEXT apart: a tree of scalar branches, with a copy and a store per element in its
// leaves, cost 200 cycles more for the column and as many for the row.  Pairs of elements share an instruction.  The caller waits for the stores (LDS
// instructions in assembly are not the compiler's to count).
template <typename T, int NV, int CASES, int CNT, int STEP, int NEXT, int OFF, bool TWO>
__device__ __forceinline__ void blk_out(int x, unsigned a0, unsigned a1, T z) {
  constexpr int W = (int)sizeof(T) / 4;
  static_assert((CNT - 1) * OFF < 256, "offset0 and offset1 are eight bits");
  constexpr int size = ((CNT + 1) / 2 * (TWO ? 2 : 1)) * 8 + 4 + CNT * 4 + 4;
  int t;
#define BLPG_OUT(ds2, ds1, mov, hi0, hi1)                                                   \
  asm volatile(                                                                             \
      "s_min_u32 %[t], %[x], %[cases] - 1\n\t"                                              \
      "s_mul_i32 %[t], %[t], %[size]\n\t"                                                   \
      "s_add_u32 %[t], %[t], 12\n\t"                                                        \
      "s_getpc_b64 vcc\n\t"                                                                 \
      "s_add_u32 vcc_lo, vcc_lo, %[t]\n\t"                                                  \
      "s_addc_u32 vcc_hi, vcc_hi, 0\n\t"                                                    \
      "s_setpc_b64 vcc\n\t"                                                                 \
      ".set blpg_c, %[nv]\n\t"                                                              \
      ".rept %[cases]\n\t"                                                                  \
      ".set blpg_a, blpg_c\n\t"                                                             \
      ".set blpg_o, 0\n\t"                                                                  \
      ".rept %[cnt] / 2\n\t"                                                                \
      ds2 " %[a0], v[blpg_a" hi0 "], v[" hi1 "] offset0:blpg_o offset1:blpg_o + %[off]\n\t" \
      ".if %[two]\n\t"                                                                      \
      ds2 " %[a1], v[blpg_a" hi0 "], v[" hi1 "] offset0:blpg_o offset1:blpg_o + %[off]\n\t" \
      ".endif\n\t"                                                                          \
      ".set blpg_a, blpg_a + 2 * %[step]\n\t"                                               \
      ".set blpg_o, blpg_o + 2 * %[off]\n\t"                                                \
      ".endr\n\t"                                                                           \
      ".if %[cnt] & 1\n\t"                                                                  \
      ds1 " %[a0], v[blpg_a" hi0 "] offset:%[bytes] * blpg_o\n\t"                           \
      ".if %[two]\n\t"                                                                      \
      ds1 " %[a1], v[blpg_a" hi0 "] offset:%[bytes] * blpg_o\n\t"                           \
      ".endif\n\t"                                                                          \
      ".endif\n\t"                                                                          \
      "s_nop 1\n\t"                                                                         \
      ".set blpg_a, blpg_c\n\t"                                                             \
      ".rept %[cnt]\n\t"                                                                    \
      mov " v[blpg_a" hi0 "], %[z]\n\t"                                                     \
      ".set blpg_a, blpg_a + %[step]\n\t"                                                   \
      ".endr\n\t"                                                                           \
      "s_branch Lout%=\n\t"                                                                 \
      ".set blpg_c, blpg_c + %[next]\n\t"                                                   \
      ".endr\n"                                                                             \
      "Lout%=:"                                                                             \
      : [t] "=&s"(t)                                                                        \
      : [x] "s"(x), [a0] "v"(a0), [a1] "v"(a1), [z] "v"(z), [nv] "n"(NV), [cases] "n"(CASES), \
        [cnt] "n"(CNT), [step] "n"(W * STEP), [next] "n"(W * NEXT), [off] "n"(OFF),         \
        [two] "n"(TWO ? 1 : 0), [size] "n"(size), [bytes] "n"(4 * W)                        \
      : "vcc", "scc", "memory")
  if constexpr (W == 2) BLPG_OUT("ds_write2_b64", "ds_write_b64", "v_mov_b64", ":blpg_a + 1", "blpg_a + %[step]:blpg_a + %[step] + 1");
  else BLPG_OUT("ds_write2_b32", "ds_write_b32", "v_mov_b32", "", "blpg_a + %[step]");
#undef BLPG_OUT
}
// the LDS address of a pointer into LDS, and the wait for blk_out's stores
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(size_t)(__attribute__((address_space(3))) const char*)p;
}
__device__ __forceinline__ void lds_settle() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

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
// binary tree of scalar branches, so that register numbers inside f stay static.
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

// lane l's value (l wave-uniform)
__device__ __forceinline__ float lane_read(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
__device__ __forceinline__ double lane_read(double x, int l) {
  const long long v = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ int lane_read(int x, int l) { return __builtin_amdgcn_readlane(x, l); }

// Minimum of a 32-bit integer over the 64 lanes: v_min with a DPP source per step (s_nop 1:
// the two wait states a DPP read needs after the write), rows outside a step's row mask keep
// their value; lane 63 ends with the minimum.
#define BLPG_DPP_MIN(op)                                                                   \
  "s_nop 1\n\t" op " %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"         \
  "s_nop 1\n\t" op " %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"         \
  "s_nop 1\n\t" op " %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"             \
  "s_nop 1\n\t" op " %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"                  \
  "s_nop 1\n\t" op " %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"                \
  "s_nop 1\n\t" op " %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"                \
  "s_nop 1"
__device__ __forceinline__ int wave_min_i32(int x) {
  asm(BLPG_DPP_MIN("v_min_i32_dpp") : "+v"(x));
  return __builtin_amdgcn_readlane(x, 63);
}
__device__ __forceinline__ unsigned wave_min_u32(unsigned x) {
  asm(BLPG_DPP_MIN("v_min_u32_dpp") : "+v"(x));
  return (unsigned)__builtin_amdgcn_readlane((int)x, 63);
}
__device__ __forceinline__ float wave_min_f32(float x) {
  asm(BLPG_DPP_MIN("v_min_f32_dpp") : "+v"(x));
  return lane_read(x, 63);
}
#undef BLPG_DPP_MIN

// index of the first set bit over the slots' ballots (slot first, then lane); -1: none
template <int CNT, class P>
__device__ __forceinline__ int first_of(P&& pred) {
  int best = -1;
#pragma unroll
  for (int u = CNT - 1; u >= 0; --u) {
    const unsigned long long b = __ballot(pred(u));
    best = b != 0ull ? 64 * u + (__ffsll((long long)b) - 1) : best;
  }
  return uniform(best);
}

// Lowest index (slot first, then lane) of the smallest key among the lanes' CNT slots with
// ok; -1 when there is none.  Keys are never NaN or zero.  neg: the smallest key is negative.
// FP32: the minimum itself, then who holds it.  FP64: the minimum of the keys' high words
// (as integers in the keys' order); only when several slots share it, of their low words.
template <int CNT>
__device__ __forceinline__ int arg_min(const float (&key)[CNT], const bool (&ok)[CNT], bool& neg) {
  float lv = inf_of<float>();
#pragma unroll
  for (int u = 0; u < CNT; ++u) lv = (ok[u] && key[u] < lv) ? key[u] : lv;
  const float w = wave_min_f32(lv);
  neg = w < 0.0f;
  return first_of<CNT>([&](int u) { return ok[u] && key[u] == w; });
}
template <int CNT>
__device__ __forceinline__ int arg_min(const double (&key)[CNT], const bool (&ok)[CNT], bool& neg) {
  int kh[CNT], lv = INT_MAX;
#pragma unroll
  for (int u = 0; u < CNT; ++u) {
    const int hi = (int)((unsigned long long)__double_as_longlong(key[u]) >> 32);
    kh[u] = ok[u] ? hi ^ ((hi >> 31) & 0x7FFFFFFF) : INT_MAX;
    lv = kh[u] < lv ? kh[u] : lv;
  }
  const int w = wave_min_i32(lv);
  neg = w < 0;
  int cnt = 0, best = -1;
#pragma unroll
  for (int u = CNT - 1; u >= 0; --u) {
    const unsigned long long b = __ballot(ok[u] && kh[u] == w);
    cnt += __popcll(b);
    best = b != 0ull ? 64 * u + (__ffsll((long long)b) - 1) : best;
  }
  if (uniform(cnt) > 1) {
    unsigned kl[CNT], ll = ~0u;
#pragma unroll
    for (int u = 0; u < CNT; ++u) {
      const unsigned lo = (unsigned)__double_as_longlong(key[u]);
      kl[u] = (ok[u] && kh[u] == w) ? lo ^ (unsigned)(w >> 31) : ~0u;
      ll = kl[u] < ll ? kl[u] : ll;
    }
    const unsigned wl = wave_min_u32(ll);
    best = first_of<CNT>([&](int u) { return ok[u] && kh[u] == w && kl[u] == wl; });
  }
  return uniform(best);
}

// BC: crash in blocks (crash_prepare).  Instantiated only for batches with warm lists, and
// only where its registers do not spill the tile; cold solves run the BC = false kernel.
template <typename T, int NW, int TC, int RPT, int CPT, bool BC, int NV>
struct TileTab {
  static constexpr int NT = NW * 64;
  static constexpr int TR = NT / TC;
  static constexpr int RCAP = TR * RPT;
  static constexpr int CCAP = TC * CPT;
  static constexpr int RP = (RCAP + 63) / 64, RB = 64 * RP;  // row form
  static constexpr int NG = (CCAP + 63) / 64, CB = 64 * NG;  // column form
  static_assert(TC <= 32 && 64 % TC == 0, "whole rows of threads per wavefront");
  static constexpr bool kEngine = true;
  // part of the block lies in accumulation registers (which blk_out does not address)
  static constexpr bool kAcc = NV + (int)sizeof(T) / 4 * RPT * CPT > 256;

  static constexpr int el(int k, int l) { return k * CPT + l; }
  T orw[NG];      // objective row orow_in, column form (kept by engine; -1: not loaded)
  int orow_in;
  int bsr[RP];    // basic variable, row form
  int nbv[NG];    // nonbasic variable, column form
  int dm;         // bit g: column lane + 64 g cannot enter
  int redm;       // bit p: row lane + 64 p is redundant
  int gr, gc, tid, lane, wv;
  int R, C, m, n;
  int col_ready;  // column published and zeroed (-1: none)
  int cph, rph;   // buffer phases
  T* colbuf;      // 2 x RB: published column, read in row form
  T* colupd;      // 2 x RB: the update's multipliers (the column, -1 at the pivot row)
  T* rhsbuf;      // RB: right-hand side, rewritten by its owners after every update
  T* rowbuf;      // 2 x CB: published row
  int* bs;        // BC: basic / nonbasic variables and the column of each nonbasic variable,
  int* nb;        //     kept during the crash stage only
  int* colof;
  uint8_t* redund;
  uint8_t* target;  // target[var] = 1: var belongs to the warm-start basis
  int* wl;          // the warm-start list (m entries), read by the crash in order
  double* s_am;     // per-wave max |A_ij| (NW entries)

  // Block crash: KB targets per block.  Their columns and pivot rows take at most 16 KB
  // of LDS, and wavefront 0 / each column thread holds KB values per row / column in
  // registers during the block's preparation (more than 8 spills the tile).
  static constexpr int KB0 = 16384 / ((RCAP + CCAP) * (int)sizeof(T));
  static constexpr int KB = !BC ? 1 : KB0 < 4 ? 4 : (KB0 > 8 ? 8 : KB0);
  static constexpr bool kBlockCrash = BC;
  static constexpr int QR = (RCAP + 63) / 64;  // rows per lane of wavefront 0
  T* cbM;    // KB x RCAP: column of target u, updated until its own step, then its negative (1 at its
             // pivot row)
  T* cbP;    // KB x CCAP: row of pivot u, updated until its own step, then scaled
  T* cbRp;   // KB: 1 / pivot element of step u
  int* cbR;  // KB + 3: pivot row of step u (-1: none); [KB] steps, [KB + 1] next ci,
             // [KB + 2] pivots made
  int* cbS;  // KB: column of target u
  int* cbW;  // KB: the block's pivots in order, packed: row | column << 12 | slot << 24 |
             // (leaving variable is an equality slack) << 30
  int blk;   // >= 0: the next pivot is the crash block's step in this slot

  // Called once per state-machine step: the per-thread indices become opaque values, so
  // the compiler recomputes index arithmetic where it is used instead of hoisting every
  // stage's invariants out of the loop (which holds registers for the whole kernel and
  // costs a wave per SIMD of occupancy).
  __device__ __forceinline__ void loop_fence() { asm volatile("" : "+v"(gr), "+v"(gc), "+v"(tid), "+v"(lane), "+s"(R), "+s"(C), "+s"(m), "+s"(n)); }

  __device__ __forceinline__ int row_of(int k) const { return gr + TR * k; }
  __device__ __forceinline__ int col_of(int l) const { return gc + TC * l; }

  template <int E>
  __device__ __forceinline__ static T get_el() { return blk_get<T, NV, E>(); }
  template <int E>
  __device__ __forceinline__ static void set_el(T x) { blk_set<T, NV, E>(x); }

  // ---- wave-uniform reads of distributed values (the empty asm keeps the selection from
  //      becoming an indexed load, which would put the array in scratch) ----
  template <int CNT, typename U>
  static __device__ __forceinline__ U pick(const U (&a)[CNT], int i) {
    U x = a[0];
    asm("" : "+v"(x));
#pragma unroll
    for (int u = 1; u < CNT; ++u) {
      U y = a[u];
      asm("" : "+v"(y));
      x = (u == (i >> 6)) ? y : x;
    }
    return lane_read(x, i & 63);
  }

  __device__ __forceinline__ void publish_rhs() {
    if (gc == 0) {
      unroll<RPT>([&](auto k) { rhsbuf[row_of(k)] = get_el<el(k, 0)>(); });
    }
  }

  // Loads the condensed tableau (row 0: -c, row 1: 0, rows 2..: A and b with '>=' rows
  // negated) and max |A_ij|.  Every thread loads each of its entries from a valid address of
  // A (clamped), so the loads are unconditional and go out together; what is not A is masked
  // to 0 and the objective row and the right-hand side are loaded over it.
  __device__ __forceinline__ void init(const double* A, const double* b, const double* c, const int8_t* sense) {
    double am = 0.0;
    unroll<RPT>([&](auto k) {
      const int i = row_of(k) - 2, r = i < 0 ? 0 : i < m ? i : m - 1;
      const unsigned ro = (unsigned)(r * n);
      const unsigned sg = sense != nullptr && sense[r] == 2 ? 0x80000000u : 0u;
      const unsigned rm = (i >= 0 && i < m) ? ~0u : 0u;
      constexpr int NP = (CPT + 8) / 9, PG = (CPT + NP - 1) / NP;
      unroll<NP>([&](auto w) {
        constexpr int l0 = w * PG, ln = CPT - l0 < PG ? CPT - l0 : PG;
        double x[ln];
#pragma unroll
        for (int l = 0; l < ln; ++l) {
          const int j = col_of(l0 + l) - 1;
          x[l] = A[ro + (unsigned)(j < 0 ? 0 : j < n ? j : n - 1)];
        }
        unroll<ln>([&](auto l) {
          const int j = col_of(l0 + l) - 1;
          const unsigned mk = (j >= 0 && j < n) ? rm : 0u;
          const unsigned long long u = (unsigned long long)__double_as_longlong(x[l]);
          const unsigned hi = (unsigned)(u >> 32) & mk, lo = (unsigned)u & mk;
          asm("v_max_f64 %0, %0, |%1|" : "+v"(am) : "v"(__longlong_as_double((long long)(((unsigned long long)hi << 32) | lo))));
          set_el<el(k, l0 + l)>(T(__longlong_as_double((long long)(((unsigned long long)(hi ^ (sg & mk)) << 32) | lo))));
        });
      });
      if (gc == 0 && rm) set_el<el(k, 0)>(T(sg ? -b[r] : b[r]));
    });
    if (gr == 0)
      unroll<CPT>([&](auto l) {
        const int j = col_of(l) - 1;
        if (j >= 0 && j < n) set_el<el(0, l)>(T(-c[j]));
      });
    // max |A_ij| in FP64 (the check scales its tolerances by it)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) am = fmax(am, __shfl_xor(am, off));
    if (lane == 0) s_am[tid >> 6] = am;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p;
      bsr[p] = (i >= 2 && i < R) ? n + i - 2 : -1;
    }
    dm = redm = 0;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = lane + 64 * g;
      nbv[g] = (j == 0 || j >= C) ? -1 : (j <= n ? j - 1 : n + m);
      if (j == 0 || j >= C - 1) dm |= 1 << g;
    }
    for (int i = tid; i < RCAP; i += NT) redund[i] = 0;
    publish_rhs();
    col_ready = -1;
    orow_in = -1;
    __syncthreads();
  }

  // marks the warm-start targets and keeps the list in LDS; false when the list holds no
  // valid variable id
  __device__ __forceinline__ bool set_target(const int32_t* warm) {
    if (!warm) return false;
    for (int x = tid; x < RCAP + CCAP; x += NT) target[x] = 0;
    if constexpr (BC) {
      for (int i = tid; i < RCAP; i += NT) bs[i] = (i >= 2 && i < R) ? n + i - 2 : -1;
      for (int j = tid; j < CCAP; j += NT) nb[j] = (j == 0 || j >= C) ? -1 : (j <= n ? j - 1 : n + m);
      for (int x = tid; x < RCAP + CCAP; x += NT) colof[x] = x < n ? x + 1 : (x == n + m ? C - 1 : -1);
    }
    __syncthreads();
    int any = 0;
    for (int i = tid; i < m; i += NT) {
      const int x = warm[i];
      wl[i] = x;
      if (x >= 0 && x < n + m) { target[x] = 1; any = 1; }
    }
    return __syncthreads_or(any) != 0;
  }

  // entry ci of the warm-start list (from LDS; uniform)
  __device__ __forceinline__ int warm_at(const int32_t*, int ci) const { return uniform(wl[ci]); }

  __device__ __forceinline__ int bs_now(int i) const { return pick(bsr, i); }
  __device__ __forceinline__ int bs_of(int i) const { return pick(bsr, i); }
  __device__ __forceinline__ int nb_of(int j) const { return pick(nbv, j); }
  __device__ __forceinline__ int find_basic(int var) const {
    return first_of<RP>([&](int p) { return bsr[p] == var; });
  }
  // column of nonbasic variable var (-1 if basic)
  __device__ __forceinline__ int find_nonbasic(int var) const {
    return first_of<NG>([&](int g) { return nbv[g] == var; });
  }

  // The owners of column s write it to LDS (with ZERO: to the update's copy too, and clear
  // it in their blocks); then every wavefront has it in row form.  Two buffers: one is
  // written again only after the barrier behind every wavefront's reads of it.
  template <bool ZERO>
  __device__ __forceinline__ void publish_col(int s, T (&acol)[RP]) {
    const int ls = s / TC, gcs = s - ls * TC;
    cph ^= 1;
    T* cb = colbuf + cph * RB;
    T* cu = colupd + cph * RB;
    if constexpr (ZERO && !kAcc) {
      if (gc == gcs)
        blk_out<T, NV, CPT, RPT, CPT, 1, TR, true>(ls, lds_addr(cb + gr), lds_addr(cu + gr), T(0));
      lds_settle();
    } else {
      dispatch<0, CPT>(ls, [&](auto l) {
        if (gc == gcs)
          unroll<RPT>([&](auto k) {
            const T x = get_el<el(k, l)>();
            cb[row_of(k)] = x;
            if constexpr (ZERO) {
              cu[row_of(k)] = x;
              set_el<el(k, l)>(T(0));
            }
          });
      });
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p;
      const T a = cb[i];
      acol[p] = i < R ? a : T(0);
    }
    col_ready = ZERO ? s : -1;
  }

  // column s back from the update's copy (after a ratio test that found no row)
  __device__ __forceinline__ void restore_col(int s) {
    const int ls = s / TC, gcs = s - ls * TC;
    const T* cu = colupd + cph * RB;
    dispatch<0, CPT>(ls, [&](auto l) {
      if (gc == gcs) unroll<RPT>([&](auto k) { set_el<el(k, l)>(cu[row_of(k)]); });
    });
    col_ready = -1;
  }

  // The owners of row r write it to LDS; with CLEAR they set it to -0.0 and one of them
  // publishes the entry of column s as 1.  Read after the next barrier.
  template <bool CLEAR>
  __device__ __forceinline__ T* write_row(int r, int s) {
    const int kr = r / TR, grr = r - kr * TR;
    rph ^= 1;
    T* rb = rowbuf + rph * CB;
    if constexpr (CLEAR && !kAcc) {
      if (gr == grr)
        blk_out<T, NV, RPT, CPT, 1, CPT, TC, false>(kr, lds_addr(rb + gc), 0, T(-0.0));
    } else {
      dispatch<0, RPT>(kr, [&](auto k) {
        if (gr == grr)
          unroll<CPT>([&](auto l) {
            rb[col_of(l)] = get_el<el(k, l)>();
            if constexpr (CLEAR) set_el<el(k, l)>(T(-0.0));
          });
      });
    }
    if constexpr (CLEAR) {
      // (same wavefront, after the row's own stores)
      if (gr == grr && gc == 0) rb[s] = T(1);
    }
    return rb;
  }

  // the objective row in column form
  __device__ __forceinline__ void load_objective(int orow) {
    const T* rb = write_row<false>(orow, 0);
    __syncthreads();
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = lane + 64 * g;
      const T d = rb[j];
      orw[g] = j < C ? d : T(0);
    }
    orow_in = orow;
  }

  // row of largest |T[i][s]| among constraint rows whose basic variable is not a target
  __device__ __forceinline__ int absmax_row(int s, T eps_p) {
    T acol[RP];
    publish_col<false>(s, acol);
    ArgMin<T> am;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p, x = bsr[p];
      const bool ok = x >= 0 && !((redm >> p) & 1) && !target[x < 0 ? 0 : x];
      am.add(ok, -tabs(acol[p]), i, i);
    }
    T bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    bp = uniform(bp);
    return (bp < 0 || !(uniform(-bv) > eps_p)) ? -1 : bp;
  }

  // Dantzig pricing on the objective row held in column form: most negative entry, lowest
  // column on ties
  __device__ __forceinline__ int price(T eps_d) const {
    bool ok[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) ok[g] = !((dm >> g) & 1) && orw[g] < -eps_d;
    bool neg;
    return arg_min<NG>(orw, ok, neg);
  }
  __device__ __forceinline__ int pricing(int orow, bool bland, T eps_d) {
    if (orow_in != orow) load_objective(orow);
    if (!bland) return price(eps_d);
    ArgMin<T> am;  // Bland: smallest nonbasic id
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = lane + 64 * g;
      am.add(!((dm >> g) & 1) && orw[g] < -eps_d, T(nbv[g]), j, j);
    }
    T bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    return uniform(bp);
  }

  // Ratio test over a published column: smallest theta = max(beta, 0) / a over a > eps_p,
  // degenerate rows by the largest a, ties to the lowest row (Bland: smallest basic id);
  // degenerate: theta is 0
  __device__ __forceinline__ int ratio(const T (&acol)[RP], bool bland, T eps_p, bool& degenerate) const {
    T key[RP];
    bool ok[RP];
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p;
      const T a = acol[p], beta = rhsbuf[i];
      ok[p] = i >= 2 && a > eps_p;
      const T th = (beta > T(0) ? beta : T(0)) / (a > eps_p ? a : T(1));
      key[p] = th > T(0) ? th : -a;
    }
    if (bland) {
      ArgMin<T> am;
#pragma unroll
      for (int p = 0; p < RP; ++p) am.add(ok[p], key[p], bsr[p], lane + 64 * p);
      T bv;
      int bk, bp;
      wave_finish(am, bv, bk, bp);
      degenerate = !(uniform(bv) > T(0));
      return uniform(bp);
    }
    return arg_min<RP>(key, ok, degenerate);
  }

  // Pivots.  Starts with the pivot (r, s), or with the ratio test of column s when r < 0;
  // with `fast` goes on -- pricing on objective row orow, ratio test, pivot -- until no
  // column prices out, the limit is reached, or Bland's rule sets in (0: the state machine
  // looks again), or no row passes the ratio test (1, column s unchanged).  With blk >= 0 the
  // pivot is the crash block's step in slot blk, whose column, scaled row and basis change
  // crash_prepare made: no barrier, every thread reads only LDS that no one writes until the
  // next barrier.
  __device__ __forceinline__ int engine(int& r, int& s, bool fast, int orow, const Opt<T>& o,
                                        int maxit, bool keep_last, int& it, int& deg, int& last) {
    if (fast && orow_in != orow) load_objective(orow);
    if (!fast) orow_in = -1;
    for (;;) {
      const T* cu;
      const T* rb;
      T rp = T(1);
      T c0 = T(0);
      bool prepared = false;
      if constexpr (BC) prepared = blk >= 0;
      if (prepared) {
        cu = cbM + blk * RCAP;
        rb = cbP + blk * CCAP;
        const int ls = s / TC, gcs = s - ls * TC, kr = r / TR, grr = r - kr * TR;
        dispatch<0, CPT>(ls, [&](auto l) {
          if (gc == gcs) unroll<RPT>([&](auto k) { set_el<el(k, l)>(T(0)); });
        });
        dispatch<0, RPT>(kr, [&](auto k) {
          if (gr == grr) unroll<CPT>([&](auto l) { set_el<el(k, l)>(T(-0.0)); });
        });
      } else {
        T acol[RP];
        publish_col<true>(s, acol);
        if (r < 0) {
          bool degenerate;
          r = ratio(acol, deg >= o.bland_after, o.eps_p, degenerate);
          if (r < 0) {
            restore_col(s);
            return 1;
          }
          deg = degenerate ? deg + 1 : 0;
        }
        rb = write_row<true>(r, s);
        cu = colupd + cph * RB;
        if (tid == 0) colupd[cph * RB + r] = T(-1);
        rp = T(-1) / pick(acol, r);
        const int e = pick(nbv, s), lv = pick(bsr, r);  // entering, leaving variable
#pragma unroll
        for (int p = 0; p < RP; ++p) bsr[p] = (lane + 64 * p == r) ? e : bsr[p];
#pragma unroll
        for (int g = 0; g < NG; ++g) nbv[g] = (lane + 64 * g == s) ? lv : nbv[g];
        if (fast) c0 = pick(orw, s);
        if constexpr (!kAcc) lds_settle();
        __syncthreads();
      }
      int sn = -1;
      if (fast) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          const int j = lane + 64 * g;
          const T pr = rb[j] * rp;
          const T d = fma_t(c0, pr, j == s ? T(0) : orw[g]);
          orw[g] = j < C ? d : T(0);
        }
        sn = price(o.eps_d);
      }
      // The block's instructions keep their order, so operands are loaded ahead of them: the
      // column, then the row in parts of at most PG entries.
      constexpr int NP = (CPT + 8) / 9, PG = (CPT + NP - 1) / NP;
      // (blocks of many rows take the column in parts too, inside the row's)
      constexpr int NK = (RPT + 7) / 8, KG = (RPT + NK - 1) / NK;
      T col[KG];
      auto load_col = [&](auto q) {
        constexpr int k0 = q * KG, kn = RPT - k0 < KG ? RPT - k0 : KG;
#pragma unroll
        for (int k = 0; k < kn; ++k) col[k] = cu[row_of(k0 + k)];
      };
      if constexpr (NK == 1) load_col(std::integral_constant<int, 0>{});
      unroll<NP>([&](auto w) {
        constexpr int l0 = w * PG, ln = CPT - l0 < PG ? CPT - l0 : PG;
        T prow[ln];
        if constexpr (NK > 1) load_col(std::integral_constant<int, 0>{});
#pragma unroll
        for (int l = 0; l < ln; ++l) prow[l] = rb[col_of(l0 + l)];
#pragma unroll
        for (int l = 0; l < ln; ++l) prow[l] *= rp;
        unroll<NK>([&](auto q) {
          constexpr int k0 = q * KG, kn = RPT - k0 < KG ? RPT - k0 : KG;
          if constexpr (q > 0) load_col(q);
          unroll<kn * ln>([&](auto e) { blk_fma<T, NV, el(k0 + e % kn, l0 + e / kn)>(col[e % kn], prow[e / kn]); });
        });
      });
      publish_rhs();
      col_ready = -1;
      blk = -1;
      last = keep_last ? r | (s << 16) : -1;
      ++it;
      if (!fast || it >= maxit || deg >= o.bland_after || sn < 0) return 0;
      s = sn;
      r = -1;
    }
  }
  __device__ __forceinline__ void pivot(int, int) {}

  // column of largest |T[r][j]| among live columns; -1 if all <= eps_p
  __device__ __forceinline__ int absmax_col(int r, T eps_p) {
    const T* rb = write_row<false>(r, 0);
    __syncthreads();
    ArgMin<T> am;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = lane + 64 * g;
      am.add(!((dm >> g) & 1), -tabs(rb[j]), j, j);
    }
    T bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    bp = uniform(bp);
    return (bp < 0 || !(uniform(-bv) > eps_p)) ? -1 : bp;
  }

  // dual simplex leaving row: most negative rhs below -tol (Bland: smallest basic id)
  __device__ __forceinline__ int dual_row(bool bland, T tol) {
    __syncthreads();
    ArgMin<T> am;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p;
      const T beta = rhsbuf[i];
      am.add(i >= 2 && i < R && !((redm >> p) & 1) && beta < -tol, bland ? T(bsr[p]) : beta, i, i);
    }
    T bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    return uniform(bp);
  }

  // dual simplex entering column for leaving row r
  __device__ __forceinline__ int dual_ratio(int r, bool bland, T eps_p, T& theta) {
    if (orow_in != 0) load_objective(0);
    const T* rb = write_row<false>(r, 0);
    __syncthreads();
    ArgMin<T> am;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = lane + 64 * g;
      const T a = rb[j];
      const T d = orw[g];
      const bool ok = !((dm >> g) & 1) && a < -eps_p;
      const T th = (d > T(0) ? d : T(0)) / (ok ? -a : T(1));
      const T key = th > T(0) ? th : a;
      am.add(ok, key, bland ? nbv[g] : j, j);
    }
    T bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    bv = uniform(bv);
    theta = bv > T(0) ? bv : T(0);
    return uniform(bp);
  }

  // A dead column never enters again, and its entries influence no other entry (the
  // update of (i, j) reads only column s and row r), so killing it only sets its bit.
  __device__ __forceinline__ void kill_col(int j) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
      if (lane + 64 * g == j) dm |= 1 << g;
  }

  // only the right-hand side (column 0) is read and written this way by the driver
  __device__ __forceinline__ T get(int i, int) {
    __syncthreads();
    return uniform(rhsbuf[i]);
  }
  __device__ __forceinline__ void set(int i, int, T val) {
    const int ki = i / TR, gri = i - ki * TR;
    __syncthreads();
    dispatch<0, RPT>(ki, [&](auto k) {
      if (gr == gri && gc == 0) set_el<el(k, 0)>(val);
    });
    if (gr == gri && gc == 0) rhsbuf[i] = val;
    __syncthreads();
  }

  __device__ __forceinline__ void mark_redund(int r) {
    if (tid == 0) redund[r] = 1;
#pragma unroll
    for (int p = 0; p < RP; ++p)
      if (lane + 64 * p == r) redm |= 1 << p;
    set(r, 0, T(0));
  }

  __device__ __forceinline__ int min_rhs_row() {
    __syncthreads();
    ArgMin<T> am;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p;
      am.add(i >= 2 && i < R && !((redm >> p) & 1), rhsbuf[i], i, i);
    }
    T bv;
    int bk, bp;
    wave_finish(am, bv, bk, bp);
    return uniform(bp);
  }

  __device__ __forceinline__ void setup_x0() {
    __syncthreads();
    const int x0 = C - 1, lx = x0 / TC, gcx = x0 - lx * TC;
    dispatch<0, CPT>(lx, [&](auto l) {
      if (gc == gcx)
        unroll<RPT>([&](auto k) {
          const int i = row_of(k);
          set_el<el(k, l)>((i >= 2 && i < R) ? (redund[i < RCAP ? i : 0] ? T(0) : T(-1)) : (i == 1 ? T(1) : T(0)));
        });
    });
    // row 1 sits in slot 1 / TR of thread row 1 % TR
    unroll<CPT>([&](auto l) {
      if (gr == 1 % TR && col_of(l) != x0) set_el<el(1 / TR, l)>(T(0));
    });
    if (gr == 1 % TR && gc == 0) rhsbuf[1] = T(0);
#pragma unroll
    for (int g = 0; g < NG; ++g)
      if (lane + 64 * g == x0) dm &= ~(1 << g);
    orow_in = -1;
    __syncthreads();
  }

  // pivot j of the prepared block, packed (wave-uniform)
  __device__ __forceinline__ int blk_word(int j) const { return uniform(cbW[j]); }

  // Prepares the next up-to-KB crash targets as one block.  Same targets, rows and
  // arithmetic as one absmax_row + pivot per target, so the tableau ends bit-identical:
  //   targets  the warm-list structurals from ci on that are nonbasic, stopping before a
  //            repeated column (its second turn must see the first one's pivot);
  //   A        wavefront 0 runs the pivots on the targets' columns alone (cbM): step t
  //            picks its row from column t as absmax_row does (rows pivoted by earlier
  //            steps no longer eligible) and updates the later columns; column t keeps
  //            the values step t multiplies by.  The steps' basis changes touch distinct
  //            rows, columns and variables, so lane u then makes step u's;
  //   B        one thread per column j runs the pivot rows alone (cbP): row r_t, updated
  //            by steps < t, becomes step t's scaled pivot row.
  // The caller then makes the block's pivots (cbW) through engine() with `blk` set to the
  // step's slot, which reads the column and row from cbM / cbP and needs no barrier.  Six
  // barriers per block instead of about five per target.  Returns the number of pivots
  // (steps without an eligible row make none), or -1 when no target is left (ci = m).
  __device__ __forceinline__ int crash_prepare(int& ci, const int8_t* sense, T eps_p) {
    __syncthreads();
    // targets: wavefront 0 reads the list 64 entries at a time and takes the nonbasic
    // structurals in order; `sel` on lane u holds target u's column
    if (wv == 0) {
      int kc = 0, c = ci, sel = -1;
      bool stop = false;
      while (!stop && c < m && kc < KB) {
        const int idx = c + lane;
        const int w = idx < m ? wl[idx] : -1;
        const int s = (w >= 0 && w < n) ? colof[w] : -1;
        unsigned long long bal = __ballot(s >= 0);
        int next = c + 64 < m ? c + 64 : m;
        while (bal != 0ull) {
          const int l = __ffsll((long long)bal) - 1;
          const int sl = __builtin_amdgcn_readlane(s, l);
          if (__ballot(lane < kc && sel == sl) != 0ull) {  // repeated: stop before it
            stop = true;
            next = c + l;
            break;
          }
          if (lane == kc) sel = sl;
          ++kc;
          bal &= bal - 1ull;
          if (kc == KB) {
            next = c + l + 1;
            break;
          }
        }
        c = next;
      }
      if (lane < kc) cbS[lane] = sel;
      if (lane == 0) {
        cbR[KB] = kc;
        cbR[KB + 1] = c;
      }
    }
    __syncthreads();
    const int kc = uniform(cbR[KB]);
    ci = uniform(cbR[KB + 1]);
    if (kc == 0) return -1;
    for (int u = 0; u < kc; ++u) {
      const int s = uniform(cbS[u]), ls = s / TC, gcs = s - ls * TC;
      dispatch<0, CPT>(ls, [&](auto l) {
        if (gc == gcs) unroll<RPT>([&](auto k) { cbM[u * RCAP + row_of(k)] = get_el<el(k, l)>(); });
      });
    }
    __syncthreads();

    // A: wavefront 0, the block's columns in registers (lane rows lane + 64 q)
    if (wv == 0) {
      T mv[QR][KB];
      bool el[QR];
#pragma unroll
      for (int q = 0; q < QR; ++q) {
        const int i = lane + 64 * q;
        const int x = (i >= 2 && i < R) ? bs[i] : -1;
        el[q] = x >= 0 && !redund[i] && !target[x];
#pragma unroll
        for (int u = 0; u < KB; ++u) mv[q][u] = (u < kc && i < RCAP) ? cbM[u * RCAP + i] : T(0);
      }
#pragma unroll
      for (int t = 0; t < KB; ++t) {
        if (t < kc) {
          T bv = inf_of<T>();
          int bk = INT_MAX, bp = -1;
          {
            ArgMin<T> am;
#pragma unroll
            for (int q = 0; q < QR; ++q) am.add(el[q], -tabs(mv[q][t]), lane + 64 * q, lane + 64 * q);
            wave_finish(am, bv, bk, bp);
          }
          const int r = uniform(bp);
          int rr = -1;
          if (r >= 0 && -bv > eps_p) {
            rr = r;
            const int rl = r & 63, rq = r >> 6;
            T pv = mv[0][t];
#pragma unroll
            for (int q = 1; q < QR; ++q) pv = (rq == q) ? mv[q][t] : pv;
            const T rp = T(1) / lane_read(pv, rl);
#pragma unroll
            for (int u = t + 1; u < KB; ++u) {
              if (u < kc) {
                T x = mv[0][u];
#pragma unroll
                for (int q = 1; q < QR; ++q) x = (rq == q) ? mv[q][u] : x;
                const T pr = lane_read(x, rl) * rp;
#pragma unroll
                for (int q = 0; q < QR; ++q)
                  mv[q][u] = (lane + 64 * q == r) ? pr : fma_t(-mv[q][t], pr, mv[q][u]);
              }
            }
#pragma unroll
            for (int q = 0; q < QR; ++q) el[q] = el[q] && (lane + 64 * q != r);
            if (lane == 0) cbRp[t] = rp;
          }
          if (lane == 0) cbR[t] = rr;
        }
      }
      // the multipliers of step t (column t negated; no later step of the block changes it),
      // 1 at its pivot row
#pragma unroll
      for (int q = 0; q < QR; ++q) {
        const int i = lane + 64 * q;
        if (i < RCAP) {
#pragma unroll
          for (int u = 0; u < KB; ++u)
            if (u < kc) cbM[u * RCAP + i] = i == cbR[u] ? T(1) : -mv[q][u];
        }
      }
      // basis changes: each step has its own row, column, entering and leaving variable,
      // so lane u makes step u's
      const int r = lane < kc ? cbR[lane] : -1;
      const unsigned long long made = __ballot(r >= 0);
      if (lane == 0) cbR[KB + 2] = __popcll(made);
      if (r >= 0) {
        {
          const int s = cbS[lane];
          const int lv = bs[r], e = nb[s];
          const int kill = (lv >= n && lv < n + m && sense && sense[lv - n] == 1) ? 1 : 0;
          cbW[__popcll(made & ((1ull << lane) - 1ull))] = r | (s << 12) | (lane << 24) | (kill << 30);
          bs[r] = e;
          nb[s] = lv;
          colof[e] = -1;
          colof[lv] = s;
        }
      }
    }
    __syncthreads();
    for (int t = 0; t < kc; ++t) {
      const int r = uniform(cbR[t]);
      if (r >= 0) {
        const int kr = r / TR, grr = r - kr * TR;
        dispatch<0, RPT>(kr, [&](auto k) {
          if (gr == grr) unroll<CPT>([&](auto l) { cbP[t * CCAP + col_of(l)] = get_el<el(k, l)>(); });
        });
      }
    }
    __syncthreads();

    // B: thread per column, the block's pivot rows in registers
    for (int j = tid; j < C; j += NT) {
      T pc[KB];
#pragma unroll
      for (int u = 0; u < KB; ++u) pc[u] = u < kc ? cbP[u * CCAP + j] : T(0);
#pragma unroll
      for (int t = 0; t < KB; ++t) {
        if (t < kc) {
          const int r = cbR[t];
          if (r >= 0) {
            const int s = cbS[t];
            const T rp = cbRp[t];
            const T pr = (j == s) ? rp : pc[t] * rp;
            pc[t] = pr;
#pragma unroll
            for (int u = t + 1; u < KB; ++u) {
              if (u < kc) {
                const int ru = cbR[u];
                if (ru >= 0) pc[u] = fma_t(cbM[t * RCAP + ru], pr, (j == s) ? T(0) : pc[u]);
              }
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < KB; ++u)
        if (u < kc) cbP[u * CCAP + j] = pc[u];
    }
    // the register copies of the basis (the maps are final here)
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int i = lane + 64 * p;
      bsr[p] = i < RCAP ? bs[i] : -1;
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = lane + 64 * g;
      nbv[g] = j < CCAP ? nb[j] : -1;
    }
    __syncthreads();
    return uniform(cbR[KB + 2]);
  }

  // column 0 is mirrored in rhsbuf (objective T[0][0], basic values T[i][0])
  __device__ __forceinline__ void write_outputs(int lp, const LpDesc& d, const Out& out, int status, int it,
                                int p1, int unb, T wfin, int last) {
    __syncthreads();
    if (tid == 0) {
      double am = s_am[0];
      for (int w = 1; w < NW; ++w) am = fmax(am, s_am[w]);
      out.amax[lp] = am;
      out.status[lp] = status;
      out.pivots[lp] = it;
      out.p1[lp] = p1;
      out.unb[lp] = unb;
      if (out.lastpiv) out.lastpiv[lp] = last;
      out.obj[lp] = (double)rhsbuf[0];
      out.wfin[lp] = (double)wfin;
    }
    double* x = out.x + d.x;
    int32_t* basis = out.basis + d.basis;
    for (int j = tid; j < n; j += NT) x[j] = 0.0;
    __syncthreads();
    if (wv == 0) {
#pragma unroll
      for (int p = 0; p < RP; ++p) {
        const int i = lane + 64 * p;
        if (i >= 2 && i < R) {
          basis[i - 2] = bsr[p];
          if (bsr[p] >= 0 && bsr[p] < n) x[bsr[p]] = (double)rhsbuf[i];
        }
      }
    }
    // final tableau and nonbasic ids for the FP64 check (B^-1 is in the slack columns)
    if (out.tab) {
      T* tp = (T*)(out.tab + 8 * d.t);
      unroll<RPT>([&](auto k) {
        const int i = row_of(k);
        unroll<CPT>([&](auto l) {
          const T x = get_el<el(k, l)>();
          if (i < R && col_of(l) < C) tp[(int64_t)i * C + col_of(l)] = x;
        });
      });
      if (wv == 0) {
        int32_t* np = (int32_t*)(out.tab + 8 * (d.t + (int64_t)R * C));
#pragma unroll
        for (int g = 0; g < NG; ++g)
          if (lane + 64 * g < C) np[lane + 64 * g] = nbv[g];
      }
    }
  }
};

// claims the block's registers for the kernel: v[NV .. ), a[0 .. ) beyond 256
template <int TOP>
__device__ __forceinline__ void claim() {
#define BLPG_CLAIM(x, r) if constexpr (TOP >= x - 3 && TOP <= x) asm volatile("" ::: r)
  // (in steps of four: registers are allocated in groups of eight)
  static_assert(TOP >= 64 && TOP <= 255);
  BLPG_CLAIM(67, "v67"); BLPG_CLAIM(71, "v71"); BLPG_CLAIM(75, "v75"); BLPG_CLAIM(79, "v79");
  BLPG_CLAIM(83, "v83"); BLPG_CLAIM(87, "v87"); BLPG_CLAIM(91, "v91"); BLPG_CLAIM(95, "v95");
  BLPG_CLAIM(99, "v99"); BLPG_CLAIM(103, "v103"); BLPG_CLAIM(107, "v107"); BLPG_CLAIM(111, "v111");
  BLPG_CLAIM(115, "v115"); BLPG_CLAIM(119, "v119"); BLPG_CLAIM(123, "v123"); BLPG_CLAIM(127, "v127");
  BLPG_CLAIM(131, "v131"); BLPG_CLAIM(135, "v135"); BLPG_CLAIM(139, "v139"); BLPG_CLAIM(143, "v143");
  BLPG_CLAIM(147, "v147"); BLPG_CLAIM(151, "v151"); BLPG_CLAIM(155, "v155"); BLPG_CLAIM(159, "v159");
  BLPG_CLAIM(163, "v163"); BLPG_CLAIM(167, "v167"); BLPG_CLAIM(171, "v171"); BLPG_CLAIM(175, "v175");
  BLPG_CLAIM(179, "v179"); BLPG_CLAIM(183, "v183"); BLPG_CLAIM(187, "v187"); BLPG_CLAIM(191, "v191");
  BLPG_CLAIM(195, "v195"); BLPG_CLAIM(199, "v199"); BLPG_CLAIM(203, "v203"); BLPG_CLAIM(207, "v207");
  BLPG_CLAIM(211, "v211"); BLPG_CLAIM(215, "v215"); BLPG_CLAIM(219, "v219"); BLPG_CLAIM(223, "v223");
  BLPG_CLAIM(227, "v227"); BLPG_CLAIM(231, "v231"); BLPG_CLAIM(235, "v235"); BLPG_CLAIM(239, "v239");
  BLPG_CLAIM(243, "v243"); BLPG_CLAIM(247, "v247"); BLPG_CLAIM(251, "v251"); BLPG_CLAIM(255, "v255");
#undef BLPG_CLAIM
}

template <typename T, int NW, int TC, int RPT, int CPT, bool BC, int NV>
__device__ __forceinline__ void tile_body(const LpDesc* __restrict__ desc, const double* __restrict__ pool,
                                          const int8_t* __restrict__ spool, const int32_t* __restrict__ idx,
                                          int32_t count, const int32_t* count_dev, int32_t* queue,
                                          const Out& out, const Opt<T>& o,
                                          const int32_t* __restrict__ warm_pool) {
  using Tab = TileTab<T, NW, TC, RPT, CPT, BC, NV>;
  constexpr int words = (int)sizeof(T) / 4 * RPT * CPT;
  claim<(NV + words < 256 ? NV + words : 256) - 1>();
  // (the comment names the block's first register in the listing, for the build's check that
  // the compiler stays below it)
  if constexpr (NV + words > 256) {
    static_assert(2 * NV + words - 256 <= 128);
    asm volatile("" ::: "a127");
    asm volatile("; block from v%0 a%0" ::"n"(NV));
  } else {
    asm volatile("; block from v%0" ::"n"(NV));
  }
  __shared__ T colbuf[2 * Tab::RB], colupd[2 * Tab::RB], rowbuf[2 * Tab::CB], rhsbuf[Tab::RB];
  __shared__ int bs[BC ? Tab::RCAP : 1], nb[BC ? Tab::CCAP : 1], colof[BC ? Tab::RCAP + Tab::CCAP : 1];
  __shared__ uint8_t redund[Tab::RCAP], target[Tab::RCAP + Tab::CCAP];
  __shared__ int wl[Tab::RCAP];
  __shared__ double s_am[NW];
  __shared__ int s_q;
  __shared__ T cbM[BC ? Tab::KB * Tab::RCAP : 1], cbP[BC ? Tab::KB * Tab::CB : 1], cbRp[Tab::KB];
  __shared__ int cbR[Tab::KB + 3], cbS[Tab::KB], cbW[Tab::KB];
  Tab t;
  t.s_am = s_am;
  t.tid = threadIdx.x;
  t.lane = threadIdx.x & 63;
  t.wv = uniform((int)(threadIdx.x >> 6));
  t.gr = threadIdx.x / TC;
  t.gc = threadIdx.x - t.gr * TC;
  t.cph = t.rph = 0;
  t.colbuf = colbuf; t.colupd = colupd; t.rhsbuf = rhsbuf; t.rowbuf = rowbuf;
  t.bs = bs; t.nb = nb; t.redund = redund; t.target = target;
  t.wl = wl; t.colof = colof;
  t.cbM = cbM; t.cbP = cbP; t.cbRp = cbRp; t.cbR = cbR; t.cbS = cbS; t.cbW = cbW;
  t.blk = -1;
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
    T wfin;
    run_simplex<T>(t, d.m, d.n, sense, o, status, it, p1, unb, wfin, last, warm);
    t.write_outputs(lp, d, out, status, it, p1, unb, wfin, last);
  }
}

// ---------------------------------------------------------------------------------
// variant table: (waves per LP, TC, RPT, CPT); capacity (64*NW/TC*RPT) x (TC*CPT)
// (the autotuner measures every variant that holds a shape; fewer waves per LP mean fewer
// barriers per pivot, more waves mean fewer registers per thread).  b32 / b64: block crash
// on (the variants whose register block leaves room for it without spilling).
// vr: vector registers left to the compiler in FP32 / FP64, cold / warm (block crash); the
// block follows them.  Chosen so that block + vr stays within the 512 / w registers of w
// waves per SIMD (128, 168, 256) where that admits one more LP per CU.
// 9, 12 and 13 are the instances for many LPs (Tuner::for_many): fewer wavefronts with more of
// the tableau each, so that one LP more fits a CU.
//   id nw  tc rpt cpt  vr32 vr32w vr64 vr64w b32 b64
#define BLPG_TILE_VARIANTS(X)                          \
  X(0, 1, 8, 4, 5, 76, 76, 88, 88, 1, 1)               \
  X(1, 1, 8, 7, 7, 78, 78, 70, 156, 1, 1)              \
  X(2, 2, 16, 8, 7, 72, 110, 144, 144, 1, 1)           \
  X(3, 2, 16, 10, 6, 68, 108, 136, 136, 1, 1)          \
  X(4, 4, 16, 7, 7, 78, 78, 70, 156, 1, 1)             \
  X(5, 8, 16, 6, 9, 74, 74, 148, 148, 1, 0)            \
  X(6, 8, 16, 7, 13, 76, 76, 74, 74, 0, 0)             \
  X(7, 1, 8, 10, 11, 144, 144, 80, 80, 0, 0)           \
  X(8, 1, 16, 16, 7, 144, 144, 80, 80, 0, 0)           \
  X(9, 2, 16, 14, 7, 156, 156, 60, 60, 0, 0)           \
  X(10, 4, 32, 14, 4, 72, 112, 144, 144, 1, 1)         \
  X(11, 8, 16, 4, 7, 100, 100, 72, 112, 1, 1)          \
  X(12, 4, 16, 11, 9, 68, 68, 58, 58, 0, 0)
#define BLPG_TILE_VARIANTS_F32(X) X(13, 4, 16, 13, 13, 86, 86, 0, 0, 0, 0)

// one kernel per variant, precision and cold / warm (the attribute takes literals only; with
// accumulation registers in use the compiler splits its share in two, without it doubles it;
// the build reads in the listing that it stayed below the block)
#define BLPG_TILE_KERNEL(name, T, nw, tc, rpt, cpt, vr, words, BC)                               \
  __global__ __launch_bounds__(nw * 64)                                                          \
  __attribute__((amdgpu_num_vgpr(vr + words * rpt * cpt > 256 ? vr : vr / 2))) void name(        \
      const LpDesc* __restrict__ desc, const double* __restrict__ pool,                          \
      const int8_t* __restrict__ spool, const int32_t* __restrict__ idx, int32_t count,          \
      const int32_t* count_dev, int32_t* queue, Out out, Opt<T> o,                               \
      const int32_t* __restrict__ warm_pool) {                                                   \
    tile_body<T, nw, tc, rpt, cpt, BC, vr>(desc, pool, spool, idx, count, count_dev, queue, out, \
                                           o, warm_pool);                                        \
  }
}  // namespace blpg
