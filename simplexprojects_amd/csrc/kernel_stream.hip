// kernel_stream.hip -- the size-generic simplex kernels: tableau in LDS, or in HBM.
//
// One workgroup per LP, persistent over a work queue (an atomic LP counter).
//
// LDS (StreamTab): the condensed tableau ((m+2) x (n+2), row-major) fits the 160 KB of a CU.
// Per pivot: a pass over the objective row, a pass over the pivot column, the rank-1 update
// T[i][j] = fma(-colbuf[i], rowbuf[j], T[i][j]); rows with colbuf[i] == 0 are skipped (their
// entries are unchanged up to the sign of zero).
//
// HBM (PanelTab), any size: the constraint rows live in a slab owned by the workgroup and a
// pivot does not touch them.  Its column and scaled row go into a panel of up to 8 pending
// pivots; the objective rows and the right-hand side (all that pricing and the ratio test
// read besides one column) are kept current.  An entering column or a pivot row is read from
// the slab and brought up to date through the panel, entry by entry the same FMAs in the same
// order as immediate updates, so results are bit-identical; every 8th pivot one pass applies
// the panel to the whole slab.  A pivot that replaced a row or column is the panel step at
// which entries of it start anew (rowstep, colstep).  Immediate updates read and wrote the
// tableau once per pivot; this does so once per 8.
//
// These replace the reference's mykernel (simplex.cu:35-385), which keeps the full tableau
// (slack identity included) in global memory, reduces through global scratch and updates
// with one thread per row looping over columns.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "simplex_device.hpp"

namespace blpg {

template <typename T, int NT>
struct StreamTab {
  static constexpr int NW = NT / 64;
  static constexpr bool kEngine = false;
  static constexpr bool kBlockCrash = false;  // crash one target per pivot
  T* tab;
  int ld, R, C, m, n;
  T* colbuf;
  T* rowbuf;
  int* bs;
  int* nb;
  uint8_t* dead;
  uint8_t* redund;
  uint8_t* target;  // target[var] = 1: var belongs to the warm-start basis
  double* s_am;     // per-wave max |A_ij| (NW entries)
  Reducer<T, NW> red;

  __device__ __forceinline__ T& at(int i, int j) { return tab[(int64_t)i * ld + j]; }
  __device__ __forceinline__ void loop_fence() {}

  __device__ __forceinline__ void init(const double* A, const double* b, const double* c, const int8_t* sense) {
    const int tid = threadIdx.x;
    for (int e = tid; e < R * C; e += NT) {
      const int i = e / C, j = e - (e / C) * C;
      at(i, j) = init_entry<T>(i, j, m, n, A, b, c, sense);
    }
    // max |A_ij| in FP64 (the check scales its tolerances by it)
    double am = 0.0;
    for (int e = tid; e < m * n; e += NT) am = fmax(am, fabs(A[e]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) am = fmax(am, __shfl_xor(am, off));
    if ((tid & 63) == 0) s_am[tid >> 6] = am;
    for (int i = tid; i < R; i += NT) { bs[i] = i >= 2 ? n + i - 2 : -1; redund[i] = 0; }
    for (int j = tid; j < C; j += NT) {
      nb[j] = j == 0 ? -1 : (j <= n ? j - 1 : n + m);
      dead[j] = (j == 0 || j == C - 1) ? 1 : 0;
    }
    __syncthreads();
  }

  // marks the warm-start targets; false when the list holds no valid variable id
  __device__ __forceinline__ bool set_target(const int32_t* warm) {
    for (int v = threadIdx.x; v < n + m; v += NT) target[v] = 0;
    __syncthreads();
    int any = 0;
    if (warm)
      for (int i = threadIdx.x; i < m; i += NT) {
        const int v = warm[i];
        if (v >= 0 && v < n + m) { target[v] = 1; any = 1; }
      }
    return __syncthreads_or(any) != 0;
  }

  // dual simplex leaving row: most negative rhs below -tol (Bland: smallest basic id)
  __device__ __forceinline__ int dual_row(bool bland, T tol) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      if (redund[i]) continue;
      const T beta = at(i, 0);
      if (!(beta < -tol)) continue;
      const T key = bland ? T(bs[i]) : beta;
      if (better(key, i, bv, bk)) { bv = key; bk = i; bp = i; }
    }
    red.argmin(bv, bk, bp);
    return bp;
  }

  // dual simplex entering column for leaving row r
  __device__ __forceinline__ int dual_ratio(int r, bool bland, T eps_p, T& theta) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int j = 1 + (int)threadIdx.x; j < C; j += NT) {
      if (dead[j]) continue;
      const T a = at(r, j);
      if (!(a < -eps_p)) continue;
      const T d = at(0, j);
      const T th = (d > T(0) ? d : T(0)) / -a;
      const T key = th > T(0) ? th : a;
      const int kk = bland ? nb[j] : j;
      if (better(key, kk, bv, bk)) { bv = key; bk = kk; bp = j; }
    }
    red.argmin(bv, bk, bp);
    theta = bv > T(0) ? bv : T(0);
    return bp;
  }

  // row of largest |T[i][s]| among constraint rows whose basic variable is not a target
  __device__ __forceinline__ int absmax_row(int s, T eps_p) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      const int v = bs[i];
      if (redund[i] || v < 0 || target[v]) continue;
      const T key = -tabs(at(i, s));
      if (better(key, i, bv, bk)) { bv = key; bk = i; bp = i; }
    }
    red.argmin(bv, bk, bp);
    if (bp < 0 || !(-bv > eps_p)) return -1;
    return bp;
  }

  __device__ __forceinline__ int bs_of(int i) {
    __syncthreads();
    return uniform(bs[i]);
  }
  __device__ __forceinline__ int bs_now(int i) { return bs_of(i); }
  __device__ __forceinline__ int warm_at(const int32_t* warm, int ci) const { return warm[ci]; }

  __device__ __forceinline__ int pricing(int orow, bool bland, T eps_d) {
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int j = 1 + (int)threadIdx.x; j < C; j += NT) {
      if (dead[j]) continue;
      const T d = at(orow, j);
      if (!(d < -eps_d)) continue;
      const T v = bland ? T(nb[j]) : d;
      if (better(v, j, bv, bk)) { bv = v; bk = j; bp = j; }
    }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ int ratio(int s, bool bland, T eps_p, T& theta) {
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = threadIdx.x; i < R; i += NT) {
      const T a = at(i, s);
      colbuf[i] = a;
      if (i >= 2 && a > eps_p) {
        const T beta = at(i, 0);
        const T th = (beta > T(0) ? beta : T(0)) / a;
        const T v = th > T(0) ? th : -a;  // degenerate rows: largest pivot first
        const int k = bland ? bs[i] : i;
        if (better(v, k, bv, bk)) { bv = v; bk = k; bp = i; }
      }
    }
    red.argmin(bv, bk, bp);
    theta = bv > T(0) ? bv : T(0);
    return bp;
  }

  __device__ __forceinline__ void pivot(int r, int s) {
    const int tid = threadIdx.x;
    // every row's pivot-column entry (the ratio pass filled colbuf; refresh it here so
    // phase-I pivots chosen without a ratio pass see it too)
    __syncthreads();
    for (int i = tid; i < R; i += NT) colbuf[i] = at(i, s);
    __syncthreads();
    const T p = uniform(colbuf[r]);
    const T rp = T(1) / p;
    for (int j = tid; j < C; j += NT) rowbuf[j] = (j == s) ? rp : at(r, j) * rp;
    if (tid == 0) { const int t = bs[r]; bs[r] = nb[s]; nb[s] = t; }
    __syncthreads();
    const int lane = tid & 63, w = tid >> 6;
    for (int i = w; i < R; i += NW) {
      const T ci = -colbuf[i];
      if (i == r) {
        for (int j = lane; j < C; j += 64) at(r, j) = rowbuf[j];
      } else if (ci != T(0)) {
        T* row = &at(i, 0);
        for (int j = lane; j < C; j += 64) {
          const T old = (j == s) ? T(0) : row[j];
          row[j] = fma_t(ci, rowbuf[j], old);
        }
      }
    }
    __syncthreads();
  }

  __device__ __forceinline__ int absmax_col(int r, T eps_p) {
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int j = 1 + (int)threadIdx.x; j < C; j += NT) {
      if (dead[j]) continue;
      const T v = -tabs(at(r, j));
      if (better(v, j, bv, bk)) { bv = v; bk = j; bp = j; }
    }
    red.argmin(bv, bk, bp);
    if (bp < 0 || !(-bv > eps_p)) return -1;
    return bp;
  }

  // A dead column never enters again and influences no other entry (an update of (i, j)
  // reads only column s and row r), so it keeps its values: B^-1 columns of fixed slacks
  // stay available to the FP64 check.
  __device__ __forceinline__ void kill_col(int j) {
    __syncthreads();
    if (threadIdx.x == 0) dead[j] = 1;
    __syncthreads();
  }

  __device__ __forceinline__ T get(int i, int j) {
    __syncthreads();
    return uniform(at(i, j));
  }

  __device__ __forceinline__ void set(int i, int j, T v) {
    __syncthreads();
    if (threadIdx.x == 0) at(i, j) = v;
    __syncthreads();
  }

  __device__ __forceinline__ void mark_redund(int r) {
    __syncthreads();
    if (threadIdx.x == 0) { redund[r] = 1; at(r, 0) = T(0); }
    __syncthreads();
  }

  __device__ __forceinline__ int min_rhs_row() {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      if (redund[i]) continue;
      const T v = at(i, 0);
      if (better(v, i, bv, bk)) { bv = v; bk = i; bp = i; }
    }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ void setup_x0() {
    __syncthreads();
    const int x0 = C - 1;
    if (threadIdx.x == 0) dead[x0] = 0;
    for (int i = threadIdx.x; i < R; i += NT)
      at(i, x0) = (i >= 2) ? (redund[i] ? T(0) : T(-1)) : (i == 1 ? T(1) : T(0));
    for (int j = threadIdx.x; j < C - 1; j += NT) at(1, j) = T(0);
    __syncthreads();
  }

  __device__ __forceinline__ int find_basic(int var) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT)
      if (bs[i] == var) { bv = T(0); bk = i; bp = i; }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ int find_nonbasic(int var) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int j = 1 + (int)threadIdx.x; j < C; j += NT)
      if (nb[j] == var) { bv = T(0); bk = j; bp = j; }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ int nb_of(int j) {
    __syncthreads();
    return uniform(nb[j]);
  }

  __device__ __forceinline__ void write_outputs(int lp, const LpDesc& d, const Out& out, int status, int it,
                                int p1, int unb, T wfin, int last) {
    __syncthreads();
    const int tid = threadIdx.x;
    if (tid == 0) {
      double am = s_am[0];
      for (int w = 1; w < NW; ++w) am = fmax(am, s_am[w]);
      out.amax[lp] = am;
      out.status[lp] = status;
      out.pivots[lp] = it;
      out.p1[lp] = p1;
      out.unb[lp] = unb;
      if (out.lastpiv) out.lastpiv[lp] = last;
      out.obj[lp] = (double)at(0, 0);
      out.wfin[lp] = (double)wfin;
    }
    double* x = out.x + d.x;
    int32_t* basis = out.basis + d.basis;
    for (int j = tid; j < n; j += NT) x[j] = 0.0;
    for (int i = tid; i < m; i += NT) basis[i] = bs[2 + i];
    __syncthreads();
    for (int i = 2 + tid; i < R; i += NT) {
      const int v = bs[i];
      if (v >= 0 && v < n) x[v] = (double)at(i, 0);
    }
    // final tableau and nonbasic ids for the FP64 check (B^-1 is in the slack columns)
    if (out.tab) {
      T* tp = (T*)(out.tab + 8 * d.t);
      for (int e = tid; e < R * C; e += NT) tp[e] = tab[e];
      int32_t* np = (int32_t*)(out.tab + 8 * (d.t + (int64_t)R * C));
      for (int j = tid; j < C; j += NT) np[j] = nb[j];
    }
  }
};

// LDS carve-up shared by host and device:
// [tab][colbuf][rowbuf][bs][nb][dead][redund][target][slots]
template <typename T>
struct StreamLayout {
  size_t tab, colbuf, rowbuf, bs, nb, dead, redund, target, slots, total;
  __host__ __device__ StreamLayout(int nw, int rcap, int ccap) {
    auto al = [](size_t x) { return (x + 15) & ~(size_t)15; };
    size_t o = 0;
    tab = o; o += al(sizeof(T) * (size_t)rcap * ccap);
    colbuf = o; o += al(sizeof(T) * rcap);
    rowbuf = o; o += al(sizeof(T) * ccap);
    bs = o; o += al(sizeof(int) * rcap);
    nb = o; o += al(sizeof(int) * ccap);
    dead = o; o += al(ccap);
    redund = o; o += al(rcap);
    target = o; o += al(rcap + ccap);
    slots = o; o += al(sizeof(RedSlot<T>) * 2 * nw);
    total = o;
  }
};

template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_stream(const LpDesc* __restrict__ desc,
                                               const double* __restrict__ pool,
                                               const int8_t* __restrict__ spool,
                                               const int32_t* __restrict__ idx, int32_t count,
                                               const int32_t* count_dev, int32_t* queue,
                                               Out out, Opt<T> o, int rcap, int ccap,
                                               const int32_t* __restrict__ warm_pool) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_q;
  __shared__ double s_am[NT / 64];
  const StreamLayout<T> L(NT / 64, rcap, ccap);
  StreamTab<T, NT> t;
  t.s_am = s_am;
  t.colbuf = (T*)(smem + L.colbuf);
  t.rowbuf = (T*)(smem + L.rowbuf);
  t.bs = (int*)(smem + L.bs);
  t.nb = (int*)(smem + L.nb);
  t.dead = smem + L.dead;
  t.redund = smem + L.redund;
  t.target = smem + L.target;
  t.red.init((RedSlot<T>*)(smem + L.slots));
  t.tab = (T*)(smem + L.tab);
  if (count_dev) count = *count_dev;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_q = atomicAdd(queue, 1);
    __syncthreads();
    const int q = uniform(s_q);
    if (q >= count) break;
    const int lp = idx ? idx[q] : q;
    const LpDesc d = desc[lp];
    t.m = d.m; t.n = d.n; t.R = d.m + 2; t.C = d.n + 2; t.ld = t.C;
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

// Vectors of a PanelTab: objective rows, right-hand side, basis, flags and the panel of
// k pending pivots; in LDS where that fits, else behind the slab in HBM.
struct PanelLayout {
  size_t row0, row1, rhs, pa, pp, bs, nb, dead, redund, target, cstep, rstep, total;
  __host__ __device__ PanelLayout(int esz, int k, int rcap, int ccap) {
    auto al = [](size_t x) { return (x + 15) & ~(size_t)15; };
    size_t o = 0;
    row0 = o; o += al((size_t)esz * ccap);
    row1 = o; o += al((size_t)esz * ccap);
    rhs = o; o += al((size_t)esz * rcap);
    pa = o; o += al((size_t)esz * k * rcap);
    pp = o; o += al((size_t)esz * k * ccap);
    bs = o; o += al(sizeof(int) * rcap);
    nb = o; o += al(sizeof(int) * ccap);
    dead = o; o += al(ccap);
    redund = o; o += al(rcap);
    target = o; o += al(rcap + ccap);
    cstep = o; o += al(ccap);
    rstep = o; o += al(rcap);
    total = o;
  }
};
constexpr int kPanel = 8;  // most pending pivots
// row pitch of the slab: whole cache lines
__host__ __device__ constexpr int panel_ld(int n) { return (n + 1 + 15) & ~15; }

template <typename T, int NT>
struct PanelTab {
  static constexpr int NW = NT / 64;
  static constexpr bool kBlockCrash = false;
  static constexpr bool kEngine = false;
  static constexpr int KB = 1;
  T* tab;        // constraint row i, nonbasic column j (both from 0) at tab[i * ld + j]
  int ld, R, C, m, n;
  int K, q;      // panel size, pending pivots
  int col_ready; // column whose multipliers are in pa[q] (-1: none)
  T *row0, *row1, *rhs;
  T* pa;         // K x R: multipliers of the pending pivots (the column negated, 1 at the row)
  T* pp;         // K x C: their scaled rows
  int *bs, *nb;
  uint8_t *dead, *redund, *target;
  int8_t *cstep, *rstep;  // pending step that replaced the column / row, -1: none
  int *stepr, *stepc;     // row / column of each pending step
  double* s_am;
  Reducer<T, NW> red;
  int blk;

  __device__ __forceinline__ void loop_fence() {}

  __device__ __forceinline__ void init(const double* A, const double* b, const double* c, const int8_t* sense) {
    const int tid = threadIdx.x, lane = tid & 63;
    q = 0;
    col_ready = -1;
    double am = 0.0;
    for_blocks([&](int i0, int c0) {
      double x[FR][FC];
#pragma unroll
      for (int u = 0; u < FR; ++u) {
        const double* t = A + (int64_t)(i0 + u < m ? i0 + u : m - 1) * n;
#pragma unroll
        for (int v = 0; v < FC; ++v) x[u][v] = t[c0 + 64 * v < n ? c0 + 64 * v : n - 1];
      }
#pragma unroll
      for (int u = 0; u < FR; ++u) {
        const int i = i0 + u;
        const bool neg = i < m && sense && sense[i] == 2;
#pragma unroll
        for (int v = 0; v < FC; ++v) {
          const int j = c0 + 64 * v;
          if (i < m && j <= n) {
            if (j < n) am = fmax(am, fabs(x[u][v]));
            tab[(int64_t)i * ld + j] = j < n ? T(neg ? -x[u][v] : x[u][v]) : T(0);
          }
        }
      }
    });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) am = fmax(am, __shfl_xor(am, off));
    if (lane == 0) s_am[tid >> 6] = am;
    for (int i = tid; i < R; i += NT) {
      const bool neg = i >= 2 && sense && sense[i - 2] == 2;
      rhs[i] = i >= 2 ? T(neg ? -b[i - 2] : b[i - 2]) : T(0);
      bs[i] = i >= 2 ? n + i - 2 : -1;
      redund[i] = 0;
      rstep[i] = -1;
    }
    for (int j = tid; j < C; j += NT) {
      row0[j] = (j >= 1 && j <= n) ? T(-c[j - 1]) : T(0);
      row1[j] = T(0);
      nb[j] = j == 0 ? -1 : (j <= n ? j - 1 : n + m);
      dead[j] = (j == 0 || j == C - 1) ? 1 : 0;
      cstep[j] = -1;
    }
    __syncthreads();
  }

  __device__ __forceinline__ bool set_target(const int32_t* warm) {
    if (!warm) return false;
    for (int v = threadIdx.x; v < n + m; v += NT) target[v] = 0;
    __syncthreads();
    int any = 0;
    for (int i = threadIdx.x; i < m; i += NT) {
      const int v = warm[i];
      if (v >= 0 && v < n + m) { target[v] = 1; any = 1; }
    }
    return __syncthreads_or(any) != 0;
  }

  // entry (i, j) brought up to date from its slab value (i, j: tableau indices)
  __device__ __forceinline__ T current(int i, int j, T x) const {
    const int rs = rstep[i], cs = cstep[j], k0 = rs > cs ? rs : cs;
    x = k0 < 0 ? x : rs >= cs ? T(-0.0) : T(0);  // replaced: starts anew at that step
    // (the whole panel's operands go out together; steps outside [k0, q) are not applied)
    T a[kPanel], p[kPanel];
#pragma unroll
    for (int k = 0; k < kPanel; ++k) {
      const int kk = k < q ? k : 0;
      a[k] = pa[kk * R + i];
      p[k] = pp[kk * C + j];
    }
#pragma unroll
    for (int k = 0; k < kPanel; ++k)
      if (k < q) x = k >= k0 ? fma_t(a[k], p[k], x) : x;
    return x;
  }
  // pa[q]: the negated column s (objective rows in front)
  __device__ __forceinline__ void fetch_col(int s) {
    __syncthreads();
    T* a = pa + q * R;
    constexpr int U = 4;  // rows per thread in flight
    for (int i0 = 2 + (int)threadIdx.x; i0 < R; i0 += U * NT) {
      T x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * NT;
        x[u] = tab[(int64_t)((i < R ? i : R - 1) - 2) * ld + s - 1];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * NT;
        if (i < R) a[i] = -current(i, s, x[u]);
      }
    }
    if (threadIdx.x == 0) {
      a[0] = -row0[s];
      a[1] = -row1[s];
    }
    __syncthreads();
    col_ready = s;
  }
  // f(j, entry (r, j)) for every nonbasic column j, each by the thread that owns it
  template <class F>
  __device__ __forceinline__ void for_row(int r, F&& f) {
    constexpr int U = 4;
    for (int j0 = 1 + (int)threadIdx.x; j0 < C; j0 += U * NT) {
      T x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 + u * NT;
        x[u] = tab[(int64_t)(r - 2) * ld + (j < C ? j : C - 1) - 1];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 + u * NT;
        if (j < C) f(j, current(r, j, x[u]));
      }
    }
  }

  // Blocks of FR rows x FC x 64 columns of the slab's m x (n + 1) entries, one after the other
  // per wavefront: f(row, first column of this lane); columns of a lane are 64 apart.
  static constexpr int FR = 8, FC = 4;
  template <class F>
  __device__ __forceinline__ void for_blocks(F&& f) const {
    const int ncb = (n + 1 + 64 * FC - 1) / (64 * FC), nrb = (m + FR - 1) / FR;
    for (int u = threadIdx.x >> 6; u < nrb * ncb; u += NW) {
      const int rb = u / ncb;
      f(rb * FR, (u - rb * ncb) * 64 * FC + (int)(threadIdx.x & 63));
    }
  }

  // Applies the pending pivots to the slab.  One pass of plain FMAs over it, all loads of a
  // block in flight together; then the rows and columns that pending pivots replaced (at most
  // one each per pivot), whose entries start anew inside the panel.
  __device__ __forceinline__ void flush() {
    __syncthreads();
    const int nc = n + 1;
    for_blocks([&](int i0, int c0) {
      T x[FR][FC];
#pragma unroll
      for (int u = 0; u < FR; ++u) {
        const T* t = tab + (int64_t)(i0 + u < m ? i0 + u : m - 1) * ld;
#pragma unroll
        for (int v = 0; v < FC; ++v) x[u][v] = t[c0 + 64 * v < nc ? c0 + 64 * v : nc - 1];
      }
      for (int k = 0; k < q; ++k) {
        T p[FC], a[FR];
#pragma unroll
        for (int v = 0; v < FC; ++v) p[v] = pp[k * C + 1 + (c0 + 64 * v < nc ? c0 + 64 * v : nc - 1)];
#pragma unroll
        for (int u = 0; u < FR; ++u) a[u] = pa[k * R + 2 + (i0 + u < m ? i0 + u : m - 1)];
#pragma unroll
        for (int u = 0; u < FR; ++u)
#pragma unroll
          for (int v = 0; v < FC; ++v) x[u][v] = fma_t(a[u], p[v], x[u][v]);
      }
#pragma unroll
      for (int u = 0; u < FR; ++u)
#pragma unroll
        for (int v = 0; v < FC; ++v)
          if (i0 + u < m && c0 + 64 * v < nc) tab[(int64_t)(i0 + u) * ld + c0 + 64 * v] = x[u][v];
    });
    __syncthreads();
    for (int k = 0; k < q; ++k) {
      const int r = uniform(stepr[k]), c = uniform(stepc[k]);
      if (uniform((int)rstep[r]) == k)
        for (int j = 1 + (int)threadIdx.x; j < C; j += NT) tab[(int64_t)(r - 2) * ld + j - 1] = current(r, j, T(0));
      if (uniform((int)cstep[c]) == k)
        for (int i = 2 + (int)threadIdx.x; i < R; i += NT) tab[(int64_t)(i - 2) * ld + c - 1] = current(i, c, T(0));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < R; i += NT) rstep[i] = -1;
    for (int j = threadIdx.x; j < C; j += NT) cstep[j] = -1;
    q = 0;
    col_ready = -1;
    __syncthreads();
  }

  __device__ __forceinline__ int bs_of(int i) {
    __syncthreads();
    return uniform(bs[i]);
  }
  __device__ __forceinline__ int bs_now(int i) { return bs_of(i); }
  __device__ __forceinline__ int warm_at(const int32_t* warm, int ci) const { return warm[ci]; }
  __device__ __forceinline__ int nb_of(int j) {
    __syncthreads();
    return uniform(nb[j]);
  }

  __device__ __forceinline__ int pricing(int orow, bool bland, T eps_d) {
    const T* row = orow == 0 ? row0 : row1;
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int j = 1 + (int)threadIdx.x; j < C; j += NT) {
      const T d = row[j];
      if (dead[j] || !(d < -eps_d)) continue;
      const T v = bland ? T(nb[j]) : d;
      if (better(v, j, bv, bk)) { bv = v; bk = j; bp = j; }
    }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ int ratio(int s, bool bland, T eps_p, T& theta) {
    fetch_col(s);
    const T* a = pa + q * R;
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      const T x = -a[i];
      if (!(x > eps_p)) continue;
      const T beta = rhs[i];
      const T th = (beta > T(0) ? beta : T(0)) / x;
      const T v = th > T(0) ? th : -x;  // degenerate rows: largest pivot first
      const int k = bland ? bs[i] : i;
      if (better(v, k, bv, bk)) { bv = v; bk = k; bp = i; }
    }
    red.argmin(bv, bk, bp);
    theta = bv > T(0) ? bv : T(0);
    return bp;
  }

  __device__ __forceinline__ void pivot(int r, int s) {
    if (col_ready != s) fetch_col(s);
    T* a = pa + q * R;
    T* p = pp + q * C;
    const T rp = T(1) / uniform(-a[r]), prow0 = uniform(rhs[r]) * rp;
    const T a0 = uniform(a[0]), a1 = uniform(a[1]);
    for_row(r, [&](int j, T x) {
      const T pr = j == s ? rp : x * rp;
      p[j] = pr;
      row0[j] = fma_t(a0, pr, j == s ? T(0) : row0[j]);
      row1[j] = fma_t(a1, pr, j == s ? T(0) : row1[j]);
    });
    __syncthreads();  // every read of rhs[r] and a[r] is behind
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) rhs[i] = i == r ? prow0 : fma_t(a[i], prow0, rhs[i]);
    if (threadIdx.x == 0) {
      row0[0] = fma_t(a0, prow0, row0[0]);
      row1[0] = fma_t(a1, prow0, row1[0]);
      const int t = bs[r];
      bs[r] = nb[s];
      nb[s] = t;
      rstep[r] = (int8_t)q;
      cstep[s] = (int8_t)q;
      stepr[q] = r;
      stepc[q] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) a[r] = T(1);
    ++q;
    col_ready = -1;
    if (q == K) flush();
    else __syncthreads();
  }

  // row of largest |T[i][s]| among constraint rows whose basic variable is not a target
  __device__ __forceinline__ int absmax_row(int s, T eps_p) {
    fetch_col(s);
    const T* a = pa + q * R;
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      const int v = bs[i];
      if (redund[i] || v < 0 || (v < n + m && target[v])) continue;
      const T key = -tabs(a[i]);
      if (better(key, i, bv, bk)) { bv = key; bk = i; bp = i; }
    }
    red.argmin(bv, bk, bp);
    if (bp < 0 || !(-bv > eps_p)) return -1;
    return bp;
  }

  __device__ __forceinline__ int absmax_col(int r, T eps_p) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for_row(r, [&](int j, T x) {
      if (dead[j]) return;
      const T v = -tabs(x);
      if (better(v, j, bv, bk)) { bv = v; bk = j; bp = j; }
    });
    red.argmin(bv, bk, bp);
    if (bp < 0 || !(-bv > eps_p)) return -1;
    return bp;
  }

  // dual simplex leaving row: most negative rhs below -tol (Bland: smallest basic id)
  __device__ __forceinline__ int dual_row(bool bland, T tol) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      const T beta = rhs[i];
      if (redund[i] || !(beta < -tol)) continue;
      const T key = bland ? T(bs[i]) : beta;
      if (better(key, i, bv, bk)) { bv = key; bk = i; bp = i; }
    }
    red.argmin(bv, bk, bp);
    return bp;
  }

  // dual simplex entering column for leaving row r
  __device__ __forceinline__ int dual_ratio(int r, bool bland, T eps_p, T& theta) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for_row(r, [&](int j, T a) {
      if (dead[j] || !(a < -eps_p)) return;
      const T d = row0[j];
      const T th = (d > T(0) ? d : T(0)) / -a;
      const T key = th > T(0) ? th : a;
      const int kk = bland ? nb[j] : j;
      if (better(key, kk, bv, bk)) { bv = key; bk = kk; bp = j; }
    });
    red.argmin(bv, bk, bp);
    theta = bv > T(0) ? bv : T(0);
    return bp;
  }

  // a dead column never enters again; it keeps its values (B^-1 columns of fixed slacks stay
  // available to the FP64 check)
  __device__ __forceinline__ void kill_col(int j) {
    __syncthreads();
    if (threadIdx.x == 0) dead[j] = 1;
    __syncthreads();
  }

  // only the right-hand side (column 0) is read and written this way by the driver
  __device__ __forceinline__ T get(int i, int) {
    __syncthreads();
    return uniform(i == 1 ? row1[0] : rhs[i]);
  }
  __device__ __forceinline__ void set(int i, int, T v) {
    __syncthreads();
    if (threadIdx.x == 0) rhs[i] = v;
    __syncthreads();
  }
  __device__ __forceinline__ void mark_redund(int r) {
    __syncthreads();
    if (threadIdx.x == 0) { redund[r] = 1; rhs[r] = T(0); }
    __syncthreads();
  }

  __device__ __forceinline__ int min_rhs_row() {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT) {
      if (redund[i]) continue;
      const T v = rhs[i];
      if (better(v, i, bv, bk)) { bv = v; bk = i; bp = i; }
    }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ void setup_x0() {
    flush();
    const int x0 = C - 1;
    for (int i = threadIdx.x; i < m; i += NT) tab[(int64_t)i * ld + n] = redund[i + 2] ? T(0) : T(-1);
    for (int j = threadIdx.x; j < C; j += NT) row1[j] = j == x0 ? T(1) : T(0);
    if (threadIdx.x == 0) { row0[x0] = T(0); dead[x0] = 0; }
    __syncthreads();
  }

  __device__ __forceinline__ int find_basic(int var) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int i = 2 + (int)threadIdx.x; i < R; i += NT)
      if (bs[i] == var) { bv = T(0); bk = i; bp = i; }
    red.argmin(bv, bk, bp);
    return bp;
  }
  __device__ __forceinline__ int find_nonbasic(int var) {
    __syncthreads();
    T bv = inf_of<T>();
    int bk = INT_MAX, bp = -1;
    for (int j = 1 + (int)threadIdx.x; j < C; j += NT)
      if (nb[j] == var) { bv = T(0); bk = j; bp = j; }
    red.argmin(bv, bk, bp);
    return bp;
  }

  __device__ __forceinline__ void write_outputs(int lp, const LpDesc& d, const Out& out, int status, int it,
                                int p1, int unb, T wfin, int last) {
    if (out.tab && q > 0) flush();
    __syncthreads();
    const int tid = threadIdx.x;
    if (tid == 0) {
      double am = s_am[0];
      for (int w = 1; w < NW; ++w) am = fmax(am, s_am[w]);
      out.amax[lp] = am;
      out.status[lp] = status;
      out.pivots[lp] = it;
      out.p1[lp] = p1;
      out.unb[lp] = unb;
      if (out.lastpiv) out.lastpiv[lp] = last;
      out.obj[lp] = (double)row0[0];
      out.wfin[lp] = (double)wfin;
    }
    double* x = out.x + d.x;
    int32_t* basis = out.basis + d.basis;
    for (int j = tid; j < n; j += NT) x[j] = 0.0;
    for (int i = tid; i < m; i += NT) basis[i] = bs[2 + i];
    __syncthreads();
    for (int i = 2 + tid; i < R; i += NT) {
      const int v = bs[i];
      if (v >= 0 && v < n) x[v] = (double)rhs[i];
    }
    // final tableau and nonbasic ids for the FP64 check (B^-1 is in the slack columns)
    if (out.tab) {
      T* tp = (T*)(out.tab + 8 * d.t);
      for (int j = tid; j < C; j += NT) {
        tp[j] = row0[j];
        tp[C + j] = row1[j];
      }
      for (int i = tid; i < m; i += NT) tp[(int64_t)(i + 2) * C] = rhs[i + 2];
      for_blocks([&](int i0, int c0) {
        T v[FR][FC];
#pragma unroll
        for (int u = 0; u < FR; ++u)
#pragma unroll
          for (int w = 0; w < FC; ++w)
            v[u][w] = tab[(int64_t)(i0 + u < m ? i0 + u : m - 1) * ld + (c0 + 64 * w <= n ? c0 + 64 * w : n)];
#pragma unroll
        for (int u = 0; u < FR; ++u)
#pragma unroll
          for (int w = 0; w < FC; ++w)
            if (i0 + u < m && c0 + 64 * w <= n) tp[(int64_t)(i0 + u + 2) * C + 1 + c0 + 64 * w] = v[u][w];
      });
      int32_t* np = (int32_t*)(out.tab + 8 * (d.t + (int64_t)R * C));
      for (int j = tid; j < C; j += NT) np[j] = nb[j];
    }
  }
};

// VLDS: the vectors are in LDS, else behind the slab.  ws_stride: bytes per workgroup, the
// first slab_bytes of them the slab.
template <typename T, int NT, bool VLDS>
__global__ __launch_bounds__(NT) void k_panel(const LpDesc* __restrict__ desc,
                                              const double* __restrict__ pool,
                                              const int8_t* __restrict__ spool,
                                              const int32_t* __restrict__ idx, int32_t count,
                                              const int32_t* count_dev, int32_t* queue,
                                              Out out, Opt<T> o, char* ws, int64_t ws_stride,
                                              int64_t slab_bytes, int panel, int rcap, int ccap,
                                              const int32_t* __restrict__ warm_pool) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_q;
  __shared__ double s_am[NT / 64];
  __shared__ RedSlot<T> slots[2 * (NT / 64)];
  __shared__ int stepr[kPanel], stepc[kPanel];
  const PanelLayout L((int)sizeof(T), panel, rcap, ccap);
  char* slab = ws + (int64_t)blockIdx.x * ws_stride;
  char* vec = VLDS ? (char*)smem : slab + slab_bytes;
  PanelTab<T, NT> t;
  t.s_am = s_am;
  t.tab = (T*)slab;
  t.row0 = (T*)(vec + L.row0); t.row1 = (T*)(vec + L.row1); t.rhs = (T*)(vec + L.rhs);
  t.pa = (T*)(vec + L.pa); t.pp = (T*)(vec + L.pp);
  t.bs = (int*)(vec + L.bs); t.nb = (int*)(vec + L.nb);
  t.dead = (uint8_t*)(vec + L.dead); t.redund = (uint8_t*)(vec + L.redund);
  t.target = (uint8_t*)(vec + L.target);
  t.cstep = (int8_t*)(vec + L.cstep); t.rstep = (int8_t*)(vec + L.rstep);
  t.stepr = stepr; t.stepc = stepc;
  t.K = panel;
  t.blk = -1;
  t.red.init(slots);
  if (count_dev) count = *count_dev;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_q = atomicAdd(queue, 1);
    __syncthreads();
    const int q = uniform(s_q);
    if (q >= count) break;
    const int lp = idx ? idx[q] : q;
    const LpDesc d = desc[lp];
    t.m = d.m; t.n = d.n; t.R = d.m + 2; t.C = d.n + 2; t.ld = panel_ld(d.n);
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
// host side

static size_t stream_layout(int precision, int nt, int rcap, int ccap) {
  return precision == 0 ? StreamLayout<double>(nt / 64, rcap, ccap).total
                        : StreamLayout<float>(nt / 64, rcap, ccap).total;
}

// Panel of a shape: 8 pending pivots in LDS where they fit 144 KB (one workgroup per CU;
// FP64 to about 800 x 800), fewer while at least 2 fit, else 8 with every vector in HBM.
static void panel_plan(int precision, int rcap, int ccap, int& k, bool& vlds) {
  const int esz = precision == 0 ? 8 : 4;
  for (k = kPanel; k >= 2; --k)
    if (PanelLayout(esz, k, rcap, ccap).total <= 144 * 1024) {
      vlds = true;
      return;
    }
  k = kPanel;
  vlds = false;
}
static int64_t panel_slab(int precision, int rcap, int ccap) {
  const int64_t b = (precision == 0 ? 8 : 4) * (int64_t)(rcap - 2) * panel_ld(ccap - 2);
  return (b + 255) & ~255ll;
}

size_t stream_lds_bytes(int precision, bool lds_tab, int nt, int rcap, int ccap) {
  if (lds_tab) return stream_layout(precision, nt, rcap, ccap);
  int k;
  bool vlds;
  panel_plan(precision, rcap, ccap, k, vlds);
  return vlds ? PanelLayout(precision == 0 ? 8 : 4, k, rcap, ccap).total : 0;
}

// HBM bytes per workgroup of the streamed kernel
size_t stream_ws_bytes(int precision, int rcap, int ccap) {
  int k;
  bool vlds;
  panel_plan(precision, rcap, ccap, k, vlds);
  size_t b = (size_t)panel_slab(precision, rcap, ccap);
  if (!vlds) b += (PanelLayout(precision == 0 ? 8 : 4, k, rcap, ccap).total + 255) & ~(size_t)255;
  return b;
}

template <typename T>
static const void* stream_fn(bool lds_tab, bool vlds, int nt) {
  switch (nt) {
#define BLPG_PICK(N)                                                                          \
  case N:                                                                                     \
    return lds_tab ? reinterpret_cast<const void*>(&k_stream<T, N>)                           \
                   : vlds ? reinterpret_cast<const void*>(&k_panel<T, N, true>)               \
                          : reinterpret_cast<const void*>(&k_panel<T, N, false>);
    BLPG_PICK(64) BLPG_PICK(128) BLPG_PICK(256) BLPG_PICK(512)
#undef BLPG_PICK
    default: return nullptr;
  }
}

static const void* stream_kernel_ptr(int precision, bool lds_tab, int nt, int rcap, int ccap) {
  int k = 0;
  bool vlds = false;
  if (!lds_tab) panel_plan(precision, rcap, ccap, k, vlds);
  return precision == 0 ? stream_fn<double>(lds_tab, vlds, nt) : stream_fn<float>(lds_tab, vlds, nt);
}

hipError_t launch_stream(const StreamLaunch& L, hipStream_t st) {
  const void* fn = stream_kernel_ptr(L.precision, L.lds_tab, L.nt, L.rcap, L.ccap);
  if (!fn) return hipErrorInvalidValue;
  const size_t lds = stream_lds_bytes(L.precision, L.lds_tab, L.nt, L.rcap, L.ccap);
  Opt<double> o64{L.eps_d, L.eps_p, L.tol, L.max_iter, L.bland_after};
  Opt<float> o32{(float)L.eps_d, (float)L.eps_p, (float)L.tol, L.max_iter, L.bland_after};
  void* o = L.precision == 0 ? (void*)&o64 : (void*)&o32;
  if (L.lds_tab) {
    void* args[] = {(void*)&L.desc, (void*)&L.pool, (void*)&L.spool, (void*)&L.idx,
                    (void*)&L.count, (void*)&L.count_dev, (void*)&L.queue, (void*)&L.out, o,
                    (void*)&L.rcap, (void*)&L.ccap, (void*)&L.warm};
    return hipLaunchKernel(fn, dim3(L.grid), dim3(L.nt), args, lds, st);
  }
  int k;
  bool vlds;
  panel_plan(L.precision, L.rcap, L.ccap, k, vlds);
  const int64_t stride = (int64_t)stream_ws_bytes(L.precision, L.rcap, L.ccap);
  const int64_t slab = panel_slab(L.precision, L.rcap, L.ccap);
  void* args[] = {(void*)&L.desc, (void*)&L.pool, (void*)&L.spool, (void*)&L.idx,
                  (void*)&L.count, (void*)&L.count_dev, (void*)&L.queue, (void*)&L.out, o,
                  (void*)&L.ws, (void*)&stride, (void*)&slab, (void*)&k,
                  (void*)&L.rcap, (void*)&L.ccap, (void*)&L.warm};
  return hipLaunchKernel(fn, dim3(L.grid), dim3(L.nt), args, lds, st);
}

int stream_max_blocks_per_cu(int precision, bool lds_tab, int nt, int rcap, int ccap) {
  const void* fn = stream_kernel_ptr(precision, lds_tab, nt, rcap, ccap);
  if (!fn) return 0;
  int nb = 0;
  const size_t lds = stream_lds_bytes(precision, lds_tab, nt, rcap, ccap);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, nt, lds) != hipSuccess) return 0;
  return nb;
}

}  // namespace blpg
