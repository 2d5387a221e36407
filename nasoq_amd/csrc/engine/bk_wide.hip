// Cooperative panel Bunch-Kaufman for very wide diagonal blocks (the root
// separators of KKT matrices), LAPACK dlasyf-style: the columns of a panel
// of nb <= 64 columns are formed left-looking from the panel's L and
// W = L D, pivots follow the dsytf2 rules (alpha = (1+sqrt(17))/8) on the
// fully updated columns, and the rank-nb trailing update runs afterwards in
// k_trailing.  Reference: LAPACKE_dsytrf on the diagonal block at
// src/ldl/parallel_blocked_ldlt_02.cpp:155 and the column permutation of the
// rows below it (LAPACKE_dlapmt, :164-165).
//
// Work split.  The rows [k0, r) of the panel are the nb "diagonal" rows
// [k0, k0+nb) and the "far" rows below them: the rest of the diagonal block
// and the supernode's off-diagonal rows [w, r), which get their L in the same
// steps (so no separate off-diagonal solve is needed) but are never pivot
// candidates.  G workgroups each own up to WCH far rows (one per thread of
// every wave but the last) and keep those rows of the panel (L for
// eliminated columns, A for pending ones) in LDS.  Every
// workgroup also keeps the diagonal rows (nb x nb) and computes their
// updated values itself, so the W row needed by each column step is always
// local.
//
// Exchange.  Per column step the workgroups publish one small record (the
// largest candidate of the column) as flag-in-word 64-bit values written
// and polled with agent-scope atomics; the flag is a per-step epoch, so the
// record is its own barrier.  A step that has to inspect a second column
// (absakk < alpha * colmax) adds the candidate row of the winning group
// (published speculatively with the record) and a second record round.
//
// Interchanges.  Within the panel nothing is written to the matrix: the
// interchange of logical rows/columns kk and kp only updates a
// logical-to-physical map (the diagonal rows' map and a table of moved far
// rows) and the LDS row copies.  At the end of the panel the accumulated
// permutation is applied in place, through a scratch copy between two group
// barriers, to the trailing block, to the earlier columns of L and to the
// columns of the rows below the diagonal block; then L and W of the panel
// are written.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

#include "engine/device_util.hpp"
#include "engine/kernels.hpp"

namespace lblg {

#define WNB 64                         // widest panel
#define WMM (2 * WNB)                  // moved indices per panel
#define OSB 16                         // columns per sub-block of the optimistic pass
#define LL_SPIN (1L << 22)

// exchange buffer layout, in 64-bit words (see kernels.hpp: LL_WORDS)
#define LL_RECA 0                            // [2][256][4]
#define LL_RECB (LL_RECA + 2 * 256 * 4)      // [2][256][8]
#define LL_PAY (LL_RECB + 2 * 256 * 8)       // [2][256][2 * WNB]

static_assert(LL_PAY + 2 * 256 * 2 * WNB == LL_WORDS, "exchange buffer size");

__device__ inline void ll_store(uint64_t* p, uint32_t v, uint32_t flag) {
  __hip_atomic_store(p, ((uint64_t)flag << 32) | (uint64_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The first wait of a factorization that runs out records where: status[8]
// = site + 16 x (word index - ll), status[9] = the waiting workgroup,
// status[10] = the flag it waited for, status[11] = the flag it last saw.
struct LlDiag {
  int* status;
  int site;
  int g;
  const uint64_t* base;
};
__device__ inline void ll_note(const LlDiag& d, const uint64_t* p, uint32_t flag, uint32_t seen) {
  if (atomicCAS(d.status + 8, 0, d.site + 16 * (int)(p - d.base)) == 0) {
    d.status[9] = d.g;
    d.status[10] = (int)flag;
    d.status[11] = (int)seen;
  }
}
// wait (bounded) for the word to carry this epoch's flag; abort != 0 skips the wait
__device__ inline uint32_t ll_load(uint64_t* p, uint32_t flag, int& abort, const LlDiag& d) {
  long spins = 0;
  while (!abort) {
    const uint64_t x = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((uint32_t)(x >> 32) == flag) return (uint32_t)x;
    if (++spins > LL_SPIN) {
      abort = 1;
      ll_note(d, p, flag, (uint32_t)(x >> 32));
    }
  }
  return 0u;
}
__device__ inline void ll_store_d(uint64_t* p, double v, uint32_t flag) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  ll_store(p, (uint32_t)b, flag);
  ll_store(p + 1, (uint32_t)(b >> 32), flag);
}
__device__ inline double ll_load_d(uint64_t* p, uint32_t flag, int& abort, const LlDiag& d) {
  const uint64_t lo = ll_load(p, flag, abort, d);
  const uint64_t hi = ll_load(p + 1, flag, abort, d);
  return __longlong_as_double((long long)((hi << 32) | lo));
}

// W(i, j) = sum_c L(i, c) D(c, j) for an eliminated panel column j; l(j) reads L(i, j)
template <typename F, typename T>
__device__ inline double w_entry(F l, int j, const T* dd, const T* dsb) {
  if (dsb[j] != 0.0) return l(j) * dd[j] + l(j + 1) * dsb[j];
  if (j > 0 && dsb[j - 1] != 0.0) return l(j - 1) * dsb[j - 1] + l(j) * dd[j];
  return l(j) * dd[j];
}

// largest value over the wave's lanes (all lanes get it): DPP row shifts and
// row broadcasts, a few cycles a stage where a shuffle through the LDS takes
// a hundred
template <int CTRL, int ROWS>
__device__ inline double dpp_max(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = (int)b, hi = (int)(b >> 32);
  const unsigned olo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
  const unsigned ohi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
  return fmax(v, __longlong_as_double((long long)(((uint64_t)ohi << 32) | olo)));
}
__device__ inline double lane_read(double v, int l);
__device__ inline double wave_max(double v) {
  v = dpp_max<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_max<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return lane_read(v, 63);
}
// Argmax over the workgroup of (v, i), v >= 0 or -1 (no candidate), i
// ascending over a wave's lanes: the smallest index of the largest value.
// redv / redi hold two sets, used in turn, so a call has one barrier.
template <int NW>
__device__ inline void wg_argmax(double& v, int& i, double (*redv)[NW], int (*redi)[NW], int& turn) {
  const int wv = threadIdx.x >> 6;
  const double m = wave_max(v);
  const int first = __ffsll((unsigned long long)__ballot(v == m)) - 1;
  const int idx = __builtin_amdgcn_readlane(i, first < 0 ? 0 : first);
  turn ^= 1;
  if ((threadIdx.x & 63) == 0) {
    redv[turn][wv] = m;
    redi[turn][wv] = idx;
  }
  __syncthreads();
  double bv[NW];
  int bi[NW];
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    bv[q] = redv[turn][q];
    bi[q] = redi[turn][q];
  }
  v = bv[0];
  i = bi[0];
#pragma unroll
  for (int q = 1; q < NW; ++q) better(v, i, bv[q], bi[q]);
}

// lane `l` (uniform) of a double
__device__ inline double lane_read(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

__device__ inline int far_phys(int a, int fstart, const unsigned* mbits, const int* mlog, const int* mphys,
                               int nm) {
  const int b = a - fstart;
  if (!(mbits[b >> 5] & (1u << (b & 31)))) return a;
  for (int q = 0; q < nm; ++q)
    if (mlog[q] == a) return mphys[q];
  return a;
}

// Waves per SIMD to compile for: the FP32 panels of many supernodes share a
// CU, four workgroups with 128 registers (two spilled) instead of three.
template <typename T, int NT, int NBM, bool ONE>
constexpr int panel_waves() {
  return ONE && NT == 256 && NBM == 32 && sizeof(T) == 4 ? 4 : 1;
}

// NT threads per workgroup: waves 0 .. NT/64 - 2 own one far row per
// thread (WCH = NT - 64 rows per workgroup), the last wave computes the
// diagonal rows; NBM is the widest panel the launch takes.
//
// ONE = false, a cooperative group of G workgroups on one supernode: 256
// threads with 64-column panels keep 192 far rows per workgroup (G <= 256:
// 49,152 rows); 512 threads keep 448 (114,688 rows) with 32-column FP64 or
// 64-column FP32 panels, whose LDS rows are the same 256 bytes.
//
// ONE = true, one workgroup per listed supernode: the far rows are those of
// the diagonal block (at most WCH), the rows below it are left to
// k_offdiag, and every exchange stays inside the workgroup.
template <typename T, int NT, int NBM, bool ONE>
__global__ __launch_bounds__(NT, (panel_waves<T, NT, NBM, ONE>())) void k_bk_wide(
    WideSn sn, PanelList pl, int G, int nb, int sub, int wcols, T* valL, T* dval, int* perm_piv, T* Wbase, int* kpos,
    int* kstart, int* sync, int* sync_next, uint64_t* ll, uint32_t ebase, int n, int* status) {
  constexpr int NW = NT / 64;                   // waves; wave NW - 1 holds the diagonal rows
  constexpr int WCH = NT - 64;                  // far rows per workgroup
  constexpr int WLDA = NBM + 1;                 // padded row length of the diagonal rows
  constexpr int WLDC = WCH + 16;                // padded column length of the far rows: the k-groups of an MFMA
                                                // operand read fall into different banks
  constexpr int MBITS_WORDS = (ONE ? 1 : 256) * WCH / 32;  // moved-far-row bitmap
  static_assert(NBM <= WNB && NT % 64 == 0 && NT >= (ONE ? 128 : 256) && WCH % 32 == 0, "wide panel launch shape");
  __shared__ T LC[NBM * WLDC];      // own far rows, column-major [column][row]
  __shared__ T Ad[NBM * WLDA];      // diagonal rows: L below the diagonal and W(j, c) at (c, j) above it
                                    // (eliminated columns c) | symmetric A (pending)
  __shared__ T wk[NBM], wi[NBM], td0[NBM], td1[NBM], dd[NBM], dsb[NBM], prow[NBM];
  __shared__ int dphys[NBM];
  __shared__ int mlog[WMM], mphys[WMM], Ml[WMM], Mp[WMM];
  __shared__ unsigned mbits[MBITS_WORDS];
  __shared__ double redv[2][NW];
  __shared__ int redi[2][NW];
  __shared__ double bcd[4];
  __shared__ int bci[4];
  __shared__ int s_nm, s_abort, s_nM, s_nMa, s_fail;

  const int g = ONE ? 0 : blockIdx.x, t = threadIdx.x, wv = t >> 6, ln = t & 63;
  // consecutive cooperative launches alternate between two barrier counters:
  // this one counts from zero, and zeroes the other for the next launch (the
  // launch before used it and has ended; the next has not started)
  if (!ONE && g == 0 && t == 0) __hip_atomic_store(sync_next, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  int s, c0, w;
  int64_t r;
  T *A, *Wp;
  if constexpr (ONE) {
    s = pl.list[blockIdx.x];
    c0 = pl.super[s];
    w = pl.super[s + 1] - c0;
    r = pl.pi[s + 1] - pl.pi[s];
    A = valL + pl.px[s];
    Wp = Wbase + pl.woff[s];
    G = 1;
  } else {
    // the supernode's shape comes with the launch: the only load before the
    // panel's own is its first column (and the block's)
    s = sn.s;
    c0 = sn.c0;
    w = sn.w;
    r = sn.r;
    A = valL + sn.px;
    Wp = Wbase + sn.woff;
  }
  const T* Pp = Wp + (int64_t)w * wcols;  // this panel's columns with the block's earlier panels applied
  // scratch of the interchanges; one workgroup: in W's place, whose columns
  // are written after them (at most min(nb, w) moved indices squared)
  T* scr = ONE ? Wp : Wp + (int64_t)w * wcols + (int64_t)r * nb;
  const int k0 = kpos[s];
  if (k0 >= w) return;
  // sub > 0: this panel continues the block of panels that started at K0.
  // The matrix holds no contribution of the block's earlier panels (the
  // trailing block is updated once per block); this panel's columns with
  // those contributions applied are in Pp, and W holds the earlier panels'
  // columns [0, off)
  const int K0 = sub == 0 ? k0 : kstart[s];
  const int off = k0 - K0;
  const int nbe = min(nb, w - k0);
  const bool last = (w - k0) <= nb;
  // far rows: the rest of the diagonal block, then (cooperative panels) the
  // rows below it (those take part in every update and get their L here, but
  // are never pivots)
  const int rend = ONE ? w : (int)r;
  const int fstart = k0 + nbe, nfar = rend - fstart;
  const int chunk = nfar > 0 ? (nfar + G - 1) / G : 0;
  if (chunk > WCH || nb > NBM || off < 0 || off + nb > wcols) {  // uniform over the grid: every workgroup returns
    if (g == 0 && t == 0) atomicOr(status, 8);
    return;
  }
  const int fbeg = fstart + g * chunk;
  const int fcnt = max(0, min(chunk, rend - fbeg));
  const bool hasrow = t < fcnt;
  const int fr = fbeg + t;
  int myphys = fr;
#define AG(i, j) A[(int64_t)(j) * r + (i)]
#define LCR(j) LC[(j) * WLDC + t]
#define ADR(i, j) Ad[(i) * WLDA + (j)]

  // ---- load the panel rows
  // panel column j, row i >= j (with the block's earlier panels applied)
  auto pcol = [&](int i, int j) -> T { return sub ? Pp[(int64_t)j * r + i] : AG(i, k0 + j); };
  // all of a thread's loads issue before its first LDS store: one round trip
  {
    // diagonal rows (lower triangle): lane = row, the waves share the columns
    constexpr int Q = (NBM + NW - 1) / NW;
    T v[Q], f[NBM];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ln, j = wv + NW * q;
      v[q] = (i < nbe && j <= i) ? pcol(k0 + i, j) : (T)0;
    }
#pragma unroll
    for (int j = 0; j < NBM; ++j) f[j] = (hasrow && j < nbe) ? pcol(fr, j) : (T)0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ln, j = wv + NW * q;
      if (i < nbe && j <= i) ADR(i, j) = v[q];
    }
    if (hasrow) {
#pragma unroll
      for (int j = 0; j < NBM; ++j)
        if (j < nbe) LCR(j) = f[j];
    }
  }
  if (t < NBM) {
    dphys[t] = k0 + t;
    dd[t] = 0.0;
    dsb[t] = 0.0;
  }
  for (int q = t; q < MBITS_WORDS; q += NT) mbits[q] = 0u;
  if (t == 0) {
    s_nm = 0;
    s_abort = 0;
  }

  // Two ways of taking steps alternate.
  //
  // ---- Optimistic pass.  Bunch-Kaufman keeps the diagonal pivot of column
  // k without interchange when |a_kk| >= alpha * max_{i>k, i<w} |a_ik| on the
  // updated column.  Every workgroup runs the steps of columns [kr, ke) on
  // that assumption with no exchange, and each thread notes the first step
  // at which one of its candidate rows breaks the test.  One exchange then
  // gives the first failing step J: the steps before it are Bunch-Kaufman's
  // own on the same values, and the columns from J on get their values back.
  // The first pass covers the whole panel (one workgroup: up to the sub-block
  // that fails); after a pivot search found RESUME columns in a row that
  // needed none, a pass covers the next OSB columns.
  // The steps run in sub-blocks of OSB columns.  A sub-block's columns first
  // receive the eliminated columns' contribution as 16x16 MFMA tiles,
  // a(i,j) -= sum_c L(i,c) W(j,c); inside the sub-block every wave computes
  // the diagonal rows itself, so the steps need no block barrier.
  // What bounds the panel is the chain of nbe dependent steps, so a step
  // keeps its operands in registers.  Per 64-column FP64 panel of a 64^3 KKT
  // (476 panels, workgroup 0, phase stamps): load 8.1 us, MFMA 11.4, steps
  // 23.3 (0.36 us each), exchange 1.8, pivot search 3.6 (averaged; 6 panels
  // take it), restore and interchanges 1.5, write 9.1.  With the columns in
  // LDS and one sum per step over the sub-block's earlier columns a launch
  // took 115 us on average, now 60 (kernel traces; FP32 panels of a 48^3 KKT:
  // 124 -> 63; where 14 of 476 panels take the search, FP64 68).
  // The price is registers: 252 vector registers for the cooperative FP64
  // form (106 before) and 150 to 290 scalar ones kept in vector lanes, which
  // costs no residency (the LDS allows one workgroup a CU); the 1024-thread
  // form has 128 and spills 19 of them in FP64 (3 in FP32).
  //
  // ---- Pivot step.  One step of the search at column kr on left-looking
  // sums over the eliminated columns: a record exchange per step, a second
  // one when another column has to be inspected.
  constexpr int RESUME = 4;
  int turn = 0;                     // wg_argmax
  int n_second = 0, n_swap = 0;     // pivoting statistics (workgroup 0)
  int kr = 0, step = 0, pass = 0, good = RESUME;
  bool plain = true;  // every step so far a 1x1 pivot in place
  const int kstop = last ? nbe : nb - 1;  // a 2x2 pivot must not straddle panels
  if constexpr (ONE) {
    // a first column that fails the test needs no pass to show it (indefinite
    // blocks fail at almost every column)
    __syncthreads();
    const double a00 = fabs((double)ADR(0, 0));
    const bool bad = !(a00 > 0.0) | (hasrow && BK_ALPHA * fabs((double)LCR(0)) > a00) |
                     (wv == NW - 1 && ln > 0 && ln < nbe && BK_ALPHA * fabs((double)ADR(ln, 0)) > a00);
    if (__syncthreads_or(bad)) {
      for (int j = wv; j < nbe; j += NW)
        if (ln > j && ln < nbe) ADR(j, ln) = ADR(ln, j);
      good = 0;
      pass = 1;
      __syncthreads();
    }
  }
  while (kr < nbe && (pass == 0 || kr < kstop)) {
    if (good >= RESUME && (pass == 0 || nbe - kr >= 8)) {
      const bool first = pass == 0;
      const int ke = first ? nbe : min(nbe, kr + OSB);
      const bool drow = ln < nbe;
      const int li = ln & 15, lk = ln >> 4;
      int myfail = ke;
      if (t == 0) s_fail = ke;
      // the sub-block's original columns of this lane's rows (cooperative
      // panels after the first pass; elsewhere they are read again)
      T vo[ONE ? 1 : OSB], vdo[ONE ? 1 : OSB];
      __syncthreads();
      int cb = kr;
      for (; cb < ke; cb += OSB) {
        const int ce = min(ke, cb + OSB);
        if constexpr (!ONE) {
          if (!first) {
#pragma unroll
            for (int q = 0; q < OSB; ++q) {
              const int j = cb + q;
              vo[q] = (hasrow && j < ce) ? LCR(j) : (T)0;
              vdo[q] = (drow && j < ce && ln >= j) ? ADR(ln, j) : (T)0;
            }
          }
        }
        if (cb > 0) {
          __syncthreads();
          if (ONE && first && s_fail < cb) break;  // uniform: written before the barrier, not again before the next
          // a wave takes its far-row tiles (rows < WCH) and at most one
          // diagonal tile (rows [cb, nbe)) in lockstep: independent
          // accumulators hide the operand loads and the MFMA latency.  Tiles
          // and columns beyond the rows compute on whatever the LDS holds
          // and store nothing.
          constexpr int NFT = WCH / 16, TPW = (NFT + NW - 1) / NW;
          static_assert(WCH % 16 == 0 && (NBM + OSB - 1) / OSB <= NW, "far-row and diagonal tiles per wave");
          const bool dtile = wv < ((nbe - cb + 15) >> 4);
          const int id0 = cb + (dtile ? 16 * wv : 0);
          typename Mfma<T>::acc acc[TPW], accd = {0, 0, 0, 0};
          int i0[TPW];
#pragma unroll
          for (int u = 0; u < TPW; ++u) {
            acc[u] = typename Mfma<T>::acc{0, 0, 0, 0};
            i0[u] = 16 * min(wv + NW * u, NFT - 1);
          }
          // operands of the next k-step are read while this step's MFMAs run;
          // columns c >= cb of the last k-step count as zero
          const int xc = min(cb + li, NBM - 1), dr = min(id0 + li, NBM - 1);
          T x, y[TPW], yd;
          auto fetch = [&](int c) {
            const int cc = min(c + lk, cb - 1);
            // first operand row = column j of the sub-block (W(j, c)), second operand col = row i (L(i, c))
            x = c + lk < cb ? ADR(cc, xc) : (T)0;
#pragma unroll
            for (int u = 0; u < TPW; ++u) y[u] = c + lk < cb ? LC[cc * WLDC + i0[u] + li] : (T)0;
            yd = c + lk < cb ? ADR(dr, cc) : (T)0;
          };
          fetch(0);
          for (int c = 0; c < cb; c += 4) {
            const T x0 = x, yd0 = yd;
            T y0[TPW];
#pragma unroll
            for (int u = 0; u < TPW; ++u) y0[u] = y[u];
            fetch(c + 4 < cb ? c + 4 : c);
#pragma unroll
            for (int u = 0; u < TPW; ++u) acc[u] = Mfma<T>::mma(x0, y0[u], acc[u]);
            accd = Mfma<T>::mma(x0, yd0, accd);
          }
          __syncthreads();  // every operand is read: pending entries may change
          // acc[e] = C(j = cb + orow(e), i = i0 + li)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = cb + Mfma<T>::orow(e, ln);
            if (j < ce) {
#pragma unroll
              for (int u = 0; u < TPW; ++u) {
                const int i = i0[u] + li;
                if (wv + NW * u < NFT && i < fcnt) LC[j * WLDC + i] -= acc[u][e];
              }
              const int i = id0 + li;
              if (dtile && i < nbe && i >= j) ADR(i, j) -= accd[e];
            }
          }
          __syncthreads();
        }
        // the steps themselves: the sub-block's columns of this lane's far row
        // (vf) and of diagonal row ln (vd, the same in every wave) in
        // registers, right-looking; the W row of a step is read across the
        // lanes (v_readlane), so a step has no LDS access and no barrier on its
        // critical path: d, its reciprocal, one multiplication, one FMA.
        // Columns beyond ce run on zeros and are neither tested nor stored.
        double vf[OSB], vd[OSB], rks = 0.0, ds = 0.0;
#pragma unroll
        for (int q = 0; q < OSB; ++q) {
          const int j = cb + q;
          vf[q] = (hasrow && j < ce) ? (double)LCR(j) : 0.0;
          vd[q] = (drow && j < ce && ln >= j) ? (double)ADR(ln, j) : 0.0;
        }
        __syncthreads();  // every wave has read the diagonal rows: the last one may store over them
        const bool fcand = hasrow && fr < w, dcand = wv == NW - 1 && drow;
        unsigned fm = 0;  // steps at which one of this lane's rows breaks the test
        double d = lane_read(vd[0], cb), rk = 1.0 / d;
#pragma unroll
        for (int q = 0; q < OSB; ++q) {
          const int kc = cb + q;
          // W and L entries as they are stored (in T)
          const T wT = (T)vd[q], lT = (T)(wT * (T)rk);
          const double wd = (double)wT, lf = (double)(T)(vf[q] * rk), ld = (double)lT;
          // the next step's pivot first: its reciprocal runs beside the other
          // columns' updates
          double dn = 0.0, rkn = 0.0;
          if (q + 1 < OSB) {
            const double wj = lane_read(wd, (kc + 1) & 63);
            vf[q + 1] -= lf * wj;
            vd[q + 1] -= ld * wj;
            dn = lane_read(vd[q + 1], (kc + 1) & 63);
            rkn = 1.0 / dn;
          }
#pragma unroll
          for (int j = q + 2; j < OSB; ++j) {
            const double wj = lane_read(wd, (cb + j) & 63);
            vf[j] -= lf * wj;
            vd[j] -= ld * wj;
          }
          const double absakk = fabs(d);
          const bool bad = !(absakk > 0.0) | (fcand & (BK_ALPHA * fabs(vf[q]) > absakk)) |
                           (dcand & (ln > kc) & (BK_ALPHA * fabs(vd[q]) > absakk));
          fm |= bad ? 1u << q : 0u;
          // keep the updates at this step: sunk to the column's own step they
          // would need every step's W row in scalar registers
#pragma unroll
          for (int j = q + 1; j < OSB; ++j) __asm__ volatile("" : "+v"(vf[j]), "+v"(vd[j]));
          vf[q] = lf;
          vd[q] = wd;
          rks = ln == q ? rk : rks;
          ds = ln == q ? d : ds;
          d = dn;
          rk = rkn;
        }
        fm &= (1u << (ce - cb)) - 1u;
        if (fm) {
          const int f = cb + __ffs(fm) - 1;
          if (f < myfail) {
            myfail = f;
            atomicMin(&s_fail, f);
          }
        }
#pragma unroll
        for (int q = 0; q < OSB; ++q) {
          const int kc = cb + q;
          if (kc < ce) {
            if (hasrow) LCR(kc) = (T)vf[q];
            if (wv == NW - 1) {
              const T rq = (T)lane_read(rks, q);
              if (drow && ln > kc) {
                ADR(kc, ln) = (T)vd[q];
                ADR(ln, kc) = (T)((T)vd[q] * rq);
              }
            }
          }
        }
        if (wv == NW - 1 && ln < ce - cb) {
          ADR(cb + ln, cb + ln) = (T)1;
          dd[cb + ln] = (T)ds;
          dsb[cb + ln] = (T)0;
        }
      }
      __syncthreads();
      int J = s_fail;
      if constexpr (!ONE) {
        if (wv == 0) {
          const uint32_t fO = ebase + (uint32_t)(3 * nb + 1 + pass);
          int abort = s_abort;
          if (ln == 0) ll_store(ll + LL_RECA + ((int64_t)(pass & 1) * 256 + g) * 4 + 3, (uint32_t)J, fO);
          int jm = ke;
          const LlDiag dg{status, 1, g, ll};
          for (int q = ln; q < G; q += 64)
            jm = min(jm, (int)ll_load(ll + LL_RECA + ((int64_t)(pass & 1) * 256 + q) * 4 + 3, fO, abort, dg));
          for (int o = 32; o > 0; o >>= 1) jm = min(jm, __shfl_xor(jm, o, 64));
          const bool any_abort = __ballot(abort) != 0;
          if (ln == 0) {
            bci[2] = any_abort ? kr : jm;
            if (any_abort) s_abort = 1;
          }
        }
        __syncthreads();
        J = bci[2];
      }
      if (!ONE && first && g == 0 && t == 0) {
        atomicAdd(status + 4, 1);
        if (J < ke) atomicAdd(status + 5, 1);
      }
      if (J < ke) {
        // columns from J on: the values before the pass
        if (ONE || first) {
          // from the matrix, through the interchanges so far (the first pass
          // of a cooperative panel has none and reads the panel buffer); the
          // columns beyond the pass (one workgroup: beyond the sub-block that
          // failed) still hold them, below the diagonal
          auto orig = [&](int pa, int pb) -> T {
            if (ONE) return pa >= pb ? AG(pa, pb) : AG(pb, pa);
            return pa >= pb ? pcol(pa, pb - k0) : pcol(pb, pa - k0);
          };
          const int te = min(cb, ke);
          for (int j0 = J; j0 < te; j0 += 16) {
            T v[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
              const int j = min(j0 + q, te - 1);
              v[q] = hasrow ? orig(ONE ? myphys : fr, ONE ? dphys[j] : k0 + j) : (T)0;
            }
#pragma unroll
            for (int q = 0; q < 16; ++q)
              if (hasrow && j0 + q < te) LCR(j0 + q) = v[q];
          }
          for (int j = J + wv; j < te; j += NW)
            if (ln >= j && ln < nbe) {
              const T v = orig(ONE ? dphys[ln] : k0 + ln, ONE ? dphys[j] : k0 + j);
              ADR(ln, j) = v;
              ADR(j, ln) = v;
            }
          if (first) {  // the pending entries above the diagonal were not loaded
            __syncthreads();
            for (int j = te + wv; j < nbe; j += NW)
              if (ln > j && ln < nbe) ADR(j, ln) = ADR(ln, j);
          }
        } else if constexpr (!ONE) {
#pragma unroll
          for (int q = 0; q < OSB; ++q) {
            const int j = kr + q;
            if (j >= J && j < ke) {
              if (hasrow) LCR(j) = vo[q];
              if (wv == NW - 1 && drow && ln >= j) {
                ADR(ln, j) = vdo[q];
                ADR(j, ln) = vdo[q];
              }
            }
          }
        }
      }
      __syncthreads();
      if (J < ke) good = 0;
      kr = J;
      ++pass;
      continue;
    }
    // ---- one step of the pivot search at column kr
    plain = false;
    const int k = k0 + kr, par = step & 1;
    const uint32_t fA = ebase + 3u * (uint32_t)step + 1u, fB = fA + 1u;
    int abort = s_abort;
    // ---- W row k over the eliminated panel columns
    if (t < kr) wk[t] = ADR(t, kr);
    __syncthreads();
    // v - sum_{j < kr} l(j) x[j], eight terms' loads together
    auto left = [&](double v, auto l, const T* x) -> double {
      int j = 0;
      for (; j + 8 <= kr; j += 8) {
        T a[8], b[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          a[q] = l(j + q);
          b[q] = x[j + q];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) v -= a[q] * b[q];
      }
      for (; j < kr; ++j) v -= l(j) * x[j];
      return v;
    };
    // ---- column k updated: own far rows and (last wave) the diagonal rows
    double v0 = 0.0, v1 = 0.0;
    const bool ldiag = wv == NW - 1 && ln >= kr && ln < nbe;
    if (hasrow) v0 = left(LCR(kr), [&](int j) { return LCR(j); }, wk);
    double av = -1.0;
    int ai = 0x7fffffff;
    if (hasrow && fr < w) {
      av = fabs(v0);
      ai = fr;
    }
    if (ldiag) {
      const double x = left(ADR(ln, kr), [&](int j) { return ADR(ln, j); }, wk);
      td0[ln] = x;
      if (ln > kr) {
        av = fabs(x);
        ai = k0 + ln;
      }
    }
    if (!(av == av)) av = -1.0;
    wg_argmax<NW>(av, ai, redv, redi, turn);
    const double absakk = fabs(td0[kr]);
    double colmax;
    int imax, gwin = 0;
    if constexpr (ONE) {
      colmax = av;
      imax = ai;
      if (hasrow && ai == fr) bcd[1] = v0;
      if (av >= 0.0 && ai >= fbeg && absakk < BK_ALPHA * av && t < nbe) prow[t] = LC[t * WLDC + (ai - fbeg)];
      __syncthreads();
    } else {
      // ---- record A: the group's largest candidate; candidate row for a second column
      {
        uint64_t* rec = ll + LL_RECA + ((int64_t)par * 256 + g) * 4;
        const bool cand = av >= 0.0;
        const bool own_far = cand && hasrow && ai == fr;
        // lanes of the last wave from nbe on hold no diagonal row (the far rows
        // k0 + nbe .. k0 + 63 must not match them)
        const bool own_diag = cand && wv == NW - 1 && ln < nbe && ai == k0 + ln;
        if (own_far || own_diag) {
          ll_store_d(rec, own_far ? v0 : td0[ln], fA);
          ll_store(rec + 2, (uint32_t)ai, fA);
        } else if (!cand && t == 0) {
          ll_store_d(rec, 0.0, fA);
          ll_store(rec + 2, 0x7fffffffu, fA);
        }
        if (cand && ai >= fbeg && ai < fbeg + fcnt && absakk < BK_ALPHA * av && t < nbe) {
          uint64_t* pay = ll + LL_PAY + ((int64_t)par * 256 + g) * 2 * WNB;
          ll_store_d(pay + 2 * t, LC[t * WLDC + (ai - fbeg)], fA);
        }
      }
      if (wv == 0) {
        double ba = -1.0, bv = 0.0;
        int bi = 0x7fffffff, bg = 0;
        for (int q = ln; q < G; q += 64) {
          uint64_t* rec = ll + LL_RECA + ((int64_t)par * 256 + q) * 4;
          const double v = ll_load_d(rec, fA, abort, LlDiag{status, 2, g, ll});
          const int idx = (int)ll_load(rec + 2, fA, abort, LlDiag{status, 3, g, ll});
          double x = fabs(v);
          if (!(x == x) || idx == 0x7fffffff) x = -1.0;
          if (x > ba || (x == ba && idx < bi)) {
            ba = x;
            bi = idx;
            bv = v;
            bg = q;
          }
        }
        for (int off = 32; off > 0; off >>= 1) {
          const double oa = __shfl_xor(ba, off, 64), ov = __shfl_xor(bv, off, 64);
          const int oi = __shfl_xor(bi, off, 64), og = __shfl_xor(bg, off, 64);
          if (oa > ba || (oa == ba && oi < bi)) {
            ba = oa;
            bi = oi;
            bv = ov;
            bg = og;
          }
        }
        const bool any_abort = __ballot(abort) != 0;
        if (ln == 0) {
          bcd[0] = ba;
          bcd[1] = bv;
          bci[0] = bi;
          bci[1] = bg;
          if (any_abort) s_abort = 1;
        }
      }
      __syncthreads();
      colmax = bcd[0];
      imax = bci[0];
      gwin = bci[1];
    }
    if (k == w - 1 || colmax < 0.0) {
      colmax = 0.0;
      imax = k;
    }
    const int imr = imax - k0;
    const bool im_diag = imr < nbe;
    const double t0imax = im_diag ? td0[imr] : bcd[1];
    int kp = k, kstep = 1, zero = 0;
    bool use_t1 = false, searched = false;
    double t1imax = 0.0;
    abort = s_abort;
    if (fmax(absakk, colmax) == 0.0 || !(absakk == absakk)) {
      zero = 1;
    } else if (!(absakk >= BK_ALPHA * colmax)) {
      searched = true;
      // ---- second column: row imax of L / A, then column imax updated
      const int pim = im_diag ? dphys[imr] : far_phys(imax, fstart, mbits, mlog, mphys, s_nm);
      double acol = 0.0;  // the matrix entry of this far row, loaded beside the row's exchange
      if (hasrow) {
        const int pa = myphys;
        acol = (pa >= pim) ? AG(pa, pim) : AG(pim, pa);
        // the matrix lacks the block's earlier panels
        for (int c = 0; c < off; ++c) acol -= AG(pa, K0 + c) * Wp[(int64_t)c * w + pim];
      }
      if (im_diag) {
        if (t < nbe) {
          prow[t] = ADR(imr, t);
          if (t < kr) wi[t] = ADR(t, imr);
        }
      } else if (!ONE && wv == 0) {
        uint64_t* pay = ll + LL_PAY + ((int64_t)par * 256 + gwin) * 2 * WNB;
        for (int j = ln; j < nbe; j += 64) prow[j] = ll_load_d(pay + 2 * j, fA, abort, LlDiag{status, 4, g, ll});
      }
      __syncthreads();
      if (!im_diag) {
        if (t < kr) wi[t] = w_entry([&](int j) { return prow[j]; }, t, dd, dsb);
        __syncthreads();
      }
      double bv2 = -1.0;
      int bi2 = 0x7fffffff;
      if (hasrow) {
        v1 = left(acol, [&](int j) { return LCR(j); }, wi);
        if (fr < w && fr != imax) {
          bv2 = fabs(v1);
          bi2 = fr;
        }
      }
      if (ldiag) {
        const double x = left(prow[ln], [&](int j) { return ADR(ln, j); }, wi);
        td1[ln] = x;
        if (k0 + ln != imax) {
          bv2 = fabs(x);
          bi2 = k0 + ln;
        }
      }
      if (!(bv2 == bv2)) bv2 = -1.0;
      if (ONE && hasrow && fr == imax) bcd[3] = v1;
      wg_argmax<NW>(bv2, bi2, redv, redi, turn);
      double rowmax;
      if constexpr (ONE) {
        rowmax = bv2;
      } else {
        {
          uint64_t* rec = ll + LL_RECB + ((int64_t)par * 256 + g) * 8;
          if (t == 0) ll_store_d(rec, bv2, fB);
          if (hasrow && fr == imax) ll_store_d(rec + 4, v1, fB);
        }
        if (wv == 0) {
          double rm = -1.0;
          for (int q = ln; q < G; q += 64) {
            const double x =
                ll_load_d(ll + LL_RECB + ((int64_t)par * 256 + q) * 8, fB, abort, LlDiag{status, 5, g, ll});
            rm = fmax(rm, x);
          }
          for (int off = 32; off > 0; off >>= 1) rm = fmax(rm, __shfl_xor(rm, off, 64));
          double ti = 0.0;
          if (!im_diag && ln == 0)
            ti = ll_load_d(ll + LL_RECB + ((int64_t)par * 256 + gwin) * 8 + 4, fB, abort, LlDiag{status, 6, g, ll});
          const bool any_abort = __ballot(abort) != 0;
          if (ln == 0) {
            bcd[2] = rm;
            bcd[3] = ti;
            if (any_abort) s_abort = 1;
          }
        }
        __syncthreads();
        rowmax = bcd[2];
      }
      if (rowmax < 0.0) rowmax = 0.0;
      t1imax = im_diag ? td1[imr] : bcd[3];
      if (absakk >= BK_ALPHA * colmax * (colmax / rowmax)) {
        kp = k;
      } else if (fabs(t1imax) >= BK_ALPHA * rowmax) {
        kp = imax;
        use_t1 = true;
      } else {
        kp = imax;
        kstep = 2;
      }
    }
    const int kk = k + kstep - 1, kkr = kk - k0, kpr = kp - k0;
    const bool swap = kp != kk;
    const bool kp_diag = kpr < nbe;
    double D1 = 0, D2 = 0, OD = 0, d11 = 0, d22 = 0, d21 = 0, rk = 0;
    if (kstep == 1) {
      D1 = use_t1 ? t1imax : td0[kr];
      rk = 1.0 / D1;
    } else {
      D1 = td0[kr];
      OD = t0imax;
      D2 = t1imax;
      d21 = OD;
      d11 = D2 / d21;
      d22 = D1 / d21;
      const double tt = 1.0 / (d11 * d22 - 1.0);
      d21 = tt / d21;
    }
    // ---- interchange kk <-> kp: row histories and the logical-to-physical map
    bool recv = false;  // this thread's far row becomes the old diagonal row kk
    if (swap) {
      if (kp_diag) {
        if (hasrow) LCR(kpr) = LCR(kkr);
      } else if (hasrow && fr == kp) {
        recv = true;
        myphys = dphys[kkr];
        for (int j = 0; j < nbe; ++j)
          if (j < kr || j > kkr) LCR(j) = ADR(kkr, j);
      }
      __syncthreads();
      if (kp_diag) {
        if (t < kr) {
          T x = ADR(kkr, t);
          ADR(kkr, t) = ADR(kpr, t);
          ADR(kpr, t) = x;
          x = ADR(t, kkr);  // and their W
          ADR(t, kkr) = ADR(t, kpr);
          ADR(t, kpr) = x;
        } else if (t > kk - k0 && t < nbe && t != kpr) {
          const T x = ADR(kkr, t);
          ADR(kpr, t) = x;
          ADR(t, kpr) = x;
        }
        if (t == 0) {
          ADR(kpr, kpr) = ADR(kkr, kkr);
          const int x = dphys[kkr];
          dphys[kkr] = dphys[kpr];
          dphys[kpr] = x;
        }
      } else {
        if (t < kr) {
          ADR(kkr, t) = prow[t];
          ADR(t, kkr) = wi[t];
        }
        if (t == 0) {
          const int old_kk = dphys[kkr];
          const int b = kp - fstart;
          int q = -1;
          if (mbits[b >> 5] & (1u << (b & 31)))
            for (int x = 0; x < s_nm; ++x)
              if (mlog[x] == kp) q = x;
          int old_kp = kp;
          if (q >= 0) {
            old_kp = mphys[q];
            mphys[q] = old_kk;
          } else {
            mlog[s_nm] = kp;
            mphys[s_nm] = old_kk;
            ++s_nm;
            mbits[b >> 5] |= 1u << (b & 31);
          }
          dphys[kkr] = old_kp;
        }
      }
      __syncthreads();
    }
    // ---- L and W column(s) of this step
    if (kstep == 1) {
      if (hasrow) {
        const double x = recv ? (use_t1 ? td1[kkr] : td0[kkr]) : (use_t1 ? v1 : v0);
        LCR(kr) = zero ? x : x * rk;
      }
      if (t > kr && t < nbe) {
        const int sr = (swap && kp_diag && t == kpr) ? kkr : t;
        const double x = use_t1 ? td1[sr] : td0[sr];
        const T l = zero ? x : x * rk;
        ADR(t, kr) = l;
        ADR(kr, t) = (T)(l * (T)D1);
      }
    } else {
      if (hasrow) {
        const double a0 = recv ? td0[kkr] : v0, a1 = recv ? td1[kkr] : v1;
        LCR(kr) = d21 * (d11 * a0 - a1);
        LCR(kr + 1) = d21 * (d22 * a1 - a0);
      }
      if (t > kr + 1 && t < nbe) {
        const int sr = (swap && kp_diag && t == kpr) ? kkr : t;
        const T l0 = d21 * (d11 * td0[sr] - td1[sr]), l1 = d21 * (d22 * td1[sr] - td0[sr]);
        ADR(t, kr) = l0;
        ADR(t, kr + 1) = l1;
        ADR(kr, t) = (T)(l0 * (T)D1 + l1 * (T)OD);
        ADR(kr + 1, t) = (T)(l0 * (T)OD + l1 * (T)D2);
      }
    }
    if (t == 0) {
      ADR(kr, kr) = 1.0;
      dd[kr] = D1;
      dsb[kr] = kstep == 2 ? OD : 0.0;
      if (kstep == 2) {
        ADR(kr + 1, kr) = 0.0;
        ADR(kr, kr + 1) = (T)OD;  // W of row kr + 1: L = 0 times D1, 1 times OD
        ADR(kr + 1, kr + 1) = 1.0;
        dd[kr + 1] = D2;
        dsb[kr + 1] = 0.0;
      }
      if (zero && g == 0) atomicOr(status, 1);
    }
    __syncthreads();
    n_second += searched;
    n_swap += swap;
    good = (searched || zero) ? 0 : good + 1;
    kr += kstep;
    ++step;
  }
  const int ker = kr, kend = k0 + kr;
  if (!ONE && t == 0 && s_abort) atomicOr(status, 4);

  // ---- moved indices of this panel: (logical, physical)
  if (t == 0 && plain) s_nM = s_nMa = 0;  // every step a 1x1 pivot in place: nothing moved
  if (t == 0 && !plain) {
    int c = 0, ca = 0;
    for (int i = 0; i < nbe; ++i)
      if (dphys[i] != k0 + i && k0 + i >= kend) {
        Ml[c] = k0 + i;
        Mp[c++] = dphys[i];
      }
    for (int q = 0; q < s_nm; ++q)
      if (mphys[q] != mlog[q]) {
        Ml[c] = mlog[q];
        Mp[c++] = mphys[q];
      }
    ca = c;  // the first ca entries lie in the trailing block
    for (int i = 0; i < nbe; ++i)
      if (dphys[i] != k0 + i && k0 + i < kend) {
        Ml[c] = k0 + i;
        Mp[c++] = dphys[i];
      }
    s_nM = c;
    s_nMa = ca;
  }
  __syncthreads();
  const int nM = s_nM, nMa = s_nMa;
  const int GT = G * NT, gt = g * NT + t;
  const int nt = w - kend;                 // trailing block size
  const int64_t no = r - w;                // rows below the diagonal block
  auto phys = [&](int j) -> int {
    if (j < k0 + nbe) return dphys[j - k0];
    return far_phys(j, fstart, mbits, mlog, mphys, s_nm);
  };
  auto sym = [&](int i, int j) -> T& { return i >= j ? AG(i, j) : AG(j, i); };
  // D, the pivot permutation of the moved indices and the statistics
  if (g == 0) {
    if (t < ker) {
      dval[c0 + k0 + t] = dd[t];
      dval[n + c0 + k0 + t] = dsb[t];
    }
    const int pold = t < nM ? perm_piv[c0 + Mp[t]] : 0;
    __syncthreads();
    if (t < nM) perm_piv[c0 + Ml[t]] = pold;
    if (!ONE && t == 0 && n_second) atomicAdd(status + 2, n_second);
    if (!ONE && t == 0 && n_swap) atomicAdd(status + 3, n_swap);
  }
  if constexpr (ONE) {
    if (nM > 0) {
      // entries (m, m') of the trailing block that both moved, through a
      // scratch copy (at most nb moved indices lie in the trailing block: one
      // per interchange)
      for (int idx = t; idx < nMa * nMa; idx += NT) {
        const int m = idx / nMa, q = idx % nMa;
        if (m >= q) scr[idx] = sym(Mp[m], Mp[q]);
      }
      __syncthreads();
      // Lines: a trailing column that did not move, a row below the diagonal
      // block, or an earlier column of L.  The moved entries of a line are
      // read by one wave's lanes and stored by them afterwards, so a line
      // needs no scratch copy; P lanes take a line, 64 / P lines an instruction.
      int P = 1;
      while (P < nM && P < 64) P *= 2;
      const int lpi = 64 / P, sub0 = ln / P, m0 = ln % P;
      auto lines = [&](int count, int mcount, auto skip, auto at) {
        constexpr int U = 8;
        for (int base = wv * lpi * U; base < count; base += NW * lpi * U) {
          T v[U][2];
          bool ok[U][2];
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int line = base + u * lpi + sub0, m = m0 + 64 * h;
              ok[u][h] = line < count && m < mcount && !skip(line);
              v[u][h] = ok[u][h] ? at(line, Mp[m]) : (T)0;
            }
          __builtin_amdgcn_wave_barrier();  // the wave's loads before its stores
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              if (ok[u][h]) at(base + u * lpi + sub0, Ml[m0 + 64 * h]) = v[u][h];
        }
      };
      auto none = [](int) { return false; };
      lines(nt, nMa, [&](int l) { return phys(kend + l) != kend + l; },
            [&](int l, int m) -> T& { return sym(m, kend + l); });
      lines((int)no, nM, none, [&](int l, int m) -> T& { return AG(w + l, m); });
      lines(k0, nM, none, [&](int l, int m) -> T& { return AG(m, l); });
      for (int idx = t; idx < nMa * nMa; idx += NT) {
        const int m = idx / nMa, q = idx % nMa;
        if (m >= q) sym(Ml[m], Ml[q]) = scr[idx];
      }
      __syncthreads();  // the panel's original columns and the scratch are read: L and W may go over them
    }
  } else {
    T* S1 = scr;                                  // [nMa][nt]
    T* S2 = scr + (int64_t)WMM * w;               // [nM][no]
    T* S3 = S2 + (int64_t)WMM * (no > 0 ? no : 0);  // [nM][k0]
    T* S4 = S3 + (int64_t)WMM * w;                 // [nM][off] rows of W of the block's earlier panels
    int epoch = 0;
    if (nM > 0) {
      // gather the permuted values from the untouched panel-start storage
      for (int64_t idx = gt; idx < (int64_t)nMa * nt; idx += GT) {
        const int m = (int)(idx / nt), j = kend + (int)(idx % nt);
        S1[idx] = sym(Mp[m], phys(j));
      }
      // rows below the diagonal block: only the trailing columns move (their
      // panel columns hold L in logical order already)
      for (int64_t idx = gt; idx < (int64_t)nMa * no; idx += GT) {
        const int m = (int)(idx / no);
        S2[idx] = AG(w + idx % no, Mp[m]);
      }
      for (int64_t idx = gt; idx < (int64_t)nM * k0; idx += GT) {
        const int m = (int)(idx / k0), j = (int)(idx % k0);
        S3[idx] = AG(Mp[m], j);
      }
      for (int64_t idx = gt; idx < (int64_t)nM * off; idx += GT) {
        const int m = (int)(idx / off), c = (int)(idx % off);
        S4[idx] = Wp[(int64_t)c * w + Mp[m]];
      }
      group_barrier(sync, G, epoch, status);
      for (int64_t idx = gt; idx < (int64_t)nMa * nt; idx += GT) {
        const int m = (int)(idx / nt), j = kend + (int)(idx % nt);
        sym(Ml[m], j) = S1[idx];
      }
      for (int64_t idx = gt; idx < (int64_t)nMa * no; idx += GT) {
        const int m = (int)(idx / no);
        AG(w + idx % no, Ml[m]) = S2[idx];
      }
      for (int64_t idx = gt; idx < (int64_t)nM * k0; idx += GT) {
        const int m = (int)(idx / k0), j = (int)(idx % k0);
        AG(Ml[m], j) = S3[idx];
      }
      for (int64_t idx = gt; idx < (int64_t)nM * off; idx += GT) {
        const int m = (int)(idx / off), c = (int)(idx % off);
        Wp[(int64_t)c * w + Ml[m]] = S4[idx];
      }
    }
  }
  // ---- L of the panel and W = L D for the rows of the trailing block
  if (hasrow) {
    if (plain) {  // all pivots 1x1: W is a scaling, sixteen columns' stores together
      for (int j0 = 0; j0 < ker; j0 += 16) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int j = j0 + q;
          if (j < ker) {
            const T l = LCR(j);
            AG(fr, k0 + j) = l;
            if (fr < w) Wp[(int64_t)(off + j) * w + fr] = l * dd[j];
          }
        }
      }
    } else {
      for (int j = 0; j < ker; ++j) {
        AG(fr, k0 + j) = LCR(j);
        if (fr < w) Wp[(int64_t)(off + j) * w + fr] = w_entry([&](int c) { return LCR(c); }, j, dd, dsb);
      }
    }
  }
  for (int idx = gt; idx < nbe * ker; idx += GT) {
    const int i = idx % nbe, j = idx / nbe;
    if (j <= i) AG(k0 + i, k0 + j) = ADR(i, j);
    if (k0 + i >= kend) Wp[(int64_t)(off + j) * w + k0 + i] = ADR(j, i);
  }
  if (g == 0 && t == 0) {
    kstart[s] = K0;
    kpos[s] = kend;
  }
#undef AG
#undef LCR
#undef ADR
}

template <typename T>
void launch_bk_wide(const WideSn& sn, int G, int nt, int nb, int sub, int wcols, int n, T* valL, T* dval,
                    int* perm_piv, T* W, int* kpos, int* kstart, int* sync, int* sync_next, uint64_t* ll,
                    uint32_t ebase, int* status, hipStream_t st) {
  if (nb > wide_panel_nb(nt, sizeof(T)) || nb < 4 || G < 1 || G > 256 || (nt != 256 && nt != WIDE_NT_TALL))
    throw std::runtime_error("bk_wide: launch shape out of range");
  PanelList pl{};
  void* args[] = {(void*)&sn, (void*)&pl, (void*)&G, (void*)&nb, (void*)&sub, (void*)&wcols, (void*)&valL, (void*)&dval,
                  (void*)&perm_piv, (void*)&W, (void*)&kpos, (void*)&kstart,
                  (void*)&sync, (void*)&sync_next, (void*)&ll, (void*)&ebase, (void*)&n, (void*)&status};
  // tall supernodes: 448 far rows per workgroup in the same 256-byte LDS rows
  // (32 FP64 or 64 FP32 columns)
  constexpr int NBT = sizeof(T) == 8 ? 32 : 64;
  const void* fn = nt == 256 ? (const void*)k_bk_wide<T, 256, 64, false>
                             : (const void*)k_bk_wide<T, WIDE_NT_TALL, NBT, false>;
  hipError_t e = hipLaunchCooperativeKernel(fn, dim3(G), dim3(nt), args, 0, st);
  if (e != hipSuccess) throw std::runtime_error(std::string("bk_wide: ") + hipGetErrorString(e));
}
template void launch_bk_wide<double>(const WideSn&, int, int, int, int, int, int, double*, double*, int*, double*,
                                     int*, int*, int*, int*, uint64_t*, uint32_t, int*, hipStream_t);
template void launch_bk_wide<float>(const WideSn&, int, int, int, int, int, int, float*, float*, int*, float*,
                                    int*, int*, int*, int*, uint64_t*, uint32_t, int*, hipStream_t);

// One-workgroup panels.  What bounds them is the chain of column steps, about
// 0.36 us each where every pivot is accepted in place; a block that searches
// at every column takes 3.4 to 4.7 us a column, launches and trailing updates
// included (65 to 256 columns), 0.94 to 1.3 times the speed of the panels
// before, by the width.  Measured per launch, before
// (columns summed left-looking from LDS or memory, 31 per launch) and now:
// 33^3 KKT 83-138 us -> 43 (64 columns) / 30 (32) / 23 (16), 24 x 150
// block-indefinite 82-102 us -> 234 / 139 / 98, that is 11.1 -> 9.1 ms a
// factorization; 40 x 40 QP's 248-wide root 42.7 -> 14.6 ms a solve.
// The shape is the smallest whose LDS holds the
// remaining rows: 256 threads and 64 columns up to 256 rows, 512 threads up
// to 448 far rows (32 FP64 or 64 FP32 columns), 1024 threads up to 960 far
// rows (16 or 32 columns): the same LDS (far rows x columns) in all three.
//
// A 64-column FP64 panel takes 146 KB of LDS, so a CU runs one (FP32: two).
// Launches of more panels than that take 32 columns, where 33 KB (128
// threads, up to 96 rows) or 66 KB (up to 224 rows) let a CU run four or two
// side by side.  All panels of one factorization, us, 64 columns / 32 columns
// (and 31-column panels with up to four workgroups a CU before): 512 blocks
// 65 wide, accepted in place 149 / 101 (274), searched at every column
// 440 / 265 (324); 1024: 278 / 117 (331), 852 / 290 (392); 512 blocks 150
// wide 325 / 252 (705), 1271 / 707 (826); FP32, 1024 blocks 65 wide
// 177 / 114 (316), 506 / 288 (376).  Up to one panel per CU (FP32: two) the
// 64-column panels win: 256 blocks 65 wide take 85 us.
struct OneShape {
  int nt, nb;  // threads, columns (0: too many rows)
};
template <typename T>
static OneShape one_shape(int rows, int count) {
  constexpr int CUS = 256, N1 = sizeof(T) == 8 ? 32 : 64, N2 = sizeof(T) == 8 ? 16 : 32;
  if (count > CUS * (sizeof(T) == 8 ? 1 : 2)) {
    if (rows <= 32 + 64) return {128, 32};
    if (rows <= 32 + 192) return {256, 32};
  }
  if (rows <= 64 + 192) return {256, 64};
  if (rows <= N1 + 448) return {512, N1};
  if (rows <= N2 + 960) return {1024, N2};
  return {0, 0};
}
template <typename T>
int one_panel_nb(int rows, int count) {
  return one_shape<T>(rows, count).nb;
}
template int one_panel_nb<double>(int, int);
template int one_panel_nb<float>(int, int);

template <typename T, int NT, int NBM>
static void launch_one(const PanelList& pl, int count, T* valL, T* dval, int* perm_piv, T* W, int* kpos, int* kstart,
                       int n, int* status, hipStream_t st) {
  int* const nosync = nullptr;
  uint64_t* const noll = nullptr;
  k_bk_wide<T, NT, NBM, true><<<count, NT, 0, st>>>(WideSn{}, pl, 1, NBM, 0, ONE_WCOLS, valL, dval, perm_piv, W, kpos,
                                                    kstart, nosync, nosync, noll, 0u, n, status);
}
template <typename T>
void launch_bk_one(const int* list, int count, int rows, const SnArgs& a, T* valL, T* dval, int* perm_piv, T* W,
                   const int64_t* woff, int* kpos, int* kstart, int* status, hipStream_t st) {
  if (count <= 0) return;
  constexpr int N1 = sizeof(T) == 8 ? 32 : 64, N2 = sizeof(T) == 8 ? 16 : 32;
  const OneShape sh = one_shape<T>(rows, count);
  const PanelList pl{list, a.super, a.pi, a.px, woff};
  if (sh.nt == 128)
    launch_one<T, 128, 32>(pl, count, valL, dval, perm_piv, W, kpos, kstart, a.n, status, st);
  else if (sh.nt == 256 && sh.nb == 32)
    launch_one<T, 256, 32>(pl, count, valL, dval, perm_piv, W, kpos, kstart, a.n, status, st);
  else if (sh.nt == 256)
    launch_one<T, 256, 64>(pl, count, valL, dval, perm_piv, W, kpos, kstart, a.n, status, st);
  else if (sh.nt == 512)
    launch_one<T, 512, N1>(pl, count, valL, dval, perm_piv, W, kpos, kstart, a.n, status, st);
  else if (sh.nt == 1024)
    launch_one<T, 1024, N2>(pl, count, valL, dval, perm_piv, W, kpos, kstart, a.n, status, st);
  else
    throw std::invalid_argument("bk_one: too many rows for a one-workgroup panel");
  HIP_LAUNCH_CHECK("bk_one");
}
template void launch_bk_one<double>(const int*, int, int, const SnArgs&, double*, double*, int*, double*,
                                    const int64_t*, int*, int*, int*, hipStream_t);
template void launch_bk_one<float>(const int*, int, int, const SnArgs&, float*, float*, int*, float*, const int64_t*,
                                   int*, int*, int*, hipStream_t);

}  // namespace lblg
