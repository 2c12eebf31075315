// One-workgroup leaf of the LU panels: partial-pivoting LU of an M x W row-major
// panel (W <= 64) whose rows all fit one workgroup, FP64 and FP32 (zml
// lapack/getrf2.zig:14-210).
//
// Rows never move while the leaf runs: each carries its LAPACK position, the
// search takes the largest |a_ik| among the rows at positions >= k, the lowest
// position on ties (iamax.zig:32's strict '>' over the interchanged rows), and
// the row that held position k takes the pivot's old one, which is the
// interchange LAPACK records. Rows are written to their final positions at the
// end, with the list of moves for the columns outside the leaf (no interchange
// list has to be composed).
//
// The 64 columns advance in groups of 8. Inside a group only its 8 columns are
// updated, column by column; a column costs the wave's candidate (largest high
// word by DPP, the tied lanes by ballot), one LDS record per wave, one barrier,
// the same search over the waves' records and the pivot row's 8 values from LDS.
// After the group the pivot rows' later columns are solved by substitution in
// LDS and every remaining row applies the group's 8 columns to its later ones.
// Every element still receives fl(a - fl(l u)) for k ascending: the factors are
// the column-by-column leaf's bit for bit.
//
// Bound by the instruction chain of a column (candidate, record, barrier, the
// records' winner, reciprocal and update: about 900 cycles with one wave per SIMD),
// then by the LDS reads of the group updates (4 cycles per value and wave). The
// column-by-column leaf (64-column updates, staging, three barriers and register
// interchanges in every column; above 256 rows an exchange between workgroups as
// well) took 146 us at 200 rows, 320 us at 500 and at 1,000 rows; this one 71, 89
// and 152 us (one MI355X, FP64, launch included).
#pragma once

#include "panel.hpp"

namespace zmlhip {
namespace panel {

constexpr int GW = 8;    // columns of a group

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int imax_step(int v) {
  const int o = __builtin_amdgcn_update_dpp((int)0x80000000, v, CTRL, ROW_MASK, 0xf, false);
  return v > o ? v : o;
}
// Largest v of the wave, in every lane.
__device__ __forceinline__ int wave_imax(int v) {
  v = imax_step<0xb1, 0xf>(v);     // quad_perm [1,0,3,2]
  v = imax_step<0x4e, 0xf>(v);     // quad_perm [2,3,0,1]
  v = imax_step<0x124, 0xf>(v);    // row_ror:4
  v = imax_step<0x128, 0xf>(v);    // row_ror:8
  v = imax_step<0x142, 0xa>(v);    // row_bcast:15 into rows 1 and 3
  v = imax_step<0x143, 0xc>(v);    // row_bcast:31 into rows 2 and 3
  return __builtin_amdgcn_readlane(v, 63);
}
// The lane (below N) with the largest v, the lowest pos among equals. N = 64, or 4
// or 8 with the same values in every group of N lanes. v >= 0, or -1 for "no
// candidate"; NaN must not occur.
template <int N>
__device__ __forceinline__ int group_imax(int v) {
  if constexpr (N == 64) return wave_imax(v);
  v = imax_step<0xb1, 0xf>(v);
  v = imax_step<0x4e, 0xf>(v);
  if constexpr (N == 8) v = imax_step<0x124, 0xf>(v);
  return v;
}
template <int N>
__device__ __forceinline__ int winner(double v, int pos) {
  constexpr uint64_t kLanes = N == 64 ? ~0ull : (1ull << N) - 1;
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const int hi = (int)(b >> 32);
  const int mh = group_imax<N>(hi);
  uint64_t m = __ballot(hi == mh) & kLanes;
  if (__builtin_expect((m & (m - 1)) != 0, 0)) {   // equal high words: the low words, then the positions
    const int lo = (int)((uint32_t)b ^ 0x80000000u);   // unsigned order as signed
    const int ml = group_imax<N>(hi == mh ? lo : (int)0x80000000);
    m = __ballot(hi == mh && lo == ml) & kLanes;
    if ((m & (m - 1)) != 0) {
      const int np = group_imax<N>(hi == mh && lo == ml ? ~pos : (int)0x80000000);
      m = __ballot(hi == mh && lo == ml && ~pos == np) & kLanes;
    }
  }
  return (int)__builtin_ctzll(m);
}

// A wave's candidate for a column: |a|, position, row (relative to the panel) and
// the row's values in the group's columns.
template <typename T>
struct __attribute__((aligned(16))) Leaf1Rec {
  double v;
  int pos, row;
  T val[GW];
};

// x[r][c] -= l[r][q] U[q ldu + c] for q = 0 .. NQ - 1 in order, 8 columns, separately
// rounded: one row of U (an LDS broadcast) is read ahead of the one being used. The
// empty asm keeps the elements in this order (reordered, the products are formed
// ahead and spill).
template <typename T, int R, int NQ>
__device__ __forceinline__ void apply_rows(T (&x)[R][GW], const T (&l)[R][NQ], const T* U, int ldu) {
#pragma clang fp contract(off)
  constexpr bool kAhead = R == 1;   // (two rows per thread leave no registers for it)
  T u[GW], un[GW];
#pragma unroll
  for (int c = 0; c < GW; ++c) un[c] = U[c];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
#pragma unroll
    for (int c = 0; c < GW; ++c) u[c] = kAhead || q == 0 ? un[c] : U[q * ldu + c];
    if (kAhead && q + 1 < NQ) {
#pragma unroll
      for (int c = 0; c < GW; ++c) un[c] = U[(q + 1) * ldu + c];
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < GW; ++c) {
        x[r][c] = x[r][c] - l[r][q] * u[c];
        asm volatile("" : "+v"(x[r][c]));
      }
  }
}

// NT threads, R rows per thread (row t + NT r), HW columns held in registers at a
// time: 64, or 32 in two halves, the second updated from the first through
// memory. moves (absolute rows): moves[0] the count, then (destination, source)
// pairs, as apply_perm_kernel reads them.
// Memory is read and written eight lanes to a row (64-byte pieces) and changed to
// one row per thread in LDS: a row per lane straight from memory touches 64 lines
// with every instruction, which took as long as the elimination itself.
template <typename T, int NT, int R, int HW>
__global__ void __launch_bounds__(NT)
leaf1_kernel(int M, int Wn, T* __restrict__ P, int64_t ld, int32_t* __restrict__ ipiv, int64_t row_base,
             int* __restrict__ info, int64_t info_base, int32_t* __restrict__ moves) {
#pragma clang fp contract(off)
  constexpr int NW = NT / 64, NG = HW / GW, TLD = GW + 1, RPP = NT / GW;   // RPP: rows of one tile pass
  __shared__ Leaf1Rec<T> rec[GW][NW];
  __shared__ __attribute__((aligned(16))) T U[GW][HW];     // the group's pivot rows, later columns
  __shared__ T tile[2][NT * TLD];
  __shared__ int32_t s_pos[NT];
  __shared__ int s_cnt;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int tr = t / GW, tc = t % GW;   // this thread's row and column in a tile pass
  const T sfmin = sizeof(T) == 8 ? T(0x1p-1022) : T(0x1p-126);   // lamch('S')
  if (t == 0) s_cnt = 0;
  int buf = 0, fz = 0, mypos = 0, myrow = 0;

  // columns [c0, c0 + 8) of rows NT r .. NT r + NT - 1, element e of this thread
  // (row tr + RPP e), clamped into the panel; keep8 makes zeros of what lies outside.
  // Apart, so that every load is on its way before the first is waited for.
  auto read8 = [&](int r, int c0, T (&v)[GW]) __attribute__((always_inline)) {
    const int row0 = NT * r + tr;
    const T* const last = P + (int64_t)(M - 1) * ld + min(c0 + tc, Wn - 1);
    const T* p = P + (int64_t)row0 * ld + min(c0 + tc, Wn - 1);
#pragma unroll
    for (int e = 0; e < GW; ++e) {
      v[e] = *(row0 + RPP * e < M ? p : last);
      p += (int64_t)RPP * ld;
    }
  };
  auto keep8 = [&](int r, int c0, T (&v)[GW]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < GW; ++e) {
      asm volatile("" : "+v"(v[e]));
      v[e] = (NT * r + tr + RPP * e < M && c0 + tc < Wn) ? v[e] : T(0);
    }
  };
  // the pass's elements to one row per thread, and back
  auto to_rows = [&](T (&v)[GW]) __attribute__((always_inline)) {
    T* const q = tile[buf];
#pragma unroll
    for (int e = 0; e < GW; ++e) q[(tr + RPP * e) * TLD + tc] = v[e];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < GW; ++c) v[c] = q[t * TLD + c];
    buf ^= 1;
  };
  auto to_pass = [&](const T (&x)[GW], T (&v)[GW]) __attribute__((always_inline)) {
    T* const q = tile[buf];
#pragma unroll
    for (int c = 0; c < GW; ++c) q[t * TLD + c] = x[c];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < GW; ++e) v[e] = q[(tr + RPP * e) * TLD + tc];
    buf ^= 1;
  };
  // a pass to memory: rows to `rows[]` (their final positions; s_pos) or to their own place
  auto write8 = [&](int r, int c0, const T (&v)[GW], const int32_t* rows) __attribute__((always_inline)) {
    const int col = c0 + tc;
#pragma unroll
    for (int e = 0; e < GW; ++e) {
      const int row = NT * r + tr + RPP * e;
      if (row < M && col < Wn) P[(int64_t)(rows ? rows[tr + RPP * e] : row) * ld + col] = v[e];
    }
  };

  int pos[R];
  T a[R][HW];
  auto load_half = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T v[NG][GW];
#pragma unroll
      for (int g = 0; g < NG; ++g) read8(r, c0 + GW * g, v[g]);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        keep8(r, c0 + GW * g, v[g]);
        to_rows(v[g]);
#pragma unroll
        for (int c = 0; c < GW; ++c) a[r][GW * g + c] = v[g][c];
      }
    }
  };
#pragma unroll
  for (int r = 0; r < R; ++r) pos[r] = t + NT * r < M ? t + NT * r : -1;   // -1: no row
  load_half(0);

  for (int h0 = 0; h0 < Wn; h0 += HW) {
    for (int g = 0; g < NG; ++g) {
      const int k0 = h0 + GW * g;
      if (k0 >= Wn) break;
      T w[R][GW];   // the group's columns
      int wins[GW] = {};   // the waves whose records hold the group's pivot rows
#pragma unroll
      for (int gg = 0; gg < NG; ++gg)
        if (gg == g) {
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < GW; ++c) w[r][c] = a[r][GW * gg + c];
        }
#pragma unroll
      for (int kk = 0; kk < GW; ++kk) {
        const int k = k0 + kk;
        if (k >= Wn) break;
        // the thread's, then the wave's candidate; a NaN at position k keeps it (as
        // +inf at the lowest position), elsewhere a NaN never wins
        double bv = -1.0;
        int bp = INT32_MAX, br = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          double f = fabs((double)w[r][kk]);
          f = f == f ? f : (pos[r] == k ? (double)INFINITY : -1.0);
          f = pos[r] >= k ? f : -1.0;
          if (f > bv || (R > 1 && f == bv && pos[r] < bp)) { bv = f; bp = pos[r]; br = r; }
        }
        const int wl = winner<64>(bv, bp);
        Leaf1Rec<T>* const my = &rec[kk][wv];
        if (lane == wl) {
          my->v = bv;
          my->pos = bp;
          my->row = t + NT * br;
#pragma unroll
          for (int c = 0; c < GW; ++c) {
            T x = w[0][c];
#pragma unroll
            for (int r = 1; r < R; ++r) x = br == r ? w[r][c] : x;
            my->val[c] = x;
          }
        }
        __syncthreads();
        const Leaf1Rec<T>* const q = &rec[kk][NW > 1 ? lane % NW : 0];
        const double qv = q->v;
        const int qp = q->pos, qr = q->row;
        const int ww = NW > 1 ? winner<NW == 1 ? 64 : NW>(qv, qp) : 0;
        const int ppos = __builtin_amdgcn_readlane(qp, ww), prow = __builtin_amdgcn_readlane(qr, ww);
        const T* const win = rec[kk][ww].val;
        T u[GW];
#pragma unroll
        for (int c = kk; c < GW; ++c) u[c] = win[c];
        const T piv = u[kk];
        // uniform over the workgroup: a zero pivot makes no interchange (getrf2.zig:55; ppos is k
        // then), one below sfmin divides
        const bool nz = __builtin_amdgcn_readfirstlane(piv != T(0)) != 0;
        const bool recip = __builtin_amdgcn_readfirstlane(fabs(piv) >= sfmin) != 0;
        if (!nz && fz == 0) fz = k + 1;
        mypos = lane == k ? ppos : mypos;   // lane k keeps column k's pivot
        myrow = lane == k ? prow : myrow;
        wins[kk] = ww;
        T l[R];
        if (recip) {
          const T rinv = T(1) / piv;
#pragma unroll
          for (int r = 0; r < R; ++r) l[r] = w[r][kk] * rinv;
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) l[r] = nz ? w[r][kk] / piv : w[r][kk];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const bool is_piv = prow == t + NT * r;
          if (pos[r] >= k && !is_piv) {
            w[r][kk] = l[r];
#pragma unroll
            for (int c = kk + 1; c < GW; ++c) w[r][c] = w[r][c] - l[r] * u[c];
            if (pos[r] == k) pos[r] = ppos;
          }
          if (is_piv) pos[r] = k;
        }
      }
#pragma unroll
      for (int gg = 0; gg < NG; ++gg)
        if (gg == g) {
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < GW; ++c) a[r][GW * gg + c] = w[r][c];
        }
      if (g + 1 >= NG || k0 + GW >= Wn) continue;
      // U of the group's rows: their later columns, u_q = a_q - sum_{j < q} l_qj u_j
      // in order (a pivot row's multipliers are the first values of its record)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (pos[r] >= k0 && pos[r] < k0 + GW) {
#pragma unroll
          for (int gg = 1; gg < NG; ++gg)
            if (gg > g) {
#pragma unroll
              for (int c = 0; c < GW; ++c) U[pos[r] - k0][GW * gg + c] = a[r][GW * gg + c];
            }
        }
      __syncthreads();
      const int cu = GW * (g + 1) + t;
      if (cu < HW) {
        T x[GW];
#pragma unroll
        for (int q = 0; q < GW; ++q) x[q] = U[q][cu];
#pragma unroll
        for (int q = 1; q < GW; ++q) {
          const T* const lq = rec[q][wins[q]].val;
#pragma unroll
          for (int j = 0; j < q; ++j) x[q] = x[q] - lq[j] * x[j];
          U[q][cu] = x[q];
        }
      }
      __syncthreads();
#pragma unroll
      for (int gg = 1; gg < NG; ++gg)
        if (gg > g) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (pos[r] >= k0 + GW) {
              T x[1][GW], l[1][GW];
#pragma unroll
              for (int c = 0; c < GW; ++c) { x[0][c] = a[r][GW * gg + c]; l[0][c] = w[r][c]; }
              apply_rows<T, 1, GW>(x, l, &U[0][GW * gg], HW);
#pragma unroll
              for (int c = 0; c < GW; ++c) a[r][GW * gg + c] = x[0][c];
            } else if (pos[r] >= k0) {   // pivoted in this group: its solved values
#pragma unroll
              for (int c = 0; c < GW; ++c) a[r][GW * gg + c] = U[pos[r] - k0][GW * gg + c];
            }
          }
        }
    }
    if constexpr (HW < W) {
      if (h0 + HW < Wn) {
        // the second half: the pivot rows' columns (U12) by substitution, then
        // every other row, 8 columns at a time; this half's columns to memory, in place
        __shared__ int32_t s_prow[W];
        __shared__ T L11[HW][HW + 1];
        __shared__ __attribute__((aligned(16))) T U12[HW][HW];
        const int h1 = h0 + HW;
        if (t < W) s_prow[t] = myrow;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (pos[r] >= 0 && pos[r] < h1) {
#pragma unroll
            for (int c = 0; c < HW; ++c) L11[pos[r]][c] = a[r][c];
          }
        for (int e = t; e < HW * HW; e += NT) {
          const int q = e / HW, c = e % HW;
          U12[q][c] = h1 + c < Wn ? P[(int64_t)s_prow[q] * ld + h1 + c] : T(0);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int g = 0; g < NG; ++g) {
            T x[GW], v[GW];
#pragma unroll
            for (int c = 0; c < GW; ++c) x[c] = a[r][GW * g + c];
            to_pass(x, v);
            write8(r, h0 + GW * g, v, nullptr);
          }
        __syncthreads();
        for (int b = 0; b < HW; b += GW) {
          if (t < HW) {   // the block's 8 rows of column t, in order
            T x[GW];
#pragma unroll
            for (int q = 0; q < GW; ++q) x[q] = U12[b + q][t];
#pragma unroll
            for (int q = 1; q < GW; ++q) {
#pragma unroll
              for (int j = 0; j < q; ++j) x[q] = x[q] - L11[b + q][b + j] * x[j];
              U12[b + q][t] = x[q];
            }
          }
          __syncthreads();
          for (int e = t; e < (HW - b - GW) * HW; e += NT) {   // the rows below it
            const int q = b + GW + e / HW, c = e % HW;
            T x = U12[q][c];
#pragma unroll
            for (int j = 0; j < GW; ++j) x = x - L11[q][b + j] * U12[b + j][c];
            U12[q][c] = x;
          }
          __syncthreads();
        }
        for (int cg = 0; cg < HW; cg += GW) {
          T x[R][GW];
#pragma unroll
          for (int r = 0; r < R; ++r) read8(r, h1 + cg, x[r]);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            keep8(r, h1 + cg, x[r]);
            to_rows(x[r]);
          }
          apply_rows<T, R, HW>(x, a, &U12[0][cg], HW);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            T v[GW];
            if (pos[r] >= 0 && pos[r] < h1) {
#pragma unroll
              for (int c = 0; c < GW; ++c) x[r][c] = U12[pos[r]][cg + c];
            }
            to_pass(x[r], v);
            write8(r, h1 + cg, v, nullptr);
          }
        }
        // (written by other threads of this workgroup: through L1, in order)
        __threadfence_block();
        __syncthreads();
        load_half(h1);
      }
    }
  }

  // rows to their final positions; every row of the panel has been read
  if constexpr (HW < W) {
    if (Wn > HW) {
      // the first half of the rows that move, 8 columns at a time
      for (int c0 = 0; c0 < HW; c0 += GW) {
        T x[R][GW];
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (pos[r] >= 0 && pos[r] != t + NT * r) {
#pragma unroll
            for (int c = 0; c < GW; ++c) x[r][c] = P[(int64_t)(t + NT * r) * ld + c0 + c];
          }
        __builtin_amdgcn_s_waitcnt(0xF70);   // (loads returned before any row is overwritten)
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (pos[r] >= 0 && pos[r] != t + NT * r) {
#pragma unroll
            for (int c = 0; c < GW; ++c) P[(int64_t)pos[r] * ld + c0 + c] = x[r][c];
          }
      }
    }
  }
  const int cl = HW < W && Wn > HW ? HW : 0;   // first column still in registers
#pragma unroll
  for (int r = 0; r < R; ++r) {
    __syncthreads();
    s_pos[t] = pos[r];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      T x[GW], v[GW];
#pragma unroll
      for (int c = 0; c < GW; ++c) x[c] = a[r][GW * g + c];
      to_pass(x, v);
      write8(r, cl + GW * g, v, s_pos);
    }
    if (pos[r] >= 0 && pos[r] != t + NT * r) {
      const int q = atomicAdd(&s_cnt, 1);
      moves[1 + 2 * q] = (int32_t)(row_base + pos[r]);
      moves[2 + 2 * q] = (int32_t)(row_base + t + NT * r);
    }
  }
  __syncthreads();
  if (t < Wn) ipiv[t] = (int32_t)(row_base + mypos + 1);
  if (t == 0) {
    moves[0] = s_cnt;
    if (fz != 0 && *info == 0) *info = (int)(info_base + fz);
  }
}

}  // namespace panel
}  // namespace zmlhip
