// Leaf of the LU panels: partial-pivoting LU of an M x W row-major panel (W <= 64)
// by one workgroup that holds all its rows, or by workgroups that exchange every
// pivot, FP64 and FP32 (zml lapack/getrf2.zig:14-210).
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
// interchanges in every column) took 146 us at 200 rows; this one 71 us, and 89 us
// at 500 rows (one MI355X, FP64, launch included).
#pragma once

#include <type_traits>

#include "panel.hpp"

namespace zmlhip {
namespace panel {

constexpr int GW = 8;    // columns of a group
template <int N> using Place = std::integral_constant<int, N>;

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

// One wave: publishes this workgroup's candidate `mine` of column k, the KK-th of
// its group (position, row and the values from column k on), and puts the best
// over all G workgroups into *out.
template <typename T, int KK>
__device__ __forceinline__ void exchange(const Leaf1Rec<T>* mine, Leaf1Rec<T>* out, int k, int G, int wg, int lane,
                                         const WS& ws, uint32_t tag_base, long spin_limit, int* s_abort) {
  constexpr int VW = (int)sizeof(T) / 4, NV = VW * (GW - KK), XW = 2 + NV;
  const uint32_t tag = tag_base + (uint32_t)k + 1u;
  uint64_t* const x = ws.x + (size_t)(k & 1) * XWMAX * GMAX;
  if (lane < XW)
    st64(x + lane * GMAX + wg,
         tagged(tag, reinterpret_cast<const uint32_t*>(mine)[2 + lane + (lane < 2 ? 0 : VW * KK)]));
  if (spin_limit < 0) {   // give-up forced by the host (error-path tests)
    if (lane == 0) { *s_abort = 1; atomicExch(ws.err, 1); }
    return;
  }
  double v = -1.0;
  int pos = INT32_MAX, row = 0;
  uint32_t val[NV];
#pragma unroll
  for (int w = 0; w < NV; ++w) val[w] = 0;
  long spins = 0;
  for (int c0 = 0; c0 < G; c0 += 64) {
    const uint64_t* const q = x + (c0 + lane < G ? c0 + lane : c0);
    uint64_t d[XW];
    while (true) {
      bool ok = true;
#pragma unroll
      for (int w = 0; w < XW; ++w) d[w] = ld64(q + w * GMAX);
#pragma unroll
      for (int w = 0; w < XW; ++w) ok = ok && tag_of(d[w]) == tag;
      if (__all(ok)) break;
      if (++spins > spin_limit) {
        if (lane == 0) { *s_abort = 1; atomicExch(ws.err, 1); }
        return;
      }
    }
    const int p = (int)payload(d[0]);
    T a;
    if constexpr (sizeof(T) == 8) a = val_of<T>(d[3], d[2]);
    else a = __uint_as_float(payload(d[2]));
    double f = fabs((double)a);
    f = f == f ? f : (double)INFINITY;   // (a NaN is a candidate only at position k)
    f = p == INT32_MAX ? -1.0 : f;
    if (f > v || (f == v && p < pos)) {
      v = f;
      pos = p;
      row = (int)payload(d[1]);
#pragma unroll
      for (int w = 0; w < NV; ++w) val[w] = payload(d[2 + w]);
    }
  }
  if (lane == winner<64>(v, pos)) {
    out->pos = pos;
    out->row = row;
#pragma unroll
    for (int w = 0; w < NV; ++w) reinterpret_cast<uint32_t*>(out->val)[VW * KK + w] = val[w];
  }
}

// x[c] -= l[q] U[q W + c] for q = 0 .. 7 in order, 8 columns, separately rounded: one
// row of U (an LDS broadcast) is read ahead of the one being used. The empty asm
// keeps the elements in this order (reordered, the products are formed ahead and
// spill).
template <typename T>
__device__ __forceinline__ void apply_group(T (&x)[GW], const T (&l)[GW], const T* U) {
#pragma clang fp contract(off)
  T u[GW], un[GW];
#pragma unroll
  for (int c = 0; c < GW; ++c) un[c] = U[c];
#pragma unroll
  for (int q = 0; q < GW; ++q) {
#pragma unroll
    for (int c = 0; c < GW; ++c) u[c] = un[c];
    if (q + 1 < GW) {
#pragma unroll
      for (int c = 0; c < GW; ++c) un[c] = U[(q + 1) * W + c];
    }
#pragma unroll
    for (int c = 0; c < GW; ++c) {
      x[c] = x[c] - l[q] * u[c];
      asm volatile("" : "+v"(x[c]));
    }
  }
}

// NT threads, one row each, its 64 values in registers. moves (absolute rows):
// moves[0] the count, then (destination, source) pairs, as apply_perm_kernel reads
// them.
// Memory is read and written eight lanes to a row (64-byte pieces) and changed to
// one row per thread in LDS: a row per lane straight from memory touches 64 lines
// with every instruction, which took 18,000 cycles of a leaf to load and 25,000 to
// store, against 9,000 and 14,000.
//
// MULTI: G workgroups of NT rows each, all resident. A workgroup's candidate of
// column k travels as tagged words (panel.hpp's protocol) that lie word by word
// over the workgroups, so that one wave reads every workgroup's whole record (lane
// = workgroup) in one poll and needs no second exchange for the winner's row; row
// k needs none either, since rows do not move. (Words 2 KB apart: 512 bytes apart
// the polls of 64 workgroups meet on fewer memory channels, 4,400 against 4,100
// cycles.) After a group the pivot rows' later columns go the same way, once for 8
// columns. Per column, 64 workgroups: exchange 1.7 us, the rest 0.9 us, 220 us a
// leaf; exchanging in two dependent polls beside 64-column updates took 360 us.
// A wait that exceeds spin_limit polls (or any, when it is negative) sets *ws.err
// and ends the kernel in every workgroup; the factors are then invalid.
template <typename T, int NT, bool MULTI>
__global__ void __launch_bounds__(NT)
leaf1_kernel(int64_t Mp, int Wn, T* __restrict__ Pp, int64_t ld, int32_t* __restrict__ ipiv, int64_t row_base,
             int* __restrict__ info, int64_t info_base, int32_t* __restrict__ moves, WS ws, uint32_t tag_base,
             long spin_limit) {
#pragma clang fp contract(off)
  constexpr int NW = NT / 64, NG = W / GW, TLD = GW + 1, RPP = NT / GW;   // RPP: rows of one load instruction
  // this workgroup's rows: M rows at P, panel rows rb ..
  const int G = MULTI ? (int)gridDim.x : 1, wg = MULTI ? (int)blockIdx.x : 0, rb = wg * NT;
  const int M = MULTI ? (int)(Mp - rb < NT ? Mp - rb : NT) : (int)Mp;
  T* const P = Pp + (int64_t)rb * ld;
  __shared__ Leaf1Rec<T> rec[GW][NW];
  __shared__ Leaf1Rec<T> grec[MULTI ? GW : 1];         // the winners over all workgroups
  __shared__ __attribute__((aligned(16))) T U[GW][W];   // the group's pivot rows
  __shared__ T tile[2][NT * TLD];
  __shared__ int32_t s_pos[NT];
  __shared__ int s_cnt, s_abort;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int tr = t / GW, tc = t % GW;   // this thread's row and column of a pass
  const T sfmin = sizeof(T) == 8 ? T(0x1p-1022) : T(0x1p-126);   // lamch('S')
  if (t == 0) { s_cnt = 0; s_abort = 0; }
  int fz = 0, mypos = 0, myrow = 0, kdone = 0;

  int pos = t < M ? rb + t : -1;   // this row's position in the panel; -1: no row
  T a[W];
  // pass g: columns [8 g, 8 g + 8) of every row, element e of this thread at row
  // tr + RPP e; all loads are on their way before the first is waited for (clamped
  // into the panel, then masked), and each pass changes layout in LDS
  {
    T v[NG][GW];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int64_t col = min(GW * g + tc, Wn - 1);
      const T* const last = P + (int64_t)(M - 1) * ld + col;
      const T* p = P + (int64_t)tr * ld + col;
#pragma unroll
      for (int e = 0; e < GW; ++e) {
        v[g][e] = *(tr + RPP * e < M ? p : last);
        p += (int64_t)RPP * ld;
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      T* const q = tile[g & 1];
#pragma unroll
      for (int e = 0; e < GW; ++e) {
        asm volatile("" : "+v"(v[g][e]));
        q[(tr + RPP * e) * TLD + tc] = (tr + RPP * e < M && GW * g + tc < Wn) ? v[g][e] : T(0);
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < GW; ++c) a[GW * g + c] = q[t * TLD + c];
    }
  }

  // gave up: the columns not reached keep their rows (identity interchanges, no moves)
  auto give_up = [&]() __attribute__((always_inline)) {
    if (wg == 0) {
      if (t < Wn) ipiv[t] = (int32_t)(row_base + (t < kdone ? mypos : t) + 1);
      if (t == 0) moves[0] = 0;
    }
  };
  for (int g = 0; g < NG; ++g) {
    const int k0 = GW * g;
    if (k0 >= Wn) break;
    T w[GW];   // the group's columns
#pragma unroll
    for (int gg = 0; gg < NG; ++gg)
      if (gg == g) {
#pragma unroll
        for (int c = 0; c < GW; ++c) w[c] = a[GW * gg + c];
      }
    // one column, its place in the group a constant (a loop over it is not unrolled
    // whole at this size, and indexing registers is slow); false: gave up
    auto column = [&](auto place) __attribute__((always_inline)) {
      constexpr int kk = decltype(place)::value;
      const int k = k0 + kk;
      if (k >= Wn) return true;
      // the wave's candidate; a NaN at position k keeps it (as +inf at the lowest
      // position), elsewhere a NaN never wins
      double f = fabs((double)w[kk]);
      f = f == f ? f : (pos == k ? (double)INFINITY : -1.0);
      f = pos >= k ? f : -1.0;
      const int bp = f >= 0.0 ? pos : INT32_MAX;
      if (lane == winner<64>(f, bp)) {
        Leaf1Rec<T>* const my = &rec[kk][wv];
        my->v = f;
        my->pos = bp;
        my->row = rb + t;
#pragma unroll
        for (int c = 0; c < GW; ++c) my->val[c] = w[c];
      }
      __syncthreads();
      const Leaf1Rec<T>* const q = &rec[kk][NW > 1 ? lane % NW : 0];
      const double qv = q->v;
      const int qp = q->pos, qr = q->row;
      const int ww = NW > 1 ? winner<NW == 1 ? 64 : NW>(qv, qp) : 0;
      int ppos, prow;
      const T* win;
      if constexpr (MULTI) {
        if (wv == 0)
          exchange<T, kk>(&rec[kk][ww], &grec[kk], k, G, wg, lane, ws, tag_base, spin_limit, &s_abort);
        __syncthreads();
        if (s_abort) return false;
        ppos = grec[kk].pos;
        prow = grec[kk].row;
        win = grec[kk].val;
      } else {
        ppos = __builtin_amdgcn_readlane(qp, ww);
        prow = __builtin_amdgcn_readlane(qr, ww);
        win = rec[kk][ww].val;
      }
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
      kdone = k + 1;
      T l = w[kk];
      if (recip) {
        const T rinv = T(1) / piv;
        l = l * rinv;
      } else if (nz) {
        l = l / piv;
      }
      const bool is_piv = prow == rb + t;
      if (pos >= k && !is_piv) {
        w[kk] = l;
#pragma unroll
        for (int c = kk + 1; c < GW; ++c) w[c] = w[c] - l * u[c];
        if (pos == k) pos = ppos;
      }
      if (is_piv) pos = k;
      return true;
    };
    if (!(column(Place<0>{}) && column(Place<1>{}) && column(Place<2>{}) && column(Place<3>{}) &&
          column(Place<4>{}) && column(Place<5>{}) && column(Place<6>{}) && column(Place<7>{}))) {
      give_up();
      return;
    }
#pragma unroll
    for (int gg = 0; gg < NG; ++gg)
      if (gg == g) {
#pragma unroll
        for (int c = 0; c < GW; ++c) a[GW * gg + c] = w[c];
      }
    if (g + 1 >= NG || k0 + GW >= Wn) continue;
    // U of the group's rows: their later columns, u_q = a_q - sum_{j < q} l_qj u_j
    // in order (with the group's columns, which hold the multipliers l)
    if (pos >= k0 && pos < k0 + GW) {
#pragma unroll
      for (int gg = 0; gg < NG; ++gg)
        if (gg >= g) {
#pragma unroll
          for (int c = 0; c < GW; ++c) U[pos - k0][GW * gg + c] = a[GW * gg + c];
        }
    }
    __syncthreads();
    if constexpr (MULTI) {
      // between the workgroups: this one's pivot rows go out, the others' come in
      // (everything goes out before anything is waited for)
      const int rest = W - k0;
      const uint32_t tag = tag_base + (uint32_t)(k0 + GW);
      uint64_t* const xu = ws.u + (size_t)(g & 1) * GW * W * 2;
      for (int e = t; e < GW * rest; e += NT) {
        const int q = e / rest, c = k0 + e % rest;
        if (grec[q].row / NT == wg) st_val<T>(xu + 2 * (q * W + c), tag, U[q][c]);
      }
      for (int e = t; e < GW * rest; e += NT) {
        const int q = e / rest, c = k0 + e % rest;
        if (grec[q].row / NT == wg) continue;
        const uint64_t* const x = xu + 2 * (q * W + c);
        long spins = 0;
        while (true) {
          const uint64_t hi = ld64(x), lo = ld64(x + 1);
          if (tag_of(hi) == tag && tag_of(lo) == tag) {
            U[q][c] = val_of<T>(hi, lo);
            break;
          }
          if (++spins > spin_limit) { s_abort = 1; atomicExch(ws.err, 1); break; }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      __syncthreads();
      if (s_abort) { give_up(); return; }
    }
    const int cu = k0 + GW + t;
    if (cu < W) {
      T x[GW];
#pragma unroll
      for (int q = 0; q < GW; ++q) x[q] = U[q][cu];
#pragma unroll
      for (int q = 1; q < GW; ++q) {
#pragma unroll
        for (int j = 0; j < q; ++j) x[q] = x[q] - U[q][k0 + j] * x[j];
        U[q][cu] = x[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int gg = 1; gg < NG; ++gg)
      if (gg > g) {
        if (pos >= k0 + GW) {
          T x[GW];
#pragma unroll
          for (int c = 0; c < GW; ++c) x[c] = a[GW * gg + c];
          apply_group<T>(x, w, &U[0][GW * gg]);
#pragma unroll
          for (int c = 0; c < GW; ++c) a[GW * gg + c] = x[c];
        } else if (pos >= k0) {   // pivoted in this group: its solved values
#pragma unroll
          for (int c = 0; c < GW; ++c) a[GW * gg + c] = U[pos - k0][GW * gg + c];
        }
      }
  }

  // rows to their final positions (every workgroup's rows were read before its
  // first exchange), pass by pass
  __syncthreads();
  s_pos[t] = pos;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    T* const q = tile[g & 1];
#pragma unroll
    for (int c = 0; c < GW; ++c) q[t * TLD + c] = a[GW * g + c];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < GW; ++e) {
      const int row = tr + RPP * e;
      if (row < M && GW * g + tc < Wn) Pp[(int64_t)s_pos[row] * ld + GW * g + tc] = q[row * TLD + tc];
    }
  }
  // the moves: every pivot row to its position, and the rows that held those
  // positions to where the interchanges left them (all known to workgroup 0)
  if (wg == 0) {
    if (t < Wn && myrow != t) {
      const int q = atomicAdd(&s_cnt, 1);
      moves[1 + 2 * q] = (int32_t)(row_base + t);
      moves[2 + 2 * q] = (int32_t)(row_base + myrow);
    }
    if (t < Wn && pos >= Wn) {
      const int q = atomicAdd(&s_cnt, 1);
      moves[1 + 2 * q] = (int32_t)(row_base + pos);
      moves[2 + 2 * q] = (int32_t)(row_base + t);
    }
    __syncthreads();
    if (t < Wn) ipiv[t] = (int32_t)(row_base + mypos + 1);
    if (t == 0) {
      moves[0] = s_cnt;
      if (fz != 0 && *info == 0) *info = (int)(info_base + fz);
    }
  }
}

}  // namespace panel
}  // namespace zmlhip
