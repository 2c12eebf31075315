// Batched mixed-precision solves of many small independent systems (n <= 256).
//
// No counterpart in zml (its getrf/potrf work on one matrix per call); per
// system the arithmetic is the one of the large mixed solves: an FP32
// factorization and FP64 iterative refinement against the FP64 A.
//
// A plan sorts the systems into size buckets (n <= 32, 64, 128, 256). The two
// smaller buckets run a persistent kernel each, whose workgroups take systems from
// an atomic work queue; a workgroup keeps its system's FP32 factor in registers
// (a TY x TX thread grid, RI x RJ values per thread, NMAX = TY RI = TX RJ) from the
// factorization through every refinement step, and reads the FP64 matrix
// from HBM only for the residuals. The thread-grid shape is chosen by timing the
// candidate shapes on the bucket's own systems (autotune). The two larger buckets
// run one workgroup per system with the factor in matrix-core accumulators. The
// queue resets plus the bucket kernels are captured once into a hipGraph, so that
// one graph launch solves the whole batch.
//
// The FP32 factorization is a Gauss-Jordan inversion in place: general
// systems pivot on the largest |a| of the column among the rows not yet
// chosen (lowest row on ties), with virtual interchanges (a pivot row is
// marked done and stays where it is); SPD systems pivot on the diagonal. The
// result M holds inv(A) up to that row order, inv(A)[k][l] =
// M[prow[k]][invp[l]], so every later solve is one parallel matrix-vector
// product instead of two sequences of n dependent steps.
// Refinement per right-hand side: x = 0, r = b; repeat x += inv32(A) r,
// r = b - A x in FP64, until ||r||_inf <= tol ||A||_inf ||x||_inf n u; a
// system whose backward error stops halving, or that runs out of steps,
// reports -1.
#include "zmlhip_internal.hpp"

#include <algorithm>
#include <cmath>
#include <memory>
#include <type_traits>
#include <vector>

#include "../../include/zmlhip.h"

namespace zmlhip {
namespace {

struct SysDesc {
  const double* a;   // column-major, ld n
  const double* b;   // column-major n x nrhs, ld n
  double* x;
  int n, nrhs, spd, pad;
};

struct BatchArgs {
  const SysDesc* sys;
  const int* list;   // systems of this bucket
  int count;
  int* counter;      // work-queue head (reset before every run)
  int* status;       // per system: refinement steps of its worst right-hand side, or -1
  int max_iter;
  double tol;
};

__device__ __forceinline__ uint64_t bkey(float v, int r) {
  if (v != v) return (uint64_t)(0x7fffffffu - (uint32_t)r);
  return ((uint64_t)__float_as_uint(v) << 32) | (0xffffffffu - (uint32_t)r);
}
__device__ __forceinline__ int bkey_row(uint64_t k) {
  const uint32_t lo = (uint32_t)k;
  return lo >= 0x80000000u ? (int)(0xffffffffu - lo) : (int)(0x7fffffffu - lo);
}

template <int NW>
__device__ __forceinline__ double block_max(double v, double* red, int t) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  double m = red[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) m = fmax(m, red[w]);
  __syncthreads();
  return m;
}

template <int TY, int TX, int RI, int RJ>
__global__ void __launch_bounds__(TY * TX) batched_solve_kernel(BatchArgs g) {
  constexpr int NT = TY * TX, NMAX = TY * RI, NW = (NT + 63) / 64, PARTS = NT / NMAX;
  static_assert(TX * RJ == NMAX && TX <= 64 && RI <= 32, "thread grid shape");
  static_assert(PARTS >= 1 && PARTS * NMAX == NT, "residual split");
  __shared__ uint64_t wbest[NW];
  __shared__ float lcol[NMAX], urow[NMAX], cv[NMAX], yv[NMAX];
  __shared__ int prow[NMAX];
  __shared__ double xv[NMAX], rv[NMAX], red[NW];
  __shared__ double psum[NT], pabs[NT];   // partial residual sums and |a| row sums
  __shared__ int s_idx, s_bad;
  const int t = threadIdx.x, tx = t % TX, ty = t / TX, lane = t & 63, wv = t >> 6;
  for (;;) {
    if (t == 0) s_idx = atomicAdd(g.counter, 1);
    __syncthreads();
    const int idx = s_idx;
    __syncthreads();
    if (idx >= g.count) break;
    const int sid = g.list[idx];
    const SysDesc d = g.sys[sid];
    const int n = d.n;

    // ---- FP32 Gauss-Jordan inversion, in registers
    // a thread row that lies inside n x n is loaded without masks (its RJ
    // loads in flight together); rows at the edge test every element
    float a[RI][RJ];
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const int row = ty + TY * i;
      if (row < n && tx + TX * (RJ - 1) < n) {
#pragma unroll
        for (int j = 0; j < RJ; ++j) a[i][j] = (float)d.a[row + (int64_t)(tx + TX * j) * n];
      } else {
#pragma unroll
        for (int j = 0; j < RJ; ++j) {
          const int col = tx + TX * j;
          a[i][j] = (row < n && col < n) ? (float)d.a[row + (int64_t)col * n] : 0.0f;
        }
      }
    }
    unsigned done = 0;
#pragma unroll
    for (int i = 0; i < RI; ++i)
      if (ty + TY * i >= n) done |= 1u << i;
    if (t == 0) s_bad = 0;
#pragma unroll
    for (int jj = 0; jj < RJ; ++jj) {
      for (int kq = 0; kq < TX; ++kq) {
        const int k = jj * TX + kq;
        if (k >= n) break;
        int p = k;
        if (!d.spd) {
          uint64_t best = 0;
          if (tx == kq) {
#pragma unroll
            for (int i = 0; i < RI; ++i)
              if (!((done >> i) & 1u)) {
                const uint64_t key = bkey(fabsf(a[i][jj]), ty + TY * i);
                best = key > best ? key : best;
              }
          }
#pragma unroll
          for (int off = TX; off < 64; off <<= 1) {
            const uint64_t o = __shfl_xor(best, off);
            best = o > best ? o : best;
          }
          if (lane == kq) wbest[wv] = best;
        }
        // also orders this step's urow / lcol writes after the previous step's reads
        __syncthreads();
        if (!d.spd) {
          uint64_t gk = wbest[0];
#pragma unroll
          for (int w = 1; w < NW; ++w) gk = wbest[w] > gk ? wbest[w] : gk;
          p = bkey_row(gk);
        }
        const int pt = p % TY, pi = p / TY;
        if (ty == pt) {   // the pivot row
#pragma unroll
          for (int i = 0; i < RI; ++i)
            if (i == pi) {
#pragma unroll
              for (int j = 0; j < RJ; ++j) urow[tx + TX * j] = a[i][j];
            }
          done |= 1u << pi;
        }
        if (tx == kq) {   // column k: the multipliers of every other row
#pragma unroll
          for (int i = 0; i < RI; ++i) lcol[ty + TY * i] = (ty + TY * i == p) ? 0.0f : a[i][jj];
        }
        if (t == 0) prow[k] = p;
        __syncthreads();
        const float pv = urow[k];
        if (t == 0 && !(pv != 0.0f && pv == pv)) s_bad = 1;
        const float rp = 1.0f / pv;
        float fi[RI], uj[RJ];
#pragma unroll
        for (int i = 0; i < RI; ++i) fi[i] = lcol[ty + TY * i];
#pragma unroll
        for (int j = 0; j < RJ; ++j) uj[j] = urow[tx + TX * j] * rp;
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
          for (int j = 0; j < RJ; ++j) a[i][j] -= fi[i] * uj[j];
        if (ty == pt) {
#pragma unroll
          for (int i = 0; i < RI; ++i)
            if (i == pi) {
#pragma unroll
              for (int j = 0; j < RJ; ++j) a[i][j] = uj[j];
            }
        }
        if (tx == kq) {
#pragma unroll
          for (int i = 0; i < RI; ++i) a[i][jj] = (ty + TY * i == p) ? rp : -fi[i] * rp;
        }
      }
    }
    __syncthreads();
    // a now holds M with inv(A)[k][l] = M[prow[k]][invp[l]]: x = inv(A) r is
    // c_j = r[prow[j]], y = M c, x_k = y[prow[k]]

    // ---- FP64 refinement of every right-hand side
    int worst = s_bad ? -1 : 0;
    double anorm = 0.0;
    for (int q = 0; q < d.nrhs && worst >= 0; ++q) {
      const double* b = d.b + (int64_t)q * n;
      if (t < NMAX) {
        xv[t] = 0.0;
        rv[t] = t < n ? b[t] : 0.0;
      }
      __syncthreads();
      double prev = INFINITY;
      int it = 0;
      for (;;) {
        if (t < NMAX) cv[t] = t < n ? (float)rv[prow[t]] : 0.0f;
        __syncthreads();
        float acc[RI];
#pragma unroll
        for (int i = 0; i < RI; ++i) {
          float s = 0.0f;
#pragma unroll
          for (int j = 0; j < RJ; ++j) s = fmaf(a[i][j], cv[tx + TX * j], s);
          acc[i] = s;
        }
#pragma unroll
        for (int off = TX / 2; off > 0; off >>= 1)
#pragma unroll
          for (int i = 0; i < RI; ++i) acc[i] += __shfl_xor(acc[i], off);
        if (tx == 0) {
#pragma unroll
          for (int i = 0; i < RI; ++i) yv[ty + TY * i] = acc[i];
        }
        __syncthreads();
        if (t < n) xv[t] += (double)yv[prow[t]];
        __syncthreads();
        // r = b - A x, ||A||_inf on the first pass. Thread t takes row t % NMAX
        // and the columns t / NMAX + PARTS l, eight loads in flight at a time (a
        // tail of fewer than eight one by one); the PARTS partial sums of a row
        // are then added in a fixed order.
        {
          const int row = t % NMAX, part = t / NMAX;
          double accd = 0.0, asum = 0.0;
          if (row < n) {
            int j0 = part;
            for (; j0 + 7 * PARTS < n; j0 += 8 * PARTS) {   // eight whole columns: no masks
              double v[8];
#pragma unroll
              for (int u = 0; u < 8; ++u) v[u] = d.a[row + (int64_t)(j0 + u * PARTS) * n];
#pragma unroll
              for (int u = 0; u < 8; ++u) {
                accd -= v[u] * xv[j0 + u * PARTS];
                asum += fabs(v[u]);
              }
            }
            for (; j0 < n; j0 += PARTS) {
              const double v = d.a[row + (int64_t)j0 * n];
              accd -= v * xv[j0];
              asum += fabs(v);
            }
          }
          psum[t] = accd;
          pabs[t] = asum;
        }
        __syncthreads();
        double ri = 0.0, ai = 0.0;
        if (t < n) {
          double accd = b[t], asum = 0.0;
#pragma unroll
          for (int q = 0; q < PARTS; ++q) {
            accd += psum[q * NMAX + t];
            asum += pabs[q * NMAX + t];
          }
          rv[t] = accd;
          ri = accd == accd ? fabs(accd) : INFINITY;   // (a maximum passes over NaN)
          ai = asum;
        }
        if (anorm == 0.0) anorm = block_max<NW>(ai, red, t);
        const double rmax = block_max<NW>(ri, red, t);
        const double xmax = block_max<NW>(t < n ? fabs(xv[t]) : 0.0, red, t);
        ++it;
        const double be = rmax / (anorm * xmax * (double)n * 0x1p-53);
        if (be <= g.tol) break;
        if (!(be < INFINITY) || it >= g.max_iter || (it >= 2 && be > 0.5 * prev)) {
          it = -1;
          break;
        }
        prev = be;
      }
      if (t < n) d.x[(int64_t)q * n + t] = xv[t];
      worst = it < 0 ? -1 : std::max(worst, it);
      __syncthreads();
    }
    if (t == 0) g.status[sid] = worst;
    __syncthreads();
  }
}

// ---- n <= 128 and n <= 256: the matrix in MFMA accumulators, 16 columns at a time
//
// ND waves hold the FP32 matrix as 32 x 32 accumulator tiles (wave w the rows
// 32 w .. 32 w + 31 of ND tiles), and ND / 2 helper waves hold nothing. The
// Gauss-Jordan steps go in chunks of 16 columns: helper wave 0 has the chunk in its
// registers (rows lane + 64 m) and runs its 16 steps there, without barriers: the
// pivot's rank through DPP, the pivot row into scalar registers, one reciprocal,
// the other rows' update (the pivot row's own factor 1 / pivot is applied at the end
// of the chunk). That leaves G, the chunk's columns of the result; with U the pivot
// rows' values in the other columns before the chunk, every other column becomes
// M + G U, pivot rows counted as zero in M: one product of inner length 16 on the
// matrix cores. The tile with the next chunk goes first, the rest while helper wave
// 0 runs the next steps. (A last chunk of fewer than 16 columns is filled up with
// the identity.)
// Refinement: the accumulator waves form inv32(A) r, the helper threads (one row
// each) the FP64 residuals, for up to four right-hand sides in one pass over A.
//
// Bound by helper wave 0's chain, about 1,000 cycles a column, with one workgroup
// on a CU at n <= 256 (its registers hold no second one): 145 of 200 us a system,
// the rest the residuals' passes over A. 4,000 systems of order 129 .. 256: 3.16 ms,
// 65 .. 128: 0.87 ms (one MI355X). A thread grid with 128 (64) entries a thread,
// two barriers, a search through LDS and a rank-1 update in every column, half of
// whose instructions moved operands between the register files, and one pass over
// A for every right-hand side and step took 7.29 and 1.32 ms.
constexpr int BQ = 4;   // right-hand sides refined together

__device__ __forceinline__ int imax_all(int v) {   // the largest v of the wave, in every lane
  auto step = [&](int o) { v = o > v ? o : v; };
  step(__builtin_amdgcn_update_dpp((int)0x80000000, v, 0xb1, 0xf, 0xf, false));    // quad_perm [1,0,3,2]
  step(__builtin_amdgcn_update_dpp((int)0x80000000, v, 0x4e, 0xf, 0xf, false));    // quad_perm [2,3,0,1]
  step(__builtin_amdgcn_update_dpp((int)0x80000000, v, 0x124, 0xf, 0xf, false));   // row_ror:4
  step(__builtin_amdgcn_update_dpp((int)0x80000000, v, 0x128, 0xf, 0xf, false));   // row_ror:8
  step(__builtin_amdgcn_update_dpp((int)0x80000000, v, 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1, 3
  step(__builtin_amdgcn_update_dpp((int)0x80000000, v, 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2, 3
  return __builtin_amdgcn_readlane(v, 63);
}

template <int ND>
struct TileShared {
  static constexpr int NMAX = 32 * ND, CW = 16, CS = CW + 4, NH = ND / 2;
  float chunk[2][NMAX * CS];   // row r of a chunk at r CS; the two together stage A at the start
  float ubuf[CW * NMAX];       // row s: the chunk's pivot row s before the chunk
  float cv[BQ][NMAX], yv[BQ][NMAX];
  double xv[NMAX][BQ], rv[BQ][NMAX];
  double red[NH][2 * BQ + 1];
  int rstep[NMAX], prow[NMAX];   // the step that chose a row (-1: none yet), the row of a step
  int bad;
  int again, solved;   // another step of this group (written before R5); the group did not fail (before R6)
};

// One chunk's steps in helper wave 0: x[m] the values of row lane + 64 m, on[m] all
// bits while the row can be chosen, else 0.
template <int RL>
__device__ __forceinline__ void chunk_inverse(float (&x)[RL][16], int (&on)[RL], int k0, bool spd, int lane,
                                              int& mine, bool& fine) {
  float sc[RL];   // the factor of a pivot row of this chunk
#pragma unroll
  for (int m = 0; m < RL; ++m) sc[m] = 1.0f;
#pragma unroll
  for (int kq = 0; kq < 16; ++kq) {
    float pr[16];
    int p = 0;
    auto take = [&](auto place, int pl) __attribute__((always_inline)) {
      constexpr int m = decltype(place)::value;
      if constexpr (m < RL) {
        p = pl + 64 * m;
#pragma unroll
        for (int c = 0; c < 16; ++c) pr[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[m][c]), pl));
      }
    };
    int pl = (k0 + kq) & 63, pm = (k0 + kq) >> 6;
    if (!spd) {
      // rank: the bits of |a|, then those of -2.0 for NaN, the lowest for a row already chosen
      int f[RL], fl = INT32_MIN;
#pragma unroll
      for (int m = 0; m < RL; ++m) {
        f[m] = min(__float_as_int(fmaxf(fabsf(x[m][kq]), -2.0f)), on[m] ^ INT32_MIN);
        fl = max(fl, f[m]);
      }
      const int fm = imax_all(fl);
      uint64_t hit = 0;   // lowest row of that rank
#pragma unroll
      for (int m = RL - 1; m >= 0; --m) {
        const uint64_t h = __ballot(f[m] == fm);
        pm = h ? m : pm;
        hit = h ? h : hit;
      }
      pl = hit ? (int)__builtin_ctzll(hit) : 0;
    }
    if (pm < 2) {
      if (pm == 0) take(std::integral_constant<int, 0>{}, pl);
      else take(std::integral_constant<int, 1>{}, pl);
    } else {
      if (pm == 2) take(std::integral_constant<int, 2>{}, pl);
      else take(std::integral_constant<int, 3>{}, pl);
    }
    const float pv = pr[kq];
    fine = fine && pv != 0.0f && pv == pv;
    mine = lane == kq ? p : mine;   // lane q keeps step q's row
    const float rp = 1.0f / pv;
    float l[RL];
#pragma unroll
    for (int m = 0; m < RL; ++m) {
      const bool sel = lane + 64 * m == p;
      const float f = x[m][kq] * rp;
      l[m] = sel ? 0.0f : f;
      x[m][kq] = sel ? 1.0f : -f;
      sc[m] = sel ? rp : sc[m];
      on[m] = sel ? 0 : on[m];
    }
#pragma unroll
    for (int c = 0; c < 16; ++c)
      if (c != kq) {
#pragma unroll
        for (int m = 0; m < RL; ++m) x[m][c] -= l[m] * pr[c];
      }
  }
#pragma unroll
  for (int m = 0; m < RL; ++m)
#pragma unroll
    for (int c = 0; c < 16; ++c) x[m][c] *= sc[m];
}

template <int ND>
__global__ void __launch_bounds__((ND + ND / 2) * 64, ND == 8 ? 3 : 4) batched_tile_kernel(BatchArgs g) {
  typedef float f32x16 __attribute__((ext_vector_type(16)));
  typedef TileShared<ND> Sh;
  constexpr int NMAX = Sh::NMAX, CW = Sh::CW, CS = Sh::CS, NH = Sh::NH, RL = NMAX / 64;
  __shared__ __align__(16) Sh sh;
  const int t = threadIdx.x, lane = t & 63, wid = __builtin_amdgcn_readfirstlane(t >> 6);
  // waves go to the four SIMDs in turn: wave 0, with the steps' chain, shares its
  // SIMD with helper waves only
  const bool holds = wid % 4 != 0 && wid != 11;
  const int wv = holds ? wid - wid / 4 - 1 : (wid == 11 ? 3 : wid / 4);
  const int li = lane & 31, hk = lane >> 5;
  const int sid = g.list[blockIdx.x];   // (larger systems come first)
  const SysDesc d = g.sys[sid];
  const int n = d.n, nch = (n + CW - 1) / CW;
  const int groups = (d.nrhs + BQ - 1) / BQ;

  // The two kinds of waves take separate paths with the same barriers, so that
  // neither carries the other's registers.
  if (!holds) {
    const int u = 64 * wv + lane;   // this thread's row
    sh.rstep[u] = -1;
    if (u == 0) sh.bad = 0;
    for (int j = 0; j < ND; ++j) {   // (the accumulator waves stage A)
      __syncthreads();
      __syncthreads();
    }
    __syncthreads();
#pragma unroll 1
    for (int ch = 0; ch < nch; ++ch) {
      const int k0 = CW * ch;
      if (wv == 0) {
        __builtin_amdgcn_s_setprio(3);
        float* const cc = sh.chunk[ch & 1];
        float x[RL][CW];
        int on[RL], mine = 0;
        bool fine = true;
#pragma unroll
        for (int m = 0; m < RL; ++m) {
          const int row = lane + 64 * m;
#pragma unroll
          for (int q = 0; q < CW / 4; ++q) {
            const float4 v = *reinterpret_cast<const float4*>(&cc[row * CS + 4 * q]);
            x[m][4 * q] = v.x;
            x[m][4 * q + 1] = v.y;
            x[m][4 * q + 2] = v.z;
            x[m][4 * q + 3] = v.w;
          }
          on[m] = row < CW * nch && sh.rstep[row] < 0 ? -1 : 0;
        }
        chunk_inverse<RL>(x, on, k0, d.spd != 0, lane, mine, fine);
#pragma unroll
        for (int m = 0; m < RL; ++m)
#pragma unroll
          for (int q = 0; q < CW / 4; ++q)
            *reinterpret_cast<float4*>(&cc[(lane + 64 * m) * CS + 4 * q]) =
                make_float4(x[m][4 * q], x[m][4 * q + 1], x[m][4 * q + 2], x[m][4 * q + 3]);
        if (lane < CW) {
          sh.prow[k0 + lane] = mine;
          sh.rstep[mine] = k0 + lane;
        }
        if (lane == 0 && !fine) sh.bad = 1;
        __builtin_amdgcn_s_setprio(0);
      }
      __syncthreads();   // B1: G is there, the last chunk's product is done
      __syncthreads();   // B2: U is there
      __syncthreads();   // B3: the next chunk is there
    }
    // ---- refinement
    int worst = sh.bad ? -1 : 0;
    const int pu = u < n ? sh.prow[u] : 0;   // (a row also when the system is bad: every step chose one)
    double anorm = 0.0;
#pragma unroll 1
    for (int gq = 0; gq < groups && worst >= 0; ++gq) {
      const int q0 = gq * BQ, nq = min(BQ, d.nrhs - q0);
      const double* const b = d.b + (int64_t)q0 * n;
      double x[BQ], prev[BQ];
      int it[BQ];
      bool act[BQ];
#pragma unroll
      for (int q = 0; q < BQ; ++q) {
        x[q] = 0.0;
        sh.rv[q][u] = q < nq && u < n ? b[(int64_t)q * n + u] : 0.0;
        prev[q] = INFINITY;
        it[q] = 0;
        act[q] = q < nq;
      }
      __syncthreads();   // R0
      for (;;) {
#pragma unroll
        for (int q = 0; q < BQ; ++q) sh.cv[q][u] = u < n ? (float)sh.rv[q][pu] : 0.0f;
        __syncthreads();   // R1
        __syncthreads();   // R2: yv
#pragma unroll
        for (int q = 0; q < BQ; ++q) {
          if (act[q] && u < n) x[q] += (double)sh.yv[q][pu];
          sh.xv[u][q] = x[q];
        }
        __syncthreads();   // R3
        // r = b - A x and the row sums of |A|, one row per thread: sums of 8 columns,
        // added up (one column after the other onto b left solutions 1.8 to 2.4 times as far
        // from the exact ones: 4.6e-16 against 2.5e-16 at n = 70, 1.16e-15 against 4.7e-16 at 256)
        double acc[BQ], sum[BQ], asum = 0.0;
#pragma unroll
        for (int q = 0; q < BQ; ++q) sum[q] = 0.0;
        if (u < n) {
          const double* pa = d.a + u;
          auto one = [&](double v, int j) __attribute__((always_inline)) {
            const double2 x01 = *reinterpret_cast<const double2*>(&sh.xv[j][0]);
            const double2 x23 = *reinterpret_cast<const double2*>(&sh.xv[j][2]);
            acc[0] += v * x01.x;
            acc[1] += v * x01.y;
            acc[2] += v * x23.x;
            acc[3] += v * x23.y;
            asum += fabs(v);
          };
          int j = 0;
          for (; j + 16 <= n; j += 16) {
            double v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = pa[(int64_t)(j + e) * n];
#pragma unroll
            for (int h = 0; h < 16; h += 8) {
#pragma unroll
              for (int q = 0; q < BQ; ++q) acc[q] = 0.0;
#pragma unroll
              for (int e = h; e < h + 8; ++e) one(v[e], j + e);
#pragma unroll
              for (int q = 0; q < BQ; ++q) sum[q] += acc[q];
            }
          }
#pragma unroll
          for (int q = 0; q < BQ; ++q) acc[q] = 0.0;
          for (; j < n; ++j) one(pa[(int64_t)j * n], j);
#pragma unroll
          for (int q = 0; q < BQ; ++q) sum[q] += acc[q];
        }
#pragma unroll
        for (int q = 0; q < BQ; ++q) acc[q] = q < nq && u < n ? b[(int64_t)q * n + u] - sum[q] : 0.0;
        double mx[2 * BQ + 1];
#pragma unroll
        for (int q = 0; q < BQ; ++q) {
          sh.rv[q][u] = acc[q];
          mx[q] = acc[q] == acc[q] ? fabs(acc[q]) : INFINITY;   // (a maximum passes over NaN)
          mx[BQ + q] = fabs(x[q]);
        }
        mx[2 * BQ] = asum;
#pragma unroll
        for (int e = 0; e < 2 * BQ + 1; ++e) {
          for (int off = 32; off > 0; off >>= 1) mx[e] = fmax(mx[e], __shfl_xor(mx[e], off));
          if (lane == 0) sh.red[wv][e] = mx[e];
        }
        __syncthreads();   // R4
#pragma unroll
        for (int e = 0; e < 2 * BQ + 1; ++e) {
          mx[e] = sh.red[0][e];
#pragma unroll
          for (int w = 1; w < NH; ++w) mx[e] = fmax(mx[e], sh.red[w][e]);
        }
        if (anorm == 0.0) anorm = mx[2 * BQ];
        bool go = false;
#pragma unroll
        for (int q = 0; q < BQ; ++q) {
          if (!act[q]) continue;
          ++it[q];
          const double be = mx[q] / (anorm * mx[BQ + q] * (double)n * 0x1p-53);
          if (be <= g.tol) {
            act[q] = false;
          } else if (!(be < INFINITY) || it[q] >= g.max_iter || (it[q] >= 2 && be > 0.5 * prev[q])) {
            it[q] = -1;
            act[q] = false;
          } else {
            prev[q] = be;
            go = true;
          }
        }
        if (u == 0) sh.again = go;
        __syncthreads();   // R5
        if (!go) break;
      }
#pragma unroll
      for (int q = 0; q < BQ; ++q) {
        if (q >= nq || worst < 0) continue;   // (nothing is written after a right-hand side that failed)
        if (u < n) d.x[(int64_t)(q0 + q) * n + u] = x[q];
        worst = it[q] < 0 ? -1 : max(worst, it[q]);
      }
      if (u == 0) sh.solved = worst >= 0;   // (a word of its own: a late wave may still be reading `again`)
      __syncthreads();   // R6
    }
    if (u == 0) g.status[sid] = worst;
    return;
  }

  const int row0 = 32 * wv + 4 * hk;   // element r of a tile: row row0 + 8 (r / 4) + r % 4, column li
  const int nj = (n + 31) / 32;        // tiles of a row (and accumulator waves) in use
  f32x16 a[ND];
  // A is column-major and a lane of a tile holds columns: tile by tile through LDS
  // (consecutive threads read consecutive rows), the next tile's reads in flight
  {
    constexpr int TS = NMAX + 4, PT = NMAX * 32 / (ND * 64);   // column stride, elements of a thread
    static_assert(32 * TS <= 2 * NMAX * CS, "a tile column fits the chunk buffers");
    float* const st = sh.chunk[0];
    const int th = 64 * wv + lane, sr = th % NMAX, sc = th / NMAX;   // row, first column (then + 2)
    double v[PT];
    auto fetch = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < PT; ++e) {
        const int c = 32 * j + sc + 2 * e;
        const double w = d.a[min(sr, n - 1) + (int64_t)min(c, n - 1) * n];
        v[e] = sr < n && c < n ? w : (sr == c && c < CW * nch ? 1.0 : 0.0);   // the rest of the last chunk: identity
      }
    };
    fetch(0);
#pragma unroll
    for (int j = 0; j < ND; ++j) {
#pragma unroll
      for (int e = 0; e < PT; ++e) st[(sc + 2 * e) * TS + sr] = (float)v[e];
      if (j + 1 < nj) fetch(j + 1);
      else {
#pragma unroll
        for (int e = 0; e < PT; ++e) v[e] = 0.0;
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 w = *reinterpret_cast<const float4*>(&st[li * TS + row0 + 8 * q]);
        a[j][4 * q] = w.x;
        a[j][4 * q + 1] = w.y;
        a[j][4 * q + 2] = w.z;
        a[j][4 * q + 3] = w.w;
      }
      __syncthreads();
    }
  }
  if (li < CW) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sh.chunk[0][(row0 + 8 * (r >> 2) + (r & 3)) * CS + li] = a[0][r];
  }
  __syncthreads();
  int hits = 0;
  auto drop = [&](f32x16& v) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = hits & (1 << r) ? 0.0f : v[r];
  };
#pragma unroll 1
  for (int ch = 0;; ++ch) {
    const int k0 = CW * ch, h = ch & 1;
    const float* const cc = sh.chunk[h];
    if (ch > 0) {
      // ---- the last chunk's G U in the tiles but this chunk's, then its own
      // columns back into their tile
      const float* const cp = sh.chunk[h ^ 1];
      const int skip = ch < nch ? ch >> 1 : ND;
      if (wv < nj) {
        float l[CW / 2];
#pragma unroll
        for (int s = 0; s < CW / 2; ++s) l[s] = cp[(32 * wv + li) * CS + 2 * s + hk];
#pragma unroll
        for (int j = 0; j < ND; ++j)
          if (j < nj && j != skip) {
            drop(a[j]);
#pragma unroll
            for (int s = 0; s < CW / 2; ++s)
              a[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(l[s], sh.ubuf[(2 * s + hk) * NMAX + 32 * j + li], a[j], 0, 0, 0);
          }
#pragma unroll
        for (int j = 0; j < ND; ++j)
          if (j == (ch - 1) >> 1 && (li / CW) != h) {
#pragma unroll
            for (int r = 0; r < 16; ++r) a[j][r] = cp[(row0 + 8 * (r >> 2) + (r & 3)) * CS + li % CW];
          }
      }
      if (ch == nch) break;
    }
    __syncthreads();   // B1
    // ---- the chunk's pivot rows to ubuf; they count as zero from here (bit r of
    // `hits`: element r's row is one)
    hits = 0;
    if (wv < nj) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int4 v = *reinterpret_cast<const int4*>(&sh.rstep[row0 + 8 * q]);
        const int rs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int st = rs[e] - k0;
          hits |= st >= 0 ? 1 << (4 * q + e) : 0;
          if (st >= 0) {
#pragma unroll
            for (int j = 0; j < ND; ++j) sh.ubuf[st * NMAX + 32 * j + li] = a[j][4 * q + e];
          }
        }
      }
    }
    __syncthreads();   // B2
    if (ch + 1 < nch && wv < nj) {
      // ---- the tile with the next chunk, and the chunk out to LDS
      const int jn = (ch + 1) >> 1;
      float l[CW / 2];
#pragma unroll
      for (int s = 0; s < CW / 2; ++s) l[s] = cc[(32 * wv + li) * CS + 2 * s + hk];
#pragma unroll
      for (int j = 0; j < ND; ++j)
        if (j == jn) {
          drop(a[j]);
#pragma unroll
          for (int s = 0; s < CW / 2; ++s)
            a[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(l[s], sh.ubuf[(2 * s + hk) * NMAX + 32 * j + li], a[j], 0, 0, 0);
        }
      float* const cn = sh.chunk[h ^ 1];
#pragma unroll
      for (int j = 0; j < ND; ++j)
        if (j == jn && (li / CW) != h) {
#pragma unroll
          for (int r = 0; r < 16; ++r) cn[(row0 + 8 * (r >> 2) + (r & 3)) * CS + li % CW] = a[j][r];
        }
    }
    __syncthreads();   // B3
  }
  // ---- refinement: y = M c, row sums over the half wave's 32 columns and the tiles
  int ok = !sh.bad;
#pragma unroll 1
  for (int gq = 0; gq < groups && ok; ++gq) {
    const int nq = min(BQ, d.nrhs - gq * BQ);
    __syncthreads();   // R0
    for (;;) {
      __syncthreads();   // R1
      if (wv < nj) {
#pragma unroll 1
        for (int q = 0; q < nq; ++q) {
          float v[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) v[r] = 0.0f;
#pragma unroll
          for (int j = 0; j < ND; ++j)
            if (j < nj) {
              const float c = sh.cv[q][32 * j + li];
#pragma unroll
              for (int r = 0; r < 16; ++r) v[r] = fmaf(a[j][r], c, v[r]);
            }
          // halves of the values change hands until lane li has row (li >> 1) & 15's sum
#pragma unroll
          for (int w = 8; w >= 1; w >>= 1) {
            const bool up = (li & (2 * w)) != 0;
#pragma unroll
            for (int r = 0; r < w; ++r) {
              const float keep = up ? v[r + w] : v[r], send = up ? v[r] : v[r + w];
              v[r] = keep + __shfl_xor(send, 2 * w);
            }
          }
          const float y = v[0] + __shfl_xor(v[0], 1);
          const int r = li >> 1;
          if ((li & 1) == 0) sh.yv[q][row0 + 8 * (r >> 2) + (r & 3)] = y;
        }
      }
      __syncthreads();   // R2
      __syncthreads();   // R3
      __syncthreads();   // R4
      __syncthreads();   // R5
      if (!sh.again) break;
    }
    __syncthreads();   // R6
    ok = sh.solved;
  }
}

__global__ void reset_counters_kernel(int* c, int k) {
  if ((int)threadIdx.x < k) c[threadIdx.x] = 0;
}

// ---- variants and buckets -------------------------------------------------------------
struct Variant {
  int ty, tx, ri, rj;   // thread grid TY x TX, RI x RJ values per thread (tiles: 32 rows, RI tiles each way)
  void (*kernel)(BatchArgs);
  int nt;               // threads
  bool queue;           // persistent workgroups on the bucket's work queue
};
const Variant kVariants[] = {
    {8, 8, 4, 4, batched_solve_kernel<8, 8, 4, 4>, 64, true},        // n <= 32, one wave
    {8, 8, 8, 8, batched_solve_kernel<8, 8, 8, 8>, 64, true},        // n <= 64, one wave
    {16, 16, 4, 4, batched_solve_kernel<16, 16, 4, 4>, 256, true},    // n <= 64, four waves
    {32, 12, 4, 4, batched_tile_kernel<4>, 384, false},           // n <= 128, accumulator tiles
    {32, 24, 8, 8, batched_tile_kernel<8>, 768, false},           // n <= 256, accumulator tiles
};
constexpr int kBuckets = 4;
const int kBucketMax[kBuckets] = {32, 64, 128, 256};
const std::vector<int> kCandidates[kBuckets] = {{0, 1, 2}, {1, 2}, {3}, {4}};

}  // namespace

struct BatchPlan {
  int count = 0;
  SysDesc* d_sys = nullptr;
  int* d_lists = nullptr;
  int* d_counters = nullptr;
  int* d_status = nullptr;
  int bucket_count[kBuckets] = {};
  int bucket_offset[kBuckets] = {};
  int variant[kBuckets] = {};
  unsigned grid[kBuckets] = {};
  BatchArgs args[kBuckets];
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  ~BatchPlan() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    for (void* p : {(void*)d_sys, (void*)d_lists, (void*)d_counters, (void*)d_status})
      if (p) (void)hipFree(p);
  }
};

namespace {

unsigned resident_grid(int v) {
  int per_cu = 0;
  const int nt = kVariants[v].nt;
  ZH_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kVariants[v].kernel),
                                                        nt, 0));
  return (unsigned)(std::max(per_cu, 1) * device_cu_count());
}

void launch_bucket(const BatchPlan& P, int b, int v, hipStream_t s) {
  const int nt = kVariants[v].nt;
  // (the tile kernels take one system per workgroup, in list order)
  const unsigned grid = kVariants[v].queue ? std::min<unsigned>(P.grid[b], (unsigned)std::max(1, P.bucket_count[b]))
                                           : (unsigned)P.bucket_count[b];
  BatchArgs args = P.args[b];
  void* kargs[] = {&args};
  ZH_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(kVariants[v].kernel), dim3(grid), dim3(nt), kargs, 0, s));
}

}  // namespace

BatchPlan* batch_plan_create(int count, const int* n, const int* nrhs, const int* spd,
                             const double* const* a, const double* const* b, double* const* x,
                             const zmlhip_ir_opts* opts, int autotune, hipStream_t s) {
  std::unique_ptr<BatchPlan> P(new BatchPlan);
  P->count = count;
  std::vector<SysDesc> h(count);
  std::vector<std::vector<int>> lists(kBuckets);
  for (int i = 0; i < count; ++i) {
    h[i] = SysDesc{a[i], b[i], x[i], n[i], nrhs[i], spd ? (spd[i] ? 1 : 0) : 0, 0};
    int bk = 0;
    while (bk < kBuckets - 1 && n[i] > kBucketMax[bk]) ++bk;
    lists[bk].push_back(i);
  }
  std::vector<int> flat;
  for (int bk = 0; bk < kBuckets; ++bk) {
    // larger systems first inside a bucket: the queue ends on the short ones
    std::stable_sort(lists[bk].begin(), lists[bk].end(), [&](int u, int v) { return n[u] > n[v]; });
    P->bucket_offset[bk] = (int)flat.size();
    P->bucket_count[bk] = (int)lists[bk].size();
    flat.insert(flat.end(), lists[bk].begin(), lists[bk].end());
  }
  ZH_CHECK(device_alloc(reinterpret_cast<void**>(&P->d_sys), sizeof(SysDesc) * std::max(count, 1)));
  ZH_CHECK(device_alloc(reinterpret_cast<void**>(&P->d_lists), sizeof(int) * std::max<size_t>(flat.size(), 1)));
  ZH_CHECK(device_alloc(reinterpret_cast<void**>(&P->d_counters), sizeof(int) * 64));
  ZH_CHECK(device_alloc(reinterpret_cast<void**>(&P->d_status), sizeof(int) * std::max(count, 1)));
  ZH_CHECK(hipMemcpyAsync(P->d_sys, h.data(), sizeof(SysDesc) * count, hipMemcpyHostToDevice, s));
  if (!flat.empty())
    ZH_CHECK(hipMemcpyAsync(P->d_lists, flat.data(), sizeof(int) * flat.size(), hipMemcpyHostToDevice, s));
  const int max_iter = opts && opts->max_iter > 0 ? opts->max_iter : 10;
  const double tol = opts && opts->tol > 0.0 ? opts->tol : 1.0;
  for (int bk = 0; bk < kBuckets; ++bk) {
    P->args[bk] = BatchArgs{P->d_sys, P->d_lists + P->bucket_offset[bk], P->bucket_count[bk],
                            P->d_counters + bk, P->d_status, max_iter, tol};
    P->variant[bk] = kCandidates[bk].back();
  }
  // autotune: time every candidate shape on the bucket's own systems
  for (int bk = 0; bk < kBuckets; ++bk) {
    const auto& cand = kCandidates[bk];
    if (P->bucket_count[bk] == 0) continue;
    float best = INFINITY;
    if (!autotune || cand.size() == 1) {
      P->grid[bk] = resident_grid(P->variant[bk]);
      continue;
    }
    hipEvent_t e0, e1;
    ZH_CHECK(hipEventCreate(&e0));
    ZH_CHECK(hipEventCreate(&e1));
    for (int v : cand) {
      P->grid[bk] = resident_grid(v);
      float ms = 0.0f;
      for (int rep = 0; rep < 2; ++rep) {   // the first run warms up
        hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(64), 0, s, P->d_counters, kBuckets);
        ZH_CHECK(hipEventRecord(e0, s));
        launch_bucket(*P, bk, v, s);
        ZH_CHECK(hipEventRecord(e1, s));
        ZH_CHECK(hipEventSynchronize(e1));
        ZH_CHECK(hipEventElapsedTime(&ms, e0, e1));
      }
      if (ms < best) {
        best = ms;
        P->variant[bk] = v;
      }
    }
    P->grid[bk] = resident_grid(P->variant[bk]);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  }
  // one graph: reset the queues, then the buckets as independent branches (their
  // workgroups only take work from their own queues, so the small buckets can use
  // the CUs the large one leaves idle as its queue drains)
  hipStream_t cs[kBuckets];
  hipEvent_t ev[kBuckets + 1];
  for (int i = 0; i < kBuckets; ++i) ZH_CHECK(hipStreamCreateWithFlags(&cs[i], hipStreamNonBlocking));
  for (int i = 0; i <= kBuckets; ++i) ZH_CHECK(hipEventCreateWithFlags(&ev[i], hipEventDisableTiming));
  ZH_CHECK(hipStreamBeginCapture(cs[0], hipStreamCaptureModeThreadLocal));
  hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(64), 0, cs[0], P->d_counters, kBuckets);
  ZH_CHECK(hipEventRecord(ev[kBuckets], cs[0]));
  for (int i = 1; i < kBuckets; ++i) ZH_CHECK(hipStreamWaitEvent(cs[i], ev[kBuckets], 0));
  for (int bk = kBuckets - 1, i = 0; bk >= 0; --bk, ++i)   // the largest bucket on the capturing stream
    if (P->bucket_count[bk] > 0) launch_bucket(*P, bk, P->variant[bk], cs[i]);
  for (int i = 1; i < kBuckets; ++i) {
    ZH_CHECK(hipEventRecord(ev[i], cs[i]));
    ZH_CHECK(hipStreamWaitEvent(cs[0], ev[i], 0));
  }
  ZH_CHECK(hipStreamEndCapture(cs[0], &P->graph));
  for (int i = 0; i < kBuckets; ++i) ZH_CHECK(hipStreamDestroy(cs[i]));
  for (int i = 0; i <= kBuckets; ++i) ZH_CHECK(hipEventDestroy(ev[i]));
  ZH_CHECK(hipGraphInstantiate(&P->exec, P->graph, nullptr, nullptr, 0));
  ZH_CHECK(hipStreamSynchronize(s));
  return P.release();
}

void batch_plan_execute(BatchPlan* P, hipStream_t s) { ZH_CHECK(hipGraphLaunch(P->exec, s)); }

void batch_plan_status(BatchPlan* P, int* status, hipStream_t s) {
  ZH_CHECK(hipMemcpyAsync(status, P->d_status, sizeof(int) * P->count, hipMemcpyDeviceToHost, s));
  ZH_CHECK(hipStreamSynchronize(s));
}

void batch_plan_variants(const BatchPlan* P, int* tg, int* r, int* counts) {
  for (int bk = 0; bk < kBuckets; ++bk) {
    tg[bk] = kVariants[P->variant[bk]].ty;
    r[bk] = kVariants[P->variant[bk]].ri;
    counts[bk] = P->bucket_count[bk];
  }
}

void batch_plan_destroy(BatchPlan* P) { delete P; }

}  // namespace zmlhip
