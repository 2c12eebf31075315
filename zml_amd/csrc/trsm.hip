// Triangular solves with several right-hand sides (TRSM), FP64 and FP32,
// column-major view (zml blas/trsm.zig:18-735).
//
// Every form is reduced to one: M x = b for many vectors x, M lower triangular
// and solved from its first row down. Element (r, c) of M is at a[r rs + c cs]
// and element r of vector v at b[r bs + v vs]; a transposed operand swaps rs and
// cs, the right-hand side forms take M = op(A)^T with the rows of B as
// vectors, and the upper (backward) forms reverse the index, so that the
// strides are negative. The arithmetic choices follow zml's trsm.zig where they
// are visible in a result: the left-side branches divide by the diagonal
// (trsm.zig:137-142,221-229,298-305,364-371), the right-side branches multiply
// by its reciprocal (trsm.zig:458-486,538-566,575-600,653-678).
//
// M is taken in blocks of QB = 512 rows: trsm_strip_kernel solves the block's
// triangle, and the rows below it are updated with K = 512 (the MFMA GEMM, or
// trsm_update_kernel for at most 64 vectors, whose GEMM tile would be mostly
// padding). A 32-row blocking with one launch for each diagonal block and one
// GEMM of K = 32 behind it, which this replaces, was bound by its 2 q / 32
// launches and by passing the whole right-hand side through memory at each of
// them: 4096 rows x 1024 vectors took 4.87 ms, against 0.99 ms now (one MI355X).
#include "zmlhip_internal.hpp"

#include <algorithm>
#include <cmath>

namespace zmlhip {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mma;
template <> struct Mma<double> {
  typedef d4 acc;
  static __device__ __forceinline__ acc step(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};
template <> struct Mma<float> {
  typedef f4 acc;
  static __device__ __forceinline__ acc step(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

constexpr int QB = 512;        // rows of one strip launch
constexpr int DB = 64;         // rows of one diagonal block inside it
constexpr int NV = 16;         // vectors per workgroup (one MFMA tile)
constexpr int XLD = NV + 1;    // LDS row stride of the solved rows
constexpr int DLD = DB + 1;    // LDS column stride of the diagonal block
constexpr int MODE_UNIT = 0, MODE_DIV = 1, MODE_MUL = 2;

// Lane N of each row of 16 lanes to the whole row.
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x150 + N, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(u >> 32), 0x150 + N, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}

// x / d from d's reciprocal with one residual correction (Markstein's scheme):
// the correctly rounded quotient while nothing leaves the normal range.
__device__ __forceinline__ double quot(double x, double d, double rinv) {
  const double q = x * rinv;
  return fma(fma(-q, d, x), rinv, q);
}
__device__ __forceinline__ float quot(float x, float d, float) { return x / d; }

template <typename T, int MODE>
__device__ __forceinline__ T scaled(T x, T dg, T rinv) {
  if constexpr (MODE == MODE_DIV) return quot(x, dg, rinv);
  if constexpr (MODE == MODE_MUL) return x * rinv;
  return x;
}

// Steps of the 16 rows of group II: 16 lanes hold one vector (lane r16: rows
// r16 + 16 ii, x[ii]). dd[kk] is the block's strictly lower element
// (r16 + 16 II, 16 II + kk), zero elsewhere, so that a step needs no lane mask (a
// row keeps its value from its own step on); D[k DLD + r] is column k of the 64 x 64
// block. One separately rounded multiply and subtract per element, k ascending,
// as zml's substitution loops. The later groups' elements are read two steps ahead
// (n0, n1; the scheduling barriers keep the reads there: left alone they move
// next to their use, and every step waits for LDS).
template <typename T, int II>
__device__ __forceinline__ void read_col(T (&n)[3], const T* D, int k, int r16) {
#pragma unroll
  for (int i2 = II + 1; i2 < 4; ++i2) n[i2 - 1] = D[k * DLD + r16 + 16 * i2];
}
template <typename T, int MODE, int II, int KK>
__device__ __forceinline__ void group_steps(T (&x)[4], const T (&dd)[16], T dg, T rinv, const T* D, int r16,
                                            T (&n0)[3], T (&n1)[3]) {
#pragma clang fp contract(off)
  if constexpr (KK < 16) {
    T n2[3];
    if constexpr (KK < 14) read_col<T, II>(n2, D, 16 * II + KK + 2, r16);
    const T xk = row_bcast<KK>(scaled<T, MODE>(x[II], dg, rinv));
    x[II] = x[II] - xk * dd[KK];
#pragma unroll
    for (int i2 = II + 1; i2 < 4; ++i2) x[i2] = x[i2] - xk * n0[i2 - 1];
    __builtin_amdgcn_sched_barrier(0);
    group_steps<T, MODE, II, KK + 1>(x, dd, dg, rinv, D, r16, n1, n2);
  }
}
template <typename T, int MODE, int II>
__device__ __forceinline__ void strip_group(T (&x)[4], T (&dd)[16], const T (&dg)[4], const T (&rinv)[4], const T* D,
                                            int r16) {
  T n0[3], n1[3];
  read_col<T, II>(n0, D, 16 * II, r16);
  read_col<T, II>(n1, D, 16 * II + 1, r16);
  __builtin_amdgcn_sched_barrier(0);
  group_steps<T, MODE, II, 0>(x, dd, dg[II], rinv[II], D, r16, n0, n1);
  x[II] = scaled<T, MODE>(x[II], dg[II], rinv[II]);
  if constexpr (II < 3) {
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) dd[kk] = D[(16 * II + 16 + kk) * DLD + 16 * II + 16 + r16];
  }
}

// Solves M x = b for q <= QB rows and the 16 vectors of each workgroup. Row
// block i of 64 in turn: the four waves form b_i - sum_{j < i} M_ij x_j on MFMA
// (one 16 x 16 tile each, the solved rows in LDS, M's values straight from memory
// one 64-column batch ahead), then solve the 64 x 64 triangle by substitution,
// 16 lanes per vector, each wave four vectors.
// Bound by the serial chain of the substitution (64 to 90 cycles a row at 2.4 GHz:
// the quotient, the row broadcast, a multiply and a subtract), then by the MFMA
// sums (1,800 cycles per 64 x 64 block): 64-68 us for 512 rows, 11.6 us for 64 with
// the launch. With lane masks and LDS reads left where the compiler puts them a row
// took 145 to 200 cycles. Sixteen vectors per workgroup, since that is one MFMA tile and
// right-hand sides are usually few: more per workgroup would leave CUs idle.
template <typename T, int MODE>
__global__ void __launch_bounds__(256, 2)
trsm_strip_kernel(int q, const T* __restrict__ a, int64_t rs, int64_t cs, T* __restrict__ b, int64_t bs, int64_t vs,
                  int64_t nvec) {
#pragma clang fp contract(off)
  typedef typename Mma<T>::acc acc_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  T* const D = reinterpret_cast<T*>(lds_raw);
  T* const X = D + DB * DLD;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t v0 = (int64_t)blockIdx.x * NV;
  const int nv = (int)(nvec - v0 < NV ? nvec - v0 : NV);
  const int nb = (q + DB - 1) / DB;
  const bool rfast = rs == 1 || rs == -1;
  b += v0 * vs;

  // the diagonal block's values, 16 per thread, along its contiguous direction,
  // and the diagonal itself in the substitution's layout (rows lr + 16 ii)
  const int dr = rfast ? lane : w, dc = rfast ? w : lane;          // element 0 of this thread
  const int64_t dstep = 4 * (rfast ? cs : rs);                     // to the next one
  T dv[16], dgn[4];
  auto load_diag = [&](int i) {
    const int64_t i0 = (int64_t)i * DB;
    const T* p = a + i0 * (rs + cs);
    if (i0 + DB <= q) {
      const T* pe = p + dr * rs + dc * cs;
#pragma unroll
      for (int e = 0; e < 16; ++e) dv[e] = pe[e * dstep];
    } else {   // the last, partial block: clamped into the matrix
      const int last = (int)(q - 1 - i0);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int sl = w + 4 * e;
        dv[e] = p[min(rfast ? lane : sl, last) * rs + min(rfast ? sl : lane, last) * cs];
      }
    }
    if (MODE != MODE_UNIT) {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int r = lr + 16 * ii;
        const T v = p[min(r, (int)(q - 1 - i0)) * (rs + cs)];
        dgn[ii] = i0 + r < q ? v : T(1);
      }
    }
  };
  // the strict triangle only; rows from q on are those of the identity
  auto store_diag = [&](int i) {
    const int left = q - i * DB;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int sl = w + 4 * e, r = rfast ? lane : sl, c = rfast ? sl : lane;
      D[c * DLD + r] = c < r && r < left ? dv[e] : T(0);
    }
  };
  // This wave's 16 rows of block row i, 64 columns (block j) at a time, k = 8 s +
  // 2 lk + e: two batches, each refilled (batch pi, pj) while it is multiplied
  T a0[16], a1[16];
  int pi = 1, pj = 0;
  const T* pa = a;      // source of the next batch
  auto next_batch = [&]() {
    const int64_t row = min(pi * DB + 16 * w + lr, q - 1);
    pa = a + row * rs + ((int64_t)pj * DB + 2 * lk) * cs;
    const bool more = pi < nb;
    if (more && ++pj == pi) { ++pi; pj = 0; }
    return more;
  };
  auto first_load = [&](T (&v)[16]) {
    if (!next_batch()) return;
#pragma unroll
    for (int s = 0; s < 16; ++s) v[s] = pa[(8 * (s >> 1) + (s & 1)) * cs];
  };
  // acc += batch v times the solved rows of block j; v is reloaded behind its use
  // (past the last batch: from a row inside the matrix, unused)
  auto multiply = [&](T (&v)[16], int j, typename Mma<T>::acc& acc) {
    int64_t step = cs;
    if (!next_batch()) { pa = a; step = 0; }
    const T* xp = X + (j * DB + 2 * lk) * XLD + lr;
    T xr[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) xr[s] = xp[(8 * (s >> 1) + (s & 1)) * XLD];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      acc = Mma<T>::step(v[s], xr[s], acc);
      v[s] = pa[(8 * (s >> 1) + (s & 1)) * step];
    }
  };
  // this wave's 16 x 16 tile of b_i in the accumulator's layout
  T bv[4];
  const int64_t vcl = min(lr, nv - 1) * vs;
  auto load_rhs = [&](int i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = min(i * DB + 16 * w + Mma<T>::row(lk, r), q - 1);
      bv[r] = b[row * bs + vcl];
    }
  };

  load_diag(0);
  load_rhs(0);
  first_load(a0);
  first_load(a1);
  bool odd = false;   // which of a0, a1 holds the next batch
  for (int i = 0; i < nb; ++i) {
    acc_t acc;   // the negated residual: M x - b
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = -bv[r];
    for (int j = 0; j < i; ++j) {
      if (odd) multiply(a1, j, acc);
      else multiply(a0, j, acc);
      odd = !odd;
    }
    T* const xi = X + i * DB * XLD;
#pragma unroll
    for (int r = 0; r < 4; ++r) xi[(16 * w + Mma<T>::row(lk, r)) * XLD + lr] = -acc[r];
    store_diag(i);
    T dg[4], rinv[4];
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      dg[ii] = MODE == MODE_UNIT ? T(1) : dgn[ii];
      rinv[ii] = MODE == MODE_UNIT ? T(1) : T(1) / dg[ii];
    }
    __syncthreads();
    if (i + 1 < nb) {   // requested now, used after the substitution
      load_diag(i + 1);
      load_rhs(i + 1);
    }
    {
      // 16 lanes per vector: vector 4 w + lk, rows lr + 16 ii
      T x[4], dd[16];
      T* const xv = xi + 4 * w + lk;
#pragma unroll
      for (int kk = 0; kk < 16; ++kk) dd[kk] = D[kk * DLD + lr];
      bool fine = true;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        x[ii] = xv[(lr + 16 * ii) * XLD];
        if (MODE == MODE_DIV && sizeof(T) == 8) {
          const T ad = fabs(dg[ii]);
          fine = fine && ad > T(0x1p-400) && ad < T(0x1p+400);
        }
      }
      // (groups past the last row are the identity's: 16 rows 18.1 us with their steps,
      // 17.0 without)
      const int left = q - i * DB;
      strip_group<T, MODE, 0>(x, dd, dg, rinv, D, lr);
      if (__builtin_expect(left > 16, 1)) strip_group<T, MODE, 1>(x, dd, dg, rinv, D, lr);
      if (__builtin_expect(left > 32, 1)) strip_group<T, MODE, 2>(x, dd, dg, rinv, D, lr);
      if (__builtin_expect(left > 48, 1)) strip_group<T, MODE, 3>(x, dd, dg, rinv, D, lr);
      // infinities and NaN (which the unmasked steps would carry to every row),
      // and for the quotients anything near the ends of the range
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const T ax = fabs(x[ii]);
        if (MODE == MODE_DIV && sizeof(T) == 8)
          fine = fine && (ax == T(0) || (ax > T(0x1p-500) && ax < T(0x1p+500)));
        else
          fine = fine && ax < T(INFINITY);
      }
      if (__builtin_expect(!__all(fine), 0)) {
        // the same steps from the start, masked and with exact quotients (the vectors of
        // this wave alone; 512 rows x 16 vectors 154 us against 75 us on the fast path, and
        // 1,030 us with each vector on one lane)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) x[ii] = xv[(lr + 16 * ii) * XLD];
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
#pragma unroll 1
          for (int kk = 0; kk < 16; ++kk) {
            const T* const dk = D + (16 * ii + kk) * DLD + lr;
            const T y = MODE == MODE_DIV ? x[ii] / dg[ii] : (MODE == MODE_MUL ? x[ii] * rinv[ii] : x[ii]);
            const T xk = __shfl(y, kk, 16);
            x[ii] = lr == kk ? xk : (lr > kk ? x[ii] - xk * dk[16 * ii] : x[ii]);
#pragma unroll
            for (int i2 = ii + 1; i2 < 4; ++i2) x[i2] = x[i2] - xk * dk[16 * i2];
          }
        }
      }
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) xv[(lr + 16 * ii) * XLD] = x[ii];
    }
    __syncthreads();
    // the solved rows to memory, along B's contiguous direction
    const int rows = min(DB, q - i * DB);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = vs == 1 ? (t >> 4) + 16 * e : t & 63, v = vs == 1 ? t & 15 : (t >> 6) + 4 * e;
      if (r < rows && v < nv) b[(int64_t)(i * DB + r) * bs + v * vs] = xi[r * XLD + v];
    }
  }
}

// Rows m below a solved block: c_r -= sum_k M_rk x_k for nv <= 16 NT vectors,
// K = the block's rows. A workgroup takes 64 rows (one 16-row tile per wave), M's
// values come straight from memory one batch of 64 columns ahead, the solved
// rows pass through LDS. Reads M's block once; below a few thousand rows it is bound
// by the latency of its eight batches (34 us at m = 1000).
template <typename T, int NT>
__global__ void __launch_bounds__(256)
trsm_update_kernel(int64_t m, int K, const T* __restrict__ a, int64_t rs, int64_t cs, const T* __restrict__ x,
                   T* __restrict__ c, int64_t bs, int64_t vs, int nv) {
  typedef typename Mma<T>::acc acc_t;
  constexpr int KC = 64, W = NV * NT, PER = KC * W / 256;
  __shared__ T X[KC][W + 1];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t r0 = (int64_t)blockIdx.x * 64 + 16 * w;
  const int64_t row = min(r0 + lr, m - 1);
  const T* const ap = a + row * rs;
  T av[16], an[16], xn[PER];
  auto load = [&](int k0) {
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int k = k0 + 8 * (s >> 1) + 2 * lk + (s & 1);
      const T v = ap[(int64_t)min(k, K - 1) * cs];
      an[s] = k < K ? v : T(0);
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int f = t + 256 * e;
      const int kk = vs == 1 ? f / W : f % KC, v = vs == 1 ? f % W : f / KC;
      const T y = x[(int64_t)min(k0 + kk, K - 1) * bs + (int64_t)min(v, nv - 1) * vs];
      xn[e] = k0 + kk < K ? y : T(0);
    }
  };
  acc_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t i = min(r0 + Mma<T>::row(lk, r), m - 1);
      acc[n][r] = c[i * bs + (int64_t)min(NV * n + lr, nv - 1) * vs];
    }
  load(0);
  for (int k0 = 0; k0 < K; k0 += KC) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int f = t + 256 * e;
      X[vs == 1 ? f / W : f % KC][vs == 1 ? f % W : f / KC] = xn[e];
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) av[s] = -an[s];
    __syncthreads();
    if (k0 + KC < K) load(k0 + KC);
#pragma unroll
    for (int s = 0; s < 16; ++s)
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[n] = Mma<T>::step(av[s], X[8 * (s >> 1) + 2 * lk + (s & 1)][NV * n + lr], acc[n]);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t i = r0 + Mma<T>::row(lk, r);
      if (i < m && NV * n + lr < nv) c[i * bs + (int64_t)(NV * n + lr) * vs] = acc[n][r];
    }
}

// At most FEW rows: one vector per thread, M in scalar registers. Bound by the launch
// and one round trip to memory: 13.2 us for 4 and 13.3 us for 8 rows, launch included,
// where the strip's block of 64 rows takes 17.1 and 16.7 us (2 to 1,000 vectors; 16
// rows 17.0 us on the strip, 64 rows 16.8).
constexpr int FEW = 8;
template <typename T>
__global__ void __launch_bounds__(64)
trsm_few_kernel(int q, int mode, const T* __restrict__ a, int64_t rs, int64_t cs, T* __restrict__ b, int64_t bs,
                int64_t vs, int64_t nvec) {
#pragma clang fp contract(off)
  const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (v >= nvec) return;
  b += v * vs;
  T m[FEW][FEW], x[FEW];   // rows from q on: row q - 1 again, not stored
#pragma unroll
  for (int r = 0; r < FEW; ++r) {
#pragma unroll
    for (int c = 0; c <= r; ++c) m[r][c] = a[min(r, q - 1) * rs + min(c, q - 1) * cs];
    x[r] = b[min(r, q - 1) * bs];
  }
#pragma unroll
  for (int k = 0; k < FEW; ++k) {
    if (k >= q) break;
    if (mode == MODE_DIV) x[k] = x[k] / m[k][k];
    else if (mode == MODE_MUL) x[k] = x[k] * (T(1) / m[k][k]);
    b[k * bs] = x[k];
#pragma unroll
    for (int i = k + 1; i < FEW; ++i) x[i] = x[i] - x[k] * m[i][k];
  }
}

template <typename T>
size_t strip_lds(int64_t q) {
  return sizeof(T) * ((size_t)DB * DLD + (size_t)((q + DB - 1) / DB * DB) * XLD);
}

template <typename T>
void strip(int mode, int q, const T* a, int64_t rs, int64_t cs, T* b, int64_t bs, int64_t vs, int64_t nvec,
           hipStream_t s) {
  const dim3 grid((unsigned)((nvec + NV - 1) / NV)), block(256);
  const size_t lds = strip_lds<T>(q);
  if (mode == MODE_UNIT)
    hipLaunchKernelGGL((trsm_strip_kernel<T, MODE_UNIT>), grid, block, lds, s, q, a, rs, cs, b, bs, vs, nvec);
  else if (mode == MODE_DIV)
    hipLaunchKernelGGL((trsm_strip_kernel<T, MODE_DIV>), grid, block, lds, s, q, a, rs, cs, b, bs, vs, nvec);
  else
    hipLaunchKernelGGL((trsm_strip_kernel<T, MODE_MUL>), grid, block, lds, s, q, a, rs, cs, b, bs, vs, nvec);
  ZH_LAUNCH_CHECK();
}

template <typename T>
void update_few(int64_t m, int K, const T* a, int64_t rs, int64_t cs, const T* x, T* c, int64_t bs, int64_t vs,
                int nv, hipStream_t s) {
  const dim3 grid((unsigned)((m + 63) / 64)), block(256);
  const int nt = (nv + NV - 1) / NV;
  if (nt == 1) hipLaunchKernelGGL((trsm_update_kernel<T, 1>), grid, block, 0, s, m, K, a, rs, cs, x, c, bs, vs, nv);
  else if (nt == 2) hipLaunchKernelGGL((trsm_update_kernel<T, 2>), grid, block, 0, s, m, K, a, rs, cs, x, c, bs, vs, nv);
  else hipLaunchKernelGGL((trsm_update_kernel<T, 4>), grid, block, 0, s, m, K, a, rs, cs, x, c, bs, vs, nv);
  ZH_LAUNCH_CHECK();
}

}  // namespace

template <typename T>
void trsm_cm(int side, int uplo, int transa, int diag, int64_t m, int64_t n, T alpha, const T* a,
             int64_t lda, T* b, int64_t ldb, hipStream_t s) {
  if (m <= 0 || n <= 0) return;
  if (alpha == T(0)) { scale_cm<T>(m, n, T(0), b, ldb, s, 0); return; }   // trsm.zig:99-113
  if (alpha != T(1)) scale_cm<T>(m, n, alpha, b, ldb, s, 0);
  const bool nt = is_notrans(transa), left = side == kLeft;
  const int mode = diag == kUnit ? MODE_UNIT : (left ? MODE_DIV : MODE_MUL);
  const int64_t q = left ? m : n, nvec = left ? n : m;
  // M = op(A) with the columns of B, or op(A)^T with its rows; lower: forward
  const bool fwd = left ? (uplo == kLower) == nt : (uplo == kUpper) == nt;
  int64_t rs = left == nt ? 1 : lda, cs = left == nt ? lda : 1;
  int64_t bs = left ? 1 : ldb;
  const int64_t vs = left ? ldb : 1;
  const T* a0 = a;
  T* b0 = b;
  if (!fwd) {
    a0 += (q - 1) * (rs + cs);
    b0 += (q - 1) * bs;
    rs = -rs; cs = -cs; bs = -bs;
  }
  if (q <= FEW) {
    hipLaunchKernelGGL(trsm_few_kernel<T>, dim3((unsigned)((nvec + 63) / 64)), dim3(64), 0, s, (int)q, mode, a0, rs, cs,
                       b0, bs, vs, nvec);
    ZH_LAUNCH_CHECK();
    return;
  }
  for (int64_t i0 = 0; i0 < q; i0 += QB) {
    const int64_t kb = std::min<int64_t>(QB, q - i0), i1 = i0 + kb, rest = q - i1;
    strip<T>(mode, (int)kb, a0 + i0 * (rs + cs), rs, cs, b0 + i0 * bs, bs, vs, nvec, s);
    if (rest <= 0) break;
    if (nvec <= 4 * NV) {
      update_few<T>(rest, (int)kb, a0 + i1 * rs + i0 * cs, rs, cs, b0 + i0 * bs, b0 + i1 * bs, bs, vs, (int)nvec, s);
      continue;
    }
    const int64_t o0 = fwd ? i0 : q - i1, r0 = fwd ? i1 : 0;   // first row of the block, of the rest
    if (left) {
      const T* a21 = nt ? a + r0 + o0 * lda : a + o0 + r0 * lda;
      gemm_cm<T>(nt ? kNoTrans : kTrans, kNoTrans, rest, n, kb, T(-1), a21, lda, b + o0, ldb, T(1), b + r0, ldb, s, 0);
    } else {
      const T* a12 = nt ? a + o0 + r0 * lda : a + r0 + o0 * lda;
      gemm_cm<T>(kNoTrans, nt ? kNoTrans : kTrans, m, rest, kb, T(-1), b + o0 * ldb, ldb, a12, lda, T(1),
                 b + r0 * ldb, ldb, s, 0);
    }
  }
}
template void trsm_cm<double>(int, int, int, int, int64_t, int64_t, double, const double*, int64_t, double*,
                              int64_t, hipStream_t);
template void trsm_cm<float>(int, int, int, int, int64_t, int64_t, float, const float*, int64_t, float*,
                             int64_t, hipStream_t);

void trsm_f64_cm(int side, int uplo, int transa, int diag, int64_t m, int64_t n, double alpha,
                 const double* a, int64_t lda, double* b, int64_t ldb, hipStream_t s) {
  trsm_cm<double>(side, uplo, transa, diag, m, n, alpha, a, lda, b, ldb, s);
}

}  // namespace zmlhip
