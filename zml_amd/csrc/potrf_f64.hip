// FP64 / FP32 Cholesky (zml lapack/potrf.zig:17-240, potrf2.zig:17-217), column-major view.
//
// zml's potrf is left-looking with NB = 64; on the GPU the same factor is
// computed right-looking (the per-element operation order of the lower,
// column-major case is the unblocked right-looking one either way, see the
// oracle's closed form), blocked on two levels: for each 512-column block
// column, in 128-column steps
//   factor the diagonal block in one workgroup (registers, separately rounded
//   multiply/subtract, l_ij = a_ij * fl(1/l_jj) as zml's right-side trsm
//   does, correctly rounded sqrt),
//   TRSM the rows below (lower) / columns right of it (upper),
//   update the rest of the block column only;
// then SYRK the trailing triangle with K = 512 on the MFMA GEMM, the next
// block column first so that its factorization overlaps the rest.
// Row-major lower is column-major upper of the same memory (and vice versa),
// which is how row-major calls are mapped.
//
// info (device int, zero on entry) receives the first non-positive or NaN
// pivot (1-based) as zml returns it (potrf2.zig:37-46, potrf.zig:100-103).
// Columns at and after a failing pivot are left unspecified.
#include "zmlhip_internal.hpp"

#include <algorithm>

namespace zmlhip {
namespace {

constexpr int DB = 128;   // diagonal block of the driver

// Cholesky of an nb x nb block (nb <= DB) by one workgroup, register resident.
// lower: A = L L^T on the lower triangle; else A = U^T U on the upper one.
// A 16 x 16 thread grid holds the elements (i + 16 ii, c + 16 cc), ii >= cc, of
// the lower-orientation block. The block advances in chunks of 16 columns:
//   the chunk goes to LDS;
//   up to three waves factor it, one row per lane with its 16 values in
//   registers: lanes 0..15 of every wave hold the chunk's own 16 rows (the same
//   values in each wave, so no step needs a barrier), lanes 16..63 the rows
//   below. A step takes l_jj = sqrt(a_jj) and r = fl(1 / l_jj) from lane j,
//   l_ij = fl(a_ij r), and the other chunk rows' multipliers by readlane;
//   every thread applies the chunk's 16 columns to its later columns, from LDS.
// Each element receives its separately rounded updates a - l_ik l_ck in the order
// of k, as in the unblocked right-looking algorithm: the same bits as one column
// at a time over the whole block, which spent its time on masks and on one
// barrier per column (158 us per 128 x 128 block alone on MI355X, against 42 us; 97 to
// 133 us inside a factorization, beside the trailing update's workgroups). Bound by
// the step chain of one wave (310 cycles a column: square root, reciprocal, up to
// 15 readlane pairs with their multiplies and subtracts), then by the later
// columns' updates (230 cycles a column on average).
__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// l = sqrt(d), r = fl(1 / l), both correctly rounded. FP64: Goldschmidt's iteration
// from the hardware's reciprocal square root with two residual corrections of
// the root, whose half reciprocal then starts Newton's iteration for 1 / l (two
// corrections, Markstein): 100 cycles against 175 for sqrt and a division. Both
// of those outside [2^-512, 2^512); d must be the same in every lane. False, with
// l = r = 1, where d is not positive.
__device__ __forceinline__ bool sqrt_and_inv(double d, double& l, double& r) {
  const uint32_t hi = (uint32_t)((uint64_t)__double_as_longlong(d) >> 32);
  constexpr uint32_t kLow = (1023u - 512u) << 20, kSpan = 1024u << 20;
  if (__builtin_expect(hi - kLow < kSpan, 1)) {
    const double y = __builtin_amdgcn_rsq(d);
    double g = d * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, d), h, g);
    g = fma(fma(-g, g, d), h, g);
    double z = h + h;
    z = fma(fma(-g, z, 1.0), z, z);
    z = fma(fma(-g, z, 1.0), z, z);
    // a root with every mantissa bit set is the one divisor whose reciprocal the
    // corrections leave one bit low (2^-k where 2^-k (1 + 2^-52) is nearest)
    constexpr uint64_t kMant = 0xfffffffffffffull;
    const uint64_t ones = ((uint64_t)__double_as_longlong(g) & kMant) == kMant ? 1u : 0u;
    l = g;
    r = __longlong_as_double((long long)((uint64_t)__double_as_longlong(z) | ones));
    return true;
  }
  const bool ok = d > 0.0;
  l = ok ? sqrt(d) : 1.0;
  r = 1.0 / l;
  return ok;
}
__device__ __forceinline__ bool sqrt_and_inv(float d, float& l, float& r) {
  const bool ok = d > 0.0f;
  l = ok ? sqrtf(d) : 1.0f;
  r = 1.0f / l;
  return ok;
}

constexpr int CW = 16;         // columns of a chunk
constexpr int PLD = CW + 1;    // LDS row stride of a chunk

// Step J of a chunk on one row per lane (p: its 16 values).
template <typename T, int J>
__device__ __forceinline__ void chunk_steps(T (&p)[CW], int lane, int j0, int& fail) {
#pragma clang fp contract(off)
  if constexpr (J < CW) {
    T ljj, rj;
    if (!sqrt_and_inv(lane_value(p[J], J), ljj, rj) && !fail) fail = j0 + J + 1;
    const T l = p[J] * rj;
    p[J] = lane == J ? ljj : l;
    // four columns at a time: their multipliers, the products, the subtractions
    // (one after the other each column would wait for its own chain)
#pragma unroll
    for (int c = J + 1; c < CW; c += 4) {
      T m[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) m[e] = c + e < CW ? lane_value(l, c + e < CW ? c + e : 0) : T(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < CW) m[e] = l * m[e];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < CW) p[c + e] = p[c + e] - m[e];
    }
    chunk_steps<T, J + 1>(p, lane, j0, fail);
  }
}

// Chunk CH of the thread's elements to LDS; the factored chunk back, and its 16
// columns, in order, into the thread's later columns.
template <typename T, int CH>
__device__ __forceinline__ void chunk_out(const T (&v)[8][8], T* P, int ri, int ci) {
#pragma unroll
  for (int ii = CH; ii < 8; ++ii) P[(ri + 16 * ii) * PLD + ci] = v[ii][CH];
}
template <typename T, int CH>
__device__ __forceinline__ void chunk_apply(T (&v)[8][8], const T* R, int ri, int ci) {
#pragma clang fp contract(off)
#pragma unroll
  for (int ii = CH; ii < 8; ++ii) v[ii][CH] = R[(ri + 16 * ii) * PLD + ci];
  if constexpr (CH < 7) {
#pragma unroll 4
    for (int k = 0; k < CW; ++k) {
      T lr[8], lc[8];
#pragma unroll
      for (int ii = CH + 1; ii < 8; ++ii) {
        lr[ii] = R[(ri + 16 * ii) * PLD + k];
        lc[ii] = R[(ci + 16 * ii) * PLD + k];
      }
#pragma unroll
      for (int ii = CH + 1; ii < 8; ++ii)
#pragma unroll
        for (int cc = CH + 1; cc <= ii; ++cc) v[ii][cc] = v[ii][cc] - lr[ii] * lc[cc];
    }
  }
}
template <typename T>
__device__ __forceinline__ void chunk_out(int ch, const T (&v)[8][8], T* P, int ri, int ci) {
  switch (ch) {
    case 0: chunk_out<T, 0>(v, P, ri, ci); break;
    case 1: chunk_out<T, 1>(v, P, ri, ci); break;
    case 2: chunk_out<T, 2>(v, P, ri, ci); break;
    case 3: chunk_out<T, 3>(v, P, ri, ci); break;
    case 4: chunk_out<T, 4>(v, P, ri, ci); break;
    case 5: chunk_out<T, 5>(v, P, ri, ci); break;
    case 6: chunk_out<T, 6>(v, P, ri, ci); break;
    default: chunk_out<T, 7>(v, P, ri, ci); break;
  }
}
template <typename T>
__device__ __forceinline__ void chunk_apply(int ch, T (&v)[8][8], const T* R, int ri, int ci) {
  switch (ch) {
    case 0: chunk_apply<T, 0>(v, R, ri, ci); break;
    case 1: chunk_apply<T, 1>(v, R, ri, ci); break;
    case 2: chunk_apply<T, 2>(v, R, ri, ci); break;
    case 3: chunk_apply<T, 3>(v, R, ri, ci); break;
    case 4: chunk_apply<T, 4>(v, R, ri, ci); break;
    case 5: chunk_apply<T, 5>(v, R, ri, ci); break;
    case 6: chunk_apply<T, 6>(v, R, ri, ci); break;
    default: chunk_apply<T, 7>(v, R, ri, ci); break;
  }
}

template <typename T>
__global__ void __launch_bounds__(256, 1)
potrf_diag_kernel(int nb, T* __restrict__ a, int64_t lda, int lower, int* __restrict__ info,
                  int64_t info_base) {
  __shared__ T P[DB * PLD], R[DB * PLD];   // the chunk before and after its 16 steps
  __shared__ int s_fail;
  if (*info != 0) return;   // an earlier block already failed
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  // memory's contiguous direction runs along the low 4 bits of the thread index
  const int ri = lower ? t & 15 : t >> 4, ci = lower ? t >> 4 : t & 15;
  if (t == 0) s_fail = 0;
  T v[8][8];
  // every address of the nb x nb block is readable: all 36 loads are issued
  // unconditionally (clamped indices; the empty asm keeps the compiler from
  // sinking each one under its mask and waiting for it), then masked; rows from nb
  // on are those of the identity
#pragma unroll
  for (int ii = 0; ii < 8; ++ii)
#pragma unroll
    for (int cc = 0; cc <= ii; ++cc) {
      const int r = ri + 16 * ii, c = ci + 16 * cc;
      const int64_t rc = r < nb ? r : nb - 1, cl = c < nb ? c : nb - 1;
      v[ii][cc] = a[lower ? rc + cl * lda : cl + rc * lda];
    }
#pragma unroll
  for (int ii = 0; ii < 8; ++ii)
#pragma unroll
    for (int cc = 0; cc <= ii; ++cc) {
      asm volatile("" : "+v"(v[ii][cc]));
      const int r = ri + 16 * ii, c = ci + 16 * cc;
      if (!(r < nb && c <= r)) v[ii][cc] = r == c ? T(1) : T(0);
    }

  const int nch = (nb + CW - 1) / CW;
  int done = nb;   // columns that were completed
  for (int ch = 0; ch < nch; ++ch) {
    const int j0 = CW * ch;
    chunk_out<T>(ch, v, P, ri, ci);
    __syncthreads();
    // the chunk's 16 columns: rows j0 .. j0 + 15 in every wave's lanes 0..15
    const int row = lane < CW ? j0 + lane : j0 + CW + (64 - CW) * w + lane - CW;
    if (w == 0 || j0 + CW + (64 - CW) * w < nb) {
      T p[CW];
      const int rl = row < DB ? row : DB - 1;
#pragma unroll
      for (int c = 0; c < CW; ++c) p[c] = P[rl * PLD + c];
      int fail = 0;
      chunk_steps<T, 0>(p, lane, j0, fail);
      if (lane >= CW ? row < DB : w == 0) {
#pragma unroll
        for (int c = 0; c < CW; ++c) R[rl * PLD + c] = p[c];
      }
      if (fail && w == 0 && lane == 0) s_fail = fail;
    }
    __syncthreads();
    chunk_apply<T>(ch, v, R, ri, ci);
    if (s_fail) {   // (s_fail only changes between this and the next barrier's far side)
      done = s_fail - 1;
      break;
    }
  }
#pragma unroll
  for (int ii = 0; ii < 8; ++ii)
#pragma unroll
    for (int cc = 0; cc <= ii; ++cc) {
      const int r = ri + 16 * ii, c = ci + 16 * cc;
      if (r < nb && c <= r && c < done) a[lower ? r + (int64_t)c * lda : c + (int64_t)r * lda] = v[ii][cc];
    }
  if (done < nb && t == 0) *info = (int)(info_base + done + 1);
}

}  // namespace

template <typename T>
void potrf_cm(int uplo, int64_t n, T* a, int64_t lda, int* info, hipStream_t s) {
  if (n <= 0) return;
  const bool lower = uplo == kLower;
  constexpr int64_t OB = 512;   // block column of the trailing updates (their K)
  auto at = [&](int64_t i, int64_t j) { return a + i + j * lda; };
  // factor block column [j0, j0 + jb) in DB-wide steps whose updates stay inside it
  auto factor_block = [&](int64_t j0, int64_t jb, hipStream_t st) {
    for (int64_t k0 = j0; k0 < j0 + jb; k0 += DB) {
      const int64_t kb = std::min<int64_t>(DB, j0 + jb - k0);
      T* d = at(k0, k0);
      hipLaunchKernelGGL(potrf_diag_kernel<T>, dim3(1), dim3(256), 0, st, (int)kb, d, lda, lower ? 1 : 0, info, k0);
      ZH_LAUNCH_CHECK();
      const int64_t r = n - k0 - kb;           // rows below (lower) / columns right (upper)
      if (r <= 0) break;
      const int64_t w = j0 + jb - (k0 + kb);   // columns of the block column still to update
      if (lower) {
        // A21 <- A21 L11^-T ; the block column's part of A22 <- A22 - A21 A21^T
        T* a21 = at(k0 + kb, k0);
        trsm_cm<T>(kRight, kLower, kTrans, kNonUnit, r, kb, T(1), d, lda, a21, lda, st);
        if (w > 0)
          gemm_cm<T>(kNoTrans, kTrans, r, w, kb, T(-1), a21, lda, a21, lda, T(1), at(k0 + kb, k0 + kb), lda, st,
                     kLower);
      } else {
        // A12 <- U11^-T A12 ; the block row's part of A22 <- A22 - A12^T A12
        T* a12 = at(k0, k0 + kb);
        trsm_cm<T>(kLeft, kUpper, kTrans, kNonUnit, kb, r, T(1), d, lda, a12, lda, st);
        if (w > 0)
          gemm_cm<T>(kTrans, kNoTrans, w, r, kb, T(-1), a12, lda, a12, lda, T(1), at(k0 + kb, k0 + kb), lda, st,
                     kUpper);
      }
    }
  };
  if (n <= OB) {
    factor_block(0, n, s);
    return;
  }
  // Look-ahead of depth one: after block column j0 is factored, the caller's
  // stream first updates the next block column and hands it to a panel stream,
  // then applies the rest of the trailing update while the panel stream
  // factors the next block column. Every update of a region stays ordered on
  // the caller's stream; the panel stream touches only its own block column.
  const hipStream_t sp = aux_stream(0);
  const hipEvent_t ev_in = aux_event(0), ev_panel = aux_event(1), ev_next = aux_event(2);
  ZH_CHECK(hipEventRecord(ev_in, s));
  ZH_CHECK(hipStreamWaitEvent(sp, ev_in, 0));
  factor_block(0, std::min<int64_t>(OB, n), sp);
  ZH_CHECK(hipEventRecord(ev_panel, sp));
  for (int64_t j0 = 0; j0 < n; j0 += OB) {
    const int64_t jb = std::min<int64_t>(OB, n - j0);
    const int64_t r = n - j0 - jb;
    if (r <= 0) break;
    const int64_t jb2 = std::min<int64_t>(OB, r), r2 = r - jb2;
    const int64_t c1 = j0 + jb, c2 = c1 + jb2;
    ZH_CHECK(hipStreamWaitEvent(s, ev_panel, 0));
    if (lower) {
      const T* l21 = at(c1, j0);
      gemm_cm<T>(kNoTrans, kTrans, r, jb2, jb, T(-1), l21, lda, l21, lda, T(1), at(c1, c1), lda, s, kLower);
      ZH_CHECK(hipEventRecord(ev_next, s));
      if (r2 > 0) syrk_cm<T>(kLower, kNoTrans, r2, jb, T(-1), at(c2, j0), lda, T(1), at(c2, c2), lda, s);
    } else {
      const T* u12 = at(j0, c1);
      gemm_cm<T>(kTrans, kNoTrans, jb2, r, jb, T(-1), u12, lda, u12, lda, T(1), at(c1, c1), lda, s, kUpper);
      ZH_CHECK(hipEventRecord(ev_next, s));
      if (r2 > 0) syrk_cm<T>(kUpper, kTrans, r2, jb, T(-1), at(j0, c2), lda, T(1), at(c2, c2), lda, s);
    }
    ZH_CHECK(hipStreamWaitEvent(sp, ev_next, 0));
    factor_block(c1, jb2, sp);
    ZH_CHECK(hipEventRecord(ev_panel, sp));
  }
  ZH_CHECK(hipStreamWaitEvent(s, ev_panel, 0));
}
template void potrf_cm<double>(int, int64_t, double*, int64_t, int*, hipStream_t);
template void potrf_cm<float>(int, int64_t, float*, int64_t, int*, hipStream_t);

void potrf_f64_cm(int uplo, int64_t n, double* a, int64_t lda, int* info, hipStream_t s) {
  potrf_cm<double>(uplo, n, a, lda, info, s);
}

}  // namespace zmlhip
