// FP64 / FP32 GEMM on CDNA4 matrix cores (v_mfma_f64_16x16x4_f64 and
// v_mfma_f32_16x16x4_f32), column-major view.
//
//   C = alpha * op(A) * op(B) + beta * C        (reference blas/gemm.zig:68-1033)
//
// Row-major calls are mapped here by swapping the operands and m/n, exactly
// as zml does (gemm.zig:48-65). Only the arithmetic differs from zml: the
// matrix cores accumulate with fused multiply-adds, so results agree with
// zml's separately rounded loop to within the usual gamma_k |A||B| bound
// (bitwise on integer-valued data such as the reference's golden vectors).
//
// Two kernels, with the same order of operations for every element of C (the same
// bits), chosen in gemm_cm:
//  - gemm_dma_kernel (whole k-slabs, 16-byte aligned operand columns): 128 x 128
//    tiles whose operand slabs go from global memory to LDS by the load unit; 71
//    TF/s FP64, 122 TF/s FP32 at 4096^3 on MI355X;
//  - gemm_small_kernel (every shape, FP64 and FP32): 64 x 64 tiles staged through
//    registers, four workgroups per CU, with k cut into parts that are summed on their
//    own, one workgroup each, where even these are few.
// A 256-thread workgroup's four waves each own a quarter of the tile. K advances in
// slabs of 16 through double-buffered LDS. The MFMA is issued as C^T = op(B)^T
// op(A)^T so that the 16 lanes of an output group hold 16 consecutive rows of one
// column of C: stores and beta-loads are 128-byte contiguous in column-major
// memory. The two element types differ only in the MFMA and in which output row a
// lane's accumulator r holds (FP64: lane / 16 + 4 r; FP32: 4 (lane / 16) + r).
// (A 128 x 128 tile staged through registers, the former kernel for everything
// the load unit does not take, was never faster than the 64 x 64 one: 59.0 against
// 58.3 TF/s at 4096^3 odd FP64, 99.6 against 101.6 FP32, and 13 against 28 TF/s
// at 1000^3.)
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "zmlhip_internal.hpp"
#include "tiles.hpp"

namespace zmlhip {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// The MFMA of each element type and its accumulator layout.
template <typename T> struct Mfma;
template <> struct Mfma<double> {
  typedef d4 acc;
  static __device__ __forceinline__ acc step(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // column (within the 16 x 16 output tile) of accumulator r of a lane group lk
  static __device__ __forceinline__ int col(int lk, int r) { return lk + 4 * r; }
};
template <> struct Mfma<float> {
  typedef f4 acc;
  static __device__ __forceinline__ acc step(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int col(int lk, int r) { return 4 * lk + r; }
};

constexpr int BM = 128, BN = 128, BK = 16, PAD = 2;
constexpr int LDA_S = BM + PAD;
constexpr int NT = 256;

// Maps the linear workgroup id to a (tile_m, tile_n) pair: consecutive ids
// land on different XCDs (dispatch is round-robin over 8 XCDs), so the ids
// are first regrouped so each XCD gets a contiguous range of tiles, and the
// range is walked in groups of 8 tile-rows to share operand panels in L2.
__device__ __forceinline__ void tile_coords(int64_t bid, int64_t ntm, int64_t ntn, int64_t& tm,
                                            int64_t& tn) {
  const int64_t nt = ntm * ntn;
  // XCD x receives the ids bid = x, x + 8, ...: give it the contiguous range
  // [x * q + min(x, r), ...) of tiles, q = nt / 8, r = nt % 8
  const int64_t x = bid & 7, q = nt >> 3, r8 = nt & 7;
  const int64_t pid = x * q + (x < r8 ? x : r8) + (bid >> 3);
  constexpr int64_t G = 8;
  const int64_t per_group = G * ntn;
  const int64_t group = pid / per_group;
  const int64_t first_m = group * G;
  const int64_t gm = (ntm - first_m) < G ? (ntm - first_m) : G;
  const int64_t r = pid - group * per_group;
  tm = first_m + r % gm;
  tn = r / gm;
}

// ---- 64 x 64 tiles, staged through registers
//
// Four waves of 32 x 32, a k-slab of 16 with clamped loads whose addresses advance
// by one addition (only the last, partial slab is masked), four workgroups per CU
// to cover the loads: bound by LDS and load latency where the CUs are full (58 TF/s
// FP64, 100 TF/s FP32 at 4096^3), by the number of tiles below about 2000^2.
// Update form C <- C +- op(A) op(B) (beta 1, alpha +-1): the accumulators start
// from C and B is staged negated for alpha -1, so the epilogue only stores.
// PARTS: k in parts of kper, each summed on its own and then added to the sum of the
// earlier ones. With part != nullptr gridDim.y workgroups take one part each and
// leave its sum in part + z m n (m x n, column-major) for splitk_sum_kernel; without,
// one workgroup goes through the parts of its tile itself: the same bits, for a call
// that has no memory for them.
// On MI355X, against 128 x 128 tiles: 1001 x 1500 x 777 143 -> 78 us, 1024^3 145 ->
// 67 us, 124 x 918 x 5130 (k split 17 ways) 838 -> 43 us.
constexpr int SM = 64, SLD = SM + 2;

// The last rounding steps of a product in parts whose sum is s, the same in both kernels.
template <typename T>
__device__ __forceinline__ T scaled_sum(T s, T alpha, T beta, T c) {
#pragma clang fp contract(off)
  const T v = alpha * s;
  return beta == T(0) ? v : (beta == T(1) ? c + v : fma(beta, c, v));
}

template <typename T, bool TA, bool TB, bool PARTS>
__global__ void __launch_bounds__(NT, PARTS ? 2 : 4)
gemm_small_kernel(int64_t m, int64_t n, int64_t k, T alpha, const T* __restrict__ A, int64_t lda,
                  const T* __restrict__ B, int64_t ldb, T beta, T* __restrict__ C, int64_t ldc, int tri,
                  int64_t tri_tiles, int64_t kper, T* __restrict__ part) {
  typedef typename Mfma<T>::acc acc_t;
  __shared__ T As[2][BK * SLD], Bs[2][BK * SLD];
  const int64_t ntm = (m + SM - 1) / SM, ntn = (n + SM - 1) / SM;
  int64_t tm, tn;
  if (tri_tiles > 0) tri_tile_coords(blockIdx.x, tri_tiles, ntm, ntn, tri, tm, tn);
  else tile_coords(blockIdx.x, ntm, ntn, tm, tn);
  const int64_t row0 = tm * SM, col0 = tn * SM;
  if (tri == kLower && row0 + SM - 1 < col0) return;
  if (tri == kUpper && col0 + SM - 1 < row0) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 15, lk = lane >> 4;
  const int64_t kb = PARTS ? blockIdx.y * kper : 0;
  int64_t ke = PARTS && kb + kper < k ? kb + kper : k;

  // element q of this thread: (i, l) = (t & 63, (t >> 6) + 4 q) where the operand is
  // contiguous along m / n, ((t >> 4) + 16 q, t & 15) where it is along k
  const T *pa[4], *pb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t ia = TA ? (t >> 4) + 16 * q : t & 63, la = TA ? t & 15 : (t >> 6) + 4 * q;
    const int64_t jb = TB ? t & 63 : (t >> 4) + 16 * q, lb = TB ? (t >> 6) + 4 * q : t & 15;
    const int64_t i = row0 + ia < m ? row0 + ia : m - 1, j = col0 + jb < n ? col0 + jb : n - 1;
    pa[q] = TA ? A + (kb + la) + i * lda : A + i + (kb + la) * lda;
    pb[q] = TB ? B + j + (kb + lb) * ldb : B + (kb + lb) + j * ldb;
  }
  const int64_t sa = TA ? BK : BK * lda, sb = TB ? BK * ldb : BK;   // to the next slab
  T ra[4], rb[4];
  auto load = [&](int64_t k0) __attribute__((always_inline)) {
    if (k0 + BK <= ke) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ra[q] = *pa[q];
        rb[q] = *pb[q];
        pa[q] += sa;
        pb[q] += sb;
      }
    } else {   // the partial slab: the last column again, masked in both operands
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t la = k0 + (TA ? t & 15 : (t >> 6) + 4 * q), lb = k0 + (TB ? (t >> 6) + 4 * q : t & 15);
        const int64_t ba = la < ke ? 0 : la - (ke - 1), bb = lb < ke ? 0 : lb - (ke - 1);
        const T va = *(pa[q] - (TA ? ba : ba * lda)), vb = *(pb[q] - (TB ? bb * ldb : bb));
        ra[q] = la < ke ? va : T(0);
        rb[q] = lb < ke ? vb : T(0);
      }
    }
  };
  const bool cinit = !PARTS && beta == T(1) && (alpha == T(1) || alpha == T(-1));
  const bool negb = cinit && alpha == T(-1);
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int ia = TA ? (t >> 4) + 16 * q : t & 63, la = TA ? t & 15 : (t >> 6) + 4 * q;
      const int jb = TB ? t & 63 : (t >> 4) + 16 * q, lb = TB ? (t >> 6) + 4 * q : t & 15;
      As[buf][la * SLD + ia] = ra[q];
      Bs[buf][lb * SLD + jb] = negb ? -rb[q] : rb[q];
    }
  };
  auto c_ok = [&](int64_t i, int64_t j) {
    return i < m && j < n && !(tri == kLower && i < j) && !(tri == kUpper && i > j);
  };
  acc_t acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[x][y][r] = T(0);
        if (cinit) {
          const int64_t i = row0 + wm * 32 + 16 * x + lr, j = col0 + wn * 32 + 16 * y + Mfma<T>::col(lk, r);
          const T v = C[(i < m ? i : m - 1) + (j < n ? j : n - 1) * ldc];
          acc[x][y][r] = v;   // (outside C, or in the other triangle: computed, not stored)
        }
      }
  auto sum = [&](int64_t k1) __attribute__((always_inline)) {   // k1 .. ke - 1 onto the accumulators
    load(k1);
    store(0);
    __syncthreads();
    int cur = 0;
    for (int64_t k0 = k1; k0 < ke; k0 += BK, cur ^= 1) {
      const bool more = k0 + BK < ke;
      if (more) load(k0 + BK);
      const T* as = As[cur] + wm * 32 + lr;
      const T* bs = Bs[cur] + wn * 32 + lr;
#pragma unroll
      for (int ks = 0; ks < BK / 4; ++ks) {
        const int kr = 4 * ks + lk;
        T av[2], bv[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) av[x] = as[kr * SLD + 16 * x];
#pragma unroll
        for (int y = 0; y < 2; ++y) bv[y] = bs[kr * SLD + 16 * y];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) acc[x][y] = Mfma<T>::step(bv[y], av[x], acc[x][y]);
      }
      if (more) store(cur ^ 1);
      __syncthreads();
    }
  };
  if (kb < ke) sum(kb);
  if constexpr (PARTS) {
    if (!part) {   // (all but the last part are whole slabs: the pointers stand at the next one's first)
      acc_t total[2][2];
#pragma unroll 1
      for (int64_t k1 = kb + kper; k1 < k; k1 += kper) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            total[x][y] = acc[x][y];
            acc[x][y] = acc_t{T(0), T(0), T(0), T(0)};
          }
        ke = k1 + kper < k ? k1 + kper : k;
        sum(k1);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) acc[x][y] = total[x][y] + acc[x][y];
      }
    }
  }
  T* const out = part ? part + (int64_t)blockIdx.y * m * n : C;
  const int64_t ldo = part ? m : ldc;
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int64_t i = row0 + wm * 32 + 16 * x + lr;
    T cv[2][4];
    const bool need_c = !part && !cinit && beta != T(0);
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t j = col0 + wn * 32 + 16 * y + Mfma<T>::col(lk, r);
        cv[y][r] = (need_c && c_ok(i, j)) ? C[i + j * ldc] : T(0);
      }
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t j = col0 + wn * 32 + 16 * y + Mfma<T>::col(lk, r);
        if (!c_ok(i, j)) continue;
        T v = acc[x][y][r];
        if constexpr (PARTS) {
          if (!part) v = scaled_sum(v, alpha, beta, cv[y][r]);
        } else if (!cinit) {
          v = alpha * v;
          v = beta == T(0) ? v : (beta == T(1) ? cv[y][r] + v : beta * cv[y][r] + v);
        }
        out[i + j * ldo] = v;
      }
  }
}

// C = alpha (sum of the nz partial products, in order) + beta C
template <typename T>
__global__ void __launch_bounds__(256)
splitk_sum_kernel(int64_t m, int64_t n, int nz, const T* __restrict__ part, T alpha, T beta, T* __restrict__ C,
                  int64_t ldc, int tri) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= m || (tri == kLower && i < j) || (tri == kUpper && i > j)) return;
  T s = part[i + j * m];
  for (int z = 1; z < nz; ++z) s += part[((int64_t)z * n + j) * m + i];
  T* const c = C + i + j * ldc;
  *c = scaled_sum(s, alpha, beta, beta == T(0) ? T(0) : *c);
}

// ---- 128 x 128 tiles with the operand slabs moved global -> LDS by the load unit
//
// MFMA order and epilogue as gemm_small_kernel (the results are identical bit for
// bit) on 128 x 128 tiles (four waves of 64 x 64); every thread issues 8 global_load_lds_dwordx4
// per slab of 128 bytes along k (16 doubles, 32 floats): each lane's 16 bytes land in LDS at 16 x its lane id
// after the instruction's (wave-uniform) base, without passing through VGPRs
// and without ds_write instructions. Two LDS buffers: slab kt + 1 is in flight
// while slab kt is multiplied; one barrier per slab, after each thread's own
// loads have landed (vmcnt 0).
// Slab layouts in LDS:
//  - operand contiguous along m (A) or n (op(B) = B^T), FP64: 16 k-rows of 128
//    elements, k-row l at l * LDA_S; a wave instruction moves one k-row (lane:
//    elements 2 lane, 2 lane + 1, so the m / n extent must be even);
//  - the same, FP32: 32 k-rows of 128 floats, an instruction moves two (32 lanes
//    of 4 floats each, so the extent must be a multiple of 4); an odd row has its
//    16-float groups exchanged in pairs, so that the four rows a fragment reads
//    lie in both halves of the LDS banks;
//  - operand contiguous along k: 128 columns of 128 bytes, its eight 16-byte chunks
//    stored at slot chunk ^ sw(c), sw(c) = (c ^ c >> 3) & 7, so that the 16
//    lanes reading one k of 16 consecutive columns hit distinct LDS banks; a
//    wave instruction moves 8 columns (lane 8 jj + s: column 8 q + jj, the chunk
//    s ^ sw).
// For the update form with alpha = -1 the A fragments are negated after their
// LDS reads (gemm_small_kernel negates B before storing it): either
// way every product enters the accumulator as fl(c - a b).
// FP32 reaches 122 TF/s at 4096^3 (1127 us against 1362 us on 64 x 64 tiles; a large
// library product reaches 148 on this card): bound by the matrix cores and, with two
// workgroups a CU, the wait at each slab's barrier.
template <typename T> constexpr int kDmaK = 128 / (int)sizeof(T);                   // k of a slab
template <typename T> constexpr int kDmaSlab = sizeof(T) == 8 ? 16 * LDA_S : 4096;   // elements per operand buffer

typedef __attribute__((address_space(3))) void* lds_void_ptr;

__device__ __forceinline__ void lds_dma16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(g, (lds_void_ptr)l, 16, 0, 0);
}
__device__ __forceinline__ double flip(double v, bool neg) {
  return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) ^ (neg ? 0x8000000000000000ull : 0ull));
}
__device__ __forceinline__ float flip(float v, bool neg) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ (neg ? 0x80000000u : 0u));
}

// One operand's slab mover and fragment reader. MNC: contiguous along m / n.
template <typename T, bool MNC>
struct DmaOperand {
  static constexpr bool kF32 = sizeof(T) == 4;
  static constexpr int CE = 16 / (int)sizeof(T);   // elements of a 16-byte chunk
  const T* p[4];        // per-thread source of each of the thread's 4 instructions (k0 = 0)
  int64_t ld;
  int o[4];             // LDS offset of fragment x at ks = 0

  __device__ __forceinline__ void init(const T* X, int64_t ldx, int64_t mn0, int64_t mn, int wave, int lane,
                                       int w, int lr, int lk) {
    ld = ldx;
    if (MNC) {
      const int rr = kF32 ? lane >> 5 : 0;   // row of the instruction's two
      const int64_t e0 = mn0 + CE * (kF32 ? (lane & 31) ^ (4 * rr) : lane), e = e0 < mn ? e0 : mn - CE;
#pragma unroll
      for (int c = 0; c < 4; ++c) p[c] = X + e + (int64_t)((kF32 ? 2 : 1) * (wave + 4 * c) + rr) * ldx;
#pragma unroll
      for (int x = 0; x < 4; ++x)
        o[x] = w * 64 + lr + (kF32 ? lk * 128 + 16 * (x ^ (lk & 1)) : lk * LDA_S + 16 * x);
    } else {
      const int jj = lane >> 3, s = lane & 7;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int q = wave + 4 * c;
        const int64_t col = mn0 + 8 * q + jj < mn ? mn0 + 8 * q + jj : mn - 1;
        p[c] = X + CE * (s ^ ((jj ^ q) & 7)) + col * ldx;
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int c = w * 64 + 16 * x + lr;
        o[x] = c * kDmaK<T> + CE * ((lk / CE) ^ ((c ^ (c >> 3)) & 7)) + lk % CE;
      }
    }
  }
  __device__ __forceinline__ void issue(int64_t k0, T* buf, int wave) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (MNC) lds_dma16(p[c] + k0 * ld, buf + (wave + 4 * c) * (kF32 ? 256 : LDA_S));
      else lds_dma16(p[c] + k0, buf + (wave + 4 * c) * 8 * kDmaK<T>);
    }
  }
  // fragment x (16 elements along m / n) at k = 4 ks + lk
  __device__ __forceinline__ T frag(const T* buf, int ks, int x) const {
    return MNC ? buf[o[x] + 4 * ks * (kF32 ? 128 : LDA_S)] : buf[o[x] ^ (4 * ks)];
  }
};

// init: the update form accumulates onto C itself (as the other kernel does);
// otherwise the products are summed first and C added once.
template <typename T, bool TA, bool TB>
__global__ void __launch_bounds__(NT, 2)
gemm_dma_kernel(int64_t m, int64_t n, int64_t k, T alpha, const T* __restrict__ A, int64_t lda,
                const T* __restrict__ B, int64_t ldb, T beta, T* __restrict__ C, int64_t ldc,
                int tri, int64_t tri_tiles, int init) {
  typedef typename Mfma<T>::acc acc_t;
  constexpr int DBK = kDmaK<T>;
  __shared__ __attribute__((aligned(16))) T As0[kDmaSlab<T>];
  __shared__ __attribute__((aligned(16))) T As1[kDmaSlab<T>];
  __shared__ __attribute__((aligned(16))) T Bs0[kDmaSlab<T>];
  __shared__ __attribute__((aligned(16))) T Bs1[kDmaSlab<T>];

  const int64_t ntm = (m + BM - 1) / BM, ntn = (n + BN - 1) / BN;
  int64_t tm, tn;
  if (tri_tiles > 0) tri_tile_coords(blockIdx.x, tri_tiles, ntm, ntn, tri, tm, tn);
  else tile_coords(blockIdx.x, ntm, ntn, tm, tn);
  const int64_t row0 = tm * BM, col0 = tn * BN;
  if (tri == kLower && row0 + BM - 1 < col0) return;
  if (tri == kUpper && col0 + BN - 1 < row0) return;

  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 15, lk = lane >> 4;

  DmaOperand<T, !TA> opa;
  DmaOperand<T, TB> opb;
  opa.init(A, lda, row0, m, wave, lane, wm, lr, lk);
  opb.init(B, ldb, col0, n, wave, lane, wn, lr, lk);

  const bool cinit = init && beta == T(1) && (alpha == T(1) || alpha == T(-1));
  const bool neg = cinit && alpha == T(-1);
  auto c_ok = [&](int64_t i, int64_t j) {
    return i < m && j < n && !(tri == kLower && i < j) && !(tri == kUpper && i > j);
  };
  acc_t acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = acc_t{T(0), T(0), T(0), T(0)};
  if (cinit) {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int64_t i = row0 + wm * 64 + 16 * x + lr;
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t j = col0 + wn * 64 + 16 * y + Mfma<T>::col(lk, r);
          if (c_ok(i, j)) acc[x][y][r] = C[i + j * ldc];
        }
    }
  }

  auto compute = [&](const T* as, const T* bs) {
#pragma unroll
    for (int ks = 0; ks < DBK / 4; ++ks) {
      T av[4], bv[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) av[x] = flip(opa.frag(as, ks, x), neg);
#pragma unroll
      for (int y = 0; y < 4; ++y) bv[y] = opb.frag(bs, ks, y);
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = Mfma<T>::step(bv[y], av[x], acc[x][y]);
    }
  };
  // vmcnt(0), expcnt and lgkmcnt left at their maxima
  constexpr int kWaitVm0 = 0x0F70;
  const int nk = (int)(k / DBK);
  opa.issue(0, As0, wave);
  opb.issue(0, Bs0, wave);
  for (int kt = 0; kt < nk; kt += 2) {
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    if (kt + 1 < nk) {
      opa.issue((int64_t)(kt + 1) * DBK, As1, wave);
      opb.issue((int64_t)(kt + 1) * DBK, Bs1, wave);
    }
    compute(As0, Bs0);
    if (kt + 1 >= nk) break;
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    if (kt + 2 < nk) {
      opa.issue((int64_t)(kt + 2) * DBK, As0, wave);
      opb.issue((int64_t)(kt + 2) * DBK, Bs0, wave);
    }
    compute(As1, Bs1);
  }

  if (cinit) {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int64_t i = row0 + wm * 64 + 16 * x + lr;
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t j = col0 + wn * 64 + 16 * y + Mfma<T>::col(lk, r);
          if (c_ok(i, j)) C[i + j * ldc] = acc[x][y][r];
        }
    }
    return;
  }
  const bool need_c = beta != T(0);
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int64_t i = row0 + wm * 64 + 16 * x + lr;
    bool ok[4][4];
    T cv[4][4];
#pragma unroll
    for (int y = 0; y < 4; ++y) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t j = col0 + wn * 64 + 16 * y + Mfma<T>::col(lk, r);
        ok[y][r] = c_ok(i, j);
        cv[y][r] = (need_c && ok[y][r]) ? C[i + j * ldc] : T(0);
      }
    }
#pragma unroll
    for (int y = 0; y < 4; ++y) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (!ok[y][r]) continue;
        const int64_t j = col0 + wn * 64 + 16 * y + Mfma<T>::col(lk, r);
        const T v = alpha * acc[x][y][r];
        C[i + j * ldc] = beta == T(0) ? v : (beta == T(1) ? cv[y][r] + v : beta * cv[y][r] + v);
      }
    }
  }
}

// Whether gemm_dma_kernel takes the product: whole k-slabs, 16-byte aligned operand
// columns, and whole 16-byte chunks along each operand's contiguous m / n direction.
template <typename T>
inline bool dma_ok(bool ta, bool tb, int64_t m, int64_t n, int64_t k, const void* a, int64_t lda,
                   const void* b, int64_t ldb) {
  constexpr int CE = 16 / (int)sizeof(T);
  if (k < kDmaK<T> || k % kDmaK<T> != 0) return false;
  if ((((uintptr_t)a) | ((uintptr_t)b)) & 15) return false;
  if (lda % CE || ldb % CE) return false;
  if (!ta && m % CE) return false;
  if (tb && n % CE) return false;
  return true;
}

template <typename T>
__global__ void scale_kernel(int64_t m, int64_t n, T beta, T* __restrict__ c, int64_t ldc, int tri) {
  const int64_t total = m * n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = e % m, j = e / m;
    if (tri == kLower && i < j) continue;
    if (tri == kUpper && i > j) continue;
    T* p = c + i + j * ldc;
    *p = beta == T(0) ? T(0) : *p * beta;
  }
}

}  // namespace

template <typename T>
void scale_cm(int64_t m, int64_t n, T beta, T* c, int64_t ldc, hipStream_t s, int tri) {
  if (m <= 0 || n <= 0 || beta == T(1)) return;
  int64_t total = m * n;
  int blocks = (int)std::min<int64_t>((total + 255) / 256, 65536);
  hipLaunchKernelGGL(scale_kernel<T>, dim3(blocks), dim3(256), 0, s, m, n, beta, c, ldc, tri);
  ZH_LAUNCH_CHECK();
}
template void scale_cm<double>(int64_t, int64_t, double, double*, int64_t, hipStream_t, int);
template void scale_cm<float>(int64_t, int64_t, float, float*, int64_t, hipStream_t, int);

// 64 x 64 tiles rather than 128 x 128 ones moved by the load unit. Both run in
// rounds over the CUs, and a round of the first costs 3.26 rounds of the second in
// FP64 (0.27 TF/s a CU on 128 x 128 tiles, 0.22 on 64 x 64 ones), 3.45 in FP32 (0.48
// and 0.40; 3.2 to 3.6 over k = 320 .. 4096), more while a CU has only one tile
// (3.64 and 4.0). FP64: 2048 x 2176 x 784 (272 tiles, two rounds for one tile more
// than a CU each) 198 against 163 us, 2048^3 (256 tiles) 277 against 322 us, 2500^2 x
// 2512 609 against 671 us. FP32: 2048 x 2176 x 768 117 against 91 us, 2048^3 186
// against 190 us, 2500^2 x 2496 349 against 386 us, 3100 x 2900 x 3008 (575 tiles)
// 664 against 581 us, 4096^3 1127 against 1362 us.
// In FP32, up to k = 128, four workgroups a CU hide the operands' first slab and the
// reads and writes of C, which the larger tiles' two do not: 6000^2 x 64 117 against
// 86 us, 5000^2 x 128 124 against 98, 12000^2 x 128 527 against 462. Beyond it depends on
// the form: k = 192 5000^2 154 against 130 us, 8192^2 333 against 354.
template <typename T>
static bool small_tiles(int64_t t128, int64_t t64, int64_t k) {
  if (sizeof(T) == 4 && k <= 128) return true;
  const int64_t cus = device_cu_count();
  const int64_t r128 = (t128 + cus - 1) / cus, r64 = (t64 + cus - 1) / cus;
  constexpr int one = sizeof(T) == 8 ? 364 : 400, more = sizeof(T) == 8 ? 326 : 345;
  return (r128 == 1 ? one : more * r128) > 100 * r64;
}

template <typename T>
static void small_gemm(bool ta, bool tb, int64_t m, int64_t n, int64_t k, T alpha, const T* a, int64_t lda, const T* b,
                       int64_t ldb, T beta, T* c, int64_t ldc, hipStream_t s, int tri, int64_t tiles, int64_t tri_tiles,
                       int nz, T* part) {
  const int64_t slabs = (k + BK - 1) / BK, kper = (slabs + nz - 1) / nz * BK;
  const dim3 grid((unsigned)tiles, part ? (unsigned)nz : 1u), block(NT);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, tri, tri_tiles, kper,
                       part);
  };
  auto form = [&](auto parts) {
    constexpr bool P = decltype(parts)::value;
    if (!ta && !tb) go(gemm_small_kernel<T, false, false, P>);
    else if (ta && !tb) go(gemm_small_kernel<T, true, false, P>);
    else if (!ta && tb) go(gemm_small_kernel<T, false, true, P>);
    else go(gemm_small_kernel<T, true, true, P>);
  };
  if (nz > 1) form(std::true_type{});
  else form(std::false_type{});
  ZH_LAUNCH_CHECK();
  if (part) {
    hipLaunchKernelGGL(splitk_sum_kernel<T>, dim3((unsigned)((m + 255) / 256), (unsigned)n), dim3(256), 0, s, m, n, nz,
                       (const T*)part, alpha, beta, c, ldc, tri);
    ZH_LAUNCH_CHECK();
  }
}

template <typename T>
static void dma_gemm(bool ta, bool tb, int64_t m, int64_t n, int64_t k, T alpha, const T* a, int64_t lda, const T* b,
                     int64_t ldb, T beta, T* c, int64_t ldc, hipStream_t s, int tri, int64_t tiles, int64_t tri_tiles,
                     int init) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(NT), 0, s, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc,
                       tri, tri_tiles, init);
  };
  if (!ta && !tb) go(gemm_dma_kernel<T, false, false>);
  else if (ta && !tb) go(gemm_dma_kernel<T, true, false>);
  else if (!ta && tb) go(gemm_dma_kernel<T, false, true>);
  else go(gemm_dma_kernel<T, true, true>);
  ZH_LAUNCH_CHECK();
}

bool gemm_f32_dma_cm(int64_t m, int64_t n, int64_t k, float alpha, const float* a, int64_t lda, const float* b,
                     int64_t ldb, float beta, float* c, int64_t ldc, hipStream_t s) {
  if (!gemm_dma_enabled() || !dma_ok<float>(false, false, m, n, k, a, lda, b, ldb)) return false;
  const int64_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  dma_gemm<float>(false, false, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s, 0, tiles, 0, 0);
  return true;
}

template <typename T>
void gemm_cm(int transa, int transb, int64_t m, int64_t n, int64_t k, T alpha, const T* a, int64_t lda,
             const T* b, int64_t ldb, T beta, T* c, int64_t ldc, hipStream_t s, int tri, int split_slot) {
  if (m <= 0 || n <= 0) return;
  if (alpha == T(0) || k <= 0) {  // gemm.zig:104-140: only the beta scaling remains
    scale_cm<T>(m, n, beta, c, ldc, s, tri);
    return;
  }
  const bool ta = !is_notrans(transa), tb = !is_notrans(transb);
  const int64_t ntm = (m + BM - 1) / BM, ntn = (n + BN - 1) / BN;
  const int64_t tri_tiles = tri_tile_count(tri, ntm, ntn);
  const int64_t tiles = tri_tiles > 0 ? tri_tiles : ntm * ntn;
  const int64_t nsm = (m + SM - 1) / SM, nsn = (n + SM - 1) / SM;
  const int64_t stri = tri_tile_count(tri, nsm, nsn), stiles = stri > 0 ? stri : nsm * nsn;
  if (gemm_dma_enabled() && dma_ok<T>(ta, tb, m, n, k, a, lda, b, ldb) && !small_tiles<T>(tiles, stiles, k)) {
    dma_gemm<T>(ta, tb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s, tri, tiles, tri_tiles, 1);
    return;
  }
  // k is cut into parts where the tiles leave CUs idle: about two workgroups per CU,
  // each with at least 128 of k (parts of 4 or 8 slabs no longer pay their sum). The
  // parts follow from the shape alone, so that a product recorded into a graph, where
  // they have no memory, has the direct one's bits. Their sums (nz m n values: at most
  // two tiles per CU, a triangle's up to four) go to a workspace of one size: it never
  // grows, which would wait for the device.
  const int64_t cus = device_cu_count();
  int nz = 1;
  if (split_slot >= 0 && stiles < cus)
    nz = (int)std::max<int64_t>(1, std::min<int64_t>({2 * cus / stiles, k / 128, 32}));
  T* part = nullptr;
  if (nz > 1) part = static_cast<T*>(try_workspace(sizeof(double) * 4 * (size_t)cus * SM * SM, split_slot, s));
  small_gemm<T>(ta, tb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s, tri, stiles, stri, nz, part);
}
template void gemm_cm<double>(int, int, int64_t, int64_t, int64_t, double, const double*, int64_t, const double*,
                              int64_t, double, double*, int64_t, hipStream_t, int, int);
template void gemm_cm<float>(int, int, int64_t, int64_t, int64_t, float, const float*, int64_t, const float*,
                             int64_t, float, float*, int64_t, hipStream_t, int, int);

void scale_f64_cm(int64_t m, int64_t n, double beta, double* c, int64_t ldc, hipStream_t s, int tri) {
  scale_cm<double>(m, n, beta, c, ldc, s, tri);
}

void gemm_f64_cm(int transa, int transb, int64_t m, int64_t n, int64_t k, double alpha,
                 const double* a, int64_t lda, const double* b, int64_t ldb, double beta,
                 double* c, int64_t ldc, hipStream_t s, int tri) {
  gemm_cm<double>(transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, s, tri);
}

}  // namespace zmlhip
