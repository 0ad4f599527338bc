// Block Gauss-Jordan elimination without pivoting, 32 columns a step, on 64 x 64
// tiles (one workgroup each): the tile update shared by the inverse of
// Q_1 - S (mak_qtrail.hip) and the batched inverse of a Hermitian positive
// definite matrix (mak_pullback.hip).
#pragma once

#include "mak_common.hpp"
#include "mak_dense32.hpp"

namespace mak {

constexpr int GB = 32;  // columns per elimination step
constexpr int GT = 64;  // tile of a step's workgroup: four waves of GB x GB

// re, im += a b (one k-group of four)
__device__ __forceinline__ void mfma_acc(v4d& re, v4d&, double a, double b) { re = mfma_f64(a, b, re); }
__device__ __forceinline__ void mfma_acc(v4d& re, v4d& im, const zd& a, const zd& b) {
  re = mfma_f64(a.x, b.x, re);
  im = mfma_f64(a.x, b.y, im);
  re = mfma_f64(-a.y, b.y, re);
  im = mfma_f64(a.y, b.x, im);
}
template <typename T> __device__ __forceinline__ T acc_get(const v4d& re, const v4d& im, int u);
template <> __device__ __forceinline__ double acc_get<double>(const v4d& re, const v4d&, int u) { return re[u]; }
template <> __device__ __forceinline__ zd acc_get<zd>(const v4d& re, const v4d& im, int u) {
  return mkz(re[u], im[u]);
}
__device__ __forceinline__ void acc_set(v4d& re, v4d&, int u, double v) { re[u] = v; }
__device__ __forceinline__ void acc_set(v4d& re, v4d& im, int u, const zd& v) {
  re[u] = v.x;
  im[u] = v.y;
}

// Step k on the tile (m0, n0) of an n x n matrix, by 256 threads.  elem(i, j)
// is the matrix before the step (any i, j: the identity outside n x n), P the
// inverse of its block k (32 x 32, column-major), dst (ld ldd) receives the
// tile.  With R_k = P_k M_kj (M_kk taken as I), every entry of the result is
// M_ij - M_ik R_kj where M_ik is taken as -I for the rows of block k, and M_ij
// as 0 for its rows and columns.  The wave whose 32 x 32 quarter is the next
// diagonal block calls next(A, Y) with it in A (LDS, 32 x 33; Y: scratch).
// Bound by launch and load latency (12 us a step at n = 1024, Float64) and by
// the serial inverse of the next block, which is why that runs right here.
template <typename T, class Elem, class Next>
__device__ __forceinline__ void gj_tile_step(int n, int k, int m0, int n0, const T* P, T* dst, int64_t ldd,
                                             const Elem& elem, const Next& next_block) {
  constexpr int LD = GT + 2;
  __shared__ T Pl[GB][33];       // P_k; then the next diagonal block
  __shared__ T Bk[GB][LD];       // M_kj as [k][j], then R_kj (each wave replaces the columns it alone reads)
  __shared__ T Lm[GB][LD];       // -M_ik as [k][i]; then the next inverse's scratch
  static_assert(GB * LD >= GB * 33, "scratch of the inverse");
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int lr = lane & 15, q = lane >> 4;
  const int k0 = k * GB;
  for (int e = tid; e < GB * GB; e += 256) Pl[e % GB][e / GB] = P[e];
  for (int e = tid; e < GB * GT; e += 256) {
    const int kk = e % GB, j = n0 + e / GB;
    Bk[kk][e / GB] = (j >= k0 && j < k0 + GB) ? (j - k0 == kk ? s_one(T()) : s_zero(T())) : elem(k0 + kk, j);
  }
  for (int e = tid; e < GB * GT; e += 256) {
    const int i = m0 + e % GT, kk = e / GT;
    Lm[kk][e % GT] = (i >= k0 && i < k0 + GB) ? (i - k0 == kk ? s_one(T()) : s_zero(T()))
                                              : s_neg(elem(i, k0 + kk));
  }
  // the tile of M: this wave's 32 x 32 quarter, lane lr holding rows, register
  // u the columns 4 u + q of each 16 x 16 block
  const int wm = w & 1, wn = w >> 1;
  v4d cr[2][2], ci[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      cr[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
      ci[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int gi = m0 + wm * 32 + i * 16 + lr, gj = n0 + wn * 32 + j * 16 + 4 * u + q;
        const bool out = (gi >= k0 && gi < k0 + GB) || (gj >= k0 && gj < k0 + GB);
        acc_set(cr[i][j], ci[i][j], u, out ? s_zero(T()) : elem(gi, gj));
      }
    }
  __syncthreads();
  // R_kj: wave w forms its columns 16 w .. 16 w + 15
  {
    v4d rr[2], ri[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      rr[b] = v4d{0.0, 0.0, 0.0, 0.0};
      ri[b] = v4d{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll
    for (int kk = 0; kk < GB; kk += 4) {
      const T bv = Bk[kk + q][16 * w + lr];
#pragma unroll
      for (int b = 0; b < 2; ++b) mfma_acc(rr[b], ri[b], Pl[16 * b + lr][kk + q], bv);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) Bk[16 * b + 4 * u + q][16 * w + lr] = acc_get<T>(rr[b], ri[b], u);
  }
  __syncthreads();
#pragma unroll
  for (int kk = 0; kk < GB; kk += 4) {
    T av[2], bv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) av[i] = Lm[kk + q][wm * 32 + i * 16 + lr];
#pragma unroll
    for (int j = 0; j < 2; ++j) bv[j] = Bk[kk + q][wn * 32 + j * 16 + lr];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) mfma_acc(cr[i][j], ci[i][j], bv[j], av[i]);
  }
  const int k1 = k0 + GB;  // the next diagonal block, if it is this wave's quarter
  const bool next = k1 < n && m0 + wm * 32 == k1 && n0 + wn * 32 == k1;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int ti = i * 16 + lr, tj = j * 16 + 4 * u + q;
        const int gi = m0 + wm * 32 + ti, gj = n0 + wn * 32 + tj;
        const T v = acc_get<T>(cr[i][j], ci[i][j], u);
        if (gi < n && gj < n) dst[gi + (int64_t)gj * ldd] = v;
        if (next) Pl[ti][tj] = v;  // Pl is no longer read (the barrier above)
      }
  if (k1 < n && m0 / GT == k1 / GT && n0 / GT == k1 / GT) __syncthreads();  // Lm is no longer read
  if (next) next_block(Pl, reinterpret_cast<T (*)[33]>(&Lm[0][0]));
}

}  // namespace mak
