// The Householder signs and the trailing columns of the full Q from the
// compact Q of the whole-matrix CholeskyQR2 (mak_cholqr2.hip), for qr_full!
// and for positive = false (src/implementations/qr.jl:106-109,132-188).
//
// Householder reconstruction (Ballard, Demmel, Grigori, Jacquelin, Nguyen,
// Solomonik, IPDPS 2014): with A = Q R (positive gauge, Q m x n) the
// Householder vectors of A are the L factor of Q - [S; 0] = L U (no pivoting),
// S = diag(s_j) unimodular with s_j = -sign(p_j) of the j-th pivot, and
// H_1 ... H_n = I - V T V^H with V = L, T = -U S^H V_1^{-H}.  Its trailing
// columns need neither V nor T: with M = Q_1 - S (Q_1, Q_2 the first n and
// the other rows of Q),
//   Q[:, n:] = [0; I] + (Q - [S; 0]) W,   W = S^H M^{-H} Q_2^H,
// two large products and one n x n inverse, against one pass over all of Q
// per 256-column reflector when the reflectors are applied one by one.  The
// Householder QR's own first columns and R are Q S^H and S R.
//
// M^{-1} comes from a block Gauss-Jordan elimination (32 columns a step, no
// pivoting: every pivot of M has magnitude >= 1), whose Schur complements are
// the LU's, so it meets the same pivots and fixes S on the way.  Step k is one
// launch over 64 x 64 tiles, out of one buffer into another; the wave that
// owns the next diagonal block inverts it (with its signs) right after its
// update, so a step is one launch and the serial part of it one wave's
// 32 x 32 inverse.
#include <algorithm>

#include "mak_common.hpp"
#include "mak_dense32.hpp"
#include "mak_gj.hpp"
#include "mak_kernels.hpp"
#include "mak_mi355x_internal.hpp"

namespace mak {

namespace {

// -sign(p) (sign_safe's convention; |p| <= 2 here)
__device__ __forceinline__ double minus_sign(double p) { return p < 0.0 ? 1.0 : -1.0; }
__device__ __forceinline__ zd minus_sign(const zd& p) {
  const double a2 = fma(p.x, p.x, p.y * p.y);
  if (!(a2 > 1e-290)) return mkz(-1.0, 0.0);
  const double r = rsqrt_nr(a2);
  return mkz(-p.x * r, -p.y * r);
}

// x -= m wx, s -= m ws with m = s of lane K of the 16-lane row (DPP source; s
// may have been written by the instruction before, and a VGPR may be a DPP
// source from two instructions after its write: s_nop 1).  In asm, so that
// the compiler cannot gather the sixteen broadcasts of a step up front (it
// spills them).
template <int K> __device__ __forceinline__ void gj_row(double& s, double& x, double ws, double wx) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %1, -%0, %3 row_newbcast:%c4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, -%0, %2 row_newbcast:%c4 row_mask:0xf bank_mask:0xf"
      : "+v"(s), "+v"(x)
      : "v"(ws), "v"(wx), "n"(K));
}
template <int K> __device__ __forceinline__ void gj_row(zd& s, zd& x, const zd& ws, const zd& wx) {
  double mr, mi;
  asm("s_nop 1\n\t"
      "v_mov_b64_dpp %4, %0 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b64_dpp %5, %1 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fma_f64 %2, -%4, %8, %2\n\t"
      "v_fma_f64 %3, -%4, %9, %3\n\t"
      "v_fma_f64 %0, -%4, %6, %0\n\t"
      "v_fma_f64 %1, -%4, %7, %1\n\t"
      "v_fma_f64 %2, %5, %9, %2\n\t"
      "v_fma_f64 %3, -%5, %8, %3\n\t"
      "v_fma_f64 %0, %5, %7, %0\n\t"
      "v_fma_f64 %1, -%5, %6, %1"
      : "+v"(s.x), "+v"(s.y), "+v"(x.x), "+v"(x.y), "=&v"(mr), "=&v"(mi)
      : "v"(ws.x), "v"(ws.y), "v"(wx.x), "v"(wx.y), "n"(K));
}

// Gauss-Jordan step K of [s | x] (lane c of a 16-lane row: column c): the
// pivot p - S, S = -sign(p) (0 from column `valid` on), of lane K; sg of lane
// K receives S.
template <typename T, int K, int R>
__device__ __forceinline__ void gj16_rows(T (&s)[16], T (&x)[16], const T& ws, const T& wx) {
  if constexpr (R < 16) {
    if constexpr (R != K) gj_row<K>(s[R], x[R], ws, wx);
    gj16_rows<T, K, R + 1>(s, x, ws, wx);
  }
}
template <typename T, int K>
__device__ __forceinline__ void gj16_step(T (&s)[16], T (&x)[16], int c0, int valid, T& sg) {
  dpp_source(s[K]);
  const T p = row_bcast<K>(s[K]);
  const T sk = K < valid ? minus_sign(p) : s_zero(T());
  const T inv = s_recip(s_sub(p, sk));
  sg = sel(step_lane(c0) == K, sk, sg);
  const T ws = s_mul(s[K], inv), wx = s_mul(x[K], inv);
  gj16_rows<T, K, 0>(s, x, ws, wx);
  s[K] = ws;
  x[K] = wx;
}
template <typename T, int... Ks>
__device__ __forceinline__ void gj16(T (&s)[16], T (&x)[16], int c, int valid, T& sg,
                                     std::integer_sequence<int, Ks...>) {
  (gj16_step<T, Ks>(s, x, c, valid, sg), ...);
}

// By one wave: A (LDS, 32 x 33) <- (A - S)^{-1}, S = diag(sg) chosen pivot by
// pivot (zero from column `valid` on, where A is the identity), sg (32) to
// global memory.  2 x 2 blocks of 16, one 16-lane row of the wave per
// right-hand side; Y (LDS, 32 x 33) and the padding column of A are scratch:
//   P11 = M11^{-1}, X12 = P11 A12;  A22 -= A21 X12, D = A21 P11;
//   P22, Z = P22 D;  inverse = [P11 + X12 Z, -X12 P22; -Z, P22].
template <typename T>
__device__ __forceinline__ void wave_sign_inv32(T (*A)[33], T (*Y)[33], int valid, T* sg) {
  const int l = lane_id(), c = l & 15, q = l >> 4;
  const auto seq = std::make_integer_sequence<int, 16>{};
  if (l < 32) A[l][32] = l == 15 ? s_one(T()) : s_zero(T());
  wave_lds_sync();
  const T* eye = &A[15 - c][32];  // rows 0 .. 15: column c of I
  T s[16], x[16], sgn = s_zero(T());
  const T* px = q == 1 ? &A[0][16 + c] : eye;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s[r] = A[r][c];
    x[r] = px[33 * r];
  }
  gj16<T>(s, x, c, valid, sgn, seq);
  if (q == 0) sg[c] = sgn;
  if (q < 2) {
    T* p = q == 0 ? &Y[0][c] : &Y[0][16 + c];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[33 * r] = x[r];
  }
  wave_lds_sync();
  {
    v4d gr = {0.0, 0.0, 0.0, 0.0}, gi = gr, hr = gr, hi = gr;
    T a[4], b1[4], b2[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[u] = A[16 + c][4 * u + q];
      b1[u] = Y[4 * u + q][16 + c];
      b2[u] = Y[4 * u + q][c];
      acc_set(gr, gi, u, A[16 + 4 * u + q][16 + c]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      mfma_acc(gr, gi, s_neg(a[u]), b1[u]);
      mfma_acc(hr, hi, a[u], b2[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      A[16 + 4 * u + q][16 + c] = acc_get<T>(gr, gi, u);
      A[16 + 4 * u + q][c] = acc_get<T>(hr, hi, u);
    }
  }
  wave_lds_sync();
  px = q == 1 ? &A[16][c] : eye;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s[r] = A[16 + r][16 + c];
    x[r] = px[33 * r];
  }
  wave_lds_sync();
  gj16<T>(s, x, c, valid - 16, sgn, seq);
  if (q == 0) sg[16 + c] = sgn;
  if (q < 2) {
    T* p = q == 0 ? &A[16][16 + c] : &A[16][c];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[33 * r] = q == 0 ? x[r] : s_neg(x[r]);
  }
  wave_lds_sync();
  {
    v4d gr = {0.0, 0.0, 0.0, 0.0}, gi = gr, hr = gr, hi = gr;
    T a[4], b1[4], b2[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[u] = s_neg(Y[c][16 + 4 * u + q]);  // -X12
      b1[u] = A[16 + 4 * u + q][16 + c];   // P22
      b2[u] = A[16 + 4 * u + q][c];        // -Z
      acc_set(hr, hi, u, Y[4 * u + q][c]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      mfma_acc(gr, gi, a[u], b1[u]);
      mfma_acc(hr, hi, a[u], b2[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      A[4 * u + q][16 + c] = acc_get<T>(gr, gi, u);
      A[4 * u + q][c] = acc_get<T>(hr, hi, u);
    }
  }
  wave_lds_sync();
}

template <typename T> struct GjArgs {
  const T* src;   // M before the step (n x n, ld lds); step 0: Q_1 (S is implicit in P)
  int64_t lds;
  T* dst;         // M after it (ld ldd)
  int64_t ldd;
  int n, k;       // k: the step (columns GB k ..)
  T* P;           // diagonal blocks' inverses, 32 x 32 each, column-major
  T* sg;          // S, padded to a multiple of GB
  int signs_only; // only the Schur complement right of and below block k is wanted
  const int* gate;
};

// P_0 and the first signs, from the leading block.
template <typename T> __global__ void __launch_bounds__(64) gj_first_kernel(GjArgs<T> a) {
  __shared__ T A[GB][33], Y[GB][33];
  if (*a.gate != 1) return;
  for (int e = threadIdx.x; e < GB * GB; e += 64) {
    const int i = e % GB, j = e / GB;
    A[i][j] = (i < a.n && j < a.n) ? a.src[i + (int64_t)j * a.lds] : (i == j ? s_one(T()) : s_zero(T()));
  }
  __syncthreads();
  wave_sign_inv32<T>(A, Y, a.n, a.sg);
  for (int e = threadIdx.x; e < GB * GB; e += 64) a.P[e] = A[e % GB][e / GB];
}

// Step k on the 64 x 64 tile (blockIdx.x, blockIdx.y).
template <typename T> __global__ void __launch_bounds__(256) gj_step_kernel(GjArgs<T> a) {
  if (*a.gate != 1) return;
  const int m0 = blockIdx.x * GT, n0 = blockIdx.y * GT, k1 = (a.k + 1) * GB, n = a.n;
  if (a.signs_only && (m0 + GT <= k1 || n0 + GT <= k1)) return;
  auto elem = [&](int i, int j) {
    return (i < n && j < n) ? a.src[i + (int64_t)j * a.lds] : (i == j ? s_one(T()) : s_zero(T()));
  };
  gj_tile_step<T>(n, a.k, m0, n0, a.P + (int64_t)a.k * GB * GB, a.dst, a.ldd, elem, [&](T (*A)[33], T (*Y)[33]) {
    wave_sign_inv32<T>(A, Y, n - k1, a.sg + k1);
    T* Pn = a.P + (int64_t)(a.k + 1) * GB * GB;
    for (int e = lane_id(); e < GB * GB; e += 64) Pn[e] = A[e % GB][e / GB];
  });
}

// K (n x n) = S^H Minv^H.
template <typename T>
__global__ void __launch_bounds__(256) scaled_adjoint_kernel(const T* Mi, const T* sg, int n, T* K, const int* gate) {
  __shared__ T tile[32][33];
  if (*gate != 1) return;
  const int r0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int i = r0 + e % 32, j = c0 + e / 32;
    if (i < n && j < n) tile[e % 32][e / 32] = Mi[i + (int64_t)j * n];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int j = c0 + e % 32, i = r0 + e / 32;  // K(j, i)
    if (i < n && j < n) K[j + (int64_t)i * n] = s_conj(s_mul(sg[j], tile[e / 32][e % 32]));
  }
}

// Qt = Q[:, n:] (m rows, nt columns): rows < n lose S W, the unit diagonal of
// [0; I] is added.
template <typename T>
__global__ void __launch_bounds__(256) trail_fix_kernel(T* Qt, int64_t ldq, int n, int nt, const T* W, const T* sg,
                                                        const int* gate) {
  if (*gate != 1) return;
  const int j = blockIdx.x;
  T* col = Qt + (int64_t)j * ldq;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < n; i += gridDim.y * 256)
    col[i] = s_sub(col[i], s_mul(sg[i], W[i + (int64_t)j * n]));
  if (blockIdx.y == 0 && threadIdx.x == 0) col[n + j] = s_add(col[n + j], s_one(T()));
}

// Q[:, j] *= conj(s_j)
template <typename T>
__global__ void __launch_bounds__(256) sign_cols_kernel(T* Q, int64_t ldq, int m, const T* sg, const int* gate) {
  if (*gate != 1) return;
  const T f = s_conj(sg[blockIdx.y]);
  T* col = Q + (int64_t)blockIdx.y * ldq;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < m; i += gridDim.x * 256) col[i] = s_mul(col[i], f);
}
// R (rows x n): rows below n are zeroed, R[i, :] *= s_i when sg is given.
template <typename T>
__global__ void __launch_bounds__(256) sign_rows_kernel(T* R, int64_t ldr, int rows, int n, const T* sg,
                                                        const int* gate) {
  if (*gate != 1) return;
  T* col = R + (int64_t)blockIdx.y * ldr;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < rows; i += gridDim.x * 256) {
    if (i >= n) col[i] = s_zero(T());
    else if (sg != nullptr) col[i] = s_mul(col[i], sg[i]);
  }
}

template <typename T>
GemmArgs gated(int M, int N, int K, const T* A, int64_t lda, const T* B, int64_t ldb, T* C, int64_t ldc,
               const int* gate) {
  GemmArgs g{};
  g.M = M; g.N = N; g.K = K;
  g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = C; g.ldc = ldc;
  g.alpha_re = 1.0;
  g.ksplit = 1; g.kchunk = K; g.batch = 1;
  g.gate = gate; g.gate_want = 1;
  return g;
}

}  // namespace

// After cholqr2_finish (same stream, its workspace cw): Q (m x m when full,
// else m x n) and R (m x n when full, else n x n, or null) of the Householder
// QR, with the positive gauge or without; runs only where the CholeskyQR2
// result was accepted.  m > n unless positive; n >= 64 (the buffers of
// cholqr2_buffers hold the inverse's blocks then).
template <typename T>
void qr_trailing_enqueue(hipStream_t s, int m, int n, T* Q, int64_t ldq, T* R, int64_t ldr, int full, int positive,
                         char* cw) {
  const Cholqr2Buffers<T> b = cholqr2_buffers<T>(cw, m, n);
  const int* gate = cholqr2_status<T>(cw, m, n);
  const int nt = full ? m - n : 0;
  T* sg = b.nn[4];
  if (nt > 0 || !positive) {
    GjArgs<T> a{};
    a.src = Q; a.lds = ldq; a.n = n; a.k = 0;
    a.P = b.nn[2]; a.sg = sg;
    a.signs_only = nt == 0;
    a.gate = gate;
    hipLaunchKernelGGL((gj_first_kernel<T>), dim3(1), dim3(64), 0, s, a);
    const int nb = cdiv(n, GB), tiles = cdiv(n, GT);
    for (int k = 0; k < nb; ++k) {
      if (a.signs_only && k + 1 == nb) break;
      a.k = k;
      a.dst = b.nn[k & 1]; a.ldd = n;
      hipLaunchKernelGGL((gj_step_kernel<T>), dim3(tiles, tiles), dim3(256), 0, s, a);
      a.src = a.dst; a.lds = n;
    }
    if (nt > 0) {
      T *K = b.nn[3], *W = b.mn;
      hipLaunchKernelGGL((scaled_adjoint_kernel<T>), dim3(cdiv(n, 32), cdiv(n, 32)), dim3(256), 0, s, a.src, sg, n, K,
                         gate);
      T* Qt = Q + (int64_t)n * ldq;
      gemm<T>(OP_N, OP_C, gated<T>(n, nt, n, K, n, Q + n, ldq, W, n, gate), s);
      gemm<T>(OP_N, OP_N, gated<T>(m, nt, n, Q, ldq, W, n, Qt, ldq, gate), s);
      hipLaunchKernelGGL((trail_fix_kernel<T>), dim3(nt, cdiv(n, 256)), dim3(256), 0, s, Qt, ldq, n, nt, W, sg, gate);
    }
    if (!positive)
      hipLaunchKernelGGL((sign_cols_kernel<T>), dim3(std::min(cdiv(m, 256), 16), n), dim3(256), 0, s, Q, ldq, m, sg,
                         gate);
  }
  const int rows = full ? m : n;
  if (R != nullptr && (rows > n || !positive))
    hipLaunchKernelGGL((sign_rows_kernel<T>), dim3(std::min(cdiv(rows, 256), 16), n), dim3(256), 0, s, R, ldr, rows, n,
                       positive ? nullptr : sg, gate);
}
template void qr_trailing_enqueue<double>(hipStream_t, int, int, double*, int64_t, double*, int64_t, int, int, char*);
template void qr_trailing_enqueue<zd>(hipStream_t, int, int, zd*, int64_t, zd*, int64_t, int, int, char*);

}  // namespace mak
