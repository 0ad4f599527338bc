// Reverse-mode rules of qr_compact! and left_polar! on MI355X, for a batch of
// equally sized matrices (strided storage, every product a batched MFMA GEMM).
//
// qr_pullback! (MatrixAlgebraKit src/pullbacks/qr.jl:73-120), rank p:
//   dQ1 -= Q1 (dR12 R12^H), dA2 += Q1 dR12                    (n > p)
//   M = triu(dR11) R11^H - Q1^H dQ1 ; M <- copyltu(M) (real diagonal)
//   dA1 += (dQ1 + Q1 M) R11^{-H}
// with Q1 = ([I; 0] - V T V_1^H) D from the compact WY factors kept by the
// primal (V strictly below the diagonal of A_wy, one 32x32 T per panel, merged
// here; D the gauge signs).  Q1 itself is never formed: with N = dR12 R12^H,
//   Z = V^H dQ1,  Q1^H dQ1 = D^H (dQ1_top - V_1 T^H Z)
//   B = D [(M - N) R11^{-H}, dR12],  G = T V_1^H B
//   dA += dQ1 [R11^{-H}, 0] + [B; 0] - V G
// Four products with m rows (V^H V, V^H dQ, dQ R^{-H}, V G) and a dozen n x n
// ones, where forming Q1 panel by panel took a pass over all of it per 32
// columns and three more products: 256 x (2048 x 256) Float64 10.0 -> 7.0 ms.
// left_polar_pullback! (src/pullbacks/polar.jl:7-29):
//   dP <- herm(dP) ; M = W^H dW - dP P ; solve P C + C P = M - M^H
//   dA += W (C + dP) + (dW - W W^H dW) P^{-1}
// The Sylvester equation (LinearAlgebra.sylvester in the reference,
// src/common/pullbacks.jl:15) is solved by preconditioned conjugate gradients
// on the SPD operator C -> P C + C P (diagonal preconditioner
// 1 / (P_ii + P_jj)); P^{-1} comes from a batched Cholesky factorisation.
// A well-conditioned batch (the usual case: tall matrices) takes the doubling
// solver of polar_pullback_doubling instead, a dozen n x n products.
// CG needs about sqrt(cond(P)) steps: when it has not converged after
// kPcgFirst steps, the batch is solved exactly through the eigendecomposition
// P = Z diag(lambda) Z^H (rocSOLVER syevd / heevd, batched):
//   C = Z [(Z^H F Z)_ij / (lambda_i + lambda_j)] Z^H,  P^{-1} = Z diag(1/lambda) Z^H,
// whose accuracy does not depend on cond(P).
#include <algorithm>
#include <cmath>
#include <vector>

#include "mak_common.hpp"
#include "mak_dense32.hpp"
#include "mak_gj.hpp"
#include "mak_kernels.hpp"
#include "mak_mi355x_internal.hpp"

namespace mak {

bool eigh_available();
size_t eigh_workspace_bytes(int n, int batch);
template <typename T>
int eigh_batched(hipStream_t s, int n, T* A, int64_t lda, int64_t strideA, double* D, int64_t strideD, int batch,
                 char* ws);

namespace {

constexpr int NB = 32;
constexpr int DBK = 64;
constexpr int kPcgFirst = 48;  // CG steps before the eigendecomposition takes over

inline size_t al256(size_t b) { return ((b + 255) / 256) * 256; }

template <typename T> GemmArgs bga(int batch, int M, int N, int K, const T* A, int64_t lda, int64_t sA, const T* B,
                                   int64_t ldb, int64_t sB, T* C, int64_t ldc, int64_t sC, double alpha,
                                   double beta) {
  GemmArgs g{};
  g.M = M; g.N = N; g.K = K;
  g.A = A; g.lda = lda; g.strideA = sA;
  g.B = B; g.ldb = ldb; g.strideB = sB;
  g.C = C; g.ldc = ldc; g.strideC = sC;
  g.alpha_re = alpha; g.beta_re = beta;
  g.ksplit = 1; g.kchunk = K; g.batch = batch;
  return g;
}

inline dim3 egrid(int64_t per, int batch) { return dim3((unsigned)cdiv64(std::max<int64_t>(per, 1), 256), 1, batch); }

// ------------------------------------------------------------------ helpers
template <typename T>
__global__ void bcopy_kernel(int m, int n, const T* X, int64_t ldx, int64_t sx, T* Y, int64_t ldy, int64_t sy) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int r = (int)(idx % m), c = (int)(idx / m);
  Y[blockIdx.z * sy + r + c * ldy] = X[blockIdx.z * sx + r + c * ldx];
}
template <typename T>
__global__ void bfill_kernel(int m, int n, T* Y, int64_t ldy, int64_t sy, int ident) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int r = (int)(idx % m), c = (int)(idx / m);
  Y[blockIdx.z * sy + r + c * ldy] = (ident && r == c) ? s_one(T()) : s_zero(T());
}
// Y = triu(X) (p x n block)
template <typename T>
__global__ void btriu_kernel(int m, int n, const T* X, int64_t ldx, int64_t sx, T* Y, int64_t ldy, int64_t sy) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int r = (int)(idx % m), c = (int)(idx / m);
  Y[blockIdx.z * sy + r + c * ldy] = (r <= c) ? X[blockIdx.z * sx + r + c * ldx] : s_zero(T());
}
// Y = (X + X^H) / 2
template <typename T>
__global__ void bherm_kernel(int n, const T* X, int64_t ldx, int64_t sx, T* Y, int64_t ldy, int64_t sy) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)n * n) return;
  const int r = (int)(idx % n), c = (int)(idx / n);
  const T* Xb = X + blockIdx.z * sx;
  Y[blockIdx.z * sy + r + c * ldy] = s_scale(s_add(Xb[r + c * ldx], s_conj(Xb[c + r * ldx])), 0.5);
}
// F = M - M^H
template <typename T>
__global__ void bskew2_kernel(int n, const T* M, int64_t ldm, int64_t sm, T* F, int64_t ldf, int64_t sf) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)n * n) return;
  const int r = (int)(idx % n), c = (int)(idx / n);
  const T* Mb = M + blockIdx.z * sm;
  F[blockIdx.z * sf + r + c * ldf] = s_sub(Mb[r + c * ldm], s_conj(Mb[c + r * ldm]));
}
// Y += a X
template <typename T>
__global__ void baxpy_kernel(int m, int n, double a, const T* X, int64_t ldx, int64_t sx, T* Y, int64_t ldy,
                             int64_t sy) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int r = (int)(idx % m), c = (int)(idx / m);
  T* y = Y + blockIdx.z * sy + r + c * ldy;
  *y = s_add(*y, s_scale(X[blockIdx.z * sx + r + c * ldx], a));
}
// V1 (p x p) = the unit lower top of V; T (p x p) = the panels' T blocks on the
// diagonal, zero elsewhere.
template <typename T>
__global__ void __launch_bounds__(256) bwy_tops_kernel(int p, const T* A, int64_t lda, int64_t sa, const T* Tp,
                                                       int64_t st, T* V1, T* Tm) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, pp = (int64_t)p * p;
  if (idx >= pp) return;
  const int r = (int)(idx % p), c = (int)(idx / p);
  const int64_t o = blockIdx.z * pp + idx;
  V1[o] = r > c ? A[blockIdx.z * sa + r + (int64_t)c * lda] : (r == c ? s_one(T()) : s_zero(T()));
  Tm[o] = r / NB == c / NB ? Tp[blockIdx.z * st + (int64_t)(c / NB) * NB * NB + r % NB + (c % NB) * NB] : s_zero(T());
}
// M - N with M = copyltu(A0 + N - D^H (dQ_top - Y)) (the upper part mirrored,
// real diagonal), by pairs of mirrored 32 x 32 tiles; A0, N, dQ may be null
// (zero).  sgn: d_i = sign_safe(A(i, i)) when sgn is 1, else 1.
template <typename T>
__global__ void __launch_bounds__(256) bqr_m_kernel(int p, const T* A0, const T* N, const T* dQ, int64_t lddq,
                                                    int64_t sdq, const T* Y, const T* A, int64_t lda, int64_t sa,
                                                    int sgn, T* Out) {
  __shared__ T tile[32][33];
  if (blockIdx.x > blockIdx.y) return;
  const int r0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  const int64_t o = (int64_t)blockIdx.z * p * p;
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int i = r0 + e % 32, j = c0 + e / 32;
    T v = s_zero(T());
    if (i < p && j < p && i <= j) {
      const int64_t x = o + i + (int64_t)j * p;
      const T n = N != nullptr ? N[x] : s_zero(T());
      if (A0 != nullptr) v = A0[x];
      v = s_add(v, n);
      if (dQ != nullptr) {
        T q = s_sub(dQ[blockIdx.z * sdq + i + (int64_t)j * lddq], Y[x]);
        if (sgn) q = s_mul(s_conj(sign_safe(A[blockIdx.z * sa + i + (int64_t)i * lda])), q);
        v = s_sub(v, q);
      }
      if (i == j) v = s_from_real<T>(s_re(v));
      Out[x] = s_sub(v, n);
    }
    tile[e % 32][e / 32] = v;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int i = c0 + e % 32, j = r0 + e / 32;  // the mirrored entry, i > j
    if (i < p && j < p && i > j) {
      const int64_t x = o + i + (int64_t)j * p;
      T v = s_conj(tile[e / 32][e % 32]);
      if (N != nullptr) v = s_sub(v, N[x]);
      Out[x] = v;
    }
  }
}
// B (p x n, packed) = D [E, dR12] (dR12 null: zero) and dA_top += B.
template <typename T>
__global__ void __launch_bounds__(256) bqr_b_kernel(int p, int n, const T* E, const T* dR, int64_t lddr, int64_t sdr,
                                                    const T* A, int64_t lda, int64_t sa, int sgn, T* B, T* dA,
                                                    int64_t ldda, int64_t sda) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p * n) return;
  const int r = (int)(idx % p), c = (int)(idx / p);
  T v = s_zero(T());
  if (c < p) v = E[(int64_t)blockIdx.z * p * p + idx];
  else if (dR != nullptr) v = dR[blockIdx.z * sdr + r + (int64_t)c * lddr];
  if (sgn) v = s_mul(sign_safe(A[blockIdx.z * sa + r + (int64_t)r * lda]), v);
  B[(int64_t)blockIdx.z * p * n + idx] = v;
  T* y = dA + blockIdx.z * sda + r + (int64_t)c * ldda;
  *y = s_add(*y, v);
}

// Inverse of a kb x kb (kb <= 64) upper-triangular diagonal block of U into Y.
// Block b of the grid's z dimension handles matrix b; the grid's x dimension
// enumerates the diagonal blocks.  Two waves invert the 32 x 32 halves by back
// substitution (lane c: column c, the rows of U read from LDS at uniform
// addresses), the off-diagonal part is -Y11 U12 Y22 on MFMA: 242 us (256
// matrices of four blocks, rank-1 steps with a barrier each) -> 36 us.
template <typename T>
__global__ void __launch_bounds__(256) btrtri_diag_kernel(int n, const T* U, int64_t ldu, int64_t su, T* Y,
                                                          int64_t ldy, int64_t sy) {
  __shared__ T Ul[3][32][33];  // U11, U22 (identity-padded), U12
  __shared__ T Yl[2][32][33];
  const int tid = threadIdx.x;
  const int k0 = blockIdx.x * DBK;
  const int kb = min(DBK, n - k0);
  const T* Ub = U + blockIdx.z * su + k0 + (int64_t)k0 * ldu;
  T* Yb = Y + blockIdx.z * sy + k0 + (int64_t)k0 * ldy;
  for (int e = tid; e < 3 * 1024; e += 256) {
    const int h = e >> 10, i = e & 31, j = (e >> 5) & 31;
    const int r = (h == 1 ? 32 : 0) + i, c = (h == 0 ? 0 : 32) + j;
    T v = s_zero(T());
    if (r < kb && c < kb && r <= c) v = Ub[r + (int64_t)c * ldu];
    else if (r == c) v = s_one(T());
    Ul[h][i][j] = v;
  }
  __syncthreads();
  const int w = tid >> 6, c = tid & 63;
  if (w < 2 && c < 32) {
    T y[32];
#pragma unroll
    for (int r = 31; r >= 0; --r) {
      T acc0 = r == c ? s_one(T()) : s_zero(T()), acc1 = s_zero(T());
#pragma unroll
      for (int k = r + 1; k < 32; ++k) {
        const T u = s_neg(Ul[w][r][k]);
        if (k & 1) acc1 = s_fma(u, y[k], acc1);
        else acc0 = s_fma(u, y[k], acc0);
      }
      y[r] = s_div(s_add(acc0, acc1), Ul[w][r][r]);
    }
#pragma unroll
    for (int r = 0; r < 32; ++r) Yl[w][r][c] = r <= c ? y[r] : s_zero(T());
  }
  __syncthreads();
  mm32<T>(Ul[2], Ul[2], false, Yl[1], false, 1.0, false);
  mm32<T>(Ul[2], Yl[0], false, Ul[2], false, -1.0, false);
  for (int e = tid; e < DBK * DBK; e += 256) {
    const int r = e % DBK, cc = e / DBK;
    if (r < kb && cc < kb) {
      T v = s_zero(T());
      if (r < 32 && cc >= 32) v = Ul[2][r][cc - 32];
      else if (r / 32 == cc / 32) v = Yl[r / 32][r % 32][cc % 32];
      Yb[r + (int64_t)cc * ldy] = v;
    }
  }
}

// X (m x kb) <- alpha X U for a kb x kb upper-triangular U (in place, batched)
template <typename T>
__global__ void __launch_bounds__(256) btrmm_kernel(T* X, int64_t ldx, int64_t sx, int m, int kb, const T* U,
                                                    int64_t ldu, int64_t su, double alpha) {
  __shared__ T Us[DBK][DBK + 1];
  __shared__ T Xs[64][DBK + 1];
  const int tid = threadIdx.x;
  const int r0 = blockIdx.x * 64;
  T* Xb = X + blockIdx.z * sx;
  const T* Ub = U + blockIdx.z * su;
  for (int i = tid; i < DBK * DBK; i += 256) {
    const int r = i % DBK, c = i / DBK;
    Us[r][c] = (r <= c && c < kb) ? Ub[r + c * ldu] : s_zero(T());
  }
  for (int i = tid; i < 64 * DBK; i += 256) {
    const int r = i % 64, c = i / 64;
    Xs[r][c] = (r0 + r < m && c < kb) ? Xb[(r0 + r) + c * ldx] : s_zero(T());
  }
  __syncthreads();
  for (int i = tid; i < 64 * DBK; i += 256) {
    const int r = i % 64, c = i / 64;
    if (r0 + r < m && c < kb) {
      T s = s_zero(T());
      for (int k = 0; k <= c; ++k) s = s_fma(Xs[r][k], Us[k][c], s);
      Xb[(r0 + r) + c * ldx] = s_scale(s, alpha);
    }
  }
}

// Y = U^{-1} for batched n x n upper-triangular U (Y fully overwritten).
template <typename T>
void btrtri_upper(int batch, int n, const T* U, int64_t ldu, int64_t su, T* Y, int64_t ldy, int64_t sy,
                  hipStream_t s) {
  hipLaunchKernelGGL((bfill_kernel<T>), egrid((int64_t)n * n, batch), dim3(256), 0, s, n, n, Y, ldy, sy, 0);
  hipLaunchKernelGGL((btrtri_diag_kernel<T>), dim3(cdiv(n, DBK), 1, batch), dim3(256), 0, s, n, U, ldu, su, Y, ldy,
                     sy);
  for (int k = DBK; k < n; k += DBK) {
    const int kb = std::min(DBK, n - k);
    T* Yc = Y + (int64_t)k * ldy;
    gemm<T>(OP_N, OP_N, bga<T>(batch, k, kb, k, Y, ldy, sy, U + (int64_t)k * ldu, ldu, su, Yc, ldy, sy, 1.0, 0.0), s);
    hipLaunchKernelGGL((btrmm_kernel<T>), dim3(cdiv(k, 64), 1, batch), dim3(256), 0, s, Yc, ldy, sy, k, kb,
                       Y + k + (int64_t)k * ldy, ldy, sy, -1.0);
  }
}

// Batched Cholesky factor kernel for one 64x64 diagonal block (upper, Z = W^H W)
template <typename T>
__global__ void __launch_bounds__(256) bpotrf_diag_kernel(T* Z, int64_t ldz, int64_t sz, int kb, int* info) {
  __shared__ T S[DBK][DBK + 1];
  __shared__ T Wl[DBK][DBK + 1];
  const int tid = threadIdx.x;
  T* Zb = Z + blockIdx.z * sz;
  for (int i = tid; i < DBK * DBK; i += 256) {
    const int r = i % DBK, c = i / DBK;
    S[r][c] = (r <= c && c < kb) ? Zb[r + c * ldz] : s_zero(T());
    Wl[r][c] = s_zero(T());
  }
  __syncthreads();
  for (int j = 0; j < kb; ++j) {
    const double d2 = s_re(S[j][j]);
    if (!(d2 > 0.0)) {
      if (tid == 0) info[0] = 1;
      break;
    }
    const double d = sqrt(d2), rd = 1.0 / d, rd2 = 1.0 / d2;
    for (int c = j + tid; c < kb; c += 256) Wl[j][c] = (c == j) ? s_from_real<T>(d) : s_scale(S[j][c], rd);
    for (int i = tid; i < DBK * DBK; i += 256) {
      const int r = i % DBK, c = i / DBK;
      if (r > j && r <= c && c < kb) S[r][c] = s_sub(S[r][c], s_scale(s_mul(s_conj(S[j][r]), S[j][c]), rd2));
    }
    __syncthreads();
  }
  __syncthreads();
  for (int i = tid; i < DBK * DBK; i += 256) {
    const int r = i % DBK, c = i / DBK;
    if (r < kb && c < kb) Zb[r + c * ldz] = (r <= c) ? Wl[r][c] : s_zero(T());
  }
}

// Batched Cholesky Z = W^H W (W upper, in place; strict lower part zeroed on the
// diagonal blocks only -- callers read the upper part).  tmp: DBK x n per matrix.
template <typename T>
void bpotrf_upper(int batch, int n, T* Z, int64_t ldz, int64_t sz, T* Ydiag, int64_t ldy, int64_t sy, T* tmp,
                  int64_t stmp, int* dinfo, hipStream_t s) {
  for (int k = 0; k < n; k += DBK) {
    const int kb = std::min(DBK, n - k);
    T* Zkk = Z + k + (int64_t)k * ldz;
    hipLaunchKernelGGL((bpotrf_diag_kernel<T>), dim3(1, 1, batch), dim3(256), 0, s, Zkk, ldz, sz, kb, dinfo);
    const int rest = n - k - kb;
    if (rest > 0) {
      // Y_kk = W_kk^{-1}
      hipLaunchKernelGGL((btrtri_diag_kernel<T>), dim3(1, 1, batch), dim3(256), 0, s, kb, Zkk, ldz, sz,
                         Ydiag, ldy, sy);
      T* Zrow = Z + k + (int64_t)(k + kb) * ldz;
      gemm<T>(OP_C, OP_N, bga<T>(batch, kb, rest, kb, Ydiag, ldy, sy, Zrow, ldz, sz, tmp, DBK, stmp, 1.0, 0.0), s);
      hipLaunchKernelGGL((bcopy_kernel<T>), egrid((int64_t)kb * rest, batch), dim3(256), 0, s, kb, rest, tmp,
                         (int64_t)DBK, stmp, Zrow, ldz, sz);
      T* Z22 = Z + (k + kb) + (int64_t)(k + kb) * ldz;
      gemm<T>(OP_C, OP_N, bga<T>(batch, rest, rest, kb, Zrow, ldz, sz, Zrow, ldz, sz, Z22, ldz, sz, -1.0, 1.0), s);
    }
  }
}

// ---- batched reductions for CG: out[b] = Re sum conj(X_b) Y_b
constexpr int kRedBlocks = 64;
template <typename T>
__global__ void __launch_bounds__(256) bdot_kernel(int m, int n, const T* X, int64_t ldx, int64_t sx, const T* Y,
                                                   int64_t ldy, int64_t sy, double* partial) {
  __shared__ double red[4];
  const int64_t tot = (int64_t)m * n;
  const T* Xb = X + blockIdx.z * sx;
  const T* Yb = Y + blockIdx.z * sy;
  double acc = 0.0;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < tot; idx += (int64_t)gridDim.x * 256) {
    const int r = (int)(idx % m), c = (int)(idx / m);
    acc += s_re(s_cfma(Xb[r + c * ldx], Yb[r + c * ldy], s_zero(T())));
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.z * kRedBlocks + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}
__global__ void bsum_kernel(const double* partial, double* out) {
  const int b = blockIdx.x;
  double acc = 0.0;
  for (int i = threadIdx.x; i < kRedBlocks; i += 64) acc += partial[b * kRedBlocks + i];
  acc = wave_sum(acc);
  if (threadIdx.x == 0) out[b] = acc;
}
template <typename T>
void bdot(int batch, int m, int n, const T* X, int64_t ldx, int64_t sx, const T* Y, int64_t ldy, int64_t sy,
          double* partial, double* out, hipStream_t s) {
  hipLaunchKernelGGL((bdot_kernel<T>), dim3(kRedBlocks, 1, batch), dim3(256), 0, s, m, n, X, ldx, sx, Y, ldy, sy,
                     partial);
  hipLaunchKernelGGL(bsum_kernel, dim3(batch), dim3(64), 0, s, partial, out);
}
// Z = R ./ (P_ii + P_jj)
template <typename T>
__global__ void bprecond_kernel(int n, const T* R, const T* P, int64_t ldp, int64_t sp, T* Z) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)n * n) return;
  const int r = (int)(idx % n), c = (int)(idx / n);
  const T* Pb = P + blockIdx.z * sp;
  const double d = s_re(Pb[r + r * ldp]) + s_re(Pb[c + c * ldp]);
  const int64_t o = blockIdx.z * (int64_t)n * n + r + (int64_t)c * n;
  Z[o] = s_scale(R[o], 1.0 / d);
}
// X += a D ; R -= a Q   with a = rz[b] / dq[b]
template <typename T>
__global__ void bcg_step_kernel(int nn, const double* rz, const double* dq, const T* D, const T* Qm, T* X, T* R) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= nn) return;
  const int b = blockIdx.z;
  const double a = (dq[b] != 0.0) ? rz[b] / dq[b] : 0.0;
  const int64_t o = (int64_t)b * nn + idx;
  X[o] = s_add(X[o], s_scale(D[o], a));
  R[o] = s_sub(R[o], s_scale(Qm[o], a));
}
// D = Z + (rz_new[b] / rz[b]) D
template <typename T>
__global__ void bcg_dir_kernel(int nn, const double* rznew, const double* rz, const T* Z, T* D) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= nn) return;
  const int b = blockIdx.z;
  const double beta = (rz[b] != 0.0) ? rznew[b] / rz[b] : 0.0;
  const int64_t o = (int64_t)b * nn + idx;
  D[o] = s_add(Z[o], s_scale(D[o], beta));
}

// ---------------------------------------------------------------------------
// Doubling (Smith's method) for P C + C P = F with P Hermitian positive
// definite.  With s > 0, G = (P + s I)^{-1}, N = 2 s G and M = I - N =
// G (P - s I), the equation is C - M C M = N (F / (2 s)) N, so
//   C = sum_k M^k C_0 M^k,   C_0 = N (F / (2 s)) N,
// and each step doubles the number of terms: C += M C M, M <- M^2.  |M| =
// max |lambda - s| / (lambda + s) < 1; for s = tr(P) / n and the spectra of
// tall Gaussian matrices it is about 0.2, and four steps reach 1e-16 (11
// products) where CG takes 20 steps of two products and six passes over n x n
// arrays.  P^{-1} and G come from one batch of 2 batch Gauss-Jordan
// eliminations.  left_polar_pullback 256 x (2048 x 256) Float64: 27.3 ms with
// CG (the solve 18 ms), 10.2 ms with the doubling (the solve 2.5 ms, the
// inverses 2.1 ms, the products with W and dW 4.2 ms).
// ---------------------------------------------------------------------------

// tr(X_b) / n (real part) to out[b].
template <typename T>
__global__ void __launch_bounds__(64) bmean_diag_kernel(int n, const T* X, int64_t ldx, int64_t sx, double* out) {
  const T* x = X + blockIdx.x * sx;
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 64) acc += s_re(x[i + (int64_t)i * ldx]);
  acc = wave_sum(acc);
  if (threadIdx.x == 0) out[blockIdx.x] = acc / n;
}

// The matrix z of the batch of 2 batch inverses before its first step: P_z, or
// P_{z - batch} + s I.
template <typename T> struct SpdGjArgs {
  const T* P;
  int64_t ldp, sp;
  const double* shift;  // s of each matrix
  int batch, n, k;
  const T* src;         // before step k > 0: n x n each, packed
  T* dst;               // after it
  T* Pd;                // 32 x 32 inverses of the diagonal blocks: two per matrix, alternating
  int* info;            // set to 1 when a diagonal block is not positive definite
};
template <typename T> __device__ __forceinline__ T spd_elem(const SpdGjArgs<T>& a, int z, int i, int j) {
  if (i >= a.n || j >= a.n) return i == j ? s_one(T()) : s_zero(T());
  if (a.k > 0) return a.src[(int64_t)z * a.n * a.n + i + (int64_t)j * a.n];
  const int b = z < a.batch ? z : z - a.batch;
  const T v = a.P[b * a.sp + i + (int64_t)j * a.ldp];
  return z >= a.batch && i == j ? s_add(v, s_from_real<T>(a.shift[b])) : v;
}
// By one wave: Pn (32 x 32, column-major, global) = A^{-1} = Y Y^H with A = W^H W,
// Y = W^{-1}; A, Y in LDS.
template <typename T>
__device__ __forceinline__ void wave_spd_inv32(T (*A)[33], T (*Y)[33], T* Pn, int* info) {
  if (wave_chol_inv32<T>(A, Y) != 0 && lane_id() == 0) *info = 1;
  const int l = lane_id(), c = l & 15, q = l >> 4;
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj) {
      v4d re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll
      for (int kk = 16 * (bi > bj ? bi : bj); kk < 32; kk += 4)  // Y is upper triangular
        mfma_acc(re, im, Y[16 * bi + c][kk + q], s_conj(Y[16 * bj + c][kk + q]));
#pragma unroll
      for (int u = 0; u < 4; ++u) Pn[16 * bi + 4 * u + q + 32 * (16 * bj + c)] = acc_get<T>(re, im, u);
    }
}
template <typename T> __global__ void __launch_bounds__(64) spd_gj_first_kernel(SpdGjArgs<T> a) {
  __shared__ T A[GB][33], Y[GB][33];
  const int z = blockIdx.x;
  for (int e = threadIdx.x; e < GB * GB; e += 64) A[e % GB][e / GB] = spd_elem(a, z, e % GB, e / GB);
  __syncthreads();
  wave_spd_inv32<T>(A, Y, a.Pd + (int64_t)z * 2 * GB * GB, a.info);
}
template <typename T> __global__ void __launch_bounds__(256) spd_gj_step_kernel(SpdGjArgs<T> a) {
  const int z = blockIdx.z;
  T* Pd = a.Pd + (int64_t)z * 2 * GB * GB;
  const int cur = a.k & 1;
  gj_tile_step<T>(
      a.n, a.k, blockIdx.x * GT, blockIdx.y * GT, Pd + cur * GB * GB, a.dst + (int64_t)z * a.n * a.n, a.n,
      [&](int i, int j) { return spd_elem(a, z, i, j); },
      [&](T (*A)[33], T (*Y)[33]) { wave_spd_inv32<T>(A, Y, Pd + (1 - cur) * GB * GB, a.info); });
}

// Out = (D - D^H) / (2 s_b) with D = K - T1 (T1 null: D = K); 32 x 32 tiles.
template <typename T>
__global__ void __launch_bounds__(256) bskew_scaled_kernel(int n, const T* K, const T* T1, const double* sh, T* Out) {
  __shared__ T Dt[32][33];
  const int64_t o = (int64_t)blockIdx.z * n * n;
  const int r0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  const double f = 0.5 / sh[blockIdx.z];
  auto at = [&](int i, int j) {
    const int64_t x = o + i + (int64_t)j * n;
    return T1 != nullptr ? s_sub(K[x], T1[x]) : K[x];
  };
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int i = c0 + e % 32, j = r0 + e / 32;  // the mirrored tile
    Dt[e % 32][e / 32] = (i < n && j < n) ? at(i, j) : s_zero(T());
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 1024; e += 256) {
    const int i = r0 + e % 32, j = c0 + e / 32;
    if (i < n && j < n) Out[o + i + (int64_t)j * n] = s_scale(s_sub(at(i, j), s_conj(Dt[e / 32][e % 32])), f);
  }
}
// N = 2 s_b G (in place) and M = I - N.
template <typename T>
__global__ void __launch_bounds__(256) bcayley_kernel(int n, T* G, T* M, const double* sh) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, nn = (int64_t)n * n;
  if (idx >= nn) return;
  const int64_t o = blockIdx.z * nn + idx;
  const T v = s_scale(G[o], 2.0 * sh[blockIdx.z]);
  G[o] = v;
  M[o] = s_sub(idx % n == idx / n ? s_one(T()) : s_zero(T()), v);
}

// The quotient q = tr(P) tr(P^{-1}) / n^2 (1 for P = c I; a tall Gaussian matrix
// of 2 n rows has 1.6) decides on the doubling solver.  P / s has its eigenvalues
// in [1 / (n q), n], so |M| <= 1 - 2 / (n q + 1), and the stop test, n^2
// |M|^(2^(K+1)) <= kDoublingRem, holds after at most kDoublingMax steps for n q up
// to kDoublingMaxSpread: a batch that is taken is finished by it, at a third of
// the products of CG and the eigendecomposition at worst.  q alone allows a
// condition number of 16 n for one small eigenvalue and of 16 n^2 for one large
// and one small one; error and residual there stay those of the
// eigendecomposition (u times the condition number).
constexpr double kDoublingMaxCond = 16.0, kDoublingMaxSpread = 16384.0;
constexpr int kDoublingMax = 18;
// Relative remainder |M^(2^K)|^2 after K steps, bounded by |M^(2^(K-1))|_F^4.
constexpr double kDoublingRem = 1e-17;
constexpr double kDoublingMinTol = 1e-15;  // requests below it keep the CG path's own test

// out[b] = |X_b|_F^2 (packed n x n): one workgroup per matrix.
template <typename T> __global__ void __launch_bounds__(256) bfro2_kernel(int64_t nn, const T* X, double* out) {
  __shared__ double red[4];
  const T* x = X + blockIdx.x * nn;
  double a0 = 0.0, a1 = 0.0;
  int64_t i = threadIdx.x;
  for (; i + 256 < nn; i += 512) {
    a0 += s_abs2(x[i]);
    a1 += s_abs2(x[i + 256]);
  }
  if (i < nn) a0 += s_abs2(x[i]);
  a0 = wave_sum(a0 + a1);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a0;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// dA += left_polar_pullback for dW given (dP may be null) on a well-conditioned
// batch; buf: ten consecutive buffers of batch n x n matrices (each a multiple
// of 256 bytes), Pd: 4096 elements per matrix, sc: 2 batch doubles.  Returns 0
// when done (steps to *iters), 1 when the batch does not qualify (nothing
// written to dA), 2 for a HIP error.
template <typename T>
int polar_pullback_doubling(hipStream_t s, int batch, int m, int n, const T* W, int64_t ldw, int64_t sw, const T* P,
                            int64_t ldp, int64_t sp, const T* dW, int64_t lddw, int64_t sdw, const T* dP,
                            int64_t lddp, int64_t sdp, T* dA, int64_t ldda, int64_t sda, T* const (&buf)[10], T* Pd,
                            double* sc, int* dinfo, int* iters) {
  const int64_t nn = (int64_t)n * n;
  const dim3 gnn = egrid(nn, batch);
  T *dPh = buf[0], *K = buf[1], *Tm = buf[2], *X = buf[3];
  double *shift = sc, *mean = sc + batch;
  auto prod = [&](int opA, int opB, const T* A, const T* B, T* C, double alpha, double beta) {
    gemm<T>(opA, opB, bga<T>(batch, n, n, n, A, n, nn, B, n, nn, C, n, nn, alpha, beta), s);
  };
  // P^{-1} and (P + s I)^{-1}, s = tr(P) / n
  zero_ints(dinfo, 1, s);
  hipLaunchKernelGGL((bmean_diag_kernel<T>), dim3(batch), dim3(64), 0, s, n, P, ldp, sp, shift);
  SpdGjArgs<T> a{P, ldp, sp, shift, batch, n, 0, nullptr, nullptr, Pd, dinfo};
  T* pair[2] = {buf[4], buf[6]};
  hipLaunchKernelGGL((spd_gj_first_kernel<T>), dim3(2 * batch), dim3(64), 0, s, a);
  const int nb = cdiv(n, GB), tiles = cdiv(n, GT);
  for (int k = 0; k < nb; ++k) {
    a.k = k;
    a.dst = pair[k & 1];
    hipLaunchKernelGGL((spd_gj_step_kernel<T>), dim3(tiles, tiles, 2 * batch), dim3(256), 0, s, a);
    a.src = a.dst;
  }
  T* Pinv = pair[(nb - 1) & 1];
  T* N = Pinv + batch * nn;
  T *Ma = pair[nb & 1], *Mb = buf[8], *F = buf[9];
  hipLaunchKernelGGL((bmean_diag_kernel<T>), dim3(batch), dim3(64), 0, s, n, (const T*)Pinv, (int64_t)n, nn, mean);
  // meanwhile K = W^H dW, F' = skew(K - herm(dP) P) / (2 s)
  gemm<T>(OP_C, OP_N, bga<T>(batch, n, n, m, W, ldw, sw, dW, lddw, sdw, K, n, nn, 1.0, 0.0), s);
  if (dP) {
    hipLaunchKernelGGL((bherm_kernel<T>), gnn, dim3(256), 0, s, n, dP, lddp, sdp, dPh, (int64_t)n, nn);
    gemm<T>(OP_N, OP_N, bga<T>(batch, n, n, n, dPh, n, nn, P, ldp, sp, Tm, n, nn, 1.0, 0.0), s);
  }
  std::vector<double> h(2 * (size_t)batch);
  int hinfo = 0;
  if (hipMemcpyAsync(h.data(), sc, h.size() * sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipMemcpyAsync(&hinfo, dinfo, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return 2;
  if (hinfo != 0) return 1;
  for (int b = 0; b < batch; ++b)
    if (!(h[b] > 0.0) || !(h[b] * h[batch + b] <= std::min(kDoublingMaxCond, kDoublingMaxSpread / n))) return 1;
  hipLaunchKernelGGL((bskew_scaled_kernel<T>), dim3(cdiv(n, 32), cdiv(n, 32), batch), dim3(256), 0, s, n, K,
                     dP ? (const T*)Tm : nullptr, (const double*)shift, F);
  hipLaunchKernelGGL((bcayley_kernel<T>), gnn, dim3(256), 0, s, n, N, Ma, (const double*)shift);
  prod(OP_N, OP_N, F, N, Tm, 1.0, 0.0);
  prod(OP_N, OP_N, N, Tm, X, 1.0, 0.0);
  int k = 0;
  for (bool done = false; !done && k < kDoublingMax;) {
    hipLaunchKernelGGL((bfro2_kernel<T>), dim3(batch), dim3(256), 0, s, nn, (const T*)Ma, mean);
    if (hipMemcpyAsync(h.data(), mean, batch * sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess) return 2;
    prod(OP_N, OP_N, X, Ma, Tm, 1.0, 0.0);  // C += M C M
    prod(OP_N, OP_N, Ma, Tm, X, 1.0, 1.0);
    ++k;
    if (hipStreamSynchronize(s) != hipSuccess) return 2;
    done = true;
    for (int b = 0; b < batch; ++b) done = done && h[b] * h[b] <= kDoublingRem;  // false for NaN
    if (!done && k < kDoublingMax) {
      prod(OP_N, OP_N, Ma, Ma, Mb, 1.0, 0.0);
      std::swap(Ma, Mb);
    } else if (!done) {
      return 1;
    }
  }
  *iters = k;
  // dA += W (C + dPh) + (dW - W K) P^{-1} = W (C + dPh - K P^{-1}) + dW P^{-1}
  if (dP)
    hipLaunchKernelGGL((baxpy_kernel<T>), gnn, dim3(256), 0, s, n, n, 1.0, dPh, (int64_t)n, nn, X, (int64_t)n, nn);
  prod(OP_N, OP_N, K, Pinv, X, -1.0, 1.0);
  GemmArgs g = bga<T>(batch, m, n, n, W, ldw, sw, X, n, nn, dA, ldda, sda, 1.0, 1.0);
  g.A2 = dW;
  g.lda2 = lddw;
  g.strideA2 = sdw;
  g.B2 = Pinv;
  g.ldb2 = n;
  g.strideB2 = nn;
  gemm_dual<T>(g, s);
  return 0;
}

}  // namespace

// ---------------------------------------------------------------------------
// workspace layouts
// ---------------------------------------------------------------------------
template <typename T> size_t qr_pullback_ws(int batch, int m, int n) {
  const size_t k = std::min(m, n);
  return al256((size_t)batch * k * k * sizeof(T)) * 10     // V1, S, T, triu(R11), R11^{-1}, N, A0, M, two scratch
         + al256((size_t)batch * k * n * sizeof(T)) * 2;   // B, G
}
// out[b] = max(out[b], max |X_ij|) over a rows x cols block of matrix b
// (upper = 1: only i <= j), by a grid-stride loop per batch member and an
// integer atomic max on the bit patterns (monotone for non-negative doubles).
template <typename T>
__global__ void bmaxabs_kernel(int rows, int cols, const T* X, int64_t ldx, int64_t sx, int upper, double* out) {
  __shared__ double red[256];
  const T* x = X + (int64_t)blockIdx.z * sx;
  const int64_t tot = (int64_t)rows * cols;
  double v = 0.0;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < tot; e += (int64_t)gridDim.x * 256) {
    const int r = (int)(e % rows), c = (int)(e / rows);
    if (!upper || r <= c) v = fmax(v, sqrt(s_abs2(x[r + (int64_t)c * ldx])));
  }
  red[threadIdx.x] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    atomicMax(reinterpret_cast<unsigned long long*>(out + blockIdx.z), (unsigned long long)__double_as_longlong(red[0]));
}
__global__ void bzero_doubles_kernel(double* p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0.0;
}
template <typename T>
void bmaxabs(int batch, int rows, int cols, const T* X, int64_t ldx, int64_t sx, int upper, double* out,
             hipStream_t s) {
  if (batch <= 0 || rows <= 0 || cols <= 0 || X == nullptr) return;
  const int64_t tot = (int64_t)rows * cols;
  const unsigned gx = (unsigned)std::min<int64_t>(cdiv64(tot, 256), 64);
  hipLaunchKernelGGL((bmaxabs_kernel<T>), dim3(gx, 1, batch), dim3(256), 0, s, rows, cols, X, ldx, sx, upper, out);
}

template <typename T>
__global__ void bsylv_divide_kernel(int n, T* X, int64_t ldx, int64_t sx, const double* lam, int64_t sl) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * n) return;
  const int r = (int)(idx % n), c = (int)(idx / n);
  const double* l = lam + (int64_t)blockIdx.z * sl;
  T* x = X + (int64_t)blockIdx.z * sx + r + (int64_t)c * ldx;
  *x = s_scale(*x, 1.0 / (l[r] + l[c]));
}
template <typename T>
__global__ void bscale_cols_inv_kernel(int m, int n, T* X, int64_t ldx, int64_t sx, const double* lam, int64_t sl) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int r = (int)(idx % m), c = (int)(idx / m);
  T* x = X + (int64_t)blockIdx.z * sx + r + (int64_t)c * ldx;
  *x = s_scale(*x, 1.0 / lam[(int64_t)blockIdx.z * sl + c]);
}

template <typename T> size_t polar_pullback_ws(int batch, int m, int n) {
  size_t b = 0;
  const size_t nn = al256((size_t)batch * n * n * sizeof(T));
  b += al256((size_t)batch * n * sizeof(double)) + al256(eigh_workspace_bytes(n, std::max(batch, 1)));  // lambda
  b += nn * 10;                                        // dPh, M, F, X, R, Z, D, Qm, Pc, Pinv
  b += al256((size_t)batch * m * n * sizeof(T));      // Zw = dW - W W^H dW
  b += al256((size_t)batch * DBK * n * sizeof(T));    // Cholesky scratch
  b += al256((size_t)batch * DBK * DBK * sizeof(T) * cdiv(n, DBK) + 256);
  b += al256((size_t)batch * kRedBlocks * sizeof(double)) + al256((size_t)batch * 4 * sizeof(double));
  b += 256;
  return b;
}

template <typename T>
int qr_pullback(hipStream_t s, int batch, int m, int n, int p, int positive, const T* A, int64_t lda, int64_t sa,
                const T* Tp, int64_t st, const T* R, int64_t ldr, int64_t sr, const T* dQ, int64_t lddq, int64_t sdq,
                const T* dR, int64_t lddr, int64_t sdr, T* dA, int64_t ldda, int64_t sda, void* work, size_t wbytes,
                double* gauge_out) {
  if (batch < 0) return -2;
  if (m < 0) return -3;
  if (n < 0) return -4;
  const int k = std::min(m, n);
  if (p < 0 || p > k) return -5;
  if (lda < std::max(1, m)) return -8;
  if (ldr < std::max(1, k)) return -13;
  if (dQ && lddq < std::max(1, m)) return -16;
  if (dR && lddr < std::max(1, k)) return -19;
  if (ldda < std::max(1, m)) return -22;
  if (work == nullptr && batch > 0 && p > 0) return -24;
  if (wbytes < qr_pullback_ws<T>(batch, m, n)) return -25;
  if (gauge_out && batch > 0) {
    // the gauge-dependent part of the cotangents (src/pullbacks/qr.jl:27-29,
    // :34-47): dQ[:, p:k] and the upper triangle of dR[p:k, p:n]
    hipLaunchKernelGGL(bzero_doubles_kernel, dim3(cdiv(batch, 256)), dim3(256), 0, s, gauge_out, batch);
    if (dQ) bmaxabs<T>(batch, m, k - p, dQ + (int64_t)p * lddq, lddq, sdq, 0, gauge_out, s);
    if (dR) bmaxabs<T>(batch, k - p, n - p, dR + p + (int64_t)p * lddr, lddr, sdr, 1, gauge_out, s);
  }
  if (batch == 0 || p == 0) return 0;
  char* w = reinterpret_cast<char*>(work);
  auto take = [&](size_t elems) { char* q = w; w += al256(elems * sizeof(T)); return reinterpret_cast<T*>(q); };
  const int64_t pp = (int64_t)p * p;
  const size_t bk = (size_t)batch * k * k;
  T *V1 = take(bk), *S = take(bk), *Tm = take(bk), *Ru = take(bk), *Rinv = take(bk), *N = take(bk), *A0 = take(bk),
    *M = take(bk), *X1 = take(bk), *X2 = take(bk);
  T *B = take((size_t)batch * k * n), *G = take((size_t)batch * k * n);
  const dim3 gpp = egrid(pp, batch);
  auto prod = [&](int opA, int opB, const T* X, const T* Y, T* C, double alpha, double beta, int tri) {
    GemmArgs g = bga<T>(batch, p, p, p, X, p, pp, Y, p, pp, C, p, pp, alpha, beta);
    g.tri = tri;
    gemm<T>(opA, opB, g, s);
  };
  // V_1, S = V^H V (upper) and the merged T: T(0:j, b) = -T(0:j, 0:j) S(0:j, b) T_b
  hipLaunchKernelGGL((bwy_tops_kernel<T>), gpp, dim3(256), 0, s, p, A, lda, sa, Tp, st, V1, Tm);
  if (p > NB) {
    GemmArgs g = bga<T>(batch, p, p, m - p, A + p, lda, sa, A + p, lda, sa, S, p, pp, 1.0, 0.0);
    g.upperC = 1;
    gemm<T>(OP_C, OP_N, g, s);
    g = bga<T>(batch, p, p, p, V1, p, pp, V1, p, pp, S, p, pp, 1.0, 1.0);
    g.upperC = 1;
    gemm<T>(OP_C, OP_N, g, s);
  }
  for (int j = NB; j < p; j += NB) {
    const int nb = std::min(NB, p - j);
    gemm<T>(OP_N, OP_N, bga<T>(batch, j, nb, nb, S + (int64_t)j * p, p, pp, Tm + j + (int64_t)j * p, p, pp, X1, p, pp,
                               1.0, 0.0), s);
    gemm<T>(OP_N, OP_N, bga<T>(batch, j, nb, j, Tm, p, pp, X1, p, pp, Tm + (int64_t)j * p, p, pp, -1.0, 0.0), s);
  }
  // R11^{-1}: only the upper triangle of R is read (UpperTriangular(R11), src/pullbacks/qr.jl:92)
  btrtri_upper<T>(batch, p, R, ldr, sr, Rinv, p, pp, s);
  const bool wide = dR != nullptr && n > p;
  if (dR) {  // A0 = triu(dR11) R11^H ; N = dR12 R12^H
    hipLaunchKernelGGL((btriu_kernel<T>), gpp, dim3(256), 0, s, p, p, dR, lddr, sdr, X1, (int64_t)p, pp);
    hipLaunchKernelGGL((btriu_kernel<T>), gpp, dim3(256), 0, s, p, p, R, ldr, sr, Ru, (int64_t)p, pp);
    prod(OP_N, OP_C, X1, Ru, A0, 1.0, 0.0, TRI_A_UPPER | TRI_B_LOWER);
    if (wide)
      gemm<T>(OP_N, OP_C, bga<T>(batch, p, p, n - p, dR + (int64_t)p * lddr, lddr, sdr, R + (int64_t)p * ldr, ldr, sr,
                                 N, p, pp, 1.0, 0.0), s);
  }
  if (dQ) {  // X2 = V_1 T^H (V^H dQ1)
    GemmArgs g = bga<T>(batch, p, p, m, A, lda, sa, dQ, lddq, sdq, X1, p, pp, 1.0, 0.0);
    g.unitLowerA = 1;
    gemm<T>(OP_C, OP_N, g, s);
    prod(OP_C, OP_N, Tm, X1, S, 1.0, 0.0, TRI_A_LOWER);
    prod(OP_N, OP_N, V1, S, X2, 1.0, 0.0, TRI_A_LOWER);
  }
  hipLaunchKernelGGL((bqr_m_kernel<T>), dim3(cdiv(p, 32), cdiv(p, 32), batch), dim3(256), 0, s, p,
                     dR ? (const T*)A0 : nullptr, wide ? (const T*)N : nullptr, dQ, lddq, sdq, (const T*)X2, A, lda, sa,
                     positive, M);
  // B = D [(M - N) R11^{-H}, dR12], dA_top += B, G = T V_1^H B
  prod(OP_N, OP_C, M, Rinv, X1, 1.0, 0.0, TRI_B_LOWER);
  const int nc = wide ? n : p;
  hipLaunchKernelGGL((bqr_b_kernel<T>), egrid((int64_t)p * nc, batch), dim3(256), 0, s, p, nc, (const T*)X1, dR, lddr,
                     sdr, A, lda, sa, positive, B, dA, ldda, sda);
  const int64_t pc = (int64_t)p * nc;
  {
    GemmArgs g = bga<T>(batch, p, nc, p, V1, p, pp, B, p, pc, G, p, pc, 1.0, 0.0);
    g.tri = TRI_A_UPPER;
    gemm<T>(OP_C, OP_N, g, s);
    g = bga<T>(batch, p, nc, p, Tm, p, pp, G, p, pc, B, p, pc, 1.0, 0.0);
    g.tri = TRI_A_UPPER;
    gemm<T>(OP_N, OP_N, g, s);
  }
  // dA += dQ1 [R11^{-H}, 0] - V G
  if (dQ) {
    GemmArgs g = bga<T>(batch, m, p, p, dQ, lddq, sdq, Rinv, p, pp, dA, ldda, sda, 1.0, 1.0);
    g.tri = TRI_B_LOWER;
    gemm<T>(OP_N, OP_C, g, s);
  }
  {
    GemmArgs g = bga<T>(batch, m, nc, p, A, lda, sa, B, p, pc, dA, ldda, sda, -1.0, 1.0);
    g.unitLowerA = 1;
    gemm<T>(OP_N, OP_N, g, s);
  }
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

template <typename T>
int polar_pullback(hipStream_t s, int batch, int m, int n, const T* W, int64_t ldw, int64_t sw, const T* P,
                   int64_t ldp, int64_t sp, const T* dW, int64_t lddw, int64_t sdw, const T* dP, int64_t lddp,
                   int64_t sdp, T* dA, int64_t ldda, int64_t sda, int maxiter, double tol, void* work, size_t wbytes,
                   int* iters_out) {
  if (batch < 0) return -2;
  if (m < n) return -3;
  if (n < 0) return -4;
  if (ldw < std::max(1, m)) return -6;
  if (ldp < std::max(1, n)) return -9;
  if (dW && lddw < std::max(1, m)) return -12;
  if (dP && lddp < std::max(1, n)) return -15;
  if (ldda < std::max(1, m)) return -18;
  if (work == nullptr && batch > 0 && n > 0) return -22;
  if (wbytes < polar_pullback_ws<T>(batch, m, n)) return -23;
  if (batch == 0 || n == 0) return 0;
  if (maxiter <= 0) maxiter = 200;
  if (!(tol > 0.0)) tol = 1e-14;
  char* w = reinterpret_cast<char*>(work);
  auto take = [&](size_t bytes) { char* q = w; w += al256(bytes); return q; };
  const int64_t snn = (int64_t)n * n, smn = (int64_t)m * n;
  const size_t nnb = (size_t)batch * snn * sizeof(T);
  double* lam = (double*)take((size_t)batch * n * sizeof(double));
  char* eigws = take(eigh_workspace_bytes(n, batch));
  T* dPh = (T*)take(nnb);
  T* M = (T*)take(nnb);
  T* F = (T*)take(nnb);
  T* X = (T*)take(nnb);
  T* R = (T*)take(nnb);
  T* Z = (T*)take(nnb);
  T* D = (T*)take(nnb);
  T* Qm = (T*)take(nnb);
  T* Pc = (T*)take(nnb);
  T* Pinv = (T*)take(nnb);
  T* Zw = (T*)take((size_t)batch * smn * sizeof(T));
  T* tmp = (T*)take((size_t)batch * DBK * n * sizeof(T));
  T* Yd = (T*)take((size_t)batch * DBK * DBK * sizeof(T) * cdiv(n, DBK) + 256);
  double* partial = (double*)take((size_t)batch * kRedBlocks * sizeof(double));
  double* sc = (double*)take((size_t)batch * 4 * sizeof(double));
  int* dinfo = (int*)take(256);
  double* rz = sc;
  double* rznew = sc + batch;
  double* dq = sc + 2 * batch;
  double* ff = sc + 3 * batch;
  const dim3 gnn = egrid(snn, batch);
  if (dW != nullptr && maxiter >= kPcgFirst && tol >= kDoublingMinTol && batch <= 32767) {  // grid z: 2 batch
    T* const buf[10] = {dPh, M, F, X, R, Z, D, Qm, Pc, Pinv};
    int steps = 0;
    const int st = polar_pullback_doubling<T>(s, batch, m, n, W, ldw, sw, P, ldp, sp, dW, lddw, sdw, dP, lddp, sdp, dA,
                                              ldda, sda, buf, Yd, sc, dinfo, &steps);
    if (st == 2) return 1;
    if (st == 0) {
      if (iters_out) *iters_out = steps;
      return hipGetLastError() == hipSuccess ? 0 : 1;
    }
  }
  // dPh = herm(dP) ; M = W^H dW - dPh P
  if (dP) hipLaunchKernelGGL((bherm_kernel<T>), gnn, dim3(256), 0, s, n, dP, lddp, sdp, dPh, (int64_t)n, snn);
  if (dW) gemm<T>(OP_C, OP_N, bga<T>(batch, n, n, m, W, ldw, sw, dW, lddw, sdw, M, n, snn, 1.0, 0.0), s);
  else hipLaunchKernelGGL((bfill_kernel<T>), gnn, dim3(256), 0, s, n, n, M, (int64_t)n, snn, 0);
  if (dP) gemm<T>(OP_N, OP_N, bga<T>(batch, n, n, n, dPh, n, snn, P, ldp, sp, M, n, snn, -1.0, 1.0), s);
  // F = M - M^H ; solve P C + C P = F  (PCG, C in X)
  hipLaunchKernelGGL((bskew2_kernel<T>), gnn, dim3(256), 0, s, n, M, (int64_t)n, snn, F, (int64_t)n, snn);
  hipLaunchKernelGGL((bfill_kernel<T>), gnn, dim3(256), 0, s, n, n, X, (int64_t)n, snn, 0);
  hipLaunchKernelGGL((bcopy_kernel<T>), gnn, dim3(256), 0, s, n, n, F, (int64_t)n, snn, R, (int64_t)n, snn);
  hipLaunchKernelGGL((bprecond_kernel<T>), gnn, dim3(256), 0, s, n, R, P, ldp, sp, Z);
  hipLaunchKernelGGL((bcopy_kernel<T>), gnn, dim3(256), 0, s, n, n, Z, (int64_t)n, snn, D, (int64_t)n, snn);
  bdot<T>(batch, n, n, R, n, snn, Z, n, snn, partial, rz, s);
  bdot<T>(batch, n, n, F, n, snn, F, n, snn, partial, ff, s);
  std::vector<double> hff(batch), hrr(batch);
  hipMemcpyAsync(hff.data(), ff, batch * sizeof(double), hipMemcpyDeviceToHost, s);
  hipStreamSynchronize(s);
  int it = 0;
  bool done = true;
  for (int b = 0; b < batch; ++b) done = done && (hff[b] == 0.0);
  const bool can_eig = eigh_available();
  const int pcg_steps = can_eig ? std::min(maxiter, kPcgFirst) : maxiter;
  for (it = 0; it < pcg_steps && !done; ++it) {
    // Qm = P D + D P
    gemm<T>(OP_N, OP_N, bga<T>(batch, n, n, n, P, ldp, sp, D, n, snn, Qm, n, snn, 1.0, 0.0), s);
    gemm<T>(OP_N, OP_N, bga<T>(batch, n, n, n, D, n, snn, P, ldp, sp, Qm, n, snn, 1.0, 1.0), s);
    bdot<T>(batch, n, n, D, n, snn, Qm, n, snn, partial, dq, s);
    hipLaunchKernelGGL((bcg_step_kernel<T>), gnn, dim3(256), 0, s, (int)snn, rz, dq, D, Qm, X, R);
    hipLaunchKernelGGL((bprecond_kernel<T>), gnn, dim3(256), 0, s, n, R, P, ldp, sp, Z);
    bdot<T>(batch, n, n, R, n, snn, Z, n, snn, partial, rznew, s);
    hipLaunchKernelGGL((bcg_dir_kernel<T>), gnn, dim3(256), 0, s, (int)snn, rznew, rz, Z, D);
    std::swap(rz, rznew);
    if ((it + 1) % 4 == 0 || it + 1 == pcg_steps) {
      bdot<T>(batch, n, n, R, n, snn, R, n, snn, partial, dq, s);
      hipMemcpyAsync(hrr.data(), dq, batch * sizeof(double), hipMemcpyDeviceToHost, s);
      hipStreamSynchronize(s);
      done = true;
      for (int b = 0; b < batch; ++b) done = done && (hrr[b] <= tol * tol * hff[b]);
    }
  }
  if (iters_out) *iters_out = it;
  // CG has not converged: solve exactly through P = Z diag(lambda) Z^H (Z in Pc)
  bool eig = false;
  if (!done && can_eig) {
    hipLaunchKernelGGL((bcopy_kernel<T>), gnn, dim3(256), 0, s, n, n, P, ldp, sp, Pc, (int64_t)n, snn);
    const int est = eigh_batched<T>(s, n, Pc, n, snn, lam, n, batch, eigws);
    if (est != 0) return est;
    std::vector<double> hl((size_t)batch * n);
    hipMemcpyAsync(hl.data(), lam, hl.size() * sizeof(double), hipMemcpyDeviceToHost, s);
    hipStreamSynchronize(s);
    for (int b = 0; b < batch; ++b)
      if (!(hl[(size_t)b * n] > 0.0)) return 2;  // P not positive definite
    gemm<T>(OP_N, OP_N, bga<T>(batch, n, n, n, F, n, snn, Pc, n, snn, Qm, n, snn, 1.0, 0.0), s);   // F Z
    gemm<T>(OP_C, OP_N, bga<T>(batch, n, n, n, Pc, n, snn, Qm, n, snn, R, n, snn, 1.0, 0.0), s);   // Z^H F Z
    hipLaunchKernelGGL((bsylv_divide_kernel<T>), gnn, dim3(256), 0, s, n, R, (int64_t)n, snn, (const double*)lam,
                       (int64_t)n);
    gemm<T>(OP_N, OP_N, bga<T>(batch, n, n, n, Pc, n, snn, R, n, snn, Qm, n, snn, 1.0, 0.0), s);   // Z Y
    gemm<T>(OP_N, OP_C, bga<T>(batch, n, n, n, Qm, n, snn, Pc, n, snn, X, n, snn, 1.0, 0.0), s);   // Z Y Z^H
    done = true;
    eig = true;
  }
  // C = X + dPh ; dA += W C
  if (dP) hipLaunchKernelGGL((baxpy_kernel<T>), gnn, dim3(256), 0, s, n, n, 1.0, dPh, (int64_t)n, snn, X, (int64_t)n, snn);
  gemm<T>(OP_N, OP_N, bga<T>(batch, m, n, n, W, ldw, sw, X, n, snn, dA, ldda, sda, 1.0, 1.0), s);
  if (dW) {
    // Zw = dW - W (W^H dW) ; dA += Zw P^{-1}
    gemm<T>(OP_C, OP_N, bga<T>(batch, n, n, m, W, ldw, sw, dW, lddw, sdw, M, n, snn, 1.0, 0.0), s);
    hipLaunchKernelGGL((bcopy_kernel<T>), egrid(smn, batch), dim3(256), 0, s, m, n, dW, lddw, sdw, Zw, (int64_t)m, smn);
    gemm<T>(OP_N, OP_N, bga<T>(batch, m, n, n, W, ldw, sw, M, n, snn, Zw, m, smn, -1.0, 1.0), s);
    if (eig) {
      // P^{-1} = (Z diag(1/lambda)) Z^H
      hipLaunchKernelGGL((bcopy_kernel<T>), gnn, dim3(256), 0, s, n, n, Pc, (int64_t)n, snn, Qm, (int64_t)n, snn);
      hipLaunchKernelGGL((bscale_cols_inv_kernel<T>), gnn, dim3(256), 0, s, n, n, Qm, (int64_t)n, snn,
                         (const double*)lam, (int64_t)n);
      gemm<T>(OP_N, OP_C, bga<T>(batch, n, n, n, Qm, n, snn, Pc, n, snn, Pinv, n, snn, 1.0, 0.0), s);
      gemm<T>(OP_N, OP_N, bga<T>(batch, m, n, n, Zw, m, smn, Pinv, n, snn, dA, ldda, sda, 1.0, 1.0), s);
    } else {
      // P = Wp^H Wp ; P^{-1} = Wp^{-1} Wp^{-H}
      hipLaunchKernelGGL((bcopy_kernel<T>), gnn, dim3(256), 0, s, n, n, P, ldp, sp, Pc, (int64_t)n, snn);
      hipMemsetAsync(dinfo, 0, sizeof(int), s);
      bpotrf_upper<T>(batch, n, Pc, n, snn, Yd, DBK, (int64_t)DBK * DBK, tmp, (int64_t)DBK * n, dinfo, s);
      btrtri_upper<T>(batch, n, Pc, n, snn, Qm, n, snn, s);
      gemm<T>(OP_N, OP_C, bga<T>(batch, n, n, n, Qm, n, snn, Qm, n, snn, Pinv, n, snn, 1.0, 0.0), s);
      gemm<T>(OP_N, OP_N, bga<T>(batch, m, n, n, Zw, m, smn, Pinv, n, snn, dA, ldda, sda, 1.0, 1.0), s);
      int hinfo = 0;
      hipMemcpyAsync(&hinfo, dinfo, sizeof(int), hipMemcpyDeviceToHost, s);
      hipStreamSynchronize(s);
      if (hinfo != 0) return 2;
    }
  }
  if (hipGetLastError() != hipSuccess) return 1;
  return done ? 0 : 6;
}

size_t qr_full_cotangent_ws_bytes(size_t elem, int batch, int m, int n) {
  const int k = std::min(m, n), r = m - k;
  return al256((size_t)batch * k * std::max(r, 0) * elem) + al256((size_t)batch * m * std::max(r, 0) * elem) + 256;
}
template <typename T> size_t qr_full_cotangent_ws(int batch, int m, int n) {
  return qr_full_cotangent_ws_bytes(sizeof(T), batch, m, n);
}

// check_and_prepare_qr_cotangents for a qr_full! cotangent (src/pullbacks/
// qr.jl:4-53): dQ (m x m, as the full Q) -> dQ1 (m x k, the compact
// cotangent the pullback takes) and gauge_out[b] (device) = max |.| of the
// gauge-dependent part: for p = k, dQ3 - Q1 Q1^H dQ3 (dQ3 = dQ[:, k:m]), with
// dQ1 = dQ[:, :k] - Q3 (Q1^H dQ3)^H; for p < k, dQ[:, p:m], with dQ1 =
// dQ[:, :k].  Q: the full Q (m x m).
template <typename T>
int qr_full_cotangent(hipStream_t s, int batch, int m, int n, int p, const T* Q, int64_t ldq, int64_t sq, const T* dQ,
                      int64_t lddq, int64_t sdq, T* dQ1, int64_t ldd1, int64_t sd1, double* gauge_out, void* work,
                      size_t wbytes) {
  if (batch < 0) return -2;
  if (m < 0) return -3;
  if (n < 0) return -4;
  const int k = std::min(m, n), r = m - k;
  if (p < 0 || p > k) return -5;
  if (ldq < std::max(1, m)) return -7;
  if (lddq < std::max(1, m)) return -10;
  if (ldd1 < std::max(1, m)) return -13;
  if (wbytes < qr_full_cotangent_ws<T>(batch, m, n) || (work == nullptr && batch > 0 && r > 0)) return -17;
  if (batch == 0 || m == 0) return 0;
  if (Q == nullptr || dQ == nullptr || dQ1 == nullptr) return -6;
  const int64_t smk = (int64_t)m * k;
  hipLaunchKernelGGL((bcopy_kernel<T>), egrid(smk, batch), dim3(256), 0, s, m, k, dQ, lddq, sdq, dQ1, ldd1, sd1);
  if (gauge_out) hipLaunchKernelGGL(bzero_doubles_kernel, dim3(cdiv(batch, 256)), dim3(256), 0, s, gauge_out, batch);
  if (r == 0) return hipGetLastError() == hipSuccess ? 0 : 1;
  if (p < k) {
    if (gauge_out) bmaxabs<T>(batch, m, m - p, dQ + (int64_t)p * lddq, lddq, sdq, 0, gauge_out, s);
    return hipGetLastError() == hipSuccess ? 0 : 1;
  }
  char* w = reinterpret_cast<char*>(work);
  T* X = reinterpret_cast<T*>(w);                                                  // Q1^H dQ3 (k x r)
  T* T3 = reinterpret_cast<T*>(w + al256((size_t)batch * k * r * sizeof(T)));     // dQ3 - Q1 X (m x r)
  const int64_t skr = (int64_t)k * r, smr = (int64_t)m * r;
  const T* dQ3 = dQ + (int64_t)k * lddq;
  const T* Q3 = Q + (int64_t)k * ldq;
  gemm<T>(OP_C, OP_N, bga<T>(batch, k, r, m, Q, ldq, sq, dQ3, lddq, sdq, X, k, skr, 1.0, 0.0), s);
  if (gauge_out) {
    hipLaunchKernelGGL((bcopy_kernel<T>), egrid(smr, batch), dim3(256), 0, s, m, r, dQ3, lddq, sdq, T3, (int64_t)m,
                       smr);
    gemm<T>(OP_N, OP_N, bga<T>(batch, m, r, k, Q, ldq, sq, X, k, skr, T3, m, smr, -1.0, 1.0), s);
    bmaxabs<T>(batch, m, r, T3, m, smr, 0, gauge_out, s);
  }
  gemm<T>(OP_N, OP_C, bga<T>(batch, m, k, r, Q3, ldq, sq, X, k, skr, dQ1, ldd1, sd1, -1.0, 1.0), s);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

#define MAK_INST_PB(T)                                                                                            \
  template size_t qr_pullback_ws<T>(int, int, int);                                                               \
  template size_t polar_pullback_ws<T>(int, int, int);                                                            \
  template int qr_pullback<T>(hipStream_t, int, int, int, int, int, const T*, int64_t, int64_t, const T*, int64_t,\
                              const T*, int64_t, int64_t, const T*, int64_t, int64_t, const T*, int64_t, int64_t, \
                              T*, int64_t, int64_t, void*, size_t, double*);                                      \
  template int qr_full_cotangent<T>(hipStream_t, int, int, int, int, const T*, int64_t, int64_t, const T*,        \
                                    int64_t, int64_t, T*, int64_t, int64_t, double*, void*, size_t);              \
  template int polar_pullback<T>(hipStream_t, int, int, int, const T*, int64_t, int64_t, const T*, int64_t,       \
                                 int64_t, const T*, int64_t, int64_t, const T*, int64_t, int64_t, T*, int64_t,    \
                                 int64_t, int, double, void*, size_t, int*);
MAK_INST_PB(double)
MAK_INST_PB(zd)

}  // namespace mak

extern "C" {

int mak_pullback_workspace_size(int kind, int dtype, int batch, int m, int n, size_t* bytes) {
  if (bytes == nullptr) return -6;
  if (batch < 0) return -3;
  if (m < 0) return -4;
  if (n < 0) return -5;
  if (kind == 0) *bytes = dtype == MAK_F64 ? mak::qr_pullback_ws<double>(batch, m, n)
                                           : mak::qr_pullback_ws<mak::zd>(batch, m, n);
  else if (kind == 1) *bytes = dtype == MAK_F64 ? mak::polar_pullback_ws<double>(batch, m, n)
                                                : mak::polar_pullback_ws<mak::zd>(batch, m, n);
  else if (kind == 2) *bytes = dtype == MAK_F64 ? mak::qr_full_cotangent_ws<double>(batch, m, n)
                                                : mak::qr_full_cotangent_ws<mak::zd>(batch, m, n);
  else return -1;
  if (dtype != MAK_F64 && dtype != MAK_C64) return -2;
  return 0;
}

#define MAK_QRPB(SUFFIX, T, CT)                                                                                     \
  int mak_qr_pullback_##SUFFIX(void* s, int batch, int m, int n, int p, int positive, const CT* A, int lda,      \
                               long long sa,                                                                       \
                               const CT* Tp, long long st, const CT* R, int ldr, long long sr, const CT* dQ,       \
                               int lddq, long long sdq, const CT* dR, int lddr, long long sdr, CT* dA, int ldda,   \
                               long long sda, void* work, size_t wbytes, double* gauge_out) {                      \
    return mak::qr_pullback<T>((hipStream_t)s, batch, m, n, p, positive, (const T*)A, lda, sa, (const T*)Tp, st,   \
                               (const T*)R, ldr, sr, (const T*)dQ, lddq, sdq, (const T*)dR, lddr, sdr, (T*)dA,    \
                               ldda, sda, work, wbytes, gauge_out);                                                \
  }
MAK_QRPB(d, double, double)
MAK_QRPB(z, mak::zd, void)

#define MAK_QRFC(SUFFIX, T, CT)                                                                                     \
  int mak_qr_full_cotangent_##SUFFIX(void* s, int batch, int m, int n, int p, const CT* Q, int ldq, long long sq,  \
                                     const CT* dQ, int lddq, long long sdq, CT* dQ1, int ldd1, long long sd1,      \
                                     double* gauge_out, void* work, size_t wbytes) {                                \
    return mak::qr_full_cotangent<T>((hipStream_t)s, batch, m, n, p, (const T*)Q, ldq, sq, (const T*)dQ, lddq,    \
                                     sdq, (T*)dQ1, ldd1, sd1, gauge_out, work, wbytes);                            \
  }
MAK_QRFC(d, double, double)
MAK_QRFC(z, mak::zd, void)

#define MAK_PPB(SUFFIX, T, CT)                                                                                      \
  int mak_left_polar_pullback_##SUFFIX(void* s, int batch, int m, int n, const CT* W, int ldw, long long sw,        \
                                       const CT* P, int ldp, long long sp, const CT* dW, int lddw, long long sdw,  \
                                       const CT* dP, int lddp, long long sdp, CT* dA, int ldda, long long sda,     \
                                       int maxiter, double tol, void* work, size_t wbytes, int* iters) {           \
    return mak::polar_pullback<T>((hipStream_t)s, batch, m, n, (const T*)W, ldw, sw, (const T*)P, ldp, sp,         \
                                  (const T*)dW, lddw, sdw, (const T*)dP, lddp, sdp, (T*)dA, ldda, sda, maxiter,    \
                                  tol, work, wbytes, iters);                                                        \
  }
MAK_PPB(d, double, double)
MAK_PPB(z, mak::zd, void)

}  // extern "C"
