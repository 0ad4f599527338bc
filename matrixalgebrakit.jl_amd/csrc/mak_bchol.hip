// CholeskyQR2 of whole blocks, many unevenly sized blocks per launch (the
// batched qr_compact! plan, mak_batched.hip):
//   G = A^H A = R1^H R1,  Q1 = A R1^{-1},  E = Q1^H Q1 - I,
//   U = the upper half of E (half of its diagonal),
//   Q = Q1 (I - U),  R = (I + U) R1.
// E is what the condition of G left of the rounding of R1; with
// ||E||_F <= 1e-8 (condition numbers to about 2e4) the terms of second order in
// U are below rounding, so that the second factorisation is U itself.  With
// ||E||_F <= 0.1 (to about 1e7) a second pass comes between: the Cholesky factor
// R2 of Q1^H Q1, Q1 <- Q1 R2^{-1}, R1 <- R2 R1.  A block whose Gram matrix has a
// pivot that is not positive, or whose E is larger, is rejected: left to the
// gated Householder launches.  A is only read.
//
// Every product runs on 64 x 64 tiles, one workgroup of four waves (32 x 32
// each) per task, over task lists of all blocks:
//   Gram      upper tiles of G, K = all rows
//   factor    block column by block column (64 wide, left-looking): step k
//             forms the tiles R_kj, and the task of tile (k, k+1) goes on to
//             factor diagonal tile k+1, so that a step is one launch
//   solve     64-row strips, block column by block column:
//             Q1_j = (A_j - sum_i Q1_i R_ij) R_jj^{-1}.  Substitution and not
//             a product with R1^{-1}, refined where R_jj is ill conditioned:
//             its residual does not grow with the condition number of R1
//   Gram      E, and its tiles' norms
//   correct   Q1 - Q1 U in place, strips from the last block column to the
//             first; the tiles of R
// 4 m n^2 flops a block, as many as blocked Householder with its orgqr, but
// with inner dimensions of up to m or n instead of 32: the panel schedule read
// and wrote the trailing matrix once per 32 columns.
// Tasks are listed so that a block stays on one XCD (workgroup b runs on XCD
// b mod 8), whose L2 then serves the operands that its tiles share.
// 4096 blocks (m log-uniform in [16, 1024], n uniform in [8, m]; 2743 of them
// whole): Float64 Gram 3.1 ms each (49 TF/s of the padded tiles), factor 2.6, solve
// 4.2, correct 5.5 ms; ComplexF64 8.7 each, 7.1, 11.0 and 13.0 ms.  All of a call,
// Float64 33.6 ms on the panel schedule, 19.0 here; 1024 ComplexF64 blocks 24.6
// and 14.7.
#include <algorithm>

#include "mak_common.hpp"
#include "mak_dense32.hpp"
#include "mak_kernels.hpp"

namespace mak {

namespace {

constexpr int BT = kBCholTile;  // 64
constexpr double kBCholMaxE = 1e-8, kBCholMaxE2 = 0.1;
constexpr double kTallMaxE = 1e-6;
// Columns of a triangular tile closer than 1 / kBCholRefine to the span of the
// others: products with the tile's inverse get a step of refinement.  The
// residual of the product alone is then about 5e-16 of ||A||, what Householder QR
// leaves, and grows in proportion.
constexpr double kBCholRefine = 8.0;

// LDS of one stage of a tile product: KB inner indices of the two operands.
// The pitches keep the fragment reads (16 rows x 4 k of a wave) off each
// other's banks; KB = 8 for ComplexF64 keeps two stages at 37 KB (four
// workgroups a CU).
template <typename T> struct BcCfg;
template <> struct BcCfg<double> {
  static constexpr int KB = 16, PK = 17, PR = 80;
  static constexpr int L = 16 * PR, R = 64 * PK, STAGE = L + R;
  static constexpr int OCC_GRAM = 4, OCC = 3;  // waves per SIMD
  static constexpr int POOL = 2 * STAGE;
};
template <> struct BcCfg<zd> {
  static constexpr int KB = 8, PK = 9, PR = 65;
  static constexpr int L = 64 * PK, R = 64 * PK, STAGE = L + R;
  static constexpr int OCC_GRAM = 2, OCC = 2;
  static constexpr int POOL = 2 * STAGE;
};
constexpr int KX = 16;  // inner indices of one stage of the product with a 64 x 64 inverse
template <typename T> struct BcX;
template <> struct BcX<double> { static constexpr int PK = 17, PR = 80; };
template <> struct BcX<zd> { static constexpr int PK = 17, PR = 65; };
static_assert(KX * BcX<double>::PR + 64 * BcX<double>::PK <= BcCfg<double>::POOL, "stage of the inverse");
static_assert(KX * BcX<zd>::PR + 64 * BcX<zd>::PK <= BcCfg<zd>::POOL, "stage of the inverse");

// 32 x 32 accumulators of a wave: row 16 i + lane % 16, column 16 j + 4 u + lane / 16
template <typename T> struct BcAcc;
template <> struct BcAcc<double> {
  v4d r[2][2];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) r[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  }
  __device__ __forceinline__ double get(int i, int j, int u) const { return r[i][j][u]; }
  template <bool CL>
  __device__ __forceinline__ void step(const double (&a)[2], const double (&b)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) r[i][j] = mfma_f64(b[j], a[i], r[i][j]);
  }
};
// three real products (Gauss): re = p - q, im = s - p - q
template <> struct BcAcc<zd> {
  v4d p[2][2], q[2][2], s[2][2];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) p[i][j] = q[i][j] = s[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  }
  __device__ __forceinline__ zd get(int i, int j, int u) const {
    return mkz(p[i][j][u] - q[i][j][u], s[i][j][u] - p[i][j][u] - q[i][j][u]);
  }
  template <bool CL>
  __device__ __forceinline__ void step(const zd (&a)[2], const zd (&b)[2]) {
    double ai[2], as[2], bs[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ai[i] = CL ? -a[i].y : a[i].y;
      as[i] = a[i].x + ai[i];
      bs[i] = b[i].x + b[i].y;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        p[i][j] = mfma_f64(b[j].x, a[i].x, p[i][j]);
        q[i][j] = mfma_f64(b[j].y, ai[i], q[i][j]);
        s[i][j] = mfma_f64(bs[j], as[i], s[i][j]);
      }
  }
};

// One 16 x 16 block of a wave: row lane % 16, column 4 u + lane / 16.
template <typename T> struct BcRow;
template <> struct BcRow<double> {
  v4d r;
  __device__ __forceinline__ void zero() { r = v4d{0.0, 0.0, 0.0, 0.0}; }
  __device__ __forceinline__ void step(double a, double b) { r = mfma_f64(b, a, r); }
  __device__ __forceinline__ double get(int u) const { return r[u]; }
};
template <> struct BcRow<zd> {
  v4d p, q, s;
  __device__ __forceinline__ void zero() { p = q = s = v4d{0.0, 0.0, 0.0, 0.0}; }
  __device__ __forceinline__ void step(const zd& a, const zd& b) {
    p = mfma_f64(b.x, a.x, p);
    q = mfma_f64(b.y, a.y, q);
    s = mfma_f64(b.x + b.y, a.x + a.y, s);
  }
  __device__ __forceinline__ zd get(int u) const { return mkz(p[u] - q[u], s[u] - p[u] - q[u]); }
};

// acc += op(L) R over K inner indices, for a 64 x 64 tile:
//   KL:  op(L)(i, k) = conj(L[k + i ldl]);  otherwise L[i + k ldl];
//   R(k, j) = R[k + j ldr].
// Rows i >= nl and columns j >= nr repeat the last valid one (the caller drops
// them); 64 ldl and 64 ldr elements stay below 2 GB.  Two LDS stages, one
// barrier per stage, and the values of two more on their way in registers.  The
// caller leaves the pool free; it is free again on return.
template <typename T, bool KL>
__device__ __forceinline__ void bc_product(BcAcc<T>& acc, T* pool, const T* L, int64_t ldl, int nl, const T* R,
                                           int64_t ldr, int nr, int K) {
  using C = BcCfg<T>;
  constexpr int KB = C::KB, NQ = BT * KB / 256;
  if (K <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int lr = lane & 15, lq = lane >> 4;
  const int wm = w & 1, wn = w >> 1;
  // byte offsets of this thread's elements from bases that advance uniformly
  unsigned ol[NQ], orr[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int e = tid + 256 * q;
    orr[q] = (unsigned)((e % KB + min(e / KB, nr - 1) * (int)ldr) * (int)sizeof(T));
    ol[q] = (unsigned)((KL ? e % KB + min(e / KB, nl - 1) * (int)ldl : min(e % BT, nl - 1) + (e / BT) * (int)ldl) *
                       (int)sizeof(T));
  }
  struct Regs {
    T l[NQ], r[NQ];
  };
  Regs v0, v1;
  auto load = [&](Regs& v, int k0) {
    const char* bl = reinterpret_cast<const char*>(L + (KL ? (int64_t)k0 : (int64_t)k0 * ldl));
    const char* br = reinterpret_cast<const char*>(R + k0);
    if (k0 + KB <= K) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        v.l[q] = *reinterpret_cast<const T*>(bl + ol[q]);
        v.r[q] = *reinterpret_cast<const T*>(br + orr[q]);
      }
    } else {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int e = tid + 256 * q;
        v.l[q] = k0 + (KL ? e % KB : e / BT) < K ? *reinterpret_cast<const T*>(bl + ol[q]) : s_zero(T());
        v.r[q] = k0 + e % KB < K ? *reinterpret_cast<const T*>(br + orr[q]) : s_zero(T());
      }
    }
  };
  auto store = [&](const Regs& v, T* st) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int e = tid + 256 * q;
      if constexpr (KL) st[(e / KB) * C::PK + e % KB] = v.l[q];
      else st[(e / BT) * C::PR + e % BT] = v.l[q];
      st[C::L + (e / KB) * C::PK + e % KB] = v.r[q];
    }
  };
  auto compute = [&](const T* st) {
#pragma unroll
    for (int kk = 0; kk < KB; kk += 4) {
      T a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = wm * 32 + i * 16 + lr, col = wn * 32 + i * 16 + lr;
        if constexpr (KL) a[i] = st[row * C::PK + kk + lq];
        else a[i] = st[(kk + lq) * C::PR + row];
        b[i] = st[C::L + col * C::PK + kk + lq];
      }
      acc.template step<KL>(a, b);
    }
  };
  // stage t is in LDS buffer t % 2, t + 1 in registers, t + 2 being loaded
  T* s0 = pool;
  T* s1 = pool + C::STAGE;
  load(v0, 0);
  if (KB < K) load(v1, KB);
  store(v0, s0);
  for (int k0 = 0; k0 < K; k0 += 2 * KB) {
    if (k0 + 2 * KB < K) load(v0, k0 + 2 * KB);
    __syncthreads();
    compute(s0);
    if (k0 + KB >= K) break;
    store(v1, s1);
    if (k0 + 3 * KB < K) load(v1, k0 + 3 * KB);
    __syncthreads();
    compute(s1);
    if (k0 + 2 * KB < K) store(v0, s0);
  }
  __syncthreads();
}

// One stage of KX inner indices held in the pool: left as [k][row], right as [col][k].
template <typename T, bool CL>
__device__ __forceinline__ void bcx_step(BcAcc<T>& acc, const T* left, const T* right) {
  using X = BcX<T>;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
#pragma unroll
  for (int kk = 0; kk < KX; kk += 4) {
    T a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[i] = left[(kk + lq) * X::PR + wm * 32 + i * 16 + lr];
      b[i] = right[(wn * 32 + i * 16 + lr) * X::PK + kk + lq];
    }
    acc.template step<CL>(a, b);
  }
}

// acc = V X, V the workgroup's 64 x 64 tile in registers (accumulator layout),
// X 64 x 64: quarters of 16 inner indices through the pool.
template <typename T>
__device__ __forceinline__ void bc_times_x(BcAcc<T>& acc, T* pool, const T (&v)[2][2][4], const T* X, int ldx) {
  using C = BcX<T>;
  T* left = pool;
  T* right = pool + KX * C::PR;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  acc.zero();
#pragma unroll
  for (int h = 0; h < BT / KX; ++h) {
    T x[BT * KX / 256];
#pragma unroll
    for (int q = 0; q < BT * KX / 256; ++q) {
      const int e = tid + 256 * q;
      x[q] = X[h * KX + e % KX + (e / KX) * ldx];
    }
    if (h > 0) __syncthreads();
    if (wn == h / 2) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int u = 0; u < 4; ++u) left[(4 * u + lq) * C::PR + wm * 32 + i * 16 + lr] = v[i][h % 2][u];
    }
#pragma unroll
    for (int q = 0; q < BT * KX / 256; ++q) {
      const int e = tid + 256 * q;
      right[(e / KX) * C::PK + e % KX] = x[q];
    }
    __syncthreads();
    bcx_step<T, false>(acc, left, right);
  }
  __syncthreads();
}

// acc = X^H V, as above
template <typename T> __device__ __forceinline__ void bc_xh_times(BcAcc<T>& acc, T* pool, const T* X, const T (&v)[2][2][4]) {
  using C = BcX<T>;
  T* left = pool;
  T* right = pool + KX * C::PR;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  acc.zero();
#pragma unroll
  for (int h = 0; h < BT / KX; ++h) {
    T x[BT * KX / 256];
#pragma unroll
    for (int q = 0; q < BT * KX / 256; ++q) {
      const int e = tid + 256 * q;
      x[q] = X[h * KX + e % KX + (e / KX) * BT];
    }
    if (h > 0) __syncthreads();
#pragma unroll
    for (int q = 0; q < BT * KX / 256; ++q) {
      const int e = tid + 256 * q;
      left[(e % KX) * C::PR + e / KX] = x[q];
    }
    if (wm == h / 2) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) right[(wn * 32 + j * 16 + 4 * u + lq) * C::PK + lr] = v[h % 2][j][u];
    }
    __syncthreads();
    bcx_step<T, true>(acc, left, right);
  }
  __syncthreads();
}

// A leading dimension whose products with column indices are formed where they
// are used, not kept in registers over the loop around.
__device__ __forceinline__ int bc_local(int64_t ld) {
  int v = (int)ld;
  asm volatile("" : "+s"(v));
  return v;
}

// Status words of a replay: nothing rejected, no panel rejected.
__global__ void bchol_init_kernel(int* state, int n, int* any, int* status, int nst) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) state[e] = 0;
  if (e < nst) status[e] = 0;
  if (e == 0) *any = 0;
}

// States of a block: 0 factored in one pass, 2 in two, 1 rejected.
__device__ __forceinline__ bool bc_skip(int state, int pass) { return state != (pass == 2 ? 2 : 0); }
// In launches that do not write the state (all but the factor and the decision).
__device__ __forceinline__ bool bc_skip(const BCholProb& p, int pass) { return bc_skip(*p.state, pass); }

// State after E of this pass; any |= rejected.  One wave per block sums the
// squared norms of E's upper tiles, in a fixed order.  (nt^2 times their
// maximum instead overestimates ||E||_F up to nt times: E sits in its last rows
// and columns, and a set of 4096 Gaussian blocks then nearly always had one in
// the second pass, 2.5 ms of 21.)
__global__ void bchol_decide_kernel(const BCholProb* P, int n, int* any, int pass) {
  const int e = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64, lane = threadIdx.x & 63;
  if (e >= n) return;
  const BCholProb p = P[e];
  const int nt = p.np / BT, st = *p.state;
  if (!bc_skip(st, pass)) {
    double s = 0.0;
    for (int t = lane; t < nt * nt; t += 64)
      if (t % nt <= t / nt) s += (t % nt < t / nt ? 2.0 : 1.0) * p.dev[t];
    s = wave_sum(s);
    const bool ok = s <= kBCholMaxE * kBCholMaxE;  // false for a NaN
    const int to = ok ? st : pass == 1 && s <= kBCholMaxE2 * kBCholMaxE2 ? 2 : 1;
    if (lane == 0) {
      *p.state = to;
      if (to == 1) *any = 1;  // every writer writes 1
    }
  } else if (st == 1 && lane == 0) {
    *any = 1;
  }
}

// Tile (a, b), a <= b: of A^H A in W, in the second pass of Q1^H Q1 in U
// (padding: the identity), or, HALF, of U from E = Q1^H Q1 - I (padding: 0)
// with the tile's norm.  Bound by the matrix cores (busy 55 % with one stage of
// operands in flight and rows 18 doubles apart in LDS: 3.5 ms; two stages and
// 17: 3.0 ms).
template <typename T, bool HALF>
__global__ void __launch_bounds__(256, BcCfg<T>::OCC_GRAM)
    bchol_gram_kernel(const BCholProb* P, const BCholTask* tasks, int pass) {
  using C = BcCfg<T>;
  __shared__ T pool[C::POOL];
  __shared__ double part[4];
  const BCholTask t = tasks[blockIdx.x];
  if (t.prob < 0) return;
  const BCholProb p = P[t.prob];
  if (bc_skip(p, pass)) return;
  const int i0 = t.a * BT, j0 = t.b * BT;
  const bool second = HALF || pass == 2;
  const T* X = reinterpret_cast<const T*>(second ? p.Q : p.A);
  const int64_t ldx = second ? p.ldq : p.lda;
  BcAcc<T> acc;
  acc.zero();
  bc_product<T, true>(acc, pool, X + (int64_t)i0 * ldx, ldx, p.n - i0, X + (int64_t)j0 * ldx, ldx, p.n - j0, p.m);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  T* G = reinterpret_cast<T*>(second ? p.U : p.W);
  double s2 = 0.0;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int gi = i0 + wm * 32 + i * 16 + lr, gj = j0 + wn * 32 + j * 16 + 4 * u + lq;
        T v = acc.get(i, j, u);
        if (gi == gj) v = s_from_real<T>(HALF ? s_re(v) - 1.0 : s_re(v));
        if (gi >= p.n || gj >= p.n) v = (!HALF && gi == gj) ? s_one(T()) : s_zero(T());
        if constexpr (HALF) {
          s2 += s_abs2(v);
          v = gi > gj ? s_zero(T()) : (gi == gj ? s_scale(v, 0.5) : v);
        }
        G[gi + (int64_t)gj * p.np] = v;
      }
  if constexpr (HALF) {
    s2 = wave_sum(s2);
    if (lane == 0) part[w] = s2;
    __syncthreads();
    if (threadIdx.x == 0) p.dev[t.a + t.b * (p.np / BT)] = part[0] + part[1] + part[2] + part[3];
  }
}

// Cholesky with inverse of a 64 x 64 Hermitian matrix by 256 threads: its upper
// 32 x 32 blocks in S[0], S[64], S[128] (rows of 33; S[32], S[96] scratch) become
// R (W, ld) and R^{-1} (X, ld 64) with zeros below the diagonal.  True if a
// pivot was not positive.  The blocks were written before a barrier here.
// cond (optional): the largest ||R(:, k)||^2 ||R^{-1}(k, :)||^2, the inverse
// square of the sine between a column and the span of the others; red: 4 in LDS.
template <typename T>
__device__ __forceinline__ bool bc_chol64(T (*S)[33], int* bad_s, T* W, int64_t ld, T* X, double* cond = nullptr,
                                          double* red = nullptr) {
  T (*S11)[33] = S;
  T (*Y11)[33] = S + 32;
  T (*S12)[33] = S + 64;  // then Y22
  T (*W12)[33] = S + 96;
  T (*S22)[33] = S + 128;  // then W12 Y22
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (threadIdx.x == 0) *bad_s = 0;
  __syncthreads();
  if (w == 0) {
    const int bad = wave_chol_inv32<T>(S11, Y11);
    if (bad && lane == 0) *bad_s = 1;
  }
  __syncthreads();
  mm32<T>(W12, Y11, true, S12, false, 1.0, false);
  mm32<T>(S22, W12, true, W12, false, -1.0, true);
  if (w == 0) {
    const int bad = wave_chol_inv32<T>(S22, S12);
    if (bad && lane == 0) *bad_s = 1;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < BT * BT; e += 256) {
    const int i = e % BT, j = e / BT;
    T wv = s_zero(T()), xv = s_zero(T());
    if (j < 32) {
      if (i < 32) {
        wv = S11[i][j];
        xv = Y11[i][j];
      }
    } else if (i < 32) {
      wv = W12[i][j - 32];
    } else {
      wv = S22[i - 32][j - 32];
      xv = S12[i - 32][j - 32];
    }
    W[i + (int64_t)j * ld] = wv;
    if (i >= 32 || j < 32) X[e] = xv;
  }
  // four threads a column
  const int kc = threadIdx.x >> 2, kr = kc & 31, kq = 8 * (threadIdx.x & 3);
  double cn = 0.0, rn = 0.0;
  if (cond != nullptr) {
    const T (*C1)[33] = kc < 32 ? S11 : W12;
#pragma unroll
    for (int i = 0; i < 8; ++i) cn += s_abs2(C1[kq + i][kr]) + (kc < 32 ? 0.0 : s_abs2(S22[kq + i][kr]));
  }
  __syncthreads();
  mm32<T>(S22, W12, false, S12, false, 1.0, false);
  mm32<T>(S22, Y11, false, S22, false, -1.0, false);
  for (int e = threadIdx.x; e < 32 * 32; e += 256) X[e % 32 + (32 + e / 32) * BT] = S22[e % 32][e / 32];
  if (cond != nullptr) {
    const T (*R1)[33] = kc < 32 ? Y11 : S12;
#pragma unroll
    for (int i = 0; i < 8; ++i) rn += s_abs2(R1[kr][kq + i]) + (kc < 32 ? s_abs2(S22[kr][kq + i]) : 0.0);
    cn += __shfl_xor(cn, 1);
    rn += __shfl_xor(rn, 1);
    cn += __shfl_xor(cn, 2);
    rn += __shfl_xor(rn, 2);
    double d = cn * rn;
#pragma unroll
    for (int h = 4; h < 64; h *= 2) d = fmax(d, __shfl_xor(d, h));
    if (lane == 0) red[w] = d;
    __syncthreads();
    if (threadIdx.x == 0) *cond = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  }
  return *bad_s != 0;
}

// Step k of the factorisation of G: tile R_kb and its term of diagonal tile b,
// then for b = k + 1 the factor of that tile (k = -1: only that).  Bound by the
// latency of that one task (about 30 us at 64 columns, 100 us at 1024): the
// diagonal tile's terms are subtracted as they come because summing them in its
// own step doubled the chain (1024 ComplexF64 blocks: 2.9 -> 2.4 ms).  The diagonal tile of 64 is factored with its
// inverse as 32 x 32 blocks by wave 0.
template <typename T>
__global__ void __launch_bounds__(256) bchol_factor_kernel(const BCholProb* P, const BCholTask* tasks, int pass) {
  using C = BcCfg<T>;
  __shared__ T pool[C::POOL > 5 * 32 * 33 ? C::POOL : 5 * 32 * 33];
  __shared__ int bad_s, state_s;
  __shared__ double red[4];
  const BCholTask t = tasks[blockIdx.x];
  if (t.prob < 0) return;
  const BCholProb p = P[t.prob];
  // The task of the block's next diagonal tile may reject the block while this
  // one starts: one thread reads the state for all (what the task writes is of
  // no use then, whichever value it sees).
  if (threadIdx.x == 0) state_s = __hip_atomic_load(p.state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (bc_skip(state_s, pass)) return;
  const int k = t.a, b = t.b;
  const int64_t ld = p.np;
  T* W = reinterpret_cast<T*>(pass == 2 ? p.U : p.W);
  T* Xd = reinterpret_cast<T*>(p.X);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  const int ri = wm * 32 + lr, cj = wn * 32 + lq;  // + 16 i, + 16 j + 4 u
  const T* Wb = W + (int64_t)b * BT * ld;
  BcAcc<T> acc;
  if (k >= 0) {
    T* Wkb = W + (int64_t)k * BT + (int64_t)b * BT * ld;
    acc.zero();
    bc_product<T, true>(acc, pool, W + (int64_t)k * BT * ld, ld, BT, Wb, ld, BT, k * BT);
    T v[2][2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          v[i][j][u] = s_sub(Wkb[ri + 16 * i + (int64_t)(cj + 16 * j + 4 * u) * ld], acc.get(i, j, u));
    bc_xh_times<T>(acc, pool, Xd + (int64_t)k * BT * BT, v);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) Wkb[ri + 16 * i + (int64_t)(cj + 16 * j + 4 * u) * ld] = acc.get(i, j, u);
    __syncthreads();  // R_kb is read by every wave below
  }
  // S = G_bb - sum_i<=k R_ib^H R_ib, one term per step: kept in G_bb, or for the
  // next diagonal block in three 32 x 32 blocks of the pool
  T (*S11)[33] = reinterpret_cast<T (*)[33]>(pool);
  T* Wbb = W + (int64_t)b * BT * (ld + 1);
  acc.zero();
  if (k >= 0) bc_product<T, true>(acc, pool, Wb + k * BT, ld, BT, Wb + k * BT, ld, BT, BT);
  if (b != k + 1) {
    if (wm <= wn)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            T* g = Wbb + ri + 16 * i + (int64_t)(cj + 16 * j + 4 * u) * ld;
            *g = s_sub(*g, acc.get(i, j, u));
          }
    return;
  }
  if (wm <= wn) {
    T (*S)[33] = S11 + 64 * (wm + wn);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          S[16 * i + lr][16 * j + 4 * u + lq] =
              s_sub(Wbb[ri + 16 * i + (int64_t)(cj + 16 * j + 4 * u) * ld], acc.get(i, j, u));
  }
  const bool bad = bc_chol64<T>(S11, &bad_s, Wbb, ld, Xd + (int64_t)b * BT * BT, p.dev + b * (p.np / BT + 1), red);
  if (threadIdx.x == 0 && bad) __hip_atomic_store(p.state, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Strip a (64 rows) of Q1 = A R1^{-1}, block column by block column; second: of
// Q1 <- Q1 R2^{-1}, in place.  A block column whose diagonal tile has a column
// closer than kBCholRefine to the span of the others (bc_chol64) gets a second
// round, Q1_j += (A_j - sum_{i<=j} Q1_i R_ij) R_jj^{-1}: the residual of the
// first is about u times that quotient, 5e-16 of ||A|| at 8 and 1e-14 at 1e3
// (Householder QR 5e-16).  Of Gaussian blocks only the last tiles of nearly
// square ones pass the limit.  R2 is near the identity and needs none.
// Bound by the operands' path through L2 (8 flops a byte; 5.4 GB of 4096 Float64
// blocks come from beyond it) and the chain of block columns.
template <typename T>
__global__ void __launch_bounds__(256, BcCfg<T>::OCC)
    bchol_solve_kernel(const BCholProb* P, const BCholTask* tasks, int pass, int second) {
  using C = BcCfg<T>;
  __shared__ T pool[C::POOL];
  const BCholTask t = tasks[blockIdx.x];
  if (t.prob < 0) return;
  const BCholProb p = P[t.prob];
  if (bc_skip(p, pass)) return;
  const int r0 = t.a * BT, rows = p.m - r0;
  const T* A = reinterpret_cast<const T*>(second ? p.Q : p.A) + r0;
  T* Q = reinterpret_cast<T*>(p.Q) + r0;
  const T* W = reinterpret_cast<const T*>(second ? p.U : p.W);
  const T* Xd = reinterpret_cast<const T*>(p.X);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  const int ri = wm * 32 + lr, cj = wn * 32 + lq;
  BcAcc<T> acc;
  for (int jb = 0, round = 0; jb * BT < p.n;) {
    const int j0 = jb * BT, lda = bc_local(second ? p.ldq : p.lda), ldq = bc_local(p.ldq);
    acc.zero();
    bc_product<T, false>(acc, pool, Q, ldq, rows, W + (int64_t)j0 * p.np, p.np, BT, min(j0 + round * BT, p.n));
    T v[2][2][4];
    const T* Aj = A + (int64_t)j0 * p.lda;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int r = ri + 16 * i, c = cj + 16 * j + 4 * u;
          v[i][j][u] = (r < rows && j0 + c < p.n) ? s_sub(Aj[r + c * lda], acc.get(i, j, u)) : s_zero(T());
        }
    bc_times_x<T>(acc, pool, v, Xd + (int64_t)jb * BT * BT, BT);
    T* Qj = Q + (int64_t)j0 * p.ldq;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int r = ri + 16 * i, c = cj + 16 * j + 4 * u;
          if (r < rows && j0 + c < p.n) {
            T* q = Qj + r + c * ldq;
            *q = round ? s_add(*q, acc.get(i, j, u)) : acc.get(i, j, u);
          }
        }
    __syncthreads();  // what follows reads this block column in every wave
    if (round == 0 && !second && p.dev[jb * (p.np / BT + 1)] > kBCholRefine * kBCholRefine) {
      round = 1;
    } else {
      round = 0;
      ++jb;
    }
  }
}

// kind 0: strip a of Q = Q1 - Q1 U, in place from the last block column to the
// first; kind 1: tile (a, b), a <= b, of R = R1 + U R1, and zeros in (b, a);
// between the passes, kind 2: the tile of R = R2 R1, kind 3: of R1 = R.
template <typename T>
__global__ void __launch_bounds__(256, BcCfg<T>::OCC)
    bchol_correct_kernel(const BCholProb* P, const BCholTask* tasks, int pass) {
  using C = BcCfg<T>;
  __shared__ T pool[C::POOL];
  const BCholTask t = tasks[blockIdx.x];
  if (t.prob < 0) return;
  const BCholProb p = P[t.prob];
  if (bc_skip(p, pass)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  const int ri = wm * 32 + lr, cj = wn * 32 + lq;
  const T* U = reinterpret_cast<const T*>(p.U);
  BcAcc<T> acc;
  if (t.kind == 0) {
    const int r0 = t.a * BT, rows = p.m - r0;
    T* Q = reinterpret_cast<T*>(p.Q) + r0;
    for (int jb = p.np / BT - 1; jb >= 0; --jb) {
      const int j0 = jb * BT, ldq = bc_local(p.ldq);
      acc.zero();
      bc_product<T, false>(acc, pool, Q, ldq, rows, U + (int64_t)j0 * p.np, p.np, BT, min(j0 + BT, p.n));
      T* Qj = Q + (int64_t)j0 * p.ldq;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int r = ri + 16 * i, c = cj + 16 * j + 4 * u;
            if (r < rows && j0 + c < p.n) {
              T* q = Qj + r + c * ldq;
              *q = s_sub(*q, acc.get(i, j, u));
            }
          }
    }
    return;
  }
  const T* W = reinterpret_cast<const T*>(p.W);
  T* R = reinterpret_cast<T*>(p.R);
  const int i0 = t.a * BT, j0 = t.b * BT;
  acc.zero();
  if (t.kind == 3) {
    T* Wij = reinterpret_cast<T*>(p.W) + i0 + (int64_t)j0 * p.np;
    for (int e = threadIdx.x; e < BT * BT; e += 256) {
      const int r = e % BT, c = e / BT;
      if (i0 + r < p.n && j0 + c < p.n) Wij[r + (int64_t)c * p.np] = R[i0 + r + (int64_t)(j0 + c) * p.ldr];
    }
    return;
  }
  bc_product<T, false>(acc, pool, U + i0 + (int64_t)i0 * p.np, p.np, BT, W + i0 + (int64_t)j0 * p.np, p.np, BT,
                       j0 + BT - i0);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = ri + 16 * i, c = cj + 16 * j + 4 * u;
        const T w1 = t.kind == 2 ? s_zero(T()) : W[i0 + r + (int64_t)(j0 + c) * p.np];
        const T v = s_add(w1, acc.get(i, j, u));
        if (i0 + r < p.n && j0 + c < p.n) R[i0 + r + (int64_t)(j0 + c) * p.ldr] = i0 + r > j0 + c ? s_zero(T()) : v;
        if (i0 < j0 && j0 + r < p.n && i0 + c < p.n) R[j0 + r + (int64_t)(i0 + c) * p.ldr] = s_zero(T());
      }
}

// ---------------------------------------------------------------------------
// One matrix with n <= m < 64 by one workgroup in LDS: the same CholeskyQR2,
// and Householder QR (xGEQR2, xORG2R, gauge) in the same kernel when it is
// rejected, so that the call stays a single launch without a host check.
//   As  the matrix, then Q1, as [row][column] (rows >= m and columns >= n: 0)
//   Wg  64 x 64 global scratch (R1)
// Products with a factor on the right belong to one wave per 16 rows and need
// no workgroup barrier.  What bounds it: latency of the two 32 x 32 in-wave
// Choleskys (3 us each Float64) and of the ~10 steps between barriers.
// 57 x 33 Float64: the call 32 us against 131 us as 22 launches; with its copy of A
// 55 against 163 us, of condition 1e9 152 against 163 us.
// ---------------------------------------------------------------------------
constexpr int SP = 65;  // pitch of As

// acc[j] (16 rows of the wave x 16 columns each) += As(rows, a0 + k) B(k, 16 j ..), k < 32
template <typename T>
__device__ __forceinline__ void small_rows_mm(BcRow<T> (&acc)[2], const T (*As)[SP], int a0, const T (*B)[33]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < 32; kk += 4) {
    const T a = As[16 * w + lr][a0 + kk + lq];
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[j].step(a, B[kk + lq][16 * j + lr]);
  }
}

// True if a column k of the upper triangular W is closer than 1 / kBCholRefine
// to the span of the others: ||W(:, k)|| ||Y(k, :)|| > kBCholRefine for Y = W^{-1}.
template <typename T> __device__ __forceinline__ bool small_ill(const T (*W)[33], const T (*Y)[33]) {
  const int k = threadIdx.x & 31, h = threadIdx.x >> 1 & 16;
  double cn = 0.0, rn = 0.0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    cn += s_abs2(W[h + i][k]);
    rn += s_abs2(Y[k][h + i]);
  }
  cn += __shfl_xor(cn, 32);
  rn += __shfl_xor(rn, 32);
  return __any(cn * rn > kBCholRefine * kBCholRefine);
}

// As(rows, a0 ..) <- V W^{-1} of its V, Y the computed inverse of the 32 x 32
// upper triangular W, with one step of refinement if W is ill conditioned:
// V - (V Y) W alone is about u cond(W) (57 x 33 Float64 with two columns 1e-3
// apart: ||A - Q R|| / ||A|| 2.7e-14 without the step, 2e-16 with it,
// Householder 4e-16; 2.4 us of the call's 34 where it always ran).
template <typename T>
__device__ __forceinline__ void small_solve(T (*As)[SP], int a0, const T (*W)[33], const T (*Y)[33]) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
  T* row = &As[16 * (threadIdx.x >> 6) + lr][a0 + lq];  // + 16 j + 4 u
  T v[2][4], x[2][4];
  BcRow<T> q[2];
  auto times = [&](const T (*B)[33]) {
    q[0].zero();
    q[1].zero();
    small_rows_mm<T>(q, As, a0, B);
    wave_lds_sync();
  };
  times(Y);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v[j][u] = row[16 * j + 4 * u];
      row[16 * j + 4 * u] = x[j][u] = q[j].get(u);
    }
  wave_lds_sync();
  if (!small_ill<T>(W, Y)) return;  // the same in every wave
  times(W);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int u = 0; u < 4; ++u) row[16 * j + 4 * u] = s_sub(v[j][u], q[j].get(u));
  wave_lds_sync();
  times(Y);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int u = 0; u < 4; ++u) row[16 * j + 4 * u] = s_add(x[j][u], q[j].get(u));
  wave_lds_sync();
}

template <typename T>
__device__ __forceinline__ void small_householder(T (*As)[SP], T (*Qs)[SP], T* tau_s, const T* A, int64_t lda, T* Q,
                                                  int64_t ldq, T* R, int64_t ldr, int m, int n) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int e = tid; e < 64 * 64; e += 256) {
    const int r = e % 64, c = e / 64;
    As[r][c] = r < m && c < n ? A[r + (int64_t)c * lda] : s_zero(T());
    Qs[r][c] = r == c ? s_one(T()) : s_zero(T());
  }
  __syncthreads();
  for (int j = 0; j < n; ++j) {
    // every wave forms the reflector; wave 0 stores it after the barrier
    const T alpha = As[j][j];
    const T x = lane > j ? As[lane][j] : s_zero(T());
    const double nu2 = wave_sum(s_abs2(x));
    const double bn = sqrt(s_abs2(alpha) + nu2);
    T tau = s_zero(T()), beta = alpha, scale = s_zero(T());
    if (!((nu2 == 0.0 && s_im(alpha) == 0.0) || !(bn > 0.0))) {
      const double br = s_re(alpha) >= 0.0 ? -bn : bn;
      beta = s_from_real<T>(br);
      tau = s_scale(s_sub(beta, alpha), 1.0 / br);
      scale = s_div(s_one(T()), s_sub(alpha, beta));
    }
    const T v = lane == j ? s_one(T()) : s_mul(x, scale);  // 0 above the diagonal
    for (int c = j + 1 + w; c < n; c += 4) {
      const T a = lane >= j ? As[lane][c] : s_zero(T());
      const T d = s_mul(s_conj(tau), wave_sum(s_mul(s_conj(v), a)));
      if (lane >= j) As[lane][c] = s_sub(a, s_mul(v, d));
    }
    __syncthreads();
    if (w == 0 && lane >= j) As[lane][j] = lane == j ? beta : v;
    if (tid == 0) tau_s[j] = tau;
    __syncthreads();
  }
  for (int j = n - 1; j >= 0; --j) {
    const T v = lane < j ? s_zero(T()) : lane == j ? s_one(T()) : As[lane][j];
    const T tau = tau_s[j];
    for (int c = j + w; c < n; c += 4) {
      const T a = Qs[lane][c];
      const T d = s_mul(tau, wave_sum(s_mul(s_conj(v), a)));
      Qs[lane][c] = s_sub(a, s_mul(v, d));
    }
    __syncthreads();
  }
  for (int e = tid; e < 64 * n; e += 256) {
    const int r = e % 64, c = e / 64;
    if (r < m) Q[r + (int64_t)c * ldq] = s_mul(Qs[r][c], sign_safe(As[c][c]));
    if (R != nullptr && r < n) {
      T v = s_zero(T());
      if (r == c) v = s_from_real<T>(s_absv(As[r][r]));
      else if (r < c) v = s_mul(s_conj(sign_safe(As[r][r])), As[r][c]);
      R[r + (int64_t)c * ldr] = v;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) qr_small_kernel(const T* A, int64_t lda, T* Q, int64_t ldq, T* R, int64_t ldr,
                                                       T* Wg, int* status, int m, int n) {
  __shared__ T As[64][SP];
  __shared__ T tiles[5][32][33];
  __shared__ T tau_s[64];
  __shared__ double part[4];
  __shared__ int bad_s;
  T (*S11)[33] = tiles[0];
  T (*Y11)[33] = tiles[1];  // then U11
  T (*S12)[33] = tiles[2];  // then Y22, U22
  T (*W12)[33] = tiles[3];  // then U12
  T (*S22)[33] = tiles[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  const bool two = n > 32;  // a second block column
  for (int e = tid; e < 64 * 64; e += 256) {
    const int r = e % 64, c = e / 64;
    As[r][c] = r < m && c < n ? A[r + (int64_t)c * lda] : s_zero(T());
  }
  if (tid == 0) bad_s = 0;
  if (status != nullptr && tid < 8) status[tid] = 0;  // [0]: 1 below if accepted
  __syncthreads();
  // pass 0: G = A^H A to S11, S12, S22; pass 1: U from E = Q1^H Q1 - I to Y11, W12, S12
  const bool quad = wm <= wn && (two || wn == 0);
  for (int pass = 0; pass < 2; ++pass) {
    double s2 = 0.0;
    if (quad) {
      BcAcc<T> acc;
      acc.zero();
      for (int kk = 0; kk < m; kk += 4) {
        T a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[i] = As[kk + lq][wm * 32 + 16 * i + lr];
          b[i] = As[kk + lq][wn * 32 + 16 * i + lr];
        }
        acc.template step<true>(a, b);
      }
      T (*D)[33] = wn == 0 ? (pass ? Y11 : S11) : wm == 0 ? (pass ? W12 : S12) : (pass ? S12 : S22);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int r = 16 * i + lr, c = 16 * j + 4 * u + lq;
            const int gr = wm * 32 + r, gc = wn * 32 + c;
            T v = acc.get(i, j, u);
            if (gr == gc) v = s_from_real<T>(gr >= n ? (pass ? 0.0 : 1.0) : s_re(v) - (pass ? 1.0 : 0.0));
            if (pass) {
              s2 += (wm < wn ? 2.0 : 1.0) * s_abs2(v);
              v = gr > gc ? s_zero(T()) : gr == gc ? s_scale(v, 0.5) : v;
            }
            D[r][c] = v;
          }
    }
    if (pass) {
      s2 = wave_sum(s2);
      if (lane == 0) part[w] = s2;
    }
    __syncthreads();
    if (pass) break;
    for (int h = 0; h < (two ? 2 : 1); ++h) {
      if (w == 0) {
        const int bad = wave_chol_inv32<T>(h ? S22 : S11, h ? S12 : Y11);
        if (bad && lane == 0) bad_s = 1;
      }
      __syncthreads();
      if (h == 0 && two) {
        mm32<T>(W12, Y11, true, S12, false, 1.0, false);
        mm32<T>(S22, W12, true, W12, false, -1.0, true);
      }
    }
    // R1 to the scratch; Q1 = A R1^{-1} by rows
    if (R != nullptr)
      for (int e = tid; e < 64 * 64; e += 256) {
        const int r = e % 64, c = e / 64;
        T v = s_zero(T());
        if (r <= c && c < (two ? 64 : 32)) v = c < 32 ? S11[r][c] : r < 32 ? W12[r][c - 32] : S22[r - 32][c - 32];
        Wg[e] = v;
      }
    small_solve<T>(As, 0, S11, Y11);
    if (two) {
      BcRow<T> q[2];
      q[0].zero();
      q[1].zero();
      small_rows_mm<T>(q, As, 0, W12);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          T* p = &As[16 * w + lr][32 + 16 * j + 4 * u + lq];
          *p = s_sub(*p, q[j].get(u));
        }
      wave_lds_sync();
      small_solve<T>(As, 32, S22, S12);
    }
    __syncthreads();
  }
  const double dev = part[0] + part[1] + part[2] + part[3];
  if (bad_s || !(dev <= kBCholMaxE * kBCholMaxE)) {  // uniform
    __syncthreads();
    small_householder<T>(As, reinterpret_cast<T (*)[SP]>(&tiles[0][0][0]), tau_s, A, lda, Q, ldq, R, ldr, m, n);
    return;
  }
  if (status != nullptr && tid == 0) status[0] = 1;
  // Q = Q1 - Q1 U
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h == 1 && !two) break;
    BcRow<T> q[2];
    q[0].zero();
    q[1].zero();
    small_rows_mm<T>(q, As, 0, h ? W12 : Y11);
    if (h) small_rows_mm<T>(q, As, 32, S12);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = 16 * w + lr, c = 32 * h + 16 * j + 4 * u + lq;
        if (r < m && c < n) Q[r + (int64_t)c * ldq] = s_sub(As[r][c], q[j].get(u));
      }
  }
  if (R == nullptr) return;
  // R = R1 + U R1, wave w its rows 16 w ..
  __syncthreads();
  for (int e = tid; e < 64 * 64; e += 256) As[e % 64][e / 64] = Wg[e];
  __syncthreads();
  for (int jp = 0; jp < (two ? 2 : 1); ++jp) {
    BcRow<T> q[2];
    q[0].zero();
    q[1].zero();
    for (int kk = 16 * w / 32 * 32; kk < 32 * (jp + 1); kk += 4) {
      const int i = 16 * w + lr, k = kk + lq;
      const T a = i >= 32 ? S12[i - 32][k - 32] : k < 32 ? Y11[i][k] : W12[i][k - 32];
#pragma unroll
      for (int j = 0; j < 2; ++j) q[j].step(a, As[k][32 * jp + 16 * j + lr]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = 16 * w + lr, c = 32 * jp + 16 * j + 4 * u + lq;
        if (r < n && c < n) R[r + (int64_t)c * ldr] = r <= c ? s_add(As[r][c], q[j].get(u)) : s_zero(T());
      }
  }
}

// ---------------------------------------------------------------------------
// One matrix with m >= 64 rows and n < 64 columns: CholeskyQR2 in three
// launches, after a small one that clears their control words.  Workgroup s has rows s rps ..; the last one of a launch to finish
// sums the partial Gram matrices in order and does the 64 x 64 work:
//   0  partial A^H A;            R1 (W), R1^{-1} (X)
//   1  Q1 = A R1^{-1}, partial Q1^H Q1;   U, D = (I + U)^{-1} - I, R = (I + U) R1
//   2  Q = Q1 + Q1 D
// What bounds it: latency (1024 x 32 Float64: 23, 20 and 7 us, most of it the
// 64 x 64 work of one workgroup).  U to second order in E (as in mak_cholqr2.hip) where ||E||_F > 1e-9; accepted
// (*state = 0) up to 1e-6.
// ---------------------------------------------------------------------------
struct TallArgs {
  const void* A;
  int64_t lda;
  void* Q;
  int64_t ldq;
  void* R;
  int64_t ldr;
  void *part, *W, *X, *D;  // gridDim.x blocks of 64 x 64; 64 x 64 each
  int* ctl;                // state (1 until accepted), a ticket per launch; set by the caller to 1, 0, 0
  int* status;             // optional: [0] = 1 when accepted
  int m, n, rps;
};

// bc_chol64's conditioning of R1, after the ints of ctl
__device__ __forceinline__ double* tall_cond(int* ctl) { return reinterpret_cast<double*>(ctl + 4); }

template <typename T, int PASS>
__global__ void __launch_bounds__(256) qr_tall_kernel(const TallArgs p) {
  using C = BcCfg<T>;
  __shared__ T pool[C::POOL > 5 * 32 * 33 ? C::POOL : 5 * 32 * 33];
  __shared__ double red[4];
  __shared__ int flag_s, bad_s;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  const int ri = wm * 32 + lr, cj = wn * 32 + lq;
  const int r0 = blockIdx.x * p.rps, rows = min(p.rps, p.m - r0), n = p.n;
  const T* A = reinterpret_cast<const T*>(p.A) + r0;
  T* Q = reinterpret_cast<T*>(p.Q) + r0;
  T* X = reinterpret_cast<T*>(p.X);
  T* W = reinterpret_cast<T*>(p.W);
  BcAcc<T> acc;
  if constexpr (PASS == 1) {
    if (p.ctl[3]) return;  // G was not positive definite
    // Q1 = A X, then Q1 += (A - Q1 R1) X: the product alone leaves a residual of
    // u cond(R1) (100 x 63 with two columns 1e-4 apart: 4e-13 of ||A||; with the
    // second round 3e-16), which well-conditioned inputs do without (512 x 32: 96 us
    // a call, 106 with it; 16384 x 32: 152 and 199)
    const bool refine = *tall_cond(p.ctl) > kBCholRefine * kBCholRefine;
    for (int b0 = 0, round = 0; b0 < rows;) {
      T v[2][2][4];
      acc.zero();
      if (round) bc_product<T, false>(acc, pool, Q + b0, p.ldq, rows - b0, W, BT, BT, n);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int r = b0 + ri + 16 * i, c = cj + 16 * j + 4 * u;
            v[i][j][u] = r < rows && c < n ? s_sub(A[r + (int64_t)c * p.lda], acc.get(i, j, u)) : s_zero(T());
          }
      bc_times_x<T>(acc, pool, v, X, BT);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int r = b0 + ri + 16 * i, c = cj + 16 * j + 4 * u;
            if (r < rows && c < n) {
              T* q = Q + r + (int64_t)c * p.ldq;
              *q = round ? s_add(*q, acc.get(i, j, u)) : acc.get(i, j, u);
            }
          }
      __syncthreads();  // the second round reads the rows in every wave
      if (round || !refine) b0 += BT;
      round = !round && refine;
    }
    __syncthreads();
  }
  {
    const T* G = PASS == 0 ? A : Q;
    const int64_t ld = PASS == 0 ? p.lda : p.ldq;
    acc.zero();
    bc_product<T, true>(acc, pool, G, ld, n, G, ld, n, rows);
  }
  // upper 32 x 32 blocks of the partial
  const bool quad = wm <= wn && 32 * wn < n;
  T* part = reinterpret_cast<T*>(p.part) + (int64_t)blockIdx.x * BT * BT;
  if (quad)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) part[ri + 16 * i + (cj + 16 * j + 4 * u) * BT] = acc.get(i, j, u);
  __threadfence();
  __syncthreads();
  if (tid == 0) flag_s = atomicAdd(p.ctl + 1 + PASS, 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!flag_s) return;
  __threadfence();
  // blocks 11, 12, 22 of the sum to S[0], S[64], S[128]; PASS 1: of U1 = up(E)
  T (*S)[33] = reinterpret_cast<T (*)[33]>(pool);
  const T* P0 = reinterpret_cast<const T*>(p.part);
  double s2 = 0.0;
  for (int e = tid; e < 3 * 32 * 32; e += 256) {
    const int q = e >> 10, r = e & 31, c = (e >> 5) & 31;
    const int gr = (q == 2 ? 32 : 0) + r, gc = (q ? 32 : 0) + c;
    T v = s_zero(T());
    if (gc < n && gr < n)
      for (int k = 0; k < (int)gridDim.x; k += 16) {
        T x[16];  // 16 loads in flight
#pragma unroll
        for (int h = 0; h < 16; ++h)
          x[h] = P0[(int64_t)min(k + h, (int)gridDim.x - 1) * BT * BT + gr + gc * BT];
#pragma unroll
        for (int h = 0; h < 16; ++h) v = k + h < (int)gridDim.x ? s_add(v, x[h]) : v;
      }
    if (gr == gc) v = s_from_real<T>(gr >= n ? (PASS ? 0.0 : 1.0) : s_re(v) - (PASS ? 1.0 : 0.0));
    if (PASS) {
      s2 += (q == 1 ? 2.0 : 1.0) * s_abs2(v);
      v = gr > gc ? s_zero(T()) : gr == gc ? s_scale(v, 0.5) : v;
    }
    S[64 * q + r][c] = v;
  }
  if constexpr (PASS == 0) {
    const bool bad = bc_chol64<T>(S, &bad_s, W, BT, X, tall_cond(p.ctl), red);
    if (tid == 0) p.ctl[3] = bad;
  } else {
    s2 = wave_sum(s2);
    if (lane == 0) red[w] = s2;
    __syncthreads();
    const double dev = red[0] + red[1] + red[2] + red[3];
    if (!(dev <= kTallMaxE * kTallMaxE)) return;  // rejected
    T (*U11)[33] = S;
    T (*T1)[33] = S + 32;
    T (*U12)[33] = S + 64;
    T (*T2)[33] = S + 96;
    T (*U22)[33] = S + 128;
    T* D = reinterpret_cast<T*>(p.D);
    const bool two = n > 32, second = dev > 1e-18;
    if (second) {  // U = up(E - U1^H U1): E's halves are U1
      auto up_sub = [&](T (*U)[33], T (*N)[33], bool diag) {
        for (int e = tid; e < 32 * 32; e += 256) {
          const int r = e & 31, c = e >> 5;
          if (!diag || r < c) U[r][c] = s_sub(U[r][c], N[r][c]);
          else if (r == c) U[r][c] = s_from_real<T>(s_re(U[r][c]) - 0.5 * s_re(N[r][c]));
        }
        __syncthreads();
      };
      if (two) {
        mm32<T>(T2, U12, true, U12, false, 1.0, false);
        mm32<T>(T2, U22, true, U22, false, 1.0, true);
        mm32<T>(T1, U11, true, U12, false, 1.0, false);
        up_sub(U22, T2, true);
        up_sub(U12, T1, false);
      }
      mm32<T>(T1, U11, true, U11, false, 1.0, false);
      up_sub(U11, T1, true);
    }
    // D = -U + U^2, block by block; R = R1 + U R1
    auto put_d = [&](T (*U)[33], T (*N)[33], int i0, int j0) {
      for (int e = tid; e < 32 * 32; e += 256) {
        const int r = e & 31, c = e >> 5;
        const T v = second ? s_sub(N[r][c], U[r][c]) : s_neg(U[r][c]);
        D[i0 + r + (j0 + c) * BT] = v;
      }
      __syncthreads();
    };
    if (second) mm32<T>(T1, U11, false, U11, false, 1.0, false);
    put_d(U11, T1, 0, 0);
    for (int e = tid; e < 32 * 32; e += 256) {  // below the diagonal blocks
      D[32 + (e & 31) + (e >> 5) * BT] = s_zero(T());
      if (!two) {
        D[(e & 31) + (32 + (e >> 5)) * BT] = s_zero(T());
        D[32 + (e & 31) + (32 + (e >> 5)) * BT] = s_zero(T());
      }
    }
    if (two) {
      if (second) {
        mm32<T>(T1, U11, false, U12, false, 1.0, false);
        mm32<T>(T1, U12, false, U22, false, 1.0, true);
        mm32<T>(T2, U22, false, U22, false, 1.0, false);
      }
      put_d(U12, T1, 0, 32);
      put_d(U22, T2, 32, 32);
    }
    if (p.R != nullptr) {
      T* R = reinterpret_cast<T*>(p.R);
      auto get_w = [&](T (*N)[33], int i0, int j0) {
        __syncthreads();
        for (int e = tid; e < 32 * 32; e += 256) N[e & 31][e >> 5] = W[i0 + (e & 31) + (j0 + (e >> 5)) * BT];
        __syncthreads();
      };
      // R block = N (+ N0), zeros below the diagonal
      auto put_r = [&](T (*N)[33], T (*N0)[33], int i0, int j0) {
        for (int e = tid; e < 32 * 32; e += 256) {
          const int r = e & 31, c = e >> 5;
          const T v = i0 + r <= j0 + c ? s_add(N[r][c], N0[r][c]) : s_zero(T());
          if (i0 + r < n && j0 + c < n) R[i0 + r + (int64_t)(j0 + c) * p.ldr] = v;
        }
      };
      get_w(T2, 0, 0);
      mm32<T>(T1, U11, false, T2, false, 1.0, false);
      put_r(T1, T2, 0, 0);
      if (two) {
        for (int e = tid; e < 32 * 32; e += 256)
          if (32 + (e & 31) < n) R[32 + (e & 31) + (int64_t)(e >> 5) * p.ldr] = s_zero(T());
        get_w(T2, 0, 32);
        mm32<T>(T1, U11, false, T2, false, 1.0, false);
        for (int e = tid; e < 32 * 32; e += 256) T1[e & 31][e >> 5] = s_add(T1[e & 31][e >> 5], T2[e & 31][e >> 5]);
        get_w(T2, 32, 32);
        mm32<T>(U11, U12, false, T2, false, 1.0, false);
        put_r(T1, U11, 0, 32);
        __syncthreads();
        mm32<T>(T1, U22, false, T2, false, 1.0, false);
        put_r(T1, T2, 32, 32);
      }
    }
    if (tid == 0) {
      p.ctl[0] = 0;
      if (p.status != nullptr) p.status[0] = 1;
    }
  }
}

// Q = Q1 + Q1 D, 64 rows a workgroup
template <typename T> __global__ void __launch_bounds__(256) qr_tall_correct_kernel(const TallArgs p) {
  using C = BcCfg<T>;
  __shared__ T pool[C::POOL];
  if (p.ctl[0]) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = w & 1, wn = w >> 1;
  const int r0 = blockIdx.x * BT, rows = p.m - r0;
  T* Q = reinterpret_cast<T*>(p.Q) + r0;
  BcAcc<T> acc;
  acc.zero();
  bc_product<T, false>(acc, pool, Q, p.ldq, rows, reinterpret_cast<const T*>(p.D), BT, BT, p.n);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = wm * 32 + lr + 16 * i, c = wn * 32 + lq + 16 * j + 4 * u;
        if (r < rows && c < p.n) {
          T* q = Q + r + (int64_t)c * p.ldq;
          *q = s_add(*q, acc.get(i, j, u));
        }
      }
}

__global__ void qr_tall_init_kernel(int* ctl, int* status, int* flags) {
  const int t = threadIdx.x;
  if (t < 4) ctl[t] = t == 0;
  if (t < 8 && status != nullptr) status[t] = 0;
  if (t < 3 && flags != nullptr) flags[t] = 0;
}

}  // namespace

void launch_bchol_init(int* state, int n, int* any, int* status, int nst, hipStream_t s) {
  const int tot = std::max(std::max(n, nst), 1);
  hipLaunchKernelGGL(bchol_init_kernel, dim3(cdiv(tot, 256)), dim3(256), 0, s, state, n, any, status, nst);
}
void launch_bchol_decide(const BCholProb* P, int n, int* any, int pass, hipStream_t s) {
  hipLaunchKernelGGL(bchol_decide_kernel, dim3(cdiv(n, 4)), dim3(256), 0, s, P, n, any, pass);
}
template <typename T>
void launch_bchol(BCholPhase phase, const BCholProb* P, const BCholTask* tasks, int n, int pass, hipStream_t s) {
  if (n <= 0) return;
  const dim3 g(n), b(256);
  switch (phase) {
    case BCHOL_GRAM1: hipLaunchKernelGGL((bchol_gram_kernel<T, false>), g, b, 0, s, P, tasks, pass); break;
    case BCHOL_FACTOR: hipLaunchKernelGGL((bchol_factor_kernel<T>), g, b, 0, s, P, tasks, pass); break;
    case BCHOL_SOLVE: hipLaunchKernelGGL((bchol_solve_kernel<T>), g, b, 0, s, P, tasks, pass, pass == 2); break;
    case BCHOL_GRAM2: hipLaunchKernelGGL((bchol_gram_kernel<T, true>), g, b, 0, s, P, tasks, pass); break;
    case BCHOL_CORRECT:
    case BCHOL_COMPOSE: hipLaunchKernelGGL((bchol_correct_kernel<T>), g, b, 0, s, P, tasks, pass); break;
  }
}
template void launch_bchol<double>(BCholPhase, const BCholProb*, const BCholTask*, int, int, hipStream_t);
template void launch_bchol<zd>(BCholPhase, const BCholProb*, const BCholTask*, int, int, hipStream_t);


template <typename T>
void launch_qr_small(const T* A, int64_t lda, T* Q, int64_t ldq, T* R, int64_t ldr, T* scratch, int* status, int m,
                     int n, hipStream_t s) {
  hipLaunchKernelGGL((qr_small_kernel<T>), dim3(1), dim3(256), 0, s, A, lda, Q, ldq, R, ldr, scratch, status,
                     m, n);
}
template void launch_qr_small<double>(const double*, int64_t, double*, int64_t, double*, int64_t, double*, int*, int,
                                      int, hipStream_t);
template void launch_qr_small<zd>(const zd*, int64_t, zd*, int64_t, zd*, int64_t, zd*, int*, int, int,
                                  hipStream_t);

template <typename T>
void qr_tall_enqueue(const T* A, int64_t lda, T* Q, int64_t ldq, T* R, int64_t ldr, T* scratch, int* status,
                     int* flags, int m, int n, hipStream_t s) {
  const int rps = cdiv(cdiv(m, kTallMaxWgs), BT) * BT, wgs = cdiv(m, rps);
  T* W = scratch + kTallCtlElems;
  const TallArgs a{A, lda, Q, ldq, R, ldr, W + 3 * BT * BT, W, W + BT * BT, W + 2 * BT * BT,
                   reinterpret_cast<int*>(scratch), status, m, n, rps};
  hipLaunchKernelGGL(qr_tall_init_kernel, dim3(1), dim3(64), 0, s, a.ctl, status, flags);
  hipLaunchKernelGGL((qr_tall_kernel<T, 0>), dim3(wgs), dim3(256), 0, s, a);
  hipLaunchKernelGGL((qr_tall_kernel<T, 1>), dim3(wgs), dim3(256), 0, s, a);
  hipLaunchKernelGGL((qr_tall_correct_kernel<T>), dim3(cdiv(m, BT)), dim3(256), 0, s, a);
}
template void qr_tall_enqueue<double>(const double*, int64_t, double*, int64_t, double*, int64_t, double*, int*, int*,
                                      int, int, hipStream_t);
template void qr_tall_enqueue<zd>(const zd*, int64_t, zd*, int64_t, zd*, int64_t, zd*, int*, int*, int, int,
                                  hipStream_t);

}  // namespace mak
