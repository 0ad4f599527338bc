// Dense 32 x 32 building blocks in LDS for one workgroup / one wave (gfx950).
#pragma once

#include <utility>

#include "mak_common.hpp"

namespace mak {

// ---------------------------------------------------------------------------
// 32x32x32 products on FP64 MFMA for one 256-thread workgroup:
//   C = alpha op(A) op(B) (+ C when acc), op = identity or conjugate transpose.
// Wave w computes the 16x16 block (w % 2, w / 2).  The result is written after
// a workgroup barrier, so C may alias A or B.  All 256 threads must call it.
// ---------------------------------------------------------------------------
template <typename T>
__device__ inline void mm32(T (*C)[33], const T (*A)[33], bool cA, const T (*B)[33], bool cB, double alpha,
                            bool acc) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int bi = w & 1, bj = w >> 1;
  v4d cr = {0.0, 0.0, 0.0, 0.0}, ci = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kk = 0; kk < 32; kk += 4) {
    const int k = kk + (lane >> 4);
    const int i = bi * 16 + (lane & 15);
    const int j = bj * 16 + (lane & 15);
    const T a = cA ? s_conj(A[k][i]) : A[i][k];
    const T b = cB ? s_conj(B[j][k]) : B[k][j];
    // transposed block: lane l holds row (l % 16) of the output
    cr = mfma_f64(s_re(b), s_re(a), cr);
    if constexpr (ScalarTraits<T>::is_complex) {
      cr = mfma_f64(-s_im(b), s_im(a), cr);
      ci = mfma_f64(s_im(b), s_re(a), ci);
      ci = mfma_f64(s_re(b), s_im(a), ci);
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = bi * 16 + (lane & 15);
    const int col = bj * 16 + mfma_f64_row(lane, r);
    T v;
    if constexpr (ScalarTraits<T>::is_complex) v = mkz(alpha * cr[r], alpha * ci[r]);
    else v = alpha * cr[r];
    C[row][col] = acc ? s_add(C[row][col], v) : v;
  }
  __syncthreads();
}

// C = alpha (op(A0) op(B0) + op(A1) op(B1)) (+ C when acc): two products
// summed in the MFMA accumulators, one write (after a barrier, so C may alias
// any operand).  A0 = nullptr drops the first product.
template <typename T>
__device__ inline void mm32_2(T (*C)[33], const T (*A0)[33], const T (*B0)[33], const T (*A1)[33],
                              const T (*B1)[33], bool cA, bool cB, double alpha, bool acc) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int bi = w & 1, bj = w >> 1;
  v4d cr = {0.0, 0.0, 0.0, 0.0}, ci = {0.0, 0.0, 0.0, 0.0};
  auto product = [&](const T (*A)[33], const T (*B)[33]) {
#pragma unroll
    for (int kk = 0; kk < 32; kk += 4) {
      const int k = kk + (lane >> 4);
      const int i = bi * 16 + (lane & 15);
      const int j = bj * 16 + (lane & 15);
      const T a = cA ? s_conj(A[k][i]) : A[i][k];
      const T b = cB ? s_conj(B[j][k]) : B[k][j];
      cr = mfma_f64(s_re(b), s_re(a), cr);
      if constexpr (ScalarTraits<T>::is_complex) {
        cr = mfma_f64(-s_im(b), s_im(a), cr);
        ci = mfma_f64(s_im(b), s_re(a), ci);
        ci = mfma_f64(s_re(b), s_im(a), ci);
      }
    }
  };
  if (A0 != nullptr) product(A0, B0);
  product(A1, B1);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = bi * 16 + (lane & 15);
    const int col = bj * 16 + mfma_f64_row(lane, r);
    T v;
    if constexpr (ScalarTraits<T>::is_complex) v = mkz(alpha * cr[r], alpha * ci[r]);
    else v = alpha * cr[r];
    C[row][col] = acc ? s_add(C[row][col], v) : v;
  }
  __syncthreads();
}

// Value of v in lane `src` (uniform over the wave) broadcast to the wave through a scalar register.
__device__ inline double rdl(double v, int src) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, src);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), src);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ inline zd rdl(zd v, int src) { return mkz(rdl(v.x, src), rdl(v.y, src)); }

// Broadcasts issued together before their arithmetic: four real or two
// complex values (eight scalar registers).
template <typename T> constexpr int kBc = ScalarTraits<T>::is_complex ? 2 : 4;

// Makes `v` appear to depend on `dep` through an empty asm (no instruction is
// emitted): broadcasts of `v` cannot then be scheduled before `dep` is
// computed.  Without it the compiler hoists all broadcasts of a factorisation
// step (or of a whole triangular inverse) into scalar registers at once and
// spills them to VGPR lanes, which costs more than the arithmetic.
__device__ __forceinline__ void order_after(double& v, double dep) { asm volatile("" : "+v"(v) : "v"(dep)); }
// The lane's column index through an empty asm, so that the per-step lane
// masks (c > j, c == j) are formed in their step instead of all being hoisted
// into scalar registers up front.
__device__ __forceinline__ int step_lane(int c) {
  asm volatile("" : "+v"(c));
  return c;
}
__device__ __forceinline__ void order_after(zd& v, double dep) { asm volatile("" : "+v"(v.x), "+v"(v.y) : "v"(dep)); }
__device__ __forceinline__ void order_after(zd& v, const zd& dep) {
  asm volatile("" : "+v"(v.x), "+v"(v.y) : "v"(dep.x));
}
// Inverse Y of an upper triangular N x N block U, lane c holding column c
// (s[r] = U(r, c)), `dinv` of lane r = 1 / U(r, r).  Rows from the
// bottom: Y(r, c) = (delta_rc - sum_{k > r} U(r, k) Y(k, c)) / U(r, r).
template <typename T, int N, int I>
__device__ __forceinline__ void trinvN_row(T (&y)[N], const T (&s)[N], const T& dinv, int c0) {
  constexpr int r = N - 1 - I;
  const int c = step_lane(c0);
  T acc0 = s_zero(T()), acc1 = s_zero(T());
  T src = s[r];
  if constexpr (r < N - 1) order_after(src, y[r < N - 1 ? r + 1 : r]);
#pragma unroll
  for (int k0 = r + 1; k0 < N; k0 += kBc<T>) {
    T b[kBc<T>];
#pragma unroll
    for (int u = 0; u < kBc<T>; ++u) b[u] = (k0 + u < N) ? rdl(src, k0 + u) : s_zero(T());   // U(r, k)
#pragma unroll
    for (int u = 0; u < kBc<T>; ++u) {
      if (k0 + u < N) {
        if (u & 1) acc1 = s_fma(b[u], y[k0 + u], acc1);
        else acc0 = s_fma(b[u], y[k0 + u], acc0);
      }
    }
    order_after(src, acc0);
  }
  const T inv = rdl(dinv, r);
  y[r] = sel(r < c, s_neg(s_mul(s_add(acc0, acc1), inv)), sel(r == c, inv, s_zero(T())));
}
template <typename T, int N, int... Is>
__device__ __forceinline__ void trinvN_rows(T (&y)[N], const T (&s)[N], const T& dinv, int c,
                                            std::integer_sequence<int, Is...>) {
  (trinvN_row<T, N, Is>(y, s, dinv, c), ...);
}
// Inverse Z of a unit lower triangular N x N block L (lane c: s[r] = L(r, c)
// for r > c), rows from the top: Z(r, c) = delta_rc - sum_{c <= k < r} L(r, k) Z(k, c).
template <typename T, int N, int R>
__device__ __forceinline__ void trilinvN_row(T (&z)[N], const T (&s)[N], int c0) {
  const int c = step_lane(c0);
  T acc0 = s_zero(T()), acc1 = s_zero(T());
  T src = s[R];
  if constexpr (R > 0) order_after(src, z[R > 0 ? R - 1 : 0]);
#pragma unroll
  for (int k0 = 0; k0 < R; k0 += kBc<T>) {
    T b[kBc<T>];
#pragma unroll
    for (int u = 0; u < kBc<T>; ++u) b[u] = (k0 + u < R) ? rdl(src, k0 + u) : s_zero(T());   // L(R, k)
#pragma unroll
    for (int u = 0; u < kBc<T>; ++u) {
      if (k0 + u < R) {
        if (u & 1) acc1 = s_fma(b[u], z[k0 + u], acc1);
        else acc0 = s_fma(b[u], z[k0 + u], acc0);
      }
    }
    order_after(src, acc0);
  }
  z[R] = sel(R == c, s_one(T()), sel(R > c, s_neg(s_add(acc0, acc1)), s_zero(T())));
}
template <typename T, int N, int... Rs>
__device__ __forceinline__ void trilinvN_rows(T (&z)[N], const T (&s)[N], int c, std::integer_sequence<int, Rs...>) {
  (trilinvN_row<T, N, Rs>(z, s, c), ...);
}

// 16 x 16 x 16 product by one wave on FP64 MFMA, operands and result in LDS
// (row stride 33): D = alpha op(A) B (+ D when acc), op(A) = A^H when CA.
// Every operand is read before D is written, so D may alias A or B.
// MFMA f64 16x16x4 layout: A operand lane l = (row l % 16, k l / 16), B
// operand lane l = (col l % 16, k l / 16), result register r of lane l =
// (row 4 r + l / 16, col l % 16).
template <typename T, bool CA>
__device__ __forceinline__ void wave_mm16(T (*D)[33], const T (*A)[33], const T (*B)[33], double alpha, bool acc) {
  const int l = lane_id();
  const int lr = l & 15, lk = l >> 4;
  v4d cr = {0.0, 0.0, 0.0, 0.0}, ci = {0.0, 0.0, 0.0, 0.0};
  T a[4], b[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = 4 * q + lk;
    a[q] = CA ? s_conj(A[k][lr]) : A[lr][k];
    b[q] = B[k][lr];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (ScalarTraits<T>::is_complex) {
      cr = mfma_f64(s_re(a[q]), s_re(b[q]), cr);
      cr = mfma_f64(-s_im(a[q]), s_im(b[q]), cr);
      ci = mfma_f64(s_re(a[q]), s_im(b[q]), ci);
      ci = mfma_f64(s_im(a[q]), s_re(b[q]), ci);
    } else {
      cr = mfma_f64(a[q], b[q], cr);
    }
  }
  T old[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) old[r] = acc ? D[4 * r + lk][lr] : s_zero(T());
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    T v;
    if constexpr (ScalarTraits<T>::is_complex) v = mkz(alpha * cr[r], alpha * ci[r]);
    else v = alpha * cr[r];
    D[4 * r + lk][lr] = s_add(old[r], v);
  }
}

// ---------------------------------------------------------------------------
// One-wave elimination of [s | x] by 16 pivots.  A 16-lane row of the wave is
// one DPP row, so the pivot row's entry r (held by lane r) reaches all its
// lanes as the DPP source of the multiply-add itself (row_newbcast, the one
// DPP control that 64-bit operations take): no LDS round trip, no readlane.
// ---------------------------------------------------------------------------

// v of lane K of each 16-lane row, in all lanes of that row.
template <int K> __device__ __forceinline__ double row_bcast(double v) {
  const long u = __builtin_bit_cast(long, v), z = 0;
  const long r = __builtin_amdgcn_update_dpp(z, u, 0x150 + K, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}

template <int K> __device__ __forceinline__ zd row_bcast(const zd& v) {
  return mkz(row_bcast<K>(v.x), row_bcast<K>(v.y));
}

// Rows R .. R + N - 1 of s and x: s -= conj(b_R) ws, x -= conj(b_R) wx with
// b_R = b of lane R of the 16-lane row.  A VGPR may be a DPP source from two
// instructions after its write, and what the register allocator puts between
// two asm blocks (a copy of b, a reload) is not known to them, so each block
// begins with the wait itself, or with two other instructions.  A wait per row
// costs a sixth of the whole factorisation, so a block holds all rows between
// two links of the chain of reciprocals (qr_compact! 1024 x 512 Float64: 375 us
// without any waits, 388 with a wait per four rows, 382 so; ComplexF64 within
// 0.5 % of each other).
#define MAK_E_OUT(i) [s##i] "+&v"(s[R + i]), [x##i] "+&v"(x[R + i])
#define MAK_E_LANE(i) [r##i] "n"(R + i)
#define MAK_E_ROW(i)                                                                                    \
  "v_fmac_f64_dpp %[s" #i "], -%[b], %[ws] row_newbcast:%c[r" #i "] row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f64_dpp %[x" #i "], -%[b], %[wx] row_newbcast:%c[r" #i "] row_mask:0xf bank_mask:0xf\n\t"
#define MAK_E_IN [b] "v"(b), [ws] "v"(ws), [wx] "v"(wx)
template <int R, int N> __device__ __forceinline__ void elim_block(double* s, double* x, double b, double ws, double wx) {
  if constexpr (N == 1)
    asm("s_nop 1\n\t" MAK_E_ROW(0)
        : MAK_E_OUT(0)
        : MAK_E_IN, MAK_E_LANE(0));
  else if constexpr (N == 2)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1)
        : MAK_E_OUT(0), MAK_E_OUT(1)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1));
  else if constexpr (N == 3)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2));
  else if constexpr (N == 4)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2) MAK_E_ROW(3)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2), MAK_E_OUT(3)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2), MAK_E_LANE(3));
  else if constexpr (N == 5)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2) MAK_E_ROW(3) MAK_E_ROW(4)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2), MAK_E_OUT(3), MAK_E_OUT(4)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2), MAK_E_LANE(3), MAK_E_LANE(4));
  else if constexpr (N == 6)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2) MAK_E_ROW(3) MAK_E_ROW(4) MAK_E_ROW(5)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2), MAK_E_OUT(3), MAK_E_OUT(4), MAK_E_OUT(5)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2), MAK_E_LANE(3), MAK_E_LANE(4), MAK_E_LANE(5));
  else if constexpr (N == 7)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2) MAK_E_ROW(3) MAK_E_ROW(4) MAK_E_ROW(5) MAK_E_ROW(6)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2), MAK_E_OUT(3), MAK_E_OUT(4), MAK_E_OUT(5), MAK_E_OUT(6)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2), MAK_E_LANE(3), MAK_E_LANE(4), MAK_E_LANE(5), MAK_E_LANE(6));
}
// The same for row R alone, forming ws = s[R - 1] inv and wx = x[R - 1] inv
// first (b = s[R - 1]); s[R] may be a DPP source afterwards.
template <int R>
__device__ __forceinline__ void elim_first(double* s, double* x, double b, double inv, double& ws, double& wx) {
  constexpr int K = R - 1;
  asm("v_mul_f64 %[ws], %[b], %[inv]\n\tv_mul_f64 %[wx], %[xk], %[inv]\n\t" MAK_E_ROW(0) "s_nop 0"
      : MAK_E_OUT(0), [ws] "=&v"(ws), [wx] "=&v"(wx)
      : [b] "v"(b), [xk] "v"(x[K]), [inv] "v"(inv), MAK_E_LANE(0));
}
#undef MAK_E_OUT
#undef MAK_E_ROW
#undef MAK_E_IN
#define MAK_E_OUT(i) \
  [sx##i] "+&v"(s[R + i].x), [sy##i] "+&v"(s[R + i].y), [xx##i] "+&v"(x[R + i].x), [xy##i] "+&v"(x[R + i].y)
#define MAK_E_FMAC(acc, i, part, w) \
  "v_fmac_f64_dpp %[" acc #i "], " part ", %[" w "] row_newbcast:%c[r" #i "] row_mask:0xf bank_mask:0xf\n\t"
#define MAK_E_ROW(i)                                                                                  \
  MAK_E_FMAC("sx", i, "-%[bx]", "wsx") MAK_E_FMAC("sy", i, "-%[bx]", "wsy")                           \
  MAK_E_FMAC("xx", i, "-%[bx]", "wxx") MAK_E_FMAC("xy", i, "-%[bx]", "wxy")                           \
  MAK_E_FMAC("sx", i, "-%[by]", "wsy") MAK_E_FMAC("sy", i, "%[by]", "wsx")                            \
  MAK_E_FMAC("xx", i, "-%[by]", "wxy") MAK_E_FMAC("xy", i, "%[by]", "wxx")
#define MAK_E_IN \
  [bx] "v"(b.x), [by] "v"(b.y), [wsx] "v"(ws.x), [wsy] "v"(ws.y), [wxx] "v"(wx.x), [wxy] "v"(wx.y)
template <int R, int N>
__device__ __forceinline__ void elim_block(zd* s, zd* x, const zd& b, const zd& ws, const zd& wx) {
  if constexpr (N == 1)
    asm("s_nop 1\n\t" MAK_E_ROW(0)
        : MAK_E_OUT(0)
        : MAK_E_IN, MAK_E_LANE(0));
  else if constexpr (N == 2)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1)
        : MAK_E_OUT(0), MAK_E_OUT(1)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1));
  else if constexpr (N == 3)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2));
  else if constexpr (N == 4)
    asm("s_nop 1\n\t" MAK_E_ROW(0) MAK_E_ROW(1) MAK_E_ROW(2) MAK_E_ROW(3)
        : MAK_E_OUT(0), MAK_E_OUT(1), MAK_E_OUT(2), MAK_E_OUT(3)
        : MAK_E_IN, MAK_E_LANE(0), MAK_E_LANE(1), MAK_E_LANE(2), MAK_E_LANE(3));
}
template <int R>
__device__ __forceinline__ void elim_first(zd* s, zd* x, const zd& b, double inv, zd& ws, zd& wx) {
  constexpr int K = R - 1;
  asm("v_mul_f64 %[wsx], %[bx], %[inv]\n\tv_mul_f64 %[wsy], %[by], %[inv]\n\t"
      "v_mul_f64 %[wxx], %[xkx], %[inv]\n\tv_mul_f64 %[wxy], %[xky], %[inv]\n\t" MAK_E_ROW(0)
      : MAK_E_OUT(0), [wsx] "=&v"(ws.x), [wsy] "=&v"(ws.y), [wxx] "=&v"(wx.x), [wxy] "=&v"(wx.y)
      : [bx] "v"(b.x), [by] "v"(b.y), [xkx] "v"(x[K].x), [xky] "v"(x[K].y), [inv] "v"(inv), MAK_E_LANE(0));
}
#undef MAK_E_OUT
#undef MAK_E_LANE
#undef MAK_E_ROW
#undef MAK_E_FMAC
#undef MAK_E_IN
// Step K: with the pivot d = s[K] of lane K and the pivot row b = s[K],
//   s[r] -= conj(b_r) s[K] / d,  x[r] -= conj(b_r) x[K] / d   (r > K).
// 1 / d is v_rcp_f64's y with its third-order correction, y (1 + e + e^2) with
// e = 1 - d y (|e| about 2^-23, so the cubic remainder is far below one ulp).
// Row K + 1, which holds the next pivot, is updated first, and the next
// pivot's reciprocal is formed between the other rows' updates (order_after
// keeps it there), so that the serial chain runs under them.
// dpp_source: the wait before a value that an asm block wrote becomes the DPP
// source of a compiler's instruction (the compiler sees no write in asm).
__device__ __forceinline__ void dpp_source(double& b) { asm("s_nop 1" : "+v"(b)); }
__device__ __forceinline__ void dpp_source(zd& b) { asm("s_nop 1" : "+v"(b.x), "+v"(b.y)); }
struct ElimPivot {
  double d, y, e, t, inv;
};
template <typename T, int K, int R0, int R1>
__device__ __forceinline__ void elim16_rows(T (&s)[16], T (&x)[16], const T& b, const T& ws, const T& wx) {
  if constexpr (R0 < R1) {
    constexpr int most = ScalarTraits<T>::is_complex ? 4 : 7, N = R1 - R0 < most ? R1 - R0 : most;
    elim_block<R0, N>(s, x, b, ws, wx);
    elim16_rows<T, K, R0 + N, R1>(s, x, b, ws, wx);
  }
}
template <typename T, int K>
__device__ __forceinline__ void elim16_step(T (&s)[16], T (&x)[16], int c0, double& piv, ElimPivot& p) {
  const T b = s[K];
  piv = sel(step_lane(c0) == K, p.d, piv);
  if constexpr (K < 15) {
    constexpr int n = 14 - K, R0 = K + 2, R1 = R0 + (n + 1) / 2, R2 = R1 + (16 - R1 + 2) / 3,
                  R3 = R2 + (16 - R2 + 1) / 2;
    T ws, wx;
    elim_first<K + 1>(s, x, b, p.inv, ws, wx);
    p.d = row_bcast<K + 1>(s_re(s[K + 1]));
    p.y = __builtin_amdgcn_rcp(p.d);
    order_after(ws, p.y);
    elim16_rows<T, K, R0, R1>(s, x, b, ws, wx);
    p.e = fma(-p.d, p.y, 1.0);
    order_after(ws, p.e);
    elim16_rows<T, K, R1, R2>(s, x, b, ws, wx);
    p.t = fma(p.e, p.e, p.e);
    order_after(ws, p.t);
    elim16_rows<T, K, R2, R3>(s, x, b, ws, wx);
    p.inv = fma(p.y, p.t, p.y);
    order_after(ws, p.inv);
    elim16_rows<T, K, R3, 16>(s, x, b, ws, wx);
  }
}
template <typename T, int... Ks>
__device__ __forceinline__ void elim16_steps(T (&s)[16], T (&x)[16], int c, double& piv,
                                             std::integer_sequence<int, Ks...>) {
  ElimPivot p;
  p.d = row_bcast<0>(s_re(s[0]));
  p.y = __builtin_amdgcn_rcp(p.d);
  p.e = fma(-p.d, p.y, 1.0);
  p.t = fma(p.e, p.e, p.e);
  p.inv = fma(p.y, p.t, p.y);
  (elim16_step<T, Ks>(s, x, c, piv, p), ...);
}
template <typename T, int... Ks>
__device__ __forceinline__ void elim16_scale(T (&x)[16], double rs, std::integer_sequence<int, Ks...>) {
  ((x[Ks] = s_scale(x[Ks], row_bcast<Ks>(rs))), ...);
}

// Lane c of every 16-lane row holds column c of the Hermitian block A in s
// (rows r <= c; the others hold anything: they only reach their own lane's
// s) and a column of any right-hand side B in x; on exit x = R^{-H} B with
// A = R^H R (B = A's upper triangle gives R, and B = I gives R^{-H}).
// Returns 0, or k + 1 for the first pivot k that is not positive (uniform;
// x is then unspecified).
template <typename T> __device__ __forceinline__ int wave_elim16(T (&s)[16], T (&x)[16], int c) {
  double piv = 1.0;
  elim16_steps<T>(s, x, c, piv, std::make_integer_sequence<int, 16>{});
  const unsigned m = (unsigned)__ballot(!(piv > 0.0)) & 0xffffu;
  elim16_scale<T>(x, rsqrt_nr(piv), std::make_integer_sequence<int, 16>{});
  return m ? __builtin_ctz(m) + 1 : 0;
}

// Cholesky with inverse of a 32 x 32 Hermitian positive definite block, by
// ONE wave (no workgroup barrier):
//   S (LDS, 32 x 33) holds the upper triangle on entry (rows/columns beyond the
//   active size padded with the identity by the caller); on exit S = W (upper,
//   zero below) with S_in = W^H W, and Y = W^{-1} (upper, zero below).  The
//   padding column of S (index 32) is used as scratch.
//   Returns 0, or j + 1 for the first pivot j that is not positive (uniform
//   over the wave; S and Y are then unspecified).
// Two eliminations by 16 pivots; all four 16-lane rows of the wave keep the
// diagonal block in s and eliminate a right-hand side each in x:
//   of S11:  I -> W11^{-H} = Y11^H,  S12 -> W12,  S11 -> W11,  0
//   then on MFMA  S22 -= W12^H W12,  H = W12^H Y11^H
//   of S22:  I -> Y22^H,  -H -> Y12^H,  S22 -> W22,  0
// (W^{-H} = [Y11^H 0; -Y22^H H, Y22^H]).  The zeros become the lower left
// blocks of W and Y, and the columns of I are read from the padding column of
// S, so that every lane loads and stores through one pointer without selects:
// one wave issues an instruction about every five cycles, and their number is
// what this costs.  Measured (one wave alone): 7.6e3 cycles Float64, 17.7e3
// ComplexF64 (of which the two eliminations 4.1e3 and 11e3), against 15.4e3 for
// an elimination of the whole [S | I] with its pivot rows through LDS
// (Float64) and 40.5e3 for 16 x 16 factorisations with readlane broadcasts
// (ComplexF64).
template <typename T> __device__ __forceinline__ int wave_chol_inv32(T (*S)[33], T (*Y)[33]) {
  const int l = lane_id(), c = l & 15, q = l >> 4;
  // loads of one array are issued together (left alone, the scheduler waits
  // for each before the next)
  auto pin = [](T (&a)[16]) {
    double* p = reinterpret_cast<double*>(&a[0]);
    constexpr int ND = 16 * sizeof(T) / sizeof(double);
#pragma unroll
    for (int h = 0; h < ND; h += 8)
      asm volatile("" : "+v"(p[h]), "+v"(p[h + 1]), "+v"(p[h + 2]), "+v"(p[h + 3]), "+v"(p[h + 4]), "+v"(p[h + 5]),
                        "+v"(p[h + 6]), "+v"(p[h + 7]));
  };
  // zeros below the diagonal of W's 16 x 16 block at D: the columns left of
  // the diagonal in row c, four per 16-lane row; the others write to the
  // padding column of Y.  A complex factor's diagonal is made exactly real.
  auto clear_lower = [&](T* D) {
    if constexpr (ScalarTraits<T>::is_complex)
      if (q == 0) D[34 * c].y = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = 4 * q + u;
      T* p = j < c ? D + 33 * c + j : &Y[c][32];
      *p = s_zero(T());
    }
  };
  if (l < 32) S[l][32] = l == 15 ? s_one(T()) : s_zero(T());
  wave_lds_sync();
  const T* eye = &S[15 - c][32];   // rows 0 .. 15: column c of I
  const T* none = &S[16][32];      // zeros
  T s[16], x[16];
  {
    const T* px = q == 0 ? eye : q == 1 ? &S[0][16 + c] : q == 2 ? &S[0][c] : none;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = S[r][c];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = px[33 * r];
    pin(s);
    pin(x);
  }
  int bad = wave_elim16<T>(s, x, c);
  if (q == 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) Y[c][r] = s_conj(x[r]);
  } else {
    T* p = q == 1 ? &S[0][16 + c] : q == 2 ? &S[0][c] : &S[16][c];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[33 * r] = x[r];
  }
  wave_lds_sync();
  {
    // The accumulators start from S22 and 0 and subtract the products, the last
    // four rows first.  Any order has the same error bound; with the rows in
    // ascending order the rounding of a 300 x 300 Gaussian matrix of condition 1.3e3
    // left ||Y^T Y - I|| above the 1e-11 that a test of the tile Cholesky asks,
    // where condition^2 u is 1.8e-10.
    v4d gr, hr = {0.0, 0.0, 0.0, 0.0}, gi = {0.0, 0.0, 0.0, 0.0}, hi = {0.0, 0.0, 0.0, 0.0};
    T w[4], h[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      w[u] = S[4 * u + q][16 + c];
      h[u] = Y[c][4 * u + q];
      const T old = S[16 + 4 * u + q][16 + c];
      gr[u] = s_re(old);
      if constexpr (ScalarTraits<T>::is_complex) gi[u] = s_im(old);
    }
    clear_lower(&S[0][0]);
#pragma unroll
    for (int u = 3; u >= 0; --u) {
      gr = mfma_f64(-s_re(w[u]), s_re(w[u]), gr);
      hr = mfma_f64(-s_re(w[u]), s_re(h[u]), hr);
      if constexpr (ScalarTraits<T>::is_complex) {
        // - conj(w) w and - conj(w) conj(h)
        gi = mfma_f64(-s_re(w[u]), s_im(w[u]), gi);
        hi = mfma_f64(s_re(w[u]), s_im(h[u]), hi);
        gr = mfma_f64(-s_im(w[u]), s_im(w[u]), gr);
        hr = mfma_f64(s_im(w[u]), s_im(h[u]), hr);
        gi = mfma_f64(s_im(w[u]), s_re(w[u]), gi);
        hi = mfma_f64(s_im(w[u]), s_re(h[u]), hi);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (ScalarTraits<T>::is_complex) {
        S[16 + 4 * u + q][16 + c] = mkz(gr[u], gi[u]);
        Y[4 * u + q][16 + c] = mkz(hr[u], hi[u]);
      } else {
        S[16 + 4 * u + q][16 + c] = gr[u];
        Y[4 * u + q][16 + c] = hr[u];
      }
    }
  }
  wave_lds_sync();
  {
    const T* px = q == 0 ? eye : q == 1 ? &Y[0][16 + c] : q == 2 ? &S[16][16 + c] : none;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = S[16 + r][16 + c];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = px[33 * r];
    pin(s);
    pin(x);
  }
  wave_lds_sync();
  const int b2 = wave_elim16<T>(s, x, c);
  if (bad == 0 && b2 != 0) bad = 16 + b2;
  if (q < 2) {
    T* p = q == 0 ? &Y[16 + c][16] : &Y[c][16];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = s_conj(x[r]);
  } else {
    T* p = q == 2 ? &S[16][16 + c] : &Y[16][c];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[33 * r] = x[r];
  }
  wave_lds_sync();
  clear_lower(&S[16][16]);
  wave_lds_sync();
  return bad;
}

}  // namespace mak
