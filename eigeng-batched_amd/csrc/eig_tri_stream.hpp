// eig_tri_stream.hpp - Householder tridiagonalisation for 256 < n <= 512, where
// the lower triangle (1 MB at n = 512 in FP64) no longer fits in one compute
// unit: it is streamed from L2 once per column.
//
// What bounds it: one workgroup per matrix reads c^2 / 2 elements for column c,
// and a compute unit takes about 64 bytes a clock from L2 (2.2 ms for n = 512 in
// FP64), so a strip is multiplied while the next one arrives, and everything else
// is kept short: five barriers a column that do not wait for memory, the vectors in
// LDS, sums through lane swaps.  FP64 with 8 waves and panels of 8 columns (16 waves
// spill: 9.0 ms), FP32 with 16 waves and panels of 16 (8 waves: 3.28 ms).
// Measured, 64 matrices: n = 512 FP64 5.5 ms (44.1 with eig_tri_large_kernel), FP32
// 3.1 ms (39.4); n = 300 FP64 1.85 ms (10.9); one matrix of 512 in FP64 5.1 ms.
//
// Storage of the live matrix: strips of 64 rows x 16 columns, contiguous, in
// 16-byte pieces of one row: strip 2 I (I + 1) + J holds rows 64 I .. and columns
// 16 J .., J < 4 (I + 1).  Below the diagonal blocks a strip gives row sums (in the
// lane) and column sums (a butterfly over the 64 rows); the four strips of a
// diagonal block hold the full symmetric block and give row sums only.  Every
// partial sum has a place of its own and they are added in a fixed order.
//
// Panels of NBP columns (the arrangement of eig_tri_large_kernel): the rank-2
// updates of a panel are kept as U_k, V_k in LDS and folded in analytically,
//   x = A(c, :) + sum_k (U_k V_k(c) + V_k U_k(c))
//   p = beta (A u + sum_k (U_k (V_k . u) + V_k (U_k . u)))
// and applied to the strips once per panel on the matrix cores ([U V] [V U]^T).
// The convention (anorm, beta, u_c in W(0:c-1, c), d, e) is that of the other
// tridiagonalisations.
#pragma once
#include "common.hpp"
#include "eig_symdmt.hpp"
#include "eig_tri_again.hpp"

namespace eigmi {

constexpr int TS_N = 512;
__host__ __device__ constexpr int ts_strips(int n) { return 2 * ((n + 63) / 64) * ((n + 63) / 64 + 1); }

template <typename T, int NBP, int TS_NW>
struct alignas(16) TriStreamLds {
  alignas(16) T U[NBP][TS_N], V[NBP][TS_N];
  alignas(16) T u[TS_N];                          // zero beyond c-1
  alignas(16) T pcol[TS_N / 64][TS_N];            // column sums of block row I
  alignas(16) T prow[TS_N / 64][TS_NW][64];       // row sums of block row I, by wave
  alignas(16) T d[TS_N], e[TS_N], beta[TS_N];
  alignas(16) T red[2][TS_NW];
  alignas(16) T dot[2 * NBP];
};

// element (row, col) of the matrix within its strip, and the strip's index
template <typename T>
__device__ __forceinline__ int ts_in(int row, int col)
{
  constexpr int VL = 16 / sizeof(T);
  const int cc = col & 15;
  return ((cc / VL) * 64 + (row & 63)) * VL + cc % VL;
}
__device__ __forceinline__ int ts_strip(int row, int col) { return 2 * (row >> 6) * ((row >> 6) + 1) + (col >> 4); }

template <typename T>
__device__ __forceinline__ void ts_load(const T *__restrict__ s, int lane, T (&v)[16])
{
  constexpr int VL = 16 / sizeof(T);
  typedef T vec __attribute__((ext_vector_type(VL)));
#pragma unroll
  for (int q = 0; q < 16 / VL; ++q) {
    const vec x = *(const vec *)(s + (q * 64 + lane) * VL);
#pragma unroll
    for (int t = 0; t < VL; ++t) v[VL * q + t] = x[t];
  }
}

template <typename T, int NBP, int TS_NT>
__global__ __launch_bounds__(TS_NT) void eig_tri_stream_kernel(int L, int nm, int n, const T *__restrict__ a,
                                                               T *__restrict__ W, T *__restrict__ strips,
                                                               long long sstride, T *__restrict__ de, int ld,
                                                               T *__restrict__ bws)
{
  typedef typename Mfma16<T>::v4 v4;
  constexpr int TS_NW = TS_NT / 64;
  __shared__ TriStreamLds<T, NBP, TS_NW> S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  bool again = false;
  for (long long mat = blockIdx.x; mat < L; mat += gridDim.x) {
    const T *__restrict__ A = a + (size_t)mat * (size_t)nm * (size_t)n;
    T *__restrict__ Wm = W + (size_t)mat * n * n;
    T *__restrict__ Sm = strips + (size_t)mat * sstride;
    // ---- the input's upper triangle into strips (zero beyond n) ---------------
    {
      const int ns = ts_strips(n);
      int I = 0;
      for (int s = wv; s < ns; s += TS_NW) {
        while (2 * (I + 1) * (I + 2) <= s) ++I;
        const int row = 64 * I + lane, col0 = 16 * (s - 2 * I * (I + 1));
        const int rc = row < n ? row : n - 1;
        T v[16];
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
          const int col = col0 + cc < n ? col0 + cc : n - 1;
          const int lo = rc < col ? rc : col, hi = rc < col ? col : rc;
          const T x = A[lo + (size_t)hi * nm];
          v[cc] = (row < n && col0 + cc < n) ? x : T(0);
        }
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) Sm[(size_t)s * 1024 + ts_in<T>(lane, cc)] = v[cc];
      }
    }
    for (int i = tid; i < TS_N; i += TS_NT) S.e[i] = S.beta[i] = T(0);
    for (int i = tid; i < NBP * TS_N; i += TS_NT) (&S.U[0][0])[i] = (&S.V[0][0])[i] = T(0);
    __syncthreads();

    // row c of the stored matrix (thread j: its element j)
    auto row_of = [&](int c) -> T {
      return (tid <= c && c >= 0) ? Sm[(size_t)ts_strip(c, tid) * 1024 + ts_in<T>(c, tid)] : T(0);
    };
    T arow = row_of(n - 1);
    int kk = 0;                                              // columns of the panel so far; U, V zero from there on
    for (int c = n - 1; c >= 1; --c) {
      // ---- 1. x = row c of the updated matrix, its norm ------------------------
      T x = T(0);
      if (wv < TS_N / 64) {
        T x1 = T(0);
        x = arow;
#pragma unroll
        for (int k = 0; k < NBP; ++k) {
          x = fma_(S.U[k][tid], S.V[k][c], x);
          x1 = fma_(S.V[k][tid], S.U[k][c], x1);
        }
        x += x1;
        if (tid == c) S.d[c] = x;
        x = (tid < c) ? x : T(0);
        const T sg = wave_sum(x * x);
        if (lane == 0) S.red[0][wv] = sg;
        S.u[tid] = x;
      }
      lds_barrier();
      T sig = T(0);
#pragma unroll
      for (int q = 0; q < TS_N / 64; ++q) sig += S.red[0][q];
      const T xl = S.u[c - 1];
      const T anorm = -sign_(sqrt_(sig), xl);
      const T ul = xl - anorm;
      const T beta = T(1) / nz(ul * anorm);
      const T u = (tid == c - 1) ? ul : x;
      if (tid < c) Wm[tid + (size_t)c * n] = u;
      arow = row_of(c - 1);                                  // arrives during the products
      const int nI = (c + 63) >> 6;
      // strip J of block row I goes to wave (J + 4 [I / 2 odd]) mod 8 (of 8; 16: the
      // upper waves take every second of them), so all waves get about the same
      // number: the k-th strip of a wave in block row I
      auto first = [&](int I) { return (wv + TS_NW - ((I >> 1) & 1) * 4) & (TS_NW - 1); };
      int I0 = 0;
      while (I0 < nI && first(I0) >= 4 * (I0 + 1)) ++I0;
      T va[16], vb[16];
      int I = I0, J = (I0 < nI) ? first(I0) : 0;
      ts_load(Sm + (size_t)(I < nI ? 2 * I * (I + 1) + J : 0) * 1024, lane, va);
      lds_barrier();                                         // every read of x(c-1) is done
      if (tid == c - 1) S.u[c - 1] = ul;
      if (tid < TS_N) S.U[kk][tid] = u;
      if (tid == 0) {
        S.e[c - 1] = anorm;
        S.beta[c] = beta;
      }
      lds_barrier();
      // ---- 2. A u by strips; the panel's dots with u -----------------------------
      for (int q = wv; q < 2 * kk; q += TS_NW) {
        const T *__restrict__ P = (q & 1) ? S.U[q >> 1] : S.V[q >> 1];
        T sm = T(0), sm1 = T(0);
#pragma unroll
        for (int j = 0; j < TS_N / 64; j += 2) {
          sm = fma_(P[64 * j + lane], S.u[64 * j + lane], sm);
          sm1 = fma_(P[64 * j + 64 + lane], S.u[64 * j + 64 + lane], sm1);
        }
        sm = wave_sum(sm + sm1);
        if (lane == 0) S.dot[q] = sm;
      }
      {
        // one block row after another; the next strip is loaded first
        auto mul = [&](T (&v)[16], int Ic, int Jc, T ur, T &rs0, T &rs1) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            T u8[8];
            ld8(&S.u[16 * Jc + 8 * h], u8);
#pragma unroll
            for (int cc = 0; cc < 8; cc += 2) {
              rs0 = fma_(v[8 * h + cc], u8[cc], rs0);
              rs1 = fma_(v[8 * h + cc + 1], u8[cc + 1], rs1);
            }
          }
          if (Jc < 4 * Ic) {
            // column sums over the 64 rows: lane ends with column lane >> 2
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = swap_sum<32>(v[i] * ur, v[i + 8] * ur);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = swap_sum<16>(v[i], v[i + 4]);
            reduce_scatter_step<2>(v, (lane & 8) != 0, MvRM());
            reduce_scatter_step<1>(v, (lane & 4) != 0, MvHM());
            v[0] += lane_move(v[0], MvX2());
            v[0] += lane_move(v[0], MvX1());
            if ((lane & 3) == 0) S.pcol[Ic][16 * Jc + (lane >> 2)] = v[0];
          }
        };
        T rs0 = T(0), rs1 = T(0);
        T ur = (I < nI) ? S.u[64 * I + lane] : T(0);
        for (int Iz = 0; Iz < I0 && Iz < nI; ++Iz) S.prow[Iz][wv][lane] = T(0);
        // (I, J) the strip in va; the one after it
        auto step = [&](T (&cur)[16], T (&nxt)[16]) {
          int In = I, Jn = J + TS_NW;
          while (In < nI && Jn >= 4 * (In + 1)) {
            ++In;
            Jn = first(In);
          }
          // always a load (of strip 0 past the last): with it under a branch the
          // wait for this strip would also wait for the next one
          ts_load(Sm + (size_t)(In < nI ? 2 * In * (In + 1) + Jn : 0) * 1024, lane, nxt);
          mul(cur, I, J, ur, rs0, rs1);
          if (In != I) {
            S.prow[I][wv][lane] = rs0 + rs1;
            rs0 = rs1 = T(0);
            for (int Iz = I + 1; Iz < In && Iz < nI; ++Iz) S.prow[Iz][wv][lane] = T(0);
            ur = (In < nI) ? S.u[64 * In + lane] : T(0);
          }
          I = In;
          J = Jn;
        };
        while (I < nI) {
          step(va, vb);
          if (I >= nI) break;
          step(vb, va);
        }
      }
      lds_barrier();
      // ---- 3. p, alpha, v ----------------------------------------------------------
      T p = T(0);
      if (wv < TS_N / 64) {
        T p1 = T(0);
#pragma unroll
        for (int q = 0; q < TS_NW; ++q) p += S.prow[wv][q][lane];
#pragma unroll
        for (int q = 1; q < TS_N / 64; ++q) {
          const T y = S.pcol[q][tid];
          p1 += (q > wv && q < nI) ? y : T(0);
        }
        p += p1;
        p1 = T(0);
#pragma unroll
        for (int k = 0; k < NBP; ++k) {
          const T du = S.dot[2 * k], dv = S.dot[2 * k + 1];
          p = fma_(S.U[k][tid], (k < kk) ? du : T(0), p);
          p1 = fma_(S.V[k][tid], (k < kk) ? dv : T(0), p1);
        }
        p = (tid < c) ? (p + p1) * beta : T(0);
        const T al = wave_sum(p * u);
        if (lane == 0) S.red[1][wv] = al;
      }
      lds_barrier();
      T alpha = T(0);
#pragma unroll
      for (int q = 0; q < TS_N / 64; ++q) alpha += S.red[1][q];
      alpha *= beta * T(0.5);
      if (tid < TS_N) S.V[kk][tid] = (tid < c) ? fma_(alpha, u, p) : T(0);
      ++kk;
      lds_barrier();
      // ---- 4. the panel into the strips -----------------------------------------------
      if (kk == NBP && c > 1) {
        // rows and columns below c, MFMA tile by tile: strip rows 16 q .., 2 NBP products deep
        const int mI = (c + 63) >> 6, ms = 2 * mI * (mI + 1);
        const int m = lane & 15, g = lane >> 4;
        int I = 0;
        for (int s = wv; s < ms; s += TS_NW) {
          while (2 * (I + 1) * (I + 2) <= s) ++I;
          const int r0 = 64 * I, j0 = 16 * (s - 2 * I * (I + 1));
          T *__restrict__ Ps = Sm + (size_t)s * 1024;
          v4 acc[4];
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[q][r] = Ps[ts_in<T>(16 * q + Mfma16<T>::row(g, r), m)];
#pragma unroll
          for (int k0 = 0; k0 < NBP; k0 += 4) {
            const T bu = S.U[k0 + g][j0 + m], bv = S.V[k0 + g][j0 + m];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              acc[q] = Mfma16<T>::op(S.U[k0 + g][r0 + 16 * q + m], bv, acc[q]);
              acc[q] = Mfma16<T>::op(S.V[k0 + g][r0 + 16 * q + m], bu, acc[q]);
            }
          }
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) Ps[ts_in<T>(16 * q + Mfma16<T>::row(g, r), m)] = acc[q][r];
        }
        kk = 0;
        __syncthreads();
        arow = row_of(c - 1);
        for (int i = tid; i < NBP * TS_N; i += TS_NT) (&S.U[0][0])[i] = (&S.V[0][0])[i] = T(0);
        lds_barrier();
      }
    }
    // d(0): row 0 of the updated matrix
    if (tid == 0) {
      T x = arow;
      for (int k = 0; k < kk; ++k) x = fma_(S.U[k][0], S.V[k][0], fma_(S.V[k][0], S.U[k][0], x));
      S.d[0] = x;
    }
    __syncthreads();
    again = again || tri_lost(S.beta, n);
    for (int i = tid; i < n; i += TS_NT) {
      de[(size_t)i * ld + mat] = S.d[i];
      de[(size_t)(n + i) * ld + mat] = S.e[i];
      bws[(size_t)mat * n + i] = S.beta[i];
    }
    __syncthreads();
  }
  if (__builtin_expect(again, 0)) {
    // as in eig_tri_reg_kernel
    for (long long mat = blockIdx.x; mat < L; mat += gridDim.x) {
      __syncthreads();
      for (int i = tid; i < n; i += TS_NT) S.beta[i] = bws[(size_t)mat * n + i];
      __syncthreads();
      if (!tri_lost(S.beta, n) ||
          !tri_again<T, TS_NT>(mat, n, nm, a, W, S.U[0], S.V[0], S.d, S.e, S.beta, S.dot))
        continue;
      for (int i = tid; i < n; i += TS_NT) {
        de[(size_t)i * ld + mat] = S.d[i];
        de[(size_t)(n + i) * ld + mat] = S.e[i];
        bws[(size_t)mat * n + i] = S.beta[i];
      }
    }
  }
}

} // namespace eigmi
