// eig_tri_wave.hpp - Householder tridiagonalisation with Q for 32 < n <= 64, and for
// 16 < n <= 32 in batches of up to 2048 matrices, one matrix per wave and no barrier: lane i holds row i of the full symmetric matrix
// in strips of 16 registers, so every product with it is lane-local and the column
// operands come from the lanes of the row inside the FMA (bcast_dot16, bcast_axpy16).
// The convention is that of the other tridiagonalisations (eig_tri_reg.hpp).
//
// The reflectors go to the place of Q; Q = H_{n-1} ... H_1 is then formed in the
// registers the matrix no longer needs, in blocks of 16 reflectors (compact WY) on
// the matrix cores: after blocks 0 .. b it differs from the identity only in its
// leading 16 (b + 1) rows and columns, so block b takes (b + 1)^2 tiles.  The
// accumulator layout of one product is the operand layout of the next (Mfma16).
//
// What bounds it: vector instructions, about 130 a column for the norm, the sums over
// lanes and the division and 48 for each strip it touches; Q is 280 matrix operations
// at n = 64.  Two sums over lanes, two LDS round trips a column, four waves a SIMD
// (FP32) to hide them.  Against eig_tri_kernel, where every column operand is moved
// across the lanes by itself and Q is formed by vector code: FP32, n = 64, 16384
// matrices 864 us, 552 here; n = 48, 65536 matrices 1774 and 1277; FP64, n = 60, 3000
// matrices 319 and 170; 16 matrices of n = 20 in FP32 21 and 15.
#pragma once
#include "common.hpp"
#include "eig_dc.hpp"
#include "eig_split.hpp"
#include "eig_symdmt.hpp"
#include "eig_tri_again.hpp"

namespace eigmi {

template <typename T>
struct alignas(16) TriWaveLds {
  alignas(16) T x[64], p[64];
  alignas(16) T G[16][16];
  alignas(16) T Tt[16][17];
};

// a[c mod 16] of strip c / 16 (c the same in every lane)
template <typename T, int NS>
__device__ __forceinline__ T tw_column(const T (&A)[NS][16], int c)
{
  T y = T(0);
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s == c >> 4) {
      T v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // as values: a conditional of two elements would be one of addresses
        const T lo = A[s][i], hi = A[s][i + 8];
        v[i] = (c & 8) ? hi : lo;
      }
#pragma unroll
      for (int h = 4; h >= 1; h >>= 1)
#pragma unroll
        for (int i = 0; i < h; ++i) {
          const T lo = v[i], hi = v[i + h];
          v[i] = (c & h) ? hi : lo;
        }
      y = v[0];
    }
  return y;
}

// NS = ceil(n / 16).  Q: n x n per matrix; d, e matrix-minor (de, ld rows apart).
// only (may be null): just the matrices flagged ST_OVERFLOW there.
template <typename T, int NS, int WPE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE))) void eig_tri_wave_kernel(
    int L, int nm, int n, const T *__restrict__ a, T *__restrict__ qws, T *__restrict__ de, int ld,
    const int *__restrict__ only)
{
  typedef typename Mfma16<T>::v4 v4;
  __shared__ TriWaveLds<T> S;
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const long long mat = blockIdx.x;
  if (mat >= L || (only && only[mat] != ST_OVERFLOW)) return;
  const T *__restrict__ Ain = a + (size_t)mat * (size_t)nm * (size_t)n;
  T *W = qws + (size_t)mat * (size_t)n * (size_t)n;
  T A[NS][16];
  const int row = lane < n ? lane : n - 1;
  // the input's upper triangle; rows and columns beyond n are zero
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int cc = 0; cc < 16; ++cc) {
      const int col = 16 * s + cc < n ? 16 * s + cc : n - 1;
      const int lo = row < col ? row : col, hi = row < col ? col : row;
      A[s][cc] = Ain[lo + (size_t)hi * nm];
    }
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int cc = 0; cc < 16; ++cc) A[s][cc] = (lane < n && 16 * s + cc < n) ? A[s][cc] : T(0);
  T dv = T(0), ev = T(0), bv = T(0);
  T x = tw_column<T, NS>(A, n - 1);
  dv = x;                                                   // lane n - 1 keeps it
  x = (lane < n - 1) ? x : T(0);
  for (int c = n - 1; c >= 1; --c) {
    const int ib = (c - 1) >> 4;
    S.x[lane] = x;
    wsync();
    T xc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) xc[s] = S.x[16 * s + m];
    const T sg = wave_sum(x * x);
    const T y = tw_column<T, NS>(A, c - 1);
    const T xl = lane_read(x, c - 1);
    const T anorm = -sign_(sqrt_(sg), xl);
    const T ul = xl - anorm;
    const T beta = T(1) / nz(ul * anorm);
    T s0 = T(0), s1 = T(0);
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s <= ib) bcast_dot16(A[s], xc[s], s0, s1);
    const T u = (lane == c - 1) ? ul : x;                   // zero from c on
    const T p = (lane < c) ? beta * fma_(-anorm, y, s0 + s1) : T(0);
    S.p[lane] = p;
    wsync();
    T pc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) pc[s] = S.p[16 * s + m];
    const T alpha2 = beta * wave_sum(p * u);
    const T w = fma_(alpha2, u, p);
    if (lane < c) W[lane + (size_t)c * n] = u;
    const T wl = lane_read(w, c - 1);
    const T xn = fma_(ul, p, fma_(wl, u, y));               // column c - 1 after the update
    dv = (lane == c - 1) ? xn : dv;
    ev = (lane == c - 1) ? anorm : ev;
    bv = (lane == c) ? beta : bv;
    x = (lane < c - 1) ? xn : T(0);
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s <= ib) {
        const T uc = (16 * s + m == c - 1) ? ul : xc[s];
        bcast_axpy16(A[s], uc, w);
        bcast_axpy16(A[s], pc[s], u);
      }
  }
  if (__builtin_expect(__ballot(tri_lost(bv)) != 0ull, 0)) {
    T *l = &S.G[0][0];
    if (tri_again<T, 64>(mat, n, nm, a, qws, S.x, S.p, l, l + 64, l + 128, l + 192)) {
      dv = lane < n ? l[lane] : T(0);
      ev = lane < n ? l[64 + lane] : T(0);
      bv = lane < n ? l[128 + lane] : T(0);
    }
  }
  if (lane < n) {
    de[(size_t)lane * ld + mat] = dv;
    de[(size_t)(n + lane) * ld + mat] = ev;
  }
  // the reflectors of the other lanes are read from here on
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  v4 Q[NS][NS];
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) Q[i][j][r] = (i == j && Mfma16<T>::row(g, r) == m) ? T(1) : T(0);
#pragma unroll
  for (int b = 0; b < NS; ++b) {
    const int cm = 16 * b + m;
    // Ut: u_{16 b + m} as rows of U^T; Ua: columns 16 b + row(g, r) of U
    T Ut[NS][4], Ua[NS][4];
#pragma unroll
    for (int t = 0; t <= b; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * t + Mfma16<T>::row(g, r), cr = 16 * b + Mfma16<T>::row(g, r), i = 16 * t + m;
        Ut[t][r] = W[(k < n ? k : n - 1) + (size_t)(cm < n ? cm : n - 1) * n];
        Ua[t][r] = W[(i < n ? i : n - 1) + (size_t)(cr < n ? cr : n - 1) * n];
      }
#pragma unroll
    for (int t = 0; t <= b; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * t + Mfma16<T>::row(g, r), cr = 16 * b + Mfma16<T>::row(g, r), i = 16 * t + m;
        Ut[t][r] = (cm < n && k < cm) ? Ut[t][r] : T(0);
        Ua[t][r] = (cr < n && i < cr) ? Ua[t][r] : T(0);
      }
    // T_jj = beta_j, T_j,0:j = beta_j (u_j^T U_0:j) T_0:j,0:j: lane m has column m
    v4 acc = v4{0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t <= b; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc = Mfma16<T>::op(Ut[t][r], Ut[t][r], acc);
    wsync();
#pragma unroll
    for (int r = 0; r < 4; ++r) S.G[Mfma16<T>::row(g, r)][m] = acc[r];
    wsync();
    T t[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      T v0 = (m == j) ? T(1) : T(0), v1 = T(0);
#pragma unroll
      for (int l0 = 0; l0 < j; l0 += 4) {
        T g4[4];
        ld4(&S.G[j][l0], g4);
#pragma unroll
        for (int l = 0; l < 4; ++l)
          if (l0 + l < j) {
            if (l & 1) v1 = fma_(g4[l], t[l0 + l], v1);
            else v0 = fma_(g4[l], t[l0 + l], v0);
          }
      }
      t[j] = (v0 + v1) * lane_read(bv, 16 * b + j);
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) S.Tt[j][m] = t[j];         // (the four rows of lanes write the same)
    wsync();
    T ta[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) ta[r] = S.Tt[m][Mfma16<T>::row(g, r)];
#pragma unroll
    for (int j = 0; j <= b; ++j) {
      v4 Y = v4{0, 0, 0, 0}, Z = v4{0, 0, 0, 0};
#pragma unroll
      for (int i = j == b ? b : 0; i <= b; ++i)             // column b of Q is still the identity's
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (i < b || j == b) Y = Mfma16<T>::op(Ut[i][r], Q[i][j][r], Y);
#pragma unroll
      for (int r = 0; r < 4; ++r) Z = Mfma16<T>::op(ta[r], Y[r], Z);
#pragma unroll
      for (int i = 0; i <= b; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) Q[i][j] = Mfma16<T>::op(Ua[i][r], Z[r], Q[i][j]);
    }
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int co = 16 * j + m;
    if (co < n) {
      T *__restrict__ o = W + (size_t)co * n;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        if (16 * i + 16 <= n) {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[16 * i + Mfma16<T>::row(g, r)] = Q[i][j][r];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (16 * i + Mfma16<T>::row(g, r) < n) o[16 * i + Mfma16<T>::row(g, r)] = Q[i][j][r];
        }
      }
    }
  }
}

} // namespace eigmi
