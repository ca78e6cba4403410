// eig_tri_again.hpp - the Householder reduction once more, for a matrix whose columns came
// so small that their squares underflowed.
//
// A matrix that is exhausted before its last column leaves rests of rounding errors, each
// eps times smaller than the one before: the all-ones matrix is at 1e-19 (FP32) or 1e-154
// (FP64) after a few columns, sums of squares there are subnormal or zero and 1 / (ul anorm)
// overflows.  The reductions of eig_tri_wave.hpp, eig_tri_reg.hpp and eig_tri_stream.hpp
// find that out from beta after their last column (a test in every column costs FP64
// n = 32, L = 1024 3 us of 84), and the workgroup starts again here (eig_tri_kernel for
// n <= 32 in its own form): the unblocked form in place in W, which sets a column to zero if its norm is below eps times the matrix's
// largest entry, a backward error of eps.  A matrix that is itself as small as that comes to
// the same end as before.
#pragma once
#include "common.hpp"

namespace eigmi {

// BETA: reflector scales above this send a matrix here.  SUM: sums of squares below this may
// have lost digits (512 of them, each off by half the smallest subnormal number).
template <typename T> struct TriTiny;
template <> struct TriTiny<float> { static constexpr float BETA = 1e38f, SUM = 1e-36f; };
template <> struct TriTiny<double> { static constexpr double BETA = 1e307, SUM = 1e-304; };

// A beta that calls for it (also one that is not a number); one of n in LDS (a wave's answer,
// the same in every wave).
template <typename T>
__device__ __forceinline__ bool tri_lost(T beta) { return !(abs_(beta) <= TriTiny<T>::BETA); }
template <typename T>
__device__ __forceinline__ bool tri_lost(const T *__restrict__ beta, int n)
{
  int i = threadIdx.x & 63;
  asm volatile("" : "+v"(i), "+s"(n));                      // as in tri_again
  bool lost = false;
#pragma unroll 1
  for (; i < n; i += 64) lost = lost || tri_lost(beta[i]);
  return __ballot(lost) != 0ull;
}

// Matrix mat of the batch a; its slot of Ws.  The convention of the callers: u_c in
// W(0:c-1, c), d, e, beta of n entries; u, p: n entries, red: one for every wave, all in LDS.
// All NT threads of the workgroup call it.  False, and nothing changed, for a matrix that is
// not finite.
template <typename T, int NT>
__device__ __forceinline__ bool tri_again(long long mat, int n, int nm, const T *__restrict__ a, T *Ws, T *u, T *p,
                                          T *d, T *e, T *beta, T *red)
{
  // opaque: nothing of this is computed, and held in registers, before the caller's columns
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid), "+s"(mat), "+s"(n), "+s"(nm));
  const T *__restrict__ Ain = a + (size_t)mat * (size_t)nm * (size_t)n;
  T *W = Ws + (size_t)mat * (size_t)n * (size_t)n;
  auto share = [&](T x) {
    __syncthreads();                                        // red of the sum before is read
    if ((tid & 63) == 0) red[tid >> 6] = x;
    __syncthreads();
  };
  auto sum = [&](T x) {
    share(wave_sum(x));
    T s = T(0);
    for (int q = 0; q < NT / 64; ++q) s += red[q];
    return s;
  };
  __syncthreads();                                          // the caller's stores to W are done
  T mx = T(0);                                              // the matrix's largest entry
  auto up = [&](T x) { mx = x > mx ? x : mx; };
  const T inf = std::numeric_limits<T>::infinity();
#pragma unroll 1
  for (int j = tid >> 6; j < n; j += NT / 64)
#pragma unroll 1
    for (int i = tid & 63; i <= j; i += 64) {
      const T x = abs_(Ain[i + (size_t)j * nm]);
      up(x < inf ? x : inf);
    }
  up(lane_move(mx, MvX1()));
  up(lane_move(mx, MvX2()));
  up(lane_move(mx, MvHM()));
  up(lane_move(mx, MvRM()));
  up(lane_move(mx, MvX16()));
  up(lane_move(mx, MvX32()));
  share(mx);
  for (int q = 0; q < NT / 64; ++q) up(red[q]);
  if (!(mx < inf)) return false;
#pragma unroll 1
  for (int j = tid >> 6; j < n; j += NT / 64)
#pragma unroll 1
    for (int i = tid & 63; i < n; i += 64)
      W[i + (size_t)j * n] = Ain[(i < j ? i : j) + (size_t)(i < j ? j : i) * nm];
  __syncthreads();
#pragma unroll 1
  for (int c = n - 1; c >= 1; --c) {
    T *col = W + (size_t)c * n;
    const T dc = col[c];
    T s = T(0);
    for (int i = tid; i < c; i += NT) s = fma_(col[i], col[i], s);
    T sg = sum(s);
    const bool zero = sg < TriTiny<T>::SUM && sqrt_(sg) <= eps_of<T>() * mx;
    if (zero) sg = T(0);
    const T xl = zero ? T(0) : col[c - 1];
    const T anorm = -sign_(sqrt_(sg), xl), ul = xl - anorm, b = T(1) / nz(ul * anorm);
    __syncthreads();                                        // every read of col[c - 1] is done
    for (int i = tid; i < c; i += NT) {
      const T x = zero ? T(0) : (i == c - 1 ? ul : col[i]);
      u[i] = col[i] = x;
    }
    if (tid == 0) {
      d[c] = dc;
      e[c - 1] = anorm;
      beta[c] = b;
    }
    __syncthreads();
    T t = T(0);
    for (int i = tid; i < c; i += NT) {
      T y = T(0);
#pragma unroll 8
      for (int j = 0; j < c; ++j) y = fma_(W[i + (size_t)j * n], u[j], y);
      y *= b;
      p[i] = y;
      t = fma_(y, u[i], t);
    }
    const T alpha = T(0.5) * b * sum(t);
    for (int i = tid; i < c; i += NT) p[i] = fma_(alpha, u[i], p[i]);
    __syncthreads();
#pragma unroll 1
    for (int j = tid >> 6; j < c; j += NT / 64) {
      const T uj = u[j], pj = p[j];
#pragma unroll 1
      for (int i = tid & 63; i < c; i += 64)
        W[i + (size_t)j * n] = fma_(u[i], pj, fma_(p[i], uj, W[i + (size_t)j * n]));
    }
    __syncthreads();
  }
  if (tid == 0) {
    d[0] = W[0];
    e[n - 1] = beta[0] = T(0);
  }
  __syncthreads();
  return true;
}

} // namespace eigmi
