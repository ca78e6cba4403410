// eig_tri_reg.hpp - workgroup-resident Householder tridiagonalisation for
// orders up to 256: the matrix lives in the registers of one workgroup from
// the load to the last column, so HBM sees the input once and the reflectors,
// d, e and beta once (the reference's hhsy2tr keeps its trailing update in
// 3 x 3 register tiles of a thread block, hhsy2tr.hpp:197-291; here the whole
// lower triangle is register-resident).
//
// Layout: strips of 64 rows x 16 columns (I, j), j < 4 (I + 1): lane l holds row
// 64 I + l, its 16 columns in 16 registers.  The strips of a diagonal block of 64
// hold the full symmetric block, so their row sums are complete and they give no
// column sums.  A wave owns whole columns of strips, so their column sums are added
// in the lane over all rows and cross the lanes once, and the waves stay balanced
// while the matrix shrinks.
//
// Column c (c = n-1 down to 1), A = the matrix after the update of column
// c + 1, A11 = A(0:c-1, 0:c-1), in the unblocked form's convention (anorm,
// beta, u_c in W(0:c-1, c), d, e of the split kernels):
//   x = A(c, 0:c-1), y = A(c-1, 0:c-1)
//   anorm = -sign(||x||, x_{c-1}), ul = x_{c-1} - anorm, beta = 1 / (ul anorm)
//   u = x with u_{c-1} = ul
//   p = beta A11 u = beta (A11 x - anorm y)      (A11 e_{c-1} = y)
//   alpha = beta / 2 (u . p)
//   A11 += u p^T + w u^T,  w = p + 2 alpha u    (= u v^T + v u^T, v = p + alpha u)
// Two workgroup barriers per column, which order LDS only (W is not waited for):
//   1. (every wave) norm, row and column sums of A11 x             | barrier
//   2. (thread i) p_i from the waves' sums in a fixed order, u_i   | barrier
//   3. (every wave) the rank-2 update of its strips; every wave forms its own copy
//      of the next column's x = row c-1 after this update from that row before it
//      and the rank-2 terms: x'_j = y_j + u_{c-1} p_j + w_{c-1} u_j, so the next
//      column starts without another barrier.
// The rows come from the strips NW at a time (a store to LDS costs the same for one
// lane as for eight), and each wave then keeps one of them up to date in LDS.
// Results do not depend on scheduling.
//
// What bounds it: 4 multiply-adds per element and column on the vector units (n = 256
// in FP64: 0.29 ms per matrix and compute unit), about as much LDS traffic for vectors
// of which every wave reads its own copy, and the chain norm - sums - p - alpha through
// two barriers; one matrix of 256 in FP64 takes 0.63 ms, 2.5 us a column.  The 16
// column operands of a strip come from the lanes of the row inside the FMA
// (bcast_dot16, bcast_axpy16): read from LDS as broadcasts, with 32 x 32 tiles in
// twelve waves, they bound the kernel.  Before and now: n = 256, FP64, 8192 matrices
// 29.8 and 20.6 ms; FP32, 2048 matrices 5.1 and 3.9; n = 128, 8192 matrices, FP64 6.1
// and 3.2, FP32 2.1 ms; 64 matrices of n = 200 in FP64 0.62 and 0.44 ms.
#pragma once
#include "common.hpp"
#include "eig_tri_again.hpp"

namespace eigmi {

// The strips of a wave.  NW = 4: wave w has the columns 4 i + w, i < NB, each down
// from its diagonal block; slots by column, known at compile time.  NW = 8 (NB = 4):
// wave w = 4 q + r has the columns w and 4 (3 - q) + r, five strips for every wave.
// The first slot of a column lies in the diagonal block.
template <int NB, int NW> struct TriSlots;
template <int NB> struct TriSlots<NB, 4> {
  static constexpr int NC = NB, KT = NB * (NB + 1) / 2;
  int wv;
  __device__ __forceinline__ explicit TriSlots(int w) : wv(w) {}
  static __device__ __forceinline__ constexpr int cidx(int k)
  {
    int i = 0;
    while (k >= NB - i) k -= NB - i, ++i;
    return i;
  }
  static __device__ __forceinline__ constexpr int row(int k)
  {
    int i = 0;
    while (k >= NB - i) k -= NB - i, ++i;
    return k + i;
  }
  __device__ __forceinline__ int col(int i) const { return 4 * i + wv; }
};
template <> struct TriSlots<4, 8> {
  static constexpr int NC = 2, KT = 5;
  int q, j0, j1;
  __device__ __forceinline__ explicit TriSlots(int w) : q(w >> 2), j0(w), j1(4 * (3 - (w >> 2)) + (w & 3)) {}
  __device__ __forceinline__ int cidx(int k) const { return (k == 4 || (k == 3 && q > 0)) ? 1 : 0; }
  __device__ __forceinline__ int row(int k) const { return cidx(k) ? k - 1 : k + q; }
  __device__ __forceinline__ int col(int i) const { return i ? j1 : j0; }
};

template <typename T, int NB, int NW>
struct alignas(16) TriRegLds {
  static constexpr int N = 64 * NB, NP = NW == 4 ? NB : NB + 1;
  alignas(16) T u[N];                                       // u of the current column, zero beyond c-1
  alignas(16) T p[N];
  alignas(16) T y[2 * NW][N];                               // rows waiting to become x: row r in slot r mod 2 NW
  alignas(16) T xw[NW][N];                                  // each wave's copy of x, zero beyond c-1
  alignas(16) T prow[NP][NW][64];                           // row sums by block row (NW = 4) or slot, and wave
  alignas(16) T pcol[N];                                    // column sums (columns left of the last active block)
  alignas(16) T d[N];
  alignas(16) T e[N];
  alignas(16) T beta[N];
  alignas(16) T red[NB];
};

// Row and column sums of the active strips (block rows <= ib).
template <typename T, int NB, int NW>
__device__ __forceinline__ void tr_sums(const T (&A)[TriSlots<NB, NW>::KT][16], const T *__restrict__ xw,
                                        TriRegLds<T, NB, NW> &S, const TriSlots<NB, NW> &sl, int wv, int lane, int c)
{
  typedef TriSlots<NB, NW> SL;
  const int ib = (c - 1) >> 6;
  T xc[SL::NC];
#pragma unroll
  for (int i = 0; i < SL::NC; ++i) xc[i] = xw[16 * sl.col(i) + (lane & 15)];
  auto reduce = [&](T (&v)[16], int j) {                    // over the 64 rows: lane ends with column lane >> 2
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = swap_sum<32>(v[i], v[i + 8]);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = swap_sum<16>(v[i], v[i + 4]);
    reduce_scatter_step<2>(v, (lane & 8) != 0, MvRM());
    reduce_scatter_step<1>(v, (lane & 4) != 0, MvHM());
    v[0] += lane_move(v[0], MvX2());
    v[0] += lane_move(v[0], MvX1());
    if ((lane & 3) == 0) S.pcol[16 * j + (lane >> 2)] = v[0];
  };
  // slots ka .. kb - 1 (the first one active)
  auto column = [&](int ka, int kb, int j) {
    T v[16];
#pragma unroll
    for (int k = ka; k < kb; ++k)
      if (k == ka || sl.row(k) <= ib) {
        const T ur = xw[64 * sl.row(k) + lane];
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) v[cc] = k == ka ? A[k][cc] * ur : fma_(A[k][cc], ur, v[cc]);
      }
    reduce(v, j);
  };
  if constexpr (NW == 4) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
      if (I <= ib) {
        T s0 = T(0), s1 = T(0);
#pragma unroll
        for (int k = 0; k < SL::KT; ++k)
          if (SL::row(k) == I) bcast_dot16(A[k], xc[SL::cidx(k)], s0, s1);
        S.prow[I][wv][lane] = s0 + s1;
      }
    int ka = 0;
#pragma unroll
    for (int i = 0; i + 1 < NB; ++i) {
      if (i < ib) column(ka + 1, ka + NB - i, sl.col(i));
      ka += NB - i;
    }
  } else {
#pragma unroll
    for (int k = 0; k < SL::KT; ++k)
      if (sl.row(k) <= ib) {
        T s0 = T(0), s1 = T(0);
        bcast_dot16(A[k], sl.cidx(k) ? xc[1] : xc[0], s0, s1);
        S.prow[k][wv][lane] = s0 + s1;
      }
    if (sl.q < ib) {
      T v[16];
      const T u1 = xw[64 * sl.row(1) + lane];
#pragma unroll
      for (int cc = 0; cc < 16; ++cc) v[cc] = A[1][cc] * u1;
#pragma unroll
      for (int k = 2; k < 4; ++k)
        if (sl.cidx(k) == 0 && sl.row(k) <= ib) {
          const T uk = xw[64 * sl.row(k) + lane];
#pragma unroll
          for (int cc = 0; cc < 16; ++cc) v[cc] = fma_(A[k][cc], uk, v[cc]);
        }
      reduce(v, sl.j0);
    }
    if (sl.q > 0 && ib == 3) column(4, 5, sl.j1);
  }
}

// The sum of row 64 b + lane over the strips of all waves and the column sums.
template <typename T, int NB, int NW>
__device__ __forceinline__ T tr_row_sum(const TriRegLds<T, NB, NW> &S, int b, int lane, int ib)
{
  T s = (b < ib) ? S.pcol[64 * b + lane] : T(0), s1 = T(0), s2 = T(0);
#pragma unroll
  for (int w = 0; w < 4; w += 2) {
    s += S.prow[b][w][lane];
    s1 += S.prow[b][w + 1][lane];
  }
  if constexpr (NW == 8) {
    // slot b of waves 0 .. 3, also slot 4 for b = 3; waves 4 .. 7: slot b - 1 of the
    // first column (b > 0), slot b + 1 of the second (b > 1)
    if (b == 3) s2 = (S.prow[4][0][lane] + S.prow[4][1][lane]) + (S.prow[4][2][lane] + S.prow[4][3][lane]);
    if (b > 0) {
#pragma unroll
      for (int w = 4; w < 8; w += 2) {
        s += S.prow[b - 1][w][lane];
        s1 += S.prow[b - 1][w + 1][lane];
      }
    }
    if (b > 1) {
#pragma unroll
      for (int w = 4; w < 8; w += 2) {
        s1 += S.prow[b + 1][w][lane];
        s2 += S.prow[b + 1][w + 1][lane];
      }
    }
  }
  return s + (s1 + s2);
}

// The rank-2 update of the active strips (row operands u, w; column operands uc, pc).
template <typename T, int NB, int NW>
__device__ __forceinline__ void tr_update(const TriSlots<NB, NW> &sl, int c, T (&A)[TriSlots<NB, NW>::KT][16],
                                          const T (&ur)[NB], const T (&wr)[NB], const T (&uc)[TriSlots<NB, NW>::NC],
                                          const T (&pc)[TriSlots<NB, NW>::NC])
{
  typedef TriSlots<NB, NW> SL;
  const int ib = (c - 1) >> 6;
#pragma unroll
  for (int k = 0; k < SL::KT; ++k) {
    if (sl.row(k) <= ib) {
      T ui, wi;
      if constexpr (NW == 4) {
        ui = ur[SL::row(k)];
        wi = wr[SL::row(k)];
        bcast_axpy16(A[k], uc[SL::cidx(k)], wi);
        bcast_axpy16(A[k], pc[SL::cidx(k)], ui);
      } else {
        constexpr int up[5] = {1, 2, 3, 2, 3};              // row(k) for q = 1; k, at most 3, for q = 0
        ui = sl.q ? ur[up[k]] : ur[k < 4 ? k : 3];
        wi = sl.q ? wr[up[k]] : wr[k < 4 ? k : 3];
        bcast_axpy16(A[k], sl.cidx(k) ? uc[1] : uc[0], wi);
        bcast_axpy16(A[k], sl.cidx(k) ? pc[1] : pc[0], ui);
      }
    }
  }
}

// Rows r, r-1, .. down to the next multiple of the number of waves into their slots
// of y (whole strips: what lies beyond the diagonal is not used).
template <typename T, int NB, int NW>
__device__ __forceinline__ void tr_publish(int r, const T (&A)[TriSlots<NB, NW>::KT][16],
                                           const TriSlots<NB, NW> &sl, int lane, TriRegLds<T, NB, NW> &S)
{
  const int lo = r & ~(NW - 1);
#pragma unroll
  for (int k = 0; k < TriSlots<NB, NW>::KT; ++k)
    if (sl.row(k) == (r >> 6)) {
      const int i = 64 * sl.row(k) + lane;
      if (i >= lo && i <= r) {
        T *__restrict__ y = &S.y[lane & (2 * NW - 1)][16 * sl.col(sl.cidx(k))];
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) y[cc] = A[k][cc];
      }
    }
}

// NB blocks of 64 rows (n <= 64 NB), NW waves; WPE waves per SIMD.
template <typename T, int NB, int NW, int WPE>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE))) void eig_tri_reg_kernel(
    int L, int nm, int n, const T *__restrict__ a, T *__restrict__ W, T *__restrict__ de, int ld,
    T *__restrict__ bws)
{
  constexpr int NT = 64 * NW, N = 64 * NB, KT = TriSlots<NB, NW>::KT, NC = TriSlots<NB, NW>::NC;
  __shared__ TriRegLds<T, NB, NW> S;
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const TriSlots<NB, NW> sl(wv);
  T *__restrict__ xw = S.xw[wv];
  T A[KT][16];
  bool again = false;

  for (long long mat = blockIdx.x; mat < L; mat += gridDim.x) {
    // n and nm re-read opaquely per matrix: otherwise the per-element load
    // addresses are hoisted out of the batch loop and held in registers for
    // the whole kernel
    int nv = n, nmv = nm, lane = tid & 63;
    asm volatile("" : "+s"(nv), "+s"(nmv), "+v"(lane));
    const T *__restrict__ Ain = a + (size_t)mat * (size_t)nm * (size_t)n;
    T *__restrict__ Wm = W + (size_t)mat * (size_t)n * (size_t)n;
    // lower (row, col) = Ain(min, max): the input's upper triangle.  Rows and
    // columns beyond n read a clamped in-range element: they only ever meet
    // zero entries of x, u and p.
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const int I = sl.row(k), col0 = 16 * sl.col(sl.cidx(k));
      if (col0 < 64 * I && 64 * I + 64 <= nv) {
        // below the diagonal block: 16 consecutive elements of input column `row`
        const T *__restrict__ src = Ain + (size_t)(64 * I + lane) * nmv + col0;
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) A[k][cc] = src[cc];
      } else {
        const int row = min(64 * I + lane, nv - 1);
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
          const int col = min(col0 + cc, nv - 1);
          const int lo = row < col ? row : col, hi = row < col ? col : row;
          A[k][cc] = Ain[lo + (size_t)hi * nmv];
        }
      }
    }
    for (int i = tid; i < N; i += NT) S.e[i] = S.beta[i] = T(0);
    // rows n-1 (x of the first column) and n-2 (its y)
    tr_publish<T, NB, NW>(nv - 1, A, sl, lane, S);
    if (((nv - 1) & (NW - 1)) == 0 && nv > 1) tr_publish<T, NB, NW>(nv - 2, A, sl, lane, S);
    __syncthreads();
    T sgl = T(0);
    // x of column c from its row before the last update, and that update's terms
    auto form_x = [&](int lane, int c, T uc, T wc, const T (&ur)[NB], const T (&pr)[NB], const T (&yr)[NB]) {
      sgl = T(0);
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        const int j = lane + 64 * m;
        const T v = fma_(wc, ur[m], fma_(uc, pr[m], yr[m]));
        const T x = (j < c) ? v : T(0);
        xw[j] = x;
        sgl = fma_(x, x, sgl);
      }
    };
    {
      T z[NB] = {}, y[NB];
#pragma unroll
      for (int m = 0; m < NB; ++m) y[m] = S.y[(nv - 1) & (2 * NW - 1)][64 * m + lane];
      form_x(lane, nv - 1, T(0), T(0), z, z, y);
    }
    if (tid == 0) S.d[nv - 1] = S.y[(nv - 1) & (2 * NW - 1)][nv - 1];

    const int lane_m = lane;
    for (int c = nv - 1; c >= 1; --c) {
      // three blocks in four waves: the lane-derived indices are formed again for every
      // column; held from before the loop they take registers that the strips need
      int lane = lane_m;
      if constexpr (NB == 3) asm volatile("" : "+v"(lane));
      // 1. norm, row and column sums of A11 x (x in this wave's copy)
      wsync();
      const T sg = wave_sum(sgl);
      const T xl = xw[c - 1];
      const T anorm = -sign_(sqrt_(sg), xl);
      const T ul = xl - anorm;
      const T beta = T(1) / nz(ul * anorm);
      const int ib = (c - 1) >> 6;                          // last active block
      tr_sums<T, NB, NW>(A, xw, S, sl, wv, lane, c);
      lds_barrier();                                        // sums complete
      // 2. p_i (thread i), u_i, the partial sums of u . p
      if (wv < NB) {
        const int i = 64 * wv + lane;
        const T s = tr_row_sum<T, NB, NW>(S, wv, lane, ib);
        const T pi = (i < c) ? beta * fma_(-anorm, S.y[(c - 1) & (2 * NW - 1)][i], s) : T(0);
        const T ui = (i == c - 1) ? ul : xw[i];             // x is 0 beyond c-1
        S.p[i] = pi;
        S.u[i] = ui;
        const T pu = wave_sum(pi * ui);
        if (lane == 0) S.red[wv] = pu;
      }
      if (tid == 0) {
        S.e[c - 1] = anorm;
        S.beta[c] = beta;
      }
      lds_barrier();                                        // p, u complete
      // every operand of the rest of the column is read at once: one latency
      const int r2 = c - 2, rw = (r2 & ~(NW - 1)) + wv;
      const bool fresh = r2 >= 0 && (r2 & (NW - 1)) == NW - 1, mine = r2 >= 0 && !fresh && rw <= r2;
      const T *__restrict__ yc = S.y[(c - 1) & (2 * NW - 1)];
      T *__restrict__ yw = S.y[rw & (2 * NW - 1)];
      const int rwc = mine ? rw : 0;
      T red[NB], ur[NB], pr[NB], yr[NB], ym[NB];
#pragma unroll
      for (int m = 0; m < NB; ++m) red[m] = S.red[m];
      const T uc = S.u[c - 1], pc = S.p[c - 1], uw = S.u[rwc], pw = S.p[rwc];
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        ur[m] = S.u[64 * m + lane];
        pr[m] = S.p[64 * m + lane];
      }
      T ucol[NC], pcol[NC];
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        ucol[i] = S.u[16 * sl.col(i) + (lane & 15)];
        pcol[i] = S.p[16 * sl.col(i) + (lane & 15)];
      }
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        yr[m] = yc[64 * m + lane];
        ym[m] = yw[64 * m + lane];
      }
      const T dd = yc[c - 1];
      T alpha = T(0);
#pragma unroll
      for (int m = 0; m < NB; ++m) alpha += red[m];
      const T alpha2 = alpha * beta;                        // 2 alpha
      // x of column c-1 = row c-1 after this update, from that row before it; d_{c-1} likewise
      const T wc = fma_(alpha2, uc, pc), ww = fma_(alpha2, uw, pw);
      form_x(lane, c - 1, uc, wc, ur, pr, yr);
      if (tid == 0) S.d[c - 1] = fma_(wc, uc, fma_(uc, pc, dd));
      if (mine) {
        // one of the rows that wait
#pragma unroll
        for (int m = 0; m < NB; ++m) yw[lane + 64 * m] = fma_(uw, pr[m], fma_(ww, ur[m], ym[m]));
      }
      if (wv == (c & (NW - 1))) {
#pragma unroll
        for (int m = 0; m < NB; ++m)
          if (lane + 64 * m < c) Wm[lane + 64 * m + (size_t)c * n] = ur[m];
      }
      // 3. rank-2 update of the active strips
#pragma unroll
      for (int m = 0; m < NB; ++m) pr[m] = fma_(alpha2, ur[m], pr[m]);
      tr_update<T, NB, NW>(sl, c, A, ur, pr, ucol, pcol);
      if (fresh) tr_publish<T, NB, NW>(r2, A, sl, lane, S);
    }
    __syncthreads();
    again = again || tri_lost(S.beta, n);
    for (int i = tid; i < nv; i += NT) {
      de[(size_t)i * ld + mat] = S.d[i];
      de[(size_t)(nv + i) * ld + mat] = S.e[i];
      bws[(size_t)mat * nv + i] = S.beta[i];
    }
    __syncthreads();
  }
  if (__builtin_expect(again, 0)) {
    // of this workgroup's matrices those that are lost (few, and none as a rule)
    for (long long mat = blockIdx.x; mat < L; mat += gridDim.x) {
      __syncthreads();                                      // every read of S is done
      for (int i = tid; i < n; i += NT) S.beta[i] = bws[(size_t)mat * n + i];
      __syncthreads();
      if (!tri_lost(S.beta, n) || !tri_again<T, NT>(mat, n, nm, a, W, S.u, S.p, S.d, S.e, S.beta, S.pcol)) continue;
      for (int i = tid; i < n; i += NT) {
        de[(size_t)i * ld + mat] = S.d[i];
        de[(size_t)(n + i) * ld + mat] = S.e[i];
        bws[(size_t)mat * n + i] = S.beta[i];
      }
    }
  }
}

} // namespace eigmi
