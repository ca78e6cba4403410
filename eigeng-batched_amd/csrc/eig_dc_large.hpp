// eig_dc_large.hpp - divide and conquer (eig_dc.hpp) for 64 < n <= 512: the blocks
// of 64 columns by eig_dc_kernel, then the merges above them, one workgroup per
// node and one product kernel per level, and the back-transformation.
//
//   eig_dc_merge_kernel   steps 1-4 of a merge for nodes of up to S columns: ranks,
//                         roots (NLR lanes each), z from the roots; U to HBM
//   eig_dc_update_kernel  Q <- diag(Q1, Q2) U of every node of the level on the
//                         matrix cores (the tile loop of eig_gemm.hpp)
//   eig_dc_wyt_kernel     T factors of the reflectors in blocks of 16 (compact WY)
//   eig_dc_back_kernel    V <- H_{n-1} ... H_1 V, 16 columns of V per wave held in
//                         registers from the first block of reflectors to the last
// A node of a tree level reads its children from one buffer and leaves its vectors
// in the other; which buffer a block starts in follows from its depth.
#pragma once
#include "common.hpp"
#include "eig_dc.hpp"
#include "eig_gemm.hpp"

namespace eigmi {

// The merges of one level: columns [base, mid) with [mid, end).
struct DcNodes {
  int cnt;
  short base[4], mid[4], end[4];
};

template <typename T, int S>
struct alignas(16) DcMergeLds {
  alignas(16) T d[S], key[S], dl[S], zq[S], zs[S];
  alignas(16) T da[S], tau[S], val[S];
  alignas(16) T zk[S], dk[S], ma[S], mt[S];
  alignas(16) int src[S], mdef[S];
  int flag[16];
  int lost;                                        // as in DcLds
};

// One workgroup per (matrix, node).  w: the eigenvalues of the blocks, replaced by
// the nodes'.  Zc: the children's vectors.  U: the node's vectors, at (base, base)
// of an n x n slot.  A node that fails leaves infinities for its eigenvalues.  The last
// level (st not null) reports per matrix: st = 1 leaves the matrix out of the final
// products (a merge failed, or not finite and nanfail), info.
template <typename T, int S, int NLR>
__global__ __launch_bounds__(S *NLR) void eig_dc_merge_kernel(int n, DcNodes nodes, const T *__restrict__ de, int ld,
                                                              T *__restrict__ w, const T *__restrict__ Zc,
                                                              T *__restrict__ U, int *__restrict__ st,
                                                              int *__restrict__ info, int nanfail, int maxit)
{
  constexpr int NTH = S * NLR, NW = NTH / 64;
  __shared__ DcMergeLds<T, S> Sh;
  const T eps = eps_of<T>(), HUGE_ = DcLim<T>::HUGE_;
  const int tid = threadIdx.x, i = tid / NLR, sub = tid % NLR, wv = tid >> 6, lane = tid & 63;
  const int mat = blockIdx.x / nodes.cnt, nd_ = blockIdx.x - mat * nodes.cnt;
  const int base = nodes.base[nd_], h = nodes.mid[nd_] - base, s = nodes.end[nd_] - base;
  T *__restrict__ wm = w + (size_t)mat * n + base;
  const T *__restrict__ Z = Zc + (size_t)mat * n * n;
  T *__restrict__ Um = U + (size_t)mat * n * n + (size_t)base * n + base;

  // ---- 1. z, scale, the poles set aside, ranks -----------------------------------
  const bool lv = i < s;
  const T er0 = de[(size_t)(n + base + h - 1) * ld + mat];
  const T d0 = lv ? wm[i] : T(0);
  T z = T(0);
  if (lv) z = (i < h) ? Z[(size_t)(base + i) * n + base + h - 1] : Z[(size_t)(base + i) * n + base + h];
  // the children are sorted, so their ends bound them
  const T q0 = abs_(wm[0]), q1 = abs_(wm[h - 1]), q2 = abs_(wm[h]), q3 = abs_(wm[s - 1]);
  const bool bad = !finite_(d0) || !finite_(z) || !finite_(er0);
  const int code = (__ballot(bad) != 0ull ? 1 : 0) | (__ballot(abs_(d0) == std::numeric_limits<T>::infinity()) != 0ull ? 2 : 0);
  if (lane == 0) Sh.flag[wv] = code;
  if (tid == 0) Sh.lost = 0;
  __syncthreads();
  int codes = 0;
#pragma unroll
  for (int q = 0; q < NW; ++q) codes |= Sh.flag[q];
  if (codes) {
    // everything of this node: NaN (the products spread it), or infinite where a merge failed
    const T nan = std::numeric_limits<T>::quiet_NaN();
    const bool fail = nanfail || (codes & 2);
    if (lv && sub == 0) wm[i] = (codes & 2) ? std::numeric_limits<T>::infinity() : nan;
    for (int m = wv; m < s; m += NW)
      for (int k = lane; k < s; k += 64) Um[(size_t)m * n + k] = nan;
    if (st && tid == 0) {
      st[mat] = fail ? 1 : 0;
      if (info) info[mat] = fail ? 1 : 0;
    }
    return;
  }
  int ex = 0;
  const T mx = max_(max_(max_(q0, q1), max_(q2, q3)), abs_(er0));
  if (mx > T(0)) (void)frexp(mx, &ex);
  ex = max(min(ex, DcLim<T>::EXP), -DcLim<T>::EXP);
  const T sc = ldexp(T(1), -ex), isc = ldexp(T(1), ex);
  const T er = er0 * sc, rho = abs_(er), dmax = mx * sc;
  const T di = lv ? d0 * sc : HUGE_ * T(2);
  if (i >= h) z *= sign_(T(1), er);
  const bool nd = lv && rho * abs_(z) > T(2) * eps * dmax;
  const T key = nd ? di : HUGE_ * (T(1) + T(i) * T(1.0 / 1024));
  if (sub == 0) {
    Sh.d[i] = di;
    Sh.key[i] = key;
  }
  __syncthreads();
  const int nq = (s + 4 * NLR - 1) / (4 * NLR);
  int c = 0, k = 0;
#pragma unroll 4
  for (int q = 0; q < nq; ++q) {
    T k4[4];
    ld4(&Sh.key[4 * (NLR * q + sub)], k4);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      c += (k4[v] < key) ? 1 : 0;
      k += (k4[v] < HUGE_) ? 1 : 0;
    }
  }
  // the slots beyond the node's count themselves
  if (i >= 4 * NLR * nq) c = i;
  else c = lanes_sum<NLR>(c);
  k = lanes_sum<NLR>(k);
  auto put = [&]() {
    if (sub == 0) {
      Sh.dl[c] = key;
      Sh.zs[c] = nd ? z : T(0);
      Sh.zq[c] = nd ? z * z : T(0);
      Sh.src[c] = i;
    }
  };
  put();
  __syncthreads();
  {
    // equal poles and poles closer than one ulp: put right in order (rare)
    const T gmin = eps * max_(abs_(Sh.dl[i > 0 ? i - 1 : 0]), dmax * T(1.0 / 4096));
    const bool rep = Sh.src[c] != i || (i > 0 && i < k && !(Sh.dl[i] - Sh.dl[i > 0 ? i - 1 : 0] >= gmin));
    const bool any = __ballot(rep) != 0ull;
    __syncthreads();
    if (lane == 0) Sh.flag[wv] = any ? 1 : 0;
    __syncthreads();
    bool fix = false;
#pragma unroll
    for (int q = 0; q < NW; ++q) fix = fix || Sh.flag[q] != 0;
    if (fix) {
      int tie = 0;
      for (int j = 0; j < i; ++j) tie += (Sh.key[j] == key) ? 1 : 0;
      c += tie;
      __syncthreads();
      put();
      __syncthreads();
      if (tid == 0) {
        T pv = Sh.dl[0];
        for (int j = 1; j < k; ++j) {
          const T g = eps * max_(abs_(pv), dmax * T(1.0 / 4096));
          T x = Sh.dl[j];
          if (x - pv < g) {
            x = pv + g;
            Sh.dl[j] = x;
          }
          pv = x;
        }
      }
      __syncthreads();
    }
  }
  // ---- 2. roots --------------------------------------------------------------------
  const bool root = i < k;
  bool ok = true;
  T da = HUGE_, tau = T(0);
  {
    T a0 = T(0), t0 = T(0);
    if (__ballot(root)) ok = dc_root<T, S, NLR, false>(Sh.dl, Sh.zq, k, i, sub, rho, root, maxit, a0, t0);
    if (root) { da = a0; tau = t0; }
  }
  const int s0 = Sh.src[i] & (S - 1);
  const T v0 = root ? da + tau : Sh.d[s0];
  if (sub == 0) {
    Sh.da[i] = da;
    Sh.tau[i] = tau;
    Sh.val[i] = v0;
  }
  __syncthreads();
  // ---- 3. z from the roots; new order ------------------------------------------------
  {
    T z2 = T(0);
    if (__ballot(root)) z2 = dc_zhat2<T, S, NLR, false>(Sh.dl, Sh.da, Sh.tau, k, root ? i : 0, sub);
    if (root && !(ok && z2 > T(0) && finite_(z2))) Sh.lost = 1;
    int nr = i;
    if (k < s) {
      nr = 0;
#pragma unroll 4
      for (int q = 0; q < nq; ++q) {
        const int j0 = 4 * (NLR * q + sub);
        T w4[4];
        ld4(&Sh.val[j0], w4);
#pragma unroll
        for (int v = 0; v < 4; ++v) nr += (w4[v] < v0 || (w4[v] == v0 && j0 + v < i)) ? 1 : 0;
      }
      if (i >= 4 * NLR * nq) nr = i;
      else nr = lanes_sum<NLR>(nr);
    }
    if (sub == 0) {
      Sh.zk[s0] = root ? sign_(qsqrt_(z2), Sh.zs[i]) : T(0);
      Sh.dk[s0] = root ? Sh.dl[i] : HUGE_;
      Sh.ma[nr] = da;
      Sh.mt[nr] = tau;
      Sh.mdef[nr] = root ? -1 : s0;
      if (nr < s) wm[nr] = v0 * isc;
    }
  }
  __syncthreads();
  const bool lost = Sh.lost != 0;
  if (st && tid == 0) {
    st[mat] = lost ? 1 : 0;
    if (info) info[mat] = lost ? 1 : 0;
  }
  if (lost && lv && sub == 0) wm[i] = std::numeric_limits<T>::infinity();
  // ---- 4. U, one column per wave at a time ----------------------------------------------
  for (int m = wv; m < s; m += NW) {
    const T a = Sh.ma[m], t0 = Sh.mt[m];
    const int def = Sh.mdef[m];
    T u[S / 64];
    T ss = T(0);
#pragma unroll
    for (int q = 0; q < S / 64; ++q) {
      const int kc = 64 * q + lane;
      const T x = (Sh.dk[kc] - a) - t0;
      T v = (def >= 0) ? (kc == def ? T(1) : T(0)) : Sh.zk[kc] * rcp_(x);
      v = (kc < s) ? v : T(0);
      u[q] = v;
      ss = fma_(v, v, ss);
    }
    ss = group_sum<64>(ss);
    const T inv = rsqrt_nr(ss);
#pragma unroll
    for (int q = 0; q < S / 64; ++q)
      if (64 * q + lane < s) Um[(size_t)m * n + 64 * q + lane] = u[q] * inv;
  }
}

// Zn <- Zc U for every node of the level: one workgroup per 64 x 64 tile of a
// node's s x s vectors; a tile's rows lie in one child (h is a multiple of 64), so
// its contraction runs over that child's columns only.
template <typename T>
__global__ __launch_bounds__(GM_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void eig_dc_update_kernel(
    int cur, int n, DcNodes nodes, int tiles, const T *__restrict__ Zc, const T *__restrict__ U, T *__restrict__ Zn)
{
  constexpr int KIND = sizeof(T) == 8 ? GK_F64 : GK_F32;
  typedef typename GemmT<KIND>::v4 v4;
  __shared__ GemmLds<KIND> Sm;
  const long long total = (long long)tiles * cur;
  const long long lid = gemm_xcd_remap(blockIdx.x, total);
  const int b = (int)(lid / tiles);
  int t = (int)(lid - (long long)b * tiles), nd = 0, base, mid, end, nt;
  for (;;) {
    base = nodes.base[nd], mid = nodes.mid[nd], end = nodes.end[nd];
    nt = (end - base + 63) >> 6;
    if (t < nt * nt || nd == nodes.cnt - 1) break;
    t -= nt * nt;
    ++nd;
  }
  const int ti = t % nt, tj = t / nt;
  const int r0 = base + 64 * ti, c0 = base + 64 * tj;
  const int cb = r0 < mid ? base : mid, ce = r0 < mid ? mid : end;
  const size_t off = (size_t)b * n * n;
  v4 acc[2][2], acc2[2][2];
  gemm_tile<KIND>(ce - cb, end - base, ce - cb, 0, 0, Zc + off + (size_t)cb * n + cb, n, U + off + (size_t)base * n + cb,
                  n, r0 - cb, c0 - base, Sm, acc, acc2);
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6, m = lane & 15, g = lane >> 4;
  T *__restrict__ O = Zn + off;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = r0 + (q & 1) * 32 + 16 * x + GemmMma<KIND>::row(g, r), j = c0 + (q >> 1) * 32 + 16 * y + m;
        if (i < ce && j < end) O[(size_t)j * n + i] = acc[x][y][r];
      }
}

// ---- back-transformation -------------------------------------------------------------
// H_c = I + beta_c u_c u_c^T, u_c in rows 0..c-1 of column c of W.  Blocks of 16:
// H_{c0+15} ... H_{c0} = I + U T U^T with T lower triangular, T_jj = beta_j and
// T_j,0:j = beta_j (u_j^T U_0:j) T_0:j,0:j.  One wave per block: G = U^T U on the
// matrix cores, then the 16 rows of T in LDS.  T is stored in A-operand order.
template <typename T>
__global__ __launch_bounds__(256) void eig_dc_wyt_kernel(long long blocks, int n, int nb16, const T *__restrict__ W,
                                                         const T *__restrict__ bw, T *__restrict__ Tm)
{
  typedef typename Mfma16<T>::v4 v4;
  __shared__ T Gs[4][16][17], Ts[4][16][17];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const long long q = (long long)blockIdx.x * 4 + wv;
  if (q >= blocks) return;                                  // the whole wave; no workgroup barrier below
  const long long mat = q / nb16;
  const int c0 = 16 * (int)(q - mat * nb16), c = c0 + m, cc = c < n ? c : n - 1;
  const T *__restrict__ u = W + (size_t)mat * n * n + (size_t)cc * n;
  v4 acc = v4{0, 0, 0, 0};
  for (int t = 0; t <= c0 / 16; ++t) {
    T a[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 16 * t + Mfma16<T>::row(g, r);
      const T x = u[k < n ? k : n - 1];
      a[r] = (c < n && k < c) ? x : T(0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) acc = Mfma16<T>::op(a[r], a[r], acc);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) Gs[wv][Mfma16<T>::row(g, r)][m] = acc[r];
  wsync();
  const T beta = (c >= 1 && c < n) ? bw[(size_t)mat * n + cc] : T(0);
  for (int j = 0; j < 16; ++j) {
    const T bj = lane_bcast(beta, j);
    if (lane < 16) {
      T v = T(0);
      for (int l = m; l < j; ++l) v = fma_(Gs[wv][j][l], Ts[wv][l][m], v);
      Ts[wv][j][m] = (m < j) ? bj * v : (m == j ? bj : T(0));
    }
    wsync();
  }
  T *__restrict__ o = Tm + (size_t)q * 256 + 4 * lane;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = Ts[wv][m][Mfma16<T>::row(g, r)];
}

// V: columns of Zs (ld n), 16 per wave, all NT row tiles in registers; per block
// of reflectors P = U^T V (rows up to the block), P <- T P, V <- V + U P, the
// accumulator layout of one product being the operand layout of the next.  The four
// waves of a workgroup share the block through LDS (columns below the diagonal as
// they are, zeros elsewhere), the next block's loads in flight meanwhile; a column
// has BS elements there, which puts the 16 columns of an operand on different banks.
// Loads are not clamped to the matrix: they stay within the workspace (16 NT - n
// rows past a column, 15 columns past the last), whose regions of eigenvectors
// follow W's, and what lies outside u_c is replaced by zero.  Result to a (ld nm,
// columns below mcols).
// What bounds it: the matrix cores wait for one LDS operand per instruction (n = 256 in
// FP64: 4 n^3 operations are 3.8 of 8192 matrices' 7.1 ms).  With every wave reading the
// reflectors for itself, twice, from L2, the whole back-transformation took 14.6 ms, now
// 8.2; n = 128 in FP32 1.14 and 0.88; 64 matrices of n = 512 in FP64 1.00 and 0.58.
template <typename T, int NT, int WPE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void eig_dc_back_kernel(
    int cur, int n, int nm, int mcols, int ncg, const T *__restrict__ W, const T *__restrict__ Tm,
    const T *__restrict__ Zs, T *__restrict__ a, const int *__restrict__ st)
{
  typedef typename Mfma16<T>::v4 v4;
  constexpr int NR = 16 * NT, BS = NR + (sizeof(T) == 8 ? 2 : 4);
  __shared__ T Ub[16 * BS];
  const long long total = (long long)cur * ncg, lid = gemm_xcd_remap(blockIdx.x, total);
  const int mat = (int)(lid / ncg), cg = (int)(lid - (long long)mat * ncg);
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, m = lane & 15, g = lane >> 4;
  if (st[mat] != 0) return;                                 // the whole workgroup
  const int col = 64 * cg + 16 * wv + m;
  const int nb16 = (n + 15) >> 4;
  const T *__restrict__ Wm = W + (size_t)mat * n * n;
  const T *__restrict__ Zm = Zs + (size_t)mat * n * n + (size_t)(col < n ? col : n - 1) * n;
  v4 V[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 16 * t + Mfma16<T>::row(g, r);
      const T x = Zm[k];
      V[t][r] = (k < n) ? x : T(0);
    }
  // thread t of the workgroup: rows (t & 63) + 64 i of the columns (t >> 6) + 4 j
  constexpr int NI = NR / 64;
  T x[NI][4];
  auto load = [&](int b) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (4 * i <= b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[i][j] = Wm[(size_t)(16 * b + (tid >> 6) + 4 * j) * n + (tid & 63) + 64 * i];
      }
  };
  load(0);
#pragma unroll 1
  for (int b = 0; b < nb16; ++b) {
    __syncthreads();                                        // the block before is used up
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (4 * i <= b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = 16 * b + (tid >> 6) + 4 * j, k = (tid & 63) + 64 * i;
          Ub[((tid >> 6) + 4 * j) * BS + k] = (k < c && c < n) ? x[i][j] : T(0);
        }
      }
    const T *__restrict__ tp = Tm + ((size_t)mat * nb16 + b) * 256 + 4 * lane;
    T ta[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) ta[r] = tp[r];
    __syncthreads();
    load(b + 1 < nb16 ? b + 1 : b);
    v4 P0 = v4{0, 0, 0, 0}, P1 = v4{0, 0, 0, 0};
#pragma unroll
    for (int G = 0; G < NT / 4; ++G) {
      if (4 * G <= b) {
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const T y = Ub[m * BS + 16 * (4 * G + tt) + Mfma16<T>::row(g, r)];
            if (tt & 1) P1 = Mfma16<T>::op(y, V[4 * G + tt][r], P1);
            else P0 = Mfma16<T>::op(y, V[4 * G + tt][r], P0);
          }
      }
    }
    v4 Q = v4{0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < 4; ++r) Q = Mfma16<T>::op(ta[r], P0[r] + P1[r], Q);
#pragma unroll
    for (int G = 0; G < NT / 4; ++G) {
      if (4 * G <= b) {
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            V[4 * G + tt] = Mfma16<T>::op(Ub[Mfma16<T>::row(g, r) * BS + 16 * (4 * G + tt) + m], Q[r], V[4 * G + tt]);
      }
    }
  }
  if (col < mcols) {
    T *__restrict__ A = a + (size_t)mat * (size_t)nm * (size_t)n + (size_t)col * nm;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * t + Mfma16<T>::row(g, r);
        if (k < n) A[k] = V[t][r];
      }
  }
}

} // namespace eigmi
