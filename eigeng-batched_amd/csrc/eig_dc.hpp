// eig_dc.hpp - divide and conquer for the symmetric tridiagonal eigenproblem
// (rank-one tearing, Cuppen, Numer. Math. 36, 1981), the default after the
// Householder reduction for the sorted IMTQL2 interface: the implicit QL
// recurrence is one serial chain per matrix and the replay of its rotations a
// second one through the columns, while here every root of a merge is
// independent and the eigenvectors are updated by matrix-core products.
//
//   T = diag(T1, T2) + rho v v^T at every second off-diagonal (rho = |e|), the
//   2 x 2 leaves in closed form, then merges 4, 8, 16, ...: with T1 = Q1 D1 Q1^T,
//   T2 = Q2 D2 Q2^T and z = (last row of Q1, sign(e) first row of Q2),
//   T = Q (D + rho z z^T) Q^T.
//
// One merge of a node of s columns:
//   1. poles with rho |z_j| <= 2 eps max(|d|, rho) are set aside as they are
//      (their column passes through); the others are ranked in ascending order
//      (counting, no sort).  Equal or nearly equal poles are not rotated away:
//      they are pushed apart by one ulp of their magnitude, a backward error of
//      eps, so that the poles are distinct and no vectors have to be mixed.
//   2. root p of 1/rho + sum z_j^2 / (d_j - lambda) = 0 in (d_p, d_p+1), as the
//      offset tau from the nearer pole (every difference d_j - lambda is formed
//      from it, so it has full relative accuracy): a start from the two nearest
//      poles' terms, then the rational interpolation that fits the sums left and
//      right of the root each with its own pole ("the middle way", Li, LAPACK
//      Working Note 89, 1993), inside a bracket.  Measured on random and LETKF
//      matrices: 3.3 evaluations per root in FP32, 4.2 in FP64.
//   3. z is recomputed from the roots (Gu & Eisenstat, SIAM J. Matrix Anal.
//      Appl. 16, 1995), so the vectors z_j / (d_j - lambda) are orthogonal to
//      working precision without extended arithmetic.
//   4. the new eigenvalues are ranked, the vectors U formed in that order, and
//      Q <- Q U on the matrix cores.
// Steps 1-3 run on nodes of order one: one that is smaller than the rest of T by more
// than DcLim::NODE is scaled by a power of two, since the products of step 3 hold one
// factor of (node's size) / HUGE_ and the derivative in step 2 is of the order of
// 1 / size (FP32: vectors off by order one from a size of 1e-16 on).
#pragma once
#include "common.hpp"
#include "eig_symdmt.hpp"
#include "eig_wave.hpp"

namespace eigmi {

// HUGE_ (a node's largest entry is between NODE and order one): from here on a value
// stands for "no pole"; slot p of a node uses HUGE_ (1 + p / 1024), so that
// these sort behind the poles in the order of their slots.  STEP: 4 sqrt(eps).
template <typename T> struct DcLim;
template <> struct DcLim<float> {
  static constexpr float HUGE_ = 1e18f, STEP = 1.3810679e-03f, NODE = 1e-6f;
  static constexpr int EXP = 120;                       // scale factors stay normal
};
template <> struct DcLim<double> {
  static constexpr double HUGE_ = 1e150, STEP = 5.9604644775390625e-08, NODE = 1e-6;
  static constexpr int EXP = 1000;
};

__device__ __forceinline__ float rcp_(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp_(double x)
{
  double y = __builtin_amdgcn_rcp(x);
  y = __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
  return y;
}
// square root to about an ulp (no correction step to the last bit)
__device__ __forceinline__ float qsqrt_(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double qsqrt_(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return x > 0.0 ? g : 0.0;
}
template <typename T> __device__ __forceinline__ T min_(T a, T b) { return a < b ? a : b; }
template <typename T> __device__ __forceinline__ T max_(T a, T b) { return a > b ? a : b; }
template <typename T> __device__ __forceinline__ bool finite_(T x) { return abs_(x) <= std::numeric_limits<T>::max(); }

// quad lane moves that fold into the instruction that uses them (every lane has a source)
template <int CTRL> struct MvQ {
  __device__ int operator()(int v) const { return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, true); }
};
// Sum and product over the NLR = 1, 2 or 4 lanes that share a root.
template <int NLR, typename T>
__device__ __forceinline__ T lanes_sum(T x)
{
  if (NLR >= 2) x += lane_move(x, MvQ<0xB1>());
  if (NLR >= 4) x += lane_move(x, MvQ<0x4E>());
  return x;
}
template <int NLR, typename T>
__device__ __forceinline__ T lanes_prod(T x)
{
  if (NLR >= 2) x *= lane_move(x, MvQ<0xB1>());
  if (NLR >= 4) x *= lane_move(x, MvQ<0x4E>());
  return x;
}

// four consecutive values from LDS (16-byte aligned)
__device__ __forceinline__ void ld4(const float *p, float (&o)[4])
{
  const float4 a = *(const float4 *)p;
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
}
__device__ __forceinline__ void ld4(const double *p, double (&o)[4])
{
  const double2 a = *(const double2 *)p, b = *(const double2 *)(p + 2);
  o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y;
}

// How the S entries of a node are dealt to the NLR lanes of a root: NQ runs of 4
// per lane, run q of lane `sub` at 4 (NLR q + sub) (nodes of fewer than 4 NLR
// entries leave lanes without any).
template <int S, int NLR> struct DcDeal {
  static constexpr int NQ = (S + 4 * NLR - 1) / (4 * NLR);
  static __device__ __forceinline__ bool has(int q, int sub) { return S >= 4 * NLR || 4 * (NLR * q + sub) < S; }
};

// Root p (0 <= p < k) of 1/rho + sum_j zq_j / (d_j - lambda), d ascending and
// distinct, zq = z^2 > 0, entries k.. of d HUGE_ and of zq zero: lambda = da + tau.
// All lanes of the wave call it (`live`: this one has a root).  REG: the lane's
// poles and weights stay in registers, otherwise every evaluation reads them
// from LDS.  False where maxit evaluations (DC_MAXIT; the most seen is 21) did not end
// in a root.
constexpr int DC_MAXIT = 64;
template <typename T, int S, int NLR, bool REG>
__device__ __forceinline__ bool dc_root(const T *__restrict__ dl, const T *__restrict__ zq, int k, int p, int sub,
                                        T rho, bool live, int maxit, T &da_out, T &tau_out)
{
  constexpr int NQ = DcDeal<S, NLR>::NQ;
  const T eps = eps_of<T>();
  const int nq = REG ? NQ : (k + 4 * NLR - 1) / (4 * NLR);
  const bool last = p >= k - 1;
  T dr[REG ? NQ : 1][4], zr[REG ? NQ : 1][4];
  T sz = T(0);
  if (REG) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const bool has = DcDeal<S, NLR>::has(q, sub);
      const int j0 = has ? 4 * (NLR * q + sub) : 0;
      ld4(dl + j0, dr[q]);
      ld4(zq + j0, zr[q]);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        zr[q][v] = has ? zr[q][v] : T(0);
        dr[q][v] = has ? dr[q][v] : DcLim<T>::HUGE_;
        sz += zr[q][v];
      }
    }
  } else {
    for (int q = 0; q < nq; ++q) {
      T z4[4];
      ld4(zq + 4 * (NLR * q + sub), z4);
      sz += (z4[0] + z4[1]) + (z4[2] + z4[3]);
    }
  }
  sz = lanes_sum<NLR>(sz);
  const T c0 = rcp_(rho);
  // poles p, p+1 and p-1 (the last root's second pole)
  const int pi = live ? p : 0;
  const T dp = dl[pi], zp = zq[pi];
  const T dn = dl[(live && !last) ? p + 1 : 0], zn = (live && !last) ? zq[p + 1] : T(0);
  const T dm = dl[pi > 0 ? pi - 1 : 0], zm = zq[pi > 0 ? pi - 1 : 0];
  const T gap = last ? rho * sz * (T(1) + T(4) * eps) : dn - dp;
  const T half = T(0.5) * gap;
  const T gl = (pi > 0) ? dm - dp : T(-1);

  // f at the middle of the interval decides which pole the root is nearer to
  T f = T(0);
  auto mid_term = [&](const T (&d4)[4], const T (&z4)[4]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) f = fma_(z4[v], rcp_((d4[v] - dp) - half), f);
  };
  if (REG) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) mid_term(dr[q], zr[q]);
  } else {
#pragma unroll 2
    for (int q = 0; q < nq; ++q) {
      T d4[4], z4[4];
      ld4(dl + 4 * (NLR * q + sub), d4);
      ld4(zq + 4 * (NLR * q + sub), z4);
      mid_term(d4, z4);
    }
  }
  f = c0 + lanes_sum<NLR>(f);
  const bool left = last || f >= T(0);
  const T da = left ? dp : dn;
  if (REG) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) dr[q][v] -= da;
  }
  T lo = left ? T(0) : -half, hi = left ? half : T(0);
  if (last && f < T(0)) { lo = half; hi = gap; }
  // start: the two nearest poles' terms, the rest frozen at its middle value
  // (the last root: poles p - 1 and p, the larger root of the quadratic)
  T tau;
  {
    const T ih = rcp_(half);
    const T zo = last ? ((pi > 0) ? zm : T(0)) : zn;
    const T c = last ? fma_(zp, ih, f) + zo * rcp_(half - gl) : fma_(zp - zn, ih, f);
    const T o = last ? gl : (left ? gap : -gap);
    const T a = fma_(c, o, zp + zo);
    const T b = last ? zp * gl : (left ? zp * gap : -(zn * gap));
    const T disc = qsqrt_(max_(fma_(a, a, T(-4) * b * c), T(0)));
    const T q = a + sign_(disc, a);
    T r2 = T(2) * b * rcp_(q);
    T r1 = T(0.5) * q * rcp_(c);
    if (last) {
      const T x = a >= T(0) ? r1 : r2;
      r1 = r2 = x;
    }
    const bool ok2 = r2 > lo && r2 < hi, ok1 = r1 > lo && r1 < hi;
    tau = ok2 ? r2 : (ok1 ? r1 : T(0.5) * (lo + hi));
  }
  // offsets of the two poles from the anchor
  const T o1 = last ? gl : (left ? T(0) : -gap), o2 = last ? T(0) : (left ? gap : T(0));
  bool act = live;
#pragma unroll 1
  for (int it = 0; it < maxit; ++it) {
    if (!__ballot(act)) break;
    // w: the sum; as: of absolute values; dal: its derivative; sd: the
    // derivative's terms right of the root minus those left of it
    T ws = T(0), as = T(0), dal = T(0), sd = T(0);
    auto term = [&](T x, T z) {
      const T r = rcp_(x);
      const T t = z * r;
      ws += t;
      as += abs_(t);
      dal = fma_(t, r, dal);
      sd = fma_(abs_(t), r, sd);
    };
    if (REG) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) term(dr[q][v] - tau, zr[q][v]);
    } else {
#pragma unroll 2
      for (int q = 0; q < nq; ++q) {
        T d4[4], z4[4];
        ld4(dl + 4 * (NLR * q + sub), d4);
        ld4(zq + 4 * (NLR * q + sub), z4);
#pragma unroll
        for (int v = 0; v < 4; ++v) term((d4[v] - da) - tau, z4[v]);
      }
    }
    ws = lanes_sum<NLR>(ws);
    as = lanes_sum<NLR>(as);
    dal = lanes_sum<NLR>(dal);
    sd = lanes_sum<NLR>(sd);
    const T w = c0 + ws;
    // within the rounding of the sum: done
    if (abs_(w) <= eps * (c0 + T(4) * as + abs_(tau) * dal)) act = false;
    T dph = T(0.5) * (dal + sd);
    if (__ballot(last)) {                                 // the last root: pole p apart from the others
      const T it_ = rcp_(tau);
      dph = last ? zp * it_ * it_ : dph;
    }
    const T dps = dal - dph;
    const T d1 = o1 - tau, d2 = o2 - tau;
    const T cc = (w - d1 * dps) - d2 * dph;
    const T d12 = d1 * d2;
    const T A = (d1 + d2) * w - d12 * dal, B = d12 * w;
    // the root between the poles, or (last) right of both
    T ds = qsqrt_(max_(fma_(A, A, T(-4) * B * cc), T(0)));
    ds = last ? -ds : ds;
    const bool far = (last ? -A : A) <= T(0);
    const T num = far ? A - ds : B + B;
    const T den = far ? cc + cc : A + ds;
    T eta = num * rcp_(den);
    if (!(w * eta < T(0))) eta = -w * rcp_(dal);
    lo = (act && w < T(0)) ? tau : lo;
    hi = (act && !(w < T(0))) ? tau : hi;
    T tn = tau + eta;
    const bool in = tn > lo && tn < hi;
    if (__builtin_expect(__ballot(act && !in) != 0ull, 0)) {
      // outside the bracket: towards its end at zero, else into its middle
      const T al = abs_(lo), ah = abs_(hi);
      T tb = T(0.5) * (lo + hi);
      if (T(16) * min_(al, ah) < max_(al, ah)) tb = sign_(qsqrt_(al) * qsqrt_(ah), lo);
      if (lo == T(0)) tb = hi * T(0.0625);
      if (hi == T(0)) tb = lo * T(0.0625);
      tn = in ? tn : tb;
    }
    // a step this small leaves an error of the order of its square
    const bool fin = tn == tau || tn == lo || tn == hi || (in && abs_(eta) <= DcLim<T>::STEP * abs_(tau));
    tau = act ? tn : tau;
    act = act && !fin;
  }
  da_out = da;
  tau_out = tau;
  return !act;
}

// z of pole p recomputed from the roots, squared, up to a factor that is the
// same for every p: prod_q (lambda_q - d_p) / prod_{q != p} (d_q - d_p) in ratios
// in (0, 1].  Entries k.. of das are HUGE_ and of taus 0, so that their ratios
// with the HUGE_ entries of dl are that common factor.
template <typename T, int S, int NLR, bool REG>
__device__ __forceinline__ T dc_zhat2(const T *__restrict__ dl, const T *__restrict__ das, const T *__restrict__ taus,
                                      int k, int p, int sub)
{
  constexpr int NQ = DcDeal<S, NLR>::NQ;
  const int nq = REG ? NQ : (k + 4 * NLR - 1) / (4 * NLR);
  const T dp = dl[p];
  T pr = T(1);
  auto run = [&](int q) {
    const bool has = DcDeal<S, NLR>::has(q, sub);
    const int j0 = has ? 4 * (NLR * q + sub) : 0;
    T d4[4], a4[4], t4[4];
    ld4(dl + j0, d4);
    ld4(das + j0, a4);
    ld4(taus + j0, t4);
    const T dx = dl[j0 + 4 < S ? j0 + 4 : 0];
    const T dnx = (j0 + 4 < S) ? dx : DcLim<T>::HUGE_;
    T pq = T(1);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const T num = (a4[v] - dp) + t4[v];
      const T dj1 = (v < 3) ? d4[v < 3 ? v + 1 : 3] : dnx;
      const T den = ((j0 + v < p) ? d4[v] : dj1) - dp;
      pq *= num * rcp_(den);
    }
    pr *= has ? pq : T(1);
  };
  if (REG) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) run(q);
  } else {
#pragma unroll 2
    for (int q = 0; q < nq; ++q) run(q);
  }
  return abs_(lanes_prod<NLR>(pr)) * DcLim<T>::HUGE_;
}

// ---- merges up to order 64: one workgroup per matrix (or 64-column block) -----

template <int NB, typename T>
struct alignas(16) DcLds {
  alignas(16) T aop[NB * NB];                    // U in matrix-core A-operand order
  alignas(16) T d[64];                           // eigenvalues by column, ascending in every node
  alignas(16) T F[2][64], B[2][64];              // first / last row of each node's vectors, by column
  alignas(16) T key[64];
  alignas(16) T dl[64], zq[64], zs[NB];          // poles in ascending order, z^2, z
  alignas(16) T da[64], tau[64];                 // roots
  alignas(16) T val[64];
  alignas(16) T zk[64], dk[64];                  // recomputed z and pole by original column
  alignas(16) T ma[NB], mt[NB];                  // root by new column
  alignas(16) int src[NB], mdef[NB];             // column that passes through, by slot / new column (-1: a root)
  alignas(16) T e[NB];
  alignas(16) int ex[NB];                        // exponent of the scale of a column's node
  alignas(16) T red[4];
  int flag[4];
  int lost;                                      // a root was not found or a vector came to nothing
};

template <int NW>
__device__ __forceinline__ void dc_sync()
{
  if (NW == 1) wsync();
  else __syncthreads();
}

// Shape of a workgroup: NLR lanes per column, NW waves; wave q carries the rows
// of the 16-row tiles CT q .. CT q + CT - 1 of the eigenvectors and forms the same
// tiles of new columns.
template <int NB, int NLR> struct DcShape {
  static constexpr int NT = NB / 16, NTH = NB * NLR, NW = NTH / 64, CT = NT / NW;
  static_assert(NTH % 64 == 0 && NT % NW == 0, "whole waves, whole tiles");
};

// WAVES: occupancy asked for (waves per SIMD).  The workgroup's chain of short
// dependent phases is hidden by other workgroups, so registers are traded for
// them: FP32 n = 64, L = 16384: 760 us at 4, 597 us at 7 (some spills); FP64 spills
// beyond 3 (n = 60, L = 3000: 333 us, 412 us at 4).  REG: bytes of poles a lane
// keeps in registers across evaluations, the smaller nodes' only; the others are
// read from LDS (n = 64 FP32 at 7 waves: 64 bytes 658 us, 16 bytes 597 us).
template <typename T, int NB> struct DcTune { static constexpr int WAVES = 6, REG = 64; };
template <> struct DcTune<float, 48> { static constexpr int WAVES = 7, REG = 32; };
template <> struct DcTune<float, 64> { static constexpr int WAVES = 7, REG = 16; };
template <> struct DcTune<double, 32> { static constexpr int WAVES = 4, REG = 64; };
template <> struct DcTune<double, 48> { static constexpr int WAVES = 4, REG = 32; };
template <> struct DcTune<double, 64> { static constexpr int WAVES = 3, REG = 32; };

// aop tile (M, t): the A operand of the new columns 16 M .. against the old
// columns 16 t' .. (t' the t-th tile of M's node), one vector of four per lane.
template <typename T>
__device__ __forceinline__ void aop_put(T *__restrict__ o, int lane, const T (&u)[4], T f)
{
  if constexpr (sizeof(T) == 4) {
    *(float4 *)(o + 4 * lane) = make_float4(u[0] * f, u[1] * f, u[2] * f, u[3] * f);
  } else {
    *(double2 *)(o + 2 * lane) = make_double2(u[0] * f, u[1] * f);
    *(double2 *)(o + 128 + 2 * lane) = make_double2(u[2] * f, u[3] * f);
  }
}
template <typename T>
__device__ __forceinline__ void aop_get(const T *__restrict__ o, int lane, T (&u)[4])
{
  if constexpr (sizeof(T) == 4) {
    ld4(o + 4 * lane, u);
  } else {
    const double2 x = *(const double2 *)(o + 2 * lane), y = *(const double2 *)(o + 128 + 2 * lane);
    u[0] = x.x; u[1] = x.y; u[2] = y.x; u[3] = y.y;
  }
}

// X <- U^T X for the nodes of TS tiles each (the last may have fewer)
template <typename T, int NB, int CT, int TS>
__device__ __forceinline__ void dc_apply(const T *__restrict__ aop, int lane, typename Mfma16<T>::v4 (&X)[CT][NB / 16])
{
  typedef typename Mfma16<T>::v4 v4;
  constexpr int NT = NB / 16;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += TS) {
      v4 acc[TS];
#pragma unroll
      for (int M = 0; M < TS; ++M) {
        if (t0 + M < NT) {
          acc[M] = v4{0, 0, 0, 0};
#pragma unroll
          for (int t = 0; t < TS; ++t) {
            if (t0 + t < NT) {
              T av[4];
              aop_get(aop + (size_t)((t0 + M) * TS + t) * 256, lane, av);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[M] = Mfma16<T>::op(av[r], X[c][t0 + t][r], acc[M]);
            }
          }
        }
      }
#pragma unroll
      for (int M = 0; M < TS; ++M)
        if (t0 + M < NT) X[c][t0 + M] = acc[M];
    }
  }
}

// The merge of all nodes of S columns (children of H; S = 48 with H = 32 is the
// last merge of 48 columns) of a block of NB columns, n of them live.  fb: which
// of the two F / B buffers holds the children's rows.  LN: lanes per root (at most
// the workgroup's lanes per column; with fewer, the first waves do steps 1-3
// alone): an evaluation costs about 7 instructions a pole and 45 more, so small
// nodes take one lane a root and large ones the whole workgroup.
// Returns DcLds::lost of all levels so far.
template <typename T, int NB, int NLR, int S, int H, int LN>
__device__ __forceinline__ bool dc_merge_level(DcLds<NB, T> &Sh,
                                               typename Mfma16<T>::v4 (&X)[DcShape<NB, NLR>::CT][NB / 16], int n,
                                               int fb, int maxit)
{
  typedef DcShape<NB, NLR> G;
  typedef DcDeal<S, LN> Deal;
  constexpr int NW = G::NW, CT = G::CT, NQ = Deal::NQ;
  constexpr int LW = (NB * LN + 63) / 64;                      // waves of steps 1-3
  constexpr int TS = S >= 16 ? S / 16 : 1;                     // tiles of a node (of several nodes: one)
  constexpr bool LAST = S >= NB;
  constexpr bool REG = S * sizeof(T) <= DcTune<T, NB>::REG * LN;
  const T eps = eps_of<T>(), HUGE_ = DcLim<T>::HUGE_;
  const int tid = threadIdx.x;
  const bool on = NB * LN >= G::NTH || tid < NB * LN;
  const int i = on ? tid / LN : 0, sub = tid % LN;
  const int wv = tid >> 6, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
  const int base = LAST ? 0 : (i & ~(S - 1)), mid = base + H, p = i - base;
  const int end = (base + S < n) ? base + S : n;               // live columns of the node end here
  const bool both = mid < n;                                   // the node has a right child
  // ---- 1. z, the poles set aside, ranks --------------------------------------
  T z = T(0), rho = T(0), key = HUGE_, dmax = T(0);
  bool nd = false, small = false;                              // small: a node of this wave is scaled
  int c = 0, k = 0;
  if (on) {
    const T er = both ? Sh.e[mid - 1] : T(0);
    T di = Sh.d[i];
    rho = abs_(er);
    z = (i < mid) ? Sh.B[fb][i] : sign_(T(1), er) * Sh.F[fb][i];
    dmax = rho;
    if (base < n) {
      // the children are sorted
      dmax = max_(dmax, max_(abs_(Sh.d[base]), abs_(Sh.d[(both ? mid : end) - 1])));
      if (both) dmax = max_(dmax, max_(abs_(Sh.d[mid]), abs_(Sh.d[end - 1])));
    }
    // steps 1-3 on a small node scaled to order one (a power of two: exact)
    const bool tiny = dmax > T(0) && dmax < DcLim<T>::NODE;
    small = __ballot(tiny) != 0ull;
    if (small) {
      int ex = 0;
      if (tiny) (void)frexp(dmax, &ex);
      ex = max(ex, -DcLim<T>::EXP);
      rho = ldexp(rho, -ex);
      dmax = ldexp(dmax, -ex);
      di = ldexp(di, -ex);
      Sh.ex[i] = ex;
    }
    nd = i < n && rho * abs_(z) > T(2) * eps * dmax;
    key = nd ? di : HUGE_ * (T(1) + T(p) * T(1.0 / 1024));
    if (sub == 0) Sh.key[i] = key;
  }
  dc_sync<LW>();
  auto put = [&]() {
    if (on && sub == 0) {
      Sh.dl[base + c] = key;
      Sh.zs[base + c] = nd ? z : T(0);
      Sh.zq[base + c] = nd ? z * z : T(0);
      Sh.src[base + c] = i;
    }
  };
  if (on) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const bool has = Deal::has(q, sub);
      T k4[4];
      ld4(&Sh.key[base + (has ? 4 * (LN * q + sub) : 0)], k4);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        c += (has && k4[v] < key) ? 1 : 0;
        k += (has && k4[v] < HUGE_) ? 1 : 0;
      }
    }
    c = lanes_sum<LN>(c);
    k = lanes_sum<LN>(k);
  }
  put();
  dc_sync<LW>();
  {
    // slots that two equal poles claimed, and poles closer than one ulp: both are
    // put right in order by a slow path (rare)
    bool rep = false;
    if (on) {
      const bool dup = Sh.src[base + c] != i;
      const T gmin = eps * max_(abs_(Sh.dl[i > 0 ? i - 1 : 0]), dmax * T(1.0 / 4096));
      rep = dup || (p > 0 && p < k && !(Sh.dl[i] - Sh.dl[i > 0 ? i - 1 : 0] >= gmin));
    }
    bool fix = __ballot(rep) != 0ull;
    if (LW > 1) {
      if (lane == 0) Sh.flag[wv] = fix ? 1 : 0;
      __syncthreads();
      fix = false;
#pragma unroll
      for (int q = 0; q < LW; ++q) fix = fix || Sh.flag[q] != 0;
    }
    if (fix) {
      if (on) {
        int tie = 0;
        for (int j = base; j < i; ++j) tie += (Sh.key[j] == key) ? 1 : 0;
        c += tie;                                          // behind the equal ones before it
      }
      dc_sync<LW>();
      put();
      dc_sync<LW>();
      if (on && p == 0 && sub == 0) {
        for (int j = base + 1; j < base + k; ++j) {
          const T pv = Sh.dl[j - 1], g = eps * max_(abs_(pv), dmax * T(1.0 / 4096));
          if (Sh.dl[j] - pv < g) Sh.dl[j] = pv + g;
        }
      }
      dc_sync<LW>();
    }
  }
  // ---- 2. roots ----------------------------------------------------------------
  const bool root = on && p < k;
  bool ok = true;
  T da = HUGE_, tau = T(0), v0 = T(0);
  int s0 = 0;
  if (on) {
    T a0, t0;
    ok = dc_root<T, S, LN, REG>(&Sh.dl[base], &Sh.zq[base], k, p, sub, rho, root, maxit, a0, t0);
    if (root) { da = a0; tau = t0; }
    s0 = Sh.src[i] & 63;
    v0 = root ? da + tau : Sh.d[s0];
    // (a slot without a column keeps HUGE_ in every scale)
    if (small && !root && s0 < n) v0 = ldexp(v0, -Sh.ex[i]);
    if (sub == 0) {
      Sh.da[i] = da;
      Sh.tau[i] = tau;
      Sh.val[i] = v0;
    }
  }
  dc_sync<LW>();
  // ---- 3. z from the roots; new order -------------------------------------------
  if (on) {
    const T z2 = dc_zhat2<T, S, LN, REG>(&Sh.dl[base], &Sh.da[base], &Sh.tau[base], k, root ? p : 0, sub);
    if (root && !(ok && z2 > T(0) && finite_(z2))) Sh.lost = 1;     // (an offset of zero gives a z of zero)
    // without a column set aside the roots are in order already
    int nr = p;
    if (__ballot(base + k < end)) {
      nr = 0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const bool has = Deal::has(q, sub);
        T w4[4];
        const int j0 = base + (has ? 4 * (LN * q + sub) : 0);
        ld4(&Sh.val[j0], w4);
#pragma unroll
        for (int v = 0; v < 4; ++v) nr += (has && (w4[v] < v0 || (w4[v] == v0 && j0 + v < i))) ? 1 : 0;
      }
      nr = lanes_sum<LN>(nr);
    }
    nr += base;
    if (sub == 0) {
      // slot i (a pole, or the column s0 that passes through): by original column
      Sh.zk[s0] = root ? sign_(qsqrt_(z2), Sh.zs[i]) : T(0);
      Sh.dk[s0] = root ? Sh.dl[i] : HUGE_;
      Sh.ma[nr] = da;
      Sh.mt[nr] = tau;
      Sh.mdef[nr] = root ? -1 : s0;
      // every read of the old values is before the last barrier
      Sh.d[nr] = (small && s0 < n) ? ldexp(v0, Sh.ex[i]) : v0;
    }
  }
  dc_sync<NW>();
  const int lost = __builtin_amdgcn_readfirstlane(Sh.lost);
  // ---- 4. U (A operand: lane = new column, slots = old columns) -------------------
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int M = wv * CT + ct, mcol = 16 * M + lm;
    const int nb = LAST ? 0 : (mcol & ~(S - 1)), nmid = nb + H;
    const int tb = LAST ? 0 : ((16 * M) & ~(16 * TS - 1));     // first old column of the tiles
    const T a = Sh.ma[mcol], t0 = Sh.mt[mcol];
    const int def = Sh.mdef[mcol];
    const bool nboth = nmid < n;
    T ss = T(0), fs = T(0), bs = T(0);
    T u[TS][4];
#pragma unroll
    for (int t = 0; t < TS; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kc = tb + 16 * t + Mfma16<T>::row(lg, r);
        const T x = (Sh.dk[kc] - a) - t0;
        T v = (def >= 0) ? (kc == def ? T(1) : T(0)) : Sh.zk[kc] * rcp_(x);
        if (S < 16) v = ((kc & ~(S - 1)) == nb) ? v : T(0);
        u[t][r] = v;
        ss = fma_(v, v, ss);
        if (!LAST) {
          const bool lft = kc < nmid;
          fs = fma_(v, lft ? Sh.F[fb][kc] : T(0), fs);
          bs = fma_(v, (lft != nboth) ? Sh.B[fb][kc] : T(0), bs);
        }
      }
    ss += lane_move(ss, MvX16());
    ss += lane_move(ss, MvX32());
    const T inv = rsqrt_nr(ss);
    if (!LAST) {
      fs += lane_move(fs, MvX16());
      fs += lane_move(fs, MvX32());
      bs += lane_move(bs, MvX16());
      bs += lane_move(bs, MvX32());
      if (lg == 0) {
        Sh.F[fb ^ 1][mcol] = fs * inv;
        Sh.B[fb ^ 1][mcol] = bs * inv;
      }
    }
#pragma unroll
    for (int t = 0; t < TS; ++t) aop_put<T>(Sh.aop + (size_t)(M * TS + t) * 256, lane, u[t], inv);
  }
  dc_sync<NW>();
  // ---- 5. X <- U^T X ----------------------------------------------------------------
  dc_apply<T, NB, CT, TS>(Sh.aop, lane, X);
  if (!LAST) dc_sync<NW>();
  return lost != 0;
}

// Full solve after the tridiagonalisation for n <= NB (NB = 16, 32, 48, 64): Q
// (n x n per matrix, from eig_tri_kernel), d / e (de, matrix-minor); one
// workgroup per matrix.  X starts as Q^T, so the last merge leaves the
// eigenvectors of A themselves.
// BLK: a 64-column block of a larger matrix (nblk per matrix) with X starting from
// the identity: the block's eigenvectors of T to z0 or z1 (bit b of zmask; ld n,
// at (64 b, 64 b)) and its eigenvalues to w (NaN for a block that is not finite,
// infinities for one whose merges failed).
// A matrix whose merges failed (DcLds::lost): info = 1 and a untouched.
// nanfail: what a matrix that is not finite gives: 1: info = 1 and a untouched,
// 0: the diagonal and Q as they are (sorted by the reference's rule), info = 0
// (the two outcomes of the QL paths, by batch size).
// only (may be null): just the matrices flagged ST_OVERFLOW there.
template <typename T, int NB, int NLR, bool BLK>
__global__ __launch_bounds__(NB *NLR) __attribute__((amdgpu_waves_per_eu(DcTune<T, NB>::WAVES))) void eig_dc_kernel(
    int L, int nm, int n_all, T *__restrict__ a, const T *__restrict__ qws, const T *__restrict__ de, int ld,
    T *__restrict__ w, int *__restrict__ info, int opts, int nanfail, int nblk, T *__restrict__ z0,
    T *__restrict__ z1, int zmask, const int *__restrict__ only)
{
  typedef typename Mfma16<T>::v4 v4;
  typedef DcShape<NB, NLR> G;
  constexpr int NT = G::NT, NW = G::NW, CT = G::CT;
  __shared__ DcLds<NB, T> Sh;
  const int tid = threadIdx.x, i = tid / NLR, sub = tid % NLR;
  const int wv = tid >> 6, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
  const int mat = BLK ? (int)(blockIdx.x / nblk) : (int)blockIdx.x;
  if (only && only[mat] != ST_OVERFLOW) return;
  const int b0 = BLK ? 64 * (int)(blockIdx.x % nblk) : 0;
  const int n = BLK ? ((n_all - b0) < NB ? n_all - b0 : NB) : n_all;
  const T HUGE_ = DcLim<T>::HUGE_;
  const T *__restrict__ dm = de + (size_t)b0 * ld + mat;
  const T *__restrict__ em = de + (size_t)(n_all + b0) * ld + mat;

  // d_i, e_i (the coupling of i and i + 1; beyond the block for its last column)
  const bool lv = i < n, cpl = lv && b0 + i + 1 < n_all;
  T dv = lv ? dm[(size_t)i * ld] : T(0);
  T ev = cpl ? em[(size_t)i * ld] : T(0);
  const T ep = (b0 + i > 0 && lv) ? em[((ptrdiff_t)i - 1) * ld] : T(0);

  // rows of Q (or of the identity)
  v4 X[CT][NT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int row = 16 * (wv * CT + c) + lm;
    const T *__restrict__ Q = qws + (size_t)mat * n_all * n_all;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kc = 16 * t + Mfma16<T>::row(lg, r);
        if (BLK) X[c][t][r] = (kc == row) ? T(1) : T(0);
        else X[c][t][r] = (kc < n && row < n) ? Q[row + (size_t)kc * n] : T(0);
      }
  }
  // the tears: the even member of a pair loses |e| to its left neighbour, the
  // odd one to its right neighbour
  dv -= abs_((i & 1) ? ev : ep);
  bool bad = !finite_(dv) || !finite_(ev);
  T mx = max_(abs_(dv), abs_(ev));
  if (NLR <= 2) mx = max_(mx, lane_move(mx, MvX2()));
  if (NLR == 1) mx = max_(mx, lane_move(mx, MvX1()));
  mx = max_(mx, lane_move(mx, MvHM()));
  mx = max_(mx, lane_move(mx, MvRM()));
  mx = max_(mx, lane_move(mx, MvX16()));
  mx = max_(mx, lane_move(mx, MvX32()));
  bad = __ballot(bad) != 0ull;
  if (NW > 1) {
    if (lane == 0) {
      Sh.red[wv] = mx;
      Sh.flag[wv] = bad ? 1 : 0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NW; ++q) {
      mx = max_(mx, Sh.red[q]);
      bad = bad || Sh.flag[q] != 0;
    }
  }
  T *__restrict__ wout = w + (size_t)mat * n_all + b0;
  if (bad) {
    if (BLK) {
      // the merges above report it
      if (sub == 0 && lv) wout[i] = std::numeric_limits<T>::quiet_NaN();
      return;
    }
    T *__restrict__ A = a + (size_t)mat * (size_t)nm * (size_t)n;
    if (info && tid == 0) info[mat] = nanfail ? 1 : 0;
    if (tid == 0) {
      for (int j = 0; j < n; ++j) {
        Sh.val[j] = dm[(size_t)j * ld];
        Sh.src[j] = j;
      }
      // the reference's selection rule on what compares (tql2_tiled.hpp:149-176)
      for (int l = 0; !nanfail && l < n - 1; ++l) {
        int il = l;
        for (int j = l + 1; j < n; ++j) il = (Sh.val[il] > Sh.val[j]) ? j : il;
        const T x = Sh.val[l];
        Sh.val[l] = Sh.val[il];
        Sh.val[il] = x;
        const int y = Sh.src[l];
        Sh.src[l] = Sh.src[il];
        Sh.src[il] = y;
      }
    }
    dc_sync<NW>();
    const T *__restrict__ Q = qws + (size_t)mat * n * n;
    const int mcols = n - kopt_mdrop(opts);
    for (int j = 0; j < n; ++j) {
      if (tid == 0) wout[j] = Sh.val[j];
      if (!nanfail && j < mcols && tid < n) A[tid + (size_t)j * nm] = Q[tid + (size_t)Sh.src[j] * n];
    }
    return;
  }
  int ex = 0;
  if (mx > T(0)) (void)frexp(mx, &ex);
  ex = max(min(ex, DcLim<T>::EXP), -DcLim<T>::EXP);
  const T sc = ldexp(T(1), -ex), isc = ldexp(T(1), ex);
  // ---- leaves: the pairs (i, i + 1), i even: [x b; b y] = V diag V^T by one rotation
  {
    if (sub == 0) {
      Sh.key[i] = lv ? dv * sc : T(0);
      Sh.e[i] = ev * sc;
    }
    if (tid == 0) Sh.lost = 0;
    if (tid < 64) {
      // entries beyond the block never hold a pole
      if (tid >= NB) {
        Sh.d[tid] = HUGE_;
        Sh.key[tid] = Sh.dl[tid] = Sh.val[tid] = HUGE_ * T(2);
        Sh.zq[tid] = Sh.tau[tid] = Sh.zk[tid] = T(0);
        Sh.da[tid] = Sh.dk[tid] = HUGE_;
        Sh.F[0][tid] = Sh.F[1][tid] = Sh.B[0][tid] = Sh.B[1][tid] = T(0);
      }
    }
    dc_sync<NW>();
    const int j = i & ~1;
    const bool pair = j + 1 < n;
    const T x = Sh.key[j], y = Sh.key[j + 1], b = pair ? Sh.e[j] : T(0);
    T cs = T(1), sn = T(0), lx = x, ly = y;
    if (b != T(0)) {
      const T th = (y - x) / (b + b);
      const T t = sign_(T(1) / (abs_(th) + sqrt_(fma_(th, th, T(1)))), th);
      cs = T(1) / sqrt_(fma_(t, t, T(1)));
      sn = t * cs;
      lx = fma_(-t, b, x);
      ly = fma_(t, b, y);
    }
    // eigenvalue lx with (cs, -sn), ly with (sn, cs); ascending
    const bool sw = pair && ly < lx;
    const bool second = (i & 1) != (sw ? 1 : 0);
    const T f = second ? sn : cs, g = second ? cs : -sn;       // rows j and j + 1 of this column
    if (sub == 0) {
      Sh.d[i] = lv ? (second ? ly : lx) : HUGE_;
      Sh.F[0][i] = lv ? f : T(0);
      Sh.B[0][i] = lv ? (pair ? g : f) : T(0);
      Sh.zk[i] = f;
      Sh.dk[i] = g;
    }
    dc_sync<NW>();
    // as the first product: U is block diagonal with the rotations
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int M = wv * CT + ct, mcol = 16 * M + lm;
      const T fm = Sh.zk[mcol], gm = Sh.dk[mcol];
      T u[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kc = 16 * M + Mfma16<T>::row(lg, r);
        u[r] = ((kc >> 1) == (mcol >> 1)) ? ((kc & 1) ? gm : fm) : T(0);
      }
      aop_put<T>(Sh.aop + (size_t)M * 256, lane, u, T(1));
    }
    dc_sync<NW>();
    dc_apply<T, NB, CT, 1>(Sh.aop, lane, X);
    dc_sync<NW>();
  }
  const int maxit = kopt_cut(opts) ? 1 : DC_MAXIT;
  constexpr int L1 = NB >= 48 ? 1 : (NB == 32 ? 2 : NLR), L2 = NB >= 48 ? 2 : NLR;
  dc_merge_level<T, NB, NLR, 4, 2, L1>(Sh, X, n, 0, maxit);
  dc_merge_level<T, NB, NLR, 8, 4, L1>(Sh, X, n, 1, maxit);
  bool lost = dc_merge_level<T, NB, NLR, 16, 8, L1>(Sh, X, n, 0, maxit);
  if constexpr (NB >= 32) lost = dc_merge_level<T, NB, NLR, 32, 16, L2>(Sh, X, n, 1, maxit);
  if constexpr (NB == 48) lost = dc_merge_level<T, NB, NLR, 48, 32, NLR>(Sh, X, n, 0, maxit);
  if constexpr (NB == 64) lost = dc_merge_level<T, NB, NLR, 64, 32, NLR>(Sh, X, n, 0, maxit);

  if (sub == 0 && lv) wout[i] = (BLK && lost) ? std::numeric_limits<T>::infinity() : Sh.d[i] * isc;
  if (!BLK && info && tid == 0) info[mat] = lost ? 1 : 0;
  if (!BLK && lost) return;
  T *__restrict__ O = BLK ? (((zmask >> (b0 / 64)) & 1) ? z1 : z0) + (size_t)mat * n_all * n_all + (size_t)b0 * n_all + b0
                          : a + (size_t)mat * (size_t)nm * (size_t)n;
  const int ldo = BLK ? n_all : nm, mcols = BLK ? n : n - kopt_mdrop(opts);
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int row = 16 * (wv * CT + c) + lm;
    if (row < n) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = 16 * t + Mfma16<T>::row(lg, r);
          if (m < mcols) O[row + (size_t)m * ldo] = X[c][t][r];
        }
    }
  }
}

} // namespace eigmi
