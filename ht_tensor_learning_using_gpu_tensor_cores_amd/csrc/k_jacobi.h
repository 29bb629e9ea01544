// Jacobi eigen solver device routines (FP64, n <= 64) shared by the small solvers and
// the batched kernel.
#pragma once
#include "ht_common.h"

namespace ht {

constexpr int SJ = 64;        // largest Jacobi problem
constexpr int SJLD = SJ + 1;  // LDS row stride of the Jacobi matrices
constexpr int SW = 16;        // waves of the 1024-thread kernels
constexpr int SR = 16;        // rows per thread there: n <= SW * SR
constexpr int SNT = SW * 64;  // threads of the 1024-thread kernels

__device__ __forceinline__ double lane_bcast(double x, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), l);
  return __hiloint2double(hi, lo);
}

// x from lane l - 1 (ROW_SR1) or l + 1 (ROW_SL1) of the same 16-lane row, by DPP moves;
// the row's first (last) lane keeps 0.
constexpr int DPP_ROW_SL1 = 0x101, DPP_ROW_SR1 = 0x111;
template <int CTRL>
__device__ __forceinline__ double dpp_row_shift(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// 1/x and 1/sqrt(x) in FP64 from the hardware approximations (v_rcp_f64, v_rsq_f64) and
// two Newton steps each (quadratic convergence from ~2^-22 leaves ~1 ulp).
__device__ __forceinline__ double rcp_nr(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  r = fma(r, fma(-x, r, 1.0), r);
  return r;
}
__device__ __forceinline__ double rsq_nr(double x) {
  double r = __builtin_amdgcn_rsq(x);
  r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
  r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
  return r;
}

// Jacobi rotation (c, s) that annihilates a_pq (Rutishauser's form: t = tan(phi) of the
// smaller angle, c = 1/sqrt(1 + t^2), s = t c; c^2 + s^2 = 1 to rounding). Without one where
// the cotangent leaves the FP64 range or is NaN: a_pq = 0, or so small that its reciprocal
// overflows (exactly dependent columns leave entries down to the subnormal numbers).
__device__ __forceinline__ void jacobi_rotation(double app, double aqq, double apq, double& c, double& s) {
  c = 1.0;
  s = 0.0;
  const double tau = (aqq - app) * rcp_nr(2.0 * apq);
  const double at = fabs(tau);
  if (!(at < 1e150)) return;
  const double h = 1.0 + tau * tau;
  double t = rcp_nr(at + h * rsq_nr(h));
  if (tau < 0.0) t = -t;
  c = rsq_nr(1.0 + t * t);
  s = t * c;
}

// Index walk of the round-robin: pair t of step s is (x, y) = ((s + t) mod m, (s - t) mod m),
// m = np - 1, and (m, s) for t = 0, so both indices move up by one from step to step (x of
// pair 0 stays). Kept times `stride`.
struct JacobiWalk {
  int x, y, incx, wrapx;
  __device__ __forceinline__ void init(int t, int m, int stride) {
    x = (t == 0 ? m : t) * stride;  // step 0
    y = (t == 0 ? 0 : m - t) * stride;
    incx = t == 0 ? 0 : stride;
    wrapx = t == 0 ? -1 : m * stride;
  }
  __device__ __forceinline__ void next(int m, int stride) {
    x += incx;
    if (x == wrapx) x = 0;
    y += stride;
    if (y == m * stride) y = 0;
  }
};

// Cyclic parallel Jacobi on the np x np symmetric matrix a (LDS, row stride LD, np even),
// accumulating the rotations into v, for a block of NT threads. A step rotates np/2 disjoint
// pairs: wave 0 forms the rotations, one per lane, while the other waves apply the step
// before's to v (rotations double-buffered in LDS); then every 2x2 block of a (rows of pair
// i, columns of pair j) becomes R_i^T A_ij R_j. Returns 1 when the off-diagonal mass fell
// below tol^2 * diagonal mass.
//
// Bound by instruction issue and the two barriers of a step, so the indices are walked, not
// computed (JacobiWalk), and the update of v hides the rotations' dependent chain: n = 64 with
// 1024 threads, full solve, 789 -> 606 us; n = 24, 165 -> 143 us.
template <int NT = SNT, int LD = SJLD>
__device__ __forceinline__ int jacobi_sweeps(double* a, double* v, int n, int np, int max_sweeps, double tol) {
  constexpr int NW = NT / 64, NV = NT - 64;  // NV threads update v
  __shared__ double2 rcs[2][SJ / 2];  // (c, s) of the pair's (smaller, larger) index
  __shared__ double red[2][NW];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int half = np / 2, m = np - 1;
  // this thread's columns of a: pair bj; its rows: pairs bi0, bi0 + di, ...
  const int bj = tid % half, bi0 = tid / half, di = NT / half;
  // its pair of columns of v and first row (threads from 64 on)
  const int tv = tid - 64, vj = tv >= 0 ? tv % half : 0, vr0 = tv >= 0 ? tv / half : np, dr = NV / half;
  const bool va = tv >= 0 && vr0 < dr, aa = bi0 < di;  // threads past the last whole row of pairs rest
  JacobiWalk wc, wr, wv2, wrot;
  wc.init(bj, m, 1);
  wr.init(min(bi0, half - 1), m, LD);
  wv2.init(vj, m, 1);
  wrot.init(min(lane, half - 1), m, 1);
  int g = 0;  // step count
  auto update_v = [&](const double2* cs) {
    const double2 r = cs[vj];
    const int P = min(wv2.x, wv2.y), Q = max(wv2.x, wv2.y);
    for (int i = vr0; i < np; i += dr) {
      double* row = v + i * LD;
      const double vP = row[P], vQ = row[Q];
      row[P] = r.x * vP - r.y * vQ;
      row[Q] = r.y * vP + r.x * vQ;
    }
    wv2.next(m, 1);
  };
  int conv = 0;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    double off = 0.0, dg = 0.0;
    for (int e = tid; e < n * n; e += NT) {
      const int i = e % n, j = e / n;
      const double x = a[i * LD + j];
      if (i == j) dg += x * x;
      else off += x * x;
    }
    off = wave_sum(off);
    dg = wave_sum(dg);
    if (lane == 0) {
      red[0][wv] = off;
      red[1][wv] = dg;
    }
    __syncthreads();
    off = 0.0;
    dg = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      off += red[0][w];
      dg += red[1][w];
    }
    __syncthreads();
    if (off <= tol * tol * dg || off == 0.0) {
      conv = 1;
      break;
    }
    for (int step = 0; step < m; ++step, ++g) {
      if (tid < 64) {
        if (tid < half) {
          const int p = min(wrot.x, wrot.y), q = max(wrot.x, wrot.y);
          double c, s;
          jacobi_rotation(a[p * LD + p], a[q * LD + q], a[p * LD + q], c, s);
          rcs[g & 1][tid] = make_double2(c, s);
          wrot.next(m, 1);
        }
      } else if (g > 0 && va) {
        update_v(rcs[(g & 1) ^ 1]);
      }
      __syncthreads();
      if (aa) {
        const double2 cj = rcs[g & 1][bj];
        const int P = min(wc.x, wc.y), Q = max(wc.x, wc.y);
        // rows of pair bi: the walk of bi0, moved on di pairs at a time
        for (int bi = bi0; bi < half; bi += di) {
          int rx = wr.x, ry = wr.y;
          if (bi != bi0) {  // (small blocks of threads) from the walk's definition
            int xs = step + bi, ys = step - bi;
            if (xs >= m) xs -= m;
            if (ys < 0) ys += m;
            rx = xs * LD;
            ry = ys * LD;
          }
          const double2 ci = rcs[g & 1][bi];
          double *p = a + min(rx, ry), *q = a + max(rx, ry);
          const double apP = p[P], apQ = p[Q], aqP = q[P], aqQ = q[Q];
          // right: columns; left: rows
          const double xpP = cj.x * apP - cj.y * apQ, xpQ = cj.y * apP + cj.x * apQ;
          const double xqP = cj.x * aqP - cj.y * aqQ, xqQ = cj.y * aqP + cj.x * aqQ;
          const double ypP = ci.x * xpP - ci.y * xqP, yqQ = ci.y * xpQ + ci.x * xqQ;
          double yqP = ci.y * xpP + ci.x * xqP, ypQ = ci.x * xpQ - ci.y * xqQ;
          if (bi == bj && ci.y != 0.0) {
            ypQ = 0.0;
            yqP = 0.0;
          }
          p[P] = ypP;
          p[Q] = ypQ;
          q[P] = yqP;
          q[Q] = yqQ;
        }
        wc.next(m, 1);
        wr.next(m, LD);
      }
      __syncthreads();
    }
  }
  if (g > 0 && va) update_v(rcs[(g & 1) ^ 1]);
  __syncthreads();
  return conv;
}

// Cyclic Jacobi on a 16 x 16 symmetric matrix in the registers of one wave, for problems
// too small to amortise block-wide barriers. Lane l = 8 I + J holds the 2 x 2 blocks (rows
// 2I, 2I+1; columns 2J, 2J+1) of A and of the rotation product V (V starts as I). A step
// rotates the eight pairs (2i, 2i+1): the diagonal lanes form the rotations, every lane
// fetches those of its row and column pair with lane permutes and applies R_I^T A R_J and
// V R_J. Then the indices move one place along the ring t1 .. t7, b7 .. b0 of the circle
// round-robin (t0 fixed; ti = 2i, bi = 2i+1) by a row and a column permutation of A and a
// column permutation of V (rows from lanes l -+ 8, columns from lanes l -+ 1 by DPP row
// shifts), so fifteen steps pair every two indices once. Diagonal entries
// equal to `pad` (decoupled padding) are left out of the convergence test, which is the
// one of jacobi_sweeps. On return a and v (LDS, ld SJLD) hold the result in the slot
// order (columns of v follow the diagonal of a); returns 1 when converged.
__device__ __forceinline__ int jacobi16_wave(double* a, double* v, int max_sweeps, double tol, double pad) {
  const int l = threadIdx.x & 63, I = l >> 3, J = l & 7;
  const bool dgl = I == J;
  double a00 = a[(2 * I) * SJLD + 2 * J], a01 = a[(2 * I) * SJLD + 2 * J + 1];
  double a10 = a[(2 * I + 1) * SJLD + 2 * J], a11 = a[(2 * I + 1) * SJLD + 2 * J + 1];
  double v00 = dgl ? 1.0 : 0.0, v01 = 0.0, v10 = 0.0, v11 = dgl ? 1.0 : 0.0;
  const int up = l >= 8 ? l - 8 : l, dn = l < 56 ? l + 8 : l;
  int conv = 0;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    double off = dgl ? a01 * a01 + a10 * a10 : a00 * a00 + a01 * a01 + a10 * a10 + a11 * a11;
    double dg = dgl ? (a00 != pad ? a00 * a00 : 0.0) + (a11 != pad ? a11 * a11 : 0.0) : 0.0;
    // one lane's sums decide for the whole wave (butterfly sums can differ in the last bit)
    off = lane_bcast(wave_sum(off), 0);
    dg = lane_bcast(wave_sum(dg), 0);
    if (off <= tol * tol * dg || off == 0.0) {
      conv = 1;
      break;
    }
    for (int step = 0; step < 15; ++step) {
      double c, s;
      jacobi_rotation(a00, a11, a01, c, s);  // used from the diagonal lanes only
      const double cI = __shfl(c, 9 * I, 64), sI = __shfl(s, 9 * I, 64);
      const double cJ = __shfl(c, 9 * J, 64), sJ = __shfl(s, 9 * J, 64);
      const double x00 = cJ * a00 - sJ * a01, x01 = sJ * a00 + cJ * a01;
      const double x10 = cJ * a10 - sJ * a11, x11 = sJ * a10 + cJ * a11;
      a00 = cI * x00 - sI * x10;
      a10 = sI * x00 + cI * x10;
      a01 = cI * x01 - sI * x11;
      a11 = sI * x01 + cI * x11;
      if (dgl && sI != 0.0) {
        a01 = 0.0;
        a10 = 0.0;
      }
      const double w00 = cJ * v00 - sJ * v01, w01 = sJ * v00 + cJ * v01;
      const double w10 = cJ * v10 - sJ * v11, w11 = sJ * v10 + cJ * v11;
      // rows: new t_I = t_{I-1} (t_1 = b_0, t_0 stays); new b_I = b_{I+1} (b_7 = t_7)
      {
        const double s0 = I == 0 ? a10 : a00, s1 = I == 0 ? a11 : a01;
        const double u00 = __shfl(s0, up, 64), u01 = __shfl(s1, up, 64);
        const double d10 = __shfl(a10, dn, 64), d11 = __shfl(a11, dn, 64);
        const double n10 = I == 7 ? a00 : d10, n11 = I == 7 ? a01 : d11;
        if (I != 0) {
          a00 = u00;
          a01 = u01;
        }
        a10 = n10;
        a11 = n11;
      }
      // columns, the same ring (A and V)
      {
        const double s0 = J == 0 ? a01 : a00, s1 = J == 0 ? a11 : a10;
        const double l00 = dpp_row_shift<DPP_ROW_SR1>(s0), l10 = dpp_row_shift<DPP_ROW_SR1>(s1);
        const double r01 = dpp_row_shift<DPP_ROW_SL1>(a01), r11 = dpp_row_shift<DPP_ROW_SL1>(a11);
        const double n01 = J == 7 ? a00 : r01, n11 = J == 7 ? a10 : r11;
        if (J != 0) {
          a00 = l00;
          a10 = l10;
        }
        a01 = n01;
        a11 = n11;
      }
      {
        const double s0 = J == 0 ? w01 : w00, s1 = J == 0 ? w11 : w10;
        const double l00 = dpp_row_shift<DPP_ROW_SR1>(s0), l10 = dpp_row_shift<DPP_ROW_SR1>(s1);
        const double r01 = dpp_row_shift<DPP_ROW_SL1>(w01), r11 = dpp_row_shift<DPP_ROW_SL1>(w11);
        v00 = J == 0 ? w00 : l00;
        v10 = J == 0 ? w10 : l10;
        v01 = J == 7 ? w00 : r01;
        v11 = J == 7 ? w10 : r11;
      }
    }
  }
  a[(2 * I) * SJLD + 2 * J] = a00;
  a[(2 * I) * SJLD + 2 * J + 1] = a01;
  a[(2 * I + 1) * SJLD + 2 * J] = a10;
  a[(2 * I + 1) * SJLD + 2 * J + 1] = a11;
  v[(2 * I) * SJLD + 2 * J] = v00;
  v[(2 * I) * SJLD + 2 * J + 1] = v01;
  v[(2 * I + 1) * SJLD + 2 * J] = v10;
  v[(2 * I + 1) * SJLD + 2 * J + 1] = v11;
  return conv;
}

// Load an n x n matrix into a (padded to even np with a decoupled, large negative
// diagonal entry that sorts last), set v = I.
template <int LD = SJLD, typename T>
__device__ __forceinline__ void jacobi_load(double* a, double* v, const T* A, int lda, int n, int np, bool symmetrise) {
  __shared__ double red[SW];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double amax = 0.0;
  for (int e = tid; e < np * np; e += blockDim.x) {
    const int i = e % np, j = e / np;
    double x = 0.0;
    if (i < n && j < n) {
      x = A[i + (long)lda * j];
      if (symmetrise) x = 0.5 * (x + A[j + (long)lda * i]);
    }
    a[i * LD + j] = x;
    v[i * LD + j] = (i == j) ? 1.0 : 0.0;
    amax = fmax(amax, fabs(x));
  }
  for (int o = 32; o > 0; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o, 64));
  if (lane == 0) red[wv] = amax;
  __syncthreads();
  if (np != n && tid == 0) {
    double m = 0.0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) m = fmax(m, red[w]);
    a[(np - 1) * LD + (np - 1)] = -(m * (double)n + 1.0) * 4.0;
  }
  __syncthreads();
}

// Descending order of the diagonal of a: thread i places index i at its rank (ties by
// index, NaN as +Inf), so order is a permutation for every matrix: its entries address LDS.
template <int LD = SJLD>
__device__ __forceinline__ void jacobi_order(const double* a, int np, int* order) {
  const int i = threadIdx.x;
  if (i < np) {
    auto key = [&](int j) {
      const double d = a[j * LD + j];
      return d == d ? d : (double)INFINITY;
    };
    const double di = key(i);
    int rank = 0;
    for (int j = 0; j < np; ++j) {
      const double dj = key(j);
      rank += (dj > di || (dj == di && j < i)) ? 1 : 0;
    }
    order[rank] = i;
  }
  __syncthreads();
}

}  // namespace ht
