// Top-k eigenpairs of a symmetric FP64 matrix with n <= 64: Householder tridiagonalisation by
// one wave, Sturm-count multisection by the work-group, then eigenvectors of the tridiagonal
// from twisted factorisations and back-transformation by one wave.
//
// What bounds it: dependent FP64 latency. The 64 x 64 matrix is 32 KB, far from any bandwidth;
// what counts is the number of dependent steps. A cyclic Jacobi solve of the same matrix takes
// ~8 sweeps of 63 steps with two work-group barriers each; this takes n - 2 reflector steps,
// each one pass over the trailing matrix (the previous step's rank-2 update is applied in the
// pass that forms the next product, so every step reads the matrix once), and then work that
// is parallel over the k wanted pairs. One wave needs no barrier: its LDS operations complete
// in order.
//
// A wave issues one instruction in ~5 cycles whatever its type (FP64 FMA latency is the same
// 5, an LDS read 64), so the time is the instruction count: each lane keeps its row in
// registers (rows in LDS cost a read and a write per entry and step: 90 of the 150 us of
// n = 64, k = 16), loops over LDS load their next values early, two Sturm recurrences share a
// lane. One problem, kernel time, rows in LDS and one wave throughout / now: n = 64, k = 16:
// 165 / 120 us; n = 32, k = 16: 72 / 62 us; n = 24, k = 4: 43 / 38 us.
//
// The result is checked before it is used: residuals in the tridiagonal basis, and mutual
// orthogonality of the k vectors, which twisted vectors of clustered eigenvalues (ranks
// above the numerical rank) lack and a Gram-Schmidt pass restores. Exactly equal
// eigenvalues fail the check and the caller takes Jacobi (rounding usually separates them:
// 64^4 with rotated identity factors stays in this solver's time).
#pragma once
#include "k_jacobi.h"

namespace ht {

constexpr int TR_N = 64;       // largest problem
constexpr int TR_K = 32;       // most pairs
constexpr double TR_RES = 5e-14;   // accepted residual, relative to the matrix's norm bound
constexpr double TR_ORTH = 1e-11;  // accepted |z_a . z_b|

// LDS of one solve besides the matrix and the 2 x n x KP vector buffer.
struct TriLds {
  alignas(16) double2 uw[TR_N + 16];  // the pending rank-2 update's (u_j, w_j), zero from TR_N on
  alignas(16) double2 de[TR_N];       // tridiagonal: diagonal and e_{i-1}^2 (0 at i = 0), floored at 1e-34
  alignas(16) double un[TR_N + 16];   // the step's reflector, zero from TR_N on
  double e[TR_N + 1];     // off-diagonal e_i between i - 1 and i (0 at both ends)
  double hinv[TR_N];      // 1/h of reflector s (0: none)
  double lam[TR_K];       // eigenvalues, descending
  double lo, hi, nrm;     // interval that holds them, bound of the norm (all scaled)
  int ex;                 // the matrix was scaled by 2^-ex
};

// LDS operations of one wave complete in order: only the compiler has to be held.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_or0(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROWS, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Sum over the wave's first n lanes (x is zero from lane n on) by DPP row shifts and row
// broadcasts (no LDS permutes), in every lane.
__device__ __forceinline__ double wave_sum_dpp(double x, int n) {
  x += dpp_or0<0x111>(x);
  x += dpp_or0<0x112>(x);
  x += dpp_or0<0x114>(x);
  x += dpp_or0<0x118>(x);
  if (n <= 16) return lane_bcast(x, 15);
  x += dpp_or0<0x142, 0xa>(x);
  if (n <= 32) return lane_bcast(x, 31);
  x += dpp_or0<0x143, 0xc>(x);
  return lane_bcast(x, 63);
}

// Sum over groups of L (1, 2, 4 or 8) neighbouring lanes, in every lane of the group.
template <int L>
__device__ __forceinline__ double group_sum(double x) {
  if constexpr (L >= 2) x += dpp_or0<0xB1>(x);   // quad_perm 1,0,3,2
  if constexpr (L >= 4) x += dpp_or0<0x4E>(x);   // quad_perm 2,3,0,1
  if constexpr (L >= 8) x += dpp_or0<0x141>(x);  // row_half_mirror
  return x;
}

// Three calls with a work-group barrier between them, all on the same L: tri_reduce_wave (one
// wave), tri_sections (every wave), tri_vectors_wave (one wave).
// tri_reduce_wave: a is the symmetric matrix in LDS, rows 0 .. n - 1 of odd stride LD; it is
// overwritten by the reflectors. n <= NR. Returns 0 (to every lane) for a matrix it refuses.
template <int LD, int NR>
__device__ __forceinline__ int tri_reduce_wave(double* __restrict__ a, int n, TriLds* __restrict__ L) {
  const int lane = threadIdx.x & 63;
  const int row = min(lane, n - 1);
  const bool act = lane < n;
  // scale to a largest diagonal entry in [1, 2): a power of two, exact
  double dmax = fabs(a[row * LD + row]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, o, 64));
  if (!(dmax > 1e-280 && dmax < 1e280)) return 0;
  const int ex = ilogb(dmax);
  double u = 0.0, w = 0.0;
  const int nc = (n + 7) >> 3;  // column chunks
  // row `lane` of the trailing matrix, from column s on at step s: r[0] is the next column
  double r[NR];
  {
    const double sc = ldexp(1.0, -ex);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const double x = a[row * LD + min(j, n - 1)];
      r[j] = act && j < n ? sc * x : 0.0;
    }
  }
  if (lane < 16) {
    L->uw[TR_N + lane] = make_double2(0.0, 0.0);
    L->un[TR_N + lane] = 0.0;
  }
  wave_fence();
  // ---- tridiagonalisation: step s reflects column s, and its pass over the trailing columns
  // applies step s - 1's rank-2 update (u, w), forms the product with its reflector and moves
  // the row down by one register (every index stays static in a loop of one body). Only the
  // vectors u, w and the reflector go through LDS, as broadcasts, a chunk of eight columns
  // ahead. Reflector s is left in row s of a, zero at and before s.
  for (int s = 0; s + 2 < n; ++s) {
    const double c = fma(-w, lane_bcast(u, s), fma(-u, lane_bcast(w, s), r[0]));
    const double ds = lane_bcast(c, s), alpha = lane_bcast(c, s + 1);
    const double tail = (act && lane > s + 1) ? c : 0.0;
    const double rest = wave_sum_dpp(tail * tail, n);
    double beta = alpha, hinv = 0.0, un = 0.0;
    if (rest > 1e-290) {
      const double sig = rest + alpha * alpha;
      beta = -copysign(sig * rsq_nr(sig), alpha);
      hinv = rcp_nr(sig - alpha * beta);
      un = lane == s + 1 ? alpha - beta : tail;
    }
    if (lane == 0) {
      L->de[s].x = ds;
      L->de[s + 1].y = fmax(beta * beta, 1e-34);
      L->e[s + 1] = beta;
      L->hinv[s] = hinv;
    }
    L->uw[lane] = make_double2(u, w);
    L->un[lane] = un;
    if (lane < LD) a[s * LD + lane] = un;
    wave_fence();
    double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
    {
      const double2* uw = L->uw + s + 1;
      const double* uv = L->un + s + 1;
      const int rem = n - s - 1;  // trailing columns
      double2 t[2][8];
      double v[2][8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        t[0][q] = uw[q];
        v[0][q] = uv[q];
      }
#pragma unroll
      for (int j = 0; j < NR / 8; ++j) {
        if (8 * j >= rem) break;
        if (j + 1 < NR / 8) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            t[(j + 1) & 1][q] = uw[8 * (j + 1) + q];
            v[(j + 1) & 1][q] = uv[8 * (j + 1) + q];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        double d[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int x = min(8 * j + 1 + q, NR - 1);  // (past the row's end: unused)
          d[q] = fma(-w, t[j & 1][q].x, fma(-u, t[j & 1][q].y, r[x]));
          r[8 * j + q] = d[q];
        }
        p0 = fma(d[0], v[j & 1][0], p0);
        p1 = fma(d[1], v[j & 1][1], p1);
        p2 = fma(d[2], v[j & 1][2], p2);
        p3 = fma(d[3], v[j & 1][3], p3);
        p0 = fma(d[4], v[j & 1][4], p0);
        p1 = fma(d[5], v[j & 1][5], p1);
        p2 = fma(d[6], v[j & 1][6], p2);
        p3 = fma(d[7], v[j & 1][7], p3);
      }
    }
    const double p = act && lane > s ? ((p0 + p1) + (p2 + p3)) * hinv : 0.0;
    const double kk = 0.5 * hinv * wave_sum_dpp(un * p, n);
    u = un;
    w = p - kk * un;
    wave_fence();
  }
  {  // the last 2 x 2 block (1 x 1 when n = 1)
    const int s = n >= 2 ? n - 2 : 0;
    const double c = r[0] - (u * lane_bcast(w, s) + w * lane_bcast(u, s));
    const double cl = (n >= 2 ? r[1] : r[0]) - (u * lane_bcast(w, n - 1) + w * lane_bcast(u, n - 1));
    const double ds = lane_bcast(c, s), es = lane_bcast(c, n - 1), dl = lane_bcast(cl, n - 1);
    if (lane == 0) {
      if (n >= 2) {
        L->de[s].x = ds;
        L->e[n - 1] = es;
        L->de[n - 1].y = fmax(es * es, 1e-34);
      }
      L->de[n - 1].x = dl;
      L->de[0].y = 0.0;
      L->e[0] = 0.0;
      L->e[n] = 0.0;
    }
    wave_fence();
  }
  // ---- Gershgorin interval
  double lo, hi;
  {
    const double d = L->de[row].x;
    const double r = fabs(L->e[row]) + fabs(L->e[row + 1]);
    lo = d - r;
    hi = d + r;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = fmin(lo, __shfl_xor(lo, o, 64));
      hi = fmax(hi, __shfl_xor(hi, o, 64));
    }
  }
  const double nrm = fmax(fabs(lo), fabs(hi));
  if (!(nrm < 1e6)) return 0;
  lo -= 1e-15 * nrm;
  hi += 1e-15 * nrm;
  const int n8 = 8 * nc;
  if (lane >= n && lane < n8) L->de[lane] = make_double2(4.0 * nrm + 4.0, 0.0);  // no sign change there
  wave_fence();
  if (lane == 0) {
    L->lo = lo;
    L->hi = hi;
    L->nrm = nrm;
    L->ex = ex;
  }
  wave_fence();
  return 1;
}

// ---- multisection for the k largest eigenvalues (descending, in L->lam): the work-group's NW
// waves share them out, G lanes per eigenvalue, two points each, narrow its interval by 2 G + 1
// each time (the two recurrences of a lane fill each other's latency)
template <int KP, int NW>
__device__ __forceinline__ void tri_sections(int n, int k, TriLds* __restrict__ L) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nc = (n + 7) >> 3, n8 = 8 * nc;
  constexpr int EW = KP > NW ? KP / NW : 1, G = 64 / EW;  // eigenvalues per wave, lanes per eigenvalue
  if (wv * EW < k) {
    constexpr int S = 2 * G;
    constexpr int IT = G == 64 ? 8 : G == 32 ? 9 : G == 16 ? 11 : G == 8 ? 14 : G == 4 ? 18 : 24;  // (S + 1)^IT >= 2^54
    const int mi = wv * EW + lane / G, m = min(mi, k - 1), jg = lane % G;
    double lo = L->lo, hi = L->hi;
    constexpr double inv = 1.0 / (S + 1);
    for (int it = 0; it < IT; ++it) {
      const double step = (hi - lo) * inv;
      const double x0 = fma(step, (double)(jg + 1), lo), x1 = fma(step, (double)(jg + 1 + G), lo);
      // p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}: its sign changes count the eigenvalues
      // below x. The pair is rescaled by a power of two every sixteen steps, over which it
      // grows by less than (2 nrm + 1)^16 < 1e102 (d, x and e are within the norm's bound, which
      // tri_reduce_wave holds under 1e6) and shrinks by no more than the floor 1e-34 of e^2
      // every two.
      double am = 0.0, ac = 1.0, bm = 0.0, bc = 1.0;
      int nega = 0, negb = 0;
      unsigned sa = 0, sb = 0;  // signs, newest lowest
      double2 t[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) t[q] = L->de[q];
      for (int i = 0; i < n8; i += 8) {
        const int in = min(i + 8, n8 - 8);
        double2 tn[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) tn[q] = L->de[in + q];
        sa &= 1;
        sb &= 1;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const double an = fma(t[q].x - x0, ac, -t[q].y * am), bn = fma(t[q].x - x1, bc, -t[q].y * bm);
          sa = __builtin_amdgcn_alignbit(sa, (unsigned)__double2hiint(an), 31);  // sa << 1 | sign
          sb = __builtin_amdgcn_alignbit(sb, (unsigned)__double2hiint(bn), 31);
          am = ac;
          ac = an;
          bm = bc;
          bc = bn;
        }
        nega += __popc((sa ^ (sa >> 1)) & 0xff);
        negb += __popc((sb ^ (sb >> 1)) & 0xff);
        if (i & 8) {
          const int ha = -max(__builtin_amdgcn_frexp_exp(ac), __builtin_amdgcn_frexp_exp(am));
          const int hb = -max(__builtin_amdgcn_frexp_exp(bc), __builtin_amdgcn_frexp_exp(bm));
          ac = ldexp(ac, ha);
          am = ldexp(am, ha);
          bc = ldexp(bc, hb);
          bm = ldexp(bm, hb);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) t[q] = tn[q];
      }
      // points below lambda_m, of the group's S
      const unsigned long long ua = __ballot(n - nega > m), ub = __ballot(n - negb > m);
      constexpr unsigned long long mask = ~0ull >> (64 - G);
      const int cnt = __popcll((ua >> (lane - jg)) & mask) + __popcll((ub >> (lane - jg)) & mask);
      if (cnt < S) hi = fma(step, (double)(cnt + 1), lo);
      lo = fma(step, (double)cnt, lo);
    }
    if (jg == 0 && mi < k) L->lam[mi] = 0.5 * (lo + hi);
  }
}

// tri_vectors_wave: a as tri_reduce_wave left it; buf: 2 * n * KP doubles, wbuf: KP * KP. On
// success (returned to every lane) store(c, i, v) has been called once for every component
// i < n of every eigenvector c < k, signed so that its largest-magnitude component is positive
// (the first one on a tie), and L->lam is in the matrix's own scale. Called by one whole wave;
// other waves must not touch a, buf or L meanwhile.
template <int KP, int LD, typename Store>
__device__ __forceinline__ int tri_vectors_wave(const double* __restrict__ a, int n, int k, TriLds* __restrict__ L,
                                                double* __restrict__ buf, double* __restrict__ wbuf, Store&& store) {
  const int lane = threadIdx.x & 63;
  const int row = min(lane, n - 1);
  const bool act = lane < n;
  const double nrm = L->nrm;
  const int ex = L->ex;
  // ---- eigenvectors of the tridiagonal. Lane c runs the top-down factorisation of
  // T - lambda_c, lane KP + c the bottom-up one (multipliers l_i = e / D_i in Lf and Lb);
  // the vector starts with 1 where the twisted pivot
  //   gamma_i = (d_i - lambda) - e_{i-1} lf_{i-1} - e_i lb_{i+1}
  // is least and continues up through lf and down through lb.
  double* Lf = buf;           // n x KP, the vectors afterwards
  double* Lb = buf + n * KP;  // n x KP
  const int c = lane % KP;
  const bool down = lane < KP;
  const bool cv = lane < 2 * KP && c < k;
  const int mate = down ? lane + KP : lane - KP;
  const double lam = L->lam[min(c, k - 1)];
  int tw = 0;  // the twist's row
  double sn = 0.0, bad = 0.0;
  if (cv) {
    const int i0 = down ? 0 : n - 1, di = down ? 1 : -1;
    double* dst = (down ? Lf : Lb) + c;
    double prod = 0.0;  // e_{i-1} l_{i-1} of the row before
    double dx = L->de[i0].x, en = L->e[down ? 1 : n - 1];
    for (int t = 0; t < n; ++t) {
      const int i = i0 + di * t;
      const int i2 = min(max(i + di, 0), n - 1);
      const double dn = L->de[i2].x, en2 = L->e[down ? i2 + 1 : i2];
      double D = (dx - lam) - prod;
      if (fabs(D) < 1e-40) D = -1e-40;
      const double l = en * rcp_nr(D);
      prod = en * l;
      dst[i * KP] = l;
      dx = dn;
      en = en2;
    }
  }
  wave_fence();
  if (cv) {
    double best = 1e300;
    // each half looks at every other row, then they agree
#pragma unroll 4
    for (int i = down ? 0 : 1; i < n; i += 2) {
      const double f = i > 0 ? L->e[i] * Lf[(i - 1) * KP + c] : 0.0;
      const double b = i + 1 < n ? L->e[i + 1] * Lb[(i + 1) * KP + c] : 0.0;
      const double g = fabs((L->de[i].x - lam) - f - b);
      if (g < best) {
        best = g;
        tw = i;
      }
    }
    const double ob = __shfl(best, mate, 64);
    const int orr = __shfl(tw, mate, 64);
    if (ob < best || (ob == best && orr < tw)) tw = orr;
  }
  wave_fence();
  if (cv) {
    double zz = 1.0, ss = down ? 1.0 : 0.0;
    const double* src = (down ? Lf : Lb) + c;
    const int cnt = down ? tw : n - 1 - tw, di = down ? -1 : 1;
    double l[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) l[q] = src[min(max(tw + di * (1 + q), 0), n - 1) * KP];
    for (int t = 1; t <= cnt; t += 4) {
      double ln[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) ln[q] = src[min(max(tw + di * (t + 4 + q), 0), n - 1) * KP];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (t + q <= cnt) {
          zz *= -l[q];
          Lf[(tw + di * (t + q)) * KP + c] = zz;
          ss += zz * zz;
        }
        l[q] = ln[q];
      }
    }
    if (down) Lf[tw * KP + c] = 1.0;
    ss += __shfl(ss, mate, 64);
    sn = rsq_nr(ss);
  }
  if (lane < 2 * KP && c >= k)
    for (int i = down ? 0 : 1; i < n; i += 2) Lf[i * KP + c] = 0.0;
  wave_fence();
  // normalise, and check the residual (T - lambda) z
  if (cv) {
    const int i0 = down ? 0 : n / 2, i1 = down ? n / 2 : n;
    double zp = i0 > 0 ? Lf[(i0 - 1) * KP + c] * sn : 0.0, zc = Lf[i0 * KP + c] * sn;
    for (int i = i0; i < i1; ++i) {
      const double zn = i + 1 < n ? Lf[(i + 1) * KP + c] * sn : 0.0;
      const double t = (L->de[i].x - lam) * zc + L->e[i] * zp + L->e[i + 1] * zn;
      bad = fmax(bad, fabs(t) < 1e300 ? fabs(t) : 1e300);
      Lb[i * KP + c] = zc;
      zp = zc;
      zc = zn;
    }
  }
  if (lane < 2 * KP && c >= k)
    for (int i = down ? 0 : 1; i < n; i += 2) Lb[i * KP + c] = 0.0;
  wave_fence();
  if (__ballot(bad > TR_RES * nrm)) return 0;
  // ---- mutual orthogonality: each lane some of the KP x KP products
  {
    constexpr int NB = KP * KP / 64;  // columns per lane
    const int ra = lane / (KP / NB), cb = (lane % (KP / NB)) * NB;
    double dot[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) dot[q] = 0.0;
#pragma unroll 2
    for (int i = 0; i < n; ++i) {
      const double za = Lb[i * KP + ra];
#pragma unroll
      for (int q = 0; q < NB; ++q) dot[q] += za * Lb[i * KP + cb + q];
    }
    double off = 0.0;
#pragma unroll
    for (int q = 0; q < NB; ++q)
      if (cb + q != ra) off = fmax(off, fabs(dot[q]));
    if (__ballot(off > 0.1)) return 0;
    if (__ballot(off > TR_ORTH)) {
      // Gram-Schmidt in order, twice per vector (row i on lane i): a vector moves by the
      // part of it along its cluster's earlier ones only, whose eigenvalues are its own to
      // the same digits, so the residuals stay
      for (int j = 1; j < k; ++j) {
        double zj = act ? Lb[row * KP + j] : 0.0;
        for (int rep = 0; rep < 2; ++rep) {
          double corr = 0.0;
          for (int b = 0; b < j; ++b) {
            const double zb = act ? Lb[row * KP + b] : 0.0;
            corr = fma(wave_sum_dpp(zb * zj, n), zb, corr);
          }
          zj -= corr;
        }
        zj *= rsq_nr(wave_sum_dpp(zj * zj, n));
        if (act) Lb[row * KP + j] = zj;
        wave_fence();
      }
    }
  }
  // ---- back-transformation z <- H_0 ... H_{n-3} z: 16 (8) vectors at a time, GB lanes per
  // vector, whose rows p + GB q stay in registers; the results go to Lf
  constexpr int VB = KP < 16 ? KP : 16, GB = 64 / VB, R = 64 / GB;
  const int cz0 = lane / GB, p = lane % GB;
  for (int v0 = 0; v0 < k; v0 += VB) {
    const int cz = v0 + cz0;
    double z[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = p + GB * q;
      z[q] = i < n ? Lb[i * KP + cz] : 0.0;
    }
    // rows are read up to the last lane's: row s has LD entries, zero from n on
    double uu[R];
    auto load = [&](int s) {
#pragma unroll
      for (int q = 0; q < R; ++q) uu[q] = (GB * (q + 1) <= LD) ? a[s * LD + p + GB * q] : 0.0;
    };
    if (n >= 3) load(n - 3);
    for (int s = n - 3; s >= 0; --s) {
      double v[R];
#pragma unroll
      for (int q = 0; q < R; ++q) v[q] = uu[q];
      const double hv = L->hinv[s];
      load(max(s - 1, 0));
      double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
#pragma unroll
      for (int q = 0; q < R; q += 4) {
        t0 = fma(v[q], z[q], t0);
        t1 = fma(v[q + 1], z[q + 1], t1);
        t2 = fma(v[q + 2], z[q + 2], t2);
        t3 = fma(v[q + 3], z[q + 3], t3);
      }
      const double t = group_sum<GB>((t0 + t1) + (t2 + t3)) * hv;
#pragma unroll
      for (int q = 0; q < R; ++q) z[q] = fma(-t, v[q], z[q]);
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (p + GB * q < n) Lf[(p + GB * q) * KP + cz] = z[q];
  }
  wave_fence();
  // ---- one Newton-Schulz step Z <- Z - Z (Z^T Z - I) / 2: the vectors' mutual products are
  // of the order of u / (relative gap) until here and of u afterwards, which error terms that
  // take the bases as orthonormal rely on
  for (int x = lane; x < KP * KP; x += 64) {
    const int i0 = x / KP, i1 = x % KP;
    double t0 = 0.0, t1 = 0.0;
    if (i0 < k && i1 < k) {
      int i = 0;
      for (; i + 2 <= n; i += 2) {
        t0 = fma(Lf[i * KP + i0], Lf[i * KP + i1], t0);
        t1 = fma(Lf[(i + 1) * KP + i0], Lf[(i + 1) * KP + i1], t1);
      }
      if (i < n) t0 = fma(Lf[i * KP + i0], Lf[i * KP + i1], t0);
    }
    wbuf[x] = 0.5 * ((i0 == i1 ? t0 - 1.0 : t0) + t1);
  }
  wave_fence();
  for (int v0 = 0; v0 < k; v0 += VB) {
    const int cz = min(v0 + cz0, k - 1);
    double z[R], dz[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      z[q] = Lf[min(p + GB * q, n - 1) * KP + cz];
      dz[q] = 0.0;
    }
    for (int b = 0; b < k; ++b) {
      const double wb = wbuf[b * KP + cz];
#pragma unroll
      for (int q = 0; q < R; ++q) dz[q] = fma(wb, Lf[min(p + GB * q, n - 1) * KP + b], dz[q]);
    }
    // canonical sign
    double best = -1.0, bv = 1.0;
    int bi = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = p + GB * q;
      z[q] -= dz[q];
      if (i < n && fabs(z[q]) > best) {
        best = fabs(z[q]);
        bi = i;
        bv = z[q];
      }
    }
#pragma unroll
    for (int o = 1; o < GB; o <<= 1) {
      const double ob = __shfl_xor(best, o, 64), ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ob > best || (ob == best && oi < bi)) {
        best = ob;
        bi = oi;
        bv = ov;
      }
    }
    const double sg = bv < 0.0 ? -1.0 : 1.0;
    if (v0 + cz0 < k) {
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (p + GB * q < n) store(cz, p + GB * q, sg * z[q]);
    }
  }
  if (lane < k) L->lam[lane] = ldexp(L->lam[lane], ex);
  wave_fence();
  return 1;
}

}  // namespace ht
