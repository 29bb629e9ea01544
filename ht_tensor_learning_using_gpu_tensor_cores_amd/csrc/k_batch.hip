// Batched HT of many small, unevenly sized 3rd-order tensors.
//
// Tree {1},{2,3} (node 0 root, 1 = {1}, 2 = {2,3}, 3 = {2}, 4 = {3}) with the reference's
// plain semantics (every non-root node's basis is the exact truncated SVD of its own
// matricisation: third_order_tensor_decompsition/CUDA/Baseline/htd_unopt.cu:65-88):
//   U1, U2, U3   top eigenvectors of the leaf Grams X_(m) X_(m)^T (FP32 MFMA Grams, FP64
//                eigen solver);
//   U23          the complementary node's basis = right singular vectors of X_(1),
//                V diag(1/sigma) with V = X_(1)^T U1, formed slab by slab and never stored;
//   B23          (U2 (x) U3)^T U23 (k2 x k3 x k23), B_root = U1^T X_(1) (U2 (x) U3) B23;
//                both come from the core M = X x1 U1^T x2 U2^T x3 U3^T:
//                B23 = M diag(1/sigma), B_root = M^T B23;
//   rel. error   ||X - X_HT||^2 = ||X||^2 - 2 ||B_root||^2 + tr(B_root B23^T B23 B_root^T)
//                (U1 and U2 (x) U3 orthonormal), all terms in FP64.
// n <= 64, ranks <= 8.
//
// Kernels on one stream: Grams, eigen problems, projections (from a hipGraph once the same
// arguments come a second time in a row). What bounds
// them differs: the Grams FP32 MFMA, the eigen problems barriers and instruction issue of
// cyclic Jacobi, the projections FP64 MFMA. One persistent kernel that ran each tensor's
// phases in turn held every phase to the occupancy of its largest and solved a tensor's three
// eigen problems one after another: 4096 tensors of 16-64 rows 30.2 -> 11.1 ms (11.9 under the
// profiler: Grams 1.0, eigen problems 10.4, projections 0.5), 40 of them 6.4 -> 0.95 ms.
#include <algorithm>

#include "k_tri.h"

namespace ht {

// ------------------------------------------------------------------ Grams
struct __attribute__((packed, aligned(4))) F4u {  // 16 bytes at 4-byte alignment
  float v[4];
};

// use(load(0)), use(load(1)), ..., use(load(count - 1)) with the next two loads in flight:
// three buffers that change roles by unrolling (a buffer copied to another would be waited
// for at the copy). load(buf) is called count times, in order.
template <typename Buf, typename Load, typename Use>
__device__ __forceinline__ void pipelined(int count, Load&& load, Use&& use) {
  Buf b0, b1, b2;
  if (count <= 0) return;
  load(b0);
  if (count > 1) load(b1);
  int i = 0;
  for (; i + 5 <= count; i += 3) {
    load(b2);
    use(b0);
    load(b0);
    use(b1);
    load(b1);
    use(b2);
  }
  // two to four left, two of them loaded
  const int left = count - i;
  if (left > 2) load(b2);
  use(b0);
  if (left > 3) load(b0);
  if (left > 1) use(b1);
  if (left > 2) use(b2);
  if (left > 3) use(b0);
}

template <int NT>
struct GramBuf {
  float v[4][NT];  // step, tile
};

// A wave's tiles of 16 rows and its tile pairs. ALL: every pair ja <= jb of NT tiles (the
// whole Gram). Panel: pairs (0, j), j < NT, of the tiles p, p + 1, p + 2 (mod tiles).
template <int NT, bool ALL>
struct GramAcc {
  static constexpr int P = ALL ? NT * (NT + 1) / 2 : NT;
  f32x4 c[P];
  __device__ __forceinline__ void step(const float (&a)[NT]) {
    int p = 0;
#pragma unroll
    for (int ja = 0; ja < (ALL ? NT : 1); ++ja)
#pragma unroll
      for (int jb = ja; jb < NT; ++jb, ++p) c[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ja], a[jb], c[p], 0, 0, 0);
  }
};

// Grams X_(m) X_(m)^T by FP32 MFMA 16x16x4. Against 32x32 tiles, 16-row ones waste at most 15
// rows of padding and leave out the lower triangle (n = 40: 6 tiles of 256 entries, not 4 of
// 1024). Lane (m = lane % 16, q = lane / 16) holds row m of each tile at column k + q of a
// step; rows past n repeat row n - 1 (their entries are not written). Columns are added in
// ascending order, each entry one chain of FMAs.
// Rows contiguous (mode 0): columns k of n floats, batches of 16 columns; a last short batch
// counts columns past K as zero.
template <int NT, bool ALL>
__device__ __forceinline__ void gram_rows(const float* __restrict__ X, int n, int K, const int (&tile)[NT],
                                          GramAcc<NT, ALL>& acc) {
  const int lane = threadIdx.x & 63, m = lane & 15, q = lane >> 4;
  unsigned off[4][NT];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int j = 0; j < NT; ++j) off[u][j] = n * (4 * u + q) + min(16 * tile[j] + m, n - 1);
  const int nb = K >> 4;
  const float* base = X;
  pipelined<GramBuf<NT>>(
      nb,
      [&](GramBuf<NT>& d) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < NT; ++j) d.v[u][j] = base[off[u][j]];
        base += 16 * n;
      },
      [&](GramBuf<NT>& d) {
#pragma unroll
        for (int u = 0; u < 4; ++u) acc.step(d.v[u]);
      });
  if (K & 15) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = 16 * nb + 4 * u + q;
      float a[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float t = X[n * min(k, K - 1) + min(16 * tile[j] + m, n - 1)];
        a[j] = k < K ? t : 0.f;
      }
      acc.step(a);
    }
  }
}

// 4 x 4 transpose between the lane groups q and the registers e: v[e] of group q goes to
// v[q] of group e (a lane's four consecutive columns become its column of four steps).
template <int NT>
__device__ __forceinline__ void transpose4(GramBuf<NT>& d) {
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    unsigned r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = __float_as_uint(d.v[e][j]);
    auto s02 = __builtin_amdgcn_permlane32_swap(r[0], r[2], false, false);
    auto s13 = __builtin_amdgcn_permlane32_swap(r[1], r[3], false, false);
    auto t01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
    auto t23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
    d.v[0][j] = __uint_as_float(t01[0]);
    d.v[1][j] = __uint_as_float(t01[1]);
    d.v[2][j] = __uint_as_float(t23[0]);
    d.v[3][j] = __uint_as_float(t23[1]);
  }
}

// Columns contiguous along memory (modes 1 and 2): nseg segments (stride sseg) of len
// columns, row r of a segment at rstride r, batches of 16 columns: 16 bytes of each row per
// lane (4-byte aligned); a segment's short last batch loads single values. With SQ also the
// FP64 sum of squares of tile 0's (ALL: every tile's) rows.
template <int NT, bool ALL, bool SQ>
__device__ __forceinline__ void gram_cols(const float* __restrict__ X, int n, int rstride, int nseg, int sseg, int len,
                                          const int (&tile)[NT], GramAcc<NT, ALL>& acc, double& sq) {
  const int lane = threadIdx.x & 63, m = lane & 15, q = lane >> 4;
  unsigned row[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) row[j] = rstride * min(16 * tile[j] + m, n - 1);
  const int nfull = len >> 4, nb = (len + 15) >> 4;  // batches per segment
  int lb = 0, ub = 0;                                // batch to load, batch in use
  const float* base = X;
  pipelined<GramBuf<NT>>(
      nb * nseg,
      [&](GramBuf<NT>& d) {
        if (lb < nfull) {
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const F4u t = *reinterpret_cast<const F4u*>(base + (row[j] + 4 * q));
#pragma unroll
            for (int e = 0; e < 4; ++e) d.v[e][j] = t.v[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < NT; ++j) d.v[e][j] = base[row[j] + min(4 * e + q, (len & 15) - 1)];
        }
        base += 16;
        if (++lb == nb) {
          lb = 0;
          base += sseg - 16 * nb;
        }
      },
      [&](GramBuf<NT>& d) {
        int steps = 4;
        if (ub < nfull) {
          transpose4<NT>(d);
        } else {
          steps = ((len & 15) + 3) >> 2;
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < NT; ++j) d.v[e][j] = 4 * e + q < (len & 15) ? d.v[e][j] : 0.f;
        }
        if (++ub == nb) ub = 0;
        if constexpr (SQ) {
#pragma unroll
          for (int j = 0; j < (ALL ? NT : 1); ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const double t = 16 * tile[j] + m < n ? d.v[e][j] : 0.f;
              sq = fma(t, t, sq);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < steps) acc.step(d.v[e]);
      });
}

// One wave's share of one Gram, written to G (n x n, both triangles), and of ||X||^2 (mode 2).
template <int NT, bool ALL>
__device__ __forceinline__ void gram_task(const float* __restrict__ X, const BatchItem& d, int mode,
                                          const int (&tile)[NT], float* __restrict__ G, double* __restrict__ xsq) {
  const int lane = threadIdx.x;
  const int n1 = d.n[0], n2 = d.n[1], n3 = d.n[2], slab = n1 * n2;
  const int n = mode == 0 ? n1 : (mode == 1 ? n2 : n3);
  GramAcc<NT, ALL> acc;
#pragma unroll
  for (int p = 0; p < acc.P; ++p) acc.c[p] = f32x4{};
  double sq = 0.0;
  if (mode == 0) gram_rows<NT, ALL>(X, n1, n2 * n3, tile, acc);
  else if (mode == 1) gram_cols<NT, ALL, false>(X, n2, n1, n3, slab, n1, tile, acc, sq);
  else gram_cols<NT, ALL, true>(X, n3, slab, 1, 0, slab, tile, acc, sq);
  if (mode == 2) {
    sq = wave_sum_dpp(sq, 64);
    if (lane == 0) *xsq = sq;
  }
  int p = 0;
#pragma unroll
  for (int ja = 0; ja < (ALL ? NT : 1); ++ja)
#pragma unroll
    for (int jb = ja; jb < NT; ++jb, ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 16 * tile[ja] + acc16_row(e, lane), c = 16 * tile[jb] + (lane & 15);
        if (r < n && c < n) {
          G[r * n + c] = acc.c[p][e];
          if (ja != jb) G[c * n + r] = acc.c[p][e];
        }
      }
}

// One wave per work-group. panels = 1: a whole Gram per wave, X read once per mode; for
// batches with waves enough to fill the GPU that way. panels = 4: tile panel p of a Gram per
// wave (T = 4 tiles: 3, 3, 2 and 2 of the 10 pairs), a quarter of the time for a handful of
// tensors at 2.5 times the reads. A tensor's three Grams are 8 work-groups apart, on one XCD
// (work-groups are dealt to the 8 XCDs in turn), whose L2 then serves two of the three reads.
__global__ __launch_bounds__(64) void batch_gram_kernel(BatchRun r, int panels) {
  const int group = blockIdx.x >> 3, pos = 8 * (group / (3 * panels)) + (blockIdx.x & 7);
  const int mode = group % 3, p = (group / 3) % panels;
  if (pos >= r.count) return;
  const int t = r.order[pos];
  const BatchItem& d = r.items[t];
  const int n1 = d.n[0], n2 = d.n[1], n3 = d.n[2];
  const int n = mode == 0 ? n1 : (mode == 1 ? n2 : n3), T = (n + 15) >> 4;
  const float* X = r.x + d.x_off;
  float* G = r.gram + d.g_off + (mode > 0 ? n1 * n1 : 0) + (mode > 1 ? n2 * n2 : 0);
  double* xsq = r.basis + d.u_scr + (long)BT_RMAX * (n1 + n2 + n3 + 3) + p;
  if (panels == 1) {
    if (mode == 2 && threadIdx.x > 0 && threadIdx.x < 4) xsq[threadIdx.x] = 0.0;  // the panels' parts
    const int tile[4] = {0, 1, 2, 3};
    if (T == 1) gram_task<1, true>(X, d, mode, {0}, G, xsq);
    else if (T == 2) gram_task<2, true>(X, d, mode, {0, 1}, G, xsq);
    else if (T == 3) gram_task<3, true>(X, d, mode, {0, 1, 2}, G, xsq);
    else gram_task<4, true>(X, d, mode, tile, G, xsq);
    return;
  }
  if (p >= T) {
    if (mode == 2 && threadIdx.x == 0) *xsq = 0.0;
    return;
  }
  const int a = p, b = (p + 1) % T, c = (p + 2) % T;
  if (T == 1 || (T == 2 && p == 1)) gram_task<1, false>(X, d, mode, {a}, G, xsq);
  else if (T < 4 || p >= 2) gram_task<2, false>(X, d, mode, {a, b}, G, xsq);
  else gram_task<3, false>(X, d, mode, {a, b, c}, G, xsq);
}

// ------------------------------------------------------------------ eigen problems
struct EigTask {
  int n, k, kl, mode;  // rows, pairs, pairs written as U, mode
  const float* G;
  double* Uc;  // n x BT_RMAX row-major, zero from column k on
  double* wc;  // BT_RMAX eigenvalues
  float *U, *s, *s2;  // packed outputs: U_t, singular values, those of node {2,3} (mode 0)
  int k2;
};

__device__ __forceinline__ EigTask eig_task(const BatchRun& r, int id) {
  const BatchItem& d = r.items[id >> 2];
  EigTask e;
  e.mode = id & 3;
  const int leaf = e.mode == 0 ? 1 : e.mode + 2;
  e.n = d.n[e.mode];
  e.kl = d.k[leaf];
  e.k2 = d.k[2];
  e.k = e.mode == 0 ? max(e.kl, e.k2) : e.kl;
  e.G = r.gram + d.g_off;
  e.Uc = r.basis + d.u_scr;
  for (int m = 0; m < e.mode; ++m) {
    e.G += d.n[m] * d.n[m];
    e.Uc += BT_RMAX * d.n[m];
  }
  e.wc = r.basis + d.u_scr + BT_RMAX * (d.n[0] + d.n[1] + d.n[2] + e.mode);
  float* O = r.out + d.out_off;
  e.U = O + d.u_off[leaf];
  e.s = O + d.s_off[leaf];
  e.s2 = O + d.s_off[2];
  return e;
}

__device__ __forceinline__ void eig_store(const EigTask& e, int c, int i, double v) {
  e.Uc[i * BT_RMAX + c] = v;
  if (c < e.kl) e.U[i + (long)e.n * c] = (float)v;
}

__device__ __forceinline__ void eig_values(const EigTask& e, int j, double lam) {
  const float s = (float)sqrt(fmax(lam, 0.0));
  e.wc[j] = lam;
  if (j < e.kl) e.s[j] = s;
  if (e.mode == 0 && j < e.k2) e.s2[j] = s;
}

// One work-group per leaf eigen problem, problems of one size class (rows at most NC) in
// descending size: cyclic Jacobi, then the top k columns with canonical signs. The class sets
// the LDS, and with it the problems per CU that hide each other's barriers and chains: 67 KB
// for 64 rows, 38 KB for 48, 17 KB for 32, 5 KB for 16.
// (The one-wave tridiagonal solver of the single decompositions takes 1.7 ms here, but with it
// the reported relative error moves by 2e-8 of itself: the formula above takes the bases as
// exactly orthonormal and cancels to 1e-6 of ||X||^2, so their squared norms' 1 + 1e-14 shows. A
// quadratic term with the bases' own Grams would cancel that and let the faster solver in.)
// Measured per class at 4096 tensors: 64 rows 8.7 ms with 256 threads a problem, 7.2 with 512;
// 48 rows 2.5 and 2.66.
template <int NC, int NT>
__global__ __launch_bounds__(NT) void batch_eig_kernel(BatchRun r, int first) {
  constexpr int LD = NC + 1;
  __shared__ double a[NC * LD];
  __shared__ double v[NC * LD];
  __shared__ int ordj[SJ];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const EigTask e = eig_task(r, r.eig[first + blockIdx.x]);
  const int n = e.n, np = (n + 1) & ~1;
  jacobi_load<LD>(a, v, e.G, n, n, np, true);
  jacobi_sweeps<NT, LD>(a, v, n, np, 30, 1e-14);
  jacobi_order<LD>(a, np, ordj);
  // canonical signs; one wave per column
  for (int j = w; j < BT_RMAX; j += NT / 64) {
    if (j >= e.k) {
      for (int i = lane; i < n; i += 64) e.Uc[i * BT_RMAX + j] = 0.0;
      continue;
    }
    const int src = ordj[j];
    double best = -1.0;
    int bi = 0;
    for (int i = lane; i < n; i += 64) {
      const double xv = fabs(v[i * LD + src]);
      if (xv > best) { best = xv; bi = i; }
    }
    for (int o = 32; o > 0; o >>= 1) {
      const double ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    const double sg = v[bi * LD + src] < 0.0 ? -1.0 : 1.0;
    for (int i = lane; i < n; i += 64) eig_store(e, j, i, sg * v[i * LD + src]);
    if (lane == 0) eig_values(e, j, a[src * LD + src]);
  }
}

// ------------------------------------------------------------------ projections
// One tensor per work-group of NW waves; wave w takes the slabs i3 = w, w + NW, ... and
// needs no other wave until the end. X is read once, in 64-byte pieces of columns. Per tile
// of 16 columns i2, FP64 MFMA 16x16x4 forms V[i2, c] = sum_i1 X[i1, i2, i3] U1[i1, c]; its
// accumulator element e (row 4 e + lane / 16, column lane % 16) is the operand of step e of
// E[a, c] = sum_i2 U2[i2, a] V[i2, c], so V never leaves the registers; E U3[i3, b] goes into
// the lane's core entries M[a, b, c]. Half of the columns c (16, ranks are at most 8) are
// padding: the matrix pipes are busy 200 us for 4096 tensors of 16 to 64 rows. With vector
// FMAs instead, U1's values from scalar loads, the waits for those took 730-870 us.
template <int NW>
__global__ __launch_bounds__(64 * NW, 3) void batch_proj_kernel(BatchRun r) {
  constexpr int R = BT_RMAX;
  __shared__ double Vs[NW][R * R * R];
  __shared__ double M[R * R * R];  // (a + 8 b) * 8 + c
  __shared__ double B23[R * R * R];
  __shared__ double U3s[BT_NMAX * R];
  __shared__ double Br[R * R];  // a * 8 + c
  __shared__ double sgn[R];
  __shared__ double u1s[16][64], u2s[16][64];
  __shared__ double bvs[NW][64];
  __shared__ int bis[NW][64];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t0 = r.order[blockIdx.x];
  const BatchItem& d = r.items[t0];
  const int n1 = d.n[0], n2 = d.n[1], n3 = d.n[2];
  const int k1 = d.k[1], k23 = d.k[2], k2 = d.k[3], k3 = d.k[4];
  const float* X = r.x + d.x_off;
  const double* U1 = r.basis + d.u_scr;
  const double* U2 = U1 + R * n1;
  const double* U3 = U2 + R * n2;
  const double* wc = U3 + R * n3;
  const int slab = n1 * n2;
  const int c = lane & 15, q = lane >> 4;
  for (int e = tid; e < R * n3; e += 64 * NW) U3s[e] = U3[e];
  // U1 as the right operand (rows i1 = 16 rb + 4 q + j for step j of block rb: the order in
  // which a lane's 16-byte loads of X hold them), U2 as the left one
  for (int f = w; f < 16; f += NW) {
    const int i1 = 16 * (f >> 2) + 4 * q + (f & 3), i2 = 4 * f + q;
    u1s[f][lane] = (i1 < n1 && c < R) ? U1[i1 * R + c] : 0.0;
    u2s[f][lane] = (i2 < n2 && c < R) ? U2[i2 * R + c] : 0.0;
  }
  __syncthreads();
  const int rb = (n1 + 15) >> 4, tb = (n2 + 15) >> 4;
  double bv = 0.0, m[2][R];
  int bi = INT32_MAX;  // nothing seen
#pragma unroll
  for (int b = 0; b < R; ++b) m[0][b] = m[1][b] = 0.0;
  // tiles (i3, t) of the wave in order, their loads two ahead
  int l3 = w, lt = 0, i3 = w, t = 0;  // tile to load, tile in use
  f64x4 E = f64x4{};
  struct Tile {
    float x[4][4];
  };
  pipelined<Tile>(
      ((n3 - w + NW - 1) / NW) * tb,
      [&](Tile& d) {
        const float* base = X + slab * l3;
        const unsigned col = n1 * min(16 * lt + c, n2 - 1);
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (b < rb) {
            if (16 * b + 16 <= n1) {
              const F4u v = *reinterpret_cast<const F4u*>(base + (col + 16 * b + 4 * q));
#pragma unroll
              for (int j = 0; j < 4; ++j) d.x[b][j] = v.v[j];
            } else {  // rows past n1 repeat the last one: U1's operand is zero there
#pragma unroll
              for (int j = 0; j < 4; ++j) d.x[b][j] = base[col + min(16 * b + 4 * q + j, n1 - 1)];
            }
          }
        if (++lt == tb) {
          lt = 0;
          l3 += NW;
        }
      },
      [&](Tile& d) {
        f64x4 V = f64x4{};
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (b < rb) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              V = __builtin_amdgcn_mfma_f64_16x16x4f64((double)d.x[b][j], u1s[4 * b + j][lane], V, 0, 0, 0);
          }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          E = __builtin_amdgcn_mfma_f64_16x16x4f64(u2s[4 * t + e][lane], V[e], E, 0, 0, 0);
          // largest |V| of the column so far (rows ascend): the sign of U23
          const int i2 = 16 * t + 4 * e + q;
          if (i2 < n2 && (fabs(V[e]) > fabs(bv) || bi == INT32_MAX)) {
            bv = V[e];
            bi = i2 + n2 * i3;
          }
        }
        if (++t == tb) {
#pragma unroll
          for (int b = 0; b < R; ++b) {
            const double u = U3s[i3 * R + b];
            m[0][b] = fma(E[0], u, m[0][b]);
            m[1][b] = fma(E[1], u, m[1][b]);
          }
          E = f64x4{};
          t = 0;
          i3 += NW;
        }
      });
  // ---- the waves' cores, and the sign of U23's columns (largest |V|, first one on a tie)
  if (c < R) {
#pragma unroll
    for (int b = 0; b < R; ++b) {
      Vs[w][(q + R * b) * R + c] = m[0][b];
      Vs[w][(4 + q + R * b) * R + c] = m[1][b];
    }
  }
  bvs[w][lane] = bv;
  bis[w][lane] = bi;
  __syncthreads();
  for (int e = tid; e < R * R * R; e += 64 * NW) {
    double s = 0.0;
#pragma unroll
    for (int v = 0; v < NW; ++v) s += Vs[v][e];
    M[e] = s;
  }
  if (tid < R) {
    double b = 0.0;
    int ix = INT32_MAX;
    for (int v = 0; v < 4 * NW; ++v) {
      const double ov = bvs[v >> 2][tid + 16 * (v & 3)];
      const int oi = bis[v >> 2][tid + 16 * (v & 3)];
      if (oi != INT32_MAX && (fabs(ov) > fabs(b) || (fabs(ov) == fabs(b) && oi < ix))) {
        b = ov;
        ix = oi;
      }
    }
    sgn[tid] = b < 0.0 ? -1.0 : 1.0;
  }
  __syncthreads();
  for (int e = tid; e < R * R * R; e += 64 * NW) {
    const int c = e & 7;
    const double s = c < k23 ? sqrt(fmax(wc[c], 0.0)) : 0.0;
    B23[e] = s > 0.0 ? sgn[c] * (M[e] / s) : 0.0;
  }
  __syncthreads();
  if (tid >= 64) return;
  // B_root[a1, c] = sum_p M[p, a1] B23[p, c]; the error terms from B23^T B23 and B_root
  const int la = lane & 7, lc = lane >> 3;
  float* O = r.out + d.out_off;
  double br = 0.0, mcc = 0.0;
#pragma unroll 8
  for (int p = 0; p < R * R; ++p) {
    const double b = B23[p * R + lc];
    br = fma(M[p * R + la], b, br);
    mcc = fma(B23[p * R + la], b, mcc);
  }
  if (la >= k1) br = 0.0;
  Br[la * R + lc] = br;
  if (la < k1 && lc < k23) O[d.b_off[0] + la + k1 * lc] = (float)br;
  for (int e = lane; e < R * R * R; e += 64) {
    const int c = e & 7, a = (e >> 3) & 7, b = e >> 6;
    if (a < k2 && b < k3 && c < k23) O[d.b_off[2] + a + k2 * (b + k3 * c)] = (float)B23[e];
  }
  wave_fence();
  double bb = 0.0;
#pragma unroll
  for (int a = 0; a < R; ++a) bb = fma(Br[a * R + la], Br[a * R + lc], bb);
  const double nb = wave_sum(br * br), tr = wave_sum(mcc * bb);
  if (lane == 0) {
    const double xsq = (wc[3 * R] + wc[3 * R + 1]) + (wc[3 * R + 2] + wc[3 * R + 3]);
    const double num = fmax(xsq - 2.0 * nb + tr, 0.0);
    r.rel_err[t0] = xsq > 0.0 ? sqrt(num / xsq) : 0.0;
  }
}

constexpr int BG_WHOLE = 1024;  // tensors from which a wave takes a whole Gram
// Tensors from which a projection has four waves, not eight: two work-groups of eight a CU hold
// fewer. A fixed rule, since the waves decide the order of sums and with it the last bits.
// Whole call, 16 to 64 rows, eight / four: 40 tensors 0.955 / 0.982 ms, 400 1.965 / 2.026, 1000
// 3.36 / 3.37, 4096 11.30 / 11.13; 8 to 24 rows: 400 0.294 / 0.295, 600 0.322 / 0.315.
constexpr int BP_FOUR = 512;

int batch_ht_launch(hipStream_t st, const BatchRun& r) {
  if (r.count < 1) return 8;
  // whole Grams once their waves outnumber the 1024 SIMDs threefold
  const int panels = r.count >= BG_WHOLE ? 1 : 4;
  hipLaunchKernelGGL(batch_gram_kernel, dim3(24 * panels * ((r.count + 7) / 8)), dim3(64), 0, st, r, panels);
  int first = 0;
  // One launch for every class, 16 waves a problem in the largest class's LDS, or the classes one
  // after another, each as long as its longest problem. Up to 512 problems (two on each of 256
  // CUs) all are resident at once: 40 tensors of 16 to 64 rows 0.96 ms, class after class 1.83.
  // With both long classes in the batch the one launch stays ahead until twice as many: 171
  // tensors 1.00 against 1.90, 300 1.55 / 2.00, 400 1.97 / 2.06, 600 2.88 / 2.58; of 48 to 64 rows
  // 200 2.03 / 2.25, 300 2.82 / 2.84, 400 3.58 / 3.46. Without them it does not: of 8 to 24 rows 170
  // 0.25 / 0.27, 200 0.30 / 0.28, 300 0.41 / 0.29.
  const bool both_long = r.eig_count[2] > 0 && r.eig_count[3] > 0;
  if (3 * r.count <= (both_long ? 1024 : 512)) {
    hipLaunchKernelGGL((batch_eig_kernel<64, 1024>), dim3(3 * r.count), dim3(1024), 0, st, r, 0);
  } else for (int c = BT_CLASSES - 1; c >= 0; --c) {  // the longest first
    const int n = r.eig_count[c];
    if (n > 0) {
      if (c == 3) hipLaunchKernelGGL((batch_eig_kernel<64, 512>), dim3(n), dim3(512), 0, st, r, first);
      else if (c == 2) hipLaunchKernelGGL((batch_eig_kernel<48, 256>), dim3(n), dim3(256), 0, st, r, first);
      else if (c == 1) hipLaunchKernelGGL((batch_eig_kernel<32, 256>), dim3(n), dim3(256), 0, st, r, first);
      else hipLaunchKernelGGL((batch_eig_kernel<16, 256>), dim3(n), dim3(256), 0, st, r, first);
    }
    first += n;
  }
  if (r.count >= BP_FOUR) hipLaunchKernelGGL(batch_proj_kernel<4>, dim3(r.count), dim3(256), 0, st, r);
  else hipLaunchKernelGGL(batch_proj_kernel<8>, dim3(r.count), dim3(512), 0, st, r);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

}  // namespace ht
