// ir.hip -- iterative refinement of tau00 against the FP64 KKR matrix.
//
// The factors P^T L U of a copy of the KKR matrix (tau_lu.hip) are a
// preconditioner; the answer is refined against the FP64 matrix M:
//   X_0 = 0;  R = B - M X (FP64, MFMA);  dX = (LU)^-1 R;  X += dX
// with B = [0; t0] in the solver layout (t0 in the central rows), until the
// central rows converge: ||dX_c||_F <= tol ||X_c||_F.  tau00 = X_c.
// Two instantiations of the correction type T:
//   float   mixed precision: complex FP32 factors and sweeps;
//   double  FP64 factors and sweeps, used when the tile-local pivots of a
//           plain FP64 factorization come out small, to recover full FP64
//           accuracy (residuals against the untouched M).
// The reference's only mixed-precision routes are LAPACK zcgesv
// (linearSolvers_CPU.cpp:148-174, which never fills its right-hand side) and
// cusolverDnIRSXgesv (linearSolvers_CUDA.cu:425-470); both refine a full
// solve the same way.
//
// Forward and backward sweeps use the block structure of the tile-pivoted
// factorization: for tile row s,
//   y_s = L_ss^-1 P_s (r_s - sum_{t<s} L_st y_t)      (L_st stored left of the diagonal tile)
//   x_s = U_ss^-1 (y_s - sum_{t>s} U_st x_t)
// with the diagonal-tile inverses and permutations kept by the factorization;
// the sums are taken right-looking, one tile column per launch (k_ir_step).
#include <type_traits>

#include "lu_common.hpp"

namespace lsmsx {

typedef GCx<double> gd2;

// X = 0 and the first residual R = B - M*0 = B ([0; t0], t0 in the central
// rows), so the first sweep needs no pass over M.  One workgroup per 64-row
// tile and solve (one per solve took 26 us for 32 solves of N = 864).
template <class T>
__global__ __launch_bounds__(256) void k_ir_init(const SolveDesc *__restrict__ descs) {
  typedef CxT<T> V;
  const SolveDesc &d = descs[blockIdx.y];
  if ((int)blockIdx.x >= d.nt) return;
  gd2 *X = (gd2 *)d.X;
  GCx<T> *R = (GCx<T> *)d.R;
  const int Ns = d.Ns, kc = d.kc;
  const int row = kTile * blockIdx.x + (threadIdx.x & 63);
  for (int col = threadIdx.x >> 6; col < kc; col += 4) {
    const long e = row + (long)Ns * col;
    X[e] = make_double2(0.0, 0.0);
    V b;
    b.x = T(0);
    b.y = T(0);
    if (row >= Ns - kc) {
      const double2 t = d.t0[(row - (Ns - kc)) + (long)d.ldt * col];
      b.x = (T)t.x;
      b.y = (T)t.y;
    }
    R[e] = b;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *d.conv = 0;
    *d.iters = 0;
    *d.dxn = 0.0;
    *d.dxn_rho2 = 0.0;
  }
}

// R = B - M X for one 64-row tile (blockIdx.x) of one solve (blockIdx.y);
// wave w handles rows 16w.. of the tile, all kc = 16 NB right-hand sides.
// FP64 MFMA in the 3M, transposed form of the LU update:
//   a-operand X(k0+kq, j0+li), b-operand M(i0+li, k0+kq).
// M streams from HBM in 32-column chunks through two register buffers: the
// loads of chunk c+1 are in flight during the MFMAs of chunk c.  The chunk's
// 32 x kc block of X is staged in LDS once per workgroup (the four waves
// share it), alternating between two buffers so that one barrier per chunk
// suffices.  The residual is stored in the correction type T.
template <class T, int NB>
__global__ __launch_bounds__(256) void k_ir_residual(const SolveDesc *__restrict__ descs) {
  typedef CxT<T> V;
  constexpr int KC = 32;               // k per chunk
  constexpr int XQ = KC * 16 * NB / 256;  // X values per thread per chunk
  const SolveDesc &d = descs[blockIdx.y];
  if (*d.conv) return;
  const int tile = blockIdx.x;
  if (tile >= d.nt) return;
  __shared__ double2 xs[2][KC][16 * NB + 1];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int w = tid >> 6;
  const int i0 = tile * kTile + 16 * w;
  const long ld = d.ld;
  const int Ns = d.Ns, kc = d.kc;
  const gd2 *__restrict__ M = (const gd2 *)d.M + i0;
  const gd2 *__restrict__ X = (const gd2 *)d.X;
  d4 q[3][NB];
  // accumulators start from B: rows >= Ns - kc hold t0
#pragma unroll
  for (int jb = 0; jb < NB; jb++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      int row = i0 + li, col = 16 * jb + kq + 4 * r;
      double2 b = make_double2(0.0, 0.0);
      if (row >= Ns - kc) b = d.t0[(row - (Ns - kc)) + (long)d.ldt * col];
      q[0][jb][r] = b.x;
      q[1][jb][r] = 0.0;
      q[2][jb][r] = b.x + b.y;
    }
  auto load = [&](int k0, double2 (&m)[KC / 4], double2 (&xv)[XQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < KC / 4; u++) m[u] = ldg<double>(M + li + ld * (k0 + 4 * u + kq));
#pragma unroll
    for (int qq = 0; qq < XQ; qq++) {
      const int e = tid + 256 * qq;
      xv[qq] = ldg<double>(X + (k0 + e % KC) + (long)Ns * (e / KC));
    }
  };
  auto compute = [&](int buf, const double2 (&m)[KC / 4], const double2 (&xv)[XQ])
                     __attribute__((always_inline)) {
#pragma unroll
    for (int qq = 0; qq < XQ; qq++) {
      const int e = tid + 256 * qq;
      xs[buf][e % KC][e / KC] = xv[qq];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < KC / 4; u++) {
      const double mr = -m[u].x, mi = -m[u].y, ms = mr + mi;
#pragma unroll
      for (int jb = 0; jb < NB; jb++) {
        const double2 x = xs[buf][4 * u + kq][16 * jb + li];
        q[0][jb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, mr, q[0][jb], 0, 0, 0);
        q[1][jb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, mi, q[1][jb], 0, 0, 0);
        q[2][jb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x + x.y, ms, q[2][jb], 0, 0, 0);
      }
    }
  };
  double2 ma[KC / 4], mb[KC / 4], xa[XQ], xb[XQ];
  load(0, ma, xa);
  for (int k0 = 0; k0 < Ns; k0 += 2 * KC) {  // Ns is a multiple of 64
    load(k0 + KC, mb, xb);
    compute(0, ma, xa);
    if (k0 + 2 * KC < Ns) load(k0 + 2 * KC, ma, xa);
    compute(1, mb, xb);
  }
  GCx<T> *R = (GCx<T> *)d.R;
#pragma unroll
  for (int jb = 0; jb < NB; jb++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      V o;
      o.x = (T)(q[0][jb][r] - q[1][jb][r]);
      o.y = (T)(q[2][jb][r] - q[0][jb][r] - q[1][jb][r]);
      R[(i0 + li) + (long)Ns * (16 * jb + kq + 4 * r)] = o;
    }
  }
}

// (-1)^l of the lm index a = l(l+1) + m, a < 16.
__device__ __forceinline__ double lsign(int a) { return (a == 0 || (a >= 4 && a < 9)) ? 1.0 : -1.0; }

// Padding rows of the residual, R = -X (identity block, B = 0), by a workgroup
// of 512 threads.
__device__ __forceinline__ void residual_g_pad(const SolveDesc &d) {
  const int tid = threadIdx.x, Ns = d.Ns, pad = d.pad, kc = d.kc;
  const gd2 *__restrict__ X = (const gd2 *)d.X;
  GCx<float> *__restrict__ R = (GCx<float> *)d.R;
  for (int e = tid; e < pad * kc; e += 512) {
    const int row = e % pad, col = e / pad;
    const double2 x = ldg<double>(X + row + (long)Ns * col);
    float2 o;
    o.x = (float)-x.x;
    o.y = (float)-x.y;
    R[row + (long)Ns * col] = o;
  }
}

// R_q = B_q - X_q + t_q Y_q (M = 1 - t G) of site q by a wave, Y_q in the MFMA
// accumulator layout; R stored in FP32.
__device__ __forceinline__ void residual_g_site(const SolveDesc &d, int q, const double2 (&yv)[4]) {
  const int n = d.numLIZ, lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  const int Ns = d.Ns, pad = d.pad, kc = d.kc;
  const gd2 *__restrict__ X = (const gd2 *)d.X;
  GCx<float> *__restrict__ R = (GCx<float> *)d.R;
  // t_q Y_q: a-operand t(li, 4u + kq), b-operand Y(4u + kq, li) = yv[u]
  const int site = site_at_pos(q, n);
  const gd2 *__restrict__ T = (const gd2 *)(d.tmat + d.ldT * d.store[site] + d.t_off);
  d4 q1 = {0.0, 0.0, 0.0, 0.0}, q2 = q1, q3 = q1;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const double2 tv = ldg<double>(T + li + (long)d.ldt * (4 * u + kq));
    q1 = mfma4(tv.x, yv[u].x, q1);
    q2 = mfma4(tv.y, yv[u].y, q2);
    q3 = mfma4(tv.x + tv.y, yv[u].x + yv[u].y, q3);
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int row = pad + 16 * q + kq + 4 * r;
    const double2 x = ldg<double>(X + row + (long)Ns * li);
    double br = 0.0, bi = 0.0;
    if (row >= Ns - kc) {
      const double2 t = d.t0[(row - (Ns - kc)) + (long)d.ldt * li];
      br = t.x;
      bi = t.y;
    }
    float2 o;
    o.x = (float)(br - x.x + (q1[r] - q2[r]));
    o.y = (float)(bi - x.y + (q3[r] - q1[r] - q2[r]));
    R[row + (long)Ns * li] = o;
  }
}

// Residual of the mixed path without an FP64 M, first half: Y = G X from the
// structure constants stored once per site pair (d.gh, G_pq for solver
// positions p < q; G_qp = D G_pq D, D = diag (-1)^l), each block read once
// and used twice:
//   y_p += G_pq X_q            (row part, kept in the wave's registers)
//   z_q += D G_pq D X_p        (the mirrored block, handed on through LDS)
// Sites go in bands of kGBand; workgroup blockIdx.x takes band rows wg and
// nbands-1-wg (equal work), each band row b the band blocks (b, c >= b).
// Wave w owns sites 2w, 2w+1 of band b; in stage st it takes the sites
// j = (w + st) mod 8 of band c, adding to their z the sums its predecessor
// left in LDS, so every z is summed in one fixed order.  y of band b goes to
// d.ybuf, the z of band block (b, c) to slot (c, b) of d.gpart (complex
// values in the MFMA accumulator layout: element r*64 + lane is row
// kq + 4r, column li).  k_ir_residual_g_finish adds them up.
__global__ __launch_bounds__(512) void k_ir_residual_g(const SolveDesc *__restrict__ descs) {
  const SolveDesc &d = descs[blockIdx.y];
  if (*d.conv) return;
  const int n = d.numLIZ, nbands = (n + kGBand - 1) / kGBand;
  const int wg = blockIdx.x;
  if (wg >= (nbands + 1) / 2 || nbands <= kGDirectBands) return;
  __shared__ double2 zs[kGWaves][kGSites][256];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int Ns = d.Ns, pad = d.pad;
  const gd2 *__restrict__ X = (const gd2 *)d.X;
  const gd2 *__restrict__ GH = (const gd2 *)d.gh;
  gd2 *__restrict__ YB = (gd2 *)d.ybuf;
  gd2 *__restrict__ GP = (gd2 *)d.gpart;
  double sk[4];
#pragma unroll
  for (int u = 0; u < 4; u++) sk[u] = lsign(4 * u + kq);
  for (int pass = 0; pass < 2; pass++) {
    const int b = pass ? nbands - 1 - wg : wg;
    if (pass && b <= wg) break;
    d4 y[kGSites][3];
    double2 xp[kGSites][4];  // D X_p, b-operand (k row 4u + kq, column li)
    int pp[kGSites];
#pragma unroll
    for (int sp = 0; sp < kGSites; sp++) {
      const int p = kGBand * b + kGSites * w + sp;
      pp[sp] = p;
#pragma unroll
      for (int m = 0; m < 3; m++) y[sp][m] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < 4; u++) {
        double2 v = make_double2(0.0, 0.0);
        if (p < n) v = ldg<double>(X + (pad + 16 * p + 4 * u + kq) + (long)Ns * li);
        xp[sp][u] = make_double2(sk[u] * v.x, sk[u] * v.y);
      }
    }
    // the band blocks (b, c >= b), stage by stage, one site q at a time: the
    // next site's blocks (p, q) and X_q are loaded before this site's MFMAs
    const int nit = (nbands - b) * kGWaves * kGSites;
    auto site_q = [&](int it) {
      const int sq = it % kGSites, st = (it / kGSites) % kGWaves;
      const int c = b + it / (kGSites * kGWaves);
      return kGBand * c + kGSites * ((w + st) % kGWaves) + sq;
    };
    auto load_q = [&](int q, double2 (&gg)[kGSites][4], double2 (&xx)[4]) {
#pragma unroll
      for (int sp = 0; sp < kGSites; sp++)
        if (pp[sp] < q && q < n) {
          const gd2 *__restrict__ G = GH + gh_index(pp[sp], q, n) * 256;
#pragma unroll
          for (int u = 0; u < 4; u++) gg[sp][u] = ldg<double>(G + li + 16 * (4 * u + kq));
        }
#pragma unroll
      for (int u = 0; u < 4; u++)
        xx[u] = q < n ? ldg<double>(X + (pad + 16 * q + 4 * u + kq) + (long)Ns * li)
                      : make_double2(0.0, 0.0);
    };
    double2 g[kGSites][4], gn[kGSites][4], xq[4], xqn[4];
    load_q(site_q(0), g, xq);
    for (int it = 0; it < nit; it++) {
      const int sq = it % kGSites, st = (it / kGSites) % kGWaves;
      const int c = b + it / (kGSites * kGWaves);
      const int j = (w + st) % kGWaves, q = kGBand * c + kGSites * j + sq;
      if (it + 1 < nit) load_q(site_q(it + 1), gn, xqn);
      // the predecessor's z sums: all four LDS reads issued together (st is
      // uniform across the wave), one wait
      double2 zv[4];
      if (st > 0) {
#pragma unroll
        for (int r = 0; r < 4; r++) zv[r] = zs[j][sq][r * 64 + lane];
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) zv[r] = make_double2(0.0, 0.0);
      }
      d4 z[3];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        z[0][r] = zv[r].x;
        z[1][r] = 0.0;
        z[2][r] = zv[r].x + zv[r].y;
      }
#pragma unroll
      for (int sp = 0; sp < kGSites; sp++) {
        if (!(pp[sp] < q && q < n)) continue;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const double gs = g[sp][u].x + g[sp][u].y;
          const double2 a = xq[u], e = xp[sp][u];
          y[sp][0] = mfma4(g[sp][u].x, a.x, y[sp][0]);
          y[sp][1] = mfma4(g[sp][u].y, a.y, y[sp][1]);
          y[sp][2] = mfma4(gs, a.x + a.y, y[sp][2]);
          z[0] = mfma4(g[sp][u].x, e.x, z[0]);
          z[1] = mfma4(g[sp][u].y, e.y, z[1]);
          z[2] = mfma4(gs, e.x + e.y, z[2]);
        }
      }
      // hand the z sums on, or write the band block's slot (c, b)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const double2 v = make_double2(z[0][r] - z[1][r], z[2][r] - z[0][r] - z[1][r]);
        if (st < kGWaves - 1) {
          zs[j][sq][r * 64 + lane] = v;
        } else if (q < n) {
          const long slot = (long)c * (c + 1) / 2 + b;
          GP[(slot * kGBand + kGSites * j + sq) * 256 + r * 64 + lane] = v;
        }
      }
      if (sq == kGSites - 1) __syncthreads();  // the stage's z sums are in LDS
#pragma unroll
      for (int sp = 0; sp < kGSites; sp++)
#pragma unroll
        for (int u = 0; u < 4; u++) g[sp][u] = gn[sp][u];
#pragma unroll
      for (int u = 0; u < 4; u++) xq[u] = xqn[u];
    }
#pragma unroll
    for (int sp = 0; sp < kGSites; sp++)
      if (pp[sp] < n)
#pragma unroll
        for (int r = 0; r < 4; r++)
          YB[(long)pp[sp] * 256 + r * 64 + lane] =
              make_double2(y[sp][0][r] - y[sp][1][r], y[sp][2][r] - y[sp][0][r] - y[sp][1][r]);
  }
}

// Second half: for site q of band c = blockIdx.x (wave w: sites 2w, 2w+1),
//   Y_q = ybuf_q + D sum_{b <= c} gpart(c, b)_q          (fixed order)
//   R_q = B_q - X_q + t_q Y_q                            (M = 1 - t G)
// and the padding rows R = -X (identity block, B = 0); R stored in FP32.
__global__ __launch_bounds__(512) void k_ir_residual_g_finish(const SolveDesc *__restrict__ descs) {
  const SolveDesc &d = descs[blockIdx.y];
  if (*d.conv) return;
  const int n = d.numLIZ, nbands = (n + kGBand - 1) / kGBand, c = blockIdx.x;
  if (c >= nbands || nbands <= kGDirectBands) return;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, kq = lane >> 4;
  const gd2 *__restrict__ YB = (const gd2 *)d.ybuf;
  const gd2 *__restrict__ GP = (const gd2 *)d.gpart;
  if (c == 0) residual_g_pad(d);
#pragma unroll
  for (int sq = 0; sq < kGSites; sq++) {
    const int q = kGBand * c + kGSites * w + sq;
    if (q >= n) continue;
    double2 yv[4], zv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      yv[r] = ldg<double>(YB + (long)q * 256 + r * 64 + lane);
      zv[r] = make_double2(0.0, 0.0);
    }
    for (int b = 0; b <= c; b++) {
      const long slot = (long)c * (c + 1) / 2 + b;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const double2 v = ldg<double>(GP + (slot * kGBand + (q - kGBand * c)) * 256 + r * 64 + lane);
        zv[r].x += v.x;
        zv[r].y += v.y;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const double sgn = lsign(kq + 4 * r);
      yv[r].x += sgn * zv[r].x;
      yv[r].y += sgn * zv[r].y;
    }
    residual_g_site(d, q, yv);
  }
}

// The residual of a solve of up to kGDirectBands bands, whole: workgroup p takes
// site p, wave w the blocks of the sites q = w, w + 8, ..., Y_p summed over the
// waves in order.  Every block is read twice, but a solve's products go to as
// many compute units as it has sites, where in bands they are one's to four's,
// in a chain of its stages (16 solves of 15 sites: 57 + 5 -> 26 us, a batch 729
// -> 659 us; 96 of 56 to 128 sites: a batch 18.0 -> 16.8 ms with the line at four
// bands, 16.3 at eight).  In large batches both run at the rate of HBM and the
// caches (2048 of those: 348 ms either way) until the second read shows: 992
// solves of 135 sites, 175 ms in bands, 178 so, and 248 of them 48.1 and 47.2.
// The line is by size alone, so that a solve's result does not depend on its
// batch.
__global__ __launch_bounds__(512) void k_ir_residual_g_site(const SolveDesc *__restrict__ descs) {
  const SolveDesc &d = descs[blockIdx.y];
  if (*d.conv) return;
  const int n = d.numLIZ, p = blockIdx.x;
  if (p >= n || n > kGBand * kGDirectBands) return;
  __shared__ double2 part[kGWaves][256];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  const int Ns = d.Ns, pad = d.pad;
  const gd2 *__restrict__ X = (const gd2 *)d.X;
  const gd2 *__restrict__ GH = (const gd2 *)d.gh;
  if (p == 0) residual_g_pad(d);
  // y over q > p, and z over q < p, where G_pq = D G_qp D is stored as G_qp
  d4 y[3], z[3];
#pragma unroll
  for (int m = 0; m < 3; m++) y[m] = z[m] = d4{0.0, 0.0, 0.0, 0.0};
  auto load_q = [&](int q, double2 (&g)[4], double2 (&x)[4]) __attribute__((always_inline)) {
    const int q1 = min(q, n - 1);
    // q == p has no block: any other one is read and not used
    const int lo = q1 == p ? 0 : min(p, q1), hi = q1 == p ? n - 1 : max(p, q1);
    const gd2 *G = GH + (lo < hi ? gh_index(lo, hi, n) * 256 : 0);
#pragma unroll
    for (int u = 0; u < 4; u++) {
      g[u] = ldg<double>(G + li + 16 * (4 * u + kq));
      x[u] = ldg<double>(X + (pad + 16 * q1 + 4 * u + kq) + (long)Ns * li);
    }
  };
  auto add = [&](d4 (&a)[3], double2 g, double2 x) __attribute__((always_inline)) {
    a[0] = mfma4(g.x, x.x, a[0]);
    a[1] = mfma4(g.y, x.y, a[1]);
    a[2] = mfma4(g.x + g.y, x.x + x.y, a[2]);
  };
  double2 g[4], x[4], gn[4], xn[4];
  if (n > 1) {
    load_q(w, g, x);
    for (int q = w; q < n; q += kGWaves) {
      load_q(q + kGWaves, gn, xn);
      if (q > p) {
#pragma unroll
        for (int u = 0; u < 4; u++) add(y, g[u], x[u]);
      } else if (q < p) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const double s = lsign(4 * u + kq);
          add(z, g[u], make_double2(s * x[u].x, s * x[u].y));
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        g[u] = gn[u];
        x[u] = xn[u];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const double s = lsign(kq + 4 * r);
    part[w][r * 64 + lane] = make_double2(y[0][r] - y[1][r] + s * (z[0][r] - z[1][r]),
                                          y[2][r] - y[0][r] - y[1][r] +
                                              s * (z[2][r] - z[0][r] - z[1][r]));
  }
  __syncthreads();
  if (w > 0) return;
  double2 yv[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    yv[r] = part[0][r * 64 + lane];
#pragma unroll
    for (int v = 1; v < kGWaves; v++) {
      yv[r].x += part[v][r * 64 + lane].x;
      yv[r].y += part[v][r * 64 + lane].y;
    }
  }
  residual_g_site(d, p, yv);
}

// 3M sums of a wave's 16 x 16nb block in the refinement sweeps: transposed
// MFMA form as in the LU update (a-operand B(k0+kq, j0+li), b-operand
// A(i0+li, k0+kq)).  Register r of lane (li, kq) holds output (row i0+li,
// column 16jb + acc_row<T>(kq, r)).
template <class T>
struct AccIR {
  Acc4<T> p[3][2];
};

// 3M sums started from C: q1 = Cre, q2 = 0, q3 = Cre + Cim; with the
// products accumulated against -A this gives C - A B = (q1 - q2, q3 - q1 - q2).
template <class T>
__device__ __forceinline__ void acc_from(AccIR<T> &q, int jb, int r, CxT<T> c) {
  q.p[0][jb][r] = c.x;
  q.p[1][jb][r] = T(0);
  q.p[2][jb][r] = c.x + c.y;
}
template <class T>
__device__ __forceinline__ CxT<T> acc_value(const AccIR<T> &q, int jb, int r) {
  CxT<T> v;
  v.x = q.p[0][jb][r] - q.p[1][jb][r];
  v.y = q.p[2][jb][r] - q.p[0][jb][r] - q.p[1][jb][r];
  return v;
}
template <class T>
__device__ __forceinline__ void acc_zero(AccIR<T> &q) {
#pragma unroll
  for (int jb = 0; jb < 2; jb++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      q.p[0][jb][r] = T(0);
      q.p[1][jb][r] = T(0);
      q.p[2][jb][r] = T(0);
    }
}

// dX = (P^T L U)^-1 R in the correction type, in place in R, by right-looking
// tile steps: one launch per step, one workgroup per (tile, solve), so a
// sweep streams the stored factors with the whole chip instead of one
// workgroup per solve.
//   forward, step s = -1 .. nt-2, workgroup tile t = s+1+bx < nt:
//     r_t -= L_ts y_s                       (s >= 0; y_s is final in rows s)
//     t == s+1:  y_t = L_tt^-1 P_t r_t       (and, t == nt-1, x_t = U_tt^-1 y_t)
//   backward, launch j = 0 .. nt-2, s = nt-1-j (x_s final), tile t = bx < s:
//     y_t -= U_ts x_s;   t == s-1:  x_t = U_tt^-1 y_t
// Solves of different sizes run the forward steps from the first tile and
// the backward steps from their own last tile.  The first sweep starts from
// R = B, zero outside the last tile; with tile-local pivoting its forward
// steps leave every earlier tile at zero, so it runs as one launch
// (step = kIrFirstSweep) that only finishes the last tile of each solve.
// Wave w handles rows 16w.. of tile t; the 64 x kc block of tile s is
// staged in LDS by the workgroup.
template <class T, bool FWD>
__global__ __launch_bounds__(256) void k_ir_step(const SolveDesc *__restrict__ descs, int step) {
  typedef CxT<T> V;
  const SolveDesc &d = descs[blockIdx.y];
  if (*d.conv || half_sweeps<T>(d.kc, d.nt)) return;
  const int nt = d.nt;
  const bool first = FWD && step == kIrFirstSweep;
  const int s = FWD ? (first ? nt - 2 : step) : nt - 1 - step;
  const int t = FWD ? s + 1 + (int)blockIdx.x : (int)blockIdx.x;
  if (FWD ? t >= nt : t >= s) return;
  __shared__ V buf[kTile][32 + 1];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int kc = d.kc, Ns = d.Ns, nb = kc / 16;
  const long ld = tile_ld(d);
  GCx<T> *R = (GCx<T> *)d.R;
  auto col_of = [&](int jb, int r) { return 16 * jb + acc_row<T>(kq, r); };
  const int i0 = t * kTile + 16 * w, rs = s * kTile;
  // factor tile (t, s), rows of this wave
  const GCx<T> *__restrict__ Wt = tile_ptr<T>(d, t, s < 0 ? 0 : s) + 16 * w;
  const bool diag = FWD ? t == s + 1 : t == s - 1;
  const GCx<T> *__restrict__ inv = (const GCx<T> *)d.inv + t * d.inv_stride + 16 * w + li;
  // every global load of the step is issued before the first wait: the
  // factor tile (t, s) in MFMA layout, r_t, the 64 x kc block of tile s, and
  // in the workgroup of the next diagonal tile that tile's inverse and pivots.
  // The launch is one link of a serial chain and as long as the latencies in
  // it: with the inverse loaded behind the product, four k-steps at a time,
  // 32 canted solves of N = 864 took 3.34 ms, so 2.93 ms.
  V a[kTile / 4], st[8], ia[kTile / 4];
  int pk[kTile / 4];
  if (diag) {
#pragma unroll
    for (int u = 0; u < kTile / 4; u++) {
      ia[u] = ldg<T>(inv + kTile * (4 * u + kq));
      pk[u] = FWD ? ((const LSMSX_GLOBAL int *)d.perm)[t * kTile + 4 * u + kq] : 4 * u + kq;
    }
  }
  if (s >= 0 && !first) {
#pragma unroll
    for (int u = 0; u < kTile / 4; u++) a[u] = ldg<T>(Wt + li + ld * (4 * u + kq));
#pragma unroll
    for (int qq = 0; qq < 8; qq++) {
      const int e = tid + 256 * qq;
      if (qq < kc / 4) st[qq] = ldg<T>(R + (rs + (e & 63)) + (long)Ns * (e >> 6));
    }
  }
  AccIR<T> q;
#pragma unroll
  for (int jb = 0; jb < 2; jb++)
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (jb < nb) acc_from<T>(q, jb, r, R[(i0 + li) + (long)Ns * col_of(jb, r)]);
  if (s >= 0 && !first) {
#pragma unroll
    for (int qq = 0; qq < 8; qq++) {
      const int e = tid + 256 * qq;
      if (qq < kc / 4) buf[e & 63][e >> 6] = st[qq];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTile / 4; u++) {
      V l = a[u];
      l.x = -l.x;
      l.y = -l.y;
      const T ls = l.x + l.y;
#pragma unroll
      for (int jb = 0; jb < 2; jb++) {
        if (jb < nb) {
          const V bb = buf[4 * u + kq][16 * jb + li];
          q.p[0][jb] = mfma4(bb.x, l.x, q.p[0][jb]);
          q.p[1][jb] = mfma4(bb.y, l.y, q.p[1][jb]);
          q.p[2][jb] = mfma4(bb.x + bb.y, ls, q.p[2][jb]);
        }
      }
    }
  }
  if (diag) {
    auto to_buf = [&]() {
      __syncthreads();
#pragma unroll
      for (int jb = 0; jb < 2; jb++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (jb < nb) buf[16 * w + li][col_of(jb, r)] = acc_value<T>(q, jb, r);
      __syncthreads();
      acc_zero<T>(q);
    };
    // the block times the unit lower L^-1 (rows of buf in pivot order) or the
    // upper U^-1, diagonal included, both from the tile in ia
    const int ii = 16 * w + li;
    auto apply = [&](auto lower) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < kTile / 4; u++) {
        const int k = 4 * u + kq;
        V l = ia[u];
        if (lower ? ii <= k : ii > k) {
          l.x = lower && ii == k ? T(1) : T(0);
          l.y = T(0);
        }
        const T ls = l.x + l.y;
#pragma unroll
        for (int jb = 0; jb < 2; jb++) {
          if (jb < nb) {
            const V bb = buf[lower ? pk[u] : k][16 * jb + li];
            q.p[0][jb] = mfma4(bb.x, l.x, q.p[0][jb]);
            q.p[1][jb] = mfma4(bb.y, l.y, q.p[1][jb]);
            q.p[2][jb] = mfma4(bb.x + bb.y, ls, q.p[2][jb]);
          }
        }
      }
    };
    to_buf();
    if (FWD) {
      apply(std::true_type{});
      if (t == nt - 1) {
        to_buf();
        apply(std::false_type{});
      }
    } else {
      apply(std::false_type{});
    }
  }
#pragma unroll
  for (int jb = 0; jb < 2; jb++)
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (jb < nb) R[(i0 + li) + (long)Ns * col_of(jb, r)] = acc_value<T>(q, jb, r);
}

// X += dX for the rows of one tile of one solve.  central = 1: the last tile
// (which holds the central rows and is final once the forward steps end),
// with the sums ||dX_c||^2 and ||X_c||^2 over the central rows; central = 0:
// tile blockIdx.x < nt-1, after the backward steps.  The convergence test runs
// between the two, so a solve that converges skips the backward half of its
// last sweep (the other rows of X are not used again).
template <class T>
__global__ __launch_bounds__(256) void k_ir_accum(const SolveDesc *__restrict__ descs, int central) {
  typedef CxT<T> V;
  const SolveDesc &d = descs[blockIdx.y];
  if (*d.conv || half_sweeps<T>(d.kc, d.nt)) return;
  const int t = central ? d.nt - 1 : (int)blockIdx.x;
  if (!central && t >= d.nt - 1) return;
  __shared__ double red[2][256];
  const int tid = threadIdx.x, Ns = d.Ns, kc = d.kc;
  gd2 *X = (gd2 *)d.X;
  const GCx<T> *R = (const GCx<T> *)d.R;
  double dn = 0.0, xn = 0.0;
  for (int e = tid; e < kTile * kc; e += 256) {
    const int row = t * kTile + (e & 63);
    const long idx = row + (long)Ns * (e >> 6);
    const V dx = R[idx];
    double2 x = X[idx];
    x.x += dx.x;
    x.y += dx.y;
    X[idx] = x;
    if (row >= Ns - kc) {
      dn += (double)dx.x * dx.x + (double)dx.y * dx.y;
      xn += x.x * x.x + x.y * x.y;
    }
  }
  if (!central) return;
  red[0][tid] = dn;
  red[1][tid] = xn;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (tid < off) {
      red[0][tid] += red[0][tid + off];
      red[1][tid] += red[1][tid + off];
    }
    __syncthreads();
  }
  if (tid == 0) {
    d.nrm[0] = red[0][0];
    d.nrm[1] = red[1][0];
    d.nrm[2] = 0.0;
    d.nrm[3] = 0.0;
  }
}

// Convergence of each unconverged solve after a sweep (one thread per solve).
// The next error is about rho ||dX|| with rho = ||dX_k|| / ||dX_{k-1}|| the
// observed contraction; converge when that estimate (and ||dX|| itself, to
// 1e-8) is below tol, or when ||dX_c|| <= tol ||X_c|| outright.
// The convergence test of one solve on ||dX_c||^2 = dn2 and ||X_c||^2 = xn2
// of the sweep just finished (one thread).
__device__ inline void ir_decide_one(const SolveDesc &d, double dn2, double xn2, double tol) {
  const int k = *d.iters;
  const double prev = *d.dxn;  // previous ||dX_c||^2
  bool ok = false;
  if (k >= 1 && prev > 0.0) {
    // the larger of the last two observed contractions, so that one
    // unusually small ratio does not end the refinement early
    const double rho2 = fmax(dn2 / prev, *d.dxn_rho2);
    ok = (rho2 < 1.0) && (rho2 * dn2 <= tol * tol * xn2) && (dn2 <= 1e-16 * xn2);
    *d.dxn_rho2 = dn2 / prev;
  }
  if (dn2 <= tol * tol * xn2) ok = true;
  *d.iters = k + 1;
  *d.dxn = dn2;
  if (ok) *d.conv = 1;
}

__global__ void k_ir_decide(const SolveDesc *__restrict__ descs, int n, double tol) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  const SolveDesc &d = descs[b];
  if (*d.conv) return;
  ir_decide_one(d, d.nrm[0] + d.nrm[2], d.nrm[1] + d.nrm[3], tol);
}

// ---------------------------------------------------------------------------
// One refinement sweep per launch, one workgroup per solve (kc = 16, complex
// FP32 factors, tile-major): dX = (P^T L U)^-1 R, the convergence test on the
// central rows between the forward and the backward halves, and X += dX.  It
// does the work of k_ir_step, k_ir_accum and k_ir_decide for one sweep.
// With kc = 32 a workgroup takes 16 of the columns, and the halves are
// launches of their own (kSweepFwd, kSweepBwd) with k_ir_decide between them,
// for the solves of a chunk that half_sweeps names.
//
// Left-looking by tile row, with the tile rows dealt round-robin to teams of
// NW = 4/RB waves (one wave, or a pair): team p of n takes t = p, p+n, ...
// (forward, ascending) and computes
//   y_t = L_tt^-1 P_t (r_t - sum_{s<t} L_ts y_s),
// 16 RB rows by each wave, with its block in MFMA accumulators (3M form), then
// publishes y_t (in place of r_t in R) by a workgroup-scope count in LDS; the
// waves that need y_s wait on it.  The backward half runs the same way from
// the last tile down (x_t = U_tt^-1 (y_t - sum_{s>t} U_ts x_s)).  Every wave
// waits only for tiles below its own (above, backward) and, before the
// diagonal product, for its partner at the same tile, and takes its tiles in
// order, so the waits always end.  The diagonal-tile inverse is applied as one
// more operand, its input staged in the team's LDS slot (a wave of a pair
// writes it once its partner has read the last one).
// All operand tiles (L_ts, U_ts, the inverses) stream from HBM through a
// ring of k-steps per wave that runs on across tiles.  The published y_s / x_s
// are kept in LDS with pairs (up to kSweepPairTiles tiles); with single waves
// they go through R and come from L2, one item ahead when the count is full.
// HBM traffic per sweep: the factors once, R and X; no launch per tile
// column.  The first sweep (R = B, zero outside the last tile, so y_t = 0
// for t < nt-1 under tile-local pivoting) runs only the last tile forward.
// With few tiles the sweep is the chain of its diagonal tiles (update with
// the last y, diagonal product, publish), half as long by pairs; with many it
// is HBM or a compute unit's MFMAs, and single waves read y half as often
// (sweep_pairs has both sides).  The arithmetic of both is the same.

template <bool FIRST, int RB, SweepPart PART>
__global__ __launch_bounds__(kSweepWaves * 64) void k_ir_sweep(const SolveDesc *__restrict__ descs,
                                                               double tol) {
  typedef float2 V;
  constexpr int NW = 4 / RB, NT = kSweepWaves / NW;  // waves of a team, teams
  constexpr bool YL = NW > 1;                        // y_s / x_s in LDS
  // k-steps (4 columns of a 16 RB x 64 operand) in flight per wave
  constexpr int kSweepD = 16 / RB;
  const SolveDesc &d = descs[blockIdx.x];
  if (*d.conv) return;
  if (PART != kSweepAll && !half_sweeps<float>(d.kc, d.nt)) return;
  const int nt = d.nt, Ns = d.Ns;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), team = w / NW, half = w % NW;
  __shared__ V slot[NT][kTile][17];  // a team's block, input of its diagonal step
  __shared__ int ready[kSweepMaxTiles], done[kSweepMaxTiles], arrived[NT], taken[NT];
  __shared__ int conv_flag;
  __shared__ __align__(16) V ybuf[YL ? kSweepPairTiles : 1][kTile][16];
  for (int i = tid; i < kSweepMaxTiles; i += kSweepWaves * 64) {
    ready[i] = 0;
    done[i] = 0;
    if (i < NT) {
      arrived[i] = 0;
      taken[i] = 0;
    }
  }
  __syncthreads();
  // kSweepFwd, kSweepBwd: the workgroup's 16 columns of 32
  const long c0 = PART == kSweepAll ? 0 : (long)Ns * (16 * blockIdx.y);
  const int central = kTile - d.kc;  // first central row in the last tile
  GCx<float> *R = (GCx<float> *)d.R + c0;
  gd2 *X = (gd2 *)d.X + c0;
  const GCx<float> *__restrict__ F = (const GCx<float> *)d.A;  // tile-major factors
  const GCx<float> *__restrict__ Inv = (const GCx<float> *)d.inv;
  const LSMSX_GLOBAL int *Perm = (const LSMSX_GLOBAL int *)d.perm;
  const long istr = d.inv_stride;
  const int row0 = 16 * RB * half;  // the wave's rows of a tile
  const int loff = row0 + li + kTile * kq;

  f4 q1[RB], q2[RB], q3[RB];  // 3M sums of the wave's block: (16 rb + li, 4 kq + r)
  V ycur[16], ynext[16];   // y_s / x_s operand: (4 kk + kq, li); ynext not with ybuf
  int phase = 0;           // diagonal products of the team so far

  // ---- operand stream.  Items are the wave's rows of 64 x 64 column-major
  // operands, consumed 4 columns (one k-step) at a time.  Forward items of
  // tile t: s < t: L_ts, s == t: the inverse (lower part), s == t+1: the
  // inverse again (upper part; last tile only).  Backward items of tile t:
  // s > t: U_ts, s == t: the inverse (upper part).
  auto item_base = [&](bool fwd, int t, int s) __attribute__((always_inline)) -> const GCx<float> * {
    const bool inv = fwd ? s >= t : s == t;
    return inv ? Inv + t * istr : F + ((long)s * nt + t) * (kTile * kTile);
  };
  auto next_item = [&](bool fwd, int &t, int &s) __attribute__((always_inline)) -> bool {
    if (fwd) {
      if (s < t || (s == t && t == nt - 1)) {
        s++;
        return true;
      }
      if (FIRST) return false;
      t += NT;
      s = 0;
      return t < nt;
    }
    if (s > t) {
      s--;
      return true;
    }
    t -= NT;
    s = nt - 1;
    return t >= 0;
  };
  // The ring holds the next kSweepD k-steps.  Every item is 16 of them, so a
  // consumer's loads are the rest of its own item and the first of the next,
  // at fixed offsets from the two bases (cb, nb) and without a branch; past
  // the last item they read it again (never consumed), so that the wait
  // counts stay static.
  V rg[kSweepD][RB];
  const GCx<float> *cb = F, *nb = F;
  int pt = 0, ps = 0;
  bool pok = false;
  auto load_slot = [&](const GCx<float> *base, int k) __attribute__((always_inline)) {
    const GCx<float> *src = base + kTile * 4 * k + loff;
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      // the factor streams through once per sweep: non-temporal, so that the
      // published y_s / x_s blocks the waves read from L2 stay there
      typedef float sv2 __attribute__((ext_vector_type(2)));
      const sv2 v = __builtin_nontemporal_load((const sv2 *)(src + 16 * rb));
      rg[k % kSweepD][rb] = make_float2(v.x, v.y);
    }
  };
  auto prime = [&](bool fwd, int t0, int s0, bool ok) __attribute__((always_inline)) {
    pt = t0;
    ps = s0;
    pok = ok;
    cb = ok ? item_base(fwd, t0, s0) : F;
#pragma unroll
    for (int u = 0; u < kSweepD; u++) load_slot(cb, u);
  };
  auto begin_item = [&](bool fwd) __attribute__((always_inline)) {
    pok = pok && next_item(fwd, pt, ps);
    nb = pok ? item_base(fwd, pt, ps) : cb;
  };
  auto refill = [&](int kk) __attribute__((always_inline)) {
    if (kk + kSweepD < 16) load_slot(cb, kk + kSweepD);
    else load_slot(nb, kk + kSweepD - 16);
    if (kk == 15) cb = nb;
    // the loads stay here, kSweepD k-steps before their use
    __builtin_amdgcn_sched_barrier(0);
  };
  // sums += operand * v, v in the MFMA's a-operand layout
  auto step = [&](int rb, V l, V v, float vs) __attribute__((always_inline)) {
    q1[rb] = mfma4(v.x, l.x, q1[rb]);
    q2[rb] = mfma4(v.y, l.y, q2[rb]);
    q3[rb] = mfma4(vs, l.x + l.y, q3[rb]);
  };
  auto consume_update = [&](bool fwd) __attribute__((always_inline)) {
    begin_item(fwd);
#pragma unroll
    for (int kk = 0; kk < 16; kk++) {
      const int u = kk % kSweepD;
      const V yv = ycur[kk];
      const float ys = yv.x + yv.y;
#pragma unroll
      for (int rb = 0; rb < RB; rb++) step(rb, rg[u][rb], yv, ys);
      refill(kk);
    }
  };
  // block - sums of the updates (set by load_block) and plain sums
  auto minus = [&](int rb, int r) __attribute__((always_inline)) {
    return make_float2(q2[rb][r] - q1[rb][r], q1[rb][r] + q2[rb][r] - q3[rb][r]);
  };
  auto plus = [&](int rb, int r) __attribute__((always_inline)) {
    return make_float2(q1[rb][r] - q2[rb][r], q3[rb][r] - q1[rb][r] - q2[rb][r]);
  };
  // What is published: LDS alone (ybuf, the slots), whose fences leave the
  // operand loads in flight, or y_s / x_s in R, whose release waits for all of
  // the wave's memory operations.
  auto release = [&]() __attribute__((always_inline)) {
    if constexpr (YL) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  };
  auto acquire = [&]() __attribute__((always_inline)) {
    if constexpr (YL) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  // Every wait ends (see above); the spin bound (about half a second) only
  // guards the GPU against a broken invariant: the solve then reports
  // kInfoSweepStall and the wave goes on, so the kernel still exits.
  auto wait_count = [&](int *count, int n) __attribute__((always_inline)) {
    unsigned spins = 0;
    while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < n) {
      if (++spins > kSweepSpinLimit) {
        if (lane == 0) *d.info = kInfoSweepStall;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    acquire();
  };
  auto count_full = [&](int *count) __attribute__((always_inline)) {
    return __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= NW;
  };
  auto publish = [&](int *count) __attribute__((always_inline)) {
    release();
    if (lane == 0)
      __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  // block = operand * In, In = the team's slot (rows in pivot order for the
  // unit lower L^-1; as stored for the upper U^-1, diagonal included): the
  // wave's half of In is already in the slot
  auto consume_diag = [&](bool fwd, bool upper, const int (&prow)[16]) __attribute__((always_inline)) {
    begin_item(fwd);
    const V(*in_slot)[17] = slot[team];
    phase++;
    if (NW > 1) {
      publish(arrived + team);
      wait_count(arrived + team, NW * phase);
    } else {
      wave_lds_fence();
    }
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      q1[rb] = f4{0.f, 0.f, 0.f, 0.f};
      q2[rb] = q1[rb];
      q3[rb] = q1[rb];
    }
#pragma unroll
    for (int kk = 0; kk < 16; kk++) ycur[kk] = in_slot[upper ? 4 * kk + kq : prow[kk]][li];
    if (NW > 1) publish(taken + team);
#pragma unroll
    for (int kk = 0; kk < 16; kk++) {
      const int u = kk % kSweepD, k = 4 * kk + kq;
      const V in = ycur[kk];
      const float is = in.x + in.y;
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        const int i = row0 + 16 * rb + li;
        V op = rg[u][rb];
        if (upper ? k < i : k >= i) {
          op.x = (!upper && k == i) ? 1.f : 0.f;
          op.y = 0.f;
        }
        step(rb, op, in, is);
      }
      refill(kk);
    }
  };
  auto load_block = [&](int t, bool fwd) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        // (the first sweep's y are zero but for the last tile)
        const V v = YL && !fwd && PART == kSweepAll ? (FIRST ? make_float2(0.f, 0.f)
                                        : ybuf[YL ? t : 0][row0 + 16 * rb + li][4 * kq + r])
                               : ldg<float>(R + (t * kTile + row0 + 16 * rb + li) + (long)Ns * (4 * kq + r));
        q1[rb][r] = -v.x;
        q2[rb][r] = 0.f;
        q3[rb][r] = -v.x - v.y;
      }
  };
  auto block_to_slot = [&](auto value) __attribute__((always_inline)) {
    V(*out)[17] = slot[team];
    if (NW > 1) wait_count(taken + team, NW * phase);  // the partner has read the last block
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int r = 0; r < 4; r++) out[row0 + 16 * rb + li][4 * kq + r] = value(rb, r);
  };
  auto store_block = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if (YL) ybuf[YL ? t : 0][row0 + 16 * rb + li][4 * kq + r] = plus(rb, r);
        if (!YL || PART == kSweepFwd)
          R[(t * kTile + row0 + 16 * rb + li) + (long)Ns * (4 * kq + r)] = plus(rb, r);
      }
  };
  // X += the block of tile t; returns the sums over the rows that are central
  // if t is the last tile (all of them in the last wave of a team)
  auto add_to_x = [&](int t, double &dn, double &xn) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const long idx = (t * kTile + row0 + 16 * rb + li) + (long)Ns * (4 * kq + r);
        const V dx = plus(rb, r);
        double2 x = X[idx];
        x.x += dx.x;
        x.y += dx.y;
        X[idx] = x;
        if (row0 + 16 * rb >= central) {
          dn += (double)dx.x * dx.x + (double)dx.y * dx.y;
          xn += x.x * x.x + x.y * x.y;
        }
      }
  };
  auto load_y = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 16; kk++) ynext[kk] = ldg<float>(R + (s * kTile + 4 * kk + kq) + (long)Ns * li);
  };
  // the update items of a tile: steps s = first, first + dir, ..., last
  // (inclusive), operand y_s / x_s published under count[s]
  auto run_updates = [&](bool fwd, int first, int last, int *count) __attribute__((always_inline)) {
    const int dir = fwd ? 1 : -1;
    bool have = false;
    for (int s = first; fwd ? s <= last : s >= last; s += dir) {
      if (YL) {
        wait_count(count + s, NW);
#pragma unroll
        for (int kk = 0; kk < 16; kk++) ycur[kk] = ybuf[YL ? s : 0][4 * kk + kq][li];
        consume_update(fwd);
        continue;
      }
      if (!have) {
        wait_count(count + s, NW);
        load_y(s);
      }
#pragma unroll
      for (int kk = 0; kk < 16; kk++) ycur[kk] = ynext[kk];
      have = false;
      const int sn = s + dir;
      if ((fwd ? sn <= last : sn >= last) && count_full(count + sn)) {
        acquire();
        load_y(sn);
        have = true;
      }
      consume_update(fwd);
    }
  };

  const int tl = nt - 1, pl = tl % NT;
  int prow[16] = {};
  // ---- forward half
  if constexpr (PART != kSweepBwd) {
    const int t0 = FIRST ? tl : team;
    const bool mine = FIRST ? team == pl : team < nt;
    prime(true, t0, FIRST ? tl : 0, mine);
    if (mine) {
      for (int t = t0; t < nt; t += NT) {
        load_block(t, true);
#pragma unroll
        for (int kk = 0; kk < 16; kk++) prow[kk] = Perm[t * kTile + 4 * kk + kq];
        if (!FIRST && t > 0) run_updates(true, 0, t - 1, ready);
        block_to_slot(minus);
        consume_diag(true, false, prow);
        if (t == tl) {
          block_to_slot(plus);
          consume_diag(true, true, prow);
          store_block(t);
          double dn = 0.0, xn = 0.0;
          add_to_x(t, dn, xn);
          for (int off = 32; off >= 1; off >>= 1) {
            dn += __shfl_xor(dn, off, 64);
            xn += __shfl_xor(xn, off, 64);
          }
          if (half == NW - 1 && lane == 0) {
            if constexpr (PART == kSweepFwd) {  // k_ir_decide adds up the column halves
              d.nrm[2 * blockIdx.y] = dn;
              d.nrm[2 * blockIdx.y + 1] = xn;
            } else {
              ir_decide_one(d, dn, xn, tol);
              conv_flag = *d.conv;
            }
          }
          publish(done + t);
        } else {
          store_block(t);
          publish(ready + t);
        }
      }
    }
  }
  if constexpr (PART == kSweepFwd) return;
  if constexpr (PART == kSweepBwd) {
    if (YL)  // the last tile's x
      for (int e = tid; e < 16 * kTile; e += kSweepWaves * 64)
        ybuf[YL ? tl : 0][e & 63][e >> 6] = ldg<float>(R + (tl * kTile + (e & 63)) + (long)Ns * (e >> 6));
    if (tid == 0) done[tl] = NW;
  }
  __syncthreads();
  if (PART == kSweepAll && conv_flag) return;

  // ---- backward half: this team's tiles below the last, descending
  {
    const int t0 = team <= nt - 2 ? team + NT * ((nt - 2 - team) / NT) : -1;
    prime(false, t0 < 0 ? 0 : t0, tl, t0 >= 0);
    for (int t = t0; t >= 0; t -= NT) {
      load_block(t, false);
      run_updates(false, tl, t + 1, done);
      block_to_slot(minus);
      consume_diag(false, true, prow);
      store_block(t);
      publish(done + t);  // the other tiles wait for it, not for X
      double dn = 0.0, xn = 0.0;
      add_to_x(t, dn, xn);
    }
  }
}

// tau00 = central rows of X.
__global__ __launch_bounds__(256) void k_ir_extract(const SolveDesc *__restrict__ descs) {
  const SolveDesc &d = descs[blockIdx.x];
  const int kc = d.kc, Ns = d.Ns;
  for (int e = threadIdx.x; e < kc * kc; e += blockDim.x) {
    int r = e % kc, c = e / kc;
    d.tau00[r + kc * c] = d.X[(Ns - kc + r) + (long)Ns * c];
  }
}

__global__ void k_count_conv(const SolveDesc *__restrict__ descs, int n, int *count) {
  __shared__ int s;
  if (threadIdx.x == 0) s = 0;
  __syncthreads();
  int local = 0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) local += *descs[i].conv;
  atomicAdd(&s, local);
  __syncthreads();
  if (threadIdx.x == 0) *count = s;
}

// Copy the FP64 matrix M into the factorization buffer A (FP64), one 64-column
// strip per workgroup, for the FP64-refined route.
__global__ __launch_bounds__(256) void k_copy_m(const SolveDesc *__restrict__ descs) {
  const SolveDesc &d = descs[blockIdx.y];
  const int strip = blockIdx.x;
  if (strip >= d.nt) return;
  const long ld = d.ld, c0 = (long)strip * kTile;
  const gd2 *__restrict__ M = (const gd2 *)d.M;
  gd2 *A = (gd2 *)d.A;
  for (long e = threadIdx.x; e < (long)kTile * d.Ns; e += 256) {
    const long c = c0 + e / d.Ns, r = e % d.Ns;
    A[r + ld * c] = M[r + ld * c];
  }
}

template __global__ void k_ir_init<float>(const SolveDesc *);
template __global__ void k_ir_init<double>(const SolveDesc *);
template __global__ void k_ir_residual<float, 1>(const SolveDesc *);
template __global__ void k_ir_residual<float, 2>(const SolveDesc *);
template __global__ void k_ir_residual<double, 1>(const SolveDesc *);
template __global__ void k_ir_residual<double, 2>(const SolveDesc *);
template __global__ void k_ir_step<float, true>(const SolveDesc *, int);
template __global__ void k_ir_step<float, false>(const SolveDesc *, int);
template __global__ void k_ir_step<double, true>(const SolveDesc *, int);
template __global__ void k_ir_step<double, false>(const SolveDesc *, int);
template __global__ void k_ir_accum<float>(const SolveDesc *, int);
template __global__ void k_ir_accum<double>(const SolveDesc *, int);
template __global__ void k_ir_sweep<true, 2, kSweepAll>(const SolveDesc *, double);
template __global__ void k_ir_sweep<true, 4, kSweepAll>(const SolveDesc *, double);
template __global__ void k_ir_sweep<false, 2, kSweepAll>(const SolveDesc *, double);
template __global__ void k_ir_sweep<false, 4, kSweepAll>(const SolveDesc *, double);
template __global__ void k_ir_sweep<true, 2, kSweepFwd>(const SolveDesc *, double);
template __global__ void k_ir_sweep<false, 2, kSweepFwd>(const SolveDesc *, double);
template __global__ void k_ir_sweep<false, 2, kSweepBwd>(const SolveDesc *, double);

}  // namespace lsmsx
