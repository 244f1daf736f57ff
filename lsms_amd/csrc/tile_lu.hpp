// tile_lu.hpp -- LU with partial pivoting of one 64 x 64 complex tile, P A = L U,
// as L^-1 and U^-1, by one workgroup of 256 threads.
//
// A tile's factorization is a serial chain (64 pivot searches, each waiting
// for the column before it) that every elimination step of a solve waits for,
// so what counts is the latency of one step, not the flops.  The tile stays in
// LDS and is taken in panels of kPanelW = 4 columns (one k-step of the MFMA):
//   - wave 0 factors the panel (panel_factor), one lane per row, without
//     barriers and without branches.  The pivot search is a wave-wide maximum
//     by DPP; rows are not moved, a mask holds those not yet used as pivots.
//     The pivot row is broadcast by readlane, and every lane's reciprocal is
//     formed beside the search.  Below U the panel is left with the row
//     operations W in the place of L: applied to the columns to the left, which
//     hold the row operations so far, they accumulate L^-1 (L itself is not
//     needed);
//   - every other column becomes a += W y on the MFMA, y the pivot rows as
//     they were before the panel: first, by all four waves, the 16-column block
//     that holds the next panel; the other three blocks by waves 1 to 3, one
//     each, while wave 0 factors the next panel (an FP64 MFMA keeps its wave
//     from issuing anything else, so this work has to be on other SIMDs).
// U^-1 then goes by blocks: 16 x 16 diagonal blocks one row per lane, then
// 16 -> 32 -> 64 with MFMA products.  (A Gauss-Jordan elimination that forms
// A^-1 instead is shorter, but the products with A^-1 lose digits where a tile
// is ill-conditioned: N = 4384, smallest pivot 0.05, tau00 to 1.5e-10 against
// 4e-12.)
// Real and imaginary parts are kept apart in LDS: four rows of an accumulator
// are then a 16- or 32-byte run.
#pragma once
#include "lu_common.hpp"

namespace lsmsx {

constexpr int kPanelW = 4;

// Column stride of a tile in LDS: 16-byte runs stay aligned, and columns lie 4
// banks apart.
template <class T>
constexpr int kTileLd = sizeof(T) == 8 ? kTile + 2 : kTile + 4;

template <class T>
struct TileLds {
  alignas(16) T re[kTile][kTileLd<T>], im[kTile][kTileLd<T>];  // [column][row]
  T wre[2][kPanelW][kTile], wim[2][kPanelW][kTile];  // W of two panels
  CxT<T> dinv[kTile];       // reciprocals of U's diagonal (0 for 0)
  int prow[kTile];          // pivot row of each column
  int info;
  double minpiv;
  __device__ __forceinline__ CxT<T> get(int c, int r) const {
    CxT<T> v;
    v.x = re[c][r];
    v.y = im[c][r];
    return v;
  }
  __device__ __forceinline__ void put(int c, int r, CxT<T> v) {
    re[c][r] = v.x;
    im[c][r] = v.y;
  }
};

// Wave-wide maximum of v (every lane of the wave active), in all lanes.
__device__ __forceinline__ int wave_max_i32(int v) {
  // INT_MIN where a lane has no source: the identity, so that the move is
  // folded into the maximum
#define LSMSX_DPP_MAX(CTRL, ROWS) \
  v = max(v, __builtin_amdgcn_update_dpp((int)0x80000000, v, CTRL, ROWS, 0xf, false))
  LSMSX_DPP_MAX(0x111, 0xf);  // row_shr:1
  LSMSX_DPP_MAX(0x112, 0xf);  // row_shr:2
  LSMSX_DPP_MAX(0x114, 0xf);  // row_shr:4
  LSMSX_DPP_MAX(0x118, 0xf);  // row_shr:8
  LSMSX_DPP_MAX(0x142, 0xa);  // row_bcast:15
  LSMSX_DPP_MAX(0x143, 0xc);  // row_bcast:31
#undef LSMSX_DPP_MAX
  return __builtin_amdgcn_readlane(v, 63);
}

__device__ __forceinline__ double lane_value(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}
// The complex value that lane `lane` (wave-uniform) holds.
template <class V>
__device__ __forceinline__ V lane_value2(V x, int lane) {
  V r;
  r.x = lane_value(x.x, lane);
  r.y = lane_value(x.y, lane);
  return r;
}

// Reciprocal by the hardware approximation and Newton steps (to about one
// ulp): a third of the instructions of a correctly rounded division, which
// every pivot step would wait for.
__device__ __forceinline__ double fast_recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ float fast_recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.f), r, r);
}

// Integer order of the magnitudes |Re| + |Im| of a pivot search (the bits of
// non-negative values order as integers; in FP64 the high words are compared:
// two magnitudes within 2^-20 of each other serve equally well as pivots).
__device__ __forceinline__ int pivot_key(double m) { return __double2hiint(m); }
__device__ __forceinline__ int pivot_key(float m) { return __float_as_int(m); }

// x + m u
template <class V>
__device__ __forceinline__ V cadd_mul(V x, V m, V u) {
  x.x = x.x + m.x * u.x - m.y * u.y;
  x.y = x.y + m.x * u.y + m.y * u.x;
  return x;
}

// x - l u
template <class V>
__device__ __forceinline__ V csub_mul(V x, V l, V u) {
  x.x = x.x - l.x * u.x + l.y * u.y;
  x.y = x.y - l.x * u.y - l.y * u.x;
  return x;
}

// Factor columns j0 .. j0+kPanelW-1 of the tile (v, one lane per row); rows not
// yet used as pivots are set in the mask `unused`, and the pivot of column j
// comes from the rows below nd while j < nd, from any row afterwards.  With p
// the pivot row and d the pivot of a column, every row i still unused gets
// -(v_i / d) times row p: the columns of the panel to the right change, and so
// do the row operations that stand in place of those to the left.  On return v
// holds, in the rows used up to a column, that column of U, and in the others
// (mask below[j]) W: the row operation of row i with the pivot row of the
// column (a zero pivot leaves everything as it is: then the whole column is 0
// in the unused rows).  pl: the pivot rows, rec: -1/d, 0 for a zero pivot.  One
// wave; no branch, so that the search of a column and the updates of the others
// interleave.
template <class T>
__device__ __forceinline__ void panel_factor(CxT<T> (&v)[kPanelW], int j0, int nd,
                                             unsigned long long &unused, int (&pl)[kPanelW],
                                             CxT<T> (&rec)[kPanelW],
                                             unsigned long long (&below)[kPanelW]) {
  typedef CxT<T> V;
#pragma unroll
  for (int j = 0; j < kPanelW; j++) {
    const T m = cabs1(v[j]);
    const unsigned long long eligible = j0 + j < nd && nd < kTile ? (1ull << nd) - 1 : ~0ull;
    const int key = __builtin_amdgcn_inverse_ballot_w64(unused & eligible) ? pivot_key(m) : -1;
    // -1 / v[j], every lane's own, beside the search
    T s = fast_recip(v[j].x * v[j].x + v[j].y * v[j].y);
    s = m == T(0) ? T(0) : s;
    V rc;
    rc.x = -v[j].x * s;
    rc.y = v[j].y * s;
    const int p = __builtin_ctzll(__ballot(key == wave_max_i32(key)));
    rec[j] = lane_value2(rc, p);
    unused &= ~(1ull << p);
    const bool rest = __builtin_amdgcn_inverse_ballot_w64(unused);
    V l = cmul2(v[j], rec[j]);
    asm volatile("" : "+v"(l.x), "+v"(l.y));  // in every lane: no branch around it
    v[j].x = rest ? l.x : v[j].x;
    v[j].y = rest ? l.y : v[j].y;
    l.x = rest ? l.x : T(0);
    l.y = rest ? l.y : T(0);
#pragma unroll
    for (int k = 0; k < kPanelW; k++)
      if (k != j) v[k] = cadd_mul(v[k], l, lane_value2(v[k], p));
    pl[j] = p;
    below[j] = unused;
  }
}

// Four consecutive rows of a column at p (one or two 16-byte accesses).
template <class T>
__device__ __forceinline__ Acc4<T> get_rows(const T *p) {
  return *(const Acc4<T> *)__builtin_assume_aligned(p, 16);
}
template <class T>
__device__ __forceinline__ void put_rows(T *p, const Acc4<T> &q) {
  *(Acc4<T> *)__builtin_assume_aligned(p, 16) = q;
}

// Element (r, c) of a tile's upper triangle, 0 below the diagonal (read first
// and masked after, so that no branch stands before the read).
template <class T>
__device__ __forceinline__ CxT<T> upper_at(const TileLds<T> &t, int r, int c) {
  CxT<T> v = t.get(c, r);
  v.x = r <= c ? v.x : T(0);
  v.y = r <= c ? v.y : T(0);
  return v;
}

// 16 x 16 complex MFMA accumulators, 4M form: register r of lane (li, kq) is
// element (li, acc_row(kq, r)).
template <class T>
struct BlockAcc {
  Acc4<T> re = {}, im = {};
};
// q += A B for 16 x 16 blocks: fa(i, k), fb(k, j).
template <class T, class FA, class FB>
__device__ __forceinline__ void block_mac(FA fa, FB fb, BlockAcc<T> &q) {
  typedef CxT<T> V;
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int k0 = 0; k0 < 16; k0 += 4) {
    const V a = fa(li, k0 + kq), b = fb(k0 + kq, li);
    q.re = mfma4(b.x, a.x, q.re);
    q.im = mfma4(b.x, a.y, q.im);
    q.re = mfma4(b.y, -a.y, q.re);
    q.im = mfma4(b.y, a.x, q.im);
  }
}

// In-place inverse of the upper triangle of t (dinv: the reciprocals of its
// diagonal).  256 threads; starts after and ends with a barrier.
template <class T>
__device__ __forceinline__ void tile_invert_upper(TileLds<T> &t) {
  typedef CxT<T> V;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // diagonal 16 x 16 block w: row li of the inverse on lane li,
  // x_c = (e_c - sum_{k<c} x_k U(k, c)) / U(c, c)
  if (lane < 16) {
    const int base = 16 * w;
    T fx[2][16], fy[2][16];
    V x[16];
    // row k of U is read while row k - 1 is eliminated (and no further ahead:
    // the 120 entries of a block do not fit the registers)
    auto read = [&](int k) __attribute__((always_inline)) {
#pragma unroll
      for (int c = k + 1; c < 16; c++) {
        fx[k & 1][c] = t.re[base + c][base + k];
        fy[k & 1][c] = t.im[base + c][base + k];
      }
    };
    read(0);
#pragma unroll
    for (int c = 0; c < 16; c++) {
      x[c].x = c == li ? T(1) : T(0);
      x[c].y = T(0);
    }
#pragma unroll
    for (int k = 0; k < 16; k++) {
      if (k < 14) read(k + 1);
      x[k] = cmul2(x[k], t.dinv[base + k]);
#pragma unroll
      for (int c = k + 1; c < 16; c++) x[c] = csub_mul(x[c], x[k], V{fx[k & 1][c], fy[k & 1][c]});
      // computed here, and not where it is stored
      asm volatile("" : "+v"(x[k].x), "+v"(x[k].y));
    }
#pragma unroll
    for (int c = 0; c < 16; c++)
      if (c >= li) t.put(base + c, base + li, x[c]);
  }
  __syncthreads();
  auto put = [&](int bi, int bj, const BlockAcc<T> &q, T sgn) {
#pragma unroll
    for (int r = 0; r < 4; r++)
      t.put(16 * bj + acc_row<T>(kq, r), 16 * bi + li, V{sgn * q.re[r], sgn * q.im[r]});
  };
  auto full = [&](int bi, int bj) {
    return [&t, bi, bj](int r, int c) { return t.get(16 * bj + c, 16 * bi + r); };
  };
  auto diag = [&](int b) {
    return [&t, b](int r, int c) { return upper_at<T>(t, 16 * b + r, 16 * b + c); };
  };
  // 16 -> 32: X_ij = -X_ii (U_ij X_jj), blocks (0,1) and (2,3)
  if (w < 2) {
    const int i = 2 * w, j = i + 1;
    BlockAcc<T> q;
    block_mac<T>(full(i, j), diag(j), q);
    put(i, j, q, T(1));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    BlockAcc<T> x;
    block_mac<T>(diag(i), full(i, j), x);
    put(i, j, x, T(-1));
  }
  __syncthreads();
  // 32 -> 64: the off-diagonal 32 x 32 part F becomes -X_a (F X_b): block
  // (i, j) = (0 or 1, 2 or 3) of either product by wave 2 i + j - 2
  const int i = w >> 1, j = 2 + (w & 1);
  {
    BlockAcc<T> q;
    if (j == 3) block_mac<T>(full(i, 2), full(2, 3), q);
    block_mac<T>(full(i, j), diag(j), q);
    __syncthreads();  // every wave has read F
    put(i, j, q, T(1));
  }
  __syncthreads();
  {
    BlockAcc<T> q;
    if (i == 0) block_mac<T>(full(0, 1), full(1, j), q);
    block_mac<T>(diag(i), full(i, j), q);
    __syncthreads();  // every wave has read F X_b
    put(i, j, q, T(-1));
  }
  __syncthreads();
}

// Factor the tile load(row, column), P A = L U: on return t holds L^-1
// below the diagonal (which is 1) and U on and above it, dinv the reciprocals of
// U's diagonal, prow the permutation (row r of P A is row prow[r] of A).  info:
// col_base + the first column with a zero pivot (1-based), or 0; minpiv: the
// smallest |pivot|.  The pivots of columns below nd come from the rows below nd,
// so the rows from nd on (the central site of the last tile) never pivot into
// the rest.  256 threads; ends with a barrier.
template <class T, class LD>
__device__ __forceinline__ void tile_lu(TileLds<T> &t, LD load, int nd, int col_base) {
  typedef CxT<T> V;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  {
    T re[kTile / 4], im[kTile / 4];  // (an array of structs would go to scratch)
#pragma unroll
    for (int q = 0; q < kTile / 4; q++) {
      const V x = load(lane, w + 4 * q);
      re[q] = x.x;
      im[q] = x.y;
    }
#pragma unroll
    for (int q = 0; q < kTile / 4; q++) {
      t.re[w + 4 * q][lane] = re[q];
      t.im[w + 4 * q][lane] = im[q];
    }
  }
  __syncthreads();
  // row of a 16-row block that lane li feeds to the MFMA as its row li, so that
  // register r of lane (li, kq) is row 4kq + r in FP64 too (there the
  // accumulator's row is kq + 4r)
  const int wrow = sizeof(T) == 8 ? 4 * (li & 3) + (li >> 2) : li;
  // rows 16 rb .. of a column block: acc += W y, W of the panel at c0
  auto operand = [&](int c0, int rb) __attribute__((always_inline)) {
    const int h = (c0 / kPanelW) & 1;
    V a;
    a.x = t.wre[h][kq][16 * rb + wrow];
    a.y = t.wim[h][kq][16 * rb + wrow];
    return a;
  };
  auto update = [&](Acc4<T> &re, Acc4<T> &im, V a, V y) __attribute__((always_inline)) {
    re = mfma4(a.x, y.x, re);
    im = mfma4(a.x, y.y, im);
    re = mfma4(-a.y, y.y, re);
    im = mfma4(a.y, y.x, im);
  };
  // column block b by one wave, for the panel at c0
  auto block_update = [&](int c0, int b) __attribute__((always_inline)) {
    const int col = 16 * b + li, pk = t.prow[c0 + kq];
    const bool on = (unsigned)(col - c0) >= kPanelW;  // not the panel itself
    V y;
    y.x = t.re[col][pk];
    y.y = t.im[col][pk];
    V a[4];
    Acc4<T> re[4], im[4];
#pragma unroll
    for (int rb = 0; rb < 4; rb++) {
      a[rb] = operand(c0, rb);
      re[rb] = get_rows<T>(&t.re[col][16 * rb + 4 * kq]);
      im[rb] = get_rows<T>(&t.im[col][16 * rb + 4 * kq]);
    }
#pragma unroll
    for (int rb = 0; rb < 4; rb++) {
      update(re[rb], im[rb], a[rb], y);
      if (on) {
        put_rows<T>(&t.re[col][16 * rb + 4 * kq], re[rb]);
        put_rows<T>(&t.im[col][16 * rb + 4 * kq], im[rb]);
      }
    }
  };
  unsigned long long unused = ~0ull;
#pragma unroll 1
  for (int c0 = 0; c0 < kTile; c0 += kPanelW) {
    if (w == 0) {
      __builtin_amdgcn_s_setprio(3);  // its reads before those of the other blocks
      V v[kPanelW], rec[kPanelW];
      int pl[kPanelW];
      unsigned long long below[kPanelW];
#pragma unroll
      for (int c = 0; c < kPanelW; c++) {
        v[c].x = t.re[c0 + c][lane];
        v[c].y = t.im[c0 + c][lane];
      }
      panel_factor<T>(v, c0, nd, unused, pl, rec, below);
      const int h = (c0 / kPanelW) & 1;
#pragma unroll
      for (int c = 0; c < kPanelW; c++) {
        const bool on = __builtin_amdgcn_inverse_ballot_w64(below[c]);
        t.put(c0 + c, lane, v[c]);
        t.wre[h][c][lane] = on ? v[c].x : T(0);
        t.wim[h][c][lane] = on ? v[c].y : T(0);
      }
      int pk = pl[0];  // lane c < kPanelW writes pivot c
      V rk = rec[0];
#pragma unroll
      for (int c = 1; c < kPanelW; c++) {
        pk = lane == c ? pl[c] : pk;
        rk.x = lane == c ? rec[c].x : rk.x;
        rk.y = lane == c ? rec[c].y : rk.y;
      }
      if (lane < kPanelW) {
        t.prow[c0 + lane] = pk;
        t.dinv[c0 + lane] = V{-rk.x, -rk.y};
      }
      __builtin_amdgcn_s_setprio(0);
    } else if (c0 > 0) {
      const int nb = c0 >> 4, b = w - 1;  // the block of this panel is up to date
      block_update(c0 - kPanelW, b + (b >= nb ? 1 : 0));
    }
    __syncthreads();  // W and the pivot rows are there; the other blocks are up to date
    const int nb = (c0 + kPanelW) >> 4;
    if (nb < 4) {
      const int col = 16 * nb + li, pk = t.prow[c0 + kq], row0 = 16 * w + 4 * kq;
      const bool on = (unsigned)(col - c0) >= kPanelW;
      V y;
      y.x = t.re[col][pk];
      y.y = t.im[col][pk];
      const V a = operand(c0, w);
      Acc4<T> re = get_rows<T>(&t.re[col][row0]), im = get_rows<T>(&t.im[col][row0]);
      __syncthreads();  // every wave has read the pivot rows
      update(re, im, a, y);
      if (on) {
        put_rows<T>(&t.re[col][row0], re);
        put_rows<T>(&t.im[col][row0], im);
      }
      __syncthreads();
    }
  }
  block_update(kTile - kPanelW, w);
  __syncthreads();
  // the rows into pivoted order, column by column (one wave's own columns)
  const int pr = t.prow[lane];
  {
    T re[kTile / 4], im[kTile / 4];
#pragma unroll
    for (int q = 0; q < kTile / 4; q++) {
      re[q] = t.re[w + 4 * q][pr];
      im[q] = t.im[w + 4 * q][pr];
    }
#pragma unroll
    for (int q = 0; q < kTile / 4; q++) t.put(w + 4 * q, lane, V{re[q], im[q]});
  }
  if (w == 0) {
    // zero pivots and the smallest pivot
    const V r = t.dinv[lane];
    const bool zero = r.x == T(0) && r.y == T(0);
    const int first = -wave_max_i32(zero ? -(lane + 1) : -(kTile + 1));
    double mn = zero ? 0.0 : 1.0 / sqrt((double)r.x * r.x + (double)r.y * r.y);
    for (int off = 32; off >= 1; off >>= 1) mn = fmin(mn, __shfl_xor(mn, off, 64));
    if (lane == 0) {
      t.minpiv = mn;
      t.info = first > kTile ? 0 : col_base + first;
    }
  }
  __syncthreads();
}

// The same for the tile at src, column stride ld.
template <class T>
__device__ __forceinline__ void tile_lu(TileLds<T> &t, const GCx<T> *src, long ld, int nd,
                                        int col_base) {
  tile_lu<T>(t, [=](int r, int c) { return ldg<T>(src + r + ld * c); }, nd, col_base);
}

}  // namespace lsmsx
