// tau_lu.hip -- batched blocked complex LU of KKR matrices on MI355X.
//
// Reference behaviour replaced: solveTau00zgetrf (linearSolvers_CPU.cpp:98-123:
// LU of M, solve [t0;0], keep the top kkrsz_ns rows) and the block-inverse
// route (zblock_lu_cpp.cpp:19-86 + tau_inv_postproc.f:33-57: eliminate the
// non-central blocks with pivoting inside diagonal blocks, then
// (1-delta)^-1 t0).  The matrix is in the solver layout (central site last,
// identity padding first) and the elimination is right-looking over 64-wide
// tiles with partial pivoting inside each 64x64 diagonal tile, the block-LU
// pivoting scheme of the reference's block-inverse solvers.
//
// Per step s (tile column c0 = 64 s), batched over all solves:
//   k_lu_diag    factor A_ss = P^T L U in LDS (tile_lu.hpp); store L^-1, U^-1 and P
//   k_lu_panel   L_is = A_is U^-1 (tiles below), U_sj = L^-1 P A_sj (right)
// with the steps taken in groups: the diagonal tile (k_lu_cross_diag) and the
// panel tiles (inside k_lu_panel) of a step first take the earlier steps of
// its group, and one trailing update per group, A_ij -= sum_k L_ik U_kj
// (k_lu_trail, MFMA, dominant), reads and writes the rest of the matrix once.
// The split-FP16 path has its own k_lu_diag_h, k_lu_panel_h and k_lu_strip_h,
// and k_lu_trail_h in update_f16.hip.  k_lu_last then factors the last tile
// with the pivots of its non-central
// rows and of the central rows kept apart.  In FP64 it also solves
// S tau00 = t0 with the Schur complement S (the plain path); in FP32 it
// stores the last tile's factors for the refinement solves (mixed path).
//
// All kernels are templated on the real type: double (complex FP64, MFMA
// v_mfma_f64_16x16x4f64) or float (complex FP32, v_mfma_f32_16x16x4f32).
#include "lu_common.hpp"
#include "tile_lu.hpp"

namespace lsmsx {

// threadIdx.x as a value the compiler does not carry over from elsewhere: a
// kernel that loops over panel tiles would otherwise keep every address and
// index of the loop body in registers across it (237 VGPRs, not 150).
__device__ __forceinline__ int fresh_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Stage a 64 x 64 tile (column stride ld) in LDS, S[col][row] =
// src[rowmap(row) + ld col]: the 16 loads of a thread are all issued before
// its first LDS write, so staging costs one memory round trip, not sixteen.
template <class T, class RM>
__device__ __forceinline__ void stage_tile(CxT<T> (*S)[kTile + 1], const GCx<T> *src, long ld,
                                           RM rowmap) {
  const int tid = fresh_tid(), r = tid & 63, c0 = tid >> 6;
  const int rr = rowmap(r);
  CxT<T> v[kTile / 4];
#pragma unroll
  for (int q = 0; q < kTile / 4; q++) v[q] = ldg<T>(src + rr + ld * (c0 + 4 * q));
#pragma unroll
  for (int q = 0; q < kTile / 4; q++) S[c0 + 4 * q][r] = v[q];
}

// Power-of-2 scale of a 64 x 64 tile for its split-FP16 planes, 256
// threads: ex with max |Re|, |Im| of get(rc, k) times 2^-ex below 2^14
// (inside the FP16 range with room for the lo part; 0 for a zero tile).
template <class F>
__device__ int plane_exponent(F get) {
  __shared__ float wmax[4];
  const int tid = fresh_tid(), w = tid >> 6, lane = tid & 63;
  __syncthreads();  // the values were written by all four waves
  float m = 0.f;
  for (int e = tid; e < kTile * kTile; e += 256) {
    const float2 v = get(e >> 6, e & 63);
    m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)));
  }
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if (lane == 0) wmax[w] = m;
  __syncthreads();
  m = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  int ex = 0;
  if (m > 0.f) {
    frexpf(m, &ex);  // m < 2^ex
    ex -= 14;
  }
  return ex;
}

// Eight complex values x 2^-ex (Re times sgn) split into hi/lo FP16 planes:
// x 2^-ex = hi + lo to 22 bits.
__device__ __forceinline__ void split8(const float2 (&v)[8], float sgn, float sc, h8 &rh, h8 &rl,
                                       h8 &ih, h8 &il) {
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const float re = sgn * v[u].x * sc, im = v[u].y * sc;
    const _Float16 a = (_Float16)re, b = (_Float16)im;
    rh[u] = a;
    rl[u] = (_Float16)(re - (float)a);
    ih[u] = b;
    il[u] = (_Float16)(im - (float)b);
  }
}

// Split the 64 x 64 values get(rc, k) (256 threads) into hi/lo FP16 planes
// with one power-of-2 scale (plane_exponent) for the split-FP16 products.
// Layout, k fastest:
//   L tile (rc = row i, k = tile column):  planes -Re, -Re lo, Im, Im lo ([i][k]);
//   U tile (k = tile row, rc = column j):  planes  Re,  Re lo, Im, Im lo ([j][k]).
// The L planes carry the sign of the update C -= L U.
template <class F>
__device__ void write_planes(F get, bool lower, _Float16 *out, int *eout) {
  const int tid = fresh_tid();
  const int ex = plane_exponent(get);
  if (tid == 0) *eout = ex;
  const float sc = ldexpf(1.f, -ex);
  const float sgn = lower ? -1.f : 1.f;
  for (int q = tid; q < kTile * 8; q += 256) {
    const int rc = q >> 3, kg = q & 7;  // row i (L) or column j (U); k group
    float2 v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = get(rc, 8 * kg + u);
    h8 rh, rl, ih, il;
    split8(v, sgn, sc, rh, rl, ih, il);
    h8 *o = (h8 *)(out + rc * kTile + 8 * kg);
    o[0] = rh;
    o[(kTile * kTile) / 8] = rl;
    o[2 * (kTile * kTile) / 8] = ih;
    o[3 * (kTile * kTile) / 8] = il;
  }
}

// The planes of an FP32 panel tile held in LDS as Ts[col][row].
__device__ __forceinline__ void write_split_planes(float2 (*Ts)[kTile + 1], bool lower,
                                                   _Float16 *out, int *eout) {
  if (lower)
    write_planes([&](int i, int k) { return Ts[k][i]; }, true, out, eout);
  else
    write_planes([&](int j, int k) { return Ts[j][k]; }, false, out, eout);
}

// ---------------------------------------------------------------------------
// The factors of a tile, as tile_lu and tile_invert_upper left them in t, to
// the solve: L^-1 (strict lower) and U^-1 (upper incl. diagonal) packed in one
// tile, the permutation and the pivot status; on the split path also the
// planes of both for the fused panel's FP16 products.  256 threads.
template <class T>
__device__ __forceinline__ void store_tile(TileLds<T> &t, const SolveDesc &d, int step) {
  typedef CxT<T> V;
  const int tid = threadIdx.x;
  if (tid < kTile) d.perm[step * kTile + tid] = t.prow[tid];
  if (tid == 0) {
    if (t.info != 0 && *d.info == 0) *d.info = t.info;
    if (t.minpiv < *d.minpiv) *d.minpiv = t.minpiv;
  }
  GCx<T> *inv = (GCx<T> *)d.inv + step * d.inv_stride;
#pragma unroll
  for (int q = 0; q < kTile / 4; q++) {
    const int r = tid & 63, c = (tid >> 6) + 4 * q;
    inv[r + kTile * c] = t.get(c, r);
  }
  if constexpr (sizeof(T) == 4) {
    if (d.ihp) {
      // L^-1 (unit lower, L layout) and U^-1 (U layout), in the step's slot
      const int slot = step % d.group;
      _Float16 *ip = (_Float16 *)d.ihp + slot * (2 * kPlaneHalves);
      int *ie = d.ihe + 2 * slot;
      write_planes(
          [&](int i, int k) {
            V v = t.get(k, i);
            v.x = i > k ? v.x : (i == k ? 1.f : 0.f);
            v.y = i > k ? v.y : 0.f;
            return v;
          },
          true, ip, ie);
      write_planes([&](int j, int k) { return upper_at<T>(t, k, j); }, false, ip + kPlaneHalves,
                   ie + 1);
    }
  }
}

// ---------------------------------------------------------------------------
// Diagonal tile of step s: L^-1, U^-1 and the permutation (the factors
// themselves are not needed again).  One tile takes 36 us in FP64 and
// 33 us in FP32 alone on the chip; the LU in LDS with a rank-1 update and
// workgroup barriers per column, and the inverses column by column, that it
// replaces took 200 and 189 us, which was most of a single solve (N = 2160: 33
// of them one after another).
template <class T>
__global__ __launch_bounds__(256) void k_lu_diag(const SolveDesc *__restrict__ descs, int step) {
  const SolveDesc &d = descs[blockIdx.x];
  const bool last = step == kLastStep;  // each solve's own last tile (full LU)
  step = last ? d.nt - 1 : step - d.step0;
  if (step < 0 || (!last && step >= d.nt - 1)) return;
  if (d.conv && *d.conv) return;
  __shared__ TileLds<T> t;
  tile_lu<T>(t, tile_ptr<T>(d, step, step), tile_ld(d), kTile, step * kTile);
  tile_invert_upper<T>(t);
  store_tile<T>(t, d, step);
}

// Cross update of tile (ti, tj) inside the split-FP16 panel, C = A - sum over
// the steps s_first .. s_first+ns-1 of L(ti, s) U(s, tj), written to
// Ts[col][rowpos[row]] (rowpos null: the identity).  The products run on the
// split planes of those steps (slot s mod group) with the FP16 MFMAs of the
// trailing update, in its orientation (a-operand a U plane, lane l: column
// l%16; b-operand an L plane, lane l: row l%16; k = 8(l/16)..+7 of a 32-wide
// chunk; register r of lane l is C(row l%16, column 4(l/16) + r)) and its
// 4M x 3 split products, FP32 accumulators that start from zero and are
// rescaled between the steps by the tile exponents (exact powers of two).
// Wave w takes rows wr.., columns wc.. (32 x 32).  Per chunk the L and U
// planes (16 KiB each) are staged in Ts's memory with the XOR-swizzled k
// groups, the next chunk's loads in flight during this chunk's MFMAs (eight
// 16-byte loads per thread).  A (the tile's FP32 values) is read during the
// last chunk and added at the end.
__device__ __forceinline__ void cross_to_lds(const SolveDesc &d, int ti, int tj, int s_first,
                                             int ns, const GCx<float> *A, long ld,
                                             float2 (*Ts)[kTile + 1], const int *rowpos) {
  __shared__ int exs[16];
  const int tid = fresh_tid(), w = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wr = 32 * (w & 1), wc = 32 * (w >> 1);
  const int nt = d.nt, gmask = d.group - 1;
  const _Float16 *hp = (const _Float16 *)d.hp;
  h8(*Ls)[kTile][4] = reinterpret_cast<h8(*)[kTile][4]>(&Ts[0][0]);  // [plane][row][k group]
  h8(*Us)[kTile][4] = Ls + 4;                                          // [plane][column][k group]
  if (tid < ns) {
    const int par = (s_first + tid) & gmask;
    exs[tid] = d.he[(par * 2 + 0) * nt + ti] + d.he[(par * 2 + 1) * nt + tj];
  }
  __syncthreads();
  // chunk ch = (step ch / 2, k half ch % 2); load q of a thread: side (L, U),
  // plane, row (column), k group
  auto src = [&](int ch, int q) __attribute__((always_inline)) -> GH8 * {
    const int s = s_first + (ch >> 1), kh = ch & 1, par = s & gmask;
    const int e8 = tid + 256 * q, side = e8 >> 10, plane = (e8 >> 8) & 3, rr = (e8 >> 2) & 63,
              grp = e8 & 3;
    return (GH8 *)(hp + (long)((par * 2 + side) * nt + (side ? tj : ti)) * kPlaneHalves) +
           ((plane * kTile + rr) * kTile + 32 * kh + 8 * grp) / 8;
  };
  auto dst = [&](int q) __attribute__((always_inline)) -> h8 * {
    const int e8 = tid + 256 * q, side = e8 >> 10, plane = (e8 >> 8) & 3, rr = (e8 >> 2) & 63,
              grp = e8 & 3;
    return &(side ? Us : Ls)[plane][rr][swz_group(rr, grp)];
  };
  f4 cr[2][2], ci[2][2];
#pragma unroll
  for (int bi = 0; bi < 2; bi++)
#pragma unroll
    for (int bj = 0; bj < 2; bj++) {
      cr[bi][bj] = f4{0.f, 0.f, 0.f, 0.f};
      ci[bi][bj] = cr[bi][bj];
    }
  int e = exs[0];
  auto rescale = [&](int ch) __attribute__((always_inline)) {
    if (ch > 0 && !(ch & 1)) {
      const int e2 = exs[ch >> 1];
      if (e2 == e) return;
      const float sc1 = ldexpf(1.f, e - e2);
#pragma unroll
      for (int bi = 0; bi < 2; bi++)
#pragma unroll
        for (int bj = 0; bj < 2; bj++) {
          cr[bi][bj] *= sc1;
          ci[bi][bj] *= sc1;
        }
      e = e2;
    }
  };
  // Cr += (-Lr) Ur + Li Ui, Ci += (-Lr) Ui + Li (-Ur): the L planes hold -Re
  auto compute = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int bj = 0; bj < 2; bj++) {
      const int col = wc + 16 * bj + l16, gu = swz_group(col, g);
      const h8 ur_h = Us[0][col][gu], ur_l = Us[1][col][gu];
      const h8 ui_h = Us[2][col][gu], ui_l = Us[3][col][gu];
      const h8 nur_h = neg8(ur_h), nur_l = neg8(ur_l);
#pragma unroll
      for (int bi = 0; bi < 2; bi++) {
        const int row = wr + 16 * bi + l16, gl = swz_group(row, g);
        const h8 nar_h = Ls[0][row][gl], nar_l = Ls[1][row][gl];
        const h8 ai_h = Ls[2][row][gl], ai_l = Ls[3][row][gl];
        f4 r = cr[bi][bj], m = ci[bi][bj];
        r = mfma_h(ur_h, nar_h, r);
        r = mfma_h(ur_l, nar_h, r);
        r = mfma_h(ur_h, nar_l, r);
        r = mfma_h(ui_h, ai_h, r);
        r = mfma_h(ui_l, ai_h, r);
        r = mfma_h(ui_h, ai_l, r);
        m = mfma_h(ui_h, nar_h, m);
        m = mfma_h(ui_l, nar_h, m);
        m = mfma_h(ui_h, nar_l, m);
        m = mfma_h(nur_h, ai_h, m);
        m = mfma_h(nur_l, ai_h, m);
        m = mfma_h(nur_h, ai_l, m);
        cr[bi][bj] = r;
        ci[bi][bj] = m;
      }
    }
  };
  const int nch = 2 * ns;
  h8 pv[8];
#pragma unroll
  for (int q = 0; q < 8; q++) pv[q] = *src(0, q);
#pragma unroll 1
  for (int ch = 0; ch < nch - 1; ch++) {
    rescale(ch);
    __syncthreads();  // the previous chunk's readers are done
#pragma unroll
    for (int q = 0; q < 8; q++) *dst(q) = pv[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; q++) pv[q] = *src(ch + 1, q);
    compute();
  }
  // the last chunk, with A's loads in the prefetch registers' place:
  // A(wr + 16 bi + l16, wc + 16 bj + 4 g + r)
  rescale(nch - 1);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 8; q++) *dst(q) = pv[q];
  __syncthreads();
  float2 av[2][2][4];
#pragma unroll
  for (int bi = 0; bi < 2; bi++)
#pragma unroll
    for (int bj = 0; bj < 2; bj++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        av[bi][bj][r] = ldg<float>(A + (wr + 16 * bi + l16) + ld * (wc + 16 * bj + 4 * g + r));
  compute();
  __syncthreads();  // every wave is done reading the staged planes
  const float sc2 = ldexpf(1.f, e);
#pragma unroll
  for (int bi = 0; bi < 2; bi++)
#pragma unroll
    for (int bj = 0; bj < 2; bj++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = wr + 16 * bi + l16, col = wc + 16 * bj + 4 * g + r;
        Ts[col][rowpos ? rowpos[row] : row] =
            make_float2(av[bi][bj][r].x + cr[bi][bj][r] * sc2, av[bi][bj][r].y + ci[bi][bj][r] * sc2);
      }
}

// Diagonal tile of step s on the split-FP16 path, after its cross update with
// the ncross (> 0) steps before s in its group, on the way into the
// factorization: a few microseconds of FP16 MFMAs, where a launch of its own
// took 14 (32 solves) to 21 (248).
__global__ __launch_bounds__(256) void k_lu_diag_h(const SolveDesc *__restrict__ descs, int step,
                                                   int ncross) {
  const SolveDesc &d = descs[blockIdx.x];
  const int s = step - d.step0;
  if (s - ncross < 0 || s >= d.nt - 1) return;
  if (d.conv && *d.conv) return;
  __shared__ TileLds<float> t;
  __shared__ __align__(16) float2 Ts[kTile][kTile + 1];
  cross_to_lds(d, s, s, s - ncross, ncross, tile_ptr<float>(d, s, s), tile_ld(d), Ts, nullptr);
  __syncthreads();
  tile_lu<float>(t, [&](int r, int c) { return Ts[c][r]; }, kTile, s * kTile);
  tile_invert_upper<float>(t);
  store_tile<float>(t, d, s);
}

// Panel tile t of step s on the split-FP16 path: lower -> L_ts = A_ts U^-1 ;
// else U_st = L^-1 P A_st.  The operand tile is staged in LDS (rows gathered
// by the pivot permutation for U_st) before it is overwritten in place, and
// takes the cross update with the ncross steps before s in its group on the
// way (cross_to_lds).
__device__ __forceinline__ void panel_tile_h(const SolveDesc &d, int step, int ncross, bool lower,
                                             int t) {
  typedef float2 V;
  __shared__ __align__(16) V Ts[kTile][kTile + 1];  // Ts[col][row]
  const int tid = fresh_tid(), w = tid >> 6;
  const int lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int wr = 32 * (w & 1), wc = 32 * (w >> 1);
  const long ld = tile_ld(d);
  const int ti = lower ? t : step, tj = lower ? step : t;
  GCx<float> *tile = tile_ptr<float>(d, ti, tj);
  if (ncross > 0) {
    // the row of C that lands at LDS row r is perm[r] (U_sj): rowpos = perm^-1
    __shared__ int rowpos[kTile];
    if (!lower && tid < kTile) rowpos[d.perm[step * kTile + tid]] = tid;
    cross_to_lds(d, ti, tj, step - ncross, ncross, tile, ld, Ts, lower ? nullptr : rowpos);
  } else {
    if (lower) {
      stage_tile<float>(Ts, tile, ld, [](int r) { return r; });
    } else {
      const int *perm = d.perm + step * kTile;
      stage_tile<float>(Ts, tile, ld, [&](int r) { return perm[r]; });
    }
  }
  __syncthreads();
  V ov[2][2][4];  // output (row wr + 16 bi + li, column wc + 16 bj + acc_row(kq, r))
  // split-FP16 product with the diagonal tile's inverse planes (written by
  // k_lu_diag): the tile's side is split here with its own scale, the
  // accumulators take -(A B) as in the cross update (b-operand rows with
  // -Re, a-operand columns with +Re), two 32-wide k chunks
  const int eC = plane_exponent([&](int a, int b) { return Ts[a][b]; });
  const float sc = ldexpf(1.f, -eC);
  const int g = kq, l16 = li;
  const int slot = step % d.group;
  GH8 *ip = (GH8 *)((const _Float16 *)d.ihp + slot * (2 * kPlaneHalves) + (lower ? kPlaneHalves : 0));
  const int eI = d.ihe[2 * slot + (lower ? 1 : 0)];
  f4 cr[2][2], ci[2][2];
#pragma unroll
  for (int bi = 0; bi < 2; bi++)
#pragma unroll
    for (int bj = 0; bj < 2; bj++) {
      cr[bi][bj] = f4{0.f, 0.f, 0.f, 0.f};
      ci[bi][bj] = cr[bi][bj];
    }
#pragma unroll 1
  for (int kh = 0; kh < 2; kh++) {
    // b-operands (rows wr + 16 bi ..): L_is = C U^-1 takes the rows of C
    // from Ts[k][i], U_sj = L^-1 (P C) the rows of L^-1 from its planes
    h8 lo[2][4];
#pragma unroll
    for (int bi = 0; bi < 2; bi++) {
      if (lower) {
        float2 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = Ts[32 * kh + 8 * g + u][wr + 16 * bi + l16];
        split8(v, -1.f, sc, lo[bi][0], lo[bi][1], lo[bi][2], lo[bi][3]);
      } else {
#pragma unroll
        for (int p = 0; p < 4; p++)
          lo[bi][p] = ip[((p * kTile + wr + 16 * bi + l16) * kTile + 32 * kh + 8 * g) / 8];
      }
    }
#pragma unroll
    for (int bj = 0; bj < 2; bj++) {
      // a-operand (columns wc + 16 bj ..): U^-1 from its planes, or P C from Ts[j][k]
      h8 uo[4];
      if (lower) {
#pragma unroll
        for (int p = 0; p < 4; p++)
          uo[p] = ip[((p * kTile + wc + 16 * bj + l16) * kTile + 32 * kh + 8 * g) / 8];
      } else {
        float2 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = Ts[wc + 16 * bj + l16][32 * kh + 8 * g + u];
        split8(v, 1.f, sc, uo[0], uo[1], uo[2], uo[3]);
      }
      const h8 nur_h = neg8(uo[0]), nur_l = neg8(uo[1]);
#pragma unroll
      for (int bi = 0; bi < 2; bi++) {
        f4 r = cr[bi][bj], m = ci[bi][bj];
        r = mfma_h(uo[0], lo[bi][0], r);
        r = mfma_h(uo[1], lo[bi][0], r);
        r = mfma_h(uo[0], lo[bi][1], r);
        r = mfma_h(uo[2], lo[bi][2], r);
        r = mfma_h(uo[3], lo[bi][2], r);
        r = mfma_h(uo[2], lo[bi][3], r);
        m = mfma_h(uo[2], lo[bi][0], m);
        m = mfma_h(uo[3], lo[bi][0], m);
        m = mfma_h(uo[2], lo[bi][1], m);
        m = mfma_h(nur_h, lo[bi][2], m);
        m = mfma_h(nur_l, lo[bi][2], m);
        m = mfma_h(nur_h, lo[bi][3], m);
        cr[bi][bj] = r;
        ci[bi][bj] = m;
      }
    }
  }
  const float so = -ldexpf(1.f, eC + eI);
#pragma unroll
  for (int bj = 0; bj < 2; bj++)
#pragma unroll
    for (int bi = 0; bi < 2; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) ov[bj][bi][r] = make_float2(cr[bi][bj][r] * so, ci[bi][bj][r] * so);
  GCx<float> *C = tile + wr + ld * wc;
  __syncthreads();  // every wave is done reading Ts
#pragma unroll
  for (int bj = 0; bj < 2; bj++)
#pragma unroll
    for (int bi = 0; bi < 2; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const V o = ov[bj][bi][r];
        // the FP32 factor tile is read again only by the refinement sweeps
        // after the whole factorization: non-temporal
        typedef float pv2 __attribute__((ext_vector_type(2)));
        __builtin_nontemporal_store(pv2{o.x, o.y},
                                    (pv2 *)&C[(16 * bi + li) + ld * (16 * bj + acc_row<float>(kq, r))]);
        Ts[wc + 16 * bj + acc_row<float>(kq, r)][wr + 16 * bi + li] = o;
      }
  // split-FP16 planes of this panel tile for the split updates
  const int side = lower ? 0 : 1;
  write_split_planes(Ts, lower, (_Float16 *)d.hp + (long)((slot * 2 + side) * d.nt + t) * kPlaneHalves,
                     d.he + (slot * 2 + side) * d.nt + t);
}

// Panel of step `step` with its cross update (panel_op): L_is = C' U^-1 for the
// tiles below the diagonal tile, U_sj = L^-1 P C' for those right of it, where
// C' has taken the ncross steps before s in its group.  N = 1: four
// workgroups a tile (lu_small_grid chooses).  Bound by the MFMAs of the group's
// steps and by the load latencies of a tile's two products (64 solves N = 2160
// in FP64: MFMAs busy 57% of 5.7 ms).
template <class T, int N>
__global__ __launch_bounds__(256) void k_lu_panel(const SolveDesc *__restrict__ descs, int step,
                                                  int ncross, int xcd_swizzle) {
  int bx = blockIdx.x, by = blockIdx.y;
  if (xcd_swizzle) xcd_remap(bx, by);
  const SolveDesc &d = descs[by];
  step -= d.step0;
  constexpr int np = N == 2 ? 1 : 4;
  const int nrest = d.nt - 1 - step, x = bx / np, piece = bx % np;
  if (step < 0 || nrest <= 0 || x >= 2 * nrest) return;
  if (d.conv && *d.conv) return;
  const long ld = tile_ld(d);
  const GCx<T> *inv = (const GCx<T> *)d.inv + step * d.inv_stride;
  const LSMSX_GLOBAL int *perm = (const LSMSX_GLOBAL int *)d.perm + step * kTile;
  const bool lower = x < nrest;
  const int ti = lower ? step + 1 + x : step, tj = lower ? step : step + 1 + x - nrest;
  const int g = step - ncross;
  const GCx<T> *A = tile_ptr<T>(d, ti, g), *B = tile_ptr<T>(d, g, tj);
  const long sa = tile_ptr<T>(d, ti, g + 1) - A, sb = tile_ptr<T>(d, g + 1, tj) - B;
  GCx<T> *C = tile_ptr<T>(d, ti, tj);
  __shared__ PanelLds<T, N> lds;
  if (lower)
    panel_op<T, N, kRightU>(C, true, false, A, sa, B, sb, ld, ncross, inv, perm, piece, lds);
  else
    panel_op<T, N, kLeftL>(C, true, false, A, sa, B, sb, ld, ncross, inv, perm, piece, lds);
}

// Panels of a group on the split-FP16 path.  k_lu_panel_h takes the tiles of
// one step: all of its column and row, or in large launches of solves of one
// size (launch_lu_steps)
// those inside the group's diagonal block alone (rows and columns up to its
// last step), which the next diagonal tiles wait for; then each tile row below
// the block, and each tile column right of it, runs through all the group's
// steps in one workgroup (k_lu_strip_h).  Both read a tile's planes of every
// earlier step of the group again, from HBM mostly; a strip shares the block's
// planes with the others at the same step through L2, and saves the launches'
// ends (248 solves N = 2160: 14.7 -> 13.4 ms a pass for the panels).
// With xcd_swizzle the workgroups of one solve run on one XCD, so that the planes
// they share are fetched into one L2.

// the last step of the group starting at solve step g
__device__ __forceinline__ int group_last(const SolveDesc &d, int g) {
  return min(g + d.group, d.nt - 1) - 1;
}

__global__ __launch_bounds__(256) void k_lu_panel_h(const SolveDesc *__restrict__ descs, int step,
                                                    int ncross, int whole, int xcd_swizzle) {
  int bx = blockIdx.x, by = blockIdx.y;
  if (xcd_swizzle) xcd_remap(bx, by);
  const SolveDesc &d = descs[by];
  const int s = step - d.step0;
  if (s - ncross < 0) return;
  const int n = (whole ? d.nt - 1 : group_last(d, s - ncross)) - s;
  if (bx >= 2 * n) return;
  if (d.conv && *d.conv) return;
  panel_tile_h(d, s, ncross, bx < n, s + 1 + (bx < n ? bx : bx - n));
}

__global__ __launch_bounds__(256, 3) void k_lu_strip_h(const SolveDesc *__restrict__ descs, int step,
                                                       int xcd_swizzle) {
  int bx = blockIdx.x, by = blockIdx.y;
  if (xcd_swizzle) xcd_remap(bx, by);
  const SolveDesc &d = descs[by];
  const int g = step - d.step0;
  if (g < 0) return;
  const int last = group_last(d, g), n = d.nt - 1 - last;
  if (last < g || bx >= 2 * n) return;
  if (d.conv && *d.conv) return;
  const bool lower = bx < n;
  const int t = last + 1 + (lower ? bx : bx - n);
#pragma unroll 1
  for (int s = g; s <= last; s++) {
    if (s > g) __syncthreads();  // the planes of step s-1 are written, Ts is read
    panel_tile_h(d, s, s - g, lower, t);
  }
}

// C(ti, tj) -= sum_{u < ns} L(ti, s0+u) U(s0+u, tj): one 64x64 tile per
// workgroup, a 32x32 quarter per wave (N = 2), or one 32x32 quarter per
// workgroup, a 16x16 block per wave (N = 1, `piece` = the quarter).
template <class T, int N>
__device__ __forceinline__ void update_tile(const SolveDesc &d, int ti, int tj, int s0, int ns,
                                            int piece) {
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = N == 2 ? 32 * (w & 1) : 32 * (piece & 1) + 16 * (w & 1);
  const int wc = N == 2 ? 32 * (w >> 1) : 32 * (piece >> 1) + 16 * (w >> 1);
  const long ld = tile_ld(d);
  GCx<T> *__restrict__ C = tile_ptr<T>(d, ti, tj) + wr + ld * wc;
  typedef T cv2 __attribute__((ext_vector_type(2)));
  Acc3<T, N> q;
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        // C is read and written once per group: non-temporal, so that the
        // panels the other tiles read stay in L2
        const cv2 c = __builtin_nontemporal_load(
            (const cv2 *)&C[(16 * bi + li) + ld * (16 * bj + acc_row<T>(kq, r))]);
        set_minus<T, N>(q, bj, bi, r, c.x, c.y);
      }
  const GCx<T> *A = tile_ptr<T>(d, ti, s0), *B = tile_ptr<T>(d, s0, tj);
  const long sa = tile_ptr<T>(d, ti, s0 + 1) - A, sb = tile_ptr<T>(d, s0 + 1, tj) - B;
  __shared__ ProductStage<T, N> st;
  tile_products<T, N>(A + wr, sa, B + ld * wc, sb, ld, ns, q, st);
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const CxT<T> v = minus_value<T, N>(q, bj, bi, r);
        __builtin_nontemporal_store(cv2{v.x, v.y},
                                    (cv2 *)&C[(16 * bi + li) + ld * (16 * bj + acc_row<T>(kq, r))]);
      }
}

// Grouped elimination: the steps g .. g+ns-1 of a group (ns = min(group,
// nt-1-g); step nt-1 is k_lu_last) are factored one after another, the
// diagonal tile and the panel of each first taking the group's earlier steps;
// then one trailing update applies all ns steps to the tiles beyond the group.
// Number of steps of the group starting at solve step g.
__device__ __forceinline__ int group_steps(const SolveDesc &d, int g) {
  return min(d.group, d.nt - 1 - g);
}

// Cross update of the diagonal tile of step t = g + U of the group starting at
// global step s with the steps g .. t-1 (the panel tiles take theirs in
// k_lu_panel): a 16x16 block per workgroup, a quarter of each step's k per
// wave, summed through LDS.  It lies between two diagonal tiles, and its
// latency counts: all operands are loaded at once, and the product's chain is
// 12 U FP64 MFMAs (with a quarter tile per workgroup and a 16x16 block per wave
// 48 U; one solve N = 2160: 7.0 -> 4.6 us a launch, of which most is the
// launch; 992 at once, at the rate of HBM: 105 -> 125 us, 0.1% of their step).
// B goes through LDS as in wave_gemm3m_staged.
template <class T, int U>
__global__ __launch_bounds__(256) void k_lu_cross_diag(const SolveDesc *__restrict__ descs,
                                                       int step) {
  typedef CxT<T> V;
  const SolveDesc &d = descs[blockIdx.y];
  const int g = step - d.step0, t = g + U;
  if (g < 0 || U >= group_steps(d, g)) return;
  if (d.conv && *d.conv) return;
  __shared__ __align__(16) V st[4][U][16][17];  // [wave][step][column][k], then [column][row]
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = 16 * (blockIdx.x & 3), c0 = 16 * (blockIdx.x >> 2);
  const long ld = tile_ld(d);
  GCx<T> *C = tile_ptr<T>(d, t, t) + (r0 + (tid & 15)) + ld * (c0 + (tid >> 4));
  V a[U][4], b[U][4];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const GCx<T> *A = tile_ptr<T>(d, t, g + u) + (r0 + li) + ld * (16 * w + kq);
    const GCx<T> *B = tile_ptr<T>(d, g + u, t) + (16 * w + li) + ld * (c0 + kq);
#pragma unroll
    for (int m = 0; m < 4; m++) b[u][m] = ldg<T>(B + 4 * m * ld);
#pragma unroll
    for (int m = 0; m < 4; m++) a[u][m] = ldg<T>(A + 4 * m * ld);
  }
  V c = ldg<T>(C);
#pragma unroll
  for (int u = 0; u < U; u++)
#pragma unroll
    for (int m = 0; m < 4; m++) st[w][u][kq + 4 * m][li] = b[u][m];
  wave_lds_fence();
  Acc3<T, 1> q;
  zero_acc(q);
#pragma unroll
  for (int u = 0; u < U; u++)
#pragma unroll
    for (int m = 0; m < 4; m++) {
      V av[1] = {a[u][m]}, bv[1] = {st[w][u][li][4 * m + kq]};
      gemm3m_step<T, 1>(av, bv, q);
    }
  wave_lds_fence();
#pragma unroll
  for (int r = 0; r < 4; r++) st[w][0][acc_row<T>(kq, r)][li] = minus_value<T, 1>(q, 0, 0, r);
  __syncthreads();
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const V p = st[v][0][tid >> 4][tid & 15];
    c.x += p.x;
    c.y += p.y;
  }
  *C = c;
}

// Trailing update of the group starting at global step s: A_ij -= sum over
// the group's steps k of L_ik U_kj for all i, j beyond the group, one pass
// over C with K = 64 ns.  64 solves N = 2160 in FP64: 18.2 ms with the MFMAs
// busy 85% (22.4 ms and 75% with groups of two steps).
template <class T, int N>
__global__ __launch_bounds__(256) void k_lu_trail(const SolveDesc *__restrict__ descs, int step,
                                                  int xcd_swizzle) {
  int bx = blockIdx.x, by = blockIdx.y;
  if (xcd_swizzle) xcd_remap(bx, by);
  const SolveDesc &d = descs[by];
  const int g = step - d.step0;
  if (g < 0) return;
  const int ns = group_steps(d, g);
  if (ns <= 0) return;
  if (d.conv && *d.conv) return;
  constexpr int np = N == 2 ? 1 : 4;
  const int last = g + ns - 1, nrest = d.nt - 1 - last, x = bx / np;
  if (x >= nrest * nrest) return;
  update_tile<T, N>(d, last + 1 + x % nrest, last + 1 + x / nrest, g, ns, bx % np);
}

// Last tile (step nt-1): factor it with the non-central rows (first nd =
// 64 - kc) pivoting among themselves and the central rows among themselves.
// The trailing kc x kc block becomes LU(S), S the Schur complement.
//   plain FP64 path: solve S tau00 = t0 from the S factors;
//   refined paths (d.X set; FP32 mixed or FP64 refined): store the tile's
//   inverses and permutation like k_lu_diag, for the refinement.
template <class T>
__global__ __launch_bounds__(256) void k_lu_last(const SolveDesc *__restrict__ descs) {
  typedef CxT<T> V;
  const SolveDesc &d = descs[blockIdx.x];
  if (d.conv && *d.conv) return;
  __shared__ TileLds<T> t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int step = d.nt - 1, kc = d.kc, nd = kTile - kc;
  tile_lu<T>(t, tile_ptr<T>(d, step, step), tile_ld(d), nd, step * kTile);
  if (d.X != nullptr) {  // refinement follows
    tile_invert_upper<T>(t);
    store_tile<T>(t, d, step);
    return;
  }
  if (tid == 0) {
    if (t.info != 0 && *d.info == 0) *d.info = t.info;
    if (t.minpiv < *d.minpiv) *d.minpiv = t.minpiv;
  }
  // one lane per row of the tile and four right-hand sides per wave at a time
  // in registers: y = L_S^-1 P_S t0, then U_S x = y column by column, the row
  // just finished broadcast by readlane (a zero diagonal of U counts as 1)
  constexpr int kRhs = 4;
  const int row = t.prow[lane] - nd;  // row of t0 in this position (central rows only)
  V ur = t.dinv[lane];
  if (ur.x == T(0) && ur.y == T(0)) ur.x = T(1);
  for (int c0 = 0; c0 < kc; c0 += 4 * kRhs) {
    V b[kRhs], y[kRhs];
#pragma unroll
    for (int q = 0; q < kRhs; q++) {
      const int c = c0 + w + 4 * q;
      b[q] = czero<V>();
      if (lane >= nd && c < kc) {
        const double2 v = d.t0[row + (long)d.ldt * c];
        b[q].x = v.x;
        b[q].y = v.y;
      }
      y[q] = b[q];
    }
    for (int j = nd; j < kTile - 1; j++) {
      V l = t.get(j, lane);
      l.x = lane > j ? l.x : T(0);
      l.y = lane > j ? l.y : T(0);
#pragma unroll
      for (int q = 0; q < kRhs; q++) y[q] = cadd_mul(y[q], l, lane_value2(b[q], j));
    }
    for (int j = kTile - 1; j >= nd; j--) {
      V u = t.get(j, lane);
      u.x = lane < j ? u.x : T(0);
      u.y = lane < j ? u.y : T(0);
      const V r = lane_value2(ur, j);
#pragma unroll
      for (int q = 0; q < kRhs; q++) {
        const V xj = cmul2(lane_value2(y[q], j), r);
        y[q] = csub_mul(y[q], u, xj);
        if (lane == j) y[q] = xj;
      }
    }
#pragma unroll
    for (int q = 0; q < kRhs; q++) {
      const int c = c0 + w + 4 * q;
      if (lane >= nd && c < kc) d.tau00[(lane - nd) + kc * c] = make_double2(y[q].x, y[q].y);
    }
  }
}

template __global__ void k_lu_diag<double>(const SolveDesc *, int);
template __global__ void k_lu_diag<float>(const SolveDesc *, int);
template __global__ void k_lu_panel<double, 2>(const SolveDesc *, int, int, int);
template __global__ void k_lu_panel<double, 1>(const SolveDesc *, int, int, int);
template __global__ void k_lu_panel<float, 2>(const SolveDesc *, int, int, int);
template __global__ void k_lu_panel<float, 1>(const SolveDesc *, int, int, int);
template __global__ void k_lu_cross_diag<double, 1>(const SolveDesc *, int);
template __global__ void k_lu_cross_diag<double, 2>(const SolveDesc *, int);
template __global__ void k_lu_cross_diag<double, 3>(const SolveDesc *, int);
template __global__ void k_lu_cross_diag<float, 1>(const SolveDesc *, int);
template __global__ void k_lu_cross_diag<float, 2>(const SolveDesc *, int);
template __global__ void k_lu_cross_diag<float, 3>(const SolveDesc *, int);
template __global__ void k_lu_trail<double, 2>(const SolveDesc *, int, int);
template __global__ void k_lu_trail<double, 1>(const SolveDesc *, int, int);
template __global__ void k_lu_trail<float, 2>(const SolveDesc *, int, int);
template __global__ void k_lu_trail<float, 1>(const SolveDesc *, int, int);
template __global__ void k_lu_last<double>(const SolveDesc *);
template __global__ void k_lu_last<float>(const SolveDesc *);

}  // namespace lsmsx
