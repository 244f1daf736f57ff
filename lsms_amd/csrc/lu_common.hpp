// lu_common.hpp -- device helpers shared by the LU, refinement and inverse
// kernels: complex types per real type, global-address-space pointers, the
// 16x16x4 MFMA wrappers with their accumulator layout, and the 3M complex
// wave product used by every trailing update.
#pragma once
#include <type_traits>

#include "lsmsx_device.hpp"

namespace lsmsx {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <class T>
struct Cplx;
template <>
struct Cplx<double> {
  typedef double2 type;
  typedef d4 acc;
};
template <>
struct Cplx<float> {
  typedef float2 type;
  typedef f4 acc;
};
template <class T>
using CxT = typename Cplx<T>::type;
template <class T>
using Acc4 = typename Cplx<T>::acc;

// Pointers read from the solve descriptors are generic; casting them to the
// global address space lets the compiler emit global (not flat) loads/stores.
// (The host pass only type-checks kernel bodies, so it sees plain types.)
#if defined(__HIP_DEVICE_COMPILE__)
#define LSMSX_GLOBAL __attribute__((address_space(1)))
#else
#define LSMSX_GLOBAL
#endif
template <class T>
using GCx = LSMSX_GLOBAL CxT<T>;

// Load of one complex value from global memory, field by field.  A struct
// copy out of a global-address-space pointer into an array element becomes a
// memcpy that keeps the array in scratch memory; two scalar loads (merged
// into one wide load) keep it in registers.
template <class T>
__device__ __forceinline__ CxT<T> ldg(const GCx<T> *p) {
  CxT<T> v;
  v.x = p->x;
  v.y = p->y;
  return v;
}

__device__ __forceinline__ d4 mfma4(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// Accumulator layout of the 16x16x4 MFMAs (measured on gfx950): register r
// of lane l holds output row l/16 + 4r (f64) or 4(l/16) + r (f32), column l%16.
template <class T>
__device__ __forceinline__ int acc_row(int kq, int r);
template <>
__device__ __forceinline__ int acc_row<double>(int kq, int r) {
  return kq + 4 * r;
}
template <>
__device__ __forceinline__ int acc_row<float>(int kq, int r) {
  return 4 * kq + r;
}

template <class V>
__device__ inline auto cabs1(V z) -> decltype(z.x) {
  return fabs(z.x) + fabs(z.y);
}
template <class V>
__device__ inline V cmul2(V a, V b) {
  V r;
  r.x = a.x * b.x - a.y * b.y;
  r.y = a.x * b.y + a.y * b.x;
  return r;
}
template <class V>
__device__ inline V crecip(V b) {
  auto s = 1 / (b.x * b.x + b.y * b.y);
  V r;
  r.x = b.x * s;
  r.y = -b.y * s;
  return r;
}
template <class V>
__device__ inline V czero() {
  V r;
  r.x = 0;
  r.y = 0;
  return r;
}

// Tile (ti, tj) of the matrix the LU kernels factor, and the stride between
// the columns of a tile: column-major with leading dimension ld, or
// tile-major (d.tiled, tiled_index) with stride 64.  Every LU, refinement and
// update kernel addresses the factored matrix tile by tile through these.
template <class T>
__device__ __forceinline__ GCx<T> *tile_ptr(const SolveDesc &d, int ti, int tj) {
  GCx<T> *A = (GCx<T> *)d.A;
  return d.tiled ? A + ((long)tj * d.nt + ti) * (kTile * kTile)
                 : A + (long)kTile * ti + (long)d.ld * (kTile * tj);
}
__device__ __forceinline__ long tile_ld(const SolveDesc &d) { return d.tiled ? kTile : d.ld; }

// ---------------------------------------------------------------------------
// Complex 32x32x64 wave product on MFMA 16x16x4, 3M form:
//   P1 = Ar Br, P2 = Ai Bi, P3 = (Ar+Ai)(Br+Bi);  re = P1 - P2, im = P3 - P1 - P2
// (three real MFMAs per complex 16x16x4 block instead of four).
// The MFMA is applied to the transposed product, D'(j,i) = sum_k B(k,j) A(i,k),
// so the accumulator of a lane covers consecutive rows i of C and every C and
// A access is a run of 16 consecutive rows.  Operands are read straight from
// L2/LDS into registers in MFMA layout (a-operand lane value B(k0+kq, j0+li),
// b-operand lane value A(i0+li, k0+kq)), loaded ahead of the MFMAs; no LDS
// staging and no barriers, so the waves of a CU run independently.
// N: a wave's block is 16N x 16N (2: the 32x32 block above; 1: 16x16, for
// launches that would leave compute units idle otherwise).
template <class T, int N = 2>
struct Acc3 {
  Acc4<T> p[3][N][N];
};

// One k-step (3 N^2 MFMAs) of the 3M product from operands already in registers.
template <class T, int N>
__device__ __forceinline__ void gemm3m_step(CxT<T> (&av)[N], CxT<T> (&bv)[N], Acc3<T, N> &q) {
  T as[N], bs[N];
#pragma unroll
  for (int t = 0; t < N; t++) {
    as[t] = av[t].x + av[t].y;
    bs[t] = bv[t].x + bv[t].y;
  }
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++) q.p[0][bj][bi] = mfma4(bv[bj].x, av[bi].x, q.p[0][bj][bi]);
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++) q.p[1][bj][bi] = mfma4(bv[bj].y, av[bi].y, q.p[1][bj][bi]);
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++) q.p[2][bj][bi] = mfma4(bs[bj], as[bi], q.p[2][bj][bi]);
}

// q += A B over nk k-steps of four.  Operand loads run PF (3 or 7) k-steps
// ahead of the MFMAs; nk is a multiple of PF + 1.  Three of a 32x32 block (768
// MFMA cycles each in FP64, 432 in FP32) cover an L2 round trip; those of a
// 16x16 block are a quarter as long.
template <class T, int N, int PF = 3, class FA, class FB>
__device__ __forceinline__ void wave_gemm3m(FA fa, FB fb, int nk, Acc3<T, N> &q) {
  typedef CxT<T> V;
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  V a[PF + 1][N], b[PF + 1][N];
  auto load = [&](int slot, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < N; t++) {
      a[slot][t] = fa(16 * t + li, 4 * ks + kq);
      b[slot][t] = fb(4 * ks + kq, 16 * t + li);
    }
  };
  auto step = [&](int slot) __attribute__((always_inline)) {
    V av[N], bv[N];
#pragma unroll
    for (int t = 0; t < N; t++) {
      av[t] = a[slot][t];
      bv[t] = b[slot][t];
    }
    gemm3m_step<T, N>(av, bv, q);
  };
#pragma unroll
  for (int i = 0; i < PF; i++) load(i, i);
  int ks = 0;
#pragma unroll 1
  for (; ks < nk - PF - 1; ks += PF + 1) {
#pragma unroll
    for (int i = 0; i <= PF; i++) {
      load((i + PF) & PF, ks + i + PF);
      step(i);
    }
  }
  load(PF, ks + PF);
#pragma unroll
  for (int i = 0; i <= PF; i++) step(i);
}

// The same in FP64 for operands in global memory, nk a multiple of 4: A(i, k)
// at A[i + ld k], B(k, j) at B[k + ld j], both wave-uniform.  An FP64 MFMA
// holds its SIMD's VALU for all of its 64 cycles, whichever wave the VALU work
// is of, so every other instruction of the loop adds to its time: the
// operands come by buffer loads whose k offset is scalar, and the only VALU
// work left of a step are the sums of the 3M form (through pointers, with A
// negated, it was 17 instructions; 64 solves of N = 2160: trailing updates
// 23.8 -> 22.4 ms at K = 128).  The offsets have 32 bits.  A's k runs over a
// group's four tiles in the LU, 4096 ld bytes, but over whole tile rows in the
// explicit inverse, 16 ld^2: LONG moves A's 64-bit base with k there, and an
// offset spans 32 columns at most.
template <bool LONG>
__device__ __forceinline__ void wave_gemm3m_k(const GCx<double> *A, const GCx<double> *B, long ld,
                                              int nk, Acc3<double, 2> &q) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef unsigned b128 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  constexpr int kRange = 0x7fffffff, kFlags = 0x00027000;  // raw buffer, byte offsets
  auto resource = [](const GCx<double> *p) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, kRange, kFlags);
  };
  auto ra = resource(A);
  const auto rb = resource(B);
  const int ld16 = (int)ld * 16;
  constexpr int N = 2, PF = 3;
  const int va = 16 * li + ld16 * kq;  // A(li, kq)
  int vb[N];                           // B(kq, 16 t + li)
#pragma unroll
  for (int t = 0; t < N; t++) vb[t] = 16 * kq + ld16 * (16 * t + li);
  double2 a[PF + 1][N], b[PF + 1][N];
  auto get = [](b128 x) __attribute__((always_inline)) {
    return double2{__hiloint2double(x[1], x[0]), __hiloint2double(x[3], x[2])};
  };
  // k-step ks0 + u; LONG: ra at ks0
  auto load = [&](int slot, int ks0, int u) __attribute__((always_inline)) {
    const int sa = 4 * (LONG ? u : ks0 + u) * ld16, sb = 64 * (ks0 + u);
#pragma unroll
    for (int t = 0; t < N; t++)
      a[slot][t] = get(__builtin_amdgcn_raw_buffer_load_b128(ra, va + 256 * t, sa, 0));
#pragma unroll
    for (int t = 0; t < N; t++)
      b[slot][t] = get(__builtin_amdgcn_raw_buffer_load_b128(rb, vb[t], sb, 0));
  };
  auto step = [&](int slot) __attribute__((always_inline)) {
    double2 av[N], bv[N];
#pragma unroll
    for (int t = 0; t < N; t++) {
      av[t] = a[slot][t];
      bv[t] = b[slot][t];
    }
    gemm3m_step<double, N>(av, bv, q);
  };
#pragma unroll
  for (int i = 0; i < PF; i++) load(i, 0, i);
  int ks = 0;
#pragma unroll 1
  for (; ks < nk - PF - 1; ks += PF + 1) {
#pragma unroll
    for (int i = 0; i <= PF; i++) {
      load((i + PF) & PF, ks, i + PF);
      step(i);
    }
    if (LONG) {
      A += 4 * (PF + 1) * ld;
      ra = resource(A);
    }
  }
  load(PF, ks, PF);
#pragma unroll
  for (int i = 0; i <= PF; i++) step(i);
#endif
}

// Wave-scope ordering of LDS traffic: what any lane has written before is there
// for the others' reads after, and what they read before is not overwritten.
// (The hardware keeps a wave's LDS operations in order; without the fence the
// compiler may still move a lane's read over its own write elsewhere.)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// LDS of one wave for the operand B of wave_gemm3m_staged: two chunks of 16 k.
struct BStage {
  __align__(16) double2 b[2][16][17];  // [chunk][column][k]
};

// The same for a 16 x 16 block, nk a multiple of 8; `st` is the wave's own
// LDS.  A's rows are contiguous over the lanes; B's are not (a lane's column,
// four k over the lane groups), and read straight into that layout every lane
// is an L1 access of its own, 64 a load.  A 16 x 16 block has a load of each a
// k-step of 192 MFMA cycles, and L1 was busy 82% of the time (the MFMAs 40%)
// in the inverse of eight solves of N = 944.  So B is read 16 k by 4 columns a
// load, 16 accesses, and turned in LDS: 1.06 -> 0.87 ms there.  A 32 x 32
// block, with half the loads to an MFMA, gains nothing (64 solves of N = 2160:
// trailing updates 18.4 ms either way, six of N = 4384 16.2 and 16.5), and
// neither do loads further ahead.  A's base always moves, an offset spans 48
// columns at most (eight adjoint solves of N = 944 2.33 ms either way).
__device__ __forceinline__ void wave_gemm3m_staged(const GCx<double> *A, const GCx<double> *B,
                                                   long ld, int nk, Acc3<double, 1> &q,
                                                   BStage &st) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef unsigned b128 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  constexpr int kRange = 0x7fffffff, kFlags = 0x00027000;  // raw buffer, byte offsets
  auto resource = [](const GCx<double> *p) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, kRange, kFlags);
  };
  auto ra = resource(A);
  const auto rb = resource(B);
  const int ld16 = (int)ld * 16;
  const int v0 = 16 * li + ld16 * kq;  // A(li, kq); B(li, kq): 16 k, columns kq + 4 m
  double2 a[8], b[4];
  auto get = [](b128 x) __attribute__((always_inline)) {
    return double2{__hiloint2double(x[1], x[0]), __hiloint2double(x[3], x[2])};
  };
  auto load_a = [&](int slot, int ks) __attribute__((always_inline)) {
    a[slot] = get(__builtin_amdgcn_raw_buffer_load_b128(ra, v0, 4 * ks * ld16, 0));
  };
  auto load_b = [&](int c) __attribute__((always_inline)) {  // chunk c: k-steps 4c .. 4c+3
#pragma unroll
    for (int m = 0; m < 4; m++)
      b[m] = get(__builtin_amdgcn_raw_buffer_load_b128(rb, v0, 256 * c + 4 * m * ld16, 0));
  };
  auto put_b = [&](int buf) __attribute__((always_inline)) {
    wave_lds_fence();
#pragma unroll
    for (int m = 0; m < 4; m++) st.b[buf][kq + 4 * m][li] = b[m];
    wave_lds_fence();
  };
  // the chunk in LDS buffer `buf` (its number mod 2), ra at the k-step 0 of a
  // chunk in buffer 0; the A k-steps of the chunk after it are loaded on the way
  // when `next`
  auto chunk = [&](int buf, bool next) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (next) load_a((4 * buf + u + 4) & 7, 4 * buf + u + 4);
      double2 av[1] = {a[4 * buf + u]}, bv[1] = {st.b[buf][li][4 * u + kq]};
      gemm3m_step<double, 1>(av, bv, q);
    }
  };
  const int nc = nk / 4;
  load_b(0);
#pragma unroll
  for (int i = 0; i < 4; i++) load_a(i, i);
  put_b(0);
  load_b(1);
  int c = 0;
#pragma unroll 1
  for (; c < nc - 2; c += 2) {
    put_b(1);
    load_b(c + 2);
    chunk(0, true);
    put_b(0);
    load_b(c + 3);
    chunk(1, true);
    A += 32 * ld;
    ra = resource(A);
  }
  put_b(1);
  chunk(0, true);
  chunk(1, false);
#endif
}

// LDS of one wave for the operand B of tile_products_f32: two chunks of 16 k.
template <int N>
struct BStage32 {
  __align__(16) float2 b[2][16 * N][18];  // [chunk][column][k]
};

// The FP32 form: q += sum_{u < ns} A_u B_u over 64-wide tiles, A_u = A + u sa,
// B_u = B + u sb, wave-uniform.  Here B read in the MFMA's layout is 128 L1
// accesses a k-step (one per lane and column block) of 432 MFMA cycles, for
// each of four waves: L1 was the bound.  Read 16 k by 8 columns a load and
// turned in LDS it is 16 (64 solves of ten tiles: panels and trailing updates
// 660 -> 495 us).
template <int N>
__device__ __forceinline__ void tile_products_f32(const GCx<float> *A, long sa,
                                                  const GCx<float> *B, long sb, long ld, int ns,
                                                  Acc3<float, N> &q, BStage32<N> &st) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef unsigned b64 __attribute__((ext_vector_type(2)));
  typedef unsigned b128 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  constexpr int kRange = 0x7fffffff, kFlags = 0x00027000;  // raw buffer, byte offsets
  const auto ra = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, kRange, kFlags);
  const auto rb = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, kRange, kFlags);
  const int ld8 = (int)ld * 8, sa8 = (int)sa * 8, sb8 = (int)sb * 8;
  const int va = 8 * li + ld8 * kq;                     // A(li, kq)
  const int bk = 2 * (lane & 7), bc = lane >> 3;        // B(bk, bc): 16 k, columns bc + 8 m
  const int vb = 8 * bk + ld8 * bc;
  constexpr int NB = 2 * N;
  float2 a[8][N];
  b128 b[NB];
  auto load_a = [&](int slot, int c, int u) __attribute__((always_inline)) {  // k-step u of chunk c
    const int off = (c >> 2) * sa8 + (16 * (c & 3) + 4 * u) * ld8;
#pragma unroll
    for (int t = 0; t < N; t++) {
      const b64 x = __builtin_amdgcn_raw_buffer_load_b64(ra, va + 128 * t, off, 0);
      a[slot][t] = make_float2(__uint_as_float(x[0]), __uint_as_float(x[1]));
    }
  };
  auto load_b = [&](int c) __attribute__((always_inline)) {
    const int off = (c >> 2) * sb8 + 128 * (c & 3);
#pragma unroll
    for (int m = 0; m < NB; m++)
      b[m] = __builtin_amdgcn_raw_buffer_load_b128(rb, vb, off + 8 * m * ld8, 0);
  };
  auto put_b = [&](int buf) __attribute__((always_inline)) {
    wave_lds_fence();
#pragma unroll
    for (int m = 0; m < NB; m++) *(b128 *)&st.b[buf][bc + 8 * m][bk] = b[m];
    wave_lds_fence();
  };
  auto chunk = [&](int c, int buf, bool next) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (next) load_a((4 * buf + u + 4) & 7, c + 1, u);
      float2 av[N], bv[N];
#pragma unroll
      for (int t = 0; t < N; t++) {
        av[t] = a[4 * buf + u][t];
        bv[t] = st.b[buf][16 * t + li][4 * u + kq];
      }
      gemm3m_step<float, N>(av, bv, q);
    }
  };
  const int nc = 4 * ns;
  load_b(0);
#pragma unroll
  for (int u = 0; u < 4; u++) load_a(u, 0, u);
  put_b(0);
  load_b(1);
  int c = 0;
#pragma unroll 1
  for (; c < nc - 2; c += 2) {
    put_b(1);
    load_b(c + 2);
    chunk(c, 0, true);
    put_b(0);
    load_b(c + 3);
    chunk(c + 1, 1, true);
  }
  put_b(1);
  chunk(c, 0, true);
  chunk(c + 1, 1, false);
#endif
}

// LDS of a workgroup's four waves for tile_products.
template <class T, int N>
struct ProductStage {
  int none;
};
template <>
struct ProductStage<double, 1> {
  BStage w[4];
};
template <int N>
struct ProductStage<float, N> {
  BStage32<N> w[4];
};

// q += sum_{u < ns} A_u B_u over 64-wide tiles: A_u = A + u sa, B_u = B + u sb
// (FP64: consecutive in k, so that ns tiles are one product).  LONG: ns is not
// bounded by a group's four steps (FP64 alone).
template <class T, int N, bool LONG = false>
__device__ __forceinline__ void tile_products(const GCx<T> *A, long sa, const GCx<T> *B, long sb,
                                              long ld, int ns, Acc3<T, N> &q,
                                              ProductStage<T, N> &st) {
  if (ns <= 0) return;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (sizeof(T) == 4) tile_products_f32<N>(A, sa, B, sb, ld, ns, q, st.w[w]);
  else if constexpr (N == 1) wave_gemm3m_staged(A, B, ld, 16 * ns, q, st.w[w]);
  else wave_gemm3m_k<LONG>(A, B, ld, 16 * ns, q);
}

template <class T, int N>
__device__ __forceinline__ void zero_acc(Acc3<T, N> &q) {
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int bj = 0; bj < N; bj++)
#pragma unroll
      for (int bi = 0; bi < N; bi++)
#pragma unroll
        for (int r = 0; r < 4; r++) q.p[m][bj][bi][r] = T(0);
}

// -C enters the 3M sums at the start (q1 = -Cre, q2 = 0, q3 = -(Cre + Cim)),
// so that C - A B = (q2 - q1, q1 + q2 - q3) at the end: C is read and written
// once however many products are taken, and no operand is negated.
template <class T, int N>
__device__ __forceinline__ void set_minus(Acc3<T, N> &q, int bj, int bi, int r, T re, T im) {
  q.p[0][bj][bi][r] = -re;
  q.p[1][bj][bi][r] = T(0);
  q.p[2][bj][bi][r] = -re - im;
}
template <class T, int N>
__device__ __forceinline__ CxT<T> minus_value(const Acc3<T, N> &q, int bj, int bi, int r) {
  CxT<T> v;
  v.x = q.p[1][bj][bi][r] - q.p[0][bj][bi][r];
  v.y = q.p[0][bj][bi][r] + q.p[1][bj][bi][r] - q.p[2][bj][bi][r];
  return v;
}
template <class T, int N>
__device__ __forceinline__ CxT<T> plus_value(const Acc3<T, N> &q, int bj, int bi, int r) {
  CxT<T> v;
  v.x = q.p[0][bj][bi][r] - q.p[1][bj][bi][r];
  v.y = q.p[2][bj][bi][r] - q.p[0][bj][bi][r] - q.p[1][bj][bi][r];
  return v;
}

// What a panel tile does with the inverse of the step's diagonal tile.
enum PanelOp {
  kRightU,  // X = C' U^-1: a tile below the diagonal tile
  kLeftL,   // X = L^-1 P C': a tile right of it, or of the inverse's forward half
  kLeftU    // X = U^-1 C': a tile of the inverse's backward half
};

// LDS of panel_op: C' (a tile, or 16 rows or columns of one) and the pivots.
template <class T, int N>
struct PanelLds {
  union {
    __align__(16) CxT<T> c[kTile * ((N == 2 ? kTile : 16) + 1)];
    ProductStage<T, N> st;  // before that: B of the earlier steps
  };
  int rowpos[kTile];
  __device__ PanelLds() {}
};

// One panel tile or a piece of it by a 256-thread workgroup:
//   C' = [C] - sum_{u < ns} A_u B_u,   X = C' U^-1, L^-1 P C' or U^-1 C',
// so that the tile takes the earlier steps of its group (of the whole inverse)
// on the way into its panel product, with no launch and no pass over C of
// their own.  N = 2: the whole 64x64 tile, a 32x32 block per wave, A read at
// 64 rows and B at 64 columns.  N = 1: 16 rows (kRightU) or 16 columns of it,
// which the product with the inverse leaves independent of the others, a
// 16x16 block per wave: a quarter of the time per tile on four times the
// workgroups, at twice the operand loads per MFMA.  `piece` = 0..3 then.
// perm: the pivots of kLeftL; identity: C' = the identity tile (nothing else).
template <class T, int N, PanelOp OP, bool LONG = false>
__device__ __forceinline__ void panel_op(GCx<T> *__restrict__ C, bool load_c, bool identity,
                                         const GCx<T> *A, long sa, const GCx<T> *B, long sb,
                                         long ld, int ns, const GCx<T> *__restrict__ inv,
                                         const LSMSX_GLOBAL int *__restrict__ perm, int piece,
                                         PanelLds<T, N> &lds) {
  typedef CxT<T> V;
  constexpr bool RIGHT = OP == kRightU;
  // Ts[column][row] of C' (rows in pivot order for kLeftL)
  constexpr int CR = N == 2 || !RIGHT ? kTile : 16, CC = N == 2 || RIGHT ? kTile : 16;
  static_assert(sizeof(V) * CC * (CR + 1) <= sizeof(lds.c), "LDS tile");
  V(*Ts)[CR + 1] = reinterpret_cast<V(*)[CR + 1]>(lds.c);
  int *rowpos = lds.rowpos;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the wave's block in the piece, and the piece in the tile
  const int wr = N == 2 ? 32 * (w & 1) : RIGHT ? 0 : 16 * w;
  const int wc = N == 2 ? 32 * (w >> 1) : RIGHT ? 16 * w : 0;
  const int r0 = N == 2 || !RIGHT ? 0 : 16 * piece, c0 = N == 2 || RIGHT ? 0 : 16 * piece;
  if (OP == kLeftL && tid < kTile) rowpos[perm[tid]] = tid;
  GCx<T> *Cw = C + (r0 + wr) + ld * (c0 + wc);
  Acc3<T, N> q;
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = 16 * bi + li, j = 16 * bj + acc_row<T>(kq, r);
        V c = czero<V>();
        if (load_c) c = ldg<T>(Cw + (i + ld * j));
        else if (identity) c.x = r0 + wr + i == c0 + wc + j ? T(1) : T(0);
        set_minus<T, N>(q, bj, bi, r, c.x, c.y);
      }
  tile_products<T, N, LONG>(A + (r0 + wr), sa, B + ld * (c0 + wc), sb, ld, ns, q, lds.st);
  // rowpos is there, the staged operands are read
  if (OP == kLeftL || sizeof(T) == 4 || N == 1) __syncthreads();
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = wr + 16 * bi + li, j = wc + 16 * bj + acc_row<T>(kq, r);
        Ts[j][OP == kLeftL ? rowpos[i] : i] = minus_value<T, N>(q, bj, bi, r);
      }
  __syncthreads();
  zero_acc(q);
  // Second product, by 16-wide strips of the triangular side (columns of U^-1,
  // rows of the left factors).  Strip t takes the k-steps up to its diagonal
  // block, or from it on: for N = 2 a wave has strips t and 3 - t, so that all
  // waves have the same work and none is done on the zero blocks.
  const int t0 = N == 2 ? (RIGHT ? w >> 1 : w & 1) : w;
  auto strip = [&](int b) { return 16 * (N == 2 && b ? 3 - t0 : t0); };
  // element k of the triangular factor at offset x of strip b
  auto tri = [&](int b, int x, int k) __attribute__((always_inline)) {
    const int ii = strip(b) + x;
    V v = ldg<T>(inv + (OP == kRightU ? k + kTile * ii : ii + kTile * k));
    if (OP == kLeftL) {
      if (ii <= k) {
        v.x = ii == k ? T(1) : T(0);
        v.y = T(0);
      }
    } else if (OP == kRightU ? k > ii : k < ii) {
      v = czero<V>();
    }
    return v;
  };
  const int pr = N == 2 ? wr : 0, pc = N == 2 ? wc : 0;  // the wave's rows (columns) of C'
  auto full = [&](int k0, int nk) __attribute__((always_inline)) {
    if constexpr (RIGHT)
      wave_gemm3m<T, N>([&](int i, int k) { return Ts[k0 + k][pr + i]; },
                        [&](int k, int j) { return tri(j >> 4, j & 15, k0 + k); }, nk, q);
    else
      wave_gemm3m<T, N>([&](int i, int k) { return tri(i >> 4, i & 15, k0 + k); },
                        [&](int k, int j) { return Ts[pc + j][k0 + k]; }, nk, q);
  };
  // k-steps of one strip alone, b the one that is longer
  auto half = [&](auto bc, int k0, int nk) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
    for (int ks = 0; ks < nk; ks += 4) {
      V av[4][2], bv[4][2];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int k = k0 + 4 * (ks + u) + kq;
        if constexpr (RIGHT) {
          bv[u][b] = tri(b, li, k);
          av[u][0] = Ts[k][pr + li];
          av[u][1] = Ts[k][pr + 16 + li];
        } else {
          av[u][b] = tri(b, li, k);
          bv[u][0] = Ts[pc + li][k];
          bv[u][1] = Ts[pc + 16 + li][k];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int o = 0; o < 2; o++) {
          const int bi = RIGHT ? o : b, bj = RIGHT ? b : o;
          const V x = av[u][bi], y = bv[u][bj];
          q.p[0][bj][bi] = mfma4(y.x, x.x, q.p[0][bj][bi]);
          q.p[1][bj][bi] = mfma4(y.y, x.y, q.p[1][bj][bi]);
          q.p[2][bj][bi] = mfma4(y.x + y.y, x.x + x.y, q.p[2][bj][bi]);
        }
    }
  };
  if constexpr (N == 1) {
    if (OP == kLeftU) full(16 * t0, 16 - 4 * t0);
    else full(0, 4 * t0 + 4);
  } else if constexpr (OP == kLeftU) {
    // strip 3 - t starts at its own block, strip t before it
    half(std::integral_constant<int, 0>(), 16 * t0, 4 * (3 - 2 * t0));
    full(16 * (3 - t0), 4 * t0 + 4);
  } else {
    full(0, 4 * t0 + 4);
    half(std::integral_constant<int, 1>(), 16 * (t0 + 1), 4 * (3 - 2 * t0));
  }
  GCx<T> *Cp = C + (RIGHT ? r0 + pr : 0) + ld * (RIGHT ? 0 : c0 + pc);
#pragma unroll
  for (int bj = 0; bj < N; bj++)
#pragma unroll
    for (int bi = 0; bi < N; bi++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = (RIGHT ? 16 * bi : strip(bi)) + li;
        const int j = (RIGHT ? strip(bj) : 16 * bj) + acc_row<T>(kq, r);
        Cp[i + ld * j] = plus_value<T, N>(q, bj, bi, r);
      }
}

// Split-FP16 operands: eight halves of a 32-wide k chunk per lane, the
// FP16 MFMA with FP32 accumulation, and a sign flip of eight halves (four
// 32-bit XORs of the packed sign bits).
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(1))) const h8 GH8;
#else
typedef const h8 GH8;
#endif
__device__ __forceinline__ f4 mfma_h(h8 a, h8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
typedef unsigned u4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ h8 neg8(h8 v) {
  return __builtin_bit_cast(h8, __builtin_bit_cast(u4v, v) ^ 0x80008000u);
}

// LDS k group of row r holding logical group g (8 halves): XOR swizzle of the
// four groups of a 64-byte row by (r >> 1) ^ (r >> 2), so that any 8 (and any
// 16) consecutive rows read at one group cover distinct 16-byte bank groups:
// rows of equal parity among 8 (equal r mod 4 among 16) get distinct masks.
__device__ __forceinline__ int swz_group(int r, int g) { return g ^ (((r >> 1) ^ (r >> 2)) & 3); }

// XCD-aware workgroup order.  Workgroups are dispatched round-robin over
// the 8 XCDs by linear id, so consecutive tiles of one solve would land on
// 8 different L2 caches.  The remap gives each XCD a contiguous range of
// the (tile, solve) grid -- whole solves, in a batched launch -- so the L
// and U panels a solve's tiles share are fetched into one L2.  A bijection
// whenever the grid size is a multiple of 8 (otherwise the order is kept).
constexpr int kNumXcd = 8;
__device__ __forceinline__ void xcd_remap(int &bx, int &by) {
  const int gx = gridDim.x;
  const long total = (long)gx * gridDim.y;
  if (total % kNumXcd) return;
  const long lin = bx + (long)gx * by;
  const long per = total / kNumXcd;
  const long l2 = (lin % kNumXcd) * per + lin / kNumXcd;
  bx = (int)(l2 % gx);
  by = (int)(l2 / gx);
}

}  // namespace lsmsx
