// 16 x 16 tile building blocks shared by the diagonal-block kernels
// (diag.hip) and the batched factorisation (batched.hip).
//
// * TileAcc / tile_mma: a 16 x 16 accumulator in the v_mfma_f64_16x16x4_f64
//   result layout (lane l, register r holds element (l / 16 + 4 r, l % 16))
//   and C += s X op(Y) over a 16-deep k range, complex as four real MFMAs.
// * leaf_factor_invert: one wave factors a 16 x 16 Hermitian positive definite
//   tile held in registers and inverts the factor, moving values between
//   lanes with row swaps and DPP row broadcasts, so the 16 sequential pivots
//   need no workgroup barrier and no LDS round trip; leaf_inverse_cols
//   inverts a factored one.
#pragma once

#include <type_traits>

#include "internal.h"

namespace hc {
namespace t16 {

constexpr int LEAF = 16;

typedef double v4d __attribute__((ext_vector_type(4)));

// Last argument of __builtin_amdgcn_mfma_f64_*: on gfx950 the FP64 MFMA's
// BLGP field holds negate modifiers (bit 0: A, bit 1: B, bit 2: C), so
// acc - A B is one instruction with no VALU negation of the operand.
constexpr int kNegA = 1;

__device__ __forceinline__ double sel(bool c, double a, double b) { return c ? a : b; }
__device__ __forceinline__ zd sel(bool c, zd a, zd b) { return make_zd(c ? a.x : b.x, c ? a.y : b.y); }

template <typename T> struct TileAcc;
template <> struct TileAcc<double> { v4d re; };
template <> struct TileAcc<zd> { v4d re, im; };

__device__ __forceinline__ void acc_zero(TileAcc<double> &c) { c.re = (v4d){0.0, 0.0, 0.0, 0.0}; }
__device__ __forceinline__ void acc_zero(TileAcc<zd> &c) {
  c.re = (v4d){0.0, 0.0, 0.0, 0.0};
  c.im = c.re;
}

__device__ __forceinline__ double acc_get(const TileAcc<double> &c, int r) { return c.re[r]; }
__device__ __forceinline__ zd acc_get(const TileAcc<zd> &c, int r) { return make_zd(c.re[r], c.im[r]); }
__device__ __forceinline__ void acc_set(TileAcc<double> &c, int r, double v) { c.re[r] = v; }
__device__ __forceinline__ void acc_set(TileAcc<zd> &c, int r, zd v) {
  c.re[r] = v.x;
  c.im[r] = v.y;
}

// Tile at C (column-major, leading dimension ls) <-> accumulator.
template <typename T>
__device__ __forceinline__ void acc_load(TileAcc<T> &c, const T *C, int ls) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
#pragma unroll
  for (int r = 0; r < 4; r++) acc_set(c, r, C[li * ls + lk + 4 * r]);
}
template <typename T>
__device__ __forceinline__ void acc_store(const TileAcc<T> &c, T *C, int ls) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
#pragma unroll
  for (int r = 0; r < 4; r++) C[li * ls + lk + 4 * r] = acc_get(c, r);
}

// acc += sx * X op(Y), 16-deep, X and Y column-major tiles; op(Y) = Y^H when
// YH.  MFMA operands: X fragment lane l = X(l % 16, k0 + l / 16), op(Y)
// fragment lane l = op(Y)(k0 + l / 16, l % 16).
template <bool YH>
__device__ __forceinline__ void tile_mma(TileAcc<double> &c, const double *X, int ldx, const double *Y,
                                         int ldy, double sx) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
#pragma unroll
  for (int k0 = 0; k0 < LEAF; k0 += 4) {
    const double a = sx * X[(k0 + lk) * ldx + li];
    const double b = YH ? Y[(k0 + lk) * ldy + li] : Y[li * ldy + k0 + lk];
    c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c.re, 0, 0, 0);
  }
}
template <bool YH>
__device__ __forceinline__ void tile_mma(TileAcc<zd> &c, const zd *X, int ldx, const zd *Y, int ldy,
                                         double sx) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
#pragma unroll
  for (int k0 = 0; k0 < LEAF; k0 += 4) {
    const zd a = sx * X[(k0 + lk) * ldx + li];
    const zd b = YH ? conjx(Y[(k0 + lk) * ldy + li]) : Y[li * ldy + k0 + lk];
    c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, c.re, 0, 0, 0);
    c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, c.re, 0, 0, 0);
    c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, c.im, 0, 0, 0);
    c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, c.im, 0, 0, 0);
  }
}

// Orders this wave's LDS writes before its following LDS reads by other lanes.
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// ---------------------------------------------------------------------------
// Row layout: lane r + 16 q holds row r of the leaf in a[0..15] (the four
// 16-lane rows of the wave, q = 0..3, hold the same matrix row; entries above
// the diagonal are not used).  A pivot's own row element is then in the lane's
// registers, and the other elements it needs come from DPP row_newbcast (lane
// m of each 16-lane row to the whole row: a VGPR move, no LDS round trip and
// no scalar register).
// ---------------------------------------------------------------------------

// f(integral_constant<int, I>) for I = B .. E - 1: loop indices that are
// compile-time constants without relying on the unroller (which declines
// large bodies, leaving register arrays indexed at run time, i.e. in scratch).
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// v from lane M of this lane's 16-lane row.
template <int M>
__device__ __forceinline__ int row_bcast_b32(int v) {
  // every lane reads a valid source lane, so no "old" value is needed
  return __builtin_amdgcn_mov_dpp(v, 0x150 + M, 0xf, 0xf, true);
}
// A 64-bit value moves in one v_mov_b64_dpp (gfx950 has 64-bit DPP moves
// with row_newbcast), not as two 32-bit halves.
template <int M>
__device__ __forceinline__ double row_bcast(double v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + M, 0xf, 0xf, true);
}
template <int M>
__device__ __forceinline__ zd row_bcast(zd v) {
  return make_zd(row_bcast<M>(v.x), row_bcast<M>(v.y));
}

// Columns q, q + 4, q + 8, q + 12 of X = inv(L) for a factored leaf L in the
// row layout (lane r + 16 q: x[j] = X(r, q + 4 j), zeros above the
// diagonal; the wave's four rows share the sixteen columns).  Forward
// substitution X(k, c) = (delta_kc - sum_{j < k} L(k, j) X(j, c)) / L(k, k):
// step k broadcasts row k of X inside each 16-lane row and every lane adds
// its L(r, k) X(k, c); with the strictly lower part of L the sums of rows
// already finished stop growing, so X is formed once after the loop.
template <typename T>
__device__ __forceinline__ void leaf_inverse_cols(const T a[LEAF], T x[4]) {
  int r = threadIdx.x & 15, q = (threadIdx.x >> 4) & 3;
  // opaque here, so that what is derived from the lane index is computed
  // here rather than hoisted out of the caller's loop and kept live (and
  // spilled) through the factorisation
  asm volatile("" : "+v"(r), "+v"(q));
  T dg = a[0];
#pragma unroll
  for (int c = 1; c < LEAF; c++) dg = sel(r == c, a[c], dg);
  const T dinv = from_real<T>(1.0) / dg;  // every lane its own row's pivot, in parallel
  T e[4], acc[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    e[j] = sel(r == q + 4 * j, from_real<T>(1.0), from_real<T>(0.0));
    acc[j] = from_real<T>(0.0);
  }
  static_for<0, LEAF>([&](auto K) {
    constexpr int k = decltype(K)::value;
    const T lk = sel(k < r, a[k], from_real<T>(0.0));  // strictly lower part of L
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const T xk = row_bcast<k>((e[j] - acc[j]) * dinv);  // X(k, q + 4 j), final in lane k
      acc[j] = acc[j] + lk * xk;
    }
  });
#pragma unroll
  for (int j = 0; j < 4; j++) x[j] = (e[j] - acc[j]) * dinv;
}

// ---------------------------------------------------------------------------
// Row fragments.  A 16 x 16 tile A is held as f[r] = A(l % 16, l / 16 + 4 r)
// in lane l: the matrix-core operand fragment of A for k-step r (either
// operand), and the result layout of A^T, so tiles enter and leave the matrix
// cores with no layout change.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void frag_load(TileAcc<T> &f, const T *C, int ls) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
#pragma unroll
  for (int r = 0; r < 4; r++) acc_set(f, r, C[(lk + 4 * r) * ls + li]);
}
template <typename T>
__device__ __forceinline__ void frag_store(const TileAcc<T> &f, T *C, int ls) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
#pragma unroll
  for (int r = 0; r < 4; r++) C[(lk + 4 * r) * ls + li] = acc_get(f, r);
}

// Rank-4 pieces (k-step s of the operands).  frag: f (row fragments) += or
// -= A conj(B)^T with A, B row fragments; acc: c (result layout) -= or += L X
// with L row fragments and X in the result layout.
template <bool NEG>
__device__ __forceinline__ void frag_rank4(TileAcc<double> &f, double a, double b) {
  f.re = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, f.re, 0, 0, NEG ? kNegA : 0);
}
template <bool NEG>
__device__ __forceinline__ void frag_rank4(TileAcc<zd> &f, zd a, zd b) {
  f.re = __builtin_amdgcn_mfma_f64_16x16x4f64(b.x, a.x, f.re, 0, 0, NEG ? kNegA : 0);
  f.im = __builtin_amdgcn_mfma_f64_16x16x4f64(b.x, a.y, f.im, 0, 0, NEG ? kNegA : 0);
  f.re = __builtin_amdgcn_mfma_f64_16x16x4f64(b.y, a.y, f.re, 0, 0, NEG ? kNegA : 0);
  f.im = __builtin_amdgcn_mfma_f64_16x16x4f64(b.y, a.x, f.im, 0, 0, NEG ? 0 : kNegA);
}
__device__ __forceinline__ void acc_rank4_sub(TileAcc<double> &c, double a, double x) {
  c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x, c.re, 0, 0, kNegA);
}
__device__ __forceinline__ void acc_rank4_sub(TileAcc<zd> &c, zd a, zd x) {
  c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.x, c.re, 0, 0, kNegA);
  c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.y, c.im, 0, 0, kNegA);
  c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, x.y, c.re, 0, 0, 0);
  c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, x.x, c.im, 0, 0, kNegA);
}

__device__ __forceinline__ void acc_rank4_add(TileAcc<double> &c, double a, double x) {
  c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x, c.re, 0, 0, 0);
}
__device__ __forceinline__ void acc_rank4_add(TileAcc<zd> &c, zd a, zd x) {
  c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.x, c.re, 0, 0, 0);
  c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.y, c.im, 0, 0, 0);
  c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, x.y, c.re, 0, 0, kNegA);
  c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, x.x, c.im, 0, 0, 0);
}

// o[j] = v of lane l % 16 + 16 j: every lane gets the four values that its
// position has in the four 16-lane rows (two row-swap stages, no LDS).
__device__ __forceinline__ void row_gather4(double v, double (&o)[4]) {
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  const v2u b = __builtin_bit_cast(v2u, v);
  const auto s0 = __builtin_amdgcn_permlane32_swap(b.x, b.x, false, false);  // {rows 0 1, rows 2 3}
  const auto s1 = __builtin_amdgcn_permlane32_swap(b.y, b.y, false, false);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const auto p0 = __builtin_amdgcn_permlane16_swap(s0[h], s0[h], false, false);
    const auto p1 = __builtin_amdgcn_permlane16_swap(s1[h], s1[h], false, false);
    const v2u even = {p0[0], p1[0]}, odd = {p0[1], p1[1]};
    o[2 * h] = __builtin_bit_cast(double, even);
    o[2 * h + 1] = __builtin_bit_cast(double, odd);
  }
}
__device__ __forceinline__ void row_gather4(zd v, zd (&o)[4]) {
  double re[4], im[4];
  row_gather4(v.x, re);
  row_gather4(v.y, im);
#pragma unroll
  for (int j = 0; j < 4; j++) o[j] = make_zd(re[j], im[j]);
}
// v[g], g = 0..3
template <typename T>
__device__ __forceinline__ T sel4(int g, const T (&v)[4]) {
  return sel((g & 2) != 0, sel((g & 1) != 0, v[3], v[2]), sel((g & 1) != 0, v[1], v[0]));
}

// c - a b
__device__ __forceinline__ double submul(double c, double a, double b) { return __builtin_fma(-a, b, c); }
__device__ __forceinline__ zd submul(zd c, zd a, zd b) {
  return make_zd(__builtin_fma(a.y, b.y, __builtin_fma(-a.x, b.x, c.x)),
                 __builtin_fma(-a.y, b.x, __builtin_fma(-a.x, b.y, c.y)));
}
// Re(c - a conj(b)) for real c
__device__ __forceinline__ double submulr(double c, double a, double b) { return __builtin_fma(-a, b, c); }
__device__ __forceinline__ double submulr(double c, zd a, zd b) {
  return __builtin_fma(-a.y, b.y, __builtin_fma(-a.x, b.x, c));
}

// 1 / sqrt(d), d > 0: the hardware estimate y corrected by the third-order
// step y (1 + e / 2 + 3 e^2 / 8), e = 1 - d y^2 (measured over [1, 4]: the
// estimate is within 5.3e-8, the result within 1.4e-16).
__device__ __forceinline__ double rsqrt_chain(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = __builtin_fma(-(d * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}
// 1 / d by the hardware estimate and the third-order step y (1 + e + e^2),
// e = 1 - d y.
__device__ __forceinline__ double recip_chain(double d) {
  const double y = __builtin_amdgcn_rcp(d);
  const double e = __builtin_fma(-d, y, 1.0);
  return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// One wave factors and inverts the Hermitian positive definite leaf f (row
// fragments; entries above the diagonal are not used) in four 4-column
// blocks.  Block r: every lane gathers its row's four entries (row_gather4)
// and the block's 4 x 4 diagonal part is broadcast to all lanes, which factor
// it redundantly (a chain of four pivots with no lane exchange) and solve
// their own row with it; the rest of the leaf takes the rank-4 update in one
// matrix-core product (complex: four).  The inverse X = inv(L) goes along as
// sixteen more rows: X starts as the identity, block r of its rows is solved
// with the same 4 x 4 part while the update of f is in the matrix pipe, and
// the rows below take their rank-4 update from it.  The elimination is
// A = L1 D L1^H (unit L1): the pivot chain has the reciprocal of d only, and
// L = L1 D^(1/2), X = D^(-1/2) inv(L1) take the square roots of a block's
// four pivots at once, one per lane group, and so do the pivot tests (one
// compare per block, looked at after the last).
// The leaf wave issues every instruction for all 64 lanes and a dependent
// FP64 operation takes about 12 cycles, so the leaf's time is its instruction
// count and its pivot chain: a column-at-a-time leaf in registers (rank-1
// updates with one DPP broadcast and one FMA per column) takes 4306 cycles,
// this one 2930 (one wave alone, real).
// Only the real part of a diagonal entry is used (complex).
// On return f holds L (entries above the diagonal unspecified).  The inverse
// (zeros above the diagonal) is handed out block by block: sink(r, l, x) gets
// l = L(lc, lg + 4 r) and x = X(lg + 4 r, lc) in lane lc + 16 lg.  Returns the
// first non-positive / NaN pivot (0-based, the same in every lane), or -1; on
// failure what was handed out and f are unspecified.
// SQ: the reciprocals of the pivots are formed as (1 / sqrt(d))^2, two dependent
// operations longer per pivot.  For the task-graph solver, whose log-determinants
// are compared with those of a factorisation that divides by the square root, at
// 10 n eps whatever the condition: on ill-conditioned 2 x 2 matrices two good
// factorisations differ by more, and this one rounds like that one.  Neither is
// the better answer (800 2 x 2 matrices, condition up to 1e9, against exact
// arithmetic: rms error 0.25 eps cond, with 1 / d 0.24), and the solver's time
// is the same (32.6 ms for 512 matrices up to n = 2048).
template <typename T, bool SQ = false, typename Sink>
__device__ __forceinline__ int leaf_factor_invert(TileAcc<T> &f, Sink sink) {
  int l = threadIdx.x & 63;
  asm volatile("" : "+v"(l));  // lane-derived values are formed here, not kept live across the caller's loop
  const int lc = l & 15, lg = l >> 4;
  unsigned long long ok[4];  // lane 16 k of ok[r]: pivot 4 r + k is positive
  TileAcc<T> L, x;
#pragma unroll
  for (int r = 0; r < 4; r++) acc_set(x, r, from_real<T>(lg + 4 * r == lc ? 1.0 : 0.0));
  static_for<0, 4>([&](auto R) {
    constexpr int r = decltype(R)::value, b = 4 * r;
    T a[4], y[4];
    double d[4];  // pivots of the block
    row_gather4(acc_get(f, r), a);
    d[0] = realx(row_bcast<b>(a[0]));
    d[1] = realx(row_bcast<b + 1>(a[1]));
    d[2] = realx(row_bcast<b + 2>(a[2]));
    d[3] = realx(row_bcast<b + 3>(a[3]));
    const T c10 = row_bcast<b + 1>(a[0]), c20 = row_bcast<b + 2>(a[0]), c30 = row_bcast<b + 3>(a[0]);
    T c21 = row_bcast<b + 2>(a[1]), c31 = row_bcast<b + 3>(a[1]), c32 = row_bcast<b + 3>(a[2]);
    auto recip = [](double v) {
      if constexpr (!SQ) return recip_chain(v);
      const double q = rsqrt_chain(v);
      return q * q;
    };
    // c_ij, a_j: unscaled columns (L1 D); l_ij = c_ij / d_j: L1
    const double rd0 = recip(d[0]);
    const T l10 = rd0 * c10, l20 = rd0 * c20, l30 = rd0 * c30;
    d[1] = submulr(d[1], l10, c10);
    c21 = submul(c21, l20, conjx(c10));
    c31 = submul(c31, l30, conjx(c10));
    d[2] = submulr(d[2], l20, c20);
    c32 = submul(c32, l30, conjx(c20));
    d[3] = submulr(d[3], l30, c30);
    a[1] = submul(a[1], a[0], conjx(l10));
    a[2] = submul(a[2], a[0], conjx(l20));
    a[3] = submul(a[3], a[0], conjx(l30));
    const double rd1 = recip(d[1]);
    const T l21 = rd1 * c21, l31 = rd1 * c31;
    d[2] = submulr(d[2], l21, c21);
    c32 = submul(c32, l31, conjx(c21));
    d[3] = submulr(d[3], l31, c31);
    a[2] = submul(a[2], a[1], conjx(l21));
    a[3] = submul(a[3], a[1], conjx(l31));
    const double rd2 = recip(d[2]);
    const T l32 = rd2 * c32;
    d[3] = submulr(d[3], l32, c32);
    a[3] = submul(a[3], a[2], conjx(l32));
    const double dv = sel4(lg, d);        // the pivot k = 4 r + lg of this lane group
    ok[r] = __ballot(dv > 0.0);           // false for NaN
    const double rs = rsqrt_chain(dv);    // 1 / L(k, k)
    const T lr = rs * sel4(lg, a);        // column k of L
    if constexpr (r < 3) frag_rank4<true>(f, lr, lr);
    __builtin_amdgcn_sched_barrier(0);    // X's block below runs in the shadow of that product
    row_gather4(acc_get(x, r), y);
    y[1] = submul(y[1], l10, y[0]);
    y[2] = submul(submul(y[2], l20, y[0]), l21, y[1]);
    y[3] = submul(submul(submul(y[3], l30, y[0]), l31, y[1]), l32, y[2]);
    const T xr = rs * sel4(lg, y);        // row k of X
    if constexpr (r < 3) acc_rank4_sub(x, sel(lc > b + 3, lr, from_real<T>(0.0)), xr);
    // the diagonal is real: an imaginary part (the caller's, which is ignored, or
    // rounding) stays in its own entry up to here
    const T lf = is_complex<T>::value ? sel(lc == b + lg, from_real<T>(realx(lr)), lr) : lr;
    acc_set(L, r, lf);
    sink(r, lf, xr);
    __builtin_amdgcn_sched_barrier(0);
  });
  f = L;
  int bad = -1;
  if ((ok[0] & ok[1] & ok[2] & ok[3]) != ~0ull) {
    asm volatile("");  // keeps the search a branch: it is off the usual path
#pragma unroll
    for (int k = LEAF - 1; k >= 0; k--) bad = ((ok[k / 4] >> (16 * (k % 4))) & 1) != 0 ? bad : k;
  }
  return bad;
}

}  // namespace t16
}  // namespace hc
