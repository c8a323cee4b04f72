// Diagonal-block kernels and reductions, double and double complex.
//
// A diagonal block of order n <= 128 (double) or n <= 64 (complex) is held in
// LDS (and, for the factor and inverse, in registers) by one workgroup and
// processed in "lower form": for an
// upper-triangle caller the block is loaded conjugate-transposed, so
// U^H U = L L^H, inv(U) = inv(L)^H and U U^H = L^H L reduce every case to a
// lower-triangular kernel, and stored back conjugate-transposed.
//
//   diag_potrf   factor + inverse (reference lapack/dpotrf.cu:23-148 and the
//                host dpotrf of lapack/dpotrf.c:268; here it never leaves the GPU)
//   diag_trtri   triangular inverse (reference lapack/dtrtri.cu:23-167)
//   diag_lauum   L^H L / U U^H      (reference lapack/dlauum.cu:23-91), single precision
//   trsm_diag_inverses  batched inverses of op(A)'s diagonal blocks
//   logdet       2 sum log(Re x_i)  (reference lapack/dlogdet.cu:53-118)
#include "internal.h"
#include "tile16.h"
#include "publish.h"

#include <climits>

namespace hc {
namespace {

// L^H L kernel: 512 threads in groups of TPR per row.
constexpr int LAUUM_THREADS = 512;

template <typename T> __device__ __forceinline__ T shfl_xor_t(T v, int m);
template <> __device__ __forceinline__ double shfl_xor_t<double>(double v, int m) {
  return __shfl_xor(v, m, 64);
}
template <> __device__ __forceinline__ zd shfl_xor_t<zd>(zd v, int m) {
  return make_zd(__shfl_xor(v.x, m, 64), __shfl_xor(v.y, m, 64));
}

// Sum over groups of G consecutive lanes (G a power of two dividing 64).
template <int G, typename T>
__device__ __forceinline__ T group_sum(T v) {
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) v = v + shfl_xor_t(v, off);
  return v;
}

// Visits the n x n block at A (column-major, 1 <= n <= NMAX) as
// use(i, k, A(i, k)), i the contiguous index: thread t takes row t % NMAX of
// columns t / NMAX + j * (THREADS / NMAX), U loads in flight together from
// clamped (always valid) addresses.  Nothing divides by the runtime n: a
// 32-bit division is a ~40-instruction sequence here, and per-element
// divisions used to cost the diagonal-block kernels more than their loads.
template <int NMAX, int THREADS, int U, typename T, typename Use>
__device__ __forceinline__ void gather_block(int n, const T *A, long lda, Use use) {
  static_assert(THREADS % NMAX == 0, "whole rows per sweep");
  constexpr int STEP = THREADS / NMAX, PER = (NMAX + STEP - 1) / STEP;
  const int i = (int)threadIdx.x % NMAX, k0 = (int)threadIdx.x / NMAX;
  const int ic = min(i, n - 1);
#pragma unroll
  for (int j0 = 0; j0 < PER; j0 += U) {
    if (k0 + j0 * STEP >= n) break;
    T v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = A[(long)min(k0 + (j0 + u) * STEP, n - 1) * lda + ic];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + (j0 + u) * STEP;
      if (i < n && k < n) use(i, k, v[u]);
    }
  }
}

// fn(i, k) for every element of an n x n block, with the thread mapping of
// gather_block (stores to column-major memory stay contiguous across lanes).
template <int NMAX, int THREADS, typename Fn>
__device__ __forceinline__ void for_block(int n, Fn fn) {
  static_assert(THREADS % NMAX == 0, "whole rows per sweep");
  constexpr int STEP = THREADS / NMAX;
  const int i = (int)threadIdx.x % NMAX, k0 = (int)threadIdx.x / NMAX;
  if (i < n)
    for (int k = k0; k < n; k += STEP) fn(i, k);
}

// S is column-major with leading dimension NMAX + 1: S(r, c) = S[c * LS + r].
template <typename T, int NMAX>
struct Lds {
  static constexpr int LS = NMAX + 1;
  static constexpr int TPR = LAUUM_THREADS / NMAX;  // threads per row in sweeps
};

// Load the lower form of the n x n block at A: S(r, c) = A(r, c) (lower) or
// conj(A(c, r)) (upper), r >= c.  Memory is read along its contiguous index.
template <typename T, int NMAX, int THREADS, typename ST = T>
__device__ __forceinline__ void load_lower_form(T *S, bool lower, int n, const ST *A, long lda) {
  constexpr int LS = Lds<T, NMAX>::LS;
  // a: contiguous index in memory; the unreferenced triangle is read but not used
  gather_block<NMAX, THREADS, 16>(n, A, lda, [&](int a, int b, ST x) {
    const T v = convert<T>(x);
    if (lower) {
      if (a >= b) S[b * LS + a] = v;
    } else {
      // A(a, b) with a <= b is upper; it is conj of lower-form (b, a)
      if (a <= b) S[a * LS + b] = conjx(v);
    }
  });
}

// Store the lower form back into the caller's triangle (diagonal included
// unless skip_diag).
template <typename T, int NMAX, int THREADS, typename ST = T>
__device__ __forceinline__ void store_lower_form(const T *S, bool lower, int n, ST *A, long lda, bool skip_diag) {
  constexpr int LS = Lds<T, NMAX>::LS;
  for_block<NMAX, THREADS>(n, [&](int a, int b) {
    if (skip_diag && a == b) return;
    if (lower) {
      if (a >= b) A[(long)b * lda + a] = convert<ST>(S[b * LS + a]);
    } else {
      if (a <= b) A[(long)b * lda + a] = convert<ST>(conjx(S[a * LS + b]));
    }
  });
}

// In-place R = L^H L of the lower form (lower part), columns left to right:
// R(r, c) = sum_{k >= r} conj(L(k, r)) L(k, c).
template <typename T, int NMAX>
__device__ __forceinline__ void lds_lauum(T *S, int n) {
  constexpr int LS = Lds<T, NMAX>::LS, TPR = Lds<T, NMAX>::TPR;
  const int tid = threadIdx.x, row = tid / TPR, part = tid % TPR;
  for (int c = 0; c < n; c++) {
    const int r = c + row;
    T sum = from_real<T>(0.0);
    if (r < n)
      for (int k = r + part; k < n; k += TPR) sum = sum + conjx(S[r * LS + k]) * S[c * LS + k];
    sum = group_sum<TPR>(sum);
    // the diagonal of L^H L is real; fused rounding of conj(a) a may leave an
    // imaginary part of order eps |a|^2, which a Hermitian result must not carry
    if (r == c) sum = from_real<T>(realx(sum));
    __syncthreads();
    if (r < n && part == 0) S[c * LS + r] = sum;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Blocked factor + inverse of one diagonal block (diag_potrf).
//
// The block is split into 16-column leaves.  Leaf p is factored and inverted
// by one wave entirely in registers (leaf_factor_invert), so its 16
// sequential pivots need no workgroup barrier.  Everything else is 16 x 16 x 16 tile products on the
// matrix cores spread over the eight waves: the panel below the leaf
// (L_Ip = A_Ip inv(L_pp)^H), the trailing update (A_IJ -= L_Ip L_Jp^H), and
// the inverse X = inv(L) row block by row block as the factor's rows
// complete (X_IJ = -X_II sum_{K=J..I-1} L_IK X_KJ, from L X = I), formed by
// the waves that are not factoring the next leaf.  Two barriers per leaf.
// ---------------------------------------------------------------------------
using t16::LEAF;
using t16::TileAcc;
using t16::acc_zero;
using t16::acc_load;
using t16::acc_store;
using t16::acc_get;
using t16::acc_rank4_add;
using t16::acc_rank4_sub;
using t16::frag_load;
using t16::frag_rank4;
using t16::frag_store;
using t16::leaf_factor_invert;
using t16::tile_mma;
using t16::wave_lds_fence;

constexpr int BLK_THREADS = 512;

// LDS holds only the lower-triangle tiles, packed: tile (I, J), I >= J, at
// index I (I + 1) / 2 + J, each 16 x 16 column-major with leading dimension
// 17 (78 KB for a 128 x 128 real block), so the kernel fits beside a
// trailing-update workgroup on the same CU.  Once leaf p is factored its tile
// holds inv(L_pp); its factor has already gone to global memory.
// T is the compute type (the LDS copy), ST the storage type of A and W
// (float for the mixed-precision factorisation, which computes the diagonal
// blocks in double).
// One workgroup per launch, run beside the trailing update's workgroups
// (256 registers per wave, up to two per SIMD): with at most 128 registers per
// wave (WPE = 4 waves per SIMD) the real-type kernel fits next to one of them
// and starts at once; the complex one needs more registers and is left free.
template <typename T>
constexpr int diag_waves_per_eu() { return is_complex<T>::value ? 2 : 4; }

// Elements of LDS that the factorisation of a diagonal block of order NMAX
// uses: the packed tiles and a buffer for the leaf's factor.
template <int NMAX>
constexpr int diag_lds_elems() {
  constexpr int NP = NMAX / LEAF;
  return (NP * (NP + 1) / 2 + 1) * LEAF * (LEAF + 1);
}

// Factor and invert the lower-form block of order n whose tiles src delivers
// (src.load<LO, HI>(I, x): the stored values of tiles (I, LO .. HI-1);
// src.fix(x, r, c): the value of an element, identity beyond n) with S as
// workspace (`flag` an LDS word).  The factor goes to A (lower form: A(r, c),
// or conj into A(c, r) when !lower) and inv(L) to the lower tiles of W (ld ldw,
// n x n only, zeros above the diagonal of the diagonal tiles; with ZEROS also
// in the tiles above them).  Nothing is done when `failed`.  Returns -1,
// or the first non-positive / NaN pivot (0-based, the same value in every
// thread; the factor is then only partly written).
//
// Wave 0 factors the leaves; workers 0 .. NW-2 are the other waves.  Worker w
// holds tile row w + 2 of the trailing matrix in registers, as row fragments
// (at once matrix-core operands and results).  Step p, after leaf p:
//   phase A: wave 0 forms the panel tile (p+1, p), worker w >= p the panel tile
//     (w+2, p), L_Ip = A_Ip X_pp^H; worker J < p finishes tile J of row p of
//     X = inv(L), X_pJ = -X_pp S_pJ (L X = I row by row);
//   phase B: wave 0 updates tile (p+1, p+1) and factors leaf p + 1; worker
//     w >= p applies step p to its row, and the owner of row p + 2 hands tiles
//     (p+2, p+1) and (p+2, p+2) to wave 0 through LDS; worker J <= p forms
//     S_{p+1,J} = sum_{K=J..p} L_{p+1,K} X_KJ.  Tiles of L and X finished in
//     phase A are written to A and W here.
// The inverse is complete with the last leaf, with no pass of its own.  Step
// p = -1 only factors leaf 0 (one call site keeps the leaf inlined once).
//
// The time is the chain leaf -> panel tile (p+1, p) -> update of tile
// (p+1, p+1) -> leaf in wave 0, so that wave does nothing else, and wave 4, on
// the same SIMD, is worker 6, which has no row; the workers, at a lower issue
// priority, keep up with it because a row in registers leaves one LDS operand
// per product.  One CU takes about 10000 cycles to read the block from HBM
// (longer than two leaves): leaf 0 overlaps the left three quarters of the tile
// columns, leaf 1 the rest.  One 128 x 128 double block alone: 24.5 us between
// events, 19.8 us in a kernel trace (36 us between events with a column-by-column
// leaf in a layout of its own, the tiles in LDS, the write-out in wave 0 and the
// block loaded element by element).
template <typename T, typename ST, int NMAX, bool ZEROS, typename Src>
__device__ __forceinline__ int diag_block_factor(const Src &src, bool failed, T *S, int &flag, int lower, int n,
                                                 ST *A, long lda, ST *W, long ldw) {
  constexpr int NPMAX = NMAX / LEAF, LL = LEAF + 1, TS = LEAF * LL, NW = BLK_THREADS / 64;
  static_assert(NPMAX <= NW && NW == 8, "a worker per tile of a row of the inverse; wave 4 shares wave 0's SIMD");
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int np = (n + LEAF - 1) / LEAF;
  int lane = tid & 63;
  asm volatile("" : "+v"(lane));
  const int lc = lane & 15, lg = lane >> 4;
  auto tile = [&](int I, int J) { return S + (I * (I + 1) / 2 + J) * TS; };
  T *const Lbuf = S + NPMAX * (NPMAX + 1) / 2 * TS;  // L_pp
  // row fragments f of L_IJ to A, of X_IJ to W (entries above the diagonal of
  // a diagonal tile: not written, zero)
  auto put_a = [&](const TileAcc<T> &f, int I, int J) {
    const int r = I * LEAF + lc, c0 = J * LEAF + lg;
    if (r < n) {
      ST *a = lower ? A + (long)c0 * lda + r : A + (long)r * lda + c0;
      const long step = lower ? 4 * lda : 4;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (r >= c0 + 4 * j) *a = lower ? convert<ST>(acc_get(f, j)) : convert<ST>(conjx(acc_get(f, j)));
        a += step;
      }
    }
  };
  auto put_w = [&](const TileAcc<T> &f, int I, int J) {
    const int r = I * LEAF + lc, c0 = J * LEAF + lg;
    if (r < n) {
      ST *w = W + (long)c0 * ldw + r;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (c0 + 4 * j < n) *w = convert<ST>(acc_get(f, j));
        w += 4 * ldw;
      }
    }
  };
  // The two roles are disjoint code (the register budget is the larger of
  // them) with the same barriers: one after phase A, one after phase B.
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(3);  // issue ahead of the workers and of any other kernel's waves
    typename Src::V x0[NPMAX][4], x1[NPMAX][4];
    const bool row1 = np > 1;
    src.template load<0, 1>(0, x0);
    if (row1) src.template load<0, 2>(1, x1);
    if (failed) return -1;
    if (tid == 0) flag = -1;
    TileAcc<T> fd, fl;  // the diagonal tile to factor, panel tile (p+1, p)
#pragma unroll
    for (int j = 0; j < 4; j++) acc_set(fd, j, src.fix(x0[0][j], lc, lg + 4 * j));
    if (row1) {
#pragma unroll
      for (int J = 0; J < 2; J++) {
#pragma unroll
        for (int j = 0; j < 4; j++) acc_set(fl, j, src.fix(x1[J][j], LEAF + lc, J * LEAF + lg + 4 * j));
        frag_store(fl, tile(1, J), LL);
      }
    }
    for (int p = -1; p < np - 1; p++) {
      if (p >= 0) {
        TileAcc<T> xf, af;
        frag_load(xf, tile(p, p), LL);
        frag_load(af, tile(p + 1, p), LL);
        frag_load(fd, tile(p + 1, p + 1), LL);
        acc_zero(fl);
#pragma unroll
        for (int s = 0; s < 4; s++) frag_rank4<false>(fl, acc_get(af, s), acc_get(xf, s));
        frag_store(fl, tile(p + 1, p), LL);
#pragma unroll
        for (int s = 0; s < 4; s++) frag_rank4<true>(fd, acc_get(fl, s), acc_get(fl, s));
        __syncthreads();
      }
      T *const xt = tile(p + 1, p + 1) + lc * LL + lg, *const lt = Lbuf + lg * LL + lc;
      const int bad = leaf_factor_invert<T>(fd, [&](int r, T l, T x) {
        lt[4 * r * LL] = l;
        xt[4 * r] = x;
      });
      if (bad >= 0 && lane == 0) flag = (p + 1) * LEAF + bad;
      __syncthreads();
      if (bad >= 0) return (p + 1) * LEAF + bad;  // padding never fails, so this is below n
    }
    put_a(fd, np - 1, np - 1);
    frag_load(fl, tile(np - 1, np - 1), LL);
    put_w(fl, np - 1, np - 1);
    return -1;
  }

  __builtin_amdgcn_s_setprio(2);
  const int wk = wave == 4 ? NW - 2 : (wave < 4 ? wave - 1 : wave - 2);  // worker
  const int row = wk + 2 < np ? wk + 2 : -1;
  TileAcc<T> R[NPMAX];  // the worker's tile row
  constexpr int FIRST = NPMAX * 6 / 8;  // tile columns loaded beside leaf 0
  // its tiles LO .. HI - 1
  auto take = [&](auto lo, auto hi) __attribute__((always_inline)) {
    constexpr int LO = decltype(lo)::value, HI = decltype(hi)::value;
    typename Src::V x[NPMAX][4];
    src.template load<LO, HI>(row, x);
    if (failed) return;
    t16::static_for<LO, HI>([&](auto Jc) {
      constexpr int J = decltype(Jc)::value;
      if (J <= row) {
#pragma unroll
        for (int j = 0; j < 4; j++) acc_set(R[J], j, src.fix(x[J][j], row * LEAF + lc, J * LEAF + lg + 4 * j));
      }
    });
  };
  take(std::integral_constant<int, 0>{}, std::integral_constant<int, FIRST>{});
  if (failed) return -1;
  __syncthreads();
  TileAcc<T> sacc;  // S_{p+1,wk}, carried from phase B to the next phase A
  TileAcc<T> lp;    // the panel tile, or tile wk of row p of L
  acc_zero(sacc);
  int zi = -1, zj = 1;  // worker NW - 2: tile above the diagonal last zeroed in W
  // panel tile (row, J), J = p; worker NW - 2, which has no tile before the
  // last row, takes L_pp instead
  auto panel = [&](auto Jc) __attribute__((always_inline)) {
    constexpr int J = decltype(Jc)::value;
    TileAcc<T> xf, acc;
    frag_load(xf, tile(J, J), LL);
    acc_zero(acc);
#pragma unroll
    for (int s = 0; s < 4; s++) frag_rank4<false>(acc, acc_get(R[J], s), acc_get(xf, s));
    frag_store(acc, tile(row, J), LL);
    lp = acc;
  };
  if (row > 0) panel(std::integral_constant<int, 0>{});
  if (wk == NW - 2 && np > 1) frag_load(lp, Lbuf, LL);
  int bad = flag;  // of leaf p (padding never fails, so it is below n)
  if (bad >= 0) return bad;
  if (np > 1) __syncthreads();
  take(std::integral_constant<int, FIRST>{}, std::integral_constant<int, NPMAX>{});
  for (int p = 0;; p++) {
    // phase B of step p
    if (wk >= p && row > 0) {  // A_IJ -= L_Ip L_Jp^H, I = row
      t16::static_for<1, NPMAX>([&](auto Jc) {
        constexpr int J = decltype(Jc)::value;
        if (J > p && J <= row) {
          TileAcc<T> b = lp;
          if (J < row) frag_load(b, tile(J, p), LL);
#pragma unroll
          for (int s = 0; s < 4; s++) frag_rank4<true>(R[J], acc_get(lp, s), acc_get(b, s));
          if (row == p + 2) frag_store(R[J], tile(row, J), LL);
        }
      });
    } else if (wk < p || (wk == NW - 2 && p < np - 1)) {
      const int J = wk < p ? wk : p;
      put_a(lp, p, J);
      TileAcc<T> x;
      frag_load(x, tile(p, J), LL);
      put_w(x, p, J);
    }
    if (p == np - 1) return -1;
    if (ZEROS && wk == NW - 2) {  // zeros of W above the diagonal tiles: its NPMAX / 2 next ones
      for (int u = 0; u < NPMAX / 2; u++) {
        if (++zi >= zj) {
          zi = 0;
          zj++;
        }
        if (zj >= np) break;
        ST *w = W + (long)(zj * LEAF + lg) * ldw + zi * LEAF + lc;
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (zj * LEAF + lg + 4 * j < n) w[j * 4 * ldw] = convert<ST>(from_real<T>(0.0));
      }
    }
    if (wk <= p) {  // S_{p+1,wk}: row p + 1 of L is complete
      acc_zero(sacc);
      for (int K = wk; K <= p; K++) tile_mma<false>(sacc, tile(p + 1, K), LL, tile(K, wk), LL, 1.0);
    }
    __syncthreads();
    // phase A of step q
    const int q = p + 1;
    if (wk >= q && row > 0) {
      t16::static_for<1, NPMAX>([&](auto Jc) {
        if (decltype(Jc)::value == q) panel(Jc);
      });
    } else if (wk < q) {
      T *tqj = tile(q, wk);
      TileAcc<T> xf, acc;
      frag_load(xf, tile(q, q), LL);
      frag_load(lp, tqj, LL);
      acc_zero(acc);
#pragma unroll
      for (int s = 0; s < 4; s++) acc_rank4_sub(acc, acc_get(xf, s), acc_get(sacc, s));
      acc_store(acc, tqj, LL);
      wave_lds_fence();
    }
    if (wk == NW - 2 && q < np - 1) frag_load(lp, Lbuf, LL);
    bad = flag;
    if (bad >= 0) return bad;
    if (q < np - 1) __syncthreads();
  }
}

// Tiles of the n x n block at A in global memory, lower form.
template <typename T, typename ST>
struct GlobalTiles {
  using V = ST;
  const ST *A;
  long lda;
  int lower, n;
  // x[J][j] <- this lane's elements of tile (I, J), LO <= J < HI and J <= I
  // (row fragments), all loads in flight together; beyond n from a clamped
  // (always valid) address, selected away by fix.  A block of whole tiles
  // walks one pointer, without the clamps and 64-bit index products.
  template <int LO, int HI, int NP>
  __device__ __forceinline__ void load(int I, V (&x)[NP][4]) const {
    const int lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4, r = I * LEAF + lc;
    if (LO > I) return;
    if (n % LEAF == 0) {
      const ST *a = lower ? A + (long)(LO * LEAF + lg) * lda + r : A + (long)r * lda + LO * LEAF + lg;
      const long step = lower ? 4 * lda : 4;
      t16::static_for<LO, HI>([&](auto Jc) {
        constexpr int J = decltype(Jc)::value;
        if (J <= I) {
#pragma unroll
          for (int j = 0; j < 4; j++, a += step) x[J][j] = *a;
        }
      });
    } else {
      const int rc = min(r, n - 1);
      t16::static_for<LO, HI>([&](auto Jc) {
        constexpr int J = decltype(Jc)::value;
        if (J <= I) {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const int c = min(J * LEAF + lg + 4 * j, n - 1);
            x[J][j] = lower ? A[(long)c * lda + rc] : A[(long)rc * lda + c];
          }
        }
      });
    }
  }
  // the value of element (r, c) loaded as x, identity beyond n
  __device__ __forceinline__ T fix(ST x, int r, int c) const {
    const T v = lower ? convert<T>(x) : conjx(convert<T>(x));
    if (n % LEAF == 0) return v;
    return t16::sel(r < n && c < n, v, from_real<T>(r == c ? 1.0 : 0.0));
  }
};

template <typename T, typename ST, int NMAX>
__global__ void __launch_bounds__(BLK_THREADS)
__attribute__((amdgpu_waves_per_eu(diag_waves_per_eu<T>(), diag_waves_per_eu<T>())))
diag_potrf_kernel(int lower, int n, ST *A, long lda, ST *W, long ldw, int *info, long info_off) {
  __shared__ T S[diag_lds_elems<NMAX>()];
  __shared__ int flag;
  const int failed = *info;  // tested once the block's loads are issued
  const GlobalTiles<T, ST> src{A, lda, lower, n};
  const int bad = diag_block_factor<T, ST, NMAX, false>(src, failed != 0, S, flag, lower, n, A, lda, W, ldw);
  if (bad >= 0 && threadIdx.x == 0) *info = (int)(info_off + bad + 1);
}

// ---------------------------------------------------------------------------
// A whole panel of the blocked factorisation in one launch (lower, real):
// the m x jb panel at A, its top jb x jb block on the diagonal, becomes L,
// left-looking by 128-column blocks J = 0 .. C-1 (C = ceil(jb / 128)).
// The reference factors a panel as a chain of diagonal-block, panel-solve
// and panel-update calls (lapack/dpotrf.c:268-326); here one workgroup owns
// each 128-row block: row block b < C is the diagonal part (rows 128 b ..),
// row block b >= C the rows jb + 128 (b - C) .. below it.  For every column
// block J left of its rows, workgroup b
//   * once row block J has published its off-diagonal blocks L_Jk (k < J),
//     accumulates S = sum_{k<J} L_bk L_Jk^T (K = 128 J, its own L_bk
//     re-read from memory);
//   * once L_JJ and inv(L_JJ) are published, stores X = A_bJ - S in place and
//     then L_bJ = X inv(L_JJ)^T.
// A diagonal workgroup b then publishes its off-diagonal blocks, factors and
// inverts A_bb - sum_k L_bk L_bk^T with diag_block_factor (FP64 for FP32
// storage; the partial sum over k < b - 1 is formed ahead of the wait for
// block b - 1 and parked in the workspace) and publishes L_bb and inv(L_bb).
// The critical path per column block is one flag hand-off, two 128^3
// products and the diagonal block; the other workgroups' accumulations run
// while a diagonal block is factored.
//
// Dependencies only point to lower workgroup indices, which the hardware
// dispatches first, so every awaited workgroup is resident or finished.
// Flags are set to the launch's epoch (a per-handle counter, so they never
// need resetting); a wait gives up when the info word becomes nonzero (a
// failed pivot anywhere) or after about four seconds, which it reports as
// kInfoAbandoned.  Publishing: every wave waits for its own stores, then one
// wave writes the L2 back once and sets the flag; waiting: one wave polls,
// then acquires with one agent-scope fence before the workgroup barrier.
// ---------------------------------------------------------------------------
typedef float pv4f __attribute__((ext_vector_type(4)));
typedef double pv4d __attribute__((ext_vector_type(4)));
typedef double pv2d __attribute__((ext_vector_type(2)));

constexpr int PK_THREADS = 512;
constexpr int PK_B = 128;          // rows and columns of a block
constexpr int PK_FLAG_STRIDE = 32; // ints between flags (one 128-byte line each)

// Matrix-core arithmetic of the panel products per storage type: K step KT
// staged in LDS as rows of LK elements (K contiguous), a 16-byte fragment of
// FV consecutive k per lane, and the result column of register r in lane
// group g (the row is lane % 16).
template <typename ST> struct PanelMma;
template <> struct PanelMma<float> {
  using V = pv4f;
  using F = pv4f;
  static constexpr int KT = 32, LK = KT + 4, FV = 4;
  __device__ static V mma(float b, float a, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, c, 0, 0, 0); }
  __device__ static int col(int g, int r) { return 4 * g + r; }
};
template <> struct PanelMma<double> {
  using V = pv4d;
  using F = pv2d;
  static constexpr int KT = 16, LK = KT + 2, FV = 2;
  __device__ static V mma(double b, double a, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, c, 0, 0, 0); }
  __device__ static int col(int g, int r) { return g + 4 * r; }
};

// 128 x 128 accumulator of the workgroup: 8 waves in 2 x 4, each 64 x 32 as
// 4 x 2 blocks of 16 x 16.
template <typename ST> struct PanelAcc {
  typename PanelMma<ST>::V v[4][2];
  __device__ void zero() {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) v[i][j][r] = ST(0);
  }
  // element <- fn(row, col, element) over the thread's 32 elements
  template <typename Fn> __device__ void map(Fn fn) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // indices formed per call, not hoisted by the caller
    const int lane = tid & 63, wave = tid >> 6;
    const int lc = lane & 15, lg = lane >> 4, wm0 = (wave & 1) * 64, wn0 = (wave >> 1) * 32;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) v[i][j][r] = fn(wm0 + 16 * i + lc, wn0 + 16 * j + PanelMma<ST>::col(lg, r), v[i][j][r]);
  }
  // fn(row, col, C(row, col) - element) where ok(row, col), C(r, c) at
  // Cp[c * ldc + r]; C is read in two halves with all loads of a half in
  // flight before its results are used (fn may store into C)
  template <typename Ok, typename Fn> __device__ void sub_from(const ST *Cp, long ldc, Ok ok, Fn fn) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6;
    const int lc = lane & 15, lg = lane >> 4, wm0 = (wave & 1) * 64, wn0 = (wave >> 1) * 32;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      ST cv[16];
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int row = wm0 + 16 * (2 * h + i) + lc, col = wn0 + 16 * j + PanelMma<ST>::col(lg, r);
            cv[8 * i + 4 * j + r] = Cp[ok(row, col) ? (long)col * ldc + row : 0];
          }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int row = wm0 + 16 * (2 * h + i) + lc, col = wn0 + 16 * j + PanelMma<ST>::col(lg, r);
            fn(row, col, cv[8 * i + 4 * j + r] - v[2 * h + i][j][r]);
          }
    }
  }
};

// acc += P Q^T over k < K: P(r, k) = Pp[k * ldp + r] (r < rp), Q(c, k) =
// Qp[k * ldq + c] (c < rq); k >= klim reads as zero.  K is a multiple of KT.
// Both operands are staged through LDS (double-buffered, the next step's
// global loads in registers during this step's products); returns with the
// LDS free (after a barrier).
template <typename ST>
__device__ __forceinline__ void panel_nt(PanelAcc<ST> &acc, const ST *Pp, long ldp, int rp, const ST *Qp, long ldq,
                                         int rq, int K, int klim, ST *lds) {
  using M = PanelMma<ST>;
  constexpr int KT = M::KT, LK = M::LK, FV = M::FV, E = KT / 4;
  using F = typename M::F;
  ST *sP = lds, *sQ = lds + 2 * PK_B * LK;
  int tid = threadIdx.x;
  // thread-derived values (and the addresses built from them) are formed here
  // at every call, not hoisted out of the caller's loop and kept live across it
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = tid >> 6;
  const int lr = tid & (PK_B - 1), kq = tid >> 7;  // loader: row lr, k = kq E .. kq E + E - 1
  const int lc = lane & 15, lg = lane >> 4, wm0 = (wave & 1) * 64, wn0 = (wave >> 1) * 32;
  ST rp_[E], rq_[E];
  auto load = [&](int k0) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int k = k0 + kq * E + e;
      const bool okp = lr < rp && k < klim, okq = lr < rq && k < klim;
      const ST a = Pp[okp ? (long)k * ldp + lr : 0];
      const ST b = Qp[okq ? (long)k * ldq + lr : 0];
      rp_[e] = okp ? a : ST(0);
      rq_[e] = okq ? b : ST(0);
    }
  };
  auto store = [&](int buf) {
    ST *dp = sP + buf * PK_B * LK + lr * LK + kq * E, *dq = sQ + buf * PK_B * LK + lr * LK + kq * E;
#pragma unroll
    for (int e = 0; e < E; e += FV) {
      F a, b;
#pragma unroll
      for (int t = 0; t < FV; t++) { a[t] = rp_[e + t]; b[t] = rq_[e + t]; }
      *reinterpret_cast<F *>(dp + e) = a;
      *reinterpret_cast<F *>(dq + e) = b;
    }
  };
  const int nk = K / KT;
  load(0);
  store(0);
  __syncthreads();
  for (int kt = 0; kt < nk; kt++) {
    const bool more = kt + 1 < nk;
    if (more) load((kt + 1) * KT);
    const ST *cP = sP + (kt & 1) * PK_B * LK, *cQ = sQ + (kt & 1) * PK_B * LK;
#pragma unroll
    for (int h = 0; h < KT; h += 4 * FV) {
      F fp[4], fq[2];
#pragma unroll
      for (int i = 0; i < 4; i++) fp[i] = *reinterpret_cast<const F *>(cP + (wm0 + 16 * i + lc) * LK + h + FV * lg);
#pragma unroll
      for (int j = 0; j < 2; j++) fq[j] = *reinterpret_cast<const F *>(cQ + (wn0 + 16 * j + lc) * LK + h + FV * lg);
#pragma unroll
      for (int t = 0; t < FV; t++)
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc.v[i][j] = M::mma(fq[j][t], fp[i][t], acc.v[i][j]);
    }
    if (more) store((kt + 1) & 1);
    __syncthreads();
  }
}

// One wave polls flag f until it holds `epoch` (or info becomes nonzero, or
// the wait times out), then acquires; the result (true: proceed) is the
// same in every thread.
__device__ __forceinline__ bool panel_wait(const int *f, int epoch, int *info, int &sh) {
  if (threadIdx.x < 64) {
    int st = 0;
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
      const int v = __builtin_amdgcn_readfirstlane(__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      const int iv = __builtin_amdgcn_readfirstlane(__hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      if (iv != 0) { st = 2; break; }
      if (v == epoch) { st = 1; break; }
      if (__builtin_amdgcn_s_memrealtime() - t0 > 400000000ull) {  // ~4 s at 100 MHz
        if (threadIdx.x == 0) {
          int expected = 0;
          __hip_atomic_compare_exchange_strong(info, &expected, kInfoAbandoned, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
        }
        st = 2;
        break;
      }
      __builtin_amdgcn_s_sleep(2);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (threadIdx.x == 0) sh = st;
  }
  __syncthreads();
  return sh == 1;
}

__device__ __forceinline__ void panel_publish(int *f, int epoch) {
  publish_wait_own();
  __syncthreads();
  if (threadIdx.x < 64) {
    publish_release();
    if (threadIdx.x == 0) __hip_atomic_store(f, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <typename ST>
constexpr int panel_lds_bytes() {
  constexpr int g = 4 * PK_B * PanelMma<ST>::LK * (int)sizeof(ST);
  constexpr int d = diag_lds_elems<PK_B>() * (int)sizeof(double);
  return g > d ? g : d;
}

// The packed lower tiles in LDS as the source of diag_block_factor, which
// reads a tile before it overwrites it (each wave only the tiles it owns).
struct LdsTiles {
  using V = double;
  const double *S;
  template <int LO, int HI, int NP>
  __device__ __forceinline__ void load(int I, double (&x)[NP][4]) const {
    const int lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4;
    t16::static_for<LO, HI>([&](auto Jc) {
      constexpr int J = decltype(Jc)::value;
      if (J <= I) {
        const double *t = S + (I * (I + 1) / 2 + J) * LEAF * (LEAF + 1);
#pragma unroll
        for (int j = 0; j < 4; j++) x[J][j] = t[(lg + 4 * j) * (LEAF + 1) + lc];
      }
    });
  }
  __device__ double fix(double x, int, int) const { return x; }
};

// ws: C inverses inv(L_JJ) (128 x 128, ld 128), then C partial sums (128 x 128).
template <typename ST>
__global__ void __launch_bounds__(PK_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4)))
panel_potrf_kernel(int m, int jb, ST *A, long lda, ST *ws, int *flags, int epoch, int *info, long info_off) {
  using T = double;  // the diagonal blocks are factored in FP64 for both storage types
  if (*info != 0) return;
  __builtin_amdgcn_s_setprio(3);
  __shared__ __attribute__((aligned(16))) char lds_raw[panel_lds_bytes<ST>()];
  __shared__ int sh_wait, sh_flag;
  ST *lds = reinterpret_cast<ST *>(lds_raw);
  const int C = (jb + PK_B - 1) / PK_B, b = blockIdx.x;
  const bool dg = b < C;
  const int r0 = dg ? PK_B * b : jb + PK_B * (b - C);
  const int ra = dg ? min(PK_B, jb - r0) : min(PK_B, m - r0);
  const int nJ = dg ? b : C;
  constexpr long BB = (long)PK_B * PK_B;
  ST *Winv = ws, *Psum = ws + C * BB;
  int *const off_flag = flags, *const diag_flag = flags + PK_FLAG_STRIDE;
  auto fo = [&](int J) { return off_flag + 2 * PK_FLAG_STRIDE * J; };
  auto fd = [&](int J) { return diag_flag + 2 * PK_FLAG_STRIDE * J; };
  PanelAcc<ST> acc;
  for (int J = 0; J < nJ; J++) {
    const int cw = min(PK_B, jb - PK_B * J);
    ST *AbJ = A + (long)PK_B * J * lda + r0;
    if (dg && J == b - 1 && b >= 2) {  // P = sum_{k < b-1} L_bk L_bk^T (own rows, no wait)
      acc.zero();
      panel_nt<ST>(acc, A + r0, lda, ra, A + r0, lda, ra, PK_B * J, PK_B * J, lds);
      ST *P = Psum + b * BB;
      acc.map([&](int r, int c, ST x) { P[(long)c * PK_B + r] = x; return x; });
    }
    acc.zero();
    if (J > 0) {
      if (!panel_wait(fo(J), epoch, info, sh_wait)) return;
      panel_nt<ST>(acc, A + r0, lda, ra, A + PK_B * J, lda, cw, PK_B * J, PK_B * J, lds);
    }
    if (!panel_wait(fd(J), epoch, info, sh_wait)) return;
    // X = A_bJ - S in place (C and the sum kept apart: they nearly cancel)
    acc.sub_from(AbJ, lda, [&](int r, int c) { return r < ra && c < cw; }, [&](int r, int c, ST v) {
      if (r < ra && c < cw) AbJ[(long)c * lda + r] = v;
    });
    publish_wait_own();
    __syncthreads();
    // L_bJ = X inv(L_JJ)^T
    acc.zero();
    panel_nt<ST>(acc, AbJ, lda, ra, Winv + J * BB, PK_B, cw, PK_B, cw, lds);
    acc.map([&](int r, int c, ST x) {
      if (r < ra && c < cw) AbJ[(long)c * lda + r] = x;
      return x;
    });
    publish_wait_own();
    __syncthreads();
  }
  if (!dg) return;
  // the diagonal workgroup's row block left of the diagonal is final
  if (b > 0) panel_publish(fo(b), epoch);
  // A_bb - sum_{k<b} L_bk L_bk^T into the packed FP64 tiles
  ST *Abb = A + (long)r0 * lda + r0;
  acc.zero();
  if (b >= 2) {
    const ST *P = Psum + b * BB;
    acc.map([&](int r, int c, ST) { return P[(long)c * PK_B + r]; });
  }
  if (b >= 1) {
    const ST *Lp = A + (long)PK_B * (b - 1) * lda + r0;
    panel_nt<ST>(acc, Lp, lda, ra, Lp, lda, ra, PK_B, PK_B, lds);
  }
  {
    constexpr int LL = LEAF + 1, TS = LEAF * LL;
    T *S = reinterpret_cast<T *>(lds_raw);
    const int npad = (ra + LEAF - 1) / LEAF * LEAF;
    acc.sub_from(Abb, lda, [&](int r, int c) { return r < ra && c < ra && r >= c; }, [&](int r, int c, ST v) {
      if (r >= c && r < npad && c < npad) {
        T *tl = S + ((r / LEAF) * (r / LEAF + 1) / 2 + c / LEAF) * TS;
        tl[(c % LEAF) * LL + r % LEAF] = (r < ra && c < ra) ? convert<T>(v) : from_real<T>(r == c ? 1.0 : 0.0);
      }
    });
  }
  __syncthreads();
  T *const S = reinterpret_cast<T *>(lds_raw);
  const int bad = diag_block_factor<T, ST, PK_B, true>(LdsTiles{S}, false, S, sh_flag, 1, ra, Abb, lda,
                                                       Winv + b * BB, PK_B);
  if (bad >= 0) {
    if (threadIdx.x == 0) {
      int expected = 0;
      __hip_atomic_compare_exchange_strong(info, &expected, (int)(info_off + r0 + bad + 1), __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }
  panel_publish(fd(b), epoch);
}

// ---------------------------------------------------------------------------
// Triangular inverse of one block in LDS (packed lower tiles as above, lower
// form, unit diagonals stored as ones): the 16 x 16 diagonal tiles first, one
// wave each, then X = inv(L) by tile rows, S = sum_{J<=K<I} L_IK X_KJ and
// L_II X_IJ = -S, one wave per tile column J (it reads row I of L, which nobody
// needs after that, and its own column of X: one barrier per row).  The solve
// with L_II is Y = -X_II S corrected once, Y -= X_II (S + L_II Y), from a copy
// of L_II kept behind the tiles.
// The inverse takes the place of L in solves, so its residual L X - I has to be
// that of a substitution, whatever the grading of L.  Measured on the factor of
// a squared-exponential covariance (n = 128, length 0.05, nugget 1e-8), residual
// of the solve A x = b from both of its triangles: substitution element by
// element 5e-14, this 4e-14, without the correction 1e-12, joining inverted
// halves (X21 = -X22 L21 X11) 3e-13 (and 7e-11 in L X - I at nugget 1e-10).
// Waves w and w + 4 share a SIMD and take columns w and 7 - w, so that every
// matrix core has the same products.  40 blocks of 128 x 128 doubles in a launch:
// 20 us (108 us as a substitution by columns in registers, one barrier per
// column).
// ---------------------------------------------------------------------------
template <int NMAX>
constexpr int tri_lds_elems() {
  constexpr int NP = NMAX / LEAF;
  return (NP * (NP + 1) / 2 + NP) * LEAF * (LEAF + 1);
}

template <typename T, int NMAX>
__device__ __forceinline__ void tiles_invert(T *S, int np) {
  constexpr int NPMAX = NMAX / LEAF, LL = LEAF + 1, TS = LEAF * LL;
  static_assert(BLK_THREADS / 64 == 8 && NPMAX <= 8, "a wave per tile column");
  const int lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto tile = [&](int I, int J) { return S + (I * (I + 1) / 2 + J) * TS; };
  T *const Ld = S + NPMAX * (NPMAX + 1) / 2 * TS;  // L_II, zeros above the diagonal
  if (wave < np) {
    T a[LEAF], x[4], l[4];
    T *t = tile(wave, wave);
#pragma unroll
    for (int c = 0; c < LEAF; c++) a[c] = t[c * LL + lc];
#pragma unroll
    for (int j = 0; j < 4; j++) l[j] = t16::sel(lg + 4 * j <= lc, t[(lg + 4 * j) * LL + lc], from_real<T>(0.0));
    t16::leaf_inverse_cols<T>(a, x);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      t[(lg + 4 * j) * LL + lc] = x[j];
      Ld[wave * TS + (lg + 4 * j) * LL + lc] = l[j];
    }
  }
  __syncthreads();
  const int J = wave < 4 ? wave : 11 - wave;
  for (int I = 1; I < np; I++) {
    TileAcc<T> s, y, xf, lf;
    acc_zero(s);
    if (J < I)
      for (int K = J; K < I; K++) tile_mma<false>(s, tile(I, K), LL, tile(K, J), LL, 1.0);
    __syncthreads();
    if (J < I) {
      frag_load(xf, tile(I, I), LL);
      frag_load(lf, Ld + I * TS, LL);
      acc_zero(y);
#pragma unroll
      for (int q = 0; q < 4; q++) acc_rank4_sub(y, acc_get(xf, q), acc_get(s, q));
#pragma unroll
      for (int q = 0; q < 4; q++) acc_rank4_add(s, acc_get(lf, q), acc_get(y, q));
#pragma unroll
      for (int q = 0; q < 4; q++) acc_rank4_sub(y, acc_get(xf, q), acc_get(s, q));
      acc_store(y, tile(I, J), LL);
      wave_lds_fence();
    }
  }
  __syncthreads();
}

// Packed lower tiles of the n x n block at A: lower-form element (r, c) is
// A(r, c), or A(c, r) when swapped, conjugated when conj; identity beyond n,
// ones on the diagonal when unit.  Lanes run along memory's contiguous index.
template <typename T, typename ST, int NMAX>
__device__ __forceinline__ void tiles_load(T *S, int n, const ST *A, long lda, bool swapped, bool conj, bool unit) {
  constexpr int LL = LEAF + 1, TS = LEAF * LL, NW = BLK_THREADS / 64, NPMAX = NMAX / LEAF;
  constexpr int PER = (NPMAX * (NPMAX + 1) / 2 + NW - 1) / NW;
  const int lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), np = (n + LEAF - 1) / LEAF;
  int ti[PER], tj[PER];
  ST x[PER][4];
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int t = q * NW + wave;  // row by row
    int I = 0;
#pragma unroll
    for (int k = 1; k <= NPMAX; k++) I += t >= k * (k + 1) / 2 ? 1 : 0;
    ti[q] = I < np ? I : -1;
    tj[q] = I < np ? t - I * (I + 1) / 2 : 0;
    const int r = max(ti[q], 0) * LEAF + (swapped ? lg : lc), c = tj[q] * LEAF + (swapped ? lc : lg);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int rr = min(swapped ? r + 4 * j : r, n - 1), cc = min(swapped ? c : c + 4 * j, n - 1);
      x[q][j] = swapped ? A[(long)rr * lda + cc] : A[(long)cc * lda + rr];
    }
  }
#pragma unroll
  for (int q = 0; q < PER; q++) {
    if (ti[q] < 0) continue;
    T *t = S + (ti[q] * (ti[q] + 1) / 2 + tj[q]) * TS;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int rl = swapped ? lg + 4 * j : lc, cl = swapped ? lc : lg + 4 * j;
      const int r = ti[q] * LEAF + rl, c = tj[q] * LEAF + cl;
      const T v = conj ? conjx(convert<T>(x[q][j])) : convert<T>(x[q][j]);
      const T e = t16::sel(r < n && c < n, v, from_real<T>(r == c ? 1.0 : 0.0));
      t[cl * LL + rl] = t16::sel(unit && r == c, from_real<T>(1.0), e);
    }
  }
}

// fn(r, c, element) over the n x n lower-form elements r >= c held in S, or
// with DENSE over all of them (zero above the diagonal); lanes along r, or
// along c when swapped.
template <typename T, int NMAX, bool DENSE, typename Fn>
__device__ __forceinline__ void tiles_each(const T *S, int n, bool swapped, Fn fn) {
  constexpr int LL = LEAF + 1, TS = LEAF * LL, NW = BLK_THREADS / 64;
  const int lane = threadIdx.x & 63, lc = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), np = (n + LEAF - 1) / LEAF;
  int t = wave + 1;
  for (int I = 0; I < np; I++)
    for (int J = 0; J < (DENSE ? np : I + 1); J++) {
      if (--t != 0) continue;
      t = NW;
      const T *p = S + (I * (I + 1) / 2 + J) * TS;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int rl = swapped ? lg + 4 * j : lc, cl = swapped ? lc : lg + 4 * j;
        const int r = I * LEAF + rl, c = J * LEAF + cl;
        T v = from_real<T>(0.0);
        if (J <= I) v = p[cl * LL + rl];
        if (r < n && c < n && (DENSE || r >= c)) fn(r, c, v);
      }
    }
}

// Workgroup b inverts the diagonal block of order min(nb, ntot - b nb) at
// (b nb, b nb) of A into the same place of B (one workgroup: nb = ntot).
// T is the compute type, ST the storage type of A and B.
template <typename T, typename ST, int NMAX>
__global__ void __launch_bounds__(BLK_THREADS)
diag_trtri_kernel(int lower, int unit, int ntot, int nb, const ST *A, long lda, ST *B, long ldb,
                  const int *abort_flag) {
  if (abort_flag != nullptr && *abort_flag != 0) return;
  __shared__ T S[tri_lds_elems<NMAX>()];
  const long off = (long)blockIdx.x * nb;
  const int n = (int)min((long)nb, (long)ntot - off);
  A += off * lda + off;
  B += off * ldb + off;
  tiles_load<T, ST, NMAX>(S, n, A, lda, !lower, !lower, unit != 0);
  __syncthreads();
  tiles_invert<T, NMAX>(S, (n + LEAF - 1) / LEAF);
  tiles_each<T, NMAX, false>(S, n, !lower, [&](int r, int c, T v) {
    if (unit && r == c) return;
    if (lower) B[(long)c * ldb + r] = convert<ST>(v);
    else B[(long)r * ldb + c] = convert<ST>(conjx(v));
  });
}

// Workgroup b squares the diagonal block of order min(nb, ntot - b nb) at
// (b nb, b nb) of A into B + b bstride (ld ldb); one workgroup in place:
// nb = ntot, B = A, ldb = lda.
template <typename T, typename ST, int NMAX>
__global__ void __launch_bounds__(LAUUM_THREADS)
diag_lauum_kernel(int lower, int ntot, int nb, const ST *A, long lda, ST *B, long ldb, long bstride,
                  const int *abort_flag) {
  if (abort_flag != nullptr && *abort_flag != 0) return;
  __shared__ T S[NMAX * (NMAX + 1)];
  const long off = (long)blockIdx.x * nb;
  const int n = (int)min((long)nb, (long)ntot - off);
  load_lower_form<T, NMAX, LAUUM_THREADS, ST>(S, lower, n, A + off * lda + off, lda);
  __syncthreads();
  lds_lauum<T, NMAX>(S, n);
  store_lower_form<T, NMAX, LAUUM_THREADS, ST>(S, lower, n, B + blockIdx.x * bstride, ldb, false);
}

// D <- S on the triangle uplo (diagonal included) of an n x n matrix, a
// 64 x 64 tile per workgroup
template <typename T>
__global__ void __launch_bounds__(256) tri_copy_kernel(int lower, int n, const T *S, long lds, T *D, long ldd,
                                                       const int *abort_flag) {
  if (abort_flag != nullptr && *abort_flag != 0) return;
  const int bi = blockIdx.x, bj = blockIdx.y;
  if (lower ? bi < bj : bi > bj) return;
  const int r = bi * 64 + (threadIdx.x & 63), c0 = bj * 64 + (threadIdx.x >> 6);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    T v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = S[(long)min(c0 + 4 * (8 * h + j), n - 1) * lds + min(r, n - 1)];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int c = c0 + 4 * (8 * h + j);
      if (r < n && c < n && (lower ? r >= c : r <= c)) D[(long)c * ldd + r] = v[j];
    }
  }
}

// Block b inverts the nb x nb diagonal block of op(A) starting at b * nb.
template <typename T, typename ST, int NMAX>
__global__ void __launch_bounds__(BLK_THREADS)
trsm_inv_kernel(int lowerlike, int op, int unit, long m, int nb, const ST *A, long lda, ST *W) {
  __shared__ T S[tri_lds_elems<NMAX>()];
  const long off = (long)blockIdx.x * nb;
  const int n = (int)((m - off) < nb ? (m - off) : nb);
  // lower form: op(A)(r, c) when op(A) is lower-like, else conj(op(A)(c, r));
  // op(A)(i, j) = A(i, j), A(j, i) or conj(A(j, i)).
  const bool swapped = (op == OP_N) != (lowerlike != 0);
  const bool conj = op == OP_N ? lowerlike == 0 : (op == OP_C) == (lowerlike != 0);
  tiles_load<T, ST, NMAX>(S, n, A + off * lda + off, lda, swapped, conj, unit != 0);
  __syncthreads();
  tiles_invert<T, NMAX>(S, (n + LEAF - 1) / LEAF);
  ST *w = W + (long)blockIdx.x * nb * nb;
  tiles_each<T, NMAX, true>(S, n, lowerlike == 0, [&](int r, int c, T v) {
    if (lowerlike) w[(long)c * nb + r] = convert<ST>(v);
    else w[(long)r * nb + c] = convert<ST>(conjx(v));
  });
}

// One workgroup scans the diagonal; info = first (upper) or last (lower)
// 1-based index of an exact zero, 0 when none.
template <typename T>
__global__ void __launch_bounds__(1024) zero_scan_kernel(int lower, long n, const T *A, long lda, int *info) {
  __shared__ int best[1024];
  int b = lower ? 0 : INT_MAX;
  for (long i = threadIdx.x; i < n; i += 1024) {
    if (is_zero(A[i * lda + i])) {
      const int v = (int)(i + 1);
      b = lower ? (v > b ? v : b) : (v < b ? v : b);
    }
  }
  best[threadIdx.x] = b;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      const int o = best[threadIdx.x + s], c = best[threadIdx.x];
      best[threadIdx.x] = lower ? (o > c ? o : c) : (o < c ? o : c);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *info = (best[0] == INT_MAX) ? 0 : best[0];
}

// ---- compensated (double-double) summation of logs ----
struct dd {
  double hi, lo;
};
__device__ __forceinline__ dd dd_add(dd a, dd b) {
  const double s = a.hi + b.hi;
  const double bb = s - a.hi;
  const double e = (a.hi - (s - bb)) + (b.hi - bb) + a.lo + b.lo;
  dd r;
  r.hi = s + e;
  r.lo = e - (r.hi - s);
  return r;
}
__device__ __forceinline__ dd dd_shfl_xor(dd v, int m) {
  dd r;
  r.hi = __shfl_xor(v.hi, m, 64);
  r.lo = __shfl_xor(v.lo, m, 64);
  return r;
}
__device__ dd block_sum(dd v) {
  __shared__ double part[2 * 16];
  for (int off = 32; off > 0; off >>= 1) v = dd_add(v, dd_shfl_xor(v, off));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 0) { part[2 * wave] = v.hi; part[2 * wave + 1] = v.lo; }
  __syncthreads();
  dd t = {0.0, 0.0};
  if (threadIdx.x == 0)
    for (int w = 0; w < nw; w++) t = dd_add(t, dd{part[2 * w], part[2 * w + 1]});
  return t;
}

template <typename T>
__global__ void __launch_bounds__(256) logdet_partial_kernel(const T *x, long incx, long n, double *partials) {
  dd acc = {0.0, 0.0};
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    acc = dd_add(acc, dd{log(realx(x[i * incx])), 0.0});
  const dd t = block_sum(acc);
  if (threadIdx.x == 0) { partials[2 * blockIdx.x] = t.hi; partials[2 * blockIdx.x + 1] = t.lo; }
}

__global__ void __launch_bounds__(256) logdet_final_kernel(const double *partials, int nblocks, double *out) {
  dd acc = {0.0, 0.0};
  for (int b = threadIdx.x; b < nblocks; b += blockDim.x)
    acc = dd_add(acc, dd{partials[2 * b], partials[2 * b + 1]});
  const dd t = block_sum(acc);
  if (threadIdx.x == 0) out[0] = 2.0 * (t.hi + t.lo);
}

}  // namespace

// Compute type of the diagonal-block kernels for a storage type.
template <typename ST> struct Compute { using type = ST; };
template <> struct Compute<float> { using type = double; };
template <> struct Compute<zf> { using type = zd; };

template <typename ST>
hipError_t diag_potrf(hipStream_t s, char uplo, int n, ST *A, long lda, ST *W, long ldw, int *info,
                      long info_off) {
  using T = typename Compute<ST>::type;
  constexpr int NMAX = diag_max<T>();
  if (n <= 0) return hipSuccess;
  if (n > NMAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((diag_potrf_kernel<T, ST, NMAX>), dim3(1), dim3(BLK_THREADS), 0, s,
                     uplo == 'L' ? 1 : 0, n, A, lda, W, ldw, info, info_off);
  return hipGetLastError();
}

template <typename ST>
hipError_t diag_trtri(hipStream_t s, char uplo, char diag, int n, const ST *A, long lda, ST *B, long ldb,
                      const int *abort_flag) {
  using T = typename Compute<ST>::type;
  constexpr int NMAX = diag_max<T>();
  if (n <= 0) return hipSuccess;
  if (n > NMAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((diag_trtri_kernel<T, ST, NMAX>), dim3(1), dim3(BLK_THREADS), 0, s, uplo == 'L' ? 1 : 0,
                     diag == 'U' ? 1 : 0, n, n, A, lda, B, ldb, abort_flag);
  return hipGetLastError();
}

template <typename ST>
hipError_t diag_trtri_blocks(hipStream_t s, char uplo, char diag, long n, int nb, ST *A, long lda,
                             const int *abort_flag) {
  using T = typename Compute<ST>::type;
  constexpr int NMAX = diag_max<T>();
  if (n <= 0) return hipSuccess;
  if (nb <= 0 || nb > NMAX || n > (long)INT32_MAX) return hipErrorInvalidValue;
  const long blocks = (n + nb - 1) / nb;
  hipLaunchKernelGGL((diag_trtri_kernel<T, ST, NMAX>), dim3((unsigned)blocks), dim3(BLK_THREADS), 0, s,
                     uplo == 'L' ? 1 : 0, diag == 'U' ? 1 : 0, (int)n, nb, static_cast<const ST *>(A), lda, A, lda,
                     abort_flag);
  return hipGetLastError();
}

template <typename ST>
hipError_t diag_lauum(hipStream_t s, char uplo, int n, ST *A, long lda, const int *abort_flag) {
  using T = typename Compute<ST>::type;
  constexpr int NMAX = diag_max<T>();
  if (n <= 0) return hipSuccess;
  if (n > NMAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((diag_lauum_kernel<T, ST, NMAX>), dim3(1), dim3(LAUUM_THREADS), 0, s,
                     uplo == 'L' ? 1 : 0, n, n, static_cast<const ST *>(A), lda, A, lda, 0L, abort_flag);
  return hipGetLastError();
}

template <typename ST>
hipError_t diag_lauum_blocks(hipStream_t s, char uplo, long n, int nb, const ST *A, long lda, ST *W,
                             const int *abort_flag) {
  using T = typename Compute<ST>::type;
  constexpr int NMAX = diag_max<T>();
  if (n <= 0) return hipSuccess;
  if (nb <= 0 || nb > NMAX || n > (long)INT32_MAX) return hipErrorInvalidValue;
  const long blocks = (n + nb - 1) / nb;
  hipLaunchKernelGGL((diag_lauum_kernel<T, ST, NMAX>), dim3((unsigned)blocks), dim3(LAUUM_THREADS), 0, s,
                     uplo == 'L' ? 1 : 0, (int)n, nb, A, lda, W, (long)nb, (long)nb * nb, abort_flag);
  return hipGetLastError();
}

template <typename T>
hipError_t tri_copy(hipStream_t s, char uplo, long n, const T *S, long lds, T *D, long ldd, const int *abort_flag) {
  if (n <= 0) return hipSuccess;
  const unsigned t = (unsigned)((n + 63) / 64);
  hipLaunchKernelGGL((tri_copy_kernel<T>), dim3(t, t), dim3(256), 0, s, uplo == 'L' ? 1 : 0, (int)n, S, lds, D, ldd,
                     abort_flag);
  return hipGetLastError();
}

template <typename ST>
hipError_t trsm_diag_inverses(hipStream_t s, char uplo, char trans, char diag, long m, int nb,
                              const ST *A, long lda, ST *W) {
  using T = typename Compute<ST>::type;
  constexpr int NMAX = diag_max<T>();
  if (m <= 0) return hipSuccess;
  if (nb > NMAX) return hipErrorInvalidValue;
  const int op = is_complex<T>::value ? op_code(trans) : (trans == 'N' ? OP_N : OP_T);
  const int lowerlike = ((uplo == 'L') == (trans == 'N')) ? 1 : 0;
  const unsigned nblk = (unsigned)((m + nb - 1) / nb);
  hipLaunchKernelGGL((trsm_inv_kernel<T, ST, NMAX>), dim3(nblk), dim3(BLK_THREADS), 0, s, lowerlike,
                     op, diag == 'U' ? 1 : 0, m, nb, A, lda, W);
  return hipGetLastError();
}

template <typename T>
hipError_t diag_zero_scan(hipStream_t s, char uplo, long n, const T *A, long lda, int *info) {
  hipLaunchKernelGGL((zero_scan_kernel<T>), dim3(1), dim3(1024), 0, s, uplo == 'L' ? 1 : 0, n, A,
                     lda, info);
  return hipGetLastError();
}

template <typename T>
hipError_t logdet(hipStream_t s, const T *x, long incx, long n, double *partials, double *out) {
  long blocks = (n + 255) / 256;
  if (blocks > kLogdetMaxBlocks) blocks = kLogdetMaxBlocks;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL((logdet_partial_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, s, x, incx,
                     n, partials);
  HC_TRY(hipGetLastError());
  hipLaunchKernelGGL(logdet_final_kernel, dim3(1), dim3(256), 0, s, partials, (int)blocks, out);
  return hipGetLastError();
}

template <typename ST>
hipError_t panel_potrf(hipStream_t s, long m, long jb, ST *A, long lda, ST *ws, int *flags, int epoch, int *info,
                       long info_off) {
  if (jb <= 0) return hipSuccess;
  if (jb > kPanelMaxCols || m < jb || m > (long)INT32_MAX) return hipErrorInvalidValue;
  const long C = (jb + PK_B - 1) / PK_B, grid = C + (m - jb + PK_B - 1) / PK_B;
  hipLaunchKernelGGL((panel_potrf_kernel<ST>), dim3((unsigned)grid), dim3(PK_THREADS), 0, s, (int)m, (int)jb, A,
                     lda, ws, flags, epoch, info, info_off);
  return hipGetLastError();
}
template hipError_t panel_potrf<float>(hipStream_t, long, long, float *, long, float *, int *, int, int *, long);
template hipError_t panel_potrf<double>(hipStream_t, long, long, double *, long, double *, int *, int, int *,
                                        long);

#define HC_INST(T)                                                                            \
  template hipError_t diag_potrf<T>(hipStream_t, char, int, T *, long, T *, long, int *, long); \
  template hipError_t diag_trtri<T>(hipStream_t, char, char, int, const T *, long, T *, long,   \
                                    const int *);                                               \
  template hipError_t diag_trtri_blocks<T>(hipStream_t, char, char, long, int, T *, long,       \
                                           const int *);                                        \
  template hipError_t tri_copy<T>(hipStream_t, char, long, const T *, long, T *, long,          \
                                  const int *);                                                 \
  template hipError_t trsm_diag_inverses<T>(hipStream_t, char, char, char, long, int,           \
                                            const T *, long, T *);                              \
  template hipError_t diag_zero_scan<T>(hipStream_t, char, long, const T *, long, int *);       \
  template hipError_t logdet<T>(hipStream_t, const T *, long, long, double *, double *);
// single / single-complex storage: computed in double / double complex
// (the mixed-precision factorisation and the s / c routines); the
// log-determinants take their logs in FP64
HC_INST(double)
HC_INST(zd)
HC_INST(float)
HC_INST(zf)
#undef HC_INST
// squares of single-precision diagonal blocks (formed in double)
#define HC_INST_SQ(T)                                                                              \
  template hipError_t diag_lauum<T>(hipStream_t, char, int, T *, long, const int *);               \
  template hipError_t diag_lauum_blocks<T>(hipStream_t, char, long, int, const T *, long, T *, const int *);
HC_INST_SQ(float)
HC_INST_SQ(zf)
#undef HC_INST_SQ

}  // namespace hc
