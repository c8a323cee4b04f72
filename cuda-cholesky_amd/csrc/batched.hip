// Batched Cholesky factorisation + log-determinant of many small SPD
// matrices of uneven sizes, packed contiguously (matrix i: n_i x n_i,
// column-major with leading dimension n_i, at element offset off_i).
//
// Persistent kernels, one per size class: workgroup w of G takes matrices
// order[w], order[w + G], ... (`order` lists the matrices by decreasing n, so
// the round-robin deal is a longest-first schedule).  The factorisation and the
// inverse of the factor are separate kernels, both with the whole triangle in
// registers.
// Storage is FP64 or FP32 (ST); arithmetic is FP64 throughout.  Only the
// referenced triangle (uplo) is read or written; tiles reaching past n read
// the identity and are not written back.
#include <algorithm>

#include "internal.h"
#include "tile16.h"

namespace hc {
namespace {

using t16::LEAF;
using t16::TileAcc;
using t16::kNegA;

constexpr int LL = LEAF + 1;                   // LDS tile leading dimension

// Lower-form view of one packed matrix: element (r, c), r >= c, is A(r, c)
// for lower storage and A(c, r) for upper storage.
template <typename ST, bool LOWER>
struct View {
  ST *M;
  int n;
  __device__ long off(int r, int c) const { return LOWER ? (long)c * n + r : (long)r * n + c; }
  // value of lower-form (r, c): zero above the diagonal, identity beyond n.
  // The load is unconditional, from a clamped (always valid) address, and the
  // value is selected afterwards: no branch per element, so loads stay in
  // flight together and register arrays filled from them stay in registers.
  __device__ double get(int r, int c) const { return fix(raw(r, c), r, c); }
  // the two halves of get: the load from the clamped address, and the select
  __device__ double raw(int r, int c) const { return (double)M[off(min(r, n - 1), min(c, n - 1))]; }
  __device__ double fix(double x, int r, int c) const {
    return (r < n && c < n) ? (r >= c ? x : 0.0) : (r == c ? 1.0 : 0.0);
  }
  __device__ void put(int r, int c, double v) const {
    if (r < n && c < n && r >= c) M[off(r, c)] = (ST)v;
  }
};

// ---------------------------------------------------------------------------
// Register-resident factorisation (factor + log-determinant, no inverse).
//
// One workgroup factors one matrix (n <= 16 NPMAX) at a time and holds the
// matrix's whole lower tile triangle in registers, so that its HBM traffic is
// one read of the triangle and one write of L.  The critical path of a
// matrix is its chain of 16-column leaves: leaf p + 1 needs tile (p + 1, p + 1)
// after its update with panel tile (p + 1, p), which needs inv(L_pp) from
// leaf p.  The roles are cut so that nothing else lies on that chain:
//   * the leaf wave (the last) holds no tiles: it waits (LDS flag `dready`)
//     for tile (D, D), factors and inverts leaf D, records its pivots (their
//     logs are taken once per matrix, off the chain), publishes inv(L_DD)
//     (flag `lready`) and waits for the next tile.  It takes part in no
//     barrier inside a matrix;
//   * the NW - 1 tile waves hold every tile.  The sub-diagonal tile
//     (J + 1, J) and the diagonal tile (J + 1, J + 1) are in the same wave,
//     (J + 1) % (NW - 1): at step p that wave forms its panel tile (p + 1, p)
//     first, updates tile (p + 1, p + 1) with it straight from registers and
//     hands it to the leaf wave before it forms its other panel tiles, so leaf
//     p + 1 starts one panel tile and one update after leaf p has finished.
//     The other off-diagonal tiles follow round-robin: in the sequence g =
//     0, 1, ... of the np - 1 sub-diagonal tiles (g: tile (g + 1, g)) and then
//     the tiles I >= J + 2 column by column, tile g is in wave
//     (g + 1) % (NW - 1), slot g / (NW - 1) (np = ceil(n / 16)).  Diagonal tile
//     (J, J) is in wave J % (NW - 1), diagonal slot J / (NW - 1).
// A tile is held as T = A_IJ^T in the MFMA result layout (lane l, register
// r: T(l / 16 + 4 r, l % 16) = A_IJ(l % 16, l / 16 + 4 r)), which is also the
// operand fragment of A_IJ for k-step r: tiles enter the matrix cores with no
// layout change.  Per step p, in the tile waves:
//   wait for inv(L_pp) (flag `lready`);
//   panel:    T_Ip <- inv(L_pp) T_Ip = L_Ip^T (I > p), to LDS buffer p % 2
//             (element (row, k) at P_I[k LL + row]) and to the matrix;
//   tile-wave barrier (an LDS counter: the leaf wave is not held);
//   trailing: T_IJ -= L_Jp L_Ip^T (p < J <= I, (p + 1, p + 1) excepted).
// The panel buffers, inv(L_pp) and the hand-off tile alternate or are
// consumed before they are written again: P and inv(L) by step parity, the
// hand-off tile (D, D) is read by the leaf wave before leaf D publishes, and
// the next hand-off waits for that.  Every wait is bounded (4 s of the
// 100 MHz real-time counter); an abandoned one makes the matrix report
// info = -1.
// ---------------------------------------------------------------------------
typedef double v4d __attribute__((ext_vector_type(4)));

// The slot code (I | J << 8, or -1) of slot s, read from lane s of `codes`
// into a scalar register.  The empty asm makes it opaque, so that nothing
// derived from it is hoisted out of the step loop and kept live per slot.
__device__ __forceinline__ int slot_code(int codes, int s) {
  int c = __builtin_amdgcn_readlane(codes, s);
  asm volatile("" : "+s"(c));
  return c;
}

// T -= L_J L_I^T with the panel tiles L_I, L_J in LDS (P_I, P_J); lo is the
// lane's fragment offset at k-step 0.  The minus sign is the instruction's
// negate-A modifier, not a VALU negation of each operand.
__device__ __forceinline__ void tile_update(v4d &T, const double *PI, const double *PJ, int lo) {
#pragma unroll
  for (int r = 0; r < 4; r++)
    T = __builtin_amdgcn_mfma_f64_16x16x4f64(PJ[r * 4 * LL + lo], PI[r * 4 * LL + lo], T, 0, 0, kNegA);
}

// The leaf wave's step: factor the leaf at g0 held in f (row fragments), write
// L_pp to the matrix, 1 / L_rr to rpiv[g0 + r] and inv(L_pp)
// to Li; returns the failing pivot's column (g0 + k) or -1.
template <typename ST, bool LOWER>
__device__ __forceinline__ int leaf_step_piv(TileAcc<double> &f, const View<ST, LOWER> &v, int g0, double *Li,
                                             double *rpiv) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int b = t16::leaf_factor_invert<double>(f, [&](int r, double, double x) {
    Li[li * LL + lk + 4 * r] = x;
    if (lk + 4 * r == li) rpiv[g0 + li] = x;  // X(r, r) = 1 / L_rr (rpiv has whole leaves)
  });
  if (b >= 0) return g0 + b;
#pragma unroll
  for (int r = 0; r < 4; r++) v.put(g0 + li, g0 + lk + 4 * r, f.re[r]);
  return -1;
}

// Size classes of the register-resident kernel, by tile rows np (order n):
//   0: np <= 4  (n <= 64):  2 waves, 3 waves per SIMD (6 workgroups per CU);
//   1: np <= 8  (n <= 128): 4 waves, 3 waves per SIMD (3 workgroups per CU);
//   2: np <= 16 (n <= 256): 8 waves, 2 waves per SIMD (1 workgroup per CU).
// More workgroups per CU for the small classes overlap more leaf chains.
template <int CLS>
struct RegClass;
template <>
struct RegClass<0> {
  static constexpr int NPMAX = 4, NW = 2, OCC = 3;
};
template <>
struct RegClass<1> {
  static constexpr int NPMAX = 8, NW = 4, OCC = 3;
};
template <>
struct RegClass<2> {
  static constexpr int NPMAX = 16, NW = 8, OCC = 2;
};

// Bounded wait of a whole wave until `pred()` holds (4 s of the 100 MHz
// real-time counter); false when abandoned.
template <typename F>
__device__ __forceinline__ bool wave_wait(F pred) {
  if (pred()) return true;
  const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
  while (!pred()) {
    __builtin_amdgcn_s_sleep(1);
    if (__builtin_amdgcn_s_memrealtime() - t0 > 400000000ull) return false;
  }
  return true;
}

__device__ __forceinline__ int lds_acquire(const int *f) {
  return __builtin_amdgcn_readfirstlane(__hip_atomic_load(f, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
}

// cnt[c]: matrices of class c; `order` lists class 2, then 1, then 0.
template <typename ST, bool LOWER, int CLS, int NPMAX = RegClass<CLS>::NPMAX, int NW = RegClass<CLS>::NW,
          int OCC = RegClass<CLS>::OCC>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(OCC, 8)))
potrf_batched_reg_kernel(const int *cnt, const int *nvec, const long *offs, const int *order, ST *A,
                         double *logdet, int *info) {
  const int count = cnt[CLS];
  order += CLS == 2 ? 0 : (CLS == 1 ? cnt[2] : cnt[2] + cnt[1]);
  constexpr int NWT = NW - 1;                                            // tile waves
  constexpr int NO = NPMAX * (NPMAX - 1) / 2, S = (NO + NWT - 1) / NWT;  // off-diagonal tiles, slots
  constexpr int SD = (NPMAX + NWT - 1) / NWT;                           // diagonal slots
  constexpr int PB = NPMAX * LEAF * LL;                                 // one panel buffer
  static_assert(S <= 64, "slot codes live in one lane each");
  __shared__ double P[2 * PB];           // panel tiles L_Ip, by step parity
  __shared__ double Li[2 * LEAF * LL];   // inv(L_pp), by step parity
  __shared__ double Dg[LEAF * LL];       // tile (D, D) on its way to the leaf wave
  __shared__ double rpiv[NPMAX * LEAF];  // 1 / L_rr
  __shared__ double red[NW];
  // flag: failing column, -1 (none) or -2 (the leaf wave abandoned a wait);
  // fleaf: the leaf that failed (set once, before lready; a large value
  // while none has), so that every tile wave decides at the same step;
  // dready: D once tile (D, D) is in Dg; lready: D once leaf D is done;
  // tbar: tile-wave barrier arrivals; werr: a tile wave abandoned a wait
  __shared__ int flag, fleaf, dready, lready, tbar, werr;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int lo = lk * LL + li;  // this lane's operand fragment in an LDS tile (k-step 0)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid == 0) {
    flag = -1;
    fleaf = 1 << 30;
    dready = -1;
    lready = -1;
    tbar = 0;
    werr = 0;
  }
  __syncthreads();
  for (int t = blockIdx.x; t < count; t += gridDim.x) {
    const int idx = order[t];
    const int n = nvec[idx];
    const View<ST, LOWER> v{A + offs[idx], n};
    if (n == 0) {
      // nothing to load: the clamped addresses below assume n >= 1
      if (tid == 0) {
        info[idx] = 0;
        if (logdet != nullptr) logdet[idx] = 0.0;
      }
      continue;
    }
    const int np = (n + LEAF - 1) / LEAF;
    if (wave == NWT) {
      // ---- leaf wave ----
      for (int D = 0; D < np; D++) {
        int b = -2;
        if (wave_wait([&] { return lds_acquire(&dready) == D; })) {
          TileAcc<double> f;
          t16::frag_load(f, Dg, LL);
          b = leaf_step_piv<ST, LOWER>(f, v, D * LEAF, Li + (D & 1) * LEAF * LL, rpiv);
        }
        if (lane == 0) {
          if (b != -1) {
            flag = b;
            fleaf = D;
          }
          __hip_atomic_store(&lready, D, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        if (b != -1) break;
      }
    } else {
      // ---- tile waves ----
      const int no = np * (np - 1) / 2;
      int codes = -1;  // lane s < S: the code of this wave's off-diagonal slot s
      {
        const int g = (wave + NWT - 1) % NWT + NWT * lane;
        if (lane < S && g < no) {
          if (g < np - 1) {
            codes = (g + 1) | (g << 8);  // sub-diagonal tile (g + 1, g)
          } else {
            int k = g - (np - 1), J = 0;  // k-th tile with I >= J + 2, column by column
            while (k >= np - 2 - J) {
              k -= np - 2 - J;
              J++;
            }
            codes = (J + 2 + k) | (J << 8);
          }
        }
      }
      v4d T[S], Td[SD];
      // every load is in flight before the first select, and each select
      // overwrites its own load (no second register set); a slot without a
      // tile loads tile (0, 0) and never uses it (no branch)
      t16::static_for<0, S>([&](auto Sc) {
        constexpr int s = decltype(Sc)::value;
        const int c = max(slot_code(codes, s), 0);
        const int I = c & 255, J = c >> 8;
#pragma unroll
        for (int r = 0; r < 4; r++) T[s][r] = v.raw(I * LEAF + li, J * LEAF + lk + 4 * r);
      });
#pragma unroll
      for (int q = 0; q < SD; q++) {
        const int J = min(q * NWT + wave, np - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) Td[q][r] = v.raw(J * LEAF + li, J * LEAF + lk + 4 * r);
      }
      t16::static_for<0, S>([&](auto Sc) {
        constexpr int s = decltype(Sc)::value;
        const int c = max(slot_code(codes, s), 0);
        const int I = c & 255, J = c >> 8;
#pragma unroll
        for (int r = 0; r < 4; r++) T[s][r] = v.fix(T[s][r], I * LEAF + li, J * LEAF + lk + 4 * r);
      });
#pragma unroll
      for (int q = 0; q < SD; q++) {
        const int J = min(q * NWT + wave, np - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) Td[q][r] = v.fix(Td[q][r], J * LEAF + li, J * LEAF + lk + 4 * r);
      }
      if (wave == 0) {  // tile (0, 0) to the leaf wave
#pragma unroll
        for (int r = 0; r < 4; r++) Dg[r * 4 * LL + lo] = Td[0][r];  // A_00(li, lk + 4 r)
        if (lane == 0) __hip_atomic_store(&dready, 0, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      // the last column has no panel tiles and no trailing update
      for (int p = 0; p + 1 < np; p++) {
        const int D = p + 1;
        if (!wave_wait([&] { return lds_acquire(&lready) >= p; })) {
          if (lane == 0) werr = 1;
          break;
        }
        // leaf p failed (a later leaf may already have failed too: the
        // decision is made on the step, the same in every tile wave)
        if (fleaf <= p) break;
        const double *Lp = Li + (p & 1) * LEAF * LL;
        double *Pp = P + (p & 1) * PB;
        // panel of column p: T_Ip <- inv(L_pp) T_Ip, to LDS and to the
        // matrix; the sub-diagonal tile (D, p) comes first (lowest slot), and
        // its owner updates tile (D, D) with it and hands that over at once
        // this lane's fragments of inv(L_pp), read once for the wave's panel
        // tiles in the largest class (the smaller ones have no registers
        // to spare and re-read them)
        double lf[4];
#pragma unroll
        for (int r = 0; r < 4; r++) lf[r] = CLS == 2 ? Lp[r * 4 * LL + lo] : 0.0;
        t16::static_for<0, S>([&](auto Sc) {
          constexpr int s = decltype(Sc)::value;
          const int c = slot_code(codes, s);
          if (c >= 0 && (c >> 8) == p) {
            v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int r = 0; r < 4; r++)
              acc = __builtin_amdgcn_mfma_f64_16x16x4f64(CLS == 2 ? lf[r] : Lp[r * 4 * LL + lo], T[s][r], acc, 0, 0, 0);
            T[s] = acc;
            const int I = c & 255;
            if (I == D) {
              // tile (D, D) -= L_Dp L_Dp^T: acc[r] is the operand fragment of
              // L_Dp for k-step r, on both sides
#pragma unroll
              for (int q = 0; q < SD; q++)
                if (q == D / NWT) {
#pragma unroll
                  for (int r = 0; r < 4; r++)
                    Td[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(acc[r], acc[r], Td[q], 0, 0, kNegA);
#pragma unroll
                  for (int r = 0; r < 4; r++) Dg[r * 4 * LL + lo] = Td[q][r];  // A_DD(li, lk + 4 r)
                }
              if (lane == 0) __hip_atomic_store(&dready, D, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            double *Pt = Pp + I * LEAF * LL;
#pragma unroll
            for (int r = 0; r < 4; r++) {
              Pt[r * 4 * LL + lo] = acc[r];
              v.put(I * LEAF + li, p * LEAF + lk + 4 * r, acc[r]);  // L_Ip(li, lk + 4 r)
            }
          }
        });
        // tile-wave barrier: every panel tile of column p is in LDS
        if (lane == 0) __hip_atomic_fetch_add(&tbar, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (!wave_wait([&] { return lds_acquire(&tbar) >= NWT * D; })) {
          if (lane == 0) werr = 1;
          break;
        }
        // the other trailing tiles
#pragma unroll
        for (int q = 0; q < SD; q++) {
          const int J = q * NWT + wave;
          if (J > D && J < np) tile_update(Td[q], Pp + J * LEAF * LL, Pp + J * LEAF * LL, lo);
        }
        t16::static_for<0, S>([&](auto Sc) {
          constexpr int s = decltype(Sc)::value;
          const int c = slot_code(codes, s);
          if (c >= 0 && (c >> 8) > p) tile_update(T[s], Pp + (c & 255) * LEAF * LL, Pp + (c >> 8) * LEAF * LL, lo);
        });
      }
    }
    __syncthreads();  // the leaf wave is done: flag, rpiv and werr are final
    const int fl = flag;
    // bad: failing column, -1 (none) or -2 (a wait was abandoned)
    const int bad = fl != -1 ? fl : (werr != 0 ? -2 : -1);
    // log-determinant: 2 sum log L_rr = -2 sum log(1 / L_rr), one pivot per thread
    double lg = 0.0;
    if (bad == -1)
      for (int r = tid; r < n; r += NW * 64) lg -= log(rpiv[r]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lg += __shfl_xor(lg, off, 64);
    if (lane == 0) red[wave] = lg;
    __syncthreads();
    if (tid == 0) {
      double sum = 0.0;
      for (int w = 0; w < NW; w++) sum += red[w];
      info[idx] = bad >= 0 ? bad + 1 : (bad == -2 ? -1 : 0);
      if (logdet != nullptr) logdet[idx] = bad != -1 ? __builtin_nan("") : 2.0 * sum;
      // every wave is past its last use of the flags
      flag = -1;
      fleaf = 1 << 30;
      dready = -1;
      lready = -1;
      tbar = 0;
      werr = 0;
    }
    __syncthreads();  // flags, rpiv and LDS tiles are reused by the next matrix
  }
}

// ---------------------------------------------------------------------------
// Register-resident inverse of factored matrices (info = 0): A^-1 = X^T X,
// X = inv(L), in place over the factor.
//
// np = ceil(n / 16) tile rows and columns; wave w of NPMAX / 2 owns first rows
// np - 1 - w and w of X, then columns w and np - 1 - w of the result (np + 1
// tiles together, equal work), held in registers in the matrix-core result
// layout (rows: transposed), which is also the operand layout of the second
// factor of every product here, so a tile never moves between lanes.
//   * the waves invert the diagonal leaves into LDS;
//   * each wave forms its rows right to left, X_IJ = -(sum_{J<K<=I} X_IK L_KJ)
//     X_JJ, with the tiles of L read from the matrix as operand fragments: no
//     exchange between waves.  k runs as 4 lk + s there, so that in lower
//     storage a lane's four elements are one load, and so are its four of X;
//   * the rows go to LDS, or for n > 128, where the triangle does not fit it,
//     replace L in the matrix; the waves read their columns of X back and form
//     their columns of the result, R_ij = sum_{K>=i} X_Ki^T X_Kj, i ascending,
//     with X_Ki from there too; R_ij takes the registers of X_ij, which no later
//     i needs;
//   * R replaces L or X in the matrix.
// X by rows has a small X L - I, which is what A X^T X - I needs.  By columns
// (X_IJ = -X_II sum L_IK X_KJ, small L X - I) the columns would stay where they
// are, but the residual of the inverse on graded factors is 30 to 500 times
// larger: squared-exponential covariances, nugget 1e-8, ||A R - I|| / (||A||
// ||R||) 3e-15 by rows, 2e-12 by columns at n = 128.
// Factor and inverse of 20000 matrices, n in [8, 256]: FP32 storage 6.4 ms
// (upper 6.6), of which the factor 2.4 (2.6), FP64 7.9 ms (8.2); by columns 7.5
// (7.0) and 7.8 ms (9.2); a 4-wave workgroup that streams every tile of a matrix
// through memory at every step 9.8 (8.4) and 11.1 ms (10.8).  10000 matrices, n in
// [65, 128], FP64: X in LDS 2.45 ms, through the matrix 2.94 ms.  The fully
// unrolled tile products are more code than the instruction cache holds, but
// rolled loops over K spilled 200 to 800 registers (rows and columns are indexed
// at compile time).
// ---------------------------------------------------------------------------
template <typename ST, bool LOWER, int CLS, int NPMAX = RegClass<CLS>::NPMAX>
__global__ void __launch_bounds__(NPMAX / 2 * 64) __attribute__((amdgpu_waves_per_eu(CLS == 0 ? 3 : 2, 8)))
potri_batched_reg_kernel(const int *cnt, const int *nvec, const long *offs, const int *order, ST *A,
                         const int *info) {
  constexpr int NWI = NPMAX / 2;
  const int count = cnt[CLS];
  order += CLS == 2 ? 0 : (CLS == 1 ? cnt[2] : cnt[2] + cnt[1]);
  constexpr bool XL = CLS < 2;             // X below the diagonal tiles in LDS
  __shared__ double D[NPMAX * LEAF * LL];  // X_II
  __shared__ double XB[XL ? NPMAX * (NPMAX - 1) / 2 * LEAF * LL : 1];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto xtile = [&](int I, int J) { return XB + (I * (I - 1) / 2 + J) * LEAF * LL; };  // I > J
  for (int t = blockIdx.x; t < count; t += gridDim.x) {
    const int idx = __builtin_amdgcn_readfirstlane(order[t]);
    const int n = __builtin_amdgcn_readfirstlane(nvec[idx]);
    if (n == 0 || __builtin_amdgcn_readfirstlane(info[idx]) != 0) continue;
    const View<ST, LOWER> v{A + offs[idx], n};
    const int np = (n + LEAF - 1) / LEAF;
    for (int I = wave; I < np; I += NWI) {
      double a[LEAF], x[4];
      t16::static_for<0, LEAF>([&](auto C) { a[decltype(C)::value] = v.get(I * LEAF + li, I * LEAF + decltype(C)::value); });
      t16::leaf_inverse_cols<double>(a, x);
#pragma unroll
      for (int j = 0; j < 4; j++) D[I * LEAF * LL + (lk + 4 * j) * LL + li] = x[j];
    }
    __syncthreads();
    // lane offsets in a tile: elements (row li, column lk) and (row lk, column li)
    const unsigned ol = LOWER ? lk * n + li : li * n + lk, ox = LOWER ? li * n + lk : lk * n + li;
    const int rstep = LOWER ? 4 : 4 * n, cstep = LOWER ? 4 * n : 4;  // four rows, four columns on
    auto tile_at = [&](int I, int J) { return v.M + (LOWER ? (long)J * LEAF * n + I * LEAF : (long)I * LEAF * n + J * LEAF); };
    // elements (row lk + 4 s, column li) of tile (K, J), the operand fragment of
    // its transpose: a whole tile, or one with rows beyond n, which are zero
    auto load_t = [&](int K, int J, auto &l) __attribute__((always_inline)) {
      const ST *p = tile_at(K, J);
#pragma unroll
      for (int s = 0; s < 4; s++) l[s] = (double)p[s * rstep + ox];
    };
    auto load_edge = [&](int K, int J, auto &l) __attribute__((always_inline)) {
      const ST *p = tile_at(K, J);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const bool ok = K * LEAF + lk + 4 * s < n;
        const double x = (double)p[ok ? s * rstep + ox : 0u];
        l[s] = ok ? x : 0.0;
      }
    };
    // in the matrix, a tile of X that is whole (all but a ragged last tile row) and
    // that lies along columns in memory is kept transposed, so that the loads of
    // X_Ki^T below run along memory; X_JJ stays in LDS
    auto transposed = [&](int I) { return LOWER && (I + 1) * LEAF <= n; };
    auto load_x = [&](int K, int J, auto &l) __attribute__((always_inline)) {
      if constexpr (XL) {
        const double *p = xtile(K, J) + li * LL + lk;
#pragma unroll
        for (int s = 0; s < 4; s++) l[s] = p[4 * s];
        return;
      }
      if (transposed(K)) {
        const ST *p = tile_at(K, J);
#pragma unroll
        for (int s = 0; s < 4; s++) l[s] = (double)p[s * cstep + ol];
      } else if (!LOWER && (K + 1) * LEAF <= n) {
        load_t(K, J, l);
      } else {
        load_edge(K, J, l);
      }
    };
    // rows 4 lk .. 4 lk + 3 of column li of tile (K, J) of L, contiguous in lower
    // storage: the operand fragment of its transpose for products whose k runs
    // as 4 lk + s; rows beyond n are zero
    typedef ST row4 __attribute__((ext_vector_type(4), aligned(sizeof(ST))));
    const unsigned of = LOWER ? li * n + 4 * lk : 4 * lk * n + li;
    const int fstep = LOWER ? 1 : n;
    auto load_l = [&](int K, int J, auto &l) __attribute__((always_inline)) {
      const ST *p = tile_at(K, J) + of;
      if (LOWER) {
        const row4 x = *reinterpret_cast<const row4 *>(p);
#pragma unroll
        for (int s = 0; s < 4; s++) l[s] = (double)x[s];
      } else {
#pragma unroll
        for (int s = 0; s < 4; s++) l[s] = (double)p[s * fstep];
      }
    };
    auto load_l_edge = [&](int K, int J, auto &l) __attribute__((always_inline)) {
      const ST *p = tile_at(K, J);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const bool ok = K * LEAF + 4 * lk + s < n;
        const double x = (double)p[ok ? of + s * fstep : 0u];
        l[s] = ok ? x : 0.0;
      }
    };
    v4d Z[NPMAX + 1];  // the long row or column: its tile t from the diagonal at t; the short one: at NPMAX - t
    const int lp = 4 * (li & 3) + (li >> 2);  // rows of a result in the order 4 lk + r: from operand rows in this order
    auto sections = [&](int longer, int shorter, auto fn) __attribute__((always_inline)) {
      if (2 * wave < np) fn(std::integral_constant<int, 0>{}, longer);
      if (2 * wave + 1 < np) fn(std::integral_constant<int, 1>{}, shorter);
    };
    auto rows = [&](auto fn) __attribute__((always_inline)) { sections(np - 1 - wave, wave, fn); };
    auto columns = [&](auto fn) __attribute__((always_inline)) { sections(wave, np - 1 - wave, fn); };
    rows([&](auto Sec, int I) __attribute__((always_inline)) {
      constexpr int sec = decltype(Sec)::value, TM = sec ? NPMAX / 2 : NPMAX;
      auto at = [](int u) { return sec ? NPMAX - u : u; };
#pragma unroll
      for (int r = 0; r < 4; r++) Z[at(0)][r] = D[I * LEAF * LL + (4 * lk + r) * LL + li];
      t16::static_for<1, TM>([&](auto Dc) {
        constexpr int d = decltype(Dc)::value;
        if (d > I) return;
        const int J = I - d;
        v4d S = {0.0, 0.0, 0.0, 0.0}, acc = {0.0, 0.0, 0.0, 0.0};
        t16::static_for<0, d>([&](auto Uc) {  // K = I - u
          constexpr int u = decltype(Uc)::value;
          double l[4];
          if (u == 0 && I == np - 1) load_l_edge(I, J, l);
          else load_l(I - u, J, l);
#pragma unroll
          for (int s = 0; s < 4; s++) S = __builtin_amdgcn_mfma_f64_16x16x4f64(l[s], Z[at(u)][s], S, 0, 0, 0);
        });
#pragma unroll
        for (int s = 0; s < 4; s++)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(D[J * LEAF * LL + lp * LL + lk + 4 * s], S[s], acc, 0, 0, kNegA);
        Z[at(d)] = acc;
      });
    });
    if (!XL) __syncthreads();  // every read of L is done
    rows([&](auto Sec, int I) __attribute__((always_inline)) {
      constexpr int sec = decltype(Sec)::value, TM = sec ? NPMAX / 2 : NPMAX;
      t16::static_for<1, TM>([&](auto Dc) {
        constexpr int d = decltype(Dc)::value;
        if (d > I) return;
        const int J = I - d;
        const v4d &z = Z[sec ? NPMAX - d : d];
        if constexpr (XL) {
#pragma unroll
          for (int r = 0; r < 4; r++) xtile(I, J)[(4 * lk + r) * LL + li] = z[r];
          return;
        }
        // X(li, 4 lk + r): along memory in upper storage, and in lower storage where the tile is transposed
        if ((I + 1) * LEAF <= n) {
          const row4 x = {(ST)z[0], (ST)z[1], (ST)z[2], (ST)z[3]};
          *reinterpret_cast<row4 *>(tile_at(I, J) + li * n + 4 * lk) = x;
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++) v.put(I * LEAF + li, J * LEAF + 4 * lk + r, z[r]);
        }
      });
    });
    __syncthreads();
    columns([&](auto Sec, int J) __attribute__((always_inline)) {
      constexpr int sec = decltype(Sec)::value, TM = sec ? NPMAX / 2 : NPMAX;
      auto at = [](int u) { return sec ? NPMAX - u : u; };
#pragma unroll
      for (int r = 0; r < 4; r++) Z[at(0)][r] = D[J * LEAF * LL + li * LL + lk + 4 * r];
      t16::static_for<1, TM>([&](auto Dc) {
        constexpr int d = decltype(Dc)::value;
        if (J + d < np) load_x(J + d, J, Z[at(d)]);
      });
    });
    columns([&](auto Sec, int J) __attribute__((always_inline)) {
      constexpr int sec = decltype(Sec)::value, TM = sec ? NPMAX / 2 : NPMAX;
      auto at = [](int u) { return sec ? NPMAX - u : u; };
      t16::static_for<0, TM>([&](auto Dc) {
        constexpr int d = decltype(Dc)::value;
        if (J + d >= np) return;
        const int i = J + d;
        v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; s++)  // K = i
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(D[i * LEAF * LL + li * LL + lk + 4 * s], Z[at(d)][s], acc, 0, 0, 0);
        t16::static_for<d + 1, TM>([&](auto Uc) {
          constexpr int u = decltype(Uc)::value;
          if (J + u >= np) return;
          double l[4];
          load_x(J + u, i, l);
#pragma unroll
          for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(l[s], Z[at(u)][s], acc, 0, 0, 0);
        });
        Z[at(d)] = acc;
      });
    });
    __syncthreads();  // every read of X is done
    columns([&](auto Sec, int J) __attribute__((always_inline)) {
      constexpr int sec = decltype(Sec)::value, TM = sec ? NPMAX / 2 : NPMAX;
      t16::static_for<0, TM>([&](auto Dc) {
        constexpr int d = decltype(Dc)::value;
        if (J + d >= np) return;
#pragma unroll
        for (int r = 0; r < 4; r++) v.put((J + d) * LEAF + lk + 4 * r, J * LEAF + li, Z[sec ? NPMAX - d : d][r]);
      });
    });
  }
}

template <typename ST, bool LOWER, int CLS>
constexpr auto reg_kernel_ptr() {
  return potrf_batched_reg_kernel<ST, LOWER, CLS>;
}

template <typename ST, bool LOWER, int CLS>
void reg_launch(hipStream_t s, int grid, const int *cnt, const int *nvec, const long *offs, const int *order, ST *A,
                double *logdet, int *info) {
  hipLaunchKernelGGL((reg_kernel_ptr<ST, LOWER, CLS>()), dim3((unsigned)std::max(1, grid)),
                     dim3(RegClass<CLS>::NW * 64), 0, s, cnt, nvec, offs, order, A, logdet, info);
}

template <typename ST, bool LOWER, int CLS>
constexpr auto inv_kernel_ptr() {
  return potri_batched_reg_kernel<ST, LOWER, CLS>;
}

template <typename ST, bool LOWER, int CLS>
void inv_launch(hipStream_t s, int grid, const int *cnt, const int *nvec, const long *offs, const int *order, ST *A,
                const int *info) {
  hipLaunchKernelGGL((inv_kernel_ptr<ST, LOWER, CLS>()), dim3((unsigned)std::max(1, grid)),
                     dim3(RegClass<CLS>::NPMAX / 2 * 64), 0, s, cnt, nvec, offs, order, A, info);
}

template <typename ST, bool LOWER, int CLS>
int inv_occupancy() {
  int nb = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, inv_kernel_ptr<ST, LOWER, CLS>(),
                                                                    RegClass<CLS>::NPMAX / 2 * 64, 0);
  return (e == hipSuccess && nb > 0) ? nb : 1;
}

template <typename ST, bool LOWER, int CLS>
int reg_occupancy() {
  int nb = 0;
  const hipError_t e =
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reg_kernel_ptr<ST, LOWER, CLS>(), RegClass<CLS>::NW * 64, 0);
  return (e == hipSuccess && nb > 0) ? nb : 1;
}

}  // namespace

template <typename ST>
hipError_t potrf_batched_reg(hipStream_t s, char uplo, const int *d_cnt, const int *h_cnt, const int grid[3],
                             const int *nvec, const long *offs, const int *order, ST *A, double *logdet, int *info) {
  for (int c = 2; c >= 0; c--) {
    if (h_cnt != nullptr && h_cnt[c] == 0) continue;
    const int g = h_cnt != nullptr ? std::min(grid[c], h_cnt[c]) : grid[c];
    if (uplo == 'L') {
      if (c == 2) reg_launch<ST, true, 2>(s, g, d_cnt, nvec, offs, order, A, logdet, info);
      else if (c == 1) reg_launch<ST, true, 1>(s, g, d_cnt, nvec, offs, order, A, logdet, info);
      else reg_launch<ST, true, 0>(s, g, d_cnt, nvec, offs, order, A, logdet, info);
    } else {
      if (c == 2) reg_launch<ST, false, 2>(s, g, d_cnt, nvec, offs, order, A, logdet, info);
      else if (c == 1) reg_launch<ST, false, 1>(s, g, d_cnt, nvec, offs, order, A, logdet, info);
      else reg_launch<ST, false, 0>(s, g, d_cnt, nvec, offs, order, A, logdet, info);
    }
    HC_TRY(hipGetLastError());
  }
  return hipSuccess;
}

template <typename ST>
int potrf_batched_reg_blocks_per_cu(char uplo, int cls) {
  if (uplo == 'L') return cls == 2 ? reg_occupancy<ST, true, 2>() : (cls == 1 ? reg_occupancy<ST, true, 1>() : reg_occupancy<ST, true, 0>());
  return cls == 2 ? reg_occupancy<ST, false, 2>() : (cls == 1 ? reg_occupancy<ST, false, 1>() : reg_occupancy<ST, false, 0>());
}

template int potrf_batched_reg_blocks_per_cu<double>(char, int);
template int potrf_batched_reg_blocks_per_cu<float>(char, int);
template hipError_t potrf_batched_reg<double>(hipStream_t, char, const int *, const int *, const int *,
                                              const int *, const long *, const int *, double *, double *, int *);
template hipError_t potrf_batched_reg<float>(hipStream_t, char, const int *, const int *, const int *,
                                             const int *, const long *, const int *, float *, double *, int *);

template <typename ST>
hipError_t potri_batched_reg(hipStream_t s, char uplo, const int *d_cnt, const int *h_cnt, const int grid[3],
                             const int *nvec, const long *offs, const int *order, ST *A, const int *info) {
  for (int c = 2; c >= 0; c--) {
    if (h_cnt[c] == 0) continue;
    const int g = std::min(grid[c], h_cnt[c]);
    if (uplo == 'L') {
      if (c == 2) inv_launch<ST, true, 2>(s, g, d_cnt, nvec, offs, order, A, info);
      else if (c == 1) inv_launch<ST, true, 1>(s, g, d_cnt, nvec, offs, order, A, info);
      else inv_launch<ST, true, 0>(s, g, d_cnt, nvec, offs, order, A, info);
    } else {
      if (c == 2) inv_launch<ST, false, 2>(s, g, d_cnt, nvec, offs, order, A, info);
      else if (c == 1) inv_launch<ST, false, 1>(s, g, d_cnt, nvec, offs, order, A, info);
      else inv_launch<ST, false, 0>(s, g, d_cnt, nvec, offs, order, A, info);
    }
    HC_TRY(hipGetLastError());
  }
  return hipSuccess;
}

template <typename ST>
int potri_batched_reg_blocks_per_cu(char uplo, int cls) {
  if (uplo == 'L') return cls == 2 ? inv_occupancy<ST, true, 2>() : (cls == 1 ? inv_occupancy<ST, true, 1>() : inv_occupancy<ST, true, 0>());
  return cls == 2 ? inv_occupancy<ST, false, 2>() : (cls == 1 ? inv_occupancy<ST, false, 1>() : inv_occupancy<ST, false, 0>());
}

template int potri_batched_reg_blocks_per_cu<double>(char, int);
template int potri_batched_reg_blocks_per_cu<float>(char, int);
template hipError_t potri_batched_reg<double>(hipStream_t, char, const int *, const int *, const int *, const int *,
                                              const long *, const int *, double *, const int *);
template hipError_t potri_batched_reg<float>(hipStream_t, char, const int *, const int *, const int *, const int *,
                                             const long *, const int *, float *, const int *);

}  // namespace hc
