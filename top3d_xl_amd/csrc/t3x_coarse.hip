// Coarsest-level direct solver of libt3x (Solving_AssembleFEAstencil chol,
// TOP3D_XL.m:1052-1065, and the triangular solves of Solving_Vcycle, 767).
//
// The coarsest Galerkin matrix is banded after an axis-permuted node order
// (bandwidth bw).  The reference factors it with CHOLMOD; here:
//
//  1. right-looking blocked banded Cholesky, 64-column panels, one launch per
//     panel: every work-group of the trailing update solves the panel tiles
//     it needs (X = A L_JJ^{-T}, blocked by 16 columns on the matrix cores
//     with the inverses of L_JJ's 16x16 diagonal blocks) and applies its
//     X_I X_K^T update on the matrix cores; the group owning the next
//     diagonal tile then factors it (register/readlane POTRF), so the only
//     serial chain per panel is that tile's pivots.  Solved panel tiles go
//     to a scratch panel and reach the band in the next launch (the band's
//     A(I, J) is still being read during the current one).  The 64x64 tile
//     inverses for the solves are formed afterwards, in parallel.
//  2. k_trsm_blocks / k_h_blocks: the band is cut into solve blocks of SB >=
//     bw rows, so each block couples only to its predecessor:
//        forward   y_b = Dinv_b v_b - G_b y_{b-1},   G_b = Dinv_b L_{b,b-1}
//        backward  x_b = Dinv_b^T y_b - H_b x_{b+1}, H_b = Dinv_b^T L_{b+1,b}^T
//     Dinv_b, G_b come from one batched blocked TRSM on [I | L_{b,b-1}],
//     H_b from a batched GEMM.
//  3. the two recurrences in one or two launches whose work-groups hand the
//     blocks on entry by entry, or as a chain of 2*nblk+1 small launches,
//     instead of one dependent step per 64 rows.
//
// Everything else synchronises at kernel boundaries: on MI355X a device-wide
// barrier inside a kernel (cooperative grid sync, or fences that write back the
// per-XCD L2) costs more than a dependent launch (~3 us).
//
// All arithmetic is FP64.  Rows beyond the true size are identity rows.
#include <hip/hip_runtime.h>

#include "t3x_coarse.h"
#include "t3x_kernels.h"
#include "t3x_reduce.h"

#include <algorithm>

namespace t3x {

constexpr int TB = 64;      // tile size
constexpr int CT = 256;     // threads per work-group

struct BandView {
  double* B;  // row-major band: L(i, i-k) at B[i*W + k]
  int n;      // padded order
  int bw;
  __device__ __forceinline__ int W() const { return bw + 1; }
  __device__ __forceinline__ bool in(int i, int k) const { return i >= k && i - k <= bw && i < n && k >= 0; }
  // branch-free: the address is clamped into the band so loads can be batched
  __device__ __forceinline__ double get(int i, int k) const {
    const int d = i - k;
    const bool ok = (d >= 0) & (d <= bw) & (i < n) & (k >= 0);
    const size_t idx = (size_t)min(max(i, 0), n - 1) * W() + min(max(d, 0), bw);
    const double v = B[idx];
    return ok ? v : 0.0;
  }
  __device__ __forceinline__ void set(int i, int k, double v) const {
    if (in(i, k)) B[(size_t)i * W() + (i - k)] = v;
  }
};

// ---- 64x64 tile helpers in LDS -----------------------------------------
__device__ __forceinline__ double readlane_d(double v, int l) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

// 1/sqrt(x) for a positive normal x: the hardware estimate and one Newton
// step (relative error below 1e-16 after the step; a factored 64x64 tile
// reproduces its matrix to 1.4e-15)
__device__ __forceinline__ double rsqrt_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double h = fma(-x * y, y, 1.0);  // 1 - x y^2
  return fma(y * h, 0.5, y);
}

typedef double cd4 __attribute__((ext_vector_type(4)));

// LDS traffic between the lanes of one wave: the hardware keeps a wave's LDS
// operations in order; this keeps the compiler from moving a lane's load over
// another lane's store (by its own addresses alone the two may be disjoint).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int PW = 8;          // waves of a factorisation work-group
constexpr int FT = 64 * PW;    // its threads

// Inverse of the 16x16 diagonal block b of the lower-triangular sL into
// sD[b], by one wave: lane c (< 16) one column, forward substitution with
// independent updates after each step; the reciprocal diagonal is formed
// first (lane k), off the dependency chain.
__device__ __forceinline__ void diag16_inverse(const double (*sL)[TB + 1], int b, double (*sD)[16][17]) {
  const int lane = threadIdx.x & 63, o = 16 * b;
  const double rdl = lane < 16 ? 1.0 / sL[o + lane][o + lane] : 0.0;
  if (lane < 16) {
    const int c = lane;
    double bvec[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) bvec[i] = (i == c) ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const double xk = bvec[k] * readlane_d(rdl, k);  // zero above the column's diagonal
      bvec[k] = xk;
#pragma unroll
      for (int i = k + 1; i < 16; ++i) bvec[i] = fma(-sL[o + i][o + k], xk, bvec[i]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sD[b][i][c] = bvec[i];
  }
}

// sC(I, J) -= X_I X_J^T for the 16x16 tile (I, J), X = sX (64x64), by one wave
__device__ __forceinline__ void tile16_syrk(double (*sC)[TB + 1], const double (*sX)[TB + 1], int I, int J) {
  const int lane = threadIdx.x & 63, i = lane & 15, kq = lane >> 4;
  cd4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kb = 0; kb < TB / 4; ++kb)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sX[16 * I + i][4 * kb + kq], sX[16 * J + i][4 * kb + kq], acc, 0, 0, 0);
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) sC[16 * I + kq + 4 * r4][16 * J + i] -= acc[r4];
}

// In-place Cholesky of the lower triangle of sA, and the inverses of its first
// three 16x16 diagonal blocks (sD), blocked in 4 panels of 16 columns, by PW
// waves.
// Wave 0 factors a 64x16 panel in registers (lane i owns row i): the pivot and
// the column entries are broadcast with readlane (compile-time lanes), the
// pivot's reciprocal square root scales the column, and the rank-1 update
// stays in registers.  Every lane applies the same operations branch-free: a
// lane's entries right of its diagonal only ever hold values that are neither
// broadcast nor stored.  The panel's rank-16 update of the trailing triangle
// runs on the matrix cores, the next panel's 16 columns first (one tile per
// wave); the other tiles, the inverse of the block just factored and the
// caller's side work (side(w, b) on waves w = 1 .. PW - 1 while panel b is
// factored; the columns before it are final) run while wave 0 factors on.  The
// upper halves of the diagonal tiles are updated too and never read.
// The next pivot is formed in every lane from entries broadcast before this
// column is scaled (the same product and update as in its own lane), so no
// broadcast lies on the chain from pivot to pivot; scaled columns go to sA as
// they are finished, and the factors of the updates further right are read back
// from there.  Bound: instruction issue of the one wave, 185 cycles a column
// (about 40 instructions at 4 to 5 cycles each; the chain itself, reciprocal
// square root, scale and update, is 64).
template <class Side>
__device__ __forceinline__ void tile_potrf(double (*sA)[TB + 1], double (*sD)[16][17], int* status, Side side) {
  constexpr int PB = 16;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, kq = lane >> 4;
  // the rank-16 update of panel b on 16x16 tile (I, J)
  auto update = [&](int b, int I, int J) {
    cd4 acc;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) acc[r4] = sA[16 * I + kq + 4 * r4][16 * J + li];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-sA[16 * I + li][PB * b + 4 * kb + kq],
                                                 sA[16 * J + li][PB * b + 4 * kb + kq], acc, 0, 0, 0);
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) sA[16 * I + kq + 4 * r4][16 * J + li] = acc[r4];
  };
#pragma unroll
  for (int b = 0; b < TB / PB; ++b) {
    const int b0 = b * PB;
    if (w == 0) {
      double p[PB];
#pragma unroll
      for (int k = 0; k < PB; ++k) p[k] = sA[lane][b0 + k];
      bool bad = false;
      double piv = readlane_d(p[0], b0);
      double rs = rsqrt_nr(piv);
      // this column's entries (b0 + k + 1, k), (b0 + k + 2, k) before scaling and
      // the next diagonal entry before this column's update, in every lane
      double a1 = readlane_d(p[0], b0 + 1), a2 = readlane_d(p[0], b0 + 2), d1 = readlane_d(p[1], b0 + 1);
      double c[PB] = {};  // column k - 1's entries (b0 + kk, k - 1), kk >= k + 2
#pragma unroll
      for (int k = 0; k < PB; ++k) {
        bad |= !(piv > 0.0);
        const double l1 = a1 * rs;
        if (k + 1 == PB) {
          p[k] *= rs;
          break;
        }
        piv = fma(-l1, l1, d1);  // what the update below leaves in the next pivot's lane
        const double y = __builtin_amdgcn_rsq(piv);  // rsqrt_nr(piv) for the next column
        __builtin_amdgcn_sched_barrier(0);
        p[k] *= rs;               // the pivot's lane gets sqrt(piv), lanes below L(i, c)
        sA[lane][b0 + k] = p[k];  // (entries right of the diagonal are never read)
        wave_lds_fence();
        double cn[PB] = {};
#pragma unroll
        for (int kk = k + 3; kk < PB; ++kk) cn[kk] = sA[b0 + kk][b0 + k];
        __builtin_amdgcn_sched_barrier(0);
        auto upd = [&](int kk) {  // column k - 1 on column kk
          if (k > 0) p[kk] = fma(-p[k - 1], c[kk], p[kk]);
        };
        p[k + 1] = fma(-p[k], l1, p[k + 1]);
        if (k + 2 < PB) {
          const double l2 = a2 * rs;
          upd(k + 2);
          p[k + 2] = fma(-p[k], l2, p[k + 2]);
          a1 = readlane_d(p[k + 1], b0 + k + 2);
          if (k + 3 < PB) a2 = readlane_d(p[k + 1], b0 + k + 3);
          d1 = readlane_d(p[k + 2], b0 + k + 2);
        }
        // the reciprocal square root's chain, other columns' updates in its waits
        const int m = (PB - k - 3 + 3) / 4;
        auto fill = [&](int q) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = k + 3 + q * m; kk < PB && kk < k + 3 + (q + 1) * m; ++kk) upd(kk);
          __builtin_amdgcn_sched_barrier(0);
        };
        const double t = -piv * y;
        fill(0);
        const double h = fma(t, y, 1.0);
        fill(1);
        const double yh = y * h;
        fill(2);
        rs = fma(yh, 0.5, y);
        fill(3);
#pragma unroll
        for (int kk = k + 3; kk < PB; ++kk) c[kk] = cn[kk];
      }
      sA[lane][b0 + PB - 1] = p[PB - 1];
      if (bad && lane == 0) *status = 1;
    } else {
      if (b > 0) {  // the rest of panel b - 1's update: tiles right of this panel
        int t = 1;
#pragma unroll
        for (int J = b + 1; J < TB / PB; ++J)
#pragma unroll
          for (int I = J; I < TB / PB; ++I, ++t)
            if (w == t) update(b - 1, I, J);
        if (w == PW - 1) diag16_inverse(sA, b - 1, sD);
      }
      side(w, b);
    }
    __syncthreads();
    if (b + 1 < TB / PB) {
      if (w < TB / PB - 1 - b) update(b, b + 1 + w, b + 1);
      __syncthreads();
    }
  }
}

// Inverse of the lower-triangular sA (64x64) into sI, blocked in 16x16:
// wave w inverts diagonal block w (lane = column, forward substitution with
// reciprocal diagonals), then the off-diagonal blocks follow by block
// diagonals d = 1, 2, 3:  X_IJ = -X_II (sum_{J<=K<I} L_IK X_KJ), I = J + d.
__device__ __forceinline__ void tile_trinv(const double (*sA)[TB + 1], double (*sI)[TB + 1], double (*sT)[TB + 1]) {
  constexpr int PB = 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int t = threadIdx.x; t < TB * TB; t += CT) sI[t / TB][t % TB] = 0.0;
  __syncthreads();
  if (lane < PB) {
    const int o = wave * PB, c = lane;
    double x[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      double s = (i == c) ? 1.0 : 0.0;
#pragma unroll
      for (int k = 0; k < i; ++k) s -= sA[o + i][o + k] * x[k];
      x[i] = (i >= c) ? s / sA[o + i][o + i] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) sI[o + i][o + c] = x[i];
  }
  __syncthreads();
  for (int d = 1; d < TB / PB; ++d) {
    const int nb = TB / PB - d;  // blocks (J + d, J), J = 0 .. nb-1
    for (int t = threadIdx.x; t < nb * PB * PB; t += CT) {  // T = sum_K L_IK X_KJ
      const int J = t / (PB * PB), a = (t / PB) % PB, c = t % PB, I = J + d;
      double s = 0.0;
      for (int k = J * PB; k < I * PB; ++k) s += sA[I * PB + a][k] * sI[k][J * PB + c];
      sT[I * PB + a][J * PB + c] = s;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < nb * PB * PB; t += CT) {  // X_IJ = -X_II T
      const int J = t / (PB * PB), a = (t / PB) % PB, c = t % PB, I = J + d;
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < PB; ++k) s += sI[I * PB + a][I * PB + k] * sT[I * PB + k][J * PB + c];
      sI[I * PB + a][J * PB + c] = -s;
    }
    __syncthreads();
  }
}


// acc = A B^T on v_mfma_f64_16x16x4 (A, B: 64x64 row-major in LDS); wave w
// owns the 32x32 quarter (32 (w / 2), 32 (w % 2)) as 2x2 tiles of 16x16.
// D[r][c] of a tile at lane c + 16 (r % 4), register r / 4.
__device__ __forceinline__ void tile_gemm_nt_mfma(const double (*sA)[TB + 1], const double (*sB)[TB + 1],
                                                  cd4 (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 15, kq = lane >> 4;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1);
#pragma unroll
  for (int kb = 0; kb < TB / 4; ++kb) {
    const double a0 = sA[r0 + i][4 * kb + kq], a1 = sA[r0 + 16 + i][4 * kb + kq];
    const double b0 = sB[c0 + i][4 * kb + kq], b1 = sB[c0 + 16 + i][4 * kb + kq];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}
// (row, col) in the 64x64 product of element (a, b, r4) of tile_gemm_nt_mfma's acc
__device__ __forceinline__ int nt_row(int a, int r4) {
  return 32 * ((threadIdx.x >> 6) >> 1) + 16 * a + ((threadIdx.x & 63) >> 4) + 4 * r4;
}
__device__ __forceinline__ int nt_col(int b) { return 32 * ((threadIdx.x >> 6) & 1) + 16 * b + (threadIdx.x & 15); }
// acc += A B (A, B: 64x64 row-major in LDS), same output layout as above.
__device__ __forceinline__ void tile_gemm_nn_mfma(const double (*sA)[TB + 1], const double (*sB)[TB + 1],
                                                  cd4 (&acc)[2][2]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 15, kq = lane >> 4;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1);
#pragma unroll
  for (int kb = 0; kb < TB / 4; ++kb) {
    const double a0 = sA[r0 + i][4 * kb + kq], a1 = sA[r0 + 16 + i][4 * kb + kq];
    const double b0 = sB[4 * kb + kq][c0 + i], b1 = sB[4 * kb + kq][c0 + 16 + i];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}

// X = A L^{-T} in place (sX: A on entry, X on exit), blocked by 16 columns on
// the matrix cores:  R_b = A_b - X_{<b} L_{b,<b}^T,  X_b = R_b Dinv_b^T,
// Dinv_b the inverses of L's diagonal blocks; column blocks [b0, b1).  Wave w of
// four owns rows 16w..16w+15 throughout, so the waves need no barrier between
// the steps.
template <int b0, int b1>
__device__ __forceinline__ void tile_trsm_rt(double (*sX)[TB + 1], const double (*sL)[TB + 1],
                                             const double (*sD)[16][17], int w) {
  const int lane = threadIdx.x & 63, i = lane & 15, kq = lane >> 4;
  const int r0 = 16 * w;
#pragma unroll
  for (int b = b0; b < b1; ++b) {
    cd4 acc;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) acc[r4] = sX[r0 + kq + 4 * r4][16 * b + i];  // D layout: row kq + 4 r4, col i
#pragma unroll
    for (int kb = 0; kb < 4 * b; ++kb)  // -= X_{<b} L_{b,<b}^T
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-sX[r0 + i][4 * kb + kq], sL[16 * b + i][4 * kb + kq], acc, 0, 0, 0);
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) sX[r0 + kq + 4 * r4][16 * b + i] = acc[r4];  // R_b
    wave_lds_fence();
    cd4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)  // X_b = R_b Dinv_b^T
      x = __builtin_amdgcn_mfma_f64_16x16x4f64(sX[r0 + i][16 * b + 4 * kb + kq], sD[b][i][4 * kb + kq], x, 0, 0, 0);
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) sX[r0 + kq + 4 * r4][16 * b + i] = x[r4];
    wave_lds_fence();
  }
}

// Stages two or three 64x64 tiles of the band in one memory round trip, by FT
// threads: (i0, k0) -> s0, (i1, k1) -> s1 and, with THREE, (i2, k2) -> s2.
// THREE is a compile-time choice: a load under a run-time condition makes the
// compiler wait for the loads before it at every branch.
template <bool THREE>
__device__ __forceinline__ void stage_tiles(BandView V, int i0, int k0, double (*s0)[TB + 1], int i1, int k1,
                                            double (*s1)[TB + 1], int i2, int k2, double (*s2)[TB + 1]) {
  constexpr int U = TB * TB / FT;
  double v0[U], v1[U], v2[THREE ? U : 1];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int t = threadIdx.x + u * FT, r = t / TB, c = t % TB;
    v0[u] = V.get(i0 + r, k0 + c);
    v1[u] = V.get(i1 + r, k1 + c);
    if constexpr (THREE) v2[u] = V.get(i2 + r, k2 + c);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int t = threadIdx.x + u * FT, r = t / TB, c = t % TB;
    s0[r][c] = v0[u];
    s1[r][c] = v1[u];
    if constexpr (THREE) s2[r][c] = v2[u];
  }
}

// ---- 1. banded Cholesky ---------------------------------------------------
// Columns [16 c, 16 c + 16) of the factored tile, and the inverse of its
// diagonal block (c < 3), from LDS to the band and to dinv [3][16][16]; t: this
// thread's place among nt
__device__ __forceinline__ void store_cols(BandView V, int d0, const double (*sA)[TB + 1], int c, int t, int nt) {
  for (int e = t; e < TB * 16; e += nt) {
    const int i = e >> 4, k = 16 * c + (e & 15);
    if (k <= i) V.set(d0 + i, d0 + k, sA[i][k]);
  }
}
__device__ __forceinline__ void store_inverse(const double (*sD)[16][17], double* __restrict__ dinv, int c, int t,
                                              int nt) {
  for (int e = t; e < 256; e += nt) dinv[256 * c + e] = sD[c][e >> 4][e & 15];
}
// what is left to store once tile_potrf has returned, if its side work called
// store_early: the last columns and the third inverse
constexpr int kStoreWaves = 2;  // waves 5 and 6
__device__ __forceinline__ void store_early(BandView V, int d0, const double (*sA)[TB + 1], const double (*sD)[16][17],
                                            double* __restrict__ dinv, int sw, int b) {
  const int t = (sw - 5) * 64 + (threadIdx.x & 63);
  if (b == 0 || t < 0 || t >= 64 * kStoreWaves) return;
  store_cols(V, d0, sA, b - 1, t, 64 * kStoreWaves);
  if (b >= 2) store_inverse(sD, dinv, b - 2, t, 64 * kStoreWaves);
}
__device__ __forceinline__ void store_rest(BandView V, int d0, const double (*sA)[TB + 1], const double (*sD)[16][17],
                                           double* __restrict__ dinv) {
  store_cols(V, d0, sA, 3, threadIdx.x, FT);
  store_inverse(sD, dinv, 2, threadIdx.x, FT);
}

__global__ __launch_bounds__(FT) void k_chol_diag(BandView V, int d0, double* __restrict__ dinv, int* status) {
  __shared__ double sA[TB][TB + 1];
  __shared__ double sD[4][16][17];
  for (int t = threadIdx.x; t < TB * TB; t += FT) sA[t / TB][t % TB] = V.get(d0 + t / TB, d0 + t % TB);
  __syncthreads();
  tile_potrf(sA, sD, status, [&](int sw, int b) { store_early(V, d0, sA, sD, dinv, sw, b); });
  store_rest(V, d0, sA, sD, dinv);
}

// One launch per 64-column panel J (right-looking, the panel solve folded into
// the trailing update).  Work-group (I, K), K <= I, over the row tiles below
// diagonal tile J that the band reaches:
//   X_I = A(I, J) L_JJ^{-T}, X_K = A(K, J) L_JJ^{-T}   (four waves each)
//   A(I, K) -= X_I X_K^T                               (matrix cores)
// The (I, I) groups keep L(I, J) = X_I in a scratch panel (the band's copy of
// A(I, J) is still being read by the other groups); the next launch's extra
// groups copy it into the band.  Group (0, 0) updates the next diagonal tile,
// factors it and leaves the inverses of its first three 16x16 diagonal blocks
// behind the scratch panel for the next launch's substitutions (the last one,
// which would prolong its chain, is formed there beside their first steps).
// Bound: group (0, 0)'s latency chain; all it does but that chain (the tiles
// of X X^T past the first 16 columns, L(I, J) to the scratch panel, the
// inverses, the stores of finished columns) runs beside the pivots.  20.9 ->
// 15.3 us a launch at 128x256x128 (20.3 -> 14.0 at 50x100x50, 14.3 at 96x192x96);
// its parts there, with four waves and in sequence / now: staging 3.6 / 2.3,
// inverses and substitution 3.3 / 2.7, product 3.0 / 0.75, pivots 8.0 / 6.8,
// store 1.6 / 0.4 us.
__global__ __launch_bounds__(FT) void k_chol_panel(BandView V, int J, int nrt, int nrtPrev, double* __restrict__ pan,
                                                   int panStride, int* status) {
  __shared__ double sL[TB][TB + 1];  // L_JJ (zeros above the diagonal)
  __shared__ double sA[TB][TB + 1];  // A(I, J) -> X_I
  __shared__ double sB[TB][TB + 1];  // A(K, J) -> X_K, or the next diagonal tile
  __shared__ double sD[4][16][17];   // inverses of L_JJ's 16x16 diagonal blocks, then of the next tile's
  const int bw = V.bw, n = V.n;
  const int j0 = J * TB, r0 = j0 + TB;
  const int npairs = nrt * (nrt + 1) / 2;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if ((int)blockIdx.x >= npairs) {  // copy row tile t of panel J - 1 into the band
    const int t = blockIdx.x - npairs;
    if (t >= nrtPrev) return;
    const double* src = pan + (size_t)((J - 1) & 1) * panStride + (size_t)t * TB * TB;
    const int i0 = j0 + t * TB, k0 = j0 - TB;
    for (int e = threadIdx.x; e < TB * TB; e += FT) V.set(i0 + e / TB, k0 + e % TB, src[e]);
    return;
  }
  const int t0 = blockIdx.x;
  int I = 0;
  while ((I + 1) * (I + 2) / 2 <= t0) ++I;
  const int K = t0 - I * (I + 1) / 2;
  const int i0 = r0 + I * TB, k0 = r0 + K * TB;
  if (i0 - (k0 + TB - 1) > bw) return;  // tile outside the band
  double* panJ = pan + (size_t)(J & 1) * panStride;
  // the inverses lie behind the panel's last row tile
  const double* dinv = panJ + panStride - TB * TB;
  const double dv0 = dinv[threadIdx.x], dv1 = dinv[FT + (threadIdx.x & 255)];  // 768 entries
  // L_JJ (zeros above the diagonal), A(I, J), and A(K, J) or, for group
  // (0, 0), the next diagonal tile (no other group of this launch writes it)
  if (K != I)
    stage_tiles<true>(V, j0, j0, sL, i0, j0, sA, k0, j0, sB);
  else if (I == 0)
    stage_tiles<true>(V, j0, j0, sL, i0, j0, sA, r0, r0, sB);
  else
    stage_tiles<false>(V, j0, j0, sL, i0, j0, sA, 0, 0, nullptr);
  sD[threadIdx.x >> 8][(threadIdx.x >> 4) & 15][threadIdx.x & 15] = dv0;
  if (threadIdx.x < 256) sD[2][threadIdx.x >> 4][threadIdx.x & 15] = dv1;
  __syncthreads();
  if (w == PW - 1) diag16_inverse(sL, 3, sD);
  if (w < 4) tile_trsm_rt<0, 3>(sA, sL, sD, w);
  else if (K != I) tile_trsm_rt<0, 3>(sB, sL, sD, w - 4);
  __syncthreads();
  if (w < 4) tile_trsm_rt<3, 4>(sA, sL, sD, w);
  else if (K != I) tile_trsm_rt<3, 4>(sB, sL, sD, w - 4);
  __syncthreads();
  if (I == 0) {  // the next diagonal tile (staged in sB): update in LDS, then factor
    if (w < 4) tile16_syrk(sB, sA, w, 0);
    __syncthreads();
    double* dinvNext = pan + (size_t)((J + 1) & 1) * panStride + panStride - TB * TB;
    tile_potrf(sB, sD, status, [&](int sw, int b) {
      if (b == 0) {
        if (sw <= 6) {  // the other lower tiles of X X^T
          const int tI = sw <= 3 ? sw : (sw <= 5 ? sw - 2 : 3), tJ = sw <= 3 ? 1 : (sw <= 5 ? 2 : 3);
          tile16_syrk(sB, sA, tI, tJ);
        }
        for (int t = (sw - 1) * 64 + lane; t < TB * TB; t += 64 * (PW - 1)) panJ[t] = sA[t / TB][t % TB];  // L(I, J)
      }
      store_early(V, r0, sB, sD, dinvNext, sw, b);
    });
    store_rest(V, r0, sB, sD, dinvNext);
    return;
  }
  if (K == I) {  // L(I, J) to the scratch panel
    double* dst = panJ + (size_t)I * TB * TB;
    for (int t = threadIdx.x; t < TB * TB; t += FT) dst[t] = sA[t / TB][t % TB];
  }
  // A(I, K) -= X_I X_K^T: wave w the 16x16 tiles (w / 2, 2 (w % 2)) and the one beside it
  const double(*sK)[TB + 1] = K == I ? sA : sB;
  const int i = lane & 15, kq = lane >> 4, R = 16 * (w >> 1), C = 32 * (w & 1);
  cd4 acc[2] = {};
#pragma unroll
  for (int kb = 0; kb < TB / 4; ++kb) {
    const double a = sA[R + i][4 * kb + kq];
#pragma unroll
    for (int c = 0; c < 2; ++c)
      acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, sK[C + 16 * c + i][4 * kb + kq], acc[c], 0, 0, 0);
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const int row = i0 + R + kq + 4 * r4, col = k0 + C + 16 * c + i;
      if (col <= row && row - col <= bw && row < n) V.B[(size_t)row * V.W() + (row - col)] -= acc[c][r4];
    }
}

// Inverses of all 64x64 diagonal tiles (after the factorization, in parallel).
__global__ __launch_bounds__(CT) void k_tile_inverses(BandView V, double* __restrict__ tinv) {
  __shared__ double sA[TB][TB + 1];
  __shared__ double sI[TB][TB + 1];
  __shared__ double sT[TB][TB + 1];
  const int d0 = blockIdx.x * TB;
  for (int t = threadIdx.x; t < TB * TB; t += CT) sA[t / TB][t % TB] = V.get(d0 + t / TB, d0 + t % TB);
  __syncthreads();
  tile_trinv(sA, sI, sT);
  double* inv = tinv + (size_t)blockIdx.x * TB * TB;
  for (int t = threadIdx.x; t < TB * TB; t += CT) inv[t] = sI[t / TB][t % TB];
}

// ---- 2. solve-block operators -------------------------------------------
// WG (b, p): columns p*64.. of X = L_bb^{-1} [I | L_{b,b-1}], SB x 2SB.
// Output: Dinv_b (SB x SB row-major) and its transpose DT_b, G_b (SB x SB).
// A step multiplies two 64x64 tiles from LDS; the next step's tiles are loaded
// into registers beside it.  Bound: the loads (64 KB a step, mostly past the
// L2, few in flight per CU); the matrix cores are busy a sixth of the time.
// 2.34 -> 1.55 ms at 256x512x256 (SB 960, 30 blocks), 81 -> 52 us at
// 50x100x50; two waves per SIMD are worth the 248 registers (one: 2.73 ms).
template <bool IDENT>
__device__ __forceinline__ void trsm_strip(BandView V, int SB, int b, int col0, const double* __restrict__ tinv,
                                           double* Out, double* __restrict__ DT, double (*sL)[TB + 1],
                                           double (*sX)[TB + 1]) {
  constexpr int U = TB * TB / CT;
  const int st = SB / TB, base = b * SB;
  const int Ist = IDENT ? col0 / TB : 0;  // rows above the diagonal panel of L^{-1} are zero
  const int tr = threadIdx.x / TB, tc = threadIdx.x % TB;  // element u of this thread: row tr + 4 u, column tc
  constexpr int RU = CT / TB;
  double vl[U], vx[U], rr[2][2][4];
  const int W = V.W();
  auto load_l = [&](int I, int K) {  // L_bb(I, K): I > K, all its rows exist, the far corner may be outside the band
    const int d = (I - K) * TB + tr - tc;
    const double* l = V.B + (size_t)(base + I * TB + tr) * W;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double v = l[RU * u * W + min(d + RU * u, V.bw)];
      vl[u] = d + RU * u <= V.bw ? v : 0.0;
    }
  };
  auto load_x = [&](int K) {
    const double* x = Out + (size_t)(K * TB + tr) * SB + col0 + tc;
#pragma unroll
    for (int u = 0; u < U; ++u) vx[u] = x[RU * u * SB];
  };
  auto load_diag = [&](int I) {  // inv(L_II) and the right-hand side
    const double* inv = tinv + (size_t)(base / TB + I) * TB * TB + threadIdx.x;
#pragma unroll
    for (int u = 0; u < U; ++u) vl[u] = inv[u * CT];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int ra = nt_row(a, r4), cc = nt_col(c);
          rr[a][c][r4] = IDENT ? ((I * TB + ra == col0 + cc) ? 1.0 : 0.0)
                               : V.get(base + I * TB + ra, base - SB + col0 + cc);
        }
  };
  // the first tile of row I inside the band
  auto first = [&](int I) { return max(Ist, (I * TB - TB + 1 - V.bw + TB - 1) / TB); };
  for (int I = 0; I < Ist; ++I)
    for (int t = threadIdx.x; t < TB * TB; t += CT) Out[(size_t)(I * TB + t / TB) * SB + col0 + t % TB] = 0.0;
  load_diag(Ist);
  for (int I = Ist; I < st; ++I) {
    // T = R_I - sum_{K<I} L_bb(I,K) X_K
    cd4 acc[2][2] = {};
    for (int K = first(I); K < I; ++K) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        sL[tr + RU * u][tc] = vl[u];
        sX[tr + RU * u][tc] = vx[u];
      }
      __syncthreads();
      if (K + 1 < I) {
        load_l(I, K + 1);
        load_x(K + 1);
      } else {
        load_diag(I);
      }
      tile_gemm_nn_mfma(sL, sX, acc);
      __syncthreads();
    }
    // X_I = inv(L_II) T
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) sX[nt_row(a, r4)][nt_col(c)] = rr[a][c][r4] - acc[a][c][r4];
#pragma unroll
    for (int u = 0; u < U; ++u) sL[tr + RU * u][tc] = vl[u];
    __syncthreads();
    const int K1 = I + 1 < st ? first(I + 1) : I + 1;  // the next row's first tile: X_I itself is not there yet
    if (K1 <= I) load_l(I + 1, K1);
    if (K1 < I) load_x(K1);
    cd4 acc2[2][2] = {};
    tile_gemm_nn_mfma(sL, sX, acc2);  // inv(L_II) is lower triangular: the zeros add nothing
#pragma unroll
    for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int a = nt_row(a2, r4), c = nt_col(c2);
          Out[(size_t)(I * TB + a) * SB + col0 + c] = acc2[a2][c2][r4];
          if (IDENT) DT[(size_t)b * SB * SB + (size_t)(col0 + c) * SB + I * TB + a] = acc2[a2][c2][r4];
        }
    __syncthreads();
    if (K1 == I) load_x(I);
    else if (K1 > I && I + 1 < st) load_diag(I + 1);
  }
}
__global__ __launch_bounds__(CT) __attribute__((amdgpu_waves_per_eu(2)))
void k_trsm_blocks(BandView V, int SB, const double* __restrict__ tinv, double* __restrict__ Dinv,
                   double* __restrict__ DT, double* __restrict__ Gm) {
  // two tiles of LDS (66.6 KB: two work-groups per CU); the right-hand side
  // minus the accumulated products is formed in sX once the products are done
  __shared__ double sL[TB][TB + 1];
  __shared__ double sX[TB][TB + 1];
  // G's strips first: their work is st(st+1)/2 tile pairs each, that of L^{-1}'s
  // falls to one (block by block 1.72 ms at 256x512x256, so 1.55; blocks kept
  // to one XCD 1.79 and 2.01: their strips start and end together)
  const int st = SB / TB, npan = 2 * st, nG = gridDim.x / npan * st;
  const bool g = (int)blockIdx.x < nG;
  const int wg = g ? blockIdx.x : blockIdx.x - nG;
  const int b = wg / st, p = wg % st + (g ? st : 0);
  if (p < st) trsm_strip<true>(V, SB, b, p * TB, tinv, Dinv + (size_t)b * SB * SB, DT, sL, sX);
  else if (b > 0)  // G_0 is unused
    trsm_strip<false>(V, SB, b, (p - st) * TB, tinv, Gm + (size_t)b * SB * SB, DT, sL, sX);
}

// H_b = Dinv_b^T L_{b+1,b}^T, i.e. H_b(i,j) = sum_k DT_b(i,k) L((b+1)SB + j, b SB + k).
// One work-group per (b, output tile I, J); the next step's tiles are loaded
// beside a step's product (0.75 -> 0.48 ms at 256x512x256, 25 -> 16.5 us at
// 50x100x50).
__global__ __launch_bounds__(CT) __attribute__((amdgpu_waves_per_eu(2)))
void k_h_blocks(BandView V, int SB, int nblk, const double* __restrict__ DT, double* __restrict__ H) {
  __shared__ double sA[TB][TB + 1];
  __shared__ double sB[TB][TB + 1];
  const int st = SB / TB;
  const int per = st * st;
  // XCD-contiguous order: one solve block's output tiles, which read the same
  // DT_b and band tiles, run on one XCD and share its L2 (0.90 -> 0.75 ms at
  // 256x512x256)
  const int wg = xcd_tile_order().x;
  const int b = wg / per, rem = wg % per;
  const int I = rem / st, J = rem % st;
  if (b >= nblk - 1) return;
  const double* D = DT + (size_t)b * SB * SB;
  cd4 acc[2][2] = {};
  // DT_b(i,k) = Dinv_b(k,i) is zero for k < i; L's tiles before K0 are outside the band
  const int rowL0 = (b + 1) * SB + J * TB;
  const int K0 = max(I, (rowL0 - b * SB - TB + 1 - V.bw + TB - 1) / TB);
  constexpr int U = TB * TB / CT, RU = CT / TB;
  const int tr = threadIdx.x / TB, tc = threadIdx.x % TB, W = V.W();
  double va[U], vb[U];
  auto load = [&](int K) {  // the next step's tiles, beside this step's product
    const double* x = D + (size_t)(I * TB + tr) * SB + K * TB + tc;
    const int d = rowL0 - (b * SB + K * TB) + tr - tc;  // > 0
    const double* l = V.B + (size_t)(rowL0 + tr) * W;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      va[u] = x[RU * u * SB];
      const double v = l[RU * u * W + min(d + RU * u, V.bw)];
      vb[u] = d + RU * u <= V.bw ? v : 0.0;
    }
  };
  if (K0 < st) load(K0);
  for (int K = K0; K < st; ++K) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      sA[tr + RU * u][tc] = va[u];
      sB[tr + RU * u][tc] = vb[u];  // row j, col k
    }
    __syncthreads();
    if (K + 1 < st) load(K + 1);
    tile_gemm_nt_mfma(sA, sB, acc);
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        H[(size_t)b * SB * SB + (size_t)(I * TB + nt_row(a, r4)) * SB + J * TB + nt_col(c)] = acc[a][c][r4];
}

// ---- 3. the solve --------------------------------------------------------
// One wave per row dot product: out[row] = base - sum_j M[row][j] v[j].  Products
// are fused explicitly: the forms of the solve agree bit for bit, and where two
// branches share a product the compiler would round it on its own.
__device__ __forceinline__ double wave_dot(const double* __restrict__ m, const double* __restrict__ v, int len) {
  const int lane = threadIdx.x & 63;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int j = lane;
  for (; j + 192 < len; j += 256) {  // four independent loads in flight per lane
    s0 = fma(m[j], v[j], s0);
    s1 = fma(m[j + 64], v[j + 64], s1);
    s2 = fma(m[j + 128], v[j + 128], s2);
    s3 = fma(m[j + 192], v[j + 192], s3);
  }
  for (; j < len; j += 64) s0 = fma(m[j], v[j], s0);
  double s = (s0 + s1) + (s2 + s3);
  return wave_sum(s);
}

// forward phase 0: gather the permuted right-hand side and va_b = Dinv_b v_b,
// a lane's columns lane + 64 c summed in order.  A work-group takes kOwnRows
// rows of one block, kOwnRows / 4 per wave, against the block's vector in LDS:
// 16 loads in flight per lane, and the vector is gathered once per group.
// HBM-bound: 110 MB at 256x512x256 in 32 us, against 42 us with a wave per row
// that gathered its own vector.
constexpr int kOwnRows = 16;  // divides TB, so a group's rows share a diagonal tile
constexpr int kOwnPerWave = kOwnRows / (CT / 64);
template <typename TR>
__global__ __launch_bounds__(CT) void k_solve_f0(int n, int np, int SB, const long long* __restrict__ map,
                                                 const TR* __restrict__ rdense, const double* __restrict__ Dinv,
                                                 double* __restrict__ va, const int* fl) {
  if (fl && fl[FL_DONE]) return;
  constexpr int SEG = 64;  // 64-column chunks of the vector in LDS at a time
  __shared__ double sv[SEG * TB];
  const int row0 = blockIdx.x * kOwnRows;  // SB is a multiple of kOwnRows
  const int b = row0 / SB, i0 = row0 % SB, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = i0 + kOwnPerWave * w;  // this wave's rows i .. i + kOwnPerWave - 1
  const double* m = Dinv + ((size_t)b * SB + i) * SB;
  const int c1 = i0 / TB + 1;  // chunks up to the diagonal's; Dinv is 0 right of the diagonal
  double s[kOwnPerWave] = {};
  for (int cs = 0; cs < c1; cs += SEG) {
    const int ce = min(c1, cs + SEG);
    __syncthreads();
    for (int j = cs * TB + threadIdx.x; j < ce * TB; j += CT) {
      const int g = b * SB + j;
      sv[j - cs * TB] = g < n ? (double)rdense[map[g]] : 0.0;
    }
    __syncthreads();
    int c = cs;
    for (; c + 4 <= ce; c += 4) {
      double t[kOwnPerWave][4];
#pragma unroll
      for (int r = 0; r < kOwnPerWave; ++r)
#pragma unroll
        for (int u = 0; u < 4; ++u) t[r][u] = m[(size_t)r * SB + lane + TB * (c + u)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double v = sv[lane + TB * (c + u - cs)];
#pragma unroll
        for (int r = 0; r < kOwnPerWave; ++r) s[r] = fma(t[r][u], v, s[r]);
      }
    }
    for (; c < ce; ++c) {
      const double v = sv[lane + TB * (c - cs)];
#pragma unroll
      for (int r = 0; r < kOwnPerWave; ++r) s[r] = fma(m[(size_t)r * SB + lane + TB * c], v, s[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < kOwnPerWave; ++r) {
    const double t = wave_sum(s[r]);
    if (lane == 0) va[row0 + kOwnPerWave * w + r] = t;
  }
}
// v[b] -= M_b v[b + d] for the SB rows of block b (d = -1 forward, +1 backward)
__global__ __launch_bounds__(CT) void k_solve_step(int SB, int b, int d, const double* __restrict__ M,
                                                   double* __restrict__ v, const int* fl) {
  if (fl && fl[FL_DONE]) return;
  const int i = blockIdx.x * (CT / 64) + (threadIdx.x >> 6);
  if (i >= SB) return;
  const double s = wave_dot(M + (size_t)b * SB * SB + (size_t)i * SB, v + (size_t)(b + d) * SB, SB);
  if ((threadIdx.x & 63) == 0) v[(size_t)b * SB + i] -= s;
}
// backward phase 0: vb_b = Dinv_b^T y_b
__global__ __launch_bounds__(CT) void k_solve_b0(int np, int SB, const double* __restrict__ DT,
                                                 const double* __restrict__ va, double* __restrict__ vb,
                                                 const int* fl) {
  if (fl && fl[FL_DONE]) return;
  const int row = blockIdx.x * (CT / 64) + (threadIdx.x >> 6);
  if (row >= np) return;
  const int b = row / SB, i = row % SB;
  const double s = wave_dot(DT + (size_t)b * SB * SB + (size_t)i * SB + i, va + (size_t)b * SB + i, SB - i);
  if ((threadIdx.x & 63) == 0) vb[row] = s;
}
template <typename TX>
__global__ void k_solve_scatter(int n, const long long* __restrict__ map, const double* __restrict__ vb,
                                TX* __restrict__ xdense, const int* fl) {
  if (fl && fl[FL_DONE]) return;
  const int i = blockIdx.x * CT + threadIdx.x;
  if (i < n) xdense[map[i]] = (TX)vb[i];
}

// ---- 3b. the recurrences without a launch per block ------------------------
// A launch per block costs ~7.5 us of dispatch, ramp and drain against
// ~1.5 us of data.  Here one launch per recurrence (forward after
// k_solve_f0, backward after k_solve_b0) walks all its blocks.  The work-groups
// form SETS sets that take the blocks in turn; a set's groups of 4 waves own
// all SB rows of its blocks, SETS rows per wave.  A block's rows carry their
// own readiness: an entry is one 64-bit word, written with an agent-scope store
// (coherent across the XCDs' L2s), and a group that needs the block before
// polls its words until none is unset.  Every vector has two places, for
// launches in turn (ChainState's count, advanced by the backward launch); the
// rows' owners clear the other one, which the launch before filled and nobody
// reads any more.  (Words of half a value and a tag each, 2 SB of them a block,
// took 2 us more of 60 a recurrence.)
// Bound: with one set, a block's hand-over (1.5 us) and then its operator rows
// (7.4 MB at SB 960, 1.6 us from HBM): a group asks for its next rows when its
// block is written, and loads return in order, so its polls see nothing before
// those rows are there.  (Asked for ahead of the product instead, in a second
// register set, they delay the store: 89 against 53 us a recurrence.)  With two
// sets one set's rows arrive while the other one's block is formed: 62.9 ->
// 48.3 us forward, 58.2 -> 49.5 us backward at 128x256x128 (18 blocks), 53 ->
// 46 us at 96x192x96.  480 groups of one row per wave: 49 us and twice the
// share of the device; 3 or 4 sets 53 to 72 us.  Above SB 1024 two rows of a
// wave do not fit its registers: one set.
// All groups must be resident together: 4 waves and SB doubles of LDS each, far
// below the device's capacity; two sets keep to 128 registers for that (see
// chain_share; 23.4% of the device at SB 960).  Each wait is bounded:
// after kChainSpin polls the launch sets fail, every group stops waiting (the
// solve is then garbage) and the caller reports the error; fail stays set.
// Measured alternatives (same operators): one launch for everything with a
// published count per block, 7.6 us per block; the same with an agent-scope
// release/acquire pair, which writes back and invalidates the L2, 30 us.
constexpr unsigned kChainSpin = 1u << 20;  // polls per wait (~1 s) before the launch gives up

// An entry of an exchanged vector is one word: the value's bits with this
// signalling NaN's taken off (exclusive or), so 0 is "not there yet": a value
// formed by arithmetic is never a signalling NaN.
constexpr unsigned long long kUnset = 0x7FF0000000000001ull;
__device__ __forceinline__ void chain_put(unsigned long long* w, double v) {
  __hip_atomic_store(w, (unsigned long long)__double_as_longlong(v) ^ kUnset, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void chain_clear(unsigned long long* w) {
  __hip_atomic_store(w, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long chain_get(const unsigned long long* w) {
  return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double chain_value(unsigned long long w) {
  return __longlong_as_double((long long)(w ^ kUnset));
}

// FWD: y_b = a_b - G_b y_{b-1} (a = Dinv_b v_b from k_solve_f0, overwritten
// by y for k_solve_b0); backward: x_b = a_b - H_b x_{b+1} (a = Dinv_b^T y_b
// from k_solve_b0), scattered to xdense as formed.  PT: block entries per
// thread (SB <= PT * CT).
template <typename TV, int PT, int SETS, bool FWD>
__global__ __launch_bounds__(CT) __attribute__((amdgpu_waves_per_eu(SETS == 2 ? 4 : 1)))
void k_solve_chain(int n, int SB, int nblk, const long long* __restrict__ map, TV* __restrict__ xdense,
                   const double* __restrict__ M, double* __restrict__ a, unsigned long long* W, ChainState* st,
                   const int* fl) {
  if (fl && fl[FL_DONE]) return;
  constexpr int NCH = PT * CT / 64;  // 64-column chunks of a row
  constexpr int RPW = SETS;          // rows per wave: the grid is as large in either form
  extern __shared__ double chainNbr[];  // the neighbour block
  const int lane = threadIdx.x & 63;
  const int set = blockIdx.x % SETS;
  const int row0 = (blockIdx.x / SETS * (CT / 64) + (threadIdx.x >> 6)) * RPW;  // RPW divides SB
  const int mine = row0 + min(lane, RPW - 1);  // the row whose entry this lane stores (lanes < RPW)
  const bool act = row0 < SB;
  const unsigned turn = st->turn[blockIdx.x];  // advanced by this group's previous backward launch
  unsigned long long *Wn = W + (size_t)(turn & 1) * nblk * SB, *Wo = W + (size_t)(~turn & 1) * nblk * SB;
  auto block_at = [&](int k) { return FWD ? k : nblk - 1 - k; };  // the k-th block of the recurrence
  double rg[RPW][NCH], ab = 0.0;
  long long to = 0;  // where the entry goes (read with the row: the store must not wait for it)
  auto load_own = [&](int b) {
    ab = a[(size_t)b * SB + mine];
    if (!FWD) to = map[min(b * SB + mine, n - 1)];
  };
  auto prefetch = [&](int b) {  // rows of M_b and their own terms, all loads in flight together
    const double* m = M + ((size_t)b * SB + row0) * SB;
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int j = lane + 64 * c;
        rg[r][c] = j < SB ? m[(size_t)r * SB + j] : 0.0;
      }
    load_own(b);
  };
  auto emit = [&](int b, double v) {
    if (lane >= RPW) return;
    const int g = b * SB + mine;
    chain_put(Wn + g, v);
    if (FWD) a[g] = v;
    else if (g < n) xdense[to] = (TV)v;
    chain_clear(Wo + g);
  };
  int k = set;
  if (act && k == 0) {  // the first block is its own term
    load_own(block_at(0));
    emit(block_at(0), ab);
  }
  if (k == 0) k = SETS;
  if (act && k < nblk) prefetch(block_at(k));
  for (; k < nblk; k += SETS) {
    {  // the block before into LDS once every entry is there
      const unsigned long long* w0 = Wn + block_at(k - 1) * SB;
      unsigned pending = 0;
#pragma unroll
      for (int u = 0; u < PT; ++u)
        if ((int)threadIdx.x + u * CT < SB) pending |= 1u << u;
      unsigned polls = 0;
      while (pending) {
        unsigned long long w[PT];
#pragma unroll
        for (int u = 0; u < PT; ++u)
          if (pending & (1u << u)) w[u] = chain_get(w0 + threadIdx.x + u * CT);
#pragma unroll
        for (int u = 0; u < PT; ++u)
          if ((pending & (1u << u)) && w[u]) {
            chainNbr[threadIdx.x + u * CT] = chain_value(w[u]);
            pending &= ~(1u << u);
          }
        if (!pending) break;
        // (given up: what is left in chainNbr makes the solve garbage, as reported)
        if (__hip_atomic_load(&st->fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        if (++polls > kChainSpin) {
          __hip_atomic_store(&st->fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
      }
    }
    __syncthreads();
    if (act) {
      // wave_dot's order over the registered row (four running sums over
      // chunk quadruples while the whole quadruple is in the row, then the
      // remaining chunks into the first), so the result is bitwise that of
      // k_solve_step
      double s = 0.0;
#pragma unroll
      for (int r = 0; r < RPW; ++r) {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
        bool quad = true;
#pragma unroll
        for (int q = 0; q < NCH / 4; ++q) {
          const int j = lane + 256 * q;
          quad = quad && j + 192 < SB;
          if (quad) {
            s0 = fma(rg[r][4 * q], chainNbr[j], s0);
            s1 = fma(rg[r][4 * q + 1], chainNbr[j + 64], s1);
            s2 = fma(rg[r][4 * q + 2], chainNbr[j + 128], s2);
            s3 = fma(rg[r][4 * q + 3], chainNbr[j + 192], s3);
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (j + 64 * u < SB) s0 = fma(rg[r][4 * q + u], chainNbr[j + 64 * u], s0);
          }
        }
        const double t = wave_sum((s0 + s1) + (s2 + s3));
        if (lane == r) s = t;
      }
      emit(block_at(k), ab - s);
      if (k + SETS < nblk) prefetch(block_at(k + SETS));
    }
    __syncthreads();  // chainNbr free
  }
  if (!FWD && threadIdx.x == 0) st->turn[blockIdx.x] = turn + 1;
}

// SB <= kFusedMaxSB: the own terms and both recurrences in one launch.  The
// operators of a block are small there (2 MB at SB 512), so a step is its
// hand-over whatever else it loads: own terms formed while waiting, the way
// back's (DT y) when the block before arrives.  Against k_solve_f0, two
// k_solve_chain and k_solve_b0 that is three launches and two passes over the
// vectors less, with the same sums in the same order.  Words and polls as in
// k_solve_chain.  Rows: one per wave, few per group, so that a block's loads
// spread over many CUs.
// Four waves a group and four groups a CU, as the other forms (chain_share): 128
// registers, for which the wave's row is in scalars and a DT row is summed before
// the next own terms are asked for (154 registers otherwise, three groups).
// Bound: the hand-over, 1.4 us a step.  50x100x50 (SB 256, 11 blocks): 38 us,
// against 54 us in four launches; at SB 384 (12 blocks) 68 against 77, at SB 512
// 108 to 113 against 122 and three launches.  Groups of two waves 39, 65 and 108
// us: two of them need not leave a slot on each SIMD for a group of four.  Two sets
// of groups in turn: 4% less and twice the share of the device.  Groups with waves
// that only poll, beside the row waves, were slower (62 us; at SB 960 163 against
// 92 us a direction: polls that do not wait for the operator rows compete with
// them for memory).
struct FusedArgs {
  int n, SB, nblk;
  const long long* map;
  const double *Dinv, *DT, *Gm, *H;
  double* vb;                 // own terms of the way back
  unsigned long long *W, *X;  // exchanged y and x, two places each
  ChainState* st;
};
// NCH: 64-column chunks of a row (SB <= 64 NCH), PT = NCH / NW entries polled per thread
template <typename TV, int NCH>
__global__ __launch_bounds__(CT) __attribute__((amdgpu_waves_per_eu(4)))
void k_solve_fused(FusedArgs A, const TV* __restrict__ rdense, TV* __restrict__ xdense, const int* fl) {
  if (fl && fl[FL_DONE]) return;
  constexpr int NW = CT / 64, PT = NCH / NW, NT = CT;
  extern __shared__ double chainNbr[];  // two neighbour blocks, in turn
  const int SB = A.SB, nblk = A.nblk;
  const int lane = threadIdx.x & 63;
  // SB is a multiple of NW: row < SB
  const int row = blockIdx.x * NW + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned turn = A.st->turn[blockIdx.x];
  const size_t wn = (size_t)(turn & 1) * nblk * SB, wo = (size_t)(~turn & 1) * nblk * SB;
  int step = 0;
  // block b of Wd into the next buffer once every entry is there
  auto poll = [&](const unsigned long long* Wd, int b) -> const double* {
    double* sY = chainNbr + (step++ & 1) * SB;
    unsigned pending = 0;
#pragma unroll
    for (int k = 0; k < PT; ++k)
      if ((int)threadIdx.x + k * NT < SB) pending |= 1u << k;
    unsigned polls = 0;
    while (pending) {
      unsigned long long w[PT];
#pragma unroll
      for (int k = 0; k < PT; ++k)
        if (pending & (1u << k)) w[k] = chain_get(Wd + b * SB + threadIdx.x + k * NT);
#pragma unroll
      for (int k = 0; k < PT; ++k)
        if ((pending & (1u << k)) && w[k]) {
          sY[threadIdx.x + k * NT] = chain_value(w[k]);
          pending &= ~(1u << k);
        }
      if (!pending) break;
      bool give = __hip_atomic_load(&A.st->fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
      if (!give && ++polls > kChainSpin) {
        __hip_atomic_store(&A.st->fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        give = true;
      }
      if (give) {
#pragma unroll
        for (int k = 0; k < PT; ++k)
          if (pending & (1u << k)) sY[threadIdx.x + k * NT] = 0.0;
        break;
      }
    }
    __syncthreads();  // (the buffer's readers of two steps ago have passed the barrier since)
    return sY;
  };
  // entries e >= len repeat the last one and enter no sum
  auto load = [&](const double* m, int len, double (&r)[NCH]) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) r[c] = m[min(lane + 64 * c, len - 1)];
  };
  // wave_dot's order over a row in registers
  auto dot = [&](const double (&r)[NCH], const double* v, int len) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    bool quad = true;
#pragma unroll
    for (int q = 0; q < NCH / 4; ++q) {
      const int j = lane + 256 * q;
      quad = quad && j + 192 < len;
      if (quad) {
        s0 = fma(r[4 * q], v[j], s0);
        s1 = fma(r[4 * q + 1], v[j + 64], s1);
        s2 = fma(r[4 * q + 2], v[j + 128], s2);
        s3 = fma(r[4 * q + 3], v[j + 192], s3);
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (j + 64 * u < len) s0 = fma(r[4 * q + u], v[j + 64 * u], s0);
      }
    }
    return wave_sum((s0 + s1) + (s2 + s3));
  };
  auto op_row = [&](const double* M, int b) { return M + ((size_t)b * SB + row) * SB; };
  // rows of G or H, of DT from the diagonal on, of Dinv; the right-hand side
  double rg[NCH], rt[NCH], rd[NCH], rv[NCH];
  auto load_own = [&](int b) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int g = b * SB + min(lane + 64 * c, SB - 1);
      const double v = (double)rdense[A.map[min(g, A.n - 1)]];
      rv[c] = g < A.n ? v : 0.0;
    }
    load(op_row(A.Dinv, b), SB, rd);
  };
  auto emit_x = [&](int b, double v) {
    const int g = b * SB + row;
    chain_put(A.X + wn + g, v);
    if (g < A.n) xdense[A.map[g]] = (TV)v;
    chain_clear(A.X + wo + g);
  };
  load_own(0);
  for (int b = 0; b < nblk; ++b) {  // forwards
    double y = 0.0;
#pragma unroll
    for (int c = 0; c < NCH; ++c)  // k_solve_f0's order
      if (lane + 64 * c <= row) y = fma(rd[c], rv[c], y);
    y = wave_sum(y);
    const double* sY = nullptr;
    if (b > 0) {
      sY = poll(A.W + wn, b - 1);
      y -= dot(rg, sY, SB);
    }
    if (lane == 0) {
      chain_put(A.W + wn + b * SB + row, y);
      chain_clear(A.W + wo + b * SB + row);
    }
    if (b + 1 < nblk) load(op_row(A.Gm, b + 1), SB, rg);
    if (b > 0) {
      const double t = dot(rt, sY + row, SB - row);
      if (lane == 0) A.vb[(size_t)(b - 1) * SB + row] = t;
    }
    if (b + 1 < nblk) load_own(b + 1);
    load(op_row(A.DT, b) + row, SB - row, rt);
  }
  {  // x of the last block is its own term
    const double* sY = poll(A.W + wn, nblk - 1);
    const double x = dot(rt, sY + row, SB - row);
    if (lane == 0) emit_x(nblk - 1, x);
  }
  for (int b = nblk - 2; b >= 0; --b) {  // backwards
    load(op_row(A.H, b), SB, rg);
    double own = 0.0;
    if (lane == 0) own = A.vb[(size_t)b * SB + row];  // this lane's own store
    const double* sY = poll(A.X + wn, b + 1);
    const double x = own - dot(rg, sY, SB);
    if (lane == 0) emit_x(b, x);
  }
  if (threadIdx.x == 0) A.st->turn[blockIdx.x] = turn + 1;
}

// ---- host side -----------------------------------------------------------
template <typename TV>
static auto fused_form(int SB) {
  return SB <= 256 ? k_solve_fused<TV, 4> : k_solve_fused<TV, 8>;
}
static size_t fused_lds(int SB) { return 2 * (size_t)SB * sizeof(double); }

template <typename TV, bool FWD>
static auto chain_form(int SB) {
  return SB > 4 * CT ? k_solve_chain<TV, kChainMaxSB / CT, 1, FWD> : k_solve_chain<TV, 4, 2, FWD>;
}

// Every form's groups have four waves, one per SIMD, and up to SB 1024 at most
// 128 registers: they count as a quarter of a CU each, whatever else is resident
// on it, also where a form alone would fit six times (77 registers up to SB
// 256).  So while the shares add up to the device, some CU has room for every
// such group that is not resident yet.  (Counted by their own occupancy, groups of
// 96 and of 128 registers could keep each other out, both launches incomplete: two
// of the one and two of the other leave 64 registers on a SIMD.)
// Above SB 1024 a group has 176 registers and counts as half a CU: it may have to
// wait for the others' launches to end, but no mix of a CU whose shares are below
// one refuses a quarter, so those do end.
long long CoarseSolver::chain_share() const {
  constexpr long long kNever = 2000000;
  constexpr int kGroupsPerCU = 4;
  if (SB > kChainMaxSB) return kNever;
  int dev = 0, cus = 0, perCU = 0, perCU2 = 0;
  if (hipGetDevice(&dev) != hipSuccess) return kNever;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return kNever;
  const int G = (SB + 3) / 4;
  if (SB <= kFusedMaxSB) {
    const size_t lds = fused_lds(SB);
    auto f64 = fused_form<double>(SB);
    auto f32 = fused_form<float>(SB);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, f64, CT, lds) != hipSuccess) return kNever;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU2, f32, CT, lds) != hipSuccess) return kNever;
  } else {
    const size_t lds = (size_t)SB * sizeof(double);
    auto fwd = chain_form<double, true>(SB);
    auto bwd = chain_form<float, false>(SB);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, fwd, CT, lds) != hipSuccess) return kNever;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU2, bwd, CT, lds) != hipSuccess) return kNever;
  }
  const long long slots = (long long)std::min({perCU, perCU2, kGroupsPerCU}) * cus;
  if (slots <= 0) return kNever;
  return (1000000LL * G + slots - 1) / slots;
}

void CoarseSolver::plan(int n_, int bw_) {
  n = n_;
  bw = bw_;
  SB = ((bw + 1 + TB - 1) / TB) * TB;
  if (SB < TB) SB = TB;
  np = ((n + SB - 1) / SB) * SB;
  nblk = np / SB;
}

size_t CoarseSolver::band_len() const { return (size_t)np * (bw + 1); }

void CoarseSolver::factor(hipStream_t s, double* band, double* tinv, double* pan, double* Dinv, double* DT,
                          double* Gm, double* H, int* status) {
  BandView V{band, np, bw};
  const int nt = np / TB;
  const int panStride = (int)(panel_len() / 2);
  // tile J's inverses lie behind scratch panel J mod 2 (its row tiles: (bw + 63) / 64)
  auto dinv = [&](int J) { return pan + (size_t)(J & 1) * panStride + panStride - TB * TB; };
  hipLaunchKernelGGL(k_chol_diag, dim3(1), dim3(FT), 0, s, V, 0, dinv(0), status);
  int nrtPrev = 0;
  for (int J = 0; J < nt; ++J) {
    const int j0 = J * TB, r0 = j0 + TB;
    const int rlast = std::min(np - 1, j0 + TB - 1 + bw);
    const int nrt = rlast >= r0 ? (rlast - r0) / TB + 1 : 0;
    const int grid = nrt * (nrt + 1) / 2 + nrtPrev;
    if (nrt > 0 || nrtPrev > 0)
      hipLaunchKernelGGL(k_chol_panel, dim3(grid), dim3(FT), 0, s, V, J, nrt, nrtPrev, pan, panStride, status);
    if (nrt == 0 && J + 1 < nt) hipLaunchKernelGGL(k_chol_diag, dim3(1), dim3(FT), 0, s, V, r0, dinv(J + 1), status);
    nrtPrev = nrt;
  }
  if (nrtPrev > 0)  // copy the last panel
    hipLaunchKernelGGL(k_chol_panel, dim3(nrtPrev), dim3(FT), 0, s, V, nt, 0, nrtPrev, pan, panStride, status);
  hipLaunchKernelGGL(k_tile_inverses, dim3(nt), dim3(CT), 0, s, V, tinv);
  const int st = SB / TB;
  hipLaunchKernelGGL(k_trsm_blocks, dim3(nblk * 2 * st), dim3(CT), 0, s, V, SB, tinv, Dinv, DT, Gm);
  if (nblk > 1) hipLaunchKernelGGL(k_h_blocks, dim3(nblk * st * st), dim3(CT), 0, s, V, SB, nblk, DT, H);
}

template <typename TV>
static void solve_impl(const CoarseSolver& C, hipStream_t s, const long long* map, const TV* rdense, TV* xdense,
                       const double* Dinv, const double* DT, const double* Gm, const double* H, double* va,
                       double* vb, const int* fl) {
  const int wpb = CT / 64;
  const int n = C.n, np = C.np, SB = C.SB, nblk = C.nblk;
  if (C.one_launch() && SB <= kFusedMaxSB) {
    const FusedArgs A{n, SB, nblk, map, Dinv, DT, Gm, H, vb, (unsigned long long*)(va + np),
                      (unsigned long long*)(vb + np), C.chain};
    hipLaunchKernelGGL(fused_form<TV>(SB), dim3(SB / wpb), dim3(CT), fused_lds(SB), s, A, rdense, xdense, fl);
    return;
  }
  const dim3 ownGrid(np / kOwnRows);
  if (C.one_launch()) {  // va, vb: np plain doubles, then 2 np words each
    auto fwd = chain_form<TV, true>(SB);
    auto bwd = chain_form<TV, false>(SB);
    const dim3 grid((SB + wpb - 1) / wpb);
    hipLaunchKernelGGL(k_solve_f0<TV>, ownGrid, dim3(CT), 0, s, n, np, SB, map, rdense, Dinv, va, fl);
    hipLaunchKernelGGL(fwd, grid, dim3(CT), SB * sizeof(double), s, n, SB, nblk, map, xdense, Gm, va,
                       (unsigned long long*)(va + np), C.chain, fl);
    hipLaunchKernelGGL(k_solve_b0, dim3((np + wpb - 1) / wpb), dim3(CT), 0, s, np, SB, DT, va, vb, fl);
    hipLaunchKernelGGL(bwd, grid, dim3(CT), SB * sizeof(double), s, n, SB, nblk, map, xdense, H, vb,
                       (unsigned long long*)(vb + np), C.chain, fl);
    return;
  }
  hipLaunchKernelGGL(k_solve_f0<TV>, ownGrid, dim3(CT), 0, s, n, np, SB, map, rdense, Dinv, va, fl);
  for (int b = 1; b < nblk; ++b)
    hipLaunchKernelGGL(k_solve_step, dim3((SB + wpb - 1) / wpb), dim3(CT), 0, s, SB, b, -1, Gm, va, fl);
  hipLaunchKernelGGL(k_solve_b0, dim3((np + wpb - 1) / wpb), dim3(CT), 0, s, np, SB, DT, va, vb, fl);
  for (int b = nblk - 2; b >= 0; --b)
    hipLaunchKernelGGL(k_solve_step, dim3((SB + wpb - 1) / wpb), dim3(CT), 0, s, SB, b, +1, H, vb, fl);
  hipLaunchKernelGGL(k_solve_scatter<TV>, dim3((n + CT - 1) / CT), dim3(CT), 0, s, n, map, vb, xdense, fl);
}

void CoarseSolver::solve(hipStream_t s, const long long* map, const double* rdense, double* xdense, const double* Dinv,
                         const double* DT, const double* Gm, const double* H, double* va, double* vb,
                         const int* fl) const {
  solve_impl(*this, s, map, rdense, xdense, Dinv, DT, Gm, H, va, vb, fl);
}
void CoarseSolver::solve(hipStream_t s, const long long* map, const float* rdense, float* xdense, const double* Dinv,
                         const double* DT, const double* Gm, const double* H, double* va, double* vb,
                         const int* fl) const {
  solve_impl(*this, s, map, rdense, xdense, Dinv, DT, Gm, H, va, vb, fl);
}

// identity rows beyond the true order (after band assembly)
__global__ void k_band_pad(double* B, int n, int np, int W) {
  const int i = n + blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) B[(size_t)i * W] = 1.0;
}
void CoarseSolver::pad_identity(hipStream_t s, double* band) {
  if (np > n) hipLaunchKernelGGL(k_band_pad, dim3((np - n + 255) / 256), dim3(256), 0, s, band, n, np, bw + 1);
}

}  // namespace t3x
