// HIP kernels of libt3x for gfx950 (CDNA4, wave64).
//
// FP64 "plain" path.  Reference lines are TOP3D_XL.m.
#include <hip/hip_runtime.h>

#include "t3x_kernels.h"
#include "t3x_reduce.h"

namespace t3x {

namespace {

__device__ __forceinline__ void node_yxz(long long n, const Geo& g, int& y, int& x, int& z) {
  const unsigned int nn = (unsigned int)n;
  const unsigned int t = nn / (unsigned int)g.NY;
  y = (int)(nn - t * (unsigned int)g.NY);
  z = (int)(t / (unsigned int)g.NX);
  x = (int)(t - (unsigned int)z * (unsigned int)g.NX);
}

__device__ __forceinline__ long long nidx(const Geo& g, int y, int x, int z) {
  return (long long)y + (long long)g.NY * ((long long)x + (long long)g.NX * z);
}

__device__ __forceinline__ bool cell_in(const Geo& g, int cy, int cx, int cz) {
  return cy >= 0 && cx >= 0 && cz >= 0 && cy < g.ny && cx < g.nx && cz < g.nz;
}

inline int grid_for(long long n) {
  long long b = (n + kBlock - 1) / kBlock;
  if (b > (1LL << 30)) b = 1LL << 30;
  return (int)(b < 1 ? 1 : b);
}

}  // namespace

// =========================================================================
// One-block finalisers: fold a reduction's partials (fixed order) and apply
// the scalar logic of the solver step that consumes it.
// =========================================================================
__global__ __launch_bounds__(kFinBlock) void k_fin1(int op, int nb, const double* __restrict__ partials, double* sc,
                                                    int* fl, double* out) {
  if (fl && fl[FL_DONE]) return;
  double v[1];
  fold_partials<1, kFinBlock>(partials, nb, v);
  if (threadIdx.x != 0) return;
  const double t = v[0];
  switch (op) {
    case FIN_PQ: {  // 615
      const double zr = sc[SC_ZRN];  // (SC_ZR: what it was an iteration ago)
      sc[SC_PQ] = t;
      sc[SC_LAMBDA] = zr / t;
      sc[SC_ZR] = zr;
    } break;
    case FIN_ZR_INIT:  // 612
      sc[SC_ZRN] = t;
      break;
    case FIN_ZR_LOOP:  // 629-631
      sc[SC_ZRN] = t;
      sc[SC_BETA] = t / sc[SC_ZR];
      break;
    case FIN_RR: {  // 618-622
      const double res = sqrt(t) / sc[SC_NORMB];
      sc[SC_RR] = t;
      sc[SC_RES] = res;
      const int it = fl[FL_ITER] + 1;
      fl[FL_ITER] = it;
      if (res < sc[SC_TOL]) {
        fl[FL_DONE] = 1;
        fl[FL_ITS] = it;
      }
    } break;
    case FIN_SUM: *out = t; break;
    case FIN_SQRT: *out = sqrt(t); break;
    default: break;
  }
}
void launch_fin1(hipStream_t s, int op, int nb, const RedWs& ws, double* sc, int* fl, double* out) {
  hipLaunchKernelGGL(k_fin1, dim3(1), dim3(kFinBlock), 0, s, op, nb, ws.partials, sc, fl, out);
}
// Whether the nb partials of a dot product are left for the kernel of `blocks`
// blocks that needs it: a launch less (2.4 to 3.3 us) against a fold in each of
// its blocks (0.4 us at 12x24x12, 1.2 at 50x100x50).  The line, in partials read
// by all its blocks together: 32x64x32 5.61 -> 5.30 ms for a design iteration,
// 50x100x50 (1.1 M) 8.63 -> 8.41; 64x128x64 (3.6 to 5 M) 10.57 -> 10.80.
constexpr long long kLateReads = 1 << 21;
static bool late_fold(const RedWs& ws, int nb, long long blocks) {
  static_assert(kLateAt + 4 * kFinBlock <= kMaxPartials, "room for a left p.q");
  // (at most kMaxPartials blocks: the kernels that fold take one element per thread)
  return ws.late && nb <= 4 * kFinBlock && blocks <= kMaxPartials && nb * blocks <= kLateReads;
}
void launch_fin_zr(hipStream_t s, int nb, long long n, const RedWs& ws, double* sc, int* fl) {
  const bool late = late_fold(ws, nb, stream_blocks(n));
  if (ws.late) ws.late->zr = late ? nb : 0;
  if (!late) launch_fin1(s, FIN_ZR_LOOP, nb, ws, sc, fl, nullptr);
}
static void fin1(hipStream_t s, int op, int nb, const RedWs& ws, double* sc, int* fl, double* out) {
  launch_fin1(s, op, nb, ws, sc, fl, out);
}

__global__ __launch_bounds__(kBlock) void k_fin_max(int nb, const double* __restrict__ partials, double* out) {
  const double m = fold_max(partials, nb);
  if (threadIdx.x == 0) *out = m;
}

// =========================================================================
// K*u on the finest level (Solving_KbyU_MatrixFree, 641-726), through the
// sum-factorised kernel of t3x_applyk_sf.hip.  The fixed DOFs are handled as
// P_free K(E) P_free + I_fixed — identical to the per-element
// uniqueKesFree_*E + uniqueKesFixed_ construction (1338-1437, 703-715): the
// fixed rows/cols of every touching element are zero and the 1/nAdj diagonal
// entries of the touching elements add up to 1.
// =========================================================================
void launch_apply_K(hipStream_t s, const Geo& g, const SfCoef& cf, const double* E, const uint8_t* fix,
                    const double* u, double* y, const RedWs& ws, double* sc, const int* fl, bool pcgStep) {
  const int nb = applyk_sf_blocks(g);
  const bool late = pcgStep && late_fold(ws, nb, stream_blocks(3 * g.NN));
  launch_apply_K_sf(s, g, cf, E, fix, u, y, pcgStep ? ws.partials + (late ? kLateAt : 0) : nullptr, fl);
  if (ws.late) ws.late->pq = late ? nb : 0;
  if (pcgStep && !late) fin1(s, FIN_PQ, nb, ws, sc, (int*)fl, nullptr);
}

// =========================================================================
// Jacobi diagonals (1001-1050).
// =========================================================================
__global__ void k_diag_fine(Geo g, const double* __restrict__ Ke, const double* __restrict__ E,
                            const uint8_t* __restrict__ fix, const uint8_t* __restrict__ nmask,
                            double* __restrict__ diag) {
  const long long n = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (n >= g.NN) return;
  double d[3] = {0.0, 0.0, 0.0};
  if (nmask[n]) {
    int iy, ix, iz;
    node_yxz(n, g, iy, ix, iz);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int dy = c & 1, dx = (c >> 1) & 1, dz = c >> 2;
      const int cy = iy - dy, cx = ix - dx, cz = iz - dz;
      if (!cell_in(g, cy, cx, cz)) continue;
      const double Ee = E[nidx(g, cy, cx, cz)];
      if (Ee == 0.0) continue;
      const int jn = loc_index(dy, dx, dz);
#pragma unroll
      for (int k = 0; k < 3; ++k) d[k] += Ke[(3 * jn + k) * 25] * Ee;
    }
    const uint8_t f = fix[n];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (f & (1 << k)) d[k] = 1.0;  // sum over touching elements of 1/nAdj
  } else {
    d[0] = d[1] = d[2] = 1.0;  // never used: vectors are 0 off the domain
  }
  diag[n] = d[0];
  diag[g.NN + n] = d[1];
  diag[2 * g.NN + n] = d[2];
}

void launch_diag_fine(hipStream_t s, const Geo& g, const double* Ke, const double* E, const uint8_t* fix,
                      const uint8_t* nmask, double* diag) {
  hipLaunchKernelGGL(k_diag_fine, dim3(grid_for(g.NN)), dim3(kBlock), 0, s, g, Ke, E, fix, nmask, diag);
}

__global__ void k_diag_coarse(Geo g, const double* __restrict__ Ks, const uint8_t* __restrict__ emask,
                              const uint8_t* __restrict__ nmask, double* __restrict__ diag) {
  const long long n = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (n >= g.NN) return;
  double d[3] = {0.0, 0.0, 0.0};
  if (nmask[n]) {
    int iy, ix, iz;
    node_yxz(n, g, iy, ix, iz);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int dy = c & 1, dx = (c >> 1) & 1, dz = c >> 2;
      const int cy = iy - dy, cx = ix - dx, cz = iz - dz;
      if (!cell_in(g, cy, cx, cz)) continue;
      const long long ce = nidx(g, cy, cx, cz);
      if (!emask[ce]) continue;
      const int jn = loc_index(dy, dx, dz);
#pragma unroll
      for (int k = 0; k < 3; ++k) d[k] += Ks[(size_t)tri_index(3 * jn + k, 3 * jn + k) * g.NN + ce];
    }
  } else {
    d[0] = d[1] = d[2] = 1.0;
  }
  diag[n] = d[0];
  diag[g.NN + n] = d[1];
  diag[2 * g.NN + n] = d[2];
}

void launch_diag_coarse(hipStream_t s, const Geo& g, const double* Ks, const uint8_t* emask,
                        const uint8_t* nmask, double* diag) {
  hipLaunchKernelGGL(k_diag_coarse, dim3(grid_for(g.NN)), dim3(kBlock), 0, s, g, Ks, emask, nmask, diag);
}

// =========================================================================
// Galerkin cell matrices (926-996).
//
// Level 2 (span 4, no BC child): Ks_c = sum_ss E_ss T_ss, T_ss = Q_ss^T Ke Q_ss
// precomputed on the host (64 x 300 upper-triangle entries, 950-954, 972-976).
// =========================================================================
// As a GEMM on v_mfma_f64_16x16x4: A = T^T (300 entries in 19 blocks of 16
// rows; K = the span^3 children in steps of 4), B = the children's moduli of
// 16 coarse cells (staged in LDS), D = 16 entries x 16 cells, stored straight
// into the entry-major Ks.  A work-group owns 64 consecutive coarse cells;
// wave w holds the A fragments of entry blocks w, w+4, ... in registers, one
// block at a time, and applies them to the 4 groups of 16 cells.  Cells that
// are void or padding get 0 (all their children's moduli are 0); the cells
// with a BC child are overwritten afterwards by k_galerkin_l2_bc.
constexpr int kL2Cells = 64;  // coarse cells per work-group
typedef double l2d4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_galerkin_l2(Geo gf, Geo gc, int span, const double* __restrict__ T,
                                                     const double* __restrict__ E, double* __restrict__ Ks) {
  const int s3 = span * span * span;  // 64 (span 4) or 8 (span 2)
  __shared__ double sE[64][kL2Cells + 1];  // [child][cell]
  const long long c0 = (long long)blockIdx.x * kL2Cells;
  for (int t = threadIdx.x; t < s3 * kL2Cells; t += 256) {
    const int j = t % kL2Cells, ss = t / kL2Cells;
    const long long cc = c0 + j;
    double v = 0.0;
    if (cc < gc.NN) {
      int cy, cx, cz;
      node_yxz(cc, gc, cy, cx, cz);
      if (cy < gc.ny && cx < gc.nx && cz < gc.nz) {
        const int ly = ss % span, lx = (ss / span) % span, lz = ss / (span * span);
        v = E[nidx(gf, span * cy + ly, span * cx + lx, span * cz + lz)];
      }
    }
    sE[ss][j] = v;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, kq = lane >> 4;
  const int nkb = s3 / 4;
  for (int m = wave; m * 16 < kTri; m += 4) {
    const int row = 16 * m + i;
    double a[16];
#pragma unroll
    for (int kb = 0; kb < 16; ++kb) a[kb] = (kb < nkb && row < kTri) ? T[(size_t)(4 * kb + kq) * kTri + row] : 0.0;
#pragma unroll
    for (int grp = 0; grp < kL2Cells / 16; ++grp) {
      l2d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kb = 0; kb < 16; ++kb)
        if (kb < nkb) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kb], sE[4 * kb + kq][16 * grp + i], acc, 0, 0, 0);
      // D[r][c] at lane c + 16 (r % 4), register r / 4
      const long long cc = c0 + 16 * grp + i;
      if (cc < gc.NN) {
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int k = 16 * m + kq + 4 * r4;
          if (k < kTri) Ks[(size_t)k * gc.NN + cc] = acc[r4];
        }
      }
    }
  }
}

void launch_galerkin_l2(hipStream_t s, const Geo& gf, const Geo& gc, int span, const double* T, const double* E,
                        const uint8_t* emaskC, const uint8_t* bcFlagC, double* Ks) {
  (void)emaskC;
  (void)bcFlagC;
  const int nb = (int)((gc.NN + kL2Cells - 1) / kL2Cells);
  hipLaunchKernelGGL(k_galerkin_l2, dim3(nb), dim3(256), 0, s, gf, gc, span, T, E, Ks);
}

// Interpolation weight of coarse local node J at fine child-local node a for
// child (ly,lx,lz) of a span-s cell: tensor product of 1-D hat weights.
__device__ __forceinline__ double hat_w(int span, int ly, int lx, int lz, int a, int J) {
  const int ty = ly + kLocDy[a], tx = lx + kLocDx[a], tz = lz + kLocDz[a];
  const double inv = 1.0 / span;
  const double wy = kLocDy[J] ? ty * inv : (span - ty) * inv;
  const double wx = kLocDx[J] ? tx * inv : (span - tx) * inv;
  const double wz = kLocDz[J] ? tz * inv : (span - tz) * inv;
  return wy * wx * wz;
}

// Level 2 cells with a child that touches a fixed node (961-971): children get
// E * P_free Ke P_free + diag(1/nAdj) on their fixed DOFs, then R += Q^T Kc Q
// with the Kronecker structure Q = N (x) I3.  One work-group per cell takes
// kBcKids children at a time, 72 threads each: thread (row, c') forms the 8
// entries T[row][3J + c'] = sum_b Kc[row][3b + c'] N[b][J], thread (q, c) the 8
// entries sum_a N[a][I] T[3a + c][q], from 8 values and with the hat weights in
// registers; then the children's entries are added in the
// children's order.  The cell's moduli, masks, node fixations and adjacency
// counts are staged once, in one memory round trip.
// Bound: a cell's latency chain (38 us: staging, then 8 rounds of 8 children).
// 277 -> 38 us at 50x100x50 (225 cells), 1.00 -> 0.58 ms at 256x512x256 (4,225
// cells, one group per CU by its 126 VGPRs; bounded to two it spills, 0.78 ms)
// against the whole group on one child at a time, one entry per thread and
// its loads behind four barriers.
constexpr int kBcKids = 8;
constexpr int kBcThreads = 72 * kBcKids;
__global__ __launch_bounds__(kBcThreads) void k_galerkin_l2_bc(Geo gf, Geo gc, int span,
                                                               const int* __restrict__ bcCells,
                                                               const double* __restrict__ Ke,
                                                               const double* __restrict__ E,
                                                               const uint8_t* __restrict__ emaskF,
                                                               const uint8_t* __restrict__ fix,
                                                               double* __restrict__ Ks) {
  __shared__ double shS[kBcKids][24][25];  // the children's entries [q][p]
  __shared__ double shT[kBcKids][24][25];
  __shared__ double shE[64];
  __shared__ uint8_t shM[64];
  __shared__ uint8_t shFix[125];
  __shared__ double shAdj[125];
  const int tid = threadIdx.x;
  const long long cc = bcCells[blockIdx.x];
  int cy, cx, cz;
  node_yxz(cc, gc, cy, cx, cz);
  const int s3 = span * span * span, sn = span + 1;
  const int kid = tid / 72, e = tid % 72, row = e / 3, cp = e % 3;
  double ke[8];  // this thread's row entries of Ke
#pragma unroll
  for (int b = 0; b < 8; ++b) ke[b] = Ke[row * 24 + 3 * b + cp];
  if (tid < s3) {
    const long long fe =
        nidx(gf, span * cy + tid % span, span * cx + (tid / span) % span, span * cz + tid / (span * span));
    shE[tid] = E[fe];
    shM[tid] = emaskF[fe];
  }
  if (tid < sn * sn * sn) {
    const int ny_ = span * cy + tid % sn, nx_ = span * cx + (tid / sn) % sn, nz_ = span * cz + tid / (sn * sn);
    shFix[tid] = fix[nidx(gf, ny_, nx_, nz_)];
    int cnt = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int qy = ny_ - (c & 1), qx = nx_ - ((c >> 1) & 1), qz = nz_ - (c >> 2);
      if (cell_in(gf, qy, qx, qz) && emaskF[nidx(gf, qy, qx, qz)]) ++cnt;
    }
    shAdj[tid] = (double)cnt;
  }
  __syncthreads();
  // entry tid of the upper triangle, t = tri_index(tp, tq)
  int tq = (int)((sqrtf(8.f * tid + 1.f) - 1.f) * 0.5f);
  tq += (tq + 1) * (tq + 2) / 2 <= tid;
  tq -= tq * (tq + 1) / 2 > tid;
  const int tp = tid - tq * (tq + 1) / 2;
  double acc = 0.0;
  const double inv = 1.0 / span;
  for (int s0 = 0; s0 < s3; s0 += kBcKids) {  // span^3 is a multiple of kBcKids
    const int ss = s0 + kid;
    const bool on = shM[ss];  // a void child contributes nothing
    const int ly = ss % span, lx = (ss / span) % span, lz = ss / (span * span);
    // hat weights per axis, [child node offset][coarse node offset]
    double wy[2][2], wx[2][2], wz[2][2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      wy[d][1] = (ly + d) * inv, wy[d][0] = (span - (ly + d)) * inv;
      wx[d][1] = (lx + d) * inv, wx[d][0] = (span - (lx + d)) * inv;
      wz[d][1] = (lz + d) * inv, wz[d][0] = (span - (lz + d)) * inv;
    }
    auto N = [&](int a, int J) {
      return wy[kLocDy[a]][kLocDy[J]] * wx[kLocDx[a]][kLocDx[J]] * wz[kLocDz[a]][kLocDz[J]];
    };
    if (on) {
      auto node = [&](int j) { return ly + kLocDy[j] + sn * (lx + kLocDx[j] + sn * (lz + kLocDz[j])); };
      // thread (row, cp): Kc's entries (row, 3b + cp) and from them its 8 entries of T
      const int nr = node(row / 3), cr = row % 3;
      const bool fr = (shFix[nr] >> cr) & 1;
      double s[8] = {};
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const bool fq = (shFix[node(b)] >> cp) & 1;
        double v = (fr || fq) ? 0.0 : ke[b] * shE[ss];
        if (row == 3 * b + cp && fr) v = v + 1.0 / shAdj[nr];
#pragma unroll
        for (int J = 0; J < 8; ++J) s[J] += v * N(b, J);
      }
#pragma unroll
      for (int J = 0; J < 8; ++J) shT[kid][row][3 * J + cp] = s[J];
    }
    __syncthreads();
    if (on) {  // thread (q = row, c = cp): the entries (3I + c, q)
      double s[8] = {};
#pragma unroll
      for (int a = 0; a < 8; ++a) {
        const double t = shT[kid][3 * a + cp][row];
#pragma unroll
        for (int I = 0; I < 8; ++I) s[I] += N(a, I) * t;
      }
#pragma unroll
      for (int I = 0; I < 8; ++I) shS[kid][row][3 * I + cp] = s[I];
    }
    __syncthreads();
    if (tid < kTri) {
#pragma unroll
      for (int k = 0; k < kBcKids; ++k)
        if (shM[s0 + k]) acc += shS[k][tq][tp];
    }
    __syncthreads();
  }
  if (tid < kTri) Ks[(size_t)tid * gc.NN + cc] = acc;
}

void launch_galerkin_l2_bc(hipStream_t s, const Geo& gf, const Geo& gc, int span, int nBc, const int* bcCells,
                           const double* Ke, const double* E, const uint8_t* emaskF, const uint8_t* fix,
                           double* Ks) {
  if (nBc <= 0) return;
  hipLaunchKernelGGL(k_galerkin_l2_bc, dim3(nBc), dim3(kBcThreads), 0, s, gf, gc, span, bcCells, Ke, E, emaskF, fix,
                     Ks);
}

// Level >= 3 (span 2): Ks_c = sum over 8 children of Q^T Ks_child Q (980-995).
// With Q = N (x) I3 (N: 8x8 hat weights of the child position) every 8x8
// component block (c, c') of the result is N^T K^{cc'} N; the 6 blocks with
// c <= c' give the 300 stored entries.  A work-group takes 16 consecutive
// coarse cells, one thread per (cell, block, column Q), the 48 threads of a
// cell adjacent (so a wave's LDS reads of a child matrix are broadcasts): per
// child it forms the column T = K^{cc'} N(:, Q) in registers and adds N^T T
// to its 8 accumulators.  The children's matrices are staged in LDS
// (expanded to 24x24, padded), with global loads shared by neighbouring cells.
constexpr int kGcCells = 16;
constexpr int kGcThreads = kGcCells * 48;
__global__ __launch_bounds__(kGcThreads) void k_galerkin_coarse(Geo gf, Geo gc, const double* __restrict__ KsF,
                                                                double* __restrict__ KsC) {
  __shared__ double sK[kGcCells][24][25];
  __shared__ double sN[8][8];
  const long long c0 = (long long)blockIdx.x * kGcCells;
  const int tid = threadIdx.x, j = tid / 48, ci = tid % 48;
  const int pr = ci / 8, Q = ci % 8;  // block pr: (0,0) (1,1) (2,2) (0,1) (0,2) (1,2)
  const int c = pr < 3 ? pr : (pr == 5 ? 1 : 0);
  const int c2 = pr < 3 ? pr : (pr == 3 ? 1 : 2);
  const long long cc = c0 + j;
  double acc[8];
#pragma unroll
  for (int P = 0; P < 8; ++P) acc[P] = 0.0;
  for (int ch = 0; ch < 8; ++ch) {
    const int ly = ch & 1, lx = (ch >> 1) & 1, lz = ch >> 2;
    __syncthreads();  // previous child's sK and sN consumed
    for (int e2 = tid; e2 < kTri * kGcCells; e2 += kGcThreads) {
      const int jj = e2 % kGcCells, k = e2 / kGcCells;
      const long long ccj = c0 + jj;
      double v = 0.0;
      if (ccj < gc.NN) {
        int qy, qx, qz;
        node_yxz(ccj, gc, qy, qx, qz);
        if (qy < gc.ny && qx < gc.nx && qz < gc.nz)
          v = KsF[(size_t)k * gf.NN + nidx(gf, 2 * qy + ly, 2 * qx + lx, 2 * qz + lz)];
      }
      int q = (int)((sqrtf(8.f * k + 1.f) - 1.f) * 0.5f);  // k = tri_index(p, q), p <= q
      q += (q + 1) * (q + 2) / 2 <= k;
      q -= q * (q + 1) / 2 > k;
      const int p = k - q * (q + 1) / 2;
      sK[jj][p][q] = v;
      sK[jj][q][p] = v;
    }
    if (tid < 64) sN[tid / 8][tid % 8] = hat_w(2, ly, lx, lz, tid / 8, tid % 8);  // N[a][J]
    __syncthreads();
    double Tc[8];
#pragma unroll
    for (int A = 0; A < 8; ++A) {
      double v = 0.0;
#pragma unroll
      for (int B = 0; B < 8; ++B) v += sK[j][3 * A + c][3 * B + c2] * sN[B][Q];
      Tc[A] = v;
    }
#pragma unroll
    for (int P = 0; P < 8; ++P) {
      double v = acc[P];
#pragma unroll
      for (int A = 0; A < 8; ++A) v += sN[A][P] * Tc[A];
      acc[P] = v;
    }
  }
  if (cc >= gc.NN) return;
#pragma unroll
  for (int P = 0; P < 8; ++P) {
    if (c == c2 && P > Q) continue;  // diagonal blocks: upper triangle only
    KsC[(size_t)tri_index(3 * P + c, 3 * Q + c2) * gc.NN + cc] = acc[P];
  }
}

void launch_galerkin_coarse(hipStream_t s, const Geo& gf, const Geo& gc, const double* KsF, const uint8_t* emaskF,
                            const uint8_t* emaskC, double* KsC) {
  (void)emaskF;
  (void)emaskC;
  const int nb = (int)((gc.NN + kGcCells - 1) / kGcCells);
  hipLaunchKernelGGL(k_galerkin_coarse, dim3(nb), dim3(kGcThreads), 0, s, gf, gc, KsF, KsC);
}

// Multigrid transfers (783-814) live in t3x_mg.hip.

// =========================================================================
// Coarsest level: assembly of its band (1052-1065; factored and solved in t3x_coarse.hip).
// Band storage: row i holds L(i, i-k) at band[i*W + k], W = bw+1.
// =========================================================================
// Assembly of the lower band: one thread per (coarsest node a, node b of its
// 3x3x3 neighbourhood) sums the 3x3 entries of rows a, columns b over the
// cells that hold both, in the cells' order, and writes them once.  Bound: one
// memory round trip per shared cell.  (One thread per node adding its 8 cells'
// 576 products into the band one after the other: 105 -> 8 us at 12x24x12, 250
// -> 19 us at 128x256x128.)
__global__ __launch_bounds__(kBlock) void k_band_assemble(Geo g, const double* __restrict__ Ks,
                                                          const uint8_t* __restrict__ emask,
                                                          const int* __restrict__ nodePos, int bw,
                                                          double* __restrict__ band) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= 27 * g.NN) return;
  const int o = (int)(t / g.NN);  // the neighbours of one offset adjacent: coalesced Ks reads
  const long long n = t - o * g.NN;
  const int pa = nodePos[n];
  if (pa < 0) return;
  int iy, ix, iz;
  node_yxz(n, g, iy, ix, iz);
  const int by = iy + o % 3 - 1, bx = ix + (o / 3) % 3 - 1, bz = iz + o / 9 - 1;
  if (by < 0 || bx < 0 || bz < 0 || by >= g.NY || bx >= g.NX || bz >= g.NZ) return;
  const int pb = nodePos[nidx(g, by, bx, bz)];
  if (pb < 0 || pb > pa) return;  // lower triangle
  double acc[3][3] = {};
  bool any = false;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int cy = iy - (c & 1), cx = ix - ((c >> 1) & 1), cz = iz - (c >> 2);
    const int dy = by - cy, dx = bx - cx, dz = bz - cz;
    if ((unsigned)dy > 1u || (unsigned)dx > 1u || (unsigned)dz > 1u) continue;  // b is no corner of this cell
    if (!cell_in(g, cy, cx, cz)) continue;
    const long long ce = nidx(g, cy, cx, cz);
    if (!emask[ce]) continue;
    any = true;
    const int ja = loc_index(c & 1, (c >> 1) & 1, c >> 2), jb = loc_index(dy, dx, dz);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int kk = 0; kk < 3; ++kk) acc[k][kk] += Ks[(size_t)tri_index(3 * ja + k, 3 * jb + kk) * g.NN + ce];
  }
  if (!any) return;
  const long long W = bw + 1;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int kk = 0; kk < 3; ++kk) {
      const long long row = 3LL * pa + k, col = 3LL * pb + kk;
      if (col <= row) band[row * W + (row - col)] = acc[k][kk];
    }
}
void launch_band_assemble(hipStream_t s, const Geo& g, const double* Ks, const uint8_t* emask, const int* nodePos,
                          int bw, double* band, long long nBand) {
  launch_fill(s, band, 0.0, nBand);
  hipLaunchKernelGGL(k_band_assemble, dim3(grid_for(27 * g.NN)), dim3(kBlock), 0, s, g, Ks, emask, nodePos, bw, band);
}

// =========================================================================
// Vector kernels of the PCG (600-639).
// =========================================================================
__global__ void k_fill(double* p, double v, long long n) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) p[i] = v;
}
struct Vals8 {
  double v[8];
};
__global__ void k_set_vals(double* dst, int n, Vals8 vals) {
  if ((int)threadIdx.x < n) dst[threadIdx.x] = vals.v[threadIdx.x];
}
void launch_set_vals(hipStream_t s, double* dst, int n, const double* vals) {
  Vals8 v{};
  for (int i = 0; i < n && i < 8; ++i) v.v[i] = vals[i];
  hipLaunchKernelGGL(k_set_vals, dim3(1), dim3(64), 0, s, dst, n < 8 ? n : 8, v);
}
__global__ void k_set_int(int* dst, int v) { *dst = v; }
void launch_set_int(hipStream_t s, int* dst, int v) { hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, s, dst, v); }
void launch_fill(hipStream_t s, double* p, double v, long long n) {
  hipLaunchKernelGGL(k_fill, dim3(stream_blocks(n)), dim3(kBlock), 0, s, p, v, n);
}
__global__ void k_copy(double* d, const double* a, long long n) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) d[i] = a[i];
}
void launch_copy(hipStream_t s, double* dst, const double* src, long long n) {
  hipLaunchKernelGGL(k_copy, dim3(stream_blocks(n)), dim3(kBlock), 0, s, dst, src, n);
}
__global__ void k_sub(double* r, const double* b, const double* q, long long n) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
    r[i] = b[i] - q[i];
}
void launch_sub(hipStream_t s, double* r, const double* b, const double* q, long long n) {
  hipLaunchKernelGGL(k_sub, dim3(stream_blocks(n)), dim3(kBlock), 0, s, r, b, q, n);
}

__global__ __launch_bounds__(kBlock) void k_dot(const double* __restrict__ a, const double* __restrict__ b,
                                                long long n, RedWs ws, double* out, int sq) {
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
    s += a[i] * b[i];
  double v[1] = {s};
  write_partials<1>(v, ws.partials);
  (void)out;
  (void)sq;
}
void launch_norm2(hipStream_t s, const double* v, long long n, const RedWs& ws, double* out) {
  hipLaunchKernelGGL(k_dot, dim3(red1_blocks(n)), dim3(kBlock), 0, s, v, v, n, ws, out, 1);
  fin1(s, FIN_SQRT, red1_blocks(n), ws, nullptr, nullptr, out);
}
void launch_dot(hipStream_t s, const double* a, const double* b, long long n, const RedWs& ws, double* out) {
  hipLaunchKernelGGL(k_dot, dim3(red1_blocks(n)), dim3(kBlock), 0, s, a, b, n, ws, out, 0);
  fin1(s, FIN_SUM, red1_blocks(n), ws, nullptr, nullptr, out);
}

// y += lambda p ; r -= lambda q ; resnorm = ||r|| / ||b|| ; convergence flag.
// r -= lambda q (617) with the r.r reduction.  With xj given (FP32 'Standard'
// V-cycle), also the first fine Jacobi step of the next preconditioner
// application, xj = omega r / dj (757), while r is in registers.
__global__ __launch_bounds__(kBlock) void k_pcg_update(double* __restrict__ r, const double* __restrict__ q,
                                                       long long n, RedWs ws, double* sc, int* fl,
                                                       const float* __restrict__ dj, float* __restrict__ xj,
                                                       double omega, Act act, double* part) {
  if (fl[FL_DONE]) return;
  // y += lambda p (616) is deferred to k_pcg_pupdate, which reads p anyway
  const double lambda = sc[SC_LAMBDA];
  double rr = 0.0;
  const long long m = act_items(act, n);
  const int nc = act_ncomp(act, n);
  for (long long g = (long long)blockIdx.x * kBlock + threadIdx.x; g < m; g += (long long)gridDim.x * kBlock) {
    const long long b = act_node(act, g);
    if (act.list && b >= act.NN) continue;
    for (int c = 0; c < nc; ++c) {
      const long long i = b + c * act.NN;
      const double ri = r[i] - lambda * q[i];     // 617
      r[i] = ri;
      rr += ri * ri;
      if (xj) {
        const double dd = (double)dj[i];
        xj[i] = dd != 0.0 ? (float)(omega * (ri / dd)) : 0.f;
      }
    }
  }
  double v[1] = {rr};
  write_partials<1>(v, part);
}
// the same with p.q still to be folded
__global__ __launch_bounds__(kBlock) void k_pcg_update_late(double* __restrict__ r, const double* __restrict__ q,
                                                            long long n, RedWs ws, double* sc, int* fl,
                                                            const float* __restrict__ dj, float* __restrict__ xj,
                                                            double omega, Act act, double* part, int nbPQ) {
  if (fl[FL_DONE]) return;
  // y += lambda p (616) is deferred to k_pcg_pupdate, which reads p anyway
  const long long m = act_items(act, n);
  const int nc = act_ncomp(act, n);
  const long long g = (long long)blockIdx.x * kBlock + threadIdx.x;  // one item per thread
  const long long b = g < m ? act_node(act, g) : 0;
  const bool on = g < m && !(act.list && b >= act.NN);
  const double r0 = on ? r[b] : 0.0, q0 = on ? q[b] : 0.0;  // on their way while the fold is made
  // FIN_PQ, in every block
  const double t = fold_here(ws.partials + kLateAt, nbPQ), zr = sc[SC_ZRN], lambda = zr / t;
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // (read by later kernels only)
    sc[SC_PQ] = t;
    sc[SC_LAMBDA] = lambda;
    sc[SC_ZR] = zr;
  }
  double rr = 0.0;
  auto element = [&](long long i, double rOld, double qi) {
    const double ri = rOld - lambda * qi;  // 617
    r[i] = ri;
    rr += ri * ri;
    if (xj) {
      const double dd = (double)dj[i];
      xj[i] = dd != 0.0 ? (float)(omega * (ri / dd)) : 0.f;
    }
  };
  if (on) {
    element(b, r0, q0);
    for (int c = 1; c < nc; ++c) element(b + c * act.NN, r[b + c * act.NN], q[b + c * act.NN]);
  }
  double v[1] = {rr};
  write_partials<1>(v, part);
}
void launch_pcg_update(hipStream_t s, double* y, double* r, const double* p, const double* q, long long n,
                       const RedWs& ws, double* sc, int* fl, const float* dj, float* xj, double omega, Act act,
                       int rrBlocks) {
  (void)y;
  (void)p;
  const int nb = red1_blocks(act_items(act, n));
  const bool late = rrBlocks && late_fold(ws, nb, rrBlocks);
  if (ws.late) ws.late->rr = late ? nb : 0;
  double* part = ws.partials + (late ? kLateRR : 0);
  const int nbPQ = ws.late ? ws.late->pq : 0;
  if (nbPQ)
    hipLaunchKernelGGL(k_pcg_update_late, dim3(nb), dim3(kBlock), 0, s, r, q, n, ws, sc, fl, dj, xj, omega, act, part,
                       nbPQ);
  else
    hipLaunchKernelGGL(k_pcg_update, dim3(nb), dim3(kBlock), 0, s, r, q, n, ws, sc, fl, dj, xj, omega, act, part);
  if (!late) fin1(s, FIN_RR, nb, ws, sc, fl, nullptr);
}

// y += lambda p (616) for the iteration just finished, then p = z + beta p (630).
template <typename TZ>
__global__ void k_pcg_pupdate(double* __restrict__ y, double* __restrict__ p, const TZ* __restrict__ z, long long n,
                              const double* sc, const int* fl, Act act) {
  if (fl[FL_DONE]) return;
  const double beta = sc[SC_BETA], lambda = sc[SC_LAMBDA];
  const long long m = act_items(act, n);
  const int nc = act_ncomp(act, n);
  for (long long g = (long long)blockIdx.x * kBlock + threadIdx.x; g < m; g += (long long)gridDim.x * kBlock) {
    const long long b = act_node(act, g);
    if (act.list && b >= act.NN) continue;
    for (int c = 0; c < nc; ++c) {
      const long long i = b + c * act.NN;
      const double pi = p[i];
      y[i] = y[i] + lambda * pi;
      p[i] = (double)z[i] + beta * pi;
    }
  }
}
// the same with z.r still to be folded (FIN_ZR_LOOP, in every block); one item per thread
template <typename TZ>
__global__ __launch_bounds__(kBlock) void k_pcg_pupdate_late(double* __restrict__ y, double* __restrict__ p,
                                                             const TZ* __restrict__ z, long long n, RedWs ws,
                                                             double* sc, const int* fl, Act act, int nbZR) {
  if (fl[FL_DONE]) return;
  const int nc = act_ncomp(act, n);
  const long long g = (long long)blockIdx.x * kBlock + threadIdx.x;
  const bool in = g < act_items(act, n);
  const long long b = in ? act_node(act, g) : 0;
  const bool on = in && !(act.list && b >= act.NN);
  const double p0 = on ? p[b] : 0.0, y0 = on ? y[b] : 0.0, z0 = on ? (double)z[b] : 0.0;  // beside the fold
  const double t = fold_here(ws.partials, nbZR), beta = t / sc[SC_ZR], lambda = sc[SC_LAMBDA];
  if (blockIdx.x == 0 && threadIdx.x == 0) sc[SC_ZRN] = t;  // (read by later kernels only)
  if (!on) return;
  y[b] = y0 + lambda * p0;
  p[b] = z0 + beta * p0;
  for (int c = 1; c < nc; ++c) {
    const long long i = b + c * act.NN;
    const double pi = p[i];
    y[i] = y[i] + lambda * pi;
    p[i] = (double)z[i] + beta * pi;
  }
}
template <typename TZ>
static void pcg_pupdate(hipStream_t s, double* y, double* p, const TZ* z, long long n, const RedWs& ws, double* sc,
                        const int* fl, Act act) {
  const dim3 grid(stream_blocks(act_items(act, n)));
  const int nbZR = ws.late ? ws.late->zr : 0;
  if (nbZR) hipLaunchKernelGGL(k_pcg_pupdate_late<TZ>, grid, dim3(kBlock), 0, s, y, p, z, n, ws, sc, fl, act, nbZR);
  else hipLaunchKernelGGL(k_pcg_pupdate<TZ>, grid, dim3(kBlock), 0, s, y, p, z, n, sc, fl, act);
}
void launch_pcg_pupdate(hipStream_t s, double* y, double* p, const double* z, long long n, const RedWs& ws, double* sc,
                        const int* fl, Act act) {
  pcg_pupdate(s, y, p, z, n, ws, sc, fl, act);
}
// After the loop: the converging iteration skipped its p-update, so its
// y += lambda p is applied here (no-op if the solve hit maxIT).
__global__ void k_pcg_finish(double* __restrict__ y, const double* __restrict__ p, long long n, const double* sc,
                             const int* fl, Act act) {
  if (!fl[FL_DONE]) return;
  const double lambda = sc[SC_LAMBDA];
  const long long m = act_items(act, n);
  const int nc = act_ncomp(act, n);
  for (long long g = (long long)blockIdx.x * kBlock + threadIdx.x; g < m; g += (long long)gridDim.x * kBlock) {
    const long long b = act_node(act, g);
    if (act.list && b >= act.NN) continue;
    for (int c = 0; c < nc; ++c) {
      const long long i = b + c * act.NN;
      y[i] = y[i] + lambda * p[i];
    }
  }
}
void launch_pcg_finish(hipStream_t s, double* y, const double* p, long long n, const double* sc, const int* fl,
                       Act act) {
  hipLaunchKernelGGL(k_pcg_finish, dim3(stream_blocks(act_items(act, n))), dim3(kBlock), 0, s, y, p, n, sc, fl, act);
}

// Mixed precision: the V-cycle output z is FP32; y, r, p and scalars FP64.
void launch_pcg_pupdate(hipStream_t s, double* y, double* p, const float* z, long long n, const RedWs& ws, double* sc,
                        const int* fl, Act act) {
  pcg_pupdate(s, y, p, z, n, ws, sc, fl, act);
}
template <typename TD, typename TS>
__global__ void k_convert(TD* __restrict__ dst, const TS* __restrict__ src, long long n) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
    dst[i] = (TD)src[i];
}
void launch_convert(hipStream_t s, float* dst, const double* src, long long n) {
  hipLaunchKernelGGL((k_convert<float, double>), dim3(stream_blocks(n)), dim3(kBlock), 0, s, dst, src, n);
}
void launch_convert(hipStream_t s, double* dst, const float* src, long long n) {
  hipLaunchKernelGGL((k_convert<double, float>), dim3(stream_blocks(n)), dim3(kBlock), 0, s, dst, src, n);
}

__global__ void k_pcg_init(double* sc, int* fl, double tol) {
  sc[SC_TOL] = tol;
  for (int i = 0; i < FL_COUNT; ++i) fl[i] = 0;
}
void launch_pcg_init(hipStream_t s, double* sc, int* fl, double tol) {
  hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(1), 0, s, sc, fl, tol);
}

// z = dinv .* r (889) with the fused z.r reduction; RR: the update before it left
// r.r to be folded here (then one element per thread).
template <bool RR>
__global__ __launch_bounds__(kBlock) void k_scale_diag(double* __restrict__ z, const double* __restrict__ dinv,
                                                       const double* __restrict__ r, long long n, RedWs ws,
                                                       const int* fl, RrFold rr) {
  if (!RR && fl && fl[FL_DONE]) return;  // RR: rr_fold looks
  double zr = 0.0;
  const long long i0 = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (RR) {
    const double r0 = i0 < n ? r[i0] : 0.0, d0 = i0 < n ? dinv[i0] : 0.0;  // beside the fold
    if (rr_fold(rr)) return;
    if (i0 < n) {
      const double zi = d0 * r0;
      z[i0] = zi;
      zr += zi * r0;
    }
  } else {
    for (long long i = i0; i < n; i += (long long)gridDim.x * kBlock) {
      const double zi = dinv[i] * r[i];
      z[i] = zi;
      zr += zi * r[i];
    }
  }
  double v[1] = {zr};
  write_partials<1>(v, ws.partials);
}
int scale_diag_blocks(long long n) { return stream_blocks(n); }
void launch_scale_diag(hipStream_t s, double* z, const double* dinv, const double* r, long long n,
                       const RedWs* ws, double* sc, const int* fl) {
  const RrFold rr{ws->partials + kLateRR, ws->late ? ws->late->rr : 0, sc, (int*)fl};
  if (fl && rr.nb)
    hipLaunchKernelGGL(k_scale_diag<true>, dim3(red1_blocks(n)), dim3(kBlock), 0, s, z, dinv, r, n, *ws, fl, rr);
  else
    hipLaunchKernelGGL(k_scale_diag<false>, dim3(red1_blocks(n)), dim3(kBlock), 0, s, z, dinv, r, n, *ws, fl, rr);
  if (!fl) fin1(s, FIN_ZR_INIT, red1_blocks(n), *ws, sc, (int*)fl, nullptr);
  else launch_fin_zr(s, red1_blocks(n), n, *ws, sc, (int*)fl);
}

__global__ void k_gather_compact(const int* __restrict__ map, int n, int ncomp, long long NN,
                                 const double* __restrict__ dense, double* __restrict__ compact) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= (long long)n * ncomp) return;
  const int i = (int)(t / ncomp), c = (int)(t % ncomp);
  compact[t] = dense[(size_t)c * NN + map[i]];
}
void launch_gather_compact(hipStream_t s, const int* map, int n, int ncomp, long long NN, const double* dense,
                           double* compact) {
  hipLaunchKernelGGL(k_gather_compact, dim3(grid_for((long long)n * ncomp)), dim3(kBlock), 0, s, map, n, ncomp, NN,
                     dense, compact);
}
__global__ void k_scatter_compact(const int* __restrict__ map, int n, int ncomp, long long NN,
                                  const double* __restrict__ compact, double* __restrict__ dense) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= (long long)n * ncomp) return;
  const int i = (int)(t / ncomp), c = (int)(t % ncomp);
  dense[(size_t)c * NN + map[i]] = compact[t];
}
void launch_scatter_compact(hipStream_t s, const int* map, int n, int ncomp, long long NN, const double* compact,
                            double* dense) {
  hipLaunchKernelGGL(k_scatter_compact, dim3(grid_for((long long)n * ncomp)), dim3(kBlock), 0, s, map, n, ncomp, NN,
                     compact, dense);
}

// =========================================================================
// PDE filter (816-917): scalar 8x8 Helmholtz kernel on the node grid.
// =========================================================================
__global__ void k_filter_e2n(Geo g, const uint8_t* __restrict__ emask, const double* __restrict__ src,
                             double* __restrict__ b) {
  const long long n = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (n >= g.NN) return;
  int iy, ix, iz;
  node_yxz(n, g, iy, ix, iz);
  double s = 0.0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int cy = iy - (c & 1), cx = ix - ((c >> 1) & 1), cz = iz - (c >> 2);
    if (!cell_in(g, cy, cx, cz)) continue;
    const long long ce = nidx(g, cy, cx, cz);
    if (emask[ce]) s += src[ce] * (1.0 / 8.0);  // 881-885
  }
  b[n] = s;
}
void launch_filter_e2n(hipStream_t s, const Geo& g, const uint8_t* emask, const double* src, double* b) {
  hipLaunchKernelGGL(k_filter_e2n, dim3(grid_for(g.NN)), dim3(kBlock), 0, s, g, emask, src, b);
}

// y = K_F u for the PDE filter's nodal operator: per node, the rows of the
// 8x8 filter kernel from its active cells.  3-D grid of 64x4 node columns,
// each thread walking zc node layers with a sliding 3x3x3 window of u and the
// masks of the 2x2x2 cells around the node in registers (32-bit offsets:
// 3 NN < 2^31 is checked at set-up).  pcgStep: per-block u.y partials.
constexpr int kFaY = 64, kFaX = 4;
__global__ __launch_bounds__(kFaY * kFaX) void k_filter_apply(Geo g, int zc, const double* __restrict__ kern,
                                                              const uint8_t* __restrict__ emask,
                                                              const double* __restrict__ u, double* __restrict__ y,
                                                              RedWs ws, const int* fl, int pcgStep) {
  if (fl && fl[FL_DONE]) return;
  const int iy = blockIdx.x * kFaY + threadIdx.x, ix = blockIdx.y * kFaX + threadIdx.y;
  const int z0 = blockIdx.z * zc, z1 = min(g.NZ, z0 + zc);
  const bool own = iy < g.NY && ix < g.NX;
  const int NY = g.NY, plane = g.NY * g.NX;
  // window: w[l][ky + 3 kx] = u(iy-1+ky, ix-1+kx, z-1+l); m[l][cy + 2 cx] = active cell (iy-1+cy, ix-1+cx, z-1+l)
  double w[3][9];
  bool m[2][4];
  auto load_u = [&](int z, double (&wl)[9]) {
#pragma unroll
    for (int kx = 0; kx < 3; ++kx)
#pragma unroll
      for (int ky = 0; ky < 3; ++ky) {
        const int yy = iy - 1 + ky, xx = ix - 1 + kx;
        const bool in = own && z >= 0 && z < g.NZ && yy >= 0 && xx >= 0 && yy < g.NY && xx < g.NX;
        wl[ky + 3 * kx] = in ? u[yy + NY * xx + plane * z] : 0.0;
      }
  };
  auto load_m = [&](int z, bool (&ml)[4]) {
#pragma unroll
    for (int cx = 0; cx < 2; ++cx)
#pragma unroll
      for (int cy = 0; cy < 2; ++cy) {
        const int yy = iy - 1 + cy, xx = ix - 1 + cx;
        const bool in = own && z >= 0 && z < g.nz && yy >= 0 && xx >= 0 && yy < g.ny && xx < g.nx;
        ml[cy + 2 * cx] = in && emask[yy + NY * xx + plane * z];
      }
  };
  load_u(z0 - 1, w[0]);
  load_u(z0, w[1]);
  load_m(z0 - 1, m[0]);
  double pq = 0.0;
  for (int z = z0; z < z1; ++z) {
    load_u(z + 1, w[2]);
    load_m(z, m[1]);
    if (own) {
      double acc = 0.0;
#pragma unroll
      for (int c = 0; c < 8; ++c) {  // cell (iy-dy, ix-dx, z-dz)
        const int dy = c & 1, dx = (c >> 1) & 1, dz = c >> 2;
        if (!m[1 - dz][(1 - dy) + 2 * (1 - dx)]) continue;
        const int jn = loc_index(dy, dx, dz);
        double sc = 0.0;
#pragma unroll
        for (int bq = 0; bq < 8; ++bq) {
          const int ky = 1 - dy + kLocDy[bq], kx = 1 - dx + kLocDx[bq], l = 1 - dz + kLocDz[bq];
          sc += w[l][ky + 3 * kx] * kern[jn * 8 + bq];
        }
        acc += sc;
      }
      y[iy + NY * ix + plane * z] = acc;
      pq += w[1][4] * acc;
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      w[0][i] = w[1][i];
      w[1][i] = w[2][i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) m[0][i] = m[1][i];
  }
  if (pcgStep) {
    __shared__ double sh[kFaY * kFaX / 64];
    const int t = threadIdx.x + kFaY * threadIdx.y;
    const double v = wave_sum(pq);
    if ((t & 63) == 0) sh[t >> 6] = v;
    __syncthreads();
    if (t == 0) {
      double s2 = 0.0;
      for (int k = 0; k < kFaY * kFaX / 64; ++k) s2 += sh[k];
      ws.partials[blockIdx.x + (size_t)gridDim.x * (blockIdx.y + (size_t)gridDim.y * blockIdx.z)] = s2;
    }
  }
}
// z chunk doubled until at most kMaxPartials work-groups; a node plane with
// more columns than that is refused at set-up (filter_plane_fits)
static dim3 filter_grid(const Geo& g, int& zc) {
  zc = 8;
  for (;;) {
    const dim3 d((g.NY + kFaY - 1) / kFaY, (g.NX + kFaX - 1) / kFaX, (g.NZ + zc - 1) / zc);
    if ((long long)d.x * d.y * d.z <= kMaxPartials || zc >= g.NZ) return d;
    zc *= 2;
  }
}
bool filter_plane_fits(int NY, int NX) {
  return (long long)((NY + kFaY - 1) / kFaY) * ((NX + kFaX - 1) / kFaX) <= kMaxPartials;
}
void launch_filter_apply(hipStream_t s, const Geo& g, const double* kern, const uint8_t* emask, const double* u,
                         double* y, const RedWs* ws, double* sc, const int* fl) {
  RedWs w{nullptr, nullptr};
  int step = 0;
  if (ws) { w = *ws; step = 1; }
  int zc = 8;
  const dim3 grid = filter_grid(g, zc);
  const int nb = (int)(grid.x * grid.y * grid.z);
  const bool late = step && late_fold(w, nb, stream_blocks(g.NN));
  RedWs at = w;
  if (late) at.partials += kLateAt;
  hipLaunchKernelGGL(k_filter_apply, grid, dim3(kFaY, kFaX), 0, s, g, zc, kern, emask, u, y, at, fl, step);
  if (w.late) w.late->pq = late ? nb : 0;
  if (step && !late) fin1(s, FIN_PQ, nb, w, sc, (int*)fl, nullptr);
}

__global__ void k_filter_n2e(Geo g, const uint8_t* __restrict__ emask, const double* __restrict__ u,
                             double* __restrict__ tar) {
  const long long n = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (n >= g.NN) return;
  if (!emask[n]) { tar[n] = 0.0; return; }
  int iy, ix, iz;
  node_yxz(n, g, iy, ix, iz);
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < 8; ++j) s += u[nidx(g, iy + kLocDy[j], ix + kLocDx[j], iz + kLocDz[j])];
  tar[n] = s * (1.0 / 8.0);  // 899-901
}
void launch_filter_n2e(hipStream_t s, const Geo& g, const uint8_t* emask, const double* u, double* tar) {
  hipLaunchKernelGGL(k_filter_n2e, dim3(grid_for(g.NN)), dim3(kBlock), 0, s, g, emask, u, tar);
}

__global__ void k_filter_diag(Geo g, const double* __restrict__ kern, const uint8_t* __restrict__ emask,
                              const uint8_t* __restrict__ nmask, double* __restrict__ dinv) {
  const long long n = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (n >= g.NN) return;
  if (!nmask[n]) { dinv[n] = 0.0; return; }
  int iy, ix, iz;
  node_yxz(n, g, iy, ix, iz);
  double s = 0.0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int dy = c & 1, dx = (c >> 1) & 1, dz = c >> 2;
    const int cy = iy - dy, cx = ix - dx, cz = iz - dz;
    if (!cell_in(g, cy, cx, cz) || !emask[nidx(g, cy, cx, cz)]) continue;
    s += kern[loc_index(dy, dx, dz) * 9];
  }
  dinv[n] = 1.0 / s;  // 867
}
void launch_filter_diag(hipStream_t s, const Geo& g, const double* kern, const uint8_t* emask,
                        const uint8_t* nmask, double* dinv) {
  hipLaunchKernelGGL(k_filter_diag, dim3(grid_for(g.NN)), dim3(kBlock), 0, s, g, kern, emask, nmask, dinv);
}

// =========================================================================
// Optimiser kernels.
// =========================================================================
__global__ void k_simp(long long n, const uint8_t* __restrict__ emask, const double* __restrict__ xPhys,
                       double Emin, double E0, double* __restrict__ E) {
  const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double x = xPhys[i];
  E[i] = emask[i] ? Emin + (x * x * x) * (E0 - Emin) : 0.0;  // 107
}
void launch_simp(hipStream_t s, long long n, const uint8_t* emask, const double* xPhys, double Emin, double E0,
                 double* E) {
  hipLaunchKernelGGL(k_simp, dim3(grid_for(n)), dim3(kBlock), 0, s, n, emask, xPhys, Emin, E0, E);
}

// Masked sums over cells: mode 0: sum a; 1: sum a*b; 2: sum a*(1-a);
// 3: sum a^16 / b^16 (p-norm, 335/360).  emask == nullptr: every cell.
__global__ __launch_bounds__(kBlock) void k_masked_sum(long long n, const uint8_t* __restrict__ emask,
                                                       const double* __restrict__ a, const double* __restrict__ b,
                                                       int mode, RedWs ws, double* out) {
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    if (emask && !emask[i]) continue;
    const double ai = a[i];
    switch (mode) {
      case 0: s += ai; break;
      case 1: s += ai * b[i]; break;
      case 2: s += ai * (1.0 - ai); break;
      case 3: {
        const double a2 = ai * ai, a4 = a2 * a2, a8 = a4 * a4;
        const double bi = b[i], b2 = bi * bi, b4 = b2 * b2, b8 = b4 * b4;
        s += (a8 * a8) / (b8 * b8);
      } break;
      default: break;
    }
  }
  double v[1] = {s};
  write_partials<1>(v, ws.partials);
  (void)out;
}
void launch_masked_sum(hipStream_t s, long long n, const uint8_t* emask, const double* a, const double* b, int mode,
                       const RedWs& ws, double* out) {
  // red_blocks, not red1_blocks: the allocation-free OC entry point runs this
  // sum with its partials in a fixed scratch sized for kMaxRedBlocks blocks
  hipLaunchKernelGGL(k_masked_sum, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, a, b, mode, ws, out);
  fin1(s, FIN_SUM, red_blocks(n), ws, nullptr, nullptr, out);
}

// ---- OC bisection (145-153) by brackets: a pass evaluates gt at 15 multipliers
// (candidates) in one sweep over the cells; the finaliser keeps the largest with
// gt > 0 and the smallest with gt <= 0 and replays the sequential bisection as
// far as these decide it.  gt(l) never rises with l: every term max(lo, min(hi,
// t / sqrt(l))) - x is monotone in l, rounded operations are, and so is a sum in
// a fixed order.  So a midpoint at or below a candidate with gt > 0 has gt > 0
// itself, bit for bit, and likewise above one with gt <= 0; the decisions, the
// final multiplier and the bisection count are the sequential loop's.  Candidates
// close in on the root: powers of 16, then quarter octaves, then clusters
// around the bracket's secant (the 2^4 - 1 midpoints the loop would visit next,
// once the bracket is as fine as they are).  Bound: a pass's FP64 issue (115
// instructions a cell) and its 16 bytes a cell about alike, so passes count: 5
// instead of the 13 that 4 levels of midpoints at a time need (33.5M cells, the
// whole update 2.74 -> 1.16 ms; 50x100x50 0.55 -> 0.2 ms).
// emask == nullptr: every cell is a design cell (compact cell arrays).
// oc[]: 0 l1, 1 l2, 2 fval, 3 done, 4 lastLmid, 5 nBisect, 6 change; the
// candidates and the bracket lie behind the pass's partials (OcSearch).
constexpr int kOcDepth = 4;
constexpr int kOcCand = (1 << kOcDepth) - 1;
constexpr int kOcMaxLevels = 256;  // bisection levels at most (no root above 1e9 2^-256)
struct OcSearch {
  double l[kOcCand + 1], rl[kOcCand + 1];  // candidates and 1 / sqrt of them
  double A, gA, B, gB;                     // bracket: gt(A) = gA > 0 (A = 0: none yet), gt(B) = gB <= 0 (B = inf: none)
};
static_assert(kOcCand * kMaxRedBlocks + sizeof(OcSearch) / 8 <= 16 * kMaxRedBlocks,
              "the search state fits behind the partials of the widest pass");
__host__ __device__ inline OcSearch* oc_search(double* partials) {
  return (OcSearch*)(partials + kOcCand * kMaxRedBlocks);
}

// x .* sqrt(-dc ./ lmid) (149) as t * rl with t = x sqrt(-dc) formed once per
// cell and rl = 1/sqrt(lmid) once per candidate, then the move limits (150).
constexpr double kOcMove = 0.2;
__device__ __forceinline__ double oc_clamp(double x, double v) {
  v = fmin(x + kOcMove, v);
  v = fmin(1.0, v);
  v = fmax(x - kOcMove, v);
  return fmax(0.0, v);
}

// fval = mean(xPhys) - V0 (145), l1 = 0, l2 = 1e9 (146), the first candidates
__global__ __launch_bounds__(64) void k_oc_begin(const double* __restrict__ vsum, double n, double V0, double* oc,
                                                 double* partials) {
  OcSearch* S = oc_search(partials);
  const int k = threadIdx.x;
  if (k == 0) {
    oc[0] = 0.0;
    oc[1] = 1e9;
    oc[2] = *vsum / n - V0;
    oc[3] = oc[4] = oc[5] = oc[6] = 0.0;
    S->A = 0.0;
    S->gA = 0.0;
    S->B = INFINITY;
    S->gB = 0.0;
  }
  if (k < kOcCand) {
    const double l = ldexp(1.0, 4 * k - 30);  // 9e-10 .. 6.7e7
    S->l[k] = l;
    S->rl[k] = 1.0 / sqrt(l);
  }
}
void launch_oc_begin(hipStream_t s, const double* vsum, double n, double V0, const RedWs& ws, double* oc) {
  hipLaunchKernelGGL(k_oc_begin, dim3(1), dim3(64), 0, s, vsum, n, V0, oc, ws.partials);
}

__global__ __launch_bounds__(kBlock) void k_oc_pass(long long n, const uint8_t* __restrict__ emask,
                                                    const uint8_t* __restrict__ passive,
                                                    const double* __restrict__ x, const double* __restrict__ dc,
                                                    RedWs ws, const double* oc) {
  if (oc[3] != 0.0) return;
  const OcSearch* S = oc_search(ws.partials);
  double s[kOcCand], rl[kOcCand];
#pragma unroll
  for (int k = 0; k < kOcCand; ++k) {
    s[k] = 0.0;
    rl[k] = S->rl[k];
  }
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    if (emask && !emask[i]) continue;
    const double xi = x[i];
    const double t = xi * sqrt(-dc[i]);
    const bool pas = passive && passive[i];
    // oc_clamp's four nested min/max as one two-sided clamp to per-cell
    // bounds: min and max are exact, so max(0, max(x - m, min(1, min(x + m,
    // v)))) = max(lo, min(hi, v)) bit for bit (a NaN v yields max(lo, hi)
    // either way); a passive cell's bounds are both 1 (xnew = 1)
    const double hi = pas ? 1.0 : fmin(1.0, xi + kOcMove), lo = pas ? 1.0 : fmax(0.0, xi - kOcMove);
#pragma unroll
    for (int k = 0; k < kOcCand; ++k) {
      const double xn = fmax(lo, fmin(hi, t * rl[k]));
      s[k] += 1.0 * (xn - xi);  // 151
    }
  }
  write_partials<kOcCand>(s, ws.partials);
}

// One wave per candidate folds its partials (as 1024 threads would: each its
// partials b, b + 1024, .., then 16 wave sums in order), then the first thread
// replays the bisection and the candidates' threads place the next ones.
__global__ __launch_bounds__(kFinBlock) void k_oc_fin(int nb, double* partials, double* oc) {
  if (oc[3] != 0.0) return;
  __shared__ double sg[kOcCand + 1], sl[kOcCand + 1], sq[8], so[8];  // gt, candidates, bracket, oc
  __shared__ double sA, sB, sL1, sL2, sEst, sE;
  __shared__ int sMode;  // 0 done; 1 powers of 16 below B; 2 quarter octaves; 3 secant cluster; 4 midpoints
  OcSearch* S = oc_search(partials);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  static_assert(kFinBlock == 1024 && kOcCand <= 15, "a wave per candidate, 16 groups of 64 partials");
  if (w == 15) {  // what the first thread reads one after the other, in one round trip
    if (lane < kOcCand) sl[lane] = S->l[lane];
    else if (lane >= 16 && lane < 20) sq[lane - 16] = (&S->A)[lane - 16];
    else if (lane >= 24 && lane < 32) so[lane - 24] = oc[lane - 24];
  }
  if (w < kOcCand) {
    const double fval = oc[2];
    const double* p = partials + (size_t)w * nb;
    static_assert(kMaxRedBlocks <= 2 * kFinBlock, "at most two partials per thread of the fold");
    double s = 0.0;
    for (int g0 = 0; g0 < 16; g0 += 8) {
      double a[8];
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const int b = 64 * (g0 + g) + lane;
        const double p0 = p[min(b, nb - 1)], p1 = p[min(b + 1024, nb - 1)];
        a[g] = b < nb ? p0 : 0.0;
        if (b + 1024 < nb) a[g] += p1;
      }
      for (int g = 0; g < 8; ++g) s += wave_sum(a[g]);
    }
    if (lane == 0) sg[w] = fval + s;  // gt (151)
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double A = sq[0], gA = sq[1], B = sq[2], gB = sq[3];
#pragma unroll
    for (int k = 0; k < kOcCand; ++k) {
      const double l = sl[k], g = sg[k];
      if (g > 0) {
        if (l > A) A = l, gA = g;
      } else if (l < B) {
        B = l, gB = g;
      }
    }
    double l1 = so[0], l2 = so[1], last = so[4];
    int nbis = (int)so[5];
    bool done = false;
    for (;;) {
      // 147; with l1 = 0 the quotient is 1
      if (nbis >= kOcMaxLevels || (l1 != 0.0 && !((l2 - l1) / (l1 + l2) > 1e-6))) { done = true; break; }
      const double lmid = 0.5 * (l2 + l1);  // 148
      if (lmid <= A) l1 = lmid;             // 152: gt > 0
      else if (lmid >= B) l2 = lmid;
      else break;
      last = lmid;
      ++nbis;
    }
    oc[0] = l1;
    oc[1] = l2;
    oc[4] = last;
    oc[5] = (double)nbis;
    if (done) oc[3] = 1.0;
    S->A = A;
    S->gA = gA;
    S->B = B;
    S->gB = gB;
    sA = A;
    sB = B;
    sL1 = l1;
    sL2 = l2;
    int mode = 4;
    if (done) {
      mode = 0;
    } else if (A == 0.0 && B < INFINITY) {
      mode = 1;
    } else if (A > 0.0 && B < INFINITY) {
      const double h = (B - A) / A;
      if (h > 0.5) {
        mode = 2;
      } else if (h > 2e-6 && gA - gB > 0.0) {
        // root of the secant; its error is about h^2 / 16 of l
        mode = 3;
        sEst = A + (B - A) * (gA / (gA - gB));
        sE = fmax(h * h * 0.0625, 1e-8);
      }
    }
    sMode = mode;
  }
  __syncthreads();
  const int k = threadIdx.x;
  if (sMode == 0 || k >= kOcCand) return;
  const double A = sA, B = sB;
  double l;
  if (sMode == 1) {
    l = ldexp(B, 4 * (k - kOcCand));
  } else if (sMode == 2) {  // quarter octaves from A (the first passes step by 16)
    const double q = (k & 1) ? ((k & 2) ? 1.0 : 1.4142135623730951) : ((k & 2) ? 1.681792830507429 : 1.189207115002721);
    l = A * ldexp(q, (k + 1) >> 2);
  } else if (sMode == 3 && k >= 9) {  // even fractions of the bracket
    l = A + (B - A) * ((k - 8) * (1.0 / 7));
  } else if (sMode == 3) {  // est and est (1 +- e 4^j), j = -2 .. 1
    const double d = k == 0 ? 0.0 : sE * ldexp(1.0, 2 * ((k - 1) >> 1) - 4);
    l = sEst * (1.0 + ((k & 1) ? d : -d));
  } else {  // the next midpoints: heap order, node 1 the root, children 2n (l2 = mid), 2n + 1 (l1 = mid)
    double a = sL1, b = sL2;
    const int node = k + 1;
    l = 0.5 * (b + a);
    for (int lev = 30 - __clz(node); lev >= 0; --lev) {
      if ((node >> lev) & 1) a = l;
      else b = l;
      l = 0.5 * (b + a);
    }
  }
  S->l[k] = l;
  S->rl[k] = 1.0 / sqrt(l);
}
void launch_oc_pass(hipStream_t s, long long n, const uint8_t* emask, const uint8_t* passive, const double* x,
                    const double* dc, const RedWs& ws, double* oc) {
  hipLaunchKernelGGL(k_oc_pass, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, passive, x, dc, ws, oc);
  hipLaunchKernelGGL(k_oc_fin, dim3(1), dim3(kFinBlock), 0, s, red_blocks(n), ws.partials, oc);
}

// xnew at the last evaluated lmid (149-150), change = max|xnew-x| (154), x = xnew.
__global__ __launch_bounds__(kBlock) void k_oc_final(long long n, const uint8_t* __restrict__ emask,
                                                     const uint8_t* __restrict__ passive, double* __restrict__ x,
                                                     const double* __restrict__ dc, RedWs ws, double* oc) {
  const double rl = 1.0 / sqrt(oc[4]);
  double m = 0.0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    if (emask && !emask[i]) continue;
    const double xi = x[i];
    const double xn = (passive && passive[i]) ? 1.0 : oc_clamp(xi, xi * sqrt(-dc[i]) * rl);
    m = fmax(m, fabs(xn - xi));
    x[i] = xn;
  }
  write_partial_max(m, ws.partials);
}
void launch_oc_final(hipStream_t s, long long n, const uint8_t* emask, const uint8_t* passive, double* x,
                     const double* dc, const RedWs& ws, double* oc) {
  hipLaunchKernelGGL(k_oc_final, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, passive, x, dc, ws, oc);
  hipLaunchKernelGGL(k_fin_max, dim3(1), dim3(kBlock), 0, s, red_blocks(n), ws.partials, oc + 6);
}

__global__ __launch_bounds__(kBlock) void k_masked_maxdiff(long long n, const uint8_t* __restrict__ emask,
                                                           const double* __restrict__ a,
                                                           const double* __restrict__ b, RedWs ws, double* out) {
  double m = 0.0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
    if (emask[i]) m = fmax(m, fabs(a[i] - b[i]));
  write_partial_max(m, ws.partials);
  (void)out;
}
void launch_masked_maxdiff(hipStream_t s, long long n, const uint8_t* emask, const double* a, const double* b,
                           const RedWs& ws, double* out) {
  hipLaunchKernelGGL(k_masked_maxdiff, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, a, b, ws, out);
  hipLaunchKernelGGL(k_fin_max, dim3(1), dim3(kBlock), 0, s, red_blocks(n), ws.partials, out);
}

// Elementwise cell operations (masked; non-domain cells are left 0).
__global__ void k_elementwise(int op, long long n, const uint8_t* __restrict__ emask, double* __restrict__ a,
                              const double* __restrict__ b, const double* __restrict__ c, double p0, double p1,
                              double p2) {
  const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  if (!emask[i]) { a[i] = 0.0; return; }
  switch (op) {
    case OP_DC: {  // a = -(p0 * x^2) * (ce / p1)   (108, 129)
      const double x = b[i];
      a[i] = -(p0 * (x * x)) * (c[i] / p1);
    } break;
    case OP_MUL: a[i] = b[i] * c[i]; break;
    case OP_DIVMAX: a[i] = a[i] / fmax(1e-3, b[i]); break;  // 137
    case OP_HEAVI: {  // 380: p0 = beta, p1 = eta
      const double beta = p0, eta = p1;
      a[i] = (tanh(beta * eta) + tanh(beta * (b[i] - eta))) / (tanh(beta * eta) + tanh(beta * (1 - eta)));
    } break;
    case OP_DHEAVI: {  // 340
      const double beta = p0, eta = p1;
      const double th = tanh(beta * (b[i] - eta));
      a[i] = beta * (1 - th * th) / (tanh(beta * eta) + tanh(beta * (1 - eta)));
    } break;
    case OP_PNORMGRAD: {  // 335: p0 = fac, p1 = numElements
      const double xh = b[i], x2 = xh * xh, x4 = x2 * x2, x8 = x4 * x4;
      const double v = c[i], v2 = v * v, v4 = v2 * v2, v8 = v4 * v4;
      a[i] = p0 * ((x8 * x4 * x2 * xh) / (v8 * v8)) / p1;
    } break;
    case OP_COPY: a[i] = b[i]; break;
    case OP_SET: a[i] = p0; break;
    case OP_DIVC: a[i] = b[i] / p0; break;
    case OP_MULC: a[i] = b[i] * p0; break;
    case OP_AXPYC: a[i] = __dadd_rn(a[i], __dmul_rn(b[i], p0)); break;  // a + b*p0, rounded twice (597)
    case OP_MMA_BOUNDS: {  // a = xmin = max(0, x - move), c-> xmax written by the caller's second call
      a[i] = p1 > 0.0 ? fmin(1.0, b[i] + p0) : fmax(0.0, b[i] - p0);  // 364-365
    } break;
    default: break;
  }
}
void launch_elementwise(hipStream_t s, int op, long long n, const uint8_t* emask, double* a, const double* b,
                        const double* c, double p0, double p1, double p2) {
  hipLaunchKernelGGL(k_elementwise, dim3(grid_for(n)), dim3(kBlock), 0, s, op, n, emask, a, b, c, p0, p1, p2);
}

// =========================================================================
// MMA for m = 1 (MMAseq, 1804-2049), every dual step on the device.
// Scalar block mm[]: see MmaSlot.  Arrays are dense cell arrays (emask).
// =========================================================================

// GenSub (1873-1928) + the xold shift of Update (1867-1868) + SolveDIP init.
__global__ __launch_bounds__(kBlock) void k_mma_gensub(long long n, const uint8_t* __restrict__ emask, int iter,
                                                       const double* __restrict__ x, const double* __restrict__ xmin,
                                                       const double* __restrict__ xmax, double* __restrict__ xold1,
                                                       double* __restrict__ xold2, double* __restrict__ low,
                                                       double* __restrict__ upp, const double* __restrict__ dfdx,
                                                       const double* __restrict__ dgdx, double* __restrict__ alpha,
                                                       double* __restrict__ beta, double* __restrict__ p0,
                                                       double* __restrict__ q0, double* __restrict__ pij,
                                                       double* __restrict__ qij, RedWs ws, double* mm, double nAct) {
  const double asyinit = 0.5, asydec = 0.7, asyinc = 1.2, feps = 1.0e-6;
  double bs = 0.0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    if (!emask[i]) continue;
    const double xv = x[i], mn = xmin[i], mx = xmax[i];
    const double o1 = xold1[i], o2 = xold2[i];
    double lo, up;
    if (iter < 3) {  // 1880-1882
      lo = xv - asyinit * (mx - mn);
      up = xv + asyinit * (mx - mn);
    } else {  // 1884-1900
      const double zzz = (xv - o1) * (o1 - o2);
      double gamma = 1.0;
      if (zzz > 0) gamma = asyinc;
      if (zzz < 0) gamma = asydec;
      lo = xv - gamma * (o1 - low[i]);
      up = xv + gamma * (upp[i] - o1);
      const double lowmin = xv - 10.0 * (mx - mn), lowmax = xv - 0.01 * (mx - mn);
      const double uppmin = xv + 0.01 * (mx - mn), uppmax = xv + 10.0 * (mx - mn);
      lo = fmax(lo, lowmin);
      lo = fmin(lo, lowmax);
      up = fmin(up, uppmax);
      up = fmax(up, uppmin);
    }
    low[i] = lo;
    upp[i] = up;
    double al = 0.9 * lo + 0.1 * xv;  // 1905-1908
    if (al - mn < 0) al = mn;
    double be = 0.9 * up + 0.1 * xv;
    if (be - mx > 0) be = mx;
    alpha[i] = al;
    beta[i] = be;
    const double ux = up - xv, xl = xv - lo, ul = up - lo;
    const double df = dfdx[i], dg = dgdx[i];
    p0[i] = ux * ux * (fmax(0.0, df) + 0.001 * fabs(df) + 0.5 * feps / ul);  // 1912
    q0[i] = xl * xl * (fmax(0.0, -1.0 * df) + 0.001 * fabs(df) + 0.5 * feps / ul);
    const double extra = 0.001 * fabs(dg) + 0.5 * feps / ul;  // 1918
    const double pp = ux * ux * (fmax(0.0, dg) + extra), qq = xl * xl * (fmax(0.0, -1.0 * dg) + extra);
    pij[i] = pp;
    qij[i] = qq;
    bs += pp / (up - xv) + qq / (xv - lo);  // 1927
    xold2[i] = o1;  // 1867
    xold1[i] = xv;  // 1868
  }
  double v[1] = {bs};
  write_partials<1>(v, ws.partials);
  (void)mm;
  (void)nAct;
}

__global__ __launch_bounds__(kBlock) void k_mma_gensub_fin(int nb, const double* __restrict__ partials, double* mm,
                                                           double nAct) {
  double v[1];
  fold_partials<1>(partials, nb, v);
  if (threadIdx.x != 0) return;
  mm[MM_B] = -mm[MM_GX] + v[0];  // 1927
  mm[MM_C] = 1000.0;             // 1815
  mm[MM_A] = 0.0;
  mm[MM_LAM] = mm[MM_C] / 2.0;   // 1933
  mm[MM_MU] = 1.0;
  mm[MM_TOL] = 1.0e-9 * sqrt(1.0 + nAct);  // 1935
  mm[MM_EPSI] = 1.0;
  mm[MM_ERR] = INFINITY;
  mm[MM_LOOP] = 0.0;
  mm[MM_DONE] = 0.0;
  mm[MM_NEWTON] = 0.0;
}

__device__ __forceinline__ double mma_x(double lam, double p0, double q0, double pij, double qij, double lo,
                                        double up, double al, double be, double* xp_out) {
  const double pj = p0 + pij * lam, qj = q0 + qij * lam;
  const double xp = (sqrt(pj) * lo + sqrt(qj) * up) / (sqrt(pj) + sqrt(qj));  // 1974
  double xv = xp;
  if (xv - al < 0) xv = al;
  if (xv - be > 0) xv = be;
  if (xp_out) *xp_out = xp;
  return xv;
}

// Newton step part A: XYZofLAMBDA, DualGrad, DualHess, solve, DualLineSearch
// (1944-1955).
__global__ __launch_bounds__(kBlock) void k_mma_stepA(long long n, const uint8_t* __restrict__ emask,
                                                      double* __restrict__ x, const double* __restrict__ low,
                                                      const double* __restrict__ upp,
                                                      const double* __restrict__ alpha,
                                                      const double* __restrict__ beta, const double* __restrict__ p0,
                                                      const double* __restrict__ q0, const double* __restrict__ pij,
                                                      const double* __restrict__ qij, RedWs ws, double* mm) {
  if (mm[MM_DONE] != 0.0) return;
  double lam = mm[MM_LAM];
  if (lam < 0.0) lam = 0.0;
  double s[2] = {0.0, 0.0};
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    if (!emask[i]) continue;
    const double lo = low[i], up = upp[i], al = alpha[i], be = beta[i];
    const double a0 = p0[i], b0 = q0[i], pp = pij[i], qq = qij[i];
    double xp;
    const double xv = mma_x(lam, a0, b0, pp, qq, lo, up, al, be, &xp);
    x[i] = xv;
    const double ux = up - xv, xl = xv - lo;
    s[0] += pp / ux + qq / xl;  // 1985
    const double pj = a0 + pp * lam, qj = b0 + qq * lam;
    const double PQ = pp / (ux * ux) - qq / (xl * xl);  // 1993
    double df2 = -1.0 / (2.0 * pj / (ux * ux * ux) + 2.0 * qj / (xl * xl * xl));
    if (xp - al < 0) df2 = 0.0;
    if (xp - be > 0) df2 = 0.0;
    s[1] += PQ * df2 * PQ;  // 2000
  }
  write_partials<2>(s, ws.partials);
}

__global__ __launch_bounds__(kBlock) void k_mma_stepA_fin(int nb, const double* __restrict__ partials, double* mm) {
  if (mm[MM_DONE] != 0.0) return;
  double s[2];
  fold_partials<2>(partials, nb, s);
  if (threadIdx.x != 0) return;
  double lam = mm[MM_LAM];
  if (lam < 0.0) lam = 0.0;
  const double c = mm[MM_C], a = mm[MM_A], epsi = mm[MM_EPSI];
  double mu = mm[MM_MU];
  // XYZofLAMBDA scalars (1967-1970)
  double y = lam - c;
  if (y < 0.0) y = 0.0;
  const double z = fmax(0.0, 10.0 * (lam * a - 1.0));
  // DualGrad (1984-1985) and 1947
  double grad = -mm[MM_B] - a * z - y + s[0];
  grad = -1.0 * grad - epsi / lam;
  // DualHess (2000-2021)
  double H = s[1];
  const double lamai = lam * a;
  if (lam > c) H = H - 1.0;
  H = H - mu / lam;
  if (lamai > 1.0) H = H - 10.0 * a * a;
  double corr = 1e-4 * H / 1.0;
  if (-1.0 * corr < 1.0e-7) corr = -1.0e-7;
  H = H + corr;
  const double s1 = grad / H;                              // 1951
  const double s2 = -mu + epsi / lam - s1 * mu / lam;      // 1953
  double theta = 1.005;                                    // 2026-2031
  if (theta < -1.01 * s1 / lam) theta = -1.01 * s1 / lam;
  if (theta < -1.01 * s2 / mu) theta = -1.01 * s2 / mu;
  theta = 1.0 / theta;
  mm[MM_LAM] = lam + theta * s1;
  mm[MM_MU] = mu + theta * s2;
  mm[MM_Y] = y;
  mm[MM_Z] = z;
  mm[MM_GRAD] = grad;
  mm[MM_HESS] = H;
  mm[MM_S1] = s1;
  mm[MM_S2] = s2;
}

// Newton step part B: XYZofLAMBDA + DualResidual and the loop control
// (1941, 1957-1960).
__global__ __launch_bounds__(kBlock) void k_mma_stepB(long long n, const uint8_t* __restrict__ emask,
                                                      double* __restrict__ x, const double* __restrict__ low,
                                                      const double* __restrict__ upp,
                                                      const double* __restrict__ alpha,
                                                      const double* __restrict__ beta, const double* __restrict__ p0,
                                                      const double* __restrict__ q0, const double* __restrict__ pij,
                                                      const double* __restrict__ qij, RedWs ws, double* mm) {
  if (mm[MM_DONE] != 0.0) return;
  double lam = mm[MM_LAM];
  if (lam < 0.0) lam = 0.0;
  double s[2] = {0.0, 0.0};
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    if (!emask[i]) continue;
    const double lo = low[i], up = upp[i];
    const double xv = mma_x(lam, p0[i], q0[i], pij[i], qij[i], lo, up, alpha[i], beta[i], nullptr);
    x[i] = xv;
    s[0] += pij[i] / (up - xv);
    s[1] += qij[i] / (xv - lo);
  }
  write_partials<2>(s, ws.partials);
}

__global__ __launch_bounds__(kBlock) void k_mma_stepB_fin(int nb, const double* __restrict__ partials, double* mm) {
  if (mm[MM_DONE] != 0.0) return;
  double s[2];
  fold_partials<2>(partials, nb, s);
  if (threadIdx.x != 0) return;
  double lam = mm[MM_LAM];
  if (lam < 0.0) lam = 0.0;
  const double c = mm[MM_C], a = mm[MM_A], epsi = mm[MM_EPSI], mu = mm[MM_MU];
  double y = lam - c;
  if (y < 0.0) y = 0.0;
  const double z = fmax(0.0, 10.0 * (lam * a - 1.0));
  mm[MM_LAM] = lam;
  mm[MM_Y] = y;
  mm[MM_Z] = z;
  double r1 = -mm[MM_B] - a * z - y + mu;  // 2039-2041
  r1 = r1 + s[0] + s[1];
  const double r2 = mu * lam - epsi;
  const double err = fmax(fabs(r1), fabs(r2));
  mm[MM_ERR] = err;
  double loop = mm[MM_LOOP] + 1.0;
  mm[MM_NEWTON] = mm[MM_NEWTON] + 1.0;
  if (!(err > 0.9 * epsi && loop < 100)) {  // 1941
    const double e2 = epsi * 0.1;          // 1960
    mm[MM_EPSI] = e2;
    loop = 0.0;
    if (!(e2 > mm[MM_TOL])) mm[MM_DONE] = 1.0;  // 1938
  }
  mm[MM_LOOP] = loop;
}

void launch_mma_gensub(hipStream_t s, long long n, const uint8_t* emask, int iter, const double* x,
                       const double* xmin, const double* xmax, double* xold1, double* xold2, double* low,
                       double* upp, const double* dfdx, const double* dgdx, double* alpha, double* beta,
                       double* p0, double* q0, double* pij, double* qij, const RedWs& ws, double* mm, double nAct) {
  hipLaunchKernelGGL(k_mma_gensub, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, iter, x, xmin, xmax, xold1,
                     xold2, low, upp, dfdx, dgdx, alpha, beta, p0, q0, pij, qij, ws, mm, nAct);
  hipLaunchKernelGGL(k_mma_gensub_fin, dim3(1), dim3(kBlock), 0, s, red_blocks(n), ws.partials, mm, nAct);
}
void launch_mma_step(hipStream_t s, long long n, const uint8_t* emask, double* x, const double* low,
                     const double* upp, const double* alpha, const double* beta, const double* p0, const double* q0,
                     const double* pij, const double* qij, const RedWs& ws, double* mm) {
  hipLaunchKernelGGL(k_mma_stepA, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, x, low, upp, alpha, beta, p0,
                     q0, pij, qij, ws, mm);
  hipLaunchKernelGGL(k_mma_stepA_fin, dim3(1), dim3(kBlock), 0, s, red_blocks(n), ws.partials, mm);
  hipLaunchKernelGGL(k_mma_stepB, dim3(red_blocks(n)), dim3(kBlock), 0, s, n, emask, x, low, upp, alpha, beta, p0,
                     q0, pij, qij, ws, mm);
  hipLaunchKernelGGL(k_mma_stepB_fin, dim3(1), dim3(kBlock), 0, s, red_blocks(n), ws.partials, mm);
}

// =========================================================================
// Streaming copy of known size: the practical HBM-bandwidth reference and
// the calibration kernel for hardware byte counters (16-byte accesses).
// =========================================================================
// 16-byte non-temporal loads and stores over a 32768-block grid: the fastest
// of the copy forms measured at 813 MB per direction (5.5 TB/s moved, against
// 4.8-5.1 for plain double2 copies over 2048-32768 blocks).
__global__ __launch_bounds__(kBlock) void k_stream_copy(double2* __restrict__ dst, const double2* __restrict__ src,
                                                        long long n) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) {
    const v2d v = __builtin_nontemporal_load((const v2d*)(src + i));
    __builtin_nontemporal_store(v, (v2d*)(dst + i));
  }
}
void launch_stream_copy(hipStream_t s, double* dst, const double* src, long long nDoubles) {
  hipLaunchKernelGGL(k_stream_copy, dim3(32768), dim3(kBlock), 0, s, (double2*)dst, (const double2*)src,
                     nDoubles / 2);
}

// a[i] = v where mask[i] (x(passiveElements) = 1, 165 / 366 / 381)
__global__ void k_set_where(long long n, const uint8_t* __restrict__ mask, double* __restrict__ a, double v) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
    if (mask[i]) a[i] = v;
}
void launch_set_where(hipStream_t s, long long n, const uint8_t* mask, double* a, double v) {
  hipLaunchKernelGGL(k_set_where, dim3(stream_blocks(n)), dim3(kBlock), 0, s, n, mask, a, v);
}

}  // namespace t3x
