// nd_factor.hip -- multifrontal Cholesky factor of the shell matrices under a
// nested-dissection order.
//
// The mesh graph is cut by short separators (nd_order.h); every separator
// and every leaf is a front of ns pivot dofs and nb boundary dofs, m = ns +
// nb.  The fronts of one distance from the root form a level and are factored
// together, deepest level first, for several designs at once.  The factor of
// a front is the m x ns panel
//
//   M = [ X ; -W ],   X = L^{-1},  W = L21 L^{-1},   F11 = L L^T, L21 = F21 X^T,
//
// so a solve needs one product with M per front and sweep:
//   up:   y = X v_J,  u_B = v_B - W v_J          (v = b plus the children's u)
//   down: x_J = X^T y - W^T x_B = M^T [y ; x_B].
//
// Factoring a level takes the pivots in blocks of 64.  At block k the panel's
// columns left of k already hold forward-eliminated columns Y of the identity
// (rows below the pivots: of zero), the columns right of it what is left of
// F.  With X_k the inverse Cholesky factor of the diagonal block and
//   Q_k = [ (X_k Y_k)^T ; X_k^T ; F_ik X_k^T ]   (rows before, at, after k)
// one update C_ij -= Q_ik Q_jk^T serves both: for columns j < k it goes on
// eliminating Y, for j = k it starts the identity's column (C_ik = 0), for j
// > k it is the Cholesky update.  After the last block the panel is M, and
// the rows of Q at the boundary are L21: the Schur complement of the front is
// one product S = (children's S) - L21 L21^T.
//
// The short separators are what this form is for: a band (level) order of the
// 200 x 400 cylinder stores 27.7 GB and needs 10.6 Tflop, this order 1.45 GB
// and 0.165 Tflop (0.074 for the panels with their inverses, 0.091 for the
// Schur complements; a plain Cholesky factor 0.128), and the largest front has
// 2,400 pivots.  A factorisation is
// bound by the chain of about 100 pivot blocks of its levels (latency), a
// solve by the two reads of M and the chain of 2 x 14 levels.
//
// Every sum has a fixed order (no atomics): a factor and its solves are
// reproducible bit for bit.
#include "nd_factor.h"

#include <algorithm>

#include "nd_layout.h"

namespace shellgpu {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const double gcdouble;
typedef __attribute__((address_space(1))) double gdouble;
typedef __attribute__((address_space(1))) const v2d gcv2d;

constexpr int kB = 64;  // pivot block

struct LevelArgs {
  const NdDev *fronts;  // the level's first front
  const NdDev *all;     // front 0
  const int *lists;
  double *M;
  double *Q;
  double *S;        // the level's Schur complements
  const double *Sc; // the children's
  long sM, sQ, sS, sSc;  // per design
  int k;            // pivot block
  int tr, tc;       // tiles per front along rows and columns
};

// one 32 x 32 block of acc += A B^T: A rows ra (clamped by the caller), B rows
// rb, columns 0 .. n of both (column stride ld); D^T layout of
// v_mfma_f64_16x16x4f64 as measured on gfx950 (gemm_f64.hip): lane l, element
// e hold row l % 16, column 4 e + l / 16
struct Frag {
  v4d c[2][2];
};

// 16 columns at a time, the loads of the next 16 in flight during the matrix
// instructions of the current; columns past n count as zero
template <typename FA, typename FB>
__device__ __forceinline__ void mma32(Frag &f, int n, FA a_at, FB b_at) {
  const int lk = (threadIdx.x & 63) >> 4;
  double a[2][4][2], b[2][4][2];
  auto load = [&](int buf, int k0) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int kk = k0 + 4 * q + lk, kc = min(kk, n - 1);
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const double v = a_at(i, kc);
        a[buf][q][i] = kk < n ? v : 0.0;
        b[buf][q][i] = b_at(i, kc);
      }
    }
  };
  auto mul = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          f.c[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[buf][q][j], a[buf][q][i], f.c[i][j], 0, 0, 0);
  };
  load(0, 0);
  for (int k0 = 0; k0 < n; k0 += 32) {
    load(1, k0 + 16);
    mul(0);
    if (k0 + 16 >= n) break;
    load(0, k0 + 32);
    mul(1);
  }
}

__device__ __forceinline__ void clear(Frag &f) {
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) f.c[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
}

// matrix blocks -> panels (zeroed before): block p of the pattern goes to
// base[p] with leading dimension ld[p] (base -1: the transposed block is
// stored).  flag[p]: bits 6 + c mark BC columns, zeroed for the symmetric
// elimination (BC rows already are), bit 12 a diagonal block, of which the
// lower triangle is stored: nothing above the diagonal of a panel is written
// before its pivot block is, and solves count it as zero.
__global__ __launch_bounds__(256) void nd_scatter_kernel(int nnzb, const double *__restrict__ vals, long vstride,
                                                         const long *__restrict__ base, const int *__restrict__ ld,
                                                         const int *__restrict__ flag, double *__restrict__ M,
                                                         long stride) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 36L * nnzb) return;
  const int p = (int)(i / 36), e = (int)(i % 36), r = e / 6, c = e % 6;
  if (base[p] < 0) return;
  const int fl = flag[p];
  const bool diag = (fl >> 12) & 1;
  if (diag && c > r) return;
  double v = vals[blockIdx.y * vstride + i];
  if (((fl >> (6 + c)) & 1) && !(diag && r == c)) v = 0.0;
  M[blockIdx.y * stride + base[p] + (long)c * ld[p] + r] = v;
}

// panel columns of a front += its children's Schur complements
__global__ __launch_bounds__(256) void nd_gather_kernel(LevelArgs a) {
  const int f = blockIdx.x / (a.tr * a.tc), t = blockIdx.x - f * a.tr * a.tc;
  const NdDev d = a.fronts[f];
  const int i = kB * (t % a.tr) + (threadIdx.x & 63), c0 = kB * (t / a.tr);
  if (d.child[0] < 0 || c0 >= d.ns || i >= d.m || kB * (t % a.tr) + kB <= c0) return;
  const int mn = d.m / 6, ri = i / 6, rr = i - 6 * ri;
  const int *lists = a.lists + d.lists;
  gdouble *C = (gdouble *)(a.M + blockIdx.y * a.sM + d.M);
  int ir[2], ldc[2];
  gcdouble *Sc[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    ir[c] = -1;
    if (d.child[c] >= 0) {
      const NdDev ch = a.all[d.child[c]];
      ir[c] = lists[(1 + c) * mn + ri];
      ldc[c] = ch.m - ch.ns;
      Sc[c] = (gcdouble *)(a.Sc + blockIdx.y * a.sSc + ch.S);
    }
  }
  if (ir[0] < 0 && ir[1] < 0) return;
  for (int j = c0 + (threadIdx.x >> 6); j < min(c0 + kB, min(d.ns, i + 1)); j += 4) {
    const int cj = j / 6, cc = j - 6 * cj;
    double v = 0.0;
    bool any = false;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (ir[c] < 0) continue;
      const int ic = lists[(1 + c) * mn + cj];
      if (ic < 0) continue;
      v += Sc[c][6 * ir[c] + rr + (long)(6 * ic + cc) * ldc[c]];
      any = true;
    }
    if (any) C[i + (long)j * d.m] += v;
  }
}

// value of one lane, as a scalar
__device__ __forceinline__ double lane_value(double v, int lane) {
  const long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double((long)hi << 32 | lo);
}

// Diagonal block k: X_k = chol(C_kk)^{-1} into C_kk (zero above the
// diagonal) and its transpose into Q_kk, by one workgroup.
//
// The chain of these blocks is what bounds a factorisation near the root, so
// the code is built for latency: the block lies in LDS as four column blocks
// of 16; a wavefront takes a column block in registers, lane i holding row i,
// and factors it with the pivot row broadcast by v_readlane (no LDS round trip
// or barrier per pivot).  Between two panels all wavefronts update the
// remaining 16 x 16 tiles with matrix instructions.  X follows two panels
// behind, on the wavefronts the panel leaves idle: first the inverse of a
// diagonal block, then the columns of X, Y_ij -= L_ib X_bj with X_bj = X_bb
// Y_bj, whose tiles stay in registers (a result of the matrix instruction is
// laid out as the second operand of the next).  Blocks shorter than 64 are
// padded with the identity.  16 us a block near the root (25 us with the
// inverses on the panels' path, 112 us with one barrier and LDS round trip per
// pivot).
struct DiagLds {
  double L[kB][kB + 1];  // by columns; odd stride: constant offsets and no bank conflicts
  double Xd[4][16][17];  // inverses of the diagonal blocks, by rows
  double rs[kB];         // 1 / L_jj
};

// 1 / sqrt(p): the hardware's estimate and one third-order step (relative
// error of the estimate below 2^-24: 5/16 of its cube is below 2^-53)
__device__ __forceinline__ double inv_sqrt(double p) {
  const double y = __builtin_amdgcn_rsq(p);
  const double e = fma(-y * p, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// all 256 threads of a workgroup; returns true (in any lane of the panel's
// wavefront) for a pivot that is not positive
__device__ __forceinline__ bool diag_block(DiagLds &lds, gdouble *C, gdouble *Q, int n, int m) {
  const int nblk = (n + 15) / 16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  double r[16];
#pragma unroll
  for (int c = 0; c < 16; c++) {
    const int j = 16 * w + c;
    const double v = C[min(lane, n - 1) + (long)min(j, n - 1) * m];
    r[c] = lane < n && j < n ? v : (lane == j ? 1.0 : 0.0);
  }
  if (w > 0 && lane >= 16 * w) {
#pragma unroll
    for (int c = 0; c < 16; c++) lds.L[16 * w + c][lane] = r[c];
  }
  // column block w of X: tile (w + t, w) in R[t], eliminated with block row b
  v4d R[4];
  auto eliminate = [&](int b) {
    if (b == w) {
#pragma unroll
      for (int e = 0; e < 4; e++) R[0][e] = lds.Xd[w][4 * e + lk][lr];
    }
#pragma unroll
    for (int s = 0; s < 4; s++) {
      if (b - w != s) continue;
      if (s > 0) {
        v4d x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; q++) x = __builtin_amdgcn_mfma_f64_16x16x4f64(lds.Xd[b][lr][4 * q + lk], R[s][q], x, 0, 0, 0);
        R[s] = x;
      }
#pragma unroll
      for (int t = s + 1; t < 4; t++) {
        if (w + t >= nblk) continue;
        if (s == 0) R[t] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; q++)
          R[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-lds.L[16 * b + 4 * q + lk][16 * (w + t) + lr], R[s][q], R[t], 0,
                                                      0, 0);
      }
    }
  };
  // inverse of diagonal block b by four rank-4 steps: with Z the inverse of
  // the 4 x 4 block s, its rows become Z Y_s and the rows below take -L_is Z
  // Y_s; lane: row lr and column lk of P_s = [Z; -L_is Z]
  auto invert = [&](int b) {
    const double *rs = &lds.rs[16 * b];
    auto at = [&](int i, int j) { return lds.L[16 * b + j][16 * b + i]; };
    double P[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int o = 4 * s;
      const double z0 = lk == 0 ? rs[o] : 0.0;
      const double z1 = ((lk == 1 ? 1.0 : 0.0) - at(o + 1, o) * z0) * rs[o + 1];
      const double z2 = ((lk == 2 ? 1.0 : 0.0) - at(o + 2, o) * z0 - at(o + 2, o + 1) * z1) * rs[o + 2];
      const double z3 =
          ((lk == 3 ? 1.0 : 0.0) - at(o + 3, o) * z0 - at(o + 3, o + 1) * z1 - at(o + 3, o + 2) * z2) * rs[o + 3];
      const int i = lr - o;
      const double in = i == 0 ? z0 : i == 1 ? z1 : i == 2 ? z2 : z3;
      const double below = -(at(lr, o) * z0 + at(lr, o + 1) * z1 + at(lr, o + 2) * z2 + at(lr, o + 3) * z3);
      P[s] = i < 0 ? 0.0 : i < 4 ? in : below;
    }
    v4d Y;
#pragma unroll
    for (int e = 0; e < 4; e++) Y[e] = 4 * e + lk == lr ? 1.0 : 0.0;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const double ys = Y[s];
      Y[s] = 0.0;  // rows 4 s + lk: replaced, not added to (Z may be tiny beside the identity)
      Y = __builtin_amdgcn_mfma_f64_16x16x4f64(P[s], ys, Y, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) lds.Xd[b][4 * e + lk][lr] = Y[e];
  };
  bool bad = false;
  for (int b = 0; b < nblk; b++) {
    if (w == b) {
      if (b > 0) {
#pragma unroll
        for (int c = 0; c < 16; c++) r[c] = lds.L[16 * b + c][max(lane, 16 * b)];
      }
      double rs_lane = 0.0;
#pragma unroll
      for (int j = 0; j < 16; j++) {
        const double p = lane_value(r[j], 16 * b + j), rs = inv_sqrt(p);
        bad = bad || !(p > 0.0);
        r[j] *= rs;
        rs_lane = lane == j ? rs : rs_lane;
#pragma unroll
        for (int c = j + 1; c < 16; c++) r[c] -= r[j] * lane_value(r[j], 16 * b + c);
      }
      if (lane >= 16 * b) {
#pragma unroll
        for (int j = 0; j < 16; j++) lds.L[16 * b + j][lane] = r[j];
      }
      if (lane < 16) lds.rs[16 * b + lane] = rs_lane;
    } else if (w == b - 1) {
      invert(b - 1);
    } else if (w < b) {
      eliminate(b - 2);
    }
    __syncthreads();
    // tiles (i, j) right of block b, dealt to the wavefronts
    int q = w;
    for (int j = b + 1; j < nblk; j++)
      for (int i = j; i < nblk; i++, q--) {
        if (q < 0) q = 3;
        if (q != 0) continue;
        v4d t;
#pragma unroll
        for (int e = 0; e < 4; e++) t[e] = -lds.L[16 * j + 4 * e + lk][16 * i + lr];
#pragma unroll
        for (int e = 0; e < 4; e++)
          t = __builtin_amdgcn_mfma_f64_16x16x4f64(lds.L[16 * b + 4 * e + lk][16 * j + lr],
                                                   lds.L[16 * b + 4 * e + lk][16 * i + lr], t, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) lds.L[16 * j + 4 * e + lk][16 * i + lr] = -t[e];
      }
    if (b + 1 < nblk) __syncthreads();
  }
  if (w == nblk - 1)
    invert(w);
  else if (w < nblk - 1)
    eliminate(nblk - 2);
  __syncthreads();
  if (w < nblk) {
    eliminate(nblk - 1);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (i >= nblk) continue;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        // entry (16 i + 4 e + lk, 16 w + lr) of X; R is indexed from the
        // diagonal block: select without a register index
        double v = 0.0;
#pragma unroll
        for (int t = 0; t < 4; t++)
          if (i - w == t) v = R[t][e];
        const int row = 16 * i + 4 * e + lk, col = 16 * w + lr;
        if (row >= n || col >= n) continue;
        C[row + (long)col * m] = v;
        Q[col + (long)row * m] = v;
      }
    }
  }
  return bad;
}

// pivot block k of every front (the first; the later ones too unless
// nd_update_kernel has factored them)
__global__ __launch_bounds__(256, 2) void nd_diag_kernel(LevelArgs a, int *info) {
  __shared__ DiagLds lds;
  const NdDev d = a.fronts[blockIdx.x];
  const int k0 = kB * a.k;
  if (k0 >= d.ns) return;
  const long o = k0 + (long)k0 * d.m;
  gdouble *C = (gdouble *)(a.M + blockIdx.y * a.sM + d.M + o);
  gdouble *Q = (gdouble *)(a.Q + blockIdx.y * a.sQ + d.Q + o);
  if (diag_block(lds, C, Q, min(kB, d.ns - k0), d.m) && (threadIdx.x & 63) == 0) info[blockIdx.y] = 1;
}

// Q_ik = C_ik X_k^T for the rows after block k (tiles 0 .. tr), and the row
// block itself, C_kj = X_k C_kj and Q_jk = C_kj^T, for the columns before it
// (tiles tr .. tr + k)
__global__ __launch_bounds__(256) void nd_scale_kernel(LevelArgs a) {
  const int tiles = a.tr + a.k;
  const int f = blockIdx.x / tiles, t = blockIdx.x - f * tiles;
  const NdDev d = a.fronts[f];
  const int k0 = kB * a.k;
  if (k0 >= d.ns) return;
  const int n = min(kB, d.ns - k0), m = d.m;
  gdouble *C = (gdouble *)(a.M + blockIdx.y * a.sM + d.M);
  gdouble *Q = (gdouble *)(a.Q + blockIdx.y * a.sQ + d.Q);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wm = 32 * (wave & 1), wn = 32 * (wave >> 1);
  Frag acc;
  clear(acc);
  if (t < a.tr) {
    const int r0 = k0 + n + kB * t + wm;
    if (r0 >= m || wn >= n) return;
    long ra[2], rb[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      ra[i] = min(r0 + 16 * i + lr, m - 1) + (long)k0 * m;
      rb[i] = k0 + min(wn + 16 * i + lr, n - 1) + (long)k0 * m;
    }
    mma32(acc, n, [&](int i, int kk) { return C[ra[i] + (long)kk * m]; },
          [&](int i, int kk) { return C[rb[i] + (long)kk * m]; });
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int r = r0 + 16 * i + lr;
      if (r >= m) continue;
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int c = wn + 16 * j + 4 * e + lk;
          if (c < n) Q[r + (long)(k0 + c) * m] = acc.c[i][j][e];
        }
    }
    return;
  }
  // rows of block k (n of them), columns of block j < k (64 of them)
  const int c0 = kB * (t - a.tr);
  long ra[2], rb[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    ra[i] = k0 + min(wm + 16 * i + lr, n - 1) + (long)k0 * m;
    rb[i] = k0 + (long)(c0 + wn + 16 * i + lr) * m;
  }
  mma32(acc, n, [&](int i, int kk) { return C[ra[i] + (long)kk * m]; },
        [&](int i, int kk) { return C[rb[i] + kk]; });
  __syncthreads();  // the tile is read in full by both row halves
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = wm + 16 * i + lr;
    if (r >= n) continue;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int c = c0 + wn + 16 * j + 4 * e + lk;
        C[k0 + r + (long)c * m] = acc.c[i][j][e];
        Q[c + (long)(k0 + r) * m] = acc.c[i][j][e];
      }
  }
}

// C_ij -= Q_ik Q_jk^T for the rows after block k: columns before k, column
// block k (from zero), and the trailing lower triangle.  AHEAD: the workgroup
// of the next diagonal block goes on to factor it, so that chain runs beside
// the other tiles' updates (those tiles come first in the grid, for all
// fronts).
template <bool AHEAD>
__global__ __launch_bounds__(256, AHEAD ? 2 : 4) void nd_update_kernel(LevelArgs a, int nf, int *info) {
  const int f = blockIdx.x % nf, t = blockIdx.x / nf;
  const NdDev d = a.fronts[f];
  const int k0 = kB * a.k, ns = d.ns, m = d.m;
  if (k0 >= ns) return;
  const int n = min(kB, ns - k0), rs = k0 + n;
  int tj = a.k + 1 + t / a.tr;  // column tiles from the next block on, then those before it
  if (tj >= a.tc) tj -= a.tc;
  const int r0 = rs + kB * (t % a.tr);
  const int c0 = tj <= a.k ? kB * tj : rs + kB * (tj - a.k - 1);
  if (r0 >= m || c0 >= ns || r0 + kB <= c0) return;
  const int cw = tj == a.k ? n : min(kB, ns - c0);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wm = 32 * (wave & 1), wn = 32 * (wave >> 1);
  gdouble *C = (gdouble *)(a.M + blockIdx.y * a.sM + d.M);
  gdouble *Qf = (gdouble *)(a.Q + blockIdx.y * a.sQ + d.Q);
  if (r0 + wm < m && wn < cw) {
    gcdouble *Q = Qf + (long)k0 * m;
    // the tile enters as the negated sum, so its loads overlap the operands'
    Frag acc;
    long ra[2], rb[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      ra[i] = min(r0 + wm + 16 * i + lr, m - 1);
      rb[i] = c0 + min(wn + 16 * i + lr, cw - 1);
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          acc.c[i][j][e] = tj == a.k ? 0.0 : -C[ra[i] + (long)(c0 + min(wn + 16 * j + 4 * e + lk, cw - 1)) * m];
    mma32(acc, n, [&](int i, int kk) { return Q[ra[i] + (long)kk * m]; },
          [&](int i, int kk) { return Q[rb[i] + (long)kk * m]; });
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int r = r0 + wm + 16 * i + lr;
      if (r >= m) continue;
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int c = wn + 16 * j + 4 * e + lk;
          if (c < cw) C[r + (long)(c0 + c) * m] = -acc.c[i][j][e];
        }
    }
  }
  if (AHEAD && tj == a.k + 1 && r0 == c0) {  // the next diagonal block (the whole workgroup)
    __shared__ DiagLds lds;
    __syncthreads();
    const long o = c0 + (long)c0 * m;
    if (diag_block(lds, C + o, Qf + o, min(kB, ns - c0), m) && lane == 0) info[blockIdx.y] = 1;
  }
}

// Schur complements: S = children's S - L21 L21^T, lower tiles
__global__ __launch_bounds__(256) void nd_schur_kernel(LevelArgs a) {
  const int nt = a.tr * (a.tr + 1) / 2;
  const int f = blockIdx.x / nt, t = blockIdx.x - f * nt;
  int ti = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
  while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
  while (ti * (ti + 1) / 2 > t) ti--;
  const int tj = t - ti * (ti + 1) / 2;
  const NdDev d = a.fronts[f];
  const int ns = d.ns, m = d.m, nb = m - ns;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int r0 = kB * ti + 32 * (wave & 1), c0 = kB * tj + 32 * (wave >> 1);
  if (r0 >= nb || c0 >= nb || r0 + 32 <= c0) return;
  gcdouble *Q = (gcdouble *)(a.Q + blockIdx.y * a.sQ + d.Q + ns);
  gdouble *S = (gdouble *)(a.S + blockIdx.y * a.sS + d.S);
  const int mn = m / 6;
  const int *lists = a.lists + d.lists;
  // the children's parts enter as the negated sum, so their loads overlap the
  // operands'
  Frag acc;
  clear(acc);
  long ra[2], rb[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    ra[i] = min(r0 + 16 * i + lr, nb - 1);
    rb[i] = min(c0 + 16 * i + lr, nb - 1);
  }
#pragma unroll
  for (int c = 0; c < 2; c++) {
    if (d.child[c] < 0) continue;
    const NdDev ch = a.all[d.child[c]];
    const int ldc = ch.m - ch.ns, *place = lists + (1 + c) * mn + ns / 6;
    gcdouble *Sc = (gcdouble *)(a.Sc + blockIdx.y * a.sSc + ch.S);
    int ir[2], rr[2], ic[2][4], cc[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      rr[i] = (int)ra[i] % 6;
      ir[i] = place[(int)ra[i] / 6];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int col = min(c0 + 16 * i + 4 * e + lk, nb - 1);
        cc[i][e] = col % 6;
        ic[i][e] = place[col / 6];
      }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int pr = 6 * ir[i] + rr[i], pc = 6 * ic[j][e] + cc[j][e];
          // entries above the diagonal of the child's block are not stored
          if (ir[i] >= 0 && ic[j][e] >= 0 && pr >= pc) acc.c[i][j][e] -= Sc[pr + (long)pc * ldc];
        }
  }
  mma32(acc, ns, [&](int i, int kk) { return Q[ra[i] + (long)kk * m]; },
        [&](int i, int kk) { return Q[rb[i] + (long)kk * m]; });
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = r0 + 16 * i + lr;
    if (r >= nb) continue;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int col = c0 + 16 * j + 4 * e + lk;
        if (col <= r) S[r + (long)col * nb] = -acc.c[i][j][e];
      }
  }
}

struct SolveArgs {
  const NdDev *fronts, *all;
  const int *lists;
  const double *M;
  double *V;
  const double *b;
  double *x;
  long sM, sV, n;
  const int *act;  // designs, or null: all
  int tiles;       // per front
};

// entry i of a front's vector from its children's u (and, for the pivots, b)
struct FrontSource {
  const int *lists;
  const double *u[2];
  int mn;
  __device__ __forceinline__ FrontSource(const SolveArgs &a, const NdDev &d, const double *V, int nv)
      : lists(a.lists + d.lists), u{nullptr, nullptr}, mn(d.m / 6) {
#pragma unroll
    for (int c = 0; c < 2; c++)
      if (d.child[c] >= 0) {
        const NdDev ch = a.all[d.child[c]];
        u[c] = V + (ch.V + ch.ns) * nv;
      }
  }
  __device__ __forceinline__ double children(int i, int nv, int v) const {
    const int q = i / 6, w = i - 6 * q;
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < 2; c++)
      if (u[c]) {
        const int p = lists[(1 + c) * mn + q];
        if (p >= 0) s += u[c][(6L * p + w) * nv + v];
      }
    return s;
  }
  __device__ __forceinline__ double pivot(const double *b, int i, int nv, int v) const {
    const int q = i / 6;
    return b[(6L * lists[q] + i - 6 * q) * nv + v] + children(i, nv, v);
  }
};

constexpr int kStage = 1024;  // vector entries staged at once
constexpr int kBatch = 8;     // columns of M per wavefront in flight

// upward sweep: y = X v_J and u_B = v_B - W v_J, 128 rows per workgroup (two
// per lane), the columns split over the NW wavefronts.  A level's launch is a
// chain of memory latencies, so the loads of M (which need nothing of the
// vector) and the children's part of the rows are issued before the vector is
// staged, and each batch of columns before the products of the last: solves of
// the 200 x 400 cylinder, several streams at once, 0.67 -> 0.61 ms each, of 16
// designs of 100 x 200 2.39 -> 2.04 ms.  With the downward sweep as it is now
// 0.59 (4.9 TB/s over both sweeps) and 1.96; solves of one stream, whose levels
// wait for each other, take 0.81 and 2.16.
template <int NW>
__global__ __launch_bounds__(64 * NW) void nd_up_kernel(SolveArgs a) {
  __shared__ double vj[kStage];
  __shared__ v2d red[NW][64];
  const int f = blockIdx.x / a.tiles, r0 = 128 * (blockIdx.x - f * a.tiles);
  const NdDev d = a.fronts[f];
  if (r0 >= d.m) return;
  const int e = a.act ? a.act[blockIdx.y] : blockIdx.y;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  double *V = a.V + e * a.sV;
  const double *b = a.b + e * a.n;
  const int cend = min(d.ns, r0 + 128), r = r0 + 2 * lane;
  gcdouble *M = (gcdouble *)(a.M + e * a.sM + d.M + min(r, d.m - 2));
  v2d mv[2][kBatch];
  auto load = [&](int buf, int j0) {
#pragma unroll
    for (int q = 0; q < kBatch; q++) mv[buf][q] = *(gcv2d *)(M + (long)min(j0 + wave + NW * q, cend - 1) * d.m);
  };
  load(0, 0);
  const FrontSource src(a, d, V, 1);
  v2d acc = {0.0, 0.0};
  if (wave == 0 && r >= d.ns && r < d.m) acc = v2d{src.children(r, 1, 0), src.children(r + 1, 1, 0)};
  auto mul = [&](int buf, int j0) {
#pragma unroll
    for (int q = 0; q < kBatch; q++) acc += mv[buf][q] * vj[(j0 & (kStage - 1)) + wave + NW * q];
  };
  static_assert(kStage % (2 * kBatch * NW) == 0, "batches do not cross a staged piece");
  for (int j0 = 0; j0 < cend; j0 += 2 * kBatch * NW) {
    if ((j0 & (kStage - 1)) == 0) {
      if (j0) __syncthreads();
      // zero past the last column, to the end of the last batch
      const int sn = min(kStage, (cend - j0 + 2 * kBatch * NW - 1) / (2 * kBatch * NW) * (2 * kBatch * NW));
      for (int i = t; i < sn; i += 64 * NW) vj[i] = j0 + i < cend ? src.pivot(b, j0 + i, 1, 0) : 0.0;
      __syncthreads();
    }
    load(1, j0 + kBatch * NW);
    mul(0, j0);
    load(0, j0 + 2 * kBatch * NW);
    mul(1, j0 + kBatch * NW);
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int w = 1; w < NW; w++) acc += red[w][lane];
  if (r >= d.m) return;
  V[d.V + r] = acc.x;
  V[d.V + r + 1] = acc.y;
}

// downward sweep: x_J = M^T [y ; x_B], CW columns per wavefront, lanes along
// the rows (two per lane), the loads of M ahead of the vector as above.  Four
// columns at every size: eight take 156 registers instead of 88, three
// wavefronts per SIMD instead of five, and no size gains by them (a solve of
// 200 x 400 831 us with eight where a level has 32,768 columns, 805 with four;
// of 64 designs of 61 x 119 3,196 and 2,921; of 256 of 20 x 40 1,168 and 1,075;
// of 1,000 of 4 x 8 149 and 126).
__global__ __launch_bounds__(256) void nd_down_kernel(SolveArgs a) {
  constexpr int CW = 4;
  constexpr int kRows = 2 * kStage;
  __shared__ __align__(16) double z[kRows];
  const int f = blockIdx.x / a.tiles, c0 = 4 * CW * (blockIdx.x - f * a.tiles);
  const NdDev d = a.fronts[f];
  if (c0 >= d.ns) return;
  const int e = a.act ? a.act[blockIdx.y] : blockIdx.y;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int *lists = a.lists + d.lists;
  const double *V = a.V + e * a.sV + d.V;
  double *x = a.x + e * a.n;
  const int cw = c0 + CW * wave;
  // rows before the first column are zero (c0 is even)
  gcdouble *M = (gcdouble *)(a.M + e * a.sM + d.M + c0);
  const int rows = d.m - c0;
  v2d mv[2][CW], acc[CW];
#pragma unroll
  for (int c = 0; c < CW; c++) acc[c] = v2d{0.0, 0.0};
  auto load = [&](int buf, int i) {
#pragma unroll
    for (int c = 0; c < CW; c++)
      mv[buf][c] = *(gcv2d *)(M + min(i + 2 * lane, rows - 2) + (long)min(cw + c, d.ns - 1) * d.m);
  };
  auto mul = [&](int buf, int i) {
    const v2d zz = *reinterpret_cast<const v2d *>(&z[(i & (kRows - 1)) + 2 * lane]);
#pragma unroll
    for (int c = 0; c < CW; c++) acc[c] += mv[buf][c] * zz;
  };
  load(0, 0);
  for (int i0 = 0; i0 < rows; i0 += 256) {
    if ((i0 & (kRows - 1)) == 0) {
      if (i0) __syncthreads();
      // zero past the last row, to the end of the last batch
      const int sn = min(kRows, (rows - i0 + 255) & ~255);
      for (int i = t; i < sn; i += 256) {
        const int r = c0 + i0 + i, q = r / 6;
        z[i] = r >= d.m ? 0.0 : r < d.ns ? V[r] : x[6L * lists[q] + r - 6 * q];
      }
      __syncthreads();
    }
    load(1, i0 + 128);
    mul(0, i0);
    load(0, i0 + 256);
    mul(1, i0 + 128);
  }
#pragma unroll
  for (int c = 0; c < CW; c++) {
    double s = acc[c].x + acc[c].y;
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w, 64);
    const int col = cw + c;
    if (lane == c && col < d.ns) {
      const int q = col / 6;
      x[6L * lists[q] + col - 6 * q] = s;
    }
  }
}

// ---- several vectors per design ------------------------------------------
//
// Load cases share one factor, so their vectors go through it together: the
// panels are read once for up to 16 of them, as matrix products with 16
// columns (v_mfma_f64_16x16x4f64).  The vectors are interleaved, entry i of
// vector v at 16 i + v, so every gather along a node list moves whole 128-byte
// lines.  16 vectors of a 32,000-quad box beam: 0.82 ms a solve (2.3 ms with
// the single-vector kernels run once per vector).
constexpr int kNv = 16;

// n-vectors b (vector v of design d at (v nd + d) n) <-> interleaved w (n x 16
// per design; the vectors past nrhs are zero)
__global__ __launch_bounds__(256) void nd_interleave_kernel(long n, int nd, int nrhs, const double *__restrict__ b,
                                                            double *__restrict__ w) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int d = blockIdx.y;
  v2d *o = reinterpret_cast<v2d *>(w + ((long)d * n + i) * kNv);
#pragma unroll
  for (int v = 0; v < kNv; v += 2) {
    v2d t;
    t.x = v < nrhs ? b[((long)v * nd + d) * n + i] : 0.0;
    t.y = v + 1 < nrhs ? b[((long)(v + 1) * nd + d) * n + i] : 0.0;
    o[v / 2] = t;
  }
}
__global__ __launch_bounds__(256) void nd_deinterleave_kernel(long n, int nd, int nrhs, const double *__restrict__ w,
                                                              double *__restrict__ x) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int d = blockIdx.y;
  const v2d *o = reinterpret_cast<const v2d *>(w + ((long)d * n + i) * kNv);
#pragma unroll
  for (int v = 0; v < kNv; v += 2) {
    const v2d t = o[v / 2];
    if (v < nrhs) x[((long)v * nd + d) * n + i] = t.x;
    if (v + 1 < nrhs) x[((long)(v + 1) * nd + d) * n + i] = t.y;
  }
}

constexpr int kStageM = 256;  // rows of 16 values staged at once

// upward sweep, 32 RG rows per workgroup: a wavefront takes 32 rows (two per
// lane, one 16-row matrix block of the even and one of the odd rows) and every
// CS-th group of four columns
template <int RG, int CS>
__global__ __launch_bounds__(64 * RG * CS) void nd_up_multi_kernel(SolveArgs a) {
  constexpr int NW = RG * CS, kU = 4, kStep = 4 * CS * kU;  // columns of a batch
  constexpr int kLds = CS > 1 && NW * 512 > kStageM * 17 ? NW * 512 : kStageM * 17;
  __shared__ double lds[kLds];
  const int f = blockIdx.x / a.tiles, r0 = 32 * RG * (blockIdx.x - f * a.tiles);
  const NdDev d = a.fronts[f];
  if (r0 >= d.m) return;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, lr = lane & 15, lk = lane >> 4;
  const int rg = wave % RG, cs = wave / RG;
  double *V = a.V + blockIdx.y * a.sV;
  const double *b = a.x + blockIdx.y * a.n * kNv;
  const int cend = min(d.ns, r0 + 32 * RG);
  const int row = r0 + 32 * rg + 2 * lr;
  gcdouble *M = (gcdouble *)(a.M + blockIdx.y * a.sM + d.M + min(row, d.m - 2));
  v2d mv[2][kU];
  auto load = [&](int buf, int c0) {
#pragma unroll
    for (int q = 0; q < kU; q++) mv[buf][q] = *(gcv2d *)(M + (long)min(c0 + 4 * (cs + CS * q) + lk, cend - 1) * d.m);
  };
  load(0, 0);
  const FrontSource src(a, d, V, kNv);
  v4d acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
  if (cs == 0) {
#pragma unroll
    for (int h = 0; h < 2; h++)
      if (row + h >= d.ns && row + h < d.m) {
#pragma unroll
        for (int e = 0; e < 4; e++) acc[h][e] = src.children(row + h, kNv, 4 * e + lk);
      }
  }
  auto mul = [&](int buf, int c0) {
#pragma unroll
    for (int q = 0; q < kU; q++) {
      const double bv = lds[17 * ((c0 & (kStageM - 1)) + 4 * (cs + CS * q) + lk) + lr];
      acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv, mv[buf][q].x, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv, mv[buf][q].y, acc[1], 0, 0, 0);
    }
  };
  static_assert(kStageM % kStep == 0, "batches do not cross a staged piece");
  for (int s0 = 0; s0 < cend; s0 += kStageM) {
    if (s0) __syncthreads();
    // zero past the last column, to the end of the last batch
    const int sn = min(kStageM, (cend - s0 + kStep - 1) / kStep * kStep);
    for (int e = t; e < kNv * sn; e += 64 * NW) {
      const int i = e / kNv, v = e % kNv;
      lds[17 * i + v] = s0 + i < cend ? src.pivot(b, s0 + i, kNv, v) : 0.0;
    }
    __syncthreads();
    int c = s0;
    for (; c + kStep < s0 + sn; c += 2 * kStep) {
      load(1, c + kStep);
      mul(0, c);
      load(0, c + 2 * kStep);
      mul(1, c + kStep);
    }
    if (c < s0 + sn) {  // one batch left: the piece is the last, or one batch
      load(1, c + kStep);
      mul(0, c);
#pragma unroll
      for (int q = 0; q < kU; q++) mv[0][q] = mv[1][q];
    }
  }
  if (CS > 1) {  // the column parts of a row group, added in order
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int e = 0; e < 4; e++) lds[512 * wave + 64 * (4 * h + e) + lane] = acc[h][e];
    __syncthreads();
    if (cs) return;
#pragma unroll 1
    for (int c = 1; c < CS; c++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[h][e] += lds[512 * (RG * c + rg) + 64 * (4 * h + e) + lane];
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int r = row + h;
    if (r >= d.m) continue;
#pragma unroll
    for (int e = 0; e < 4; e++) V[(d.V + r) * kNv + 4 * e + lk] = acc[h][e];
  }
}

// downward sweep, 16 CW columns per workgroup: a wavefront takes 16 columns
// and every RS-th group of 16 rows (four consecutive rows per lane, the sum
// over rows in any order)
template <int CW, int RS>
__global__ __launch_bounds__(64 * CW * RS) void nd_down_multi_kernel(SolveArgs a) {
  constexpr int NW = CW * RS, kU = kStageM / (16 * RS) < 2 ? 1 : 2, kStep = 16 * RS * kU;  // rows of a batch
  constexpr int kLds = RS > 1 && NW * 256 > kStageM * 17 ? NW * 256 : kStageM * 17;
  __shared__ double lds[kLds];
  const int f = blockIdx.x / a.tiles, t0 = 16 * CW * (blockIdx.x - f * a.tiles);
  const NdDev d = a.fronts[f];
  if (t0 >= d.ns) return;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, lr = lane & 15, lk = lane >> 4;
  const int cw = wave % CW, rs = wave / CW;
  const int *lists = a.lists + d.lists;
  const double *V = a.V + blockIdx.y * a.sV + d.V * kNv;
  double *x = a.x + blockIdx.y * a.n * kNv;
  const int col = t0 + 16 * cw + lr;
  // rows before the first column are zero (t0 is even)
  gcdouble *M = (gcdouble *)(a.M + blockIdx.y * a.sM + d.M + t0 + (long)min(col, d.ns - 1) * d.m);
  const int rows = d.m - t0;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  v2d mv[2][kU][2];
  auto load = [&](int buf, int i0) {
#pragma unroll
    for (int q = 0; q < kU; q++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        mv[buf][q][h] = *(gcv2d *)(M + min(i0 + 16 * (rs + RS * q) + 4 * lk + 2 * h, rows - 2));
  };
  auto mul = [&](int buf, int i0) {
#pragma unroll
    for (int q = 0; q < kU; q++)
#pragma unroll
      for (int h = 0; h < 4; h++)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(lds[17 * ((i0 & (kStageM - 1)) + 16 * (rs + RS * q) + 4 * lk + h) + lr],
                                                   mv[buf][q][h >> 1][h & 1], acc, 0, 0, 0);
  };
  static_assert(kStageM % kStep == 0, "batches do not cross a staged piece");
  load(0, 0);
  for (int s0 = 0; s0 < rows; s0 += kStageM) {
    if (s0) __syncthreads();
    // zero past the last row, to the end of the last batch
    const int sn = min(kStageM, (rows - s0 + kStep - 1) / kStep * kStep);
    for (int e = t; e < kNv * sn; e += 64 * NW) {
      const int i = e / kNv, v = e % kNv, r = t0 + s0 + i, q = r / 6;
      lds[17 * i + v] = r >= d.m ? 0.0 : r < d.ns ? V[(long)r * kNv + v] : x[(6L * lists[q] + r - 6 * q) * kNv + v];
    }
    __syncthreads();
    int i = s0;
    for (; i + kStep < s0 + sn; i += 2 * kStep) {
      load(1, i + kStep);
      mul(0, i);
      load(0, i + 2 * kStep);
      mul(1, i + kStep);
    }
    if (i < s0 + sn) {  // one batch left
      load(1, i + kStep);
      mul(0, i);
#pragma unroll
      for (int q = 0; q < kU; q++)
#pragma unroll
        for (int h = 0; h < 2; h++) mv[0][q][h] = mv[1][q][h];
    }
  }
  if (RS > 1) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; e++) lds[256 * wave + 64 * e + lane] = acc[e];
    __syncthreads();
    if (rs) return;
#pragma unroll
    for (int c = 1; c < RS; c++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[e] += lds[256 * (CW * c + cw) + 64 * e + lane];
  }
  if (col >= d.ns) return;
  const int q = col / 6;
#pragma unroll
  for (int e = 0; e < 4; e++) x[(6L * lists[q] + col - 6 * q) * kNv + 4 * e + lk] = acc[e];
}

template <typename T>
hipError_t upload(T **dst, const std::vector<T> &src) {
  hipError_t e = hipMalloc((void **)dst, sizeof(T) * std::max<size_t>(1, src.size()));
  if (e == hipSuccess && !src.empty()) e = hipMemcpy(*dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice);
  return e;
}

// workspace for F.chunk designs at once, for fewer where the memory left does
// not hold it
hipError_t alloc_work(NdFactor &F) {
  for (;; F.chunk = (F.chunk + 1) / 2) {
    hipError_t e = hipMalloc((void **)&F.Q, sizeof(double) * (size_t)F.q_len * F.chunk);
    for (int k = 0; k < 2 && e == hipSuccess; k++)
      e = hipMalloc((void **)&F.S[k], sizeof(double) * (size_t)F.s_len[k] * F.chunk);
    if (e != hipErrorOutOfMemory || F.chunk == 1) return e;
    (void)hipGetLastError();  // handled here
    for (double **p : {&F.Q, &F.S[0], &F.S[1]}) {
      if (*p) (void)hipFree(*p);
      *p = nullptr;
    }
  }
}

}  // namespace

std::string nd_create(int nn, const NdLayout &L, int nbatch, int nrhs, NdFactor &F) {
  F.nbatch = nbatch;
  F.levels = L.levels;
  F.per_design = L.per_design;
  F.v_len = L.v_len;
  F.q_len = L.q_len;
  F.s_len[0] = L.s_len[0];
  F.s_len[1] = L.s_len[1];
  // workspace copies: at most as many designs at once as 4 GiB hold (15 of the
  // 100 x 200 cylinder), which leaves no level short of workgroups
  const double ws = 8.0 * (F.q_len + F.s_len[0] + F.s_len[1]);
  F.chunk = std::max(1, (int)std::min<double>(nbatch, 4294967296.0 / ws));
  F.n = 6L * nn;
  hipError_t e = upload(&F.d_fronts, L.fronts);
  if (e == hipSuccess) e = upload(&F.d_lists, L.lists);
  if (e == hipSuccess) e = hipMalloc((void **)&F.M, sizeof(double) * (size_t)F.per_design * nbatch);
  if (e == hipSuccess) e = nd_reserve(F, nrhs);
  if (e == hipSuccess) e = alloc_work(F);
  if (e != hipSuccess)
    return std::string("factor allocation (") + std::to_string((long)(8.0 * F.per_design * nbatch) >> 20) +
           " MiB): " + hipGetErrorString(e);
  return "";
}

void nd_destroy(NdFactor &F) {
  void *bufs[] = {F.d_fronts, F.d_lists, F.M, F.Q, F.S[0], F.S[1], F.V, F.W};
  for (void *p : bufs)
    if (p) (void)hipFree(p);
  F = NdFactor();
}

hipError_t nd_reserve(NdFactor &F, int nrhs) {
  // several vectors take the buffers of 16
  const int cap = nrhs > 1 ? kNv : 1;
  if (cap <= F.rhs_cap) return hipSuccess;
  if (nrhs > kNv) return hipErrorInvalidValue;
  F.rhs_cap = 0;
  for (double **p : {&F.V, &F.W}) {
    if (*p) (void)hipFree(*p);
    *p = nullptr;
  }
  hipError_t e = hipMalloc((void **)&F.V, sizeof(double) * (size_t)F.v_len * F.nbatch * cap);
  if (e == hipSuccess && cap > 1) e = hipMalloc((void **)&F.W, sizeof(double) * (size_t)F.n * F.nbatch * cap);
  if (e == hipSuccess) F.rhs_cap = cap;
  return e;
}

hipError_t nd_compute(NdFactor &F, int nnzb, const double *vals, const long *blk_base, const int *blk_ld,
                      const int *blk_flag, int *info, hipStream_t stream) {
  hipError_t e = hipMemsetAsync(F.M, 0, sizeof(double) * (size_t)F.per_design * F.nbatch, stream);
  if (e == hipSuccess) e = hipMemsetAsync(info, 0, sizeof(int) * F.nbatch, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(nd_scatter_kernel, dim3((unsigned)((36L * nnzb + 255) / 256), F.nbatch), dim3(256), 0, stream,
                     nnzb, vals, 36L * nnzb, blk_base, blk_ld, blk_flag, F.M, F.per_design);
  for (int d0 = 0; d0 < F.nbatch; d0 += F.chunk) {
    const unsigned nd = (unsigned)std::min(F.chunk, F.nbatch - d0);
    for (size_t l = 0; l < F.levels.size(); l++) {
      const NdLevel &lv = F.levels[l];
      LevelArgs a;
      a.all = F.d_fronts;
      a.fronts = F.d_fronts + lv.f0;
      a.lists = F.d_lists;
      a.M = F.M + (size_t)d0 * F.per_design;
      a.Q = F.Q;
      a.S = F.S[l & 1];
      a.Sc = F.S[(l & 1) ^ 1];
      a.sM = F.per_design;
      a.sQ = F.q_len;
      a.sS = F.s_len[l & 1];
      a.sSc = F.s_len[(l & 1) ^ 1];
      const int tm = (lv.max_m + kB - 1) / kB, tn = (lv.max_ns + kB - 1) / kB;
      if (lv.inner) {
        a.tr = tm;
        a.tc = tn;
        hipLaunchKernelGGL(nd_gather_kernel, dim3((unsigned)lv.nf * tm * tn, nd), dim3(256), 0, stream, a);
      }
      // few fronts: the chain of pivot blocks bounds the level, and the update
      // factors the next one; many: the updates' throughput does, and the
      // registers of the pivot code would halve their occupancy (panels of a
      // level of the 200 x 400 cylinder: 1 front 2,760 -> 1,870 us, 64 350 ->
      // 314, 256 276 -> 268, 512 332 -> 344, 2,048 1,120 -> 1,445)
      const bool ahead = (long)lv.nf * nd <= 256;
      for (a.k = 0; a.k < tn; a.k++) {
        if (a.k == 0 || !ahead)
          hipLaunchKernelGGL(nd_diag_kernel, dim3(lv.nf, nd), dim3(256), 0, stream, a, info + d0);
        // rows after block k of the tallest front (a front whose block k is
        // its last, of n < 64 pivots, has its boundary left)
        a.tr = std::max((lv.max_m - kB * (a.k + 1) + kB - 1) / kB, (lv.max_nb + kB - 1) / kB);
        a.tc = tn;
        if (a.tr + a.k > 0)
          hipLaunchKernelGGL(nd_scale_kernel, dim3((unsigned)lv.nf * (a.tr + a.k), nd), dim3(256), 0, stream, a);
        if (a.tr > 0)
          hipLaunchKernelGGL(ahead ? nd_update_kernel<true> : nd_update_kernel<false>,
                             dim3((unsigned)lv.nf * a.tr * a.tc, nd), dim3(256), 0, stream, a, lv.nf, info + d0);
      }
      if (lv.max_nb > 0) {
        a.tr = (lv.max_nb + kB - 1) / kB;
        hipLaunchKernelGGL(nd_schur_kernel, dim3((unsigned)lv.nf * (a.tr * (a.tr + 1) / 2), nd), dim3(256), 0, stream,
                           a);
      }
    }
  }
  return hipGetLastError();
}

hipError_t nd_solve(const NdFactor &F, const double *b, double *x, long n, int nrhs, const int *act, int nact,
                    hipStream_t stream) {
  SolveArgs a;
  a.all = F.d_fronts;
  a.lists = F.d_lists;
  a.M = F.M;
  a.V = F.V;
  a.b = b;
  a.x = x;
  a.sM = F.per_design;
  a.sV = F.v_len;
  a.n = n;
  a.act = act;
  if (nrhs > 1 && !act) {
    a.x = F.W;
    a.sV = F.v_len * kNv;
    const dim3 ig((unsigned)((n + 255) / 256), F.nbatch);
    hipLaunchKernelGGL(nd_interleave_kernel, ig, dim3(256), 0, stream, n, F.nbatch, nrhs, b, F.W);
    for (const NdLevel &lv : F.levels) {
      a.fronts = F.d_fronts + lv.f0;
      const long rows = (long)lv.nf * F.nbatch * ((lv.max_m + 31) / 32);
      // 32-row pieces of the level: enough of them fill the GPU with whole
      // columns, fewer split the columns over the wavefronts of a workgroup
      // (16 vectors, us.  First line at 1,024 / 8,192 / none: 61 x 119 309 / 319 /
      // 319, 200 x 400 1,923 / 1,998 / 2,148, 32,000-quad box beam 771 / 817 / 831.
      // Second at 0 / 1,024 / 4,096: 329 / 319 / 355, 2,061 / 1,999 / 2,162, 841 /
      // 816 / 907).  The lines here and below also set the order of the sums: the
      // lower ones that would be faster move box-beam KS gradients, which lose
      // digits to cancellation, by 2e-9.
      if (rows >= 8192) {
        a.tiles = (lv.max_m + 127) / 128;
        hipLaunchKernelGGL((nd_up_multi_kernel<4, 1>), dim3((unsigned)(lv.nf * a.tiles), F.nbatch), dim3(256), 0,
                           stream, a);
      } else if (rows >= 1024) {
        a.tiles = (lv.max_m + 63) / 64;
        hipLaunchKernelGGL((nd_up_multi_kernel<2, 4>), dim3((unsigned)(lv.nf * a.tiles), F.nbatch), dim3(512), 0,
                           stream, a);
      } else {
        a.tiles = (lv.max_m + 31) / 32;
        hipLaunchKernelGGL((nd_up_multi_kernel<1, 16>), dim3((unsigned)(lv.nf * a.tiles), F.nbatch), dim3(1024), 0,
                           stream, a);
      }
    }
    for (size_t l = F.levels.size(); l-- > 0;) {
      const NdLevel &lv = F.levels[l];
      a.fronts = F.d_fronts + lv.f0;
      const long cols = (long)lv.nf * F.nbatch * ((lv.max_ns + 15) / 16);
      // 16-column pieces: many split the rows over fewer wavefronts (16 vectors,
      // us.  First line at 512 / 4,096 / none: 61 x 119 322 / 319 / 319, 200 x 400
      // 2,014 / 2,001 / 1,845, box beam 841 / 816 / 762: whole rows per wavefront
      // are not the faster form, but see above.  Second at 0 / 512 / 4,096: 363 /
      // 319 / 320, 2,095 / 2,001 / 1,974, 872 / 817 / 809)
      if (cols >= 4096) {
        a.tiles = (lv.max_ns + 127) / 128;
        hipLaunchKernelGGL((nd_down_multi_kernel<8, 1>), dim3((unsigned)(lv.nf * a.tiles), F.nbatch), dim3(512), 0,
                           stream, a);
      } else if (cols >= 512) {
        a.tiles = (lv.max_ns + 31) / 32;
        hipLaunchKernelGGL((nd_down_multi_kernel<2, 4>), dim3((unsigned)(lv.nf * a.tiles), F.nbatch), dim3(512), 0,
                           stream, a);
      } else {
        a.tiles = (lv.max_ns + 15) / 16;
        hipLaunchKernelGGL((nd_down_multi_kernel<1, 16>), dim3((unsigned)(lv.nf * a.tiles), F.nbatch), dim3(1024), 0,
                           stream, a);
      }
    }
    hipLaunchKernelGGL(nd_deinterleave_kernel, ig, dim3(256), 0, stream, n, F.nbatch, nrhs, F.W, x);
    return hipGetLastError();
  }
  const unsigned ne = (unsigned)(act ? nact : F.nbatch);
  for (const NdLevel &lv : F.levels) {
    a.fronts = F.d_fronts + lv.f0;
    a.tiles = (lv.max_m + 127) / 128;
    const long groups = (long)lv.nf * a.tiles * ne;
    // few row tiles (the fronts near the root): more wavefronts share a
    // tile's columns, so that enough loads are in flight (line at 0 / 256 /
    // 1,024 / none, us: 61 x 119 147 / 144 / 148 / 148, 100 x 200 284 / 277 / 285 /
    // 294, 200 x 400 802 / 783 / 792 / 867, 16 designs of 20 x 40 108 / 108 / 114 /
    // 114, of 61 x 119 788 / 786 / 791 / 875)
    if (groups < 1024)
      hipLaunchKernelGGL(nd_up_kernel<16>, dim3((unsigned)(lv.nf * a.tiles), ne), dim3(1024), 0, stream, a);
    else
      hipLaunchKernelGGL(nd_up_kernel<4>, dim3((unsigned)(lv.nf * a.tiles), ne), dim3(256), 0, stream, a);
  }
  for (size_t l = F.levels.size(); l-- > 0;) {
    const NdLevel &lv = F.levels[l];
    a.fronts = F.d_fronts + lv.f0;
    a.tiles = (lv.max_ns + 15) / 16;
    hipLaunchKernelGGL(nd_down_kernel, dim3((unsigned)(lv.nf * a.tiles), ne), dim3(256), 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace shellgpu
