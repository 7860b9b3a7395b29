// xpt_kernels.hip -- coordinate, thickness and path derivatives of the
// element scalars of the buckling sensitivities:
//
//   s_K = phi^T K_e phi,   s_G = phi^T G_e(u) phi,   s_R = psi^T R_e(u)
//
// The reference differentiates these products with respect to Xpts by
// central differences (TACSElement::addMatXptSensInnerProduct and
// addAdjResXptProduct, src/elements/TACSElement.cpp:270-332, 434-507,
// dh = 1e-7).  Here they are exact, by the adjoint of the strain evaluation:
// one backward sweep gives all 12 coordinates of an element.  The scalars are
// written through strains only,
//
//   e(q) = e1(q) + Q(q, q) / 2           (Q symmetric bilinear)
//   s_K = sum_qp det e1(phi)^T C e1(phi)
//   s_G = sum_qp det [2 Q(u, phi)^T C e1(phi) + (e1(u) - e_th)^T C Q(phi, phi)]
//   s_R = sum_qp det e1(psi)^T C (e1(u) - e_th)                  (linear model)
//       = sum_qp det (e1(psi) + Q(u, psi))^T C (e(u) - e_th)     (nonlinear)
//   s_M = phi^T M_e phi = sum_qp det (m0 |u0(phi)|^2 + m2 |d0(phi)|^2)
//
// The last is the consistent mass of the linearized-rotation shell
// (TACSShellElement.h:613-648 with the moments of
// TACSIsoShellConstitutive::evalMassMoments, m0 = rho t, m2 = rho t^3/12):
// its rotational block -[t_i]x S_ij [t_j]x contracts with phi to
// S_ij (q_i x t_i).(q_j x t_j), and the interpolated director is
// d0 = sum N_m (q_m x t_m).
//
// with the strain evaluation of the element kernels: node normals and
// drilling strains (TACSShellUtilities.h:301-343, 649-707), MITC tying
// strains (TACSShellElementModel.h:32-77, 643-697) interpolated and
// transformed at the quadrature points, bending strains from the
// displacement gradients (TACSShellUtilities.h:361-422) and the natural
// transform with its un-orthogonalised in-plane axis.
//
// Four lanes share an element: lane p takes node p, quadrature point p and
// the tying points p, p + 4, p + 8, and they exchange normals, tying strains
// and their adjoints through LDS.  The element gradients go to a buffer and a
// second kernel adds them up per node, in element order, so all elements run
// in one launch whatever the colouring (a colour of a 20,000-element mesh has
// too few wavefronts to fill the GPU).
//
// Bound by the registers: the strains of two vectors and two pairs with their
// adjoints hold all 512 of a lane, one wavefront per SIMD.  Against one lane
// per (element, coordinate) in forward-mode dual numbers, which evaluated
// every strain 12 times: s_G + s_K of 19,691 elements 6 x 246 us -> 45 us,
// s_R 34, s_K 25, and 4.5 us for the sums per node; a lane per element would
// need four times the registers and leave three quarters of the GPU idle.
// The thickness derivatives need the forward half only (two wavefronts per
// SIMD): against half a wavefront per element with the 24 columns of B in LDS,
// s_G of 19,691 elements 6 x 58 us -> 15 us, s_R 6 x 24 -> 13, s_K 6 x 26 -> 12.
#include "elem_common.h"
#include "shellgpu_internal.h"

namespace shellgpu {
namespace {

constexpr int kElems = 32;  // per workgroup of 128 threads
enum { kCoord, kThick, kThickPath };

struct V3 {
  double x, y, z;
};
__device__ __forceinline__ V3 operator+(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 operator-(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ V3 operator*(double s, V3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ V3 &operator+=(V3 &a, V3 b) { return a = a + b; }
__device__ __forceinline__ double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ V3 load3(const double *p) { return {p[0], p[1], p[2]}; }
__device__ __forceinline__ V3 zero3() { return {0.0, 0.0, 0.0}; }
// a x_0 + b x_1 + c x_2 of a triple of vectors
__device__ __forceinline__ V3 comb(V3 x, V3 a, V3 b, V3 c) { return x.x * a + x.y * b + x.z * c; }

// natural transform (elem_common.h) of the surface direction a and the normal
// n0: T = [t1 t2 n], and its adjoint
struct Frame {
  V3 T[3];
  double iv, in, d;
  __device__ __forceinline__ void set(V3 a, V3 n0) {
    in = 1.0 / sqrt(dot(n0, n0));
    const V3 n = in * n0;
    d = dot(n, a);
    V3 v = a;
    v.x = a.x - d * n.x;
    v.x = v.x - d * n.x;
    v.x = v.x - d * n.x;
    iv = 1.0 / sqrt(dot(v, v));
    T[0] = iv * v;
    T[1] = cross(n, T[0]);
    T[2] = n;
  }
  __device__ __forceinline__ void adjoint(V3 a, const V3 Tb[3], V3 &ab, V3 &n0b) const {
    const V3 n = T[2], t1 = T[0];
    V3 nb = Tb[2] + cross(t1, Tb[1]);
    const V3 t1b = Tb[0] + cross(Tb[1], n);
    const V3 vb = iv * (t1b - dot(t1, t1b) * t1);
    const double db = -3.0 * n.x * vb.x;
    nb.x -= 3.0 * d * vb.x;
    nb += db * a;
    ab += vb + db * n;
    n0b += in * (nb - dot(n, nb) * n);
  }
};

// inverse of [a b c]: rows r, determinant; and the adjoint: Gi[i] is the
// adjoint of row i
struct Inverse {
  V3 r[3];
  double det;
  __device__ __forceinline__ void set(V3 a, V3 b, V3 c) {
    const V3 bc = cross(b, c);
    det = dot(a, bc);
    const double i = 1.0 / det;
    r[0] = i * bc;
    r[1] = i * cross(c, a);
    r[2] = i * cross(a, b);
  }
  __device__ __forceinline__ V3 mul(V3 v) const { return {dot(r[0], v), dot(r[1], v), dot(r[2], v)}; }
  __device__ __forceinline__ V3 mul_t(V3 v) const { return comb(v, r[0], r[1], r[2]); }
  __device__ __forceinline__ V3 column(int l, const V3 Gi[3], double detb) const {
    return (detb * det) * r[l] - comb({dot(Gi[0], r[l]), dot(Gi[1], r[l]), dot(Gi[2], r[l])}, r[0], r[1], r[2]);
  }
};

__device__ __forceinline__ void apply_c(const Section &c, const double b[9], double y[9]) {
  y[0] = c.A[0] * b[0] + c.A[1] * b[1] + c.A[2] * b[2];
  y[1] = c.A[1] * b[0] + c.A[3] * b[1] + c.A[4] * b[2];
  y[2] = c.A[2] * b[0] + c.A[4] * b[1] + c.A[5] * b[2];
  y[3] = c.D[0] * b[3] + c.D[1] * b[4] + c.D[2] * b[5];
  y[4] = c.D[1] * b[3] + c.D[3] * b[4] + c.D[4] * b[5];
  y[5] = c.D[2] * b[3] + c.D[4] * b[4] + c.D[5] * b[5];
  y[6] = c.As[0] * b[6] + c.As[1] * b[7];
  y[7] = c.As[1] * b[6] + c.As[2] * b[7];
  y[8] = c.drill * b[8];
}
__device__ __forceinline__ double dot9(const double a[9], const double b[9]) {
  double s = a[0] * b[0];
#pragma unroll
  for (int i = 1; i < 9; i++) s += a[i] * b[i];
  return s;
}

// vectors: 0 phi, 1 u, 2 psi; bilinear pairs (u,phi), (phi,phi), (u,psi), (u,u)
constexpr int kPairA[4] = {1, 0, 1, 1};
constexpr int kPairB[4] = {0, 0, 2, 1};
constexpr int bits(int m) { return (m & 1) + ((m >> 1) & 1) + ((m >> 2) & 1) + ((m >> 3) & 1); }

// LDS of one element.  The sources of tying strains are the vectors of WM,
// then the pairs of PM.
template <int WM, int PM, int W>
struct XptSmem {
  static constexpr int kNw = bits(WM), kNs = kNw + bits(PM);
  double q[kNw][24];
  double fn[12];
  union {
    struct {
      double et[kNw][4];   // drilling strains at the nodes
      double ty[kNs][9];   // tying strains
    } f;
    struct {
      double g[4][kNs][5];  // per quadrature point, adjoints of the tying fields
      double e8[4][kNw];    // and of the drilling strain
    } b;
    double part[4][W];      // per lane, adjoints of the normals, then of the result
  };
};

// WM: the vectors a variant evaluates (bit w), PM: the pairs (bit p).  Each
// scalar needs: s_K and s_M phi; s_G phi, u and the pairs (u,phi),
// (phi,phi); s_R u, psi and, for the nonlinear model, (u,psi), (u,u).
// Vectors and pairs outside the masks are never formed.
//
// OUT: kCoord, the gradient in the coordinates; kThick, the scalars with the
// section's thickness derivative, into a.dv; kThickPath, those and
// d s_G / du (s_G is affine in u: the adjoint of Q(u, phi) and e1(u) alone)
template <int WM, int PM, int OUT>
__global__ __launch_bounds__(4 * kElems) void xpt_kernel(XptArgs a, double *out) {
  using SM = XptSmem<WM, PM, OUT == kThickPath ? 24 : 12>;
  constexpr int NW = SM::kNw, NS = SM::kNs;
  constexpr bool kPhi = WM & 1, kU = (WM >> 1) & 1, kPsi = (WM >> 2) & 1;
  constexpr bool kGeo = kPhi && kU && (PM & 3) == 3;
  constexpr bool kRes = kU && kPsi;
  constexpr bool kResNl = kRes && (PM & 12) == 12;
  // places of the vectors and pairs among the sources
  constexpr int wi[3] = {0, bits(WM & 1), bits(WM & 3)};
  constexpr int pi[4] = {NW, NW + bits(PM & 1), NW + bits(PM & 3), NW + bits(PM & 7)};
  __shared__ SM smem[kElems];
  SM &sm = smem[threadIdx.x >> 2];
  const int p = threadIdx.x & 3;
  const long le = (long)blockIdx.x * kElems + (threadIdx.x >> 2);
  const bool active = le < a.nelems;
  const int e = active ? (int)le : a.nelems - 1;
  const long design = blockIdx.y;
  const int *cn = a.conn + 4 * e;
  const double c[4] = {a.coef[4 * design], a.coef[4 * design + 1], a.coef[4 * design + 2], a.coef[4 * design + 3]};
  {
    // a vector whose coefficients are zero does not enter
    const bool has[3] = {c[0] != 0.0 || c[1] != 0.0 || c[3] != 0.0, c[1] != 0.0 || c[2] != 0.0, c[2] != 0.0};
    const double *src[3] = {a.phi, a.u, a.psi};
    const long o = design * a.stride + 6 * cn[p];
#pragma unroll
    for (int w = 0; w < 3; w++)
      if ((WM >> w) & 1) {
#pragma unroll
        for (int i = 0; i < 6; i++) sm.q[wi[w]][6 * p + i] = src[w] && has[w] ? src[w][o + i] : 0.0;
      }
  }
  V3 X[4];
#pragma unroll
  for (int m = 0; m < 4; m++) X[m] = load3(a.Xpts + 3 * cn[m]);
  auto sum = [](const double N[4], const V3 v[4]) { return N[0] * v[0] + N[1] * v[1] + N[2] * v[2] + N[3] * v[3]; };
  double u_, v_, nN[4], nNa[4], nNb[4];
  // ---- node p: normal, frame, drilling strains (et = 0.5 (Ct[3] + u0x[3] -
  // Ct[1] - u0x[1]), TacsShellComputeDrillStrain) ----
  node_point(p, u_, v_);
  shape4(u_, v_, nN, nNa, nNb);
  const V3 an = sum(nNa, X), bn = sum(nNb, X);
  V3 fnp = cross(an, bn);
  const double fl = sqrt(dot(fnp, fnp)), fi = fl != 0.0 ? 1.0 / fl : 1.0;
  fnp = fi * fnp;
  sm.fn[3 * p] = fnp.x;
  sm.fn[3 * p + 1] = fnp.y;
  sm.fn[3 * p + 2] = fnp.z;
  __syncthreads();
  // gradient of a vector's displacements, and its nodal directors d = q x n
  auto grad_u = [&](int s, const double Na[4], const double Nb[4], V3 &ux, V3 &ue) {
    ux = zero3();
    ue = zero3();
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const V3 q = load3(&sm.q[s][6 * m]);
      ux += Na[m] * q;
      ue += Nb[m] * q;
    }
  };
  auto director = [&](int s, int m) { return cross(load3(&sm.q[s][6 * m + 3]), load3(&sm.fn[3 * m])); };
  Frame nf;
  Inverse ni;
  nf.set(an, fnp);
  ni.set(an, bn, fnp);
  const V3 nx1 = ni.mul(nf.T[0]), nx2 = ni.mul(nf.T[1]);
#pragma unroll
  for (int s = 0; s < NW; s++) {
    V3 ux, ue;
    grad_u(s, nNa, nNb, ux, ue);
    const V3 rot = load3(&sm.q[s][6 * p + 3]);
    sm.f.et[s][p] = -dot(rot, cross(nf.T[0], nf.T[1])) +
                    0.5 * (dot(nf.T[1], nx1.x * ux + nx1.y * ue) - dot(nf.T[0], nx2.x * ux + nx2.y * ue));
  }
  // ---- tying strains at points p, p + 4, p + 8 ----
#pragma unroll 1
  for (int t = p; t < 9; t += 4) {
    double u, v, N[4], Na[4], Nb[4];
    tying_point(t, u, v);
    shape4(u, v, N, Na, Nb);
    const V3 at = sum(Na, X), bt = sum(Nb, X);
    V3 n0 = zero3(), ux[NW], ue[NW], d0[NW];
#pragma unroll
    for (int m = 0; m < 4; m++) n0 += N[m] * load3(&sm.fn[3 * m]);
    const int f = tying_field(t);
#pragma unroll
    for (int s = 0; s < NW; s++) {
      grad_u(s, Na, Nb, ux[s], ue[s]);
      d0[s] = zero3();
#pragma unroll
      for (int m = 0; m < 4; m++) d0[s] += N[m] * director(s, m);
      sm.f.ty[s][t] = f == kG11   ? dot(ux[s], at)
                      : f == kG22 ? dot(ue[s], bt)
                      : f == kG12 ? 0.5 * (dot(ux[s], bt) + dot(ue[s], at))
                      : f == kG23 ? 0.5 * (dot(bt, d0[s]) + dot(n0, ue[s]))
                                  : 0.5 * (dot(at, d0[s]) + dot(n0, ux[s]));
    }
#pragma unroll
    for (int k = 0; k < 4; k++)
      if ((PM >> k) & 1) {
        const int A = wi[kPairA[k]], B = wi[kPairB[k]];
        sm.f.ty[pi[k]][t] = f == kG11   ? dot(ux[A], ux[B])
                            : f == kG22 ? dot(ue[A], ue[B])
                            : f == kG12 ? 0.5 * (dot(ux[A], ue[B]) + dot(ux[B], ue[A]))
                            : f == kG23 ? 0.5 * (dot(d0[A], ue[B]) + dot(d0[B], ue[A]))
                                        : 0.5 * (dot(d0[A], ux[B]) + dot(d0[B], ux[A]));
      }
  }
  __syncthreads();
  // ---- quadrature point p ----
  double N[4], Na[4], Nb[4], Nt[9];
  quad_point(p, u_, v_);
  shape4(u_, v_, N, Na, Nb);
  tying_interp(u_, v_, Nt);
  const V3 aq = sum(Na, X), bq = sum(Nb, X);
  V3 n0 = zero3(), na = zero3(), nb = zero3();
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const V3 f = load3(&sm.fn[3 * m]);
    n0 += N[m] * f;
    na += Na[m] * f;
    nb += Nb[m] * f;
  }
  Frame F;
  Inverse I;
  F.set(aq, n0);
  I.set(aq, bq, n0);
  V3 x[3], z[2], h[2];  // columns of X_d^{-1} T and of the normal-gradient part
#pragma unroll
  for (int k = 0; k < 3; k++) x[k] = I.mul(F.T[k]);
#pragma unroll
  for (int k = 0; k < 2; k++) {
    h[k] = x[k].x * na + x[k].y * nb;
    z[k] = -1.0 * I.mul(h[k]);
  }
  // tying fields of a source, interpolated here
  auto fields = [&](int s, double g[5]) {
    const double *t = sm.f.ty[s];
    g[kG11] = Nt[0] * t[0] + Nt[1] * t[1];
    g[kG22] = Nt[2] * t[2] + Nt[3] * t[3];
    g[kG12] = Nt[4] * t[4];
    g[kG23] = Nt[5] * t[5] + Nt[6] * t[6];
    g[kG13] = Nt[7] * t[7] + Nt[8] * t[8];
  };
  auto sym_mul = [](const double g[5], V3 v) -> V3 {
    return {g[kG11] * v.x + g[kG12] * v.y + g[kG13] * v.z, g[kG12] * v.x + g[kG22] * v.y + g[kG23] * v.z,
            g[kG13] * v.x + g[kG23] * v.y};
  };
  // displacement fields of the vectors at the point
  V3 ux[NW], ue[NW], d0[NW], dx[NW], de[NW], U0[NW][2], U1[NW][2];
#pragma unroll
  for (int s = 0; s < NW; s++) {
    grad_u(s, Na, Nb, ux[s], ue[s]);
    d0[s] = dx[s] = de[s] = zero3();
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const V3 d = director(s, m);
      d0[s] += N[m] * d;
      dx[s] += Na[m] * d;
      de[s] += Nb[m] * d;
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const V3 P = comb(x[k], ux[s], ue[s], d0[s]);
      const V3 S = x[k].x * dx[s] + x[k].y * de[s] + comb(z[k], ux[s], ue[s], d0[s]);
      U0[s][k] = {dot(F.T[0], P), dot(F.T[1], P), dot(F.T[2], P)};
      U1[s][k] = {dot(F.T[0], S), dot(F.T[1], S), dot(F.T[2], S)};
    }
  }
  auto tensor_strains = [&](int s, double e9[9]) {
    double g[5];
    fields(s, g);
    const V3 y0 = sym_mul(g, x[0]), y1 = sym_mul(g, x[1]);
    e9[0] = dot(x[0], y0);
    e9[1] = dot(x[1], y1);
    e9[2] = 2.0 * dot(x[0], y1);
    e9[6] = 2.0 * dot(x[2], y1);
    e9[7] = 2.0 * dot(x[2], y0);
  };
  auto linear_strain = [&](int s, double e9[9]) {
    tensor_strains(s, e9);
    e9[3] = U1[s][0].x;
    e9[4] = U1[s][1].y;
    e9[5] = U1[s][1].x + U1[s][0].y;
    e9[8] = N[0] * sm.f.et[s][0] + N[1] * sm.f.et[s][1] + N[2] * sm.f.et[s][2] + N[3] * sm.f.et[s][3];
  };
  auto pair_strain = [&](int k, double e9[9]) {
    const int A = wi[kPairA[k]], B = wi[kPairB[k]];
    tensor_strains(pi[k], e9);
    e9[3] = dot(U0[A][0], U1[B][0]) + dot(U0[B][0], U1[A][0]);
    e9[4] = dot(U0[A][1], U1[B][1]) + dot(U0[B][1], U1[A][1]);
    e9[5] = dot(U0[A][0], U1[B][1]) + dot(U1[A][0], U0[B][1]) + dot(U0[B][0], U1[A][1]) + dot(U1[B][0], U0[A][1]);
    e9[8] = 0.0;
  };
  // ---- the scalar's terms and the adjoints of its strains ----
  const double thick = a.thick[design * a.nelems + e];
  const Section sec = make_section(a.mat, thick);
  const Section vsec = OUT == kCoord ? sec : make_section_dt(a.mat, thick);  // of the value
  const double eth = a.temp ? a.mat.cte * a.temp[design * a.nelems + e] : 0.0;
  const double det = I.det;
  double value = 0.0;  // of the integrand: the adjoint of the determinant
  double sb[NS][9];    // adjoints of the sources' strains
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int i = 0; i < 9; i++) sb[s][i] = 0.0;
  double eu[9], Ceu[9];
  if constexpr (kU) {
    linear_strain(wi[1], eu);
    eu[0] -= eth;
    eu[1] -= eth;
  }
  if constexpr (kPhi) {
    double ep[9], Cep[9];
    linear_strain(wi[0], ep);
    apply_c(vsec, ep, Cep);
    value += c[0] * dot9(ep, Cep);
    if constexpr (OUT == kCoord) {
#pragma unroll
      for (int i = 0; i < 9; i++) sb[wi[0]][i] += 2.0 * c[0] * det * Cep[i];
    }
    if constexpr (kGeo) {
      double q0[9], q1[9], Cq[9];
      pair_strain(0, q0);
      pair_strain(1, q1);
      apply_c(vsec, eu, Ceu);
      value += c[1] * (2.0 * dot9(q0, Cep) + dot9(q1, Ceu));
      const double w = c[1] * det;
      if constexpr (OUT == kCoord) {
        apply_c(sec, q0, Cq);
#pragma unroll
        for (int i = 0; i < 9; i++) {
          sb[wi[0]][i] += 2.0 * w * Cq[i];
          sb[pi[1]][i] += w * Ceu[i];
        }
      }
      if constexpr (OUT == kThickPath) apply_c(sec, ep, Cep);
      if constexpr (OUT != kThick) {
        apply_c(sec, q1, Cq);
#pragma unroll
        for (int i = 0; i < 9; i++) {
          sb[pi[0]][i] += 2.0 * w * Cep[i];
          sb[wi[1]][i] += w * Cq[i];
        }
      }
    }
  }
  if constexpr (kRes) {
    double es[9], Ces[9];
    linear_strain(wi[2], es);
    double et[9];
#pragma unroll
    for (int i = 0; i < 9; i++) et[i] = eu[i];
    if constexpr (kResNl) {
      if (a.nonlin) {
        double q[9];
        pair_strain(2, q);
#pragma unroll
        for (int i = 0; i < 9; i++) es[i] += q[i];
        pair_strain(3, q);
#pragma unroll
        for (int i = 0; i < 9; i++) et[i] += 0.5 * q[i];
      }
    }
    apply_c(vsec, et, Ceu);
    value += c[2] * dot9(es, Ceu);
    const double w = c[2] * det;
    apply_c(sec, es, Ces);
#pragma unroll
    for (int i = 0; i < 9; i++) {
      sb[wi[1]][i] += w * Ces[i];
      sb[wi[2]][i] += w * Ceu[i];
    }
    if constexpr (kResNl) {
      if (a.nonlin) {
#pragma unroll
        for (int i = 0; i < 9; i++) {
          sb[pi[2]][i] += w * Ceu[i];
          sb[pi[3]][i] += 0.5 * w * Ces[i];
        }
      }
    }
  }
  if constexpr (OUT != kCoord) {
    double dv = value * det;
    dv += __shfl_xor(dv, 1);
    dv += __shfl_xor(dv, 2);
    if (active && p == 0 && a.dv) a.dv[design * a.nelems + e] += dv;
    if constexpr (OUT == kThick) return;
  }
  // adjoint of a source's tying fields here
  auto fields_adjoint = [&](const double b[9], double g[5]) {
    const V3 m0 = b[0] * x[0] + b[2] * x[1] + b[7] * x[2], m1 = b[2] * x[0] + b[1] * x[1] + b[6] * x[2],
             m2 = b[7] * x[0] + b[6] * x[1];
    g[kG11] = x[0].x * m0.x + x[1].x * m1.x + x[2].x * m2.x;
    g[kG22] = x[0].y * m0.y + x[1].y * m1.y + x[2].y * m2.y;
    g[kG12] = 2.0 * (x[0].x * m0.y + x[1].x * m1.y + x[2].x * m2.y);
    g[kG23] = 2.0 * (x[0].y * m0.z + x[1].y * m1.z + x[2].y * m2.z);
    g[kG13] = 2.0 * (x[0].x * m0.z + x[1].x * m1.z + x[2].x * m2.z);
  };
  // weight of the source s at tying point t: its field's adjoints of the four
  // quadrature points
  auto tying_weight = [&](int t, int s) {
    double w = 0.0;
#pragma unroll
    for (int iq = 0; iq < 4; iq++) {
      double u, v, Nq[9];
      quad_point(iq, u, v);
      tying_interp(u, v, Nq);
      double Nqt = Nq[0];
#pragma unroll
      for (int k = 1; k < 9; k++) Nqt = t == k ? Nq[k] : Nqt;
      w += Nqt * sm.b.g[iq][s][tying_field(t)];
    }
    return w;
  };
  // adjoint of the drilling strain of node p
  auto drill_weight = [&](int s) {
    double w = 0.0;
#pragma unroll
    for (int iq = 0; iq < 4; iq++) {
      double u, v, qN[4], qa[4], qb[4];
      quad_point(iq, u, v);
      shape4(u, v, qN, qa, qb);
      w += (p == 0 ? qN[0] : p == 1 ? qN[1] : p == 2 ? qN[2] : qN[3]) * sm.b.e8[iq][s];
    }
    return w;
  };
  if constexpr (OUT == kThickPath) {
    constexpr int A = wi[1], B = wi[0], P = pi[0];
    const double *b = sb[P], *l = sb[A];
    const V3 U0b[2] = {b[3] * U1[B][0] + b[5] * U1[B][1], b[5] * U1[B][0] + b[4] * U1[B][1]};
    const V3 U1b[2] = {V3{l[3], l[5], 0.0} + b[3] * U0[B][0] + b[5] * U0[B][1],
                       V3{l[5], l[4], 0.0} + b[5] * U0[B][0] + b[4] * U0[B][1]};
    V3 uxb = zero3(), ueb = zero3(), d0b = zero3(), dxb = zero3(), deb = zero3();
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const V3 P0 = comb(U0b[k], F.T[0], F.T[1], F.T[2]), P1 = comb(U1b[k], F.T[0], F.T[1], F.T[2]);
      uxb += x[k].x * P0 + z[k].x * P1;
      ueb += x[k].y * P0 + z[k].y * P1;
      d0b += x[k].z * P0 + z[k].z * P1;
      dxb += x[k].x * P1;
      deb += x[k].y * P1;
    }
    double gl[5], gp[5];
    fields_adjoint(l, gl);
    fields_adjoint(b, gp);
    V3 qb[4], db[4];  // displacements and directors of the nodes
#pragma unroll
    for (int m = 0; m < 4; m++) {
      qb[m] = Na[m] * uxb + Nb[m] * ueb;
      db[m] = N[m] * d0b + Na[m] * dxb + Nb[m] * deb;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 5; i++) {
      sm.b.g[p][A][i] = gl[i];
      sm.b.g[p][P][i] = gp[i];
    }
    sm.b.e8[p][A] = l[8];
    __syncthreads();
#pragma unroll 1
    for (int t = p; t < 9; t += 4) {
      double u, v, tN[4], tNa[4], tNb[4];
      const int f = tying_field(t);
      const double wl = tying_weight(t, A), wp = tying_weight(t, P);
      tying_point(t, u, v);
      shape4(u, v, tN, tNa, tNb);
      V3 fx, fe, d = zero3(), tn = zero3(), tux = zero3(), tue = zero3(), td = zero3();
      const V3 at = sum(tNa, X), bt = sum(tNb, X);
      grad_u(B, tNa, tNb, fx, fe);
#pragma unroll
      for (int m = 0; m < 4; m++) {
        d += tN[m] * director(B, m);
        tn += tN[m] * load3(&sm.fn[3 * m]);
      }
      if (f == kG11) {
        tux = wl * at + wp * fx;
      } else if (f == kG22) {
        tue = wl * bt + wp * fe;
      } else if (f == kG12) {
        tux = 0.5 * (wl * bt + wp * fe);
        tue = 0.5 * (wl * at + wp * fx);
      } else if (f == kG23) {
        td = 0.5 * (wl * bt + wp * fe);
        tue = 0.5 * (wl * tn + wp * d);
      } else {
        td = 0.5 * (wl * at + wp * fx);
        tux = 0.5 * (wl * tn + wp * d);
      }
#pragma unroll
      for (int m = 0; m < 4; m++) {
        qb[m] += tNa[m] * tux + tNb[m] * tue;
        db[m] += tN[m] * td;
      }
    }
    const double w = drill_weight(A), hw = 0.5 * w;
    const V3 sxb = hw * (nx1.x * nf.T[1] - nx2.x * nf.T[0]), seb = hw * (nx1.y * nf.T[1] - nx2.y * nf.T[0]);
    const V3 rotb = -w * cross(nf.T[0], nf.T[1]);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const V3 qm = qb[m] + nNa[m] * sxb + nNb[m] * seb;
      V3 rm = cross(load3(&sm.fn[3 * m]), db[m]);
      if (m == p) rm += rotb;
      double *o = &sm.part[p][6 * m];
      o[0] = qm.x;
      o[1] = qm.y;
      o[2] = qm.z;
      o[3] = rm.x;
      o[4] = rm.y;
      o[5] = rm.z;
    }
    __syncthreads();
    if (!active) return;
    double *dst = out + (design * a.nelems + e) * 24 + 6 * p;
#pragma unroll
    for (int i = 0; i < 6; i++)
      dst[i] = ((sm.part[0][6 * p + i] + sm.part[1][6 * p + i]) + sm.part[2][6 * p + i]) + sm.part[3][6 * p + i];
    return;
  }
  // adjoints of the directors at the point (values and gradients)
  V3 d0b[NW], dxb[NW], deb[NW];
#pragma unroll
  for (int s = 0; s < NW; s++) d0b[s] = dxb[s] = deb[s] = zero3();
  if constexpr (kPhi && OUT == kCoord) {
    if (c[3] != 0.0) {
      // mass moments of TACSIsoShellConstitutive with tOffset = 0
      const double m0 = a.mat.rho * thick, m2 = a.mat.rho * thick * thick * thick / 12.0;
      V3 u0 = zero3();
#pragma unroll
      for (int m = 0; m < 4; m++) u0 += N[m] * load3(&sm.q[wi[0]][6 * m]);
      value += c[3] * (m0 * dot(u0, u0) + m2 * dot(d0[wi[0]], d0[wi[0]]));
      d0b[wi[0]] += (2.0 * c[3] * det * m2) * d0[wi[0]];
    }
  }
  // ---- back through the strains ----
  V3 xb[3] = {zero3(), zero3(), zero3()}, zb[2] = {zero3(), zero3()};
  double gb[NS][5], e8b[NW];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    // E = x^T G x with E's adjoint symmetric: rows 0, 1, 2, 6, 7
    double g[5];
    fields(s, g);
    const double *b = sb[s];
    const V3 y0 = sym_mul(g, x[0]), y1 = sym_mul(g, x[1]), y2 = sym_mul(g, x[2]);
    xb[0] += 2.0 * (b[0] * y0 + b[2] * y1 + b[7] * y2);
    xb[1] += 2.0 * (b[2] * y0 + b[1] * y1 + b[6] * y2);
    xb[2] += 2.0 * (b[7] * y0 + b[6] * y1);
    fields_adjoint(b, gb[s]);
  }
  V3 Tb[3] = {zero3(), zero3(), zero3()};
#pragma unroll
  for (int s = 0; s < NW; s++) {
    e8b[s] = sb[s][8];
    // adjoints of the columns of U0, U1: bending strains, then the pairs
    V3 U0b[2] = {zero3(), zero3()}, U1b[2];
    U1b[0] = {sb[s][3], sb[s][5], 0.0};
    U1b[1] = {sb[s][5], sb[s][4], 0.0};
#pragma unroll
    for (int k = 0; k < 4; k++)
      if ((PM >> k) & 1) {
        const double *b = sb[pi[k]];
        const int A = wi[kPairA[k]], B = wi[kPairB[k]];
        if (s == A) {
          U0b[0] += b[3] * U1[B][0] + b[5] * U1[B][1];
          U0b[1] += b[5] * U1[B][0] + b[4] * U1[B][1];
          U1b[0] += b[3] * U0[B][0] + b[5] * U0[B][1];
          U1b[1] += b[5] * U0[B][0] + b[4] * U0[B][1];
        }
        if (s == B) {
          U0b[0] += b[3] * U1[A][0] + b[5] * U1[A][1];
          U0b[1] += b[5] * U1[A][0] + b[4] * U1[A][1];
          U1b[0] += b[3] * U0[A][0] + b[5] * U0[A][1];
          U1b[1] += b[5] * U0[A][0] + b[4] * U0[A][1];
        }
      }
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const V3 P = comb(x[k], ux[s], ue[s], d0[s]);
      const V3 S = x[k].x * dx[s] + x[k].y * de[s] + comb(z[k], ux[s], ue[s], d0[s]);
      const V3 P0 = comb(U0b[k], F.T[0], F.T[1], F.T[2]), P1 = comb(U1b[k], F.T[0], F.T[1], F.T[2]);
      Tb[0] += U0b[k].x * P + U1b[k].x * S;
      Tb[1] += U0b[k].y * P + U1b[k].y * S;
      Tb[2] += U0b[k].z * P + U1b[k].z * S;
      xb[k] += V3{dot(ux[s], P0) + dot(dx[s], P1), dot(ue[s], P0) + dot(de[s], P1), dot(d0[s], P0)};
      zb[k] += V3{dot(ux[s], P1), dot(ue[s], P1), dot(d0[s], P1)};
      d0b[s] += x[k].z * P0 + z[k].z * P1;
      dxb[s] += x[k].x * P1;
      deb[s] += x[k].y * P1;
    }
  }
  // ---- back through the frame of the point ----
  V3 Gi[3] = {zero3(), zero3(), zero3()}, nab = zero3(), nbb = zero3();
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const V3 hb = -1.0 * I.mul_t(zb[k]);
    Gi[0] += -zb[k].x * h[k];
    Gi[1] += -zb[k].y * h[k];
    Gi[2] += -zb[k].z * h[k];
    nab += x[k].x * hb;
    nbb += x[k].y * hb;
    xb[k].x += dot(na, hb);
    xb[k].y += dot(nb, hb);
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    Tb[k] += I.mul_t(xb[k]);
    Gi[0] += xb[k].x * F.T[k];
    Gi[1] += xb[k].y * F.T[k];
    Gi[2] += xb[k].z * F.T[k];
  }
  V3 ab = I.column(0, Gi, value), bb = I.column(1, Gi, value), n0b = I.column(2, Gi, value);
  F.adjoint(aq, Tb, ab, n0b);
  V3 Xb[4], fb[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    Xb[m] = Na[m] * ab + Nb[m] * bb;
    fb[m] = N[m] * n0b + Na[m] * nab + Nb[m] * nbb;
#pragma unroll
    for (int s = 0; s < NW; s++)
      fb[m] += cross(N[m] * d0b[s] + Na[m] * dxb[s] + Nb[m] * deb[s], load3(&sm.q[s][6 * m + 3]));
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int i = 0; i < 5; i++) sm.b.g[p][s][i] = gb[s][i];
#pragma unroll
  for (int s = 0; s < NW; s++) sm.b.e8[p][s] = e8b[s];
  __syncthreads();
  // ---- back through the tying points ----
#pragma unroll 1
  for (int t = p; t < 9; t += 4) {
    double u, v, tN[4], tNa[4], tNb[4], w[NS];
    const int f = tying_field(t);
#pragma unroll
    for (int s = 0; s < NS; s++) w[s] = tying_weight(t, s);
    tying_point(t, u, v);
    shape4(u, v, tN, tNa, tNb);
    const V3 at = sum(tNa, X), bt = sum(tNb, X);
    V3 tux[NW], tue[NW], td[NW];
#pragma unroll
    for (int s = 0; s < NW; s++) grad_u(s, tNa, tNb, tux[s], tue[s]);
    V3 atb = zero3(), btb = zero3(), tnb = zero3();
#pragma unroll
    for (int s = 0; s < NW; s++) {
      V3 d = zero3();
      td[s] = zero3();
#pragma unroll
      for (int m = 0; m < 4; m++) d += tN[m] * director(s, m);
      if (f == kG11) {
        atb += w[s] * tux[s];
      } else if (f == kG22) {
        btb += w[s] * tue[s];
      } else if (f == kG12) {
        atb += (0.5 * w[s]) * tue[s];
        btb += (0.5 * w[s]) * tux[s];
      } else if (f == kG23) {
        btb += (0.5 * w[s]) * d;
        td[s] += (0.5 * w[s]) * bt;
        tnb += (0.5 * w[s]) * tue[s];
      } else {
        atb += (0.5 * w[s]) * d;
        td[s] += (0.5 * w[s]) * at;
        tnb += (0.5 * w[s]) * tux[s];
      }
    }
    if (f == kG23 || f == kG13) {
#pragma unroll
      for (int k = 0; k < 4; k++)
        if ((PM >> k) & 1) {
          const int A = wi[kPairA[k]], B = wi[kPairB[k]];
          const double hw = 0.5 * w[pi[k]];
          td[A] += hw * (f == kG23 ? tue[B] : tux[B]);
          td[B] += hw * (f == kG23 ? tue[A] : tux[A]);
        }
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
      Xb[m] += tNa[m] * atb + tNb[m] * btb;
      V3 s3 = tnb;
#pragma unroll
      for (int s = 0; s < NW; s++) s3 += cross(td[s], load3(&sm.q[s][6 * m + 3]));
      fb[m] += tN[m] * s3;
    }
  }
  // ---- back through the drilling strains of node p ----
  V3 Tnb[3] = {zero3(), zero3(), zero3()}, x1b = zero3(), x2b = zero3(), cb = zero3();
#pragma unroll
  for (int s = 0; s < NW; s++) {
    const double w = drill_weight(s);
    V3 sx, se;
    grad_u(s, nNa, nNb, sx, se);
    cb += -w * load3(&sm.q[s][6 * p + 3]);
    const double hw = 0.5 * w;
    Tnb[1] += hw * (nx1.x * sx + nx1.y * se);
    Tnb[0] += -hw * (nx2.x * sx + nx2.y * se);
    x1b.x += hw * dot(nf.T[1], sx);
    x1b.y += hw * dot(nf.T[1], se);
    x2b.x -= hw * dot(nf.T[0], sx);
    x2b.y -= hw * dot(nf.T[0], se);
  }
  Tnb[0] += cross(nf.T[1], cb) + ni.mul_t(x1b);
  Tnb[1] += cross(cb, nf.T[0]) + ni.mul_t(x2b);
  V3 nGi[3];
  nGi[0] = x1b.x * nf.T[0] + x2b.x * nf.T[1];
  nGi[1] = x1b.y * nf.T[0] + x2b.y * nf.T[1];
  nGi[2] = zero3();
  V3 anb = ni.column(0, nGi, 0.0), bnb = ni.column(1, nGi, 0.0), fnb = ni.column(2, nGi, 0.0);
  nf.adjoint(an, Tnb, anb, fnb);
  // ---- the normals' adjoints, summed over the lanes, through node p's normal ----
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; m++) {
    sm.part[p][3 * m] = fb[m].x;
    sm.part[p][3 * m + 1] = fb[m].y;
    sm.part[p][3 * m + 2] = fb[m].z;
  }
  __syncthreads();
#pragma unroll
  for (int l = 0; l < 4; l++) fnb += load3(&sm.part[l][3 * p]);
  const V3 cb3 = fi * (fnb - dot(fnp, fnb) * fnp);
  anb += cross(bn, cb3);
  bnb += cross(cb3, an);
#pragma unroll
  for (int m = 0; m < 4; m++) Xb[m] += nNa[m] * anb + nNb[m] * bnb;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; m++) {
    sm.part[p][3 * m] = Xb[m].x;
    sm.part[p][3 * m + 1] = Xb[m].y;
    sm.part[p][3 * m + 2] = Xb[m].z;
  }
  __syncthreads();
  if (!active) return;
  const V3 o = ((load3(&sm.part[0][3 * p]) + load3(&sm.part[1][3 * p])) + load3(&sm.part[2][3 * p])) +
               load3(&sm.part[3][3 * p]);
  double *dst = out + (design * a.nelems + e) * 12 + 3 * p;
  dst[0] = o.x;
  dst[1] = o.y;
  dst[2] = o.z;
}

// dst[node] += the node's W values of its elements' gradients, in element order
template <int W>
__global__ __launch_bounds__(256) void xpt_gather_kernel(int n, int nelems, const int *__restrict__ ptr,
                                                         const int *__restrict__ corner, const double *__restrict__ g,
                                                         double *dst, long stride) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= W * n) return;
  const int node = i / W, d = i - W * node;
  const long o = blockIdx.y * (long)nelems * (4 * W) + d;
  double s = 0.0;
  for (int k = ptr[node]; k < ptr[node + 1]; k++) s += g[o + (long)W * corner[k]];
  dst[blockIdx.y * stride + i] += s;
}

template <int W>
void gather(const XptArgs &a, int nnodes, int nbatch, const int *node_ptr, const int *node_corner, const double *work,
            double *dst, long stride, hipStream_t stream) {
  hipLaunchKernelGGL(xpt_gather_kernel<W>, dim3((W * nnodes + 255) / 256, nbatch), dim3(256), 0, stream, nnodes,
                     a.nelems, node_ptr, node_corner, work, dst, stride);
}

}  // namespace

hipError_t launch_xpt_kernel(const XptArgs &args, int nnodes, int nbatch, const int *node_ptr, const int *node_corner,
                             double *work, hipStream_t stream) {
  if (args.nelems <= 0) return hipSuccess;
  const dim3 grid((args.nelems + kElems - 1) / kElems, nbatch), block(4 * kElems);
  const int t = args.terms;
  if (t & kXptR)  // u, psi; (u, psi) and (u, u) for the nonlinear model
    if (args.nonlin)
      hipLaunchKernelGGL((xpt_kernel<6, 12, kCoord>), grid, block, 0, stream, args, work);
    else
      hipLaunchKernelGGL((xpt_kernel<6, 0, kCoord>), grid, block, 0, stream, args, work);
  else if (t & kXptG)  // phi, u; (u, phi) and (phi, phi)
    hipLaunchKernelGGL((xpt_kernel<3, 3, kCoord>), grid, block, 0, stream, args, work);
  else  // phi alone: s_K, s_M
    hipLaunchKernelGGL((xpt_kernel<1, 0, kCoord>), grid, block, 0, stream, args, work);
  gather<3>(args, nnodes, nbatch, node_ptr, node_corner, work, args.dfdX, args.dX_stride, stream);
  return hipGetLastError();
}

hipError_t launch_dv_kernel(const XptArgs &args, int nnodes, int nbatch, const int *node_ptr, const int *node_corner,
                            double *work, hipStream_t stream) {
  if (args.nelems <= 0) return hipSuccess;
  const dim3 grid((args.nelems + kElems - 1) / kElems, nbatch), block(4 * kElems);
  if (args.terms & kXptR)
    if (args.nonlin)
      hipLaunchKernelGGL((xpt_kernel<6, 12, kThick>), grid, block, 0, stream, args, work);
    else
      hipLaunchKernelGGL((xpt_kernel<6, 0, kThick>), grid, block, 0, stream, args, work);
  else if (args.res) {
    hipLaunchKernelGGL((xpt_kernel<3, 3, kThickPath>), grid, block, 0, stream, args, work);
    gather<6>(args, nnodes, nbatch, node_ptr, node_corner, work, args.res, args.stride, stream);
  } else if (args.terms & kXptG)
    hipLaunchKernelGGL((xpt_kernel<3, 3, kThick>), grid, block, 0, stream, args, work);
  else
    hipLaunchKernelGGL((xpt_kernel<1, 0, kThick>), grid, block, 0, stream, args, work);
  return hipGetLastError();
}

}  // namespace shellgpu
