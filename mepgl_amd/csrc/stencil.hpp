// Per-site Ginzburg-Landau arithmetic of the relaxation loop, shared by the
// HIP kernels.  Each function restates one reference kernel's per-site body
// (mepgl/src/nlcg.cu) on values already gathered into registers, in the
// compute type T (double for the FP64 path, float for the mixed path).
//
// Neighbour slots: 0 = own site, 1 = +x, 2 = -x, 3 = +y, 4 = -y.
// A is also needed on the diagonals for the curl gradient: ax[dy+1][dx+1].
#pragma once

#include "common.hpp"

namespace mepgl {

__device__ __forceinline__ int bitof(int m, int k) { return (m >> k) & 1; }

template <class T>
__device__ __forceinline__ T sq(T v) { return v * v; }

// Neighbour-pair and quadrant presence of an 8-bit neighbour mask, as bit
// masks: bit k of pair_bits is set when neighbours k and k + 1 (mod 8) are
// both present; bit 2q of quad_bits when quadrant q (neighbours 2q, 2q + 1,
// 2q + 2 mod 8) is complete.  Weights and flags below are popcounts and bits
// of these, so they are the same small integers as the products of single
// bits they replace.
__device__ __forceinline__ unsigned pair_bits(int m) {
  const unsigned w = (unsigned)m | ((unsigned)m << 8);
  return w & (w >> 1);
}
__device__ __forceinline__ unsigned quad_bits(int m) {
  const unsigned p = pair_bits(m);
  return p & (p >> 1) & 0x55u;
}
__device__ __forceinline__ int popc(unsigned v) { return __builtin_popcount(v); }

// Quadrant area weight (S0S1S2 + S2S3S4 + S4S5S6 + S6S7S0)/4, nlcg.cu:140-143.
__device__ __forceinline__ int quad_count(int m) { return popc(quad_bits(m)); }

// Bond weights of nlcg.cu:188-189 and 552-571 as pair counts:
// (S1S2 + S6S7)/2 (forward x), (S2S3 + S5S6)/2 (backward x),
// (S0S1 + S3S4)/2 (forward y), (S4S5 + S7S0)/2 (backward y).
__device__ __forceinline__ int wx_fwd(unsigned p) { return popc(p & 0x42u); }
__device__ __forceinline__ int wx_bwd(unsigned p) { return popc(p & 0x24u); }
__device__ __forceinline__ int wy_fwd(unsigned p) { return popc(p & 0x09u); }
__device__ __forceinline__ int wy_bwd(unsigned p) { return popc(p & 0x90u); }

// Per-site constants of one component.
template <class T>
struct CompConst {
  T q;       // charge
  T two_a;   // 2 a
  T two_b;   // 2 b
  T b;       // b
  T ab;      // a / b
  T hx, hy;  // 0.5 / m_xx, 0.5 / m_yy
};

template <class T>
__device__ __forceinline__ double param_at(const DevParam& p, long long off) {
  // Parameter planes live in global memory: a global (not flat) load.
  using gd = __attribute__((address_space(1))) const double*;
  return p.p ? ((gd)p.p)[off] : p.v;
}

template <class T, int NC>
__device__ __forceinline__ void load_comp_const(const DevString& s, long long off,
                                                CompConst<T> (&k)[NC]) {
  if (!s.planes) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      k[c].q = (T)s.kc[c][0];
      k[c].two_a = (T)s.kc[c][1];
      k[c].two_b = (T)s.kc[c][2];
      k[c].b = (T)s.kc[c][3];
      k[c].ab = (T)s.kc[c][4];
      k[c].hx = (T)s.kc[c][5];
      k[c].hy = (T)s.kc[c][6];
    }
    return;
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double a = param_at<T>(s.a[c], off), b = param_at<T>(s.b[c], off);
    const double mx = param_at<T>(s.mxx[c], off), my = param_at<T>(s.myy[c], off);
    k[c].q = (T)s.q[c];
    k[c].two_a = (T)(2.0 * a);
    k[c].two_b = (T)(2.0 * b);
    k[c].b = (T)b;
    k[c].ab = (T)(a / b);
    k[c].hx = (T)(0.5 / mx);
    k[c].hy = (T)(0.5 / my);
  }
}

// The parameter descriptors of a string, read once into registers before a
// row loop (reading them from the descriptor inside the loop would be a
// memory load per row).
template <int NC>
struct ParamView {
  int planes;
  DevParam a[NC], b[NC], mxx[NC], myy[NC];
  double q[NC];
};

template <int NC>
__device__ __forceinline__ ParamView<NC> param_view(const DevString& s) {
  ParamView<NC> v;
  v.planes = s.planes;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    v.a[c] = s.a[c];
    v.b[c] = s.b[c];
    v.mxx[c] = s.mxx[c];
    v.myy[c] = s.myy[c];
    v.q[c] = s.q[c];
  }
  return v;
}

// Per-site constants of plane parameters (ParamView::planes != 0).
template <class T, int NC>
__device__ __forceinline__ void load_comp_planes(const ParamView<NC>& v, long long off,
                                                 CompConst<T> (&k)[NC]) {
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double a = param_at<T>(v.a[c], off), b = param_at<T>(v.b[c], off);
    const double mx = param_at<T>(v.mxx[c], off), my = param_at<T>(v.myy[c], off);
    k[c].q = (T)v.q[c];
    k[c].two_a = (T)(2.0 * a);
    k[c].two_b = (T)(2.0 * b);
    k[c].b = (T)b;
    k[c].ab = (T)(a / b);
    k[c].hx = (T)(0.5 / mx);
    k[c].hy = (T)(0.5 / my);
  }
}

// Gathered neighbourhood of one site.
template <class T, int NC>
struct Nbhd {
  T ax[3][3], ay[3][3];  // A on the 3x3 stencil, [dy+1][dx+1]
  T u[NC][5], v[NC][5];  // order parameters on the 5-point stencil
  T h[5];                // applied field on the 5-point stencil
};

// ---------------------------------------------------------------------------
// Kinetic bond of one component, gradient with respect to psi and A.
// Forward bond (+x or +y): nlcg.cu:529-549 / 573-593 and 769-776 / 787-794.
// Backward bond (-x or -y): nlcg.cu:551-571 / 595-615 and 778-785 / 796-803.
// u0,v0,A0: own site; un,vn,An: neighbour; hm = 0.5/m; w = bond weight.
template <class T>
__device__ __forceinline__ void bond_fwd(T u0, T v0, T A0, T un, T vn, T An, T q, T hm, T w,
                                         T idx, T& gu, T& gv, T& gA) {
  const T du = (un - u0) * idx, dv = (vn - v0) * idx;
  const T t1 = -du - q * A0 * v0;
  const T t2 = -du - q * An * vn;
  const T t3 = dv - q * A0 * u0;
  const T t4 = dv - q * An * un;
  const T hw = hm * w;
  gu += hw * (idx * t1 + idx * t2 - q * A0 * t3);
  gv += hw * (-idx * t3 - idx * t4 - q * A0 * t1);
  gA += -q * hw * (v0 * t1 + u0 * t3);
}

template <class T>
__device__ __forceinline__ void bond_bwd(T u0, T v0, T A0, T um, T vm, T Am, T q, T hm, T w,
                                         T idx, T& gu, T& gv, T& gA) {
  const T du = (u0 - um) * idx, dv = (v0 - vm) * idx;
  const T s1 = -du - q * A0 * v0;
  const T s2 = -du - q * Am * vm;
  const T s3 = dv - q * A0 * u0;
  const T s4 = dv - q * Am * um;
  const T hw = hm * w;
  gu += hw * (-idx * s1 - idx * s2 - q * A0 * s3);
  gv += hw * (idx * s3 + idx * s4 - q * A0 * s1);
  gA += -q * hw * (v0 * s1 + u0 * s3);
}

// Full gradient of one site (gradientPsi + gradientA, nlcg.cu:504-888),
// already multiplied by dx^2.  do_a = false skips the A part
// (NO_SELF_FIELD).  The psi part is always evaluated: its kinetic bonds also
// give the bond terms of the A gradient, and in Maxwell mode (nlcg.cu:1521)
// the caller keeps the frozen psi gradient instead of gpsi.
template <class T, int NC>
__device__ __forceinline__ void site_gradient(const Nbhd<T, NC>& s, const CompConst<T> (&k)[NC],
                                              T eta, T gamma, T delta, T idx, T dx2, int sc,
                                              int cm, bool do_a, T (&gpsi)[NC][2], T (&ga)[2]) {
  const unsigned sp = pair_bits(sc);
  const T af = (T)quad_count(sc) * (T)0.25;
  const T wxf = (T)wx_fwd(sp) * (T)0.5;
  const T wxb = (T)wx_bwd(sp) * (T)0.5;
  const T wyf = (T)wy_fwd(sp) * (T)0.5;
  const T wyb = (T)wy_bwd(sp) * (T)0.5;
  const T AX0 = s.ax[1][1], AY0 = s.ay[1][1];
  T gax = 0, gay = 0;

  // Each bond contributes only when its neighbour exists (bits 0, 4, 2, 6).
  // Its presence is folded into its weight once per site: an absent bond
  // gets weight 0, and every term it adds is then an exact zero (the fields
  // are finite), so no lane diverges and no term needs a select.
  const T wxf0 = bitof(sc, 0) ? wxf : (T)0, wxb0 = bitof(sc, 4) ? wxb : (T)0;
  const T wyf0 = bitof(sc, 2) ? wyf : (T)0, wyb0 = bitof(sc, 6) ? wyb : (T)0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T u0 = s.u[c][0], v0 = s.v[c][0];
    const T n2 = u0 * u0 + v0 * v0;
    T gu = (k[c].two_a * u0 + k[c].two_b * u0 * n2) * af;
    T gv = (k[c].two_a * v0 + k[c].two_b * v0 * n2) * af;
    T bu, bv, bA;
    bu = bv = bA = 0;
    bond_fwd(u0, v0, AX0, s.u[c][1], s.v[c][1], s.ax[1][2], k[c].q, k[c].hx, wxf0, idx, bu, bv, bA);
    gu += bu;
    gv += bv;
    gax += bA;
    bu = bv = bA = 0;
    bond_bwd(u0, v0, AX0, s.u[c][2], s.v[c][2], s.ax[1][0], k[c].q, k[c].hx, wxb0, idx, bu, bv, bA);
    gu += bu;
    gv += bv;
    gax += bA;
    bu = bv = bA = 0;
    bond_fwd(u0, v0, AY0, s.u[c][3], s.v[c][3], s.ay[2][1], k[c].q, k[c].hy, wyf0, idx, bu, bv, bA);
    gu += bu;
    gv += bv;
    gay += bA;
    bu = bv = bA = 0;
    bond_bwd(u0, v0, AY0, s.u[c][4], s.v[c][4], s.ay[0][1], k[c].q, k[c].hy, wyb0, idx, bu, bv, bA);
    gu += bu;
    gv += bv;
    gay += bA;
    gpsi[c][0] = gu;
    gpsi[c][1] = gv;
  }
  if (NC == 2) {
    // Couplings, nlcg.cu:623-650.
    const T u1 = s.u[0][0], v1 = s.v[0][0], u2 = s.u[NC - 1][0], v2 = s.v[NC - 1][0];
    const T n1 = u1 * u1 + v1 * v1, n2 = u2 * u2 + v2 * v2;
    const T P = u1 * u2 + v1 * v2, Q = u1 * v2 - v1 * u2;
    const T ea = eta * af, ga_ = gamma * af, da = delta * af;
    gpsi[0][0] += ea * u2 + ga_ * u1 * n2 + da * (u2 * P - v2 * Q);
    gpsi[0][1] += ea * v2 + ga_ * v1 * n2 + da * (v2 * P + u2 * Q);
    gpsi[NC - 1][0] += ea * u1 + ga_ * u2 * n1 + da * (u1 * P + v1 * Q);
    gpsi[NC - 1][1] += ea * v1 + ga_ * v2 * n1 + da * (v1 * P - u1 * Q);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    gpsi[c][0] *= dx2;
    gpsi[c][1] *= dx2;
  }

  if (do_a) {
    // Curl terms, nlcg.cu:852-883: 8 own-quadrant and 8 neighbour-quadrant
    // contributions, gated on the own site's quadrant bits.
    const T c4 = (T)0.25 * idx;
    const T(&X)[3][3] = s.ax;
    const T(&Y)[3][3] = s.ay;
    const T dyf = (Y[1][2] - Y[1][1]) * idx;  // forward x-difference of A_y
    const T dyb = (Y[1][1] - Y[1][0]) * idx;
    const T dxf = (X[2][1] - X[1][1]) * idx;  // forward y-difference of A_x
    const T dxb = (X[1][1] - X[0][1]) * idx;
    const T h0 = s.h[0];
    // Quadrant presence folded into the quadrant's weight, as for the bonds.
    const unsigned cq = quad_bits(cm);
    const T c0 = (cq & 0x01u) ? c4 : (T)0;
    const T c1 = (cq & 0x04u) ? c4 : (T)0;
    const T c2 = (cq & 0x10u) ? c4 : (T)0;
    const T c3 = (cq & 0x40u) ? c4 : (T)0;
    {
      const T e = dyf - dxf - h0;
      const T n1 = dyf - (X[2][2] - X[1][2]) * idx - s.h[1];
      const T n2 = (Y[2][2] - Y[2][1]) * idx - dxf - s.h[3];
      gax += c0 * e + c0 * n2;
      gay += -c0 * e - c0 * n1;
    }
    {
      const T e = dyb - dxf - h0;
      const T n1 = (Y[2][1] - Y[2][0]) * idx - dxf - s.h[3];
      const T n2 = dyb - (X[2][0] - X[1][0]) * idx - s.h[2];
      gax += c1 * e + c1 * n1;
      gay += c1 * e + c1 * n2;
    }
    {
      const T e = dyb - dxb - h0;
      const T n1 = dyb - (X[1][0] - X[0][0]) * idx - s.h[2];
      const T n2 = (Y[0][1] - Y[0][0]) * idx - dxb - s.h[4];
      gax += -c2 * e - c2 * n2;
      gay += c2 * e + c2 * n1;
    }
    {
      const T e = dyf - dxb - h0;
      const T n1 = (Y[0][2] - Y[0][1]) * idx - dxb - s.h[4];
      const T n2 = dyf - (X[1][2] - X[0][2]) * idx - s.h[1];
      gax += -c3 * e - c3 * n1;
      gay += -c3 * e - c3 * n2;
    }
    ga[0] = gax * dx2;
    ga[1] = gay * dx2;
  }
}

// ---------------------------------------------------------------------------
// Line-search quartic of one site, polynomialExpansion nlcg.cu:997-1370.
// x and direction d on the 5-point stencil (A and psi); returns A..E.
template <class T, int NC>
struct PolyNbhd {
  T ax[5], ay[5];            // slots 0 own, 1 +x, 2 -x, 3 +y, 4 -y
  T dax[5], day[5];
  T u[NC][3], v[NC][3];      // slots 0 own, 1 +x, 2 +y
  T du[NC][3], dv[NC][3];
  T h0;
};

template <class T>
struct Quartic {
  T c[5];
};

// One kinetic bond (+x: A = A_x, +y: A = A_y) of one component, in units of
// dx: differences are not divided by dx, q0 = q dx A and b0 = q dx d_A at the
// own site (qn, bn at the neighbour), c0 and cn the first-order coefficient
// times d_A there.  f is the bond's weight 0.5 / m, f3 its weight on the cubic
// term.
template <class T>
__device__ __forceinline__ void poly_bond(T u0, T v0, T un, T vn, T du0, T dv0, T dun, T dvn, T q0,
                                          T qn, T b0, T bn, T c0, T cn, T f, T f3, Quartic<T>& r) {
  const T Du = u0 - un, Dv = vn - v0, Ddu = du0 - dun, Ddv = dvn - dv0;
  T k0[4], k1[4], k2[4];
  k0[0] = fma(-q0, v0, Du);
  k0[1] = fma(-qn, vn, Du);
  k0[2] = fma(-q0, u0, Dv);
  k0[3] = fma(-qn, un, Dv);
  k1[0] = fma(c0, v0, fma(-q0, dv0, Ddu));
  k1[1] = fma(cn, vn, fma(-qn, dvn, Ddu));
  k1[2] = fma(c0, u0, fma(-q0, du0, Ddv));
  k1[3] = fma(cn, un, fma(-qn, dun, Ddv));
  k2[0] = -b0 * dv0;
  k2[1] = -bn * dvn;
  k2[2] = -b0 * du0;
  k2[3] = -bn * dun;
  T s00 = k0[0] * k0[0], s01 = k0[0] * k1[0], s11 = k1[0] * k1[0];
  T s02 = k0[0] * k2[0], s12 = k1[0] * k2[0], s22 = k2[0] * k2[0];
#pragma unroll
  for (int t = 1; t < 4; ++t) {
    s00 = fma(k0[t], k0[t], s00);
    s01 = fma(k0[t], k1[t], s01);
    s11 = fma(k1[t], k1[t], s11);
    s02 = fma(k0[t], k2[t], s02);
    s12 = fma(k1[t], k2[t], s12);
    s22 = fma(k2[t], k2[t], s22);
  }
  const T fh = (T)0.5 * f;
  r.c[0] = fma(s00, fh, r.c[0]);
  r.c[1] = fma(s01, f, r.c[1]);
  r.c[2] = fma(s11, fh, fma(s02, f, r.c[2]));
  r.c[3] = fma(s12, f3, r.c[3]);
  r.c[4] = fma(s22, fh, r.c[4]);
}

// Constants of the quartic, with the factors of dx that its units leave.
template <class T, int NC>
struct PolyConst {
  struct {
    T ab;       // a / b
    T kb;       // b dx^2 / 4
    T q;        // q dx
    T c1;       // first-order coefficient of d_A on the x bond, times dx
    T hx, hy;   // 0.25 / m
    T hy3;      // hy, halved on the cubic term of the reference's quartic
  } k[NC];
  T eta, gam, del;  // eta dx^2 / 4, gamma dx^2 / 8, delta dx^2 / 8
};

template <class T, int NC>
__device__ __forceinline__ PolyConst<T, NC> poly_const(const CompConst<T> (&k)[NC], T eta, T gamma,
                                                       T delta, T dx, T dx2, bool exact) {
  PolyConst<T, NC> p;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    p.k[c].ab = k[c].ab;
    p.k[c].kb = k[c].b * ((T)0.25 * dx2);
    p.k[c].q = k[c].q * dx;
    p.k[c].c1 = exact ? -p.k[c].q : dx;
    p.k[c].hx = (T)0.5 * k[c].hx;
    p.k[c].hy = (T)0.5 * k[c].hy;
    p.k[c].hy3 = exact ? p.k[c].hy : (T)0.5 * p.k[c].hy;
  }
  p.eta = eta * ((T)0.25 * dx2);
  p.gam = gamma * ((T)0.125 * dx2);
  p.del = delta * ((T)0.125 * dx2);
  return p;
}

// The quartic's arithmetic is most of what the P kernel issues.  Bonds and
// plaquettes are evaluated in units of dx, where their weights lose the
// factors dx^2 and 1 / dx, and each sum of products takes its weight once:
// about 30 % fewer operations per site than with every term scaled by itself.
// P took 140 us before and 135 us after on 24 two-component images of 512^2 in
// mixed precision, 76.4 and 71.7 us on a film of 8 images of 768^2, 59.9 and
// 58.4 us on 64 one-component images of 256^2.
// h0: the site's applied field times dx.
template <class T, int NC>
__device__ __forceinline__ Quartic<T> site_poly(const PolyNbhd<T, NC>& s,
                                                const PolyConst<T, NC>& pc, int sc, int cm,
                                                bool nsf) {
  Quartic<T> r;
#pragma unroll
  for (int t = 0; t < 5; ++t) r.c[t] = 0;
  const T qc = (T)quad_count(sc);
  // Nonlinear terms, nlcg.cu:1024-1112.
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T u = s.u[c][0], v = s.v[c][0], ud = s.du[c][0], vd = s.dv[c][0];
    const T n0 = fma(v, v, fma(u, u, pc.k[c].ab));
    const T pd = fma(v, vd, u * ud);
    const T n1 = pd + pd;
    const T n2 = fma(vd, vd, ud * ud);
    const T kb = pc.k[c].kb * qc;
    const T kh = (T)0.5 * kb, m0 = kb * n0;
    r.c[0] = fma(kh * n0, n0, r.c[0]);
    r.c[1] = fma(m0, n1, r.c[1]);
    r.c[2] = fma(m0, n2, fma(kh * n1, n1, r.c[2]));
    r.c[3] = fma(kb * n1, n2, r.c[3]);
    r.c[4] = fma(kh * n2, n2, r.c[4]);
  }
  if (NC == 2) {
    const T u1 = s.u[0][0], v1 = s.v[0][0], u2 = s.u[NC - 1][0], v2 = s.v[NC - 1][0];
    const T ud1 = s.du[0][0], vd1 = s.dv[0][0], ud2 = s.du[NC - 1][0], vd2 = s.dv[NC - 1][0];
    const T n1 = u1 * u1 + v1 * v1, n2 = u2 * u2 + v2 * v2;
    const T pd1 = u1 * ud1 + v1 * vd1, pd2 = u2 * ud2 + v2 * vd2;
    const T dd1 = ud1 * ud1 + vd1 * vd1, dd2 = ud2 * ud2 + vd2 * vd2;
    const T P = u1 * u2 + v1 * v2, Q = u1 * v2 - v1 * u2;
    const T P1 = u1 * ud2 + ud1 * u2 + v1 * vd2 + vd1 * v2;
    const T Q1 = u1 * vd2 + ud1 * v2 - v1 * ud2 - vd1 * u2;
    const T P2 = ud1 * ud2 + vd1 * vd2, Q2 = ud1 * vd2 - vd1 * ud2;
    // P, P1 and P2 are also the terms of the Josephson coupling.
    const T e = pc.eta * qc, g = pc.gam * qc, dl = pc.del * qc;
    const T g2 = g + g, dl2 = dl + dl;
    r.c[0] += e * P + g * n1 * n2 + dl * (P * P - Q * Q);
    r.c[1] += e * P1 + g2 * (pd1 * n2 + pd2 * n1) + dl2 * (P1 * P - Q1 * Q);
    r.c[2] += e * P2 + g * ((T)4 * pd1 * pd2 + n1 * dd2 + n2 * dd1) + dl * (P1 * P1 - Q1 * Q1) +
              dl2 * (P * P2 - Q * Q2);
    r.c[3] += g2 * (pd1 * dd2 + pd2 * dd1) + dl2 * (P1 * P2 - Q1 * Q2);
    r.c[4] += g * (dd1 * dd2) + dl * (P2 * P2 - Q2 * Q2);
  }
  // Magnetic term, nlcg.cu:1116-1157.
  if (!nsf) {
    const T yf = s.ay[1] - s.ay[0] - s.h0, yb = s.ay[0] - s.ay[2] - s.h0;
    const T xf = s.ax[3] - s.ax[0], xb = s.ax[0] - s.ax[4];
    const T dyf = s.day[1] - s.day[0], dyb = s.day[0] - s.day[2];
    const T dxf = s.dax[3] - s.dax[0], dxb = s.dax[0] - s.dax[4];
    // Quadrant presence as the quadrant's weight (absent: 0).
    const unsigned cq = quad_bits(cm);
    const T w[4] = {(cq & 0x01u) ? (T)1 : (T)0, (cq & 0x04u) ? (T)1 : (T)0,
                    (cq & 0x10u) ? (T)1 : (T)0, (cq & 0x40u) ? (T)1 : (T)0};
    const T e0[4] = {yf - xf, yb - xf, yb - xb, yf - xb};
    const T e1[4] = {dyf - dxf, dyb - dxf, dyb - dxb, dyf - dxb};
    T s00 = 0, s01 = 0, s11 = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const T we = w[t] * e0[t];
      s00 = fma(we, e0[t], s00);
      s01 = fma(we, e1[t], s01);
      s11 = fma(w[t] * e1[t], e1[t], s11);
    }
    r.c[0] = fma((T)0.125, s00, r.c[0]);
    r.c[1] = fma((T)0.25, s01, r.c[1]);
    r.c[2] = fma((T)0.125, s11, r.c[2]);
  }
  // Kinetic bonds, nlcg.cu:1160-1366; an absent bond (bits 0 and 2) has
  // weight 0.
  const unsigned sp = pair_bits(sc);
  const T cx = bitof(sc, 0) ? (T)wx_fwd(sp) : (T)0;
  const T cy = bitof(sc, 2) ? (T)wy_fwd(sp) : (T)0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const auto& k = pc.k[c];
    const T q = k.q, fx = k.hx * cx;
    const T bx0 = q * s.dax[0], bx1 = q * s.dax[1], by0 = q * s.day[0], by3 = q * s.day[3];
    poly_bond(s.u[c][0], s.v[c][0], s.u[c][1], s.v[c][1], s.du[c][0], s.dv[c][0], s.du[c][1],
              s.dv[c][1], q * s.ax[0], q * s.ax[1], bx0, bx1, k.c1 * s.dax[0], k.c1 * s.dax[1], fx,
              fx, r);
    poly_bond(s.u[c][0], s.v[c][0], s.u[c][2], s.v[c][2], s.du[c][0], s.dv[c][0], s.du[c][2],
              s.dv[c][2], q * s.ay[0], q * s.ay[3], by0, by3, -by0, -by3, k.hy * cy,
              k.hy3 * cy, r);
  }
  return r;
}

// ---------------------------------------------------------------------------
// Energy density of one site in double, freeEnergyDensity nlcg.cu:105-214.
// The fused operations are written out and the compiler forms no others, so
// every kernel that evaluates a site gets the same bits.
template <int NC>
__device__ __forceinline__ double site_energy(const PolyNbhd<double, NC>& s,
                                              const CompConst<double> (&k)[NC], double eta,
                                              double gamma, double delta, double idx,
                                              double dx2, int sc, int cm, bool nsf) {
#pragma clang fp contract(off)
  const double af = quad_count(sc) * 0.25;
  double nl = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double u = s.u[c][0], v = s.v[c][0];
    const double n0 = fma(v, v, fma(u, u, k[c].ab));
    nl = fma((0.5 * k[c].b) * n0, n0, nl);
  }
  if (NC == 2) {
    const double u1 = s.u[0][0], v1 = s.v[0][0], u2 = s.u[NC - 1][0], v2 = s.v[NC - 1][0];
    const double P = fma(v1, v2, u1 * u2), Q = fma(-v1, u2, u1 * v2);
    nl = fma(eta, P, nl);
    nl = fma((gamma * 0.5) * fma(v1, v1, u1 * u1), fma(v2, v2, u2 * u2), nl);
    nl = fma(delta * 0.5, fma(P, P, -(Q * Q)), nl);
  }
  nl *= af;
  // One kinetic bond: the sum of the squares at both of its ends.
  auto bond = [&](double u0, double v0, double A0, double un, double vn, double An, double q) {
#pragma clang fp contract(off)
    const double Du = (un - u0) * idx, Dv = (vn - v0) * idx, q0 = q * A0, qn = q * An;
    const double t1 = fma(q0, v0, Du), t2 = fma(qn, vn, Du);
    const double t3 = fma(-q0, u0, Dv), t4 = fma(-qn, un, Dv);
    return fma(t4, t4, fma(t3, t3, fma(t2, t2, t1 * t1)));
  };
  // Nothing of an absent bond (bits 0 and 2) or plaquette enters the sum: what
  // lies outside the sample need not be finite (a mass of zero, A).
  const unsigned sp = pair_bits(sc);
  const bool has_x = bitof(sc, 0), has_y = bitof(sc, 2);
  const double wx = wx_fwd(sp) * 0.25, wy = wy_fwd(sp) * 0.25;
  double e = nl;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double q = k[c].q;
    const double bx = bond(s.u[c][0], s.v[c][0], s.ax[0], s.u[c][1], s.v[c][1], s.ax[1], q);
    e = has_x ? fma(wx * k[c].hx, bx, e) : e;
    const double by = bond(s.u[c][0], s.v[c][0], s.ay[0], s.u[c][2], s.v[c][2], s.ay[3], q);
    e = has_y ? fma(wy * k[c].hy, by, e) : e;
  }
  if (!nsf) {
    const double yf = (s.ay[1] - s.ay[0]) * idx, yb = (s.ay[0] - s.ay[2]) * idx;
    const double xf = (s.ax[3] - s.ax[0]) * idx, xb = (s.ax[0] - s.ax[4]) * idx;
    const unsigned cq = quad_bits(cm);
    const double e0 = (cq & 0x01u) ? yf - xf - s.h0 : 0.0, e1 = (cq & 0x04u) ? yb - xf - s.h0 : 0.0;
    const double e2 = (cq & 0x10u) ? yb - xb - s.h0 : 0.0, e3 = (cq & 0x40u) ? yf - xb - s.h0 : 0.0;
    const double em = fma(e3, e3, fma(e2, e2, fma(e1, e1, e0 * e0)));
    e = fma(0.125, em, e);
  }
  return e * dx2;
}

// Magnetic field and supercurrents of one site, computeJBKernel
// nlcg.cu:243-364, in R (double for the JB output and the FP64 arclength;
// float in the mixed-precision arclength, as the mixed step kernels' own
// stencils).  Uses own-site A and no bond weights.
template <class R, int NC>
__device__ __forceinline__ void site_jb(const PolyNbhd<R, NC>& s, const R (&um)[NC],
                                        const R (&vm)[NC], const R (&uym)[NC],
                                        const R (&vym)[NC], const CompConst<R> (&k)[NC], R idx,
                                        int sc, int cm, R& b, R (&j)[NC][2]) {
  const R yf = (s.ay[1] - s.ay[0]) * idx, yb = (s.ay[0] - s.ay[2]) * idx;
  const R xf = (s.ax[3] - s.ax[0]) * idx, xb = (s.ax[0] - s.ax[4]) * idx;
  const R qr = (R)0.25;
  R bb = 0;
  if (bitof(cm, 0) && bitof(cm, 1) && bitof(cm, 2)) bb += qr * (yf - xf);
  if (bitof(cm, 2) && bitof(cm, 3) && bitof(cm, 4)) bb += qr * (yb - xf);
  if (bitof(cm, 4) && bitof(cm, 5) && bitof(cm, 6)) bb += qr * (yb - xb);
  if (bitof(cm, 6) && bitof(cm, 7) && bitof(cm, 0)) bb += qr * (yf - xb);
  if (bb != 0) bb /= (R)quad_count(cm) * qr;
  b = bb;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const R q = k[c].q, u0 = s.u[c][0], v0 = s.v[c][0];
    const R ax0 = s.ax[0], ay0 = s.ay[0];
    R jx = 0, jy = 0;
    const R fx = q * k[c].hx, fy = q * k[c].hy;  // 0.5 q / m
    if (bitof(sc, 0)) {
      const R Du = (s.u[c][1] - u0) * idx, Dv = (s.v[c][1] - v0) * idx;
      jx += fx * (v0 * (-Du - q * ax0 * v0) + u0 * (Dv - q * ax0 * u0));
    }
    if (bitof(sc, 4)) {
      const R Du = (u0 - um[c]) * idx, Dv = (v0 - vm[c]) * idx;
      jx += fx * (v0 * (-Du - q * ax0 * v0) + u0 * (Dv - q * ax0 * u0));
    }
    if (bitof(sc, 2)) {
      const R Du = (s.u[c][2] - u0) * idx, Dv = (s.v[c][2] - v0) * idx;
      jy += fy * (v0 * (-Du - q * ay0 * v0) + u0 * (Dv - q * ay0 * u0));
    }
    if (bitof(sc, 6)) {
      const R Du = (u0 - uym[c]) * idx, Dv = (v0 - vym[c]) * idx;
      jy += fy * (v0 * (-Du - q * ay0 * v0) + u0 * (Dv - q * ay0 * u0));
    }
    j[c][0] = jx;
    j[c][1] = jy;
  }
}

}  // namespace mepgl
