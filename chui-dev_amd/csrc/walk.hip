// walk.hip — wavefront-cooperative periodic short-range residual walk.
//
// One wave64 owns 64 consecutive tree-order targets. The tree is stored in
// preorder with subtree sizes, so each lane's depth-first walk is a monotone
// sequence of node indices: opening node i continues at i + 1, pruning or
// accepting it continues at i + skip(i). The wave always processes the smallest
// pending node index of its lanes (a wave-uniform index, so node records and
// leaf sources come through the scalar cache); lanes whose next node is larger
// sit that node out. Every lane therefore sees exactly the node sequence,
// acceptance decisions and summation order of the reference's per-target DFS
// (tree_pm_coupling.cpp:4026-4272), and leaf pairs are evaluated with the
// source shared by the whole wave.
//
// walk64_kernel  : FP64, the reference's arithmetic (erf/exp split
//                  kernel, nearbyint minimum image, monopole + quadrupole residual).
// walkmix_kernel : 32-bit fixed-point positions (minimum image = int32
//                  subtraction), FP32 pair kernel with a cubic-cell LDS table
//                  for the Gaussian coefficient H(t), per-drain partial sums
//                  folded into a Kahan-compensated FP32 accumulator.
#include "walk.hpp"

#include "primitives.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <vector>

namespace chui {
namespace {

constexpr double kInvSqrtPi = 0.564189583547756286948079451560772586;
constexpr int kWalkThreads = 256;

// ---- FP64 split kernel (tree_pm_split_kernel.hpp:66-228) -------------------
__device__ __forceinline__ double series_h(double t) {
  constexpr double c = 2.25675833419102514779231780624309034;
  return c * (1.0 / 3.0 + t * (-1.0 / 5.0 + t * (1.0 / 14.0 + t * (-1.0 / 54.0 + t * (1.0 / 264.0 +
         t * (-1.0 / 1560.0 + t * (1.0 / 10800.0 - t / 85680.0)))))));
}
__device__ __forceinline__ double short_factor(double r, double a) {
  if (r <= 0.0) return 1.0;
  const double q = (0.5 * r) / a;
  if (isinf(q)) return 0.0;
  return erfc(q) + 2.0 * kInvSqrtPi * q * exp(-q * q);
}
__device__ __forceinline__ double long_factor(double r, double a) {
  if (r <= 0.0) return 0.0;
  const double q = (0.5 * r) / a;
  if (isinf(q)) return 1.0;
  if (q < 0.125) {
    const double t = q * q;
    const double h = 4.0 * kInvSqrtPi * (1.0 / 3.0 + t * (-1.0 / 5.0 + t * (1.0 / 14.0 + t * (-1.0 / 54.0 +
        t * (1.0 / 264.0 + t * (-1.0 / 1560.0 + t * (1.0 / 10800.0 - t / 85680.0)))))));
    return q * q * q * h;
  }
  return erf(q) - 2.0 * kInvSqrtPi * q * exp(-q * q);
}
__device__ __forceinline__ double long_inv_r3(double r, double a) {
  const double q = (0.5 * r) / a;
  if (q < 0.125) return ((0.125 * series_h(q * q) / a) / a) / a;
  return ((long_factor(r, a) / r) / r) / r;
}
__device__ __forceinline__ double softened_inv_r3(double r2, double eps) {
  const double s = r2 + eps * eps;
  if (s <= 0.0) return 0.0;
  return 1.0 / (s * sqrt(s));
}
__device__ __forceinline__ double residual_inv_r3(double r2, double eps, double a) {
  if (r2 <= 0.0) {
    if (eps == 0.0) return softened_inv_r3(r2, eps);
    constexpr double k = 0.094031597257959381158013241926795431;
    if (eps <= a) {
      const double ratio = eps / a;
      return (((1.0 - k * ratio * ratio * ratio) / eps) / eps) / eps;
    }
    const double ratio = a / eps;
    return (((ratio * ratio * ratio - k) / a) / a) / a;
  }
  return softened_inv_r3(r2, eps) - long_inv_r3(sqrt(r2), a);
}

// d/dt of residual_inv_r3 at t = r^2. With q = r/(2a) and
// L(r) = erf(q) - 2q exp(-q^2)/sqrt(pi):
//   d/dt (t + eps^2)^{-3/2} = -1.5 (t + eps^2)^{-5/2},
//   d/dt [L(r)/r^3] = exp(-q^2) / (4 sqrt(pi) a^3 r^2) - 1.5 L(r)/r^5,
// the latter from the series of L(r)/r^3 = H(q^2)/(8a^3) below q = 1/8.
__device__ __forceinline__ double residual_inv_r3_dt(double r2, double eps, double a) {
  const double s = r2 + eps * eps;
  const double dsoft = s > 0.0 ? -1.5 / (s * s * sqrt(s)) : 0.0;
  const double r = sqrt(r2);
  const double q = (0.5 * r) / a;
  double dlong;
  if (q < 0.125) {
    constexpr double c = 2.25675833419102514779231780624309034;
    const double u = q * q;
    const double dh = c * (-1.0 / 5.0 + u * (2.0 / 14.0 + u * (-3.0 / 54.0 + u * (4.0 / 264.0 +
                      u * (-5.0 / 1560.0 + u * (6.0 / 10800.0 - 7.0 * u / 85680.0))))));
    dlong = (0.125 / (a * a * a)) * dh * (0.25 / (a * a));  // dH/du * du/dt, u = t / (4 a^2)
  } else {
    dlong = exp(-q * q) * kInvSqrtPi / (4.0 * a * a * a * r2) - 1.5 * long_factor(r, a) / (r2 * r2 * r);
  }
  return dsoft - dlong;
}

// Minimum image (tree_pm_geometry.hpp:12-25): nearbyint semantics, with the
// division skipped whenever |d| <= L lies outside the half-box tie band.
__device__ __forceinline__ double mi64(double d, double L) {
  const double ad = fabs(d), half = 0.5 * L;
  if (ad <= L && fabs(ad - half) > 4.0 * 2.220446049250313e-16 * L)
    return d > half ? d - L : (d < -half ? d + L : d);
  return d - L * rint(d / L);
}

// tree_pm_geometry.hpp:51-60
__device__ __forceinline__ bool within_cutoff(double d2, double c, double c2) {
  if (!isnormal(c2) || !isfinite(d2) || fabs(d2 - c2) <= 8.0 * 2.220446049250313e-16 * c2) return sqrt(d2) <= c;
  return d2 <= c2;
}

// Forward-mode derivative of a scalar with respect to the node offset d
// (three partials), for the Jacobian of the node expansion in the force VJP.
struct D3 {
  double v, x, y, z;
};
__device__ __forceinline__ D3 d3c(double c) { return D3{c, 0.0, 0.0, 0.0}; }
__device__ __forceinline__ D3 operator+(D3 a, D3 b) { return D3{a.v + b.v, a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ D3 operator-(D3 a, D3 b) { return D3{a.v - b.v, a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ D3 operator-(D3 a) { return D3{-a.v, -a.x, -a.y, -a.z}; }
__device__ __forceinline__ D3 operator*(D3 a, D3 b) {
  return D3{a.v * b.v, a.x * b.v + a.v * b.x, a.y * b.v + a.v * b.y, a.z * b.v + a.v * b.z};
}
__device__ __forceinline__ D3 operator*(D3 a, double c) { return D3{a.v * c, a.x * c, a.y * c, a.z * c}; }
__device__ __forceinline__ D3 operator*(double c, D3 a) { return a * c; }
__device__ __forceinline__ D3 operator+(D3 a, double c) { return D3{a.v + c, a.x, a.y, a.z}; }
__device__ __forceinline__ D3 operator+(double c, D3 a) { return a + c; }
__device__ __forceinline__ D3 operator-(D3 a, double c) { return D3{a.v - c, a.x, a.y, a.z}; }
__device__ __forceinline__ D3 operator-(double c, D3 a) { return D3{c - a.v, -a.x, -a.y, -a.z}; }
__device__ __forceinline__ D3 operator/(D3 a, D3 b) {
  const double q = a.v / b.v, ib = 1.0 / b.v;
  return D3{q, (a.x - q * b.x) * ib, (a.y - q * b.y) * ib, (a.z - q * b.z) * ib};
}
__device__ __forceinline__ D3 operator/(D3 a, double c) { return D3{a.v / c, a.x / c, a.y / c, a.z / c}; }
__device__ __forceinline__ D3 operator/(double c, D3 b) { return d3c(c) / b; }
__device__ __forceinline__ D3 d_scale(D3 a, double v, double dv) { return D3{v, a.x * dv, a.y * dv, a.z * dv}; }
__device__ __forceinline__ double f_max(double a, double c) { return fmax(a, c); }
__device__ __forceinline__ D3 f_max(D3 a, double c) { return a.v > c ? a : d3c(fmax(a.v, c)); }
__device__ __forceinline__ double f_sqrt(double a) { return sqrt(a); }
__device__ __forceinline__ D3 f_sqrt(D3 a) {
  const double v = sqrt(a.v);
  return d_scale(a, v, 0.5 / v);
}
__device__ __forceinline__ double f_exp(double a) { return exp(a); }
__device__ __forceinline__ D3 f_exp(D3 a) {
  const double v = exp(a.v);
  return d_scale(a, v, v);
}
// short_factor of a dual r: d/dr [erfc(q) + 2 q exp(-q^2)/sqrt(pi)] = -2 q^2 exp(-q^2) / (sqrt(pi) a), q = r/2a
__device__ __forceinline__ double f_short(double r, double a) { return short_factor(r, a); }
__device__ __forceinline__ D3 f_short(D3 r, double a) {
  const double q = (0.5 * r.v) / a;
  const double dv = (r.v <= 0.0 || isinf(q)) ? 0.0 : -2.0 * kInvSqrtPi * q * q * exp(-q * q) / a;
  return d_scale(r, short_factor(r.v, a), dv);
}

// monopolePlusQuadrupoleAccelPeriodicReference (tree_pm_coupling.cpp:743-827),
// on double (the walks) or on D3 (its Jacobian with respect to the offset).
template <class T>
__device__ __forceinline__ void node_accel_t(double mass, const NodeQuad64& Q, T dx, T dy, T dz,
                                             const WalkParams& P, T& cx, T& cy, T& cz) {
  const T r2 = dx * dx + dy * dy + dz * dz;
  const T safe_r2 = f_max(r2, 1.0e-30);
  const T r = f_sqrt(safe_r2);
  const double pe = P.eps;  // uniform softening: max(node eps, target eps) = eps
  const double eps2 = pe * pe;
  const T denom = f_max(r2 + eps2, 1.0e-30);
  const T soft = 1.0 / (denom * f_sqrt(denom));
  const T split = f_short(r, P.a);
  const T newton = 1.0 / (safe_r2 * r);
  const T radial = soft + (split - 1.0) * newton;
  const double pref = P.G;
  cx = pref * mass * radial * dx;
  cy = pref * mass * radial * dy;
  cz = pref * mass * radial * dz;
  if (P.quad) {
    const double tr = Q.trace;
    const double mxx = (Q.qxx + tr) / 3.0, mxy = Q.qxy / 3.0, mxz = Q.qxz / 3.0;
    const double myy = (Q.qyy + tr) / 3.0, myz = Q.qyz / 3.0, mzz = (Q.qzz + tr) / 3.0;
    const T mdx = mxx * dx + mxy * dy + mxz * dz;
    const T mdy = mxy * dx + myy * dy + myz * dz;
    const T mdz = mxz * dx + myz * dy + mzz * dz;
    const T dmd = dx * mdx + dy * mdy + dz * mdz;
    const double a = P.a, a2 = a * a;
    const T ex = f_exp(-r2 / (4.0 * a2));
    const T s1 = -0.5 * kInvSqrtPi * r2 * ex / (a * a2);
    const T s2 = kInvSqrtPi * ex * (-r / (a * a2) + 0.25 * r * r2 / (a * a2 * a2));
    const T f1 = -3.0 * r / (denom * denom * f_sqrt(denom));
    const T f2 = -3.0 / (denom * denom * f_sqrt(denom)) + 15.0 * r2 / (denom * denom * denom * f_sqrt(denom));
    const T n1 = -3.0 / (safe_r2 * safe_r2);
    const T n2 = 12.0 / (safe_r2 * safe_r2 * r);
    const T rf = f1 + s1 * newton + (split - 1.0) * n1;
    const T rs = f2 + s2 * newton + 2.0 * s1 * n1 + (split - 1.0) * n2;
    const T fo = rf / r;
    const T cr = rs / r2 - rf / (r2 * r);
    cx = cx + pref * (mdx * fo + 0.5 * tr * dx * fo + 0.5 * dx * dmd * cr);
    cy = cy + pref * (mdy * fo + 0.5 * tr * dy * fo + 0.5 * dy * dmd * cr);
    cz = cz + pref * (mdz * fo + 0.5 * tr * dz * fo + 0.5 * dz * dmd * cr);
  }
}

__device__ __forceinline__ void node_accel64(const NodeMom64& M, const NodeQuad64& Q, double dx, double dy, double dz,
                                             const WalkParams& P, double& ax, double& ay, double& az) {
  double cx, cy, cz;
  node_accel_t<double>(M.mass, Q, dx, dy, dz, P, cx, cy, cz);
  ax += cx;
  ay += cy;
  az += cz;
}

// Force VJP at an accepted node N of target t (offset d = COM_N - x_t, lam of
// t): the node's force a(d, Q) depends on x_t through d, and on the positions
// of N's particles through COM_N (= d + x_t) and the quadrupole Q.
//   g = J^T lam with J = da/dd (forward-mode D3);
//   s_t -= g (da/dx_t = -J);
//   U_N += g, V_N[p] += lam . da/dQ_p (a is linear in the seven stored Q
//   components qxx..qzz, trace: each column is the expansion with mass 0 and
//   Q = e_p).
// U_N and V_N are spread over N's particles afterwards (vjp_node_push).
__device__ __attribute__((noinline)) void jvp_node64(const NodeMom64& M, const NodeQuad64& Q, double dx, double dy,
                                                     double dz, const WalkParams& P, double lx, double ly,
                                                     double lz, double* __restrict__ acc, double& sx, double& sy,
                                                     double& sz) {
  D3 cx, cy, cz;
  node_accel_t<D3>(M.mass, Q, D3{dx, 1.0, 0.0, 0.0}, D3{dy, 0.0, 1.0, 0.0}, D3{dz, 0.0, 0.0, 1.0}, P, cx, cy, cz);
  const double gx = lx * cx.x + ly * cy.x + lz * cz.x;
  const double gy = lx * cx.y + ly * cy.y + lz * cz.y;
  const double gz = lx * cx.z + ly * cy.z + lz * cz.z;
  sx -= gx;
  sy -= gy;
  sz -= gz;
  atomicAdd(acc + 0, gx);
  atomicAdd(acc + 1, gy);
  atomicAdd(acc + 2, gz);
  if (!P.quad) return;
  for (int q = 0; q < 7; ++q) {
    NodeQuad64 e{0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    switch (q) {
      case 0: e.qxx = 1.0; break;
      case 1: e.qxy = 1.0; break;
      case 2: e.qxz = 1.0; break;
      case 3: e.qyy = 1.0; break;
      case 4: e.qyz = 1.0; break;
      case 5: e.qzz = 1.0; break;
      default: e.trace = 1.0; break;
    }
    double ex, ey, ez;
    node_accel_t<double>(0.0, e, dx, dy, dz, P, ex, ey, ez);
    atomicAdd(acc + 3 + q, lx * ex + ly * ey + lz * ez);
  }
}

// Strict-reference acceptance of an internal node (tree_pm_acceptance.hpp:54-139,
// tree_interaction_common.hpp:36-89) for uniform softening and no history.
__device__ __forceinline__ bool accept64(double h, double offset, bool inside, bool contained, double r2,
                                         const WalkParams& P) {
  const double r = sqrt(fmax(r2, 1.0e-30));
  const bool env_ok = P.quad && (2.0 * h / r) < 0.08;
  bool mac = false;
  if (!inside) {
    if (P.criterion == 0) mac = (2.0 * h / sqrt(r2 + 1.0e-30)) < P.theta;
    else mac = ((2.0 * h + offset) / sqrt(r2 + 1.0e-30)) < P.theta;
  }
  return mac && env_ok && contained && !inside && isfinite(r2);
}

// ---- adaptive acceptance pieces (FP64) -------------------------------------------
// Gaussian Hermite table (tree_pm_split_kernel.hpp:130-183): knots (H, step dH/dt)
// at t = i / 64, i = 0..4096.
constexpr int kGaussCells = 4096;
__device__ __forceinline__ double gauss_hermite(const double2* __restrict__ tab, double t) {
  const double cell = t * 64.0;
  const int i = static_cast<int>(cell);
  const double u = cell - static_cast<double>(i), u2 = u * u, u3 = u2 * u;
  const double2 k0 = tab[i], k1 = tab[i + 1];
  return (2 * u3 - 3 * u2 + 1) * k0.x + (u3 - 2 * u2 + u) * k0.y + (-2 * u3 + 3 * u2) * k1.x + (u3 - u2) * k1.y;
}
// dimensionlessCoefficient: series below t = 1/64, analytic from t = 64
__device__ __forceinline__ double gauss_coefficient(const double2* __restrict__ tab, double t) {
  if (t < 0.015625) return series_h(t);
  if (!(t < 64.0)) return long_inv_r3(sqrt(t), 0.5);
  return gauss_hermite(tab, t);
}
// Leaf-pair residual of the per-target walk with the Gaussian lookup
// (tree_pm_coupling.cpp:4216-4227), r2 > 0.
__device__ __forceinline__ double table_residual64(const double2* __restrict__ tab, double r2, const WalkParams& P) {
  const double t = r2 * P.inv2a2;
  double lr;
  if (t < 64.0) {
    lr = gauss_coefficient(tab, t) * P.inv8a3;
  } else {
    const double tt = 0.25 * (r2 / P.a) / P.a;  // longRangeInvR3 beyond the table
    lr = (!(tt >= 0.0) || tt >= 64.0) ? long_inv_r3(sqrt(r2), P.a)
                                      : ((0.125 * gauss_coefficient(tab, tt) / P.a) / P.a) / P.a;
  }
  return softened_inv_r3(r2, P.eps) - lr;
}

// treePmResidualRadialCoefficients (tree_pm_split_kernel.hpp:245-282).
__device__ __forceinline__ void residual_radial64(double x, double eps, double a, double& value, double& first,
                                                  double& second) {
  const double d = x + eps * eps;
  const double soft = 1.0 / (d * sqrt(d));
  const double t = (0.25 * x / a) / a;
  constexpr double c = 2.25675833419102514779231780624309034;
  double h, dh, ddh;
  if (t < 0.015625) {
    constexpr double k[8] = {1.0 / 3.0, -1.0 / 5.0, 1.0 / 14.0, -1.0 / 54.0,
                             1.0 / 264.0, -1.0 / 1560.0, 1.0 / 10800.0, -1.0 / 85680.0};
    h = k[7]; dh = 0.0; ddh = 0.0;
#pragma unroll
    for (int i = 7; i > 0; --i) {
      ddh = ddh * t + 2.0 * dh;
      dh = dh * t + h;
      h = h * t + k[i - 1];
    }
    h *= c; dh *= c; ddh *= c;
  } else {
    const double q = sqrt(t);
    const double e = exp(-t);
    h = (erf(q) - 0.5 * c * q * e) / (t * q);
    dh = (0.5 * c * e - 1.5 * h) / t;
    ddh = (-0.5 * c * e - 2.5 * dh) / t;
  }
  const double scale = ((0.125 / a) / a) / a;
  const double dt_dx = (0.25 / a) / a;
  value = soft - scale * h;
  first = -3.0 * soft / d - 2.0 * scale * dt_dx * dh;
  second = 15.0 * soft / (d * d) - 4.0 * scale * dt_dx * dt_dx * ddh;
}

// monopolePlusQuadrupoleAccelPeriodic (tree_pm_coupling.cpp:829-894); non-finite
// coefficients use the reference expansion.
__device__ __forceinline__ void node_accel_radial64(const NodeMom64& M, const NodeQuad64& Q, double dx, double dy,
                                                    double dz, const WalkParams& P, double& ax, double& ay,
                                                    double& az) {
  const double r2 = dx * dx + dy * dy + dz * dz;
  const double safe_r2 = fmax(r2, 1.0e-30);
  double v, fo, cr;
  residual_radial64(safe_r2, P.eps, P.a, v, fo, cr);
  if (!isfinite(v) || !isfinite(fo) || !isfinite(cr)) {
    node_accel64(M, Q, dx, dy, dz, P, ax, ay, az);
    return;
  }
  const double pref = P.G;
  double cx = pref * M.mass * v * dx;
  double cy = pref * M.mass * v * dy;
  double cz = pref * M.mass * v * dz;
  if (P.quad) {
    const double tr = Q.trace;
    const double mxx = (Q.qxx + tr) / 3.0, mxy = Q.qxy / 3.0, mxz = Q.qxz / 3.0;
    const double myy = (Q.qyy + tr) / 3.0, myz = Q.qyz / 3.0, mzz = (Q.qzz + tr) / 3.0;
    const double mdx = mxx * dx + mxy * dy + mxz * dz;
    const double mdy = mxy * dx + myy * dy + myz * dz;
    const double mdz = mxz * dx + myz * dy + mzz * dz;
    const double dmd = dx * mdx + dy * mdy + dz * mdz;
    cx += pref * (mdx * fo + 0.5 * tr * dx * fo + 0.5 * dx * dmd * cr);
    cy += pref * (mdy * fo + 0.5 * tr * dy * fo + 0.5 * dy * dmd * cr);
    cz += pref * (mdz * fo + 0.5 * tr * dz * fo + 0.5 * dz * dmd * cr);
  }
  ax += cx;
  ay += cy;
  az += cz;
}

// Out-of-line forms for kernels whose register budget the inlined expansions
// would exceed (accepted nodes are rare next to leaf pairs).
__device__ __attribute__((noinline)) void node_accel64_call(const NodeMom64& M, const NodeQuad64& Q, double dx,
                                                            double dy, double dz, const WalkParams& P, double& ax,
                                                            double& ay, double& az) {
  if (P.radial) node_accel_radial64(M, Q, dx, dy, dz, P, ax, ay, az);
  else node_accel64(M, Q, dx, dy, dz, P, ax, ay, az);
}

// residualAccuracyProxy (tree_pm_acceptance.hpp:14-51) for uniform softening.
__device__ __forceinline__ double residual_proxy64(double h, double offset, double mass, double r2,
                                                   const WalkParams& P) {
  if (!(r2 > 0.0) || !isfinite(r2)) return INFINITY;
  const double a = P.a;
  const double r = sqrt(r2);
  const double d = r2 + P.eps * P.eps;
  const double inv_d5 = 1.0 / (d * d * sqrt(d));
  const double inv_r3 = 1.0 / (r2 * r);
  const double inv_r4 = 1.0 / (r2 * r2);
  const double lf = long_factor(r, a);
  const double q = r / (2.0 * a);
  const double e = exp(-q * q);
  const double a3 = a * a * a;
  const double s1 = -0.5 * kInvSqrtPi * r2 * e / a3;
  const double s2 = kInvSqrtPi * e * (-r / a3 + 0.25 * r * r2 / (a3 * a * a));
  const double first = -3.0 * r * inv_d5 + s1 * inv_r3 - 3.0 * (-lf) * inv_r4;
  const double second = -3.0 * inv_d5 + 15.0 * r2 * inv_d5 / d + s2 * inv_r3 - 6.0 * s1 * inv_r4 +
                        12.0 * (-lf) * inv_r4 / r;
  const double width = 2.0 * h;
  const double rho = 1.7320508075688772935274463415058723 * h + offset;
  const double proxy = P.G * mass * fmax(width * width * inv_r4,
                                         0.5 * rho * rho * (3.0 * fabs(first) + fabs(r * second - first)));
  return isfinite(proxy) && proxy >= 0.0 ? proxy : INFINITY;
}

// acceptTreePmNode (tree_pm_acceptance.hpp:54-139) under the adaptive policy for
// an internal node that neither holds the target nor leaves the cutoff
// container (those are opened first, tree_pm_coupling.cpp:4094-4104).
__device__ __forceinline__ bool accept_adaptive64(double h, double offset, double mass, double r2, bool history,
                                                  double prev, const WalkParams& P) {
  const double r = sqrt(fmax(r2, 1.0e-30));
  const bool env_ok = (2.0 * h / r) < P.amax;
  bool mac;
  if (history && isfinite(prev) && prev > P.accel_floor) {
    const double allowance = P.alpha * prev;
    const double width = 2.0 * h;
    const double inv_r4 = 1.0 / (r2 * r2);
    const double lower = P.G * mass * (width * width * inv_r4);
    if (isfinite(allowance) && isfinite(lower) && lower > allowance) {
      mac = false;
    } else if (P.estimator == 1) {  // relative monopole
      mac = isfinite(allowance) && isfinite(lower);
    } else {
      const double est = residual_proxy64(h, offset, mass, r2, P);
      mac = isfinite(est) && isfinite(allowance) && est <= allowance;
    }
  } else {
    mac = ((2.0 * h + offset) / sqrt(r2 + 1.0e-30)) < P.theta;
  }
  return mac && env_ok && isfinite(r2);
}

// ---- PM interpolation (pm_solver.cpp:925-951, :5900-5957) --------------------
__device__ __forceinline__ double wrap_position(double x, double L) {
  const double w = fmod(x, L);
  return w < 0.0 ? w + L : w;
}
__device__ __forceinline__ int wrap_index(long i, int n) {
  long w = i % n;
  if (w < 0) w += n;
  return static_cast<int>(w);
}

// Stencil of one axis with a compile-time point count (CIC 2, TSC 3) so the
// gather below is fully unrolled and stays in registers.
template <int SCHEME>
__device__ __forceinline__ void stencil64(double g, int n, int (&idx)[SCHEME + 2], double (&w)[SCHEME + 2]) {
  if constexpr (SCHEME == 0) {
    const double base = floor(g);
    const long i0 = static_cast<long>(base);
    const double t = g - base;
    idx[0] = wrap_index(i0, n);
    idx[1] = wrap_index(i0 + 1, n);
    w[0] = 1.0 - t;
    w[1] = t;
  } else {
    const double c = floor(g + 0.5);
    const long ic = static_cast<long>(c);
    const double d = g - c;
    idx[0] = wrap_index(ic - 1, n);
    idx[1] = wrap_index(ic, n);
    idx[2] = wrap_index(ic + 1, n);
    w[0] = 0.5 * (0.5 - d) * (0.5 - d);
    w[1] = 0.75 - d * d;
    w[2] = 0.5 * (0.5 + d) * (0.5 + d);
  }
}

template <int SCHEME>
__device__ void interp64(const WalkParams& P, const double* __restrict__ fx, const double* __restrict__ fy,
                         const double* __restrict__ fz, double x, double y, double z, double& gx, double& gy,
                         double& gz) {
  constexpr int K = SCHEME + 2;
  int ix[K], iy[K], iz[K];
  double wx[K], wy[K], wz[K];
  stencil64<SCHEME>(wrap_position(x, P.L[0]) * (static_cast<double>(P.mesh[0]) / P.L[0]), P.mesh[0], ix, wx);
  stencil64<SCHEME>(wrap_position(y, P.L[1]) * (static_cast<double>(P.mesh[1]) / P.L[1]), P.mesh[1], iy, wy);
  stencil64<SCHEME>(wrap_position(z, P.L[2]) * (static_cast<double>(P.mesh[2]) / P.L[2]), P.mesh[2], iz, wz);
  gx = gy = gz = 0.0;
#pragma unroll
  for (int a = 0; a < K; ++a)
#pragma unroll
    for (int b = 0; b < K; ++b) {
      const std::size_t row = (static_cast<std::size_t>(ix[a]) * P.mesh[1] + iy[b]) * P.mesh_row;
#pragma unroll
      for (int c = 0; c < K; ++c) {
        const double w = wx[a] * wy[b] * wz[c];
        const std::size_t i = row + iz[c];
        gx += w * fx[i];
        gy += w * fy[i];
        gz += w * fz[i];
      }
    }
}

// Stencil weights and their derivatives with respect to the mesh coordinate g
// (multiply by n/L for a length derivative).
template <int SCHEME>
__device__ __forceinline__ void stencil64_grad(double g, int n, int (&idx)[SCHEME + 2], double (&w)[SCHEME + 2],
                                               double (&dw)[SCHEME + 2]) {
  stencil64<SCHEME>(g, n, idx, w);
  if constexpr (SCHEME == 0) {
    dw[0] = -1.0;
    dw[1] = 1.0;
  } else {
    const double d = g - floor(g + 0.5);
    dw[0] = -(0.5 - d);
    dw[1] = -2.0 * d;
    dw[2] = 0.5 + d;
  }
}

// Transpose of the PM force's Jacobian for one source k (FP64):
//   s_k = grad_{x_k} sum_c W(x_k, c) [lam_k . F(c) + m_k nu(c)]
// with F the force meshes (interpolation's own dependence on x_k) and nu the
// adjoint potential sum_a S_a^T mu_a of the deposited lam (deposit's
// dependence on x_k).
template <int SCHEME>
__device__ void vjp_gather64(const WalkParams& P, const double* __restrict__ fx, const double* __restrict__ fy,
                             const double* __restrict__ fz, const double* __restrict__ nu, double lx, double ly,
                             double lz, double mk, double x, double y, double z, double& sx, double& sy,
                             double& sz) {
  constexpr int K = SCHEME + 2;
  int ix[K], iy[K], iz[K];
  double wx[K], wy[K], wz[K], dx[K], dy[K], dz[K];
  const double hx = static_cast<double>(P.mesh[0]) / P.L[0];
  const double hy = static_cast<double>(P.mesh[1]) / P.L[1];
  const double hz = static_cast<double>(P.mesh[2]) / P.L[2];
  stencil64_grad<SCHEME>(wrap_position(x, P.L[0]) * hx, P.mesh[0], ix, wx, dx);
  stencil64_grad<SCHEME>(wrap_position(y, P.L[1]) * hy, P.mesh[1], iy, wy, dy);
  stencil64_grad<SCHEME>(wrap_position(z, P.L[2]) * hz, P.mesh[2], iz, wz, dz);
  sx = sy = sz = 0.0;
#pragma unroll
  for (int a = 0; a < K; ++a)
#pragma unroll
    for (int b = 0; b < K; ++b) {
      const std::size_t row = (static_cast<std::size_t>(ix[a]) * P.mesh[1] + iy[b]) * P.mesh_row;
#pragma unroll
      for (int c = 0; c < K; ++c) {
        const std::size_t i = row + iz[c];
        const double u = lx * fx[i] + ly * fy[i] + lz * fz[i] + mk * nu[i];
        sx += dx[a] * wy[b] * wz[c] * u;
        sy += wx[a] * dy[b] * wz[c] * u;
        sz += wx[a] * wy[b] * dz[c] * u;
      }
    }
  sx *= hx;
  sy *= hy;
  sz *= hz;
}

// Stencil from a 32-bit fixed-point coordinate q (x = q L / 2^32) on a mesh of
// n cells: q n / 2^32 = cell + t exactly in 64-bit integers (for n = 2^lg the
// cell is the top lg bits and t the remaining bits).
__device__ __forceinline__ int wrap_once(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

template <int SCHEME>
__device__ __forceinline__ void stencil32(uint32_t q, int n, int lg, int (&idx)[SCHEME + 2], float (&w)[SCHEME + 2]) {
  (void)lg;
  const uint64_t p = static_cast<uint64_t>(q) * static_cast<uint32_t>(n);
  const int cell = static_cast<int>(p >> 32);
  const float t = static_cast<float>(static_cast<uint32_t>(p)) * 0x1p-32f;
  if constexpr (SCHEME == 0) {
    idx[0] = cell;
    idx[1] = wrap_once(cell + 1, n);
    w[0] = 1.0f - t;
    w[1] = t;
  } else {
    const int c = t >= 0.5f ? cell + 1 : cell;
    const float d = t >= 0.5f ? t - 1.0f : t;
    idx[0] = wrap_once(c - 1, n);
    idx[1] = wrap_once(c, n);
    idx[2] = wrap_once(c + 1, n);
    w[0] = 0.5f * (0.5f - d) * (0.5f - d);
    w[1] = 0.75f - d * d;
    w[2] = 0.5f * (0.5f + d) * (0.5f + d);
  }
}

template <int SCHEME>
__device__ void interp32(const WalkParams& P, const float* __restrict__ fx, const float* __restrict__ fy,
                         const float* __restrict__ fz, uint32_t qx, uint32_t qy, uint32_t qz, float& gx, float& gy,
                         float& gz) {
  constexpr int K = SCHEME + 2;
  int ix[K], iy[K], iz[K];
  float wx[K], wy[K], wz[K];
  stencil32<SCHEME>(qx, P.mesh[0], P.mesh_log2[0], ix, wx);
  stencil32<SCHEME>(qy, P.mesh[1], P.mesh_log2[1], iy, wy);
  stencil32<SCHEME>(qz, P.mesh[2], P.mesh_log2[2], iz, wz);
  gx = gy = gz = 0.0f;
#pragma unroll
  for (int a = 0; a < K; ++a)
#pragma unroll
    for (int b = 0; b < K; ++b) {
      const std::size_t row = (static_cast<std::size_t>(ix[a]) * P.mesh[1] + iy[b]) * P.mesh_row;
      const float wab = wx[a] * wy[b];
#pragma unroll
      for (int c = 0; c < K; ++c) {
        const float w = wab * wz[c];
        const std::size_t i = row + iz[c];
        gx = fmaf(w, fx[i], gx);
        gy = fmaf(w, fy[i], gy);
        gz = fmaf(w, fz[i], gz);
      }
    }
}

// XCD-aware block order: the dispatcher sends block b to XCD b % 8; each XCD
// takes runs of kXcdChunk consecutive target chunks, so neighbouring targets
// share an L2 and the dense regions spread over the XCDs (one contiguous
// eighth per XCD left the XCDs unevenly loaded: the 256^3 mixed walk took 20.7
// ms so, 18.6 ms in runs of 4, 18.8 of 16 and 19.1 of 64).
constexpr uint32_t kXcdChunk = 4;
__device__ __forceinline__ uint32_t xcd_logical_block() {
  constexpr uint32_t C = kXcdChunk;
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t full = nb / (8 * C) * (8 * C);
  if (b >= full) return b;
  const uint32_t x = b % 8, j = b / 8;
  return ((j / C) * 8 + x) * C + j % C;
}

__device__ __forceinline__ void flush_counters(unsigned long long* counters, const uint32_t* c) {
  for (int i = 0; i < kWalkCounters; ++i) {
    const unsigned long long v = wave_sum(static_cast<unsigned long long>(c[i]));
    if (lane_id() == 0 && v) atomicAdd(&counters[i], v);
  }
}

// ---- mixed-precision pair pieces -----------------------------------------------
__device__ __forceinline__ float fx_delta(uint32_t a, uint32_t b, float scale) {
  return static_cast<float>(static_cast<int32_t>(a - b)) * scale;
}

__device__ __forceinline__ void node_accel32(const NodeMom32& M, const NodeQuad32& Q, float dx, float dy, float dz,
                                          const WalkParams& P, float& ax, float& ay, float& az) {
  const float r2 = dx * dx + dy * dy + dz * dz;
  const float safe_r2 = fmaxf(r2, 1.0e-30f);
  const float r = sqrtf(safe_r2);
  const float eps = static_cast<float>(P.eps);
  const float denom = fmaxf(r2 + eps * eps, 1.0e-30f);
  const float rs_d = rsqrtf(denom);
  const float soft = rs_d * rs_d * rs_d;
  const float a = static_cast<float>(P.a);
  const float q = 0.5f * r / a;
  const float split = erfcf(q) + 2.0f * static_cast<float>(kInvSqrtPi) * q * expf(-q * q);
  const float newton = 1.0f / (safe_r2 * r);
  const float radial = soft + (split - 1.0f) * newton;
  const float pref = static_cast<float>(P.G);
  float cx = pref * M.mass * radial * dx;
  float cy = pref * M.mass * radial * dy;
  float cz = pref * M.mass * radial * dz;
  if (P.quad) {
    const float tr = Q.trace;
    const float third = 1.0f / 3.0f;
    const float mxx = (Q.qxx + tr) * third, mxy = Q.qxy * third, mxz = Q.qxz * third;
    const float myy = (Q.qyy + tr) * third, myz = Q.qyz * third, mzz = (Q.qzz + tr) * third;
    const float mdx = mxx * dx + mxy * dy + mxz * dz;
    const float mdy = mxy * dx + myy * dy + myz * dz;
    const float mdz = mxz * dx + myz * dy + mzz * dz;
    const float dmd = dx * mdx + dy * mdy + dz * mdz;
    const float a2 = a * a;
    const float ex = expf(-r2 / (4.0f * a2));
    const float isp = static_cast<float>(kInvSqrtPi);
    const float s1 = -0.5f * isp * r2 * ex / (a * a2);
    const float s2 = isp * ex * (-r / (a * a2) + 0.25f * r * r2 / (a * a2 * a2));
    const float d52 = soft / denom;  // denom^-5/2
    const float f1 = -3.0f * r * d52;
    const float f2 = -3.0f * d52 + 15.0f * r2 * d52 / denom;
    const float n1 = -3.0f / (safe_r2 * safe_r2);
    const float n2 = 12.0f / (safe_r2 * safe_r2 * r);
    const float rf = f1 + s1 * newton + (split - 1.0f) * n1;
    const float rsec = f2 + s2 * newton + 2.0f * s1 * n1 + (split - 1.0f) * n2;
    const float fo = rf / r;
    const float cr = rsec / r2 - rf / (r2 * r);
    cx += pref * (mdx * fo + 0.5f * tr * dx * fo + 0.5f * dx * dmd * cr);
    cy += pref * (mdy * fo + 0.5f * tr * dy * fo + 0.5f * dy * dmd * cr);
    cz += pref * (mdz * fo + 0.5f * tr * dz * fo + 0.5f * dz * dmd * cr);
  }
  ax = cx;
  ay = cy;
  az = cz;
}

// Node-test units of the mixed walk: per-axis scale of fixed-point
// differences (1 for a cubic box, whose tests run in fixed-point units),
// separation unit -> length and back, the containment radius^2 and theta^2.
struct MixFrame {
  float s0, s1, s2, to_len, inv_len, contain2, theta2;
};

// Strict acceptance of internal node n (tree_pm_acceptance.hpp:54-66: the
// node's cell inside r_cut, the opening criterion and 2h/r < 0.08 with
// quadrupoles) for the target at fixed point (px, py, pz), with the COM
// separation in lengths left in mf* for the multipole evaluation.
__device__ __forceinline__ bool strict_accept32(const WalkParams& P, const MixFrame& F, const NodeGeo32& g,
                                                const NodeMom32& M, const NodeQuad32* __restrict__ node_quad,
                                                uint32_t n, uint32_t px, uint32_t py, uint32_t pz, float& mfx,
                                                float& mfy, float& mfz) {
  const float h = g.half * F.inv_len;
  const float ax_ = fabsf(fx_delta(g.cx, px, F.s0)), ay_ = fabsf(fx_delta(g.cy, py, F.s1)),
              az_ = fabsf(fx_delta(g.cz, pz, F.s2));
  const bool inside = ax_ <= h && ay_ <= h && az_ <= h;
  const float mx = ax_ + h, my = ay_ + h, mz = az_ + h;
  const bool contained = fmaf(mx, mx, fmaf(my, my, mz * mz)) <= F.contain2;
  mfx = fx_delta(M.comx, px, F.s0) * F.to_len;
  mfy = fx_delta(M.comy, py, F.s1) * F.to_len;
  mfz = fx_delta(M.comz, pz, F.s2) * F.to_len;
  const float r2 = mfx * mfx + mfy * mfy + mfz * mfz;
  const float w2 = 2.0f * g.half;
  // 2h/r < 0.08 and (2h [+ |c - COM|]) / r < theta, squared (no sqrt/div)
  const bool env_ok = P.quad && w2 * w2 < 0.0064f * fmaxf(r2, 1.0e-30f);
  const float lead = P.criterion == 0 ? w2 : w2 + node_quad[n].offset;
  const bool mac = !inside && lead * lead < F.theta2 * (r2 + 1.0e-30f);
  return mac && env_ok && contained;
}

__device__ __forceinline__ void kahan_add(float& s, float& c, float v) {
  const float y = v - c;
  const float t = s + y;
  c = (t - s) - y;
  s = t;
}

// ---- the walk -------------------------------------------------------------------
// Per node, every lane whose next node it is applies the reference's cutoff
// prune; whether the node is a leaf is wave-uniform, so leaf and internal-node
// work are scalar branches. While the wave streams a leaf's sources (wave-
// uniform scalar loads of packed records) each lane only forms the separation,
// applies the cutoff and self test and appends the source index to its own LDS
// queue; the residual kernel then runs over the queues, so lanes spend it only
// on pairs inside r_cut. A queue is drained before it can overflow and before
// any lane adds an accepted multipole, so each lane's contributions are summed
// in the order of the reference's sequential walk. The next node is i + 1
// whenever any lane is waiting on it (one ballot), otherwise the DPP wave
// minimum of the lanes' next nodes.
constexpr int kWalkWaves = kWalkThreads / kWave;
constexpr int kQueue = 32;
constexpr int kChunk = 16;

struct WalkData {
  const NodeLink* link;
  const NodeGeo64* geo64;
  const NodeMom64* mom64;
  const NodeQuad64* quad64;
  const uint32_t* child_index;  // group walks
  const NodeGeo32* geo32;
  const NodeMom32* mom32;
  const NodeQuad32* quad32;
  const NodeBox32* box32;
  const uint32_t* order;
  const double4* src64;
  const uint4* src32;
  const float4* htab;
  int uniform_mass;
  const uint32_t *tpos, *tslot;
  const double *f64x, *f64y, *f64z;
  const float *f32x, *f32y, *f32z;
  // force VJP: tree-ordered lam (x, y, z, unused) and the adjoint potential
  const double4* lam64;
  const double* nu64;
  // adaptive policy: Gaussian Hermite knots and |a_prev| per output slot (nullable)
  const double2* gtab;
  const double* prev;
  // group walk: the same Gaussian cells as monomial coefficients (a0..a3)
  const double4* gcoef;
  // FP64 box walk: degree-5 cells of H (a0..a5 as three double2 per cell)
  const double2* h64tab;
  // mixed timed walk: residual cells indexed by the float bits of r^2 + eps^2
  const float4* ltab;
  // force VJP with accepted nodes: per preorder node U (3) and V (7)
  // accumulators, and the (target tree position << 32 | node) list
  double* vjp_node_acc;
  unsigned long long* vjp_accepted;
  unsigned int* vjp_accepted_count;
  unsigned int vjp_accepted_cap;
  // after a capture-safe build the node count is on the device (P.node_count
  // is then the capacity); the mixed walks bound their traversal with it
  const uint32_t* node_count_dev;
  // breadth-first records of the box-classified walks
  const WalkNode* wnode;
};

// splitmix64 finaliser of the pair (target row, source row): the pair-set
// checksum adds it over every direct pair inside r_cut.
__device__ __forceinline__ unsigned long long pair_mix(uint32_t target_row, uint32_t source_row) {
  unsigned long long z = (static_cast<unsigned long long>(target_row) << 32) | source_row;
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ uint32_t next_node(uint32_t n, uint32_t nxt) {
  return __ballot(nxt == n + 1) ? n + 1 : wave_min_u32(nxt);
}

// ---- FP64 walk (reference arithmetic) ---------------------------------------------
// JVP: instead of the acceleration, each target k accumulates the transpose of
// the acceleration Jacobian applied to lam (see vjp_gather64 for the PM part).
// For the residual pairs, with r = x_j - x_k, t = r^2 and the pair force
// G m_j F(t) r, the contribution is G (F w + 2 F'(t) (r . w) r) with
// w = m_k lam_j - m_j lam_k; the sum runs over the same interaction lists.
// ADAPT: the adaptive acceptance policy with the target's acceleration history,
// the cutoff node policy, optional Gaussian-table leaf pairs and the optional
// radial-coefficient node expansion (tree_pm_coupling.cpp:4026-4272 with
// TreePmAcceptancePolicy::kAdaptiveRelative).
template <int SCHEME, bool JVP, bool ADAPT = false>
__global__ __launch_bounds__(kWalkThreads) void walk64_kernel(WalkParams P, WalkData D, WalkOutputs out,
                                                               unsigned long long* __restrict__ counters) {
  __shared__ uint32_t queue[kWalkWaves][kQueue][kWave];
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const uint32_t k = xcd_logical_block() * kWalkThreads + threadIdx.x;
  const bool valid = k < P.n_targets;
  const uint32_t tp = valid ? (P.identity_targets ? k : D.tpos[k]) : 0u;
  const uint32_t slot = valid ? (P.identity_targets ? D.order[k] : D.tslot[k]) : 0u;
  uint32_t cnt[kWalkCounters] = {0, 0, 0, 0, 0, 0, 0, 0};
  uint32_t qlen = 0, queued = 0;
  uint32_t nxt = valid ? 0u : P.node_count;
  double nearest = INFINITY;  // r^2 of the nearest distinct direct-summed source inside r_cut
  const uint32_t target_row = valid ? D.order[tp] : 0u;
  unsigned long long pair_sum = 0;  // pair-set checksum (wrapping)
  double px = 0.0, py = 0.0, pz = 0.0;
  double gx = 0.0, gy = 0.0, gz = 0.0;
  double4 lk_ = make_double4(0.0, 0.0, 0.0, 0.0);  // JVP: lam of the target
  double mk = 0.0;                                  // JVP: mass of the target
  if (valid) {
    const double4 t = D.src64[tp];
    px = t.x;
    py = t.y;
    pz = t.z;
    if constexpr (JVP) {
      lk_ = D.lam64[tp];
      mk = D.uniform_mass ? P.uniform_mass : t.w;
      if (P.pm_enabled)
        vjp_gather64<SCHEME>(P, D.f64x, D.f64y, D.f64z, D.nu64, lk_.x, lk_.y, lk_.z, mk, px, py, pz, gx, gy, gz);
    } else {
      if (P.pm_enabled) interp64<SCHEME>(P, D.f64x, D.f64y, D.f64z, px, py, pz, gx, gy, gz);
    }
  }
  double ax = 0.0, ay = 0.0, az = 0.0;
  const double L0 = P.L[0], L1 = P.L[1], L2 = P.L[2];
  bool history = false;
  double prev = 0.0;
  if constexpr (ADAPT) {
    if (valid && D.prev != nullptr) {
      prev = D.prev[slot];
      history = isfinite(prev);
      if (!history) prev = 0.0;
    }
  }

  auto drain = [&]() {
    const uint32_t m = wave_max_u32(qlen);
    for (uint32_t q = 0; q < m; ++q) {
      if (q < qlen) {
        const uint32_t j = queue[w][q][lane];
        const double4 sj = D.src64[j];
        const double qx = mi64(sj.x - px, L0), qy = mi64(sj.y - py, L1), qz = mi64(sj.z - pz, L2);
        const double r2 = qx * qx + qy * qy + qz * qz;
        const double mj = D.uniform_mass ? P.uniform_mass : sj.w;
        double f;
        if constexpr (ADAPT) {
          f = (P.lookup ? table_residual64(D.gtab, r2, P) : residual_inv_r3(r2, P.eps, P.a)) * P.G;
        } else {
          f = residual_inv_r3(r2, P.eps, P.a) * P.G;
        }
        if constexpr (JVP) {
          const double4 lj = D.lam64[j];
          const double wx = mk * lj.x - mj * lk_.x, wy = mk * lj.y - mj * lk_.y, wz = mk * lj.z - mj * lk_.z;
          const double c = 2.0 * residual_inv_r3_dt(r2, P.eps, P.a) * P.G * (qx * wx + qy * wy + qz * wz);
          ax += f * wx + c * qx;
          ay += f * wy + c * qy;
          az += f * wz + c * qz;
        } else {
          ax += f * mj * qx;
          ay += f * mj * qy;
          az += f * mj * qz;
        }
      }
    }
    queued += qlen;
    qlen = 0;
  };

  uint32_t n = wave_min_u32(nxt);
  while (n < P.node_count) {
    if (lane == 0) ++cnt[5];
    const NodeLink lk = D.link[n];
    const NodeGeo64 g = D.geo64[n];
    const bool act = nxt == n;
    if (!__ballot(act)) {  // the chosen node must be some lane's next node
      if (lane == 0) atomicOr(&counters[kFaultSlot], 1ull);
      break;
    }
    cnt[0] += act;
    const double h = g.half;
    const double ndx = mi64(g.cx - px, L0), ndy = mi64(g.cy - py, L1), ndz = mi64(g.cz - pz, L2);
    const double ax_ = fabs(ndx), ay_ = fabs(ndy), az_ = fabs(ndz);
    const double ex = fmax(0.0, ax_ - h), ey = fmax(0.0, ay_ - h), ez = fmax(0.0, az_ - h);
    const bool keep = act && within_cutoff(ex * ex + ey * ey + ez * ez, P.rcut, P.rcut2);
    if (act && !keep) {
      ++cnt[1];
      nxt = n + lk.skip;
    }
    if (lk.child_count == 0) {
      if (keep) {
        ++cnt[4];
        nxt = n + 1;
      }
      if (__ballot(keep)) {
        const uint32_t e0 = lk.begin + lk.count;
        for (uint32_t c0 = lk.begin; c0 < e0; c0 += kChunk) {
          const uint32_t c1 = c0 + kChunk < e0 ? c0 + kChunk : e0;
          if (lane == 0) cnt[6] += c1 - c0;
          for (uint32_t j = c0; j < c1; ++j) {
            const double4 sj = D.src64[j];
            const double qx = mi64(sj.x - px, L0), qy = mi64(sj.y - py, L1), qz = mi64(sj.z - pz, L2);
            const double r2 = qx * qx + qy * qy + qz * qz;
            if (keep && j != tp && r2 <= P.rcut2) {
              nearest = fmin(nearest, r2);
              pair_sum += pair_mix(target_row, D.order[j]);
              // a coincident pair has a zero force but, in the JVP, the
              // Jacobian F(0) I
              if (!JVP && qx == 0.0 && qy == 0.0 && qz == 0.0) {
                ++cnt[2];  // counted coincident pair, zero vector
              } else {
                queue[w][qlen][lane] = j;
                ++qlen;
              }
            }
          }
          if (wave_max_u32(qlen) > static_cast<uint32_t>(kQueue - kChunk)) drain();
        }
      }
    } else if (__ballot(keep)) {
      bool take_mp = false;
      double mdx = 0.0, mdy = 0.0, mdz = 0.0;
      if (keep) {
        const bool inside = ax_ <= h && ay_ <= h && az_ <= h;
        const double mx = ax_ + h, my = ay_ + h, mz = az_ + h;
        if constexpr (ADAPT) {
          const bool contained = P.com_cut || within_cutoff(mx * mx + my * my + mz * mz, P.rcut, P.rcut2);
          bool cut = false;
          if (!inside && contained) {
            const NodeMom64 M = D.mom64[n];
            mdx = mi64(M.comx - px, L0);
            mdy = mi64(M.comy - py, L1);
            mdz = mi64(M.comz - pz, L2);
            const double r2 = mdx * mdx + mdy * mdy + mdz * mdz;
            take_mp = accept_adaptive64(h, D.quad64[n].offset, M.mass, r2, history, prev, P);
            // kComDistance: an accepted node whose COM lies beyond r_cut is pruned
            if (take_mp && P.com_cut && r2 > P.rcut2) {
              take_mp = false;
              cut = true;
              ++cnt[1];
            }
          }
          nxt = (take_mp || cut) ? n + lk.skip : n + 1;
        } else {
          const bool contained = within_cutoff(mx * mx + my * my + mz * mz, P.rcut, P.rcut2);
          const NodeMom64 M = D.mom64[n];
          mdx = mi64(M.comx - px, L0);
          mdy = mi64(M.comy - py, L1);
          mdz = mi64(M.comz - pz, L2);
          const double r2 = mdx * mdx + mdy * mdy + mdz * mdz;
          take_mp = accept64(h, D.quad64[n].offset, inside, contained, r2, P);
          nxt = take_mp ? n + lk.skip : n + 1;
        }
      }
      if (__ballot(take_mp)) {
        drain();
        if (take_mp) {
          ++cnt[3];
          if (ADAPT && P.radial) node_accel_radial64(D.mom64[n], D.quad64[n], mdx, mdy, mdz, P, ax, ay, az);
          else node_accel64(D.mom64[n], D.quad64[n], mdx, mdy, mdz, P, ax, ay, az);
        }
      }
    }
    n = next_node(n, nxt);
  }
  drain();
  cnt[2] += queued;
  flush_counters(counters, cnt);
  {
    const unsigned long long v = wave_sum(pair_sum);
    if (lane == 0 && v) atomicAdd(&counters[kPairChecksumSlot], v);
  }
  if (!valid) return;
  static_cast<double*>(out.ax)[slot] = gx + ax;
  static_cast<double*>(out.ay)[slot] = gy + ay;
  static_cast<double*>(out.az)[slot] = gz + az;
  if (out.pm_x) {
    static_cast<double*>(out.pm_x)[slot] = gx;
    static_cast<double*>(out.pm_y)[slot] = gy;
    static_cast<double*>(out.pm_z)[slot] = gz;
  }
  const uint32_t row = D.order[tp];
  if (out.sr_x) {
    static_cast<double*>(out.sr_x)[row] = ax;
    static_cast<double*>(out.sr_y)[row] = ay;
    static_cast<double*>(out.sr_z)[row] = az;
  }
  if (out.near2) static_cast<double*>(out.near2)[row] = nearest;
}

// ---- group walk (FP64) -----------------------------------------------------------
// One wave per residual block of visit-ordered targets (tree_pm_coupling.cpp:
// 4451-4546). The wave splits its block into target groups (the targets of one
// leaf, or up to group_size consecutive targets whose box stays within
// max_extent per axis), then per group:
//   1. checks every target's history and bounded metric; a failing group is
//      appended to the per-target fallback list (tree_pm_coupling.cpp:4341-4370);
//   2. walks the tree once for the group box (buildTreePmGroupInteractionList,
//      tree_pm_group_walk.hpp:78-163): eight opened nodes are popped from an
//      LDS stack and the lanes decide their children, so every lane's node is
//      one the walk visits. (Deciding 64 consecutive preorder nodes and
//      following the visited chain through them left most of each window
//      unused and was half of the kernel's time.) Listed leaves and accepted
//      nodes are appended to LDS lists;
//   3. whenever a list fills (and at the end) the listed leaves' sources are
//      taken 64 at a time; those beyond r_cut of the group box (beyond it of
//      every target, so their pairs are zero) are dropped, the rest compacted
//      into an LDS window, and every full window of 64 is evaluated by all
//      targets: a group of T targets gives each target S lanes (the largest
//      power of two with S T <= 64), each taking every S-th source and every
//      S-th accepted node (accumulateTreePmGroupCulledLeaves, :290-341); the
//      lanes' sums are added at the end. The per-target leaf cull is evaluated
//      only for its counters, when they are read.
// Four waves share a block for the FP64 pair table's cells up to r_cut: 12 KB
// of LDS instead of gathers from a 128 KB table in memory. What bounds it is
// waiting, most of it for the walk's dependent loads: of 2 (FP64) or 3 (mixed)
// possible waves per SIMD 1.4 are resident on average and wait in 59 % of their
// cycles, and the SIMDs issue vector instructions in a third. Kernel time,
// 128^3 bodies and a 256^3 mesh in FP64: 23.1 ms, with the window and the table
// in LDS 21, with the stack 12.2; 1500001 bodies mixed: 15.0 to 10.8 ms.
// Groups above 64 targets are evaluated 64 targets at a time, repeating the
// (identical) tree walk for each.
//
// Mixed precision (MIX, group_walkmix_kernel): groups, histories, the tree
// walk and every acceptance decision stay in FP64, so the lists equal the FP64
// walk's; the accepted nodes' expansions stay in FP64 as well (a few per
// target). Only the listed-source pairs change: sources are staged as 32-bit
// fixed-point coordinates (16 B instead of 32 B), a separation is the wrapped
// int32 difference scaled to H-table units, and the pair term is the FP32
// residual of the mixed strict walk (reciprocal square root, the 128-cell
// cubic table of H in LDS). Each staged chunk's FP32 sums are added to the
// FP64 totals, so no FP32 sum runs over more than 64 sources per lane. PM
// interpolation reads the FP32 force meshes at the fixed-point position.
constexpr int kGroupLeafCap = 192;
constexpr int kGroupNodeCap = 128;
constexpr int kGroupStage = 64;  // sources evaluated in a pass
// Open nodes of the tree walk: eight are expanded at a time, one at a time from
// kGroupWide on, so that a depth of 21 levels cannot overflow the stack.
constexpr uint32_t kNoNode = 0xFFFFFFFFu;  // child_index without a child
constexpr uint32_t kGroupWide = 96;
constexpr uint32_t kGroupStack = kGroupWide + 56 + 7 * 21 + 13;
constexpr int kGroupCells = 384;  // FP64 pair table cells held in LDS (12 KB; r_cut = 4.5 a needs 326)

struct GroupLeaf {
  double ox, oy, oz, h;  // cell centre relative to the group centre, cell half size
  uint32_t b, e;         // tree-order source range
};

__device__ __forceinline__ double nearest_image(double d, double L) { return d - L * rint(d / L); }
// The same with 1/L precomputed: rint(d * iL) equals rint(d / L) unless d / L
// lies within an ulp of a half-integer, where both images are equally near.
__device__ __forceinline__ double nearest_image_inv(double d, double L, double iL) {
  return d - L * rint(d * iL);
}
__device__ __forceinline__ double wrap_half(double d, double L) {
  const double hl = 0.5 * L;
  return d > hl ? d - L : (d < -hl ? d + L : d);
}
template <class T> __device__ __forceinline__ T scan_min(T v, int lane) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const T o = __shfl_up(v, off, kWave);
    if (lane >= off) v = o < v ? o : v;
  }
  return v;
}
template <class T> __device__ __forceinline__ T scan_max(T v, int lane) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const T o = __shfl_up(v, off, kWave);
    if (lane >= off) v = o > v ? o : v;
  }
  return v;
}

// inclusive sum / maximum over the lanes up to this one (all 64 active)
__device__ __forceinline__ uint32_t wave_scan_sum(uint32_t v) {
  v += CHUI_DPP(v, 0x111, 0xf, 0u);  // row_shr:1
  v += CHUI_DPP(v, 0x112, 0xf, 0u);  // row_shr:2
  v += CHUI_DPP(v, 0x114, 0xf, 0u);  // row_shr:4
  v += CHUI_DPP(v, 0x118, 0xf, 0u);  // row_shr:8
  v += CHUI_DPP(v, 0x142, 0xa, 0u);  // row_bcast:15
  v += CHUI_DPP(v, 0x143, 0xc, 0u);  // row_bcast:31
  return v;
}
__device__ __forceinline__ uint32_t wave_scan_max(uint32_t v) {
  v = dpp_max_step(v, CHUI_DPP(v, 0x111, 0xf, 0u));
  v = dpp_max_step(v, CHUI_DPP(v, 0x112, 0xf, 0u));
  v = dpp_max_step(v, CHUI_DPP(v, 0x114, 0xf, 0u));
  v = dpp_max_step(v, CHUI_DPP(v, 0x118, 0xf, 0u));
  v = dpp_max_step(v, CHUI_DPP(v, 0x142, 0xa, 0u));
  v = dpp_max_step(v, CHUI_DPP(v, 0x143, 0xc, 0u));
  return v;
}
// LDS written by some lanes of the wave is read by others after this
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One wave's lists and window.
template <bool MIX>
struct GroupLds {
  GroupLeaf leaves[kGroupLeafCap];
  uint32_t nodes[kGroupNodeCap];
  uint32_t leaf_pre[kGroupLeafCap + 1];
  uint32_t open[kGroupStack];
  uint32_t mark[kWave];
  std::conditional_t<MIX, uint4, double4> stage[2 * kGroupStage];
  uint32_t stage_j[2 * kGroupStage];
};

// TAB: the FP64 pair table's cells up to r_cut lie in LDS.
template <int SCHEME, bool MIX, bool NODE32, bool TAB>
__device__ __forceinline__ void group_walk_body(const WalkParams& P, const GroupParams& G, const WalkData& D,
                                                const uint32_t* __restrict__ leaf_of_pos, const WalkOutputs& out,
                                                uint32_t* __restrict__ fb_pos, uint32_t* __restrict__ fb_slot,
                                                uint32_t* __restrict__ fb_count,
                                                unsigned long long* __restrict__ counters) {
  __shared__ GroupLds<MIX> lds_all[kWalkWaves];
  __shared__ float4 htab[MIX ? kHTableCells : 1];
  __shared__ double4 gtab[TAB ? kGroupCells : 1];
  const int w = static_cast<int>(readlane_u32(threadIdx.x / kWave, 0));
  const int lane = threadIdx.x % kWave;
  if constexpr (MIX) {
    for (int i = threadIdx.x; i < kHTableCells; i += kWalkThreads) htab[i] = D.htab[i];
  }
  if constexpr (TAB) {
    for (int i = threadIdx.x; i < static_cast<int>(G.table_cells); i += kWalkThreads) gtab[i] = D.gcoef[i];
  }
  if constexpr (MIX || TAB) __syncthreads();
  GroupLeaf* const leaves = lds_all[w].leaves;
  uint32_t* const nodes = lds_all[w].nodes;
  uint32_t* const leaf_pre = lds_all[w].leaf_pre;
  uint32_t* const mark = lds_all[w].mark;
  uint32_t* const open = lds_all[w].open;
  auto* const stage = lds_all[w].stage;
  uint32_t* const stage_j = lds_all[w].stage_j;
  const uint64_t bb64 = (static_cast<uint64_t>(xcd_logical_block()) * kWalkWaves + w) * G.block;
  if (bb64 >= P.n_targets) return;
  const uint32_t bb = static_cast<uint32_t>(bb64);
  const uint32_t be = min(bb + G.block, P.n_targets);
  const double L0 = P.L[0], L1 = P.L[1], L2 = P.L[2];
  const double cull2 = P.rcut2 * (1.0 + 1.0e-9);
  // table coordinates end below 64, or within the cells held in LDS (every
  // pair inside r_cut lies below)
  const double tlim = TAB ? (G.table_cells - 0.5) / 64.0 : 0x1.fffffffffffffp+5;
  const double iL0 = 1.0 / P.L[0], iL1 = 1.0 / P.L[1], iL2 = 1.0 / P.L[2];
  const double eps2 = P.eps * P.eps;
  uint32_t cnt[kGroupCounters] = {};
  unsigned long long size_max = 0, entries_max = 0;
  auto tpos = [&](uint32_t v) { return P.identity_targets ? v : D.tpos[v]; };
  auto tslot = [&](uint32_t v) { return P.identity_targets ? D.order[v] : D.tslot[v]; };

  uint32_t v = bb;
  while (v < be) {
    const double4 p0 = D.src64[tpos(v)];
    // ---- the group [v, ge) (tree_pm_coupling.cpp:4491-4523)
    uint32_t ge;
    if (G.group_size == 0) {
      const uint32_t leaf0 = leaf_of_pos[tpos(v)];
      ge = be;
      for (uint32_t c = v + 1; c < be; c += kWave) {
        const uint32_t k = c + lane;
        const unsigned long long m = __ballot(k < be && leaf_of_pos[tpos(k)] != leaf0);
        if (m) {
          ge = c + static_cast<uint32_t>(__ffsll(static_cast<long long>(m)) - 1);
          break;
        }
      }
    } else {
      const uint32_t lim = min(be, v + G.group_size);
      double lo0 = 0.0, lo1 = 0.0, lo2 = 0.0, hi0 = 0.0, hi1 = 0.0, hi2 = 0.0;
      ge = lim;
      for (uint32_t c = v + 1; c < lim; c += kWave) {
        const uint32_t k = c + lane;
        const bool in = k < lim;
        double d0 = 0.0, d1 = 0.0, d2 = 0.0;  // 0 is neutral: every running box holds 0
        if (in) {
          const double4 q = D.src64[tpos(k)];
          d0 = nearest_image(q.x - p0.x, L0);
          d1 = nearest_image(q.y - p0.y, L1);
          d2 = nearest_image(q.z - p0.z, L2);
        }
        const double a0 = scan_min(fmin(lo0, d0), lane), a1 = scan_min(fmin(lo1, d1), lane),
                     a2 = scan_min(fmin(lo2, d2), lane);
        const double b0 = scan_max(fmax(hi0, d0), lane), b1 = scan_max(fmax(hi1, d1), lane),
                     b2 = scan_max(fmax(hi2, d2), lane);
        const bool within = b0 - a0 <= G.max_extent && b1 - a1 <= G.max_extent && b2 - a2 <= G.max_extent;
        const unsigned long long bad = __ballot(in && !within);
        if (bad) {
          ge = c + static_cast<uint32_t>(__ffsll(static_cast<long long>(bad)) - 1);
          break;
        }
        lo0 = readlane_f64(a0, 63); lo1 = readlane_f64(a1, 63); lo2 = readlane_f64(a2, 63);
        hi0 = readlane_f64(b0, 63); hi1 = readlane_f64(b1, 63); hi2 = readlane_f64(b2, 63);
      }
    }
    const uint32_t count = ge - v;

    // ---- history / bounded metric, minimum |a_prev| and the group box (:4333-4370)
    int fall = 0;  // 1 history, 2 geometry (first failing target decides)
    double amin = INFINITY, lo0 = 0.0, lo1 = 0.0, lo2 = 0.0, hi0 = 0.0, hi1 = 0.0, hi2 = 0.0;
    for (uint32_t c = v; c < ge; c += kWave) {
      const uint32_t k = c + lane;
      const bool in = k < ge;
      double pv = INFINITY, d0 = 0.0, d1 = 0.0, d2 = 0.0;
      bool hist = true, bounded = true;
      if (in) {
        pv = D.prev != nullptr ? D.prev[tslot(k)] : NAN;
        hist = isfinite(pv) && pv > P.accel_floor;
        const double4 q = D.src64[tpos(k)];
        bounded = G.lo[0] - q.x >= -L0 && G.hi[0] - q.x <= L0 && G.lo[1] - q.y >= -L1 && G.hi[1] - q.y <= L1 &&
                  G.lo[2] - q.z >= -L2 && G.hi[2] - q.z <= L2;
        d0 = nearest_image(q.x - p0.x, L0);
        d1 = nearest_image(q.y - p0.y, L1);
        d2 = nearest_image(q.z - p0.z, L2);
      }
      const unsigned long long bad = __ballot(in && !(hist && bounded));
      if (bad) {
        const uint32_t l = static_cast<uint32_t>(__ffsll(static_cast<long long>(bad)) - 1);
        fall = readlane_u32(hist ? 2u : 1u, l);
        break;
      }
      amin = fmin(amin, wave_min(in ? pv : INFINITY));
      lo0 = fmin(lo0, wave_min(d0)); lo1 = fmin(lo1, wave_min(d1)); lo2 = fmin(lo2, wave_min(d2));
      hi0 = fmax(hi0, wave_max(d0)); hi1 = fmax(hi1, wave_max(d1)); hi2 = fmax(hi2, wave_max(d2));
    }
    if (fall) {
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(fb_count, count);
      base = readlane_u32(base, 0);
      for (uint32_t c = v; c < ge; c += kWave) {
        const uint32_t k = c + lane;
        if (k < ge) {
          fb_pos[base + (k - v)] = tpos(k);
          fb_slot[base + (k - v)] = tslot(k);
        }
      }
      if (lane == 0) {
        cnt[8] += count;
        if (fall == 1) cnt[9] += count;
        else cnt[10] += count;
      }
      v = ge;
      continue;
    }
    // wave-uniform group box and minimum |a_prev| (scalar registers)
    amin = readlane_f64(amin, 0);
    const double c0x = readlane_f64(p0.x + 0.5 * (lo0 + hi0), 0), c0y = readlane_f64(p0.y + 0.5 * (lo1 + hi1), 0),
                 c0z = readlane_f64(p0.z + 0.5 * (lo2 + hi2), 0);
    const double hg0 = readlane_f64(0.5 * (hi0 - lo0), 0), hg1 = readlane_f64(0.5 * (hi1 - lo1), 0),
                 hg2 = readlane_f64(0.5 * (hi2 - lo2), 0);
    if (lane == 0) {
      cnt[5] += 1;
      cnt[6] += count;
    }
    // all sources in [0, L] and r_cut around the group inside the box on every
    // axis: its pairs need no image (a source within r_cut of the group box has
    // none nearer)
    const double rcm = P.rcut * (1.0 + 1.0e-9);
    const auto clear = [&](double c, double hg, double L, int a) {
      return G.lo[a] >= 0.0 && G.hi[a] <= L && c - hg - rcm > 0.0 && c + hg + rcm < L && 2.0 * hg + rcm < 0.4999 * L;
    };
    const bool inner = clear(c0x, hg0, L0, 0) && clear(c0y, hg1, L1, 1) && clear(c0z, hg2, L2, 2);
    // MIX: the group box in fixed point and table units, widened by the
    // roundings of its centre and of the offsets
    uint32_t gcx = 0, gcy = 0, gcz = 0;
    float gt0 = 0.0f, gt1 = 0.0f, gt2 = 0.0f;
    if constexpr (MIX) {
      const double f0 = 4294967296.0 / L0, f1 = 4294967296.0 / L1, f2 = 4294967296.0 / L2;
      gcx = readlane_u32(static_cast<uint32_t>(static_cast<int64_t>(floor(c0x * f0))), 0);
      gcy = readlane_u32(static_cast<uint32_t>(static_cast<int64_t>(floor(c0y * f1))), 0);
      gcz = readlane_u32(static_cast<uint32_t>(static_cast<int64_t>(floor(c0z * f2))), 0);
      gt0 = static_cast<float>(hg0 * f0 + 4.0) * P.tab_scale[0] * 1.000001f;
      gt1 = static_cast<float>(hg1 * f1 + 4.0) * P.tab_scale[1] * 1.000001f;
      gt2 = static_cast<float>(hg2 * f2 + 4.0) * P.tab_scale[2] * 1.000001f;
    }
    size_max = count > size_max ? count : size_max;

    // ---- targets, 64 at a time
    for (uint32_t t0 = v; t0 < ge; t0 += kWave) {
      const uint32_t T = min(ge - t0, static_cast<uint32_t>(kWave));
      int S = 1;  // lanes per target: the largest power of two with S * T <= 64
      while (S < kWave && static_cast<uint32_t>(2 * S) * T <= static_cast<uint32_t>(kWave)) S *= 2;
      const int TT = kWave / S;
      const int t = lane & (TT - 1), s = lane / TT;
      const bool valid = static_cast<uint32_t>(t) < T;
      const bool first = t0 == v;  // count the (repeated) tree walk once per group
      uint32_t tp = 0, slot = 0;
      uint32_t tx = 0, ty = 0, tz = 0;  // MIX: fixed-point target position
      double px = 0.0, py = 0.0, pz = 0.0, ox = 0.0, oy = 0.0, oz = 0.0;
      if (valid) {
        tp = tpos(t0 + t);
        slot = tslot(t0 + t);
        if constexpr (MIX) {
          const uint4 f = D.src32[tp];
          tx = f.x;
          ty = f.y;
          tz = f.z;
        }
        const double4 q = D.src64[tp];
        px = q.x;
        py = q.y;
        pz = q.z;
        ox = nearest_image(px - c0x, L0);
        oy = nearest_image(py - c0y, L1);
        oz = nearest_image(pz - c0z, L2);
      }
      double ax = 0.0, ay = 0.0, az = 0.0, nearest = INFINITY;
      uint32_t listed = 0, nl = 0, nm = 0;

      uint32_t wn = 0;  // sources in the window, below kGroupStage between batches
      // the first gn staged sources: each of a target's S lanes takes every
      // S-th one
      auto pairs = [&]<bool WRAP>(uint32_t gn) {
        if (!valid) return;
        if constexpr (MIX) {
          // FP32 pairs in H-table units (the mixed strict walk's pair term)
          const float u0 = P.tab_scale[0], u1 = P.tab_scale[1], u2 = P.tab_scale[2];
          const float rc2 = P.rcut2_tab, e2 = P.eps2_tab, c8 = P.c8_tab;
          float lx = 0.0f, ly = 0.0f, lz = 0.0f, near_t = INFINITY;
          uint32_t inside_n = 0;
          for (uint32_t q = s; q < gn; q += S) {
            const uint4 sv = stage[q];
            const uint32_t j = stage_j[q];
            const float dx = fx_delta(sv.x, tx, u0), dy = fx_delta(sv.y, ty, u1), dz = fx_delta(sv.z, tz, u2);
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            const float rinv = __builtin_amdgcn_rsqf(r2 + e2);
            const float soft = rinv * rinv * rinv;
            const int ci = static_cast<int>(fminf(r2, static_cast<float>(kHTableCells - 1)));
            const float fu = __builtin_amdgcn_fractf(r2);
            const float4 c = htab[ci];
            const float hcoef = fmaf(fmaf(fmaf(c.w, fu, c.z), fu, c.y), fu, c.x);
            float fr = fmaf(-hcoef, c8, soft);
            if (!D.uniform_mass) fr *= __uint_as_float(sv.w);
            const bool inside = j != tp && r2 <= rc2;
            const float f = inside ? fr : 0.0f;
            lx = fmaf(f, dx, lx);
            ly = fmaf(f, dy, ly);
            lz = fmaf(f, dz, lz);
            inside_n += inside ? 1u : 0u;
            near_t = inside ? fminf(near_t, r2) : near_t;
          }
          const double gm = P.force_scale;
          ax = fma(gm, static_cast<double>(lx), ax);
          ay = fma(gm, static_cast<double>(ly), ay);
          az = fma(gm, static_cast<double>(lz), az);
          cnt[2] += inside_n;
          nearest = fmin(nearest, static_cast<double>(near_t) * static_cast<double>(P.tab_to_len2));
        } else {
          for (uint32_t q = s; q < gn; q += S) {
            const double4 sj = stage[q];
            const uint32_t j = stage_j[q];
            // minimum image by rounding: the same separations as wrap_half
            // wherever |d| <= L/2 or d - L is exact (every pair inside r_cut)
            const double ex = sj.x - px, ey = sj.y - py, ez = sj.z - pz;
            const double dx = WRAP ? fma(-L0, rint(ex * iL0), ex) : ex, dy = WRAP ? fma(-L1, rint(ey * iL1), ey) : ey,
                         dz = WRAP ? fma(-L2, rint(ez * iL2), ez) : ez;
            const double r2 = dx * dx + dy * dy + dz * dz;
            const bool inside = j != tp && r2 <= P.rcut2;
            // the Hermite cell as a cubic in u (Horner with fused steps)
            const double cell = fmin(r2 * P.inv2a2, tlim) * 64.0;
            const int ci = static_cast<int>(cell);
            const double u = cell - static_cast<double>(ci);
            const double4 hc = TAB ? gtab[ci] : D.gcoef[ci];
            const double lr = fma(fma(fma(hc.w, u, hc.z), u, hc.y), u, hc.x) * P.inv8a3;
            // (r^2 + eps^2)^(-3/2): hardware reciprocal square root and two
            // Newton steps y <- y + y (1 - dd y^2) / 2 (r2 = 0 is masked below)
            const double dd = r2 + eps2;
            double y = __builtin_amdgcn_rsq(dd);
            y = fma(0.5 * y, fma(-dd * y, y, 1.0), y);
            y = fma(0.5 * y, fma(-dd * y, y, 1.0), y);
            const double soft = y * y * y;
            const double mj = D.uniform_mass ? P.uniform_mass : sj.w;
            const double f = inside && r2 > 0.0 ? (soft - lr) * P.G * mj : 0.0;
            ax += f * dx;
            ay += f * dy;
            az += f * dz;
            cnt[2] += inside ? 1u : 0u;
            nearest = inside ? fmin(nearest, r2) : nearest;
          }
        }
      };
      auto evaluate = [&](bool last) {
        wave_sync();
        // candidate and culled leaves per target (the counters of
        // accumulateTreePmGroupCulledLeaves): a culled leaf lies beyond r_cut
        // of the target, so its sources add nothing to the pair sums below
        if (G.count) {
          for (uint32_t e = s; e < nl; e += S) {
            if (!valid) continue;
            const GroupLeaf Lf = leaves[e];
            const double gx = fmax(0.0, fabs(wrap_half(Lf.ox - ox, L0)) - Lf.h);
            const double gy = fmax(0.0, fabs(wrap_half(Lf.oy - oy, L1)) - Lf.h);
            const double gz = fmax(0.0, fabs(wrap_half(Lf.oz - oz, L2)) - Lf.h);
            const bool cull = gx * gx + gy * gy + gz * gz > cull2;
            ++cnt[11];
            if (cull) ++cnt[12];
            else cnt[13] += Lf.e - Lf.b;
          }
        }
        // exclusive prefix of the listed leaves' source counts
        uint32_t total = 0;
        for (uint32_t c = 0; c < nl; c += kWave) {
          const uint32_t e = c + lane;
          const uint32_t own = e < nl ? leaves[e].e - leaves[e].b : 0u;
          const uint32_t incl = wave_scan_sum(own);
          if (e < nl) leaf_pre[e] = total + incl - own;
          total += readlane_u32(incl, kWave - 1);
        }
        wave_sync();
        // the listed sources, 64 at a time: leaves (none is empty) mark the
        // lane where they start and a running maximum gives every lane its
        // leaf; sources beyond r_cut of the group box are dropped
        uint32_t e0 = 0;  // the leaf of the last batch's last source
        for (uint32_t g0 = 0;; g0 += kWave) {
          mark[lane] = 0;
          wave_sync();
          const uint32_t e = e0 + 1u + lane;
          const uint32_t st = e < nl ? leaf_pre[e] - g0 : static_cast<uint32_t>(kWave);
          if (st < static_cast<uint32_t>(kWave)) mark[st] = lane + 1u;
          wave_sync();
          const uint32_t lf = e0 + wave_scan_max(mark[lane]);
          const uint32_t g = g0 + lane;
          const bool on = g < total;
          const uint32_t j = on ? leaves[lf].b + (g - leaf_pre[lf]) : 0u;
          e0 = readlane_u32(lf, kWave - 1);
          bool keep;
          std::conditional_t<MIX, uint4, double4> rec;
          if constexpr (MIX) {
            rec = D.src32[j];
            const float ex = fmaxf(fabsf(fx_delta(rec.x, gcx, P.tab_scale[0])) - gt0, 0.0f);
            const float ey = fmaxf(fabsf(fx_delta(rec.y, gcy, P.tab_scale[1])) - gt1, 0.0f);
            const float ez = fmaxf(fabsf(fx_delta(rec.z, gcz, P.tab_scale[2])) - gt2, 0.0f);
            keep = on && !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > P.rcut2_tab * 1.00001f);
          } else {
            rec = D.src64[j];
            const double ex = fmax(0.0, fabs(nearest_image_inv(rec.x - c0x, L0, iL0)) - hg0);
            const double ey = fmax(0.0, fabs(nearest_image_inv(rec.y - c0y, L1, iL1)) - hg1);
            const double ez = fmax(0.0, fabs(nearest_image_inv(rec.z - c0z, L2, iL2)) - hg2);
            keep = on && !(ex * ex + ey * ey + ez * ez > cull2);
          }
          const unsigned long long km = __ballot(keep);
          if (keep) {
            const uint32_t at = wn + static_cast<uint32_t>(__popcll(km & ((1ull << lane) - 1ull)));
            stage[at] = rec;
            stage_j[at] = j;
          }
          wn += static_cast<uint32_t>(__popcll(km));
          const bool end = g0 + kWave >= total;
          while (wn >= static_cast<uint32_t>(kGroupStage) || (last && end && wn)) {
            const uint32_t gn = wn < static_cast<uint32_t>(kGroupStage) ? wn : static_cast<uint32_t>(kGroupStage);
            wave_sync();
            if (MIX || !inner) pairs.template operator()<true>(gn);
            else pairs.template operator()<false>(gn);
            wave_sync();
            wn -= gn;
            // the records past the window move to its front
            if (static_cast<uint32_t>(lane) < wn) {
              stage[lane] = stage[kGroupStage + lane];
              stage_j[lane] = stage_j[kGroupStage + lane];
            }
          }
          wave_sync();
          if (end) break;
        }
        for (uint32_t e = s; e < nm; e += S) {
          if (!valid) continue;
          const uint32_t nd = nodes[e];
          const NodeMom64 M = D.mom64[nd];
          const double dx = mi64(M.comx - px, L0), dy = mi64(M.comy - py, L1), dz = mi64(M.comz - pz, L2);
          if (P.com_cut && dx * dx + dy * dy + dz * dz > P.rcut2) {
            ++cnt[1];
            continue;
          }
          if constexpr (NODE32) {
            // the mixed strict walk's FP32 expansion from the fixed-point
            // centre of mass (the cutoff decision above stays FP64)
            const NodeMom32 M32 = D.mom32[nd];
            const float s0 = P.cubic ? 1.0f : P.fx_to_len[0], s1 = P.cubic ? 1.0f : P.fx_to_len[1],
                        s2 = P.cubic ? 1.0f : P.fx_to_len[2], tl = P.cubic ? P.fx_to_len[0] : 1.0f;
            float cx = 0.0f, cy = 0.0f, cz = 0.0f;
            node_accel32(M32, D.quad32[nd], fx_delta(M32.comx, tx, s0) * tl, fx_delta(M32.comy, ty, s1) * tl,
                         fx_delta(M32.comz, tz, s2) * tl, P, cx, cy, cz);
            ax += cx;
            ay += cy;
            az += cz;
          } else {
            // inline: an out-of-line call here saves and restores the live
            // registers through scratch on every accepted node
            if (P.radial) node_accel_radial64(M, D.quad64[nd], dx, dy, dz, P, ax, ay, az);
            else node_accel64(M, D.quad64[nd], dx, dy, dz, P, ax, ay, az);
          }
        }
        wave_sync();
        nl = 0;
        nm = 0;
      };

      uint32_t sp = 0;
      bool root = true;
      while (true) {
        const bool done = !root && sp == 0;
        if (done || nl > static_cast<uint32_t>(kGroupLeafCap - kWave) ||
            nm > static_cast<uint32_t>(kGroupNodeCap - kWave))
          evaluate(done);
        if (done) break;
        // decide the children of up to eight open nodes (or the root) for the
        // group box, one to a lane
        uint32_t q = kNoNode;
        wave_sync();
        if (root) {
          if (lane == 0) q = 0;
          root = false;
        } else {
          const uint32_t m = sp > kGroupWide ? 1u : min(sp, 8u);
          sp -= m;
          const uint32_t k = static_cast<uint32_t>(lane) >> 3;
          if (k < m) q = D.child_index[8ull * open[sp + k] + (lane & 7)];
        }
        wave_sync();
        const bool on = q != kNoNode;
        uint32_t lb = 0, le = 0;
        int kind = 3;  // 0 pruned, 1 listed leaf, 2 accepted node, 3 opened
        double dc0 = 0.0, dc1 = 0.0, dc2 = 0.0, h = 0.0;
        if (on) {
          const NodeLink lk = D.link[q];
          const NodeGeo64 g = D.geo64[q];
          h = g.half;
          dc0 = nearest_image_inv(g.cx - c0x, L0, iL0);
          dc1 = nearest_image_inv(g.cy - c0y, L1, iL1);
          dc2 = nearest_image_inv(g.cz - c0z, L2, iL2);
          const double v0 = fabs(dc0), v1 = fabs(dc1), v2 = fabs(dc2);
          const double g0 = fmax(0.0, v0 - h - hg0), g1 = fmax(0.0, v1 - h - hg1), g2 = fmax(0.0, v2 - h - hg2);
          const double f0 = v0 + h + hg0, f1 = v1 + h + hg1, f2 = v2 + h + hg2;
          const double gap2 = g0 * g0 + g1 * g1 + g2 * g2;
          const double far2 = f0 * f0 + f1 * f1 + f2 * f2;
          if (gap2 > P.rcut2) {
            kind = 0;
          } else if (lk.child_count == 0) {
            kind = 1;
            lb = lk.begin;
            le = lk.begin + lk.count;
          } else {
            bool acc = gap2 > 0.0 && (!G.contain || far2 <= P.rcut2);
            if (acc) {
              const NodeMom64 M = D.mom64[q];
              const double m0 = fmax(0.0, fabs(nearest_image_inv(M.comx - c0x, L0, iL0)) - hg0);
              const double m1 = fmax(0.0, fabs(nearest_image_inv(M.comy - c0y, L1, iL1)) - hg1);
              const double m2 = fmax(0.0, fabs(nearest_image_inv(M.comz - c0z, L2, iL2)) - hg2);
              const double rmin2 = m0 * m0 + m1 * m1 + m2 * m2;
              const double width2 = 4.0 * h * h;
              acc = rmin2 > 0.0 && width2 < G.amax2 * rmin2 && M.mass * width2 <= G.tolg * amin * rmin2 * rmin2;
            }
            kind = acc ? 2 : 3;
          }
        }
        const unsigned long long vm = __ballot(on);
        const unsigned long long lm = __ballot(on && kind == 1);
        const unsigned long long mm = __ballot(on && kind == 2);
        const unsigned long long below = (1ull << lane) - 1ull;
        if (on && kind == 1) {
          GroupLeaf& Lf = leaves[nl + __popcll(lm & below)];
          Lf.ox = dc0;
          Lf.oy = dc1;
          Lf.oz = dc2;
          Lf.h = h;
          Lf.b = lb;
          Lf.e = le;
        }
        if (on && kind == 2) nodes[nm + __popcll(mm & below)] = q;
        const unsigned long long pm = __ballot(on && kind == 0), om = __ballot(on && kind == 3);
        if (on && kind == 3) open[sp + __popcll(om & below)] = q;
        sp += __popcll(om);
        nl += __popcll(lm);
        nm += __popcll(mm);
        listed += __popcll(lm) + __popcll(mm);
        if (first && lane == 0) {
          cnt[0] += __popcll(vm);
          cnt[1] += __popcll(pm);
          cnt[3] += __popcll(mm);
          cnt[4] += __popcll(lm);
        }
      }
      entries_max = listed > entries_max ? listed : entries_max;
      // sums of a target's lanes
      for (int off = TT; off < kWave; off <<= 1) {
        ax += __shfl_xor(ax, off, kWave);
        ay += __shfl_xor(ay, off, kWave);
        az += __shfl_xor(az, off, kWave);
        nearest = fmin(nearest, __shfl_xor(nearest, off, kWave));
      }
      if (MIX && valid && s == 0) {
        float gx = 0.0f, gy = 0.0f, gz = 0.0f;
        if (P.pm_enabled) interp32<SCHEME>(P, D.f32x, D.f32y, D.f32z, tx, ty, tz, gx, gy, gz);
        const float sx = static_cast<float>(ax), sy = static_cast<float>(ay), sz = static_cast<float>(az);
        static_cast<float*>(out.ax)[slot] = gx + sx;
        static_cast<float*>(out.ay)[slot] = gy + sy;
        static_cast<float*>(out.az)[slot] = gz + sz;
        if (out.pm_x) {
          static_cast<float*>(out.pm_x)[slot] = gx;
          static_cast<float*>(out.pm_y)[slot] = gy;
          static_cast<float*>(out.pm_z)[slot] = gz;
        }
        const uint32_t row = D.order[tp];
        if (out.sr_x) {
          static_cast<float*>(out.sr_x)[row] = sx;
          static_cast<float*>(out.sr_y)[row] = sy;
          static_cast<float*>(out.sr_z)[row] = sz;
        }
        if (out.near2) static_cast<float*>(out.near2)[row] = static_cast<float>(nearest);
      } else if (!MIX && valid && s == 0) {
        double gx = 0.0, gy = 0.0, gz = 0.0;
        if (P.pm_enabled) interp64<SCHEME>(P, D.f64x, D.f64y, D.f64z, px, py, pz, gx, gy, gz);
        static_cast<double*>(out.ax)[slot] = gx + ax;
        static_cast<double*>(out.ay)[slot] = gy + ay;
        static_cast<double*>(out.az)[slot] = gz + az;
        if (out.pm_x) {
          static_cast<double*>(out.pm_x)[slot] = gx;
          static_cast<double*>(out.pm_y)[slot] = gy;
          static_cast<double*>(out.pm_z)[slot] = gz;
        }
        const uint32_t row = D.order[tp];
        if (out.sr_x) {
          static_cast<double*>(out.sr_x)[row] = ax;
          static_cast<double*>(out.sr_y)[row] = ay;
          static_cast<double*>(out.sr_z)[row] = az;
        }
        if (out.near2) static_cast<double*>(out.near2)[row] = nearest;
      }
    }
    v = ge;
  }
#pragma unroll
  for (int i = 0; i < kGroupCounters; ++i) {
    if (i == 7 || i == 14) continue;
    const unsigned long long sum = wave_sum(static_cast<unsigned long long>(cnt[i]));
    if (lane == 0 && sum) atomicAdd(&counters[i], sum);
  }
  if (lane == 0) {
    if (size_max) atomicMax(&counters[7], size_max);
    if (entries_max) atomicMax(&counters[14], entries_max);
  }
}

// Two waves per SIMD (256 VGPRs) where the FP64 node expansions are inline:
// the body needs about that many; at 168 VGPRs (3 waves) it spilled 384-512
// bytes per lane and ran 2% (FP64) to 29% (mixed) slower at 256^3 (the walk
// before the stack; now 256 VGPRs spill 24 to 27 of them). The mixed walk with
// FP32 node expansions (RADIAL false) holds 152 VGPRs without spills and runs 3
// waves per SIMD (4 waves: 128 VGPRs with spills, 16% slower, before the stack).
template <int SCHEME, bool TAB>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(2))) void group_walk64_kernel(
    WalkParams P, GroupParams G, WalkData D, const uint32_t* __restrict__ leaf_of_pos, WalkOutputs out,
    uint32_t* __restrict__ fb_pos, uint32_t* __restrict__ fb_slot, uint32_t* __restrict__ fb_count,
    unsigned long long* __restrict__ counters) {
  group_walk_body<SCHEME, false, false, TAB>(P, G, D, leaf_of_pos, out, fb_pos, fb_slot, fb_count, counters);
}

// RADIAL: the radial-coefficient node expansion (FP64; the FP32 expansion is
// the plain monopole + quadrupole one).
template <int SCHEME, bool RADIAL>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(RADIAL ? 2 : 3))) void group_walkmix_kernel(
    WalkParams P, GroupParams G, WalkData D, const uint32_t* __restrict__ leaf_of_pos, WalkOutputs out,
    uint32_t* __restrict__ fb_pos, uint32_t* __restrict__ fb_slot, uint32_t* __restrict__ fb_count,
    unsigned long long* __restrict__ counters) {
  group_walk_body<SCHEME, true, !RADIAL, false>(P, G, D, leaf_of_pos, out, fb_pos, fb_slot, fb_count, counters);
}

// Mixed adaptive solves: targets the group walk hands back (or every target
// when the group walk does not run) take the FP64 per-target adaptive walk
// without PM, written into FP64 lanes by output slot (nearest pair by source
// row). This kernel adds the FP32 PM interpolation at the fixed-point
// position and writes the FP32 outputs of those targets. pos/slot: the
// targets' tree positions and output slots (identity: position k, slot
// order[k]).
template <int SCHEME>
__global__ __launch_bounds__(256) void adaptive_mixed_finish_kernel(WalkParams P, WalkData D,
                                                                    const uint32_t* __restrict__ pos,
                                                                    const uint32_t* __restrict__ slot, uint32_t n,
                                                                    int identity, const double* __restrict__ sx,
                                                                    const double* __restrict__ sy,
                                                                    const double* __restrict__ sz,
                                                                    const double* __restrict__ near64,
                                                                    WalkOutputs out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t tp = identity ? i : pos[i];
  const uint32_t sl = identity ? D.order[i] : slot[i];
  const uint4 f = D.src32[tp];
  float gx = 0.0f, gy = 0.0f, gz = 0.0f;
  if (P.pm_enabled) interp32<SCHEME>(P, D.f32x, D.f32y, D.f32z, f.x, f.y, f.z, gx, gy, gz);
  const float ax = static_cast<float>(sx[sl]), ay = static_cast<float>(sy[sl]), az = static_cast<float>(sz[sl]);
  static_cast<float*>(out.ax)[sl] = gx + ax;
  static_cast<float*>(out.ay)[sl] = gy + ay;
  static_cast<float*>(out.az)[sl] = gz + az;
  if (out.pm_x) {
    static_cast<float*>(out.pm_x)[sl] = gx;
    static_cast<float*>(out.pm_y)[sl] = gy;
    static_cast<float*>(out.pm_z)[sl] = gz;
  }
  const uint32_t row = D.order[tp];
  if (out.sr_x) {
    static_cast<float*>(out.sr_x)[row] = ax;
    static_cast<float*>(out.sr_y)[row] = ay;
    static_cast<float*>(out.sr_z)[row] = az;
  }
  if (out.near2) static_cast<float*>(out.near2)[row] = static_cast<float>(near64[row]);
}

__global__ void leaf_of_pos_kernel(const NodeLink* __restrict__ link, std::size_t nodes,
                                   uint32_t* __restrict__ leaf_of_pos) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= nodes) return;
  const NodeLink lk = link[i];
  if (lk.child_count != 0) return;
  for (uint32_t p = lk.begin; p < lk.begin + lk.count; ++p) leaf_of_pos[p] = static_cast<uint32_t>(i);
}

// ---- mixed walk -----------------------------------------------------------------
// CUBIC: equal box lengths, so separations stay in fixed-point units (one
// scale factor for all axes) and only the pair kernel converts to lengths.
//
// A leaf that any lane keeps is staged in the wave's LDS window with one
// coalesced load (one source per lane). Every lane then evaluates the residual
// pair kernel against each staged source in turn, reading it with a broadcast
// LDS load, and keeps the term when the pair lies inside r_cut (a lane that
// pruned the leaf compares against a negative cutoff). A leaf's pair terms
// are summed in registers and added to a per-lane partial sum in LDS, which is
// folded into the lane's Kahan-compensated totals (also in LDS) every kWindow
// sources. Keeping these sums out of the node loop's registers spares the
// loop-carried copies the compiler would otherwise make on every node.
//
// Window format. Most waves hold 64 consecutive tree-order targets inside a
// small region: their window stores float offsets from the wave origin O (the
// centre of the targets' fixed-point bounding box), so a separation is three
// float subtractions. The exact minimum image is kept because every offset
// int32(q - O) is exact and, when all targets lie within min(L/16, L/2 - r_cut)
// of O (per axis), a pair inside r_cut cannot straddle the wrap of O's frame.
// Waves that straddle a jump of the space-filling order (targets far apart)
// store raw fixed-point coordinates and form int32(q_s - q_t) per pair.
//
// The timed walk is walkmix_box_kernel below: the same pairs and multipoles
// from a traversal per box of targets, summed in another order.
constexpr int kWindow = 64;
constexpr int kPairGroup = 2;  // box walk: table reads in flight together

//
// Residual table indexed by the float bits (LOG, the timed walk): the whole
// pair coefficient F(s) = s^{-3/2} - c8 H((s/scale - eps^2) / 4a^2) as a
// function of s = r^2 + eps^2 in table units, whose scale puts r_cut^2 + eps^2
// at s = 1. The cell of s is its exponent and top 5 mantissa bits (32 cubic
// Hermite cells per octave, from the octave of eps^2 up to s = 1, then one
// zero cell), the position in the cell its low 18 mantissa bits as an integer
// (the coefficients carry the 2^-18 powers). eps^2 enters the FMA chain of
// r^2, the chain's last FMA clamps s to [0, 1] (so every pair beyond r_cut
// lands in the zero cell, the cell of s = 1), and the octave base is folded
// into the table's LDS address. A pair then costs a shift, an address add, an
// LDS read, the position (and, convert) and three FMAs instead of a
// reciprocal square root, the Gaussian table and a cutoff select. Cubic
// Hermite cells of relative width 1/32 to 1/64 keep F within 1.5e-7 of its
// value.
//
// 16-byte cell `cell` of an LDS table at LDS address `base`: the address is
// one shift-add (the compiler folds a constant shift of a shifted value into
// shift, and, add). Inline asm counts as convergent, so a loop holding it is
// unrolled only with a constant trip count: the box walk's windows use it
// (groups of kPairGroup), the lane-by-lane walk indexes the table plainly.
typedef float f32x4 __attribute__((ext_vector_type(4)));
using lds_f32x4 = __attribute__((address_space(3))) const f32x4;
__device__ __forceinline__ float4 lds_cell(uint32_t base, uint32_t cell) {
  uint32_t a;
  asm("v_lshl_add_u32 %0, %1, 4, %2" : "=v"(a) : "v"(cell), "s"(base));
  const f32x4 v = *(lds_f32x4*)static_cast<uintptr_t>(a);
  return make_float4(v.x, v.y, v.z, v.w);
}

// The counting walk (diagnostics, counters, the nearest-pair lane): lane by
// lane, one pair kernel with the reciprocal square root and the Gaussian table.
template <int SCHEME, bool CUBIC>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(4)))
void walkmix_kernel(WalkParams P, WalkData D, WalkOutputs out, unsigned long long* __restrict__ counters,
                    const NodeLink* __restrict__ node_link, const NodeGeo32* __restrict__ node_geo,
                    const NodeMom32* __restrict__ node_mom, const NodeQuad32* __restrict__ node_quad,
                    const NodeBox32* __restrict__ node_box) {
  // node records are read-only for the kernel's lifetime and indexed by the
  // wave-uniform node number, so they come through the scalar cache
  __shared__ float4 win[kWalkWaves][kWindow];
  __shared__ float4 htab[kHTableCells];
  // per lane: force totals [0..2] and their Kahan compensations [3..5]
  __shared__ float ksum[kWalkWaves][6][kWave];
  for (int i = threadIdx.x; i < kHTableCells; i += kWalkThreads) htab[i] = D.htab[i];
  __syncthreads();
  const uint32_t node_count = P.node_count;
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const uint32_t k = xcd_logical_block() * kWalkThreads + threadIdx.x;
  const bool valid = k < P.n_targets;
  const uint32_t tp = valid ? (P.identity_targets ? k : D.tpos[k]) : 0u;
  const uint32_t slot = valid ? (P.identity_targets ? D.order[k] : D.tslot[k]) : 0u;
  uint32_t cnt[kWalkCounters] = {0, 0, 0, 0, 0, 0, 0, 0};
  uint32_t nxt = valid ? 0u : node_count;
  float nearest = INFINITY;  // counting variant: nearest distinct pair, table units
  uint32_t px = 0, py = 0, pz = 0;
  float gx = 0.0f, gy = 0.0f, gz = 0.0f;
  if (valid) {
    const uint4 t = D.src32[tp];
    px = t.x;
    py = t.y;
    pz = t.z;
    if (P.pm_enabled) interp32<SCHEME>(P, D.f32x, D.f32y, D.f32z, px, py, pz, gx, gy, gz);
  }
  // node tests: fixed-point units (CUBIC) or lengths
  const float s0 = CUBIC ? 1.0f : P.fx_to_len[0];
  const float s1 = CUBIC ? 1.0f : P.fx_to_len[1];
  const float s2 = CUBIC ? 1.0f : P.fx_to_len[2];
  const float to_len = CUBIC ? P.fx_to_len[0] : 1.0f;          // node separation unit -> length
  const float inv_len = CUBIC ? 1.0f / P.fx_to_len[0] : 1.0f;  // length -> node separation unit
  const float prune2 = P.prune2_sep;
  const float contain2 = P.contain2_sep;
  const float theta2 = static_cast<float>(P.theta * P.theta);
  // pairs: table units (lengths * sqrt(t_to_cell)), so r^2 is the H-table coordinate
  const float u0 = P.tab_scale[0], u1 = P.tab_scale[1], u2 = P.tab_scale[2];
  const float rc2 = P.rcut2_tab;
  const float eps2 = P.eps2_tab;
  const float c8 = P.c8_tab;
  // wave origin: centre of the valid targets' bounding box in fixed point
  uint32_t org[3];
  bool near = true;
  {
    const uint32_t pp[3] = {px, py, pz};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t o0 = readlane_u32(pp[a], 0);
      const int32_t off = valid ? static_cast<int32_t>(pp[a] - o0) : 0;
      // wave-uniform through readlane, so the box lives in scalar registers
      const int32_t lo = static_cast<int32_t>(readlane_u32(static_cast<uint32_t>(wave_min(off)), 0));
      const int32_t hi = static_cast<int32_t>(readlane_u32(static_cast<uint32_t>(wave_max(off)), 0));
      const int64_t mid = (static_cast<int64_t>(lo) + static_cast<int64_t>(hi)) / 2;
      org[a] = o0 + static_cast<uint32_t>(static_cast<int32_t>(mid));
      const int64_t half_extent = (static_cast<int64_t>(hi) - static_cast<int64_t>(lo)) / 2 + 1;
      near = near && half_extent <= static_cast<int64_t>(P.fast_half_extent[a]);
    }
  }
  const uint32_t ox = org[0], oy = org[1], oz = org[2];
  const float tx = fx_delta(px, ox, u0), ty = fx_delta(py, oy, u1), tz = fx_delta(pz, oz, u2);
#pragma unroll
  for (int c = 0; c < 6; ++c) ksum[w][c][lane] = 0.0f;
  auto accumulate = [&](float vx, float vy, float vz) {
    const float v[3] = {vx, vy, vz};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      float sum = ksum[w][c][lane], comp = ksum[w][3 + c][lane];
      kahan_add(sum, comp, v[c]);
      ksum[w][c][lane] = sum;
      ksum[w][3 + c][lane] = comp;
    }
  };

  // source -> window record, and window record -> separation from this lane
  auto stage_record = [&]<bool NEAR>(const uint4& sv, float mj) -> float4 {
    if constexpr (NEAR)
      return make_float4(fx_delta(sv.x, ox, u0), fx_delta(sv.y, oy, u1), fx_delta(sv.z, oz, u2), mj);
    else
      return make_float4(__uint_as_float(sv.x), __uint_as_float(sv.y), __uint_as_float(sv.z), mj);
  };
  auto separation = [&]<bool NEAR>(const float4& sj, float& dx, float& dy, float& dz) {
    if constexpr (NEAR) {
      dx = sj.x - tx;
      dy = sj.y - ty;
      dz = sj.z - tz;
    } else {
      dx = fx_delta(__float_as_uint(sj.x), px, u0);
      dy = fx_delta(__float_as_uint(sj.y), py, u1);
      dz = fx_delta(__float_as_uint(sj.z), pz, u2);
    }
  };

  uint32_t pend = 0;  // wave-uniform count of sources in the partial sums
  float psx = 0.0f, psy = 0.0f, psz = 0.0f;  // partial pair sums since the last fold
  auto fold = [&]() {
    const float gm = P.force_scale;
    accumulate(psx * gm, psy * gm, psz * gm);
    psx = psy = psz = 0.0f;
    pend = 0;
    if (lane == 0) ++cnt[7];
  };

  // the residual pair kernel against the cn staged sources; UMASS: every
  // source has the uniform mass, which the force scale already carries; lanes
  // with a negative cutoff (they pruned the leaf or accepted an ancestor) drop
  // their terms
  auto pairs = [&]<bool NEAR, bool UMASS>(uint32_t c0, uint32_t cn, float lim) {
    float lx = 0.0f, ly = 0.0f, lz = 0.0f;
#pragma unroll 4
    for (uint32_t si = 0; si < cn; ++si) {
      const float4 sj = win[w][si];
      float dx, dy, dz;
      separation.template operator()<NEAR>(sj, dx, dy, dz);
      const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));  // = table coordinate
      const float rinv = __builtin_amdgcn_rsqf(r2 + eps2);
      const float soft = rinv * rinv * rinv;
      const int ci = static_cast<int>(fminf(r2, static_cast<float>(kHTableCells - 1)));
      const float fu = __builtin_amdgcn_fractf(r2);
      const float4 c = htab[ci];
      const float hcoef = fmaf(fmaf(fmaf(c.w, fu, c.z), fu, c.y), fu, c.x);
      float fr = fmaf(-hcoef, c8, soft);
      if constexpr (!UMASS) fr *= sj.w;
      // The target itself has r2 == 0 exactly (same fixed-point value), as
      // does any coincident source: its term is exactly zero (dx = dy = dz = 0
      // against a finite softened value). Coincident sources are counted as
      // the reference does.
      const bool pair = r2 <= lim;
      const bool distinct = pair && (r2 != 0.0f || (c0 + si) != tp);
      cnt[2] += distinct;
      nearest = distinct ? fminf(nearest, r2) : nearest;
      const float f = pair ? fr : 0.0f;
      lx = fmaf(f, dx, lx);
      ly = fmaf(f, dy, ly);
      lz = fmaf(f, dz, lz);
    }
    psx += lx;
    psy += ly;
    psz += lz;
  };

  // Strict acceptance of internal node n (cell centre and half from g) for
  // this lane, with the COM separation it needs left in mf*. Nodes with
  // h >= 0.041 r_cut are never accepted (2h/r < 0.08 with r inside r_cut), so
  // the caller skips the test for them.
  const MixFrame F{s0, s1, s2, to_len, inv_len, contain2, theta2};
  auto accepts = [&](uint32_t n, const NodeGeo32& g, float& mfx, float& mfy, float& mfz) -> bool {
    return strict_accept32(P, F, g, node_mom[n], node_quad, n, px, py, pz, mfx, mfy, mfz);
  };

  // The evaluating walk prunes against each node's tight particle box. Every
  // pair inside r_cut still lies in a kept leaf, and a node the reference
  // accepts as a multipole (its whole cell inside r_cut) is always kept, so
  // the pairs and multipoles are the reference's; only nodes whose particles
  // all lie beyond r_cut are skipped earlier than with the octree cells.
  auto walk = [&]<bool NEAR>(uint32_t end) {
    uint32_t n = wave_min_u32(nxt);
    while (n < end) {
      if (lane == 0) ++cnt[5];
      const NodeLink lk = node_link[n];
      const NodeBox32 b = node_box[n];
      const bool act = nxt == n;
      if (!__ballot(act)) {
        if (lane == 0) atomicOr(&counters[kFaultSlot], 1ull);
        break;
      }
      const float ax_ = fabsf(fx_delta(b.cx, px, s0)), ay_ = fabsf(fx_delta(b.cy, py, s1)),
                  az_ = fabsf(fx_delta(b.cz, pz, s2));
      const float ex = fmaxf(0.0f, ax_ - b.hx), ey = fmaxf(0.0f, ay_ - b.hy), ez = fmaxf(0.0f, az_ - b.hz);
      const bool keep = act && !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > prune2);
      if (lk.child_count == 0) {
        // a leaf's subtree is itself: every waiting lane moves on to n + 1,
        // so that is the wave's next node too
        nxt = act ? n + 1 : nxt;
        if (__ballot(keep)) {
          const float lim = keep ? rc2 : -1.0f;
          const uint32_t e0 = lk.begin + lk.count;
          for (uint32_t c0 = lk.begin; c0 < e0; c0 += kWindow) {
            const uint32_t cn = e0 - c0 < static_cast<uint32_t>(kWindow) ? e0 - c0 : static_cast<uint32_t>(kWindow);
            if (lane == 0) cnt[6] += cn;
            if (pend + cn > static_cast<uint32_t>(kWindow)) fold();
            pend += cn;
            {
              const uint4 sv = D.src32[c0 + (static_cast<uint32_t>(lane) < cn ? lane : 0)];
              const float mj = D.uniform_mass ? 1.0f : __uint_as_float(sv.w);
              if (static_cast<uint32_t>(lane) < cn) win[w][lane] = stage_record.template operator()<NEAR>(sv, mj);
            }
            __builtin_amdgcn_wave_barrier();
            if (D.uniform_mass) pairs.template operator()<NEAR, true>(c0, cn, lim);
            else pairs.template operator()<NEAR, false>(c0, cn, lim);
            __builtin_amdgcn_wave_barrier();
          }
        }
        ++n;
        continue;
      }
      nxt = (act && !keep) ? n + lk.skip : nxt;
      if (__ballot(keep)) {
        bool take_mp = false;
        float mfx = 0.0f, mfy = 0.0f, mfz = 0.0f;
        if (b.cell_half < P.accept_half_max) {
          if (keep) take_mp = accepts(n, node_geo[n], mfx, mfy, mfz);
        }
        if (keep) nxt = take_mp ? n + lk.skip : n + 1;
        if (__ballot(take_mp) && take_mp) {
          float cx = 0.0f, cy = 0.0f, cz = 0.0f;
          node_accel32(node_mom[n], node_quad[n], mfx, mfy, mfz, P, cx, cy, cz);
          accumulate(cx, cy, cz);
        }
      }
      n = next_node(n, nxt);
    }
  };

  if (near) walk.template operator()<true>(node_count);
  else walk.template operator()<false>(node_count);
  fold();

  // Replay the reference's walk over the octree cells (no pair work) for its
  // per-target node counters.
  {
    const float cell_prune2 = P.cell_prune2_sep;
    uint32_t cnxt = valid ? 0u : node_count;
    uint32_t n = wave_min_u32(cnxt);
    while (n < node_count) {
      const NodeLink lk = node_link[n];
      const NodeGeo32 g = node_geo[n];
      const bool act = cnxt == n;
      if (!__ballot(act)) break;  // reported by the evaluating walk
      cnt[0] += act;
      const float h = g.half * inv_len;
      const float ax_ = fabsf(fx_delta(g.cx, px, s0)), ay_ = fabsf(fx_delta(g.cy, py, s1)),
                  az_ = fabsf(fx_delta(g.cz, pz, s2));
      const float ex = fmaxf(0.0f, ax_ - h), ey = fmaxf(0.0f, ay_ - h), ez = fmaxf(0.0f, az_ - h);
      const bool keep = act && !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > cell_prune2);
      cnt[1] += act && !keep;
      if (lk.child_count == 0) {
        cnt[4] += keep;
        cnxt = act ? n + 1 : cnxt;
        ++n;
        continue;
      }
      cnxt = (act && !keep) ? n + lk.skip : cnxt;
      bool take_mp = false;
      if (keep && g.half < P.accept_half_max) {
        float mfx, mfy, mfz;
        take_mp = accepts(n, g, mfx, mfy, mfz);
      }
      cnt[3] += take_mp;
      if (keep) cnxt = take_mp ? n + lk.skip : n + 1;
      n = next_node(n, cnxt);
    }
  }

  flush_counters(counters, cnt);
  if (!valid) return;
  const float ax = ksum[w][0][lane] - ksum[w][3][lane];
  const float ay = ksum[w][1][lane] - ksum[w][4][lane];
  const float az = ksum[w][2][lane] - ksum[w][5][lane];
  static_cast<float*>(out.ax)[slot] = gx + ax;
  static_cast<float*>(out.ay)[slot] = gy + ay;
  static_cast<float*>(out.az)[slot] = gz + az;
  if (out.pm_x) {
    static_cast<float*>(out.pm_x)[slot] = gx;
    static_cast<float*>(out.pm_y)[slot] = gy;
    static_cast<float*>(out.pm_z)[slot] = gz;
  }
  const uint32_t row = D.order[tp];
  if (out.sr_x) {
    static_cast<float*>(out.sr_x)[row] = ax;
    static_cast<float*>(out.sr_y)[row] = ay;
    static_cast<float*>(out.sr_z)[row] = az;
  }
  if (out.near2) static_cast<float*>(out.near2)[row] = nearest * P.tab_to_len2;
}


// ---- box-classified traversal -----------------------------------------------------
// The timed strict walks traverse the tree once per segment of consecutive
// visit-ordered targets, against the segment's target box. A segment is a
// power-of-two run of T targets inside a wave's targets: the whole run when
// its box fits (half-extents up to box_half_max), else halves of it, down to
// single targets, so a run that straddles a jump of the space-filling curve
// costs two or three compact traversals instead of a lane-by-lane walk of the
// union of distant neighbourhoods. The 64 lanes are T targets times 64 / T
// source slices: every lane sums its slice of the staged sources for its
// target, and the slices are added at the end. Small target sets launch fewer
// targets per wave, so that they still fill the chip.
//
// Traversal: breadth-first records (WalkNode) keep a node's children
// consecutive. The wave pops eight opened nodes from an LDS stack and its
// lanes test their children with one load each; kept children are pushed,
// kept leaves listed. A 256^3 walk visits about 500 nodes per wave, which
// took one dependent load and a scalar chain for each of some 100 windows of
// consecutive preorder nodes (11 of the walk's 24 ms); eight nodes per step
// take 15 to 20 loads. The stack pops one node per step above kBoxWide
// entries, so it never holds more than kBoxWide + 56 + 7 * 21 + 8 entries.
//
// Listed leaves are expanded 64 sources at a time: the leaves' source counts
// are scanned across the lanes, each leaf marks its first slot of the batch,
// and a running maximum spreads the leaf over its slots. The next batch's
// records are in flight while the current one is culled and evaluated.
constexpr uint32_t kBoxGroup = 16;     // FP64: targets per evaluation group, a DPP row
constexpr uint32_t kBoxWindow = 128;   // records staged between evaluations
constexpr uint32_t kBoxList = 80;      // 64 records in up to 16 slices, one slot of padding each (LDS banks)
// FP64: half-extent in r_cut up to which a segment stays one group. The value
// hardly matters: with 0.15 and 0.6 solves of 96^3, VJPs of 64^3 and steps of
// 32^3 take the time they take with 0.3, to 1 %.
constexpr float kBoxCompact = 0.3f;
constexpr int kBoxWide = 96;
constexpr int kBoxStack = kBoxWide + 56 + 7 * 21 + 13;

struct BoxLds {
  uint32_t stack[kBoxStack];
  uint32_t leaf[2 * kWave];
  uint32_t mark[kWave];
};

// Target box of a segment in fixed point: centre, half-extents in separation
// units (they cover every target's fixed-point position), the node tests'
// scales and cutoffs.
struct BoxFrame {
  uint32_t ox, oy, oz;
  float hx, hy, hz;
  float s0, s1, s2;
  float prune2;
  float accept_half_max;  // no acceptance for cells of this half size or more (length)
  float to_len;
};

// centre and half-extent of v over this lane's row of 16 lanes (all active);
// the half-extent covers the rounding of the centre
__device__ __forceinline__ void row_bounds(float v, float& centre, float& half) {
  auto step = [](float x, uint32_t y, bool mx) {
    const float o = __uint_as_float(y);
    return mx ? fmaxf(x, o) : fminf(x, o);
  };
#define CHUI_ROW(ctrl)                                                                                          \
  {                                                                                                             \
    const uint32_t a_ = __float_as_uint(lo), b_ = __float_as_uint(hi);                                          \
    lo = step(lo, CHUI_DPP(a_, ctrl, 0xf, a_), false);                                                          \
    hi = step(hi, CHUI_DPP(b_, ctrl, 0xf, b_), true);                                                           \
  }
  float lo = v, hi = v;
  CHUI_ROW(0x121)  // row_ror:1
  CHUI_ROW(0x122)  // row_ror:2
  CHUI_ROW(0x124)  // row_ror:4
  CHUI_ROW(0x128)  // row_ror:8
#undef CHUI_ROW
  centre = 0.5f * (lo + hi);
  half = fmaxf(hi - centre, centre - lo);
}
__device__ __forceinline__ uint32_t lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
}

// Walks the tree (breadth-first records nodes, root 0) for one box. Wave-
// uniform control flow throughout.
//   load(j)        the source record of tree position j (any valid j)
//   take(rec, on, last)  one batch of up to 64 records, `on` marking the lanes
//                  with one; last: no batch follows
//   candidate(pre, end)  an internal node [pre, end) in preorder that some
//                  target may accept: true when no target does (it is opened
//                  like any node), false when the callee has walked it
template <class Load, class Take, class Candidate>
__device__ __forceinline__ void box_traverse(const WalkNode* __restrict__ nodes, BoxLds& s, int lane,
                                             const BoxFrame& F, Load&& load, Take&& take, Candidate&& candidate) {
  const uint4* const raw = reinterpret_cast<const uint4*>(nodes);
  uint32_t sp = 0, nleaf = 0;
  // sources of the last m listed leaves; last: no leaf is left and none will come
  auto drain = [&](uint32_t m, bool last) {
    nleaf -= m;
    __builtin_amdgcn_wave_barrier();
    uint32_t begin = 0, count = 0;
    if (static_cast<uint32_t>(lane) < m) {
      const WalkNode& q = nodes[s.leaf[nleaf + lane]];
      begin = q.first;
      count = q.count;
    }
    const uint32_t incl = wave_scan_sum(count);
    const uint32_t excl = incl - count;
    const uint32_t total = readlane_u32(incl, kWave - 1);
    const uint32_t shift = begin - excl;
    uint32_t carry = 0;
    auto index = [&](uint32_t base) -> uint32_t {
      s.mark[lane] = 0;
      __builtin_amdgcn_wave_barrier();
      if (count && excl - base < static_cast<uint32_t>(kWave)) s.mark[excl - base] = static_cast<uint32_t>(lane);
      __builtin_amdgcn_wave_barrier();
      uint32_t v = s.mark[lane];
      __builtin_amdgcn_wave_barrier();
      if (lane == 0) v = v > carry ? v : carry;
      v = wave_scan_max(v);
      carry = readlane_u32(v, kWave - 1);
      const uint32_t j = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(static_cast<int>(v << 2),
                                                                            static_cast<int>(shift))) + base + lane;
      const uint32_t j0 = readlane_u32(j, 0);
      return base + lane < total ? j : j0;
    };
    auto cur = load(index(0));  // leaves are never empty: total > 0
    for (uint32_t base = 0; base < total; base += kWave) {
      const bool more = base + kWave < total;
      auto nxt = cur;
      if (more) nxt = load(index(base + kWave));
      take(cur, base + lane < total, last && !more);
      cur = nxt;
    }
  };
  // children of the top entries: lane group g = lane / 8 takes entry sp - 1 - g
  uint4 a, b, c;
  uint32_t idx = 0;
  bool in = false;
  auto pop = [&]() {
    const uint32_t m = sp > static_cast<uint32_t>(kBoxWide) ? 1u : (sp < 8u ? sp : 8u);
    const uint32_t g = static_cast<uint32_t>(lane) >> 3;
    __builtin_amdgcn_wave_barrier();
    in = g < m;
    idx = s.stack[sp - 1 - (in ? g : 0u)] + (lane & 7u);
    sp -= m;
    const uint4* r = raw + 3ull * idx;
    a = r[0];
    b = r[1];
    c = r[2];
  };
  if (lane == 0) s.stack[0] = 0;
  sp = 1;
  pop();
  bool open = true;  // a, b, c hold popped nodes
  do {
    if (open) {
      // a: cx cy cz hx | b: hy hz cell_half kids | c: first count pre skip
      const uint32_t kids = b.w;
      const uint32_t lastbits =
          static_cast<uint32_t>(__ballot(in && (kids & kLastSibling)) >> (lane & 56)) & 0xFFu;
      const bool on = in && !(lastbits & ((1u << (lane & 7)) - 1u));  // no last sibling before this lane
      const float ex = fmaxf(0.0f, fabsf(fx_delta(a.x, F.ox, F.s0)) - __uint_as_float(a.w) - F.hx);
      const float ey = fmaxf(0.0f, fabsf(fx_delta(a.y, F.oy, F.s1)) - __uint_as_float(b.x) - F.hy);
      const float ez = fmaxf(0.0f, fabsf(fx_delta(a.z, F.oz, F.s2)) - __uint_as_float(b.y) - F.hz);
      const bool keep = on && !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > F.prune2);
      const bool leaf = (kids & 0xFFu) == 0;
      bool cand = false;
      if (keep && !leaf) {
        const float h = __uint_as_float(b.z);
        if (h < F.accept_half_max) {
          // a target within 25 h of the node fails 2h/r < 0.08: no candidate
          // when the whole box (and the node's own extent) lies within 25 h
          const float dx = (fabsf(fx_delta(a.x, F.ox, F.s0)) + __uint_as_float(a.w) + F.hx) * F.to_len;
          const float dy = (fabsf(fx_delta(a.y, F.oy, F.s1)) + __uint_as_float(b.x) + F.hy) * F.to_len;
          const float dz = (fabsf(fx_delta(a.z, F.oz, F.s2)) + __uint_as_float(b.y) + F.hz) * F.to_len;
          cand = !(fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= 624.9f * h * h);
        }
      }
      const unsigned long long lm = __ballot(keep && leaf);
      if (keep && leaf) s.leaf[nleaf + lanes_below(lm)] = idx;
      nleaf += static_cast<uint32_t>(__popcll(lm));
      const unsigned long long om = __ballot(keep && !leaf && !cand);
      if (keep && !leaf && !cand) s.stack[sp + lanes_below(om)] = c.x;
      sp += static_cast<uint32_t>(__popcll(om));
      unsigned long long rest = __ballot(cand);
      while (rest) {
        const uint32_t l = static_cast<uint32_t>(__ffsll(static_cast<long long>(rest)) - 1);
        rest &= rest - 1ull;
        // the lane reads come before any branch on the lane: an inactive
        // lane's register may hold nothing (a spilled value is reloaded for
        // the active lanes only)
        const uint32_t pre = readlane_u32(c.z, l), end = pre + readlane_u32(c.w, l), child = readlane_u32(c.x, l);
        if (candidate(pre, end)) {
          if (lane == 0) s.stack[sp] = child;
          ++sp;
        }
      }
      open = sp != 0;
      if (open) pop();  // the next nodes' loads are in flight while leaves are drained
    }
    // one leaf stays listed while nodes are open, so the last drain comes last
    if (nleaf > static_cast<uint32_t>(kWave) || (!open && nleaf)) {
      const uint32_t m = nleaf < static_cast<uint32_t>(kWave) ? nleaf : static_cast<uint32_t>(kWave);
      drain(m, !open && m == nleaf);
    }
  } while (open || nleaf);
}

// Bounds of a segment [seg, seg + T) of the wave's targets: halves T until
// fits() accepts the run (a single target always fits). Wave-uniform.
template <class Fits>
__device__ __forceinline__ uint32_t box_segment(uint32_t seg, uint32_t per_wave, Fits&& fits) {
  uint32_t T = seg ? (seg & (0u - seg)) : per_wave;
  while (!fits(T) && T > 1) T >>= 1;
  return T;
}

// ---- mixed box walk ----------------------------------------------------------------
// The timed mixed walk: fused PM interpolation and the residual walk of the
// comment above walkmix_kernel, box-classified. Staged sources farther than
// r_cut from the target box (all their pairs are zero) are dropped; the rest
// are compacted into an LDS window and evaluated 64 at a time. Window slot of
// record r for S = 64 / TL slices: (r % S) (TL + 1) + r / S, so a lane's TL
// records are consecutive and the slices start in different LDS banks. The
// second half of the window takes a batch's overflow and stages the leaves of
// the lane-by-lane walks.
//
// The pairs' separations are FP32 differences of offsets from an origin (or
// fixed-point differences where the origin's targets span too much for it). In
// FP32 a pair within about 1e-7 of r_cut may fall on either side of it, and the
// residual is still 1.8e-2 of Newtonian there, so one pair moves a 32^3 box's
// force field by up to 2e-6 in relative L2 (1e-7 otherwise). Up to 2^20 sources
// the origin is that of the 64 targets that share a wave of the counting walk
// (SHARED), so the side does not depend on how the targets are cut into waves
// and segments. It may still differ from the counting walk's, whose offsets
// are scaled to other units: one pair in 6e6 of a random 2^20 box does, one in
// 6e6 of a 96^3 lattice, one in 5e5 of a 32^3 one, no fewer than with segment
// origins (65 and 64 targets, 14 and 20, 6 and 4). The errors against FP64 are
// alike too (1.2e-6 and 1.0e-6, 3.5e-6 and 2.7e-6, 1.0e-6 and 0.7e-6). Beyond,
// where single pairs do not show, the origin is the segment's centre, which the
// box test can share (256^3: 4 % of the solve). SHARED holds both forms of a
// pair: 4 waves per SIMD without spills instead of 5 with 27 registers spilled
// (eleven boxes of 32^3 to 96^3: 6.01 to 5.34 ms; one of 100003: 1083 to 1020
// us). FP64 decisions took 27 VALU instructions per pair against 16.
// With segment origins 5 waves (96 VGPRs, 11 spilled, 18 KB of LDS) are bound
// by VALU issue at 256^3: the SIMDs issue vector instructions in every cycle.
template <int SCHEME, bool CUBIC, bool LOG, int WAVES, bool FRAME, bool SHARED>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(SHARED ? 4 : 5)))
void walkmix_box_kernel(WalkParams P, WalkData D, WalkOutputs out, unsigned long long* __restrict__ counters,
                        const NodeLink* __restrict__ node_link, const NodeGeo32* __restrict__ node_geo,
                        const NodeMom32* __restrict__ node_mom, const NodeQuad32* __restrict__ node_quad,
                        const NodeBox32* __restrict__ node_box, const WalkNode* __restrict__ wnode) {
  __shared__ float4 win_all[WAVES][2 * kBoxList];
  __shared__ BoxLds box_all[WAVES];
  __shared__ float4 htab[LOG ? 1 : kHTableCells];
  extern __shared__ float4 ltab[];  // LOG: P.log_cells cells
  if constexpr (LOG) {
    for (int i = threadIdx.x; i < static_cast<int>(P.log_cells); i += (WAVES * kWave)) ltab[i] = D.ltab[i];
  } else {
    for (int i = threadIdx.x; i < kHTableCells; i += (WAVES * kWave)) htab[i] = D.htab[i];
  }
  __syncthreads();
  const uint32_t node_count = D.node_count_dev ? *D.node_count_dev : P.node_count;
  const int w = static_cast<int>(readlane_u32(threadIdx.x / kWave, 0));
  const int lane = threadIdx.x % kWave;
  float4* const win = win_all[w];
  BoxLds& lds = box_all[w];
  const uint32_t per_wave = P.targets_per_wave;
  const uint64_t k64 = (static_cast<uint64_t>(xcd_logical_block()) * WAVES + w) * per_wave;
  if (k64 >= P.n_targets || node_count == 0) return;
  const uint32_t k0 = static_cast<uint32_t>(k64);
  const uint32_t here = P.n_targets - k0 < per_wave ? P.n_targets - k0 : per_wave;  // targets of this wave
  // node tests: fixed-point units (CUBIC) or lengths
  const float s0 = CUBIC ? 1.0f : P.fx_to_len[0];
  const float s1 = CUBIC ? 1.0f : P.fx_to_len[1];
  const float s2 = CUBIC ? 1.0f : P.fx_to_len[2];
  const float to_len = CUBIC ? P.fx_to_len[0] : 1.0f;          // node separation unit -> length
  const float inv_len = CUBIC ? 1.0f / P.fx_to_len[0] : 1.0f;  // length -> node separation unit
  const float prune2 = P.prune2_sep;
  // pairs: table units (lengths * sqrt(t_to_cell), or of the residual table)
  const float u0 = P.tab_scale[0], u1 = P.tab_scale[1], u2 = P.tab_scale[2];
  const float rc2 = P.rcut2_tab;
  const float eps2 = P.eps2_tab;
  const float c8 = P.c8_tab;
  const MixFrame F{s0, s1, s2, to_len, inv_len, P.contain2_sep, static_cast<float>(P.theta * P.theta)};
  const float4* const lcell = ltab - P.log_base;
  const uint32_t lbase = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_f32x4*)ltab - P.log_base));

  // beyond r_cut of every target whose offset the origin admits (2^28 units per axis)
  const float far = 2.0f * fmaf(268435456.0f, fmaxf(u0, fmaxf(u1, u2)), sqrtf(rc2));
  // --- the origin of the 64 targets around (SHARED), else the segment's ---
  uint32_t wox = 0, woy = 0, woz = 0;
  bool wave_origin = false;
  if constexpr (!SHARED) {
    wave_origin = FRAME;
  } else {
    const uint32_t i = (k0 & ~(static_cast<uint32_t>(kWave) - 1u)) + lane;
    const bool in = i < P.n_targets;
    const uint32_t v = in ? i : k0;
    const uint4 t = D.src32[P.identity_targets ? v : D.tpos[v]];
    const uint32_t pp[3] = {t.x, t.y, t.z};
    uint32_t o[3];
    wave_origin = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t o0 = readlane_u32(pp[a], 0);
      const uint32_t off = in ? (pp[a] - o0) ^ 0x80000000u : 0x80000000u;  // ordered as unsigned
      const int32_t lo = static_cast<int32_t>(wave_min_u32(off) ^ 0x80000000u);
      const int32_t hi = static_cast<int32_t>(wave_max_u32(off) ^ 0x80000000u);
      const int64_t mid = (static_cast<int64_t>(lo) + static_cast<int64_t>(hi)) / 2;
      o[a] = o0 + static_cast<uint32_t>(static_cast<int32_t>(mid));
      const int64_t half = (static_cast<int64_t>(hi) - static_cast<int64_t>(lo)) / 2 + 1;
      wave_origin = wave_origin && half <= static_cast<int64_t>(P.fast_half_extent[a]);
    }
    wox = o[0]; woy = o[1]; woz = o[2];
  }
  for (uint32_t seg = 0; seg < here;) {
    // --- the segment and its box ---
    uint32_t px, py, pz;
    uint32_t ox = 0, oy = 0, oz = 0;
    float bh0 = 0.0f, bh1 = 0.0f, bh2 = 0.0f;  // half-extents, separation units
    float bt0 = 0.0f, bt1 = 0.0f, bt2 = 0.0f;  // the same in table units
    uint32_t T;
    if constexpr (!FRAME) {
      T = per_wave;
    } else {
      // lane i: target seg + i (the last valid one past the end)
      const uint32_t i = seg + lane < here ? seg + lane : here - 1;
      const uint4 t = D.src32[P.identity_targets ? k0 + i : D.tpos[k0 + i]];
      T = box_segment(seg, per_wave, [&](uint32_t want) -> bool {
        const bool in = static_cast<uint32_t>(lane) < want;
        const uint32_t pp[3] = {t.x, t.y, t.z};
        const float sa[3] = {s0, s1, s2};
        uint32_t o[3];
        float bh[3], bt[3];
        bool ok = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const uint32_t o0 = readlane_u32(pp[a], 0);
          // offsets from the first target, ordered as unsigned
          const uint32_t off = in ? (pp[a] - o0) ^ 0x80000000u : 0x80000000u;
          const int32_t lo = static_cast<int32_t>(wave_min_u32(off) ^ 0x80000000u);
          const int32_t hi = static_cast<int32_t>(wave_max_u32(off) ^ 0x80000000u);
          const int64_t mid = (static_cast<int64_t>(lo) + static_cast<int64_t>(hi)) / 2;
          o[a] = o0 + static_cast<uint32_t>(static_cast<int32_t>(mid));
          const int64_t half = (static_cast<int64_t>(hi) - static_cast<int64_t>(lo)) / 2 + 1;
          bh[a] = static_cast<float>(half + 1) * sa[a];
          bt[a] = static_cast<float>(half + 1) * P.tab_scale[a];
          ok = ok && half <= static_cast<int64_t>(P.fast_half_extent[a]) && bh[a] <= P.box_half_max[a];
        }
        ox = o[0]; oy = o[1]; oz = o[2];
        bh0 = bh[0]; bh1 = bh[1]; bh2 = bh[2];
        bt0 = bt[0]; bt1 = bt[1]; bt2 = bt[2];
        return ok;
      });
    }
    // T targets as TL columns (at least 4) and 64 / TL source slices
    const uint32_t TL = T < 4u ? 4u : T;
    const uint32_t lgT = 31u - static_cast<uint32_t>(__builtin_clz(TL));
    const uint32_t lgS = 6u - lgT;
    const uint32_t col = static_cast<uint32_t>(lane) & (TL - 1u), slice = static_cast<uint32_t>(lane) >> lgT;
    const bool valid = col < T && seg + col < here;
    const uint32_t k = k0 + seg + (valid ? col : 0u);
    const uint32_t tp = P.identity_targets ? k : D.tpos[k];
    {
      const uint4 t = D.src32[tp];
      px = t.x;
      py = t.y;
      pz = t.z;
    }
    if constexpr (!SHARED) {
      wox = ox;
      woy = oy;
      woz = oz;
    }
    const float tx = fx_delta(px, wox, u0), ty = fx_delta(py, woy, u1), tz = fx_delta(pz, woz, u2);
    float sum[3] = {0.0f, 0.0f, 0.0f}, comp[3] = {0.0f, 0.0f, 0.0f};  // Kahan totals of this lane's slice
    auto accumulate = [&](float vx, float vy, float vz) {
      kahan_add(sum[0], comp[0], vx);
      kahan_add(sum[1], comp[1], vy);
      kahan_add(sum[2], comp[2], vz);
    };
    uint32_t pend = 0;                         // sources in this lane's partial sums (wave-uniform)
    float psx = 0.0f, psy = 0.0f, psz = 0.0f;  // partial pair sums since the last fold
    auto fold = [&]() {
      const float gm = P.force_scale;
      accumulate(psx * gm, psy * gm, psz * gm);
      psx = psy = psz = 0.0f;
      pend = 0;
    };
    auto stage_record = [&]<bool NEAR>(const uint4& sv, float mj) -> float4 {
      if constexpr (NEAR)
        return make_float4(fx_delta(sv.x, wox, u0), fx_delta(sv.y, woy, u1), fx_delta(sv.z, woz, u2), mj);
      else
        return make_float4(__uint_as_float(sv.x), __uint_as_float(sv.y), __uint_as_float(sv.z), mj);
    };
    // One pair term; NEAR: offsets from the origin, else fixed point.
    // UMASS: the force scale carries the mass. SEL: lanes with a negative
    // cutoff drop the term.
    auto pair = [&]<bool NEAR, bool UMASS, bool SEL>(const float4& sj, float lim, float& lx, float& ly, float& lz) {
      float dx, dy, dz;
      if constexpr (NEAR) {
        dx = sj.x - tx;
        dy = sj.y - ty;
        dz = sj.z - tz;
      } else {
        dx = fx_delta(__float_as_uint(sj.x), px, u0);
        dy = fx_delta(__float_as_uint(sj.y), py, u1);
        dz = fx_delta(__float_as_uint(sj.z), pz, u2);
      }
      float f;
      if constexpr (LOG) {
        // s = r^2 + eps^2 clamped to [0, 1]: s >= eps^2 >= 2^first_octave, and
        // s = 1 (r_cut and beyond) is the zero cell
        float sc = __builtin_amdgcn_fmed3f(fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2))), 0.0f, 1.0f);
        const uint32_t bits = __float_as_uint(sc);
        const float4 c = lcell[bits >> kLogMantissaShift];
        const float u = static_cast<float>(bits & ((1u << kLogMantissaShift) - 1u));
        float fr = fmaf(fmaf(fmaf(c.w, u, c.z), u, c.y), u, c.x);
        if constexpr (!UMASS) fr *= sj.w;
        f = (SEL && lim < 0.0f) ? 0.0f : fr;
      } else {
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));  // = table coordinate
        const float rinv = __builtin_amdgcn_rsqf(r2 + eps2);
        const float soft = rinv * rinv * rinv;
        const int ci = static_cast<int>(fminf(r2, static_cast<float>(kHTableCells - 1)));
        const float fu = __builtin_amdgcn_fractf(r2);
        const float4 c = htab[ci];
        const float hcoef = fmaf(fmaf(fmaf(c.w, fu, c.z), fu, c.y), fu, c.x);
        float fr = fmaf(-hcoef, c8, soft);
        if constexpr (!UMASS) fr *= sj.w;
        // the target itself (and any coincident source) has r2 == 0 exactly:
        // zero separation against a finite softened value
        f = r2 <= lim ? fr : 0.0f;
      }
      lx = fmaf(f, dx, lx);
      ly = fmaf(f, dy, ly);
      lz = fmaf(f, dz, lz);
    };
    // the cn leaf sources staged in the second half (lane-by-lane walks)
    auto leaf_pairs = [&]<bool NEAR, bool UMASS>(uint32_t cn, float lim) {
      float lx = 0.0f, ly = 0.0f, lz = 0.0f;
#pragma unroll 2
      for (uint32_t si = 0; si < cn; ++si)
        pair.template operator()<NEAR, UMASS, true>(win[kBoxList + si], lim, lx, ly, lz);
      psx += lx;
      psy += ly;
      psz += lz;
    };
    // Strict acceptance of internal node n for this lane, with the COM
    // separation it needs left in mf*.
    auto accepts = [&](uint32_t n, const NodeGeo32& g, float& mfx, float& mfy, float& mfz) -> bool {
      return strict_accept32(P, F, g, node_mom[n], node_quad, n, px, py, pz, mfx, mfy, mfz);
    };
    // Lane-by-lane walk of the preorder range [nxt, end) (walkmix_kernel's
    // walk): candidate subtrees, and whole walks without a box frame.
    uint32_t nxt = 0;
    auto walk = [&]<bool NEAR>(uint32_t end) {
      uint32_t n = wave_min_u32(nxt);
      while (n < end) {
        const NodeLink lk = node_link[n];
        const NodeBox32 b = node_box[n];
        const bool act = nxt == n;
        if (!__ballot(act)) {
          if (lane == 0) atomicOr(&counters[kFaultSlot], 1ull);
          break;
        }
        const float ax_ = fabsf(fx_delta(b.cx, px, s0)), ay_ = fabsf(fx_delta(b.cy, py, s1)),
                    az_ = fabsf(fx_delta(b.cz, pz, s2));
        const float ex = fmaxf(0.0f, ax_ - b.hx), ey = fmaxf(0.0f, ay_ - b.hy), ez = fmaxf(0.0f, az_ - b.hz);
        const bool keep = act && !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > prune2);
        if (lk.child_count == 0) {
          // a leaf's subtree is itself: every waiting lane moves on to n + 1,
          // so that is the wave's next node too
          nxt = act ? n + 1 : nxt;
          if (__ballot(keep)) {
            const float lim = keep ? rc2 : -1.0f;
            const uint32_t e0 = lk.begin + lk.count;
            for (uint32_t c0 = lk.begin; c0 < e0; c0 += kWindow) {
              const uint32_t cn = e0 - c0 < static_cast<uint32_t>(kWindow) ? e0 - c0 : static_cast<uint32_t>(kWindow);
              if (pend + cn > static_cast<uint32_t>(kWindow)) fold();
              pend += cn;
              const uint4 sv = D.src32[c0 + (static_cast<uint32_t>(lane) < cn ? lane : 0)];
              const float mj = D.uniform_mass ? 1.0f : __uint_as_float(sv.w);
              if (static_cast<uint32_t>(lane) < cn)
                win[kBoxList + lane] = stage_record.template operator()<NEAR>(sv, mj);
              __builtin_amdgcn_wave_barrier();
              if (D.uniform_mass) leaf_pairs.template operator()<NEAR, true>(cn, lim);
              else leaf_pairs.template operator()<NEAR, false>(cn, lim);
              __builtin_amdgcn_wave_barrier();
            }
          }
          ++n;
          continue;
        }
        nxt = (act && !keep) ? n + lk.skip : nxt;
        if (__ballot(keep)) {
          bool take_mp = false;
          float mfx = 0.0f, mfy = 0.0f, mfz = 0.0f;
          if (b.cell_half < P.accept_half_max) {
            if (keep) take_mp = accepts(n, node_geo[n], mfx, mfy, mfz);
          }
          if (keep) nxt = take_mp ? n + lk.skip : n + 1;
          if (__ballot(take_mp) && take_mp) {
            float cx = 0.0f, cy = 0.0f, cz = 0.0f;
            node_accel32(node_mom[n], node_quad[n], mfx, mfy, mfz, P, cx, cy, cz);
            accumulate(cx, cy, cz);
          }
        }
        n = next_node(n, nxt);
      }
    };
    const bool owner = valid && slice == 0;  // the lane-by-lane walks run on the first slice
    if constexpr (FRAME) {
      // a source whose offset from the box centre lies beyond r_cut of the box
      // (outside half-extent + 1 fixed-point unit per axis) is beyond r_cut of
      // every target; the 1e-5 margin covers the rounding of the offsets, so
      // every dropped source is one whose pairs are all zero
      const float cull2 = rc2 * 1.00001f;
      // SHARED: the box centre in the origin's frame; the offsets there reach
      // L/16 + r_cut, so their roundings may take 3e-7 of that off the gap
      float obx = 0.0f, oby = 0.0f, obz = 0.0f;
      if (SHARED && wave_origin) {
        obx = fx_delta(ox, wox, u0);
        oby = fx_delta(oy, woy, u1);
        obz = fx_delta(oz, woz, u2);
        const float far_r = sqrtf(rc2);
        bt0 += 6.0e-7f * (268435456.0f * u0 + far_r);
        bt1 += 6.0e-7f * (268435456.0f * u1 + far_r);
        bt2 += 6.0e-7f * (268435456.0f * u2 + far_r);
      }
      uint32_t wn = 0;  // records in the window, below kWindow between batches
      const float4* const mine = win + slice * (TL + 1u);
      // iters records of every slice (a multiple of 4)
      auto window_pairs = [&]<bool NEAR, bool UMASS>(uint32_t iters) {
        float lx = 0.0f, ly = 0.0f, lz = 0.0f;
        if constexpr (LOG) {
          // two table reads in flight before their polynomials are evaluated
          for (uint32_t i0 = 0; i0 < iters; i0 += 4) {
#pragma unroll
            for (int h = 0; h < 4; h += kPairGroup) {
              float dx[kPairGroup], dy[kPairGroup], dz[kPairGroup], mj[kPairGroup];
              uint32_t bits[kPairGroup];
              float4 c[kPairGroup];
#pragma unroll
              for (int q = 0; q < kPairGroup; ++q) {
                const float4 sj = mine[i0 + h + q];
                mj[q] = sj.w;
                dx[q] = NEAR ? sj.x - tx : fx_delta(__float_as_uint(sj.x), px, u0);
                dy[q] = NEAR ? sj.y - ty : fx_delta(__float_as_uint(sj.y), py, u1);
                dz[q] = NEAR ? sj.z - tz : fx_delta(__float_as_uint(sj.z), pz, u2);
                bits[q] = __float_as_uint(__builtin_amdgcn_fmed3f(
                    fmaf(dx[q], dx[q], fmaf(dy[q], dy[q], fmaf(dz[q], dz[q], eps2))), 0.0f, 1.0f));
              }
#pragma unroll
              for (int q = 0; q < kPairGroup; ++q) c[q] = lds_cell(lbase, bits[q] >> kLogMantissaShift);
#pragma unroll
              for (int q = 0; q < kPairGroup; ++q) {
                const float u = static_cast<float>(bits[q] & ((1u << kLogMantissaShift) - 1u));
                float fr = fmaf(fmaf(fmaf(c[q].w, u, c[q].z), u, c[q].y), u, c[q].x);
                if constexpr (!UMASS) fr *= mj[q];
                lx = fmaf(fr, dx[q], lx);
                ly = fmaf(fr, dy[q], ly);
                lz = fmaf(fr, dz[q], lz);
              }
            }
          }
        } else {
#pragma unroll 4
          for (uint32_t i0 = 0; i0 < iters; ++i0)
            pair.template operator()<NEAR, UMASS, false>(mine[i0], rc2, lx, ly, lz);
        }
        psx += lx;
        psy += ly;
        psz += lz;
      };
      // every lane sums its slice of the first cn records (pairs beyond r_cut
      // are zero; lanes without a target are never written out)
      auto evaluate = [&](uint32_t cn) {
        __builtin_amdgcn_wave_barrier();
        const uint32_t iters = (((cn + (1u << lgS) - 1u) >> lgS) + 3u) & ~3u;
        if (pend + iters > static_cast<uint32_t>(kWindow)) fold();
        pend += iters;
        if (!SHARED || wave_origin) {
          if (D.uniform_mass) window_pairs.template operator()<true, true>(iters);
          else window_pairs.template operator()<true, false>(iters);
        } else if (D.uniform_mass) {
          window_pairs.template operator()<false, true>(iters);
        } else {
          window_pairs.template operator()<false, false>(iters);
        }
        __builtin_amdgcn_wave_barrier();
      };
      auto slot_of = [&](uint32_t r) -> uint32_t {
        const uint32_t q = r & (kWindow - 1u);
        return (r >= static_cast<uint32_t>(kWindow) ? kBoxList : 0u) + (q & ((1u << lgS) - 1u)) * (TL + 1u) + (q >> lgS);
      };
      const BoxFrame frame{ox, oy, oz, bh0, bh1, bh2, s0, s1, s2, prune2, P.quad ? P.accept_half_max : 0.0f, to_len};
      box_traverse(
          wnode, lds, lane, frame, [&](uint32_t j) -> uint4 { return D.src32[j]; },
          [&](const uint4& sv, bool on, bool last) {
            const float mj = D.uniform_mass ? 1.0f : __uint_as_float(sv.w);
            const float4 rec = !SHARED || wave_origin ? stage_record.template operator()<true>(sv, mj)
                                           : stage_record.template operator()<false>(sv, mj);
            const float ex = fmaxf(fabsf(!SHARED ? rec.x : wave_origin ? rec.x - obx : fx_delta(sv.x, ox, u0)) - bt0, 0.0f);
            const float ey = fmaxf(fabsf(!SHARED ? rec.y : wave_origin ? rec.y - oby : fx_delta(sv.y, oy, u1)) - bt1, 0.0f);
            const float ez = fmaxf(fabsf(!SHARED ? rec.z : wave_origin ? rec.z - obz : fx_delta(sv.z, oz, u2)) - bt2, 0.0f);
            const bool keep = on && !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > cull2);
            const unsigned long long km = __ballot(keep);
            __builtin_amdgcn_wave_barrier();
            if (keep) win[slot_of(wn + lanes_below(km))] = rec;
            wn += static_cast<uint32_t>(__popcll(km));
            while (wn >= static_cast<uint32_t>(kWindow) || (last && wn)) {
              const uint32_t cn = wn < static_cast<uint32_t>(kWindow) ? wn : static_cast<uint32_t>(kWindow);
              if (static_cast<uint32_t>(lane) >= cn) {
                // dummies beyond r_cut of every target fill the last window (in
                // fixed point half a period from the box centre per axis)
                win[slot_of(lane)] = !SHARED || wave_origin ? make_float4(far, far, far, 0.0f)
                                                 : make_float4(__uint_as_float(ox ^ 0x80000000u),
                                                               __uint_as_float(oy ^ 0x80000000u),
                                                               __uint_as_float(oz ^ 0x80000000u), 0.0f);
              }
              evaluate(cn);
              wn -= cn;
              // the records past the window move to its front, same slots
              const uint32_t at = slot_of(lane);
              win[at] = win[kBoxList + at];
            }
          },
          [&](uint32_t pre, uint32_t end) -> bool {
            float mx, my, mz;
            if (!__ballot(owner && accepts(pre, node_geo[pre], mx, my, mz))) return true;
            nxt = owner ? pre : end;
            if (!SHARED || wave_origin) walk.template operator()<true>(end);
            else walk.template operator()<false>(end);
            return false;
          });
    } else {
      nxt = owner ? 0u : node_count;
      walk.template operator()<false>(node_count);
    }
    fold();
    // --- slices -> targets ---
    double tot[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) tot[a] = static_cast<double>(sum[a]) - static_cast<double>(comp[a]);
    for (uint32_t o = TL; o < static_cast<uint32_t>(kWave); o <<= 1) {
#pragma unroll
      for (int a = 0; a < 3; ++a) tot[a] += __shfl_xor(tot[a], static_cast<int>(o), kWave);
    }
    if (owner) {
      const float ax = static_cast<float>(tot[0]), ay = static_cast<float>(tot[1]), az = static_cast<float>(tot[2]);
      float gx = 0.0f, gy = 0.0f, gz = 0.0f;
      if (P.pm_enabled) interp32<SCHEME>(P, D.f32x, D.f32y, D.f32z, px, py, pz, gx, gy, gz);
      const uint32_t row = D.order[tp];
      const uint32_t slot = P.identity_targets ? row : D.tslot[k];
      static_cast<float*>(out.ax)[slot] = gx + ax;
      static_cast<float*>(out.ay)[slot] = gy + ay;
      static_cast<float*>(out.az)[slot] = gz + az;
      if (out.pm_x) {
        static_cast<float*>(out.pm_x)[slot] = gx;
        static_cast<float*>(out.pm_y)[slot] = gy;
        static_cast<float*>(out.pm_z)[slot] = gz;
      }
      if (out.sr_x) {
        static_cast<float*>(out.sr_x)[row] = ax;
        static_cast<float*>(out.sr_y)[row] = ay;
        static_cast<float*>(out.sr_z)[row] = az;
      }
    }
    seg += T;
  }
}

// ---- mixed walk, one target per wave --------------------------------------------
// For sparse active sets the 64 targets of a walkmix_kernel wave lie far
// apart, and the wave walks the union of 64 distant neighbourhoods. Here a
// wave serves one target. Its lanes classify 64 consecutive preorder nodes at
// a time with walkmix_kernel's tests (the cutoff prune against the tight
// particle boxes, strict_accept32 for internal nodes whose cell is small
// enough), follow the visited chain through that window, list the kept
// leaves' sources and the accepted nodes in LDS and evaluate the lists 64
// entries at a time with walkmix_kernel's pair and multipole arithmetic. The
// pairs and multipoles are walkmix_kernel's; per-lane partial sums are
// reduced in FP64 at the end.
constexpr int kTargetList = 1024;  // listed sources per wave before an evaluation
constexpr int kTargetNodes = 128;  // listed multipoles per wave before an evaluation

// The tree walk of the per-wave kernels: the lanes classify preorder nodes
// p .. p + 63 (classify(q, next, lb, lc) returns 0 pruned, 1 kept leaf with
// sources [lb, lb + lc), 2 accepted node or 3 opened, and sets next to q + 1
// to descend or q + skip to move past the subtree), a scalar loop follows the
// visited chain through the window with readlane, and the chain's kept
// leaves' sources and accepted nodes are appended to the wave's LDS lists
// (list: kTargetList entries, mps: kTargetNodes). evaluate() consumes the
// lists and resets nl and nm; it runs whenever a list would overflow and at
// the end.
template <class Classify, class Evaluate>
__device__ __forceinline__ void walk_target_wave(uint32_t node_count, int lane, uint32_t* list, uint32_t* mps,
                                                 uint32_t& nl, uint32_t& nm, Classify&& classify,
                                                 Evaluate&& evaluate) {
  const unsigned long long below = (1ull << lane) - 1ull;
  uint32_t p = 0;
  while (p < node_count) {
    const uint32_t q = p + lane;
    uint32_t next = q + 1, lb = 0, lc = 0;
    const int kind = q < node_count ? classify(q, next, lb, lc) : 3;
    unsigned long long chain = 0;
    uint32_t cur = p;
    while (cur < p + kWave && cur < node_count) {
      const uint32_t l = cur - p;
      chain |= 1ull << l;
      cur = readlane_u32(next, l);
    }
    p = cur;
    const bool on = (chain >> lane) & 1ull;
    const unsigned long long mm = __ballot(on && kind == 2);
    if (nm + static_cast<uint32_t>(__popcll(mm)) > static_cast<uint32_t>(kTargetNodes)) evaluate();
    if (on && kind == 2) mps[nm + __popcll(mm & below)] = q;
    nm += __popcll(mm);
    unsigned long long rest = __ballot(on && kind == 1);
    while (rest) {
      const uint32_t l = static_cast<uint32_t>(__ffsll(static_cast<long long>(rest)) - 1);
      rest &= rest - 1ull;
      const uint32_t b0 = readlane_u32(lb, l), c = readlane_u32(lc, l);
      for (uint32_t c0 = 0; c0 < c; c0 += kWave) {
        const uint32_t cn = c - c0 < static_cast<uint32_t>(kWave) ? c - c0 : static_cast<uint32_t>(kWave);
        if (nl + cn > static_cast<uint32_t>(kTargetList)) evaluate();
        if (static_cast<uint32_t>(lane) < cn) list[nl + lane] = b0 + c0 + lane;
        nl += cn;
      }
    }
  }
  evaluate();
}

template <int SCHEME, bool CUBIC>
__global__ __launch_bounds__(kWalkThreads) void walkmix_target_kernel(WalkParams P, WalkData D, WalkOutputs out) {
  __shared__ float4 htab[kHTableCells];
  __shared__ uint32_t list[kWalkWaves][kTargetList];
  __shared__ uint32_t mps[kWalkWaves][kTargetNodes];
  for (int i = threadIdx.x; i < kHTableCells; i += kWalkThreads) htab[i] = D.htab[i];
  __syncthreads();
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const uint32_t k = xcd_logical_block() * kWalkWaves + w;
  if (k >= P.n_targets) return;  // wave-uniform; no block barrier follows
  const uint32_t tp = P.identity_targets ? k : D.tpos[k];
  const uint32_t slot = P.identity_targets ? D.order[k] : D.tslot[k];
  const uint4 t = D.src32[tp];
  const uint32_t px = t.x, py = t.y, pz = t.z;
  const float s0 = CUBIC ? 1.0f : P.fx_to_len[0];
  const float s1 = CUBIC ? 1.0f : P.fx_to_len[1];
  const float s2 = CUBIC ? 1.0f : P.fx_to_len[2];
  const float to_len = CUBIC ? P.fx_to_len[0] : 1.0f;
  const float inv_len = CUBIC ? 1.0f / P.fx_to_len[0] : 1.0f;
  const MixFrame F{s0, s1, s2, to_len, inv_len, P.contain2_sep, static_cast<float>(P.theta * P.theta)};
  const float prune2 = P.prune2_sep;
  const float u0 = P.tab_scale[0], u1 = P.tab_scale[1], u2 = P.tab_scale[2];
  const float rc2 = P.rcut2_tab, eps2 = P.eps2_tab, c8 = P.c8_tab;

  float lx = 0.0f, ly = 0.0f, lz = 0.0f;  // pair sums (force-scale units)
  float mx = 0.0f, my = 0.0f, mz = 0.0f;  // multipole accelerations
  uint32_t nl = 0, nm = 0;
  auto evaluate = [&]() {
    __builtin_amdgcn_wave_barrier();
    for (uint32_t e = lane; e < nl; e += kWave) {
      const uint4 sv = D.src32[list[w][e]];
      const float dx = fx_delta(sv.x, px, u0), dy = fx_delta(sv.y, py, u1), dz = fx_delta(sv.z, pz, u2);
      const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));  // = H-table coordinate
      const float rinv = __builtin_amdgcn_rsqf(r2 + eps2);
      const float soft = rinv * rinv * rinv;
      const int ci = static_cast<int>(fminf(r2, static_cast<float>(kHTableCells - 1)));
      const float fu = __builtin_amdgcn_fractf(r2);
      const float4 c = htab[ci];
      const float hcoef = fmaf(fmaf(fmaf(c.w, fu, c.z), fu, c.y), fu, c.x);
      float fr = fmaf(-hcoef, c8, soft);
      if (!D.uniform_mass) fr *= __uint_as_float(sv.w);
      const float f = r2 <= rc2 ? fr : 0.0f;  // the target itself: dx = dy = dz = 0
      lx = fmaf(f, dx, lx);
      ly = fmaf(f, dy, ly);
      lz = fmaf(f, dz, lz);
    }
    for (uint32_t e = lane; e < nm; e += kWave) {
      const uint32_t n = mps[w][e];
      const NodeMom32 M = D.mom32[n];
      const float dx = fx_delta(M.comx, px, s0) * to_len, dy = fx_delta(M.comy, py, s1) * to_len,
                  dz = fx_delta(M.comz, pz, s2) * to_len;
      float cx = 0.0f, cy = 0.0f, cz = 0.0f;
      node_accel32(M, D.quad32[n], dx, dy, dz, P, cx, cy, cz);
      mx += cx;
      my += cy;
      mz += cz;
    }
    __builtin_amdgcn_wave_barrier();
    nl = 0;
    nm = 0;
  };

  // walkmix_kernel's tests: the prune against the tight particle box and the
  // strict acceptance of small internal nodes
  auto classify = [&](uint32_t q, uint32_t& next, uint32_t& lb, uint32_t& lc) -> int {
    const NodeLink lk = D.link[q];
    const NodeBox32 b = D.box32[q];
    const float ax_ = fabsf(fx_delta(b.cx, px, s0)), ay_ = fabsf(fx_delta(b.cy, py, s1)),
                az_ = fabsf(fx_delta(b.cz, pz, s2));
    const float ex = fmaxf(0.0f, ax_ - b.hx), ey = fmaxf(0.0f, ay_ - b.hy), ez = fmaxf(0.0f, az_ - b.hz);
    const bool keep = !(fmaf(ex, ex, fmaf(ey, ey, ez * ez)) > prune2);
    if (lk.child_count == 0) {
      lb = lk.begin;
      lc = lk.count;
      return keep ? 1 : 0;
    }
    if (!keep) {
      next = q + lk.skip;
      return 0;
    }
    bool take = false;
    if (b.cell_half < P.accept_half_max) {
      float mfx, mfy, mfz;
      take = strict_accept32(P, F, D.geo32[q], D.mom32[q], D.quad32, q, px, py, pz, mfx, mfy, mfz);
    }
    next = take ? q + lk.skip : q + 1;
    return take ? 2 : 3;
  };
  walk_target_wave(D.node_count_dev ? *D.node_count_dev : P.node_count, lane, list[w], mps[w], nl, nm, classify, evaluate);
  const double gm = P.force_scale;
  const double sx = gm * wave_sum(static_cast<double>(lx)) + wave_sum(static_cast<double>(mx));
  const double sy = gm * wave_sum(static_cast<double>(ly)) + wave_sum(static_cast<double>(my));
  const double sz = gm * wave_sum(static_cast<double>(lz)) + wave_sum(static_cast<double>(mz));
  if (lane != 0) return;
  const float ax = static_cast<float>(sx), ay = static_cast<float>(sy), az = static_cast<float>(sz);
  float gx = 0.0f, gy = 0.0f, gz = 0.0f;
  if (P.pm_enabled) interp32<SCHEME>(P, D.f32x, D.f32y, D.f32z, px, py, pz, gx, gy, gz);
  static_cast<float*>(out.ax)[slot] = gx + ax;
  static_cast<float*>(out.ay)[slot] = gy + ay;
  static_cast<float*>(out.az)[slot] = gz + az;
  if (out.pm_x) {
    static_cast<float*>(out.pm_x)[slot] = gx;
    static_cast<float*>(out.pm_y)[slot] = gy;
    static_cast<float*>(out.pm_z)[slot] = gz;
  }
  const uint32_t row = D.order[tp];
  if (out.sr_x) {
    static_cast<float*>(out.sr_x)[row] = ax;
    static_cast<float*>(out.sr_y)[row] = ay;
    static_cast<float*>(out.sr_z)[row] = az;
  }
}

// ---- FP64 walk, one target per wave ----------------------------------------------
// walkmix_target_kernel's mapping for the FP64 strict walk: the lanes classify
// 64 consecutive preorder nodes with walk64_kernel's tests (the cutoff prune
// against the octree cell, accept64 for internal nodes), the visited chain
// lists kept leaves' sources and accepted nodes in LDS, and the lists are
// evaluated 64 entries at a time with walk64_kernel's pair and node
// arithmetic. The pairs and multipoles are walk64_kernel's; the sum runs in
// another order (per-lane partial sums, then a wave reduction).
template <int SCHEME>
__global__ __launch_bounds__(kWalkThreads) void walk64_target_kernel(WalkParams P, WalkData D, WalkOutputs out) {
  __shared__ uint32_t list[kWalkWaves][kTargetList];
  __shared__ uint32_t mps[kWalkWaves][kTargetNodes];
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const uint32_t k = xcd_logical_block() * kWalkWaves + w;
  if (k >= P.n_targets) return;  // wave-uniform
  const uint32_t tp = P.identity_targets ? k : D.tpos[k];
  const uint32_t slot = P.identity_targets ? D.order[k] : D.tslot[k];
  const double4 t = D.src64[tp];
  const double px = t.x, py = t.y, pz = t.z;
  const double L0 = P.L[0], L1 = P.L[1], L2 = P.L[2];

  double ax = 0.0, ay = 0.0, az = 0.0;
  uint32_t nl = 0, nm = 0;
  auto evaluate = [&]() {
    __builtin_amdgcn_wave_barrier();
    for (uint32_t e = lane; e < nl; e += kWave) {
      const uint32_t j = list[w][e];
      const double4 sj = D.src64[j];
      const double qx = mi64(sj.x - px, L0), qy = mi64(sj.y - py, L1), qz = mi64(sj.z - pz, L2);
      const double r2 = qx * qx + qy * qy + qz * qz;
      // coincident pairs have a zero vector; the target itself is skipped
      if (j != tp && r2 <= P.rcut2 && !(qx == 0.0 && qy == 0.0 && qz == 0.0)) {
        const double f = residual_inv_r3(r2, P.eps, P.a) * P.G;
        const double mj = D.uniform_mass ? P.uniform_mass : sj.w;
        ax += f * mj * qx;
        ay += f * mj * qy;
        az += f * mj * qz;
      }
    }
    for (uint32_t e = lane; e < nm; e += kWave) {
      const uint32_t n = mps[w][e];
      const NodeMom64 M = D.mom64[n];
      const double dx = mi64(M.comx - px, L0), dy = mi64(M.comy - py, L1), dz = mi64(M.comz - pz, L2);
      node_accel64_call(M, D.quad64[n], dx, dy, dz, P, ax, ay, az);  // out of line: register pressure
    }
    __builtin_amdgcn_wave_barrier();
    nl = 0;
    nm = 0;
  };

  // walk64_kernel's tests: the prune against the octree cell and accept64
  auto classify = [&](uint32_t q, uint32_t& next, uint32_t& lb, uint32_t& lc) -> int {
    const NodeLink lk = D.link[q];
    const NodeGeo64 g = D.geo64[q];
    const double h = g.half;
    const double ax_ = fabs(mi64(g.cx - px, L0)), ay_ = fabs(mi64(g.cy - py, L1)), az_ = fabs(mi64(g.cz - pz, L2));
    const double ex = fmax(0.0, ax_ - h), ey = fmax(0.0, ay_ - h), ez = fmax(0.0, az_ - h);
    const bool keep = within_cutoff(ex * ex + ey * ey + ez * ez, P.rcut, P.rcut2);
    if (lk.child_count == 0) {
      lb = lk.begin;
      lc = lk.count;
      return keep ? 1 : 0;
    }
    if (!keep) {
      next = q + lk.skip;
      return 0;
    }
    const bool inside = ax_ <= h && ay_ <= h && az_ <= h;
    const double mx = ax_ + h, my = ay_ + h, mz = az_ + h;
    const bool contained = within_cutoff(mx * mx + my * my + mz * mz, P.rcut, P.rcut2);
    const NodeMom64 M = D.mom64[q];
    const double mdx = mi64(M.comx - px, L0), mdy = mi64(M.comy - py, L1), mdz = mi64(M.comz - pz, L2);
    const bool take = accept64(h, D.quad64[q].offset, inside, contained, mdx * mdx + mdy * mdy + mdz * mdz, P);
    next = take ? q + lk.skip : q + 1;
    return take ? 2 : 3;
  };
  walk_target_wave((D.node_count_dev ? *D.node_count_dev : P.node_count), lane, list[w], mps[w], nl, nm, classify, evaluate);
  ax = wave_sum(ax);
  ay = wave_sum(ay);
  az = wave_sum(az);
  if (lane != 0) return;
  double gx = 0.0, gy = 0.0, gz = 0.0;
  if (P.pm_enabled) interp64<SCHEME>(P, D.f64x, D.f64y, D.f64z, px, py, pz, gx, gy, gz);
  static_cast<double*>(out.ax)[slot] = gx + ax;
  static_cast<double*>(out.ay)[slot] = gy + ay;
  static_cast<double*>(out.az)[slot] = gz + az;
  if (out.pm_x) {
    static_cast<double*>(out.pm_x)[slot] = gx;
    static_cast<double*>(out.pm_y)[slot] = gy;
    static_cast<double*>(out.pm_z)[slot] = gz;
  }
  const uint32_t row = D.order[tp];
  if (out.sr_x) {
    static_cast<double*>(out.sr_x)[row] = ax;
    static_cast<double*>(out.sr_y)[row] = ay;
    static_cast<double*>(out.sr_z)[row] = az;
  }
}

// ---- FP64 strict walk, box-classified (the timed FP64 path) ----------------------
// The box-classified traversal in FP64 for solves without counters and for
// the force VJP. Staged sources beyond r_cut of the segment's box are dropped,
// the rest fill an LDS window of kBoxWindow records (half that in the JVP,
// which also stages lam). A full window is evaluated group by group:
// kBoxGroup consecutive targets of the segment, whose own box drops the
// window's records again (the kept ones are copied to a list of 64) and whose
// pairs all 64 lanes share, as 64 / kBoxGroup source slices. In the evenly
// filled parts of a box the 64 targets of a segment span more than r_cut and a
// record reaches few of them: groups of 16 cut the pair slots per 64 targets
// from 1171 to 674 at 96^3 (10% in halos; counted on a CPU model of the walk).
// An FP64 pair costs enough for that to pay (96^3: 3.27 ms without groups,
// 2.97 with; the VJP of 64^3 3.10 against 2.75 ms); a mixed pair does not
// (256^3: 18.2 against 21.9 ms). Segments whose box is small against r_cut
// (kBoxCompact) stay one group. List slot of record r for S slices of TL
// records: (r % S) (TL + 1) + r / S, so a lane's records are consecutive and
// the slices start in different LDS banks. Subtrees some target may accept as
// a multipole are walked lane by lane with walk64_kernel's tests (cell prune,
// accept64, node_accel64). The pairs and multipoles are walk64_kernel's; the
// pair arithmetic and the summation order differ at the round-off level.
// What bounds it at 96^3 is waiting: 1.4 of 3 possible waves are resident per
// SIMD on average (13824 waves of uneven length), spend half of their cycles
// waiting, and spill 114 VGPRs (444 bytes per lane); the SIMDs issue vector
// instructions in 36 % of the cycles. The JVP at 64^3: 1.2 of 2 waves, 167
// VGPRs spilled, 30 %.
constexpr int kH64Cells = kH64MaxCells;

// JVP: the transpose of the acceleration Jacobian applied to lam, as in
// walk64_kernel<..., JVP> (pair term G (F w + 2 F'(t) (r . w) r), w = m_k
// lam_j - m_j lam_k, with F' = dF/d(r^2) from the same table); accepted nodes
// add their Jacobian terms and are listed for vjp_node_corrections.
template <int SCHEME, bool JVP, bool FRAME>
__global__ __launch_bounds__(kWalkThreads) __attribute__((amdgpu_waves_per_eu(JVP ? 2 : 3))) void walk64_box_kernel(
    WalkParams P, WalkData D, WalkOutputs out, unsigned long long* __restrict__ counters) {
  constexpr uint32_t kWin = JVP ? kBoxWindow / 2 : kBoxWindow;
  __shared__ double4 win_all[kWalkWaves][kWin];
  __shared__ double4 list_all[kWalkWaves][kBoxList];
  // JVP: lam of the staged sources
  __shared__ double4 winl_all[JVP ? kWalkWaves : 1][JVP ? kWin : 1];
  __shared__ double4 listl_all[JVP ? kWalkWaves : 1][JVP ? kBoxList : 1];
  __shared__ BoxLds box_all[kWalkWaves];
  __shared__ double2 htab[3 * (kH64Cells + 1)];
  for (int i = threadIdx.x; i < 3 * (P.h64_cells + 1); i += kWalkThreads) htab[i] = D.h64tab[i];
  __syncthreads();
  const uint32_t node_count = D.node_count_dev ? *D.node_count_dev : P.node_count;
  const int w = static_cast<int>(readlane_u32(threadIdx.x / kWave, 0));
  const int lane = threadIdx.x % kWave;
  double4* const win = win_all[w];
  double4* const list = list_all[w];
  double4* const winl = winl_all[JVP ? w : 0];
  double4* const listl = listl_all[JVP ? w : 0];
  const uint32_t per_wave = P.targets_per_wave;
  const uint64_t k64 = (static_cast<uint64_t>(xcd_logical_block()) * kWalkWaves + w) * per_wave;
  if (k64 >= P.n_targets || node_count == 0) return;
  const uint32_t k0 = static_cast<uint32_t>(k64);
  const uint32_t here = P.n_targets - k0 < per_wave ? P.n_targets - k0 : per_wave;  // targets of this wave
  const double L0 = P.L[0], L1 = P.L[1], L2 = P.L[2];
  const double iL0 = 1.0 / L0, iL1 = 1.0 / L1, iL2 = 1.0 / L2;
  // minimum image by a reciprocal multiply: d - L rint(d / L) up to the
  // rounding of d / L, which only matters at |d| within an ulp of L/2, far
  // outside r_cut
  auto mi_fast = [&](double d, int a) -> double {
    const double L = a == 0 ? L0 : (a == 1 ? L1 : L2);
    const double iL = a == 0 ? iL0 : (a == 1 ? iL1 : iL2);
    return fma(-L, rint(d * iL), d);
  };
  auto image = [&](double v, double b, int a) -> double {
    const double L = a == 0 ? L0 : (a == 1 ? L1 : L2);
    const double iL = a == 0 ? iL0 : (a == 1 ? iL1 : iL2);
    return fma(-L, rint((v - b) * iL), v);
  };
  const double rc = P.rcut, rc2 = P.rcut2;
  const double eps2 = P.eps2_64, tscale = P.h64_scale;
  const uint32_t last_cell = static_cast<uint32_t>(P.h64_cells);
  // node tests against the fixed-point tight boxes
  const float s0 = P.cubic ? 1.0f : P.fx_to_len[0];
  const float s1 = P.cubic ? 1.0f : P.fx_to_len[1];
  const float s2 = P.cubic ? 1.0f : P.fx_to_len[2];
  const float to_len = P.cubic ? P.fx_to_len[0] : 1.0f;
  // F at r = 0 (the reference's limit: 0 without softening), for coincident pairs in the JVP
  const double f_zero = JVP ? residual_inv_r3(0.0, P.eps, P.a) : 0.0;
  // Residual pair kernel in FP64: G m_j [(r^2+eps^2)^{-3/2} - H(r^2/4a^2)/8a^3] r_vec
  // (G m_j applied by the caller); with the derivative fp = dF/d(r^2) when asked (JVP).
  // s^{-3/2} from the FP32 reciprocal square root y (whose square is exact in
  // FP64): with e = 1 - s y^2, |e| < 2^-21, s^{-3/2} = y^3 (1 + 3/2 e + 15/8 e^2)
  // up to e^3 < 2^-63. The cell of H is the integer nearest to r^2 tscale, read
  // from the low word of the sum with 1.5 2^52; the cell's polynomial (-1/8a^3
  // folded into it) runs in the offset from the cell's centre. The pair loop
  // takes 36 VALU instructions per pair against 53 with two Newton steps and a
  // truncated cell index.
  constexpr double kRound = 6755399441055744.0;  // 1.5 * 2^52
  auto residual = [&](double r2, double* fp) -> double {
    const double s = r2 + eps2;  // eps2 > 0: coincident unsoftened pairs stay finite, times a zero vector
    const double y = static_cast<double>(__builtin_amdgcn_rsqf(static_cast<float>(s)));
    const double y2 = y * y;
    const double e = fma(-s, y2, 1.0);
    const double y3 = y2 * y;
    const double soft = fma(y3, e * fma(1.875, e, 1.5), y3);
    const double tm = fma(r2, tscale, kRound);
    const uint32_t c = static_cast<uint32_t>(__double2loint(tm));
    const uint32_t ci = c < last_cell ? c : last_cell;
    const double u = fma(r2, tscale, kRound - tm);
    const double2 a01 = htab[3 * ci], a23 = htab[3 * ci + 1], a45 = htab[3 * ci + 2];
    const double hv = fma(fma(fma(fma(fma(a45.y, u, a45.x), u, a23.y), u, a23.x), u, a01.y), u, a01.x);
    if (fp) {
      const double dh = fma(fma(fma(fma(5.0 * a45.y, u, 4.0 * a45.x), u, 3.0 * a23.y), u, 2.0 * a23.x), u, a01.y);
      const double is = fma(y2, fma(e, e, e), y2);  // 1 / s
      *fp = fma(-1.5 * soft, is, dh * tscale);
    }
    return soft + hv;
  };

  for (uint32_t seg = 0; seg < here;) {
    // --- the segment and its box (offsets from its first target) ---
    double bx = 0.0, by = 0.0, bz = 0.0, ex = 0.0, ey = 0.0, ez = 0.0;
    uint32_t T;
    if constexpr (!FRAME) {
      T = per_wave;
    } else {
      const uint32_t i = seg + lane < here ? seg + lane : here - 1;
      const double4 t = D.src64[P.identity_targets ? k0 + i : D.tpos[k0 + i]];
      const double o0 = readlane_f64(t.x, 0), o1 = readlane_f64(t.y, 0), o2 = readlane_f64(t.z, 0);
      const double vx = mi_fast(t.x - o0, 0), vy = mi_fast(t.y - o1, 1), vz = mi_fast(t.z - o2, 2);
      T = box_segment(seg, per_wave, [&](uint32_t want) -> bool {
        const bool in = static_cast<uint32_t>(lane) < want;
        const double ux = in ? vx : 0.0, uy = in ? vy : 0.0, uz = in ? vz : 0.0;
        // wave-uniform values through readlane, so they live in scalar registers
        const double lox = readlane_f64(wave_min(ux), 0), hix = readlane_f64(wave_max(ux), 0),
                     loy = readlane_f64(wave_min(uy), 0), hiy = readlane_f64(wave_max(uy), 0),
                     loz = readlane_f64(wave_min(uz), 0), hiz = readlane_f64(wave_max(uz), 0);
        bx = o0 + 0.5 * (lox + hix);
        by = o1 + 0.5 * (loy + hiy);
        bz = o2 + 0.5 * (loz + hiz);
        ex = 0.5 * (hix - lox) * (1.0 + 1.0e-12);
        ey = 0.5 * (hiy - loy) * (1.0 + 1.0e-12);
        ez = 0.5 * (hiz - loz) * (1.0 + 1.0e-12);
        return ex <= P.box_max64 && ey <= P.box_max64 && ez <= P.box_max64 && ex + rc < 0.5 * L0 * (1.0 - 1.0e-9) &&
               ey + rc < 0.5 * L1 * (1.0 - 1.0e-9) && ez + rc < 0.5 * L2 * (1.0 - 1.0e-9);
      });
    }
    const uint32_t TL = T < 4u ? 4u : T;
    const uint32_t lgT = 31u - static_cast<uint32_t>(__builtin_clz(TL));
    const uint32_t col = static_cast<uint32_t>(lane) & (TL - 1u), slice = static_cast<uint32_t>(lane) >> lgT;
    const bool valid = col < T && seg + col < here;
    const bool owner = valid && slice == 0;  // the lane-by-lane walks run on the first slice
    const uint32_t k = k0 + seg + (valid ? col : 0u);
    const uint32_t tp = P.identity_targets ? k : D.tpos[k];
    double px, py, pz;
    double4 lk_ = make_double4(0.0, 0.0, 0.0, 0.0);  // JVP: lam of the target
    double mk = 0.0;                                  // JVP: mass of the target
    {
      const double4 t = D.src64[tp];
      px = t.x;
      py = t.y;
      pz = t.z;
      if constexpr (JVP) {
        lk_ = D.lam64[tp];
        mk = D.uniform_mass ? P.uniform_mass : t.w;
      }
    }
    // Boxed segments stage each source as its image nearest the box centre and
    // take the target's image likewise: away from the seam both are the
    // tree-frame coordinates themselves (the shift is zero), so r = x_j - x_k
    // is the reference's difference exactly.
    const double qx = image(px, bx, 0), qy = image(py, by, 1), qz = image(pz, bz, 2);
    double ax = 0.0, ay = 0.0, az = 0.0;
    // One staged record against a target: NEAR = images nearest the box centre,
    // else tree-frame coordinates with a minimum image per pair. tl, tm: lam
    // and mass of the target (JVP).
    auto pair = [&]<bool NEAR>(const double4& sj, const double4* lj_, double x, double y, double z, const double4& tl,
                               double tm, double lim, double& lx, double& ly, double& lz) {
      double dx, dy, dz;
      if constexpr (NEAR) {
        dx = sj.x - x;
        dy = sj.y - y;
        dz = sj.z - z;
      } else {
        dx = mi_fast(sj.x - x, 0);
        dy = mi_fast(sj.y - y, 1);
        dz = mi_fast(sj.z - z, 2);
      }
      const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
      if constexpr (JVP) {
        // the target itself: w = 0; a coincident source: F(0) w
        double fp = 0.0;
        double f = residual(r2, &fp);
        f = r2 > 0.0 ? f : f_zero;
        const double4 lj = *lj_;
        double wx, wy, wz;
        if (D.uniform_mass) {  // w / m (the mass goes into the final scale)
          wx = lj.x - tl.x;
          wy = lj.y - tl.y;
          wz = lj.z - tl.z;
        } else {
          wx = tm * lj.x - sj.w * tl.x;
          wy = tm * lj.y - sj.w * tl.y;
          wz = tm * lj.z - sj.w * tl.z;
        }
        const bool in = r2 <= lim;
        f = in ? f : 0.0;
        const double cr = in ? 2.0 * fp * fma(dx, wx, fma(dy, wy, dz * wz)) : 0.0;
        lx = fma(f, wx, fma(cr, dx, lx));
        ly = fma(f, wy, fma(cr, dy, ly));
        lz = fma(f, wz, fma(cr, dz, lz));
      } else {
        double f = residual(r2, nullptr);
        if (!D.uniform_mass) f *= sj.w;
        f = r2 <= lim ? f : 0.0;  // the target itself and coincident sources: zero vector
        lx = fma(f, dx, lx);
        ly = fma(f, dy, ly);
        lz = fma(f, dz, lz);
      }
    };
    const double gm = D.uniform_mass ? P.G * P.uniform_mass : P.G;
    // the n leaf sources staged in the list (lane-by-lane walks; the list is
    // free between evaluations)
    auto leaf_pairs = [&]<bool NEAR>(uint32_t n, double lim) {
      double lx = 0.0, ly = 0.0, lz = 0.0;
      const double x = NEAR ? qx : px, y = NEAR ? qy : py, z = NEAR ? qz : pz;
      for (uint32_t si = 0; si < n; ++si)
        pair.template operator()<NEAR>(list[si], listl + (JVP ? si : 0u), x, y, z, lk_, mk, lim, lx, ly, lz);
      ax = fma(gm, lx, ax);
      ay = fma(gm, ly, ay);
      az = fma(gm, lz, az);
    };

    // lane-by-lane walk of the preorder range [nxt, end) with walk64_kernel's tests
    uint32_t nxt = 0;
    auto walk = [&]<bool NEAR>(uint32_t end) {
      uint32_t n = wave_min_u32(nxt);
      while (n < end) {
        const NodeLink lk = D.link[n];
        const NodeGeo64 g = D.geo64[n];
        const bool act = nxt == n;
        if (!__ballot(act)) {
          if (lane == 0) atomicOr(&counters[kFaultSlot], 1ull);
          break;
        }
        const double h = g.half;
        const double ndx = mi_fast(g.cx - px, 0), ndy = mi_fast(g.cy - py, 1), ndz = mi_fast(g.cz - pz, 2);
        const double ax_ = fabs(ndx), ay_ = fabs(ndy), az_ = fabs(ndz);
        const double fx_ = fmax(0.0, ax_ - h), fy_ = fmax(0.0, ay_ - h), fz_ = fmax(0.0, az_ - h);
        const bool keep = act && within_cutoff(fx_ * fx_ + fy_ * fy_ + fz_ * fz_, P.rcut, P.rcut2);
        if (act && !keep) nxt = n + lk.skip;
        if (lk.child_count == 0) {
          if (keep) nxt = n + 1;
          if (__ballot(keep)) {
            const double lim = keep ? rc2 : -1.0;
            const uint32_t e0 = lk.begin + lk.count;
            for (uint32_t c0 = lk.begin; c0 < e0; c0 += kWindow) {
              const uint32_t cn = e0 - c0 < static_cast<uint32_t>(kWindow) ? e0 - c0 : static_cast<uint32_t>(kWindow);
              __builtin_amdgcn_wave_barrier();
              if (static_cast<uint32_t>(lane) < cn) {
                const double4 sv = D.src64[c0 + lane];
                if constexpr (JVP) listl[lane] = D.lam64[c0 + lane];
                list[lane] =
                    NEAR ? make_double4(image(sv.x, bx, 0), image(sv.y, by, 1), image(sv.z, bz, 2), sv.w) : sv;
              }
              __builtin_amdgcn_wave_barrier();
              leaf_pairs.template operator()<NEAR>(cn, lim);
            }
            __builtin_amdgcn_wave_barrier();
          }
        } else if (__ballot(keep)) {
          // the forward's strict acceptance; in the JVP an accepted node's
          // Jacobian terms go to the target and to the node's accumulators
          bool take_mp = false;
          double mdx = 0.0, mdy = 0.0, mdz = 0.0;
          if (keep && P.quad) {
            const bool inside = ax_ <= h && ay_ <= h && az_ <= h;
            const double mx = ax_ + h, my = ay_ + h, mz = az_ + h;
            const bool contained = within_cutoff(mx * mx + my * my + mz * mz, P.rcut, P.rcut2);
            const NodeMom64 M = D.mom64[n];
            mdx = mi_fast(M.comx - px, 0);
            mdy = mi_fast(M.comy - py, 1);
            mdz = mi_fast(M.comz - pz, 2);
            take_mp = accept64(h, D.quad64[n].offset, inside, contained, mdx * mdx + mdy * mdy + mdz * mdz, P);
          }
          if (keep) nxt = take_mp ? n + lk.skip : n + 1;
          if (__ballot(take_mp) && take_mp) {
            if constexpr (JVP) {
              jvp_node64(D.mom64[n], D.quad64[n], mdx, mdy, mdz, P, lk_.x, lk_.y, lk_.z, D.vjp_node_acc + 10ull * n,
                         ax, ay, az);
              const unsigned int slot_i = atomicAdd(D.vjp_accepted_count, 1u);
              if (slot_i < D.vjp_accepted_cap)
                D.vjp_accepted[slot_i] = (static_cast<unsigned long long>(tp) << 32) | n;
            } else {
              node_accel64(D.mom64[n], D.quad64[n], mdx, mdy, mdz, P, ax, ay, az);
            }
          }
        }
        n = next_node(n, nxt);
      }
    };

    if constexpr (FRAME) {
      // staged sources beyond r_cut of the target box (every pair with them
      // lies beyond r_cut, so their terms are zero) are dropped
      const double cull2 = rc2 * (1.0 + 1.0e-9);
      uint32_t wn = 0;  // records in the window
      // evaluation groups of kBoxGroup targets, or the whole segment
      const double compact = kBoxCompact * rc;
      const bool one = TL <= kBoxGroup || (ex <= compact && ey <= compact && ez <= compact);
      const uint32_t lgG = one ? lgT : 4u, GL = 1u << lgG, lgGS = 6u - lgG;
      const uint32_t groups = one ? 1u : TL >> lgG;
      const uint32_t gcol = static_cast<uint32_t>(lane) & (GL - 1u), gslice = static_cast<uint32_t>(lane) >> lgG;
      const uint32_t mine = gslice * (GL + 1u);
      // group boxes about the box centre in FP32; the half-extents' margin
      // covers the rounding of the offsets (box and r_cut are of one order)
      const float bm = static_cast<float>(1.0e-6 * (rc + ex + ey + ez));
      float qc0 = 0.0f, qc1 = 0.0f, qc2 = 0.0f;
      float qh0 = static_cast<float>(ex) + bm, qh1 = static_cast<float>(ey) + bm, qh2 = static_cast<float>(ez) + bm;
      if (!one) {
        row_bounds(static_cast<float>(qx - bx), qc0, qh0);
        row_bounds(static_cast<float>(qy - by), qc1, qh1);
        row_bounds(static_cast<float>(qz - bz), qc2, qh2);
        qh0 += bm;
        qh1 += bm;
        qh2 += bm;
      }
      const float gcull2 = static_cast<float>(cull2) * 1.000001f;
      auto slot_of = [&](uint32_t r) -> uint32_t { return (r & ((1u << lgGS) - 1u)) * (GL + 1u) + (r >> lgGS); };
      const double far = 8.0 * (rc + ex + ey + ez);
      auto process = [&]() {
        __builtin_amdgcn_wave_barrier();
        for (uint32_t g = 0; g < groups; ++g) {
          const uint32_t row = g << lgG;
          const int from = static_cast<int>(row + gcol);
          const double x = __shfl(qx, from, kWave), y = __shfl(qy, from, kWave), z = __shfl(qz, from, kWave);
          double4 tl = make_double4(0.0, 0.0, 0.0, 0.0);
          double tm = 0.0;
          if constexpr (JVP) {
            tl.x = __shfl(lk_.x, from, kWave);
            tl.y = __shfl(lk_.y, from, kWave);
            tl.z = __shfl(lk_.z, from, kWave);
            tm = __shfl(mk, from, kWave);
          }
          const float c0 = readlane_f32(qc0, row), c1 = readlane_f32(qc1, row), c2 = readlane_f32(qc2, row);
          const float h0 = readlane_f32(qh0, row), h1 = readlane_f32(qh1, row), h2 = readlane_f32(qh2, row);
          double lx = 0.0, ly = 0.0, lz = 0.0;
          uint32_t n2 = 0;
          for (uint32_t b = 0;; b += kWave) {
            const bool end = b >= wn;
            double4 rec = make_double4(0.0, 0.0, 0.0, 0.0);
            bool keep = false;
            if (b + lane < wn) {
              rec = win[b + lane];
              const float dx = fmaxf(fabsf(static_cast<float>(rec.x - bx) - c0) - h0, 0.0f);
              const float dy = fmaxf(fabsf(static_cast<float>(rec.y - by) - c1) - h1, 0.0f);
              const float dz = fmaxf(fabsf(static_cast<float>(rec.z - bz) - c2) - h2, 0.0f);
              keep = !(fmaf(dx, dx, fmaf(dy, dy, dz * dz)) > gcull2);
            }
            const unsigned long long km = __ballot(keep);
            const uint32_t kept = static_cast<uint32_t>(__popcll(km));
            if (n2 && (end || n2 + kept > static_cast<uint32_t>(kWindow))) {
              // dummies beyond r_cut of every target fill the last iterations
              const uint32_t iters = (((n2 + (1u << lgGS) - 1u) >> lgGS) + 1u) & ~1u;
              if (static_cast<uint32_t>(lane) >= n2 && static_cast<uint32_t>(lane) < iters << lgGS) {
                list[slot_of(lane)] = make_double4(bx + far, by + far, bz + far, 0.0);
                if constexpr (JVP) listl[slot_of(lane)] = make_double4(0.0, 0.0, 0.0, 0.0);
              }
              __builtin_amdgcn_wave_barrier();
#pragma unroll 2
              for (uint32_t si = 0; si < iters; ++si)
                pair.template operator()<true>(list[mine + si], listl + (JVP ? mine + si : 0u), x, y, z, tl, tm, rc2,
                                               lx, ly, lz);
              __builtin_amdgcn_wave_barrier();
              n2 = 0;
            }
            if (end) break;
            if (keep) {
              const uint32_t at = slot_of(n2 + lanes_below(km));
              list[at] = rec;
              if constexpr (JVP) listl[at] = winl[b + lane];
            }
            n2 += kept;
          }
          // slices -> the group's own lanes
          for (uint32_t o = GL; o < static_cast<uint32_t>(kWave); o <<= 1) {
            lx += __shfl_xor(lx, static_cast<int>(o), kWave);
            ly += __shfl_xor(ly, static_cast<int>(o), kWave);
            lz += __shfl_xor(lz, static_cast<int>(o), kWave);
          }
          if (gslice == g) {
            ax = fma(gm, lx, ax);
            ay = fma(gm, ly, ay);
            az = fma(gm, lz, az);
          }
        }
        wn = 0;
        __builtin_amdgcn_wave_barrier();
      };
      // the box in fixed point: the centre's floor and the conversion of the
      // half-extents move a face by less than four units
      const double fs0 = 4294967296.0 * iL0, fs1 = 4294967296.0 * iL1, fs2 = 4294967296.0 * iL2;
      auto fixed = [](double v, double scale) -> uint32_t {
        return static_cast<uint32_t>(static_cast<uint64_t>(static_cast<int64_t>(floor(v * scale))));
      };
      auto half = [&](double e, double fs, float unit) -> float {
        return static_cast<float>((e * fs + 4.0) * (1.0 + 1.0e-6)) * unit;
      };
      const BoxFrame frame{fixed(bx, fs0), fixed(by, fs1), fixed(bz, fs2), half(ex, fs0, s0), half(ey, fs1, s1),
                           half(ez, fs2, s2), s0, s1, s2, P.prune2_sep,
                           P.quad ? static_cast<float>(0.041 * rc) : 0.0f, to_len};
      struct Record {
        double4 s;
        uint32_t j;
      };
      box_traverse(
          D.wnode, box_all[w], lane, frame, [&](uint32_t j) -> Record { return Record{D.src64[j], j}; },
          [&](const Record& r, bool on, bool last) {
            const double4 rec =
                make_double4(image(r.s.x, bx, 0), image(r.s.y, by, 1), image(r.s.z, bz, 2), r.s.w);
            const double fx_ = fmax(0.0, fabs(rec.x - bx) - ex), fy_ = fmax(0.0, fabs(rec.y - by) - ey),
                         fz_ = fmax(0.0, fabs(rec.z - bz) - ez);
            const bool keep = on && fx_ * fx_ + fy_ * fy_ + fz_ * fz_ <= cull2;
            const unsigned long long km = __ballot(keep);
            const uint32_t kept = static_cast<uint32_t>(__popcll(km));
            bool todo = true, go = wn + kept > kWin;
            do {  // evaluate a full window, add the batch, evaluate the last window
              if (go) process();
              if (todo) {
                if (keep) {
                  const uint32_t at = wn + lanes_below(km);
                  win[at] = rec;
                  if constexpr (JVP) winl[at] = D.lam64[r.j];
                }
                wn += kept;
                todo = false;
              }
              go = last && wn;
            } while (go);
          },
          [&](uint32_t pre, uint32_t end) -> bool {
            const NodeGeo64 g = D.geo64[pre];
            const NodeMom64 M = D.mom64[pre];
            const double h = g.half;
            const double ax_ = fabs(mi_fast(g.cx - px, 0)), ay_ = fabs(mi_fast(g.cy - py, 1)),
                         az_ = fabs(mi_fast(g.cz - pz, 2));
            const double mx = ax_ + h, my = ay_ + h, mz = az_ + h;
            const double mdx = mi_fast(M.comx - px, 0), mdy = mi_fast(M.comy - py, 1), mdz = mi_fast(M.comz - pz, 2);
            const bool acc = accept64(h, D.quad64[pre].offset, ax_ <= h && ay_ <= h && az_ <= h,
                                      within_cutoff(mx * mx + my * my + mz * mz, P.rcut, P.rcut2),
                                      mdx * mdx + mdy * mdy + mdz * mdz, P);
            if (!__ballot(owner && acc)) return true;
            nxt = owner ? pre : end;
            walk.template operator()<true>(end);
            return false;
          });
    } else {
      nxt = owner ? 0u : node_count;
      walk.template operator()<false>(node_count);
    }
    if (owner) {
      double gx = 0.0, gy = 0.0, gz = 0.0;
      if (P.pm_enabled) {
        if constexpr (JVP)
          vjp_gather64<SCHEME>(P, D.f64x, D.f64y, D.f64z, D.nu64, lk_.x, lk_.y, lk_.z, mk, px, py, pz, gx, gy, gz);
        else
          interp64<SCHEME>(P, D.f64x, D.f64y, D.f64z, px, py, pz, gx, gy, gz);
      }
      const uint32_t row = D.order[tp];
      const uint32_t slot = P.identity_targets ? row : D.tslot[k];
      static_cast<double*>(out.ax)[slot] = gx + ax;
      static_cast<double*>(out.ay)[slot] = gy + ay;
      static_cast<double*>(out.az)[slot] = gz + az;
      if (out.pm_x) {
        static_cast<double*>(out.pm_x)[slot] = gx;
        static_cast<double*>(out.pm_y)[slot] = gy;
        static_cast<double*>(out.pm_z)[slot] = gz;
      }
      if (out.sr_x) {
        static_cast<double*>(out.sr_x)[row] = ax;
        static_cast<double*>(out.sr_y)[row] = ay;
        static_cast<double*>(out.sr_z)[row] = az;
      }
    }
    seg += T;
  }
}

// ---- force VJP: accepted-node terms ----------------------------------------
// For a direct pair (t sees p) the symmetric pair term of p's walk adds
// M_tp lam_t to s_p, M_tp = d a_t / d x_p = G m_p [F I + 2 F' r r^T]; it is
// right only if t also sees p directly. For an accepted (t, N) and p in N
// within r_cut that sees t directly (p accepts no node holding t): remove
// M_tp lam_t from s_p, and add to s_t the term p's force contributes,
// M_pt lam_p = G m_t [F lam_p + 2 F' (r . lam_p) r]. rec is sorted.
// A recorded VJP: more accepted (target, node) pairs than list slots.
__global__ void vjp_count_check_kernel(const unsigned int* __restrict__ count, unsigned int cap,
                                       unsigned long long* __restrict__ fault) {
  if (threadIdx.x == 0 && *count > cap) atomicOr(fault, kFaultPrepared);
}

// nrec_dev (a recorded VJP): the list's real length on the device, nrec its capacity.
__global__ __launch_bounds__(256) void vjp_pair_fix_kernel(const unsigned long long* __restrict__ rec, uint32_t nrec_cap,
                                                           const unsigned int* __restrict__ nrec_dev,
                                                           const NodeLink* __restrict__ link,
                                                           const double4* __restrict__ src,
                                                           const double4* __restrict__ lam, int uniform, double um,
                                                           WalkParams P, double* __restrict__ corr) {
  const uint32_t nrec = nrec_dev ? min(*nrec_dev, nrec_cap) : nrec_cap;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrec) return;
  const uint32_t t = static_cast<uint32_t>(rec[i] >> 32), node = static_cast<uint32_t>(rec[i] & 0xFFFFFFFFull);
  const double4 xt = src[t], lt = lam[t];
  const double mt = uniform ? um : xt.w;
  const NodeLink lk = link[node];
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (uint32_t pp = lk.begin; pp < lk.begin + lk.count; ++pp) {
    const double4 xp = src[pp];
    const double dx = mi64(xp.x - xt.x, P.L[0]), dy = mi64(xp.y - xt.y, P.L[1]), dz = mi64(xp.z - xt.z, P.L[2]);
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (!(r2 <= P.rcut2) || !(r2 > 0.0)) continue;
    const unsigned long long key = static_cast<unsigned long long>(pp) << 32;
    uint32_t lo = 0, hi = nrec;
    while (lo < hi) {
      const uint32_t mid = lo + ((hi - lo) >> 1);
      if (rec[mid] < key) lo = mid + 1;
      else hi = mid;
    }
    bool mutual = false;
    for (uint32_t j = lo; j < nrec && static_cast<uint32_t>(rec[j] >> 32) == pp; ++j) {
      const NodeLink l2 = link[static_cast<uint32_t>(rec[j] & 0xFFFFFFFFull)];
      if (t >= l2.begin && t < l2.begin + l2.count) {
        mutual = true;
        break;
      }
    }
    if (mutual) continue;
    const double f = residual_inv_r3(r2, P.eps, P.a), fd = residual_inv_r3_dt(r2, P.eps, P.a);
    const double4 lp = lam[pp];
    const double mp = uniform ? um : xp.w;
    const double rt = dx * lt.x + dy * lt.y + dz * lt.z, rp = dx * lp.x + dy * lp.y + dz * lp.z;
    const double gp = P.G * mp, gt = P.G * mt;
    atomicAdd(&corr[3ull * pp + 0], -gp * (f * lt.x + 2.0 * fd * rt * dx));
    atomicAdd(&corr[3ull * pp + 1], -gp * (f * lt.y + 2.0 * fd * rt * dy));
    atomicAdd(&corr[3ull * pp + 2], -gp * (f * lt.z + 2.0 * fd * rt * dz));
    s0 += gt * (f * lp.x + 2.0 * fd * rp * dx);
    s1 += gt * (f * lp.y + 2.0 * fd * rp * dy);
    s2 += gt * (f * lp.z + 2.0 * fd * rp * dz);
  }
  atomicAdd(&corr[3ull * t + 0], s0);
  atomicAdd(&corr[3ull * t + 1], s1);
  atomicAdd(&corr[3ull * t + 2], s2);
}

// U and V of node N spread over its particles p (d_p = x_p - COM_N):
// s_p += (m_p / M) U + m_p G_V d_p, with G_V the symmetric matrix of
// sum_q V_q d Q_q / d d_p for the stored components (Q_q of one particle:
// m (3 d d^T - |d|^2 I) traceless parts qxx..qzz and the trace m |d|^2).
__global__ __launch_bounds__(256) void vjp_node_push_kernel(uint32_t nodes, const double* __restrict__ acc,
                                                            const NodeLink* __restrict__ link,
                                                            const NodeMom64* __restrict__ mom,
                                                            const double4* __restrict__ src, int uniform, double um,
                                                            WalkParams P, double* __restrict__ corr) {
  const uint32_t n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nodes) return;
  const double* a = acc + 10ull * n;
  bool any = false;
#pragma unroll
  for (int k = 0; k < 10; ++k) any = any || a[k] != 0.0;
  if (!any) return;
  const NodeMom64 M = mom[n];
  if (!(M.mass > 0.0)) return;
  const double ux = a[0] / M.mass, uy = a[1] / M.mass, uz = a[2] / M.mass;
  const double v0 = a[3], v1 = a[4], v2 = a[5], v3 = a[6], v4 = a[7], v5 = a[8], v6 = a[9];
  const double gxx = 4.0 * v0 - 2.0 * v3 - 2.0 * v5 + 2.0 * v6, gxy = 3.0 * v1, gxz = 3.0 * v2;
  const double gyy = -2.0 * v0 + 4.0 * v3 - 2.0 * v5 + 2.0 * v6, gyz = 3.0 * v4;
  const double gzz = -2.0 * v0 - 2.0 * v3 + 4.0 * v5 + 2.0 * v6;
  const NodeLink lk = link[n];
  for (uint32_t pp = lk.begin; pp < lk.begin + lk.count; ++pp) {
    const double4 xp = src[pp];
    const double mp = uniform ? um : xp.w;
    const double dx = mi64(xp.x - M.comx, P.L[0]), dy = mi64(xp.y - M.comy, P.L[1]), dz = mi64(xp.z - M.comz, P.L[2]);
    atomicAdd(&corr[3ull * pp + 0], mp * (ux + gxx * dx + gxy * dy + gxz * dz));
    atomicAdd(&corr[3ull * pp + 1], mp * (uy + gxy * dx + gyy * dy + gyz * dz));
    atomicAdd(&corr[3ull * pp + 2], mp * (uz + gxz * dx + gyz * dy + gzz * dz));
  }
}

__global__ __launch_bounds__(256) void vjp_apply_kernel(uint32_t n, const uint32_t* __restrict__ order,
                                                        const double* __restrict__ corr, double* __restrict__ ox,
                                                        double* __restrict__ oy, double* __restrict__ oz) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t row = order[k];
  ox[row] += corr[3ull * k + 0];
  oy[row] += corr[3ull * k + 1];
  oz[row] += corr[3ull * k + 2];
}

// H(t) = L(sqrt t) / t^{3/2} (tree_pm_split_kernel.hpp:109-128).
double gaussian_h_exact(double t) {
  if (t < 0.015625) {
    constexpr double c = 2.25675833419102514779231780624309034;
    return c * (1.0 / 3.0 + t * (-1.0 / 5.0 + t * (1.0 / 14.0 + t * (-1.0 / 54.0 + t * (1.0 / 264.0 +
           t * (-1.0 / 1560.0 + t * (1.0 / 10800.0 - t / 85680.0)))))));
  }
  const double q = std::sqrt(t);
  return (std::erf(q) - 2.0 * kInvSqrtPi * q * std::exp(-t)) / (t * q);
}

// dH/dt: derivative of the series below t = 1/64, of the closed form above
// (the same split as tree_pm_split_kernel.hpp:248-285).
double gaussian_h_slope(double t) {
  constexpr double c = 2.25675833419102514779231780624309034;
  if (t < 0.015625) {
    const double coef[8] = {1.0 / 3.0, -1.0 / 5.0, 1.0 / 14.0, -1.0 / 54.0,
                            1.0 / 264.0, -1.0 / 1560.0, 1.0 / 10800.0, -1.0 / 85680.0};
    double d = 0.0;
    for (int i = 7; i >= 1; --i) d = d * t + i * coef[i];
    return c * d;
  }
  return (0.5 * c * std::exp(-t) - 1.5 * gaussian_h_exact(t)) / t;
}

template <int SCHEME, bool JVP = false>
void launch64(const WalkParams& p, const WalkData& d, const WalkOutputs& out, unsigned long long* counters,
              hipStream_t s) {
  walk64_kernel<SCHEME, JVP><<<grid_for(p.n_targets, kWalkThreads), kWalkThreads, 0, s>>>(p, d, out, counters);
  CHUI_LAUNCH_CHECK("walk64_kernel");
}
// Targets per wave of the box walks: 64, or fewer (down to 8) until the
// launch has kBoxMinWaves waves, four for each of the 1024 SIMDs.
constexpr uint32_t kBoxMinWaves = 4096;
WalkParams box_params(const WalkParams& p) {
  WalkParams q = p;
  q.targets_per_wave = kWave;
  if (q.box_single)
    while (q.targets_per_wave > 8 && p.n_targets / q.targets_per_wave < kBoxMinWaves) q.targets_per_wave >>= 1;
  return q;
}
unsigned box_blocks(const WalkParams& p, unsigned waves) {
  return grid_for((static_cast<std::size_t>(p.n_targets) + p.targets_per_wave - 1) / p.targets_per_wave, waves);
}

template <int SCHEME, bool CUBIC, bool LOG, int WAVES>
void launch_box(const WalkParams& p, const WalkData& d, const WalkOutputs& out, unsigned long long* counters,
                hipStream_t s) {
  const WalkParams q = box_params(p);
  const std::size_t lds = LOG ? p.log_cells * sizeof(float4) : 0;
  const unsigned grid = box_blocks(q, WAVES);
  const auto go = [&](auto kernel) {
    kernel<<<grid, WAVES * kWave, lds, s>>>(q, d, out, counters, d.link, d.geo32, d.mom32, d.quad32, d.box32, d.wnode);
  };
  if (q.box_single && q.shared_origin) go(walkmix_box_kernel<SCHEME, CUBIC, LOG, WAVES, true, true>);
  else if (q.box_single) go(walkmix_box_kernel<SCHEME, CUBIC, LOG, WAVES, true, false>);
  else go(walkmix_box_kernel<SCHEME, CUBIC, LOG, WAVES, false, false>);
  CHUI_LAUNCH_CHECK("walkmix_box_kernel");
}

template <bool JVP>
void launch_box64(const WalkParams& p, const WalkData& d, const WalkOutputs& out, unsigned long long* counters,
                  hipStream_t s) {
  const WalkParams q = box_params(p);
  const unsigned grid = box_blocks(q, kWalkWaves);
  if (q.box_single && p.assignment == 0)
    walk64_box_kernel<0, JVP, true><<<grid, kWalkThreads, 0, s>>>(q, d, out, counters);
  else if (q.box_single)
    walk64_box_kernel<1, JVP, true><<<grid, kWalkThreads, 0, s>>>(q, d, out, counters);
  else if (p.assignment == 0)
    walk64_box_kernel<0, JVP, false><<<grid, kWalkThreads, 0, s>>>(q, d, out, counters);
  else
    walk64_box_kernel<1, JVP, false><<<grid, kWalkThreads, 0, s>>>(q, d, out, counters);
  CHUI_LAUNCH_CHECK("walk64_box_kernel");
}

template <int SCHEME, bool CUBIC>
void launchmix(const WalkParams& p, const WalkData& d, const WalkOutputs& out, unsigned long long* counters,
               hipStream_t s) {
  if (p.count) {
    if (d.node_count_dev) throw std::logic_error("counting walk after a capture-safe build");
    walkmix_kernel<SCHEME, CUBIC><<<grid_for(p.n_targets, kWalkThreads), kWalkThreads, 0, s>>>(
        p, d, out, counters, d.link, d.geo32, d.mom32, d.quad32, d.box32);
    CHUI_LAUNCH_CHECK("walkmix_kernel");
  } else if (p.target_per_wave) {
    walkmix_target_kernel<SCHEME, CUBIC><<<grid_for(p.n_targets, kWalkWaves), kWalkThreads, 0, s>>>(p, d, out);
    CHUI_LAUNCH_CHECK("walkmix_target_kernel");
  } else if (p.log_cells > 0) {
    if (p.walk_waves == 8) launch_box<SCHEME, CUBIC, true, 8>(p, d, out, counters, s);
    else if (p.walk_waves == 2) launch_box<SCHEME, CUBIC, true, 2>(p, d, out, counters, s);
    else launch_box<SCHEME, CUBIC, true, 4>(p, d, out, counters, s);
  } else {
    launch_box<SCHEME, CUBIC, false, 4>(p, d, out, counters, s);
  }
}

}  // namespace

std::vector<float> log_residual_table(double scale, double eps, double a, int32_t& first_octave,
                                      uint32_t& cells) {
  // s = (r^2 + eps^2) * scale; F(s) = s^{-3/2} - c H(x(s)) with
  // x(s) = (s / scale - eps^2) / (4 a^2) and c = scale^{-3/2} / (8 a^3).
  cells = 0;
  const float eps2_tab = static_cast<float>(eps * eps * scale);
  if (!(eps2_tab > 0.0f) || !std::isfinite(eps2_tab)) return {};
  const int e0 = std::ilogb(eps2_tab);
  const int octaves = -e0;
  if (octaves < 1 || octaves > kLogMaxOctaves) return {};
  const double c = std::pow(scale, -1.5) / (8.0 * a * a * a);
  const double dxds = 1.0 / (scale * 4.0 * a * a);
  auto F = [&](double sv) { return std::pow(sv, -1.5) - c * gaussian_h_exact((sv / scale - eps * eps) / (4.0 * a * a)); };
  auto dF = [&](double sv) {
    return -1.5 * std::pow(sv, -2.5) - c * gaussian_h_slope((sv / scale - eps * eps) / (4.0 * a * a)) * dxds;
  };
  const int K = octaves * kLogCellsPerOctave;
  std::vector<float> tab(4 * static_cast<std::size_t>(K + 1), 0.0f);
  const double u1 = std::ldexp(1.0, -kLogMantissaShift), u2 = u1 * u1, u3 = u2 * u1;
  for (int o = 0; o < octaves; ++o) {
    const double base = std::ldexp(1.0, e0 + o);
    for (int j = 0; j < kLogCellsPerOctave; ++j) {
      const double s0 = base * (1.0 + static_cast<double>(j) / kLogCellsPerOctave);
      const double s1 = base * (1.0 + static_cast<double>(j + 1) / kLogCellsPerOctave);
      const double h = s1 - s0;
      const double f0 = F(s0), f1 = F(s1), d0 = h * dF(s0), d1 = h * dF(s1);
      float* t = &tab[4 * static_cast<std::size_t>(o * kLogCellsPerOctave + j)];
      t[0] = static_cast<float>(f0);
      t[1] = static_cast<float>(d0 * u1);
      t[2] = static_cast<float>((3.0 * (f1 - f0) - 2.0 * d0 - d1) * u2);
      t[3] = static_cast<float>((2.0 * (f0 - f1) + d0 + d1) * u3);
    }
  }
  first_octave = e0;
  cells = static_cast<uint32_t>(K + 1);  // the last cell is zero: s >= 1, beyond r_cut
  return tab;
}

std::vector<double> gaussian_quintic_table(double t_max, int cells, double factor) {
  // Interpolation at the Chebyshev points of each cell: error below
  // 2 (h/4)^6 max|H^(6)| / 6!, largest in the first whole cell: 4e-16 for cells
  // of width 0.04 (r_cut up to 6.4 a), 9e-14 at width 0.1 (10 a) and 6e-12 at
  // width 0.2 (14 a; t_max = 50 on 255 cells). The 6 x 6
  // Vandermonde system in u is solved in long double. The first cell covers
  // t >= 0 only, u in [0, 1/2].
  const double h = t_max / cells;
  std::vector<double> tab(6 * static_cast<std::size_t>(cells + 1));
  constexpr int D = 6;
  for (int i = 0; i <= cells; ++i) {
    const long double lo = i == 0 ? 0.0L : -0.5L, hi = 0.5L;
    long double A[D][D + 1];
    for (int j = 0; j < D; ++j) {
      const long double cj = std::cos(static_cast<long double>(3.14159265358979323846264338327950288L) * (2 * j + 1) /
                                      (2 * D));
      const long double un = 0.5L * (lo + hi) + 0.5L * (hi - lo) * cj;
      long double pw = 1.0L;
      for (int c = 0; c < D; ++c) {
        A[j][c] = pw;
        pw *= un;
      }
      A[j][D] = gaussian_h_exact((i + static_cast<double>(un)) * h);
    }
    for (int c = 0; c < D; ++c) {  // Gaussian elimination with partial pivoting
      int piv = c;
      for (int r = c + 1; r < D; ++r)
        if (std::fabs(static_cast<double>(A[r][c])) > std::fabs(static_cast<double>(A[piv][c]))) piv = r;
      for (int q = 0; q <= D; ++q) std::swap(A[c][q], A[piv][q]);
      for (int r = 0; r < D; ++r) {
        if (r == c) continue;
        const long double f = A[r][c] / A[c][c];
        for (int q = c; q <= D; ++q) A[r][q] -= f * A[c][q];
      }
    }
    for (int c = 0; c < D; ++c)
      tab[6 * static_cast<std::size_t>(i) + c] = static_cast<double>(factor * A[c][D] / A[c][c]);
  }
  return tab;
}

std::vector<float> gaussian_coefficient_table(WalkParams& p, double t_max) {
  // Cubic Hermite cells on [0, t_max]: value c0 + c1 u + c2 u^2 + c3 u^3 with u
  // the position inside the cell; interpolation error <= h^4/384 max|d4H/dt4|,
  // about 2e-9 for 128 cells on t <= 6, far below FP32 round-off.
  const int K = kHTableCells;
  const double h = t_max / K;
  std::vector<float> tab(4 * K);
  for (int i = 0; i < K; ++i) {
    const double t0 = i * h, t1 = (i + 1) * h;
    const double f0 = gaussian_h_exact(t0), f1 = gaussian_h_exact(t1);
    const double d0 = h * gaussian_h_slope(t0), d1 = h * gaussian_h_slope(t1);
    tab[4 * i + 0] = static_cast<float>(f0);
    tab[4 * i + 1] = static_cast<float>(d0);
    tab[4 * i + 2] = static_cast<float>(3.0 * (f1 - f0) - 2.0 * d0 - d1);
    tab[4 * i + 3] = static_cast<float>(2.0 * (f0 - f1) + d0 + d1);
  }
  p.t_to_cell = static_cast<float>(static_cast<double>(p.c4) / h);
  return tab;
}

void walk_fp64(const Tree& t, const WalkParams& p, const double4* src, int uniform_mass,
               const uint32_t* target_pos, const uint32_t* target_slot, const double* fx, const double* fy,
               const double* fz, const WalkOutputs& out, unsigned long long* counters, const double2* h64tab,
               hipStream_t s) {
  if (!t.records64 && t.node_count > 0) throw std::logic_error("FP64 walk on a tree without FP64 records");
  if (p.n_targets == 0) return;
  WalkData d{};
  d.link = t.link.as<NodeLink>();
  d.geo64 = t.geo64.as<NodeGeo64>();
  d.mom64 = t.mom64.as<NodeMom64>();
  d.quad64 = t.quad64.as<NodeQuad64>();
  d.order = t.order.as<uint32_t>();
  d.node_count_dev = device_node_count(t);
  d.src64 = src;
  d.uniform_mass = uniform_mass;
  d.tpos = target_pos;
  d.tslot = target_slot;
  d.f64x = fx;
  d.f64y = fy;
  d.f64z = fz;
  if (p.target_per_wave) {
    if (p.assignment == 0)
      walk64_target_kernel<0><<<grid_for(p.n_targets, kWalkWaves), kWalkThreads, 0, s>>>(p, d, out);
    else
      walk64_target_kernel<1><<<grid_for(p.n_targets, kWalkWaves), kWalkThreads, 0, s>>>(p, d, out);
    CHUI_LAUNCH_CHECK("walk64_target_kernel");
    return;
  }
  if (p.box64) {
    d.h64tab = h64tab;
    d.wnode = t.wnode.as<WalkNode>();
    launch_box64<false>(p, d, out, counters, s);
    return;
  }
  if (p.assignment == 0) launch64<0>(p, d, out, counters, s);
  else launch64<1>(p, d, out, counters, s);
}

void walk_fp64_adaptive(const Tree& t, const WalkParams& p, const double4* src, int uniform_mass,
                        const double2* gtab, const double* prev, const uint32_t* target_pos,
                        const uint32_t* target_slot, const double* fx, const double* fy, const double* fz,
                        const WalkOutputs& out, unsigned long long* counters, hipStream_t s) {
  if (!t.records64 && t.node_count > 0) throw std::logic_error("FP64 walk on a tree without FP64 records");
  if (p.n_targets == 0) return;
  WalkData d{};
  d.link = t.link.as<NodeLink>();
  d.geo64 = t.geo64.as<NodeGeo64>();
  d.mom64 = t.mom64.as<NodeMom64>();
  d.quad64 = t.quad64.as<NodeQuad64>();
  d.order = t.order.as<uint32_t>();
  d.src64 = src;
  d.uniform_mass = uniform_mass;
  d.tpos = target_pos;
  d.tslot = target_slot;
  d.f64x = fx;
  d.f64y = fy;
  d.f64z = fz;
  d.gtab = gtab;
  d.prev = prev;
  const unsigned grid = grid_for(p.n_targets, kWalkThreads);
  if (p.assignment == 0) walk64_kernel<0, false, true><<<grid, kWalkThreads, 0, s>>>(p, d, out, counters);
  else walk64_kernel<1, false, true><<<grid, kWalkThreads, 0, s>>>(p, d, out, counters);
  CHUI_LAUNCH_CHECK("walk64_kernel (adaptive)");
}

void walk_fp64_group(const Tree& t, const WalkParams& p, const GroupParams& g, const double4* src,
                     int uniform_mass, const double2* gtab, const double4* gcoef, const double* prev,
                     const uint32_t* leaf_of_pos,
                     const uint32_t* target_pos, const uint32_t* target_slot, const double* fx, const double* fy,
                     const double* fz, const WalkOutputs& out, uint32_t* fallback_pos, uint32_t* fallback_slot,
                     uint32_t* fallback_count, unsigned long long* counters, hipStream_t s) {
  if (!t.records64 && t.node_count > 0) throw std::logic_error("FP64 walk on a tree without FP64 records");
  if (p.n_targets == 0) return;
  if (g.block == 0 || g.block > 256) throw std::invalid_argument("group walk residual block must be in [1, 256]");
  WalkData d{};
  d.link = t.link.as<NodeLink>();
  d.geo64 = t.geo64.as<NodeGeo64>();
  d.mom64 = t.mom64.as<NodeMom64>();
  d.quad64 = t.quad64.as<NodeQuad64>();
  d.child_index = t.child_index.as<uint32_t>();
  d.order = t.order.as<uint32_t>();
  d.src64 = src;
  d.uniform_mass = uniform_mass;
  d.tpos = target_pos;
  d.tslot = target_slot;
  d.f64x = fx;
  d.f64y = fy;
  d.f64z = fz;
  d.gtab = gtab;
  d.gcoef = gcoef;
  d.prev = prev;
  // the table's cells up to r_cut in LDS when they fit (one more for rounding)
  GroupParams gp = g;
  const double cells = std::floor(p.rcut2 * p.inv2a2 * 64.0 * (1.0 + 1.0e-12)) + 2.0;
  gp.table_cells = cells <= kGroupCells ? static_cast<uint32_t>(cells) : 0u;
  const unsigned blocks = grid_for((static_cast<std::size_t>(p.n_targets) + g.block - 1) / g.block, kWalkWaves);
  const auto go = [&](auto kernel) {
    kernel<<<blocks, kWalkThreads, 0, s>>>(p, gp, d, leaf_of_pos, out, fallback_pos, fallback_slot, fallback_count,
                                           counters);
  };
  if (p.assignment == 0) {
    if (gp.table_cells) go(group_walk64_kernel<0, true>);
    else go(group_walk64_kernel<0, false>);
  } else {
    if (gp.table_cells) go(group_walk64_kernel<1, true>);
    else go(group_walk64_kernel<1, false>);
  }
  CHUI_LAUNCH_CHECK("group_walk64_kernel");
}

void walk_mixed_group(const Tree& t, const WalkParams& p, const GroupParams& g, const double4* src64,
                      const uint4* src32, int uniform_mass, const float4* htab, const double* prev,
                      const uint32_t* leaf_of_pos, const uint32_t* target_pos, const uint32_t* target_slot,
                      const float* fx, const float* fy, const float* fz, const WalkOutputs& out,
                      uint32_t* fallback_pos, uint32_t* fallback_slot, uint32_t* fallback_count,
                      unsigned long long* counters, hipStream_t s) {
  if (!t.records64 && t.node_count > 0) throw std::logic_error("mixed group walk on a tree without FP64 records");
  if (p.n_targets == 0) return;
  if (g.block == 0 || g.block > 256) throw std::invalid_argument("group walk residual block must be in [1, 256]");
  if (!htab || !src32 || !src64) throw std::logic_error("mixed group walk without its source lanes or pair table");
  WalkData d{};
  d.link = t.link.as<NodeLink>();
  d.geo64 = t.geo64.as<NodeGeo64>();
  d.mom64 = t.mom64.as<NodeMom64>();
  d.quad64 = t.quad64.as<NodeQuad64>();
  d.child_index = t.child_index.as<uint32_t>();
  d.order = t.order.as<uint32_t>();
  d.src64 = src64;
  d.src32 = src32;
  d.htab = htab;
  d.mom32 = t.mom32.as<NodeMom32>();
  d.quad32 = t.quad32.as<NodeQuad32>();
  d.uniform_mass = uniform_mass;
  d.tpos = target_pos;
  d.tslot = target_slot;
  d.f32x = fx;
  d.f32y = fy;
  d.f32z = fz;
  d.prev = prev;
  const unsigned blocks = grid_for((static_cast<std::size_t>(p.n_targets) + g.block - 1) / g.block, kWalkWaves);
  if (!t.mom32.ptr || !t.quad32.ptr) throw std::logic_error("mixed group walk on a tree without FP32 node records");
  auto go = [&](auto kernel) {
    kernel<<<blocks, kWalkThreads, 0, s>>>(p, g, d, leaf_of_pos, out, fallback_pos, fallback_slot, fallback_count,
                                           counters);
  };
  if (p.assignment == 0) {
    if (p.radial) go(group_walkmix_kernel<0, true>);
    else go(group_walkmix_kernel<0, false>);
  } else {
    if (p.radial) go(group_walkmix_kernel<1, true>);
    else go(group_walkmix_kernel<1, false>);
  }
  CHUI_LAUNCH_CHECK("group_walkmix_kernel");
}

void adaptive_mixed_finish(const Tree& t, const WalkParams& p, const uint4* src32, const uint32_t* pos,
                           const uint32_t* slot, uint32_t n, int identity, const double* sx, const double* sy,
                           const double* sz, const double* near64, const float* fx, const float* fy,
                           const float* fz, const WalkOutputs& out, hipStream_t s) {
  if (n == 0) return;
  if (out.near2 && !near64) throw std::logic_error("mixed adaptive finish: nearest-pair lane without its FP64 source");
  if (!identity && (!pos || !slot)) throw std::logic_error("mixed adaptive finish: target lists are null");
  WalkData d{};
  d.order = t.order.as<uint32_t>();
  d.src32 = src32;
  d.f32x = fx;
  d.f32y = fy;
  d.f32z = fz;
  const unsigned grid = grid_for(n, 256);
  if (p.assignment == 0)
    adaptive_mixed_finish_kernel<0><<<grid, 256, 0, s>>>(p, d, pos, slot, n, identity, sx, sy, sz, near64, out);
  else
    adaptive_mixed_finish_kernel<1><<<grid, 256, 0, s>>>(p, d, pos, slot, n, identity, sx, sy, sz, near64, out);
  CHUI_LAUNCH_CHECK("adaptive_mixed_finish_kernel");
}

void build_leaf_of_pos(const Tree& t, uint32_t* leaf_of_pos, hipStream_t s) {
  if (t.node_count == 0) return;
  leaf_of_pos_kernel<<<grid_for(t.node_count, 256), 256, 0, s>>>(t.link.as<NodeLink>(), t.node_count, leaf_of_pos);
  CHUI_LAUNCH_CHECK("leaf_of_pos_kernel");
}

std::vector<double> gaussian_hermite_knots() {
  // tree_pm_split_kernel.hpp:159-170: H(t_i) from the closed form (series at
  // t = 0) and step * dH/dt(t_i), t_i = i / 64, interleaved (value, slope).
  constexpr double c = 2.25675833419102514779231780624309034;  // 4 / sqrt(pi)
  constexpr double step = 64.0 / kGaussCells;
  std::vector<double> k(2 * (kGaussCells + 1));
  for (int i = 0; i <= kGaussCells; ++i) {
    const double t = static_cast<double>(i) * step;
    const double q = std::sqrt(t);
    double h, dh;
    if (i == 0) {
      h = c * (1.0 / 3.0);
      dh = -4.0 * kInvSqrtPi / 5.0;
    } else {
      const double qq = (0.5 * q) / 0.5;  // L(q) at split scale 1/2
      const double lf = std::erf(qq) - 2.0 * kInvSqrtPi * qq * std::exp(-qq * qq);
      h = lf / (t * q);
      dh = (2.0 * kInvSqrtPi * std::exp(-t) - 1.5 * h) / t;
    }
    k[2 * i] = h;
    k[2 * i + 1] = step * dh;
  }
  return k;
}

std::vector<double> gaussian_hermite_monomials(const std::vector<double>& knots) {
  // the cubic Hermite cell i on u in [0, 1) as a0 + u (a1 + u (a2 + u a3))
  std::vector<double> a(4 * kGaussCells);
  for (int i = 0; i < kGaussCells; ++i) {
    const double v0 = knots[2 * i], s0 = knots[2 * i + 1], v1 = knots[2 * i + 2], s1 = knots[2 * i + 3];
    a[4 * i] = v0;
    a[4 * i + 1] = s0;
    a[4 * i + 2] = 3.0 * (v1 - v0) - 2.0 * s0 - s1;
    a[4 * i + 3] = 2.0 * (v0 - v1) + s0 + s1;
  }
  return a;
}

void walk_fp64_vjp(const Tree& t, const WalkParams& p, const double4* src, int uniform_mass, const double4* lam,
                   const double* fx, const double* fy, const double* fz, const double* nu, const WalkOutputs& out,
                   unsigned long long* counters, const double2* h64tab, const VjpNodeTerms* nt, hipStream_t s) {
  if (!t.records64 && t.node_count > 0) throw std::logic_error("FP64 walk on a tree without FP64 records");
  if (p.n_targets == 0) return;
  WalkData d{};
  d.link = t.link.as<NodeLink>();
  d.geo64 = t.geo64.as<NodeGeo64>();
  d.mom64 = t.mom64.as<NodeMom64>();
  d.quad64 = t.quad64.as<NodeQuad64>();
  d.order = t.order.as<uint32_t>();
  d.node_count_dev = device_node_count(t);
  d.src64 = src;
  d.uniform_mass = uniform_mass;
  d.f64x = fx;
  d.f64y = fy;
  d.f64z = fz;
  d.lam64 = lam;
  d.nu64 = nu;
  if (p.quad) {
    if (!nt || !p.box64) throw std::logic_error("force VJP with accepted nodes needs the node-term buffers");
    d.vjp_node_acc = nt->node_acc;
    d.vjp_accepted = nt->accepted;
    d.vjp_accepted_count = nt->count;
    d.vjp_accepted_cap = nt->cap;
  }
  if (p.box64) {
    d.h64tab = h64tab;
    d.wnode = t.wnode.as<WalkNode>();
    launch_box64<true>(p, d, out, counters, s);
    return;
  }
  if (p.assignment == 0) launch64<0, true>(p, d, out, counters, s);
  else launch64<1, true>(p, d, out, counters, s);
}

void vjp_node_corrections(const Tree& t, const WalkParams& p, const double4* src, int uniform_mass,
                          double uniform_mass_value, const double4* lam, const VjpNodeTerms& nt, unsigned int count,
                          const WalkOutputs& out, hipStream_t s, const unsigned int* count_dev,
                          unsigned long long* fault) {
  const std::size_t n = t.n;
  if (n == 0) return;
  if (count_dev) {
    vjp_count_check_kernel<<<1, 64, 0, s>>>(count_dev, count, fault);
    CHUI_LAUNCH_CHECK("vjp_count_check_kernel");
  }
  if (count > 0) {
    radix_sort_pairs(reinterpret_cast<uint64_t*>(nt.accepted), nt.vals, reinterpret_cast<uint64_t*>(nt.accepted_alt),
                     nt.vals_alt, count, 0, 64, nt.sort_scratch, s);
    vjp_pair_fix_kernel<<<grid_for(count, 256), 256, 0, s>>>(nt.accepted, count, count_dev, t.link.as<NodeLink>(),
                                                             src, lam, uniform_mass, uniform_mass_value, p, nt.corr);
    CHUI_LAUNCH_CHECK("vjp_pair_fix_kernel");
    vjp_node_push_kernel<<<grid_for(t.node_count, 256), 256, 0, s>>>(
        static_cast<uint32_t>(t.node_count), nt.node_acc, t.link.as<NodeLink>(), t.mom64.as<NodeMom64>(), src,
        uniform_mass, uniform_mass_value, p, nt.corr);
    CHUI_LAUNCH_CHECK("vjp_node_push_kernel");
  }
  vjp_apply_kernel<<<grid_for(n, 256), 256, 0, s>>>(static_cast<uint32_t>(n), t.order.as<uint32_t>(), nt.corr,
                                                    static_cast<double*>(out.ax), static_cast<double*>(out.ay),
                                                    static_cast<double*>(out.az));
  CHUI_LAUNCH_CHECK("vjp_apply_kernel");
}

void walk_mixed(const Tree& t, const WalkParams& p, const uint4* src, int uniform_mass, const float4* htab,
                const float4* ltab, const uint32_t* target_pos, const uint32_t* target_slot, const float* fx,
                const float* fy, const float* fz, const WalkOutputs& out, unsigned long long* counters,
                hipStream_t s) {
  if (p.n_targets == 0) return;
  WalkData d{};
  d.link = t.link.as<NodeLink>();
  d.geo32 = t.geo32.as<NodeGeo32>();
  d.mom32 = t.mom32.as<NodeMom32>();
  d.quad32 = t.quad32.as<NodeQuad32>();
  d.box32 = t.box32.as<NodeBox32>();
  d.order = t.order.as<uint32_t>();
  d.src32 = src;
  d.htab = htab;
  d.ltab = ltab;
  d.wnode = t.wnode.as<WalkNode>();
  d.uniform_mass = uniform_mass;
  d.tpos = target_pos;
  d.tslot = target_slot;
  d.f32x = fx;
  d.f32y = fy;
  d.f32z = fz;
  d.node_count_dev = device_node_count(t);
  const bool cic = p.assignment == 0;
  if (p.cubic) {
    if (cic) launchmix<0, true>(p, d, out, counters, s);
    else launchmix<1, true>(p, d, out, counters, s);
  } else {
    if (cic) launchmix<0, false>(p, d, out, counters, s);
    else launchmix<1, false>(p, d, out, counters, s);
  }
}

}  // namespace chui
