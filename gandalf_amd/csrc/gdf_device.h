// Device-side helpers: smoothing kernels, periodic images, wave primitives.
//
// Kernel polynomials restate src/Headers/SmoothingKernel.h:132-408 (M4 and quintic, 3D) with
// the reference's own constants; powers are formed by multiplication.  Tabulated lookups follow
// SmoothingKernel.h:611-657 (nearest-lower entry of a 1000-entry table).
#pragma once

#include <hip/hip_runtime.h>
#include "gdf_internal.h"

namespace gdf {

// ---- fast reciprocal and square-root forms ----
// FP32: the hardware approximations (about 1 ulp), for the mixed-precision pair sums
__device__ __forceinline__ float rcp_f(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float rsq_f(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float sqrt_f(float x) { return __builtin_amdgcn_sqrtf(x); }
// FP64 1/sqrt(x) for x > 0: hardware estimate (about 2^-23 relative) refined by one third-order
// step y <- y (1 + e/2 + 3 e^2/8), e = 1 - x y^2, whose error is 5 e^3/16: rounding only
__device__ __forceinline__ double rsq_d(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x*y), y, 1.0);
  return fma(y*e, fma(0.375, e, 0.5), y);
}
// sqrt(x) for x >= 0 from it
__device__ __forceinline__ double sqrt_d(double x) { return x*rsq_d(fmax(x, 1.0e-280)); }
__device__ __forceinline__ float rsq_t(float x) { return rsq_f(x); }
__device__ __forceinline__ double rsq_t(double x) { return rsq_d(x); }
__device__ __forceinline__ float sqrt_t(float x) { return sqrt_f(x); }
__device__ __forceinline__ double sqrt_t(double x) { return sqrt_d(x); }

enum { KW0 = 0, KW1, KWOMEGA, KWZETA, KWGRAV, KWPOT, KW0S2, KWOMEGAS2, KWZETAS2 };

template <typename T> __device__ __forceinline__ const T* ktab(const KernelDesc& k);
template <> __device__ __forceinline__ const double* ktab<double>(const KernelDesc& k) { return k.tab; }
template <> __device__ __forceinline__ const float* ktab<float>(const KernelDesc& k) { return k.tabf; }

// ---- M4 (SmoothingKernel.h:132-240) ----
template <typename T> __device__ __forceinline__ T m4_w0(T norm, T s) {
  if (s < T(1)) return norm*(T(1) - T(1.5)*s*s + T(0.75)*s*s*s);
  if (s < T(2)) { T q = T(2) - s; return T(0.25)*norm*(q*q*q); }
  return T(0);
}
template <typename T> __device__ __forceinline__ T m4_w1(T norm, T s) {
  if (s < T(1)) return norm*(T(-3)*s + T(2.25)*s*s);
  if (s < T(2)) return T(-0.75)*norm*(T(2) - s)*(T(2) - s);
  return T(0);
}
template <typename T> __device__ __forceinline__ T m4_wzeta(T s) {
  const T s2 = s*s, s4 = s2*s2, s5 = s4*s;
  if (s < T(1)) return T(1.4) - T(2)*s2 + T(1.5)*s4 - T(0.6)*s5;
  if (s < T(2)) return T(1.6) - T(4)*s2 + T(4)*s2*s - T(1.5)*s4 + T(0.2)*s5;
  return T(0);
}
template <typename T> __device__ __forceinline__ T m4_wgrav(T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2;
  if (s < T(1)) return T(1.333333333333333333333)*s - T(1.2)*s3 + T(0.5)*s4;
  if (s < T(2))
    return T(2.6666666666666666667)*s - T(3)*s2 + T(1.2)*s3 - T(0.166666666666666666667)*s4 -
           T(0.06666666666666666667)/s2;
  return T(1)/s2;
}
template <typename T> __device__ __forceinline__ T m4_wpot(T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2, s5 = s4*s;
  if (s < T(1)) return T(1.4) - T(0.666666666666666666666666)*s2 + T(0.3)*s4 - T(0.1)*s5;
  if (s < T(2))
    return T(-1)/(T(15)*s) + T(1.6) - T(1.33333333333333333333333333)*s2 + s3 - T(0.3)*s4 +
           T(1.0/30.0)*s5;
  return T(1)/s;
}

// ---- quintic (SmoothingKernel.h:282-408) ----
template <typename T> __device__ __forceinline__ T q_w0(T norm, T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2, s5 = s4*s;
  if (s < T(1)) return norm*(T(66) - T(60)*s2 + T(30)*s4 - T(10)*s5);
  if (s < T(2)) return norm*(T(51) + T(75)*s - T(210)*s2 + T(150)*s3 - T(45)*s4 + T(5)*s5);
  if (s < T(3)) return norm*(T(243) - T(405)*s + T(270)*s2 - T(90)*s3 + T(15)*s4 - s5);
  return T(0);
}
template <typename T> __device__ __forceinline__ T q_w1(T norm, T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2;
  if (s < T(1)) return norm*(T(-120)*s + T(120)*s3 - T(50)*s4);
  if (s < T(2)) return norm*(T(75) - T(420)*s + T(450)*s2 - T(180)*s3 + T(25)*s4);
  if (s < T(3)) return norm*(T(-405) + T(540)*s - T(270)*s2 + T(60)*s3 - T(5)*s4);
  return T(0);
}
template <typename T> __device__ __forceinline__ T q_wzeta(T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2, s5 = s4*s, s6 = s3*s3, s7 = s6*s;
  if (s < T(1)) return T(33)*s2 - T(15)*s4 + T(5)*s6 - T(1.42857142857)*s7 - T(34.14285714);
  if (s < T(2))
    return T(25.5)*s2 + T(25)*s3 - T(52.5)*s4 + T(30)*s5 - T(7.5)*s6 + T(0.7142857143)*s7 -
           T(33.785714286);
  if (s < T(3))
    return T(121.5)*s2 - T(135)*s3 + T(67.5)*s4 - T(18)*s5 + T(2.5)*s6 - T(0.142857143)*s7 -
           T(52.07142857);
  return T(0);
}
template <typename T> __device__ __forceinline__ T q_wgrav(T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2, s5 = s4*s, s6 = s3*s3;
  const T c = T(12.0/359.0);
  if (s < T(1)) return c*(T(22)*s - T(12)*s3 + T(30.0/7.0)*s5 - T(5.0/4.0)*s6);
  if (s < T(2))
    return c*(T(17)*s + T(75.0/4.0)*s2 - T(42)*s3 + T(25)*s4 - T(45.0/7.0)*s5 +
              T(5.0/8.0)*s6 + T(5.0/56.0)/s2);
  if (s < T(3))
    return c*(T(81)*s - T(405.0/4.0)*s2 + T(54)*s3 - T(15)*s4 + T(15.0/7.0)*s5 -
              T(1.0/8.0)*s6 - T(507.0/56.0)/s2);
  return T(1)/s2;
}
template <typename T> __device__ __forceinline__ T q_wpot(T s) {
  const T s2 = s*s, s3 = s2*s, s4 = s2*s2, s5 = s4*s, s6 = s3*s3, s7 = s6*s;
  const T c = T(12.0/359.0);
  if (s < T(1))
    return c*(T(-11)*s2 + T(3)*s4 - T(5.0/7.0)*s6 + T(5.0/28.0)*s7 + T(478.0/14.0));
  if (s < T(2))
    return c*(T(-17.0/2.0)*s2 - T(25.0/4.0)*s3 + T(21.0/2.0)*s4 - T(5)*s5 + T(15.0/14.0)*s6 -
              T(5.0/56.0)*s7 + T(473.0/14.0) + T(5.0/56.0)/s);
  if (s < T(3))
    return c*(T(-81.0/2.0)*s2 + T(135.0/4.0)*s3 - T(27.0/2.0)*s4 + T(3)*s5 - T(5.0/14.0)*s6 +
              T(1.0/56.0)*s7 + T(729.0/14.0) - T(507.0/56.0)/s);
  return T(1)/s;
}

// ---- dispatch; s is r/h (or (r/h)^2 for the _s2 forms) ----
template <typename T> __device__ __forceinline__ T tab_lin(const KernelDesc& k, int w, T s) {
  if (s >= T(k.range)) return T(0);
  return ktab<T>(k)[w*k.res + (int) (s*T(k.resinv))];
}
template <typename T> __device__ __forceinline__ T kw0(const KernelDesc& k, T s) {
  if (k.tabulated) return tab_lin<T>(k, KW0, s);
  return k.type == 0 ? m4_w0<T>(T(k.norm), s) : q_w0<T>(T(k.norm), s);
}
// ---- branch-free analytic forms for the pair loops ----
// W and dW/ds as truncated powers, i.e. the reference's piecewise polynomials summed without the
// cancellation of their expanded form: M4 W = (norm/4)[(2-s)^3_+ - 4(1-s)^3_+], quintic
// W = norm[(3-s)^5_+ - 6(2-s)^5_+ + 15(1-s)^5_+]; womega = -3 w0 - s w1 exactly for both.
// With W = norm sum_k c_k (a_k - s)^n_+ (M4: n = 3, a = 2, 1, c = 1, -4; quintic: n = 5,
// a = 3, 2, 1, c = 1, -6, 15), the enclosed mass M(s) and the outer potential integral
// P(s) = 4 pi int_s^inf u W du are polynomials in x_k = (a_k - s)_+:
//   M = 1 - sum_k c_k x_k^(n+1) (a_k^2/(n+1) - 2 a_k x_k/(n+2) + x_k^2/(n+3)) * C,
//   P = sum_k c_k x_k^(n+1) (a_k/(n+1) - x_k/(n+2)) * C      (C = 1 for M4, 1/30 quintic),
// and wgrav = M/s^2, wpot = M/s + P, wzeta = wpot - s wgrav = P.  These are the reference's
// piecewise polynomials (SmoothingKernel.h:132-408) summed without branches; the reference's
// quintic wgrav and wpot carry 360/359 inside the kernel (its 12/359 in place of 1/30) and its
// quintic wzeta is -30 P, both kept.  Below s = 1 the mass comes from the inner polynomial,
// which avoids the cancellation of 1 - (...) at small s.
template <typename T> __device__ __forceinline__ T tpos(T x) { return x > T(0) ? x : T(0); }

template <typename T> __device__ __forceinline__ T kw1(const KernelDesc& k, T s) {
  if (k.tabulated) return tab_lin<T>(k, KW1, s);
  const T norm = T(k.norm);
  if (k.type == 0) {
    const T A = tpos(T(2) - s), B = tpos(T(1) - s);
    return T(-0.75)*norm*(A*A - T(4)*(B*B));
  }
  const T A = tpos(T(3) - s), B = tpos(T(2) - s), C = tpos(T(1) - s);
  const T A2 = A*A, B2 = B*B, C2 = C*C;
  return T(-5)*norm*(A2*A2 - T(6)*(B2*B2) + T(15)*(C2*C2));
}

template <typename T> __device__ __forceinline__ T kwgrav(const KernelDesc& k, T s) {
  if (k.tabulated) {
    if (s >= T(k.range)) return T(1)/(s*s);
    return ktab<T>(k)[KWGRAV*k.res + (int) (s*T(k.resinv))];
  }
  return k.type == 0 ? m4_wgrav<T>(s) : q_wgrav<T>(s);
}
template <typename T> __device__ __forceinline__ T kwpot(const KernelDesc& k, T s) {
  if (k.tabulated) {
    if (s >= T(k.range)) return T(1)/s;
    return ktab<T>(k)[KWPOT*k.res + (int) (s*T(k.resinv))];
  }
  return k.type == 0 ? m4_wpot<T>(s) : q_wpot<T>(s);
}
// ---- sums of the h-rho pass ----
// KT: 0 M4, 1 quintic, 2 tabulated; the sums of the density triple at s^2 (GradhSph.cpp:197-204).
// The analytic kernels in truncated powers, their constant factors taken out of the sums: with w0, w1
// and P without the norm, womega = -3 w0 - s w1 makes sum(m womega) two sums, and wzeta is P (M4)
// or -30 P (quintic).  The reference's quintic wzeta polynomials are rounded to ten digits: their
// differences from -30 P, a constant and an s^7 term per segment, are added in FP64.
// sum(m w0), which decides when the iteration stops, is FP64 in both precisions, at 2 % of the mixed
// pass: the relative error of rho over 64 bits is 5.1e-8 (M4, 262144 particles) and 6.7e-8 (quintic,
// 100003), against 5.9e-8 and 7.7e-8 with each term's FP32 norm and FP32 sums.
template <typename T, int KT> struct DensSums {
  double r = 0.0;
  T o = T(0), z = T(0);
  __device__ __forceinline__ void add(const KernelDesc& k, T ssqd, T m) {
    if (KT == 2) {
      if (ssqd >= T(k.rangesqd)) return;
      const int i = (int) (ssqd*T(k.resinvsqd));
      const T* t = ktab<T>(k);
      r += (double) (m*t[KW0S2*k.res + i]); o += m*t[KWOMEGAS2*k.res + i]; z += m*t[KWZETAS2*k.res + i];
      return;
    }
    const T s = sqrt_t(ssqd);
    const T c = tpos(T(1) - s), b = tpos(T(2) - s);
    const T c2 = c*c, b2 = b*b;
    if (KT == 0) {
      const T w1 = b2 - T(4)*c2;                        // -4/3 w1
      const T c4 = c2*c2, b4 = b2*b2;
      r += (double) (m*(b*b2 - T(4)*(c*c2)));                      // 4 w0
      o += (m*s)*w1;
      z += m*(b4*(T(0.5) - T(0.2)*b) - T(4)*c4*(T(0.25) - T(0.2)*c));
    } else {
      const T a = tpos(T(3) - s);
      const T a2 = a*a;
      const T a4 = a2*a2, b4 = T(-6)*(b2*b2), c4 = T(15)*(c2*c2);
      r += (double) (m*(a4*a + b4*b + c4*c));                      // w0
      o += (m*s)*(a4 + b4 + c4);                        // -w1/5
      T p = (a4*a2)*(T(0.5) - T(1.0/7.0)*a) + (b4*b2)*(T(1.0/3.0) - T(1.0/7.0)*b) +
            (c4*c2)*(T(1.0/6.0) - T(1.0/7.0)*c);        // 30 P
      if (sizeof(T) == 8) {
        const double d0 = s < T(1) ? 34.14285714 - 239.0/7.0
                                   : s < T(2) ? 33.785714286 - 236.5/7.0
                                              : 52.07142857 - 364.5/7.0;
        const double d7 = s < T(1) ? 1.42857142857 - 10.0/7.0
                                   : s < T(2) ? 5.0/7.0 - 0.7142857143 : 0.142857143 - 1.0/7.0;
        const T s2 = s*s;
        const T d = T(d0) + T(d7)*((s2*s2)*(s2*s));
        p += s < T(3) ? d : T(0);
      }
      z += m*p;
    }
  }
  // sum(m w0), sum(m womega), sum(m wzeta) of these sums
  __device__ __forceinline__ static void finish(const KernelDesc& k, double& r_, double& o_,
                                                double& z_) {
    if (KT == 2) return;
    const double norm = (double) (T) k.norm;      // the norm of the precision's own kernel
    if (KT == 0) {
      r_ *= 0.25*norm;
      o_ = -3.0*r_ + 0.75*norm*o_;
    } else {
      r_ *= norm;
      o_ = -3.0*r_ + 5.0*norm*o_;
      z_ = -z_;
    }
  }
};

// ---- kernels of the hydro pairs ----
// KT as DensSums.  set(s): w1 without its constant factor (w1_factor).  grav: the enclosed mass M
// and outer potential integral P above, with the reference's 360/359 (quintic, inside the
// kernel): wgrav = M/s^2, wpot = M/s + P.  The truncated-power forms are the reference's
// piecewise polynomials exactly, so the FP64 path takes them too: no branches, and the terms of
// the force and the potential share their powers.  (Tabulated kernels: M = s^2 wgrav, and P is
// what then remains of wpot.)
template <typename T, int KT> struct HydroKern {
  T w1, s, a, b, c, a2, b2, c2, a4, b4, c4;
  __device__ __forceinline__ static double w1_factor(const KernelDesc& k) {
    return KT == 0 ? -0.75*k.norm : KT == 1 ? -5.0*k.norm : 1.0;
  }
  __device__ __forceinline__ void set(const KernelDesc& k, T s_) {
    s = s_;
    if (KT == 2) { w1 = tab_lin<T>(k, KW1, s); return; }
    b = tpos(T(2) - s); c = tpos(T(1) - s);
    b2 = b*b; c2 = c*c;
    if (KT == 0) { w1 = b2 - T(4)*c2; return; }
    a = tpos(T(3) - s);
    a2 = a*a;
    a4 = a2*a2; b4 = T(-6)*(b2*b2); c4 = T(15)*(c2*c2);
    w1 = a4 + b4 + c4;
  }
  __device__ __forceinline__ void grav(const KernelDesc& k, T& M, T& P) const {
    if (KT == 2) {
      M = kwgrav<T>(k, s)*(s*s);
      P = s > T(0) ? kwpot<T>(k, s) - M/s : kwpot<T>(k, s);
    } else if (KT == 0) {
      const T x = b2*b2, y = T(-4)*(c2*c2);
      const T D = x*(T(1) + b*(b*T(1.0/6.0) - T(0.8))) + y*(T(0.25) + c*(c*T(1.0/6.0) - T(0.4)));
      P = x*(T(0.5) - T(0.2)*b) + y*(T(0.25) - T(0.2)*c);
      const T s2 = s*s;
      const T in = (s2*s)*(T(4.0/3.0) + s2*(T(0.5)*s - T(1.2)));
      M = s < T(1) ? in : T(1) - D;
    } else {
      const T x = a4*a2, y = b4*b2, z = c4*c2;
      const T D = x*(T(1.5) + a*(T(0.125)*a - T(6.0/7.0))) +
                  y*(T(2.0/3.0) + b*(T(0.125)*b - T(4.0/7.0))) +
                  z*(T(1.0/6.0) + c*(T(0.125)*c - T(2.0/7.0)));
      const T f = T(12.0/359.0);
      P = f*(x*(T(0.5) - T(1.0/7.0)*a) + y*(T(1.0/3.0) - T(1.0/7.0)*b) +
             z*(T(1.0/6.0) - T(1.0/7.0)*c));
      const T s2 = s*s;
      const T in = (f*(s2*s))*(T(22) + s2*(T(-12) + s2*(T(30.0/7.0) - T(1.25)*s)));
      M = s < T(1) ? in : (s < T(3) ? T(360.0/359.0) : T(1)) - f*D;
    }
  }
};

// wzeta at s^2 alone (the stars' zeta terms, GradhSph.cpp:289-303)
__device__ __forceinline__ double kwzeta_s2(const KernelDesc& k, double s2) {
  if (k.tabulated) {
    if (s2 >= k.rangesqd) return 0.0;
    return k.tab[KWZETAS2*k.res + (int) (s2*k.resinvsqd)];
  }
  const double s = sqrt(s2);
  return k.type == 0 ? m4_wzeta<double>(s) : q_wzeta<double>(s);
}

// ---- periodic nearest image (GhostNeighbours.hpp:119-138) ----
template <typename T>
__device__ __forceinline__ void nearest_image(const PhysParams& p, T& dx, T& dy, T& dz) {
  if (!p.periodic) return;
  if (dx > T(p.boxhalf[0])) dx -= T(p.boxsize[0]); else if (dx < -T(p.boxhalf[0])) dx += T(p.boxsize[0]);
  if (dy > T(p.boxhalf[1])) dy -= T(p.boxsize[1]); else if (dy < -T(p.boxhalf[1])) dy += T(p.boxsize[1]);
  if (dz > T(p.boxhalf[2])) dz -= T(p.boxsize[2]); else if (dz < -T(p.boxhalf[2])) dz += T(p.boxsize[2]);
}

// Ewald::CalculatePeriodicCorrection (src/Common/Ewald.cpp:500-650) for a fully periodic box:
// the periodic correction of mass m at separation d = r_source - r_target.  A separation outside
// the half box first swaps its Newtonian term for that of its nearest image (the reference's
// repair of a non-nearest separation); the acceleration is trilinear in the table, the
// potential the value at the lower corner node, signs restored per axis.
template <typename T>
__device__ __forceinline__ void ewald_corr(const PhysParams& p, T dx, T dy, T dz, T m, T& ax,
                                           T& ay, T& az, T& pot) {
  T d[3] = {dx, dy, dz};
  const T half[3] = {T(p.boxhalf[0]), T(p.boxhalf[1]), T(p.boxhalf[2])};
  if (fabs(d[0]) > half[0] || fabs(d[1]) > half[1] || fabs(d[2]) > half[2]) {
    T inv = T(1)/sqrt(d[0]*d[0] + d[1]*d[1] + d[2]*d[2] + T(1.0e-20));
    T inv3 = inv*inv*inv;
    ax -= m*d[0]*inv3; ay -= m*d[1]*inv3; az -= m*d[2]*inv3;
    pot -= m*inv;
    for (int k = 0; k < 3; k++) {
      if (d[k] > half[k]) d[k] -= T(2)*half[k];
      else if (d[k] < -half[k]) d[k] += T(2)*half[k];
    }
    inv = T(1)/sqrt(d[0]*d[0] + d[1]*d[1] + d[2]*d[2] + T(1.0e-20));
    inv3 = inv*inv*inv;
    ax += m*d[0]*inv3; ay += m*d[1]*inv3; az += m*d[2]*inv3;
    pot += m*inv;
  }
  int il[3];
  T w[3];
  for (int k = 0; k < 3; k++) {
    const T b = T(p.edI[k])*fabs(d[k]);
    // |d| <= L/2 keeps b in [0, eng - 2] already; the clamp keeps any input in the table
    il[k] = max(0, min((int) b, p.eng[k] - 2));
    w[k] = b - (T) il[k];
  }
  const int n0 = p.eng[0], n01 = p.eng[0]*p.eng[1];
  const int b0 = il[0] + il[1]*n0 + il[2]*n01;
  T g0 = T(0), g1 = T(0), g2 = T(0), p0;
  auto corner = [&](int off, T wt) {
    if (sizeof(T) == 4) {
      const float4 t = p.etabf[b0 + off];
      g0 += wt*(T) t.y; g1 += wt*(T) t.z; g2 += wt*(T) t.w;
    } else {
      const double4 t = p.etab[b0 + off];
      g0 += wt*(T) t.y; g1 += wt*(T) t.z; g2 += wt*(T) t.w;
    }
  };
  const T u0 = T(1) - w[0], u1 = T(1) - w[1], u2 = T(1) - w[2];
  corner(0, u2*u1*u0);             corner(1, u2*u1*w[0]);
  corner(n0, u2*w[1]*u0);          corner(n0 + 1, u2*w[1]*w[0]);
  corner(n01, w[2]*u1*u0);         corner(n01 + 1, w[2]*u1*w[0]);
  corner(n01 + n0, w[2]*w[1]*u0);  corner(n01 + n0 + 1, w[2]*w[1]*w[0]);
  if (sizeof(T) == 4) p0 = (T) p.etabf[b0].x;
  else p0 = (T) p.etab[b0].x;
  pot += m*p0;
  const T sx = d[0] > T(0) ? T(1) : (d[0] < T(0) ? T(-1) : T(0));
  const T sy = d[1] > T(0) ? T(1) : (d[1] < T(0) ? T(-1) : T(0));
  const T sz = d[2] > T(0) ? T(1) : (d[2] < T(0) ? T(-1) : T(0));
  ax += m*g0*sx; ay += m*g1*sy; az += m*g2*sz;
}

// squared distance with the reference's operation order and no fused multiply-add, so
// neighbour-set membership is decided exactly as the oracle decides it.  (HIP's __dadd_rn and
// __dmul_rn are plain operators that the compiler may still contract; the pragma may not.)
__device__ __forceinline__ double dot3_rn(double a, double b, double c) {
#pragma clang fp contract(off)
  return a*a + b*b + c*c;
}
__device__ __forceinline__ double range2_rn(double krsqd, double h) {
#pragma clang fp contract(off)
  return krsqd*h*h;
}

// FP32 squared distance of the mixed path with a fixed operation order (explicit fused
// multiply-adds): the scatter-gather walk and the gravity walk both classify a pair with it,
// so each pair lands in exactly one of the two sums
__device__ __forceinline__ float dot3_f(float a, float b, float c) {
  return fmaf(c, c, fmaf(b, b, a*a));
}

__device__ __forceinline__ float dot3_t(float a, float b, float c) { return dot3_f(a, b, c); }
__device__ __forceinline__ double dot3_t(double a, double b, double c) { return dot3_rn(a, b, c); }

// Kernel-range box test of the gravity walk with a relative slack: a node whose box comes within
// (1 + slack) k max(h) of the group is resolved to particles, so no pair of the scatter-gather
// set (decided per pair in FP64 or FP32) can end up inside an accepted multipole.
constexpr double kGravNeibSlack = 1.0 + 1.0e-4;

// ---- wave primitives (wave64) ----
__device__ __forceinline__ int lane_id() { return __lane_id(); }
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned) (mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned) mask, 0));
}
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = __lane_id();
  #pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    int o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}
__device__ __forceinline__ int wave_max_int(int v) {
  #pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = max(v, __shfl_xor(v, d, 64));
  return v;
}
__device__ __forceinline__ double wave_max_d(double v) {
  #pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmax(v, __shfl_xor(v, d, 64));
  return v;
}
__device__ __forceinline__ int wave_bcast(int v, int src) { return __shfl(v, src, 64); }
// sum over the wavefront, one atomic add by lane 0; every lane of the wave must take part
__device__ __forceinline__ void wave_add_ll(long long* dst, long long v) {
  #pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if (__lane_id() == 0 && v != 0) atomicAdd((unsigned long long*) dst, (unsigned long long) v);
}

// The same over a whole workgroup (blockDim.x a multiple of 64, at most 1024; every thread
// calls it): one atomic per workgroup.  Atomics on one address from every wavefront of a
// million-particle pass serialise at the memory side (about 0.2 ms for 16384 of them).
__device__ __forceinline__ void block_add_ll(long long* dst, long long v) {
  __shared__ long long part[16];
  #pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if (__lane_id() == 0) part[threadIdx.x/64] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    long long t = 0;
    for (int w = 0; w < (int) blockDim.x/64; w++) t += part[w];
    if (t != 0) atomicAdd((unsigned long long*) dst, (unsigned long long) t);
  }
}

// GradhSph::ComputeThermalProperties (GradhSph.cpp:335-347) with the adiabatic
// (AdiabaticEOS.cpp), isothermal (IsothermalEOS.cpp) and barotropic (BarotropicEOS.cpp) closures:
// u (replaced for the last two), sound speed and pressure from rho and u
__device__ __forceinline__ void eos_state(const PhysParams& p, double rho, double& u,
                                          double& snd, double& press) {
  if (p.eos == 1) { u = p.temp0/p.gammam1/p.mu_bar; snd = sqrt(p.gammam1*u); }
  else if (p.eos == 2) {
    u = p.temp0*(1.0 + pow(rho*p.invrho_bary, p.gammam1))/p.gammam1/p.mu_bar;
    snd = sqrt(p.gammam1*u);
  } else snd = sqrt(p.gamma*p.gammam1*u);
  press = p.gammam1*rho*u;
}

// MI355X has 8 XCDs, each with its own L2, and workgroups are dispatched to them round-robin by
// workgroup id.  Work that neighbours other work in memory (Morton-ordered particles, walk
// groups) is therefore remapped so each XCD takes one contiguous eighth.
constexpr int kXcds = 8;

// logical block of physical block b in a grid of nb: XCD x = b % 8 gets the x-th contiguous
// run of blocks (a bijection for any nb)
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int x = b % kXcds, k = b / kXcds, q = nb / kXcds, r = nb % kXcds;
  return x*q + min(x, r) + k;
}

// ---- a group's targets on the lanes ----
// The members of a walk group that take part (the set bits of a mask, at least one) on the lanes of
// a wavefront: target `slot` on the lanes slot, slot + span, ..., which share its sources, copy k of
// them taking every copies-th from the k-th on, and add their sums (over_copies) at the end.  Groups
// hold 44 members on average and a sparse block step's few active ones; the lanes that had no target
// stood idle.  Steps of a million-particle cloud with a few per cent of its particles active: hydro
// pass 172 -> 70 us, gravity walk 251 -> 141, h-rho pass 72 -> 41; with a third, 1083 -> 588, 839 ->
// 587, 341 -> 259.
struct TargetLanes {
  int span, copies, slot, copy, member;    // span: a power of two, at least the number of targets
  bool has;
  // alone: no copies, whatever the number of targets
  __device__ __forceinline__ explicit TargetLanes(unsigned long long on, bool alone = false) {
    const int n = __popcll(on), lane = lane_id();
    span = alone ? kWave : n <= 2 ? 2 : 1 << (32 - __clz(n - 1));
    copies = kWave/span;
    slot = lane & (span - 1);
    copy = lane/span;
    has = slot < n;
    // the member of the slot-th set bit
    int s = slot;
    member = 0;
    unsigned long long m = on;
    #pragma unroll
    for (int w = 32; w > 0; w >>= 1) {
      const int c = __popcll(m & ((1ULL << w) - 1));
      if (s >= c) { s -= c; m >>= w; member += w; }
    }
  }
  // this copy's share of a word of 32 sources
  __device__ __forceinline__ unsigned share() const {
    const unsigned every = copies == 1 ? 0xffffffffu : copies == 2 ? 0x55555555u :
                           copies == 4 ? 0x11111111u : copies == 8 ? 0x01010101u :
                           copies == 16 ? 0x00010001u : 1u;
    return every << copy;
  }
  template <class T> __device__ __forceinline__ T over_copies(T v) const {
    for (int o = span; o < kWave; o <<= 1) v += __shfl_xor(v, o, kWave);
    return v;
  }
};

// ---- tree walks ----
// A walk's node stack: the first kLdsStack entries live in LDS, deeper ones in the wave's
// global stack region (kStackCap entries), so the common case never waits on global memory.
constexpr int kLdsStack = 512;

__device__ __forceinline__ int stack_get(const int* lstk, const int* gstk, int s) {
  return s < kLdsStack ? lstk[s] : gstk[s - kLdsStack];
}
__device__ __forceinline__ void stack_put(int* lstk, int* gstk, int s, int v) {
  if (s < kLdsStack) lstk[s] = v;
  else gstk[s - kLdsStack] = v;
}

// particle range and children of a node (unified index: leaf l is node N - 1 + l), loaded
// together with the node's box so that a walk step waits on global memory once
struct NodeLinks {
  int first, count, left, right;
};
__device__ __forceinline__ void load_links(int n, int N, const int4* __restrict__ lnk,
                                           NodeLinks& l) {
  if (n >= N - 1) {
    l.first = n - (N - 1); l.count = 1; l.left = -1; l.right = -1;
  } else {
    const int4 k = lnk[n];           // (first, last, left, right)
    l.first = k.x; l.count = k.y - k.x + 1; l.left = k.z; l.right = k.w;
  }
}

// The walk groups of a persistent workgroup: nq entries (all groups, or a compacted list of the
// groups with targets) in eight contiguous ranges, one an XCD, whose workgroups take every
// (their number)-th entry of it.  Neighbouring groups are walked at the same time and share the
// XCD's L2.  (Fetching each entry from a counter a range, and on from the other ranges', took an
// atomic an entry and eight a workgroup on one line: 0.1 ms of a walk of 2048 groups.)
struct GroupQueue {
  int first, end, step;
};
__device__ __forceinline__ GroupQueue group_queue(int nq) {
  const int x = blockIdx.x % kXcds, nb = gridDim.x;
  const int q = nq/kXcds, r = nq % kXcds, lo = x*q + min(x, r);
  return {lo + (int) blockIdx.x/kXcds, lo + q + (x < r), nb/kXcds + (x < nb % kXcds)};
}

// The same ranges handed out entry by entry, for walks whose groups cost unequally: one counter a
// range, kQueueStride apart (the line is the unit that atomics are serialised by), and from the
// other ranges once a workgroup's own is empty.  Called by one lane; returns nq at the end.
constexpr int kQueueStride = 32;
__device__ __forceinline__ int group_fetch(int* counters, int nq, int& range) {
  const int q = nq/kXcds, r = nq % kXcds;
  for (int t = 0; t < kXcds; t++) {
    const int x = (range + t) % kXcds;
    const int k = atomicAdd(&counters[x*kQueueStride], 1);
    if (k < q + (x < r)) { range = x; return x*q + min(x, r) + k; }
  }
  return nq;
}

// Kahan-compensated accumulator for the mixed-precision pair sums
struct KahanF {
  float s = 0.f, c = 0.f;
  __device__ __forceinline__ void add(float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
};

}  // namespace gdf
