// Device-side superelastic SMA law (Alya solidz stress model 160) for gfx950.
//
// Reference: sld_stress_model_160.f90 (compute_kirchoff_stress :212-500,
// eval_loading_function :513-537, eval_beta :539-556 with beta forced to 1,
// INV2x2 :558-573), dsyevq3.f90:22-137 + dsytrd3.f90:22-109 (Kopp's
// Householder + QL), eigsrt.f90:19-48 (descending selection sort).
//
// The strain comes from the series artanh(Z) (hencky_fp64, hencky_fp32) where it
// reaches, else from one of two spectral front ends; all feed one FP64 return
// map:
//   * spectral_fp64: b = F F^T, Kopp QL on b, sqrt/pow/log exactly as the
//     reference sequences them (point-wise law, parity <= 1e-10);
//   * spectral_fp32: the same QL on b - I = H + H^T + H H^T (H = F - I) in
//     FP32, with e_i = log1p(mu_i)/2 - theta/3.  Working on b - I keeps the
//     small strains at full FP32 relative precision (FP32 kinematics mode).
// The loading functions, branch flags and the 2x2 Newton on (dh_AS, dh_SA)
// always run in FP64, with FMA contraction off so that every branch decision
// sees the same rounding as the reference.
//
// All loops over the 3 eigenpairs are written with compile-time indices so
// that the state stays in VGPRs (no dynamically indexed private arrays).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sma {

constexpr uint32_t FLAG_KF_AS = 0x01u;
constexpr uint32_t FLAG_KF_SA = 0x02u;
constexpr uint32_t FLAG_NEWTON_FAIL = 0x04u;
constexpr uint32_t FLAG_EIGEN_FAIL = 0x08u;
constexpr uint32_t FLAG_DETF_NONPOS = 0x10u;
constexpr uint32_t FLAG_SURR_USED = 0x20u;
constexpr uint32_t FLAG_SURR_FALLBACK = 0x40u;
constexpr uint32_t FLAG_BAD_INPUT = 0x80u;
constexpr int FLAG_ITER_SHIFT = 8;

// Material constants derived once per point from props(18) and E
// (compute_kirchoff_stress :263-289).
struct Mat {
  double K, G, eL, alfa, Rf_AS, Rs_AS, Rf_SA, Rs_SA, G_1, C_AS, C_SA;
};

// Bulk and shear modulus from Young's modulus E and props(2) = nu.
__host__ __device__ __forceinline__ void elastic_moduli(const double* __restrict__ p, double E,
                                                       double& K, double& G) {
#pragma clang fp contract(off)
  const double v = p[1];
  K = E / (3.0 - 6.0 * v);
  G = E / (2.0 + 2.0 * v);
}

// Material constants with K, G given (precomputed per element).
__host__ __device__ __forceinline__ Mat make_mat_kg(const double* __restrict__ p, double K, double G) {
#pragma clang fp contract(off)
  Mat m;
  m.eL = p[2];
  m.alfa = p[14];
  m.C_AS = p[5];
  m.C_SA = p[11];
  m.K = K;
  m.G = G;
  double aux = sqrt(2.0 / 3.0) + m.alfa;
  m.Rf_AS = p[4] * aux + p[5] * p[6];
  m.Rs_AS = p[3] * aux + p[5] * p[7];
  m.Rf_SA = p[10] * aux + p[11] * p[12];
  m.Rs_SA = p[9] * aux + p[11] * p[13];
  m.G_1 = (2.0 * m.G + 9.0 * (m.alfa * m.alfa) * m.K) * m.eL;
  return m;
}

// Constants of make_mat_kg that depend on props(18) alone, per material (the
// same operations): c[0..7] = eL, alfa, C_AS, C_SA, Rf_AS, Rs_AS, Rf_SA, Rs_SA.
__host__ __device__ __forceinline__ void law_constants(const double* __restrict__ p, double* c) {
  const Mat m = make_mat_kg(p, 0.0, 0.0);
  c[0] = m.eL;
  c[1] = m.alfa;
  c[2] = m.C_AS;
  c[3] = m.C_SA;
  c[4] = m.Rf_AS;
  c[5] = m.Rs_AS;
  c[6] = m.Rf_SA;
  c[7] = m.Rs_SA;
}

// make_mat_kg from c = law_constants(p).
__host__ __device__ __forceinline__ Mat make_mat_const(const double* c, double K, double G) {
#pragma clang fp contract(off)
  Mat m;
  m.eL = c[0];
  m.alfa = c[1];
  m.C_AS = c[2];
  m.C_SA = c[3];
  m.K = K;
  m.G = G;
  m.Rf_AS = c[4];
  m.Rs_AS = c[5];
  m.Rf_SA = c[6];
  m.Rs_SA = c[7];
  m.G_1 = (2.0 * m.G + 9.0 * (m.alfa * m.alfa) * m.K) * m.eL;
  return m;
}

__host__ __device__ __forceinline__ Mat make_mat(const double* __restrict__ p, double E) {
  double K, G;
  elastic_moduli(p, E, K, G);
  return make_mat_kg(p, K, G);
}

// 1/x: the hardware reciprocal (1 ulp) on the device, for FP32-only paths.
__host__ __device__ __forceinline__ float fast_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.0f / x;
#endif
}

// 1/x in FP64 for the element step: the hardware estimate refined by two
// Newton steps, within 1 ulp (the IEEE division: 0.5) in 5 instructions
// against its 11.  0, infinities and an x whose reciprocal overflows give NaN
// (0 times infinity in the steps), which the step's health check treats as it
// does infinity.  Not for values that a caller is handed (inv3's EXACT).
__host__ __device__ __forceinline__ double rcp64(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
#else
  return 1.0 / x;
#endif
}

// sqrt(s) and 1/sqrt(s) of s >= 0 together: the hardware estimate refined by
// two Newton steps (1 ulp), the root corrected once more by its residual;
// 12 instructions against ~25 for an IEEE root and a division by it.  Below
// 1e-290 (where the refinement would lose digits) s is scaled first; the
// reciprocal of 0 is 0.
__host__ __device__ __forceinline__ void sqrt_rsqrt64(double s, double& root, double& inv) {
  const bool small = !(s >= 1e-290);
  double t = s;
  if (small) t = s * 0x1p600;
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rsq(t);
#else
  double y = 1.0 / sqrt(t);
#endif
  y = fma(0.5 * y, fma(-t * y, y, 1.0), y);
  y = fma(0.5 * y, fma(-t * y, y, 1.0), y);
  const double r = t * y;
  root = fma(fma(-r, r, t), 0.5 * y, r);
  inv = y;
  if (small) {
    root = s == 0.0 ? 0.0 : root * 0x1p-300;
    inv = s > 0.0 ? y * 0x1p300 : 0.0;
  }
}

// J^(-2/3) in FP64 (the neo-Hookean law's volumetric factor).  On the
// device: y = J^(-1/3) from the hardware single-precision log2 and exp2
// (relative error ~3e-7), refined by two Newton steps on y^-3 = J,
// y <- y + y (1 - J y^3) / 3 (error e -> -2 e^2: 3e-7 -> 2e-13 -> rounding),
// then squared: within 2 ulps of the exact value (pow: 1), in ~20
// instructions against pow's ~170.  J outside [2^-100, 2^100] is first scaled
// by a power of 8 and the result by the power of 4 (both exact); a J that is
// not positive and finite gives what pow gives.  (A call of pow there put its
// 38 constants into vector registers at the start of every wave: 6% of the
// neo-Hookean element kernel's instructions, 28 of its 108 registers.)
__host__ __device__ __forceinline__ double pow_m23(double J) {
  int k = 0;
  if (!(J >= 0x1p-100 && J <= 0x1p100)) {
    if (!(J > 0.0 && J < __builtin_inf()))
      return J == 0.0 ? __builtin_inf() : J == __builtin_inf() ? 0.0 : __builtin_nan("");
#if defined(__HIP_DEVICE_COMPILE__)
    k = __builtin_amdgcn_frexp_exp(J) / 3;
#else
    k = (ilogb(J) + 1) / 3;
#endif
    J = ldexp(J, -3 * k);
  }
#if defined(__HIP_DEVICE_COMPILE__)
  double y = (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)J) * (-1.0f / 3.0f));
#else
  double y = (double)exp2f(log2f((float)J) * (-1.0f / 3.0f));
#endif
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const double r = fma(-J * y, y * y, 1.0);
    y = fma(y * (1.0 / 3.0), r, y);
  }
  return ldexp(y * y, -2 * k);
}

// One Givens step of the implicit-shift QL sweep (dsyevq3.f90:99-129) on
// scalar state: off-diagonals ej, ej1, diagonals wj, wj1, eigenvector columns
// (a0,a1,a2) = column j and (b0,b1,b2) = column j+1.  Scalars, not arrays, so
// that every value stays in a VGPR.
template <typename R>
__host__ __device__ __forceinline__ void ql_rot(R& s, R& c, R& p, R& g, R ej, R& ej1, R wj, R& wj1,
                                       R& a0, R& a1, R& a2, R& b0, R& b1, R& b2) {
#pragma clang fp contract(off)
  R f = s * ej;
  R b = c * ej;
  // Both branches of :102-114 as one select (identical arithmetic per branch):
  // |f| > |g|: c = g/f, r = sqrt(1+c^2), e = f r, s = 1/r, c = c s
  // else     : s = f/g, r = sqrt(1+s^2), e = g r, c = 1/r, s = s c
  const bool big = fabs(f) > fabs(g);
  const R num = big ? g : f, den = big ? f : g;
  const R t0 = num / den;
  R r = sqrt(R(1) + t0 * t0);
  ej1 = den * r;
  const R inv = R(1) / r;
  const R tr = t0 * inv;
  c = big ? tr : inv;
  s = big ? inv : tr;
  g = wj1 - p;
  r = (wj - g) * s + R(2) * c * b;
  p = s * r;
  wj1 = g + p;
  g = c * r - b;
  R t;
  t = b0; b0 = s * a0 + c * t; a0 = c * a0 - s * t;
  t = b1; b1 = s * a1 + c * t; a1 = c * a1 - s * t;
  t = b2; b2 = s * a2 + c * t; a2 = c * a2 - s * t;
}

// Shift of dsyevq3.f90:87-94 for (L, M): wl, wl1 = W(L), W(L+1); wm = W(M).
template <typename R>
__host__ __device__ __forceinline__ R ql_shift(R wl, R wl1, R wm, R el) {
#pragma clang fp contract(off)
  R g = (wl1 - wl) / (R(2) * el);
  R r = sqrt(R(1) + g * g);
  if (g >= R(0)) return wm - wl + el / (g + r);
  return wm - wl + el / (g - r);
}

// Symmetric 3x3 eigen-decomposition: dsytrd3 + dsyevq3 + eigsrt (largest
// eigenvalue first).  Eigenvectors in q[9] column-major.  Returns false on
// the 30-iteration bail-out (dsyevq3.f90:82-84).
template <typename R>
__host__ __device__ __forceinline__ bool eig3(R a00, R a01, R a02, R a11, R a12, R a22,
                                     R& w0, R& w1, R& w2, R (&q)[9]) {
#pragma clang fp contract(off)
  // dsytrd3.f90:22-109 (Q starts as the identity)
  R q00 = 1, q01 = 0, q02 = 0, q10 = 0, q11 = 1, q12 = 0, q20 = 0, q21 = 0, q22 = 1;
  R e0, e1, e2 = 0;
  R h = a01 * a01 + a02 * a02;
  R g = (a01 > R(0)) ? -sqrt(h) : sqrt(h);
  e0 = g;
  R f = g * a01;
  R u1 = a01 - g, u2 = a02;
  R omega = h - f;
  if (omega > R(0)) {
    omega = R(1) / omega;
    R f1 = a11 * u1 + a12 * u2;          // I = 2: A(2,2)U(2) + A(2,3)U(3)
    R p1 = omega * f1;
    R K = R(0) + u1 * f1;
    R f2 = a12 * u1 + a22 * u2;          // I = 3: A(2,3)U(2) + A(3,3)U(3)
    R p2 = omega * f2;
    K = K + u2 * f2;
    if constexpr (sizeof(R) == 8) K = R(0.5) * K * (omega * omega);   // reference order
    else K = R(0.5) * (K * omega) * omega;                            // no FP32 overflow
    p1 = p1 - K * u1;
    p2 = p2 - K * u2;
    w0 = a00;
    w1 = a11 - R(2) * p1 * u1;
    w2 = a22 - R(2) * p2 * u2;
    R fa = omega * u1;
    q11 = q11 - fa * u1;
    q21 = q21 - fa * u2;
    R fb = omega * u2;
    q12 = q12 - fb * u1;
    q22 = q22 - fb * u2;
    e1 = a12 - p1 * u2 - u1 * p2;
  } else {
    w0 = a00; w1 = a11; w2 = a22;
    e1 = a12;
  }
  // dsyevq3.f90:64-134: L = 1 (0-based 0), then L = 2
  bool ok = true;
  {
    int niter = 0;
    for (int it = 0; it < 50; ++it) {
      R g0 = fabs(w0) + fabs(w1);
      if (fabs(e0) + g0 == g0) break;                 // M = L
      R g1 = fabs(w1) + fabs(w2);
      const bool m1 = (fabs(e1) + g1 == g1);          // M = 2, else M = 3
      if (++niter >= 30) { ok = false; break; }
      R s = 1, c = 1, p = 0;
      if (m1) {
        R gg = ql_shift<R>(w0, w1, w1, e0);
        ql_rot<R>(s, c, p, gg, e0, e1, w0, w1, q00, q10, q20, q01, q11, q21);
        w0 = w0 - p; e0 = gg; e1 = 0;
      } else {
        R gg = ql_shift<R>(w0, w1, w2, e0);
        ql_rot<R>(s, c, p, gg, e1, e2, w1, w2, q01, q11, q21, q02, q12, q22);
        ql_rot<R>(s, c, p, gg, e0, e1, w0, w1, q00, q10, q20, q01, q11, q21);
        w0 = w0 - p; e0 = gg; e2 = 0;
      }
    }
  }
  if (ok) {
    int niter = 0;
    for (int it = 0; it < 50; ++it) {
      R g1 = fabs(w1) + fabs(w2);
      if (fabs(e1) + g1 == g1) break;
      if (++niter >= 30) { ok = false; break; }
      R s = 1, c = 1, p = 0;
      R gg = ql_shift<R>(w1, w2, w2, e1);
      ql_rot<R>(s, c, p, gg, e1, e2, w1, w2, q01, q11, q21, q02, q12, q22);
      w1 = w1 - p; e1 = gg; e2 = 0;
    }
  }
  // eigsrt.f90:19-48 as selects.  Pass 1 moves the last maximum ('>=') to
  // slot 1; pass 2 swaps slots 2 and 3 whenever d(3) >= d(2).
  {
    const bool k1 = (w1 >= w0) && !(w2 >= w1);
    const bool k2 = (w2 >= ((w1 >= w0) ? w1 : w0));
    const R pmax = k2 ? w2 : (k1 ? w1 : w0);
    const R nw1 = k1 ? w0 : w1, nw2 = k2 ? w0 : w2;
    R c00 = k1 ? q01 : (k2 ? q02 : q00), c10 = k1 ? q11 : (k2 ? q12 : q10),
      c20 = k1 ? q21 : (k2 ? q22 : q20);
    R c01 = k1 ? q00 : q01, c11 = k1 ? q10 : q11, c21 = k1 ? q20 : q21;
    R c02 = k2 ? q00 : q02, c12 = k2 ? q10 : q12, c22 = k2 ? q20 : q22;
    w0 = pmax;
    const bool sw = nw2 >= nw1;
    w1 = sw ? nw2 : nw1;
    w2 = sw ? nw1 : nw2;
    q00 = c00; q10 = c10; q20 = c20;
    q01 = sw ? c02 : c01; q11 = sw ? c12 : c11; q21 = sw ? c22 : c21;
    q02 = sw ? c01 : c02; q12 = sw ? c11 : c12; q22 = sw ? c21 : c22;
  }
  q[0] = q00; q[1] = q10; q[2] = q20;
  q[3] = q01; q[4] = q11; q[5] = q21;
  q[6] = q02; q[7] = q12; q[8] = q22;
  return ok;
}

// Log-strain invariants that the return map consumes, plus the principal
// directions and deviatoric strains the stress needs.
template <typename R>
struct Spectral {
  double theta, e_n;            // FP64 for the return map
  R e[3], d[3];                 // principal log strains and e_i / e_n
  R n[9];                       // principal directions (columns)
  bool eig_ok;
};

// Plain FP64: compute_kirchoff_stress :293-332 in reference order.
__host__ __device__ __forceinline__ Spectral<double> spectral_fp64(const double (&F)[9]) {
#pragma clang fp contract(off)
  Spectral<double> s;
  // b = matmul(F, transpose(F)) (col-major F: F(i,k) = F[i + 3k])
  double b00 = F[0] * F[0] + F[3] * F[3] + F[6] * F[6];
  double b01 = F[0] * F[1] + F[3] * F[4] + F[6] * F[7];
  double b02 = F[0] * F[2] + F[3] * F[5] + F[6] * F[8];
  double b11 = F[1] * F[1] + F[4] * F[4] + F[7] * F[7];
  double b12 = F[1] * F[2] + F[4] * F[5] + F[7] * F[8];
  double b22 = F[2] * F[2] + F[5] * F[5] + F[8] * F[8];
  double w0, w1, w2;
  s.eig_ok = eig3<double>(b00, b01, b02, b11, b12, b22, w0, w1, w2, s.n);
  double h1 = sqrt(w0), h2 = sqrt(w1), h3 = sqrt(w2);
  double J = h1 * h2 * h3;
  s.theta = log(J);
  double Jd = pow(J, -1.0 / 3.0);
  s.e[0] = log(Jd * h1);
  s.e[1] = log(Jd * h2);
  s.e[2] = log(Jd * h3);
  s.e_n = sqrt(s.e[0] * s.e[0] + s.e[1] * s.e[1] + s.e[2] * s.e[2]);
  const double eps = 2.220446049250313080847e-16;  // epsilon(0.0_rp)
  if (s.e_n > eps) {
    s.d[0] = s.e[0] / s.e_n; s.d[1] = s.e[1] / s.e_n; s.d[2] = s.e[2] / s.e_n;
  } else {
    s.d[0] = s.d[1] = s.d[2] = 0.0;
  }
  return s;
}

// FP32 kinematics: spectral decomposition of b - I from H = F - I.
__host__ __device__ __forceinline__ Spectral<float> spectral_fp32(const float (&H)[9]) {
  Spectral<float> s;
  // (b - I)_ij = H_ij + H_ji + sum_k H_ik H_jk
  float c00 = 2.f * H[0] + (H[0] * H[0] + H[3] * H[3] + H[6] * H[6]);
  float c11 = 2.f * H[4] + (H[1] * H[1] + H[4] * H[4] + H[7] * H[7]);
  float c22 = 2.f * H[8] + (H[2] * H[2] + H[5] * H[5] + H[8] * H[8]);
  float c01 = H[3] + H[1] + (H[0] * H[1] + H[3] * H[4] + H[6] * H[7]);
  float c02 = H[6] + H[2] + (H[0] * H[2] + H[3] * H[5] + H[6] * H[8]);
  float c12 = H[7] + H[5] + (H[1] * H[2] + H[4] * H[5] + H[7] * H[8]);
  // scale to unit magnitude so no intermediate of the FP32 Householder/QL
  // steps under- or overflows for strains from 1e-12 to 1
  float sc = fmaxf(fmaxf(fmaxf(fabsf(c00), fabsf(c11)), fmaxf(fabsf(c22), fabsf(c01))),
                   fmaxf(fabsf(c02), fabsf(c12)));
  // below 1e-30 the strain is zero to FP32 precision; a denormal scale would
  // overflow its reciprocal
  const float inv = sc > 1e-30f ? 1.0f / sc : 0.f;
  float mu0, mu1, mu2;
  s.eig_ok = eig3<float>(c00 * inv, c01 * inv, c02 * inv, c11 * inv, c12 * inv, c22 * inv,
                         mu0, mu1, mu2, s.n);
  mu0 *= sc;
  mu1 *= sc;
  mu2 *= sc;
  float l0 = 0.5f * log1pf(mu0), l1 = 0.5f * log1pf(mu1), l2 = 0.5f * log1pf(mu2);
  float th = l0 + l1 + l2;
  float t3 = th * (1.0f / 3.0f);
  s.e[0] = l0 - t3; s.e[1] = l1 - t3; s.e[2] = l2 - t3;
  float en = sqrtf(s.e[0] * s.e[0] + s.e[1] * s.e[1] + s.e[2] * s.e[2]);
  s.theta = (double)th;
  s.e_n = (double)en;
  if (en > 1.1920929e-07f) {
    float r = 1.0f / en;
    s.d[0] = s.e[0] * r; s.d[1] = s.e[1] * r; s.d[2] = s.e[2] * r;
  } else {
    s.d[0] = s.d[1] = s.d[2] = 0.f;
  }
  return s;
}

// FP32 kinematics without eigenvectors.  The stress of the law needs only
// theta = tr E, the deviatoric Hencky strain e' = dev E and |e'|, because
// tau = c_vol I + sum_i 2G (e_i - eL xS e_i/|e'|) n_i n_i^T
//     = c_vol I + 2G (1 - eL xS/|e'|) e'          (compute_kirchoff_stress
// :293-332 with d_i = e_i/|e'|).  E = 1/2 log b is formed as a tensor:
// 1/2 log b = artanh(Z) = sum_k Z^(2k+1)/(2k+1), Z = (b - I)(b + I)^-1, whose
// terms all commute with b; with |Z|_F <= 0.6 the terms fall by >= 0.36 each.
struct Hencky32 {
  double theta, e_n;   // FP64 for the return map
  float ed[6];         // e' (00, 01, 02, 11, 12, 22)
  bool ok;             // false: |Z|_F > 0.6, use the spectral path
};

// Principal values, descending, of a symmetric deviatoric 3x3 tensor
// s = (00, 01, 02, 11, 12, 22), in closed form: the roots of the
// characteristic polynomial l^3 - J2 l - J3 = 0 by the trigonometric
// solution, l_k = 2 r cos(a - 2 pi k / 3) with r = sqrt(J2 / 3),
// cos 3a = J3 / (2 r^3), a in [0, pi / 3] (k = 0, 1, 2 give the descending
// order).  Any trace left by rounding is removed first.  Below J2 = 1e-24
// (|s| ~ 1e-12) the values are returned as zero.
__host__ __device__ __forceinline__ void principal_dev_fp32(const float (&s)[6], float& l0, float& l1,
                                                           float& l2) {
  const float m = (s[0] + s[3] + s[5]) * (1.0f / 3.0f);
  const float d0 = s[0] - m, d1 = s[3] - m, d2 = s[5] - m;
  const float J2 = 0.5f * (d0 * d0 + d1 * d1 + d2 * d2) + s[1] * s[1] + s[2] * s[2] + s[4] * s[4];
  if (!(J2 > 1e-24f)) {
    l0 = l1 = l2 = 0.f;
    return;
  }
  const float J3 = d0 * (d1 * d2 - s[4] * s[4]) - s[1] * (s[1] * d2 - s[4] * s[2]) +
                   s[2] * (s[1] * s[4] - d1 * s[2]);
  const float r = sqrtf(J2 * (1.0f / 3.0f));
  const float c3 = fminf(1.0f, fmaxf(-1.0f, J3 / (2.0f * r * r * r)));
  const float a = acosf(c3) * (1.0f / 3.0f);
  const float c = cosf(a), sn = sinf(a);
  const float h = 1.7320508075688772f;   // 2 sin(2 pi / 3)
  l0 = 2.0f * r * c;
  l1 = r * (h * sn - c);
  l2 = -r * (c + h * sn);
}

// c = a b for symmetric a, b that commute (the product is symmetric).
__host__ __device__ __forceinline__ void sym_mul_commuting(const float (&a)[6], const float (&b)[6],
                                                          float (&c)[6]) {
  c[0] = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
  c[1] = a[0] * b[1] + a[1] * b[3] + a[2] * b[4];
  c[2] = a[0] * b[2] + a[1] * b[4] + a[2] * b[5];
  c[3] = a[1] * b[1] + a[3] * b[3] + a[4] * b[4];
  c[4] = a[1] * b[2] + a[3] * b[4] + a[4] * b[5];
  c[5] = a[2] * b[2] + a[4] * b[4] + a[5] * b[5];
}

__host__ __device__ __forceinline__ Hencky32 hencky_fp32(const float (&H)[9]) {
  Hencky32 h;
  // C = b - I from H = F - I without cancellation
  float c[6];
  c[0] = 2.f * H[0] + (H[0] * H[0] + H[3] * H[3] + H[6] * H[6]);
  c[3] = 2.f * H[4] + (H[1] * H[1] + H[4] * H[4] + H[7] * H[7]);
  c[5] = 2.f * H[8] + (H[2] * H[2] + H[5] * H[5] + H[8] * H[8]);
  c[1] = H[3] + H[1] + (H[0] * H[1] + H[3] * H[4] + H[6] * H[7]);
  c[2] = H[6] + H[2] + (H[0] * H[2] + H[3] * H[5] + H[6] * H[8]);
  c[4] = H[7] + H[5] + (H[1] * H[2] + H[4] * H[5] + H[7] * H[8]);
  // (b + I)^-1 = (2I + C)^-1 by cofactors (det(b + I) >= 1)
  const float m00 = 2.f + c[0], m11 = 2.f + c[3], m22 = 2.f + c[5];
  float a[6];
  a[0] = m11 * m22 - c[4] * c[4];
  a[1] = c[2] * c[4] - c[1] * m22;
  a[2] = c[1] * c[4] - c[2] * m11;
  a[3] = m00 * m22 - c[2] * c[2];
  a[4] = c[1] * c[2] - m00 * c[4];
  a[5] = m00 * m11 - c[1] * c[1];
  const float r = fast_rcp(m00 * a[0] + c[1] * a[1] + c[2] * a[2]);
#pragma unroll
  for (int q = 0; q < 6; ++q) a[q] *= r;
  float z[6];
  sym_mul_commuting(c, a, z);
  const float zf2 = z[0] * z[0] + z[3] * z[3] + z[5] * z[5] +
                    2.f * (z[1] * z[1] + z[2] * z[2] + z[4] * z[4]);
  h.ok = zf2 <= 0.36f;
  // terms after Z^(2n+1) sum to below 2^-24 of |E| ~ |Z| when
  // |Z|^(2n+2) / ((2n+3)(1 - |Z|^2)) <= 2^-24 (|Z| <= |Z|_F)
  const int nterms = zf2 <= 1.7e-7f ? 0 : zf2 <= 5.4e-4f ? 1 : zf2 <= 7.3e-3f ? 2
                   : zf2 <= 2.6e-2f ? 3 : zf2 <= 5.2e-2f ? 4 : zf2 <= 8.4e-2f ? 5
                   : zf2 <= 0.115f ? 6 : zf2 <= 0.17f ? 8 : zf2 <= 0.22f ? 10
                   : zf2 <= 0.28f ? 14 : 20;
  float z2[6], t[6], e[6];
  sym_mul_commuting(z, z, z2);
#pragma unroll
  for (int q = 0; q < 6; ++q) t[q] = e[q] = z[q];
  if (h.ok) {
    // written out term by term: constant weights 1/(2k+1), no loop-carried
    // register copies; each lane takes its own number of terms
    auto term = [&](float w) {
      float tn[6];
      sym_mul_commuting(t, z2, tn);
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        t[q] = tn[q];
        e[q] += w * tn[q];
      }
    };
    if (nterms >= 1) { term(1.0f / 3.0f);
    if (nterms >= 2) { term(1.0f / 5.0f);
    if (nterms >= 3) { term(1.0f / 7.0f);
    if (nterms >= 4) { term(1.0f / 9.0f);
    if (nterms >= 5) { term(1.0f / 11.0f);
    if (nterms >= 6) { term(1.0f / 13.0f);
    if (nterms >= 7) {
      for (int k = 7; k <= nterms; ++k) term(1.0f / (float)(2 * k + 1));
    } } } } } } }
  }
  const float th = e[0] + e[3] + e[5];
  const float t3 = th * (1.0f / 3.0f);
  h.ed[0] = e[0] - t3;
  h.ed[1] = e[1];
  h.ed[2] = e[2];
  h.ed[3] = e[3] - t3;
  h.ed[4] = e[4];
  h.ed[5] = e[5] - t3;
  const float en = sqrtf(h.ed[0] * h.ed[0] + h.ed[3] * h.ed[3] + h.ed[5] * h.ed[5] +
                         2.f * (h.ed[1] * h.ed[1] + h.ed[2] * h.ed[2] + h.ed[4] * h.ed[4]));
  h.theta = (double)th;
  h.e_n = (double)en;
  return h;
}

// ---------------------------------------------------------------------------
// The Hencky strain E = 1/2 log b = artanh(Z) = sum_k Z^(2k+1)/(2k+1),
// Z = (b - I)(b + I)^-1, as a polynomial in Z.  By Cayley-Hamilton Z^3 = J1 Z^2
// - J2 Z + J3 I (J1..J3 the invariants of Z), so a polynomial is three scalars
// (on I, Z, Z^2), and a Horner step of the series, r <- Z^2 r + 1/(2k+1), is 6
// scalar operations; a product of symmetric tensors and its sum into E, which
// a term took before, is 30.  The identity divides by nothing, so equal or
// nearly equal principal values need no care.  (FP64 on C1: the same count of
// VALU instructions fell by 8% in all; measured errors of theta and e' against
// extended precision: rms 5.5e-17 |E|, 6.5e-17 term by term.)  FP64 only: the
// FP32 mode keeps the arithmetic its runs had, since a run amplifies a change of
// rounding in FP32 to 2e-4 of the velocities in 200 steps.
// ---------------------------------------------------------------------------

// 1/x of the element step's precision (1 ulp)
template <typename R>
__host__ __device__ __forceinline__ R rcp_r(R x) {
  if constexpr (sizeof(R) == 4) return fast_rcp(x);
  else return rcp64(x);
}

// Z = (b - I)(b + I)^-1 from c = b - I.  With A = adj(c) and the invariants
// I1..I3 of c, c adj(2I + c) = 4c - 2A + (2 I2 + I3) I (Cayley-Hamilton; the
// terms of order 1 cancel in the identity, not in the arithmetic) and
// det(2I + c) = 8 + 4 I1 + 2 I2 + I3 >= 1: 36 operations and a reciprocal,
// without the product of c with an inverse.
template <typename R>
__host__ __device__ __forceinline__ void cayley(const R (&c)[6], R (&z)[6]) {
  const R a0 = c[3] * c[5] - c[4] * c[4], a1 = c[2] * c[4] - c[1] * c[5],
          a2 = c[1] * c[4] - c[2] * c[3], a3 = c[0] * c[5] - c[2] * c[2],
          a4 = c[1] * c[2] - c[0] * c[4], a5 = c[0] * c[3] - c[1] * c[1];
  const R i2 = a0 + a3 + a5, i3 = c[0] * a0 + c[1] * a1 + c[2] * a2;
  const R q = R(2) * i2 + i3;
  const R r = rcp_r<R>(R(4) * (R(2) + (c[0] + c[3] + c[5])) + q);
  z[0] = (R(4) * c[0] + (q - R(2) * a0)) * r;
  z[1] = (R(4) * c[1] - R(2) * a1) * r;
  z[2] = (R(4) * c[2] - R(2) * a2) * r;
  z[3] = (R(4) * c[3] + (q - R(2) * a3)) * r;
  z[4] = (R(4) * c[4] - R(2) * a4) * r;
  z[5] = (R(4) * c[5] + (q - R(2) * a5)) * r;
}

// w = z^2 of a symmetric z; its trace is |z|_F^2.
template <typename R>
__host__ __device__ __forceinline__ void sym_square(const R (&z)[6], R (&w)[6]) {
  w[0] = z[0] * z[0] + z[1] * z[1] + z[2] * z[2];
  w[1] = z[0] * z[1] + z[1] * z[3] + z[2] * z[4];
  w[2] = z[0] * z[2] + z[1] * z[4] + z[2] * z[5];
  w[3] = z[1] * z[1] + z[3] * z[3] + z[4] * z[4];
  w[4] = z[1] * z[2] + z[3] * z[4] + z[4] * z[5];
  w[5] = z[2] * z[2] + z[4] * z[4] + z[5] * z[5];
}

// true when x holds on any active lane of the wave (on the host: for x)
__host__ __device__ __forceinline__ bool any_lane(bool x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __ballot(x) != 0ull;
#else
  return x;
#endif
}

// Horner evaluation of the series' polynomial r = a I + b Z + c Z^2.
template <typename R>
struct SeriesPoly {
  R j1, j2, j3, a, b, c;
  __host__ __device__ __forceinline__ SeriesPoly(const R (&z)[6], R zf2) {
    j1 = z[0] + z[3] + z[5];
    j2 = R(0.5) * (j1 * j1 - zf2);
    j3 = z[0] * (z[3] * z[5] - z[4] * z[4]) + z[1] * (z[2] * z[4] - z[1] * z[5]) +
         z[2] * (z[1] * z[4] - z[2] * z[3]);
  }
  // the two highest terms: Z^2 (w0 I) + w1 I
  __host__ __device__ __forceinline__ void start(R w1, R w0) {
    a = w1;
    b = R(0);
    c = w0;
  }
  // r <- Z^2 r + w I, by Z (a, b, c) = (c J3, a - c J2, b + c J1) twice
  __host__ __device__ __forceinline__ void step(R w) {
    const R ya = c * j3, yb = a - c * j2, yc = b + c * j1;
    a = yc * j3 + w;
    b = ya - yc * j2;
    c = yb + yc * j1;
  }
  // E = scale Z r = e0 I + e1 Z + e2 Z^2: theta = tr E, e' = dev E, |e'|^2
  __host__ __device__ __forceinline__ void strain(const R (&z)[6], const R (&w)[6], R zf2, R scale,
                                                  double& theta, R (&ed)[6], R& en2) const {
    const R e0 = scale * (c * j3), e1 = scale * (a - c * j2), e2 = scale * (b + c * j1);
    const R t = e1 * j1 + e2 * zf2, t3 = t * R(1.0 / 3.0);
    theta = (double)(R(3) * e0 + t);
    ed[0] = e1 * z[0] + (e2 * w[0] - t3);
    ed[1] = e1 * z[1] + e2 * w[1];
    ed[2] = e1 * z[2] + e2 * w[2];
    ed[3] = e1 * z[3] + (e2 * w[3] - t3);
    ed[4] = e1 * z[4] + e2 * w[4];
    ed[5] = e1 * z[5] + (e2 * w[5] - t3);
    en2 = ed[0] * ed[0] + ed[3] * ed[3] + ed[5] * ed[5] +
          R(2) * (ed[1] * ed[1] + ed[2] * ed[2] + ed[4] * ed[4]);
  }
};

// The same strain by the spectral form, for stretches beyond the series'
// range: e' = sum_k e_k n_k n_k^T.  Returns false where the eigen-solver gave
// up.
__host__ __device__ __forceinline__ bool hencky_spectral_fp32(const float (&H)[9], Hencky32& h) {
  const Spectral<float> sp = spectral_fp32(H);
  const float* n = sp.n;
  auto sum = [&](int i, int j) {
    return sp.e[0] * n[i] * n[j] + sp.e[1] * n[3 + i] * n[3 + j] + sp.e[2] * n[6 + i] * n[6 + j];
  };
  h.ed[0] = sum(0, 0);
  h.ed[1] = sum(0, 1);
  h.ed[2] = sum(0, 2);
  h.ed[3] = sum(1, 1);
  h.ed[4] = sum(1, 2);
  h.ed[5] = sum(2, 2);
  h.theta = sp.theta;
  h.e_n = sp.e_n;
  return sp.eig_ok;
}

// FP64 Hencky strain by the same series, for the plain FP64 element step:
// E = 1/2 log b = sum_k Z^(2k+1)/(2k+1), Z = (b - I)(b + I)^-1, b - I formed
// from H = F - I.  theta = tr E and e' = dev E are what the loading functions
// and the stress consume (theta = log J, |e'| = e_n of compute_kirchoff_stress
// :313-322), so no eigenvectors, square roots of eigenvalues, logarithms or
// powers are needed; the terms run until the remainder is below 2^-54 of
// |Z|.  Stretches with |Z|_F > 0.6 (principal stretches beyond about 1/2..2)
// first halve the logarithm by symmetric square roots, log b = 2^k
// log b^(1/2^k), until |Z|_F <= 0.6.
struct Hencky64 {
  double theta, e_n;
  double inv_en;       // 1 / e_n (0 where e_n is 0)
  double ed[6];        // e' (00, 01, 02, 11, 12, 22)
  bool ok;             // false: no finite strain (a non-finite or non-positive b)
};

// Inverse of a symmetric 3x3 matrix (00, 01, 02, 11, 12, 22) by its adjugate.
__host__ __device__ __forceinline__ void sym_inv64(const double (&m)[6], double (&r)[6]) {
  r[0] = m[3] * m[5] - m[4] * m[4];
  r[1] = m[2] * m[4] - m[1] * m[5];
  r[2] = m[1] * m[4] - m[2] * m[3];
  r[3] = m[0] * m[5] - m[2] * m[2];
  r[4] = m[1] * m[2] - m[0] * m[4];
  r[5] = m[0] * m[3] - m[1] * m[1];
  const double d = 1.0 / (m[0] * r[0] + m[1] * r[1] + m[2] * r[2]);
#pragma unroll
  for (int q = 0; q < 6; ++q) r[q] *= d;
}

// Square root of a symmetric positive definite 3x3 matrix by the
// Denman-Beavers iteration Y <- (Y + W^-1)/2, W <- (W + Y^-1)/2 (Y -> b^1/2,
// W -> b^-1/2), run to convergence (quadratic; ~6-10 iterations for the
// stretches a solid reaches).
__host__ __device__ __forceinline__ void sym_sqrt64(double (&y)[6]) {
  double w[6] = {1.0, 0.0, 0.0, 1.0, 0.0, 1.0};
  for (int it = 0; it < 40; ++it) {
    double yi[6], wi[6];
    sym_inv64(y, yi);
    sym_inv64(w, wi);
    double d2 = 0.0, n2 = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const double yn = 0.5 * (y[q] + wi[q]);
      const double f = (q == 1 || q == 2 || q == 4) ? 2.0 : 1.0;
      d2 += f * (yn - y[q]) * (yn - y[q]);
      n2 += f * yn * yn;
      y[q] = yn;
      w[q] = 0.5 * (w[q] + yi[q]);
    }
    if (!(d2 > 1e-32 * n2)) break;   // converged (or not finite)
  }
}

// Number n of series terms after Z: the remainder |Z|^(2n+3) / ((2n+3)
// (1 - |Z|^2)) stays below 2^-54 |Z| (|Z| <= |Z|_F, zf2 = |Z|_F^2): strains
// of 1% take 4 terms, of 5% 6; beyond 2% of zf2 the steps get coarser.  A
// lane's n depends on its own zf2 alone, so that a point's result does not
// depend on which points share its wave; the wave runs the Horner steps of its
// largest n, and a lane whose series is shorter joins with its first term
// (its coefficients before are zero, and so is its r).
struct HenckyTerms {
  int n;           // the wave's largest n
  double w1, w0;   // the lane's coefficients of terms n - 1 and n
};
constexpr double kTerms3 = 1.4949e-04, kTerms4 = 9.0589e-04, kTerms5 = 2.9934e-03,
                 kTerms6 = 7.0039e-03, kTerms7 = 1.3216e-02, kTerms8 = 2.1619e-02,
                 kTerms10 = 4.4078e-02, kTerms15 = 1.1898e-01, kTerms22 = 2.2961e-01;
// 1/N, formed where it is used: the empty asm keeps the compiler from holding
// the coefficients of all series lengths in vector registers from the start of
// a wave (34 instructions of ~800 and 26 of 126 registers of the element kernel).
template <int N>
__host__ __device__ __forceinline__ double odd64() {
  double c = 1.0 / N;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(c));
#endif
  return c;
}
__host__ __device__ __forceinline__ HenckyTerms hencky64_terms(double zf2) {
  const bool m3 = zf2 > kTerms3;
  if (!any_lane(m3)) return {3, odd64<5>(), odd64<7>()};
  const bool m4 = zf2 > kTerms4;
  if (!any_lane(m4)) return {4, odd64<7>(), m3 ? odd64<9>() : 0.0};
  const bool m5 = zf2 > kTerms5;
  if (!any_lane(m5)) return {5, m3 ? odd64<9>() : 0.0, m4 ? odd64<11>() : 0.0};
  const bool m6 = zf2 > kTerms6;
  if (!any_lane(m6)) return {6, m4 ? odd64<11>() : 0.0, m5 ? odd64<13>() : 0.0};
  const bool m7 = zf2 > kTerms7;
  if (!any_lane(m7)) return {7, m5 ? odd64<13>() : 0.0, m6 ? odd64<15>() : 0.0};
  if (!any_lane(zf2 > kTerms8)) return {8, m6 ? odd64<15>() : 0.0, m7 ? odd64<17>() : 0.0};
  if (!any_lane(zf2 > kTerms10)) return {10, zf2 > kTerms8 ? odd64<19>() : 0.0, zf2 > kTerms8 ? odd64<21>() : 0.0};
  if (!any_lane(zf2 > kTerms15)) return {15, zf2 > kTerms10 ? odd64<29>() : 0.0, zf2 > kTerms10 ? odd64<31>() : 0.0};
  if (!any_lane(zf2 > kTerms22)) return {22, zf2 > kTerms15 ? odd64<43>() : 0.0, zf2 > kTerms15 ? odd64<45>() : 0.0};
  return {32, zf2 > kTerms22 ? odd64<63>() : 0.0, zf2 > kTerms22 ? odd64<65>() : 0.0};   // zf2 <= 0.36
}
// 1/(2k+1), k = 7..30: the coefficients of the long series
constexpr double kInvOdd64[24] = {
    1.0 / 15, 1.0 / 17, 1.0 / 19, 1.0 / 21, 1.0 / 23, 1.0 / 25, 1.0 / 27, 1.0 / 29,
    1.0 / 31, 1.0 / 33, 1.0 / 35, 1.0 / 37, 1.0 / 39, 1.0 / 41, 1.0 / 43, 1.0 / 45,
    1.0 / 47, 1.0 / 49, 1.0 / 51, 1.0 / 53, 1.0 / 55, 1.0 / 57, 1.0 / 59, 1.0 / 61};

// LARGE false: no halvings, stretches beyond the series' range give ok = false.
template <bool LARGE = true>
__host__ __device__ __forceinline__ Hencky64 hencky_fp64(const double (&H)[9]) {
  Hencky64 h;
  double c[6];
  c[0] = 2.0 * H[0] + (H[0] * H[0] + H[3] * H[3] + H[6] * H[6]);
  c[3] = 2.0 * H[4] + (H[1] * H[1] + H[4] * H[4] + H[7] * H[7]);
  c[5] = 2.0 * H[8] + (H[2] * H[2] + H[5] * H[5] + H[8] * H[8]);
  c[1] = H[3] + H[1] + (H[0] * H[1] + H[3] * H[4] + H[6] * H[7]);
  c[2] = H[6] + H[2] + (H[0] * H[2] + H[3] * H[5] + H[6] * H[8]);
  c[4] = H[7] + H[5] + (H[1] * H[2] + H[4] * H[5] + H[7] * H[8]);
  double z[6], w[6];
  cayley<double>(c, z);
  sym_square<double>(z, w);
  double zf2 = w[0] + w[3] + w[5];
  // large stretches: b <- b^(1/2) until |Z|_F <= 0.6 (each halves log b)
  int halvings = 0;
  if (LARGE && zf2 > 0.36) {
    double b[6] = {1.0 + c[0], c[1], c[2], 1.0 + c[3], c[4], 1.0 + c[5]};
    while (zf2 > 0.36 && halvings < 10) {
      sym_sqrt64(b);
      ++halvings;
      const double cb[6] = {b[0] - 1.0, b[1], b[2], b[3] - 1.0, b[4], b[5] - 1.0};
      cayley<double>(cb, z);
      sym_square<double>(z, w);
      zf2 = w[0] + w[3] + w[5];
    }
  }
  h.ok = zf2 <= 0.36;
  if (!LARGE && !h.ok) return h;
  const HenckyTerms nt = hencky64_terms(zf2);
  const int n = nt.n;
  SeriesPoly<double> r(z, zf2);
  r.start(nt.w1, nt.w0);
  if (n > 8) {
    const int nl = zf2 > kTerms22 ? 32 : zf2 > kTerms15 ? 22 : zf2 > kTerms10 ? 15
                 : zf2 > kTerms8 ? 10 : zf2 > kTerms7 ? 8 : zf2 > kTerms6 ? 7 : 6;
    for (int k = n - 2; k > 6; --k) r.step(k <= nl ? kInvOdd64[k - 7] : 0.0);
  }
  if (n > 7) r.step(zf2 > kTerms5 ? odd64<13>() : 0.0);   // k = 6
  if (n > 6) r.step(zf2 > kTerms4 ? odd64<11>() : 0.0);
  if (n > 5) r.step(zf2 > kTerms3 ? odd64<9>() : 0.0);
  if (n > 4) r.step(odd64<7>());
  if (n > 3) r.step(odd64<5>());
  r.step(1.0 / 3.0);                                      // k = 1
  r.step(1.0);
  double en2;
  r.strain(z, w, zf2, (double)(1 << halvings), h.theta, h.ed, en2);
  sqrt_rsqrt64(en2, h.e_n, h.inv_en);
  return h;
}

// The law's Kirchhoff stress from the Hencky tensor (FP64):
// tau = c_vol I + 2G (1 - eL xS/e_n) e', the direction term dropped for
// e_n <= epsilon(0.0_rp) as d_i = 0 in compute_kirchoff_stress :323-332.
__host__ __device__ __forceinline__ void kirchhoff_hencky64(const Mat& m, const Hencky64& h,
                                                           double xS, double (&t)[6]) {
  const double cvol = m.K * (h.theta - 3.0 * m.alfa * m.eL * xS);
  const double twoG = 2.0 * m.G;
  const double coef =
      h.e_n > 2.220446049250313080847e-16 ? twoG * (1.0 - m.eL * xS * h.inv_en) : twoG;
  t[0] = cvol + coef * h.ed[0];
  t[1] = coef * h.ed[1];
  t[2] = coef * h.ed[2];
  t[3] = cvol + coef * h.ed[3];
  t[4] = coef * h.ed[4];
  t[5] = cvol + coef * h.ed[5];
}

// tau = c_vol I + 2G (1 - eL xS/|e'|) e'; for |e'| below FP32 epsilon the
// direction term is dropped, as d_i = 0 in the spectral form.
__host__ __device__ __forceinline__ void kirchhoff_dev(const Mat& m, const Hencky32& h, double xS,
                                                      float (&t)[6]) {
  const float cvol = (float)(m.K * (h.theta - 3.0 * m.alfa * m.eL * xS));
  const float twoG = (float)(2.0 * m.G);
  const float en = (float)h.e_n;
  const float coef = en > 1.1920929e-07f ? twoG * (1.0f - (float)(m.eL * xS) * fast_rcp(en)) : twoG;
  t[0] = cvol + coef * h.ed[0];
  t[1] = coef * h.ed[1];
  t[2] = coef * h.ed[2];
  t[3] = cvol + coef * h.ed[3];
  t[4] = coef * h.ed[4];
  t[5] = cvol + coef * h.ed[5];
}

// Neo-Hookean (Ansys form) Kirchhoff stress, sld_stress_model_102.f90:116-119
// pushed forward: tau = F S F^T with S = ((-mu/3) J^(-2/3) tr C + J K (J-1))
// C^-1 + mu J^(-2/3) I gives tau = mu J^(-2/3) dev(b) + J K (J-1) I.  Formed
// from H = F - I: dev(b) = dev(b - I) and J - 1 = tr H + I2(H) + det H, so
// small strains lose nothing to cancellation (in FP32 as in FP64).
template <typename R>
__host__ __device__ __forceinline__ void neo_hookean_tau(double mu, double K, const R (&H)[9],
                                                        R (&t)[6], R& jm1_out) {
  R c[6];   // b - I = H + H^T + H H^T
  c[0] = R(2) * H[0] + (H[0] * H[0] + H[3] * H[3] + H[6] * H[6]);
  c[3] = R(2) * H[4] + (H[1] * H[1] + H[4] * H[4] + H[7] * H[7]);
  c[5] = R(2) * H[8] + (H[2] * H[2] + H[5] * H[5] + H[8] * H[8]);
  c[1] = H[3] + H[1] + (H[0] * H[1] + H[3] * H[4] + H[6] * H[7]);
  c[2] = H[6] + H[2] + (H[0] * H[2] + H[3] * H[5] + H[6] * H[8]);
  c[4] = H[7] + H[5] + (H[1] * H[2] + H[4] * H[5] + H[7] * H[8]);
  // det(I + H) - 1 (H column-major: H(i,k) = H[i + 3k])
  const R trH = H[0] + H[4] + H[8];
  const R i2 = (H[0] * H[4] - H[3] * H[1]) + (H[0] * H[8] - H[6] * H[2]) + (H[4] * H[8] - H[7] * H[5]);
  const R dH = H[0] * (H[4] * H[8] - H[7] * H[5]) - H[3] * (H[1] * H[8] - H[7] * H[2]) +
               H[6] * (H[1] * H[5] - H[4] * H[2]);
  const R jm1 = trH + i2 + dH;
  const R J = R(1) + jm1;
  R jm23;
  if constexpr (sizeof(R) == 8) jm23 = pow_m23(J);
  else jm23 = expf((-2.0f / 3.0f) * log1pf(jm1));
  const R tr3 = (c[0] + c[3] + c[5]) * (R(1) / R(3));
  const R m = (R)mu * jm23;
  const R p = J * (R)K * jm1;
  t[0] = m * (c[0] - tr3) + p;
  t[3] = m * (c[3] - tr3) + p;
  t[5] = m * (c[5] - tr3) + p;
  t[1] = m * c[1];
  t[2] = m * c[2];
  t[4] = m * c[4];
  jm1_out = jm1;
}

// eval_loading_function :513-537 (beta = 1 per :554, temperature inert).
__host__ __device__ __forceinline__ double loading(const Mat& m, double C, double theta,
                                          double enor, double xS) {
#pragma clang fp contract(off)
  double pres = m.K * (theta - 3.0 * m.alfa * m.eL * xS);
  double trac = 2.0 * m.G * (enor - m.eL * xS);
  return trac * 1.0 + 3.0 * m.alfa * pres - C * 0.0;
}

// Branch flags and return map (:334-484).  sdv in = TIME_N (xS_0, F_AS_0,
// F_SA_0); sdv out = ITER_K.  Returns status bits; xS is the clamped value.
struct ReturnMap {
  double xS, F_AS, F_SA;
  uint32_t flags;
};

__host__ __device__ __forceinline__ bool flags_only(const Mat& m, double theta, double e_n,
                                           double xS_0, double F_AS_0, double F_SA_0,
                                           bool& kf_AS, bool& kf_SA,
                                           double& F_AS, double& F_SA) {
#pragma clang fp contract(off)
  F_AS = loading(m, m.C_AS, theta, e_n, xS_0);
  kf_AS = (F_AS > F_AS_0) && (F_AS - m.Rs_AS > 0.0) && (xS_0 < 1.0);
  F_SA = loading(m, m.C_SA, theta, e_n, xS_0);
  kf_SA = (F_SA < F_SA_0) && (F_SA - m.Rs_SA < 0.0) && (xS_0 > 0.0);
  return kf_AS || kf_SA;
}

// One active branch: the other's increment and residual stay zero, the 2x2
// system is its first (or second) equation, and the residual is linear in the
// increment, so one division solves it (the full system takes four and the
// inverse of a matrix).  Taken where the reference's first iteration converges
// as well: stresses below 1e5 and terms below 1e6, whose rounding (~1e-10) is
// far below its tolerance of 1e-8 (absolute: in Pa it is not, and the
// reference's iteration runs, to its cap if need be), and an idle diagonal
// that is not zero (the reference divides by it).
// Returns true when r is final: so solved, or no iteration to be made
// (no branch active, residual within the tolerance at the start).
__host__ __device__ __forceinline__ bool return_map_closed(const Mat& m, double theta, double e_n,
                                                  double xS_0, double F_AS_0, double F_SA_0,
                                                  ReturnMap& r) {
#pragma clang fp contract(off)
  bool kf_AS, kf_SA, done = true;
  double F_AS, F_SA;
  flags_only(m, theta, e_n, xS_0, F_AS_0, F_SA_0, kf_AS, kf_SA, F_AS, F_SA);
  r.flags = (kf_AS ? FLAG_KF_AS : 0u) | (kf_SA ? FLAG_KF_SA : 0u);
  double xS = xS_0;
  if (kf_AS || kf_SA) {
    const double RHS_AS = kf_AS ? (F_AS - F_AS_0) * (1.0 - xS) : 0.0;
    const double RHS_SA = kf_SA ? 0.0 - (F_SA - F_SA_0) * xS : 0.0;
    done = !(RHS_AS * RHS_AS + RHS_SA * RHS_SA > 1.0e-8);   // squared first (:403)
    if (!done && kf_AS != kf_SA && (kf_AS ? F_SA - m.Rf_SA : F_AS - m.Rf_AS) != 0.0) {
      const double Rf = kf_AS ? m.Rf_AS : m.Rf_SA, F_0 = kf_AS ? F_AS_0 : F_SA_0;
      const double F = kf_AS ? F_AS : F_SA, RHS = kf_AS ? RHS_AS : RHS_SA;
      const double g = 0.0 - ((F - F_0) + (kf_AS ? (1.0 - xS) * m.G_1 : -(xS * m.G_1)));
      const double dh = 0.0 - RHS / (g + (F - Rf));
      const double x1 = xS + dh;
      const double F1 = loading(m, kf_AS ? m.C_AS : m.C_SA, theta, e_n, x1);
      const double t1 = (F1 - Rf) * dh, t2 = (F1 - F_0) * (kf_AS ? 1.0 - x1 : -x1);
      // what the loading functions' rounding, and so the residual's, scales with
      const double size = m.G * e_n + fabs(m.K * theta) + m.G_1 + fabs(F_0) + fabs(Rf);
      if (fabs(t1 + t2) <= 1.0e-9 && fabs(t1) + fabs(t2) < 1.0e6 && size < 1.0e5) {
        xS = x1;
        F_AS = loading(m, m.C_AS, theta, e_n, xS);
        F_SA = loading(m, m.C_SA, theta, e_n, xS);
        r.flags |= 1u << FLAG_ITER_SHIFT;
        done = true;
      }
    }
  }
  r.F_AS = F_AS;
  r.F_SA = F_SA;
  r.xS = fmax(fmin(1.0, xS), 0.0);                      // clamp after storing F's
  return done;
}

// The largest q whose square root, rounded, is at most 1.0e-8: sqrt(q) > 1.0e-8
// is q > kResi2.
constexpr double kResi2 = 0x1.cd2b297d889bdp-54;
__host__ __device__ __forceinline__ ReturnMap return_map(const Mat& m, double theta, double e_n,
                                                double xS_0, double F_AS_0, double F_SA_0) {
#pragma clang fp contract(off)
  ReturnMap r;
  if (return_map_closed(m, theta, e_n, xS_0, F_AS_0, F_SA_0, r)) return r;
  const bool kf_AS = r.flags & FLAG_KF_AS, kf_SA = r.flags & FLAG_KF_SA;
  double xS = xS_0, F_AS = r.F_AS, F_SA = r.F_SA;       // at xS_0: nothing solved yet
  const double H_AS = kf_AS ? 1.0 : 0.0, H_SA = kf_SA ? 1.0 : 0.0;
  double F_AS_dot = F_AS - F_AS_0, F_SA_dot = F_SA - F_SA_0;
  double dh_AS = 0.0, dh_SA = 0.0;
  double RHS_AS = (F_AS - m.Rf_AS) * dh_AS + H_AS * F_AS_dot * (1.0 - xS);
  double RHS_SA = (F_SA - m.Rf_SA) * dh_SA - H_SA * F_SA_dot * xS;
  bool more = RHS_AS * RHS_AS + RHS_SA * RHS_SA > 1.0e-8;   // squared first (:403)
  int iter = 0;
  while (iter < 65 && more) {
    ++iter;
    double m11 = -m.G_1 * dh_AS - (H_AS * F_AS_dot + H_AS * (1.0 - xS) * m.G_1) + (F_AS - m.Rf_AS);
    double m12 = -m.G_1 * dh_AS - (H_AS * F_AS_dot + H_AS * (1.0 - xS) * m.G_1);
    double m21 = -m.G_1 * dh_SA - (H_SA * F_SA_dot - H_SA * xS * m.G_1);
    double m22 = -m.G_1 * dh_SA - (H_SA * F_SA_dot - H_SA * xS * m.G_1) + (F_SA - m.Rf_SA);
    double det = m11 * m22 - m12 * m21;
    double r11 = m22 / det, r12 = -m12 / det, r21 = -m21 / det, r22 = m11 / det;
    double sol1 = r11 * RHS_AS + r12 * RHS_SA;
    double sol2 = r21 * RHS_AS + r22 * RHS_SA;
    dh_AS = dh_AS - sol1;
    dh_SA = dh_SA - sol2;
    xS = xS + dh_SA + dh_AS;                         // running totals (:429-432)
    F_AS = loading(m, m.C_AS, theta, e_n, xS);
    F_AS_dot = F_AS - F_AS_0;
    F_SA = loading(m, m.C_SA, theta, e_n, xS);
    F_SA_dot = F_SA - F_SA_0;
    RHS_AS = (F_AS - m.Rf_AS) * dh_AS + H_AS * F_AS_dot * (1.0 - xS);
    RHS_SA = (F_SA - m.Rf_SA) * dh_SA - H_SA * F_SA_dot * xS;
    more = RHS_AS * RHS_AS + RHS_SA * RHS_SA > kResi2;
  }
  if (iter >= 65) {                                  // revert (:459-465)
    r.flags |= FLAG_NEWTON_FAIL;
    xS = xS_0;
    F_AS = F_AS_0;
    F_SA = F_SA_0;
  }
  r.flags |= (uint32_t)(iter & 0xff) << FLAG_ITER_SHIFT;
  r.F_AS = F_AS;
  r.F_SA = F_SA;
  r.xS = fmax(fmin(1.0, xS), 0.0);                      // clamp after storing F's
  return r;
}

// Return map with the transformation update supplied by a surrogate: the
// branch flags are evaluated exactly (:342-374); on a flagged point xS takes
// the supplied value x_hat instead of the Newton iterate, and F_AS/F_SA are
// the loading functions at x_hat (stored before the clamp, as :484-498).
__host__ __device__ __forceinline__ ReturnMap return_map_given(const Mat& m, double theta, double e_n,
                                                               double xS_0, double F_AS_0, double F_SA_0,
                                                               double x_hat) {
#pragma clang fp contract(off)
  ReturnMap r;
  bool kf_AS, kf_SA;
  double F_AS, F_SA;
  flags_only(m, theta, e_n, xS_0, F_AS_0, F_SA_0, kf_AS, kf_SA, F_AS, F_SA);
  r.flags = (kf_AS ? FLAG_KF_AS : 0u) | (kf_SA ? FLAG_KF_SA : 0u);
  double xS = xS_0;
  if (kf_AS || kf_SA) {
    xS = x_hat;
    F_AS = loading(m, m.C_AS, theta, e_n, xS);
    F_SA = loading(m, m.C_SA, theta, e_n, xS);
  }
  r.F_AS = F_AS;
  r.F_SA = F_SA;
  r.xS = fmax(fmin(1.0, xS), 0.0);
  return r;
}

// Distance, in xS, from a candidate x to the return map's solution on a
// single-branch point.  With one branch active the reference's residual
// (:449-450) is linear in the increment dh = x - xS_0 (the dh^2 terms of
// (F(x) - R_f) dh and (F(x) - F_0)(1 - x) cancel because F is linear in x),
// so R(x) / R'(x) is exactly x minus the root, i.e. the size of the Newton
// correction the reference's first iteration would apply from x.  Returns a
// large value for two-branch points (always solved exactly) and when the
// slope vanishes.
__host__ __device__ __forceinline__ double consistency_residual(const Mat& m, double theta, double e_n,
                                                                double xS_0, double F_AS_0, double F_SA_0,
                                                                double x) {
  bool kf_AS, kf_SA;
  double F_AS, F_SA;
  flags_only(m, theta, e_n, xS_0, F_AS_0, F_SA_0, kf_AS, kf_SA, F_AS, F_SA);
  if (kf_AS == kf_SA) return 1e30;
  const double d = x - xS_0;
  // dF/dx of the loading function (eval_loading_function, beta = 1)
  const double k = -(2.0 * m.G * m.eL + 9.0 * m.alfa * m.alfa * m.K * m.eL);
  double R, dR;
  if (kf_AS) {
    const double Fx = loading(m, m.C_AS, theta, e_n, x);
    R = (Fx - m.Rf_AS) * d + (Fx - F_AS_0) * (1.0 - x);
    dR = k * d + (Fx - m.Rf_AS) + k * (1.0 - x) - (Fx - F_AS_0);
  } else {
    const double Fx = loading(m, m.C_SA, theta, e_n, x);
    R = (Fx - m.Rf_SA) * d - (Fx - F_SA_0) * x;
    dR = k * d + (Fx - m.Rf_SA) - k * x - (Fx - F_SA_0);
  }
  if (!(fabs(dR) > 0.0)) return 1e30;
  return fabs(R / dR);
}

// Kirchhoff stress (:487-491) as a symmetric tensor t00 t01 t02 t11 t12 t22.
template <typename R>
__host__ __device__ __forceinline__ void kirchhoff(const Mat& m, const Spectral<R>& s, double xS,
                                          R (&t)[6]) {
  R cvol = (R)(m.K * (s.theta - 3.0 * m.alfa * m.eL * xS));
  R exS = (R)(m.eL * xS);
  R twoG = (R)(2.0 * m.G);
  R c0 = twoG * (s.e[0] - exS * s.d[0]);
  R c1 = twoG * (s.e[1] - exS * s.d[1]);
  R c2 = twoG * (s.e[2] - exS * s.d[2]);
  const R* n = s.n;
  t[0] = cvol + c0 * n[0] * n[0] + c1 * n[3] * n[3] + c2 * n[6] * n[6];
  t[3] = cvol + c0 * n[1] * n[1] + c1 * n[4] * n[4] + c2 * n[7] * n[7];
  t[5] = cvol + c0 * n[2] * n[2] + c1 * n[5] * n[5] + c2 * n[8] * n[8];
  t[1] = c0 * n[0] * n[1] + c1 * n[3] * n[4] + c2 * n[6] * n[7];
  t[2] = c0 * n[0] * n[2] + c1 * n[3] * n[5] + c2 * n[6] * n[8];
  t[4] = c0 * n[1] * n[2] + c1 * n[4] * n[5] + c2 * n[7] * n[8];
}

// The law at a point of given F (plain FP64): branch flags, return map and
// Kirchhoff stress.  The Hencky strain comes from the series (no eigenvectors,
// logarithms or powers: ~300 operations for a few percent of strain, the
// spectral form ~1700), whose strains are relative to |E| as exact as the
// spectral form's are relative to 1.  The spectral form, which follows the
// reference operation by operation, stays where the series does not reach
// (stretches beyond about 1/2..2, non-finite or singular F), for deviatoric
// strains up to 1e-5 of a point with a history (there its own rounding, 1e-16, is
// seen in the direction e'/|e'| and so in the stress), for a rotation's strains of
// rounding size, where the return map needs the reference's iteration, whose count
// and end can hang on the last bit, and where an off-diagonal of b is so small
// (1e-162 .. 1e-77 beside any stretch) that the reference's Householder step
// underflows: its NaN is kept.
// Points at rest (xS = 0, loading function well below its threshold), as much of a
// loaded body is, take the series also below 1e-5 and at F = I: no direction enters
// their stress.  A wave that holds points of both kinds goes through both forms:
// 500 points, 2% of them at rest, 14.4 us with the spectral form for those, 4.2 with
// the series for all, 8.3 with the spectral form for all.
constexpr double kSeriesMinEn = 1.0e-5, kSeriesMinB = 1.0e-60;
constexpr double kNoiseEn = 1.0e-13, kNoiseTurn = 1.0e-10;
__host__ __device__ __forceinline__ ReturnMap law_point(const Mat& m, const double (&F)[9], double xS_0,
                                                        double F_AS_0, double F_SA_0, double (&tau)[6]) {
  ReturnMap rm;
  bool done = false;
  {
    const double H[9] = {F[0] - 1.0, F[1], F[2], F[3], F[4] - 1.0, F[5], F[6], F[7], F[8] - 1.0};
    const Hencky64 h = hencky_fp64<false>(H);
    auto tiny = [](double x) { return x != 0.0 && fabs(x) < kSeriesMinB; };
    const bool under = tiny(F[0] * F[1] + F[3] * F[4] + F[6] * F[7]) ||
                       tiny(F[0] * F[2] + F[3] * F[5] + F[6] * F[8]) ||
                       tiny(F[1] * F[2] + F[4] * F[5] + F[7] * F[8]);
    if (h.ok && !under) {
      done = return_map_closed(m, h.theta, h.e_n, xS_0, F_AS_0, F_SA_0, rm);
      // small strains: at rest (F_AS is that of the strain) by a margin that no
      // rounding of either form crosses, and not a rotation alone (a half turn's b is
      // exact in both forms)
      const double turn = fmax(fmax(fabs(H[1]), fabs(H[2])), fabs(H[5]));
      const bool rest = xS_0 == 0.0 && rm.flags == 0 && m.Rs_AS - rm.F_AS > 1.0e-9 * m.G &&
                        (h.e_n > kNoiseEn || turn <= kNoiseTurn);
      done = done && (h.e_n > kSeriesMinEn || rest);
      kirchhoff_hencky64(m, h, rm.xS, tau);
    }
  }
  if (!done) {
    const Spectral<double> sp = spectral_fp64(F);
    rm = return_map(m, sp.theta, sp.e_n, xS_0, F_AS_0, F_SA_0);
    if (!sp.eig_ok) rm.flags |= FLAG_EIGEN_FAIL;
    kirchhoff<double>(m, sp, rm.xS, tau);
  }
  return rm;
}

// Column-major cofactor matrix: C(i,k) = d det(M) / d M(i,k), M^-1 = C^T / det.
template <typename R>
__host__ __device__ __forceinline__ void cof3(const R (&M)[9], R (&C)[9]) {
  C[0] = M[4] * M[8] - M[5] * M[7];
  C[1] = M[5] * M[6] - M[3] * M[8];
  C[2] = M[3] * M[7] - M[4] * M[6];
  C[3] = M[2] * M[7] - M[1] * M[8];
  C[4] = M[0] * M[8] - M[2] * M[6];
  C[5] = M[1] * M[6] - M[0] * M[7];
  C[6] = M[1] * M[5] - M[2] * M[4];
  C[7] = M[2] * M[3] - M[0] * M[5];
  C[8] = M[0] * M[4] - M[1] * M[3];
}

template <typename R>
__host__ __device__ __forceinline__ R det3(const R (&M)[9]) {
  return M[0] * (M[4] * M[8] - M[5] * M[7]) + M[3] * (M[2] * M[7] - M[1] * M[8]) +
         M[6] * (M[1] * M[5] - M[2] * M[4]);
}

// Column-major 3x3 inverse by cofactors (one reciprocal); returns det.  EXACT:
// the IEEE reciprocal in FP64, so that a singular M gives the infinities of a
// division by 0; else 1 ulp, for values of the element step.
template <typename R, bool EXACT = false>
__host__ __device__ __forceinline__ R inv3(const R (&M)[9], R (&Mi)[9]) {
  R C[9];
  cof3<R>(M, C);
  const R det = M[0] * C[0] + M[3] * C[3] + M[6] * C[6];
  R r;
  if constexpr (EXACT && sizeof(R) == 8) r = R(1) / det;
  else r = rcp_r<R>(det);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) Mi[i + 3 * k] = C[k + 3 * i] * r;
  return det;
}

// S = F^-1 tau F^-T (col-major result) from Finv and symmetric tau.
template <typename R>
__host__ __device__ __forceinline__ void pk2(const R (&Fi)[9], const R (&t)[6], R (&S)[9]) {
  R T[9] = {t[0], t[1], t[2], t[1], t[3], t[4], t[2], t[4], t[5]};
  R A[9];  // A = Finv * tau
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      A[i + 3 * j] = Fi[i] * T[3 * j] + Fi[i + 3] * T[1 + 3 * j] + Fi[i + 6] * T[2 + 3 * j];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      S[i + 3 * j] = A[i] * Fi[j] + A[i + 3] * Fi[j + 3] + A[i + 6] * Fi[j + 6];
}

}  // namespace sma
