// HIP kernels of the explicit solid-mechanics step (gfx950, wave64).
//
// Per step, on one stream (captured into a hipGraph by the host):
//   sld_predict   nodal predictor, Dirichlet overwrite at t^{n+1}
//                 (mod_sld_solution_methods.f90:122-145 CD, :406-429 TW;
//                 sld_updbcs.f90:79-114 + sld_funbou.f90:95-136); clears
//                 f_int for the coloured scatter
//   sld_element   SoA gather, one node per lane (coordinates and
//                 displacements relative to the element's first node),
//                 reference Jacobian + deformation gradient at the 8 Gauss
//                 points, SMA return map, Kirchhoff stress, internal force
//                 (sld_element_operations.f90:119-256, elmca2.f90:105-111,
//                 sld_elmpre.f90:149-162, sld_builtin_materials.f90:316-371,
//                 sld_elmmat.f90:137-150, mod_matrix.f90:2327-2431).
//                 Two assemblies, both deterministic and bitwise equal:
//                 coloured scatter (one launch per colour, read-modify-write
//                 of f_int) or gather (one launch over all elements writing
//                 each corner force into its node-sorted slot; the
//                 corrector sums each node's contiguous slots in colour
//                 order, i.e. the same additions in the same order)
//   sld_face_load Neumann loads of boundary faces (sld_bouope.f90), when set
//   sld_correct   [gather f_int], f_ext (faces + nodal pattern + m g),
//                 a = (f_ext - f_int) / m, velocity corrector / TW Dirichlet
//                 zeroing (solric.f90:294-330; mod_sld_solution_methods.f90:
//                 181-210 CD, :494-527 TW); writes t^{n+1} = t^n + dt
//                 (setgts.f90:98); inside a captured run of steps it also
//                 runs the next step's predictor; optional energy sums
//                 (mod_sld_energy.f90) reduced by sld_energy_reduce
// The history (xS, F_AS, F_SA) and the clock live in two slots that swap
// roles every step (sld_updunk.f90:149-186, svegm TIME_N <- ITER_K): slot
// tn holds TIME_N / t^n, the step writes slot 1 - tn.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "sma_law.hpp"
#include "surrogate_features.hpp"

namespace sld {

// HEX08 natural derivatives at the 2x2x2 Gauss points: dN_a/dxi_k at GP g is
// 0.5 * s_ak * f(a,g,m1) * f(a,g,m2) where f = 0.5*(1 +- 0.577350269189626)
// depending on whether node a and GP g lie on the same side in direction m
// (mod_lagrange.f90:935-1000, mod_quadrature_gauss.f90:2320-2321,2372-2385).
__host__ __device__ __forceinline__ int node_sign(int a, int k) {
  // node order (-,-,-) (+,-,-) (+,+,-) (-,+,-) (-,-,+) (+,-,+) (+,+,+) (-,+,+)
  const int sx = 0x66, sy = 0xCC, sz = 0xF0;  // bit a set = +1
  int m = (k == 0) ? sx : (k == 1) ? sy : sz;
  return ((m >> a) & 1) ? 1 : -1;
}
__host__ __device__ __forceinline__ int gp_sign(int g, int k) {
  // GP order: xi outer, eta, zeta inner; bit = 1 means +0.5773...
  int bit = (k == 0) ? (g >> 2) & 1 : (k == 1) ? (g >> 1) & 1 : g & 1;
  return bit ? 1 : -1;
}
template <typename R>
__host__ __device__ __forceinline__ R hex_deriv(int a, int g, int k) {
  const double gpos = 0.577350269189626;
  const R cp = (R)(0.5 * (1.0 + gpos)), cm = (R)(0.5 * (1.0 - gpos));
  R f[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) f[m] = (node_sign(a, m) == gp_sign(g, m)) ? cp : cm;
  R s = (R)(0.5 * node_sign(a, k));
  if (k == 0) return s * f[1] * f[2];
  if (k == 1) return s * f[0] * f[2];
  return s * f[0] * f[1];
}
// The same derivatives, direction by direction.  With node signs s_am, GP signs
// s_gm and c the GP coordinate,
//   dN_a/dxi_k(g) = s_ak / 2 * w(s_a1 s_g1) * w(s_a2 s_g2),
// (m1, m2) the two directions other than k, w(+1) = (1 + c) / 2 and w(-1) =
// (1 - c) / 2: a half difference along k and interpolations along m1 and m2.
// An element's eight lanes hold one node and one Gauss point each, both with
// the lane's sign bits, so each of the three combines the lane's own value with
// that of one partner lane.  Lane l = 0..7 of an element has the sign bits
// x = l2, y = l1 ^ l2, z = l0 ^ l2, which makes the partners across x, y and z
// the lanes l ^ 7, l ^ 2 and l ^ 1: the three exchanges that are one DPP move
// each (row_half_mirror and two quad permutations).
//   Scales and signs are left out of the combinations: an interpolation is
// v + r v', r = (1 - c) / (1 + c), and a difference v - v'.  The derivatives
// they give are the true ones over HEX_SC = ((1 + c) / 2)^2 / 2, column k with
// the factor s_gk.  Both cancel in H = G_u J^-1; the cofactors of the current
// Jacobian carry HEX_SC^-2 and the product of the other two signs, and the
// transposed combinations give back HEX_SC and, where column k of Q keeps the
// factor s_gk, differences again: one constant, +-HEX_SC^3 by the product of
// the lane's signs, stands for them all.
constexpr double HEX_GPOS = 0.577350269189626;
constexpr double HEX_R = (1.0 - HEX_GPOS) / (1.0 + HEX_GPOS);
constexpr double HEX_CP = 0.5 * (1.0 + HEX_GPOS);
constexpr double HEX_SC = 0.5 * HEX_CP * HEX_CP;
__device__ __forceinline__ int lane_bits(int l) { return l ^ (3 * ((l >> 2) & 1)); }   // 4 x + 2 y + z
// reference node (-,-,-) (+,-,-) (+,+,-) (-,+,-) (-,-,+) ... of sign bits b;
// the Gauss point of sign bits b is b itself (xi outer, zeta inner)
__host__ __device__ constexpr int hex_node(int b) {
  return 4 * (b & 1) + ((b & 2) ? 3 - ((b >> 2) & 1) : (b >> 2) & 1);
}

// The value v of the partner lane across direction DIR (0 = x, 1 = y, 2 = z).
template <int DIR>
__device__ __forceinline__ float partner(float v) {
  constexpr int ctrl = DIR == 0 ? 0x141 : DIR == 1 ? 0x4E : 0xB1;
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ctrl, 0xf, 0xf, true));
}
template <int DIR>
__device__ __forceinline__ double partner(double v) {
  constexpr int ctrl = DIR == 0 ? 0x141 : DIR == 1 ? 0x4E : 0xB1;
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true));
}

// v + r v' of a lane's own value and its partner's
__device__ __forceinline__ float interp_of(float v, float w) { return __builtin_fmaf((float)HEX_R, w, v); }
__device__ __forceinline__ double interp_of(double v, double w) { return __builtin_fma(HEX_R, w, v); }

// Interpolation along DIR over (1 + c) / 2 (its transpose is the same
// combination).  In FP32 the exchange folds into the sum.
template <int DIR>
__device__ __forceinline__ float interp(float v) {
  return v + partner<DIR>((float)HEX_R * v);
}
template <int DIR>
__device__ __forceinline__ double interp(double v) {
  return __builtin_fma(HEX_R, partner<DIR>(v), v);
}

// Derivatives over HEX_SC, columns with their signs left out, of a nodal value:
// the three share their first exchanges (6 in all).
template <typename R>
__device__ __forceinline__ void hex_grad(R x, R (&d)[3]) {
  const R xz = partner<2>(x);
  const R a = interp_of(x, xz), dz = x - xz;
  const R ay = partner<1>(a);
  const R b = interp_of(a, ay), dy = a - ay;
  d[0] = b - partner<0>(b);
  d[1] = interp<0>(dy);
  d[2] = interp<0>(interp<1>(dz));
}

// The transpose: sum_g sum_k q_k(g) dN_a/dxi_k(g) over HEX_SC at the lane's
// node, column k of q with the factor s_gk.
template <typename R>
__device__ __forceinline__ R hex_grad_t(R qx, R qy, R qz) {
  const R b = qx - partner<0>(qx), c = interp<0>(qy), g = interp<1>(interp<0>(qz));
  const R a = (b + c) + partner<1>((R)HEX_R * b - c);
  return (a + g) + partner<2>((R)HEX_R * a - g);
}

// x less the value of the element's first lane (a broadcast within each half
// of a 16-lane row)
__device__ __forceinline__ double minus_first(double x) {
  const long long v = __double_as_longlong(x);
  long long t = __builtin_amdgcn_update_dpp(v, v, 0x150, 0xf, 0x3, false);   // row_newbcast:0
  t = __builtin_amdgcn_update_dpp(t, v, 0x158, 0xf, 0xc, false);             // row_newbcast:8
  return x - __longlong_as_double(t);
}

// The FP32 kernels form the same derivatives by Walsh-Hadamard sums: with V(h) = sum_a (prod_{m in h} s_am) x_a,
//   sum_a x_a dN_a/dxi_k(g) = 1/8 [V(k) + c s_g1 V(k|m1) + c s_g2 V(k|m2)
//   + c^2 s_g1 s_g2 V(7)],
//   sum_g Q(g) dN_a/dxi_k(g) = 1/8 s_ak [U0 + c s_a1 U1 + c s_a2 U2
//   + c^2 s_a1 s_a2 U12],
// U the sums over g of Q(g), s_g1 Q(g), s_g2 Q(g), s_g1 s_g2 Q(g).  V and U are
// per element and go through LDS.
// in-place Walsh-Hadamard butterfly over bit m of an 8-slot array: slot
// b | m becomes the signed difference (+ side minus - side)
template <typename R>
__device__ __forceinline__ void wht_stage(R (&v)[8], int m) {
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    if (b & m) continue;
    const R lo = v[b], hi = v[b | m];
    v[b] = lo + hi;
    v[b | m] = hi - lo;
  }
}

// U0, U1, U2, U12 of the 8 GP values q[b] of Q(3i+k): pair sums over the
// k-sign, then the two-direction Hadamard over (m1, m2).
template <typename R>
__device__ __forceinline__ void u4_of_q(const R* q, int k, R* u) {
  const int hk = 4 >> k, h1 = k == 0 ? 2 : 4, h2 = k == 2 ? 2 : 1;
  R p[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    // t = 2 b1 + b2: the GPs with m1-sign b1 and m2-sign b2
    const int b = ((t >> 1) ? h1 : 0) | ((t & 1) ? h2 : 0);
    p[t] = q[b] + q[b | hk];
  }
  const R s0 = p[0] + p[1], d0 = p[1] - p[0], s1 = p[2] + p[3], d1 = p[3] - p[2];
  u[0] = s0 + s1;   // sum
  u[1] = s1 - s0;   // m1-signed
  u[2] = d0 + d1;   // m2-signed
  u[3] = d1 - d0;   // m1 m2-signed
}

template <typename R>
__host__ __device__ __forceinline__ R hex_shape(int a, int g) {
  const double gpos = 0.577350269189626;
  const R cp = (R)(0.5 * (1.0 + gpos)), cm = (R)(0.5 * (1.0 - gpos));
  R f0 = (node_sign(a, 0) == gp_sign(g, 0)) ? cp : cm;
  R f1 = (node_sign(a, 1) == gp_sign(g, 1)) ? cp : cm;
  R f2 = (node_sign(a, 2) == gp_sign(g, 2)) ? cp : cm;
  return f0 * f1 * f2;
}

// Load tables: DISCRETE[,SMOOTH] (sld_funbou.f90 itask 2), rows (vx,vy,vz,t).
__device__ __forceinline__ double funbou(const double* __restrict__ tab, int npts,
                                         int smooth, int c, double t) {
#pragma clang fp contract(off)
  double x = 0.0;
  for (int i = 0; i < npts - 1; ++i) {
    double t1 = tab[4 * i + 3], t2 = tab[4 * (i + 1) + 3];
    if (t >= t1 && t <= t2) {
      double p1 = tab[4 * i + c], p2 = tab[4 * (i + 1) + c], m;
      if (smooth == 1) {
        m = (t - t1) / (t2 - t1);
        x = p1 + (p2 - p1) * (m * m * m) * (10.0 - 15.0 * m + 6.0 * (m * m));
      } else {
        m = (p2 - p1) / (t2 - t1);
        x = p1 + m * (t - t1);
      }
      break;
    }
  }
  double tlast = tab[4 * (npts - 1) + 3];
  if (t > tlast) x = tab[4 * (npts - 1) + c] * t / tlast;
  return x;
}

// The same value with the table's length, interpolation and first 4 rows loaded
// at once (tables are [..][maxpts][4]): one trip to memory for a table of up
// to 4 rows, where the search by rows makes one for each.  A node's chain of
// such trips and the interpolation were 0.7 to 1.3 of the ~9 us a step of a
// small mesh takes; so loaded, 0.1 to 0.2 less (2583 elements 9.34 -> 9.14 us,
// 7200 9.67 -> 9.48).  Rows taken by scalar loads ahead of the node's own: 9.53.
struct LoadRows {
  double r[4][4];
  int npts, smooth;
};
__device__ __forceinline__ LoadRows load_rows(const double* __restrict__ tab, const int32_t* __restrict__ npts,
                                              const int32_t* __restrict__ smooth, int maxpts, int fn) {
  LoadRows q;
  q.npts = npts[fn];
  q.smooth = smooth[fn];
  const double* f = tab + (size_t)fn * maxpts * 4;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = min(j, maxpts - 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) q.r[j][c] = f[4 * row + c];
  }
  return q;
}
__device__ __forceinline__ double funbou_rows(const LoadRows& q, const double* __restrict__ tab, int maxpts,
                                              int fn, int c, double t) {
#pragma clang fp contract(off)
  if (q.npts > 4) return funbou(tab + (size_t)fn * maxpts * 4, q.npts, q.smooth, c, t);
  bool in = false;
  double t1 = 0.0, t2 = 1.0, p1 = 0.0, p2 = 0.0, tlast = q.r[0][3], plast = q.r[0][c];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i >= q.npts - 1) continue;
    const double a = q.r[i][3], b = q.r[i + 1][3];
    if (!in && t >= a && t <= b) {
      in = true;
      t1 = a;
      t2 = b;
      p1 = q.r[i][c];
      p2 = q.r[i + 1][c];
    }
    tlast = b;
    plast = q.r[i + 1][c];
  }
  double x = 0.0, m;
  if (in) {
    if (q.smooth == 1) {
      m = (t - t1) / (t2 - t1);
      x = p1 + (p2 - p1) * (m * m * m) * (10.0 - 15.0 * m + 6.0 * (m * m));
    } else {
      m = (p2 - p1) / (t2 - t1);
      x = p1 + m * (t - t1);
    }
  }
  if (t > tlast) x = plast * t / tlast;
  return x;
}

// Run health.  The reference stops the run on a non-positive Jacobian det F
// at a Gauss point (sld_elmpre.f90:229-240 keeps the smallest one and its
// element, sld_elmope.f90:106 -> sld_detjac.f90:93 calls runend) and on a
// NaN or infinite displacement or force residual (sld_cvgunk.f90:195-199).
// Here the kernel that meets such a state records it and sets `halted`;
// every step kernel returns at once while `halted` is set, so the device
// state stays as it was when the failure was found and the host reports it.
struct Health {
  // 0 = none; else (|det F| as FP32 bits) << 32 | (0xffffffff - element):
  // atomicMax keeps the most negative det F, ties to the lowest element
  unsigned long long detf;
  unsigned long long node;   // ~0 = none; else the lowest node with a non-finite value
  unsigned halted;           // bit 0: det F <= 0, bit 1: non-finite state
  unsigned pad;
};
constexpr unsigned HALT_DETF = 1u, HALT_NONFINITE = 2u;

__device__ __forceinline__ void report_detf(Health* h, int64_t e, double detF) {
  const float mag = fabsf((float)detF);
  const unsigned long long key = ((unsigned long long)__float_as_uint(mag) << 32) |
                                 (unsigned long long)(0xffffffffu - (uint32_t)e);
  atomicMax(&h->detf, key);
  atomicOr(&h->halted, HALT_DETF);
}
__device__ __forceinline__ void report_nonfinite(Health* h, int64_t node) {
  atomicMin(&h->node, (unsigned long long)node);
  atomicOr(&h->halted, HALT_NONFINITE);
}

// fixmask bits: 1, 2, 4 = prescribed x, y, z; FIX_FORCE = the node carries
// a nonzero entry of the nodal force pattern fext0 (set by the library); the
// upper four bits = the node's load function + 1 (0 = none), FIX_FUNC_LOOKUP =
// in func_of_node: the mask says which table to load without a trip of its own.
constexpr int FIX_FORCE = 8, FIX_FUNC_SHIFT = 4, FIX_FUNC_LOOKUP = 15;

struct NodalArgs {
  int64_t npoin;
  double* u[3];
  double* v[3];
  double* a[3];
  void* fint[3];               // double or float per precision mode
  int fint_fp32;
  const double* rmass;         // 1/m per node
  const uint8_t* fixmask;
  const int32_t* func_of_node; // may be null
  const double* func_table;    // [nfunc][maxpts][4]
  const int32_t* func_npts;
  const int32_t* func_smooth;
  int32_t func_maxpts;
  const double* fext0[3];      // may be null
  int32_t fext_func;           // -1 = none
  double* clock;               // [2] device time, slot tn = t^n
  int32_t tn;
  int32_t zero_fint;           // coloured scatter: the predictor clears f_int
  const int32_t* node_ptr;     // gather: [npoin+1] slot ranges per node, else null
  int32_t slot_width;          // gather with W slots per node (node i: W i ..), or 0
  const void* efor;            // gather: corner forces [slot][3] (double or float),
                               // slots of a node in ascending element order
  unsigned* sur_count;         // surrogate list segment counters, cleared per step
  // energy balance (mod_sld_energy.f90), when du is non-null: the predictor
  // stores du = u^{n+1} - u^n, the corrector writes per-block partial sums of
  // (f_int^{n+1} + f_int^n).du, (f_ext^{n+1} + f_ext^n).du and m v.v
  double* du[3];
  double* fint_prev[3];
  double* fext_prev[3];
  const double* mass;
  double* energy_part;         // [3][gridDim of the corrector]
  // boundary-face loads: [npoin+1] slot ranges per node (null = no faces)
  // and the face-corner forces of the step [slot][3]
  const int32_t* node_face_ptr;
  const double* fface;
  // gravity (sld_dev_set_gravity): f_ext += m g at every dof; mass is set
  int32_t gravity;
  double grav[3];
  // body force (sld_dev_set_body_force): f_ext += m b(t^{n+1}), b from load
  // function body_func by the rule of sld_funbou.f90 itask 3; mass is set
  int32_t body_func;           // -1 = none
  // Rayleigh damping (sld_dev_set_damping): the central-difference
  // predictor keeps v^n in vdamp (the element's veloc_sld(ITER_K)); the
  // corrector sums each node's corner damping forces (edamp, laid out as
  // efor) into the residual and stores them in fdamp at a run's last step
  double* vdamp[3];            // null: no damping or Tchamwa-Wielgosz
  const void* edamp;           // null: no damping
  double* fdamp[3];
  Health* health;              // run health (never null)
};

// Body-force value of component c at time t (sld_funbou.f90:142-167, itask
// 3): linear between the rows with t1 <= t < t2, value m t + b with
// m = (p2 - p1)/(t2 - t1), b = p1 - m t1; zero outside the table.
__device__ __forceinline__ double funbou_body(const double* __restrict__ tab, int npts, int c,
                                              double t) {
#pragma clang fp contract(off)
  for (int i = 0; i < npts - 1; ++i) {
    const double t1 = tab[4 * i + 3], t2 = tab[4 * (i + 1) + 3];
    if (t >= t1 && t < t2) {
      const double p1 = tab[4 * i + c], p2 = tab[4 * (i + 1) + c];
      const double m = (p2 - p1) / (t2 - t1);
      const double b = p1 - m * t1;
      return m * t + b;
    }
  }
  return 0.0;
}

// Boundary faces with Neumann loads (sld_bouope.f90), one QUA04 face per
// thread; corner forces go to node-sorted slots that the corrector sums.
struct FaceArgs {
  int64_t nface;
  const int32_t* lnodb;        // [nface][4]
  const int32_t* code;         // [nface] 3 pressure, 6 traction
  const double* value;         // [nface][3]
  const int32_t* func;         // [nface] or null
  int32_t transient, follower;
  const double* coord[3];
  const double* u[3];          // u^{n+1} (follower loads)
  const uint8_t* fixmask;
  const double* func_table;
  const int32_t* func_npts;
  const int32_t* func_smooth;
  int32_t func_maxpts;
  const int32_t* slot;         // [4 nface] slot of each face corner
  double* fface;               // [4 nface][3]
  const double* clock;
  int32_t tn;
};

// Predictor of node i from the step-n state (u, v, a): u^{n+1} with the
// Dirichlet values at t^{n+1} = cutim, and v^{n+1/2} (CD) or v^{n+1} (TW).
// scheme: 0 = central difference, 1 = Tchamwa-Wielgosz.  uvw = the state,
// already loaded.
__device__ __forceinline__ void predict_vals(const NodalArgs& A, int64_t i, int scheme, double dt,
                                             double phi, double cutim, int fix, const double u0[3],
                                             const double v0[3], const double a0[3], double un[3],
                                             double vn[3]) {
#pragma clang fp contract(off)
  const double t_end = cutim + dt, t_mid = 0.5 * (cutim + t_end);
  double fv[3] = {0.0, 0.0, 0.0};
  if ((fix & 7) && (fix >> FIX_FUNC_SHIFT)) {
    const int fc = fix >> FIX_FUNC_SHIFT, fn = fc == FIX_FUNC_LOOKUP ? A.func_of_node[i] : fc - 1;
    const LoadRows q = load_rows(A.func_table, A.func_npts, A.func_smooth, A.func_maxpts, fn);
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if ((fix >> d) & 1) fv[d] = funbou_rows(q, A.func_table, A.func_maxpts, fn, d, cutim);
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double u = u0[d], v = v0[d], a = a0[d];
    if (scheme == 0) {
      vn[d] = v + (t_mid - cutim) * a;
      un[d] = u + dt * vn[d];
    } else {
      vn[d] = v + dt * a;
      un[d] = u + dt * v + phi * (dt * dt) * a;
    }
    if ((fix >> d) & 1) un[d] = fv[d];
  }
}

// Stores the predicted state (and du for the energy balance); the coloured
// scatter also clears f_int for the element launches that add into it.
__device__ __forceinline__ void store_prediction(const NodalArgs& A, int64_t i, const double u0[3],
                                                 const double un[3], const double vn[3],
                                                 const double vprev[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (A.vdamp[0]) A.vdamp[d][i] = vprev[d];
    if (A.du[0]) A.du[d][i] = un[d] - u0[d];
    A.u[d][i] = un[d];
    A.v[d][i] = vn[d];
    if (A.zero_fint) {
      if (A.fint_fp32) ((float*)A.fint[d])[i] = 0.f;
      else ((double*)A.fint[d])[i] = 0.0;
    }
  }
}

template <int SCHEME>  // 0 = central difference, 1 = Tchamwa-Wielgosz
__global__ void __launch_bounds__(256) sld_predict(NodalArgs A, double dt, double phi) {
  if (A.health->halted) return;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.npoin) return;
  double u[3], v[3], a[3], un[3], vn[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    u[d] = A.u[d][i];
    v[d] = A.v[d][i];
    a[d] = A.a[d][i];
  }
  predict_vals(A, i, SCHEME, dt, phi, A.clock[A.tn] + dt, A.fixmask[i], u, v, a, un, vn);
  store_prediction(A, i, u, un, vn, v);
  if (!(isfinite(un[0]) && isfinite(un[1]) && isfinite(un[2]))) report_nonfinite(A.health, i);
}

// Gather assembly: f_int at node i = 0 + f_(e1) + f_(e2) + ... over the
// element corners at the node in ascending (colour-sorted) element order,
// which is the order in which the coloured scatter adds them.
// Slots padded to W per node (W = the mesh's largest corner count, unused
// slots zero): node i's values sit at a fixed place, so the loads need no
// slot range and the wave's loads are contiguous; W = 8 (hex meshes) loads
// all 24 values at once.  Trailing zeros leave the ordered sum unchanged.
// Without padding, a node with 8 corners still loads them in one round trip.
template <typename R>
__device__ __forceinline__ void gather_fint(const NodalArgs& A, int64_t i, double fi[3],
                                            bool store, const void* slots = nullptr) {
  const int W = A.slot_width;
  const int32_t k0 = W ? W * (int32_t)i : A.node_ptr[i];
  const int32_t k1 = W ? k0 + W : A.node_ptr[i + 1];
  const R* ef = (const R*)(slots ? slots : A.efor) + 3 * (int64_t)k0;
  R s0 = R(0), s1 = R(0), s2 = R(0);
  if (k1 - k0 == 8) {
    R c[24];
#pragma unroll
    for (int j = 0; j < 24; ++j) c[j] = ef[j];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s0 += c[3 * j];
      s1 += c[3 * j + 1];
      s2 += c[3 * j + 2];
    }
  } else {
    for (int32_t k = 0; k < k1 - k0; ++k) {
      s0 += ef[3 * k];
      s1 += ef[3 * k + 1];
      s2 += ef[3 * k + 2];
    }
  }
  if (store && !slots) {
    ((R*)A.fint[0])[i] = s0;
    ((R*)A.fint[1])[i] = s1;
    ((R*)A.fint[2])[i] = s2;
  }
  fi[0] = (double)s0;
  fi[1] = (double)s1;
  fi[2] = (double)s2;
}

// Per-node energy terms of one step: internal-force and external-force work
// over the displacement increment (trapezoidal, mod_sld_energy.f90:113-131)
// and m v.v (mod_sld_energy.f90:134-140); f_int^{n+1} and f_ext^{n+1} replace
// the previous step's.
__device__ __forceinline__ void node_energy(const NodalArgs& A, int64_t i, const double fg[3],
                                            const double fe[3], const double vel[3],
                                            double e[3]) {
#pragma clang fp contract(off)
  double ie = 0.0, wk = 0.0, ke = 0.0;
  const double m = A.mass[i];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double du = A.du[d][i];
    ie = ie + (fg[d] + A.fint_prev[d][i]) * du;
    wk = wk + (fe[d] + A.fext_prev[d][i]) * du;
    A.fext_prev[d][i] = fe[d];
    const double v = vel[d];
    ke = ke + v * v * m;
    A.fint_prev[d][i] = fg[d];
  }
  e[0] = ie;
  e[1] = wk;
  e[2] = ke;
}

// Corrector of node i.  FUSE (inside a captured run of steps): the
// corrected a and v stay in registers and the next step's predictor runs
// on them at t^{n+2} = t^{n+1} + dt, with the same arithmetic as its own
// kernel; a, v^{n+1} and f_int reach memory only at the last step of the run.
// The node's loads are all issued first; the load function of the nodal
// force pattern is evaluated only at nodes that carry one (FIX_FORCE).
template <int SCHEME, bool FUSE>
__device__ __forceinline__ void correct_node(const NodalArgs& A, int64_t i, double dt, double phi,
                                             double e[3]) {
#pragma clang fp contract(off)
  const double rm = A.rmass[i];
  const int fix = A.fixmask[i];
  double fg[3];
  if (A.node_ptr) {
    if (A.fint_fp32) gather_fint<float>(A, i, fg, !FUSE);
    else gather_fint<double>(A, i, fg, !FUSE);
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d)
      fg[d] = A.fint_fp32 ? (double)((const float*)A.fint[d])[i] : ((const double*)A.fint[d])[i];
  }
  double v0[3], u0[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    v0[d] = A.v[d][i];
    if (FUSE) u0[d] = A.u[d][i];
  }
  const double cutim = A.clock[A.tn] + dt;  // t^{n+1}
  const double t_end = cutim + dt, t_mid = 0.5 * (cutim + t_end);
  // f_ext: face loads (summed per node in face order) + fx fext0
  double fe[3] = {0.0, 0.0, 0.0};
  if (A.node_face_ptr) {
    const int32_t k0 = A.node_face_ptr[i], k1 = A.node_face_ptr[i + 1];
    for (int32_t k = k0; k < k1; ++k) {
#pragma unroll
      for (int d = 0; d < 3; ++d) fe[d] = fe[d] + A.fface[3 * (int64_t)k + d];
    }
  }
  if (A.fext_func >= 0 && (fix & FIX_FORCE)) {
    const LoadRows q = load_rows(A.func_table, A.func_npts, A.func_smooth, A.func_maxpts, A.fext_func);
    const double fx = funbou_rows(q, A.func_table, A.func_maxpts, A.fext_func, 0, cutim);
#pragma unroll
    for (int d = 0; d < 3; ++d) fe[d] = fe[d] + fx * A.fext0[d][i];
  }
  if (A.gravity || A.body_func >= 0) {
    // the element load sum_g N_a rho (g + b) w detJ (sld_elmmat.f90:152-157)
    // of every element at the node: the lumped mass times g + b(t^{n+1})
    const double m = A.mass[i];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double gb = A.gravity ? A.grav[d] : 0.0;
      if (A.body_func >= 0)
        gb = gb + funbou_body(A.func_table + (size_t)A.body_func * A.func_maxpts * 4,
                              A.func_npts[A.body_func], d, cutim);
      fe[d] = fe[d] + m * gb;
    }
  }
  // Rayleigh damping forces of the node's element corners
  double fd[3] = {0.0, 0.0, 0.0};
  if (A.edamp) {
    if (A.fint_fp32) gather_fint<float>(A, i, fd, false, A.edamp);
    else gather_fint<double>(A, i, fd, false, A.edamp);
    if (!FUSE) {
#pragma unroll
      for (int d = 0; d < 3; ++d) A.fdamp[d][i] = fd[d];
    }
  }
  double an[3], vn[3];
  bool finite = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    double fi = fg[d];
    double r = 0.0 - fi;
    r = r - fd[d];
    r = r + fe[d];
    finite = finite && isfinite(r);
    double acc = 0.0 + r * rm;
    if (SCHEME == 0) {
      an[d] = acc;
      vn[d] = v0[d] + (t_end - t_mid) * acc;
    } else {
      vn[d] = v0[d];
      if ((fix >> d) & 1) { vn[d] = 0.0; acc = 0.0; }
      an[d] = acc;
    }
    if (!FUSE) {
      A.a[d][i] = an[d];
      if (SCHEME == 0 || ((fix >> d) & 1)) A.v[d][i] = vn[d];
    }
  }
  if (A.energy_part) node_energy(A, i, fg, fe, vn, e);
  if (!finite) report_nonfinite(A.health, i);
  if (FUSE) {
    double un[3], vp[3];
    predict_vals(A, i, SCHEME, dt, phi, cutim + dt, fix, u0, vn, an, un, vp);
    store_prediction(A, i, u0, un, vp, vn);
    if (!(isfinite(un[0]) && isfinite(un[1]) && isfinite(un[2]))) report_nonfinite(A.health, i);
  }
  if (i == 0) {
    A.clock[1 - A.tn] = cutim;
  }
}

// Fixed-order block sum of three values; thread 0 writes part[k*gridDim.x + b].
__device__ __forceinline__ void block_sum3(double e[3], double* part) {
  __shared__ double red[3][256];
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 3; ++k) red[k][t] = e[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
#pragma unroll
      for (int k = 0; k < 3; ++k) red[k][t] = red[k][t] + red[k][t + w];
    }
    __syncthreads();
  }
  if (t == 0) {
#pragma unroll
    for (int k = 0; k < 3; ++k) part[(size_t)k * gridDim.x + blockIdx.x] = red[k][0];
  }
}

template <int SCHEME, bool FUSE>
__global__ void __launch_bounds__(256) sld_correct(NodalArgs A, double dt, double phi) {
#pragma clang fp contract(off)
  if (A.health->halted) return;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double e[3] = {0.0, 0.0, 0.0};
  if (i < A.npoin) correct_node<SCHEME, FUSE>(A, i, dt, phi, e);
  // the next step's surrogate list starts empty
  if (A.sur_count)
    for (int64_t k = i; k < mlp::LIST_SEGS; k += (int64_t)gridDim.x * blockDim.x)
      A.sur_count[k * mlp::LIST_STRIDE] = 0u;
  if (A.energy_part) block_sum3(e, A.energy_part);
}

// Sums the corrector's partials in a fixed order and advances the totals
// acc = {allie, allwk, allke, etota, steps} (mod_sld_energy.f90:141-162): the
// first step after a reset takes the full increment, later ones half the
// trapezoid.
__global__ void __launch_bounds__(256) sld_energy_reduce(const double* part, int nparts,
                                                         double* acc, const Health* health) {
#pragma clang fp contract(off)
  if (health->halted) return;
  double e[3] = {0.0, 0.0, 0.0};
  for (int b = threadIdx.x; b < nparts; b += 256) {
#pragma unroll
    for (int k = 0; k < 3; ++k) e[k] = e[k] + part[(size_t)k * nparts + b];
  }
  __shared__ double red[3][256];
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 3; ++k) red[k][t] = e[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
#pragma unroll
      for (int k = 0; k < 3; ++k) red[k][t] = red[k][t] + red[k][t + w];
    }
    __syncthreads();
  }
  if (t == 0) {
    const double w = acc[4] == 0.0 ? 1.0 : 0.5;
    acc[0] = acc[0] + w * fabs(red[0][0]);
    acc[1] = acc[1] + w * fabs(red[1][0]);
    acc[2] = 0.5 * red[2][0];
    acc[3] = acc[0] + acc[2] - acc[1];
    acc[4] = acc[4] + 1.0;
  }
}

// Face loads of one step at t^{n+1} (sld_bouope.f90:88-277 with the values
// of sld_updbcs.f90:153-181): geometry of the face's 4 nodes (reference, or
// current with follower loads); value = the constant one, or under transient
// conditions (column x of the face's function, 0, 0) and 0 without one
// (sld_funbou.f90 itask 1); at the 2x2 Gauss points (s outer, t inner,
// mod_quadrature_gauss.f90:2361-2370) the tangents of bouder
// (mod_bouder.f90:74-89), n = t_s x t_t, |n|, the unit normal of chenor, the
// traction (code 3: value_1 n/|n|, code 6: value) and the corner forces
// |n| tract N_a on dofs that are not prescribed (QUA04 of mod_lagrange.f90).
__global__ void __launch_bounds__(256) sld_face_load(FaceArgs F, double dt) {
#pragma clang fp contract(off)
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= F.nface) return;
  const double cutim = F.clock[F.tn] + dt;
  int32_t nb[4];
  double x[4][3];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    nb[a] = F.lnodb[4 * f + a];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      x[a][d] = F.coord[d][nb[a]];
      if (F.follower) x[a][d] = x[a][d] + F.u[d][nb[a]];
    }
  }
  double val[3];
  if (F.transient) {
    const int fn = F.func ? F.func[f] : -1;
    val[0] = fn >= 0 ? funbou(F.func_table + (size_t)fn * F.func_maxpts * 4, F.func_npts[fn],
                              F.func_smooth[fn], 0, cutim)
                     : 0.0;
    val[1] = 0.0;
    val[2] = 0.0;
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d) val[d] = F.value[3 * f + d];
  }
  const int code = F.code[f];
  const double g = 0.577350269189626;
  double elfex[4][3];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int d = 0; d < 3; ++d) elfex[a][d] = 0.0;
  for (int ig = 0; ig < 4; ++ig) {
    const double s = ig < 2 ? -g : g, t = (ig & 1) ? g : -g, st = s * t;
    const double N[4] = {(1.0 - t - s + st) * 0.25, (1.0 - t + s - st) * 0.25,
                         (1.0 + t + s + st) * 0.25, (1.0 + t - s - st) * 0.25};
    const double ds[4] = {(-1.0 + t) * 0.25, (1.0 - t) * 0.25, (1.0 + t) * 0.25,
                          (-1.0 - t) * 0.25};
    const double dtt[4] = {(-1.0 + s) * 0.25, (-1.0 - s) * 0.25, (1.0 + s) * 0.25,
                           (1.0 - s) * 0.25};
    double t1[3], t2[3], n[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      t1[d] = 0.0;
      t2[d] = 0.0;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        t1[d] = t1[d] + x[a][d] * ds[a];
        t2[d] = t2[d] + x[a][d] * dtt[a];
      }
    }
    n[0] = t1[1] * t2[2] - t1[2] * t2[1];
    n[1] = t1[2] * t2[0] - t1[0] * t2[2];
    n[2] = t1[0] * t2[1] - t1[1] * t2[0];
    const double eucta = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    const double gbsur = 1.0 * eucta;
    double tract[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) tract[d] = code == 3 ? (n[d] / eucta) * val[0] : val[d];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int fix = F.fixmask[nb[a]];
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (!((fix >> d) & 1)) elfex[a][d] = elfex[a][d] + gbsur * tract[d] * N[a];
    }
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int64_t k = F.slot[4 * f + a];
#pragma unroll
    for (int d = 0; d < 3; ++d) F.fface[3 * k + d] = elfex[a][d];
  }
}

// ----------------------------------------------------------------------------
// Element kernel
// ----------------------------------------------------------------------------
struct ElemArgs {
  int32_t e_begin, e_end;       // range of the launch in elem_list (or of elements)
  const int32_t* elem_list;     // scatter: elements sorted by colour; gather: null (identity)
  int64_t nelem;
  const int32_t* lnods;         // [nelem][8]
  const double* coord[3];       // SoA reference coordinates
  const double* u[3];           // SoA displacement (ITER_K)
  const double* props;          // [nmat][18]
  const double* law_const;      // [nmat][8] sma::law_constants of each material
  const int32_t* mat_of_elem;   // [nelem] or null
  const double* E_of_elem;      // [nelem] or null
  const double* kg;             // [nelem][2] bulk and shear modulus per element
  const uint8_t* law_of_elem;   // [nelem] 1 = neo-Hookean (model 102), 0 = SMA; null = all SMA
  const double* sdv_n[3];       // TIME_N history, SoA over GP = 8*e + g
  double* sdv_k[3];             // ITER_K history
  void* fint[3];                // scatter: nodal internal force (double or float)
  void* efor;                   // gather: corner forces [slot][3] (double or float)
  const int32_t* corner_slot;   // gather: [8 * e + a] -> slot of the corner at its node
  double* S_out;                // optional PK2 [9][ngp]
  double* P_out;                // optional first Piola F S [9][ngp] (with S_out)
  uint32_t* flags_out;          // optional [ngp]
  unsigned long long* counters; // [COUNTER_SLOTS][8] per-flag Gauss-point counts
  Health* health;               // run health (never null)
  // Rayleigh damping (DAMP kernels): veloc_sld(ITER_K) of the step (v^n in
  // the central difference, the predicted v^{n+1} in Tchamwa-Wielgosz),
  // (alpha, beta) and density per material, corner damping forces
  const double* vel[3];
  const double* damping;        // [nmat][2]
  const double* rho;            // [nmat]
  void* edamp;                  // [slot][3] (double or float)
  int32_t one_f;                // F_AS = F_SA: sdv_n[2], sdv_k[2] are sdv_n[1], sdv_k[1]
  int32_t xcd_remap;            // 1 = spread consecutive tiles per XCD
  int32_t tiles_per_block;      // > 0: persistent launch, tiles per workgroup
  // surrogate (mode 2): per-GP status from the prepass (0 not flagged,
  // 1 listed, 2 flagged and not listed), the listed points' slots, their
  // features and the network's outputs by slot
  uint8_t* sur_status;
  int32_t* sur_slot;            // [gp], valid where status is 1
  float* sur_feat;              // [cap][16]
  const float* sur_Y;           // [cap][12]
  double sur_tol;               // acceptance tolerance on xS
  unsigned* sur_count;          // the list's segment counters (mlp::LIST_SEGS)
  int64_t sur_seg_cap;          // slots per segment
  double T_feat;                // temperature fed to the surrogate (inert in the law)
  // surrogate candidates: per element, 1 when one of its points transformed
  // in the previous step (the prepass lists points of those elements only;
  // every other point takes the exact map), and the flags the step writes
  // for the next one; null: every element is a candidate
  const uint8_t* sur_cand;
  uint8_t* sur_cand_next;
};

// Flag counters live in COUNTER_SLOTS slots of 8 (one 64-byte line each);
// workgroup b adds into slot b % COUNTER_SLOTS, so the per-wave atomics of a
// launch spread over many addresses instead of serialising on one.  The host
// sums the slots.
constexpr int COUNTER_SLOTS = 256;

// Surrogate mode, one Gauss point: a listed point takes the network's xS
// when it lies within tol of the return map's solution (|R(x)/R'(x)| of the
// single-branch consistency residual, exact because that residual is linear
// in the increment on one branch) and in [-1e-3, 1 + 1e-3]; every other
// point takes the exact map.  Flags: FLAG_SURR_USED on accepted transforming
// points, FLAG_SURR_FALLBACK on flagged points that took the exact map.
__device__ inline sma::ReturnMap surrogate_or_exact(const ElemArgs& A, const sma::Mat& m, int64_t gp,
                                                   double theta, double e_n, double xS0,
                                                   double FAS0, double FSA0) {
  const uint8_t st = A.sur_status[gp];
  bool ok = false;
  double x = 0.0;
  if (st == 1) {
    const int64_t slot = A.sur_slot[gp];
    x = xS0 + (double)A.sur_Y[slot * mlp::NOUT + 11] / mlp::Scale::dx;
    ok = (x >= -1e-3) && (x <= 1.0 + 1e-3) &&
         sma::consistency_residual(m, theta, e_n, xS0, FAS0, FSA0, x) <= A.sur_tol;
  }
  sma::ReturnMap rm;
  if (ok) {
    rm = sma::return_map_given(m, theta, e_n, xS0, FAS0, FSA0, x);
    if (rm.flags & 3u) rm.flags |= sma::FLAG_SURR_USED;
  } else {
    rm = sma::return_map(m, theta, e_n, xS0, FAS0, FSA0);
    if (st != 0 && (rm.flags & 3u)) rm.flags |= sma::FLAG_SURR_FALLBACK;
  }
  return rm;
}

// The value of x, opaque to the optimiser: quantities derived from the lane
// index (shape-function derivatives at the lane's Gauss point or node) are
// then recomputed where they are used instead of being hoisted out of the
// tile loop and held in registers through the constitutive update.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Wave-level flag counters: 64-bit atomics on the wave's counter line, lane 0
// adding its KF_AS count and lane 1 its KF_SA count in one instruction; the
// other bits (rare) one by one.
__device__ __forceinline__ void count_flags(unsigned long long* ctr, uint32_t fl, bool valid) {
  if (!valid) fl = 0u;
  if (__ballot(fl != 0u) == 0ull) return;   // wave-uniform: nothing to count
  ctr += 8 * (blockIdx.x % COUNTER_SLOTS);
  static_assert(sma::FLAG_KF_AS == 1u && sma::FLAG_KF_SA == 2u, "counters 0 and 1");
  const int lane = opaque(threadIdx.x) & 63;
  const int n0 = __popcll(__ballot(fl & sma::FLAG_KF_AS));
  const int n1 = __popcll(__ballot(fl & sma::FLAG_KF_SA));
  const int n = lane == 0 ? n0 : n1;
  if (lane < 2 && n) atomicAdd(ctr + lane, (unsigned long long)n);
  const uint32_t bits[5] = {sma::FLAG_NEWTON_FAIL, sma::FLAG_EIGEN_FAIL, sma::FLAG_DETF_NONPOS,
                            sma::FLAG_SURR_USED, sma::FLAG_SURR_FALLBACK};
  if (__ballot(fl & (bits[0] | bits[1] | bits[2] | bits[3] | bits[4])) == 0ull) return;
#pragma unroll
  for (int b = 0; b < 5; ++b) {
    const unsigned long long m = __ballot(fl & bits[b]);
    if (m && lane == 0) atomicAdd(ctr + 2 + b, (unsigned long long)__popcll(m));
  }
}

// Orders one wave's LDS accesses (an element's eight lanes sit in one wave,
// whose LDS operations complete in order): no wait and no workgroup barrier.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// EPB elements per block, 8 threads (one per Gauss point) per element.
// What bounds it (counters): in FP64 on C1, whose state stays in the 256 MB cache,
// VALU issue, 0.86 of the busy cycles (663 instructions a wave, 3 of 4 in FP64, 4
// cycles each); on meshes whose state does not (631 000 elements and more) it
// issues 0.5 to 0.6, as much of a wave's time being waits for memory at 2.7 TB/s.
// FP32 (675 instructions) issues one in 4 cycles on C1 and 0.9 beyond the cache with
// 4 waves a SIMD; that is no ceiling (the neo-Hookean launch reaches 1.3 with 8).
// In FP64 an element's lanes exchange values by DPP moves (hex_grad, hex_grad_t)
// instead of through LDS: with Walsh-Hadamard sums and Gauss-point rows in LDS
// (175 FP64 values read or written per lane) the LDS of a CU, shared by its four
// SIMDs, was as busy as the VALU, and the two overlapped poorly.  FP64 element launch, before -> with exchanges: C1
// 400x20x20 46.7 -> 39.2 us; 631 000 elements in 64 specimens 191 -> 167;
// 691 000 elements of SMA tube in tissue 159 -> 125; 2583 damped elements
// 8.0 -> 6.5.
// R = kinematics/stress precision; the return map is always FP64.
// SUR = 0 plain; 1 surrogate prepass (flags + features of transforming
// points, no stress, no scatter); 2 element step using accepted surrogate
// answers (exact return map otherwise).
// GATHER = false: read-modify-write of f_int (the launch covers one colour);
// true: per-corner forces to efor (the launch may cover every element).
#ifndef SLD_WAVES_F64
#define SLD_WAVES_F64 3
#endif
#ifndef SLD_WAVES_F32
#define SLD_WAVES_F32 4
#endif
#ifndef SLD_WAVES_F64_SMA
#define SLD_WAVES_F64_SMA 5
#endif
// LAWS = 0: each element takes its own law (law_of_elem); LAWS = 1: every
// element of the launch is SMA (a mesh without neo-Hookean elements, or the
// SMA range of a law-grouped mesh), without the neo-Hookean path, whose
// registers would otherwise add to the SMA path's; LAWS = 2: every element of
// the launch is neo-Hookean (the tissue range of a law-grouped mesh), without
// the SMA path (FP64: 72 VGPRs, 7 waves per SIMD; FP32: 63, 8).  The FP64 SMA
// kernel needs 94 VGPRs (5 waves) since nothing of the rarely taken branches
// is held through it: constants of long series and of library functions were
// 32 of its 126 registers (4 waves) and 40 of its ~800 instructions.  C1 38.6
// -> 35.5 us, 64 specimens 158 -> 154.5, tube 117 -> 113; 3 waves: 40 and 178,
// and with 5 registers spilled at 5 waves 38 and 182.  FP32 SMA kernels stay
// at 4 waves (5 spill and are slower).  Kernels that also store the stresses
// (STORE) keep 3 waves in FP64 and 6 in the FP32 neo-Hookean kernel.
template <typename R, int LAWS = 0, bool DAMP = false, bool STORE = false>
struct ElemOccupancy {
  static constexpr int waves = DAMP ? (sizeof(R) == 8 ? 1 : 2)
                               : LAWS == 2 ? (sizeof(R) == 8 ? 4 : (STORE ? 6 : 8))
                               : LAWS == 1 ? (sizeof(R) == 8 ? (STORE ? 3 : SLD_WAVES_F64_SMA)
                                                             : SLD_WAVES_F32)
                                           : (sizeof(R) == 8 ? SLD_WAVES_F64 : SLD_WAVES_F32);
};

// Elements of R in one element's LDS block, padded from n: a multiple of 16
// bytes whose size in 4-byte words is an odd multiple of 4, so that the
// blocks of 8 consecutive elements start 4 banks apart (mod 32) and values
// read at the same offset by the 8 elements of a wave fall in 8 different
// 4-bank groups.
constexpr int lds_block(int n, int rsize) {
  int m = n;
  while ((m * rsize) % 16 != 0 || ((m * rsize) / 4) % 8 != 4) ++m;
  return m;
}

// c with its sign flipped when neg is 1 (neg is 0 or 1): an integer xor on
// the sign bit, so that a lane-dependent signed weight costs no pair of
// constant registers held through the kernel
template <typename R>
__device__ __forceinline__ R sign_if(R c, int neg) {
  if constexpr (sizeof(R) == 8)
    return __longlong_as_double(__double_as_longlong(c) ^ ((long long)(neg & 1) << 63));
  else
    return __int_as_float(__float_as_int(c) ^ (int)((unsigned)(neg & 1) << 31));
}

// DAMP: Rayleigh damping (sld_elmmat.f90:160-163, :174-194) -- the
// element also gathers the velocity, forms at each Gauss point the
// consistent-mass term q = alpha rho detJ v(g) and the beta term's
// z_k = detJ sum_j J^-1_kj w_j, w_j = sum_k L_kj S_jk (L the velocity
// gradient, S the PK2 stress), and writes per corner the damping force
// alpha sum_g N_a q(g) - sum_g sum_k dN_a/dxi_k z_k to edamp.
// ONE_F: the history's two loading functions are one value, read and written
// once, and C_AS and C_SA are finite, so that their terms, times a temperature
// of 0, are left out (FP64: a step of C1 43.3 -> 41.8 us, of 64 specimens
// 188.8 -> 186.6; FP32 keeps one form, whose rounding must not move).
template <typename R, int EPB, bool STORE, int SUR = 0, bool GATHER = false, int LAWS = 0,
          bool DAMP = false, bool ONE_F = false>
__global__ void __launch_bounds__(EPB * 8, (ElemOccupancy<R, LAWS, DAMP, STORE>::waves))
    sld_element(ElemArgs A) {
  constexpr int NC = DAMP ? 9 : 6;        // gathered components: x, u (, v)
  // Two forms of the element's sums.  FP64 (XCH): exchanges between the lanes
  // (hex_grad, hex_grad_t).  FP32: Walsh-Hadamard sums through LDS, the
  // arithmetic that mode's runs have had: a change of rounding in FP32 grows to
  // 2e-4 of the velocities in 200 steps of a cantilever.  (With exchanges the
  // FP32 element launch takes 27.8 instead of 30 us on C1.)
  constexpr bool XCH = sizeof(R) == 8;
  constexpr int NQ = DAMP ? 15 : 9;
  // One LDS block per element (byte offsets; an element's eight lanes sit in
  // one wave, so wave_sync orders them and no workgroup barrier is needed).
  // XCH: the rows of j through the law (FP64), the material constants.  FP32:
  // the relative nodal values, then the Gauss-point rows of Q; V(h), then
  // (without damping) the U sums; the material constants.
  // Blocks are padded (lds_block) so that the 8 elements of a wave start in
  // different LDS banks: the eight lanes of an element read one value at once,
  // and unpadded power-of-two strides put all eight elements' values in one
  // bank.  Rows of 9 let the lanes of an element that read different rows hit
  // different banks.
  constexpr bool JLDS = sizeof(R) == 8;
  constexpr int ROW = 9, VC = DAMP ? 10 : LAWS == 2 ? 6 : 8, U4R = DAMP ? 11 : 8;
  constexpr int V_OFF = XCH ? (JLDS ? 9 * 8 * 8 : 0) : (NQ * ROW * 4 + 15) / 16 * 16;
  constexpr int U_OFF = !XCH && DAMP ? V_OFF + 8 * VC * 4 : V_OFF;
  constexpr int W_OFF = U_OFF + (XCH ? 0 : DAMP ? U4R * 16 : 8 * VC * 4);   // damping: WHT of q_i
  constexpr int C_OFF = W_OFF + (!XCH && DAMP ? 3 * 8 * 4 : 0);
  constexpr int BLK = lds_block(C_OFF + 10 * 8, 1);
  __shared__ __align__(16) unsigned char s_blk[EPB][BLK];
  auto s_row = [&](int l) { return reinterpret_cast<double(*)[8]>(&s_blk[l][0]); };
  auto s_q = [&](int l) { return reinterpret_cast<R(*)[ROW]>(&s_blk[l][0]); };
  auto s_v = [&](int l) { return reinterpret_cast<R(*)[VC]>(&s_blk[l][V_OFF]); };
  auto s_u4 = [&](int l) { return reinterpret_cast<R(*)[4]>(&s_blk[l][U_OFF]); };
  auto s_wq = [&](int l) { return reinterpret_cast<R(*)[8]>(&s_blk[l][W_OFF]); };
  auto s_c = [&](int l) { return reinterpret_cast<double*>(&s_blk[l][C_OFF]); };
  __shared__ double s_v0[!XCH && DAMP ? EPB : 1][3];   // node 0's velocity

  if (A.health->halted) return;
  int bid = blockIdx.x;
  if (A.xcd_remap) {
    // workgroups are dealt round-robin to the 8 XCDs: workgroup b runs on
    // XCD b % 8 as that XCD's (b / 8)-th.  Give each XCD a contiguous run of
    // tiles so neighbouring elements share its L2: XCD x owns q + (x < r)
    // workgroups (nb = 8 q + r), its run starts at x q + min(x, r).
    const int nb = gridDim.x, q = nb >> 3, r = nb & 7;
    const int xcd = bid & 7, k = bid >> 3;
    bid = xcd * q + min(xcd, r) + k;
  }
  // persistent launches give each workgroup a contiguous run of tiles
  const int ntiles = (A.e_end - A.e_begin + EPB - 1) / EPB;
  const int per = A.tiles_per_block > 0 ? A.tiles_per_block : 1;
  const int t_begin = bid * per, t_end = min(ntiles, t_begin + per);
  for (int blk = t_begin; blk < t_end; ++blk) {
  // the thread index passes through an empty asm in every phase, so that what
  // is derived from it (LDS addresses, the element, signed weights) is formed
  // again where it is used and not held in registers through the law
  const int tid = opaque(threadIdx.x);
  // element, and the lane's Gauss point (its sign bits) and corner
  const int le = tid >> 3, lb = XCH ? lane_bits(tid & 7) : tid & 7;
  const int corner = XCH ? hex_node(lb) : tid & 7;
  // lanes beyond the range repeat the last element: they load and compute as
  // the others do and only their stores and counts are left out
  const int i0 = A.e_begin + blk * EPB;
  const bool valid = i0 + le < A.e_end;
  const int lel = min(le, A.e_end - 1 - i0);
  const int e = (!GATHER && A.elem_list) ? A.elem_list[i0 + lel] : i0 + lel;
  // entry k (Gauss point or corner) of the lane's element: the tile's first
  // one, the same for all lanes, plus a 32-bit offset where the elements
  // follow each other
  auto at = [&](auto* ptr, int k) {
    if constexpr (GATHER) return ptr + (int64_t)i0 * 8 + (unsigned)(lel * 8 + k);
    else return ptr + ((int64_t)e * 8 + k);
  };
  if constexpr (SUR == 1) {
    // prepass: a workgroup without a candidate element only marks its
    // points as not listed (workgroup-uniform, before any barrier)
    if (A.sur_cand && !__syncthreads_or(valid && A.sur_cand[e])) {
      if (valid) *at(A.sur_status, lb) = 0;
      continue;
    }
  }

  // -- phase 1: the lane's node.  All of the tile's loads are issued here, in
  // the order of their use: the indices (connectivity, material, corner slot),
  // the nodal values, one material constant per lane (the element's 8
  // constants and 2 moduli go through LDS) and the point's history, so that a
  // wave waits for memory twice and not at every use.
  const int node = *at(A.lnods, corner);
  const int mat = A.mat_of_elem ? A.mat_of_elem[e] : 0;
  int slot = 0;
  if constexpr (GATHER) slot = *at(A.corner_slot, corner);
  double xa[NC];
#pragma unroll
  for (int c = 0; c < 3; ++c) xa[c] = A.coord[c][node];
#pragma unroll
  for (int c = 0; c < 3; ++c) xa[3 + c] = A.u[c][node];
  if constexpr (DAMP) {
#pragma unroll
    for (int c = 0; c < 3; ++c) xa[6 + c] = A.vel[c][node];
  }
  const bool neo = LAWS == 2 || (LAWS == 0 && A.law_of_elem && A.law_of_elem[e]);
  // constant l of the element's material, and its bulk (even l) or shear modulus
  const int l8 = tid & 7;
  const double c8 = LAWS == 2 ? A.props[18 * (int64_t)mat + (l8 & 1)] : A.law_const[8 * (int64_t)mat + l8];
  double c2 = 0.0;
  if constexpr (LAWS != 2) c2 = A.kg[2 * (int64_t)e + (l8 & 1)];
  // a neo-Hookean element has no history: its values stay as they are in
  // both slots (equal from creation and every set), so they are neither
  // read nor written
  double xS0 = 0.0, FAS0 = 0.0, FSA0 = 0.0;
  if (!neo) {
    xS0 = *at(A.sdv_n[0], lb);
    FAS0 = *at(A.sdv_n[1], lb);
    FSA0 = ONE_F ? FAS0 : *at(A.sdv_n[2], lb);
  }
  // nodal values relative to the element's first node (formed in FP64), so that
  // coordinates far from the origin lose no more digits than one subtraction
  R xr[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) xr[c] = (R)(c < 6 || !XCH ? minus_first(xa[c]) : xa[c]);
  if constexpr (!XCH) {
#pragma unroll
    for (int c = 0; c < NC; ++c) s_q(le)[c][corner] = xr[c];
    if constexpr (DAMP)
      if (lb == 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) s_v0[le][c] = xa[6 + c];
      }
    wave_sync();
    // lane c: V(h) of component c
    const int t1 = opaque(tid), l1 = t1 >> 3;
    for (int c = t1 & 7; c < NC; c += 8) {
      R v[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) v[b] = s_q(l1)[c][hex_node(b)];
      wht_stage(v, 4);
      wht_stage(v, 2);
      wht_stage(v, 1);
#pragma unroll
      for (int h = 0; h < 8; ++h) s_v(l1)[h][c] = v[h];
    }
  }
  {
    const int t1 = opaque(tid), l1 = t1 >> 3, c = t1 & 7;
    if (LAWS != 2 || c < 2) s_c(l1)[c] = c8;
    if (LAWS != 2 && c < 2) s_c(l1)[8 + c] = c2;
  }
  wave_sync();

  // -- phase 2: the Gauss point of the lane's sign bits
  uint32_t fl = 0;
  R Q[9], rF, detJ;
  R qd[DAMP ? 3 : 1], zd[DAMP ? 3 : 1];   // damping terms at the point
  {
    const int t2 = opaque(tid), le = t2 >> 3;
    R H[9], detF;
    R jr[9];    // XCH: the rows of j; else j^-1
    if constexpr (XCH) {
      // J^-1, then row by row G_u, H = F - I = G_u J^-1 and the current
      // Jacobian j = J + G_u = F J (J, G_u and j without HEX_SC and the column
      // signs).  FP64: the rows of j go to LDS until the force needs their
      // cofactors (Q = detJ tau j^-T = tau cof(j) / det F),
      // so that neither they nor an inverse of F or j live through the law.
      {
        R J[9], Ji[9];  // col-major: J(i,k) = J[i + 3k]
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          R r3[3];
          hex_grad(xr[i], r3);
#pragma unroll
          for (int k = 0; k < 3; ++k) J[i + 3 * k] = r3[k];
        }
        detJ = sma::inv3<R>(J, Ji);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          R gu[3];
          hex_grad(xr[3 + i], gu);
#pragma unroll
          for (int j = 0; j < 3; ++j)
            H[i + 3 * j] = gu[0] * Ji[3 * j] + gu[1] * Ji[1 + 3 * j] + gu[2] * Ji[2 + 3 * j];
          if constexpr (SUR != 1) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              if constexpr (JLDS) s_row(le)[i + 3 * k][t2 & 7] = J[i + 3 * k] + gu[k];
              else jr[i + 3 * k] = J[i + 3 * k] + gu[k];
            }
          }
        }
      }
      {
        R Fm1[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) Fm1[q] = H[q] + ((q % 4 == 0) ? R(1) : R(0));
        detF = sma::det3<R>(Fm1);
      }
    } else {
      const int gk = t2 & 7;
      // signed weights of the lane's GP: c s_gm / 8 and c^2 s_gm s_gn / 8;
      // row i of J (i < 3) or of G_u (i = 3..5) at the GP, column k
      auto grad_row = [&](int i, R (&out)[3]) {
        const R c1 = (R)(0.125 * HEX_GPOS), c2 = (R)(0.125 * HEX_GPOS * HEX_GPOS);
        const R k0 = (R)0.125;
        const R ax = sign_if(c1, ((gk >> 2) & 1) ^ 1), ay = sign_if(c1, ((gk >> 1) & 1) ^ 1),
                az = sign_if(c1, (gk & 1) ^ 1);
        const R byz = sign_if(c2, ((gk >> 1) ^ gk) & 1);
        const R bxz = sign_if(c2, ((gk >> 2) ^ gk) & 1);
        const R bxy = sign_if(c2, ((gk >> 2) ^ (gk >> 1)) & 1);
        const R* V7 = s_v(le)[7];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int hk = 4 >> k, h1 = k == 0 ? 2 : 4, h2 = k == 2 ? 2 : 1;
          const R w1 = k == 0 ? ay : ax, w2 = k == 2 ? ay : az, w3 = k == 0 ? byz : k == 1 ? bxz : bxy;
          out[k] = k0 * s_v(le)[hk][i] + w1 * s_v(le)[hk | h1][i] + w2 * s_v(le)[hk | h2][i] +
                   w3 * V7[i];
        }
      };
      // J^-1 first (J is then dead), H = F - I = G_u J^-1 (G_u row by row)
      R Ji[9];
      {
        R J[9];  // col-major: J(i,k) = J[i + 3k]
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          R r3[3];
          grad_row(i, r3);
#pragma unroll
          for (int k = 0; k < 3; ++k) J[i + 3 * k] = r3[k];
        }
        detJ = sma::inv3<R>(J, Ji);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        R gu[3];
        grad_row(3 + i, gu);
#pragma unroll
        for (int j = 0; j < 3; ++j)
          H[i + 3 * j] = gu[0] * Ji[3 * j] + gu[1] * Ji[1 + 3 * j] + gu[2] * Ji[2 + 3 * j];
      }
      // current Jacobian j = J + G_u = F J: j^-1 = J^-1 F^-1 and det j =
      // det J det F, formed before the constitutive update
      {
        R Fm1[9], Fi[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) Fm1[q] = H[q] + ((q % 4 == 0) ? R(1) : R(0));
        detF = sma::inv3<R>(Fm1, Fi);
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
          for (int c = 0; c < 3; ++c)
            jr[r + 3 * c] = Ji[r] * Fi[3 * c] + Ji[r + 3] * Fi[1 + 3 * c] + Ji[r + 6] * Fi[2 + 3 * c];
      }
    }

    // det F > 0 (false for NaN); det F <= 0 stops the run (NaN is left to
    // the residual check)
    const bool detf_pos = detF > R(0);
    if constexpr (SUR != 1) {
      if (detF <= R(0)) report_detf(A.health, e, (double)detF);
    }
    const double* pr = A.props + 18 * (int64_t)mat;   // surrogate features, mixed laws
    sma::Mat m{};
    if constexpr (LAWS != 2) m = sma::make_mat_const(s_c(le), s_c(le)[8], s_c(le)[9]);
    if constexpr (ONE_F) m.C_AS = m.C_SA = 0.0;

    R tau[6];
    R Fm[9];
    sma::ReturnMap rm;
    if (neo) {
      // neo-Hookean element: no history, no flags
      R jm1;
      if constexpr (LAWS == 2) sma::neo_hookean_tau<R>(s_c(le)[0], s_c(le)[1], H, tau, jm1);
      else sma::neo_hookean_tau<R>(pr[0], pr[1], H, tau, jm1);
      rm.xS = xS0;
      rm.F_AS = FAS0;
      rm.F_SA = FSA0;
      rm.flags = 0;
#pragma unroll
      for (int q = 0; q < 9; ++q) Fm[q] = H[q] + ((q % 4 == 0) ? R(1) : R(0));
      if constexpr (SUR == 1) {
        if (valid) *at(A.sur_status, lb) = 0;
      }
    } else if constexpr (sizeof(R) == 8) {
      // the Hencky tensor by series (theta, e' and e_n, no eigenvectors;
      // large stretches first halve log b by symmetric square roots)
      const sma::Hencky64 hk = sma::hencky_fp64(H);
      rm = sma::return_map(m, hk.theta, hk.e_n, xS0, FAS0, FSA0);
      sma::kirchhoff_hencky64(m, hk, rm.xS, tau);
      if (!hk.ok) rm.flags |= sma::FLAG_EIGEN_FAIL;
#pragma unroll
      for (int q = 0; q < 9; ++q) Fm[q] = H[q] + ((q % 4 == 0) ? 1.0 : 0.0);
    } else {
      float Hf[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) Hf[q] = H[q];
      // FP32: Hencky strain tensor by series (theta and |e'| are all the
      // return map and the stress need); the spectral form serves stretches
      // beyond the series' range
      sma::Hencky32 hk = sma::hencky_fp32(Hf);
      bool eig_ok = true;
      if (!hk.ok) eig_ok = sma::hencky_spectral_fp32(Hf, hk);
      if constexpr (SUR == 1) {
        const double th = hk.theta, en = hk.e_n;
        bool kf_AS, kf_SA;
        double FAS, FSA;
        const bool flagged = sma::flags_only(m, th, en, xS0, FAS0, FSA0, kf_AS, kf_SA, FAS, FSA);
        // single-branch points whose features lie in the trained range
        // (|f| <= 8) go to the list
        float f[mlp::NIN];
        bool want = false;
        if (valid && flagged && kf_AS != kf_SA) {
          // the features' principal deviatoric strains, in closed form
          float e1, e2, e3;
          sma::principal_dev_fp32(hk.ed, e1, e2, e3);
          const double E = A.E_of_elem ? A.E_of_elem[e] : pr[0];
          mlp::make_features(pr, E, A.T_feat, e1, e2, e3, th, xS0, FAS0, FSA0, FAS, f);
          want = true;
#pragma unroll
          for (int k = 0; k < mlp::NIN; ++k) want = want && fabsf(f[k]) <= 8.0f;
        }
        // one atomic per wave, on the counter of the wave's segment (wave
        // index mod LIST_SEGS; the wave covers elements 8 w .. 8 w + 7 of
        // the launch)
        const unsigned long long wm = __ballot(want);
        const int lane = threadIdx.x & 63;
        const int leader = wm ? __ffsll((long long)wm) - 1 : 0;
        const int seg = ((A.e_begin + blk * EPB) / 8 + (tid >> 6)) % mlp::LIST_SEGS;
        unsigned base = 0;
        if (wm && lane == leader)
          base = atomicAdd(A.sur_count + seg * mlp::LIST_STRIDE, (unsigned)__popcll(wm));
        base = __shfl(base, leader);
        if (want) {
          const int64_t slot = (int64_t)seg * A.sur_seg_cap + base +
                               (unsigned)__popcll(wm & ((1ull << lane) - 1ull));
          float4* dst = reinterpret_cast<float4*>(A.sur_feat + slot * mlp::NIN);
#pragma unroll
          for (int k = 0; k < mlp::NIN / 4; ++k)
            dst[k] = make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
          *at(A.sur_slot, lb) = (int32_t)slot;
        }
        if (valid) *at(A.sur_status, lb) = !flagged ? 0 : want ? 1 : 2;
      } else {
        if constexpr (SUR == 2) {
          rm = surrogate_or_exact(A, m, (int64_t)e * 8 + lb, hk.theta, hk.e_n, xS0, FAS0, FSA0);
        } else {
          rm = sma::return_map(m, hk.theta, hk.e_n, xS0, FAS0, FSA0);
        }
        sma::kirchhoff_dev(m, hk, rm.xS, tau);
        if (!eig_ok) rm.flags |= sma::FLAG_EIGEN_FAIL;
      }
#pragma unroll
      for (int q = 0; q < 9; ++q) Fm[q] = H[q] + ((q % 4 == 0) ? R(1) : R(0));
    }
    if constexpr (SUR != 1) {
    if (!neo && valid) {
      *at(A.sdv_k[0], lb) = rm.xS;
      *at(A.sdv_k[1], lb) = rm.F_AS;
      if constexpr (!ONE_F) *at(A.sdv_k[2], lb) = rm.F_SA;
    }
    fl = rm.flags;
    if (!detf_pos) fl |= sma::FLAG_DETF_NONPOS;

    const int neg = (__popc(lb) & 1) ^ 1;   // the product of the lane's signs is -1
    R jq[9];
    if constexpr (XCH) {
      // Q = tau cof(j) / det F, with the constants of HEX_SC; column k keeps the
      // factor s_gk
      {
        rF = sma::rcp_r(detF);
        if constexpr (JLDS) {
          const int t3 = opaque(tid);
#pragma unroll
          for (int q = 0; q < 9; ++q) jr[q] = s_row(t3 >> 3)[q][t3 & 7];
        }
        sma::cof3<R>(jr, jq);
        const R sF = rF * sign_if((R)(HEX_SC * HEX_SC * HEX_SC), neg);
        const R T[6] = {tau[0] * sF, tau[1] * sF, tau[2] * sF, tau[3] * sF, tau[4] * sF, tau[5] * sF};
        const R Tf[9] = {T[0], T[1], T[2], T[1], T[3], T[4], T[2], T[4], T[5]};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int k = 0; k < 3; ++k)
            Q[3 * i + k] = Tf[i] * jq[3 * k] + Tf[i + 3] * jq[1 + 3 * k] + Tf[i + 6] * jq[2 + 3 * k];
      }
    } else {
      // Q = detJ tau j^-T
      const R T[9] = {tau[0], tau[1], tau[2], tau[1], tau[3], tau[4], tau[2], tau[4], tau[5]};
      const int t3 = opaque(tid), l3 = t3 >> 3, g = t3 & 7;
#pragma unroll
      for (int q = 0; q < 9; ++q) jq[q] = jr[q];
      wave_sync();
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k)
          s_q(l3)[3 * i + k][g] =
              detJ * (T[i] * jq[k] + T[i + 3] * jq[k + 3] + T[i + 6] * jq[k + 6]);
    }

    if constexpr (DAMP && XCH) {
      // Rayleigh damping at the Gauss point: q = alpha rho detJ gpvel, the
      // velocity interpolated there (sld_elmpre.f90:110-114), and z
      const double alpha = A.damping[2 * mat], beta = A.damping[2 * mat + 1];
      const R arho = (R)(alpha * A.rho[mat]);
      const R dJ = detJ * sign_if((R)(HEX_SC * HEX_SC * HEX_SC), neg);   // det J
      constexpr double cp3 = HEX_CP * HEX_CP * HEX_CP;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const R gv = (R)cp3 * interp<0>(interp<1>(interp<2>(xr[6 + i])));
        qd[i] = (R)cp3 * arho * dJ * gv;
        zd[i] = R(0);
      }
      if (__ballot(beta > 0.0) != 0ull) {
        // the beta term as written (sld_elmmat.f90:174-194):
        // z_k = beta detJ sum_j J^-1_kj w_j, w_j = sum_k L_kj S_jk with the
        // velocity gradient L = G_v J^-1 (gprat, sld_elmpre.f90:150-157); the
        // exchanges of hex_grad need every lane of the element
        R Jd[9], Gv[9];   // without HEX_SC and the column signs
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          R a3[3], b3[3];
          hex_grad(xr[i], a3);
          hex_grad(xr[6 + i], b3);
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            Jd[i + 3 * k] = a3[k];
            Gv[i + 3 * k] = b3[k];
          }
        }
        R Jid[9];
        sma::inv3<R>(Jd, Jid);
        R L[9], Fi[9], S[9];
        const R rj = rF * sma::rcp_r(detJ);   // 1 / det j
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            L[r + 3 * c] = Gv[r] * Jid[3 * c] + Gv[r + 3] * Jid[1 + 3 * c] + Gv[r + 6] * Jid[2 + 3 * c];
            // F^-1 = J j^-1 (j = F J), j^-1 = cof(j)^T / det j
            Fi[r + 3 * c] = rj * (Jd[r] * jq[c] + Jd[r + 3] * jq[c + 3] + Jd[r + 6] * jq[c + 6]);
          }
        sma::pk2<R>(Fi, tau, S);
        R w[3];
#pragma unroll
        for (int j = 0; j < 3; ++j)
          w[j] = L[3 * j] * S[j] + L[1 + 3 * j] * S[j + 3] + L[2 + 3 * j] * S[j + 6];
        // z_k s_gk HEX_SC: row k of Jid is that of J^-1 times HEX_SC s_gk
        const R bd = (R)beta * dJ;
#pragma unroll
        for (int k = 0; k < 3; ++k)
          zd[k] = bd * (Jid[k] * w[0] + Jid[k + 3] * w[1] + Jid[k + 6] * w[2]);
      }
    }
    if constexpr (DAMP && !XCH) {
      // Rayleigh damping at Gauss point g.  J and the velocity's natural
      // derivatives are formed again from the V(h) rows (they are not kept
      // through the constitutive update); the velocity interpolated at g is
      // gpvel = v_0 + 1/8 sum_h c^|h| s_g(h) V_v(h) (sld_elmpre.f90:110-114)
      const int gd = opaque(tid) & 7, g = gd;
      const R c1 = (R)(0.125 * HEX_GPOS), c2 = (R)(0.125 * HEX_GPOS * HEX_GPOS);
      const R c3 = (R)(0.125 * HEX_GPOS * HEX_GPOS * HEX_GPOS), k0 = (R)0.125;
      const R ax = sign_if(c1, ((gd >> 2) & 1) ^ 1), ay = sign_if(c1, ((gd >> 1) & 1) ^ 1),
              az = sign_if(c1, (gd & 1) ^ 1);
      const R byz = sign_if(c2, ((gd >> 1) ^ gd) & 1);
      const R bxz = sign_if(c2, ((gd >> 2) ^ gd) & 1);
      const R bxy = sign_if(c2, ((gd >> 2) ^ (gd >> 1)) & 1);
      const R bxyz = sign_if(c3, (((gd >> 2) ^ (gd >> 1) ^ gd) & 1) ^ 1);
      // weights of V(h): h = 0, z, y, yz, x, xz, xy, xyz (bits x = 4, y = 2, z = 1)
      const R wv[8] = {k0, az, ay, byz, ax, bxz, bxy, bxyz};
      const double alpha = A.damping[2 * mat], beta = A.damping[2 * mat + 1];
      const R arho = (R)(alpha * A.rho[mat]);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        R gv = R(0);
#pragma unroll
        for (int h = 0; h < 8; ++h) gv += wv[h] * s_v(le)[h][6 + i];
        gv += (R)s_v0[le][i];
        s_q(le)[9 + i][g] = arho * detJ * gv;
      }
      R z[3] = {R(0), R(0), R(0)};
      if (beta > 0.0) {
        // the beta term as written (sld_elmmat.f90:174-194):
        // z_k = beta detJ sum_j J^-1_kj w_j, w_j = sum_k L_kj S_jk with the
        // velocity gradient L = G_v J^-1 (gprat, sld_elmpre.f90:150-157)
        R Jd[9], Gv[9];
        const R* V7 = s_v(le)[7];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int hk = 4 >> k, h1 = k == 0 ? 2 : 4, h2 = k == 2 ? 2 : 1;
          const R w1 = k == 0 ? ay : ax, w2 = k == 2 ? ay : az, w3 = k == 0 ? byz : k == 1 ? bxz : bxy;
          const R* Vk = s_v(le)[hk];
          const R* V1 = s_v(le)[hk | h1];
          const R* V2 = s_v(le)[hk | h2];
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            Jd[i + 3 * k] = k0 * Vk[i] + w1 * V1[i] + w2 * V2[i] + w3 * V7[i];
            Gv[i + 3 * k] = k0 * Vk[6 + i] + w1 * V1[6 + i] + w2 * V2[6 + i] + w3 * V7[6 + i];
          }
        }
        R Jid[9];
        sma::inv3<R>(Jd, Jid);
        R L[9], Fi[9], S[9];
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            L[r + 3 * c] = Gv[r] * Jid[3 * c] + Gv[r + 3] * Jid[1 + 3 * c] + Gv[r + 6] * Jid[2 + 3 * c];
            // F^-1 = J j^-1 (j = F J)
            Fi[r + 3 * c] = Jd[r] * jq[3 * c] + Jd[r + 3] * jq[1 + 3 * c] + Jd[r + 6] * jq[2 + 3 * c];
          }
        sma::pk2<R>(Fi, tau, S);
        R w[3];
#pragma unroll
        for (int j = 0; j < 3; ++j)
          w[j] = L[3 * j] * S[j] + L[1 + 3 * j] * S[j + 3] + L[2 + 3 * j] * S[j + 6];
        const R bd = (R)beta * detJ;
#pragma unroll
        for (int k = 0; k < 3; ++k)
          z[k] = bd * (Jid[k] * w[0] + Jid[k + 3] * w[1] + Jid[k + 6] * w[2]);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) s_q(le)[12 + k][g] = z[k];
    }

    if constexpr (STORE) {
      R Fi[9], S[9];
      sma::inv3<R, true>(Fm, Fi);
      sma::pk2<R>(Fi, tau, S);
      const int64_t ngp = A.nelem * 8, gp = (int64_t)e * 8 + lb;
      if (valid) {
#pragma unroll
      for (int q = 0; q < 9; ++q) A.S_out[q * ngp + gp] = (double)S[q];
      // P_jk = sum_i F_ji S_ik (sld_builtin_materials.f90:355-371), column-major
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int j = 0; j < 3; ++j)
          A.P_out[(j + 3 * k) * ngp + gp] =
              (double)(Fm[j] * S[3 * k] + Fm[j + 3] * S[1 + 3 * k] + Fm[j + 6] * S[2 + 3 * k]);
      A.flags_out[gp] = fl;
      }
    }
    }  // SUR != 1
  }
  if constexpr (SUR == 1) continue;   // uniform: the prepass has no scatter
  count_flags(A.counters, fl, valid);
  if constexpr (SUR == 2) {
    // the next step's candidates: elements with a transforming point now
    if (A.sur_cand_next) {
      const unsigned long long tm = __ballot(valid && (fl & 3u));
      if (valid && lb == 0) A.sur_cand_next[e] = ((tm >> (8 * (le & 7))) & 0xffull) != 0ull;
    }
  }


  // Walsh-Hadamard sums: lane j forms U of Q(j) (Q(8) in phase 3, by every
  // lane); with damping lanes 0-2 also form U of z_0..2 and lanes 3-5 the
  // Walsh-Hadamard coefficients of q_0..2
  if constexpr (!XCH) {
    const int t4 = opaque(tid), le = t4 >> 3, j = t4 & 7;
    wave_sync();
    u4_of_q(s_q(le)[j], j % 3, s_u4(le)[j]);
    if constexpr (DAMP) {
      if (j < 3) {
        u4_of_q(s_q(le)[12 + j], j, s_u4(le)[8 + j]);
      } else if (j < 6) {
        R v[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) v[b] = s_q(le)[9 + j - 3][b];
        wht_stage(v, 4);
        wht_stage(v, 2);
        wht_stage(v, 1);
#pragma unroll
        for (int h = 0; h < 8; ++h) s_wq(le)[j - 3][h] = v[h];
      }
    }
  }

  // -- phase 3: the lane's corner, f_a = sum_g sum_k Q_k(g) dN_a/dxi_k(g)
  {
    R f[3];
    R fd[DAMP ? 3 : 1];
    if constexpr (XCH) {
#pragma unroll
      for (int i = 0; i < 3; ++i) f[i] = hex_grad_t(Q[3 * i], Q[3 * i + 1], Q[3 * i + 2]);
      if constexpr (DAMP) {
        // damping force of the corner: alpha sum_g N_a(g) q(g) less the beta
        // sum sum_g sum_k dN_a/dxi_k z_k (one value for the three components)
        const R cb = hex_grad_t(zd[0], zd[1], zd[2]);
#pragma unroll
        for (int i = 0; i < 3; ++i) fd[i] = interp<0>(interp<1>(interp<2>(qd[i]))) - cb;
      }
    } else {
      // f_ai = sum_k s_ak/8 [U0 + c s_a1 U1 + c s_a2 U2 + c^2 s_a1 s_a2 U12](3i+k)
      wave_sync();
      const int t5 = opaque(tid), le = t5 >> 3, a = t5 & 7;
      const int sx = (0x66 >> a) & 1, sy = (0xCC >> a) & 1, sz = (0xF0 >> a) & 1;
      const R c0 = (R)0.125, c1 = (R)(0.125 * HEX_GPOS), c2 = (R)(0.125 * HEX_GPOS * HEX_GPOS);
      R u8[4];
      u4_of_q(s_q(le)[8], 2, u8);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int sk = k == 0 ? sx : k == 1 ? sy : sz;
        const int s1 = k == 0 ? sy : sx, s2 = k == 2 ? sy : sz;
        // signs s_ak, s_ak s_a1, s_ak s_a2, s_ak s_a1 s_a2 as bit parities
        const R l0 = sign_if(c0, sk ^ 1);
        const R l1 = sign_if(c1, sk ^ s1);
        const R l2 = sign_if(c1, sk ^ s2);
        const R l3 = sign_if(c2, (sk ^ s1 ^ s2) ^ 1);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const R* u = (3 * i + k == 8) ? u8 : s_u4(le)[3 * i + k];
          const R term = l0 * u[0] + l1 * u[1] + l2 * u[2] + l3 * u[3];
          f[i] = k == 0 ? term : f[i] + term;
        }
      }
      if constexpr (DAMP) {
        // damping force of corner a: alpha sum_g N_a(g) q(g) =
        // 1/8 sum_h c^|h| s_a(h) Q_q(h), less the beta sum
        // sum_g sum_k dN_a/dxi_k z_k (one value for the three components)
        R cb = R(0);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int sk = k == 0 ? sx : k == 1 ? sy : sz;
          const int s1 = k == 0 ? sy : sx, s2 = k == 2 ? sy : sz;
          const R l0 = sign_if(c0, sk ^ 1);
          const R l1 = sign_if(c1, sk ^ s1);
          const R l2 = sign_if(c1, sk ^ s2);
          const R l3 = sign_if(c2, (sk ^ s1 ^ s2) ^ 1);
          const R* u = s_u4(le)[8 + k];
          cb += l0 * u[0] + l1 * u[1] + l2 * u[2] + l3 * u[3];
        }
        const R c3 = (R)(0.125 * HEX_GPOS * HEX_GPOS * HEX_GPOS);
        const R px = sign_if(c1, sx ^ 1), py = sign_if(c1, sy ^ 1), pz = sign_if(c1, sz ^ 1);
        const R pyz = sign_if(c2, sy ^ sz), pxz = sign_if(c2, sx ^ sz), pxy = sign_if(c2, sx ^ sy);
        const R pxyz = sign_if(c3, (sx ^ sy ^ sz) ^ 1);
        const R wa[8] = {c0, pz, py, pyz, px, pxz, pxy, pxyz};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          R r = R(0);
#pragma unroll
          for (int h = 0; h < 8; ++h) r += wa[h] * s_wq(le)[i][h];
          fd[i] = r - cb;
        }
      }
    }
    if constexpr (DAMP) {
      R* ed = (R*)A.edamp + 3 * (int64_t)slot;
      if (valid) {
        ed[0] = fd[0];
        ed[1] = fd[1];
        ed[2] = fd[2];
      }
    }
    if constexpr (GATHER) {
      R* ef = (R*)A.efor + 3 * (int64_t)slot;
      if (valid) {
        ef[0] = f[0];
        ef[1] = f[1];
        ef[2] = f[2];
      }
    } else if (valid) {
      // coloured scatter: no other element of this colour touches this node
      R* fx = (R*)A.fint[0];
      R* fy = (R*)A.fint[1];
      R* fz = (R*)A.fint[2];
      fx[node] += f[0];
      fy[node] += f[1];
      fz[node] += f[2];
    }
  }
  wave_sync();   // the next tile's gather writes the LDS rows phase 3 has just read
  }  // tile loop
}

// ----------------------------------------------------------------------------
// Setup: lumped mass (sld_elmmat.f90:199-209), one thread per element, per colour.
// ----------------------------------------------------------------------------
struct MassArgs {
  int32_t e_begin, e_end;       // colour range in elem_list
  const int32_t* elem_list;
  const int32_t* lnods;
  const double* coord[3];
  const double* rho;
  const int32_t* mat_of_elem;
  double* mass;
};

__global__ void sld_mass(MassArgs A) {
#pragma clang fp contract(off)
  const int i_el = A.e_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (i_el >= A.e_end) return;
  const int e = A.elem_list[i_el];
  double x[8][3];
  int nodes[8];
  for (int a = 0; a < 8; ++a) {
    nodes[a] = A.lnods[(int64_t)e * 8 + a];
    for (int d = 0; d < 3; ++d) x[a][d] = A.coord[d][nodes[a]];
  }
  const double rho = A.rho[A.mat_of_elem ? A.mat_of_elem[e] : 0];
  double elmuu[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int g = 0; g < 8; ++g) {
    double J[9] = {0};
    for (int a = 0; a < 8; ++a)
      for (int k = 0; k < 3; ++k) {
        double D = hex_deriv<double>(a, g, k);
        for (int i = 0; i < 3; ++i) J[i + 3 * k] = J[i + 3 * k] + x[a][i] * D;
      }
    // jacobi.f90 ndime==3 determinant by first-row cofactors
    double t1 = J[4] * J[8] - J[5] * J[7];
    double t2 = -J[1] * J[8] + J[2] * J[7];
    double t3 = J[1] * J[5] - J[2] * J[4];
    double vol = 1.0 * (J[0] * t1 + J[3] * t2 + J[6] * t3);
    for (int a = 0; a < 8; ++a)
      for (int b = 0; b < 8; ++b)
        elmuu[a] = elmuu[a] + rho * vol * hex_shape<double>(a, g) * hex_shape<double>(b, g);
  }
  for (int a = 0; a < 8; ++a) A.mass[nodes[a]] += elmuu[a];
}

// Setup: bulk and shear modulus per element (the expressions of make_mat).
__global__ void sld_elem_moduli(int64_t ne, const double* __restrict__ props,
                                const int32_t* __restrict__ mat_of_elem,
                                const double* __restrict__ E_of_elem, double* __restrict__ kg) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  const double* pr = props + 18 * (mat_of_elem ? mat_of_elem[e] : 0);
  sma::elastic_moduli(pr, E_of_elem ? E_of_elem[e] : pr[0], kg[2 * e], kg[2 * e + 1]);
}

__global__ void sld_reciprocal(const double* __restrict__ m, double* __restrict__ rm, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) rm[i] = 1.0 / m[i];
}

// ----------------------------------------------------------------------------
// Read-back: components of a field (one array each) interleaved by rows, with
// the caller's element order, as the host wants them.  One value a thread, so
// a wave writes 512 consecutive bytes; the output is pinned host memory, whose
// link (55 GB/s) is the bound.
// ----------------------------------------------------------------------------
struct PackArgs {
  const void* src[9];
  int32_t fp32;                 // the sources are float
  const int32_t* stored;        // rows are Gauss points: stored position of each element, or null
  int64_t row0, same;           // component 2 of stored rows below `same` is component 1
  int32_t rows;
  double* out;                  // [rows][NC]
};

template <int NC>
__global__ void __launch_bounds__(256) sld_pack(PackArgs A) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= A.rows * NC) return;
  const int r = j / NC;
  int k = j - r * NC;
  int64_t i = A.row0 + r;
  if (A.stored) i = 8 * (int64_t)A.stored[i >> 3] + (i & 7);
  if (NC == 3 && k == 2 && i < A.same) k = 1;
  A.out[j] = A.fp32 ? (double)((const float*)A.src[k])[i] : ((const double*)A.src[k])[i];
}

// ----------------------------------------------------------------------------
// Point-wise law (drop-in for eval_sld_stress_model_160 with flagt = 0).
// Bound by memory: 212 bytes a point (F, S, history, E, material, flags).  The
// stresses, a third of it, are stored past the caches: nothing here reads them
// again, and the inputs of a call, or what its caller just wrote, stay in.
// 1.28 million points, 256 materials: 125 us with the spectral form at every
// point, 54 with the series strain, 41 with the streaming stores (the inputs
// then fit the 256 MB cache; loads past the caches: 59).  Five sets of inputs in
// turn, plain -> streaming stores: 300 000 points 18.9 -> 12.8 us, 640 000 33.5 ->
// 32.8, 1.28 million 61.4 -> 60.3; with a kernel after each that reads S back, which
// it then has to fetch from memory, 26.8 -> 28.4, 47.8 -> 50.7 and 94.5 -> 96.4.
// ----------------------------------------------------------------------------
struct LawArgs {
  int64_t n;
  int32_t nmat;
  const double* props;
  const int32_t* mat_of_gp;
  const double* E_of_gp;
  const double* F;        // [9][n]
  const double* sdv_old;  // [3][n]
  double* sdv_new;        // [3][n]
  double* S;              // [9][n]
  uint32_t* flags;        // [n] or null
};

template <bool FP32_KIN>
__global__ void __launch_bounds__(256) sma160_points(LawArgs A) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n) return;
  int mat = A.mat_of_gp ? A.mat_of_gp[i] : 0;
  uint32_t bad = 0;
  if (mat < 0 || mat >= A.nmat) {  // device arrays cannot be checked on the host
    bad = sma::FLAG_BAD_INPUT;
    mat = 0;
  }
  const double* pr = A.props + 18 * mat;
  const double E = A.E_of_gp ? A.E_of_gp[i] : pr[0];
  const sma::Mat m = sma::make_mat(pr, E);
  double F[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) F[q] = A.F[q * A.n + i];
  const double xS0 = A.sdv_old[i], FAS0 = A.sdv_old[A.n + i], FSA0 = A.sdv_old[2 * A.n + i];
  sma::ReturnMap rm;
  double S[9];
  if constexpr (!FP32_KIN) {
    double tau[6], Fi[9];
    rm = sma::law_point(m, F, xS0, FAS0, FSA0, tau);
    double det = sma::inv3<double, true>(F, Fi);
    if (!(det > 0.0)) rm.flags |= sma::FLAG_DETF_NONPOS;
    sma::pk2<double>(Fi, tau, S);
  } else {
    float H[9], Ff[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      H[q] = (float)(F[q] - ((q % 4 == 0) ? 1.0 : 0.0));
      Ff[q] = (float)F[q];
    }
    sma::Spectral<float> sp = sma::spectral_fp32(H);
    rm = sma::return_map(m, sp.theta, sp.e_n, xS0, FAS0, FSA0);
    if (!sp.eig_ok) rm.flags |= sma::FLAG_EIGEN_FAIL;
    float tau[6], Fi[9], Sf[9];
    sma::kirchhoff<float>(m, sp, rm.xS, tau);
    float det = sma::inv3<float>(Ff, Fi);
    if (!(det > 0.f)) rm.flags |= sma::FLAG_DETF_NONPOS;
    sma::pk2<float>(Fi, tau, Sf);
#pragma unroll
    for (int q = 0; q < 9; ++q) S[q] = Sf[q];
  }
  A.sdv_new[i] = rm.xS;
  A.sdv_new[A.n + i] = rm.F_AS;
  A.sdv_new[2 * A.n + i] = rm.F_SA;
#pragma unroll
  for (int q = 0; q < 9; ++q) __builtin_nontemporal_store(S[q], A.S + q * A.n + i);
  if (A.flags) A.flags[i] = rm.flags | bad;
}

}  // namespace sld
