// Device-side building blocks of the WENO5 flux divergence fe() for CDNA4 (gfx950), FP64.
//
// Data layout in HBM (the reference's ManyVector layout, euler3D.hpp:62-65):
//   fluid fields rho, mx, my, mz, et: 5 separate arrays, cell index i + nx*(j + ny*k);
//   advected species: one AoS array, species fastest: v + nchem*(i + nx*(j + ny*k)).
//
// Two face-flux implementations live here:
//   face_flux_ref  - the reference recipe (utilities.cpp:270-479) operation by operation,
//                    with FMA contraction disabled; used by the plain comparator kernels
//                    and reproducible bit for bit against a non-FMA CPU build.
//   face_flux_lds  - the same mathematics rearranged for the FP64 pipes: primitive values
//                    computed once per point (staged in LDS), the characteristic projection
//                    taken relative to the Roe velocity, the smoothness indicators as
//                    completed squares, the WENO weights over one common denominator and
//                    one reciprocal per component for both split sides.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace mvd {

constexpr int BC_PERIODIC = 0, BC_NEUMANN = 1, BC_DIRICHLET = 2, BC_REFLECTING = 3;
constexpr int NCHEM_MAX = 16;
constexpr int NV_MAX = 5 + NCHEM_MAX;

// Grid and boundary description passed by value to every fe() kernel.
struct Grid {
  int nx, ny, nz, nchem;
  int bc[6];               // xl, xr, yl, yr, zl, zr
  double gamma, dx, dy, dz;
  double igm;              // 1 / (gamma - 1)
};

__host__ __device__ inline int extent(const Grid &g, int d) {
  return d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
}

// Source position and sign of extended index e (ghost layer 3 deep) along direction d.
// Physical boundaries follow the reference's ghost fill (euler3D.hpp:793-1166):
// low faces mirror (e -> -1-e), high faces copy shifted (e -> e-3); periodic wraps.
// sgn_all = -1 for Dirichlet (all fields negated); sgn_norm = -1 for the normal momentum
// under reflecting (and Dirichlet) boundaries.
struct GhostMap {
  int src;
  double sgn_all, sgn_norm;
};

__device__ inline GhostMap ghost_map(const Grid &g, int d, int e) {
  const int n = extent(g, d);
  GhostMap m{e, 1.0, 1.0};
  if (e < 0 || e >= n) {
    const bool lo = e < 0;
    const int bc = g.bc[2 * d + (lo ? 0 : 1)];
    if (bc == BC_PERIODIC) {
      m.src = lo ? e + n : e - n;
    } else {
      m.src = lo ? -1 - e : e - 3;
      if (bc == BC_DIRICHLET) { m.sgn_all = -1.0; m.sgn_norm = -1.0; }
      else if (bc == BC_REFLECTING) { m.sgn_norm = -1.0; }
    }
  }
  return m;
}

// SUNRsqrt (sundials_math.h): non-positive arguments give 0.
__device__ inline double sun_sqrt(double x) { return (x <= 0.0) ? 0.0 : sqrt(x); }

// Reciprocal from the hardware estimate (v_rcp_f64, relative error e of about 2^-24) times
// 1 + e + e^2: the error left is e^3, below rounding, for one FMA less than two Newton
// steps. Within 1 ulp. fast_div refines the estimate once (2^-48) and corrects the quotient
// by its residual, which squares that error again: the correctly rounded quotient but for
// rare ties. Denominators: normal numbers whose reciprocal is normal (0, infinity and
// denormals give NaN where an IEEE divide gives infinity or 0).
__device__ inline double fast_rcp(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

__device__ inline double fast_div(double n, double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  const double q = n * r;
  return fma(fma(-d, q, n), r, q);
}

// sqrt(x) for normal x > 0, 0 for x <= 0 (SUNRsqrt's rule): Goldschmidt's iteration from
// v_rsq_f64 with a residual correction, within 1 ulp in half the library's instructions
// (no scaling of denormals).
__device__ inline double fast_sqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double gq = x * y, h = 0.5 * y;
  const double e = fma(-h, gq, 0.5);
  gq = fma(gq, e, gq);
  h = fma(h, e, h);
  gq = fma(fma(-gq, gq, x), h, gq);
  return x <= 0.0 ? 0.0 : gq;
}

// ---------------------------------------------------------------------------------
// Reference-order face flux (no contraction). s[l][v], l = stencil point, v = field in
// direction-local order (rho, m_normal, m_t1, m_t2, et, species...).
// ---------------------------------------------------------------------------------
template <int NC>
__device__ inline void face_flux_ref(double (&s)[6][5 + NC], double gamma, double *ff_out) {
#pragma clang fp contract(off)
  constexpr int NV = 5 + NC;
  const double bc = 1.083333333333333333333333333333333333333;
  const double eps = 1e-6;
  const double c13 = 0.3333333333333333333333333333333333333333;
  const double c56 = 0.8333333333333333333333333333333333333333;
  const double c16 = 0.1666666666666666666666666666666666666667;
  const double c76 = 1.166666666666666666666666666666666666667;
  const double c116 = 1.833333333333333333333333333333333333333;
  double p[6];
#pragma unroll
  for (int l = 0; l < 6; l++)
    p[l] = (gamma - 1.0) * (s[l][4] - (s[l][1] * s[l][1] + s[l][2] * s[l][2] + s[l][3] * s[l][3]) * 0.5 / s[l][0]);
  const double sL = sun_sqrt(s[2][0]), sR = sun_sqrt(s[3][0]);
  const double sbar = 0.5 * (sL + sR);
  const double u = 0.5 * (s[2][1] / sL + s[3][1] / sR) / sbar;
  const double v = 0.5 * (s[2][2] / sL + s[3][2] / sR) / sbar;
  const double w = 0.5 * (s[2][3] / sL + s[3][3] / sR) / sbar;
  const double H = 0.5 * ((p[2] + s[2][4]) / sL + (p[3] + s[3][4]) / sR) / sbar;
  const double qsq = u * u + v * v + w * w;
  const double gm = gamma - 1.0;
  const double cs = gm * (H - 0.5 * qsq);
  const double ci = 1.0 / cs;
  const double RV[5][5] = {{1.0, 0.0, 0.0, 1.0, 1.0},
                           {u - cs, 0.0, 0.0, u, u + cs},
                           {v, 1.0, 0.0, v, v},
                           {w, 0.0, 1.0, w, w},
                           {H - u * cs, v, w, 0.5 * qsq, H + u * cs}};
  const double LV[5][5] = {
      {0.5 * ci * (u + 0.5 * gm * qsq), -0.5 * ci * (gm * u + 1.0), -0.5 * v * gm * ci,
       -0.5 * w * gm * ci, 0.5 * gm * ci},
      {-v, 0.0, 1.0, 0.0, 0.0},
      {-w, 0.0, 0.0, 1.0, 0.0},
      {(-gm) * ci * (qsq - H), u * gm * ci, v * gm * ci, w * gm * ci, (-gm) * ci},
      {-0.5 * ci * (u - 0.5 * gm * qsq), -0.5 * ci * (gm * u - 1.0), -0.5 * v * gm * ci,
       -0.5 * w * gm * ci, 0.5 * gm * ci}};
  double flux[6][NV];
  double alpha = 0.0;
#pragma unroll
  for (int l = 0; l < 6; l++) {
    const double ul = s[l][1] / s[l][0];
    flux[l][0] = s[l][1];
    flux[l][1] = ul * s[l][1] + p[l];
    flux[l][2] = ul * s[l][2];
    flux[l][3] = ul * s[l][3];
    flux[l][4] = ul * (s[l][4] + p[l]);
#pragma unroll
    for (int c = 0; c < NC; c++) flux[l][5 + c] = ul * s[l][5 + c];
    const double cl = sun_sqrt(gamma * p[l] / s[l][0]);
    const double al = fabs(ul) + cl;
    alpha = (alpha < al) ? al : alpha;
  }
  double ff[NV];
#pragma unroll
  for (int side = 0; side < 2; side++) {
    double fp[5][NV];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      double fs[NV];
#pragma unroll
      for (int c = 0; c < NV; c++)
        fs[c] = side == 0 ? 0.5 * (flux[l][c] + alpha * s[l][c])
                          : 0.5 * (flux[l + 1][c] - alpha * s[l + 1][c]);
#pragma unroll
      for (int a = 0; a < 5; a++)
        fp[l][a] = LV[a][0] * fs[0] + LV[a][1] * fs[1] + LV[a][2] * fs[2] + LV[a][3] * fs[3] + LV[a][4] * fs[4];
#pragma unroll
      for (int c = 0; c < NC; c++) fp[l][5 + c] = fs[5 + c];
    }
#pragma unroll
    for (int c = 0; c < NV; c++) {
      const double f0 = fp[0][c], f1 = fp[1][c], f2 = fp[2][c], f3 = fp[3][c], f4 = fp[4][c];
      const double x1 = f2 - 2.0 * f3 + f4, y1 = 3.0 * f2 - 4.0 * f3 + f4;
      const double x2 = f1 - 2.0 * f2 + f3, y2 = f1 - f3;
      const double x3 = f0 - 2.0 * f1 + f2, y3 = f0 - 4.0 * f1 + 3.0 * f2;
      const double b1 = bc * (x1 * x1) + 0.25 * (y1 * y1);
      const double b2 = bc * (x2 * x2) + 0.25 * (y2 * y2);
      const double b3 = bc * (x3 * x3) + 0.25 * (y3 * y3);
      if (side == 0) {
        const double w1 = 0.3 / ((eps + b1) * (eps + b1));
        const double w2 = 0.6 / ((eps + b2) * (eps + b2));
        const double w3 = 0.1 / ((eps + b3) * (eps + b3));
        const double q1 = c13 * f2 + c56 * f3 - c16 * f4;
        const double q2 = (-c16) * f1 + c56 * f2 + c13 * f3;
        const double q3 = c13 * f0 - c76 * f1 + c116 * f2;
        ff[c] = (q1 * w1 + q2 * w2 + q3 * w3) / (w1 + w2 + w3);
      } else {
        const double w1 = 0.1 / ((eps + b1) * (eps + b1));
        const double w2 = 0.6 / ((eps + b2) * (eps + b2));
        const double w3 = 0.3 / ((eps + b3) * (eps + b3));
        const double q1 = c116 * f2 - c76 * f3 + c13 * f4;
        const double q2 = c13 * f1 + c56 * f2 - c16 * f3;
        const double q3 = (-c16) * f0 + c56 * f1 + c13 * f2;
        ff[c] += (q1 * w1 + q2 * w2 + q3 * w3) / (w1 + w2 + w3);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 5; a++)
    ff_out[a] = RV[a][0] * ff[0] + RV[a][1] * ff[1] + RV[a][2] * ff[2] + RV[a][3] * ff[3] + RV[a][4] * ff[4];
#pragma unroll
  for (int c = 0; c < NC; c++) ff_out[5 + c] = ff[5 + c];
}

// ---------------------------------------------------------------------------------
// Fast face flux.
// ---------------------------------------------------------------------------------

// A stencil point as the face fluxes read it from LDS, field q at base[q * FS]: the
// primitive state, sqrt(rho), c^2 = gamma p / rho (signed) and c.
enum { PT_R = 0, PT_U, PT_V, PT_W, PT_P, PT_SR, PT_C2, PT_C, PT_NF };

// Converts a conserved state; returns p.
__device__ inline double store_point(double *pp, int FS, double r, double mx, double my,
                                     double mz, double e, double gamma) {
  const double ir = fast_rcp(r);
  const double p = (gamma - 1.0) * (e - 0.5 * (mx * mx + my * my + mz * mz) * ir);
  const double c2 = gamma * p * ir;
  pp[PT_R * FS] = r;
  pp[PT_U * FS] = mx * ir;
  pp[PT_V * FS] = my * ir;
  pp[PT_W * FS] = mz * ir;
  pp[PT_P * FS] = p;
  pp[PT_SR * FS] = fast_sqrt(r);
  pp[PT_C2 * FS] = c2;
  pp[PT_C * FS] = fast_sqrt(c2);
  return p;
}

// WENO5-JS over f0..f4 (the f+ formula; the f- one is the same function of the reversed
// values): the reconstruction is f2 + (2/3) S / den. With the differences a, b, c, d of
// neighbouring values the smoothness indicators are completed squares,
//   beta_3 = 4/3 ((a - 11/8 b)^2 + 39/64 b^2), beta_2 = 4/3 ((b - 5/8 c)^2 + 39/64 c^2),
//   beta_1 = 4/3 ((d - 11/8 c)^2 + 39/64 c^2),
// whose second squares are shared; the common factor (4/3)^2 cancels in the weight ratio, so
// eps enters as 3/4 eps. Over the common denominator the weights are d_k times products of
// the other two (eps + beta)^2; den = (10/3) sum of them, and the candidate stencils are
// written relative to f2: c - d/4, c + b/2, 5/12 b - a/6 (times 2/3 and the linear weights'
// ratios 1, 2, 1/3). 29 operations. epsb is 3/4 eps for the values as given; WENO5 is
// homogeneous in the sense WENO(l f; eps) = l WENO(f; eps / l^2), so a caller that
// reconstructs f / l passes WENO_EPSB / l^2 and multiplies the result by l.
constexpr double WENO_EPSB = 0.75e-6;

// A constant in a scalar register pair. Given as a literal the compiler puts it into a
// two-address FMA and copies the addend it would overwrite (40 64-bit moves per face).
__device__ inline double scalar_const(double v) {
  __asm__("" : "+s"(v));
  return v;
}

__device__ inline void weno5_sd(double f0, double f1, double f2, double f3, double f4,
                                double epsb, double &S, double &den) {
  const double a = f1 - f0, b = f2 - f1, c = f3 - f2, d = f4 - f3;
  const double c1375 = scalar_const(-1.375), c0625 = scalar_const(-0.625);
  const double c025 = scalar_const(-0.25);
  const double t3 = fma(c1375, b, a), t2 = fma(c0625, c, b), t1 = fma(c1375, c, d);
  const double wb = fma(0.609375 * b, b, epsb), wc = fma(0.609375 * c, c, epsb);
  const double b1 = fma(t1, t1, wc), b2 = fma(t2, t2, wc), b3 = fma(t3, t3, wb);
  const double p1 = b2 * b3, p2 = b1 * b3, p3 = b1 * b2;
  const double s1 = p1 * p1, s2 = p2 * p2, s3 = p3 * p3;
  const double q1 = fma(c025, d, c), q2 = fma(0.5, b, c);
  const double q3 = fma(-1.0 / 6.0, a, (5.0 / 12.0) * b);
  S = fma(q1, s1, fma(q2, s2, q3 * s3));
  den = fma(1.0 / 3.0, s3, fma(2.0, s2, s1));
}

// The corrections of the f+ and f- reconstructions together, with a single reciprocal:
//   q = S+ / den+ + S- / den-,   f+ + f- = f2+ + f2- + (2/3) q
// (den+ den- is a product of eight (eps + beta) factors: finite for |beta| < 1e38, and normal for
// eps > 1e-38, which holds the acoustic components, with their 12e-6 cs^2, to cs > 3e-17).
// fp: f+ at points 0..4; fm: f- at points 5..1 (reversed).
__device__ inline double weno5_q(const double (&fp)[5], const double (&fm)[5], double epsb) {
  double Sp, dp, Sm, dm;
  weno5_sd(fp[0], fp[1], fp[2], fp[3], fp[4], epsb, Sp, dp);
  weno5_sd(fm[0], fm[1], fm[2], fm[3], fm[4], epsb, Sm, dm);
  return fma(Sp, dm, Sm * dp) * fast_rcp(dp * dm);
}

__device__ inline double weno5_both(const double (&fp)[5], const double (&fm)[5], double epsb) {
  return fma(2.0 / 3.0, weno5_q(fp, fm, epsb), fp[2] + fm[2]);
}

// Lax-Friedrichs speed of a face: the largest |u_n| + c of its six points.
template <int UN>
__device__ inline double face_alpha(const double *base, int FS, int LS) {
  double alpha = 0.0;
#pragma unroll
  for (int l = 0; l < 6; l++)
    alpha = fmax(alpha, fabs(base[UN * FS + l * LS]) + base[PT_C * FS + l * LS]);
  return alpha;
}

// Face flux with the 6-point stencil read from LDS as it is needed (point l, field q at
// base[q*FS + l*LS]), one split side at a time. UN, U1, U2: the normal and transverse velocity fields; F in direction-local order.
// The split flux of a point is (F +- alpha U) / 2 with, for x0 = rho (u +- alpha),
//   mass x0, normal momentum x0 u + p, transverse x0 v, x0 w, energy x0 E + u p,
// and its products with the left eigenvectors, taken in the frame of the Roe velocity
// (du, dv, dw the velocity differences, D = du^2 + dv^2 + dw^2), are
//   A = x0 du + p,  K = p (u +- alpha + (gamma-1) du) + (gamma-1)/2 x0 D,
//   K - A, x0 dv, x0 dw, x0 - K / cs, K + A
// up to constant factors: no cancellation of the mean flow, five fields per point. The Roe
// cs (the reference's csnd, the squared sound speed) is the weighted mean of the points' c^2
// plus (gamma-1)/2 w_L w_R |V_L - V_R|^2.
template <int UN, int U1, int U2>
__device__ inline void face_flux_lds(const double *base, int FS, int LS, double gamma,
                                     double igm, double alpha, double (&F)[5]) {
  const double gm = gamma - 1.0, gmh = 0.5 * gm;
  double u, v, w, cs;
  {
    const double *L = base + 2 * LS, *R = base + 3 * LS;
    const double Lsr = L[PT_SR * FS], Rsr = R[PT_SR * FS];
    const double iden = fast_rcp(Lsr + Rsr);
    const double wl = Lsr * iden, wr = Rsr * iden;
    const double uL = L[UN * FS], vL = L[U1 * FS], zL = L[U2 * FS];
    const double uR = R[UN * FS], vR = R[U1 * FS], zR = R[U2 * FS];
    u = fma(uL, wl, uR * wr);
    v = fma(vL, wl, vR * wr);
    w = fma(zL, wl, zR * wr);
    const double du = uR - uL, dv = vR - vL, dw = zR - zL;
    cs = fma(L[PT_C2 * FS], wl, R[PT_C2 * FS] * wr) +
         gmh * (wl * wr) * fma(du, du, fma(dv, dv, dw * dw));
  }
  const double ci = fast_rcp(cs);
  // The characteristic values are reconstructed without their constant factors (hci = 1/(4
  // cs) for components 0 and 4, 1/2 for 1..3), with eps scaled to match (1 / hci^2 = 16
  // cs^2).
  // ff1, ff2, ff3: the shear and entropy components (times 1/2); h04 and d04: half the sum
  // and half the difference of the acoustic ones (times hci), formed from K and A so that
  // the pressure-sized parts of K - A and K + A never meet in a rounded sum
  double ff1, ff2, ff3, h04, d04, xp[5], xm[5], D[6];            // xp[l]: point l, xm[l]: point 5 - l
  {
    double dv[6], dw[6];
#pragma unroll
    for (int l = 0; l < 6; l++) {
      const double *q = base + l * LS;
      const double un = q[UN * FS], r = q[PT_R * FS];
      if (l < 5) xp[l] = r * (un + alpha);
      if (l > 0) xm[5 - l] = r * (un - alpha);
      const double du = un - u;
      dv[l] = q[U1 * FS] - v;
      dw[l] = q[U2 * FS] - w;
      D[l] = gmh * fma(du, du, fma(dv[l], dv[l], dw[l] * dw[l]));
    }
    // the shear components (times 1/2)
    const double eps13 = 4.0 * WENO_EPSB;
    double fp[5], fm[5];
#pragma unroll
    for (int l = 0; l < 5; l++) { fp[l] = xp[l] * dv[l]; fm[l] = xm[l] * dv[5 - l]; }
    ff1 = weno5_both(fp, fm, eps13);
    __asm__ volatile("" : "+v"(ff1));
#pragma unroll
    for (int l = 0; l < 5; l++) { fp[l] = xp[l] * dw[l]; fm[l] = xm[l] * dw[5 - l]; }
    ff2 = weno5_both(fp, fm, eps13);
    __asm__ volatile("" : "+v"(ff2));
  }
  // an offset the compiler does not know to be zero: the points are read again here instead
  // of being kept in registers through the shear components
  int again = 0;
  __asm__ volatile("" : "+v"(again));
  {
    double Kp[5], Km[5], Ap[5], Am[5], fp[5], fm[5];
    const double tp = fma(-gm, u, alpha), tm = fma(-gm, u, -alpha);
#pragma unroll
    for (int l = 0; l < 6; l++) {
      const double *q = base + l * LS + again;
      const double un = q[UN * FS], p = q[PT_P * FS];
      const double du = un - u;
      if (l < 5) {
        Kp[l] = fma(p, fma(gamma, un, tp), xp[l] * D[l]);
        Ap[l] = fma(xp[l], du, p);
      }
      if (l > 0) {
        Km[5 - l] = fma(p, fma(gamma, un, tm), xm[5 - l] * D[l]);
        Am[5 - l] = fma(xm[5 - l], du, p);
      }
    }
    // the entropy component (times 1/2), then the acoustic ones (times hci)
#pragma unroll
    for (int l = 0; l < 5; l++) { fp[l] = fma(-ci, Kp[l], xp[l]); fm[l] = fma(-ci, Km[l], xm[l]); }
    ff3 = weno5_both(fp, fm, 4.0 * WENO_EPSB);
    __asm__ volatile("" : "+v"(ff3));
    const double eps04 = (16.0 * WENO_EPSB) * (cs * cs);
#pragma unroll
    for (int l = 0; l < 5; l++) { fp[l] = Kp[l] - Ap[l]; fm[l] = Km[l] - Am[l]; }
    double q0 = weno5_q(fp, fm, eps04);
    __asm__ volatile("" : "+v"(q0));
#pragma unroll
    for (int l = 0; l < 5; l++) { fp[l] = Kp[l] + Ap[l]; fm[l] = Km[l] + Am[l]; }
    const double q4 = weno5_q(fp, fm, eps04);
    h04 = fma(1.0 / 3.0, q0 + q4, Kp[2] + Km[2]);
    d04 = fma(1.0 / 3.0, q4 - q0, Ap[2] + Am[2]);
  }
  // the factors back (cs hci = 1/4); H = cs / (gamma-1) + q^2/2
  const double d40 = 0.5 * d04, f1 = 0.5 * ff1, f2t = 0.5 * ff2;
  const double hq = 0.5 * fma(u, u, fma(v, v, w * w));
  F[0] = 0.5 * fma(ci, h04, ff3);
  F[1] = fma(u, F[0], d40);
  F[2] = fma(v, F[0], f1);
  F[3] = fma(w, F[0], f2t);
  F[4] = fma(0.5 * igm, h04, fma(hq, F[0], fma(u, d40, fma(v, f1, w * f2t))));
}

// Species (passive tracer) face flux for one component from its 6 point values c[l]
// (utilities.cpp:376-377,395,439,473): component-wise WENO5 of the split fluxes
// (u c +- alpha c) / 2, no characteristic projection. The split fluxes are formed as
// c[l] hp[l] and c[5-l] hm[l] with the face's split factors hp[l] = (u_l + alpha) / 2 and
// hm[l] = (u_{5-l} - alpha) / 2 (tracer_split), which every tracer of the face shares.
__device__ inline void tracer_split(const double (&un)[6], double alpha, double (&hp)[5],
                                    double (&hm)[5]) {
#pragma unroll
  for (int l = 0; l < 5; l++) {
    hp[l] = 0.5 * (un[l] + alpha);
    hm[l] = 0.5 * (un[5 - l] - alpha);
  }
}

__device__ inline double tracer_face_flux(const double (&c)[6], const double (&hp)[5],
                                          const double (&hm)[5]) {
  double fp[5], fm[5];
#pragma unroll
  for (int l = 0; l < 5; l++) {
    fp[l] = c[l] * hp[l];
    fm[l] = c[5 - l] * hm[l];
  }
  return weno5_both(fp, fm, WENO_EPSB);
}

}  // namespace mvd
