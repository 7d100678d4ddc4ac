// Vector-Jacobian product of fe(): wbar = (d fe / d w)^T v.
//
// fe(w) = -div F with every face flux a function of its 6-point stencil, so
//   Fbar(face between cells c-1 | c) = (v_c - v_{c-1}) / delta   (no cell: 0)
// and each face's stencil adjoint sbar = (dF/ds)^T Fbar goes back to the stencil's source
// cells (ghost points are +-copies of interior cells). Every face recomputes its flux in the
// form of face_flux_lds and sweeps it in reverse. No face buffer: per direction a kernel walks
// along the lines and writes each cell once its last face is in:
//   fe_vjp_tracers - tracers, each lane its own (column, tracer), any direction;
//   fe_vjp_lines   - fluid along x: a wave walks whole x-lines 64 faces at a time;
//   fe_vjp_walk    - fluid along y or z: each lane its own column.
// The x kernels store wbar, the others add. No atomics between waves: the result is
// deterministic. The tracer kernel of a direction runs before the fluid one, which takes over
// the velocity and wave-speed adjoints that the tracers produce. 128^3 with ten tracers: per
// direction 0.28 (tracers) and 0.24 ms (fluid), 1.55 ms in all; one kernel for both, with tracer-
// major copies of w and wbar and the reference's formula order, took 2.77 ms at one wave per
// SIMD (480 registers, 38 KB of LDS).
#include <algorithm>

#include "mvd_device.hpp"
#include "mvd_internal.hpp"
#include "../../include/mvd_rhs.h"

namespace mvd {

namespace {

// The adjoint of a WENO5 reconstruction over f0..f4 (the f+ formula; the f- one is the same
// function of the reversed values): x_i = y d(weno)/d f_i for the cotangent y. weno =
// f2 + (2/3) Q with Q = sum o_k q_k over the normalised weights o_k = d_k e_k^-2 / sum, in the
// differences a, b, c, d of neighbouring values and the completed squares e_k of weno5_sd:
//   dQ = sum o_k dq_k - 2 sum (o_k / e_k) (q_k - Q) de_k,
//   de_1 = 2 t1 dt1 + (39/32) c dc and so on.
// One reciprocal (of the common denominator times e_1 e_2 e_3: seven factors, finite for
// |beta| < 1e43 and normal for eps > 1e-43); 77 operations. Returns Q.
__device__ inline double weno5_adj(double f0, double f1, double f2, double f3, double f4,
                                   double epsb, double y, double (&x)[5]) {
  const double a = f1 - f0, b = f2 - f1, c = f3 - f2, d = f4 - f3;
  const double c1375 = scalar_const(-1.375), c0625 = scalar_const(-0.625);
  const double c025 = scalar_const(-0.25), c025p = scalar_const(0.25);
  const double c125 = scalar_const(1.25), c13 = scalar_const(1.0 / 3.0);
  const double t3 = fma(c1375, b, a), t2 = fma(c0625, c, b), t1 = fma(c1375, c, d);
  const double hb = 0.609375 * b, hc = 0.609375 * c;
  const double wb = fma(hb, b, epsb), wc = fma(hc, c, epsb);
  const double e1 = fma(t1, t1, wc), e2 = fma(t2, t2, wc), e3 = fma(t3, t3, wb);
  const double p1 = e2 * e3, p2 = e1 * e3, p3 = e1 * e2;
  const double s1 = p1 * p1, s2 = 2.0 * (p2 * p2), s3 = c13 * (p3 * p3);
  const double q1 = fma(c025, d, c), q2 = fma(c025p, b, 0.5 * c), q3 = fma(-0.5, a, c125 * b);
  const double den = s1 + s2 + s3, E = p1 * e1;
  const double r = fast_rcp(den * E);
  const double iden = E * r, iE = (-4.0 * den) * r;
  const double Q = fma(q1, s1, fma(q2, s2, q3 * s3)) * iden;
  const double yd = ((2.0 / 3.0) * y) * iden;
  const double o1 = s1 * yd, o2 = s2 * yd, o3 = s3 * yd;
  const double m1 = (o1 * (p1 * iE)) * (q1 - Q), m2 = (o2 * (p2 * iE)) * (q2 - Q);
  const double m3 = (o3 * (p3 * iE)) * (q3 - Q);
  const double u1 = m1 * t1, u2 = m2 * t2, u3 = m3 * t3;
  const double ga = fma(-0.5, o3, u3), gd = fma(c025, o1, u1);
  const double gb = fma(m3, hb, fma(c1375, u3, fma(c125, o3, fma(c025p, o2, u2))));
  const double gc = fma(m1 + m2, hc, fma(c0625, u2, fma(c1375, u1, fma(0.5, o2, o1))));
  x[0] = -ga;
  x[1] = ga - gb;
  x[2] = y + (gb - gc);
  x[3] = gc - gd;
  x[4] = gd;
  return Q;
}

// The lines of cells along a direction D ("columns"), the rows of a line and its ghosts.
struct Walk {
  long rs, bs_in, bs_out, ncol;  // row stride; column col starts at (col % nin) bs_in + (col / nin) bs_out
  long afs, acs;                 // alb strides of a face and of a column
  int nin, n, ncb, nseg, per, add;
  double sa_lo, su_lo, sa_hi, su_hi;   // ghost signs: all conserved fields, normal velocity
  double idelta, gamma, igm;
};

struct TrWalk : Walk {
  const double *r, *m0, *m1, *m2, *e, *mn;   // fluid; mn: the momentum along the walk
  const double *t, *v;
  double *out, *ub, *alb;
};

// Fluid fields in direction-local order: rho, m_normal, m_t1, m_t2, et.
struct FlWalk : Walk {
  const double *w[5], *v[5];
  double *out[5];
  const double *ub, *alb;        // of the tracers, or null
};

// Row of extended index e: wrapped, mirrored or shifted (ghost_map); rows further out than
// the ghosts, which no face reads, are clamped.
__device__ inline int walk_row(const Walk &k, int e, double &sa, double &su) {
  sa = su = 1.0;
  const int n = k.n;
  if (e >= 0 && e < n) return e;
  if (k.per) {
    e = e < 0 ? e + n : e - n;
    return e < 0 ? e + n : e >= n ? e - n : e;
  }
  if (e < 0) { sa = k.sa_lo; su = k.su_lo; return min(-1 - e, n - 1); }
  sa = k.sa_hi; su = k.su_hi;
  return min(e - 3, n - 1);
}

__device__ inline long walk_cell(const Walk &k, long col) {
  const unsigned q = (unsigned)col / (unsigned)k.nin;
  return (long)((unsigned)col - q * (unsigned)k.nin) * k.bs_in + (long)q * k.bs_out;
}

__device__ inline void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------------------------------
// Tracers. With u_l the normal velocities and alpha the Lax-Friedrichs speed of a face, a
// tracer's flux reconstructs t_l (u_l +- alpha) / 2; its adjoint goes to the tracer, to the
// velocities and to alpha. A lane walks one tracer of one column along D over the rows
// [c0, c1), the lanes of a wave being consecutive (column, tracer) pairs: cell-major tracer
// rows along y and z are read as they lie. The stencil and the open rows' adjoints slide
// through registers (six faces per round, so that every index is a constant); a row is
// written out with its last face. Segments do the faces that reach into them again instead
// of exchanging rows, ghost rows are added to their source rows in the lane: no side
// buffer and no fix-up pass. The velocity adjoint of each cell and the alpha adjoint of each
// face are summed over a cell's tracers (in tracer order) once per round and handed to the
// fluid sweep in ub [cell] and alb [face]; so are the velocities and alphas that the lanes
// of a cell share, which one lane computes for all. About 280 instructions per
// face and tracer, 216 of them FP64 (0.2 ms to issue at 128^3 with ten tracers; 0.28 ms taken at
// three waves per SIMD, 0.31 at two; the row offsets come from LDS, computed in the scalar unit
// they spilled).
// ------------------------------------------------------------------------------------
template <int NC>
__global__ void __launch_bounds__(64, 3)
fe_vjp_tracers(TrWalk k) {
  constexpr int GPW = 64 / NC;                 // columns per wave
  constexpr int STEP = 64 / GPW;               // lanes lane / GPW + STEP * pass take the rows
  __shared__ double ring_u[12][GPW], ring_a[12][GPW], alpha[6][GPW];
  __shared__ double red[6][2][GPW * NC + 4], rsign[24];
  __shared__ long roff[24];
  const int lane = threadIdx.x, n = k.n;
  const int blk = blockIdx.x % k.ncb, seg = blockIdx.x / k.ncb;
  const int c0 = (int)((long)seg * n / k.nseg), c1 = (int)((long)(seg + 1) * n / k.nseg);
  const int fa = k.per ? c0 - 2 : max(c0 - 2, 0);       // first face
  const int fend = c1 + 2, fb = k.per ? fend : min(fend, n);   // faces past fb only close rows
  const int grp = min(lane / NC, GPW - 1), c = lane % NC;
  const long col0 = (long)blk * GPW;
  const bool act = lane < GPW * NC && col0 + grp < k.ncol;
  const long base = walk_cell(k, min(col0 + grp, k.ncol - 1)) * NC + c;
  const double *tp = k.t + base, *vp = k.v + base;
  double *op = k.out + base;
  // what the lanes of a cell share: one lane per (row, column) of a round
  const int gg = lane % GPW, gr = lane / GPW;
  const bool gact = col0 + gg < k.ncol;
  const long gbase = walk_cell(k, min(col0 + gg, k.ncol - 1));
  // offsets and signs of rows ra, ra+1, ... (cnt <= 64) into slots rho, rho+1, ... of 24
  const auto fill_rows = [&](int ra, int rho, int cnt) {
    if (lane < cnt) {
      double sa, su;
      const int sl = (rho + lane) % 24;
      roff[sl] = (long)walk_row(k, min(ra + lane, fend + 2), sa, su) * k.rs * NC;
      rsign[sl] = sa;
    }
  };
  // velocities and wave speeds of rows ra, ra+1, ... into ring slots rho, rho+1, ... of 12
  const auto fill = [&](int ra, int rho, int cnt) {
    for (int rr = gr; rr < cnt; rr += STEP) {
      double sa, su;
      const long cc = gbase + walk_row(k, min(ra + rr, fend + 2), sa, su) * k.rs;
      const double m0 = k.m0[cc], m1 = k.m1[cc], m2 = k.m2[cc];
      const double ir = fast_rcp(k.r[cc]);
      const double p = (k.gamma - 1.0) * (k.e[cc] - 0.5 * (m0 * m0 + m1 * m1 + m2 * m2) * ir);
      const double u = k.mn[cc] * ir;
      const int sl = (rho + rr) % 12;
      ring_u[sl][gg] = 0.5 * su * u;
      ring_a[sl][gg] = fabs(u) + fast_sqrt(k.gamma * p * ir);
    }
  };
  fill_rows(fa - 3, 0, 17);
  fill(fa - 3, 0, 11);
  wave_sync_lds();
  // window slot (j + l) % 6 holds point l of the round's face j: tracer, half velocity and
  // the adjoints so far
  double tw[6], hu[6], at[6], au[6], tn[6], vn[6], on[6];
#pragma unroll
  for (int l = 0; l < 6; l++) at[l] = au[l] = tw[l] = hu[l] = 0.0;
#pragma unroll
  for (int l = 0; l < 5; l++) {
    tw[l] = rsign[l] * tp[roff[l]];
    hu[l] = ring_u[l][grp];
  }
  // face f's new tracer row f+2, cotangent row f and open row f-3; rt: slot of row f-3
  const auto load_face = [&](int f, int rt, double &t, double &v, double &o) {
    t = tp[roff[(rt + 5) % 24]];
    v = vp[roff[(rt + 3) % 24]];
    if (k.add) o = f - 3 >= c0 && f - 3 < c1 ? op[roff[rt % 24]] : 0.0;
  };
#pragma unroll
  for (int j = 0; j < 6; j++) on[j] = 0.0;
#pragma unroll
  for (int j = 0; j < 6; j++) load_face(fa + j, j, tn[j], vn[j], on[j]);
  double vprev = fa > 0 || k.per ? vp[roff[2]] : 0.0;
  int par = 0, rt = 0;              // this round's slots of row f0-3: 0 or 6 of 12; of 24
#pragma unroll 1
  for (int f0 = fa; f0 <= fend; f0 += 6) {
    for (int jj = gr; jj < 6; jj += STEP) {
      double a = 0.0;
#pragma unroll
      for (int l = 0; l < 6; l++) a = fmax(a, ring_a[(par + jj + l) % 12][gg]);
      alpha[jj][gg] = a;
    }
    fill_rows(f0 + 14, rt + 17, 6);
    wave_sync_lds();
#pragma unroll
    for (int j = 0; j < 6; j++) {
      const int f = f0 + j;
      double alphab = 0.0, vu = 0.0;
      tw[(j + 5) % 6] = tn[j] * rsign[(rt + j + 5) % 24];
      hu[(j + 5) % 6] = ring_u[(par + j + 5) % 12][grp];
      at[(j + 5) % 6] = au[(j + 5) % 6] = 0.0;
      const double vcur = (f < n || k.per) ? vn[j] : 0.0;
      const double old = on[j];
      const double y = (vcur - vprev) * k.idelta;
      vprev = vcur;
      load_face(f + 6, rt + j + 6, tn[j], vn[j], on[j]);
      if (f <= fb) {
        const double ha = 0.5 * alpha[j][grp];
        double xp[5], xm[5], hp[5], hm[5];
        {
          double fp[5];
#pragma unroll
          for (int l = 0; l < 5; l++) {
            hp[l] = hu[(j + l) % 6] + ha;
            fp[l] = tw[(j + l) % 6] * hp[l];
          }
          (void)weno5_adj(fp[0], fp[1], fp[2], fp[3], fp[4], WENO_EPSB, y, xp);
#pragma unroll
          for (int l = 0; l < 5; l++) at[(j + l) % 6] = fma(xp[l], hp[l], at[(j + l) % 6]);
        }
        {
          double fm[5];                          // point 5 - l
#pragma unroll
          for (int l = 0; l < 5; l++) {
            hm[l] = hu[(j + 5 - l) % 6] - ha;
            fm[l] = tw[(j + 5 - l) % 6] * hm[l];
          }
          (void)weno5_adj(fm[0], fm[1], fm[2], fm[3], fm[4], WENO_EPSB, y, xm);
#pragma unroll
          for (int l = 0; l < 5; l++)
            at[(j + 5 - l) % 6] = fma(xm[l], hm[l], at[(j + 5 - l) % 6]);
        }
        // u_l: half of t (x+ + x-), alpha: half of the sum of t (x+ - x-)
#pragma unroll
        for (int l = 0; l < 6; l++) {
          const double t = tw[(j + l) % 6];
          const double xs = l == 0 ? xp[0] : l == 5 ? xm[0] : xp[l] + xm[5 - l];
          const double xd = l == 0 ? xp[0] : l == 5 ? -xm[0] : xp[l] - xm[5 - l];
          au[(j + l) % 6] = fma(t, xs, au[(j + l) % 6]);
          alphab = fma(t, xd, alphab);
        }
      }
      // row f-3 is complete; ghost rows are added to their source rows: -1-e (faces 0..2,
      // which only a column's first round has) and e-3
      const int e = f - 3;
      if (!k.per) {
        if (j < 3 && f == j) {
          at[(j + 5 - 2 * j) % 6] = fma(k.sa_lo, at[j], at[(j + 5 - 2 * j) % 6]);
          au[(j + 5 - 2 * j) % 6] = fma(k.su_lo, au[j], au[(j + 5 - 2 * j) % 6]);
        }
        if (f >= n) {
          at[j] = fma(k.sa_hi, at[(j + 3) % 6], at[j]);
          au[j] = fma(k.su_hi, au[(j + 3) % 6], au[j]);
        }
      }
      if (e >= c0 && e < c1 && act) op[roff[(rt + j) % 24]] = k.add ? old + at[j] : at[j];
      if (lane < GPW * NC) {
        red[j][0][lane] = au[j];
        red[j][1][lane] = alphab;
      }
    }
    wave_sync_lds();
    // sums over the tracers; each face's alpha adjoint is written by the segment it opens
    // (face n by the last one, as zero if it is face 0 again)
    for (int jq = gr; jq < 12; jq += STEP) {
      const int f = f0 + (jq >> 1), e = f - 3, q = jq & 1;
      const double *r = &red[jq >> 1][q][gg * NC];
      double a = r[0];
#pragma unroll
      for (int cc = 1; cc < NC; cc++) a += r[cc];
      a *= 0.5;
      if (gact) {
        if (q == 0) {
          if (e >= c0 && e < c1) k.ub[gbase + e * k.rs] = a;
        } else if (f >= c0 && (f < c1 || (f == n && c1 == n))) {
          k.alb[f * k.afs + (col0 + gg) * k.acs] = k.per && f == n ? 0.0 : a;
        }
      }
    }
    fill(f0 + 8, par + 11, 6);
    par = 6 - par;
    rt = rt == 18 ? 0 : rt + 6;
    wave_sync_lds();
  }
}

// ------------------------------------------------------------------------------------
// Fluid. The adjoint of face_flux_lds: with G = W / (4 cs) for the acoustic reconstructions
// W (K -+ A), S = G4 + G0, T = G4 - G0 and half the shear and entropy ones g1, g2, g3,
//   F0 = S + g3, F1 = u F0 + cs T, F2 = v F0 + g1, F3 = w F0 + g2,
//   F4 = cs S / (gamma-1) + (u^2 + v^2 + w^2)/2 F0 + u cs T + v g1 + w g2.
// The cotangents of the reconstructions need only the Roe state, so one pass forms each
// reconstruction and its adjoint, one split side at a time. W depends on cs through its eps,
// which is the derivative of a homogeneous function: d(G)/d(1/(4 cs)) = sum f dW/df.
// Adjoints are those of the points' (rho, u_n, u_t1, u_t2, p); a cell's go back to the
// conserved fields once all of its faces are in (fluid_store). Bound by issue at two waves per
// SIMD: 0.15 ms of instructions in 0.23 - 0.24 ms per direction at 128^3 (the reference's
// formula order with the tracers taken out: 0.46 ms at one wave per SIMD).
// ------------------------------------------------------------------------------------
enum { Q_R = 0, Q_U, Q_V, Q_W, Q_P, Q_A };     // Q_A: |u_n| + c

// Waits for a before b is used: keeps the compiler from starting on the next reconstruction
// (and from reading its points) while the registers of the current one are taken.
__device__ inline void then_on(const double (&a)[5], double (&b)[5]) {
  __asm__ volatile("" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(b[4])
                   : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]));
}
__device__ inline int then_at(const double (&a)[5], int o) {
  __asm__ volatile("" : "+v"(o) : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]));
  return o;
}

// Forms the sums here and not where they are used next (the compiler moves them into a later
// block and keeps both terms in registers until then).
__device__ inline void hold(double (&acc)[6][5]) {
#pragma unroll
  for (int l = 0; l < 6; l++)
    __asm__ volatile("" : "+v"(acc[l][0]), "+v"(acc[l][1]), "+v"(acc[l][2]), "+v"(acc[l][3]), "+v"(acc[l][4]));
}

// Stencil point l, field q at P[off[l] + q * FS]. lstar: the first point with the largest
// |u_n| + c. acc[l] += the adjoint of point l. About 1250 FP64 instructions; the points are read
// again from LDS wherever they are used, which is what makes it fit into 256 registers.
template <int FS>
__device__ inline void face_adjoint(const double *P, const int (&off)[6], double gamma, double igm,
                                    double alpha, int lstar, const double (&Fb)[5], double alphab,
                                    double (&acc)[6][5]) {
  const double gm = gamma - 1.0, gmh = 0.5 * gm;
  double u, v, w, cs, wl, wr;
  {
    const double *L = P + off[2], *R = P + off[3];
    const double rL = L[Q_R * FS], rR = R[Q_R * FS], sL = fast_sqrt(rL), sR = fast_sqrt(rR);
    const double iden = fast_rcp(sL + sR);
    wl = sL * iden;
    wr = sR * iden;
    const double uL = L[Q_U * FS], vL = L[Q_V * FS], zL = L[Q_W * FS];
    const double uR = R[Q_U * FS], vR = R[Q_V * FS], zR = R[Q_W * FS];
    u = fma(uL, wl, uR * wr);
    v = fma(vL, wl, vR * wr);
    w = fma(zL, wl, zR * wr);
    const double du = uR - uL, dv = vR - vL, dw = zR - zL;
    const double cL = gamma * L[Q_P * FS] * fast_rcp(rL), cR = gamma * R[Q_P * FS] * fast_rcp(rR);
    cs = fma(cL, wl, cR * wr) + gmh * (wl * wr) * fma(du, du, fma(dv, dv, dw * dw));
  }
  const double ci = fast_rcp(cs), hci = 0.25 * ci;
  const double tb = fma(u, Fb[4], Fb[1]), y1 = 0.5 * fma(v, Fb[4], Fb[2]);
  const double y2 = 0.5 * fma(w, Fb[4], Fb[3]);
  double y0, y4, y3;
  {
    const double hq = 0.5 * fma(u, u, fma(v, v, w * w));
    const double B0 = fma(hq, Fb[4], fma(u, Fb[1], fma(v, Fb[2], fma(w, Fb[3], Fb[0]))));
    const double Sb = fma(igm * cs, Fb[4], B0), Tb = cs * tb;
    y0 = hci * (Sb - Tb);
    y4 = hci * (Sb + Tb);
    y3 = 0.5 * B0;
  }
  // The acoustic values are reconstructed times the power of two next to 1 / cs: the seven factors
  // of size eps04 in weno5_adj's denominator stay of order 1e-5 each however small cs is (with
  // eps in units of cs^2 their product underflows below cs = 3e-20). W0, W4 and sfx carry
  // that factor until the end.
  const int ecs = __builtin_amdgcn_frexp_exp(cs);
  const double css = ldexp(cs, -ecs);
  const double eps04 = (16.0 * WENO_EPSB) * (css * css), eps13 = 4.0 * WENO_EPSB;
  double W0 = 0.0, W1 = 0.0, W2 = 0.0, W3 = 0.0, W4 = 0.0;
  double sfx = 0.0, skx = 0.0, ub = 0.0, vb = 0.0, wb = 0.0;
  double X[5] = {y0, y1, y2, y3, y4};
#pragma unroll
  for (int sd = 0; sd < 2; sd++) {
    const double al = sd == 0 ? alpha : -alpha;
    const double tt = fma(-gm, u, al);
    const auto pt = [&](int l, int o) { return P + off[sd == 0 ? l : 5 - l] + o; };
    double x[5], K[5], D[5], Kb[5], Ab[5], f[5];
    int o = then_at(X, 0);
#pragma unroll
    for (int l = 0; l < 5; l++) {
      const double *q = pt(l, o);
      const double un = q[Q_U * FS], p = q[Q_P * FS], du = un - u;
      const double dv = q[Q_V * FS] - v, dw = q[Q_W * FS] - w;
      x[l] = q[Q_R * FS] * (un + al);
      D[l] = gmh * fma(du, du, fma(dv, dv, dw * dw));
      K[l] = fma(p, fma(gamma, un, tt), x[l] * D[l]);
      f[l] = ldexp(K[l] - fma(x[l], du, p), -ecs);
    }
    {
      const double Q0 = weno5_adj(f[0], f[1], f[2], f[3], f[4], eps04, y0, Ab);
      W0 += fma(2.0 / 3.0, Q0, f[2]);
#pragma unroll
      for (int l = 0; l < 5; l++) sfx = fma(f[l], Ab[l], sfx);
      __asm__ volatile("" : "+v"(sfx), "+v"(W0));
    }
    o = then_at(Ab, 0);
#pragma unroll
    for (int l = 0; l < 5; l++) {
      const double *q = pt(l, o);
      f[l] = ldexp(K[l] + fma(x[l], q[Q_U * FS] - u, q[Q_P * FS]), -ecs);
    }
    {
      double x4[5];
      const double Q4 = weno5_adj(f[0], f[1], f[2], f[3], f[4], eps04, y4, x4);
      W4 += fma(2.0 / 3.0, Q4, f[2]);
#pragma unroll
      for (int l = 0; l < 5; l++) {
        sfx = fma(f[l], x4[l], sfx);
        Kb[l] = Ab[l] + x4[l];
        Ab[l] = x4[l] - Ab[l];
      }
      __asm__ volatile("" : "+v"(sfx), "+v"(W4));
    }
#pragma unroll
    for (int l = 0; l < 5; l++) f[l] = fma(-ci, K[l], x[l]);
    then_on(Ab, f);
    {
      const double Q3 = weno5_adj(f[0], f[1], f[2], f[3], f[4], eps13, y3, X);
      W3 += fma(2.0 / 3.0, Q3, f[2]);
      __asm__ volatile("" : "+v"(W3));
    }
    o = then_at(X, 0);
#pragma unroll
    for (int l = 0; l < 5; l++) {
      const int a = sd == 0 ? l : 5 - l;
      const double *q = pt(l, o);
      const double un = q[Q_U * FS], p = q[Q_P * FS], du = un - u;
      skx = fma(K[l], X[l], skx);
      Kb[l] = fma(-ci, X[l], Kb[l]);
      X[l] = fma(Kb[l], D[l], fma(Ab[l], du, X[l]));
      acc[a][4] += fma(Kb[l], fma(gamma, un, tt), Ab[l]);
      const double pk = p * Kb[l];
      K[l] = gm * (Kb[l] * x[l]);                 // the adjoint of D, times gamma - 1
      const double dub = fma(Ab[l], x[l], du * K[l]);
      acc[a][1] += fma(gamma, pk, dub);
      ub -= fma(gm, pk, dub);
      alphab += sd == 0 ? pk : -pk;
    }
    hold(acc);
    then_on(X, K);
    // the shear components
#pragma unroll
    for (int c = 2; c < 4; c++) {
      double xs[5], d[5];
      o = then_at(X, 0);
#pragma unroll
      for (int l = 0; l < 5; l++) {
        d[l] = pt(l, o)[c * FS] - (c == 2 ? v : w);
        f[l] = x[l] * d[l];
      }
      const double Q = weno5_adj(f[0], f[1], f[2], f[3], f[4], eps13, c == 2 ? y1 : y2, xs);
      (c == 2 ? W1 : W2) += fma(2.0 / 3.0, Q, f[2]);
#pragma unroll
      for (int l = 0; l < 5; l++) {
        const double b = fma(xs[l], x[l], d[l] * K[l]);
        X[l] = fma(xs[l], d[l], X[l]);
        acc[sd == 0 ? l : 5 - l][c] += b;
        (c == 2 ? vb : wb) -= b;
      }
      hold(acc);
    }
    o = then_at(X, 0);
#pragma unroll
    for (int l = 0; l < 5; l++) {
      const int a = sd == 0 ? l : 5 - l;
      const double *q = pt(l, o);
      const double xr = X[l] * q[Q_R * FS];
      acc[a][0] = fma(X[l], q[Q_U * FS] + al, acc[a][0]);
      acc[a][1] += xr;
      alphab += sd == 0 ? xr : -xr;
    }
    hold(acc);
    __asm__ volatile("" : "+v"(skx), "+v"(W1), "+v"(W2));
    X[0] = alphab; X[1] = ub; X[2] = vb; X[3] = wb; X[4] = sfx;
  }
  // the Roe state: from the back-projection, then to the two points
  double csb;
  {
    const double h04 = ldexp(hci, ecs), S = h04 * (W4 + W0), T = h04 * (W4 - W0);
    const double F0 = fma(0.5, W3, S);
    csb = fma(ci, fma(ci, skx, -ldexp(sfx, ecs)), fma(igm * Fb[4], S, T * tb));
    ub += fma(Fb[1], F0, Fb[4] * fma(u, F0, cs * T));
    vb += fma(Fb[2], F0, Fb[4] * fma(v, F0, 0.5 * W1));
    wb += fma(Fb[3], F0, Fb[4] * fma(w, F0, 0.5 * W2));
  }
  {
    const int o = then_at(X, 0);
    const double *L = P + off[2] + o, *R = P + off[3] + o;
    const double rL = L[Q_R * FS], irL = fast_rcp(rL), cL = gamma * L[Q_P * FS] * irL;
    const double rR = R[Q_R * FS], irR = fast_rcp(rR), cR = gamma * R[Q_P * FS] * irR;
    const double du = R[Q_U * FS] - L[Q_U * FS], dv = R[Q_V * FS] - L[Q_V * FS];
    const double dw = R[Q_W * FS] - L[Q_W * FS];
    const double Qb = gmh * csb, Qv = fma(du, du, fma(dv, dv, dw * dw)), ww = wl * wr;
    // the adjoint of w_L minus that of w_R
    const double wd = fma(Qb * Qv, wr - wl, csb * (cL - cR)) - fma(ub, du, fma(vb, dv, wb * dw));
    const double q2 = 2.0 * Qb * ww;
    acc[2][1] += fma(ub, wl, -q2 * du);
    acc[3][1] += fma(ub, wr, q2 * du);
    acc[2][2] += fma(vb, wl, -q2 * dv);
    acc[3][2] += fma(vb, wr, q2 * dv);
    acc[2][3] += fma(wb, wl, -q2 * dw);
    acc[3][3] += fma(wb, wr, q2 * dw);
    // dw_L = w_L w_R / 2 (drho_L / rho_L - drho_R / rho_R); c^2 = gamma p / rho
    const double h = 0.5 * wd * ww, cl = csb * wl * irL, cr = csb * wr * irR;
    acc[2][0] += fma(-cl, cL, rL > 0.0 ? h * irL : 0.0);
    acc[3][0] -= fma(cr, cR, rR > 0.0 ? h * irR : 0.0);
    acc[2][4] = fma(gamma, cl, acc[2][4]);
    acc[3][4] = fma(gamma, cr, acc[3][4]);
  }
  hold(acc);
  // Lax-Friedrichs speed: alpha = |u_l*| + c_l*
  {
    int o = off[0];
#pragma unroll
    for (int l = 1; l < 6; l++) o = l == lstar ? off[l] : o;
    const double uS = P[o + Q_U * FS], pS = P[o + Q_P * FS], ir = fast_rcp(P[o + Q_R * FS]);
    const double c2 = gamma * pS * ir;
    const double cc = c2 > 0.0 ? 0.5 * ir * fast_rcp(fast_sqrt(c2)) : 0.0;
    const double kp = gamma * cc, kr = -c2 * cc, ku = uS < 0.0 ? -1.0 : 1.0;
#pragma unroll
    for (int l = 0; l < 6; l++) {
      const double ab = l == lstar ? alphab : 0.0;
      acc[l][0] = fma(kr, ab, acc[l][0]);
      acc[l][1] = fma(ku, ab, acc[l][1]);
      acc[l][4] = fma(kp, ab, acc[l][4]);
    }
  }
}

// A conserved state as a stencil point, with its ghost signs.
template <int FS>
__device__ inline void put_point(const Walk &k, const double (&x)[5], double sa, double su,
                                 double *q) {
  const double ir = fast_rcp(x[0]), u = x[1] * ir;
  const double p = (k.gamma - 1.0) * (x[4] - 0.5 * (x[1] * x[1] + x[2] * x[2] + x[3] * x[3]) * ir);
  q[Q_R * FS] = sa * x[0];
  q[Q_U * FS] = su * u;
  q[Q_V * FS] = x[2] * ir;
  q[Q_W * FS] = x[3] * ir;
  q[Q_P * FS] = sa * p;
  q[Q_A * FS] = fabs(u) + fast_sqrt(k.gamma * p * ir);
}

// Adjoint of a cell's (rho, u, p) back to its conserved fields, into wbar (local order).
__device__ inline void fluid_store(const FlWalk &k, long cell, const double (&b)[5], double r,
                                   double u, double v, double w) {
  double old[5];
#pragma unroll
  for (int a = 0; a < 5; a++) old[a] = k.add ? k.out[a][cell] : 0.0;
  const double ir = fast_rcp(r), pb = (k.gamma - 1.0) * b[4];
  double x[5];
  x[0] = fma(0.5 * pb, fma(u, u, fma(v, v, w * w)), b[0]) -
         fma(b[1], u, fma(b[2], v, b[3] * w)) * ir;
  x[1] = fma(-pb, u, b[1] * ir);
  x[2] = fma(-pb, v, b[2] * ir);
  x[3] = fma(-pb, w, b[3] * ir);
  x[4] = pb;
#pragma unroll
  for (int a = 0; a < 5; a++) k.out[a][cell] = k.add ? old[a] + x[a] : x[a];
}

// y and z: each lane walks its own column over the rows [c0, c1) of a segment, with the
// stencil in an LDS ring of six rows and the open rows' adjoints in registers. Segments do
// the five faces that reach into them from outside again, ghost rows are added to their
// source rows in the lane. The loads for the next face are issued between the split sides and
// the Roe state, where registers are free.
__global__ void __launch_bounds__(64, 2)
fe_vjp_walk(FlWalk k) {
  constexpr int FS = 64, LS = 6 * 64;
  __shared__ double P[6 * LS];
  const int lane = threadIdx.x, n = k.n;
  const int blk = blockIdx.x % k.ncb, seg = blockIdx.x / k.ncb;
  const int c0 = (int)((long)seg * n / k.nseg), c1 = (int)((long)(seg + 1) * n / k.nseg);
  const int fa = k.per ? c0 - 2 : max(c0 - 2, 0);
  const int fend = c1 + 2, fb = k.per ? fend : min(fend, n);
  const long col0 = (long)blk * 64 + lane;
  const bool act = col0 < k.ncol;
  const long col = act ? col0 : k.ncol - 1, base = walk_cell(k, col);
  double nw[5], nv[5], vl[5], nal = 0.0, acc[6][5];
  const auto load_row = [&](int e) {
    double sa, su;
    const long c = base + walk_row(k, min(e, fend + 2), sa, su) * k.rs;
#pragma unroll
    for (int a = 0; a < 5; a++) nw[a] = k.w[a][c];
  };
  const auto put_row = [&](int e, int slot) {
    double sa, su;
    (void)walk_row(k, min(e, fend + 2), sa, su);
    put_point<FS>(k, nw, sa, su, P + slot * LS + lane);
  };
  // the cotangents of the cells either side of face f, and its alpha adjoint
  const auto load_v = [&](int f) {
    double sa, su;
    f = min(f, fend + 2);
    const int row = walk_row(k, f, sa, su);
    const long cr = base + row * k.rs;
    const long cl = base + walk_row(k, k.per ? f - 1 : max(f - 1, 0), sa, su) * k.rs;
#pragma unroll
    for (int a = 0; a < 5; a++) { nv[a] = k.v[a][cr]; vl[a] = k.v[a][cl]; }
    if (k.alb) nal = k.alb[(k.per ? row : min(f, n)) * k.afs + col * k.acs];
  };
#pragma unroll
  for (int l = 0; l < 6; l++)
#pragma unroll
    for (int a = 0; a < 5; a++) acc[l][a] = 0.0;
#pragma unroll 1
  for (int l = 0; l < 5; l++) {
    load_row(fa - 3 + l);
    put_row(fa - 3 + l, l);
  }
  load_v(fa);
  load_row(fa + 2);
  int s0 = 0;
#pragma unroll 1
  for (int f = fa; f <= fend; f++) {
    const int e = f - 3;
    const bool own = e >= c0 && e < c1;
    put_row(f + 2, s0 >= 1 ? s0 - 1 : 5);
    int off[6];
#pragma unroll
    for (int l = 0; l < 6; l++) off[l] = (s0 + l >= 6 ? s0 + l - 6 : s0 + l) * LS + lane;
    if (f <= fb) {
      double Fb[5], alpha = 0.0;
      const double mr = f < n || k.per ? k.idelta : 0.0, ml = f > 0 || k.per ? k.idelta : 0.0;
#pragma unroll
      for (int a = 0; a < 5; a++)
        Fb[a] = mr == ml ? (nv[a] - vl[a]) * k.idelta : mr != 0.0 ? nv[a] * mr : -(vl[a] * ml);
      int lstar = -1;
#pragma unroll
      for (int l = 0; l < 6; l++) {
        const double a = P[off[l] + Q_A * FS];
        if (alpha < a) { alpha = a; lstar = l; }
      }
      face_adjoint<FS>(P, off, k.gamma, k.igm, alpha, lstar, Fb, nal, acc);
    }
    load_row(f + 3);
    load_v(f + 1);
    // row f-3 is complete; ghost rows: -1-e and e-3 are their source rows
    if (!k.per) {
      const auto fold = [&](int to, int from, double sa, double su) {
        acc[to][0] = fma(sa, acc[from][0], acc[to][0]);
        acc[to][1] = fma(su, acc[from][1], acc[to][1]);
        acc[to][2] += acc[from][2];
        acc[to][3] += acc[from][3];
        acc[to][4] = fma(sa, acc[from][4], acc[to][4]);
      };
      if (f == 0) fold(5, 0, k.sa_lo, k.su_lo);
      else if (f == 1) fold(3, 0, k.sa_lo, k.su_lo);
      else if (f == 2) fold(1, 0, k.sa_lo, k.su_lo);
      if (f >= n) fold(0, 3, k.sa_hi, k.su_hi);
    }
    if (own && act) {
      const long cell = base + e * k.rs;
      const double *q = P + off[0];
      if (k.ub) acc[0][1] += k.ub[cell];
      fluid_store(k, cell, acc[0], q[Q_R * FS], q[Q_U * FS], q[Q_V * FS], q[Q_W * FS]);
    }
#pragma unroll
    for (int l = 0; l < 5; l++)
#pragma unroll
      for (int a = 0; a < 5; a++) acc[l][a] = acc[l + 1][a];
#pragma unroll
    for (int a = 0; a < 5; a++) acc[5][a] = 0.0;
    s0 = s0 == 5 ? 0 : s0 + 1;
  }
}

// x: a wave walks whole lines 64 faces at a time, the lanes along x; lines follow one
// another, each with its ghost points (and, if periodic, with the faces around its ends done
// again) at consecutive positions, whose points and adjoints live in a ring of RING positions.
// The six points of a face are added with six LDS adds per component: within one
// instruction the lanes hit distinct positions and a wave's LDS operations complete in order,
// so the order of the sums is fixed. A position is final once the faces up to three beyond it
// are in. RING holds the positions of 64 faces and the six below them: 64 + 5 per line begun
// + 6, 128 for lines of eight faces or more.
template <int RING>
__global__ void __launch_bounds__(64, 2)
fe_vjp_lines(FlWalk k, int lps) {
  constexpr int FS = RING;
  __shared__ double P[6 * RING], A[5 * RING];
  const int lane = threadIdx.x, n = k.n;
  const int fa = k.per ? -2 : 0, nf = k.per ? n + 5 : n + 1, np = nf + 5;
  // faces and positions are counted from the wave's first line
  const long line0 = (long)blockIdx.x * lps;
  const int nl = (int)min((long)lps, k.ncol - line0);
  const double inf = 1.0 / nf, inp = 1.0 / np;
  const auto div = [](int a, double inv) { return (int)(((double)a + 0.5) * inv); };   // exact below 2^31
  const int Q1 = nl * nf;
  int loaded = 0, done = 0;                        // next position to load, to write out
#pragma unroll 1
  for (int B = 0; B < Q1; B += 64) {
    const int qe = min(B + 64, Q1) - 1;            // last face of this pass
    const int le = div(qe, inf), last = qe + le * (np - nf) + 5;
    for (int p = loaded + lane; p <= last; p += 64) {
      const int line = div(p, inp), e = p - line * np + fa - 3;
      const int slot = p & (RING - 1);
      double sa, su;
      const long c = (line0 + line) * n + walk_row(k, e, sa, su);
      double x[5];
#pragma unroll
      for (int a = 0; a < 5; a++) x[a] = k.w[a][c];
      put_point<FS>(k, x, sa, su, P + slot);
#pragma unroll
      for (int a = 0; a < 5; a++) A[a * RING + slot] = 0.0;
    }
    loaded = last + 1;
    wave_sync_lds();
    const int q = min(B + lane, qe);
    const bool mine = B + lane <= qe;
    const int line = div(q, inf), f = q - line * nf + fa;
    int off[6];
#pragma unroll
    for (int l = 0; l < 6; l++) off[l] = (q + line * (np - nf) + l) & (RING - 1);
    double acc[6][5];
    {
      double Fb[5], alphab = 0.0, alpha = 0.0;
      double sa, su;
      const bool hr = k.per || f < n, hl = k.per || f > 0;
      const long cr = (line0 + line) * n + walk_row(k, hr ? f : n - 1, sa, su);
      const long cl = (line0 + line) * n + walk_row(k, hl ? f - 1 : 0, sa, su);
#pragma unroll
      for (int a = 0; a < 5; a++) {
        const double vr = k.v[a][cr], vl = k.v[a][cl];
        Fb[a] = ((hr ? vr : 0.0) - (hl ? vl : 0.0)) * k.idelta;
      }
      if (k.alb) alphab = k.alb[(k.per ? walk_row(k, f, sa, su) : f) + (line0 + line) * (n + 1)];
      int lstar = -1;
#pragma unroll
      for (int l = 0; l < 6; l++) {
        const double a = P[Q_A * FS + off[l]];
        if (alpha < a) { alpha = a; lstar = l; }
#pragma unroll
        for (int b = 0; b < 5; b++) acc[l][b] = 0.0;
      }
      face_adjoint<FS>(P, off, k.gamma, k.igm, alpha, lstar, Fb, alphab, acc);
    }
    if (mine) {
#pragma unroll
      for (int l = 0; l < 6; l++) {
#pragma unroll
        for (int a = 0; a < 5; a++) atomicAdd(&A[a * RING + off[l]], acc[l][a]);
        wave_sync_lds();
      }
    }
    wave_sync_lds();
    // positions below the next face's stencil are final
    const int hi = qe + 1 + div(qe + 1, inf) * (np - nf);
    for (int p = done + lane; p < hi; p += 64) {
      const int ln = div(p, inp), e = p - ln * np + fa - 3;
      if (e < 0 || e >= n) continue;
      const int slot = p & (RING - 1);
      const long cell = (line0 + ln) * n + e;
      double b[5];
#pragma unroll
      for (int a = 0; a < 5; a++) b[a] = A[a * RING + slot];
      const auto ghost = [&](int pg, double sa, double su) {
        const int sl = pg & (RING - 1);
        b[0] = fma(sa, A[sl], b[0]);
        b[1] = fma(su, A[RING + sl], b[1]);
        b[2] += A[2 * RING + sl];
        b[3] += A[3 * RING + sl];
        b[4] = fma(sa, A[4 * RING + sl], b[4]);
      };
      if (!k.per && e < 3) ghost(p - 2 * e - 1, k.sa_lo, k.su_lo);
      if (!k.per && e >= n - 3) ghost(p + 3, k.sa_hi, k.su_hi);
      if (k.ub) b[1] += k.ub[cell];
      fluid_store(k, cell, b, P[Q_R * FS + slot], P[Q_U * FS + slot], P[Q_V * FS + slot],
                  P[Q_W * FS + slot]);
    }
    done = hi;
    wave_sync_lds();
  }
}

// Waves that a direction's walk is split into at least, where columns allow: four per SIMD
// for the tracers, two for the fluid (what its registers allow).
constexpr long TRACER_WAVES = 4096, FLUID_WAVES = 2048;

static Walk walk_of(const Grid &g, int d) {
  const long nx = g.nx, nxy = nx * g.ny;
  Walk k{};
  k.n = extent(g, d);
  k.ncol = nxy * g.nz / k.n;
  k.nin = (int)(d == 0 ? 1 : d == 1 ? nx : nxy);
  k.bs_in = d == 0 ? 0 : 1;
  k.bs_out = d == 0 ? nx : nxy;
  k.rs = d == 0 ? 1 : d == 1 ? nx : nxy;
  k.afs = d == 0 ? 1 : k.ncol;
  k.acs = d == 0 ? k.n + 1 : 1;
  k.per = g.bc[2 * d] == BC_PERIODIC;
  k.add = d != 0;
  const int lo = g.bc[2 * d], hi = g.bc[2 * d + 1];
  k.sa_lo = lo == BC_DIRICHLET ? -1.0 : 1.0;
  k.sa_hi = hi == BC_DIRICHLET ? -1.0 : 1.0;
  k.su_lo = lo == BC_REFLECTING ? -1.0 : 1.0;      // Dirichlet negates m and rho: u stays
  k.su_hi = hi == BC_REFLECTING ? -1.0 : 1.0;
  k.idelta = 1.0 / (d == 0 ? g.dx : d == 1 ? g.dy : g.dz);
  k.gamma = g.gamma;
  k.igm = g.igm;
  return k;
}

// Column blocks of gpw columns and the segments that give at least `waves` waves, of
// minrows rows or more.
static void walk_split(Walk &k, long gpw, long waves, int minrows) {
  k.ncb = (int)((k.ncol + gpw - 1) / gpw);
  const long maxseg = std::max(1, k.n / minrows);
  k.nseg = (int)std::min(maxseg, (waves + k.ncb - 1) / k.ncb);
}

template <int NC>
static void tracers_launch(const Grid &g, int d, const Fields &w, const double *v, double *out,
                           double *ub, double *alb, hipStream_t st) {
  TrWalk k{};
  (Walk &)k = walk_of(g, d);
  k.r = w.w[0]; k.m0 = w.w[1]; k.m1 = w.w[2]; k.m2 = w.w[3]; k.e = w.w[4]; k.mn = w.w[1 + d];
  k.t = w.chem; k.v = v; k.out = out; k.ub = ub; k.alb = alb;
  walk_split(k, 64 / NC, TRACER_WAVES, 8);
  hipLaunchKernelGGL(fe_vjp_tracers<NC>, dim3((unsigned)(k.ncb * k.nseg)), dim3(64), 0, st, k);
}

static int tracers_run(const Grid &g, int d, const Fields &w, const double *v, double *out,
                       double *ub, double *alb, hipStream_t st) {
  switch (g.nchem) {
    case 1: tracers_launch<1>(g, d, w, v, out, ub, alb, st); return 0;
    case 2: tracers_launch<2>(g, d, w, v, out, ub, alb, st); return 0;
    case 4: tracers_launch<4>(g, d, w, v, out, ub, alb, st); return 0;
    case 6: tracers_launch<6>(g, d, w, v, out, ub, alb, st); return 0;
    case 10: tracers_launch<10>(g, d, w, v, out, ub, alb, st); return 0;
    default: return MVD_UNSUPPORTED;
  }
}

static void fluid_run(const Grid &g, int d, const Fields &w, const Fields &v, const FieldsOut &out,
                      const double *ub, const double *alb, hipStream_t st) {
  FlWalk k{};
  (Walk &)k = walk_of(g, d);
  k.ub = ub;
  k.alb = alb;
  for (int a = 0; a < 5; a++) {
    const int q = a == 1 ? 1 + d : a == 1 + d ? 1 : a;
    k.w[a] = w.w[q];
    k.v[a] = v.w[q];
    k.out[a] = out.w[q];
  }
  if (d == 0) {
    const int lps = (int)((k.ncol + FLUID_WAVES - 1) / FLUID_WAVES);
    const dim3 grid((unsigned)((k.ncol + lps - 1) / lps));
    if (k.n + (k.per ? 5 : 1) >= 8)
      hipLaunchKernelGGL(fe_vjp_lines<128>, grid, dim3(64), 0, st, k, lps);
    else hipLaunchKernelGGL(fe_vjp_lines<256>, grid, dim3(64), 0, st, k, lps);
  } else {
    walk_split(k, 64, FLUID_WAVES, 4);
    hipLaunchKernelGGL(fe_vjp_walk, dim3((unsigned)(k.ncb * k.nseg)), dim3(64), 0, st, k);
  }
}

}  // namespace

static long max_faces(const Grid &g) {
  const long nx = g.nx, ny = g.ny, nz = g.nz;
  return std::max({(nx + 1) * ny * nz, nx * (ny + 1) * nz, nx * ny * (nz + 1)});
}

// Scratch, with tracers only: ub (cells), alb (faces of a direction) and a tracer array for
// calls whose wbar tracers overlap an input's.
size_t fe_vjp_buffer_doubles(const Grid &g) {
  const long ncell = (long)g.nx * g.ny * g.nz;
  return g.nchem ? (size_t)(1 + g.nchem) * ncell + max_faces(g) : 0;
}

int fe_vjp_launch(const Grid &g, const Fields &w, const Fields &v, const FieldsOut &out,
                  double *buf, hipStream_t st) {
  const long ncell = (long)g.nx * g.ny * g.nz, nt = g.nchem * ncell;
  double *ub = nullptr, *alb = nullptr, *tr = out.chem;
  if (g.nchem) {
    ub = buf;
    alb = ub + ncell;
    const auto overlaps = [&](const double *a) { return a < out.chem + nt && out.chem < a + nt; };
    if (overlaps(w.chem) || overlaps(v.chem)) tr = alb + max_faces(g);
  }
  for (int d = 0; d < 3; d++) {
    if (g.nchem) {
      const int rc = tracers_run(g, d, w, v.chem, tr, ub, alb, st);
      if (rc) return rc;
    }
    fluid_run(g, d, w, v, out, ub, alb, st);
  }
  if (tr != out.chem &&
      hipMemcpyAsync(out.chem, tr, sizeof(double) * nt, hipMemcpyDeviceToDevice, st) != hipSuccess)
    return -1;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mvd
