// WENO5 flux divergence fe() kernels for gfx950 (FP64).
//
// Plain path (the comparator; fEuler, utilities.cpp:17-253, transcribed for the GPU):
//   fe_plain_faces : one thread per cell computes the lower x/y/z faces of its cell
//                    (plus the domain's upper boundary faces) with the reference-order
//                    face flux, into SoA face-flux buffers;
//   fe_plain_div   : one thread per cell forms the divergence in the reference order.
// Small grids without tracers (one launch; also a Runge-Kutta stage with its combination):
//   fe_box         : faces of all three directions of a box of 8 x 4 x 4 cells, one per
//                    thread, and the divergence.
// Fast path without tracers (two launches):
//   fe_xyface_div  : x- and y-faces of 16 x 15-cell plane tiles from one LDS staging of the
//                    tile and its x/y halos, and their part of the divergence into wdot
//                    (the x and y face fluxes stay in LDS); the legal-state check;
//   fe_zface_div_xy: z-faces (blocks walk up columns of 16 x-cells 16 faces at a time, their
//                    primitives staged in LDS) and the divergence of the cells between
//                    them, adding the x/y part read from wdot.
// Fast path with tracers (three launches):
//   fe_xyface_div<NC>: as without tracers, then the tracers on the same x- and y-faces
//                    (their values staged in LDS, up to five tracers at a time, after the
//                    fluid phase)
//                    and their part of the divergence into wdot;
//   fe_zface_div_xy: the fluid z-faces, as without tracers;
//   fe_zface_tracers: the tracer z-faces (tiles of 16 x-cells by 16 faces; per point the
//                    normal velocity, wave speed and tracer values in LDS), adding their
//                    part of the divergence.
// The divergence is accumulated as -((dFx/dx + dFy/dy) + dFz/dz), the reference's
// association (utilities.cpp:202-207).
#include "mvd_device.hpp"
#include "mvd_internal.hpp"

namespace mvd {

// ------------------------------------------------------------------------------------
// shared helpers
// ------------------------------------------------------------------------------------

__device__ inline long cell_index(const Grid &g, long i, long j, long k) {
  return i + (long)g.nx * (j + (long)g.ny * k);
}

// Cell index of extended index e along direction d through (i,j,k), and its ghost signs.
__device__ inline long stencil_cell(const Grid &g, int d, int i, int j, int k, int e,
                                    GhostMap &m) {
  m = ghost_map(g, d, e);
  if (d == 0) i = m.src; else if (d == 1) j = m.src; else k = m.src;
  return cell_index(g, i, j, k);
}

// Conserved state of one stencil point in direction-local order
// (rho, m_normal, m_t1, m_t2, et) with ghost signs applied; the momentum permutation is
// the reference's swap of component 1 with component 1+d (utilities.cpp:283-285).
__device__ inline void load_local(const Grid &g, const Fields &f, int d, long c,
                                  const GhostMap &m, double (&s)[5]) {
  const double r = f.w[0][c], mx = f.w[1][c], my = f.w[2][c], mz = f.w[3][c], e = f.w[4][c];
  double mn, m1, m2;
  if (d == 0) { mn = mx; m1 = my; m2 = mz; }
  else if (d == 1) { mn = my; m1 = mx; m2 = mz; }
  else { mn = mz; m1 = my; m2 = mx; }
  s[0] = r * m.sgn_all;
  s[1] = mn * m.sgn_norm;
  s[2] = m1 * m.sgn_all;
  s[3] = m2 * m.sgn_all;
  s[4] = e * m.sgn_all;
}

// direction-local flux components back to global momentum order
__device__ inline int global_comp(int d, int a) {
  if (a == 1) return 1 + d;
  if (a == 1 + d) return 1;
  return a;
}

__device__ inline void legal_check(const Grid &g, const Fields &f, long c, unsigned *flag) {
  const double r = f.w[0][c], mx = f.w[1][c], my = f.w[2][c], mz = f.w[3][c], e = f.w[4][c];
  const double p = (g.gamma - 1.0) * (e - (mx * mx + my * my + mz * mz) * 0.5 / r);
  unsigned bits = 0;
  if (!(r > 0.0)) bits |= 1u;
  if (!(e > 0.0)) bits |= 2u;
  if (!(p > 0.0)) bits |= 4u;
  if (bits) atomicOr(flag, bits);
}

// ------------------------------------------------------------------------------------
// plain comparator
// ------------------------------------------------------------------------------------

template <int NC>
__global__ void __launch_bounds__(256)
fe_plain_faces(Grid g, Fields f, double *Fx, double *Fy, double *Fz, unsigned *flag) {
  constexpr int NV = 5 + NC;
  const long nxp = g.nx + 1, nyp = g.ny + 1, nzp = g.nz + 1;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= nxp * nyp * nzp) return;
  const int i = (int)(tid % nxp);
  const int j = (int)((tid / nxp) % nyp);
  const int k = (int)(tid / (nxp * nyp));
  if (i < g.nx && j < g.ny && k < g.nz) legal_check(g, f, cell_index(g, i, j, k), flag);
  const long nfx = nxp * g.ny * g.nz, nfy = (long)g.nx * nyp * g.nz, nfz = (long)g.nx * g.ny * nzp;
  for (int d = 0; d < 3; d++) {
    const bool ok = (d == 0) ? (j < g.ny && k < g.nz) : (d == 1) ? (i < g.nx && k < g.nz)
                                                               : (i < g.nx && j < g.ny);
    if (!ok) continue;
    const int c0 = (d == 0) ? i : (d == 1) ? j : k;
    double s[6][NV];
    for (int l = 0; l < 6; l++) {
      GhostMap m;
      const long c = stencil_cell(g, d, i, j, k, c0 - 3 + l, m);
      double loc[5];
      load_local(g, f, d, c, m, loc);
      for (int v = 0; v < 5; v++) s[l][v] = loc[v];
      for (int v = 0; v < NC; v++) s[l][5 + v] = f.chem[(long)NC * c + v] * m.sgn_all;
    }
    double ff[NV];
    face_flux_ref<NC>(s, g.gamma, ff);
    double *F = (d == 0) ? Fx : (d == 1) ? Fy : Fz;
    const long nf = (d == 0) ? nfx : (d == 1) ? nfy : nfz;
    const long face = (d == 0) ? (i + nxp * (j + (long)g.ny * k))
                    : (d == 1) ? (i + (long)g.nx * (j + nyp * k))
                               : (i + (long)g.nx * (j + (long)g.ny * k));
    for (int a = 0; a < NV; a++) F[(long)global_comp(d, a) * nf + face] = ff[a];
  }
}

template <int NC>
__global__ void __launch_bounds__(256)
fe_plain_div(Grid g, const double *Fx, const double *Fy, const double *Fz, FieldsOut out) {
#pragma clang fp contract(off)
  constexpr int NV = 5 + NC;
  const long ncell = (long)g.nx * g.ny * g.nz;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const long i = c % g.nx, j = (c / g.nx) % g.ny, k = c / ((long)g.nx * g.ny);
  const long nxp = g.nx + 1, nyp = g.ny + 1, nzp = g.nz + 1;
  const long nfx = nxp * g.ny * g.nz, nfy = (long)g.nx * nyp * g.nz, nfz = (long)g.nx * g.ny * nzp;
  const long x0 = i + nxp * (j + g.ny * k);
  const long y0 = i + g.nx * (j + nyp * k);
  const long z0 = c;
  for (int v = 0; v < NV; v++) {
    const double dv = (Fx[v * nfx + x0 + 1] - Fx[v * nfx + x0]) / g.dx +
                      (Fy[v * nfy + y0 + g.nx] - Fy[v * nfy + y0]) / g.dy +
                      (Fz[v * nfz + z0 + (long)g.nx * g.ny] - Fz[v * nfz + z0]) / g.dz;
    if (v < 5) out.w[v][c] = 0.0 - dv;
    else out.chem[(long)NC * c + (v - 5)] = 0.0 - dv;
  }
}

// ------------------------------------------------------------------------------------
// fast path
// ------------------------------------------------------------------------------------

// Raw conserved state of a stencil point of a z line with the ghost signs applied.
struct RawPt {
  double r, mx, my, mz, e;
};

__device__ inline RawPt load_raw_z(const Fields &f, int c, double sa, double sn) {
  RawPt q;
  q.r = f.w[0][c] * sa;
  q.mx = f.w[1][c] * sa;
  q.my = f.w[2][c] * sa;
  q.mz = f.w[3][c] * sn;
  q.e = f.w[4][c] * sa;
  return q;
}

// Cell of extended index e along direction D of the line whose e = 0 cell is `base`
// (cells `stride` apart), with ghost signs. Interior points take the short path.
template <int D>
__device__ inline int line_cell(const Grid &g, int base, int stride, int n, int e, double &sa,
                                double &sn) {
  if (e >= 0 && e < n) {
    sa = 1.0;
    sn = 1.0;
    return base + e * stride;
  }
  const GhostMap m = ghost_map(g, D, e);
  sa = m.sgn_all;
  sn = m.sgn_norm;
  return base + m.src * stride;
}

// local (rho, m_normal, m_t1, m_t2, e) flux of direction D into global component order
template <int D>
__device__ inline void to_global(const double (&Fl)[5], double *Fg) {
  Fg[0] = Fl[0];
  Fg[4] = Fl[4];
  if (D == 1) { Fg[2] = Fl[1]; Fg[1] = Fl[2]; Fg[3] = Fl[3]; }
  else { Fg[3] = Fl[1]; Fg[2] = Fl[2]; Fg[1] = Fl[3]; }
}

// Tracer z-faces, adding their part to the x/y part that fe_xyface_div<NC> left in
// out.chem (the fluid z-faces are fe_zface_div_xy's). A block of 16 x 16 threads covers 16
// x-cells of row j and 16 consecutive z-faces, i.e. the 15 cells between them. Per point
// of the tile (21 per column) LDS holds the normal velocity w, the wave speed |w| + c
// (store_point's c, so the face's alpha is the fluid flux's bit for bit) and the NC tracer
// values; each thread forms its face's alpha and split factors once and then the NC
// tracer fluxes. Without the fluid flux's registers the kernel runs at a higher occupancy
// than a fused fluid + tracer z kernel.
//
// ST: doubles per cell record of f.chem and out.chem. MODE (fslow's rates, NC = 9 species of
// records of 10): 1 also moves the total-energy rate out.w[4] (final: the fluid kernels have
// run) into the record's tenth slot and leaves zero there; 2 in addition converts the whole
// record to the scaled variables (FeSlow).
enum { TR_PLAIN = 0, TR_SLOW, TR_SLOW_SCALED };
template <int NC, int ST, int MODE>
__global__ void __launch_bounds__(256)
fe_zface_tracers(Grid g, Fields f, FieldsOut out, double idz, FeSlow slow) {
  constexpr int TX = 16, TF = 16, TPTS = TF + 5, TC = TF - 1, NPT = TPTS * TX;
  constexpr int NR = (NPT + 255) / 256;
  constexpr int PT_SZ = (2 + NC) * NPT, FL_SZ = NC * TF * TX;
  __shared__ double s_buf[PT_SZ > FL_SZ ? PT_SZ : FL_SZ];   // [w | speed | tracers][point]
  const int t = threadIdx.x, tx = t % TX, ty = t / TX;
  const int nxc = (g.nx + TX - 1) / TX, ncc = (g.nz + TC - 1) / TC;
  int b = blockIdx.x;
  const int xc = b % nxc;
  b /= nxc;
  const int cc = b % ncc;
  const int j = b / ncc;
  const int k0 = cc * TC;
  const int i = xc * TX + tx, k = k0 + ty;
  // the x/y part of the thread's cell, loaded first (its latency passes under the staging)
  const bool cell_ok = ty < TC && i < g.nx && k < g.nz;
  const long cell = i + (long)g.nx * (j + (long)g.ny * k);
  double dxy[NC];
#pragma unroll
  for (int v = 0; v < NC; v++) dxy[v] = cell_ok ? out.chem[(long)ST * cell + v] : 0.0;
  double erate = 0.0;
  if (MODE != TR_PLAIN && cell_ok) erate = out.w[4][cell];
  // points k0 - 3 .. k0 + TF + 1 of the 16 columns: located, loaded, then converted
  {
    const int stride = g.nx * g.ny;
    int cs[NR];
    double sa[NR], sn[NR];
    bool use[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int s = t + 256 * r;
      const int row = s / TX, x = s - row * TX;
      const int e = k0 - 3 + row;
      use[r] = s < NPT && xc * TX + x < g.nx && e <= g.nz + 2;
      cs[r] = use[r] ? line_cell<2>(g, xc * TX + x + g.nx * j, stride, g.nz, e, sa[r], sn[r])
                     : 0;
    }
    RawPt raw[NR];
    double tv[NR][NC];
#pragma unroll
    for (int r = 0; r < NR; r++) {
      if (!use[r]) continue;
      raw[r] = load_raw_z(f, cs[r], sa[r], sn[r]);
#pragma unroll
      for (int v = 0; v < NC; v++) tv[r][v] = f.chem[(long)ST * cs[r] + v] * sa[r];
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
      if (!use[r]) continue;
      const int s = t + 256 * r;
      const RawPt &q = raw[r];
      const double ir = fast_rcp(q.r);
      const double p = (g.gamma - 1.0) * (q.e - 0.5 * (q.mx * q.mx + q.my * q.my + q.mz * q.mz) * ir);
      const double un = q.mz * ir;
      s_buf[s] = un;
      s_buf[NPT + s] = fabs(un) + fast_sqrt(g.gamma * p * ir);
#pragma unroll
      for (int v = 0; v < NC; v++) s_buf[(2 + v) * NPT + s] = tv[r][v];
    }
  }
  __syncthreads();
  const bool face_ok = i < g.nx && k <= g.nz;
  double Fz[NC];
  if (face_ok) {
    const double *pb = s_buf + ty * TX + tx;
    double alpha = 0.0, un[6];
#pragma unroll
    for (int l = 0; l < 6; l++) alpha = fmax(alpha, pb[NPT + l * TX]);
#pragma unroll
    for (int l = 0; l < 6; l++) un[l] = pb[l * TX];
    double hp[5], hm[5];
    tracer_split(un, alpha, hp, hm);
#pragma unroll
    for (int v = 0; v < NC; v++) {
      double cv[6];
#pragma unroll
      for (int l = 0; l < 6; l++) cv[l] = pb[(2 + v) * NPT + l * TX];
      Fz[v] = tracer_face_flux(cv, hp, hm);
    }
  }
  __syncthreads();   // the points are dead; LDS takes the face fluxes [tracer][face][x]
  if (face_ok) {
#pragma unroll
    for (int v = 0; v < NC; v++) s_buf[(v * TF + ty) * TX + tx] = Fz[v];
  }
  __syncthreads();
  if (!cell_ok) return;
  const double *const sc = MODE == TR_SLOW_SCALED ? slow.scale + (long)ST * cell : nullptr;
#pragma unroll
  for (int v = 0; v < NC; v++) {
    const double dz = (s_buf[(v * TF + ty + 1) * TX + tx] - s_buf[(v * TF + ty) * TX + tx]) * idz;
    const double r = 0.0 - (dxy[v] + dz);
    out.chem[(long)ST * cell + v] = MODE == TR_SLOW_SCALED ? r / sc[v] : r;
  }
  if (MODE != TR_PLAIN) {
    out.chem[(long)ST * cell + NC] = MODE == TR_SLOW_SCALED ? erate * slow.eunits / sc[NC] : erate;
    out.w[4][cell] = 0.0;
  }
}

// z-faces of the fluid fields, adding their part to the x/y part that fe_xyface_div left in
// out. A block of 16 x 16 threads walks up a segment of `len` cells of the columns of 16
// x-cells of row j, ZC faces at a time (one per thread). Each chunk's points (its faces' and
// five more rows) are in LDS as primitive values; the next chunk's 16 new rows and the x/y
// part of the cells it completes are loaded while the fluxes are formed, so only a segment's
// first loads are waited for, no point is loaded or converted twice within a segment, and
// the last five rows and the last face's flux are carried over. A kernel that loaded 37
// rows for 32 faces and then computed them issued 65% of the time; at 256^3 the z faces went
// from 0.78 to 0.56 ms with this form (0.74 at four waves per SIMD, where it spills).
constexpr int ZX = 16, ZC = 16, ZROWS = ZC + 5;
__global__ void __launch_bounds__(256, 3)
fe_zface_div_xy(Grid g, Fields f, FieldsOut out, double idz, int nseg, int len) {
  constexpr int FS = ZROWS * ZX;                        // points per field
  constexpr int FF = (ZC + 1) * ZX;                     // fluxes per field (one carried row)
  __shared__ double s_pt[PT_NF * FS], s_f[5 * FF];
  const int t = threadIdx.x, tx = t % ZX, ty = t / ZX;
  const int nxc = (g.nx + ZX - 1) / ZX;
  int b = blockIdx.x;
  const int xc = b % nxc;
  b /= nxc;
  const int seg = b % nseg;
  const int j = b / nseg;
  const int ks = seg * len, ke = min(ks + len, g.nz);   // cells [ks, ke), faces ks..ke
  const int i = xc * ZX + tx;
  const int plane = g.nx * g.ny;
  const int col = i + g.nx * j;
  const bool iok = i < g.nx;
  // point (row e, this thread's column) or nothing
  const auto load = [&](int e, RawPt &q) {
    const bool use = iok && e <= g.nz + 2;
    double sa = 1.0, sn = 1.0;
    const int c = use ? line_cell<2>(g, col, plane, g.nz, e, sa, sn) : 0;
    if (use) q = load_raw_z(f, c, sa, sn);
    return use;
  };
  const auto store = [&](int row, const RawPt &q) {
    (void)store_point(s_pt + row * ZX + tx, FS, q.r, q.mx, q.my, q.mz, q.e, g.gamma);
  };
  {
    RawPt q0, q1;                                       // rows ty, and 16 + ty of the first chunk
    const bool u0 = load(ks - 3 + ty, q0);
    const bool u1 = ty < ZROWS - 16 && load(ks - 3 + 16 + ty, q1);
    if (u0) store(ty, q0);
    if (u1) store(16 + ty, q1);
  }
  for (int f0 = ks;; f0 += ZC) {
    const bool more = f0 + ZC <= ke;
    RawPt qn;
    bool un = false;
    if (more) un = load(f0 + ZC + 2 + ty, qn);          // row 5 + ty of the next chunk
    const int k = f0 - 1 + ty;                          // the cell this chunk's faces complete
    const bool own = iok && k >= ks && k < ke;
    const int cell = col + plane * k;
    double dxy[5];
#pragma unroll
    for (int a = 0; a < 5; a++) dxy[a] = own ? out.w[a][cell] : 0.0;
    __syncthreads();                                    // the chunk's points are there
    if (iok && f0 + ty <= ke) {
      double Fl[5], Fz[5];
      const double *base = s_pt + ty * ZX + tx;
      face_flux_lds<PT_W, PT_V, PT_U>(base, FS, ZX, g.gamma, g.igm,
                                      face_alpha<PT_W>(base, FS, ZX), Fl);
      to_global<2>(Fl, Fz);
#pragma unroll
      for (int a = 0; a < 5; a++) s_f[a * FF + (ty + 1) * ZX + tx] = Fz[a];
    }
    __syncthreads();                                    // fluxes there, points read
    if (own) {
#pragma unroll
      for (int a = 0; a < 5; a++) {
        const double *F = s_f + a * FF + ty * ZX + tx;
        out.w[a][cell] = 0.0 - (dxy[a] + (F[ZX] - F[0]) * idz);
      }
    }
    if (!more) break;
    // carry rows 16..20 of every field to rows 0..4 and the last face's flux to row 0
    constexpr int NP = PT_NF * 5 * ZX, NALL = NP + 5 * ZX, NR = (NALL + 255) / 256;
    double cv[NR];
#pragma unroll
    for (int n = 0; n < NR; n++) {
      const int e = t + 256 * n;
      const int fp = e / (5 * ZX), pp = e % (5 * ZX), ef = e - NP;
      cv[n] = e < NP ? s_pt[fp * FS + ZC * ZX + pp]
                     : e < NALL ? s_f[(ef / ZX) * FF + ZC * ZX + ef % ZX] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NR; n++) {
      const int e = t + 256 * n;
      const int fp = e / (5 * ZX), pp = e % (5 * ZX), ef = e - NP;
      if (e < NP) s_pt[fp * FS + pp] = cv[n];
      else if (e < NALL) s_f[(ef / ZX) * FF + ef % ZX] = cv[n];
    }
    if (un) store(5 + ty, qn);
  }
}

// x- and y-faces of one z-plane tile together: a block covers XY_TX x XY_TY cells of plane k
// and forms (Fx[i+1]-Fx[i])/dx + (Fy[j+1]-Fy[j])/dy for them into out (the z kernel then
// adds the z part), so the x and y face fluxes never go to HBM. The points of the tile and
// of its x and y halos (a cross, 3 deep) are converted once into LDS and serve both
// directions; x-faces (XY_TX+1 per row) and y-faces (XY_TY+1 per column) are 255 and 256
// with the 16 x 15 tile: one of each per thread.
//
// With NC tracers further phases follow on the same faces, at most XY_TP tracers at a time:
// their values on the cross (issued before the previous divergence) go to LDS where dead
// point fields were, one tracer per field; u, v and c stay, for the faces' split factors;
// each thread forms its x- and y-face's tracer fluxes from LDS. The kernel is bound by its
// FP64 instructions: 8 point fields and the y fluxes (40 KB) let four blocks share a CU, so
// that four waves per SIMD hide the LDS and dependency latency (128 registers, vector
// instructions issued in 81% of the cycles). At 256^3: 0.94 ms, 1.26 before (three waves per
// SIMD, ten point fields, 786 FP64 instructions per face with its share of the staging; now 638).
constexpr int XY_TX = 16, XY_TY = 15;
constexpr int XY_PX = XY_TX + 6, XY_PY = XY_TY + 6;      // point window 22 x 21
constexpr int XY_NP = XY_PX * XY_PY;
constexpr int XY_NXF = (XY_TX + 1) * XY_TY, XY_NYF = XY_TX * (XY_TY + 1);   // 255, 256
constexpr int XY_LDS = PT_NF * XY_NP + 5 * XY_NYF;          // points + y-face fluxes
constexpr int XY_TP = 5;     // fields per divergence pass: the fluid's, or at most as many tracers
// the x-face fluxes go over dead point fields, from PT_W on; u, v (PT_U, PT_V) and c survive
static_assert(PT_W * XY_NP + XY_TP * XY_NXF <= PT_C * XY_NP, "x fluxes over w, p, sr, c2");

// LDS field that holds tracer v of a pass (the fields a tracer phase may overwrite)
__device__ constexpr int xy_slot(int v) { return v < 4 ? PT_W + v : PT_R; }

// Point q of the cross of the tile at (x0, y0) in plane k: its cell, ghost signs (all
// fields, mx, my) and whether it is used (inside the cross and the extended grid) and a
// cell of the tile (`own`), with the boundary mapping of ghost_map.
struct XYPoint {
  int cell;
  double s_all, s_mx, s_my;
  bool use, own, row, col;
};

__device__ inline XYPoint xy_point(const Grid &g, int x0, int y0, int k, int q) {
  XYPoint P;
  const int yy = q / XY_PX, xx = q - yy * XY_PX;
  const int ex = x0 - 3 + xx, ey = y0 - 3 + yy;
  P.row = yy >= 3 && yy < 3 + XY_TY && ey < g.ny;          // x-line point
  P.col = xx >= 3 && xx < 3 + XY_TX && ex < g.nx;          // y-column point
  int i = ex, j = ey;
  P.s_all = P.s_mx = P.s_my = 1.0;
  P.use = q < XY_NP && (P.row ? ex <= g.nx + 2 : (P.col && ey <= g.ny + 2));
  P.own = P.row && P.col && ex >= 0;   // a cell of the tile: legal_state once
  if (P.row) {
    if (ex < 0 || ex >= g.nx) {
      const GhostMap m = ghost_map(g, 0, ex);
      i = m.src;
      P.s_all = P.s_my = m.sgn_all;
      P.s_mx = m.sgn_norm;
    }
  } else if (P.col) {
    if (ey < 0 || ey >= g.ny) {
      const GhostMap m = ghost_map(g, 1, ey);
      j = m.src;
      P.s_all = P.s_mx = m.sgn_all;
      P.s_my = m.sgn_norm;
    }
  }
  P.cell = P.use ? (int)(i + (long)g.nx * (j + (long)g.ny * k)) : 0;
  return P;
}

// (Fx[i+1]-Fx[i])/dx + (Fy[j+1]-Fy[j])/dy of field a of a pass, cell (ci, cj) of the tile
__device__ inline double xy_div(const double *sfx, const double *sfy, int a, int ci, int cj,
                                double idx, double idy) {
  const double *fx = sfx + (a * XY_TY + cj) * (XY_TX + 1) + ci;
  const double *fy = sfy + (a * (XY_TY + 1) + cj) * XY_TX + ci;
  return (fx[1] - fx[0]) * idx + (fy[XY_TX] - fy[0]) * idy;
}

template <int NC, int ST>
__global__ void __launch_bounds__(256, 4)
fe_xyface_div(Grid g, Fields f, FieldsOut out, double idx, double idy, unsigned *flag) {
  // points [PT_NF][XY_NP], then the y-face fluxes [5][XY_TY+1][XY_TX]
  __shared__ double sh[XY_LDS];
  double *const sfy = sh + PT_NF * XY_NP;
  double *const sfx = sh + PT_W * XY_NP;     // [5][XY_TY][XY_TX+1], once the points are dead
  const int t = threadIdx.x;
  const int nxb = (g.nx + XY_TX - 1) / XY_TX, nyb = (g.ny + XY_TY - 1) / XY_TY;
  // The hardware deals blocks to the 8 XCDs in turn, and each XCD has its own L2. Tiles are
  // renumbered so that consecutive tiles (x neighbours, which read the same halo lines)
  // run on the same XCD one after another: block b takes tile (b % 8) * m + b / 8 (m = the
  // blocks per XCD; the remainder past 8 m keeps its own number).
  const unsigned m8 = gridDim.x / 8;
  int b = blockIdx.x < 8 * m8 ? (int)((blockIdx.x % 8) * m8 + blockIdx.x / 8) : (int)blockIdx.x;
  const int xb = b % nxb;
  b /= nxb;
  const int yb = b % nyb;
  const int k = b / nyb;
  const int x0 = xb * XY_TX, y0 = yb * XY_TY;
  // stage the cross: points of the tile's rows (real y) over the x window, with x ghosts,
  // then the other points of the tile's columns (real x) over the y window, with y ghosts.
  // A thread's points (q = t + 256 r) are located first and all their loads issued before
  // any is converted, so that their latencies overlap.
  constexpr int NR = (XY_NP + 255) / 256;
  {
    XYPoint pt[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) pt[r] = xy_point(g, x0, y0, k, t + 256 * r);
    double raw[NR][5];
#pragma unroll
    for (int r = 0; r < NR; r++) {
#pragma unroll
      for (int a = 0; a < 5; a++) raw[r][a] = pt[r].use ? f.w[a][pt[r].cell] : 1.0;
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
      if (!pt[r].use) continue;
      const double rr = raw[r][0] * pt[r].s_all, mx = raw[r][1] * pt[r].s_mx;
      const double my = raw[r][2] * pt[r].s_my;
      const double mz = raw[r][3] * pt[r].s_all, e = raw[r][4] * pt[r].s_all;
      const double p = store_point(sh + t + 256 * r, XY_NP, rr, mx, my, mz, e, g.gamma);
      if (pt[r].own) {
        unsigned bits = 0;
        if (!(rr > 0.0)) bits |= 1u;
        if (!(e > 0.0)) bits |= 2u;
        if (!(p > 0.0)) bits |= 4u;
        if (bits) atomicOr(flag, bits);
      }
    }
  }
  __syncthreads();
  // y-face t: column cx, faces between rows y0+fy-1 and y0+fy (points yy = fy..fy+5)
  const int cx = t % XY_TX, fy = t / XY_TX;
  const bool yok = x0 + cx < g.nx && y0 + fy <= g.ny;
  const double *const yb0 = sh + fy * XY_PX + cx + 3;
  // x-face t: row ry, faces between columns x0+fx-1 and x0+fx (points xx = fx..fx+5)
  const int ry = t / (XY_TX + 1), fx = t % (XY_TX + 1);
  const bool xok = t < XY_NXF && y0 + ry < g.ny && x0 + fx <= g.nx;
  const double *const xb0 = sh + (ry + 3) * XY_PX + fx;
  if (yok) {
    double Fl[5], Fy[5];
    face_flux_lds<PT_V, PT_U, PT_W>(yb0, XY_NP, XY_PX, g.gamma, g.igm,
                                    face_alpha<PT_V>(yb0, XY_NP, XY_PX), Fl);
    to_global<1>(Fl, Fy);
#pragma unroll
    for (int a = 0; a < 5; a++) sfy[(a * (XY_TY + 1) + fy) * XY_TX + cx] = Fy[a];
  }
  double Fx[5];
  if (xok)
    face_flux_lds<PT_U, PT_V, PT_W>(xb0, XY_NP, 1, g.gamma, g.igm,
                                    face_alpha<PT_U>(xb0, XY_NP, 1), Fx);
  __syncthreads();                    // points dead: their LDS takes the x-face fluxes
  if (xok)
#pragma unroll
    for (int a = 0; a < 5; a++) sfx[(a * XY_TY + ry) * (XY_TX + 1) + fx] = Fx[a];
  __syncthreads();
  const int ci = t % XY_TX, cj = t / XY_TX;
  const bool cok = cj < XY_TY && x0 + ci < g.nx && y0 + cj < g.ny;
  const long cell = (x0 + ci) + (long)g.nx * ((y0 + cj) + (long)g.ny * k);
  if constexpr (NC == 0) {
    if (cok)
#pragma unroll
      for (int a = 0; a < 5; a++) out.w[a][cell] = xy_div(sfx, sfy, a, ci, cj, idx, idy);
  } else {
    // the faces' alpha for the tracers, formed again (as the fluid flux forms it) rather
    // than held through the fluid fluxes
    double alpha_y = 0.0, alpha_x = 0.0;
    if (yok) alpha_y = face_alpha<PT_V>(yb0, XY_NP, XY_PX);
    if (xok) alpha_x = face_alpha<PT_U>(xb0, XY_NP, 1);
    constexpr int NPASS = (NC + XY_TP - 1) / XY_TP, TP = (NC + NPASS - 1) / NPASS;
#pragma unroll 1
    for (int v0 = 0; v0 < NC; v0 += TP) {
      // the pass's tracer values of the thread's cross points, loaded now so that their
      // latency passes under the divergence of the previous pass. The points are located
      // again rather than kept: made opaque, the tile origin keeps the compiler from
      // holding the staging's values.
      double tv[NR][TP];
      {
        int ox = x0, oy = y0, ok = k;
        __asm__ volatile("" : "+s"(ox), "+s"(oy), "+s"(ok));
#pragma unroll
        for (int r = 0; r < NR; r++) {
          const XYPoint P = xy_point(g, ox, oy, ok, t + 256 * r);
#pragma unroll
          for (int v = 0; v < TP; v++)
            tv[r][v] = P.use && v0 + v < NC ? f.chem[(long)ST * P.cell + v0 + v] * P.s_all : 0.0;
        }
      }
      if (cok) {
        if (v0 == 0) {
#pragma unroll
          for (int a = 0; a < 5; a++) out.w[a][cell] = xy_div(sfx, sfy, a, ci, cj, idx, idy);
        } else {
#pragma unroll
          for (int v = 0; v < TP; v++)
            out.chem[(long)ST * cell + v0 - TP + v] = xy_div(sfx, sfy, v, ci, cj, idx, idy);
        }
      }
      __syncthreads();                  // the previous pass's fluxes are read
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const int q = t + 256 * r;
        if (q < XY_NP)
#pragma unroll
          for (int v = 0; v < TP; v++) sh[xy_slot(v) * XY_NP + q] = tv[r][v];
      }
      __syncthreads();
      double Fxt[TP];
      if (yok) {
        double un[6], hp[5], hm[5];
#pragma unroll
        for (int l = 0; l < 6; l++) un[l] = yb0[PT_V * XY_NP + l * XY_PX];
        tracer_split(un, alpha_y, hp, hm);
#pragma unroll
        for (int v = 0; v < TP; v++) {
          double cv[6];
#pragma unroll
          for (int l = 0; l < 6; l++) cv[l] = yb0[xy_slot(v) * XY_NP + l * XY_PX];
          sfy[(v * (XY_TY + 1) + fy) * XY_TX + cx] = tracer_face_flux(cv, hp, hm);
        }
      }
      if (xok) {
        double un[6], hp[5], hm[5];
#pragma unroll
        for (int l = 0; l < 6; l++) un[l] = xb0[PT_U * XY_NP + l];
        tracer_split(un, alpha_x, hp, hm);
#pragma unroll
        for (int v = 0; v < TP; v++) {
          double cv[6];
#pragma unroll
          for (int l = 0; l < 6; l++) cv[l] = xb0[xy_slot(v) * XY_NP + l];
          Fxt[v] = tracer_face_flux(cv, hp, hm);
        }
      }
      __syncthreads();                  // tracer values dead
      if (xok)
#pragma unroll
        for (int v = 0; v < TP; v++) sfx[(v * XY_TY + ry) * (XY_TX + 1) + fx] = Fxt[v];
      __syncthreads();
    }
    if (cok)
#pragma unroll
      for (int v = 0; v < TP; v++) {
        constexpr int v0 = (NPASS - 1) * TP;
        if (v0 + v < NC)
          out.chem[(long)ST * cell + v0 + v] = xy_div(sfx, sfy, v, ci, cj, idx, idy);
      }
  }
}

// ------------------------------------------------------------------------------------
// one-launch fe() of small grids
// ------------------------------------------------------------------------------------

// fe() of a grid too small to fill the device is bound by latency: each launch costs its
// start, its staging and one face flux per thread in turn (Sod's 128x3x3 cells: 7 us for the
// x/y kernel, which forms two fluxes per thread, then 4 us for z and 2 us for the stage's
// linear combination). Here a block of 512 threads does all of it for a box of 8 x 4 x 4
// cells: the 464 faces of the three directions, one per thread. The box's points and their
// 3-deep halos are staged line by line, once per direction, with the velocities in
// direction-local order, so that every thread runs the same code whatever its face's
// direction. A Runge-Kutta stage's linear combination is formed while the points are loaded,
// and its value, or the step's, is stored by the cells' own threads. Faces and points are
// recomputed between boxes (464 against 384 faces, 608 points for 128 cells).
constexpr int BX = 8, BY = 4, BZ = 4, BCELLS = BX * BY * BZ;
constexpr int BPX = 15, BPY = 11;                       // padded lines of 14 and 10 points
constexpr int BOFY = BY * BZ * BPX, BOFZ = BOFY + BX * BZ * BPY, BFS = BOFZ + BX * BY * BPY;
constexpr int BNFX = BY * BZ * (BX + 1), BNFY = BX * BZ * (BY + 1), BNFZ = BX * BY * (BZ + 1);
constexpr int BNF = BNFX + BNFY + BNFZ;                 // 464
constexpr int BNP = BCELLS + 6 * (BY * BZ + BX * BZ + BX * BY);   // 608
static_assert(BNF <= 512 && 5 * BNF <= PT_NF * BFS, "one face per thread; fluxes over points");

// Point p of the staging of the box at (x0, y0, z0): its local coordinates, the cell it is
// read from, its signs, and which lines it belongs to.
struct BoxPoint {
  int lx, ly, lz, cell;
  double sa, sx, sy, sz;
  bool use, core, ox, oy, oz;
  __device__ bool in_x() const { return lx >= 0 && lx < BX; }
  __device__ bool in_y() const { return ly >= 0 && ly < BY; }
  __device__ bool in_z() const { return lz >= 0 && lz < BZ; }
  // on a line of the box along x, y, z, and its place in the staged field
  __device__ bool on_x() const { return in_y() && in_z() && !oy && !oz; }
  __device__ bool on_y() const { return in_x() && in_z() && !ox && !oz; }
  __device__ bool on_z() const { return in_x() && in_y() && !ox && !oy; }
  __device__ int at_x() const { return (ly + BY * lz) * BPX + lx + 3; }
  __device__ int at_y() const { return BOFY + (lx + BX * lz) * BPY + ly + 3; }
  __device__ int at_z() const { return BOFZ + (lx + BX * ly) * BPY + lz + 3; }
};

__device__ inline BoxPoint box_point(const Grid &g, int x0, int y0, int z0, int p) {
  BoxPoint P;
  // local coordinates: the box's cells, then the halos of the x, y and z lines
  if (p < BCELLS) {
    P.lx = p % BX; P.ly = p / BX % BY; P.lz = p / (BX * BY);
  } else if (p < BCELLS + 6 * BY * BZ) {
    const int q = p - BCELLS, h = q % 6;
    P.lx = h < 3 ? h - 3 : BX - 3 + h; P.ly = q / 6 % BY; P.lz = q / (6 * BY);
  } else if (p < BCELLS + 6 * (BY * BZ + BX * BZ)) {
    const int q = p - (BCELLS + 6 * BY * BZ), h = q / BX % 6;
    P.lx = q % BX; P.ly = h < 3 ? h - 3 : BY - 3 + h; P.lz = q / (6 * BX);
  } else {
    const int q = p - (BCELLS + 6 * (BY * BZ + BX * BZ)), h = q / (BX * BY);
    P.lx = q % BX; P.ly = q / BX % BY; P.lz = h < 3 ? h - 3 : BZ - 3 + h;
  }
  const int ex = x0 + P.lx, ey = y0 + P.ly, ez = z0 + P.lz;
  // which dimension the point lies outside the grid in: none, or one (a ghost of lines along
  // it); a point outside in two, or past the third ghost, is not used
  P.ox = ex < 0 || ex >= g.nx;
  P.oy = ey < 0 || ey >= g.ny;
  P.oz = ez < 0 || ez >= g.nz;
  P.use = p < BNP && P.ox + P.oy + P.oz <= 1 && ex <= g.nx + 2 && ey <= g.ny + 2 &&
          ez <= g.nz + 2;
  P.core = P.use && p < BCELLS && !P.ox && !P.oy && !P.oz;   // a cell of the box
  int i = ex, j = ey, k = ez;
  P.sa = P.sx = P.sy = P.sz = 1.0;
  if (P.ox) {
    const GhostMap m = ghost_map(g, 0, ex);
    i = m.src; P.sa = P.sy = P.sz = m.sgn_all; P.sx = m.sgn_norm;
  } else if (P.oy) {
    const GhostMap m = ghost_map(g, 1, ey);
    j = m.src; P.sa = P.sx = P.sz = m.sgn_all; P.sy = m.sgn_norm;
  } else if (P.oz) {
    const GhostMap m = ghost_map(g, 2, ez);
    k = m.src; P.sa = P.sx = P.sy = m.sgn_all; P.sz = m.sgn_norm;
  }
  P.cell = P.use ? i + g.nx * (j + g.ny * k) : 0;
  return P;
}

// With NC tracers (NT = 0) their faces follow, at most BTP tracers at a time: values of the
// points loaded before the previous fields' divergence, staged over the dead points, one flux
// per thread and tracer with the split factors kept from the fluid's face. ST and MODE as in
// fe_zface_tracers.
constexpr int BTP = 5;
template <int NT, int NC = 0, int ST = NC, int MODE = TR_PLAIN>
__global__ void __launch_bounds__(512, NC > 0 ? 1 : 2)
fe_box(Grid g, Fields y, BoxStage s, FieldsOut out, double idx, double idy, double idz,
       unsigned *flag, FeSlow slow) {
  __shared__ double sh[PT_NF * BFS];
  const int t = threadIdx.x;
  const int nbx = (g.nx + BX - 1) / BX, nby = (g.ny + BY - 1) / BY;
  int b = blockIdx.x;
  const int x0 = (b % nbx) * BX;
  b /= nbx;
  const int y0 = (b % nby) * BY, z0 = (b / nby) * BZ;
  const int ncell = g.nx * g.ny * g.nz;
  // all loads of the thread's one or two points are issued before any is used
  constexpr int NR = (BNP + 511) / 512;
  BoxPoint P[NR];
#pragma unroll
  for (int n = 0; n < NR; n++) P[n] = box_point(g, x0, y0, z0, t + 512 * n);
  double raw[NR][5], Kv[NR][NT > 0 ? NT : 1][5];
#pragma unroll
  for (int n = 0; n < NR; n++) {
    if (!P[n].use) continue;
#pragma unroll
    for (int q = 0; q < 5; q++) raw[n][q] = y.w[q][P[n].cell];
#pragma unroll
    for (int m = 0; m < NT; m++)
#pragma unroll
      for (int q = 0; q < 5; q++) Kv[n][m][q] = s.K[m][q * ncell + P[n].cell];
  }
#pragma unroll
  for (int n = 0; n < NR; n++) {
    const BoxPoint &Q = P[n];
    if (!Q.use) continue;
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int m = 0; m < NT; m++)
#pragma unroll
        for (int q = 0; q < 5; q++) raw[n][q] += s.c[m] * Kv[n][m][q];
    }
    if (Q.core && s.z) {
#pragma unroll
      for (int q = 0; q < 5; q++) s.z[q * ncell + Q.cell] = raw[n][q];
    }
    const double r = raw[n][0] * Q.sa, e = raw[n][4] * Q.sa;
    const double mx = raw[n][1] * Q.sx, my = raw[n][2] * Q.sy, mz = raw[n][3] * Q.sz;
    double pt[PT_NF];
    const double pr = store_point(pt, 1, r, mx, my, mz, e, g.gamma);
    if (Q.core) {
      unsigned bits = 0;
      if (!(r > 0.0)) bits |= 1u;
      if (!(e > 0.0)) bits |= 2u;
      if (!(pr > 0.0)) bits |= 4u;
      if (bits) atomicOr(flag, bits);
    }
    const auto put = [&](int at, double un, double u1, double u2) {
      double *d = sh + at;
      d[PT_R * BFS] = pt[PT_R]; d[PT_U * BFS] = un; d[PT_V * BFS] = u1; d[PT_W * BFS] = u2;
      d[PT_P * BFS] = pt[PT_P]; d[PT_SR * BFS] = pt[PT_SR]; d[PT_C2 * BFS] = pt[PT_C2];
      d[PT_C * BFS] = pt[PT_C];
    };
    if (Q.on_x()) put(Q.at_x(), pt[PT_U], pt[PT_V], pt[PT_W]);
    if (Q.on_y()) put(Q.at_y(), pt[PT_V], pt[PT_U], pt[PT_W]);
    if (Q.on_z()) put(Q.at_z(), pt[PT_W], pt[PT_V], pt[PT_U]);
  }
  __syncthreads();
  // face t: lines of BX + 1, BY + 1, BZ + 1 faces
  int at = 0;
  bool ok = false;
  if (t < BNFX) {
    const int f = t % (BX + 1), line = t / (BX + 1);
    at = line * BPX + f;
    ok = x0 + f <= g.nx && y0 + line % BY < g.ny && z0 + line / BY < g.nz;
  } else if (t < BNFX + BNFY) {
    const int q = t - BNFX, f = q % (BY + 1), line = q / (BY + 1);
    at = BOFY + line * BPY + f;
    ok = y0 + f <= g.ny && x0 + line % BX < g.nx && z0 + line / BX < g.nz;
  } else if (t < BNF) {
    const int q = t - (BNFX + BNFY), f = q % (BZ + 1), line = q / (BZ + 1);
    at = BOFZ + line * BPY + f;
    ok = z0 + f <= g.nz && x0 + line % BX < g.nx && y0 + line / BX < g.ny;
  }
  double F[5], hp[NC > 0 ? 5 : 1], hm[NC > 0 ? 5 : 1];
  if (ok) {
    const double alpha = face_alpha<PT_U>(sh + at, BFS, 1);
    face_flux_lds<PT_U, PT_V, PT_W>(sh + at, BFS, 1, g.gamma, g.igm, alpha, F);
    if constexpr (NC > 0) {
      double un[6];
#pragma unroll
      for (int l = 0; l < 6; l++) un[l] = sh[PT_U * BFS + at + l];
      tracer_split(un, alpha, hp, hm);
    }
  }
  // the first tracers' values, their latency under the fluid's divergence
  constexpr int NPASS = NC > 0 ? (NC + BTP - 1) / BTP : 0, TP = NC > 0 ? (NC + NPASS - 1) / NPASS : 1;
  double tv[NR][TP];
  const auto load_tracers = [&](int v0) {
#pragma unroll
    for (int n = 0; n < NR; n++)
#pragma unroll
      for (int v = 0; v < TP; v++)
        tv[n][v] = P[n].use && v0 + v < NC ? y.chem[(long)ST * P[n].cell + v0 + v] * P[n].sa : 0.0;
  };
  if constexpr (NC > 0) load_tracers(0);
  __syncthreads();                    // points dead: their LDS takes the fluxes [comp][face]
  if (ok) {
#pragma unroll
    for (int a = 0; a < 5; a++) sh[a * BNF + t] = F[a];
  }
  __syncthreads();
  // one value per thread and turn: field a of cell q
  for (int n = t; n < 5 * BCELLS; n += 512) {
    const int a = n / BCELLS, q = n % BCELLS;
    const int lx = q % BX, ly = q / BX % BY, lz = q / (BX * BY);
    if (x0 + lx >= g.nx || y0 + ly >= g.ny || z0 + lz >= g.nz) continue;
    const int ay = a == 1 ? 2 : a == 2 ? 1 : a, az = a == 1 ? 3 : a == 3 ? 1 : a;
    const double *Fx = sh + a * BNF + (ly + BY * lz) * (BX + 1) + lx;
    const double *Fy = sh + ay * BNF + BNFX + (lx + BX * lz) * (BY + 1) + ly;
    const double *Fz = sh + az * BNF + BNFX + BNFY + (lx + BX * ly) * (BZ + 1) + lz;
    const double dxy = (Fx[1] - Fx[0]) * idx + (Fy[1] - Fy[0]) * idy;
    double rate = 0.0 - (dxy + (Fz[1] - Fz[0]) * idz);
    const int c = (x0 + lx) + g.nx * ((y0 + ly) + g.ny * (z0 + lz));
    if (MODE != TR_PLAIN && a == 4) {
      const long rec = (long)ST * c + NC;
      out.chem[rec] = MODE == TR_SLOW_SCALED ? rate * slow.eunits / slow.scale[rec] : rate;
      rate = 0.0;
    }
    // (selected, not indexed: an index that is not constant would copy the arguments to
    // scratch memory)
    double *o = out.w[0];
    const double *ya = y.w[0];
#pragma unroll
    for (int m = 1; m < 5; m++)
      if (a == m) { o = out.w[m]; ya = y.w[m]; }
    o[c] = rate;
    if (s.y1) {
#pragma clang fp contract(off)
      double v = ya[c];
      for (int m = 0; m < s.nb; m++) v += s.b[m] * s.Kb[m][a * ncell + c];
      s.y1[a * ncell + c] = v + s.blast * rate;
    }
  }
  if constexpr (NC > 0) {
#pragma unroll 1
    for (int v0 = 0; v0 < NC; v0 += TP) {
      __syncthreads();                // the previous fluxes are read
#pragma unroll
      for (int n = 0; n < NR; n++) {
        const BoxPoint &Q = P[n];
        if (!Q.use) continue;
        const bool ox = Q.on_x(), oy = Q.on_y(), oz = Q.on_z();
#pragma unroll
        for (int v = 0; v < TP; v++) {
          if (ox) sh[v * BFS + Q.at_x()] = tv[n][v];
          if (oy) sh[v * BFS + Q.at_y()] = tv[n][v];
          if (oz) sh[v * BFS + Q.at_z()] = tv[n][v];
        }
      }
      __syncthreads();
      double Ft[TP];
      if (ok) {
#pragma unroll
        for (int v = 0; v < TP; v++) {
          double cv[6];
#pragma unroll
          for (int l = 0; l < 6; l++) cv[l] = sh[v * BFS + at + l];
          Ft[v] = tracer_face_flux(cv, hp, hm);
        }
      }
      if (v0 + TP < NC) load_tracers(v0 + TP);
      __syncthreads();                // the values are read
      if (ok) {
#pragma unroll
        for (int v = 0; v < TP; v++) sh[v * BNF + t] = Ft[v];
      }
      __syncthreads();
      for (int n = t; n < TP * BCELLS; n += 512) {
        const int v = n / BCELLS, q = n % BCELLS;
        const int lx = q % BX, ly = q / BX % BY, lz = q / (BX * BY);
        if (v0 + v >= NC || x0 + lx >= g.nx || y0 + ly >= g.ny || z0 + lz >= g.nz) continue;
        const double *Fx = sh + v * BNF + (ly + BY * lz) * (BX + 1) + lx;
        const double *Fy = sh + v * BNF + BNFX + (lx + BX * lz) * (BY + 1) + ly;
        const double *Fz = sh + v * BNF + BNFX + BNFY + (lx + BX * ly) * (BZ + 1) + lz;
        const double dxy = (Fx[1] - Fx[0]) * idx + (Fy[1] - Fy[0]) * idy;
        const double rate = 0.0 - (dxy + (Fz[1] - Fz[0]) * idz);
        const long rec = (long)ST * ((x0 + lx) + g.nx * ((y0 + ly) + g.ny * (z0 + lz))) + v0 + v;
        out.chem[rec] = MODE == TR_SLOW_SCALED ? rate / slow.scale[rec] : rate;
      }
    }
  }
}
static_assert(BTP <= PT_NF, "tracer values over point fields");

__global__ void reset_flag(unsigned *flag) { *flag = 0u; }

// ------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------

static inline unsigned nblocks(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// The flag at zero before a call, by a launch only where it is not known to be (33x31x17 cells
// with four tracers: 38.4 -> 36.4 us a call).
static void clear_flag(FeScratch &s, hipStream_t st) {
  if (!s.flag_zero) hipLaunchKernelGGL(reset_flag, dim3(1), dim3(1), 0, st, s.flag);
  s.flag_zero = false;
}

constexpr int TILE_X = 16, TILE_F = 16;   // fe_zface_tracers' tile

// the number of boxes
static long fe_boxes(const Grid &g) {
  return (long)((g.nx + BX - 1) / BX) * ((g.ny + BY - 1) / BY) * ((g.nz + BZ - 1) / BZ);
}

// NC tracers in records of ST doubles
template <int NC, int ST = NC, int MODE = TR_PLAIN>
static int launch_fe(const Grid &g, const Fields &f, const FieldsOut &o, FeScratch &s,
                     hipStream_t st, bool plain, unsigned *accum, const FeSlow &slow = {}) {
  const long nxp = g.nx + 1, nyp = g.ny + 1, nzp = g.nz + 1;
  unsigned *const flag = accum ? accum : s.flag;
  if (!accum) clear_flag(s, st);
  KernelTimer &tm = s.timer;
  if constexpr (NC > 0) if (!plain && !(tm.on && tm.faces) && fe_boxes(g) <= FE_BOX_TRACER_MAX) {
    tm.begin(PROF_FE_BOX, st);
    hipLaunchKernelGGL((fe_box<0, NC, ST, MODE>), dim3((unsigned)fe_boxes(g)), dim3(512), 0, st, g,
                       f, BoxStage{}, o, 1.0 / g.dx, 1.0 / g.dy, 1.0 / g.dz, flag, slow);
    tm.end(PROF_FE_BOX, st);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  if constexpr (MODE == TR_PLAIN) if (plain) {
    tm.begin(PROF_PLAIN_FACES, st);
    hipLaunchKernelGGL(fe_plain_faces<NC>, dim3(nblocks(nxp * nyp * nzp, 256)), dim3(256), 0, st,
                       g, f, s.Fx, s.Fy, s.Fz, flag);
    tm.end(PROF_PLAIN_FACES, st);
    tm.begin(PROF_PLAIN_DIV, st);
    hipLaunchKernelGGL(fe_plain_div<NC>, dim3(nblocks((long)g.nx * g.ny * g.nz, 256)), dim3(256),
                       0, st, g, s.Fx, s.Fy, s.Fz, o);
    tm.end(PROF_PLAIN_DIV, st);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  // x and y faces of each plane tile (fluid, then the tracers) in one kernel, then the z
  // faces adding their part
  constexpr int TX = TILE_X, TF = TILE_F;
  const long nxc = (g.nx + TX - 1) / TX;
  const long nxyb = ((long)(g.nx + XY_TX - 1) / XY_TX) * ((g.ny + XY_TY - 1) / XY_TY) * g.nz;
  tm.begin(PROF_XYFACE_DIV, st);
  hipLaunchKernelGGL((fe_xyface_div<NC, ST>), dim3((unsigned)nxyb), dim3(256), 0, st, g, f, o,
                     1.0 / g.dx, 1.0 / g.dy, flag);
  tm.end(PROF_XYFACE_DIV, st);
  tm.begin(PROF_ZFACE_DIV, st);
  // column segments: whole columns when they fill the device with four blocks per CU, else
  // as many segments (of 16 m - 1 cells, the cells between 16 m faces) as that takes
  const long want = (4L * 256 + nxc * g.ny - 1) / (nxc * g.ny);
  const int zlen = ZC * (int)(((g.nz + want - 1) / want + ZC) / ZC) - 1;
  const int nseg = (g.nz + zlen - 1) / zlen;
  hipLaunchKernelGGL(fe_zface_div_xy, dim3((unsigned)(nxc * nseg * g.ny)), dim3(256), 0, st, g,
                     f, o, 1.0 / g.dz, nseg, zlen);
  if constexpr (NC > 0)
    hipLaunchKernelGGL((fe_zface_tracers<NC, ST, MODE>),
                       dim3((unsigned)(nxc * ((g.nz + TF - 2) / (TF - 1)) * g.ny)),
                       dim3(TX * TF), 0, st, g, f, o, 1.0 / g.dz, slow);
  tm.end(PROF_ZFACE_DIV, st);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// 32-bit cell indices in the fast kernels
static bool fe_too_large(const Grid &g) {
  return (long)(g.nx + 1) * (g.ny + 1) * (g.nz + 1) >= (1L << 31) / 16;
}

int fe_slow_launch(const Grid &g, const Fields &f, const FieldsOut &o, FeScratch &s,
                   hipStream_t st, unsigned *accum, const FeSlow &slow) {
  if (fe_too_large(g) || g.nchem != 10) return -2;
  return slow.scale ? launch_fe<9, 10, TR_SLOW_SCALED>(g, f, o, s, st, false, accum, slow)
                    : launch_fe<9, 10, TR_SLOW>(g, f, o, s, st, false, accum, slow);
}

bool fe_box_fits(const Grid &g) {
  return g.nchem == 0 && (long)g.nx * g.ny * g.nz <= FE_BOX_MAX;
}

int fe_box_launch(const Grid &g, const Fields &y, const BoxStage &bs, const FieldsOut &o,
                  hipStream_t st, unsigned *flag) {
  const long nb = fe_boxes(g);
  const auto kern = bs.nt == 0   ? fe_box<0>
                    : bs.nt == 1 ? fe_box<1>
                    : bs.nt == 2 ? fe_box<2>
                    : bs.nt == 3 ? fe_box<3>
                    : bs.nt == 4 ? fe_box<4>
                                 : fe_box<5>;
  hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(512), 0, st, g, y, bs, o, 1.0 / g.dx,
                     1.0 / g.dy, 1.0 / g.dz, flag, FeSlow{});
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fe_launch(const Grid &g, const Fields &f, const FieldsOut &o, FeScratch &s,
              hipStream_t st, bool plain, unsigned *accum) {
  if (fe_too_large(g)) return -2;
  if (!plain && fe_box_fits(g) && !(s.timer.on && s.timer.faces)) {
    if (!accum) clear_flag(s, st);
    s.timer.begin(PROF_FE_BOX, st);
    const int rc = fe_box_launch(g, f, BoxStage{}, o, st, accum ? accum : s.flag);
    s.timer.end(PROF_FE_BOX, st);
    return rc;
  }
  switch (g.nchem) {
    case 0: return launch_fe<0>(g, f, o, s, st, plain, accum);
    case 1: return launch_fe<1>(g, f, o, s, st, plain, accum);
    case 2: return launch_fe<2>(g, f, o, s, st, plain, accum);
    case 4: return launch_fe<4>(g, f, o, s, st, plain, accum);
    case 6: return launch_fe<6>(g, f, o, s, st, plain, accum);
    case 10: return launch_fe<10>(g, f, o, s, st, plain, accum);
    default: return -2;
  }
}

bool fe_nchem_supported(int nchem) {
  return nchem == 0 || nchem == 1 || nchem == 2 || nchem == 4 || nchem == 6 || nchem == 10;
}

}  // namespace mvd
