// Fixed-step explicit Runge-Kutta evolution of fEuler on the device: the path of the
// fluid driver with an explicit table and a fixed step (euler3D_main.cpp:194 ARKStepCreate
// with fEuler explicit, :209 ARKStepSetOrder, :280 ARKStepSetFixedStep). ARKStep's stage
// loop (SUNDIALS 6.2.0 arkode_erkstep.c; not in the reference tree) is restated:
//   z_i = y_n + sum_{j<i} (h a_ij) F_j,  F_i = fe(z_i),  y_{n+1} = y_n + sum_i (h b_i) F_i.
// The state, the stage state and the stage derivatives live in contiguous device blocks
// ([rho][mx][my][mz][et][chem], the ManyVector's subvectors back to back). The steps are
// queued on the caller's stream, one after another, without waiting; the legal-state bits of
// every stage are OR-ed into one word that is read back once, after the last step.
//
// Grids that fe_box takes run a stage in one launch, its linear combination included; the
// last stage also forms the new state (into a second state buffer, since neighbouring boxes
// still read the old one). Other grids run fe()'s kernels, with every stage combination one
// fused kernel over the whole vector.
//
// Tables whose last stage is taken at the new state (last row of A equal to b, and so b_s =
// 0, as Bogacki-Shampine's): the stage value is y_{n+1} itself, bit for bit, and the rate
// found there is the next step's first one, which is not evaluated a second time.
//
// Sod, 128x3x3 cells, 200 steps of Bogacki-Shampine 3 (three launches a step): 10.7 -> 4.8 ms
// (before: twelve kernels a step, replayed as a graph); 64^3, ten steps: 2.2 -> 1.3 ms.
#include "mvd_internal.hpp"

namespace mvd {

namespace {

// z = y + sum_{j<nt} c_j K_j
struct Coefs { double c[ERK_MAXSTAGE]; };
struct StagePtrs { const double *K[ERK_MAXSTAGE]; };

__global__ void __launch_bounds__(256)
mv_lincomb(long len, const double *y, int nt, Coefs c, StagePtrs p, double *z) {
#pragma clang fp contract(off)
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= len) return;
  double acc = y[i];
  for (int j = 0; j < nt; j++) acc += c.c[j] * p.K[j][i];
  z[i] = acc;
}

__global__ void zero_flag(unsigned *dst) { *dst = 0u; }

inline Fields fields_at(const double *base, long ncell, int nchem) {
  Fields f;
  for (int q = 0; q < 5; q++) f.w[q] = base + q * ncell;
  f.chem = nchem > 0 ? base + 5 * ncell : nullptr;
  return f;
}

inline FieldsOut fields_out_at(double *base, long ncell, int nchem) {
  FieldsOut f;
  for (int q = 0; q < 5; q++) f.w[q] = base + q * ncell;
  f.chem = nchem > 0 ? base + 5 * ncell : nullptr;
  return f;
}

// last row of A equal to b: the last stage's state is the new one
bool fsal(const ErkTable &tab) {
  const int s = tab.stages;
  if (s < 2 || tab.b[s - 1] != 0.0) return false;
  for (int j = 0; j < s - 1; j++)
    if (tab.A[(s - 1) * ERK_MAXSTAGE + j] != tab.b[j]) return false;
  return true;
}

}  // namespace

void erk_free(ErkState &e) {
  if (e.Y[0]) (void)hipFree(e.Y[0]);
  if (e.flag) (void)hipFree(e.flag);
  e = ErkState{};
}

int erk_evolve(const Grid &g, FeScratch &fe, ErkState &e, const ErkTable &tab, double h,
               int nsteps, const Fields &w_in, const FieldsOut &w_out, hipStream_t st,
               unsigned *host_flag) {
  const long ncell = (long)g.nx * g.ny * g.nz;
  const long len = (5L + g.nchem) * ncell;
  const unsigned nb = (unsigned)((len + 255) / 256);
  if (!e.Y[0]) {
    if (hipMalloc(&e.Y[0], sizeof(double) * len * (3 + ERK_MAXSTAGE)) != hipSuccess ||
        hipMalloc(&e.flag, sizeof(unsigned)) != hipSuccess) {
      erk_free(e);                          // (all or nothing: the next call tries again)
      return -1;
    }
    e.Y[1] = e.Y[0] + len;
    e.Z = e.Y[1] + len;
    e.K = e.Z + len;
  }
  // state in
  for (int q = 0; q < 5; q++)
    if (hipMemcpyAsync(e.Y[0] + q * ncell, w_in.w[q], sizeof(double) * ncell,
                       hipMemcpyDeviceToDevice, st) != hipSuccess)
      return -1;
  if (g.nchem > 0 &&
      hipMemcpyAsync(e.Y[0] + 5 * ncell, w_in.chem, sizeof(double) * g.nchem * ncell,
                     hipMemcpyDeviceToDevice, st) != hipSuccess)
    return -1;
  hipLaunchKernelGGL(zero_flag, dim3(1), dim3(1), 0, st, e.flag);
  const bool timer_on = fe.timer.on;
  fe.timer.on = false;                      // the kernel timer covers fe() calls only
  const int S = tab.stages;
  const bool last_is_new = fsal(tab), box = fe_box_fits(g);
  // stage derivative j's buffer; with last_is_new the first and the last change places from
  // step to step
  bool swap = false;
  const auto K = [&](int j) {
    if (last_is_new && swap) j = j == 0 ? S - 1 : j == S - 1 ? 0 : j;
    return e.K + (long)j * len;
  };
  int rc = 0, cur = 0;
  for (int n = 0; n < nsteps && rc == 0; n++) {
    double *const Y = e.Y[cur], *const Y1 = e.Y[1 - cur];
    const Fields fy = fields_at(Y, ncell, g.nchem);
    bool stored = false;                    // Y1 holds the new state
    for (int i = last_is_new && n > 0 ? 1 : 0; i < S && rc == 0; i++) {
      const bool last = i == S - 1, to_new = last && last_is_new;
      const FieldsOut ki = fields_out_at(K(i), ncell, g.nchem);
      Coefs c{};
      for (int j = 0; j < i; j++) c.c[j] = h * tab.A[i * ERK_MAXSTAGE + j];
      if (box) {
        BoxStage b;
        b.nt = i;
        for (int j = 0; j < i; j++) {
          b.K[j] = K(j);
          b.c[j] = c.c[j];
        }
        if (to_new) b.z = Y1;
        else if (last) {
          b.nb = S - 1;
          for (int j = 0; j < S - 1; j++) {
            b.Kb[j] = K(j);
            b.b[j] = h * tab.b[j];
          }
          b.blast = h * tab.b[S - 1];
          b.y1 = Y1;
        }
        stored = last;
        rc = fe_box_launch(g, fy, b, ki, st, e.flag);
        continue;
      }
      double *const Z = to_new ? Y1 : e.Z;
      if (i > 0) {
        StagePtrs p{};
        for (int j = 0; j < i; j++) p.K[j] = K(j);
        hipLaunchKernelGGL(mv_lincomb, dim3(nb), dim3(256), 0, st, len, (const double *)Y, i, c, p,
                           Z);
      }
      stored = to_new;
      // the stage's legal-state bits go straight into the run's flag
      rc = fe_launch(g, i > 0 ? fields_at(Z, ncell, g.nchem) : fy, ki, fe, st, false, e.flag);
    }
    if (rc) break;
    if (!stored) {
      Coefs c{};
      StagePtrs p{};
      for (int j = 0; j < S; j++) {
        c.c[j] = h * tab.b[j];
        p.K[j] = K(j);
      }
      hipLaunchKernelGGL(mv_lincomb, dim3(nb), dim3(256), 0, st, len, (const double *)Y, S, c, p,
                         Y1);
    }
    cur = 1 - cur;
    swap = !swap;
  }
  fe.timer.on = timer_on;
  if (rc) return rc;
  if (hipGetLastError() != hipSuccess) return -1;
  // state out, flag back
  for (int q = 0; q < 5; q++)
    if (hipMemcpyAsync(w_out.w[q], e.Y[cur] + q * ncell, sizeof(double) * ncell,
                       hipMemcpyDeviceToDevice, st) != hipSuccess)
      return -1;
  if (g.nchem > 0 &&
      hipMemcpyAsync(w_out.chem, e.Y[cur] + 5 * ncell, sizeof(double) * g.nchem * ncell,
                     hipMemcpyDeviceToDevice, st) != hipSuccess)
    return -1;
  if (hipMemcpyAsync(host_flag, e.flag, sizeof(unsigned), hipMemcpyDeviceToHost, st) !=
          hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return -1;
  return 0;
}

}  // namespace mvd
