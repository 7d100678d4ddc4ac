// Internal (non-ABI) declarations shared by the kernel translation units and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include "mvd_device.hpp"

namespace mvd {

struct Fields {
  const double *w[5];   // rho, mx, my, mz, et
  const double *chem;   // species, AoS [cell][nchem] (may be null when nchem == 0)
};

struct FieldsOut {
  double *w[5];
  double *chem;
};

// Kernel timing slots (HIP events recorded on the launch stream around each kernel).
// (slots 0 and 1 are unused; the numbering is part of mvd_profile_read's interface)
enum { PROF_UNUSED0 = 0, PROF_UNUSED1, PROF_ZFACE_DIV, PROF_PLAIN_FACES, PROF_PLAIN_DIV,
       PROF_XYFACE_DIV, PROF_FE_BOX, PROF_NSLOT };

struct KernelTimer {
  bool on = false;
  bool faces = false;        // while on: fe() by its face kernels on every grid (no fe_box)
  hipEvent_t ev[2 * PROF_NSLOT] = {};
  bool pending[PROF_NSLOT] = {};
  double ms[PROF_NSLOT] = {};
  long count[PROF_NSLOT] = {};
  void begin(int slot, hipStream_t st) {
    if (on) (void)hipEventRecord(ev[2 * slot], st);
  }
  void end(int slot, hipStream_t st) {
    if (on) { (void)hipEventRecord(ev[2 * slot + 1], st); pending[slot] = true; }
  }
  // after the stream has been synchronized
  void collect() {
    if (!on) return;
    for (int s = 0; s < PROF_NSLOT; s++) {
      if (!pending[s]) continue;
      float t = 0.f;
      if (hipEventElapsedTime(&t, ev[2 * s], ev[2 * s + 1]) == hipSuccess) {
        ms[s] += t;
        count[s] += 1;
      }
      pending[s] = false;
    }
  }
};

// Device scratch owned by the context (EulerData keeps xflux/yflux/zflux for the same
// purpose, euler3D.hpp:496-499).
struct FeScratch {
  double *Fx = nullptr, *Fy = nullptr, *Fz = nullptr;   // face fluxes, [component][face]
  unsigned *flag = nullptr;                             // legal-state bits of the last call
  // The flag is known to be zero: the last call waited for its kernels and read it so. Never
  // again once fe() has been queued without waiting (async_used): such a call may sit in a
  // graph that writes the flag whenever it is replayed.
  bool flag_zero = false, async_used = false;
  double *red = nullptr;                                // reduction partials
  long red_len = 0;
  KernelTimer timer;
};

// accum: when not null, the legal-state bits are OR-ed into *accum (a stage loop's running
// flag) instead of into the scratch flag, which is then neither reset nor written.
int fe_launch(const Grid &g, const Fields &f, const FieldsOut &o, FeScratch &s,
              hipStream_t st, bool plain, unsigned *accum = nullptr);
bool fe_nchem_supported(int nchem);
// fe() as the slow right-hand side takes it (records of 10 species): the gas energy is not
// advected as a tracer (its slot's rate is overwritten), the total-energy rate goes into its
// slot of o.chem and o.w[4] becomes 0. With a scale ([cell][10]) the record is converted to
// the scaled variables: species rates divided by their scale, the energy rate times eunits
// divided by the gas energy's.
struct FeSlow {
  const double *scale = nullptr;
  double eunits = 1.0;
};
int fe_slow_launch(const Grid &g, const Fields &f, const FieldsOut &o, FeScratch &s,
                   hipStream_t st, unsigned *accum, const FeSlow &slow);

// fe() of a small grid without tracers in one launch (fe_box). With nt > 0 the state it is
// taken at is y + sum_n c[n] K[n] (summed in order; K as contiguous [field][cell] blocks);
// z (nullable) receives that state, y1 (nullable) the vector y + sum_m b[m] Kb[m] + blast *
// rate. z and y1 must not be read by the same launch.
constexpr int BOX_TERMS = 5;
struct BoxStage {
  int nt = 0, nb = 0;
  const double *K[BOX_TERMS] = {}, *Kb[BOX_TERMS] = {};
  double c[BOX_TERMS] = {}, b[BOX_TERMS] = {}, blast = 0.0;
  double *z = nullptr, *y1 = nullptr;
};
// Largest grid it is taken for: fe() of 40^3 cells 38.4 us against 43.4 with the x/y and z
// kernels, 48^3 46.2 / 48.3, 56^3 54.8 / 55.8, 64^3 62.1 / 59.4 (its boxes recompute a fifth
// of the faces and load every point five times).
constexpr long FE_BOX_MAX = 50 * 50 * 50;
// With tracers, the most boxes: two per CU. fe() of 32^3 cells (256 boxes) with four tracers 39.0
// us against 49.6 with the three kernels, with ten 42.8 / 56.5 (fslow 47.8 / 61.8); 40^3 (500
// boxes) with ten 56.8 / 68.5; 48^3 (864) with four 65.4 / 66.7, with ten 81.6 / 80.3.
constexpr long FE_BOX_TRACER_MAX = 512;
bool fe_box_fits(const Grid &g);
int fe_box_launch(const Grid &g, const Fields &y, const BoxStage &bs, const FieldsOut &o,
                  hipStream_t st, unsigned *flag);

// CFL wave speed: max over cells of |mx/rho| + c (stability, utilities.cpp:483-528).
int max_wave_speed_launch(const Grid &g, const Fields &f, FeScratch &s, hipStream_t st,
                          double *host_out);

// fslow (multirate_chem_hydro_main.cpp:996-1083), queued: et of w rebuilt from the gas energy,
// wdot its rates; converted: the chemistry rates in the scaled variables (as FeSlow). accum as
// for fe_launch. Returns 0, -2 (unsupported grid) or -1.
int fslow_launch(const Grid &g, double *const *w, double *const *wdot, const double *scale,
                 double eunit_inv, bool converted, FeScratch &s, hipStream_t st,
                 unsigned *accum = nullptr);
// PostprocessStep (imex_chem_hydro_main.cpp:1002-1050): et from the gas energy, and the
// chemistry through its scaling and back (x * s / s)
int postprocess_launch(const Grid &g, double *const *w, const double *scale, double eunit_inv,
                       hipStream_t st);
int chem_scale_launch(long n, double *chem, const double *scale, int apply, hipStream_t st);
// N_VConst: z[0..len) = c
int const_launch(double c, double *z, long len, hipStream_t st);

// fe() vector-Jacobian product (fe_vjp.hip); buf holds fe_vjp_buffer_doubles(g) doubles
size_t fe_vjp_buffer_doubles(const Grid &g);
int fe_vjp_launch(const Grid &g, const Fields &w, const Fields &v, const FieldsOut &out,
                  double *buf, hipStream_t st);

// N_Vector operations (nvec.hip)
constexpr int LC_MAX = 16;        // vectors per linear-combination launch
constexpr int WRMS_MAXSUB = 8;    // subvectors per WRMS norm
// ghost exchange buffers (W, E, S, N, B, F; null entries skipped) and stencil packs
int exchange_launch(const Grid &g, const Fields &f, double *const *recv, hipStream_t st);
int pack1d_launch(const Grid &g, const Fields &f, int d, long ncell, const int *ijk,
                  double *out, int *scratch, hipStream_t st, int *host_bad);

// y = 1 y + a x, nsteps times in turn (one launch)
int axpy_steps_launch(int nsteps, double a, const double *x, double *y, long len,
                      hipStream_t st);
int linear_combination_launch(int nv, const double *c, const double *const *X, double *z,
                              long len, hipStream_t st);
int wrms_norm_launch(int nsub, const double *const *x, const double *const *w, const long *len,
                     FeScratch &s, hipStream_t st, double *host_out);

// fixed-step explicit Runge-Kutta evolution of fe() (erk.hip)
constexpr int ERK_MAXSTAGE = 6;
struct ErkTable {
  int stages = 0;
  double A[ERK_MAXSTAGE * ERK_MAXSTAGE] = {};
  double b[ERK_MAXSTAGE] = {}, c[ERK_MAXSTAGE] = {};
};
struct ErkState {
  double *Y[2] = {}, *Z = nullptr, *K = nullptr;     // one allocation: Y_0, Y_1, Z, K_0..K_5
  unsigned *flag = nullptr;
};
int erk_evolve(const Grid &g, FeScratch &fe, ErkState &e, const ErkTable &tab, double h,
               int nsteps, const Fields &w_in, const FieldsOut &w_out, hipStream_t st,
               unsigned *host_flag);
void erk_free(ErkState &e);

}  // namespace mvd
