// One diagonally implicit RK step of the per-cell primordial chemistry (the fast implicit
// stage of the reacting-flow demo), two ways:
//
//   batched  - one persistent launch. Each wave pulls chunks of up to 64 cells from an atomic
//              work queue (work stealing across waves and CUs: cells need 3 to 9+ Newton
//              iterations) and each lane runs all stages and Newton iterations of its cell:
//              RHS with the temperature solve, analytic Jacobian, M = I - h a_ii s J, 10x10
//              LU with partial pivoting, triangular solves, WRMS convergence test, re-setup
//              after max_iters. The iterate and the LU factors stay in the register file for
//              the whole step (one wave per SIMD: 512 VGPR + AGPR); what is read once per
//              pass or stage is in LDS. Statistics are accumulated per block in LDS.
//   plain    - the reference's structure (primordial_ode_main.cpp with SUNDIALS + MAGMA):
//              one-thread-per-cell kernels for the RHS, the Jacobian into column-major 10x10
//              blocks, the batched LU factorisation, and the Newton update with the
//              triangular solves, the iterate and stage values in global memory, and a host
//              round trip per Newton iteration to test convergence.
//
// Both follow the same per-cell algorithm (stage predictor, modified Newton with the
// Jacobian from y_n, whose RHS evaluation is also the first iteration's, re-setup after
// max_iters) and share their arithmetic, so they agree with each other bitwise and with the
// CPU oracle iteration for iteration.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include "mvd_chem.hpp"
#include "mvd_dirk.hpp"
#include "../../include/mvd_rhs.h"

namespace mvd {

// Per-cell inputs: scale factors at sc[s*st] / isc[s*st] (st = 1 for the per-cell AoS
// arrays, 64 for the element-major chunk block) and the cell's auxiliary values.
struct CellIn {
  const double *sc, *isc;
  long st;
  CellAux ax;
  __device__ double s(int k) const { return sc[k * st]; }
  __device__ double is(int k) const { return isc[k * st]; }
};

__device__ inline CellIn load_cell(const ChemPtrsD &p, long i) {
  return CellIn{p.scale + NSP * i, p.iscale + NSP * i, 1,
                CellAux{p.md[i], p.imd[i], p.cie[i], p.h2o[i]}};
}

// calculate_rhs_cvklu for one cell in scaled variables, times srhs; updates Ts/dTs. The
// temperature solve reads the gamma tables from gt (global memory or an LDS copy).
// With solve_t false, Ts/dTs already hold the solution at y and the solve is skipped.
// PAIRS: the rates come from the bin-major pair table (same values), or, where the caller
// keeps a RateBin, from the lane's copy of its bin.
constexpr int RATE_BATCH = 25;        // pairs per wait: each group of tables at once
struct NoRateBin {
  static constexpr bool on = false, pairs = false;
};
struct PairTable : NoRateBin {         // the matrix, too, from the bin-major pairs
  static constexpr bool pairs = true;
};

// The pairs of the table bin a lane's temperature lies in, copied to LDS: pair r at
// row[64 r], bin -1 when none is held. From one Newton iteration to the next the bin (1.1%
// of T wide) hardly ever changes, and a read back costs 46 conflict-free 16-byte LDS loads
// instead of as many gathers of up to 64 lines each.
struct RateBin {
  static constexpr bool on = true, pairs = false;
  double2 *row;
  int bin;
  __device__ void hold(const ChemConst &cc, int b) {
    if (b == bin) return;
    bin = b;
    const double2 *src = cc.tabp + (long)b * NRATE;
    constexpr int PART = NRATE / 2;
    static_assert(2 * PART == NRATE, "two parts");
    copy<0, PART>(src);
    __asm__ volatile("" ::: "memory");                     // bounds the loads in flight
    copy<PART, NRATE>(src);
  }
  template <int R0, int R1>
  __device__ void copy(const double2 *src) {
    double a[R1 - R0], b[R1 - R0];
#pragma unroll
    for (int r = R0; r < R1; r++) {
      const double2 v = src[r];
      a[r - R0] = v.x;
      b[r - R0] = v.y;
    }
#pragma unroll
    for (int r = R0; r < R1; r++) row[r * 64] = make_double2(a[r - R0], b[r - R0]);
  }
};

template <bool PAIRS = false, class Bin>
__device__ inline void cell_rhs(const ChemConst &cc, const GammaTabs &gt, const CellIn &c,
                                double &Ts, double &dTs, const double (&y)[NSP], double srhs,
                                double (&f)[NSP], bool solve_t, Bin &rb) {
#pragma clang fp contract(on)
  double ya[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) ya[s] = y[s] * c.s(s);
  if (solve_t) chem_temperature_near(cc, gt, ya, Ts, dTs);
  // species rows from the reaction tables, then the energy row from the cooling tables;
  // the fence keeps the two groups of table loads from being scheduled together
  double k[NRATE];
#pragma unroll
  for (int r = 0; r < NRATE; r++) k[r] = 0.0;
  double Tdef = 0.0;
  const double2 *pairs = nullptr;
  if constexpr (Bin::on) {
    rb.hold(cc, chem_locate(cc, chem_log(Ts), Tdef));
    chem_rates_only_batch<0, C_BREM, 64, RATE_BATCH>(rb.row, Tdef, k);
  } else if (PAIRS) {
    pairs = cc.tabp + (long)chem_locate(cc, chem_log(Ts), Tdef) * NRATE;
    chem_rates_only_batch<0, C_BREM, 1, RATE_BATCH>(pairs, Tdef, k);
  }
  else chem_rates_only_range<0, C_BREM>(cc, Ts, k);
  chem_rhs_species(ya, k, f);
  __asm__ volatile("" ::: "memory");
  if constexpr (Bin::on) chem_rates_only_batch<C_BREM, NRATE, 64, RATE_BATCH>(rb.row, Tdef, k);
  else if (PAIRS) chem_rates_only_batch<C_BREM, NRATE, 1, RATE_BATCH>(pairs, Tdef, k);
  else chem_rates_only_range<C_BREM, NRATE>(cc, Ts, k);
  f[9] = chem_rhs_energy(ya, k, Ts, cc.z, c.ax);
#pragma unroll
  for (int s = 0; s < NSP; s++) f[s] *= c.is(s);
  f[9] *= c.ax.inv_mdensity;
#pragma unroll
  for (int s = 0; s < NSP; s++) f[s] *= srhs;
}

template <bool PAIRS = false>
__device__ inline void cell_rhs(const ChemConst &cc, const GammaTabs &gt, const CellIn &c,
                                double &Ts, double &dTs, const double (&y)[NSP], double srhs,
                                double (&f)[NSP], bool solve_t = true) {
  NoRateBin none;
  cell_rhs<PAIRS>(cc, gt, c, Ts, dTs, y, srhs, f, solve_t, none);
}

template <bool PAIRS = false>
__device__ inline void cell_rhs(const ChemConst &cc, const CellIn &c, double &Ts, double &dTs,
                                const double (&y)[NSP], double srhs, double (&f)[NSP]) {
  cell_rhs<PAIRS>(cc, gamma_tabs(cc), c, Ts, dTs, y, srhs, f);
}

// Packed pivots of a factorisation without row exchanges (pivot k at step k).
constexpr unsigned long long PIV_IDENTITY = 0x9876543210ULL;

// LU with partial pivoting (first maximum wins, LAPACK getrf row interchanges) with the
// whole matrix in registers (right-looking, predicated row exchanges so that the runtime
// pivot never indexes a register array; a column in which no lane of the wave pivots skips
// them, 1800 selects in all). Returns the pivots packed 4 bits each.
// INVD (the Newton solvers' form): FMA updates, fast_rcp pivots, and the diagonal of U left
// as its reciprocals for lu_solve_regs. Without it: LAPACK's separate products and IEEE
// reciprocals, which meet an exact zero pivot (a singular block) as its getrf would.
template <bool INVD>
__device__ inline unsigned long long lu_factor_regs(double (&a)[NSP][NSP]) {
#pragma clang fp contract(off)
  unsigned long long pv = 0;
#pragma unroll
  for (int k = 0; k < NSP; k++) {
    int p = k;
    double best = fabs(a[k][k]);
#pragma unroll
    for (int r = k + 1; r < NSP; r++) {
      const double v = fabs(a[r][k]);
      if (v > best) { best = v; p = r; }
    }
    pv |= (unsigned long long)p << (4 * k);
    if (p != k) {
#pragma unroll
      for (int r = k + 1; r < NSP; r++) {
        const bool sw = (r == p);
#pragma unroll
        for (int q = 0; q < NSP; q++) {
          const double x = a[k][q], y = a[r][q];
          a[k][q] = sw ? y : x;
          a[r][q] = sw ? x : y;
        }
      }
    }
    const double ik = INVD ? fast_rcp(a[k][k]) : 1.0 / a[k][k];
#pragma unroll
    for (int r = k + 1; r < NSP; r++) {
      const double l = a[r][k] * ik;
      a[r][k] = l;
#pragma unroll
      for (int q = k + 1; q < NSP; q++)
        a[r][q] = INVD ? fma(-l, a[k][q], a[r][q]) : a[r][q] - l * a[k][q];
    }
    if (INVD) a[k][k] = ik;
  }
  return pv;
}

// b's rows exchanged as step k of the factorisation exchanged the matrix's, and as all steps did
__device__ inline void lu_exchange(unsigned long long pv, int k, double (&b)[NSP]) {
  const int p = (int)((pv >> (4 * k)) & 15);
#pragma unroll
  for (int r = k + 1; r < NSP; r++) {
    const bool sw = (r == p);
    const double bk = b[k], br = b[r];
    b[k] = sw ? br : bk;
    b[r] = sw ? bk : br;
  }
}

__device__ inline void lu_exchange(unsigned long long pv, double (&b)[NSP]) {
#pragma unroll
  for (int k = 0; k < NSP; k++) lu_exchange(pv, k, b);
}

__device__ inline double wrms_norm(const double (&d)[NSP], const double (&z)[NSP],
                                   double rtol, double atol) {
#pragma clang fp contract(on)
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < NSP; k++) {
    const double w = d[k] * fast_rcp(rtol * fabs(z[k]) + atol);
    s += w * w;
  }
  return sqrt(s * (1.0 / NSP));
}

// ARKODE's Newton convergence test (arkStep_NlsConvTest, ARKODE 5.2 / SUNDIALS 6.2.0, the
// version the reference builds against): with del the WRMS norm of the correction
// (weights of the updated iterate, as wrms_norm; ARKODE weighs by the step start, with which
// fast steps of the multirate blast fail where a species starts near zero) and m the
// iteration of the stage solve (0 first), the rate
// estimate crate = max(0.3 crate, del / del_prev) for m > 0 (1 after every setup, carried
// from stage to stage); converged when min(crate, 1) del / tol <= 1; diverging, handled as
// a failed iteration budget, when m > 0 and del > 2.3 del_prev.
__device__ inline double conv_rate(double crate, double del, double delp) {
  const double a = 0.3 * crate, b = del / delp;
  return a > b ? a : b;
}

__device__ inline bool conv_ok(double crate, double del, double tol) {
#pragma clang fp contract(on)
  return (crate < 1.0 ? crate : 1.0) * del <= tol;
}

__device__ inline bool conv_diverging(double del, double delp) {
#pragma clang fp contract(on)
  return del > 2.3 * delp;
}

// a_{st,j} for a stage index held per lane, with constant indices only (no dynamic indexing
// of the by-value argument): selected among the rows 1..QMAX-1 (QMAX: the most stages the
// caller's kernel handles)
template <int QMAX = MAXSTAGE>
__device__ inline double dirk_coef(const DirkDev &o, int st, int j) {
  double v = 0.0;
#pragma unroll
  for (int q = 1; q < QMAX; q++)
    if (q == st) v = o.A[q * MAXSTAGE + j];
  return v;
}

// ------------------------------------------------------------------------------------
// statistics: per-wave partial rows, summed by one block at the end (no same-address
// atomics on the hot path)
// ------------------------------------------------------------------------------------

// Per-lane accumulators and the wave's histogram (uniform) of one wave.
struct WaveStats {
  int iters = 0, maxit = 0, failed = 0, setups = 0;
  int hist[NHIST] = {};
  // called by the lanes that finished a cell (the others inactive)
  __device__ void add(int nit, int nsetup, bool fail) {
    iters += nit;
    maxit = nit > maxit ? nit : maxit;
    failed += fail ? 1 : 0;
    setups += nsetup;
    const int bin = nit < NHIST - 1 ? nit : NHIST - 1;
#pragma unroll
    for (int b = 0; b < NHIST; b++) hist[b] += (int)__popcll(__ballot(bin == b));
  }
  // called by the whole wave: lane 0 writes the wave's row
  __device__ void flush(int *row) const {
    int it = iters, mx = maxit, fl = failed, su = setups;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      it += __shfl_xor(it, off, 64);
      fl += __shfl_xor(fl, off, 64);
      su += __shfl_xor(su, off, 64);
      const int m2 = __shfl_xor(mx, off, 64);
      mx = m2 > mx ? m2 : mx;
    }
    if ((threadIdx.x & 63) == 0) {
      row[STAT_ITERS] = it;
      row[STAT_MAXIT] = mx;
      row[STAT_FAILED] = fl;
      row[STAT_SETUPS] = su;
#pragma unroll
      for (int b = 0; b < NHIST; b++) row[STAT_HIST + b] = hist[b];
    }
  }
};

// sums nrow rows of NSTAT partials into out (zeroed beforehand): LDS accumulation per
// block, then one global atomic per statistic and block
__global__ void __launch_bounds__(256)
stats_reduce(const int *rows, long nrow, int *out) {
  __shared__ int acc[NSTAT];
  const int t = threadIdx.x;
  if (t < NSTAT) acc[t] = 0;
  __syncthreads();
  const long m = nrow * NSTAT;
  for (long e = (long)blockIdx.x * blockDim.x + t; e < m; e += (long)gridDim.x * blockDim.x) {
    const int s = (int)(e % NSTAT);
    if (s == STAT_MAXIT) atomicMax(&acc[s], rows[e]);
    else atomicAdd(&acc[s], rows[e]);
  }
  __syncthreads();
  if (t < NSTAT) {
    if (t == STAT_MAXIT) atomicMax(&out[t], acc[t]);
    else atomicAdd(&out[t], acc[t]);
  }
}

static inline unsigned stats_blocks(long nrow) {
  const long b = (nrow * NSTAT + 2047) / 2048;
  return (unsigned)(b < 1 ? 1 : (b > 64 ? 64 : b));
}

// ------------------------------------------------------------------------------------
// batched path
// ------------------------------------------------------------------------------------

// The structural nonzeros of the analytic Jacobian (chem_jac_species, chem_jac_energy).
__device__ constexpr bool CHEM_JNZ[NSP][NSP] = {
    {1, 1, 1, 1, 1, 0, 0, 0, 1, 1}, {1, 1, 1, 1, 1, 0, 0, 0, 1, 1}, {1, 1, 1, 1, 1, 0, 0, 0, 1, 1},
    {1, 1, 1, 1, 1, 0, 0, 0, 1, 1}, {0, 1, 1, 1, 1, 0, 0, 0, 1, 1}, {0, 0, 0, 0, 0, 1, 1, 0, 1, 1},
    {0, 0, 0, 0, 0, 1, 1, 1, 1, 1}, {0, 0, 0, 0, 0, 0, 1, 1, 1, 1}, {0, 1, 1, 1, 1, 1, 1, 1, 1, 1},
    {1, 0, 1, 1, 0, 1, 1, 1, 1, 1}};

// M = I - hg * srhs * J into registers, J = calculate_jacobian_cvklu from the current
// temperature: the species rows (reaction tables), then the gas-energy row (cooling tables),
// so that both groups of rates never occupy registers at once. The rates come from the
// rate-major tables here: with the factors held in registers, the pair table's wider loads
// cost the batched kernel spills, and it measured faster this way. (Where the lane keeps its
// bin's pairs in LDS they come from there; the RHS evaluation at this Ts has set it. The adjoint
// kernels take them from the pair table, loads issued together: 1.37 -> 1.33 ms for 32^3 cells
// and 20 steps, while the batched kernel loses 1 to 2% that way.)
template <class Bin>
__device__ inline void cell_matrix_regs(const ChemConst &cc, const CellIn &c, double Ts,
                                        double dTs, const double (&y)[NSP], double hg,
                                        double srhs, double (&M)[NSP][NSP], const Bin &rb) {
#pragma clang fp contract(on)
  double ya[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) ya[s] = y[s] * c.s(s);
  double k[NRATE], dk[NRATE];
#pragma unroll
  for (int r = 0; r < NRATE; r++) k[r] = dk[r] = 0.0;
  const double hs = hg * srhs;
  double Tdef = 0.0, Tfactor = 0.0;
  const double2 *pairs = nullptr;
  if constexpr (Bin::on) {
    chem_locate(cc, chem_log(Ts), Tdef);
    Tfactor = fast_rcp(Ts) * cc.idbin;
    chem_rates_at<0, C_BREM, 64>(rb.row, Tdef, Tfactor, k, dk);
  } else if constexpr (Bin::pairs) {
    pairs = cc.tabp + (long)chem_locate(cc, chem_log(Ts), Tdef) * NRATE;
    Tfactor = fast_rcp(Ts) * cc.idbin;
    chem_rates_batch<0, C_BREM, 1, RATE_BATCH>(pairs, Tdef, Tfactor, k, dk);
  } else chem_rates_range<0, C_BREM>(cc, Ts, k, dk);
  chem_jac_species(ya, k, dk, dTs, M);
#pragma unroll
  for (int r = 0; r < NSP - 1; r++) {
    const double row = hs * c.is(r);
#pragma unroll
    for (int q = 0; q < NSP; q++) {
      const double eye = r == q ? 1.0 : 0.0;
      M[r][q] = CHEM_JNZ[r][q] ? eye - row * (M[r][q] * c.s(q)) : eye;
    }
  }
  if constexpr (Bin::on) chem_rates_at<C_BREM, NRATE, 64>(rb.row, Tdef, Tfactor, k, dk);
  else if constexpr (Bin::pairs)
    chem_rates_batch<C_BREM, NRATE, 1, RATE_BATCH>(pairs, Tdef, Tfactor, k, dk);
  else chem_rates_range<C_BREM, NRATE>(cc, Ts, k, dk);
  chem_jac_energy(ya, k, dk, Ts, cc.z, dTs, c.ax, M);
  const double row = hs * c.is(NSP - 1);
#pragma unroll
  for (int q = 0; q < NSP; q++) {
    const double eye = NSP - 1 == q ? 1.0 : 0.0;
    M[NSP - 1][q] = CHEM_JNZ[NSP - 1][q] ? eye - row * (M[NSP - 1][q] * c.s(q)) : eye;
  }
}

__device__ inline void cell_matrix_regs(const ChemConst &cc, const CellIn &c, double Ts,
                                        double dTs, const double (&y)[NSP], double hg,
                                        double srhs, double (&M)[NSP][NSP]) {
  cell_matrix_regs(cc, c, Ts, dTs, y, hg, srhs, M, NoRateBin());
}

// Solve with the factors of lu_factor_regs<true> (reciprocal diagonal). Row exchanges are
// applied step by step, and only where some lane of the wave pivoted in that step: for
// I - h*gamma*J of the stiff network the diagonal is the column maximum in nearly every cell
// and column, and applying all packed pivots costs 180 selects per solve. Column by column, so
// that a row's update waits for one new value only: row by row the back substitution is a chain
// of 55 dependent operations, this way of 20. (167 forced seven-stage steps of 4096 cells 11.7 ->
// 10.8 ms.)
__device__ inline void lu_solve_regs(const double (&a)[NSP][NSP], unsigned long long pv,
                                     double (&b)[NSP]) {
#pragma clang fp contract(on)
  const unsigned long long moved = pv ^ PIV_IDENTITY;
  if (__builtin_amdgcn_ballot_w64(moved != 0) != 0) {            // wave-uniform
#pragma unroll
    for (int k = 0; k < NSP - 1; k++)
      if (__builtin_amdgcn_ballot_w64(((moved >> (4 * k)) & 15) != 0) != 0) lu_exchange(pv, k, b);
  }
#pragma unroll
  for (int q = 0; q < NSP - 1; q++)
#pragma unroll
    for (int r = q + 1; r < NSP; r++) b[r] -= a[r][q] * b[q];
#pragma unroll
  for (int q = NSP - 1; q >= 0; q--) {
    b[q] *= a[q][q];
#pragma unroll
    for (int r = 0; r < q; r++) b[r] -= a[r][q] * b[q];
  }
}

// Per-cell values a wave keeps in LDS, element-major ([word][64 lanes]): scale, inv_scale,
// mdensity, inv_mdensity, the two optical-depth factors, the (sub)step start y_n, then the
// work slots of NSP words each.
// Narrow tables (SDIRK of up to FST_LDS_MAX stages): slot j keeps the stage derivative F_j.
// The current stage's right-hand side r sits in the slot that the stage's own F will take
// (the last stage, whose F is not needed: in slot 0, whose F_0 is consumed when that r is
// formed), and the first correction of a step across its matrix set-up in slot 1, free until
// the second stage; tables of one or two stages have two slots for these.
// Wide tables (an explicit first stage or more than FST_LDS_MAX stages): slot 0 is r, slot 1
// the correction, and the stage derivatives live in a global buffer, [(j*10+s)][thread of the
// grid], so that four waves still share a block.
constexpr int CELL_WORDS = 2 * NSP + 4;
constexpr int FST_LDS_MAX = 4;
__host__ __device__ inline bool dirk_wide(int nstage, bool esdirk) {
  return esdirk || nstage > FST_LDS_MAX;
}
// What else a launch keeps in LDS when its waves leave room (DirkMem):
//   MEM_SHARED  nothing: four waves share a block;
//   MEM_STAGES  the forcing and the wide tables' stage derivatives (after the work slots):
//               at most two waves per CU;
//   MEM_RATES   these and the rate pairs of each cell's table bin (RateBin): one wave per CU.
enum DirkMem { MEM_SHARED = 0, MEM_STAGES, MEM_RATES };
__host__ __device__ inline int dirk_slot_words(int nstage, bool wide) {
  return (wide || nstage <= 3 ? 2 : nstage - 1) * NSP;
}
__host__ __device__ inline int dirk_wave_words(int nstage, bool wide, int mem = MEM_SHARED) {
  return CELL_WORDS + NSP + dirk_slot_words(nstage, wide) +
         (mem >= MEM_STAGES ? NSP + (wide ? (nstage - 1) * NSP : 0) : 0) +
         (mem >= MEM_RATES ? 2 * NRATE : 0);
}
// dynamic LDS of the batched kernel for `wpb` waves per block
inline size_t dirk_lds_bytes(int wpb, int nstage, bool wide, int mem = MEM_SHARED) {
  return sizeof(double) *
         ((size_t)4 * TLEN + (size_t)wpb * dirk_wave_words(nstage, wide, mem) * 64);
}

// Threads per block of a batched launch asked for `block` threads: blocks whose LDS (the
// dynamic part for their waves plus the kernel's static part) would exceed the per-block
// limit are halved (fewer waves then share one copy of the gamma tables); 0 when not even
// one wave fits.
static int fit_block(int block, int nstage, size_t static_lds, size_t limit, bool wide, int mem) {
  for (; block >= 64; block /= 2)
    if (dirk_lds_bytes(block / 64, nstage, wide, mem) + static_lds <= limit) return block;
  return 0;
}
int dirk_fit_block(int block, int nstage, size_t static_lds, size_t limit, bool esdirk) {
  return fit_block(block, nstage, static_lds, limit, dirk_wide(nstage, esdirk), MEM_SHARED);
}

// queue += chunk by one lane of the wave; returns the old value to all of them. Called with all
// lanes. The lane mask is set and restored within the statement, so that there is no branch and
// no join for the compiler: `if (lane == 0) atomicAdd(...)` in the chunk loop once had the register
// allocator save live values at the join, ahead of the mask's restoration, for lane 0 only. (64
// lanes adding 0 to other words instead: one SDIRK3 step of 131072 cells 212 -> 276 us.)
__device__ inline int queue_take(int *queue, int chunk) {
  int old;
  unsigned long long mask;
  __asm__ volatile("s_mov_b64 %1, exec\n\t"
                   "s_mov_b64 exec, 1\n\t"
                   "global_atomic_add %0, %2, %3, %4 sc0\n\t"
                   "s_waitcnt vmcnt(0)\n\t"
                   "s_mov_b64 exec, %1"
                   : "=&v"(old), "=&s"(mask)
                   : "v"(0), "v"(chunk), "s"(queue)
                   : "memory");
  return __builtin_amdgcn_readfirstlane(old);
}

// FORCED: y' = s_rhs f(y) + force, force constant over the step ([cell][10], the forcing an
// MRI method hands its fast stepper, multirate_chem_hydro_main.cpp:922-946).
// SUBSTEP (o.max_halvings > 0): per-cell step rejection. When a cell's Newton budget runs
// out, the cell returns to the start of its current substep (state and temperature warm
// start) and retries it in halves, up to max_halvings times; accepted substeps are
// counted in units of the finest one (h / 2^max_halvings), so their sizes add up to h
// exactly. A cell that fails at the finest size keeps its last accepted state and counts
// as failed. Without SUBSTEP a failed cell keeps its last Newton iterate (the plain
// solver's behaviour).
// nsteps: steps of size h per cell in this launch (a fixed-step run with constant forcing,
// such as the fast steps of one multirate slow stage); each cell runs them back to back,
// its state and temperature staying in registers, every step exactly as a launch of its
// own would run it (a failed step counts and the next starts from the state it kept).
// With nsteps > 1 the statistics are per cell over all its steps (failures: failed steps).
// WIDE: tables with an explicit first stage (ESDIRK) or more than FST_LDS_MAX stages (the
// stage derivatives then in the global buffer fglob); the other instantiations are the
// plain SDIRK form, without that code.
// MEM: what is kept in LDS beyond the cells' constants and work slots (DirkMem).
template <bool FORCED, bool SUBSTEP, bool WIDE, int MEM>
__global__ void __launch_bounds__(256)
chem_dirk_batched(long n, ChemConst cc, ChemPtrsD p, DirkDev o, double h, double *y,
                  const double *force, const int *order, const double2 *tdt, int *queue,
                  int *rows, int nsteps, double *fglob, int chunk) {
#pragma clang fp contract(on)
  // block statistics in LDS (the per-cell updates are LDS atomics; one row per block).
  // Dynamic LDS: the gamma tables of the temperature solve (32 KB; the ten-step Newton loop
  // gathers from them at every step of every RHS evaluation), then per wave the values of
  // its cells (dirk_wave_words): the constants read at every RHS evaluation, loaded from HBM
  // once per cell, and the stage derivatives and step start read at stage changes.
  __shared__ int bs[NSTAT];
  // (16-byte accesses: the rate pairs of MEM_RATES, whose rows lie at multiples of 64 doubles)
  extern __shared__ __attribute__((aligned(16))) double lds[];
  static_assert(4 * TLEN % 64 == 0 && sizeof(double2) == 16, "rate pairs at 16-byte addresses");
  if (threadIdx.x < NSTAT) bs[threadIdx.x] = 0;
  // the wide tables' matrix, for a stage index held per lane
  __shared__ double tabA[WIDE ? MAXSTAGE * MAXSTAGE : 1];
  if (WIDE && threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < MAXSTAGE * MAXSTAGE; k++) tabA[k] = o.A[k];
  }
  for (int e = threadIdx.x; e < 4 * TLEN; e += blockDim.x) lds[e] = cc.tab[G_GH2_1 * TLEN + e];
  __syncthreads();
  const GammaTabs gt = gamma_tabs(lds);
  const int lane = threadIdx.x & 63;
  double *const cst =
      lds + 4 * TLEN + (threadIdx.x >> 6) * (dirk_wave_words(o.nstage, WIDE, MEM) * 64);
  double *const yst = cst + CELL_WORDS * 64 + lane;        // y_n[s] at s*64
  double *const slots = yst + NSP * 64;                    // work slot k, element s: (10 k + s)*64
  // F_j[s] at (j*10 + s) * fstr: in the work slots (fstr 64), or for the wide tables in the
  // global buffer (one column per thread of the grid)
  // (or, MEM_STAGES, in LDS behind the forcing)
  constexpr bool FLDS = MEM >= MEM_STAGES;
  double *const frc = slots + dirk_slot_words(o.nstage, WIDE) * 64;      // forcing s at s*64
  const long fstr = WIDE && !FLDS ? (long)gridDim.x * blockDim.x : 64;
  double *const Fst = !WIDE ? slots : FLDS ? frc + NSP * 64
                                          : fglob + (long)blockIdx.x * blockDim.x + threadIdx.x;
  typename std::conditional<MEM >= MEM_RATES, RateBin, NoRateBin>::type rb;
  if constexpr (MEM >= MEM_RATES) {
    const int at = CELL_WORDS + NSP + dirk_slot_words(o.nstage, WIDE) + NSP +
                   (WIDE ? (o.nstage - 1) * NSP : 0);
    rb.row = reinterpret_cast<double2 *>(cst + at * 64) + lane;
    rb.bin = -1;
  }
  // The first chunk of each wave is its global wave index; later ones come from the queue
  // (which starts after them), asked for when a chunk is done.
  const int nwaves = (int)(gridDim.x * (blockDim.x >> 6));
  int next = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * chunk;
  for (;;) {
    const int base = next;
    if ((long)base >= n) break;
    if (lane < chunk && (long)base + lane < n) {   // the other lanes idle to the chunk's end
    // the lane's cell: queue positions run over the cells in temperature order
    const int cell = order ? order[base + lane] : base + lane;
    // per-lane state for the whole step: iterate and LU factors
    double Ts, dTs, Ts0, dTs0, z[NSP], lu[NSP][NSP];
    {
      const long i = cell;
      Ts0 = p.Ts[i];                                       // warm start at the substep start
      dTs0 = p.dTs[i];
      if (!SUBSTEP && tdt) {                               // solved at y_n by the ordering pass
        const double2 t = tdt[i];
        Ts = t.x;
        dTs = t.y;
      } else {
        Ts = Ts0;
        dTs = dTs0;
      }
#pragma unroll
      for (int s = 0; s < NSP; s++) z[s] = y[NSP * i + s];
#pragma unroll
      for (int s = 0; s < NSP; s++) {
        yst[s * 64] = z[s];
        cst[s * 64 + lane] = p.scale[NSP * i + s];
        cst[(NSP + s) * 64 + lane] = p.iscale[NSP * i + s];
      }
      cst[(2 * NSP) * 64 + lane] = p.md[i];
      cst[(2 * NSP + 1) * 64 + lane] = p.imd[i];
      cst[(2 * NSP + 2) * 64 + lane] = p.cie[i];
      cst[(2 * NSP + 3) * 64 + lane] = p.h2o[i];
      if (FORCED && FLDS) {
#pragma unroll
        for (int s = 0; s < NSP; s++) frc[s * 64] = force[NSP * i + s];
      }
    }
    // the cell's forcing (0 without) in registers. Every loop below that writes LDS has its
    // LDS reads taken out in front of it: the compiler must keep reads behind writes that may
    // overlap them, and one by one each pays the latency (a stage change: 3300 cycles, 10 of
    // them in turn at two places).
    auto forcing = [&](long i, double (&fo)[NSP]) {
#pragma unroll
      for (int s = 0; s < NSP; s++)
        fo[s] = !FORCED ? 0.0 : FLDS ? frc[s * 64] : force[NSP * i + s];
    };
    // One loop, one RHS evaluation per pass. A pass is one Newton iteration of the cell's
    // stage; where a setup is due (at y_n, or after max_iters without convergence) the pass
    // forms and factors the matrix at the iterate between that evaluation and the update,
    // so the evaluation serves both.
    // The cells of a wave keep step with each other: one whose stage has converged waits
    // until the others' have too, and the stage changes (and the next step's setups, which
    // fall due together) are taken by all lanes at once. A wave runs to its slowest cell
    // anyway; without the waiting, the lanes' stage changes and setups spread over nearly
    // every pass and each of them was paid for by the whole wave. r and the first correction
    // live in LDS: in registers across the matrix set-up they cost 170 spilled VGPRs. With
    // the contracted arithmetic (mvd_chem.hpp) and the even chunks, against lanes that ran
    // on alone and evaluated the RHS again after a setup: 4096 cells, 167 forced
    // seven-stage steps 72.4 -> 19.7 ms; one multirate slow step of 32^3 cells 77.3 -> 31.6
    // ms; one SDIRK3 step of 64^3 cells 0.471 -> 0.382 ms (ordering pass included). With what
    // followed (DirkMem, loads issued together, the shorter temperature solve, the column-wise
    // substitution): 10.8, 16.9 and 0.33 ms.
    // (the substepping variants, which hold more state, solve it again: skipping there
    // costs registers that are worth more than the solve)
    bool setup = true, solved = !SUBSTEP && tdt != nullptr;
    bool busy = true;                                      // iterating (else waiting)
    bool fend = false;                                     // the step ended by failing
    bool start = true;                                     // z is the (sub)step start y_n
    int rslot = 0;                                         // offset of r's slot
    int st = 0, it = 0, setups = 0, nit = 0, nsetup = 0, nst = 0, nfail = 0;
    double crate = 1.0, delp = 0.0;                        // Newton rate estimate, last norm
    int lsetup = 0;                                        // step of the last Jacobian setup
    double hs = h;                                         // current (sub)step
    double hg = h * o.gamma;                               // one implicit diagonal value
    int halv = 0, done = 0;                                // substep level, units done
    unsigned long long pv = 0;
    // With forcing, r holds the stage's right-hand side plus hg * force, the constant part
    // of z - hg f(z) - r; the forcing is then read at stage changes only.
    {
      double fo[NSP];
      forcing(cell, fo);
#pragma unroll
      for (int s = 0; s < NSP; s++) slots[s * 64] = FORCED ? z[s] + hg * fo[s] : z[s];
    }
    for (;;) {
      // The lane offset and cell index are made opaque on every pass so that the per-lane
      // addresses of the cell's inputs are formed where they are used instead of being held
      // in registers.
      long lo = lane;
      int ci = cell;
      __asm__ volatile("" : "+v"(lo), "+v"(ci));
      const long i = ci;
      if (busy) {
        const double *cl = cst + lo;
        const CellIn c{cl, cl + NSP * 64, 64,
                       CellAux{cl[(2 * NSP) * 64], cl[(2 * NSP + 1) * 64],
                               cl[(2 * NSP + 2) * 64], cl[(2 * NSP + 3) * 64]}};
        double f[NSP];
        cell_rhs<true>(cc, gt, c, Ts, dTs, z, o.rhs_scale, f, !solved, rb);
        solved = false;
        if (WIDE && o.esdirk && st == 0) {
          // explicit first stage (ESDIRK): its value is y_n and F_0 = f(y_n), this pass's
          // RHS; the first implicit stage's r = y_n + hs a_10 F_0. The pass goes on as that
          // stage's first Newton iteration, with this f at its predictor y_n.
          double fo[NSP], yn[NSP];
          forcing(i, fo);
#pragma unroll
          for (int s = 0; s < NSP; s++) yn[s] = yst[s * 64];
#pragma unroll
          for (int s = 0; s < NSP; s++) {
            const double F0 = FORCED ? f[s] + fo[s] : f[s];
            Fst[s * fstr] = F0;
            double a = 0.0;
            a += dirk_coef(o, 1, 0) * F0;
            double rs = yn[s] + hs * a;
            if (FORCED) rs += hg * fo[s];
            slots[s * 64] = rs;
          }
          st = 1;
        }
        double *const rs = slots + rslot + (lo - lane);
        double d[NSP];
#pragma unroll
        for (int s = 0; s < NSP; s++) d[s] = -(z[s] - hg * f[s] - rs[s * 64]);
        if (setup) {
          // at a step's start the correction waits in its slot (and z is y_n), so that
          // neither occupies registers while the matrix is formed and factored; a setup at
          // a later iterate (rare) evaluates the RHS again in the next pass instead
          double *const ds = slots + NSP * 64 + (lo - lane);
          if (start) {
#pragma unroll
            for (int s = 0; s < NSP; s++) ds[s * 64] = d[s];
          }
          cell_matrix_regs(cc, c, Ts, dTs, z, hg, o.rhs_scale, lu, rb);
          pv = lu_factor_regs<true>(lu);
          nsetup++;
          setup = false;
          it = 0;
          crate = 1.0;
          lsetup = nst;
          if (!start) continue;
          __asm__ volatile("" ::: "memory");
#pragma unroll
          for (int s = 0; s < NSP; s++) {
            d[s] = ds[s * 64];
            z[s] = yst[s * 64 + (lo - lane)];
          }
        }
        start = false;
        lu_solve_regs(lu, pv, d);
#pragma unroll
        for (int s = 0; s < NSP; s++) z[s] += d[s];
        nit++;
        it++;
        const double del = wrms_norm(d, z, o.rtol, o.atol);
        if (it > 1) crate = conv_rate(crate, del, delp);
        const bool diverging = it > 1 && conv_diverging(del, delp);
        delp = del;
        if (conv_ok(crate, del, o.ntol)) {
          busy = false;
        } else if (it == o.max_iters || diverging) {
          if (++setups > o.max_setups) {
            bool retry = false;
            if (SUBSTEP) {
              // back to the substep start
#pragma unroll
              for (int s = 0; s < NSP; s++) z[s] = yst[s * 64];
              Ts = Ts0;
              dTs = dTs0;
              if (halv < o.max_halvings) {
                retry = true;
                halv++;
                hs = ldexp(h, -halv);
                hg = hs * o.gamma;
                double fo[NSP];
                forcing(i, fo);
#pragma unroll
                for (int s = 0; s < NSP; s++) slots[s * 64] = FORCED ? z[s] + hg * fo[s] : z[s];
                rslot = 0;
                st = 0;
                it = 0;
                setups = 0;
                setup = true;
                start = true;
              }
            }
            if (!retry) {                                  // the step failed
              nfail++;
              fend = true;
              busy = false;
            }
          } else {
            setup = true;
          }
        }
      }
      if (__ballot(busy) != 0) continue;                   // some cell of the wave iterates
      busy = true;
      if (!fend && ++st < o.nstage) {
        // F_{st-1} = (z - r)/hg (ARKODE's implicit-stage derivative; with forcing r holds
        // hg * force too); the next stage's r
        const double ihg = 1.0 / hg;
        double *const rold = slots + rslot;
        // (narrow: r_{st-1} and F_{st-1} share slot st - 1; the last stage's r takes slot 0)
        if (!WIDE) rslot = st + 1 < o.nstage ? st * NSP * 64 : 0;
        double *const rnew = slots + rslot;
        double fo[NSP], yn[NSP];
        forcing(i, fo);
        {
          double ro[NSP];
#pragma unroll
          for (int s = 0; s < NSP; s++) ro[s] = rold[s * 64];
#pragma unroll
          for (int s = 0; s < NSP; s++) yn[s] = yst[s * 64];
#pragma unroll
          for (int s = 0; s < NSP; s++) {
            const double F = (z[s] - ro[s]) * ihg;
            Fst[((st - 1) * NSP + s) * fstr] = FORCED ? F + fo[s] : F;
          }
        }
        double a[NSP];
#pragma unroll
        for (int s = 0; s < NSP; s++) a[s] = 0.0;
        if (WIDE) {
          // two earlier stages' loads in flight at a time: all of them at once cost this
          // variant 70 spilled VGPRs
#pragma unroll 1
          for (int j = 0; j < st; j += 2) {
            const double c0 = tabA[st * MAXSTAGE + j], c1 = tabA[st * MAXSTAGE + j + 1];
            const bool two = j + 1 < st;
            const double *const F0 = Fst + (long)j * NSP * fstr;
            const double *const F1 = two ? F0 + NSP * fstr : F0;
            double u[NSP], v[NSP];
#pragma unroll
            for (int s = 0; s < NSP; s++) u[s] = F0[s * fstr];
#pragma unroll
            for (int s = 0; s < NSP; s++) v[s] = F1[s * fstr];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < NSP; s++) {
              a[s] += c0 * u[s];
              if (two) a[s] += c1 * v[s];
            }
          }
        } else {
#pragma unroll
          for (int s = 0; s < NSP; s++)
#pragma unroll
            for (int j = 0; j < FST_LDS_MAX - 1; j++)
              if (j < st) a[s] += dirk_coef<FST_LDS_MAX>(o, st, j) * Fst[(j * NSP + s) * 64];
        }
#pragma unroll
        for (int s = 0; s < NSP; s++) {
          double rs = yn[s] + hs * a[s];                   // the (sub)step start
          if (FORCED) rs += hg * fo[s];
          rnew[s * 64] = rs;
        }
        it = 0;
        setups = 0;
        continue;
      }
      // end of the (sub)step
      bool step_end = true;
      if (SUBSTEP && !fend) {
        done += 1 << (o.max_halvings - halv);
        step_end = done >= (1 << o.max_halvings);
      }
      if (step_end) {
        if (++nst >= nsteps) break;
        // the next step from the state the cell kept (as the next launch would start it).
        // ARKODE's lsetup frequency: a setup at y_n after a failed or split step and once
        // msbp steps have passed since the last one; else Newton starts with the held factors
        setup = fend || halv > 0 || nst - lsetup >= o.msbp;
        fend = false;
        hs = h;
        hg = h * o.gamma;
        halv = 0;
        done = 0;
      } else {
        setup = true;                                      // substep accepted: the next one
      }
      double fo[NSP];
      forcing(i, fo);
#pragma unroll
      for (int s = 0; s < NSP; s++) {
        yst[s * 64] = z[s];
        slots[s * 64] = FORCED ? z[s] + hg * fo[s] : z[s];
      }
      rslot = 0;
      start = true;
      Ts0 = Ts;
      dTs0 = dTs;
      st = 0;
      it = 0;
      setups = 0;
    }
    {
      const long i = cell;
#pragma unroll
      for (int s = 0; s < NSP; s++) y[NSP * i + s] = z[s];
      p.Ts[i] = Ts;
      p.dTs[i] = dTs;
    }
    atomicAdd(&bs[STAT_ITERS], nit);
    atomicMax(&bs[STAT_MAXIT], nit);
    atomicAdd(&bs[STAT_SETUPS], nsetup);
    if (nfail) atomicAdd(&bs[STAT_FAILED], nfail);
    atomicAdd(&bs[STAT_HIST + (nit < NHIST - 1 ? nit : NHIST - 1)], 1);
    }
    next = queue_take(queue, chunk) + nwaves * chunk;
  }
  __syncthreads();
  // block statistics: one row per block; the last block to finish sums the rows into
  // queue[1 .. NSTAT] (the ticket counter at queue[1 + NSTAT] starts at zero)
  if (threadIdx.x < NSTAT) rows[(long)blockIdx.x * NSTAT + threadIdx.x] = bs[threadIdx.x];
  __threadfence();
  __shared__ unsigned ticket;
  if (threadIdx.x == 0) ticket = atomicAdd((unsigned *)(queue + 1 + NSTAT), 1u);
  __syncthreads();
  if (ticket != gridDim.x - 1) return;
  __threadfence();
  // each thread reads whole rows (independent loads, issued together), then LDS atomics
  __shared__ int tot[NSTAT];
  if (threadIdx.x < NSTAT) tot[threadIdx.x] = 0;
  __syncthreads();
  for (unsigned b = threadIdx.x; b < gridDim.x; b += blockDim.x) {
    int v[NSTAT];
#pragma unroll
    for (int st = 0; st < NSTAT; st++)
      v[st] = __hip_atomic_load(rows + (long)b * NSTAT + st, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int st = 0; st < NSTAT; st++) {
      if (st == STAT_MAXIT) atomicMax(&tot[st], v[st]);
      else if (v[st]) atomicAdd(&tot[st], v[st]);
    }
  }
  __syncthreads();
  if (threadIdx.x < NSTAT) queue[1 + threadIdx.x] = tot[threadIdx.x];
}

// ------------------------------------------------------------------------------------
// plain (reference-structured) kernels
// ------------------------------------------------------------------------------------

// Plain-path cell states (`active`): 0 done with the stage (converged or failed), 1
// iterating, 2 diverged and waiting for the re-setup.
constexpr int PLAIN_ITERATING = 1 << 1, PLAIN_UNCONVERGED = (1 << 1) | (1 << 2);

// f = s * rhs(z) for the cells whose state is in `mask` (updates Ts/dTs of those cells)
__global__ void __launch_bounds__(256)
plain_rhs(long n, ChemConst cc, ChemPtrsD p, double srhs, const double *z, double *f,
          const int *active, int mask) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !((mask >> active[i]) & 1)) return;
  const CellIn c = load_cell(p, i);
  double Ts = p.Ts[i], dTs = p.dTs[i];
  double zz[NSP], ff[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) zz[s] = z[NSP * i + s];
  cell_rhs(cc, c, Ts, dTs, zz, srhs, ff);
  p.Ts[i] = Ts;
  p.dTs[i] = dTs;
#pragma unroll
  for (int s = 0; s < NSP; s++) f[NSP * i + s] = ff[s];
}

// calculate_jacobian_cvklu at z from the current temperature and M = I - hg s J into the
// column-major 10x10 blocks (SUNMatrix_MagmaDenseBlock) of the cells flagged in `todo`
__global__ void __launch_bounds__(256)
plain_jac(long n, ChemConst cc, ChemPtrsD p, double hg, double srhs, const double *z,
          double *LU, const int *todo) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !todo[i]) return;
  const CellIn c = load_cell(p, i);
  double zz[NSP], M[NSP][NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) zz[s] = z[NSP * i + s];
  cell_matrix_regs(cc, c, p.Ts[i], p.dTs[i], zz, hg, srhs, M);
  double *blk = LU + (long)NSP * NSP * i;
#pragma unroll
  for (int q = 0; q < NSP; q++)
#pragma unroll
    for (int r = 0; r < NSP; r++) blk[NSP * q + r] = M[r][q];
}

// batched getrf: each thread factors its cell's block in registers
__global__ void __launch_bounds__(256)
plain_getrf(long n, double *LU, unsigned long long *piv, const int *todo) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !todo[i]) return;
  double *blk = LU + (long)NSP * NSP * i;
  double a[NSP][NSP];
#pragma unroll
  for (int q = 0; q < NSP; q++)
#pragma unroll
    for (int r = 0; r < NSP; r++) a[r][q] = blk[NSP * q + r];
  piv[i] = lu_factor_regs<true>(a);
#pragma unroll
  for (int q = 0; q < NSP; q++)
#pragma unroll
    for (int r = 0; r < NSP; r++) blk[NSP * q + r] = a[r][q];
}

// stage start: r = y_n + h sum_{j<st} a_st,j F_j; activate the cells that have not failed
__global__ void __launch_bounds__(256)
plain_stage_init(long n, int st, double h, DirkDev o, const double *yn, const double *F,
                 double *r, int *active, const int *failed) {
#pragma clang fp contract(on)
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int s = 0; s < NSP; s++) {
    double a = 0.0;
#pragma unroll
    for (int j = 0; j < MAXSTAGE - 1; j++)
      if (j < st) a += dirk_coef(o, st, j) * F[(long)j * n * NSP + NSP * i + s];
    r[NSP * i + s] = yn[NSP * i + s] + h * a;
  }
  active[i] = failed[i] ? 0 : 1;
}

// Newton update (getrs + z += d + ARKODE's convergence test, iteration m of the stage
// solve) of the iterating cells; converged cells are done, diverging ones wait for the
// re-setup; the still iterating (count[0]) and the diverged (count[1]) are counted.
__global__ void __launch_bounds__(256)
plain_newton(long n, double hg, DirkDev o, double *LU, const unsigned long long *piv,
             const double *f, const double *r, double *z, int *active, int *cell_iters,
             double *crate, double *delp, int m, int *count) {
#pragma clang fp contract(on)
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || active[i] != 1) return;
  double d[NSP], zz[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) {
    zz[s] = z[NSP * i + s];
    d[s] = -(zz[s] - hg * f[NSP * i + s] - r[NSP * i + s]);
  }
  double a[NSP][NSP];
  const double *blk = LU + (long)NSP * NSP * i;
#pragma unroll
  for (int q = 0; q < NSP; q++)
#pragma unroll
    for (int r = 0; r < NSP; r++) a[r][q] = blk[NSP * q + r];
  lu_solve_regs(a, piv[i], d);
#pragma unroll
  for (int s = 0; s < NSP; s++) {
    zz[s] += d[s];
    z[NSP * i + s] = zz[s];
  }
  cell_iters[i] += 1;
  const double del = wrms_norm(d, zz, o.rtol, o.atol), dp = delp[i];
  double cr = crate[i];
  if (m > 0) cr = conv_rate(cr, del, dp);
  crate[i] = cr;
  delp[i] = del;
  if (conv_ok(cr, del, o.ntol)) active[i] = 0;
  else if (m > 0 && conv_diverging(del, dp)) {
    active[i] = 2;
    atomicAdd(count + 1, 1);
  } else {
    atomicAdd(count, 1);
  }
}

// after a setup: its cells iterate again, with the rate estimate back at 1
__global__ void __launch_bounds__(256)
plain_resume(long n, int *active, double *crate) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !active[i]) return;
  active[i] = 1;
  crate[i] = 1.0;
}

// stage end: F_st = (z - r)/hg
__global__ void __launch_bounds__(256)
plain_stage_finish(long n, int st, double hg, const double *z, const double *r, double *F) {
#pragma clang fp contract(on)
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int s = 0; s < NSP; s++)
    F[(long)st * n * NSP + NSP * i + s] = (z[NSP * i + s] - r[NSP * i + s]) * (1.0 / hg);
}

// per-wave statistics rows of the plain path
__global__ void __launch_bounds__(256)
plain_finish(long n, const int *cell_iters, const int *cell_setups, const int *failed,
             int *rows) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  WaveStats ws;
  if (i < n) ws.add(cell_iters[i], cell_setups[i], failed[i] != 0);
  if (((long)blockIdx.x * blockDim.x + (threadIdx.x & ~63)) < n) ws.flush(rows + (i >> 6) * NSTAT);
}

__global__ void __launch_bounds__(256)
fill_int(long n, int *a, int v) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// zero a[0..na) and b[0..nb) (b may be null)
__global__ void __launch_bounds__(256)
zero_two(long na, int *a, long nb, int *b) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < na) a[i] = 0;
  if (b && i < nb) b[i] = 0;
}

__global__ void __launch_bounds__(256)
copy_double(long n, const double *a, double *b) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// the cells still active after the last allowed setup have failed
__global__ void __launch_bounds__(256)
mark_failed(long n, const int *active, int *failed) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && active[i]) failed[i] = 1;
}

__global__ void __launch_bounds__(256)
count_setups(long n, const int *active, int *cell_setups) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && active[i]) cell_setups[i] += 1;
}

// ------------------------------------------------------------------------------------
// host drivers
// ------------------------------------------------------------------------------------

static inline unsigned nb(long n) { return (unsigned)((n + 255) / 256); }

static ChemPtrsD ptrs_d(ChemState &s) {
  return ChemPtrsD{s.scale, s.inv_scale, s.mdensity, s.inv_mdensity, s.cie_oda, s.h2_oda,
                   s.Ts, s.dTs_ge};
}

static int ensure_work(ChemState &s, size_t bytes) {
  if (s.work_bytes >= bytes) return 0;
  if (s.work) (void)hipFree(s.work);
  s.work = nullptr;
  s.work_bytes = 0;
  s.gen++;
  if (hipMalloc(&s.work, bytes) != hipSuccess) return -1;
  s.work_bytes = bytes;
  return 0;
}

static constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// ------------------------------------------------------------------------------------
// Cell order of the batched step: a counting sort of the cells by a two-level key, so that
// the 64 lanes of a wave gather from the same few lines of every rate table and need
// similar Newton work (a wave runs to its slowest cell). Major: the table bin of the
// temperature at y_n in groups of 8 bins. Minor: the size of the first Newton correction,
// classed by log10(h * max_s |y'_s(y_n)|) over the nine species in half decades over
// [1e-8, 1) (16 classes; the energy row adds nothing to the grouping):
// cells whose scaled rate change over the step is tiny converge in one iteration per
// stage, the others in two or more, and the temperature alone does not tell them apart
// (for the 64^3 synthetic cells the sum over chunks of the slowest cell's iterations is
// 1.19 times the mean work in temperature order, 1.07 with the minor key). The queue then
// hands out positions of this order. Per-cell results do not depend on the order. The
// temperature is the solved one at y_n (the warm start alone may be a common guess such
// as the 1000 K of a fresh preparation).
// ------------------------------------------------------------------------------------
constexpr int TORD_TB = 128;                  // temperature buckets: table bin (0..1022) / 8
constexpr int TORD_RC = 16;                   // rate classes within a temperature bucket
constexpr int TORD_NBK = TORD_TB * TORD_RC;   // keys
constexpr long TORD_MIN = 4096;               // smaller batches keep the natural order
// Bucket counters sit 32 bytes apart so that the blocks' atomics on different buckets
// rarely share an address: total of bucket k at cnt[k * TORD_PAD], its running offset at
// cnt[(TORD_NBK + k) * TORD_PAD].
constexpr int TORD_PAD = 8;

// rate class of a cell from m = h * max_s |y'_s|: 0 below 1e-8 (or not finite), 15 at 1 and
// above, else floor(2 log10 m) + 16
__device__ inline int tord_rate_class(double m) {
  if (!(m > 1e-8)) return 0;
  if (m >= 1.0) return TORD_RC - 1;
  const int c = (int)floor(2.0 * log10(m)) + 16;
  return c < 0 ? 0 : (c > TORD_RC - 1 ? TORD_RC - 1 : c);
}

// Keys (two bytes per cell) and the bucket totals, accumulated per block in LDS first. One
// cell per thread, blocks of TORD_CBLOCK threads. The temperature is solved from the
// cell's warm start exactly as the step's first RHS evaluation solves it (same function,
// same inputs, so the same bits); the solution goes to tdt and that evaluation skips its
// solve. The rate class uses the species rows of the RHS at that temperature (times the
// RHS scale, plus the forcing when the step is forced).
constexpr int TORD_CBLOCK = 256;
__global__ void __launch_bounds__(TORD_CBLOCK)
tord_count(long n, ChemConst cc, ChemPtrsD p, const double *y, const double *force, double h,
           double srhs, unsigned short *key, int *cnt, double2 *tdt) {
#pragma clang fp contract(on)
  __shared__ int hc[TORD_NBK];
  __shared__ double gl[4 * TLEN];        // the gamma tables of the temperature solve
  for (int e = threadIdx.x; e < TORD_NBK; e += blockDim.x) hc[e] = 0;
  for (int e = threadIdx.x; e < 4 * TLEN; e += blockDim.x) gl[e] = cc.tab[G_GH2_1 * TLEN + e];
  __syncthreads();
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    double ya[NSP], T = p.Ts[i], dT = p.dTs[i];
#pragma unroll
    for (int s = 0; s < NSP; s++) ya[s] = y[NSP * i + s] * p.scale[NSP * i + s];
    chem_temperature_near(cc, gamma_tabs(gl), ya, T, dT);
    tdt[i] = make_double2(T, dT);
    double kr[NRATE], f[NSP];
#pragma unroll
    for (int r = 0; r < NRATE; r++) kr[r] = 0.0;
    chem_rates_only_pairs<0, C_BREM>(cc, T, kr);
    chem_rhs_species(ya, kr, f);
    double m = 0.0;
#pragma unroll
    for (int s = 0; s < NSP - 1; s++) {
      double v = f[s] * p.iscale[NSP * i + s] * srhs;
      if (force) v += force[NSP * i + s];
      v = fabs(v);
      m = v > m ? v : m;
    }
    const int kt = chem_bin(cc, chem_log(T > cc.tmin ? (T < cc.tmax ? T : cc.tmax) : cc.tmin)) >> 3;
    const int k = kt * TORD_RC + tord_rate_class(h * m);
    key[i] = (unsigned short)k;
    atomicAdd(&hc[k], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < TORD_NBK; e += blockDim.x)
    if (hc[e]) atomicAdd(&cnt[e * TORD_PAD], hc[e]);
}

// order[start of bucket k + reserved range of this block + local rank] = cell. Each block
// takes the exclusive prefix of the bucket totals, ranks its cells per bucket in LDS and
// reserves one range per bucket from the running counters (zeroed beforehand).
constexpr int TORD_BLOCK = 1024;
static_assert(TORD_NBK == 2 * TORD_BLOCK, "the scan below gives each thread two buckets");
__global__ void __launch_bounds__(TORD_BLOCK)
tord_scatter(long n, const unsigned short *key, int *cnt, int *order) {
  __shared__ int pre[TORD_NBK], hc[TORD_NBK], res[TORD_NBK], wsum[TORD_BLOCK / 64];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const int a = cnt[(2 * t) * TORD_PAD], b = cnt[(2 * t + 1) * TORD_PAD];
  hc[2 * t] = 0;
  hc[2 * t + 1] = 0;
  // inclusive scan of the pair sums: within each wave by shuffles, then over the waves'
  // totals by the first wave
  int v = a + b;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  if (lane == 63) wsum[wid] = v;
  __syncthreads();
  if (wid == 0) {
    int w = lane < TORD_BLOCK / 64 ? wsum[lane] : 0;
#pragma unroll
    for (int o = 1; o < TORD_BLOCK / 64; o <<= 1) {
      const int u = __shfl_up(w, o, 64);
      if (lane >= o) w += u;
    }
    if (lane < TORD_BLOCK / 64) wsum[lane] = w;
  }
  __syncthreads();
  const int ex = v + (wid > 0 ? wsum[wid - 1] : 0) - (a + b);   // totals of buckets < 2t
  pre[2 * t] = ex + a;                                     // inclusive prefix per bucket
  pre[2 * t + 1] = ex + a + b;
  const long i = (long)blockIdx.x * blockDim.x + t;
  int k = 0, r = 0;
  if (i < n) {
    k = key[i];
    r = atomicAdd(&hc[k], 1);
  }
  __syncthreads();
  for (int e = t; e < TORD_NBK; e += TORD_BLOCK)
    if (hc[e]) res[e] = atomicAdd(&cnt[(TORD_NBK + e) * TORD_PAD], hc[e]);
  __syncthreads();
  if (i < n) order[(k ? pre[k - 1] : 0) + res[k] + r] = (int)i;
}

using DirkKernel = void (*)(long, ChemConst, ChemPtrsD, DirkDev, double, double *, const double *,
                            const int *, const double2 *, int *, int *, int, double *, int);

template <bool FORCED, bool SUBSTEP>
static DirkKernel dirk_kernel(bool wide, int mem) {
  if (wide)
    return mem == MEM_RATES    ? chem_dirk_batched<FORCED, SUBSTEP, true, MEM_RATES>
           : mem == MEM_STAGES ? chem_dirk_batched<FORCED, SUBSTEP, true, MEM_STAGES>
                               : chem_dirk_batched<FORCED, SUBSTEP, true, MEM_SHARED>;
  return mem == MEM_RATES ? chem_dirk_batched<FORCED, SUBSTEP, false, MEM_RATES>
                          : chem_dirk_batched<FORCED, SUBSTEP, false, MEM_SHARED>;
}

static DirkKernel dirk_kernel(bool forced, bool sub, bool wide, int mem) {
  if (forced) return sub ? dirk_kernel<true, true>(wide, mem) : dirk_kernel<true, false>(wide, mem);
  return sub ? dirk_kernel<false, true>(wide, mem) : dirk_kernel<false, false>(wide, mem);
}

// Launch plan of one batched step: kernel variant, block after the LDS split, grid, and the
// layout of its work buffer (per-block statistics rows | cell order | bucket totals and
// running offsets | keys | temperatures at y_n).
struct BatchedPlan {
  DirkKernel kern;
  int block, wpb, chunk, mem;
  long grid, nrow;
  bool sorted;
  size_t b_rows, b_ord, b_cnt, b_key, b_tdt, b_fst;
  size_t bytes() const { return b_rows + b_ord + b_cnt + b_key + b_tdt + b_fst; }
};

// max_rows: the most blocks (statistics rows) the caller has room for (0: any number).
static int batched_plan(long n, const DirkDev &o, int grid_waves, int block, bool forced,
                        int nsteps, BatchedPlan &p, long max_rows = 0) {
  if (n <= 0 || n > (1L << 30)) return -1;
  if (block != 64 && block != 128 && block != 256) return -1;
  if (o.nstage < 1 || o.nstage > MAXSTAGE) return -1;
  const bool sub = o.max_halvings > 0;
  const bool wide = dirk_wide(o.nstage, o.esdirk != 0);
  // LDS by the number of waves: one or two per CU leave room for more than four do.
  // 167 forced seven-stage steps of 4096 cells: 19.7 ms without, 17.0 (as many full waves),
  // 13.5 with MEM_RATES; one multirate slow step of 32^3 cells 31.0 -> 23.5 ms with
  // MEM_STAGES; one seven-stage step of 20000 cells 270 -> 192 us. (Before loads were
  // issued together and the temperature solve shortened: 11.7, 17.4 ms since.)
  int dev = 0, lim = 0, ncu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return -1;
  const long want = grid_waves > 0 ? grid_waves : 1;
  const long full = std::min<long>(want, (n + 63) / 64);   // waves with every lane taken
  p.mem = full <= ncu ? MEM_RATES : wide && full <= 2L * ncu ? MEM_STAGES : MEM_SHARED;
  // blocks whose LDS would not fit are split: the kernel's static LDS as compiled and the
  // device's per-block limit, both asked of the runtime
  for (;; p.mem = MEM_SHARED) {
    p.kern = dirk_kernel(forced, sub, wide, p.mem);
    hipFuncAttributes fa{};
    if (hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(p.kern)) != hipSuccess) return -1;
    p.block = fit_block(block, o.nstage, fa.sharedSizeBytes, (size_t)lim, wide, p.mem);
    // (MEM_STAGES in one-wave blocks would leave every second wave waiting for a CU)
    if (p.block != 0 && (p.mem != MEM_STAGES || p.block >= 128)) break;
    if (p.mem == MEM_SHARED) return -1;
  }
  p.wpb = p.block / 64;
  // Cells per wave and turn. Four waves share a block: 32 to 64, spread evenly over the waves
  // of the grid and the turns each of them takes, so that a batch that does not fill every
  // lane of the device's waves leaves fewer cells waiting for a wave's slowest one.
  // With more LDS per wave: full waves. Two neighbouring CUs share an instruction cache, and
  // waves that do run this long code 15% slower (4096 cells, 167 steps: 64 full waves 13.5 ms,
  // 128 half full ones 16.0). From half as many full waves as there are CUs on they share it
  // anyhow, and the cells are spread over one wave per CU (9000 cells, 40 forced SDIRK3
  // steps: 141 waves 3.85 ms, 256 waves 3.53). A single step of few cells, whose waves pull
  // their cells from memory for most of its time, takes 32 to a wave (1500 cells: 115 -> 111
  // us; 3000: 119 -> 122).
  const long spread = p.mem == MEM_SHARED                      ? want
                      : p.mem == MEM_RATES && 2 * full > ncu   ? std::min<long>(want, ncu)
                                                               : full;
  const long turns = (n + 64 * spread - 1) / (64 * spread);
  p.chunk = (int)((n + turns * spread - 1) / (turns * spread));
  if (p.chunk < 32) p.chunk = 32;
  if (p.mem != MEM_SHARED && full == spread && full < want)
    p.chunk = nsteps == 1 && n <= 32 * 64 ? 32 : 64;
  // full waves where spreading the cells would take more blocks than there are rows for
  if (max_rows && std::min<long>(want, (n + p.chunk - 1) / p.chunk) > max_rows * p.wpb)
    p.chunk = 64;
  const long chunks = (n + p.chunk - 1) / p.chunk;
  const long waves = want < chunks ? want : chunks;
  p.grid = (waves + p.wpb - 1) / p.wpb;
  p.nrow = p.grid;                                         // one statistics row per block
  p.sorted = n >= TORD_MIN;
  p.b_rows = align256((size_t)p.nrow * NSTAT * sizeof(int));
  p.b_ord = p.sorted ? align256((size_t)n * sizeof(int)) : 0;
  p.b_cnt = p.sorted ? align256((size_t)2 * TORD_NBK * TORD_PAD * sizeof(int)) : 0;
  p.b_key = p.sorted ? align256((size_t)n * sizeof(unsigned short)) : 0;
  p.b_tdt = p.sorted ? align256((size_t)n * sizeof(double2)) : 0;
  // stage derivatives of tables too long for LDS: one column per thread of the grid
  p.b_fst = wide && p.mem == MEM_SHARED
                ? align256((size_t)p.grid * p.block * (o.nstage - 1) * NSP * sizeof(double))
                : 0;
  return 0;
}

// Queue one planned step: the cell order (unless reused), the counters cleared, the
// persistent kernel (whose last block sums the statistics into counters[1..NSTAT]). work
// holds p.bytes(); counters 2 + NSTAT ints (the work-queue position, the statistics, the
// kernel's finishing ticket).
static int batched_enqueue(const BatchedPlan &p, ChemState &s, const DirkDev &o, double h,
                           double *y, const double *force, bool reuse_order, char *work,
                           int *counters, hipStream_t st, int nsteps = 1) {
  const long n = s.n;
  int *rows = (int *)(work);
  int *order = p.sorted ? (int *)(work + p.b_rows) : nullptr;
  double2 *tdt = nullptr;                                  // temperatures at y_n, if solved
  if (p.sorted && !reuse_order) {
    int *cnt = (int *)(work + p.b_rows + p.b_ord);
    unsigned short *key = (unsigned short *)(work + p.b_rows + p.b_ord + p.b_cnt);
    tdt = (double2 *)(work + p.b_rows + p.b_ord + p.b_cnt + p.b_key);
    hipLaunchKernelGGL(zero_two, dim3(2 * TORD_NBK * TORD_PAD / 256), dim3(256), 0, st,
                       (long)(2 * TORD_NBK * TORD_PAD), cnt, (long)(2 + NSTAT), counters);
    const unsigned cb = (unsigned)((n + TORD_CBLOCK - 1) / TORD_CBLOCK);
    hipLaunchKernelGGL(tord_count, dim3(cb), dim3(TORD_CBLOCK), 0, st, n, s.cc, ptrs_d(s),
                       (const double *)y, force, h, o.rhs_scale, key, cnt, tdt);
    const unsigned tb = (unsigned)((n + TORD_BLOCK - 1) / TORD_BLOCK);
    hipLaunchKernelGGL(tord_scatter, dim3(tb), dim3(TORD_BLOCK), 0, st, n,
                       (const unsigned short *)key, cnt, order);
  }
  if (!(p.sorted && !reuse_order))   // (else cleared with the bucket counters above)
    hipLaunchKernelGGL(fill_int, dim3(1), dim3(64), 0, st, (long)(2 + NSTAT), counters, 0);
  const unsigned lds = (unsigned)dirk_lds_bytes(p.wpb, o.nstage, dirk_wide(o.nstage, o.esdirk != 0), p.mem);
  const bool sub = o.max_halvings > 0;
  double *fglob =
      p.b_fst ? (double *)(work + p.b_rows + p.b_ord + p.b_cnt + p.b_key + p.b_tdt) : nullptr;
  hipLaunchKernelGGL(p.kern, dim3((unsigned)p.grid), dim3(p.block), lds, st, n, s.cc,
                     ptrs_d(s), o, h, y, force, (const int *)order,
                     sub ? nullptr : (const double2 *)tdt, counters, rows, nsteps, fglob,
                     p.chunk);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int dirk_batched_launch(ChemState &s, const DirkDev &o, double h, double *y, hipStream_t st,
                        int grid_waves, int block, const double *force, bool reuse_order,
                        int nsteps) {
  if (nsteps < 1) return -1;
  BatchedPlan p;
  if (batched_plan(s.n, o, grid_waves, block, force != nullptr, nsteps, p)) return -1;
  const void *work0 = s.work;
  if (ensure_work(s, p.bytes())) return -1;
  if (s.work != work0) reuse_order = false;                // a new buffer holds no order
  return batched_enqueue(p, s, o, h, y, force, reuse_order, (char *)s.work, s.counters, st,
                         nsteps);
}

// ------------------------------------------------------------------------------------
// Allocation-free batched step: the same kernels with their work buffer and counters in
// one file-scope device array per GPU instead of the context's lazily sized buffer, for
// callers that cannot allocate device memory (graph capture, tight serving loops). Each
// GPU holds its own copy for the life of the process; every call on a GPU uses that GPU's
// copy, so calls that overlap on one GPU (other streams, other threads, other contexts)
// race and must not be issued. Everything a step needs to start from zero (bucket counters,
// work-queue position, statistics) is cleared by the step itself.
// ------------------------------------------------------------------------------------
constexpr size_t NOALLOC_COUNTERS = 256;                   // 2 + NSTAT ints, padded
constexpr size_t NOALLOC_WORK =
    align256((size_t)NOALLOC_MAX_ROWS * NSTAT * sizeof(int)) +
    align256((size_t)NOALLOC_MAX_CELLS * sizeof(int)) +
    align256((size_t)2 * TORD_NBK * TORD_PAD * sizeof(int)) +
    align256((size_t)NOALLOC_MAX_CELLS * sizeof(unsigned short)) +
    align256((size_t)NOALLOC_MAX_CELLS * sizeof(double2));
static __device__ __align__(256) unsigned char scratch[NOALLOC_COUNTERS + NOALLOC_WORK];

constexpr int NOALLOC_MAX_DEV = 64;
static std::mutex noalloc_mu;
static unsigned char *noalloc_ptr[NOALLOC_MAX_DEV] = {};

// The current device's address of `scratch`, looked up once per device (with that device
// current); nullptr on failure.
unsigned char *dirk_noalloc_scratch() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEV) return nullptr;
  std::lock_guard<std::mutex> lk(noalloc_mu);
  if (!noalloc_ptr[dev]) {
    void *a = nullptr;
    if (hipGetSymbolAddress(&a, HIP_SYMBOL(scratch)) != hipSuccess || !a) return nullptr;
    noalloc_ptr[dev] = (unsigned char *)a;
  }
  return noalloc_ptr[dev];
}

int dirk_batched_launch_noalloc(ChemState &s, const DirkDev &o, double h, double *y,
                                hipStream_t st, int grid_waves, int block, const double *force,
                                int **counters_out) {
  if (s.n > NOALLOC_MAX_CELLS) return MVD_BAD_ARGUMENT;
  if (dirk_wide(o.nstage, o.esdirk != 0)) return MVD_UNSUPPORTED;   // no room for its stage buffer
  BatchedPlan p;
  if (batched_plan(s.n, o, grid_waves, block, force != nullptr, 1, p, NOALLOC_MAX_ROWS)) return -1;
  if (p.nrow > NOALLOC_MAX_ROWS || p.bytes() > NOALLOC_WORK) return MVD_BAD_ARGUMENT;
  unsigned char *base = dirk_noalloc_scratch();
  if (!base) return -1;
  int *counters = (int *)base;
  *counters_out = counters;
  return batched_enqueue(p, s, o, h, y, force, false, (char *)(base + NOALLOC_COUNTERS),
                         counters, st);
}

int dirk_plain_run(ChemState &s, const DirkDev &o, double h, double *y, hipStream_t st) {
  const long n = s.n;
  if (n <= 0 || n > (1L << 30)) return -1;
  // scratch: yn, z, f, r, F[MAXSTAGE-1], LU blocks, rate estimate, last correction norm |
  // pivots | active, iters, setups, failed, counts | per-wave statistics rows
  const size_t b_dbl = align256(((size_t)n * NSP * (4 + (MAXSTAGE - 1)) + (size_t)n * NSP * NSP +
                                 (size_t)2 * n) * sizeof(double));
  const size_t b_piv = align256((size_t)n * sizeof(unsigned long long));
  const size_t b_int = align256(((size_t)n * 4 + 64) * sizeof(int));
  const long nrow = (n + 63) / 64;
  const size_t b_rows = align256((size_t)nrow * NSTAT * sizeof(int));
  if (ensure_work(s, b_dbl + b_piv + b_int + b_rows)) return -1;
  char *w = (char *)s.work;
  double *yn = (double *)w, *z = yn + n * NSP, *f = z + n * NSP, *r = f + n * NSP;
  double *acc = r + n * NSP, *LU = acc + (long)(MAXSTAGE - 1) * n * NSP;
  double *crate = LU + (long)NSP * NSP * n, *delp = crate + n;
  unsigned long long *piv = (unsigned long long *)(w + b_dbl);
  int *active = (int *)(w + b_dbl + b_piv), *iters = active + n, *csetups = iters + n,
      *failed = csetups + n, *nact = failed + n;
  int *rows = (int *)(w + b_dbl + b_piv + b_int);
  const ChemPtrsD p = ptrs_d(s);
  hipLaunchKernelGGL(copy_double, dim3(nb(n * NSP)), dim3(256), 0, st, n * NSP, y, yn);
  hipLaunchKernelGGL(copy_double, dim3(nb(n * NSP)), dim3(256), 0, st, n * NSP, y, z);
  // iters, setups, failed are contiguous
  hipLaunchKernelGGL(fill_int, dim3(nb(3 * n)), dim3(256), 0, st, 3 * n, iters, 0);
  hipLaunchKernelGGL(fill_int, dim3(nb(n)), dim3(256), 0, st, n, active, 1);
  // temperature at y_n, Jacobian at y_n, factor (the first stage's a_ii)
  hipLaunchKernelGGL(plain_rhs, dim3(nb(n)), dim3(256), 0, st, n, s.cc, p, o.rhs_scale, z, f,
                     active, PLAIN_UNCONVERGED);
  // an explicit first stage (ESDIRK) keeps that RHS as F_0
  if (o.esdirk)
    hipLaunchKernelGGL(copy_double, dim3(nb(n * NSP)), dim3(256), 0, st, n * NSP,
                       (const double *)f, acc);
  hipLaunchKernelGGL(plain_jac, dim3(nb(n)), dim3(256), 0, st, n, s.cc, p, h * o.gamma,
                     o.rhs_scale, z, LU, active);
  hipLaunchKernelGGL(plain_getrf, dim3(nb(n)), dim3(256), 0, st, n, LU, piv, active);
  hipLaunchKernelGGL(count_setups, dim3(nb(n)), dim3(256), 0, st, n, active, csetups);
  hipLaunchKernelGGL(plain_resume, dim3(nb(n)), dim3(256), 0, st, n, active, crate);
  int *hcnt = s.host_counters;
  bool fresh = true;              // f holds the RHS at the iterate y_n (the setup's evaluation)
  for (int stg = o.esdirk ? 1 : 0; stg < o.nstage; stg++) {
    const double hg = h * o.A[stg * MAXSTAGE + stg];
    hipLaunchKernelGGL(plain_stage_init, dim3(nb(n)), dim3(256), 0, st, n, stg, h, o, yn, acc, r,
                       active, failed);
    int setups = 0;
    for (;;) {
      bool all_done = false;
      hipLaunchKernelGGL(fill_int, dim3(1), dim3(64), 0, st, 2L, nact, 0);
      for (int it = 0; it < o.max_iters; it++) {
        if (!fresh)
          hipLaunchKernelGGL(plain_rhs, dim3(nb(n)), dim3(256), 0, st, n, s.cc, p, o.rhs_scale,
                             z, f, active, PLAIN_ITERATING);
        fresh = false;
        hipLaunchKernelGGL(fill_int, dim3(1), dim3(64), 0, st, 1L, nact, 0);
        hipLaunchKernelGGL(plain_newton, dim3(nb(n)), dim3(256), 0, st, n, hg, o, LU, piv, f, r,
                           z, active, iters, crate, delp, it, nact);
        // convergence test on the host, as the reference's Newton loop does: stop when no
        // cell iterates; done when none diverged either
        if (hipMemcpyAsync(hcnt, nact, 2 * sizeof(int), hipMemcpyDeviceToHost, st) !=
                hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
          return -1;
        if (hcnt[0] == 0) { all_done = hcnt[1] == 0; break; }
      }
      if (all_done) break;
      if (++setups > o.max_setups) {
        hipLaunchKernelGGL(mark_failed, dim3(nb(n)), dim3(256), 0, st, n, active, failed);
        break;
      }
      hipLaunchKernelGGL(plain_rhs, dim3(nb(n)), dim3(256), 0, st, n, s.cc, p, o.rhs_scale, z, f,
                         active, PLAIN_UNCONVERGED);
      hipLaunchKernelGGL(plain_jac, dim3(nb(n)), dim3(256), 0, st, n, s.cc, p, hg, o.rhs_scale,
                         z, LU, active);
      hipLaunchKernelGGL(plain_getrf, dim3(nb(n)), dim3(256), 0, st, n, LU, piv, active);
      hipLaunchKernelGGL(count_setups, dim3(nb(n)), dim3(256), 0, st, n, active, csetups);
      hipLaunchKernelGGL(plain_resume, dim3(nb(n)), dim3(256), 0, st, n, active, crate);
    }
    if (stg + 1 < o.nstage)
      hipLaunchKernelGGL(plain_stage_finish, dim3(nb(n)), dim3(256), 0, st, n, stg, hg, z, r,
                         acc);
  }
  hipLaunchKernelGGL(copy_double, dim3(nb(n * NSP)), dim3(256), 0, st, n * NSP, z, y);
  hipLaunchKernelGGL(plain_finish, dim3(nb(n)), dim3(256), 0, st, n, (const int *)iters,
                     (const int *)csetups, (const int *)failed, rows);
  hipLaunchKernelGGL(fill_int, dim3(1), dim3(64), 0, st, (long)(1 + NSTAT), s.counters, 0);
  hipLaunchKernelGGL(stats_reduce, dim3(stats_blocks(nrow)), dim3(256), 0, st,
                     (const int *)rows, nrow, s.counters + 1);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------------
// Block linear solver of the chemistry subvector: the Setup/Solve of
// SUNLinSol_RankLocalLS (multirate_chem_hydro_main.cpp:1348-1411) over MAGMA's batched
// getrf/getrs. Setup forms A = I - gamma J per cell from the dense column-major blocks
// (DENSEIDX(b,r,c) = 100b + 10c + r) and factors it with partial pivoting (first maximum,
// LAPACK row interchanges); Solve applies the factors to one right-hand side per cell
// ([cell][10], x may alias b). A block whose U has an exact zero on the diagonal counts as
// singular, as getrf's info > 0.
// ---------------------------------------------------------------------------------
// The factors are kept wave by wave, element-major ([wave][10 q + r][lane]): setup stores
// and solve loads them straight from registers, 512 contiguous bytes per access. The caller's
// blocks come in through LDS (blk_load). Both are bound by that traffic: 64^3 cells, setup
// (1608 bytes per cell) 141 -> 89 us, solve (968 bytes) 165 -> 50 us.
__global__ void __launch_bounds__(64)
ls_setup_kernel(long n, double gamma, const double *J, double *LU, unsigned long long *piv,
                int *nsing, bool formed) {
#pragma clang fp contract(off)
  __shared__ double lds[BLK_LDS];
  const long base = (long)blockIdx.x * 64;
  const int ncell = (int)min(n - base, 64L), lane = threadIdx.x;
  double a[NSP][NSP];
#pragma unroll
  for (int r = 0; r < NSP; r++)
#pragma unroll
    for (int q = 0; q < NSP; q++) a[r][q] = r == q ? 1.0 : 0.0;
  blk_load(J + (long)BLK * base, ncell, lds, a);
  if (lane >= ncell) return;
  if (!formed) {
#pragma unroll
    for (int q = 0; q < NSP; q++)
#pragma unroll
      for (int r = 0; r < NSP; r++) a[r][q] = (r == q ? 1.0 : 0.0) - gamma * a[r][q];
  }
  piv[base + lane] = lu_factor_regs<false>(a);
  bool sing = false;
  double *o = LU + (long)BLK * base + lane;
#pragma unroll
  for (int q = 0; q < NSP; q++) {
    sing |= a[q][q] == 0.0;
#pragma unroll
    for (int r = 0; r < NSP; r++) o[(NSP * q + r) * 64] = a[r][q];
  }
  if (sing) atomicAdd(nsing, 1);
}

__global__ void __launch_bounds__(64)
ls_solve_kernel(long n, const double *LU, const unsigned long long *piv, const double *b,
                double *x) {
#pragma clang fp contract(off)
  const long i = (long)blockIdx.x * 64 + threadIdx.x;
  if (i >= n) return;
  // every factor is loaded before the substitutions start
  const double *p = LU + (long)BLK * 64 * blockIdx.x + threadIdx.x;
  double a[NSP][NSP], v[NSP];
#pragma unroll
  for (int q = 0; q < NSP; q++)
#pragma unroll
    for (int r = 0; r < NSP; r++) a[r][q] = p[(NSP * q + r) * 64];
#pragma unroll
  for (int s = 0; s < NSP; s++) v[s] = b[NSP * i + s];
  lu_exchange(piv[i], v);
#pragma unroll
  for (int r = 1; r < NSP; r++)
#pragma unroll
    for (int q = 0; q < r; q++) v[r] -= a[r][q] * v[q];
#pragma unroll
  for (int r = NSP - 1; r >= 0; r--) {
#pragma unroll
    for (int q = r + 1; q < NSP; q++) v[r] -= a[r][q] * v[q];
    v[r] /= a[r][r];
  }
#pragma unroll
  for (int s = 0; s < NSP; s++) x[NSP * i + s] = v[s];
}

int chem_ls_setup(long n, double gamma, const double *J, double *LU, unsigned long long *piv,
                  int *nsing, hipStream_t st, bool formed) {
  hipLaunchKernelGGL(fill_int, dim3(1), dim3(64), 0, st, 1L, nsing, 0);
  hipLaunchKernelGGL(ls_setup_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, n, gamma, J,
                     LU, piv, nsing, formed);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int chem_ls_solve(long n, const double *LU, const unsigned long long *piv, const double *b,
                  double *x, hipStream_t st) {
  hipLaunchKernelGGL(ls_solve_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, n, LU, piv,
                     b, x);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------------
// Checkpointed discrete adjoint of nsteps DIRK steps (no counterpart in the reference; for
// sensitivity drivers): lam0 = (d y_N / d y_0)^T lamT, per cell, for the stage equations
// solved exactly along the computed trajectory. One thread per cell:
//   forward  - advances the cell nsteps steps with the per-cell step below, storing
//              (y, Ts, dTs) every K steps;
//   backward - segment by segment, last first: recomputes the segment's steps from its
//              checkpoint, keeping every step's stage values Y_k and end temperature in
//              scratch, then walks them backwards; the exact stage Jacobians
//              J_k = s_rhs dF/dy(Y_k) (rows from the exact vector-Jacobian product of the
//              RHS, its cotangent-independent part formed once per stage) enter
//                for k = s..1: Ybar_k = h J_k^T (b_k lam + sum_{m>k} a_mk nu_m),
//                              nu_k = (I - h a_kk J_k)^{-T} Ybar_k;   lam += sum_k nu_k,
//              b = the last row of A (the stiffly accurate tables of mvd_chem_dirk_step).
// The per-cell step is the plain solver's algorithm (modified Newton, J at y_n, refactor
// after max_iters), thread-local, so that recomputation repeats the forward run bit for bit.
// Scratch per cell (element-major, coalesced): nckpt x 12 + K x (nstage x 10 + 1) doubles, the
// second part twice where pairs of waves run (adj_pipe).
// A wave's steps are one long dependent chain at one wave per SIMD, so what shortens it is work
// taken out or handed to an idle SIMD: gamma tables, scales and stage derivatives in LDS, the last
// segment kept by the forward run instead of recomputed, and for small batches a second
// wave that recomputes ahead of the backward walk. 32^3 cells, 20 steps, K = 5: forward 1.02 ->
// 0.79 ms, backward 2.43 -> 0.92 ms (1.05 with the nu_k in registers, which spilled); with one
// loop over the stages and the table loads issued together 0.57 and 0.68 ms.
// ---------------------------------------------------------------------------------

// a_{row,col} of an adjoint table, both uniform in the wave (scalar selects; see dirk_coef)
__device__ inline double adj_coef(const DirkDev &o, int row, int col) {
  double v = 0.0;
#pragma unroll
  for (int r = 0; r < ADJ_MAXSTAGE; r++)
#pragma unroll
    for (int q = 0; q <= r; q++)
      if (r == row && q == col) v = o.A[r * MAXSTAGE + q];
  return v;
}

// One step of the lane's cell. Fl: y_n, then the stage derivatives but the last; a stage's
// right-hand side r lies where its own F will (the last of four stages: where F_0 was, which
// r has consumed), a step's first correction across the matrix set-up where F_1 will. One loop
// over all stages and iterations with one RHS evaluation, one matrix and one solve in it, the
// cells of a wave changing stage together (chem_dirk_batched): unrolled over the stages the
// two adjoint kernels had 113 and 207 KB of code, and two CUs share 64 KB of instruction cache.
__device__ inline bool cell_step(const ChemConst &cc, const GammaTabs &gt, const CellIn &c,
                                 double &Ts, double &dTs, const DirkDev &o, double h,
                                 double (&y)[NSP], double *Fl, double *Ys, long n, long i) {
#pragma clang fp contract(on)
  double z[NSP], a[NSP][NSP];
  unsigned long long pv = 0;
#pragma unroll
  for (int s = 0; s < NSP; s++) {
    z[s] = y[s];
    Fl[s * 64] = y[s];
    Fl[(NSP + s) * 64] = y[s];                        // r of the first stage
  }
  bool ok = true, solved = false, setup = true, start = true, busy = true;
  double crate = 1.0, delp = 0.0;                     // Newton rate estimate, last norm
  int setups = 0, it = 0;
#pragma unroll 1
  for (int st = 0;;) {
    const double hg = h * adj_coef(o, st, st);
    double *const rs = Fl + (st + 1 < ADJ_MAXSTAGE ? st + 1 : 1) * NSP * 64;
    if (busy) {
      double f[NSP];
      cell_rhs<true>(cc, gt, c, Ts, dTs, z, o.rhs_scale, f, !solved);
      solved = false;
      double d[NSP];
#pragma unroll
      for (int s = 0; s < NSP; s++) d[s] = -(z[s] - hg * f[s] - rs[s * 64]);
      bool update = true;
      if (setup) {
        if (start) {
#pragma unroll
          for (int s = 0; s < NSP; s++) Fl[(2 * NSP + s) * 64] = d[s];
        }
        cell_matrix_regs(cc, c, Ts, dTs, z, hg, o.rhs_scale, a, PairTable());
        pv = lu_factor_regs<true>(a);
        setup = false;
        crate = 1.0;
        it = 0;
        if (start) {
          __asm__ volatile("" ::: "memory");
#pragma unroll
          for (int s = 0; s < NSP; s++) {
            d[s] = Fl[(2 * NSP + s) * 64];
            z[s] = Fl[s * 64];
          }
        } else {
          solved = true;                              // the next pass evaluates f here again
          update = false;
        }
        start = false;
      }
      if (update) {
        lu_solve_regs(a, pv, d);
#pragma unroll
        for (int s = 0; s < NSP; s++) z[s] += d[s];
        const double del = wrms_norm(d, z, o.rtol, o.atol);
        if (it > 0) crate = conv_rate(crate, del, delp);
        const bool diverging = it > 0 && conv_diverging(del, delp);
        delp = del;
        it++;
        if (conv_ok(crate, del, o.ntol)) {
          busy = false;
        } else if (it >= o.max_iters || diverging) {
          setup = true;
          if (++setups > o.max_setups) ok = busy = false;
        }
      }
    }
    if (__builtin_amdgcn_ballot_w64(busy) != 0) continue;   // some cell of the wave iterates
    // all cells' stages ended. (One that failed, here or at an earlier stage of the step, keeps
    // its iterate and stops: its later stages store nothing.)
    if (setups >= 0) {
      double r[NSP];
#pragma unroll
      for (int s = 0; s < NSP; s++) r[s] = rs[s * 64];
      const double ihg = 1.0 / hg;
      if (st + 1 < ADJ_MAXSTAGE)
#pragma unroll
        for (int s = 0; s < NSP; s++) Fl[((st + 1) * NSP + s) * 64] = (z[s] - r[s]) * ihg;
      if (Ys)
#pragma unroll
        for (int s = 0; s < NSP; s++) Ys[(long)(st * NSP + s) * n + i] = z[s];
    }
    if (++st >= o.nstage) break;
    busy = ok;
    setups = ok ? 0 : -1;
    it = 0;
    if (__builtin_amdgcn_ballot_w64(busy) == 0) break;
    double acc[NSP], yn[NSP];
#pragma unroll
    for (int s = 0; s < NSP; s++) acc[s] = 0.0;
#pragma unroll
    for (int j = 0; j < ADJ_MAXSTAGE - 1; j++)
      if (j < st) {
        const double aj = adj_coef(o, st, j);
#pragma unroll
        for (int s = 0; s < NSP; s++) acc[s] += aj * Fl[((j + 1) * NSP + s) * 64];
      }
#pragma unroll
    for (int s = 0; s < NSP; s++) yn[s] = Fl[s * 64];
    double *const rn = Fl + (st + 1 < ADJ_MAXSTAGE ? st + 1 : 1) * NSP * 64;
#pragma unroll
    for (int s = 0; s < NSP; s++) rn[s * 64] = yn[s] + h * acc[s];
  }
#pragma unroll
  for (int s = 0; s < NSP; s++) y[s] = z[s];
  return ok;
}

constexpr int ADJ_REC = NSP + 2;     // y, Ts, dTs

// LDS of an adjoint block: the gamma tables, then scale and inv_scale of each group of 64 cells
// ([20][64]), which every RHS reads, y_n and the stage derivatives but the last
// ([10 ADJ_MAXSTAGE][64]). 63.5 KB for 64 cells, 156 KB for 256; a pair of waves adds 15 KB
// (two pairs per CU).
constexpr int ADJ_CELLS = (2 + ADJ_MAXSTAGE) * NSP * 64;

__device__ inline CellIn adj_cell(const ChemPtrsD &p, const ChemConst &cc, long i, int group,
                                  int part, double *lds) {
  for (int e = threadIdx.x; e < 4 * TLEN; e += blockDim.x) lds[e] = cc.tab[G_GH2_1 * TLEN + e];
  double *q = lds + 4 * TLEN + group * ADJ_CELLS + (threadIdx.x & 63);
  if (part == 0) {
#pragma unroll
    for (int s = 0; s < NSP; s++) {
      q[s * 64] = p.scale[NSP * i + s];
      q[(NSP + s) * 64] = p.iscale[NSP * i + s];
    }
  }
  __syncthreads();
  return CellIn{q, q + NSP * 64, 64, CellAux{p.md[i], p.imd[i], p.cie[i], p.h2o[i]}};
}

__global__ void __launch_bounds__(256)
chem_adjoint_forward(long n, ChemConst cc, ChemPtrsD p, DirkDev o, double h, int nsteps, int K,
                     const int *order, double *y, double *ck, double *Te, double *Ys, int *nfail) {
  extern __shared__ double lds[];
  // thread u takes the u-th cell of the temperature order; scratch is indexed by u
  const long u0 = (long)blockIdx.x * blockDim.x + threadIdx.x, u = min(u0, n - 1);
  const long i = order ? order[u] : u;
  const CellIn c = adj_cell(p, cc, i, threadIdx.x >> 6, 0, lds);
  const GammaTabs gt = gamma_tabs(lds);
  double *Fl = lds + 4 * TLEN + (threadIdx.x >> 6) * ADJ_CELLS + 2 * NSP * 64 + (threadIdx.x & 63);
  if (u0 >= n) return;
  const int last = (nsteps - 1) / K * K;       // first step of the last segment
  double Ts = p.Ts[i], dTs = p.dTs[i];
  double z[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) z[s] = y[NSP * i + s];
  bool ok = true;
  for (int st = 0; st < nsteps; st++) {
    if (st % K == 0) {
      double *rec = ck + (long)(st / K) * ADJ_REC * n;
#pragma unroll
      for (int s = 0; s < NSP; s++) rec[s * n + u] = z[s];
      rec[NSP * n + u] = Ts;
      rec[(NSP + 1) * n + u] = dTs;
    }
    double *Yst = st >= last ? Ys + (long)(st - last) * o.nstage * NSP * n : nullptr;
    ok = cell_step(cc, gt, c, Ts, dTs, o, h, z, Fl, Yst, n, u) && ok;
    if (Yst) Te[(long)(st - last) * n + u] = Ts;
  }
#pragma unroll
  for (int s = 0; s < NSP; s++) y[NSP * i + s] = z[s];
  p.Ts[i] = Ts;
  p.dTs[i] = dTs;
  if (!ok) atomicAdd(nfail, 1);
}

// M^T = (I - hg J)^T of one stage from the exact Jacobian rows at the scaled state Y
// (temperature solved from the warm start T); also yb = h J^T w.
__device__ inline void stage_adjoint_matrix(const ChemConst &cc, const GammaTabs &gt, const CellIn &c,
                                            double T,
                                            const double (&Y)[NSP], double srhs, double h,
                                            double hg, const double (&w)[NSP],
                                            double (&Mt)[NSP][NSP], double (&yb)[NSP]) {
#pragma clang fp contract(on)
  double ya[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) ya[s] = Y[s] * c.s(s);
  double dT;
  chem_temperature(cc, gt, ya, T, dT);
  const bool clamped = !(T > cc.tmin && T < cc.tmax);
  ChemVjpPre P;                  // rates, gas-energy tangents, temperature path: once
  chem_vjp_prepare(cc, ya, T, clamped, c.ax, P);
  double acc[NSP];
#pragma unroll
  for (int q = 0; q < NSP; q++) acc[q] = 0.0;
#pragma unroll
  for (int r = 0; r < NSP; r++) {
    // row r of the RHS Jacobian in scaled variables: the VJP of the cotangent is(r) e_r
    // (times inv_mdensity on the gas-energy row)
    double row[NSP];
    chem_vjp_row(P, ya, r, r == NSP - 1 ? c.is(r) * c.ax.inv_mdensity : c.is(r), row);
#pragma unroll
    for (int q = 0; q < NSP; q++) {
      const double J = row[q] * c.s(q);                 // scaled dF_r/dy_q
      acc[q] += (srhs * J) * w[r];
      Mt[q][r] = (q == r ? 1.0 : 0.0) - hg * (srhs * J);
    }
  }
#pragma unroll
  for (int q = 0; q < NSP; q++) yb[q] = h * acc[q];
}

// One segment's steps from its checkpoint: stage values and end temperatures.
__device__ inline void adj_recompute(const ChemConst &cc, const GammaTabs &gt, const CellIn &c,
                                     const DirkDev &o, double h, int nst, double *Fl,
                                     const double *rec, double *Te, double *Ys, long n, long u) {
  double z[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) z[s] = rec[s * n + u];
  double Ts = rec[NSP * n + u], dTs = rec[(NSP + 1) * n + u];
  for (int st = 0; st < nst; st++) {
    (void)cell_step(cc, gt, c, Ts, dTs, o, h, z, Fl, Ys + (long)st * o.nstage * NSP * n, n, u);
    Te[(long)st * n + u] = Ts;   // the warm start of the step's stage solves
  }
}

// One segment's steps backwards. Nl: the nu_k of the stages but the first, as Fl.
__device__ inline void adj_backward(const ChemConst &cc, const GammaTabs &gt, const CellIn &c,
                                    const DirkDev &o, double h, int nst, double *Nl,
                                    const double *Te, const double *Ys, long n, long u, double (&lam)[NSP]) {
#pragma clang fp contract(on)
  const int ns = o.nstage;
  for (int st = nst - 1; st >= 0; st--) {
    const double Ts = Te[(long)st * n + u];
    const double *Yst = Ys + (long)st * ns * NSP * n;
    double nu[NSP];                                   // of the stage at hand; nu_0 at the end
#pragma unroll 1
    for (int k = ns - 1; k >= 0; k--) {
      double w[NSP], Y[NSP];
#pragma unroll
      for (int s = 0; s < NSP; s++) Y[s] = Yst[(long)(k * NSP + s) * n + u];
      const double bk = adj_coef(o, ns - 1, k);
#pragma unroll
      for (int s = 0; s < NSP; s++) w[s] = bk * lam[s];
#pragma unroll
      for (int m = 1; m < ADJ_MAXSTAGE; m++)
        if (m > k && m < ns) {
          const double am = adj_coef(o, m, k);
#pragma unroll
          for (int s = 0; s < NSP; s++) w[s] += am * Nl[((m - 1) * NSP + s) * 64];
        }
      double Mt[NSP][NSP];
      stage_adjoint_matrix(cc, gt, c, Ts, Y, o.rhs_scale, h, h * adj_coef(o, k, k), w, Mt, nu);
      const unsigned long long pv = lu_factor_regs<true>(Mt);
      lu_solve_regs(Mt, pv, nu);
      if (k > 0)
#pragma unroll
        for (int s = 0; s < NSP; s++) Nl[((k - 1) * NSP + s) * 64] = nu[s];
    }
#pragma unroll
    for (int s = 0; s < NSP; s++) lam[s] += nu[s];
#pragma unroll 1
    for (int k = 1; k < ns; k++)
#pragma unroll
      for (int s = 0; s < NSP; s++) lam[s] += Nl[((k - 1) * NSP + s) * 64];
  }
}

// The last segment's stage values are there already (chem_adjoint_forward keeps them).
// PIPE: two waves per 64 cells, one walking segment sg backwards while the other recomputes
// segment sg-1 into the second half of Te and Ys (blocks of 128 threads).
template <bool PIPE>
__global__ void __launch_bounds__(PIPE ? 128 : 256)
chem_adjoint_backward(long n, ChemConst cc, ChemPtrsD p, DirkDev o, double h, int nsteps, int K,
                      const int *order, const double *ck, double *Te, double *Ys,
                      const double *lamT, double *lam0) {
  extern __shared__ double lds[];
  const int role = PIPE ? threadIdx.x >> 6 : 0;
  const long u0 = PIPE ? (long)blockIdx.x * 64 + (threadIdx.x & 63)
                       : (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long u = min(u0, n - 1);                   // as in chem_adjoint_forward
  const long i = order ? order[u] : u;
  const CellIn c = adj_cell(p, cc, i, PIPE ? 0 : threadIdx.x >> 6, role, lds);
  const GammaTabs gt = gamma_tabs(lds);
  double *Fl = lds + 4 * TLEN + (PIPE ? 0 : threadIdx.x >> 6) * ADJ_CELLS + 2 * NSP * 64 +
               (threadIdx.x & 63);
  double *Nl = PIPE ? lds + 4 * TLEN + ADJ_CELLS + (threadIdx.x & 63) : Fl;
  if (!PIPE && u0 >= n) return;                    // (spare lanes of a pair stay for the barriers)
  double lam[NSP];
#pragma unroll
  for (int s = 0; s < NSP; s++) lam[s] = lamT[NSP * i + s];
  const int nseg = (nsteps + K - 1) / K;
  const auto steps_of = [&](int sg) { return min(K, nsteps - sg * K); };
  const long half = (long)K * n, halfY = half * o.nstage * NSP;
  for (int sg = nseg - 1; sg >= 0; sg--) {
    if (PIPE) {
      if (role == 0) {
        if (sg > 0 && u0 < n)
          adj_recompute(cc, gt, c, o, h, K, Fl, ck + (long)(sg - 1) * ADJ_REC * n,
                        Te + ((sg - 1) & 1) * half, Ys + ((sg - 1) & 1) * halfY, n, u);
      } else if (u0 < n) {
        adj_backward(cc, gt, c, o, h, steps_of(sg), Nl, Te + (sg & 1) * half, Ys + (sg & 1) * halfY,
                     n, u, lam);
      }
      __syncthreads();
    } else {
      if (sg < nseg - 1)
        adj_recompute(cc, gt, c, o, h, K, Fl, ck + (long)sg * ADJ_REC * n, Te, Ys, n, u);
      adj_backward(cc, gt, c, o, h, steps_of(sg), Nl, Te, Ys, n, u, lam);
    }
  }
  if ((!PIPE || role == 1) && u0 < n)
#pragma unroll
    for (int s = 0; s < NSP; s++) lam0[NSP * i + s] = lam[s];
}

// Pairs of waves where the cells fill at most half of the SIMDs and there is something to
// recompute; the second set of stage values stays below 4 GiB.
static bool adj_pipe(long n, int nsteps, int K, int nstage) {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  return (n + 63) / 64 <= 2L * ncu && nsteps > K &&
         (double)n * K * (nstage * NSP + 1) * sizeof(double) < 4.0 * (1 << 30);
}

// Scratch: checkpoints | end temperatures | stage values | the cell order (order, keys,
// temperatures at y_0, bucket counters of the ordering pass).
static size_t adj_order_doubles(long n) {
  const size_t b = align256((size_t)n * sizeof(int)) + align256((size_t)n * sizeof(short)) +
                   align256((size_t)n * sizeof(double2)) +
                   align256((size_t)2 * TORD_NBK * TORD_PAD * sizeof(int));
  return (b + 256) / sizeof(double);     // (+ the alignment of its start)
}

size_t chem_adjoint_scratch_doubles(long n, int nsteps, int K, int nstage) {
  const long nckpt = (nsteps + K - 1) / K;
  const long sets = adj_pipe(n, nsteps, K, nstage) ? 2 : 1;
  return (size_t)n * (nckpt * ADJ_REC + sets * K * (nstage * NSP + 1)) + adj_order_doubles(n);
}

int chem_adjoint_run(ChemState &s, const DirkDev &o, double h, int nsteps, int K, double *y,
                     const double *lamT, double *lam0, double *scratch, hipStream_t st,
                     int *host_fail) {
  const long n = s.n;
  const long nckpt = (nsteps + K - 1) / K;
  const bool pipe = adj_pipe(n, nsteps, K, o.nstage);
  const long sets = pipe ? 2 : 1, keep = pipe ? (nckpt - 1) & 1 : 0;   // where the last segment lies
  double *ck = scratch, *Te = ck + nckpt * ADJ_REC * n, *Ys = Te + sets * K * n;
  const ChemPtrsD p = ptrs_d(s);
  int *nfail = s.counters;
  hipLaunchKernelGGL(fill_int, dim3(1), dim3(64), 0, st, 1L, nfail, 0);
  // cells in the batched step's order at y_0 (temperature bucket, rate class), so that the
  // cells of a wave take similar Newton paths; kept for the whole run
  int *order = nullptr;
  if (n >= TORD_MIN) {
    const uintptr_t a = (uintptr_t)(Ys + sets * K * o.nstage * NSP * n);
    char *w = (char *)((a + 255) & ~(uintptr_t)255);
    order = (int *)w;
    unsigned short *key = (unsigned short *)(w + align256((size_t)n * sizeof(int)));
    double2 *tdt = (double2 *)((char *)key + align256((size_t)n * sizeof(short)));
    int *cnt = (int *)((char *)tdt + align256((size_t)n * sizeof(double2)));
    hipLaunchKernelGGL(fill_int, dim3(2 * TORD_NBK * TORD_PAD / 256), dim3(256), 0, st,
                       (long)(2 * TORD_NBK * TORD_PAD), cnt, 0);
    hipLaunchKernelGGL(tord_count, dim3((unsigned)((n + TORD_CBLOCK - 1) / TORD_CBLOCK)),
                       dim3(TORD_CBLOCK), 0, st, n, s.cc, p, (const double *)y,
                       (const double *)nullptr, h, o.rhs_scale, key, cnt, tdt);
    hipLaunchKernelGGL(tord_scatter, dim3((unsigned)((n + TORD_BLOCK - 1) / TORD_BLOCK)),
                       dim3(TORD_BLOCK), 0, st, n, (const unsigned short *)key, cnt, order);
  }
  // one group of 64 cells per block while that spreads them over more CUs, else four
  const int groups = pipe || (n + 63) / 64 <= 512 ? 1 : 4;
  const unsigned nbk = (unsigned)((n + 64 * groups - 1) / (64 * groups));
  const size_t shmem = sizeof(double) * (4 * TLEN + groups * ADJ_CELLS);
  const size_t pairmem = sizeof(double) * (ADJ_MAXSTAGE - 1) * NSP * 64;   // Nl of a pair
  hipLaunchKernelGGL(chem_adjoint_forward, dim3(nbk), dim3(64 * groups), shmem, st, n, s.cc, p, o, h,
                     nsteps, K, (const int *)order, y, ck, Te + keep * K * n,
                     Ys + keep * K * o.nstage * NSP * n, nfail);
  if (pipe)
    hipLaunchKernelGGL(chem_adjoint_backward<true>, dim3(nbk), dim3(128), shmem + pairmem, st, n, s.cc, p, o,
                       h, nsteps, K, (const int *)order, (const double *)ck, Te, Ys, lamT, lam0);
  else
    hipLaunchKernelGGL(chem_adjoint_backward<false>, dim3(nbk), dim3(64 * groups), shmem, st, n,
                       s.cc, p, o, h, nsteps, K, (const int *)order, (const double *)ck, Te, Ys,
                       lamT, lam0);
  if (hipGetLastError() != hipSuccess) return -1;
  if (hipMemcpyAsync(host_fail, nfail, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return -1;
  return 0;
}

}  // namespace mvd
